"""Wide LayerNorm rows of whole aligned vectors: workgroups walk rows in steps of two behind buffer descriptors, so what
counts is the number of steps (one, two, odd, even), lanes without a vector and rows past the last one."""
import pytest
import torch

from _util import randn, ulp_distance

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def guarded(t):
    """t on the GPU with 64 sevens on either side of it, and a check that they are still there."""
    flat = torch.full((t.numel() + 128,), 7.0, dtype=t.dtype, device="cuda")
    flat[64:-64].copy_(t.reshape(-1))
    return flat[64:-64].view(t.shape), lambda: (flat[:64] == 7).all() and (flat[-64:] == 7).all()


@pytest.mark.parametrize("C,dtype", [(2056, BF16), (2560, F16), (3592, BF16), (5120, BF16), (8192, F16), (1028, F32), (3076, F32), (4096, F32)])
@pytest.mark.parametrize("rows", [1, 255, 257, 512, 513, 769, 1025, 1281])
def test_steps(C, dtype, rows):
    from core_scheduler_amd import ops

    x, res, dy, dres = (randn((rows, C), 40 + i, dtype=dtype).cuda() for i in range(4))
    gamma, beta = randn(C, 44, 0.2, 1.0).cuda(), randn(C, 45, 0.2).cuda()
    gx, kept_x = guarded(x)
    total, y, mean, rstd = ops.add_layernorm_forward(gx, res, gamma, beta, inplace=True)
    assert kept_x() and torch.equal(total, x + res)
    assert all(torch.equal(a, b) for a, b in zip((y, mean, rstd), ops.layernorm_forward(total, gamma, beta)))
    t = total.double()
    mu = t.mean(1, keepdim=True)
    rs = (t.var(1, unbiased=False, keepdim=True) + 1e-5).rsqrt()
    xh = (t - mu) * rs
    # fp32 statistics: a mean of C terms, pairwise below 2^-18 of their size
    assert ((mean.double() - mu[:, 0]).abs() <= 1e-6).all() and ((rstd.double() / rs[:, 0] - 1).abs() <= 4e-6).all()

    def close(got, want, tol):
        ok = (got.double() - want).abs() <= tol
        return (ok if dtype == F32 else ok | (ulp_distance(got.cpu(), want.to(dtype).cpu()) <= 1).cuda()).all()

    assert close(y, xh * gamma.double() + beta.double(), 2e-5)
    g = dy.double() * gamma.double()
    want = rs * (g - g.mean(1, keepdim=True) - xh * (g * xh).mean(1, keepdim=True))
    dx, dgamma, dbeta = ops.layernorm_backward(dy, total, mean, rstd, gamma)
    assert close(dx, want, 2e-5)
    d64 = dy.double()
    for got, terms in ((dgamma, d64 * xh), (dbeta, d64)):
        # x-hat in fp32 (2^-22 with its inputs' roundings), sums of up to `rows` terms in fp32 where they ride in fp32
        assert ((got.double() - terms.sum(0)).abs() <= 2.0 ** -20 * terms.abs().sum(0) + 1e-6).all()
    apart = ops.layernorm_backward(dy, total, mean, rstd, gamma, dresidual=dres)
    assert torch.equal(apart[0], (dx + dres)) and torch.equal(apart[1], dgamma) and torch.equal(apart[2], dbeta)


@pytest.mark.parametrize("rows,C", [(513, 2056), (1281, 5120)])
def test_gradient_over_the_residuals(rows, C):
    """dx written over dresidual, as the residual stream's gradient is updated in place."""
    from core_scheduler_amd import _capi, ops

    x, dy, dres = (randn((rows, C), 50 + i, dtype=BF16).cuda() for i in range(3))
    gamma = randn(C, 53, 0.2, 1.0).cuda()
    _, mean, rstd = ops.layernorm_forward(x, gamma)
    want = ops.layernorm_backward(dy, x, mean, rstd, gamma, dresidual=dres)
    over, kept = guarded(dres)
    dgamma, dbeta = torch.empty_like(gamma), torch.empty_like(gamma)
    lib = _capi.load()
    size = lib.cs_layernorm_backward_workspace_bytes(rows, C)
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    code = lib.cs_layernorm_backward_add(dy.data_ptr(), x.data_ptr(), mean.data_ptr(), rstd.data_ptr(), gamma.data_ptr(),
                                         over.data_ptr(), over.data_ptr(), dgamma.data_ptr(), dbeta.data_ptr(), ws.data_ptr(),
                                         size, rows, C, _capi.BF16, _capi.BF16, _capi.BF16, _capi.F32, 0,
                                         torch.cuda.current_stream().cuda_stream)
    assert code == _capi.OK and kept()
    assert all(torch.equal(a, b) for a, b in zip((over, dgamma, dbeta), want))
