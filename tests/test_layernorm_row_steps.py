"""Forward LayerNorm, a wave per row: 512 workgroups walk the rows in steps of one, two or four rows a wave, so what counts
is row counts on either side of a full step, and of the line where the rows per step change."""
import pytest
import torch

from _util import randn, ulp_distance

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("C,dtype", [(1024, BF16), (520, F16), (260, F32), (1600, BF16), (1032, F16), (1024, F32), (768, BF16), (512, BF16), (2056, BF16)])
@pytest.mark.parametrize("rows", [2049, 4096, 4097, 6145, 8191, 8193, 16385])
def test_row_steps(C, dtype, rows):
    from core_scheduler_amd import ops

    x, res = (randn((rows, C), 60 + i, dtype=dtype).cuda() for i in range(2))
    gamma, beta = randn(C, 62, 0.2, 1.0).cuda(), randn(C, 63, 0.2).cuda()
    total, y, mean, rstd = ops.add_layernorm_forward(x, res, gamma, beta)
    assert torch.equal(total, x + res)
    alone = ops.layernorm_forward(total, gamma, beta)
    assert all(torch.equal(a, b) for a, b in zip((y, mean, rstd), alone))
    t = total.double()
    mu = t.mean(1, keepdim=True)
    rs = (t.var(1, unbiased=False, keepdim=True) + 1e-5).rsqrt()
    # fp32 statistics: a mean of C terms, pairwise below 2^-18 of their size
    assert ((mean.double() - mu[:, 0]).abs() <= 1e-6).all() and ((rstd.double() / rs[:, 0] - 1).abs() <= 4e-6).all()
    want = (t - mu) * rs * gamma.double() + beta.double()
    ok = (y.double() - want).abs() <= 2e-5
    assert (ok if dtype == F32 else ok | (ulp_distance(y.cpu(), want.to(dtype).cpu()) <= 1).cuda()).all()


@pytest.mark.parametrize("C,dtype", [(264, F16), (512, BF16), (520, BF16), (640, F16), (1024, BF16), (132, F32), (260, F32), (512, F32)])
@pytest.mark.parametrize("rows", [1, 9, 512, 513, 2047, 2049, 4097])
def test_backward_a_wave_per_row(C, dtype, rows):
    """256 workgroups of eight waves, a row a wave and step: row counts on either side of a workgroup and of a step."""
    from core_scheduler_amd import ops

    x, dy, dres = (randn((rows, C), 70 + i, dtype=dtype).cuda() for i in range(3))
    gamma = randn(C, 73, 0.2, 1.0).cuda()
    _, mean, rstd = ops.layernorm_forward(x, gamma, gamma)
    mu, rs = mean.double()[:, None], rstd.double()[:, None]
    xh, d64 = (x.double() - mu) * rs, dy.double()
    g = d64 * gamma.double()
    want = rs * (g - g.mean(1, keepdim=True) - xh * (g * xh).mean(1, keepdim=True))
    dx, dgamma, dbeta = ops.layernorm_backward(dy, x, mean, rstd, gamma)
    # some ten fp32 roundings of terms of up to 40: 2^-24 * 10 * 40
    ok = (dx.double() - want).abs() <= 2.4e-5
    assert (ok if dtype == F32 else ok | (ulp_distance(dx.cpu(), want.to(dtype).cpu()) <= 1).cuda()).all()
    for got, terms in ((dgamma, d64 * xh), (dbeta, d64)):
        # x-hat in fp32 (2^-22 with its inputs' roundings), chains of up to 17 + 16 + 16 fp32 additions
        assert ((got.double() - terms.sum(0)).abs() <= 2.0 ** -18 * terms.abs().sum(0) + 1e-6).all()
    apart = ops.layernorm_backward(dy, x, mean, rstd, gamma, dresidual=dres)
    assert torch.equal(apart[0], dx + dres) and torch.equal(apart[1], dgamma) and torch.equal(apart[2], dbeta)
    chain = ops.LayerNormBackwardChain()
    one, two = (chain.backward(dy, x, mean, rstd, gamma, dresidual=dres) for _ in range(2))
    chain.flush()
    assert all(torch.equal(a, b) and torch.equal(a, c) for a, b, c in zip(apart, one, two))
