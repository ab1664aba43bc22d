"""Forward LayerNorm, a wave per row: 512 or 1024 workgroups walk the rows in steps of one, two or four rows a wave, so what counts
is row counts on either side of a full step, and of the lines where the rows per step and the workgroups change."""
import pytest
import torch

from _util import randn, ulp_distance

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("C,dtype", [(1024, BF16), (520, F16), (260, F32), (1600, BF16), (1032, F16), (1024, F32), (768, BF16), (512, BF16), (2056, BF16)])
@pytest.mark.parametrize("rows", [2049, 4096, 4097, 6145, 8191, 8193, 10241, 12289, 14337, 16385, 20481, 32769])
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
@pytest.mark.parametrize("rows", [1, 9, 512, 513, 2047, 2049, 4097, 10241, 24577])
def test_backward_a_wave_per_row(C, dtype, rows):
    """256 or, of many narrow rows, 512 workgroups of eight waves, a row a wave and step: row counts on either side of a
    workgroup, of a step and of the lines between the two."""
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


def _dx_in_fp32(dy, x, mean, rstd, gamma):
    """dx in fp32 as a wave forms it: 64 lanes of four columns, chains over a lane's columns, a tree over the lanes, the
    products dy * gamma unrounded in the last line.  (A fused multiply-add: the product of two floats is exact in 64 bits.)"""
    def fma(a, b, c):
        return (a.double() * b.double() + c.double()).float()

    def tree(t):
        while t.shape[1] > 1:
            t = t[:, 0::2] + t[:, 1::2]
        return t

    rows, C = x.shape
    xh = (x - mean[:, None]) * rstd[:, None]
    s1, s2 = (torch.zeros(rows, 64, device=x.device) for _ in range(2))
    for j in range(0, C, 256):
        for k in range(4):
            at = torch.arange(j + k, min(j + 256, C), 4)
            n = len(at)
            t = dy[:, at] * gamma[at]
            s1[:, :n] += t
            s2[:, :n] = fma(t, xh[:, at], s2[:, :n])
    s1, s2 = (tree(s) * torch.tensor(1.0 / C, dtype=torch.float32, device=x.device) for s in (s1, s2))
    return rstd[:, None] * fma(-xh, s2, fma(dy, gamma, -s1))


@pytest.mark.parametrize("C", [132, 200, 256, 396, 512])  # 33 to 64 vectors, and 97 to 128
@pytest.mark.parametrize("rows", [400, 2049])  # one launch with the sums, and two
@pytest.mark.parametrize("along", [0.0, 0.9, 0.999])
def test_dx_is_as_exact_as_its_formula(C, rows, along):
    """dy that lies along x-hat leaves little of dx, and what was rounded ahead of the subtraction shows."""
    from core_scheduler_amd import ops

    x, noise = (randn((rows, C), 75 + i).cuda() for i in range(2))
    gamma = randn(C, 77, 0.2, 1.0).cuda()
    _, mean, rstd = ops.layernorm_forward(x, gamma, gamma)
    rs = rstd.double()[:, None]
    xh = (x.double() - mean.double()[:, None]) * rs
    dy = (along * xh + (1 - along ** 2) ** 0.5 * noise.double()).float()
    g = dy.double() * gamma.double()
    want = rs * (g - g.mean(1, keepdim=True) - xh * (g * xh).mean(1, keepdim=True))
    dx = ops.layernorm_backward(dy, x, mean, rstd, gamma)[0]
    formula = _dx_in_fp32(dy, x, mean, rstd, gamma)

    def error(t):
        return (t.double() - want).pow(2).mean().sqrt().item()

    # (the product rounded, and rstd multiplied into the terms: 8 to 18% more where along is 0.9 or more)
    assert error(dx) <= 1.02 * error(formula)


@pytest.mark.parametrize("C,dtype", [(512, BF16), (1024, BF16), (520, F16), (132, F32), (400, F32)])
@pytest.mark.parametrize("rows", [1, 513, 4095, 4096, 4097, 8193, 20480, 20481])  # where the launch of dx alone changes
def test_dx_alone_has_the_bits_of_the_full_call(C, dtype, rows):
    from core_scheduler_amd import ops

    x, dy, dres = (torch.randn(rows, C, device="cuda", generator=torch.Generator("cuda").manual_seed(78 + i)).to(dtype) for i in range(3))
    gamma = randn(C, 81, 0.2, 1.0).cuda()
    args = (dy, x, *ops.layernorm_forward(x, gamma)[1:], gamma)
    for more in ({}, {"dresidual": dres}):
        alone = ops.layernorm_backward(*args, need_dgamma=False, need_dbeta=False, **more)
        assert alone[1] is None and alone[2] is None
        assert torch.equal(alone[0], ops.layernorm_backward(*args, **more)[0])


@pytest.mark.parametrize("C,dtype", [(8, BF16), (72, F16), (132, F32), (264, BF16), (640, BF16), (1000, F16), (400, F32), (1600, BF16),
                                     (2056, BF16), (1001, BF16), (3, F32)])
@pytest.mark.parametrize("rows", [3, 700])  # one launch with the sums, and two
def test_infinite_gamma_of_the_last_column(C, dtype, rows):
    """An infinity in gamma makes a row's sums infinite, and its dx where the two infinities do not meet; lanes that have no
    part of the row add nothing to them."""
    from core_scheduler_amd import ops

    x = randn((rows, C), 82).to(dtype).cuda()
    dy = (randn((rows, C), 83).abs() + 0.5).to(dtype).cuda()
    gamma = torch.ones(C, device="cuda")
    _, mean, rstd = ops.layernorm_forward(x, gamma)
    gamma[-1] = float("inf")
    xh = (x.double() - mean.double()[:, None]) * rstd.double()[:, None]
    g = dy.double() * gamma.double()
    want = rstd.double()[:, None] * (g - g.mean(1, keepdim=True) - xh * (g * xh).mean(1, keepdim=True))
    assert torch.isinf(want).any()
    for sums in (True, False):
        dx = ops.layernorm_backward(dy, x, mean, rstd, gamma, need_dgamma=sums, need_dbeta=sums)[0].double()
        assert torch.equal(dx.isnan(), want.isnan()) and torch.equal(dx.isinf(), want.isinf())
        assert torch.equal(dx[dx.isinf()], want[want.isinf()])


@pytest.mark.parametrize("C,dtype", [(256, F32), (512, F32), (1000, BF16)])
def test_sums_of_very_many_rows(C, dtype):
    """A wave's chain of fp32 sums grows with the rows: 4096 waves share them, as close to 64 bits as such sums are."""
    from core_scheduler_amd import ops

    rows, waves = 262147, 4096
    random = torch.Generator("cuda").manual_seed(84)
    x, dy = (torch.randn(rows, C, device="cuda", generator=random).to(dtype) for _ in range(2))
    gamma = torch.ones(C, device="cuda")
    _, mean, rstd = ops.layernorm_forward(x, gamma)
    _, dgamma, dbeta = ops.layernorm_backward(dy, x, mean, rstd, gamma)

    chains = [torch.zeros(waves, C, device="cuda") for _ in range(2)]
    want = [torch.zeros(C, dtype=torch.float64, device="cuda") for _ in range(2)]
    for r in range(0, rows, waves):
        at = slice(r, min(r + waves, rows))
        n = at.stop - r
        xh, dv = (x[at].float() - mean[at, None]) * rstd[at, None], dy[at].float()
        for s, total, term in zip(chains, want, (dv.double() * xh.double(), dv.double())):
            s[:n] = (s[:n].double() + term).float()  # (a fused multiply-add)
            total += term.sum(0)
    for s, total, got in zip(chains, want, (dgamma, dbeta)):
        for groups in (8, 32, 16):  # a workgroup's waves, every 16th partial row, and those: each one after the other
            s = s.view(-1, 8, C) if groups == 8 else s.view(32, 16, C).transpose(0, 1) if groups == 32 else s[None]
            t = torch.zeros_like(s[:, 0])
            for g in range(groups):
                t = t + s[:, g]
            s = t
        formula, error = ((v.double() - total).pow(2).mean().sqrt().item() for v in (s[0], got))
        assert error <= 1.02 * formula  # (2048 waves: 1.2 of it)
