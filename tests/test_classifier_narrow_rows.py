"""Fused classifier rows that one workgroup holds in its registers, padded or not, at the edges of the plan: widths of less
than a vector, up to the last one for few and for many rows, rows that share a vector, the array's last vector."""
import pytest
import torch

from _util import gen, randint, randn, ulp_distance

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("N,V,stride,dtype,gdt", [
    (5, 1, 1, BF16, BF16),           # five rows in one vector, which is not whole
    (9, 3, 7, F16, F32), (4, 63, 65, BF16, BF16), (4, 255, 257, F32, F32),
    (3, 2041, 2041, BF16, BF16),     # a wave and a bit
    (3, 2048, 2048, F16, F16), (3, 2049, 2056, F16, F32),
    (2, 16321, 16321, BF16, BF16),   # the widest unpadded row of few rows, and the next one
    (2, 16322, 16322, BF16, BF16),
    (2, 16384, 16384, BF16, BF16), (2, 16377, 16392, BF16, BF16),
    (2, 8161, 8161, F32, F32), (2, 8192, 8192, F32, F32),
    (2, 16321, 16321, F16, F32), (2, 16384, 16384, BF16, F32),
    # three accesses a lane of two waves, and of three: the widest rows, and the next ones
    (3, 3072, 3072, BF16, BF16), (3, 3073, 3080, F16, F16), (3, 4545, 4545, F16, F16), (3, 4546, 4546, BF16, BF16),
    (3, 1536, 1536, F32, F32), (3, 1540, 1540, F32, F32), (3, 2257, 2257, F32, F32), (3, 3009, 3009, F16, F32),
    (3, 3010, 3010, BF16, F32), (3, 4608, 4608, BF16, F32),
    (513, 24513, 24513, BF16, BF16), (513, 24514, 24514, BF16, BF16), (513, 32767, 32768, F16, F16),
    (513, 12257, 12257, F32, F32), (513, 24512, 24513, BF16, F32), (513, 32760, 32768, BF16, F32),
])
@pytest.mark.parametrize("weighted", [False, True])
def test_rows_in_registers(N, V, stride, dtype, gdt, weighted):
    from core_scheduler_amd import ops

    x, t = randn((N, stride), 60, std=2.0, dtype=dtype).cuda(), randint(0, V, (N,), 61).cuda()
    t[0], t[-1] = V - 1, 0
    if N > 2:
        t[1] = -100
    w = (torch.rand(V, generator=gen(62)) + 0.5).cuda() if weighted else None
    keep = t >= 0
    at = t.clamp(min=0)
    wt = (w.double()[at] if weighted else torch.ones(N, dtype=torch.float64, device="cuda")) * keep
    logp = x[:, :V].double().log_softmax(1)
    want_rows = -logp.gather(1, at[:, None])[:, 0] * wt
    total = wt.sum()
    want = torch.zeros(N, stride, dtype=torch.float64, device="cuda")
    want[:, :V] = logp.exp()
    onehot = torch.zeros_like(want).scatter_(1, at[:, None], 1.0)
    sizes = (want + onehot) * (wt / total)[:, None]
    want = (want - onehot) * (wt / total)[:, None]

    logits = x.clone()
    loss, rows, d, weight = ops.fused_classifier(logits, t, V, class_weight=w, dlogits_dtype=gdt)
    # exponents of up to 2^4 rounded to 2^-24 of 24, sums by trees of 2^-24 each: 2^-19 of a probability, and the loss to
    # 2^-20 of itself and of the logits
    assert ((rows.double() - want_rows).abs() <= 2.0 ** -19 * (want_rows.abs() + 8)).all()
    assert abs(weight.item() - total.item()) <= 1e-5 * total.item()
    assert abs(loss.item() - (want_rows.sum() / total).item()) <= 2.0 ** -18 * (8 + want_rows.abs().max().item())
    ok = (d.double() - want).abs() <= 2.0 ** -19 * sizes
    if gdt != F32:
        ok |= (ulp_distance(d.cpu(), want.to(gdt).cpu()) <= 1).cuda()
    assert ok.all() and not d[:, V:].any() and torch.equal(logits, x)
    alone = ops.fused_classifier(x, t, V, class_weight=w, want_dlogits=False)[1]
    assert ((alone.double() - want_rows).abs() <= 2.0 ** -19 * (want_rows.abs() + 8)).all()
    if N <= 512 and gdt == dtype:  # the loss alone goes the same way
        assert torch.equal(alone, rows)
    if gdt == dtype and not weighted:  # the gradient over the logits
        _, rows2, d2, _ = ops.fused_classifier(logits, t, V, inplace=True)
        assert torch.equal(d2, d) and torch.equal(rows2, rows) and d2.data_ptr() == logits.data_ptr()


@pytest.mark.parametrize("stride", [500, 501])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_rows_that_are_not_finite(stride, bad):
    from core_scheduler_amd import ops

    x, t = randn((3, stride), 63, dtype=BF16).cuda(), torch.tensor([1, 2, 3], device="cuda")
    x[1, :499] = bad if bad == float("-inf") else x[1, :499]
    x[1, 7] = bad
    _, rows, d, _ = ops.fused_classifier(x, t, 499)
    clean = ops.fused_classifier(torch.where(torch.isfinite(x), x, torch.zeros_like(x)), t, 499)
    assert torch.isnan(rows[1]) and torch.isnan(d[1, :499]).all() and not d[:, 499:].any()
    assert torch.equal(rows[0], clean[1][0]) and torch.equal(d[0], clean[2][0]) and torch.equal(d[2], clean[2][2])


@pytest.mark.parametrize("N", [1023, 1024, 1025, 8193])  # one row a lane of the last launch, and eight under way
@pytest.mark.parametrize("weighted", [False, True])
def test_sums_over_the_rows(N, weighted):
    from core_scheduler_amd import ops

    V = 40
    x, t = randn((N, V), 64, dtype=F32).cuda(), randint(-1, V + 1, (N,), 65).cuda()  # some rows out of range
    w = (torch.rand(V, generator=gen(66)) + 0.5).cuda() if weighted else None
    keep = (t >= 0) & (t < V)
    at = t.clamp(0, V - 1)
    wt = (w.double()[at] if weighted else torch.ones(N, dtype=torch.float64, device="cuda")) * keep
    want = (-x.double().log_softmax(1).gather(1, at[:, None])[:, 0] * wt).sum()
    for reduction, by in (("sum", 1.0), ("mean", wt.sum())):
        for gradient in (True, False):
            loss, _, _, total = ops.fused_classifier(x, t, V, reduction=reduction, class_weight=w, want_dlogits=gradient)
            # sums of positive terms, 2^-24 a level of a tree of at most 20
            assert abs(loss.item() - (want / by).item()) <= 20 * 2.0 ** -24 * (want / by).item()
            assert abs(total.item() - wt.sum().item()) <= 20 * 2.0 ** -24 * wt.sum().item()
