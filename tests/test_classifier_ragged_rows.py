"""Fused classifier rows that start anywhere (a vocabulary used unpadded) at the edges of the kernels'
plans, against the CPU oracle."""
import pytest
import torch

from _util import assert_bit_exact, assert_close, randint, randn

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(scope="module")
def ops():
    from core_scheduler_amd import ops as o
    return o


@pytest.fixture(scope="module")
def co():
    from oracle import c_oracle
    return c_oracle


@pytest.mark.parametrize("N,V,stride,dtype,gdt", [
    (3, 16385, 16385, BF16, None),      # 2048 vectors and an element: the narrowest streamed row
    (259, 16390, 16391, F16, None),     # more rows than workgroups, a padding column
    (5, 32705, 32705, BF16, None),      # the four-vector plan with the line's 63 elements in front: its last width
    (5, 32706, 32707, BF16, None),      # the next one
    (3, 57279, 57279, F16, None),       # the widest streamed 16-bit row
    (3, 57281, 57281, BF16, None),      # the next one
    (2, 53183, 53183, BF16, F32),       # the widest with fp32 gradients
    (2, 53185, 53185, F16, F32),
    (260, 20011, 20011, BF16, F32),     # two sweeps up to 24576 columns with fp32 gradients
    (3, 24575, 24575, BF16, F32),
    (3, 24577, 24577, F16, F32),        # streamed
    (520, 33001, 33001, BF16, None),    # the loss alone: two sweeps where rows are a few per CU
    (3, 8193, 8193, F32, None),         # fp32: 2048 vectors and an element
    (2, 32735, 32735, F32, None),       # the widest streamed fp32 row
    (2, 32737, 32737, F32, None),
    (1, 50257, 50257, BF16, None),      # a single row, its last vector not whole
    (7, 50255, 50257, F16, None),
])
@pytest.mark.parametrize("weighted", [False, True])
def test_unpadded_rows(ops, co, N, V, stride, dtype, gdt, weighted):
    x = randn((N, stride), 950, std=2.0, dtype=dtype)
    t = randint(0, V, (N,), 951)
    t[0] = V - 1
    if N > 1:
        t[N - 1] = 0
    if N > 2:
        t[1] = -100
    kw = dict(dlogits_dtype=gdt) if gdt else {}
    w = randn(V, 952).abs() + 0.1 if weighted else None
    gw = w.to("cuda:0") if weighted else None
    gx, gt = x.to("cuda:0"), t.to("cuda:0")
    loss, row, d, tw = ops.fused_classifier(gx, gt, V, class_weight=gw, **kw)
    loss2, row2, d2, tw2 = co.cross_entropy(x, t, V, class_weight=w, **kw)
    scale = 1.0 if w is None else float(w.max())
    assert_close(tw, tw2.float(), atol=1e-5 * N, name="total weight")
    assert_close(loss, loss2.float(), atol=1e-5 * scale, name="loss")
    assert_close(row, row2.float(), atol=1e-5 * scale, name="row loss")
    assert_close(d, d2, atol=1e-10 * scale, name="dlogits")
    assert (d[:, V:] == 0).all()
    if N > 2:
        assert (d[1] == 0).all()
    # the loss alone, and in place: nothing of a neighbouring row is touched
    loss3, row3, none, _ = ops.fused_classifier(gx, gt, V, class_weight=gw, want_dlogits=False)
    assert none is None
    assert_close(row3, row2.float(), atol=1e-5 * scale, name="row loss alone")
    if not gdt:
        ops.fused_classifier(gx, gt, V, class_weight=gw, inplace=True)
        assert_bit_exact(gx, d, "in place")


@pytest.mark.parametrize("V,stride,dtype,gdt", [
    (50257, 50257, BF16, None), (50255, 50257, F16, None), (40011, 40011, BF16, F32), (32001, 32003, F32, None),
])
def test_rows_that_are_not_finite(ops, V, stride, dtype, gdt):
    """An unpadded row without a finite logit, or with a NaN or +inf, is NaN in every class and 0 in the padding, as a
    softmax in 64 bits gives it; -inf elsewhere has no share."""
    N, inf, nan = 10, float("inf"), float("nan")
    x = randn((N, stride), 953, std=2.0, dtype=dtype)
    t = randint(0, V, (N,), 954)
    x[0, :V] = -inf
    x[1, V // 2] = nan
    x[2, 17] = inf
    x[3, :V] = nan
    x[4, :V - 1], t[4] = -inf, V - 1
    x[5, 100:], t[5] = -inf, 7
    x[6], t[6] = -inf, -100
    x[7, 0], x[7, 5:V] = nan, -inf
    x[8, 1000:], x[8, 30000], t[8] = -inf, nan, 50  # the NaN's lane holds no finite value
    kw = dict(dlogits_dtype=gdt) if gdt else {}
    loss, row, d, _ = ops.fused_classifier(x.to("cuda:0"), t.to("cuda:0"), V, reduction="sum", **kw)
    want = x[:, :V].double().softmax(dim=1)
    keep = t >= 0
    want[keep, t[keep]] -= 1.0
    want[~keep] = 0.0
    # one rounding of the result, and 1e-6 for the target element that cancels
    assert_close(d[:, :V], want.to(d.dtype), atol=1e-6, name="dlogits")
    assert (d[:, V:] == 0).all()
    want_row = torch.nn.functional.cross_entropy(x[:, :V].double(), t, reduction="none")
    assert_close(row, want_row.float(), atol=1e-5, name="row loss")
    assert torch.isnan(loss)


@pytest.mark.parametrize("V,stride,dtype", [
    (50257, 50257, BF16), (40001, 40001, BF16), (35000, 35003, F16), (30001, 30001, F32), (9001, 9001, F32),
    (100003, 100003, BF16),  # the row-holding kernel
])
def test_every_gradient_element_keeps_its_digits(ops, V, stride, dtype):
    """The relative error of the probabilities, which a norm over the gradient hides behind the target's.

    Exponents lie mostly in [8, 16) (logits of deviation 2, 50 thousand of them: the maximum is 8.5 above the
    middle), where rounding is uniform in half a unit of 2^-20: 2.75e-7 rms times ln 2 = 1.9e-7 of the value.
    The exponential, the scale and the product add 0.5e-7 each, the row's sum 1e-7: 2.3e-7, here with a fifth more.
    """
    N = 64
    x = randn((N, stride), 955, std=2.0, dtype=dtype)
    t = randint(0, V, (N,), 956)
    d = ops.fused_classifier(x.to("cuda:0"), t.to("cuda:0"), V, dlogits_dtype=F32)[2][:, :V].cpu().double()
    want = x[:, :V].double().softmax(dim=1) / N
    rel = (d - want) / want
    rel[torch.arange(N), t] = 0.0
    assert rel.square().mean().sqrt().item() < 2.8e-7


@pytest.mark.parametrize("N,V,dtype,grad", [
    (2000, 50257, BF16, "same"), (2000, 50257, F16, "fp32"), (2000, 32001, F32, "same"), (2000, 20001, BF16, "same"),
    (1000, 50257, BF16, None), (1000, 57001, F16, None), (1000, 30001, F32, None),
])
def test_loss_of_confident_rows(ops, N, V, dtype, grad):
    """Rows whose target holds nearly all of the sum: their loss, near 0, is the sum's distance from 1.

    Every add onto a term of 1 rounds by 3.4e-8 rms (half a unit of 2^-23, uniform); a lane adds its columns in
    groups of 16, at most four groups, then come ten levels of lanes and waves: 1.3e-7, here with a tenth more.
    """
    x = randn((N, V), 957, std=2.0, dtype=dtype).to("cuda:0")
    t = randint(0, V, (N,), 958).to("cuda:0")
    x[torch.arange(N, device="cuda:0"), t] = (18.0 + randn((N,), 959).abs()).to(dtype).to("cuda:0")
    kw = dict(dlogits_dtype=F32) if grad == "fp32" else {}
    row = ops.fused_classifier(x, t, V, want_dlogits=grad is not None, **kw)[1].double()
    want = torch.cat([torch.nn.functional.cross_entropy(x[i:i + 100].double(), t[i:i + 100], reduction="none")
                      for i in range(0, N, 100)])
    assert (row - want).square().mean().sqrt().item() < 1.45e-7
