"""Fused classifier rows too wide for two register sets, at the edges of the plans that hold one row in
registers, against the CPU oracle."""
import pytest
import torch

from _util import assert_bit_exact, assert_close, randint, randn

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
INF = float("inf")


@pytest.fixture(scope="module")
def ops():
    from core_scheduler_amd import ops as o
    return o


@pytest.fixture(scope="module")
def co():
    from oracle import c_oracle
    return c_oracle


@pytest.mark.parametrize("N,V,stride,dtype,gdt", [
    (3, 57345, 57352, BF16, None),      # the narrowest 16-bit row of whole vectors
    (330, 57347, 57352, F16, None),     # more rows than workgroups, too few for a second round: two sweeps
    (390, 57347, 57352, F16, None),     # enough
    (300, 40000, 40000, F32, None),     # fp32: a row per workgroup in registers
    (3, 98304, 98304, BF16, None),      # the last width of the first plan, no padding
    (3, 98305, 98312, F16, None),
    (3, 131072, 131072, F16, None),
    (3, 131073, 131080, BF16, None),
    (2, 163840, 163840, BF16, None),    # the widest
    (260, 57345, 57352, BF16, None),    # a few rows more than CUs: two sweeps
    (2, 163841, 163848, BF16, None),    # the next one: two sweeps
    (3, 53252, 53252, BF16, F32),       # 8-byte accesses: fp32 gradients
    (3, 98300, 98304, F16, F32),
    (2, 163839, 163840, BF16, F32),
    (3, 32772, 32772, F32, None),
    (260, 49152, 49152, F32, None),
    (3, 65533, 65536, F32, None),
    (2, 81920, 81920, F32, None),
    (2, 81921, 81924, F32, None),
    # rows that start anywhere
    (4, 57281, 57281, BF16, None),
    (3, 98241, 98241, F16, None),       # the last width of the first plan, 63 elements of the line in front
    (3, 98240, 98243, BF16, None),
    (2, 163775, 163775, BF16, None),
    (2, 163777, 163777, BF16, None),    # two sweeps
    (330, 53187, 53187, BF16, F32),
    (3, 32738, 32739, F32, None),
    (2, 81887, 81887, F32, None),
    (1, 100003, 100003, BF16, None),    # a single row, its last vector not whole
])
@pytest.mark.parametrize("weighted", [False, True])
def test_wide_rows(ops, co, N, V, stride, dtype, gdt, weighted):
    x = randn((N, stride), 960, std=2.0, dtype=dtype)
    t = randint(0, V, (N,), 961)
    t[0] = V - 1
    if N > 1:
        t[N - 1] = 0
    if N > 2:
        t[1] = -100
    kw = dict(dlogits_dtype=gdt) if gdt else {}
    w = randn(V, 962).abs() + 0.1 if weighted else None
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
    if not gdt:  # in place: nothing of a neighbouring row is touched
        ops.fused_classifier(gx, gt, V, class_weight=gw, inplace=True)
        assert_bit_exact(gx, d, "in place")


@pytest.mark.parametrize("V,dtype", [(100003, BF16), (57281, F16), (32739, F32)])
def test_unpadded_rows_in_place(ops, V, dtype):
    """More rows than workgroups, each reading vectors that it shares with a neighbour whose gradient may be there."""
    N = 400
    x = (randn((N, V), 975, std=2.0)).to(dtype).to("cuda:0")
    t = randint(0, V, (N,), 976)
    t[::7] = -100
    t = t.to("cuda:0")
    loss, row, d, _ = ops.fused_classifier(x, t, V)
    loss2, row2, d2, _ = ops.fused_classifier(x, t, V, inplace=True)
    assert d2.data_ptr() == x.data_ptr()
    assert_bit_exact(x, d, "in place")
    assert_bit_exact(row2, row, "row loss")
    assert_bit_exact(loss2, loss, "loss")


@pytest.mark.parametrize("stride", [70016, 70001])
def test_values_that_are_not_finite(ops, stride):
    """-inf logits have no share; a NaN or +inf makes its row NaN and no other; padding stays zero;
    whole lanes of -inf (columns 16384 apart are one lane's) and the type's lowest value are no maxima."""
    V, N = 70001, 6
    x = randn((N, stride), 970, std=2.0, dtype=BF16)
    x[1, :60000] = -INF
    x[2, 40000] = float("nan")
    x[3, 5] = INF
    x[4, 100:] = torch.finfo(BF16).min
    x[5] = -INF
    x[5, 69999] = 1.0
    t = torch.tensor([7, 69000, 3, 9, 50, 69999])
    loss, row, d, _ = ops.fused_classifier(x.to("cuda:0"), t.to("cuda:0"), V, reduction="sum")
    p = x[:, :V].double().softmax(-1)
    want = p.clone()
    want[torch.arange(N), t] -= 1
    d, row = d.cpu().double(), row.cpu().double()
    for i in (0, 1, 4, 5):
        # one bf16 rounding of the result, and 1e-6 for the cancelling target element
        assert ((d[i, :V] - want[i]).abs() <= 2.0 ** -8 * want[i].abs() + 1e-6).all(), i
        ref = -p[i, t[i]].log()
        assert abs(row[i] - ref) <= 1e-5 * max(1.0, ref), i
    for i in (2, 3):
        assert torch.isnan(d[i, :V]).any() and torch.isnan(row[i])
    assert (d[:, V:] == 0).all()
