"""Fused classifier calls whose last launch counts the rows (everything but the gradient of a mean): the
count, the class weights' sum and the loss at the edges of that launch's loop, against the CPU oracle."""
import pytest
import torch

from _util import assert_close, randint, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 1023, 1025, 8193, 20001])
@pytest.mark.parametrize("reduction,want_dlogits", [("mean", False), ("sum", False), ("sum", True), ("none", True), ("none", False)])
@pytest.mark.parametrize("weighted", [False, True])
def test_count_in_the_last_launch(N, reduction, want_dlogits, weighted):
    from core_scheduler_amd import ops
    from oracle import c_oracle as co

    V = 40
    x = randn((N, V), 980, std=2.0)
    t = randint(0, V, (N,), 981)
    if N > 1:
        t[::7] = -100
        t[N - 1] = V - 1
    w = randn(V, 982).abs() + 0.1 if weighted else None
    args = dict(reduction=reduction, want_dlogits=want_dlogits)
    loss, row, d, tw = ops.fused_classifier(x.cuda(), t.cuda(), class_weight=None if w is None else w.cuda(), **args)
    loss2, row2, d2, tw2 = co.cross_entropy(x, t, V, class_weight=w, reduction=reduction)
    counts = t >= 0
    total = float(counts.sum() if w is None else w.double()[t[counts]].sum())
    assert_close(row, row2.float(), atol=1e-5, name="row loss")
    if w is None:
        assert tw.item() == total
    else:  # positive terms: at most 3 + 3 + 10 roundings of 2^-24 lie between a weight and the sum
        assert abs(tw.item() - total) <= 1e-6 * total
    if reduction != "none":  # the same, and 1e-5 for each row's loss as above
        want = float(row2.double().sum()) / (total if reduction == "mean" else 1.0)
        assert abs(loss.item() - want) <= 2e-5 * want
    if want_dlogits:
        assert_close(d, d2, atol=1e-6, name="dlogits")


def test_no_row_counts():
    from core_scheduler_amd import ops

    x, t = randn((5, 40), 990).cuda(), torch.full((5,), -100, device="cuda:0")
    loss, row, d, tw = ops.fused_classifier(x, t, want_dlogits=False)
    assert torch.isnan(loss) and tw.item() == 0 and (row == 0).all()
    loss, row, d, tw = ops.fused_classifier(x, t, reduction="sum")
    assert loss.item() == 0 and tw.item() == 0 and (d == 0).all()


# one width of each row kernel: 64 and 256 lanes, streamed (padded, ragged, 16-bit to fp32), held, two sweeps, general
@pytest.mark.parametrize("V,stride,dtype,out", [
    (40, 40, torch.bfloat16, None), (5003, 5008, torch.bfloat16, None), (50257, 50304, torch.bfloat16, None),
    (50257, 50257, torch.bfloat16, torch.float32), (60000, 60000, torch.float16, None), (60001, 60001, torch.float16, None),
    (18001, 18001, torch.bfloat16, torch.float32), (1003, 1003, torch.float32, None), (40, 41, torch.float64, None)])
def test_few_rows_count_themselves(V, stride, dtype, out):
    """The gradient of a mean of up to 512 rows: the bits of the call whose count is a launch ahead of the rows."""
    from core_scheduler_amd import _capi, ops

    lib = _capi.load()
    x = randn((513, stride), 983, std=2.0).to(dtype).cuda()
    targets = randint(0, V, (513,), 984).cuda()
    targets[1::5] = -100
    for N in (1, 2, 63, 64, 65, 300, 512, 513):
        got = ops.fused_classifier(x[:N], targets[:N], V, dlogits_dtype=out)
        want = [torch.empty((), device="cuda"), torch.empty(N, device="cuda"),
                torch.empty(N, stride, dtype=out or dtype, device="cuda"), torch.empty((), device="cuda")]
        n = lib.cs_fused_classifier_workspace_bytes(N)
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        for phase in (1, 2, 4):
            code = lib.cs_fused_classifier_phases(
                x.data_ptr(), want[2].data_ptr(), targets.data_ptr(), want[1].data_ptr(), want[0].data_ptr(),
                want[3].data_ptr(), ws.data_ptr(), n, N, V, stride, -100, _capi.REDUCTION_MEAN, 1.0, ops._DTYPES[dtype],
                ops._DTYPES[out or dtype], phase, torch.cuda.current_stream().cuda_stream)
            assert code == _capi.OK
        for g, w in zip(got, want):
            assert torch.equal(g, w)
        assert got[3].item() == (targets[:N] >= 0).sum().item()
