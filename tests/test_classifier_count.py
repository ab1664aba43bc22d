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
