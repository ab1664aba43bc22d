"""The loss alone of up to 1024 long rows, each split over several workgroups: against the double-precision loss.

The sum's terms round at 2^-23 and their tree, at most 6 + 6 + 2 + 32 additions deep, at 2^-24 each: 3e-6 of it, so as much in
its logarithm; the exponents' argument rounds at |x log2 e| 2^-24 < 2e-6 for these logits.  1e-5 bounds their sum."""
import pytest
import torch

from _util import randint, randn


# widths at the edges of the vectors a lane holds (2, 4, 8 of them) and of the rule (more than 2048 vectors; 32 splits)
@pytest.mark.gpu
@pytest.mark.parametrize("N,V,stride,dtype", [
    (1, 16392, 16392, torch.bfloat16), (3, 16385, 16400, torch.float16), (64, 50257, 50304, torch.bfloat16),
    (509, 50257, 50257, torch.bfloat16), (1024, 16399, 16399, torch.bfloat16), (1025, 16399, 16399, torch.bfloat16),
    (700, 32768, 32768, torch.float16), (130, 8197, 8197, torch.float32), (257, 20001, 20004, torch.float32),
    (2, 262144, 262144, torch.float32), (2, 262145, 262145, torch.float32), (5, 524289, 524289, torch.bfloat16),
    (40, 1, 16640, torch.bfloat16), (40, 9, 16641, torch.float16)])
def test_split_loss(N, V, stride, dtype):
    from core_scheduler_amd import ops

    x = randn((N, stride), 1, std=2.0).to(dtype)
    x[:, V:] = 1e4  # padding takes no part
    t = randint(0, V, (N,), 2)
    if N > 2:
        x[1, :V] -= 3000.0
        x[2, V // 2 + 1:V] = float("-inf")
        t[2] = 0
        t[5::7] = -100
        t[N - 1] = V - 1 if N != 3 else 0
    w = randn(V, 3).abs() + 0.1
    counts = t >= 0
    at = t.clamp(min=0)
    exact = torch.logsumexp(x[:, :V].double(), 1) - x[torch.arange(N), at].double()
    for weight in (None, w):
        rows = torch.where(counts, exact if weight is None else exact * weight[at].double(), torch.zeros((), dtype=torch.double))
        total = (counts if weight is None else weight[at].double() * counts).sum().item()
        for reduction in ("mean", "sum", "none"):
            loss, row, d, tw = ops.fused_classifier(x.cuda(), t.cuda(), V, reduction=reduction, want_dlogits=False,
                                                    class_weight=None if weight is None else weight.cuda())
            assert d is None and abs(tw.item() - total) <= 1e-6 * total
            assert ((row.cpu().double() - rows).abs() <= 1e-5 * rows.abs().clamp(min=1)).all()
            if reduction != "none":
                want = rows.sum().item() / (total if reduction == "mean" else 1.0)
                assert abs(loss.item() - want) <= 2e-5 * max(1.0, abs(want))


@pytest.mark.gpu
def test_split_rows_that_have_no_loss():
    from core_scheduler_amd import ops

    N, V = 6, 40001
    x = randn((N, V), 4).to(torch.bfloat16)
    x[0], x[1, 39999], x[2, 3], x[3] = float("-inf"), float("nan"), float("inf"), float("nan")
    x[4, :39999] = float("-inf")  # the first splits hold nothing finite
    t = torch.tensor([1, 2, 5, 7, 39999, -100])
    loss, row, _, tw = ops.fused_classifier(x.cuda(), t.cuda(), want_dlogits=False, reduction="sum")
    assert row[:4].isnan().all() and loss.isnan() and tw.item() == 5 and row[5].item() == 0
    exact = torch.logsumexp(x[4].double(), 0) - x[4, 39999].double()
    assert abs(row[4].item() - exact.item()) <= 1e-5


@pytest.mark.gpu
def test_workspace_without_the_splits():
    """A caller that brings the header and a row loss each is served by whole rows, as before."""
    from core_scheduler_amd import _capi, ops

    lib = _capi.load()
    x, t = randn((33, 20000), 6).cuda(), randint(0, 20000, (33,), 7).cuda()
    out = [torch.empty(n, device="cuda") for n in (33, 1, 1)]
    ws = torch.empty(512, dtype=torch.uint8, device="cuda")
    code = lib.cs_fused_classifier(x.data_ptr(), None, t.data_ptr(), out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(),
                                   ws.data_ptr(), 512, 33, 20000, 20000, -100, _capi.REDUCTION_MEAN, 1.0, _capi.F32, _capi.F32,
                                   torch.cuda.current_stream().cuda_stream)
    assert code == _capi.OK
    row = ops.fused_classifier(x, t, want_dlogits=False)[1]
    assert (row - out[0]).abs().max().item() <= 1e-5


def test_workspace_never_falls_with_the_rows():
    """One buffer for the longest batch gives every shorter one the splits that a buffer of its own size gives it."""
    from core_scheduler_amd import _capi

    size = _capi.load().cs_fused_classifier_workspace_bytes
    sizes = [size(n) for n in (*range(0, 3000), 8192, 100000, 1 << 20)]
    assert sizes == sorted(sizes)
