"""Embedding backward with the position table, where its launches divide the work: the position sums move from the
reduce launch to the finish launch beyond 256 windows of 32 entries, the finish launch deals columns to workgroups of
256, and its probe for a segment's end takes 256 windows a round.  And the ranking of short lists, which has 16 or
32 keys to a workgroup by their number and by the size of the table."""
import pytest
import torch

from _util import gen, randn, sum_tolerance, ulp_distance

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,C,hot,dtype", [
    (8, 1024, 264, 0.3, torch.bfloat16),   # 256 windows: positions in the reduce launch; one column slice and 8 columns
    (9, 911, 256, 0.3, torch.float32),     # 257 windows: positions in the finish launch; whole slices
    (1, 1, 8, 0.0, torch.float16),         # one entry
    (1, 33, 776, 0.5, torch.float32),      # two windows, a last slice of 8 columns
    (20, 500, 252, 1.0, torch.float32),    # one id in every entry: 313 windows, two rounds of probing; sliced batch
    (40, 15, 516, 0.9, torch.bfloat16),    # sliced batch in the reduce launch
])
def test_positions_and_table(B, T, C, hot, dtype):
    from core_scheduler_amd import ops

    V = 700
    ids = torch.randint(0, V, (B, T), generator=gen(1))
    ids[torch.rand((B, T), generator=gen(2)) < hot] = 3
    dout = randn((B, T, C), 3, dtype=dtype)
    dwte, dwpe = ops.embedding_backward_fused(dout.cuda(), ids.cuda(), V)
    terms = dout.double().reshape(-1, C)
    want_t = torch.zeros(V, C, dtype=torch.float64).index_add_(0, ids.reshape(-1), terms)
    squares = torch.zeros(V, C, dtype=torch.float64).index_add_(0, ids.reshape(-1), terms * terms)
    # sum_tolerance's bound, for sums of different lengths
    tol_t = 7.0 * 2.0 ** -24 * torch.sqrt(torch.log2(torch.tensor(float(max(2, B * T)))) * squares)
    for got, want, tol, name in ((dwte, want_t, tol_t, "dwte"),
                                 (dwpe, dout.double().sum(0), sum_tolerance(dout), "dwpe")):
        got = got.cpu()
        ok = (got.double() - want).abs() <= tol
        if dtype != torch.float32:
            ok |= ulp_distance(got, want.to(dtype)) <= 1
        assert ok.all(), (name, (got.double() - want).abs().max().item())
    again = ops.embedding_backward_fused(dout.cuda(), ids.cuda(), V)
    assert torch.equal(again[0], dwte) and torch.equal(again[1], dwpe)
    # += of both tables, and the position sums by themselves
    base_t, base_p = randn((V, C), 4, dtype=dtype), randn((T, C), 5, dtype=dtype)
    acc_t, acc_p = ops.embedding_backward_fused(dout.cuda(), ids.cuda(), V, base_t.cuda(), base_p.cuda())
    for got, want, tol in ((acc_t, want_t + base_t.double(), tol_t), (acc_p, dout.double().sum(0) + base_p.double(),
                                                                     sum_tolerance(dout))):
        got = got.cpu()
        ok = (got.double() - want).abs() <= tol + 2.0 ** -23 * want.abs()
        if dtype != torch.float32:
            ok |= ulp_distance(got, want.to(dtype)) <= 1
        assert ok.all()
    assert torch.equal(ops.embedding_backward_positions(dout.cuda()), dwpe)


@pytest.mark.parametrize("n", [15, 17, 4095, 4096, 4097])
@pytest.mark.parametrize("V", [40, 60000])  # tables on either side of 32 MB at 192 columns fp32
def test_short_lists(n, V):
    from core_scheduler_amd import ops

    C = 192
    ids = torch.randint(-1, V + 1, (n,), generator=gen(6))  # some out of range
    dout = torch.randint(-8, 9, (n, C), generator=gen(7)).float()  # whole numbers: every order gives the same sums
    want = torch.zeros(V, C)
    keep = (ids >= 0) & (ids < V) & (ids != 5)
    want.index_add_(0, ids[keep], dout[keep])
    assert torch.equal(ops.embedding_backward(dout.cuda(), ids.cuda(), V, padding_idx=5).cpu(), want)


@pytest.mark.parametrize("V", [24576, 24577])  # 3 * 2^20 vectors of fill, with which the sort launch still has the sums
@pytest.mark.parametrize("n_batch", [9, 20])   # one lane per vector of the position table, and a sliced batch
def test_positions_of_a_long_list(V, n_batch):
    from core_scheduler_amd import ops

    T, C = 911, 512
    ids = torch.randint(0, V, (n_batch, T), generator=gen(8))
    dout = torch.randint(-8, 9, (n_batch, T, C), generator=gen(9)).float()  # whole numbers: every order gives the same sums
    want_t = torch.zeros(V, C).index_add_(0, ids.reshape(-1), dout.reshape(-1, C))
    want_p = dout.sum(0)
    dwte, dwpe = ops.embedding_backward_fused(dout.cuda(), ids.cuda(), V)
    assert torch.equal(dwte.cpu(), want_t) and torch.equal(dwpe.cpu(), want_p)
    dwte, dwpe = ops.embedding_backward_fused(dout.cuda(), ids.cuda().int(), V, dwte, dwpe)  # nothing to fill
    assert torch.equal(dwte.cpu(), 2 * want_t) and torch.equal(dwpe.cpu(), 2 * want_p)


@pytest.mark.parametrize("C", [1020, 1024, 1028, 1100, 1600])  # one column a lane up to 1024, two beyond; a last slice that is not full
@pytest.mark.parametrize("n,hot", [(1500, 0.5), (13200, 0.0), (13200, 0.5)])  # few workgroups (one column), and more than 2048
def test_finish_of_wide_rows(C, n, hot):
    from core_scheduler_amd import ops

    V = 600  # nearly every window is left by a run; a hot id has partial rows of its own to add
    ids = torch.randint(0, V, (n,), generator=gen(10))
    ids[torch.rand(n, generator=gen(11)) < hot] = 7
    dout = torch.randint(-8, 9, (n, C), generator=gen(12)).float()  # whole numbers: every order gives the same sums
    want = torch.zeros(V, C).index_add_(0, ids, dout)
    got = ops.embedding_backward(dout.cuda(), ids.cuda(), V)
    assert torch.equal(got.cpu(), want)
    assert torch.equal(ops.embedding_backward(dout.cuda(), ids.cuda(), V, dweight=got).cpu(), 2 * want)
    mean = ops.embedding_backward(dout.cuda(), ids.cuda(), V, scale_grad_by_freq=True).cpu()
    exact = want.double() / torch.bincount(ids, minlength=V).clamp(min=1).double()[:, None]
    assert ((mean.double() - exact).abs() <= 2.0 ** -22 * exact.abs()).all()  # a reciprocal and a product, rounded each
