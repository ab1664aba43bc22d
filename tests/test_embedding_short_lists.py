"""Embedding backward of lists of up to 1024 entries: one launch that compares the list with its entries (whole segments
up to 192 entries, runs cut at windows of 32 sorted entries and a second launch beyond), the zeros of the rows that no
entry names in the same launch."""
import pytest
import torch

from _util import gen, randn, ulp_distance, zipf_ids

pytestmark = pytest.mark.gpu


def _ids(kind, n, V):
    if kind == "one":
        return torch.full((n,), min(3, V - 1))
    if kind == "zipf":
        return zipf_ids(n, V, 21)
    return torch.randint(-1, V + 1, (n,), generator=gen(20))  # some out of range


@pytest.mark.parametrize("kind", ["one", "zipf", "any"])
@pytest.mark.parametrize("n", [1, 2, 3, 33, 191, 192, 193, 256, 511, 513, 1023, 1024, 1025])
def test_sums_and_zeros(n, kind):
    from core_scheduler_amd import ops

    # C: less than a vector slice, one slice and a bit, several (fp32: 128 vectors of 4 columns each)
    for C, V, pad in ((8, 5000, 4), (516, 40, -1), (1544, 300, 3)):
        ids = _ids(kind, n, V)
        dout = torch.randint(-8, 9, (n, C), generator=gen(22)).float()  # whole numbers: every order gives the same sums
        keep = (ids >= 0) & (ids < V) & (ids != pad)
        want = torch.zeros(V, C).index_add_(0, ids[keep], dout[keep])
        for cast in (torch.int64, torch.int32):
            got = ops.embedding_backward(dout.cuda(), ids.to(cast).cuda(), V, padding_idx=pad)
            assert torch.equal(got.cpu(), want), (C, cast)
        assert torch.equal(ops.embedding_backward(dout.cuda(), ids.cuda(), V, padding_idx=pad, dweight=got).cpu(), 2 * want)
        mean = ops.embedding_backward(dout.cuda(), ids.cuda(), V, padding_idx=pad, scale_grad_by_freq=True).cpu()
        exact = want.double() / torch.bincount(ids[keep], minlength=V).clamp(min=1).double()[:, None]
        assert ((mean.double() - exact).abs() <= 2.0 ** -22 * exact.abs()).all()  # a reciprocal and a product, rounded each


@pytest.mark.parametrize("B,T", [(1, 123), (3, 64), (17, 60), (1000, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rounded_once_with_positions(B, T, dtype):
    from core_scheduler_amd import ops

    V, C = 900, 264
    ids, dout = zipf_ids(B * T, V, 23).view(B, T), randn((B, T, C), 24, dtype=dtype)
    dwte, dwpe = ops.embedding_backward_fused(dout.cuda(), ids.cuda(), V)
    terms = dout.double().view(-1, C)
    want = torch.zeros(V, C, dtype=torch.float64).index_add_(0, ids.view(-1), terms)
    sizes = torch.zeros(V, C, dtype=torch.float64).index_add_(0, ids.view(-1), terms.abs())
    # n - 1 additions of at most the sum of the terms' sizes, each rounded by 2^-24 of it
    ok = (dwte.cpu().double() - want).abs() <= B * T * 2.0 ** -24 * sizes
    assert (ok | (ulp_distance(dwte.cpu(), want.to(dtype)) <= 1)).all()
    assert torch.equal(ops.embedding_backward_positions(dout.cuda()), dwpe)
    assert torch.equal(ops.embedding_backward_fused(dout.cuda(), ids.cuda(), V)[0], dwte)


@pytest.mark.parametrize("n", [0, 5, 700])
def test_nothing_outside_the_table_is_written(n):
    from core_scheduler_amd import _capi

    lib, V, C, edge = _capi.load(), 9001, 8, 256  # more rows than a zero-filling workgroup has bits for
    ids, dout = torch.randint(0, V, (max(n, 1),), generator=gen(25)), torch.ones(max(n, 1), C)
    size = lib.cs_embedding_backward_workspace_bytes(n, C, V)
    ws = torch.full((size + 4096,), 77, dtype=torch.uint8, device="cuda")
    buf = torch.full((edge + V * C + edge,), 7.0, device="cuda")
    dev_dout, dev_ids = dout.cuda(), ids.cuda()
    code = lib.cs_embedding_backward(dev_dout.data_ptr(), dev_ids.data_ptr(), buf.data_ptr() + 4 * edge, ws.data_ptr(), size,
                                     n, C, V, -1, _capi.F32, _capi.I64, 0, torch.cuda.current_stream().cuda_stream)
    assert code == _capi.OK and (ws[size:] == 77).all()
    want = torch.full_like(buf, 7.0).cpu()
    want[edge:edge + V * C] = torch.zeros(V, C).index_add_(0, ids[:n], dout[:n]).view(-1)
    assert torch.equal(buf.cpu(), want)


@pytest.mark.parametrize("n", [4096, 4097, 6144, 6145])  # either side of the lines for two slices, and for three or more
@pytest.mark.parametrize("C", [256, 260, 516, 1100])  # fp32: a slice of 64 vectors, one more, three, five
def test_windows_in_slices(n, C):
    from core_scheduler_amd import ops

    V = 900
    ids = zipf_ids(n, V, 26)
    dout = torch.randint(-8, 9, (n, C), generator=gen(27)).float()  # whole numbers: every order gives the same sums
    want = torch.zeros(V, C).index_add_(0, ids, dout)
    got = ops.embedding_backward(dout.cuda(), ids.cuda(), V)
    assert torch.equal(got.cpu(), want)
    assert torch.equal(ops.embedding_backward(dout.cuda(), ids.cuda(), V, dweight=got).cpu(), 2 * want)
    dwte, dwpe = ops.embedding_backward_fused(dout.view(1, n, C).cuda(), ids.view(1, n).cuda(), V)
    assert torch.equal(dwte.cpu(), want) and torch.equal(dwpe.cpu(), dout)


@pytest.mark.parametrize("kind", ["one", "zipf", "any"])
@pytest.mark.parametrize("n", [5, 64, 65, 129, 192])  # a run of a step of 16 rows for each of four waves, and more
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_whole_runs_of_16_bits(n, kind, dtype):
    from core_scheduler_amd import ops

    for C, V in ((8, 5000), (520, 40), (1032, 300), (3080, 60)):  # up to one slice of 64 vectors, two, three, and 128 to a lane's two
        ids = _ids(kind, n, V)
        dout = torch.randint(-8, 9, (n, C), generator=gen(28)).float()  # whole numbers: every order gives the same sums
        keep = (ids >= 0) & (ids < V)
        want = torch.zeros(V, C).index_add_(0, ids[keep], dout[keep])
        got = ops.embedding_backward(dout.to(dtype).cuda(), ids.cuda(), V)
        assert torch.equal(got.cpu(), want.to(dtype)), C
