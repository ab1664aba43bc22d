"""Embedding rows that are not whole aligned 16-byte vectors (and fp64): gather by vectors moved back to the row's end,
scatter-add by windows of 64 sorted entries in double.  Each backward result is one rounding of a double sum, so it is
held to half a unit in the last place of the exact sum (p significant bits: at most 2^-p of the value), next to what
the double sum is off by."""
import pytest
import torch

from _util import randint, randn

pytestmark = pytest.mark.gpu

# p = 53, 24, 11, 8; 16-bit results are rounded to fp32 first, which moves them by 2^-24 at most
HALF_ULP = {torch.float64: 2.0 ** -53, torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11 + 2.0 ** -23,
            torch.bfloat16: 2.0 ** -8 + 2.0 ** -23}
SMALLEST = {torch.float64: 0.0, torch.float32: 0.0, torch.float16: 2.0 ** -25, torch.bfloat16: 0.0}


def off_by_one(t):
    """The same values one element past a 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")[1:]
    flat.copy_(t.reshape(-1))
    return flat.view(t.shape)


def rounded_once(got, exact, terms):
    # the double sum is off by at most n 2^-53 of the sum of magnitudes, n <= 9001
    bound = HALF_ULP[got.dtype] * exact.abs() + SMALLEST[got.dtype] + 2.0 ** -38 * terms
    return ((got.double() - exact).abs() <= bound).all()


# remainders of a vector, rows of one to three workgroups' columns, rows shorter than a vector, and whole unaligned rows
@pytest.mark.parametrize("C,dtype,shift", [(1, torch.bfloat16, False), (7, torch.float16, True), (9, torch.bfloat16, False),
                                           (255, torch.float32, False), (257, torch.bfloat16, True), (301, torch.float16, False),
                                           (513, torch.float32, True), (64, torch.bfloat16, True), (3, torch.float64, False),
                                           (300, torch.float64, False)])
@pytest.mark.parametrize("n,V", [(0, 5), (1, 3), (63, 1), (64, 7), (65, 2), (129, 40), (256, 9), (257, 9), (1000, 30),
                                 (2731, 500), (3072, 70), (3073, 70), (4097, 3000), (9001, 90)])
def test_ragged_rows(C, dtype, shift, n, V):
    from core_scheduler_amd import ops

    place = off_by_one if shift else (lambda t: t.cuda())
    ids = randint(0, V, (n,), 1)
    ids[n // 3: n // 3 + n // 2] = V // 2  # a hot row: half of the windows lie in it whole
    if n > 10:
        ids[3], ids[7] = -1, V  # out of range: no row
    dout, wte = randn((n, C), 2, dtype=dtype), randn((V, C), 3, dtype=dtype)
    ok = (ids >= 0) & (ids < V)
    want = torch.where(ok[:, None], wte[ids.clamp(0, V - 1)], torch.zeros((), dtype=dtype))
    d_ids, d_dout = ids.cuda(), place(dout)
    assert torch.equal(ops.embedding_forward(place(wte), d_ids).cpu(), want)
    got = ops.embedding_backward(d_dout, d_ids, V)
    keep, at = dout.double()[ok], ids[ok]
    exact = torch.zeros(V, C, dtype=torch.float64).index_add_(0, at, keep)
    terms = torch.zeros(V, C, dtype=torch.float64).index_add_(0, at, keep.abs())
    assert rounded_once(got.cpu(), exact, terms)
    assert torch.equal(got, ops.embedding_backward(d_dout, d_ids.int(), V))
    # padding index, gradient that is there already, division by the count
    pad = V // 2
    base = randn((V, C), 4, dtype=dtype)
    acc = ops.embedding_backward(d_dout, d_ids, V, padding_idx=pad, dweight=place(base)).cpu()
    other = torch.arange(V) != pad
    assert torch.equal(acc[pad], base[pad])
    assert rounded_once(acc[other], exact[other] + base.double()[other], terms[other] + base.double()[other].abs())
    count = torch.bincount(at, minlength=V).clamp(min=1).double()[:, None]
    mean = ops.embedding_backward(d_dout, d_ids, V, scale_grad_by_freq=True).cpu()
    assert rounded_once(mean, exact / count, terms)


@pytest.mark.parametrize("n,C,positions,want", [(300, 301, False, "scalar"), (1000, 65, True, "scalar"), (2000, 301, True, "vec"),
                                                (2, 3, False, "scalar"), (300000, 7, False, "scalar")])
def test_gather_by_elements_or_vectors(n, C, positions, want):
    """Few elements are gathered one by one, rows shorter than a vector always: the same bits."""
    from core_scheduler_amd import ops

    ids, wte, wpe = randint(-1, 52, (1, n), 1).cuda(), randn((50, C), 2).bfloat16().cuda(), randn((n, C), 3).bfloat16().cuda()
    call = (lambda: ops.embedding_forward_add(wte, wpe, ids)) if positions else (lambda: ops.embedding_forward(wte, ids))
    call()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        got = call()
        torch.cuda.synchronize()
    assert [e.name.split("emb_fwd_")[1].split("_")[0] for e in prof.events() if "emb_fwd_" in e.name] == [want]
    ok = ((ids >= 0) & (ids < 50))[..., None]
    rows = wte[ids.clamp(0, 49)]
    rows = (rows.float() + wpe.float()).bfloat16() if positions else rows
    assert torch.equal(got, torch.where(ok, rows, torch.zeros((), dtype=rows.dtype, device="cuda")))


@pytest.mark.parametrize("n,C,want", [(256, 301, ["runs"]), (257, 301, ["runs", "finish"]), (3072, 301, ["runs", "finish"]),
                                      (3073, 301, ["reduce", "finish"]), (2731, 513, ["reduce", "finish"])])
def test_launches_of_a_list(n, C, want):
    """A short list has a workgroup per entry, and no second launch where that adds whole runs."""
    from core_scheduler_amd import ops

    ids, dout = randint(0, 50, (n,), 1).cuda(), randn((n, C), 2).cuda()
    ops.embedding_backward(dout, ids, 50)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        ops.embedding_backward(dout, ids, 50)
        torch.cuda.synchronize()
    names = [e.name.split("_ragged")[0].split("emb_bwd_")[1] for e in prof.events() if "_ragged_kernel" in e.name]
    assert names == want


@pytest.mark.parametrize("B,T,C,dtype,shift", [(1, 1, 9, torch.bfloat16, False), (3, 50, 301, torch.float32, False),
                                               (17, 65, 257, torch.float16, False), (9, 33, 64, torch.bfloat16, True),
                                               (40, 65, 301, torch.bfloat16, False), (10, 900, 64, torch.bfloat16, True)])
def test_ragged_positions(B, T, C, dtype, shift):
    from core_scheduler_amd import ops

    place = off_by_one if shift else (lambda t: t.cuda())
    V = 70
    ids = randint(0, V, (B, T), 5)
    wte, wpe, dout = randn((V, C), 6, dtype=dtype), randn((T + 2, C), 7, dtype=dtype), randn((B, T, C), 8, dtype=dtype)
    got = ops.embedding_forward_add(place(wte), place(wpe), ids.cuda()).cpu()
    assert torch.equal(got, (wte[ids].float() + wpe[None, :T].float()).to(dtype))
    dwte, dwpe = ops.embedding_backward_fused(place(dout), ids.cuda(), V)
    d = dout.double()
    assert rounded_once(dwpe.cpu(), d.sum(0), d.abs().sum(0))
    exact = torch.zeros(V, C, dtype=torch.float64).index_add_(0, ids.reshape(-1), d.reshape(-1, C))
    assert rounded_once(dwte.cpu(), exact, torch.zeros_like(exact).index_add_(0, ids.reshape(-1), d.reshape(-1, C).abs()))


def test_nothing_beside_the_table_is_written():
    """A table that starts and ends off a 16-byte boundary, inside a larger buffer."""
    from core_scheduler_amd import _capi

    lib = _capi.load()
    for V, C, lead in ((5, 3, 1), (1, 1, 3), (11, 9, 7), (4, 2, 5)):
        buf = torch.full((V * C + 32,), 7.0, dtype=torch.bfloat16, device="cuda")
        ids, dout = torch.zeros(2, dtype=torch.int64, device="cuda"), torch.ones(2, C, dtype=torch.bfloat16, device="cuda")
        size = lib.cs_embedding_backward_workspace_bytes(2, C, V)
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        code = lib.cs_embedding_backward(dout.data_ptr(), ids.data_ptr(), buf.data_ptr() + 2 * lead, ws.data_ptr(), size, 2, C,
                                         V, -1, _capi.BF16, _capi.I64, 0, torch.cuda.current_stream().cuda_stream)
        assert code == _capi.OK
        want = torch.full_like(buf, 7.0)
        want[lead:lead + V * C] = 0
        want[lead:lead + C] = 2
        assert torch.equal(buf, want)


@pytest.mark.parametrize("n", [33, 64, 65, 97, 4129])
def test_nothing_behind_the_workspace_is_written(n):
    """The partial rows fit the workspace of a float row per slot of each 32 entries, whatever the remainder."""
    from core_scheduler_amd import _capi

    lib, V, C = _capi.load(), 3, 301
    ids, dout = torch.ones(n, dtype=torch.int64, device="cuda"), randn((n, C), 1).cuda()
    size = lib.cs_embedding_backward_workspace_bytes(n, C, V)
    assert size <= 4 * 1024 * -(-n // 1024) + 8 * n + 8 * C * -(-n // 32) + 4 * 256
    ws = torch.full((size + 65536,), 77, dtype=torch.uint8, device="cuda")
    dw = torch.empty(V, C, device="cuda")
    code = lib.cs_embedding_backward(dout.data_ptr(), ids.data_ptr(), dw.data_ptr(), ws.data_ptr(), size, n, C, V, -1, _capi.F32,
                                     _capi.I64, 0, torch.cuda.current_stream().cuda_stream)
    assert code == _capi.OK and (ws[size:] == 77).all()
    assert rounded_once(dw[1].cpu(), dout.cpu().double().sum(0), dout.cpu().double().abs().sum(0))
