"""LayerNorm backward of up to 512 rows takes its column sums straight from the rows, in one launch; the bits are those
of the row pass followed by the sum of its partial rows, which more rows take."""
import pytest
import torch

from _util import gen, randn

pytestmark = pytest.mark.gpu


# widths of each plan: two rows per wave (1 and 3 vectors a lane), a wave per row (1, 2, 4 vectors a lane)
@pytest.mark.parametrize("C,dtype", [(8, torch.bfloat16), (256, torch.float16), (264, torch.bfloat16),
                                     (768, torch.bfloat16), (776, torch.float16), (1600, torch.bfloat16),
                                     (2048, torch.bfloat16), (4, torch.float32), (384, torch.float32),
                                     (260, torch.float32), (1024, torch.float32)])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 257, 511, 512, 513])
def test_bits_of_two_launches(rows, C, dtype):
    from core_scheduler_amd import ops

    x, dy, res = (randn((rows, C), s, dtype=dtype).cuda() for s in (1, 2, 3))
    if rows == 17:
        x[16, 0] = float("inf")  # the last row is also what missing rows read
    gamma = randn((C,), 4, 0.02, 1.0).cuda()
    _, mean, rstd = ops.layernorm_forward(x, gamma)

    def two_launches(dresidual=None, **acc):
        dx, partials = ops.layernorm_backward_rows(dy, x, mean, rstd, gamma, dresidual=dresidual)
        return (dx, *ops.layernorm_backward_finalize(partials, x.dtype, gamma.dtype, **acc))

    for dresidual in (None, res):
        want = two_launches(dresidual)
        chain = ops.LayerNormBackwardChain()
        chained = chain.backward(dy, x, mean, rstd, gamma, dresidual=dresidual)
        assert (chain._pending is None) == (rows <= 512)
        chain.flush()
        got = ops.layernorm_backward(dy, x, mean, rstd, gamma, dresidual=dresidual)
        for g, w in zip(got + chained, want + want):
            assert torch.equal(torch.nan_to_num(g), torch.nan_to_num(w)) and torch.equal(g.isnan(), w.isnan())
    base = [randn((C,), s).cuda() for s in (5, 6)]
    want = two_launches(dgamma=base[0].clone(), dbeta=base[1].clone())
    got = ops.layernorm_backward(dy, x, mean, rstd, gamma, dgamma=base[0].clone(), dbeta=base[1].clone())
    only = ops.layernorm_backward(dy, x, mean, rstd, gamma, need_dgamma=False)
    assert only[1] is None and torch.equal(torch.nan_to_num(only[0]), torch.nan_to_num(want[0]))
    for g, w in zip(got, want):
        assert torch.equal(torch.nan_to_num(g), torch.nan_to_num(w))


# partial rows of 8 rows (a wave per row) and of 16 (two rows per wave) that are not full, and rows on several waves
@pytest.mark.parametrize("rows,C,dtype", [(1, 768, torch.bfloat16), (2, 1600, torch.bfloat16), (17, 768, torch.float16),
                                          (77, 1024, torch.float32), (130, 256, torch.bfloat16), (9, 257, torch.bfloat16)])
def test_rows_that_do_not_exist_add_nothing(rows, C, dtype):
    """An infinite x-hat in the last row, which stands in for missing rows: infinite in that column's dgamma, not NaN."""
    from core_scheduler_amd import ops

    x, dy = (randn((rows, C), s, dtype=dtype).cuda() for s in (1, 2))
    x[rows - 1, 5] = float("inf")
    dy[rows - 1, 5] = 2.0
    mean, rstd = torch.zeros(rows, device="cuda"), torch.ones(rows, device="cuda")  # a caller's own statistics
    _, dgamma, dbeta = ops.layernorm_backward(dy, x, mean, rstd, torch.ones(C, device="cuda"))
    assert dgamma[5] == float("inf")
    terms = dy.double() * x.double()
    bound = 2.0 ** -24 * rows * terms.abs().sum(0) + 2.0 ** -149  # fp32 terms and sums of `rows` of them
    others = torch.arange(C, device="cuda") != 5
    assert ((dgamma.double() - terms.sum(0)).abs() <= bound)[others].all()
    assert ((dbeta.double() - dy.double().sum(0)).abs() <= 2.0 ** -24 * rows * dy.double().abs().sum(0)).all()


def test_chain_of_many_and_few_rows():
    """What many rows left is added up before a call of few rows that accumulates into the same gradients."""
    from core_scheduler_amd import ops

    gamma = randn((768,), 4, 0.02, 1.0).cuda()
    calls = []
    for rows in (600, 40, 1000, 33):
        x, dy = (randn((rows, 768), s + rows, dtype=torch.bfloat16).cuda() for s in (1, 2))
        calls.append((dy, x, *ops.layernorm_forward(x, gamma)[1:], gamma))
    sums = [[torch.zeros(768, device="cuda") for _ in range(2)] for _ in range(2)]
    chain = ops.LayerNormBackwardChain()
    for c in calls:
        chain.backward(*c, dgamma=sums[0][0], dbeta=sums[0][1])
        ops.layernorm_backward(*c, dgamma=sums[1][0], dbeta=sums[1][1])
    fresh = [chain.backward(*c) for c in calls]
    chain.flush()
    assert all(torch.equal(a, b) for a, b in zip(*sums))
    for c, f in zip(calls, fresh):
        assert all(torch.equal(a, b) for a, b in zip(f, ops.layernorm_backward(*c)))


# rows of the register plans, on several waves, and of the general kernels
@pytest.mark.parametrize("rows,C,dtype", [(300, 768, torch.bfloat16), (300, 1003, torch.bfloat16), (33, 100, torch.float64)])
def test_dx_over_an_input(rows, C, dtype):
    """dx written over dy or x (a row is read before it is written, and the sums before either): as in separate buffers."""
    from core_scheduler_amd import _capi, ops

    lib, code = _capi.load(), {torch.bfloat16: _capi.BF16, torch.float64: _capi.F64}[dtype]
    x, dy = (randn((rows, C), s, dtype=dtype).cuda() for s in (1, 2))
    pt = dtype if dtype == torch.float64 else torch.float32
    gamma = randn((C,), 4, 0.02, 1.0, dtype=pt).cuda()
    _, mean, rstd = ops.layernorm_forward(x, gamma)
    want = ops.layernorm_backward(dy, x, mean, rstd, gamma)
    n = lib.cs_layernorm_backward_workspace_bytes(rows, C)
    ws = torch.empty(max(n, 256), dtype=torch.uint8, device="cuda")
    for over in (0, 1):
        ins = [dy.clone(), x.clone()]
        dg, db = torch.empty_like(gamma), torch.empty_like(gamma)
        status = lib.cs_layernorm_backward(ins[0].data_ptr(), ins[1].data_ptr(), mean.data_ptr(), rstd.data_ptr(),
                                           gamma.data_ptr(), ins[over].data_ptr(), dg.data_ptr(), db.data_ptr(), ws.data_ptr(),
                                           n, rows, C, code, code, code, _capi.F64 if pt == dtype else _capi.F32, 0,
                                           torch.cuda.current_stream().cuda_stream)
        assert status == _capi.OK
        assert torch.equal(ins[over], want[0])
        for got, w in zip((dg, db), want[1:]):  # the two forms of the several-waves sums differ by roundings of a double
            assert torch.equal(got, w) if C != 1003 else ((got - w).abs() <= 2.0 ** -23 * w.abs() + 1e-12).all()


@pytest.mark.parametrize("over,rows,C", [("gamma", 300, 768), ("gamma", 300, 1003), ("mean", 300, 300), ("mean", 301, 301),
                                         ("rstd", 300, 300), ("rstd", 301, 301)])
def test_sums_over_an_input(over, rows, C):
    """A parameter gradient written over an input, which the rows' workgroups read: the bits of separate buffers."""
    from core_scheduler_amd import _capi, ops

    lib = _capi.load()
    x, dy = (randn((rows, C), s, dtype=torch.float32).cuda() for s in (1, 2))
    gamma = randn((C,), 4, 0.02, 1.0).cuda()
    _, mean, rstd = ops.layernorm_forward(x, gamma)
    want = ops.layernorm_backward(dy, x, mean, rstd, gamma)
    n = lib.cs_layernorm_backward_workspace_bytes(rows, C)
    ws = torch.empty(max(n, 256), dtype=torch.uint8, device="cuda")
    for which in (0, 1):
        ins = dict(gamma=gamma.clone(), mean=mean.clone(), rstd=rstd.clone())
        dx, outs = torch.empty_like(x), [torch.empty_like(gamma) for _ in range(2)]
        outs[which] = ins[over]
        code = lib.cs_layernorm_backward(dy.data_ptr(), x.data_ptr(), ins["mean"].data_ptr(), ins["rstd"].data_ptr(),
                                         ins["gamma"].data_ptr(), dx.data_ptr(), outs[0].data_ptr(), outs[1].data_ptr(),
                                         ws.data_ptr(), n, rows, C, *[_capi.F32] * 4, 0,
                                         torch.cuda.current_stream().cuda_stream)
        assert code == _capi.OK
        torch.testing.assert_close(dx, want[0], rtol=0, atol=0)
        for got, w in zip(outs, want[1:]):
            # the two forms of the several-waves sums differ by roundings of a double
            assert ((got - w).abs() <= 2.0 ** -23 * w.abs() + 1e-12).all()


# the plans of the row forward, with rows at the edges of their rule (few_forward_rows)
@pytest.mark.parametrize("C,dtype,rows", [(8, torch.bfloat16, 9216), (256, torch.float16, 4608), (768, torch.bfloat16, 3072),
                                          (776, torch.bfloat16, 4096), (512, torch.float16, 4096), (4, torch.float32, 9216),
                                          (384, torch.float32, 1536), (1024, torch.float32, 2048), (1600, torch.bfloat16, 1024),
                                          (2048, torch.bfloat16, 2048)])
def test_forward_bits_of_many_rows(C, dtype, rows):
    """A short batch is normalised by a wave per row or pair of rows: the bits that a long one's waves give."""
    from core_scheduler_amd import ops

    many = 9217 + 512
    x, res = (randn((many, C), s, dtype=dtype).cuda() for s in (1, 2))
    x[0, 0], x[2, C - 1] = float("inf"), float("nan")
    gamma, beta = randn((C,), 4, 0.02, 1.0).cuda(), randn((C,), 5).cuda()
    for b, out in ((beta, None), (None, torch.float32)):
        want = ops.layernorm_forward(x, gamma, b, out_dtype=out), ops.add_layernorm_forward(x, res, gamma, b, out_dtype=out)
        for n in (1, 2, 77, rows // 2 + 1, rows, rows + 1):
            got = (ops.layernorm_forward(x[:n], gamma, b, out_dtype=out),
                   ops.add_layernorm_forward(x[:n], res[:n], gamma, b, out_dtype=out))
            for g, w in zip(sum(got, ()), sum(want, ())):
                assert torch.equal(torch.nan_to_num(g), torch.nan_to_num(w[:n])) and torch.equal(g.isnan(), w[:n].isnan())
    s = x[:77].clone()  # the sum over x itself
    got = ops.add_layernorm_forward(s, res[:77], gamma, beta, inplace=True)
    assert got[0].data_ptr() == s.data_ptr()
    for g, w in zip(got, ops.add_layernorm_forward(x, res, gamma, beta)):
        assert torch.equal(torch.nan_to_num(g), torch.nan_to_num(w[:77]))


# ragged, wide and unaligned rows: one, two and four vectors a lane, a tile of 32 columns that ends inside, the general kernels' range
@pytest.mark.parametrize("C,dtype,shift", [(257, torch.bfloat16, 0), (1003, torch.float32, 0), (768, torch.bfloat16, 1),
                                           (4099, torch.float16, 0), (5120, torch.bfloat16, 0), (9001, torch.float32, 0),
                                           (3, torch.float32, 0), (2056, torch.float32, 1)])
@pytest.mark.parametrize("rows", [1, 16, 17, 63, 300, 512, 513, 1024])
def test_wide_rows_in_one_launch(rows, C, dtype, shift):
    """dx has the bits it has in a long batch; each column sum is the double sum of its fp32 terms, rounded once."""
    from core_scheduler_amd import ops

    def put(t):
        flat = torch.empty(t.numel() + shift, dtype=t.dtype, device="cuda")[shift:]
        return flat.copy_(t.reshape(-1)).view(t.shape)

    many = 1100
    x, dy, res = (randn((many, C), s, dtype=dtype) for s in (1, 2, 3))
    gamma = randn((C,), 4, 0.02, 1.0).cuda()
    _, mean, rstd = ops.layernorm_forward(put(x), gamma)
    want = ops.layernorm_backward(put(dy), put(x), mean, rstd, gamma, dresidual=put(res))[0][:rows]
    m, r = mean[:rows].contiguous(), rstd[:rows].contiguous()
    args = put(dy[:rows]), put(x[:rows]), m, r, gamma
    dx, dgamma, dbeta = ops.layernorm_backward(*args, dresidual=put(res[:rows]))
    assert torch.equal(dx, want)
    terms_b = dy[:rows].float()
    terms_g = terms_b * ((x[:rows].float() - m.cpu()[:, None]) * r.cpu()[:, None])
    base = randn((C,), 5)
    acc = ops.layernorm_backward(*args, dgamma=base.clone().cuda(), dbeta=base.clone().cuda())
    for got, again, terms in ((dgamma, acc[1], terms_g), (dbeta, acc[2], terms_b)):
        exact, size = terms.double().sum(0), terms.double().abs().sum(0)
        assert ((got.cpu().double() - exact).abs() <= 2.0 ** -24 * exact.abs() + 2.0 ** -40 * size).all()
        exact, size = exact + base.double(), size + base.double().abs()
        assert ((again.cpu().double() - exact).abs() <= 2.0 ** -24 * exact.abs() + 2.0 ** -40 * size).all()
    for mask in (dict(need_dx=False), dict(need_dgamma=False, need_dbeta=False)):  # the bits of the full call
        part = ops.layernorm_backward(*args, **mask)
        full = ops.layernorm_backward(*args)
        assert all(p is None or torch.equal(p, f) for p, f in zip(part, full))
    only = ops.layernorm_backward(*args, need_dgamma=False)
    assert only[1] is None and torch.equal(only[2], dbeta)
