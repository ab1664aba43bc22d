"""LayerNorm rows shared by several waves: widths beyond one wave's registers, ragged widths and
unaligned tensors, at the edges of the kernels' tiles, against the CPU oracle."""
import ctypes

import pytest
import torch

from _util import assert_bit_exact, assert_close, assert_sum_close, randn, sum_tolerance

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


def place(t, offset):
    """t on the GPU, its first element `offset` elements past an aligned address."""
    flat = torch.empty(t.numel() + offset, dtype=t.dtype, device="cuda:0")
    flat[offset:].copy_(t.reshape(-1))
    return flat[offset:].view(t.shape)


@pytest.mark.parametrize("rows,C,x_dtype,p_dtype,wide_dy,offset", [
    (700, 2056, BF16, F32, False, 0),    # just past a wave's 256 vectors: five waves, the last nearly empty
    (515, 4096, F16, F16, False, 0),     # 512 vectors: two per lane in the plain forward
    (260, 4104, BF16, F32, True, 0),     # 513: one per lane again; fp32 gradients of 16-bit rows
    (300, 8192, BF16, BF16, False, 0),   # 16 full waves
    (70, 8200, BF16, F32, False, 0),     # one vector more: two per lane, sums and dx in two passes
    (33, 16384, F16, F32, False, 0),     # the widest row
    (20, 16392, BF16, F32, False, 0),    # past it: the general kernels
    (1100, 1028, F32, F32, False, 0),    # fp32: 257 vectors
    (40, 16380, F32, F32, False, 0),     # four fp32 vectors per lane
    (16, 8200, F32, F32, False, 0),      # too few rows for them in the backward
    (17, 8200, F32, F32, False, 0),
    (513, 8197, F32, F32, False, 0),     # enough at a ragged width
    (64, 4100, F16, F16, False, 0),      # as many rows as the general backward kernels take, up to 512 vectors
    (65, 4100, BF16, F32, False, 0),     # one more
    (5000, 1, F32, F32, False, 0),       # no whole vector, one column
    (3000, 7, BF16, F32, False, 0),      # no whole vector
    (777, 71, F16, F16, False, 0),       # 8 vectors and 7 columns
    (4099, 513, BF16, F32, False, 0),    # 64 vectors and a column; several rows per group, the last step ragged
    (1, 1001, F32, F32, False, 0),       # a single row
    (300, 4099, F32, F32, False, 0),     # 1024 vectors (16 waves) and 3 columns
    (600, 768, BF16, F32, False, 1),     # an aligned width at an unaligned address
    (600, 768, BF16, F32, True, 3),
])
def test_layernorm_rows_on_several_waves(ops, co, rows, C, x_dtype, p_dtype, wide_dy, offset):
    g_dtype = F32 if wide_dy else x_dtype
    x, res = randn((rows, C), 900, dtype=x_dtype), randn((rows, C), 901, dtype=x_dtype)
    gamma, beta = randn(C, 902, std=0.02, mean=1.0, dtype=p_dtype), randn(C, 903, std=0.02, dtype=p_dtype)
    dy, dres = randn((rows, C), 904, dtype=g_dtype), randn((rows, C), 905, dtype=g_dtype)
    total_ref = (x.float() + res.float()).to(x_dtype)
    gx, gres, gg, gb = place(x, offset), place(res, offset), place(gamma, 0), place(beta, 0)
    y2, mean2, rstd2 = co.layernorm_forward(total_ref, gamma, beta, 1e-5)
    # with one column the variance is 0 and rstd = 1/sqrt(eps) multiplies every rounding by 316
    loose = 316 if C == 1 else 1
    total, y, mean, rstd = ops.add_layernorm_forward(gx, gres, gg, gb, 1e-5)
    assert_bit_exact(total, total_ref, "x + residual")
    assert_close(y, y2, atol=2e-6 * loose, name="y")
    assert_close(mean, mean2, atol=1e-7, name="mean")
    assert_close(rstd, rstd2, atol=1e-6 * loose, name="rstd")
    y_sep, mean_sep, rstd_sep = ops.layernorm_forward(place(total_ref, offset), gg, gb, 1e-5)
    assert_bit_exact(y_sep, y, "y without residual")
    assert_bit_exact(mean_sep, mean, "mean without residual")
    assert_bit_exact(rstd_sep, rstd, "rstd without residual")
    ops.add_layernorm_forward(gx, gres, gg, gb, 1e-5, inplace=True)
    assert_bit_exact(gx, total_ref, "in-place sum")

    gdy, gt, gm, gr, gdr = place(dy, offset), place(total_ref, offset), place(mean2, 0), place(rstd2, 0), place(dres, offset)
    dx, dg, db = ops.layernorm_backward(gdy, gt, gm, gr, gg, dx_dtype=g_dtype)
    dx2, dg2, db2 = co.layernorm_backward(dy, total_ref, mean2, rstd2, gamma, **({"out_dtype": F32} if wide_dy else {}))
    # dx = rstd * (three terms of size |dy gamma|): rstd scales their rounding
    assert_close(dx, dx2, atol=5e-6 * max(1.0, float(rstd2.max())), name="dx")
    xhat = (total_ref.double() - mean2.double().reshape(-1, 1)) * rstd2.double().reshape(-1, 1)
    assert_sum_close(dg, dg2, sum_tolerance(dy.double() * xhat), name="dgamma")
    assert_sum_close(db, db2, sum_tolerance(dy), name="dbeta")
    # each output mask gives the bits of the full call; dresidual is added to the rounded dx
    only_dx = ops.layernorm_backward(gdy, gt, gm, gr, gg, dx_dtype=g_dtype, need_dgamma=False, need_dbeta=False)[0]
    assert_bit_exact(only_dx, dx, "dx alone")
    _, dg1, db1 = ops.layernorm_backward(gdy, gt, gm, gr, gg, need_dx=False)
    assert_bit_exact(dg1, dg, "dgamma alone")
    assert_bit_exact(db1, db, "dbeta alone")
    dxr, dgr, dbr = ops.layernorm_backward(gdy, gt, gm, gr, gg, dx_dtype=g_dtype, dresidual=gdr)
    assert_bit_exact(dxr, (dx.cpu().float() + dres.float()).to(g_dtype), "dx + dresidual")
    assert_bit_exact(dgr, dg, "dgamma with dresidual")
    assert_bit_exact(dbr, db, "dbeta with dresidual")
    # += into existing gradients
    acc_g, acc_b = gg.clone(), gb.clone()
    ops.layernorm_backward(gdy, gt, gm, gr, gg, dx_dtype=g_dtype, dgamma=acc_g, dbeta=acc_b)
    # the sum is added in fp32 and rounded once: 2^-24 of the result (2^-8 or 2^-11 of it at 16 bit: one unit)
    for acc, old, terms, name in ((acc_g, gamma, dy.double() * xhat, "dgamma +="), (acc_b, beta, dy, "dbeta +=")):
        exact = terms.double().sum(0) + old.double()
        assert_sum_close(acc, exact.to(p_dtype), sum_tolerance(terms) + 1e-6, name=name)


@pytest.mark.parametrize("rows,C,dtype,offset", [
    # 257 to 512 vectors: one or two per lane of several waves, or a wave per row, by rows and residual
    (300, 2056, BF16, 0), (512, 4096, F16, 0), (513, 3072, BF16, 0), (1024, 2056, F16, 0), (1025, 4096, BF16, 0),
    (300, 1028, F32, 0), (512, 2048, F32, 0), (513, 2044, F32, 0),
    (300, 4099, BF16, 0), (300, 2051, F32, 0), (64, 4096, BF16, 3),  # the same at element alignment
    (300, 5120, BF16, 0), (40, 8200, BF16, 0), (40, 16380, F32, 0), (40, 16383, BF16, 0),  # the same plan for both
])
def test_added_residual_gives_the_bits_of_two_calls(ops, rows, C, dtype, offset):
    """x + residual inside the norm: y, mean and rstd are those of the norm of the rounded sum, bit for bit."""
    x, res = place(randn((rows, C), 920, dtype=dtype), offset), place(randn((rows, C), 921, dtype=dtype), offset)
    gamma, beta = place(randn(C, 922, std=0.02, mean=1.0), 0), place(randn(C, 923, std=0.02), 0)
    total, y, mean, rstd = ops.add_layernorm_forward(x, res, gamma, beta, 1e-5)
    y_sep, mean_sep, rstd_sep = ops.layernorm_forward(place(total, offset), gamma, beta, 1e-5)
    assert_bit_exact(mean, mean_sep, "mean")
    assert_bit_exact(rstd, rstd_sep, "rstd")
    assert_bit_exact(y, y_sep, "y")


@pytest.mark.parametrize("C,dtype,offset", [(c, F32, 0) for c in (1, 3, 41, 47, 55, 61, 1003, 6145, 16380)] + [
    (768, BF16, 1), (5120, BF16, 0), (4099, F16, 0), (12295, BF16, 0)])
@pytest.mark.parametrize("residual", [False, True])
def test_rows_of_one_value(ops, C, dtype, offset, residual):
    """Sums of one small whole number are exact, so the mean is that number and y is beta."""
    rows = 64
    v = torch.arange(1, rows + 1, dtype=F32)
    x = v[:, None].expand(rows, C).contiguous().to(dtype)
    gamma, beta = place(randn(C, 940, std=0.02, mean=1.0), 0), randn(C, 941)
    if residual:
        zero = place(torch.zeros_like(x), offset)
        y, mean, _ = ops.add_layernorm_forward(place(x, offset), zero, gamma, place(beta, 0), 1e-5, out_dtype=F32)[1:]
    else:
        y, mean, _ = ops.layernorm_forward(place(x, offset), gamma, place(beta, 0), 1e-5, out_dtype=F32)
    assert_bit_exact(mean, v, "mean")
    assert_bit_exact(y, beta.expand(rows, C), "y")


@pytest.mark.parametrize("rows,C,dtype,offset", [
    (4096, 1003, F32, 0), (515, 4099, F32, 0), (5000, 71, F16, 0), (3000, 4, F32, 1), (2000, 5, BF16, 0),  # ragged
    (600, 768, BF16, 1), (1000, 2056, BF16, 1),   # unaligned
    (3000, 4104, BF16, 0), (300, 8200, BF16, 0), (100, 16380, F32, 0), (40, 16391, F32, 0), (520, 16391, F32, 0),  # wide, and the widest
])
def test_column_sums_are_rounded_once(ops, rows, C, dtype, offset):
    """dgamma and dbeta are the double sums of the fp32 terms, rounded once: half a unit in the last place, and
    2^-53 of the terms for every add in double."""
    x, dy = randn((rows, C), 930, mean=1.0, dtype=dtype), randn((rows, C), 931, dtype=dtype)
    gamma = randn(C, 932, std=0.02, mean=1.0)
    mean, rstd = randn(rows, 933, mean=1.0, std=0.1), randn(rows, 934).abs() + 0.5
    _, dg, db = ops.layernorm_backward(place(dy, offset), place(x, offset), place(mean, 0), place(rstd, 0), place(gamma, 0))
    terms = (dy.float() * ((x.float() - mean[:, None]) * rstd[:, None])).double()
    for got, t, name in ((dg, terms, "dgamma"), (db, dy.double(), "dbeta")):
        want = t.sum(0)
        bound = 2.0 ** -24 * want.abs() + 2.0 ** -53 * rows * t.abs().sum(0)
        err = (got.cpu().double() - want).abs()
        assert (err <= bound).all(), f"{name}: {(err > bound).sum().item()} of {C} sums off"


@pytest.mark.parametrize("rows,C,dtype,offset", [
    (300, 2056, BF16, 0), (600, 3072, F16, 0), (600, 1003, F32, 0), (300, 4099, BF16, 1), (300, 5120, BF16, 0),
    (70, 8200, F16, 0), (70, 16380, F32, 0)])
@pytest.mark.parametrize("residual", [False, True])
def test_values_that_are_not_finite_stay_in_their_rows(ops, rows, C, dtype, offset, residual):
    """A row with a NaN or an infinity is NaN throughout, forward and backward; every other row has the bits it has
    without them, although rows share a wave's registers in turn and workgroups share partial rows."""
    x, dy, res = (randn((rows, C), s, dtype=dtype) for s in (980, 981, 982))
    gamma, beta = place(randn(C, 983, std=0.02, mean=1.0), 0), place(randn(C, 984, std=0.02), 0)
    bad = x.clone()
    bad[1, 0], bad[rows // 2, C - 1], bad[rows - 1, C // 2] = float("nan"), float("inf"), float("-inf")
    good_rows = torch.ones(rows, dtype=torch.bool)
    good_rows[[1, rows // 2, rows - 1]] = False
    out = []
    for v in (x, bad):
        gv, gdy, gres = place(v, offset), place(dy, offset), place(res, offset)
        if residual:
            total, y, mean, rstd = ops.add_layernorm_forward(gv, gres, gamma, beta)
        else:
            total, (y, mean, rstd) = gv, ops.layernorm_forward(gv, gamma, beta)
        dx, dg, db = ops.layernorm_backward(gdy, place(total.cpu(), offset), mean, rstd, gamma)
        out.append([t.cpu() for t in (y, mean, rstd, dx, dg, db)])
    for clean, got, name in zip(out[0][:4], out[1][:4], ("y", "mean", "rstd", "dx")):
        assert_bit_exact(got[good_rows], clean[good_rows], name)
        if name in ("y", "dx"):
            assert torch.isnan(got[~good_rows]).all(), name
    assert torch.isnan(out[1][4]).all()              # every column of dgamma sums a NaN xhat
    assert_bit_exact(out[1][5], out[0][5], "dbeta")  # dy is finite


@pytest.mark.parametrize("C,dtype", [(4096, BF16), (1003, F32), (4099, F16), (5120, BF16)])
def test_a_long_batchs_workspace_serves_a_short_one(ops, C, dtype):
    from core_scheduler_amd import _capi
    lib = _capi.load()
    dt = {F32: _capi.F32, F16: _capi.F16, BF16: _capi.BF16}[dtype]
    size = lib.cs_layernorm_backward_workspace_bytes(300, C)
    ws = torch.empty(size, dtype=torch.uint8, device="cuda:0")
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    for rows in (300, 257, 256, 200, 1):
        x, dy = place(randn((rows, C), 910, dtype=dtype), 0), place(randn((rows, C), 911, dtype=dtype), 0)
        gamma = place(randn(C, 912, std=0.02, mean=1.0), 0)
        _, mean, rstd = ops.layernorm_forward(x, gamma)
        want = ops.layernorm_backward(dy, x, mean, rstd, gamma)
        dx, dg, db = torch.empty_like(x), torch.empty_like(gamma), torch.empty_like(gamma)
        code = lib.cs_layernorm_backward(P(dy), P(x), P(mean), P(rstd), P(gamma), P(dx), P(dg), P(db), P(ws), size, rows, C,
                                         dt, dt, dt, _capi.F32, 0,
                                         ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert code == _capi.OK, rows
        for got, ref, name in zip((dx, dg, db), want, ("dx", "dgamma", "dbeta")):
            assert_bit_exact(got, ref, name)


def test_wide_rows_without_a_workspace(ops):
    """A caller that brings no workspace for a ragged width still gets its gradients."""
    from core_scheduler_amd import _capi
    rows, C = 64, 50
    x, dy = place(randn((rows, C), 910), 0), place(randn((rows, C), 911), 0)
    gamma = place(randn(C, 912, std=0.02, mean=1.0), 0)
    _, mean, rstd = ops.layernorm_forward(x, gamma)
    want = ops.layernorm_backward(dy, x, mean, rstd, gamma)
    dx, dg, db = torch.empty_like(x), torch.empty_like(gamma), torch.empty_like(gamma)
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    code = _capi.load().cs_layernorm_backward(P(dy), P(x), P(mean), P(rstd), P(gamma), P(dx), P(dg), P(db), None, 0, rows,
                                              C, 0, 0, 0, 0, 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert code == _capi.OK
    for got, ref, name in zip((dx, dg, db), want, ("dx", "dgamma", "dbeta")):
        assert_close(got, ref.cpu(), atol=1e-5, name=name)
