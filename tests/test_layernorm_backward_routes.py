"""Which kernels a LayerNorm backward of few ragged or wide rows runs on: the one launch that takes the column sums with
dx only where a call wants both and lays no output over an input, the general kernels where they are shorter."""
import pytest
import torch

from _util import randn


def kernels(call):
    """Names of the LayerNorm kernels of a call, in order."""
    call()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    names = ("ln_bwd_block", "ln_bwd_dx_general", "ln_bwd_param_general", "ln_bwd_finalize")
    found = [n for e in prof.events() for n in names if n in e.name]
    assert found, [e.name for e in prof.events()]
    return found


def operands(rows, C, dtype):
    from core_scheduler_amd import ops

    x, dy = (randn((rows, C), s, dtype=dtype).cuda() for s in (1, 2))
    gamma = randn((C,), 4, 0.02, 1.0).cuda()
    return (dy, x, *ops.layernorm_forward(x, gamma)[1:], gamma)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,C,dtype", [
    (64, 257, torch.bfloat16), (64, 4099, torch.bfloat16), (16, 9001, torch.float32),
    (65, 257, torch.bfloat16), (384, 9001, torch.float32)])
def test_all_three_are_one_launch(rows, C, dtype):
    from core_scheduler_amd import ops

    args = operands(rows, C, dtype)
    assert kernels(lambda: ops.layernorm_backward(*args)) == ["ln_bwd_block"]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,C,dtype,want", [
    (16, 257, torch.bfloat16, "param_general"), (64, 4099, torch.bfloat16, "param_general"),
    (64, 9001, torch.float32, "param_general"), (64, 1003, torch.bfloat16, "block"), (64, 3, torch.float32, "param_general"),
    (65, 257, torch.bfloat16, "block"), (65, 9001, torch.float32, "block")])
def test_sums_alone(rows, C, dtype, want):
    from core_scheduler_amd import ops

    args = operands(rows, C, dtype)
    assert kernels(lambda: ops.layernorm_backward(*args, need_dx=False)) == ["ln_bwd_" + want]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,C,dtype", [(64, 9, torch.bfloat16), (64, 65, torch.float32), (16, 8200, torch.float32)])
def test_dx_alone(rows, C, dtype):
    from core_scheduler_amd import ops

    args = operands(rows, C, dtype)
    call = lambda: ops.layernorm_backward(*args, need_dgamma=False, need_dbeta=False)
    assert kernels(call) == ["ln_bwd_block"] and torch.equal(call()[0], ops.layernorm_backward(*args)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("rows,C,dtype,general", [
    (64, 257, torch.bfloat16, True), (65, 257, torch.bfloat16, False), (16, 8200, torch.float32, True),
    (17, 8200, torch.float32, False), (384, 9001, torch.float32, True), (385, 9001, torch.float32, False)])
def test_dx_over_dy(rows, C, dtype, general):
    from core_scheduler_amd import _capi, ops

    lib, code = _capi.load(), {torch.float32: _capi.F32, torch.bfloat16: _capi.BF16}[dtype]
    dy, x, mean, rstd, gamma = operands(rows, C, dtype)
    want = ops.layernorm_backward(dy, x, mean, rstd, gamma)
    n = lib.cs_layernorm_backward_workspace_bytes(rows, C)
    ws = torch.empty(max(n, 256), dtype=torch.uint8, device="cuda")
    over, dg, db = torch.empty_like(dy), torch.empty_like(gamma), torch.empty_like(gamma)

    def call():
        over.copy_(dy)
        assert lib.cs_layernorm_backward(over.data_ptr(), x.data_ptr(), mean.data_ptr(), rstd.data_ptr(), gamma.data_ptr(),
                                         over.data_ptr(), dg.data_ptr(), db.data_ptr(), ws.data_ptr(), n, rows, C, code, code,
                                         code, _capi.F32, 0, torch.cuda.current_stream().cuda_stream) == _capi.OK

    # (four vectors a lane: dx and the sums are two passes there)
    assert set(kernels(call)) == ({"ln_bwd_dx_general", "ln_bwd_param_general"} if general
                                  else {"ln_bwd_block", "ln_bwd_finalize"})
    # dx: one rounding of the stored type of results of O(1), and fp32 sums of C terms in another order
    eps = torch.finfo(dtype).eps
    assert ((over.float() - want[0].float()).abs() <= eps * want[0].float().abs() + 2.0 ** -20).all()
    for got, w in zip((dg, db), want[1:]):  # double sums, rounded once
        assert ((got - w).abs() <= 2.0 ** -23 * w.abs() + 1e-12).all()


def test_workspace_of_few_rows():
    """Rows that every call takes in one launch or on the general kernels need none; its size never falls with the rows."""
    from core_scheduler_amd import _capi

    size = _capi.load().cs_layernorm_backward_workspace_bytes
    assert size(64, 257) == size(64, 1003) == size(16, 65) == 0 < size(65, 257)
    for C in (65, 257, 1003, 9001, 16383):
        sizes = [size(rows, C) for rows in range(1, 1100)]
        assert sizes == sorted(sizes)
