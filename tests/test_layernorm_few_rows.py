"""LayerNorm backward of up to 512 rows takes its column sums straight from the rows, in one launch; the bits are those
of the row pass followed by the sum of its partial rows (LayerNormBackwardChain), which more rows take."""
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
    for dresidual in (None, res):
        chain = ops.LayerNormBackwardChain()
        want = chain.backward(dy, x, mean, rstd, gamma, dresidual=dresidual)
        chain.flush()
        got = ops.layernorm_backward(dy, x, mean, rstd, gamma, dresidual=dresidual)
        for g, w in zip(got, want):
            assert torch.equal(torch.nan_to_num(g), torch.nan_to_num(w)) and torch.equal(g.isnan(), w.isnan())
    base = [randn((C,), s).cuda() for s in (5, 6)]
    chain = ops.LayerNormBackwardChain()
    want = chain.backward(dy, x, mean, rstd, gamma, dgamma=base[0].clone(), dbeta=base[1].clone())
    chain.flush()
    got = ops.layernorm_backward(dy, x, mean, rstd, gamma, dgamma=base[0].clone(), dbeta=base[1].clone())
    only = ops.layernorm_backward(dy, x, mean, rstd, gamma, need_dgamma=False)
    assert only[1] is None and torch.equal(torch.nan_to_num(only[0]), torch.nan_to_num(want[0]))
    for g, w in zip(got, want):
        assert torch.equal(torch.nan_to_num(g), torch.nan_to_num(w))
