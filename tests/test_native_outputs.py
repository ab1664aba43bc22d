"""Outputs of the native calls are the tensors that torch's own factories would have made."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _kind(t):
    return (type(t), t.device, t.dtype, t.shape, t.stride(), t.storage_offset(), t.untyped_storage().nbytes(), t.is_inference(),
            t.requires_grad)


@pytest.mark.parametrize("inside", ["plain", "inference", "no_grad", "autocast", "deterministic"])
def test_outputs_are_ordinary_tensors(inside):
    from core_scheduler_amd import ops

    x = torch.randn(5, 768, device="cuda").bfloat16()
    row = torch.empty_strided((1, 64), (5, 1), device="cuda").normal_()
    g = torch.ones(768, device="cuda")
    modes = {"plain": torch.enable_grad(), "inference": torch.inference_mode(), "no_grad": torch.no_grad(),
             "autocast": torch.autocast("cuda", torch.bfloat16), "deterministic": torch.enable_grad()}
    torch.use_deterministic_algorithms(inside == "deterministic")
    try:
        with modes[inside]:
            y, mean, rstd = ops.layernorm_forward(x, g)
            assert _kind(y) == _kind(torch.empty_like(x)) and _kind(mean) == _kind(torch.empty(5, device="cuda"))
            dx, dg, db = ops.layernorm_backward(x, x, mean, rstd, g)
            assert _kind(dx) == _kind(torch.empty_like(x)) and _kind(db) == _kind(torch.empty(768, device="cuda"))
            assert _kind(ops.gelu_forward(row)) == _kind(torch.empty_like(row))
            loss = ops.fused_classifier(x, torch.arange(5, device="cuda"))[0]
            assert _kind(loss) == _kind(torch.empty((), device="cuda"))
            empty = ops.gelu_forward(x[:0])
            assert _kind(empty) == _kind(torch.empty_like(x[:0]))
    finally:
        torch.use_deterministic_algorithms(False)


def test_a_profiler_sees_the_outputs():
    from core_scheduler_amd import ops

    x, g = torch.randn(5, 768, device="cuda"), torch.ones(768, device="cuda")
    _, mean, rstd = ops.layernorm_forward(x, g)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as trace:
        ops.layernorm_backward(x, x, mean, rstd, g)
    made = [e for e in trace.key_averages() if e.key == "aten::empty"]
    assert made and made[0].count >= 3  # dx, dgamma, dbeta
