"""Argument checks of core_scheduler_amd.ops that run before anything touches a device.

The kernels take one element type and one element count for a parameter, its gradient and its
optimizer state, and add into an existing embedding gradient with the incoming gradient's type
and row length; a mismatch must raise instead of reading or writing past a buffer.
"""
import pytest
import torch

from core_scheduler_amd import ops

HP = dict(lr=1e-3, beta1=0.9, beta2=0.999, eps=1e-8, weight_decay=0.0, t=1)


@pytest.mark.parametrize("which", ["dw", "m", "v", "v_max"])
@pytest.mark.parametrize("fault", ["dtype", "numel"])
def test_adamw_step_rejects_mismatched_tensors(which, fault):
    t = {k: torch.zeros(16) for k in ("w", "dw", "m", "v", "v_max")}
    t[which] = torch.zeros(16, dtype=torch.bfloat16) if fault == "dtype" else torch.zeros(8)
    with pytest.raises(ValueError, match="AdamW"):
        ops.adamw_step(t["w"], t["dw"], t["m"], t["v"], v_max=t["v_max"], **HP)


def test_multi_tensor_adamw_rejects_mixed_parameter_dtypes():
    with pytest.raises(ValueError, match="one dtype"):
        ops.MultiTensorAdamW([torch.zeros(4), torch.zeros(4, dtype=torch.bfloat16)],
                             [torch.zeros(4), torch.zeros(4, dtype=torch.bfloat16)])


@pytest.mark.parametrize("bad", [torch.zeros(10, 8, dtype=torch.float64), torch.zeros(10, 4), torch.zeros(9, 8)])
def test_embedding_backward_rejects_a_gradient_of_another_type_or_shape(bad):
    dout, ids = torch.zeros(4, 8), torch.zeros(4, dtype=torch.int64)
    with pytest.raises(ValueError, match="dweight"):
        ops.embedding_backward(dout, ids, 10, dweight=bad)
    with pytest.raises(ValueError, match="dwte"):
        ops.embedding_backward_fused(dout.reshape(1, 4, 8), ids.reshape(1, 4), 10, dwte=bad, dwpe=torch.zeros(4, 8))


def test_ops_refuse_cpu_tensors():
    with pytest.raises(RuntimeError, match="no CPU path"):
        ops.gelu_forward(torch.zeros(8))


@pytest.mark.parametrize("short", ["dy", "mean", "rstd", "gamma", "mean type", "rstd type"])
@pytest.mark.parametrize("call", [ops.layernorm_backward, ops.layernorm_backward_rows,
                                  lambda *t: ops.LayerNormBackwardChain().backward(*t)])
def test_layernorm_backward_rejects_operands_it_would_read_past(call, short):
    t = dict(dy=torch.zeros(4, 16), x=torch.zeros(4, 16), mean=torch.zeros(4), rstd=torch.ones(4), gamma=torch.ones(16))
    name = short.split()[0]
    t[name] = t[name].bfloat16() if short.endswith("type") else t[name][:3]
    with pytest.raises(ValueError, match="must"):
        call(*t.values())


@pytest.mark.parametrize("bad", [torch.zeros(15), torch.zeros(16, dtype=torch.float64)])
@pytest.mark.parametrize("which", ["dgamma", "dbeta"])
def test_layernorm_backward_rejects_sums_it_would_write_past(which, bad):
    sums = dict(dgamma=torch.zeros(16), dbeta=torch.zeros(16))
    sums[which] = bad
    with pytest.raises(ValueError, match="dgamma / dbeta"):
        ops.layernorm_backward(torch.zeros(4, 16), torch.zeros(4, 16), torch.zeros(4), torch.ones(4), torch.ones(16), **sums)


def test_embedding_backward_rejects_rows_or_indices_it_would_read_past():
    with pytest.raises(ValueError, match="dout"):
        ops.embedding_backward(torch.zeros(3, 8), torch.zeros(4, dtype=torch.int64), 10)
    with pytest.raises(ValueError, match="indices"):
        ops.embedding_backward_fused(torch.zeros(1, 4, 8), torch.zeros(1, 3, dtype=torch.int64), 10)
