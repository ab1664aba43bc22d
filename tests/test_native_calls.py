"""The native forms of the calls of ops.py (csrc/host/src/calls.cpp): the same results as the Python bodies, and every
call that is not the plain case is left to them."""
import importlib
import timeit
import warnings

import pytest
import torch

from core_scheduler_amd import ops

NATIVE = [n for n in vars(ops) if n.startswith("_") and n[1:] in dir(ops._calls) and not n.startswith("__")]


class Sub(torch.Tensor):
    pass


def test_every_native_form_is_built_and_used():
    assert sorted(n[1:] for n in NATIVE) == sorted(n for n in dir(ops._calls) if not n.startswith("_"))


def test_a_broken_extension_is_reported(monkeypatch):
    def load(error):
        def fail(name):
            raise error
        monkeypatch.setattr(importlib, "import_module", fail)
        return ops._load_calls()

    with pytest.warns(RuntimeWarning, match="undefined symbol"):
        assert load(ImportError("_cs_calls.so: undefined symbol: cs_gelu_forward")) is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert load(ModuleNotFoundError("not built", name="core_scheduler_amd._cs_calls")) is None


def test_what_is_not_plain_is_left_alone():
    x, ids = torch.zeros(4, 8), torch.zeros(4, dtype=torch.int64)  # on the CPU
    c = ops._calls
    for out in (c.gelu_forward(x, "none"), c.gelu_forward(None, "none"), c.gelu_forward(x), c.gelu_backward(x, x, 3),
                c.layernorm_forward(x, x, None, 1e-5, None), c.embedding_forward(x, ids),
                c.embedding_backward(x, ids, 10, -1, False), c.embedding_backward_fused(x, ids, 10),
                c.fused_classifier(x, ids, None, -100, "mean", 1.0, True, None, None)):
        assert out is NotImplemented


def test_leaving_a_call_alone_is_cheap():
    """The Python body's call comes on top: no exception may stand between (2.5 us and more; the whole body takes 7)."""
    x, c = torch.zeros(4, 8), ops._calls

    def best(fn, *args):
        return min(timeit.repeat(lambda: fn(*args), number=2000, repeat=15)) / 2000

    nothing = best(c.gelu_forward, x)  # a wrong number of arguments: the way there and back
    for fn, args in ((c.gelu_forward, (x, "none")), (c.add_layernorm_forward, (x, x, x, None, 1, None)),
                     (c.layernorm_backward_chained, (x, x, x, x, x, None, None, None, None, None, False)),
                     (c.fused_classifier, (x, x, None, -100, "mean", 1, True, None, None))):
        assert fn(*args) is NotImplemented
        assert best(fn, *args) < 5 * nothing + 0.5e-6


def _calls(dt):
    g = torch.Generator(device="cuda").manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dt)
    x, res, dy = r(2, 33, 72), r(2, 33, 72), r(2, 33, 72)
    pt = dt if dt == torch.float64 else torch.float32
    gamma, beta = r(72).to(pt) + 1, r(72).to(pt)
    ids = torch.randint(0, 50, (2, 33), generator=g, device="cuda")
    w, p = r(50, 72), r(40, 72)
    logits, t = r(66, 72), torch.randint(0, 70, (66,), generator=g, device="cuda")
    mean, rstd = ops.layernorm_forward(x, gamma, beta)[1:]
    cw = torch.rand(70, generator=g, device="cuda")

    def chain():
        c = ops.LayerNormBackwardChain()
        a = c.backward(dy, x, mean, rstd, gamma)
        b = c.backward(res, x, mean, rstd, gamma, dresidual=a[0])
        c.flush()
        return a + b

    return [lambda: ops.gelu_forward(x, "tanh"), lambda: ops.gelu_forward(x[:0]), lambda: ops.gelu_backward(dy, x),
            lambda: ops.layernorm_forward(x, gamma), lambda: ops.layernorm_forward(x, gamma, beta, 1e-3, torch.float32),
            lambda: ops.layernorm_forward(x, gamma, beta, 1), lambda: ops.add_layernorm_forward(x, res, gamma, beta),
            lambda: ops.layernorm_backward(dy, x, mean, rstd, gamma),
            lambda: ops.layernorm_backward(dy, x, mean, rstd, gamma, dresidual=res),
            lambda: ops.layernorm_backward(dy, x, mean, rstd, gamma, need_dbeta=False), chain,
            lambda: ops.embedding_forward(w, ids), lambda: ops.embedding_forward(w, ids.int()[0, 0]),
            lambda: ops.embedding_forward_add(w, p, ids), lambda: ops.embedding_backward(dy, ids, 50, padding_idx=4),
            lambda: ops.embedding_backward(dy, ids, 50, scale_grad_by_freq=True),
            lambda: ops.embedding_backward_fused(dy, ids, 50), lambda: ops.fused_classifier(logits, t, 70, reduction="sum"),
            lambda: ops.fused_classifier(logits, t, 70, class_weight=cw, dlogits_dtype=torch.float32),
            lambda: ops.fused_classifier(logits, t, want_dlogits=False, reduction="none", dloss=2),
            lambda: ops.gelu_forward(torch.nn.Parameter(x)), lambda: ops.gelu_forward(x.as_subclass(Sub))]


def _raises(dt):
    x, gamma = torch.zeros(4, 16, device="cuda", dtype=dt), torch.ones(16, device="cuda")
    ids, st = torch.zeros(4, dtype=torch.int64, device="cuda"), torch.float64 if dt == torch.float64 else torch.float32
    return [lambda: ops.gelu_forward(x, "sigmoid"), lambda: ops.gelu_forward(x.t()), lambda: ops.gelu_forward(x.int()),
            lambda: ops.gelu_backward(x, x[:2]), lambda: ops.layernorm_forward(x, gamma[:8]),
            lambda: ops.layernorm_forward(x.cpu(), gamma), lambda: ops.add_layernorm_forward(x, x[:2], gamma),
            lambda: ops.layernorm_backward(x, x, gamma, gamma, gamma, dresidual=x[:2]),
            lambda: ops.layernorm_backward(x[:3], x, gamma.to(st)[:4], gamma.to(st)[:4], gamma),
            lambda: ops.layernorm_backward(x, x, gamma.to(st)[:3], gamma.to(st)[:4], gamma),
            lambda: ops.layernorm_backward(x, x, gamma.half()[:4], gamma.to(st)[:4], gamma),
            lambda: ops.LayerNormBackwardChain().backward(x, x, gamma.to(st)[:4], gamma.to(st)[:3], gamma),
            lambda: ops.LayerNormBackwardChain().backward(x, x, gamma.to(st)[:4], gamma.to(st)[:4], gamma[:8]),
            lambda: ops.embedding_backward(x[:3], ids, 10), lambda: ops.embedding_backward_fused(x[None], ids[:3], 10),
            lambda: ops.embedding_forward(x, ids.float()), lambda: ops.embedding_forward_add(x, x[:, :8], ids[None]),
            lambda: ops.embedding_backward(x, ids, 0), lambda: ops.fused_classifier(x, ids.int()),
            lambda: ops.fused_classifier(x, ids, 17), lambda: ops.fused_classifier(x, ids, reduction="max")]


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float64])
def test_same_results_and_refusals(dt, monkeypatch):
    def outcomes(calls):
        out = []
        for call in calls:
            try:
                r = call()
                out.append([t if t is None else (type(t), t.dtype, t.stride(), t.cpu()) for t in
                            (r if isinstance(r, tuple) else (r,))])
            except Exception as e:
                out.append((type(e), str(e)))
        return out

    native = outcomes(_calls(dt)), outcomes(_raises(dt))
    with torch.inference_mode():
        assert ops.gelu_forward(torch.ones(8, device="cuda")).is_inference()
    for n in NATIVE:
        monkeypatch.setattr(ops, n, lambda *args: NotImplemented)
    plain = outcomes(_calls(dt)), outcomes(_raises(dt))
    for a, b in zip(native[0], plain[0]):
        assert len(a) == len(b) and all((p is None and q is None) or (p[:3] == q[:3] and torch.equal(p[3], q[3]))
                                        if not isinstance(p, (type, str)) else p == q for p, q in zip(a, b)), (a, b)
    assert native[1] == plain[1] and all(isinstance(r, tuple) for r in native[1]), native[1]
