"""The native forms of the calls of ops.py (csrc/host/src/calls.cpp): the same results as the Python bodies, and every
call that is not the plain case is left to them."""
import importlib
import timeit
import warnings

import pytest
import torch

from core_scheduler_amd import ops

NATIVE = ["_" + n for n in ("add_layernorm_forward", "embedding_backward", "embedding_backward_fused", "embedding_forward",
                            "embedding_forward_add", "fused_classifier", "gelu_backward", "gelu_forward", "layernorm_backward",
                            "layernorm_backward_chained", "layernorm_forward")]


class Sub(torch.Tensor):
    pass


def test_every_native_form_is_built_and_used():
    assert ops._calls is not None
    assert NATIVE == sorted("_" + n for n in dir(ops._calls) if not n.startswith("_"))
    for n in NATIVE:
        assert getattr(ops, n) is getattr(ops._calls, n[1:])


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

    # (call, the native forms that take it: a chain's calls are several)
    return [(lambda: ops.gelu_forward(x, "tanh"), "gelu_forward"), (lambda: ops.gelu_forward(x[:0]), "gelu_forward"),
            (lambda: ops.gelu_backward(dy, x), "gelu_backward"), (lambda: ops.layernorm_forward(x, gamma), "layernorm_forward"),
            (lambda: ops.layernorm_forward(x, gamma, beta, 1e-3, torch.float32),
             "layernorm_forward" if dt != torch.float64 else None),
            (lambda: ops.layernorm_forward(x, gamma, beta, 1), None),
            (lambda: ops.add_layernorm_forward(x, res, gamma, beta), "add_layernorm_forward"),
            (lambda: ops.layernorm_backward(dy, x, mean, rstd, gamma), "layernorm_backward"),
            (lambda: ops.layernorm_backward(dy, x, mean, rstd, gamma, dresidual=res), "layernorm_backward"),
            (lambda: ops.layernorm_backward(dy, x, mean, rstd, gamma, need_dbeta=False), None),
            # (fp64 rows have no split form: the chain's Python body asks for the whole call instead)
            (chain, "layernorm_backward_chained" if dt != torch.float64 else "layernorm_backward"),
            (lambda: ops.embedding_forward(w, ids), "embedding_forward"),
            (lambda: ops.embedding_forward(w, ids.int()[0, 0]), "embedding_forward"),
            (lambda: ops.embedding_forward_add(w, p, ids), "embedding_forward_add"),
            (lambda: ops.embedding_backward(dy, ids, 50, padding_idx=4), "embedding_backward"),
            (lambda: ops.embedding_backward(dy, ids, 50, scale_grad_by_freq=True), "embedding_backward"),
            (lambda: ops.embedding_backward_fused(dy, ids, 50), "embedding_backward_fused"),
            (lambda: ops.fused_classifier(logits, t, 70, reduction="sum"), "fused_classifier"),
            (lambda: ops.fused_classifier(logits, t, 70, class_weight=cw, dlogits_dtype=torch.float32),
             "fused_classifier" if dt != torch.float64 else None),
            (lambda: ops.fused_classifier(logits, t, want_dlogits=False, reduction="none", dloss=2), None),
            (lambda: ops.gelu_forward(torch.nn.Parameter(x)), "gelu_forward"),
            (lambda: ops.gelu_forward(x.as_subclass(Sub)), None)]


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
    taken = []  # the native forms that took a call

    def noted(name, native):
        def call(*args):
            out = native(*args)
            if out is not NotImplemented:
                taken.append(name[1:])
            return out
        return call

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

    calls, raises = _calls(dt), _raises(dt)
    for n in NATIVE:
        monkeypatch.setattr(ops, n, noted(n, getattr(ops, n)))
    native = []
    for call, form in calls:
        taken.clear()
        native += outcomes([call])
        assert set(taken) == ({form} if form and not isinstance(native[-1], tuple) else set()), (form, taken, native[-1])
    taken.clear()
    refused = outcomes(raises)
    assert not taken
    with torch.inference_mode():
        assert ops.gelu_forward(torch.ones(8, device="cuda")).is_inference()
    for n in NATIVE:
        monkeypatch.setattr(ops, n, lambda *args: NotImplemented)
    plain = outcomes([call for call, _ in calls])
    for a, b in zip(native, plain):
        assert len(a) == len(b) and all((p is None and q is None) or (p[:3] == q[:3] and torch.equal(p[3], q[3]))
                                        if not isinstance(p, (type, str)) else p == q for p, q in zip(a, b)), (a, b)
    assert refused == outcomes(raises) and all(isinstance(r, tuple) for r in refused), refused
