"""What this framework's speed is measured on: calls of `core_scheduler_amd.ops` as a training
program makes them, over the sizes, element types and options it makes them with.

Six kinds of case (the key "op"):
  classifier   softmax + cross-entropy + gradient of [N, V] logits; padded or unpadded rows, 16- or
               32-bit logits, gradients in the logits' type or (autocast) in fp32, ignored rows,
               per-class weights, or the loss alone (validation)
  layernorm    forward and backward of one norm, with or without the residual stream
  gelu         forward and backward of one activation, exact or tanh form
  embedding    gather (+ positions) and its scatter-add backward, uniform or Zipf-distributed ids
  adamw        one optimizer step of a whole GPT-2-shaped parameter set, optionally clipped
  blocks       the ops of a two-block GPT-2 training step in the order a step runs them (the matrix
               products and attention between them belong to no op of this framework)

No imports besides torch and the framework.  Inputs come from the seed alone.
"""
import math

import torch

from core_scheduler_amd import ops

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}
ADAMW = dict(lr=6e-4, beta1=0.9, beta2=0.95, eps=1e-8, weight_decay=0.1)
N_BLOCKS = 2  # of the "blocks" cases: few enough that every output can be handed back


def listed():
    return [
        # ---- the smallest calls
        # one norm of a short prompt's tokens: launches and host work are everything
        _layernorm("norm_short", rows=77, C=768, dtype="bf16", residual=True),
        # the step of a small model in fp32, the reference's default type: three blocks of width 384
        _adamw("adamw_small_model", n_layer=3, C=384, V=4095, T=256, dtype="fp32", amsgrad=False, clip=1.0),
        # two blocks of GPT-2 small on one short sequence (fine-tuning, gradient accumulation)
        _blocks("blocks_short", B=1, T=123, C=768, V=50257, dtype="bf16"),
        # validation of a few sequences: the loss alone, vocabulary unpadded as the reference keeps it
        _classifier("loss_only", N=509, V=50257, stride=50257, dtype="bf16", grad="none", reduction="mean", ignored=0.1),
        # ---- ordinary ones
        # fp32 activations through the exact form, both of them the reference's defaults
        _gelu("gelu_fp32", rows=4096, C=3072, dtype="fp32", mode="none"),
        # a table trained in fp32 with a padding index, int32 ids (the reference's test width)
        _embedding("embedding_fp32", B=8, T=500, C=512, V=4095, dtype="fp32", ids="int32", zipf=False, positions=False),
        # GPT-2 XL tokens as text distributes them: hot rows
        _embedding("embedding_xl", B=16, T=1024, C=1600, V=50257, dtype="bf16", ids="int64", zipf=True, positions=True),
        # a wide model's norm
        _layernorm("norm_wide", rows=4096, C=5120, dtype="bf16", residual=True),
        # ---- the largest
        # the classifier of the headline benchmark: GPT-2 vocabulary, padded rows
        _classifier("classifier_padded", N=8192, V=50257, stride=50304, dtype="bf16", grad="same", reduction="mean", ignored=0.0),
        # the same vocabulary unpadded, as at::log_softmax's callers hold it, gradients by the autocast rule
        _classifier("classifier_unpadded", N=6000, V=50257, stride=50257, dtype="bf16", grad="fp32", reduction="mean", ignored=0.1),
        # a vocabulary twice as large
        _classifier("classifier_wide", N=4096, V=128256, stride=128256, dtype="bf16", grad="same", reduction="sum", ignored=0.0),
        # all 124M parameters of GPT-2 small, gradients clipped by their global norm
        _adamw("adamw_gpt2", n_layer=12, C=768, V=50257, T=1024, dtype="fp32", amsgrad=False, clip=1.0),
    ]


# What a drawn case may move at most, below the largest listed one (4.0 GB).
MOST_BYTES = 3.4e9


def draw(rng):
    while True:
        case = _draw_one(rng)
        if work(case)["bytes"] <= MOST_BYTES:
            return case


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, odd=0.25):
    """A model width: mostly a multiple of 64, now and then any number."""
    c = _log_int(rng, lo, hi)
    return c if rng.random() < odd else max(64, (c + 32) // 64 * 64)


def _draw_one(rng):
    op = rng.choice(("classifier", "classifier", "layernorm", "layernorm", "gelu", "embedding", "adamw", "blocks"))
    dtype = rng.choice(("bf16", "bf16", "fp16", "fp32"))
    if op == "classifier":
        V = _log_int(rng, 1000, 152064)
        stride = V if rng.random() < 0.5 else (V + 63) // 64 * 64
        grad = rng.choice(("same", "same", "fp32", "none"))
        return _classifier(None, N=_log_int(rng, 8, 16384), V=V, stride=stride, dtype=dtype, grad=grad,
                           reduction=rng.choice(("mean", "mean", "sum", "none")),
                           ignored=rng.choice((0.0, 0.1)), weighted=rng.random() < 0.15)
    if op == "layernorm":
        return _layernorm(None, rows=_log_int(rng, 16, 16384), C=_width(rng, 64, 8192), dtype=dtype,
                          residual=rng.random() < 0.6)
    if op == "gelu":
        return _gelu(None, rows=_log_int(rng, 16, 16384), C=_width(rng, 256, 8192), dtype=dtype,
                     mode=rng.choice(("none", "tanh")))
    if op == "embedding":
        return _embedding(None, B=_log_int(rng, 1, 32), T=_log_int(rng, 16, 1024), C=_width(rng, 64, 1600, odd=0.1),
                          V=_log_int(rng, 1000, 100000), dtype=dtype, ids=rng.choice(("int32", "int64")),
                          zipf=rng.random() < 0.5, positions=rng.random() < 0.6)
    if op == "adamw":
        return _adamw(None, n_layer=rng.randint(1, 12), C=_width(rng, 64, 1024, odd=0.1), V=_log_int(rng, 1000, 50304),
                      T=1024, dtype=rng.choice(("fp32", "fp32", "bf16")), amsgrad=rng.random() < 0.25,
                      clip=rng.choice((0.0, 1.0)))
    return _blocks(None, B=_log_int(rng, 1, 8), T=_log_int(rng, 32, 1024), C=_width(rng, 256, 1600, odd=0.0),
                   V=_log_int(rng, 4095, 50257), dtype=rng.choice(("bf16", "bf16", "fp16")))


def _named(name, case):
    return case if name is None else dict(case, name=name)


def _classifier(name, *, N, V, stride, dtype, grad, reduction, ignored, weighted=False):
    return _named(name, dict(op="classifier", N=N, V=V, stride=stride, dtype=dtype, grad=grad, reduction=reduction,
                             ignored=ignored, weighted=weighted))


def _layernorm(name, *, rows, C, dtype, residual):
    return _named(name, dict(op="layernorm", rows=rows, C=C, dtype=dtype, residual=residual))


def _gelu(name, *, rows, C, dtype, mode):
    return _named(name, dict(op="gelu", rows=rows, C=C, dtype=dtype, mode=mode))


def _embedding(name, *, B, T, C, V, dtype, ids, zipf, positions):
    return _named(name, dict(op="embedding", B=B, T=T, C=C, V=V, dtype=dtype, ids=ids, zipf=zipf, positions=positions))


def _adamw(name, *, n_layer, C, V, T, dtype, amsgrad, clip):
    return _named(name, dict(op="adamw", n_layer=n_layer, C=C, V=V, T=T, dtype=dtype, amsgrad=amsgrad, clip=clip))


def _blocks(name, *, B, T, C, V, dtype):
    return _named(name, dict(op="blocks", B=B, T=T, C=C, V=V, dtype=dtype))


class _Inputs:
    """Random tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, shape, dtype, std=1.0, mean=0.0):
        return torch.empty(shape, dtype=torch.float32, device=DEVICE).normal_(mean, std, generator=self.gen).to(dtype)

    def ints(self, high, shape, dtype=torch.int64):
        return torch.randint(0, high, shape, generator=self.gen, device=DEVICE, dtype=dtype)

    def uniform(self, shape, dtype=torch.float32):
        return torch.rand(shape, generator=self.gen, device=DEVICE, dtype=dtype)

    def token_ids(self, V, shape, dtype, zipf):
        if not zipf:
            return self.ints(V, shape, dtype)
        # ranks by Zipf's law with exponent 1.1, as byte-pair tokens of text are distributed
        cdf = torch.arange(1, V + 1, dtype=torch.float64, device=DEVICE).pow(-1.1).cumsum(0)
        u = self.uniform(shape, torch.float64) * cdf[-1]
        return torch.searchsorted(cdf, u).clamp_(max=V - 1).to(dtype)


# ------------------------------------------------------------------ inputs
def prepare(case, seed):
    return _PREPARE[case["op"]](case, _Inputs(seed))


def _prepare_classifier(c, inp):
    N, V = c["N"], c["V"]
    targets = inp.ints(V, (N,))
    if c["ignored"]:
        targets[inp.uniform((N,)) < c["ignored"]] = -100
        targets[0] = 0  # not every row
    kwargs = dict(reduction=c["reduction"], want_dlogits=c["grad"] != "none")
    if c["grad"] == "fp32":
        kwargs["dlogits_dtype"] = torch.float32
    if c["weighted"]:
        kwargs["class_weight"] = inp.uniform((V,)) + 0.5
    return dict(op="classifier", logits=inp.normal((N, c["stride"]), DTYPES[c["dtype"]], 2.0), targets=targets, V=V,
                kwargs=kwargs)


def _prepare_layernorm(c, inp):
    shape, dt = (c["rows"], c["C"]), DTYPES[c["dtype"]]
    s = dict(op="layernorm", x=inp.normal(shape, dt), dy=inp.normal(shape, dt), residual=None,
             gamma=inp.normal(c["C"], torch.float32, 0.02, 1.0), beta=inp.normal(c["C"], torch.float32, 0.02))
    if c["residual"]:
        s.update(residual=inp.normal(shape, dt), dresidual=inp.normal(shape, dt))
    return s


def _prepare_gelu(c, inp):
    shape, dt = (c["rows"], c["C"]), DTYPES[c["dtype"]]
    return dict(op="gelu", x=inp.normal(shape, dt, 1.5), dy=inp.normal(shape, dt), mode=c["mode"])


def _prepare_embedding(c, inp):
    B, T, C, V, dt = c["B"], c["T"], c["C"], c["V"], DTYPES[c["dtype"]]
    ids = inp.token_ids(V, (B, T), torch.int32 if c["ids"] == "int32" else torch.int64, c["zipf"])
    return dict(op="embedding", wte=inp.normal((V, C), dt, 0.02), ids=ids, dout=inp.normal((B, T, C), dt), V=V,
                wpe=inp.normal((T, C), dt, 0.02) if c["positions"] else None)


def _gpt2_sizes(c):
    C, sizes = c["C"], [c["V"] * c["C"], c["T"] * c["C"]]
    for _ in range(c["n_layer"]):
        sizes += [C, C, 3 * C * C, 3 * C, C * C, C, C, C, 4 * C * C, 4 * C, 4 * C * C, C]
    return sizes + [C, C]


def _prepare_adamw(c, inp):
    sizes, dt = _gpt2_sizes(c), DTYPES[c["dtype"]]
    offsets, total = [], 0
    for n in sizes:
        offsets.append(total)
        total += (n + 63) // 64 * 64  # a flat buffer per kind, every tensor on an aligned offset in it

    def views(flat):
        return [flat[o:o + n] for o, n in zip(offsets, sizes)]

    w, g = inp.normal(total, dt, 0.02), inp.normal(total, dt, 1e-3)
    m, v = inp.normal(total, dt, 1e-4), inp.normal(total, torch.float32, 1e-3).square_().to(dt)
    opt = ops.MultiTensorAdamW(views(w), views(g), amsgrad=c["amsgrad"], t=100, **ADAMW)
    opt.m, opt.v = views(m), views(v)
    state = dict(op="adamw", opt=opt, w=w, m=m, v=v, v_max=None, clip=c["clip"] or None)
    if c["amsgrad"]:
        state["v_max"] = v.clone()
        opt.v_max = views(state["v_max"])
    opt.refresh(views(g))
    return state


def _prepare_blocks(c, inp):
    B, T, C, V, dt = c["B"], c["T"], c["C"], c["V"], DTYPES[c["dtype"]]
    n = 2 * N_BLOCKS + 1
    rows = B * T
    return dict(
        op="blocks", V=V, wte=inp.normal((V, C), dt, 0.02), wpe=inp.normal((T, C), dt, 0.02),
        ids=inp.token_ids(V, (B, T), torch.int64, True), targets=inp.ints(V, (rows,)),
        gamma=[inp.normal(C, torch.float32, 0.02, 1.0) for _ in range(n)],
        beta=[inp.normal(C, torch.float32, 0.02) for _ in range(n)],
        # what attention and the MLP add to the residual stream, and the gradients that come back
        branch=[inp.normal((B, T, C), dt, 0.5) for _ in range(n - 1)],
        dbranch=[inp.normal((B, T, C), dt) for _ in range(n)],
        hidden=[inp.normal((B, T, 4 * C), dt, 1.5) for _ in range(N_BLOCKS)],
        dhidden=[inp.normal((B, T, 4 * C), dt) for _ in range(N_BLOCKS)],
        logits=inp.normal((rows, (V + 63) // 64 * 64), dt, 2.0))


_PREPARE = dict(classifier=_prepare_classifier, layernorm=_prepare_layernorm, gelu=_prepare_gelu,
                embedding=_prepare_embedding, adamw=_prepare_adamw, blocks=_prepare_blocks)


# ------------------------------------------------------------------- passes
def run(state):
    return _RUN[state["op"]](state)


def _run_classifier(s):
    return ops.fused_classifier(s["logits"], s["targets"], s["V"], **s["kwargs"])


def _run_layernorm(s):
    x, gamma, beta = s["x"], s["gamma"], s["beta"]
    if s["residual"] is None:
        y, mean, rstd = ops.layernorm_forward(x, gamma, beta)
        return y, mean, rstd, ops.layernorm_backward(s["dy"], x, mean, rstd, gamma)
    total, y, mean, rstd = ops.add_layernorm_forward(x, s["residual"], gamma, beta)
    return total, y, mean, rstd, ops.layernorm_backward(s["dy"], total, mean, rstd, gamma, dresidual=s["dresidual"])


def _run_gelu(s):
    return ops.gelu_forward(s["x"], s["mode"]), ops.gelu_backward(s["dy"], s["x"], s["mode"])


def _run_embedding(s):
    if s["wpe"] is None:
        return ops.embedding_forward(s["wte"], s["ids"]), ops.embedding_backward(s["dout"], s["ids"], s["V"], padding_idx=0)
    return (ops.embedding_forward_add(s["wte"], s["wpe"], s["ids"]),
            ops.embedding_backward_fused(s["dout"], s["ids"], s["V"]))


def _run_adamw(s):
    norm = s["opt"].step(max_grad_norm=s["clip"])
    return s["w"], s["m"], s["v"], s["v_max"], norm


def _run_blocks(s):
    gamma, beta = s["gamma"], s["beta"]
    n = len(gamma)
    out = []
    # forward: embeddings, then two norms per block on the residual stream and the final one
    stream = ops.embedding_forward_add(s["wte"], s["wpe"], s["ids"])
    y, mean, rstd = ops.layernorm_forward(stream, gamma[0], beta[0])
    saved = [(stream, mean, rstd)]
    out += [stream, y, mean, rstd]
    for j in range(1, n):
        stream, y, mean, rstd = ops.add_layernorm_forward(stream, s["branch"][j - 1], gamma[j], beta[j])
        saved.append((stream, mean, rstd))
        out += [stream, y, mean, rstd]
    out += [ops.gelu_forward(h, "tanh") for h in s["hidden"]]
    out += ops.fused_classifier(s["logits"], s["targets"], s["V"])
    # backward
    out += [ops.gelu_backward(d, h, "tanh") for d, h in zip(s["dhidden"], s["hidden"])]
    chain = ops.LayerNormBackwardChain()
    dstream = None
    for j in reversed(range(n)):
        x, mean, rstd = saved[j]
        dstream, dgamma, dbeta = chain.backward(s["dbranch"][j], x, mean, rstd, gamma[j], dresidual=dstream)
        out += [dstream, dgamma, dbeta]
    chain.flush()
    out += ops.embedding_backward_fused(dstream, s["ids"], s["V"])
    return out


_RUN = dict(classifier=_run_classifier, layernorm=_run_layernorm, gelu=_run_gelu, embedding=_run_embedding,
            adamw=_run_adamw, blocks=_run_blocks)


# --------------------------------------------------------------------- work
def work(case):
    """Each input read once, each output written once; the arithmetic of the formulas as written."""
    c, op, e = case, case["op"], BYTES[case["dtype"]]
    if op == "classifier":
        n = c["N"] * c["V"]
        grad = {"same": e, "fp32": 4, "none": 0}[c["grad"]]
        # padding columns are no input; the gradient is written over the whole row
        nbytes = n * e + c["N"] * c["stride"] * grad + c["N"] * 12
        return dict(bytes=nbytes, flops=n * (8 if grad else 5))
    if op == "layernorm":
        return _layernorm_work(c["rows"], c["C"], e, c["residual"])
    if op == "gelu":
        n = c["rows"] * c["C"]
        return dict(bytes=5 * n * e, flops=40 * n)
    if op == "embedding":
        return _embedding_work(c["B"], c["T"], c["C"], c["V"], e, 4 if c["ids"] == "int32" else 8, c["positions"], c["zipf"])
    if op == "adamw":
        n = sum(_gpt2_sizes(c))
        arrays = 7 + (2 if c["amsgrad"] else 0) + (1 if c["clip"] else 0)
        return dict(bytes=arrays * n * e, flops=20 * n)
    rows, C, V = c["B"] * c["T"], c["C"], c["V"]
    hidden = rows * 4 * C
    parts = [_embedding_work(c["B"], c["T"], C, V, e, 8, True, True), _layernorm_work(rows, C, e, False)]
    parts += [_layernorm_work(rows, C, e, True)] * (2 * N_BLOCKS)
    parts += [dict(bytes=5 * hidden * e, flops=40 * hidden)] * N_BLOCKS
    parts += [dict(bytes=rows * V * e + rows * ((V + 63) // 64 * 64) * e + rows * 12, flops=8 * rows * V)]
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def _layernorm_work(rows, C, e, residual):
    n = rows * C
    return dict(bytes=(8 if residual else 5) * n * e + rows * 16 + C * 20, flops=25 * n)


def _embedding_work(B, T, C, V, e, id_bytes, positions, zipf):
    n = B * T
    # distinct table rows among n ids: all but a few where ids are uniform over a large table
    if zipf:
        norm = sum(k ** -1.1 for k in range(1, V + 1))
        distinct = sum(-math.expm1(n * math.log1p(-(k ** -1.1) / norm)) for k in range(1, V + 1))
    else:
        distinct = -V * math.expm1(n * math.log1p(-1.0 / V))
    elements = distinct * C + n * C + n * C + V * C + (2 * T * C if positions else 0)
    return dict(bytes=int(elements * e) + 2 * n * id_bytes, flops=2 * n * C)


# ---------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times what the path differs by from itself on 64-bit inputs, the worst of some
    sixty cases: 1.8e-7 of the norm and 4e-6 at one value where everything that comes back is fp32,
    3.4e-3 and 1e-2 at bf16 (one rounding of a result is 1.7e-3 and 3.9e-3), 3e-4 and 1.2e-3 at
    fp16.  A chain of blocks rounds its residual stream several times and adds it up in table rows
    of very different sizes (0.36 at one value, against the root mean square of a table that is
    mostly zeros); fp16 gradients of a mean over many rows are subnormal (3e-3)."""
    op, dtype = case["op"], case["dtype"]
    if dtype == "fp32" or case.get("grad") in ("fp32", "none"):
        return dict(rel=1e-6, max=2e-5)
    if op == "blocks":
        return dict(rel=1e-2, max=0.8)
    if dtype == "bf16":
        return dict(rel=1e-2, max=0.04)
    return dict(rel=1e-2, max=0.15) if op == "classifier" else dict(rel=1.2e-3, max=5e-3)
