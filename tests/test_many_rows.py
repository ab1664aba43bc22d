"""More rows than one dimension of a launch counts work-items for: kernels of a workgroup per row."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _some(n):
    """Rows on either side of where the work-items of whole rows pass 2^31 and 2^32, the first and the last ones."""
    edges = [1 << 21, 1 << 23, 1 << 24, 1 << 25, 1 << 26, n]
    rows = torch.tensor(sorted({r for e in [1] + edges for r in range(e - 3, e + 3) if 0 <= r < n}), device="cuda")
    return torch.cat([rows, torch.randint(0, n, (2000,), generator=torch.Generator().manual_seed(80)).cuda()])


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("stride", [3, 8])  # unpadded, and whole vectors
def test_classifier(stride, weighted):
    from core_scheduler_amd import ops

    N, V = (1 << 26) + 5, 3
    x = torch.empty(N, stride, device="cuda", dtype=torch.bfloat16).normal_()
    t = torch.randint(-1, V, (N,), device="cuda")
    w = torch.tensor([0.5, 1.0, 1.5], device="cuda") if weighted else None
    loss, rows, d, total = ops.fused_classifier(x, t, V, reduction="sum", class_weight=w)
    at = _some(N)
    keep = t[at] >= 0
    wt = (w.double()[t[at].clamp(min=0)] if weighted else 1.0) * keep.double()
    logp = x[at, :V].double().log_softmax(1)
    want = -logp.gather(1, t[at].clamp(min=0)[:, None])[:, 0] * wt
    # as for any narrow row: 2^-19 of a probability and of a loss of this size
    assert ((rows[at].double() - want).abs() <= 2.0 ** -19 * (want.abs() + 8)).all()
    grad = (logp.exp() - torch.nn.functional.one_hot(t[at].clamp(min=0), V)) * wt[:, None]
    assert ((d[at, :V].double() - grad).abs() <= 2.0 ** -8 * grad.abs() + 2.0 ** -18).all() and not d[at, V:].any()
    # every row has its own value: positive terms, chains of 2^13 and their sums, 2^-24 each
    assert abs(loss.item() / rows.double().sum().item() - 1) <= 2.0 ** -10


def test_classifier_fp64():
    from core_scheduler_amd import ops

    N, V = (1 << 24) + 5, 3
    x = torch.empty(N, V, device="cuda", dtype=torch.float64).normal_()
    t = torch.randint(-1, V, (N,), device="cuda")
    _, rows, d, _ = ops.fused_classifier(x, t, V, reduction="sum")
    at = _some(N)
    keep = (t[at] >= 0).double()
    logp = x[at].log_softmax(1)
    want = -logp.gather(1, t[at].clamp(min=0)[:, None])[:, 0] * keep
    assert ((rows[at].double() - want).abs() <= 2.0 ** -23 * want.abs()).all()  # an fp32 number
    grad = (logp.exp() - torch.nn.functional.one_hot(t[at].clamp(min=0), V)) * keep[:, None]
    assert ((d[at] - grad).abs() <= 1e-14).all()


def test_layernorm_fp64():
    from core_scheduler_amd import ops

    N, C = (1 << 24) + 5, 3
    x, dy = (torch.empty(N, C, device="cuda", dtype=torch.float64).normal_() for _ in range(2))
    gamma = torch.tensor([0.5, 1.0, 1.5], device="cuda", dtype=torch.float64)
    y, mean, rstd = ops.layernorm_forward(x, gamma)
    dx, _, _ = ops.layernorm_backward(dy, x, mean, rstd, gamma, need_dgamma=False, need_dbeta=False)
    at = _some(N)
    mu = x[at].mean(1, keepdim=True)
    rs = (x[at].var(1, unbiased=False, keepdim=True) + 1e-5).rsqrt()
    xh, g = (x[at] - mu) * rs, dy[at] * gamma
    # up to 2^8 of rstd on a handful of roundings of 2^-53
    assert ((y[at] - xh * gamma).abs() <= 1e-12).all()
    assert ((dx[at] - rs * (g - g.mean(1, keepdim=True) - xh * (g * xh).mean(1, keepdim=True))).abs() <= 1e-10).all()
