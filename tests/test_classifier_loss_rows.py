"""The loss alone of many wide rows (one workgroup per row, two chunks in registers): odd and even numbers of
chunks, rows that start off every boundary, the array's last vector, values that are not finite."""
import pytest
import torch

pytestmark = pytest.mark.gpu

N = 1200  # more than four rows per CU
CASES = [
    # (dtype, V, row stride): a chunk is 256 or 512 lanes x 4 vectors
    (torch.bfloat16, 16392, 16392), (torch.bfloat16, 16447, 16447), (torch.bfloat16, 24576, 24576),
    (torch.bfloat16, 24513, 24513), (torch.bfloat16, 32705, 32768), (torch.bfloat16, 40001, 40001),
    (torch.bfloat16, 65537, 65537), (torch.bfloat16, 5, 16401), (torch.float16, 32767, 32767),
    (torch.float16, 33000, 33003), (torch.float16, 81921, 81921), (torch.float32, 8196, 8196),
    (torch.float32, 8193, 8200), (torch.float32, 10000, 10000), (torch.float32, 12289, 12289),
    (torch.float32, 16385, 16385), (torch.float32, 32770, 32770), (torch.float32, 50257, 50257),
]


def reference(x, t, V):
    x = x[:, :V]
    out = []
    for i in range(0, x.shape[0], 100):
        out.append(torch.nn.functional.cross_entropy(x[i:i + 100].double(), t[i:i + 100], reduction="none", ignore_index=-100))
    return torch.cat(out)


@pytest.mark.parametrize("dtype,V,stride", CASES)
def test_loss_of_many_rows(dtype, V, stride):
    from core_scheduler_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(V)
    x = torch.empty((N, stride), device="cuda").normal_(0, 2.0, generator=gen).to(dtype)
    x[:, V:] = 1e4  # padding counts for nothing
    t = torch.randint(0, V, (N,), generator=gen, device="cuda")
    t[::9] = -100
    t[1], t[N - 2], t[N - 1] = 0, V - 1, V - 1
    x[N - 1, V - 1] = 20.0  # the row's sum hangs on the last column
    x[2, 0] = 20.0
    loss, row, d, tw = ops.fused_classifier(x, t, V, want_dlogits=False)
    want = reference(x, t, V)
    # the sum's relative error is at most 2^-24 times the depth of its additions (below 64 in a lane, 10
    # across the workgroup) and exp2's two ulp; the logarithm and its difference round at 2^-24 of |x_max|
    torch.testing.assert_close(row.double(), want, rtol=0, atol=76 * 2.0 ** -24 + 4 * 2.0 ** -24 * 32)
    assert d is None and tw.item() == int((t >= 0).sum())
    torch.testing.assert_close(loss.double(), want.sum() / (t >= 0).sum(), rtol=2e-6, atol=0)
    w = torch.rand(V, generator=gen, device="cuda") + 0.5
    _, row_w, _, _ = ops.fused_classifier(x, t, V, want_dlogits=False, class_weight=w)
    torch.testing.assert_close(row_w, row * torch.where(t >= 0, w[t.clamp(min=0)], 0.0), rtol=1e-6, atol=0)


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 16447), (torch.float32, 12289)])
def test_not_finite(dtype, V):
    from core_scheduler_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.empty((N, V), device="cuda").normal_(0, 2.0, generator=gen).to(dtype)
    t = torch.randint(0, V, (N,), generator=gen, device="cuda")
    x[0, :] = float("-inf")
    x[1, 7] = float("nan")
    x[2, V - 1] = float("inf")
    x[3, :V // 2] = float("-inf")
    x[4, :] = torch.finfo(dtype).min
    x[5, :V - 1] = float("-inf")
    t[5] = V - 1
    x[N - 1, V - 1] = float("nan")
    _, row, _, _ = ops.fused_classifier(x, t, V, want_dlogits=False)
    want = reference(x, t, V)
    assert torch.equal(row.isnan(), want.isnan())
    fin = want.isfinite()
    assert torch.equal(row.isposinf(), want.isposinf())
    # row 4: fp32's rounding of values of that size leaves nothing of the logarithm
    fin[4] = False
    torch.testing.assert_close(row[fin].double(), want[fin], rtol=0, atol=76 * 2.0 ** -24 + 4 * 2.0 ** -24 * 32)


@pytest.mark.parametrize("N,V,dtype", [
    (2000, 50257, torch.bfloat16), (2000, 100003, torch.float16), (2000, 30001, torch.float32), (1500, 70000, torch.float32)])
def test_loss_of_confident_rows(N, V, dtype):
    """Rows whose target holds nearly all of the sum: their loss, near 0, is the sum's distance from 1.

    Every add onto a term of 1 rounds by 3.4e-8 rms (half a unit of 2^-23, uniform): up to four steps within the
    pair of chunks that holds it, and ten levels of lanes and waves: 1.3e-7, here with a tenth more.
    """
    from core_scheduler_amd import ops
    g = torch.Generator().manual_seed(967)
    x = (torch.randn((N, V), generator=g) * 2).to(dtype).to("cuda:0")
    t = torch.randint(0, V, (N,), generator=g).to("cuda:0")
    x[torch.arange(N, device="cuda:0"), t] = (18.0 + torch.randn(N, generator=g).abs()).to(dtype).to("cuda:0")
    row = ops.fused_classifier(x, t, V, want_dlogits=False)[1].double()
    want = torch.cat([torch.nn.functional.cross_entropy(x[i:i + 100].double(), t[i:i + 100], reduction="none")
                      for i in range(0, N, 100)])
    assert (row - want).square().mean().sqrt().item() < 1.4e-7
