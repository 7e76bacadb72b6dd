"""Softmax around the channel count its registers hold, and the loss around the size one block adds, against 64 bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C", [1, 2, 10, 15, 16, 17, 40])
@pytest.mark.parametrize("B,H,W", [(1, 1, 1), (33, 1, 1), (5, 3, 7)])
def test_softmax(C, B, H, W):
    import torch
    from n2d2_amd import capi, runtime as rt
    print("softmax", C, B, H, W, flush=True)
    x = np.random.default_rng(C + B).normal(0, 5, size=(B, C, H, W)).astype(np.float32)
    dx, y = torch.from_numpy(x).cuda(), torch.full((B, C, H, W), 7.0, device="cuda")
    capi.check(capi.lib.n2d2hip_softmax_f32_forward(dx.data_ptr(), y.data_ptr(), B, C, H, W, rt.stream_ptr()))
    e = np.exp(x.astype(np.float64) - x.max(1, keepdims=True))
    want = e / e.sum(1, keepdims=True)
    # x - max is rounded once (2^-24 of up to 40), expf is good to 2 ulp, the sum to C / 2 ulp and the quotient to half of one
    assert np.max(np.abs(y.cpu().numpy() - want) / want) < (40 + 2 + C / 2 + 1) * 2.0 ** -23


@pytest.mark.parametrize("n", [1, 255, 257, 4095, 4096, 4097, 70001])
def test_loss(n):
    import torch
    from n2d2_amd import capi, runtime as rt
    print("loss", n, flush=True)
    rng = np.random.default_rng(n)
    t, o = (rng.normal(size=n).astype(np.float32) for _ in range(2))
    dt, do, diff, loss = torch.from_numpy(t).cuda(), torch.from_numpy(o).cuda(), torch.empty(n, device="cuda"), torch.zeros(1, dtype=torch.float64, device="cuda")
    ws = torch.empty(int(capi.lib.n2d2hip_loss_workspace_bytes(n)), dtype=torch.uint8, device="cuda")
    capi.check(capi.lib.n2d2hip_loss_f32(dt.data_ptr(), do.data_ptr(), diff.data_ptr(), n, 3, loss.data_ptr(), ws.data_ptr(), ws.numel(), rt.stream_ptr()))
    e = t.astype(np.float64) - o
    assert np.array_equal(diff.cpu().numpy(), e.astype(np.float32))
    assert abs(float(loss) - (e * e).sum() / 3) <= n * 2.0 ** -53 * (e * e).sum()
