"""The unpadded forward convolution of square kernels of 4 to 7 against the same sum in float32 on the host, term for term: equal bits.
Odd and even channel counts, windows that end at the input's last row and column and before it, strides, depthwise, and the
cases it leaves to the masked walk."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Ci,H,W,O,k,stride,groups", [
    (2, 1, 5, 5, 3, 5, 1, 1), (3, 2, 9, 7, 5, 5, 1, 1), (2, 3, 10, 11, 4, 4, 2, 1), (1, 6, 14, 14, 16, 5, 1, 1), (2, 5, 8, 9, 3, 6, 1, 1),
    (2, 4, 15, 16, 2, 7, 3, 1), (1, 7, 12, 13, 7, 4, 1, 7), (5, 1, 32, 32, 6, 5, 1, 1)])
@pytest.mark.parametrize("pad", [0, 1])
def test_equals_ordered_float32_sum(B, Ci, H, W, O, k, stride, groups, pad):
    import torch
    from n2d2_amd import capi, runtime as rt
    print("window", B, Ci, H, W, O, k, stride, groups, pad, flush=True)
    rng = np.random.default_rng(B + H + k)
    cw = Ci // groups
    x, w = (rng.normal(size=s).astype(np.float32) for s in ((B, Ci, H, W), (O, cw, k, k)))
    bias, y0 = rng.normal(size=O).astype(np.float32), None
    oh, ow = (H + 2 * pad - k) // stride + 1, (W + 2 * pad - k) // stride + 1
    y0 = rng.normal(size=(B, O, oh, ow)).astype(np.float32)
    xp = np.pad(x, ((0, 0), (0, 0), (pad, pad), (pad, pad)))
    want = np.zeros((B, O, oh, ow), np.float32)
    for c in range(cw):
        for i in range(k):
            for j in range(k):
                src = xp[:, :, i:i + stride * (oh - 1) + 1:stride, j:j + stride * (ow - 1) + 1:stride]
                src = src[:, c:c + 1] if groups == 1 else src       # (depthwise: one channel each)
                want = want + w[None, :, c, i, j, None, None] * src  # (a tap in the padding adds a signed zero)
    want = bias[None, :, None, None] + (want + np.float32(0.5) * y0)
    d = capi.ConvDesc(Ci, O, k, k, stride, stride, pad, pad, pad, pad, 1, 1, groups, 0, capi.KERNEL_F32_DIRECT)
    dev = lambda a: torch.from_numpy(a).cuda()
    dx, dw, db, dy = dev(x), dev(w), dev(bias), dev(y0)
    n = int(capi.lib.n2d2hip_conv2d_f32_workspace_bytes(C.byref(d), B, H, W))
    ws = torch.empty(max(n, 8), dtype=torch.uint8, device="cuda")
    capi.check(capi.lib.n2d2hip_conv2d_f32_forward(C.byref(d), B, H, W, dx.data_ptr(), dw.data_ptr(), db.data_ptr(), 0.5, dy.data_ptr(), ws.data_ptr(), n,
                                                   rt.stream_ptr()))
    torch.cuda.synchronize()
    got = dy.cpu().numpy()
    if H == k + 2 * pad or (oh == 1 and ow == 1):        # (a kernel that spans its input has one more order: 4 running sums)
        assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))
    else:
        assert np.array_equal(got, want)
