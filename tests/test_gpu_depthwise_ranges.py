"""The filter gradient of float depthwise layers with the workspace that the query names: a channel's sum in several ranges."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# B, C, H, W, k, stride, pad: several ranges with a short last one, one range, rows shorter than a strip, blocks of one tap row
@pytest.mark.parametrize("case", [(40, 3, 31, 29, 3, 1, 1), (33, 2, 62, 61, 5, 2, 3), (64, 5, 28, 27, 3, 2, 1), (2, 4, 9, 7, 3, 1, 1), (700, 1, 3, 3, 5, 1, 2), (9, 60, 31, 30, 3, 1, 1)])
@pytest.mark.parametrize("workspace", ["whole", "short", "none", "odd address"])
def test_filter_gradient_in_ranges(case, workspace):
    import torch
    from n2d2_amd import capi, runtime
    B, Cn, H, W, k, s, p = case
    print(case, workspace, flush=True)
    rng = np.random.default_rng(sum(case))
    oH, oW = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    x, dy = (rng.normal(size=z).astype(np.float32) for z in ((B, Cn, H, W), (B, Cn, oH, oW)))
    w64 = torch.zeros(Cn, 1, k, k, dtype=torch.float64, requires_grad=True)
    mags = []
    for f in (lambda v: v, np.abs):
        w64.grad = None
        torch.nn.functional.conv2d(torch.from_numpy(f(x)).double(), w64, stride=s, padding=p, groups=Cn).backward(torch.from_numpy(f(dy)).double())
        mags.append(w64.grad.numpy().copy())
    want, mag = mags
    d = capi.ConvDesc(Cn, Cn, k, k, s, s, p, p, p, p, 1, 1, Cn, 0)
    need = int(capi.lib.n2d2hip_conv2d_f32_workspace_bytes(C.byref(d), B, H, W))
    items = B * oH * ((oW + 3) // 4)
    assert (need > 0) == (items > 6 * 256 and Cn < 40)
    ws = torch.empty(need + 16, dtype=torch.uint8, device="cuda")
    ptr, n = {"whole": (ws.data_ptr(), need), "short": (ws.data_ptr(), max(need - 8, 0)), "none": (None, 0), "odd address": (ws.data_ptr() + 4, need)}[workspace]
    xd, dyd, dw = torch.from_numpy(x).cuda(), torch.from_numpy(dy).cuda(), torch.full((Cn, 1, k, k), 2.0, device="cuda")
    for _ in range(2):          # the second adds to the first
        capi.check(capi.lib.n2d2hip_conv2d_f32_backward_filter(C.byref(d), B, H, W, xd.data_ptr(), dyd.data_ptr(), 0.0 if _ == 0 else 1.0, dw.data_ptr(), ptr, n,
                                                               runtime.stream_ptr()))
    # products rounded to float (2^-24 each), their sum in double, the result and the sum of the two rounded to float
    bound = 2 * mag * 2.0 ** -24 + 2 * np.abs(want) * 2.0 ** -23 + 1e-30
    assert (np.abs(dw.cpu().numpy().astype(np.float64) - 2 * want) <= bound).all()
