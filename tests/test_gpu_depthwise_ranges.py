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


@pytest.mark.parametrize("B,C,k,H,W,s,pl,pr", [(2, 3, 3, 6, 8, 1, 1, 1), (2, 3, 3, 6, 8, 1, 0, 2), (2, 3, 3, 6, 8, 1, 2, 0), (2, 3, 3, 5, 4, 1, 1, 1), (3, 2, 3, 7, 9, 1, 1, 1),
                                               (2, 2, 3, 9, 16, 2, 1, 1), (2, 2, 3, 9, 15, 2, 1, 2), (2, 2, 3, 9, 17, 2, 0, 0), (2, 2, 5, 8, 12, 1, 2, 2), (2, 2, 5, 8, 12, 1, 3, 1),
                                               (2, 2, 5, 9, 16, 2, 2, 2), (2, 2, 5, 9, 8, 1, 2, 2), (40, 4, 3, 56, 56, 1, 1, 1)])
def test_filter_of_rows_whose_ends_are_infinite(B, C, k, H, W, s, pl, pr):
    """Rows of whole and broken strips, with little and with more padding: against 64 bits (a product is rounded once, the sum in double
    and once more), and with an infinity at either end of a row, and of a row of dy, in the taps that it reaches and in no other."""
    import ctypes as ct
    import torch
    from n2d2_amd import capi, runtime as rt
    print("depthwise row ends", B, C, k, H, W, s, pl, pr, flush=True)
    rng = np.random.default_rng(k * H + W)
    pt, oH, oW = k // 2, (H + 2 * (k // 2) - k) // s + 1, (W + pl + pr - k) // s + 1
    d = capi.ConvDesc(C, C, k, k, s, s, pl, pt, pr, pt, 1, 1, C, 0, 0)
    nws = int(capi.lib.n2d2hip_conv2d_f32_workspace_bytes(ct.byref(d), B, H, W))
    ws = torch.empty(max(nws, 16), dtype=torch.uint8, device="cuda")
    for place in (None, ("x", 0), ("x", W - 1), ("dy", 0), ("dy", oW - 1)):
        x, dy = (rng.uniform(0.5, 1.5, n).astype(np.float32) for n in ((B, C, H, W), (B, C, oH, oW)))
        if place:
            (x if place[0] == "x" else dy)[1, 0, 2, place[1]] = np.inf
        X, Y, dw = torch.from_numpy(x).cuda(), torch.from_numpy(dy).cuda(), torch.empty(C * k * k, device="cuda")
        capi.check(capi.lib.n2d2hip_conv2d_f32_backward_filter(ct.byref(d), B, H, W, X.data_ptr(), Y.data_ptr(), 0.0, dw.data_ptr(), ws.data_ptr(), nws,
                                                               rt.stream_ptr()))
        want = np.zeros((C, k, k))
        for ty in range(k):
            for tx in range(k):
                oy, ox = np.arange(oH), np.arange(oW)
                iy, ix = oy * s - pt + ty, ox * s - pl + tx
                vy, vx = (iy >= 0) & (iy < H), (ix >= 0) & (ix < W)
                xs = x[:, :, iy[vy]][:, :, :, ix[vx]].astype(np.float64)
                want[:, ty, tx] = (xs * dy[:, :, oy[vy]][:, :, :, ox[vx]].astype(np.float64)).sum((0, 2, 3))
        got = dw.cpu().numpy().reshape(C, k, k).astype(np.float64)
        assert np.array_equal(np.isinf(got), np.isinf(want)) and not np.isnan(got).any()
        ok = np.isfinite(want)
        assert np.max(np.abs(got[ok] - want[ok]) / want[ok].clip(1e-9)) < 2 * 2.0 ** -24
