"""The filter gradient of float depthwise layers where a block takes a tap row: which form runs on either side of its lines, and the
values against 64 bits."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# B, C, H, W, k, stride -> threads of a block and its tap rows: up to 512 strips a channel, 2048, past it; many channels; too many
# strips (a channel's, all channels'); strides and both kernels.  A strip is 4 outputs of a row.
@pytest.mark.parametrize("case,form", [
    ((1, 5, 3, 2, 3, 1), (256, 1)), ((8, 6, 16, 13, 3, 1), (256, 1)), ((9, 6, 16, 13, 3, 1), (512, 1)), ((8, 171, 9, 32, 3, 1), (256, 1)),
    ((16, 7, 32, 16, 3, 1), (512, 1)), ((17, 7, 32, 16, 3, 1), (1024, 1)), ((9, 342, 33, 30, 3, 1), (256, 1)), ((20, 342, 33, 30, 3, 1), (256, 3)), ((3, 300, 26, 110, 3, 1), (1024, 1)),
    ((64, 3, 32, 16, 3, 1), (1024, 1)), ((65, 3, 32, 16, 3, 1), (256, 3)), ((5, 30, 23, 22, 3, 2), (256, 1)), ((20, 30, 57, 56, 3, 2), (1024, 1)),
    ((1, 860, 40, 118, 3, 1), (256, 3)), ((2, 9, 7, 9, 5, 1), (256, 1)), ((30, 9, 19, 17, 5, 1), (1024, 1)), ((100, 2, 32, 16, 5, 1), (1024, 1)),
    ((101, 2, 32, 16, 5, 1), (256, 5)), ((4, 11, 61, 37, 5, 2), (512, 1)), ((2, 520, 15, 30, 5, 2), (256, 1)), ((25, 520, 15, 30, 5, 2), (256, 5)),
], ids=lambda v: "x".join(map(str, v)))
def test_filter_gradient_by_tap_rows(case, form):
    import torch
    from n2d2_amd import capi, runtime
    B, Cn, H, W, k, s = case
    p = k // 2
    print(case, form, flush=True)
    rng = np.random.default_rng(sum(case))
    oH, oW = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    x, dy = (torch.from_numpy(rng.normal(size=z).astype(np.float32)) for z in ((B, Cn, H, W), (B, Cn, oH, oW)))
    # in 64 bits, tap by tap; and the same sum of magnitudes
    xp = torch.nn.functional.pad(x, (p, p, p, p)).double()
    want, mag = (torch.empty(Cn, 1, k, k, dtype=torch.float64) for _ in range(2))
    for ty in range(k):
        for tx in range(k):
            t = xp[:, :, ty:ty + s * oH:s, tx:tx + s * oW:s][:, :, :oH, :oW] * dy.double()
            want[:, 0, ty, tx], mag[:, 0, ty, tx] = t.sum((0, 2, 3)), t.abs().sum((0, 2, 3))
    d = capi.ConvDesc(Cn, Cn, k, k, s, s, p, p, p, p, 1, 1, Cn, 0)
    ws = torch.empty(int(capi.lib.n2d2hip_conv2d_f32_workspace_bytes(C.byref(d), B, H, W)) + 8, dtype=torch.uint8, device="cuda")
    xd, dyd, dw = x.cuda(), dy.cuda(), torch.full((Cn, 1, k, k), 7.0, device="cuda")
    with capi.launch_log() as log:
        capi.check(capi.lib.n2d2hip_conv2d_f32_backward_filter(C.byref(d), B, H, W, xd.data_ptr(), dyd.data_ptr(), 0.0, dw.data_ptr(), ws.data_ptr(), ws.numel(),
                                                               runtime.stream_ptr()))
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:          # (the lines were measured there)
        assert [e[0] for e in log.entries] == ["depthwise_f32_filter_kernel<%d, %d, %d, %d>" % ((k, s) + form)]
    # products rounded to float (2^-24 each), their sum in double, the result rounded to float
    assert bool(((dw.cpu().double() - want).abs() <= mag * 2.0 ** -24 + want.abs() * 2.0 ** -24 + 1e-30).all())
