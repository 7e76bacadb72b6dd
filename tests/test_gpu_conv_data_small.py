"""Data gradients of small float layers, added in double: a rounding to float and what sums of K terms in double lose.  Channels and
pixels that do not fill a tile of 16, terms that do not fill a wave's 16 or the block's round, strides with and without a pixel
that no tap reaches, unequal paddings, one image and one channel, layers that span their input."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# B, C, H, W, O, kH, kW, stride x, y, pad left, top
CASES = [(32, 6, 14, 14, 16, 5, 5, 1, 1, 0, 0), (1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0), (3, 17, 9, 11, 5, 3, 3, 1, 1, 1, 1), (2, 16, 13, 7, 29, 3, 3, 2, 2, 1, 1), (5, 33, 8, 8, 40, 1, 1, 1, 1, 0, 0),
         (4, 3, 10, 9, 8, 2, 3, 3, 2, 0, 1), (1, 64, 14, 14, 256, 3, 3, 1, 1, 1, 1), (2, 5, 30, 4, 33, 31, 2, 1, 1, 1, 15), (2, 20, 7, 7, 11, 3, 3, 1, 3, 2, 0),
         (32, 16, 5, 5, 120, 5, 5, 1, 1, 0, 0), (7, 30, 1, 1, 9, 1, 1, 1, 1, 0, 0), (3, 2, 8, 8, 100, 8, 8, 1, 1, 0, 0)]
# A tile to each wave: tiles and channels left over, one term and the most, a tap and nine; beside them one tile and one term less or more than
# the line.  Sixteen waves to a tile, and the last K of eight.
WAVES = [((1, 17, 151, 190, 1, 1, 1, 1, 1, 0, 0), "<4, 4>"), ((31, 20, 40, 47, 8, 1, 1, 1, 1, 0, 0), "<4, 4>"), ((33, 16, 31, 30, 12, 3, 3, 2, 2, 1, 1), "<4, 4>"),
         ((7, 9, 64, 65, 112, 1, 1, 1, 1, 0, 0), "<4, 4>"), ((7, 9, 64, 65, 113, 1, 1, 1, 1, 0, 0), "<4, 1>"), ((28, 16, 32, 32, 9, 3, 3, 1, 1, 1, 1), "<4, 1>"),
         ((1, 16, 64, 449, 9, 3, 3, 1, 1, 1, 1), "<4, 4>"), ((2, 30, 9, 7, 1025, 1, 1, 1, 1, 0, 0), "<16, 1>"), ((1, 17, 5, 9, 256, 3, 3, 1, 1, 1, 1), "<16, 1>"),
         ((2, 30, 9, 7, 1024, 1, 1, 1, 1, 0, 0), "<8, 1>")]


@pytest.mark.parametrize("beta", [0.0, 0.5])
@pytest.mark.parametrize("case", CASES)
def test_adds_in_double(case, beta):
    import torch
    from n2d2_amd import capi, runtime as rt
    B, Ci, H, W, O, kH, kW, sx, sy, pl, pt = case
    print("small data gradient", case, beta, flush=True)
    rng = np.random.default_rng(sum(case))
    oH, oW = (H + 2 * pt - kH) // sy + 1, (W + 2 * pl - kW) // sx + 1
    w, dy = rng.normal(size=(O, Ci, kH, kW)).astype(np.float32), rng.normal(size=(B, O, oH, oW)).astype(np.float32)
    start = rng.normal(size=(B, Ci, H, W)).astype(np.float32)

    def data(w_, dy_):
        x = torch.zeros(B, Ci, H, W, dtype=torch.float64, requires_grad=True)
        torch.nn.functional.conv2d(x, torch.from_numpy(w_).double(), stride=(sy, sx), padding=(pt, pl)).backward(torch.from_numpy(dy_).double())
        return x.grad.numpy()
    want, mag = data(w, dy), data(np.abs(w), np.abs(dy))
    d = capi.ConvDesc(Ci, O, kW, kH, sx, sy, pl, pt, pl, pt, 1, 1, 1, 0, 0)
    dev = lambda a: torch.from_numpy(np.array(a)).cuda()
    w_, dy_, dx = dev(w), dev(dy), dev(start if beta else np.full_like(start, np.nan))
    n = int(capi.lib.n2d2hip_conv2d_f32_workspace_bytes(C.byref(d), B, H, W))
    ws = torch.empty(max(n, 16), dtype=torch.uint8, device="cuda")
    capi.check(capi.lib.n2d2hip_conv2d_f32_backward_data(C.byref(d), B, H, W, w_.data_ptr(), dy_.data_ptr(), beta, dx.data_ptr(), ws.data_ptr(), n, rt.stream_ptr()))
    torch.cuda.synchronize()
    got = dx.cpu().numpy()
    bound = np.abs(want) * 2.0 ** -24 + mag * O * kH * kW * 2.0 ** -52
    if beta:                            # (the product with beta and the sum are rounded to float)
        want = want + 0.5 * start
        bound = bound + 2.0 ** -24 * (np.abs(want) + bound) + 2.0 ** -25 * np.abs(start)
    assert (np.abs(got - want) <= bound).all()


@pytest.mark.parametrize("case,shape", WAVES, ids=str)
def test_waves_of_a_tile(case, shape):
    from n2d2_amd import capi
    with capi.launch_log() as log:
        test_adds_in_double(case, 0.0)
        test_adds_in_double(case, 0.5)
    assert [e[0] for e in log.entries] == ["conv_f32_data_small_kernel" + shape] * 2


@pytest.mark.parametrize("joint", [False, True])
def test_more_channel_tiles_than_a_grids_second_dimension(joint):
    """One output, 1x1: a gradient is one product.  65537 tiles of channels and the rest of one, two pixels."""
    import torch
    from n2d2_amd import capi, runtime as rt
    Ci = 16 * 65535 + 17
    print("small data gradient, channels", Ci, joint, flush=True)
    rng = np.random.default_rng(7)
    d = capi.ConvDesc(Ci, 1, 1, 1, 1, 1, 0, 0, 0, 0, 1, 1, 1, 0, 0)
    dev = lambda *n: torch.from_numpy(rng.normal(size=n).astype(np.float32)).cuda()
    x, w, dy = dev(1, Ci, 1, 2), dev(1, Ci, 1, 1), dev(1, 1, 1, 2)
    dw, dx = torch.full_like(w, np.nan), torch.full_like(x, np.nan)
    with capi.launch_log() as log:
        if joint:
            capi.check(capi.lib.n2d2hip_conv2d_f32_backward(C.byref(d), 1, 1, 2, x.data_ptr(), w.data_ptr(), dy.data_ptr(), 0.0, dw.data_ptr(), 0.0, dx.data_ptr(),
                                                            None, 0, rt.stream_ptr()))
        else:
            capi.check(capi.lib.n2d2hip_conv2d_f32_backward_data(C.byref(d), 1, 1, 2, w.data_ptr(), dy.data_ptr(), 0.0, dx.data_ptr(), None, 0, rt.stream_ptr()))
    torch.cuda.synchronize()
    assert any("small" in e[0] for e in log.entries)
    assert torch.equal(dx, w.reshape(1, Ci, 1, 1) * dy)
    if joint:
        want = (x.double() * dy.double()).sum(dim=3).reshape(w.shape)
        assert bool(((dw.double() - want).abs() <= 2.0 ** -24 * want.abs()).all())
