"""Float convolutions on the bf16 matrix cores, operands in three parts: forward, data and filter gradient against float64 at the edges of the
tiles, runs and channel chunks, and infinities, NaN and floats near the largest where a float sum has them."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# B, C, H, W, O, kH, kW, stride, pad, forward and data gradient, whichever kernel takes them (ROUTES names those of the parts): rows and channels left over (97 rows, 39 channels), runs that cross images, pixels past
# the last tile, 32 rows and less, other kernels than 3x3, strides, K ranges, sums in double
CASES = [(33, 64, 32, 32, 64, 3, 3, 1, 1), (9, 39, 31, 33, 97, 3, 3, 1, 1), (70, 32, 13, 11, 31, 3, 3, 1, 1), (5, 64, 20, 112, 40, 3, 3, 1, 0), (21, 128, 27, 27, 70, 3, 3, 2, 1),
         (12, 48, 29, 17, 80, 5, 5, 1, 2), (17, 64, 15, 40, 64, 2, 7, 1, 0), (2, 256, 14, 14, 256, 3, 3, 1, 1), (40, 96, 14, 15, 160, 3, 3, 1, 1), (64, 512, 7, 7, 129, 3, 3, 1, 1),
         (4, 64, 60, 61, 33, 1, 9, 1, 4)]


def _passes(x, w, dy, s, pad):
    import torch
    x64, w64 = (torch.from_numpy(v).double().requires_grad_() for v in (x, w))
    y = torch.nn.functional.conv2d(x64, w64, stride=s, padding=pad)
    y.backward(torch.from_numpy(dy).double())
    return y.detach().numpy(), x64.grad.numpy()


def _run(x, w, dy, s, pad, bias=None, beta=0.0, start=0.0, workspace=True, less=0, choice=0):
    import torch
    from n2d2_amd import capi, runtime as rt
    (B, Ci, H, W), (O, _, kH, kW) = x.shape, w.shape
    d = capi.ConvDesc(Ci, O, kW, kH, s, s, pad[1], pad[0], pad[1], pad[0], 1, 1, 1, 0, choice)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    x_, w_, dy_, y, dx = dev(x), dev(w), dev(dy), torch.full(dy.shape, start, device="cuda"), torch.full(x.shape, start, device="cuda")
    b_ = None if bias is None else dev(bias)
    n = int(capi.lib.n2d2hip_conv2d_f32_workspace_bytes(C.byref(d), B, H, W)) if workspace else 0
    n = max(0, n - (less(n) if callable(less) else less))
    ws = torch.empty(max(n, 16), dtype=torch.uint8, device="cuda")
    p = ws.data_ptr() if n else None
    capi.check(capi.lib.n2d2hip_conv2d_f32_forward(C.byref(d), B, H, W, x_.data_ptr(), w_.data_ptr(), None if b_ is None else b_.data_ptr(), beta, y.data_ptr(), p, n,
                                                   rt.stream_ptr()))
    capi.check(capi.lib.n2d2hip_conv2d_f32_backward_data(C.byref(d), B, H, W, w_.data_ptr(), dy_.data_ptr(), beta, dx.data_ptr(), p, n, rt.stream_ptr()))
    torch.cuda.synchronize()
    return y.cpu().numpy(), dx.cpu().numpy()


def _inputs(case, seed=0):
    B, Ci, H, W, O, kH, kW, s, p = case
    pad = (p if kH > 1 else 0, p if kW > 1 else 0)
    rng = np.random.default_rng(sum(case) + seed)
    x, w = rng.normal(size=(B, Ci, H, W)).astype(np.float32), rng.normal(size=(O, Ci, kH, kW)).astype(np.float32)
    dy = rng.normal(size=(B, O, (H + 2 * pad[0] - kH) // s + 1, (W + 2 * pad[1] - kW) // s + 1)).astype(np.float32)
    return x, w, dy, s, pad, rng


@pytest.mark.parametrize("case", CASES)
def test_against_float64(case):
    """A sum of K terms is rounded 5 times in 32 terms (and no longer than the sums in float that it stands for, K times), each time by
    2.53e-8 of it in the root mean square; the i-th of L equal steps is sqrt(i / L) of the last."""
    print("parts", case, flush=True)
    x, w, dy, s, pad, rng = _inputs(case)
    want, mag = _passes(x, w, dy, s, pad), _passes(np.abs(x), np.abs(w), np.abs(dy), s, pad)
    got = _run(x, w, dy, s, pad)
    T = w.shape[2] * w.shape[3]
    for g, t, m, k in zip(got, want, mag, (w.shape[1] * T, w.shape[0] * T)):
        assert (np.abs(g - t) <= 2.0 ** -24 * (np.abs(t) + (k + 4) * m)).all()
    # (the other kernels, which take short and padded passes, round once a term)
    for g, t, k in zip(got, want, (w.shape[1] * T, w.shape[0] * T)):
        assert np.linalg.norm(g - t) <= 1.1 * 2.53e-8 * np.sqrt(1 + k / 2) * np.linalg.norm(t)
    bias = rng.normal(size=w.shape[0]).astype(np.float32)
    y, dx = _run(x, w, dy, s, pad, bias=bias, beta=0.5, start=3.0)
    assert np.abs(y - (got[0] + np.float32(1.5) + bias[None, :, None, None])).max() <= 2.0 ** -22 * (np.abs(got[0]).max() + 5)
    assert np.abs(dx - (got[1] + np.float32(1.5))).max() <= 2.0 ** -22 * (np.abs(got[1]).max() + 2)


@pytest.mark.parametrize("case", [(9, 39, 31, 33, 97, 3, 3, 1, 1), (40, 96, 14, 15, 160, 3, 3, 1, 1), (21, 128, 27, 27, 70, 3, 3, 2, 1)])
def test_infinities_nan_and_the_largest_floats(case):
    """An infinity in one operand gives infinities of the products' signs, NaN only against a zero or another infinity; a float that
    rounds to infinity in bf16 is finite here."""
    print("parts, special values", case, flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 1)
    big = np.float32(3.4e38)
    w *= np.float32(1e-3)
    w[np.abs(w) < 1e-5] = 1e-5
    w[3, 5, 1, 1] = 0.0
    for t in (x, dy):
        flat = t.reshape(-1)
        at = rng.permutation(flat.size)[:12]
        flat[at] = [np.inf, -np.inf, np.nan, big, -big, big, -big, big, np.inf, -big, 1e-42, -1e-42]
    got = _run(x, w, dy, s, pad)
    want = _passes(x, w, dy, s, pad)
    fin = _passes(np.where(np.isfinite(x), x, 0), w, np.where(np.isfinite(dy), dy, 0), s, pad)
    mag = _passes(np.abs(np.where(np.isfinite(x), x, 0)), np.abs(w), np.abs(np.where(np.isfinite(dy), dy, 0)), s, pad)
    k = w.shape[1] * 9, w.shape[0] * 9
    for g, t, f, m, n in zip(got, want, fin, mag, k):
        assert np.array_equal(np.isnan(g), np.isnan(t)) and np.array_equal(g == np.inf, t == np.inf) and np.array_equal(g == -np.inf, t == -np.inf)
        ok = np.isfinite(t)
        assert (np.abs(g - f)[ok] <= 2.0 ** -24 * (np.abs(f) + (n + 4) * m)[ok]).all()


@pytest.mark.parametrize("case", [(2, 256, 14, 14, 256, 3, 3, 1, 1), (40, 96, 14, 15, 160, 3, 3, 1, 1), (21, 128, 27, 27, 70, 3, 3, 2, 1), (64, 512, 7, 7, 129, 3, 3, 1, 1)])
def test_workspaces_of_every_size(case):
    """A workspace that holds the laid-out weights but not the partial results, half of it, and none: all of K, within the bound of a sum that
    rounds every term."""
    print("parts, workspaces", case, flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 2)
    want, mag = _passes(x, w, dy, s, pad), _passes(np.abs(x), np.abs(w), np.abs(dy), s, pad)
    T = w.shape[2] * w.shape[3]
    for less in (16, 4 * dy.size + 16, lambda n: n // 2, lambda n: n):
        for g, t, m, k in zip(_run(x, w, dy, s, pad, less=less), want, mag, (w.shape[1] * T, w.shape[0] * T)):
            assert (np.abs(g - t) <= 2.0 ** -24 * (np.abs(t) + (k + 4) * m)).all(), less


# The kernel's stride-1 instances: tiles of 32 rows x 128 pixels, 64 x 64 and 64 x 128, runs of up to 256 positions (4) and 384 (6), nine taps and any (0), with
# sums in double and without.  Odd batches, rows, pixels and channels left over, runs of 256, 260 and 384 positions, images with and
# without rows between them; beside them what the kernel leaves to the others: too much padding of channels, too few flops, runs of 385.
ROUTES = [((65, 64, 31, 33, 70, 3, 3, 1, 1), "2, 2, 2, 4, 4, 9, false", "2, 2, 2, 4, 4, 9, false"), ((9, 64, 60, 100, 70, 3, 3, 1, 1), "2, 2, 2, 4, 6, 9, false", "2, 2, 2, 4, 6, 9, false"),
          ((40, 48, 37, 41, 80, 5, 5, 1, 2), "2, 2, 2, 4, 6, 0, false", "2, 2, 2, 4, 6, 0, false"), ((65, 64, 31, 33, 64, 2, 5, 1, 0), "2, 2, 2, 4, 4, 0, false", None),
          ((22, 256, 28, 28, 64, 1, 5, 1, 2), "2, 2, 2, 2, 4, 0, true", "2, 2, 2, 4, 4, 0, false"), ((22, 160, 28, 28, 64, 9, 1, 1, 4), "2, 2, 2, 2, 6, 0, true", "2, 2, 2, 4, 6, 0, false"),
          ((4, 160, 43, 100, 64, 3, 3, 1, 1), "2, 2, 2, 2, 6, 9, true", "2, 2, 2, 4, 6, 9, false"), ((40, 96, 14, 15, 160, 3, 3, 1, 1), "2, 2, 2, 2, 4, 9, false", "2, 2, 2, 2, 4, 9, true"),
          ((6, 64, 22, 100, 48, 3, 3, 1, 1), "2, 2, 2, 2, 6, 9, false", "2, 2, 2, 2, 6, 9, false"), ((12, 48, 29, 17, 80, 5, 5, 1, 2), "2, 2, 2, 2, 4, 0, false", "2, 2, 2, 2, 4, 0, false"),
          ((9, 47, 31, 33, 97, 3, 3, 1, 1), "2, 2, 2, 2, 4, 9, false", "2, 2, 2, 2, 4, 9, false"), ((5, 256, 14, 14, 256, 3, 3, 1, 1), "2, 2, 2, 2, 4, 9, false", "2, 2, 2, 2, 4, 9, false"),
          ((3, 64, 40, 159, 40, 3, 3, 1, 1), "2, 2, 2, 2, 6, 9, false", None), ((3, 64, 40, 160, 40, 3, 3, 1, 1), None, None),
          ((200, 32, 13, 11, 31, 3, 3, 1, 1), "1, 4, 2, 2, 4, 9, false", "1, 4, 2, 2, 4, 9, false"), ((5, 32, 71, 90, 31, 3, 3, 1, 1), "1, 4, 2, 2, 6, 9, false", "1, 4, 2, 2, 6, 9, false"),
          ((40, 32, 29, 31, 32, 5, 5, 1, 2), "1, 4, 2, 2, 4, 0, false", "1, 4, 2, 2, 4, 0, false"), ((38, 32, 29, 32, 24, 5, 5, 1, 2), "1, 4, 2, 2, 6, 0, false", "1, 4, 2, 2, 6, 0, false"),
          ((28, 160, 16, 28, 32, 9, 1, 1, 4), "1, 4, 2, 2, 6, 0, false", "2, 2, 2, 2, 6, 0, false"), ((21, 128, 27, 27, 70, 3, 3, 2, 1), "2, 2, 2, 2, 6, 9, false", None),
          ((9, 39, 31, 33, 97, 3, 3, 1, 1), None, "2, 2, 2, 2, 4, 9, false"), ((70, 32, 13, 11, 31, 3, 3, 1, 1), None, None), ((2, 256, 14, 14, 256, 3, 3, 1, 1), None, None)]


def _patch_kernels(log):
    return [e[0][len("conv_f32_patch_kernel<"):-1] for e in log.entries if e[0].startswith("conv_f32_patch_kernel")]


@pytest.mark.parametrize("case,forward,data", ROUTES, ids=str)
def test_kernel_of_every_tile_and_run(case, forward, data):
    """The kernel that each pass is to take, and what only that one gives: 5 roundings in 32 terms, of which the rests of channels are some."""
    from n2d2_amd import capi
    print("parts, kernels", case, flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 6)
    want, T = _passes(x, w, dy, s, pad), w.shape[2] * w.shape[3]
    with capi.launch_log() as log:
        got = _run(x, w, dy, s, pad)
    assert _patch_kernels(log) == [k for k in (forward, data) if k]
    assert [e[0] for e in log.entries].count("conv_f32_lay_parts_kernel") == (forward is not None) + (data is not None)
    for g, t, kernel, channels in zip(got, want, (forward, data), (w.shape[1], w.shape[0])):
        roundings = 5 * -(-channels // 32) * T if kernel else channels * T
        assert np.linalg.norm(g - t) <= 1.1 * 2.53e-8 * np.sqrt(1 + roundings / 2) * np.linalg.norm(t)
    bias = rng.normal(size=w.shape[0]).astype(np.float32)
    y, dx = _run(x, w, dy, s, pad, bias=bias, beta=0.5, start=3.0)
    assert np.abs(y - (got[0] + np.float32(1.5) + bias[None, :, None, None])).max() <= 2.0 ** -22 * (np.abs(got[0]).max() + 5)
    assert np.abs(dx - (got[1] + np.float32(1.5))).max() <= 2.0 ** -22 * (np.abs(got[1]).max() + 2)


# Forward with room for the laid-out weights alone, which adds all of K in one range: tiles of 32 rows with sums in double
@pytest.mark.parametrize("case,forward", [((50, 160, 16, 16, 32, 3, 3, 1, 1), "1, 4, 2, 2, 4, 9, true"), ((2, 160, 64, 100, 32, 3, 3, 1, 1), "1, 4, 2, 2, 6, 9, true"),
                                          ((50, 256, 16, 16, 32, 1, 5, 1, 2), "1, 4, 2, 2, 4, 0, true"), ((28, 160, 16, 28, 32, 9, 1, 1, 4), "1, 4, 2, 2, 6, 0, true")], ids=str)
def test_rows_of_32_in_one_range(case, forward):
    from n2d2_amd import capi
    print("parts, one range", case, flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 7)
    want = _passes(x, w, dy, s, pad)[0]
    with capi.launch_log() as log:
        got = _run(x, w, dy, s, pad, less=4 * dy.size + 16)[0]
    assert _patch_kernels(log)[0] == forward
    assert np.linalg.norm(got - want) <= 1.1 * 2.53e-8 * np.sqrt(1 + 5 * w.shape[1] * w.shape[2] * w.shape[3] / 64) * np.linalg.norm(want)


@pytest.mark.parametrize("case", [(65, 64, 31, 33, 70, 3, 3, 1, 1), (9, 47, 31, 33, 97, 3, 3, 1, 1), (200, 32, 13, 11, 31, 3, 3, 1, 1)])
def test_infinities_nan_and_the_largest_floats_of_every_tile(case):
    """(the kernels of these are in ROUTES)"""
    assert any(r[0] == case and r[1] and r[2] for r in ROUTES)
    test_infinities_nan_and_the_largest_floats(case)


def test_sums_term_by_term_where_they_are_asked_for():
    """N2D2HIP_KERNEL_F32_TERMS: forward rounds once a term, on the kernel that has no parts; backward is as without it."""
    import torch
    from n2d2_amd import capi, runtime as rt
    case = (33, 64, 32, 32, 64, 3, 3, 1, 1)
    print("parts, sums term by term", case, flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 8)
    plain = _run(x, w, dy, s, pad)
    with capi.launch_log() as log:
        got = _run(x, w, dy, s, pad, choice=capi.KERNEL_F32_TERMS)
    assert _patch_kernels(log) == ["2, 2, 2, 2, 4, 9, false"]        # (of the data gradient)
    assert np.array_equal(got[1], plain[1]) and not np.array_equal(got[0], plain[0])
    want = _passes(x, w, dy, s, pad)[0]
    assert np.linalg.norm(got[0] - want) <= 1.1 * 2.53e-8 * np.sqrt(1 + 64 * 9 / 2) * np.linalg.norm(want)


# Data gradients at stride 2 whose four pixels a place run together: odd and even sizes, rows, channels and pixels left over, 0 to 2 of padding, K
# ranges, runs of one unit and of two, each beside a neighbour that does not qualify (tiles between the limits, long sums, a step back, few rows)
FOURS = [((64, 64, 32, 32, 128, 3, 3, 2, 1), 2), ((66, 100, 31, 33, 70, 3, 3, 2, 1), 2), ((12, 70, 31, 30, 390, 3, 3, 2, 1), 2), ((70, 64, 32, 32, 64, 3, 3, 2, 1), 2),
         ((10, 128, 40, 41, 400, 3, 3, 2, 2), 4), ((3, 100, 57, 100, 385, 3, 3, 2, 1), 4), ((3, 64, 16, 200, 512, 3, 3, 2, 1), 0),
         ((33, 128, 27, 27, 256, 3, 3, 2, 1), 0), ((9, 70, 29, 30, 390, 3, 3, 2, 1), 0), ((70, 64, 33, 33, 64, 3, 3, 2, 0), 0), ((128, 32, 32, 32, 128, 3, 3, 2, 1), 0), ((64, 36, 48, 48, 48, 3, 3, 2, 1), 0)]


@pytest.mark.parametrize("case,units", FOURS, ids=str)
def test_strided_data_gradient_of_four_pixels_a_place(case, units):
    from n2d2_amd import capi
    with capi.launch_log() as log:
        test_against_float64(case)
        test_workspaces_of_every_size(case)
    kernels = {e[0] for e in log.entries if e[0].endswith("4>") and e[0].startswith("conv_f32_patch_kernel")}
    assert kernels == ({"conv_f32_patch_kernel<2, 2, 2, 2, %d, 9, false, 4>" % units} if units else set())


@pytest.mark.parametrize("case", [(66, 100, 31, 33, 70, 3, 3, 2, 1), (10, 128, 40, 41, 400, 3, 3, 2, 2)])
def test_strided_data_gradient_infinities_nan_and_the_largest_floats(case):
    test_infinities_nan_and_the_largest_floats(case)


# B, C, H, W, O, stride, pad y: rows of one octet, of two, three (a step of one each, of two with one left over), four and eight, ends inside an
# octet, tiles left over in both directions, no padding and two rows above, images whose last row no output reads
FILTER = [(260, 64, 7, 7, 128, 1, 1), (70, 64, 13, 15, 100, 1, 1), (44, 70, 19, 24, 64, 1, 1), (33, 64, 31, 30, 64, 1, 1), (11, 32, 40, 57, 120, 1, 0), (6, 64, 64, 64, 64, 1, 2),
          (290, 96, 14, 14, 64, 2, 1), (33, 128, 27, 27, 120, 2, 1), (21, 64, 41, 50, 128, 2, 0), (22, 64, 57, 64, 64, 2, 2), (300, 64, 9, 16, 128, 2, 1)]


def _filter(x, w_shape, dy, s, pt, beta=0.0, start=0.0):
    import torch
    from n2d2_amd import capi, runtime as rt
    B, Ci, H, W = x.shape
    d = capi.ConvDesc(Ci, w_shape[0], 3, 3, s, s, 1, pt, 1, pt, 1, 1, 1, 0, 0)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    x_, dy_, dw = dev(x), dev(dy), torch.full(w_shape, start, device="cuda")
    n = int(capi.lib.n2d2hip_conv2d_f32_workspace_bytes(C.byref(d), B, H, W))
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    capi.check(capi.lib.n2d2hip_conv2d_f32_backward_filter(C.byref(d), B, H, W, x_.data_ptr(), dy_.data_ptr(), beta, dw.data_ptr(), ws.data_ptr(), n, rt.stream_ptr()))
    torch.cuda.synchronize()
    return dw.cpu().numpy()


def _filter64(x, dy, s, pt):
    B, Ci, H, W = x.shape
    xp = np.zeros((B, Ci, dy.shape[2] * s + 2, dy.shape[3] * s + 2))
    h, w = min(H, xp.shape[2] - pt), min(W, xp.shape[3] - 1)
    xp[:, :, pt:pt + h, 1:1 + w] = x[:, :, :h, :w]
    dw = np.empty((dy.shape[1], Ci, 3, 3))
    d = dy.astype(np.float64).transpose(1, 0, 2, 3).reshape(dy.shape[1], -1)
    for i in range(3):
        for j in range(3):
            dw[:, :, i, j] = d @ xp[:, :, i:i + s * dy.shape[2]:s, j:j + s * dy.shape[3]:s].transpose(1, 0, 2, 3).reshape(Ci, -1).T
    return dw


@pytest.mark.parametrize("case", FILTER)
def test_filter_gradient_against_float64(case):
    from n2d2_amd import capi
    B, Ci, H, W, O, s, pt = case
    print("parts, filter gradient", case, flush=True)
    rng = np.random.default_rng(sum(case))
    oH, oW = (H + 2 * pt - 3) // s + 1, (W - 1) // s + 1
    assert 2.0 * B * O * oH * oW * Ci * 9 >= 1.5e9
    octets = -(-oW // 8)                         # a step has 8 of them, 4 at stride 2: the most of a row that leave the fewest beyond its end
    nol = min(range(4 - s, -1, -1), key=lambda n: -(-octets // 2 ** n) * 2 ** n)
    x, dy = rng.normal(size=(B, Ci, H, W)).astype(np.float32), rng.normal(size=(B, O, oH, oW)).astype(np.float32)
    want, mag = _filter64(x, dy, s, pt), _filter64(np.abs(x), np.abs(dy), s, pt)
    with capi.launch_log() as log:
        got = _filter(x, (O, Ci, 3, 3), dy, s, pt)
    assert [e[0] for e in log.entries] == ["conv_f32_filter_rows_kernel<%d, %d>" % (s, nol), "conv_f32_reduce_rows_kernel"]
    # (ranges, of which each is a sum in float, are added in double; one range is at most all pixels: 5 roundings in 32)
    K = B * oH * oW
    assert (np.abs(got - want) <= 2.0 ** -24 * (np.abs(want) + (5 * K / 32 + 4) * mag)).all()
    assert np.linalg.norm(got - want) <= 1.1 * 2.53e-8 * np.sqrt(1 + 5 * K / 64) * np.linalg.norm(want)
    again = _filter(x, (O, Ci, 3, 3), dy, s, pt, beta=0.5, start=2.0)
    assert np.abs(again - (got + np.float32(1.0))).max() <= 2.0 ** -23 * (np.abs(got).max() + 2)


def test_filter_gradient_infinities_nan_and_the_largest_floats():
    B, Ci, H, W, O, s, pt = 33, 128, 27, 27, 120, 2, 1
    print("parts, filter gradient, special values", flush=True)
    rng = np.random.default_rng(5)
    x, dy = rng.normal(size=(B, Ci, H, W)).astype(np.float32), (1e-3 * rng.normal(size=(B, O, 14, 14))).astype(np.float32)
    dy[np.abs(dy) < 1e-5] = 1e-5
    dy[2, 7] = 0.0
    for c, v in enumerate([np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 1e-42]):
        x[rng.integers(B), 3 * c + 1, rng.integers(H), rng.integers(W)] = v
    x[2, 50, 5, 6] = np.inf
    with np.errstate(invalid="ignore"):
        want = _filter64(x, dy, s, pt)
    got = _filter(x, (O, Ci, 3, 3), dy, s, pt)
    # (a padded position is no product here, in the reference a zero: only NaN of `want` against infinities outside the windows would differ)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got == np.inf, want == np.inf) and np.array_equal(got == -np.inf, want == -np.inf)
    ok = np.isfinite(want)
    fin = np.where(np.isfinite(x), x, 0)
    mag = _filter64(np.abs(fin), np.abs(dy), s, pt)
    assert (np.abs(got - _filter64(fin, dy, s, pt))[ok] <= 2.0 ** -24 * ((5 * B * 196 / 32 + 4) * mag)[ok]).all()


@pytest.mark.parametrize("small", [2.0 ** -112, 2.0 ** -118, 2.0 ** -126])
def test_small_floats_keep_their_bits(small):
    """One operand of a size whose parts would lie below the smallest bf16, against the other of size 1, and of 2^100: the bound of
    values of size 1, and half a step of the results where they are below the normal floats."""
    case = (33, 64, 32, 32, 64, 3, 3, 1, 1)
    print("parts, small floats", small, flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 3)
    small = np.float32(small)
    for of_x, of_w in ((small, 1), (1, small), (small, np.float32(2.0 ** 100)), (np.float32(2.0 ** 100), small)):
        a, b, d = x * of_x, w * of_w, dy * of_x
        for g, t, k in zip(_run(a, b, d, s, pad), _passes(a, b, d, s, pad), (64 * 9, 64 * 9)):
            assert np.linalg.norm(g - t) <= 1.1 * 2.53e-8 * np.sqrt(1 + k / 2) * np.linalg.norm(t) + 2.0 ** -150 * np.sqrt(t.size)
    K = dy.size // 64
    for of_x, of_dy in ((small, 1), (1, small), (small, np.float32(2.0 ** 100)), (np.float32(2.0 ** 100), small)):
        a, d = x * of_x, dy * of_dy
        got, want = _filter(a, w.shape, d, 1, 1), _filter64(a, d, 1, 1)
        assert np.linalg.norm(got - want) <= 1.1 * 2.53e-8 * np.sqrt(1 + 5 * K / 64) * np.linalg.norm(want) + 2.0 ** -150 * np.sqrt(want.size)


def _clipped(x, w, dy, s, pad):
    """Forward and data gradient in float64 whose windows end at the borders: of a tap outside there is no product, not one with 0."""
    (B, Ci, H, W), (O, _, kH, kW), (oH, oW) = x.shape, w.shape, dy.shape[2:]
    y, dx, w64 = np.zeros(dy.shape), np.zeros(x.shape), w.astype(np.float64)

    def axis(t, p, size, out):
        at = [o for o in range(out) if 0 <= o * s + t - p < size]
        return slice(at[0], at[-1] + 1), slice(at[0] * s + t - p, at[-1] * s + t - p + 1, s)
    for i in range(kH):
        for j in range(kW):
            (oy, iy), (ox, ix) = axis(i, pad[0], H, oH), axis(j, pad[1], W, oW)
            xs, ds = x[:, :, iy, ix].astype(np.float64), dy[:, :, oy, ox].astype(np.float64)
            y[:, :, oy, ox] += np.matmul(w64[:, :, i, j], xs.reshape(B, Ci, -1)).reshape(ds.shape)
            dx[:, :, iy, ix] += np.matmul(w64[:, :, i, j].T, ds.reshape(B, O, -1)).reshape(xs.shape)
    return y, dx


@pytest.mark.parametrize("weights", ["some", "every weight NaN"])
@pytest.mark.parametrize("case", [(9, 47, 31, 33, 97, 3, 3, 1, 1), (66, 100, 31, 33, 70, 3, 3, 2, 1)])
def test_weights_that_are_not_finite(case, weights):
    """What is NaN or infinite follows from the products inside the borders alone: beside them a weight meets no zero."""
    print("parts, weights not finite", case, weights, flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 4)
    x[1, 5], dy[1, 3, ::2] = 0.0, 0.0
    if weights == "some":
        w[3, 5, 1, 1], w[7, 2, 0, 2], w[9, 1, 2, 2], w[12, 3, 0, 0], w[12, 30, 2, 1], w[60, 46, 2, 2] = np.inf, np.nan, -np.inf, np.inf, -np.inf, np.nan
    else:
        w[:] = np.nan
    with np.errstate(invalid="ignore"):
        want = _clipped(x, w, dy, s, pad)
    fin = np.where(np.isfinite(w), w, np.float32(0))
    mag = _clipped(np.abs(x), np.abs(fin), np.abs(dy), s, pad)
    for g, t, m, k in zip(_run(x, w, dy, s, pad), want, mag, (w.shape[1] * 9, w.shape[0] * 9)):
        assert np.array_equal(np.isnan(g), np.isnan(t)) and np.array_equal(g == np.inf, t == np.inf) and np.array_equal(g == -np.inf, t == -np.inf)
        ok = np.isfinite(t)
        assert (np.abs(g[ok] - t[ok]) <= 2.0 ** -24 * (np.abs(t) + (k + 4) * m)[ok]).all()


def test_sums_beyond_the_scaled_range():
    """Operands of size 2^50 and 1e30, whose sums are past 2^96: added again, no further off than the sums of ordinary size."""
    case = (33, 64, 32, 32, 64, 3, 3, 1, 1)
    print("parts, large sums", flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 5)
    for of_x, of_w in ((np.float32(1e30), np.float32(1)), (np.float32(2.0 ** 50), np.float32(2.0 ** 50)), (np.float32(2.0 ** 115), np.float32(2.0 ** -20))):
        a, b, d = x * of_x, w * of_w, dy * of_x
        for g, t in zip(_run(a, b, d, s, pad), _passes(a, b, d, s, pad)):
            assert np.linalg.norm(g / 1e30 - t / 1e30) <= 1.1 * 2.53e-8 * np.sqrt(1 + 5 * 64 * 9 / 64) * np.linalg.norm(t / 1e30)
        d = dy * of_w
        got, want = _filter(a, w.shape, d, 1, 1) / 1e30, _filter64(a, d, 1, 1) / 1e30
        assert np.linalg.norm(got - want) <= 1.1 * 2.53e-8 * np.sqrt(1 + 5 * 33 * 1024 / 64) * np.linalg.norm(want)
