"""Both gradients of a convolution in one call: the bits of backward-filter followed by backward-data, in one launch where both
sums are small, and also where a result lies over an operand, which takes the two passes."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PAIR, BOTH = "conv_f32_small_pair_kernel", "conv_f32_small_both_kernel"
# (B, C, O, k, H, W, stride, pad, groups, the kernel of both)
CASES = [(32, 84, 10, 1, 1, 1, 1, 0, 1, PAIR), (32, 120, 84, 1, 1, 1, 1, 0, 1, PAIR), (32, 16, 120, 5, 5, 5, 1, 0, 1, PAIR), (1, 1, 1, 1, 1, 1, 1, 0, 1, PAIR),
         (17, 15, 17, 1, 1, 1, 1, 0, 1, PAIR), (16, 16, 16, 1, 1, 1, 1, 0, 1, PAIR), (255, 33, 65, 1, 1, 1, 1, 0, 1, PAIR), (3, 2, 130, 2, 2, 2, 1, 0, 1, PAIR),
         (600, 8, 8, 1, 1, 1, 1, 0, 1, None), (4, 2, 3000, 1, 1, 1, 1, 0, 1, None),           # (sums in ranges)
         (8, 6, 16, 5, 14, 14, 1, 0, 1, BOTH), (4, 16, 16, 3, 12, 10, 2, 1, 1, BOTH), (1, 17, 28, 3, 9, 9, 1, 1, 1, BOTH), (2, 16, 29, 3, 9, 9, 1, 0, 1, BOTH),
         (1, 1, 1, 2, 3, 3, 1, 0, 1, BOTH), (32, 3, 8, 3, 15, 17, 1, 1, 1, BOTH), (32, 6, 16, 5, 14, 14, 1, 0, 1, BOTH),
         (31, 20, 8, 1, 40, 47, 1, 0, 1, BOTH), (9, 5, 3, 3, 71, 64, 1, 1, 1, BOTH), (1, 9, 130, 3, 9, 9, 1, 1, 1, BOTH),      # (a tile to a wave; sixteen waves to a tile)
         (4, 16, 16, 3, 12, 10, 1, 1, 16, None),
         (64, 64, 64, 3, 24, 24, 1, 1, 1, None), (64, 512, 1000, 1, 1, 1, 1, 0, 1, None), (2, 4, 10, 16, 16, 16, 1, 0, 1, None)]


def _larger(case):
    """diff_x than diff_y: it does not fit over it"""
    _, Ci, O, k, H, W, s, p, _, _ = case
    return Ci * H * W > O * ((H + 2 * p - k) // s + 1) * ((W + 2 * p - k) // s + 1)


@pytest.mark.parametrize("over,case", [(o, c) for o in (None, "x", "dy") for c in CASES if o != "dy" or not _larger(c)], ids=str)
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_equals_the_two_passes(case, beta, over):
    import torch
    from n2d2_amd import capi, runtime as rt
    B, Ci, O, k, H, W, s, p, groups, kernel = case
    print("both gradients", case, beta, over, flush=True)
    lib, rng = capi.lib, np.random.default_rng(sum(case[:8]))
    oH, oW = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    d = capi.ConvDesc(Ci, O, k, k, s, s, p, p, p, p, 1, 1, groups, 0, 0)
    dev = lambda *n: torch.from_numpy(rng.normal(size=n).astype(np.float32)).cuda()
    x, w, dy, dw0, dx0 = dev(B, Ci, H, W), dev(O, Ci // groups, k, k), dev(B, O, oH, oW), dev(O, Ci // groups, k, k), dev(B, Ci, H, W)
    nws = int(lib.n2d2hip_conv2d_f32_workspace_bytes(C.byref(d), B, H, W))
    ws = torch.empty(max(nws, 16), dtype=torch.uint8, device="cuda")
    out = []
    for both in (False, True):
        X, Y, dw, dx = x.clone(), dy.clone(), dw0.clone(), dx0.clone()
        if over:                                # diff_x over an operand that the pass before it has read
            dx = X if over == "x" else Y
        with capi.launch_log() as log:
            if both:
                capi.check(lib.n2d2hip_conv2d_f32_backward(C.byref(d), B, H, W, X.data_ptr(), w.data_ptr(), Y.data_ptr(), beta, dw.data_ptr(), beta,
                                                           dx.data_ptr(), ws.data_ptr(), nws, rt.stream_ptr()))
            else:
                capi.check(lib.n2d2hip_conv2d_f32_backward_filter(C.byref(d), B, H, W, X.data_ptr(), Y.data_ptr(), beta, dw.data_ptr(), ws.data_ptr(), nws,
                                                                  rt.stream_ptr()))
                if over != "dy":                 # (backward-data reads what it would write: only the weights' gradient is compared)
                    capi.check(lib.n2d2hip_conv2d_f32_backward_data(C.byref(d), B, H, W, w.data_ptr(), Y.data_ptr(), beta, dx.data_ptr(), ws.data_ptr(), nws,
                                                                    rt.stream_ptr()))
        out.append((dw, None if over == "dy" else dx))
    torch.cuda.synchronize()
    assert [e[0].split("<")[0] for e in log.entries if e[0].startswith((PAIR, BOTH))] == ([kernel] if kernel and not over else [])
    for a, b in zip(*out):
        assert a is None or (torch.equal(a, b) and bool(torch.isfinite(a).all()))


def test_refuses_what_the_passes_refuse():
    import torch
    from n2d2_amd import capi
    t = torch.zeros(4096, device="cuda")
    call = lambda d, *a: capi.lib.n2d2hip_conv2d_f32_backward(C.byref(d), 2, 1, 1, *a)
    q = [t[1024 * i:].data_ptr() for i in range(4)] + [t.data_ptr()]
    fc, dilated = capi.ConvDesc(8, 4, 1, 1, 1, 1, 0, 0, 0, 0, 1, 1, 1, 0, 0), capi.ConvDesc(8, 4, 1, 1, 1, 1, 0, 0, 0, 0, 2, 2, 1, 0, 0)
    good = lambda n: [None if i == n else q[i] for i in range(5)]
    for n in range(5):
        x, w, dy, dw, dx = good(n)
        assert call(fc, x, w, dy, 0.0, dw, 0.0, dx, None, 0, None) == capi.ERR_INVALID
    x, w, dy, dw, dx = q
    assert call(dilated, x, w, dy, 0.0, dw, 0.0, dx, None, 0, None) != 0
