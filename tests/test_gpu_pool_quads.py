"""Max pooling's gradient for rows of whole quads against the kernel that takes an input at a time, which a result off 16-byte
boundaries goes to: equal bits, windows that overlap, leave gaps, are larger than a quad or padded."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 3, 7, 4), (3, 2, 6, 8), (1, 1, 1, 4), (2, 5, 9, 12), (40, 16, 28, 28)], ids=str)
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_quads_equal_single_inputs(shape, beta):
    import torch
    from n2d2_amd import capi, runtime as rt
    B, Cn, H, W = shape
    lib, rng = capi.lib, np.random.default_rng(sum(shape))
    for pw, ph, sx, sy, px, py in itertools.product((1, 2, 3, 7), (1, 3), (1, 2, 3, 5), (1, 2), (0, 1, 2), (0, 1)):
        if px >= pw or py >= ph or pw > W + 2 * px or ph > H + 2 * py:
            continue
        oH, oW = (H + 2 * py - ph) // sy + 1, (W + 2 * px - pw) // sx + 1
        x = torch.from_numpy(rng.integers(-3, 4, size=shape).astype(np.float32)).cuda()
        dy = torch.from_numpy(rng.normal(size=(B, Cn, oH, oW)).astype(np.float32)).cuda()
        y, argmax = torch.empty_like(dy), torch.empty(dy.shape, dtype=torch.int32, device="cuda")
        rc = lib.n2d2hip_pool_max_f32_forward(B, Cn, H, W, pw, ph, sx, sy, px, py, x.data_ptr(), y.data_ptr(), argmax.data_ptr(), rt.stream_ptr())
        capi.check(rc)
        start = torch.from_numpy(rng.normal(size=shape).astype(np.float32)).cuda()
        out = []
        for off in (0, 1):
            dx = torch.empty(x.numel() + 4, device="cuda")[off:off + x.numel()]
            dx.copy_(start.view(-1))
            capi.check(lib.n2d2hip_pool_max_f32_backward(B, Cn, H, W, pw, ph, sx, sy, px, py, dy.data_ptr(), argmax.data_ptr(), beta, dx.data_ptr(), rt.stream_ptr()))
            out.append(dx.clone())
        assert torch.equal(*out), (shape, pw, ph, sx, sy, px, py)
