"""What a learning net's cells leave in one launch against the calls it stands for, through the C ABI: a layer with the SAT quantizer
behind it (n2d2hip_conv2d_f32_forward_sat: the same sums, so the same bits) and the softmax with its loss
(n2d2hip_softmax_loss_f32: the same bits, the loss of the same squares added in double in another order)."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

# (images, C, H, W, outputs, kernel): spanning layers of few sums, of up to a block a compute unit and of more; 3x3 spanning and not a
# multiple of four terms (direct kernels); the matrix cores; a layer that does not span its input
LAYERS = [(1, 4, 1, 1, 1, 1), (33, 120, 1, 1, 84, 1), (7, 16, 2, 2, 11, 2), (70, 100, 1, 1, 210, 1), (130, 64, 1, 1, 300, 1), (5, 7, 3, 3, 9, 3),
          (5, 3, 1, 1, 6, 1), (64, 512, 1, 1, 512, 1), (3, 6, 9, 8, 5, 3)]


@pytest.mark.parametrize("layer", LAYERS)
@pytest.mark.parametrize("learning", [True, False])
def test_layer_with_quantizer(layer, learning):
    import torch
    from n2d2_amd import capi, runtime
    lib, sp = capi.lib, runtime.stream_ptr
    B, Cn, H, W, O, k = layer
    g = torch.Generator(device="cuda").manual_seed(B * O)
    oH, oW = H - k + 1, W - k + 1
    d = capi.ConvDesc(Cn, O, k, k, 1, 1, 0, 0, 0, 0, 1, 1, 1, 0)
    x, w = torch.randn(B, Cn, H, W, device="cuda", generator=g), torch.randn(O, Cn, k, k, device="cuda", generator=g)
    bias, alpha = torch.randn(O, device="cuda", generator=g), torch.full((1,), -2.5, device="cuda")
    ws = torch.empty(max(int(lib.n2d2hip_conv2d_f32_workspace_bytes(C.byref(d), B, H, W)), 4), dtype=torch.uint8, device="cuda")
    for b in (None, bias.data_ptr()):
        want, fp = torch.empty(B, O, oH, oW, device="cuda"), torch.full((B, O, oH, oW), -9.0, device="cuda")
        capi.check(lib.n2d2hip_conv2d_f32_forward(C.byref(d), B, H, W, x.data_ptr(), w.data_ptr(), b, 0.0, want.data_ptr(), ws.data_ptr(), ws.numel(), sp()))
        capi.check(lib.n2d2hip_sat_act_forward(want.data_ptr(), fp.data_ptr() if learning else None, want.numel(), 15.0, alpha.data_ptr(), sp()))
        got, gfp = torch.full_like(want, -9.0), torch.full_like(want, -9.0)
        capi.check(lib.n2d2hip_conv2d_f32_forward_sat(C.byref(d), B, H, W, x.data_ptr(), w.data_ptr(), b, got.data_ptr(), gfp.data_ptr() if learning else None,
                                                      15.0, alpha.data_ptr(), ws.data_ptr(), ws.numel(), sp()))
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(gfp, fp)
    assert lib.n2d2hip_conv2d_f32_forward_sat(C.byref(d), B, H, W, x.data_ptr(), w.data_ptr(), None, got.data_ptr(), got.data_ptr(), 15.0,
                                              alpha.data_ptr(), ws.data_ptr(), ws.numel(), sp()) == capi.ERR_INVALID


@pytest.mark.parametrize("B,Cn,H,W", [(1, 1, 1, 1), (32, 10, 1, 1), (256, 16, 1, 1), (257, 16, 1, 1), (3, 17, 1, 1), (2, 5, 13, 7), (64, 1000, 1, 1)])
@pytest.mark.parametrize("below", [True, False])
def test_softmax_with_loss(B, Cn, H, W, below):
    import torch
    from n2d2_amd import capi, runtime
    lib, sp = capi.lib, runtime.stream_ptr
    g = torch.Generator(device="cuda").manual_seed(B + Cn)
    x, t = (torch.randn(B, Cn, H, W, device="cuda", generator=g) for _ in range(2))
    x[0, 0] = float("nan") if B > 200 else 80.0
    ws = torch.empty(int(lib.n2d2hip_loss_workspace_bytes(x.numel())), dtype=torch.uint8, device="cuda")
    y, diff = torch.empty_like(x), torch.empty_like(x)
    loss, got_loss = (torch.zeros(1, dtype=torch.float64, device="cuda") for _ in range(2))
    capi.check(lib.n2d2hip_softmax_f32_forward(x.data_ptr(), y.data_ptr(), B, Cn, H, W, sp()))
    capi.check(lib.n2d2hip_loss_f32(t.data_ptr(), y.data_ptr(), diff.data_ptr(), x.numel(), B, loss.data_ptr(), ws.data_ptr(), ws.numel(), sp()))
    gy, gd, gx = (torch.full_like(x, -9.0) for _ in range(3))
    capi.check(lib.n2d2hip_softmax_loss_f32(x.data_ptr(), t.data_ptr(), gy.data_ptr(), gd.data_ptr(), gx.data_ptr() if below else None, B, Cn, H, W,
                                            got_loss.data_ptr(), ws.data_ptr(), ws.numel(), sp()))
    torch.cuda.synchronize()
    same = lambda a, b: torch.equal(a.view(torch.int32), b.view(torch.int32)) or torch.equal(torch.nan_to_num(a, 7.0), torch.nan_to_num(b, 7.0))  # noqa: E731
    assert same(gy, y) and same(gd, diff) and (same(gx, diff) if below else bool((gx == -9.0).all()))
    # (n squares, each half an ulp of a double, in two orders)
    assert torch.isclose(got_loss, loss, rtol=x.numel() * 2.0 ** -52 + 2.0 ** -51, atol=0.0, equal_nan=True).all()
