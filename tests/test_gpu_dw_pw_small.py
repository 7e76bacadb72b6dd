"""The one-launch depthwise + 1x1 kernel for few pixels against the two separate launches, byte for byte: remainders of its 16 pixels,
one and several chunks of 64 channels a wave, both strides, every rescale it takes, and the sizes where it hands over."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,C,O,stride,H,W,pad", [
    (1, 64, 32, 1, 1, 1, 1),           # one pixel
    (1, 32, 96, 1, 7, 5, 1),           # half a chunk; 96 outputs (the other kernel does not take them)
    (3, 64, 64, 2, 9, 11, 0),          # pixels of three images in one work-group, no padding
    (2, 192, 160, 1, 6, 9, 1),         # three waves
    (1, 512, 64, 2, 14, 14, 1),        # eight waves
    (1, 640, 32, 1, 5, 4, 1),          # ten chunks: two waves have two
    (2, 1024, 1024, 1, 7, 7, 1),
    (2, 64, 128, 1, 33, 31, 1),        # 256 + groups: all on the chip
    (2, 64, 128, 1, 48, 47, 1),        # 1128 work-groups: the kernel for many pixels
    (1, 32, 64, 1, 20, 9, 1),          # 32 channels: the kernel for many pixels
    (6, 64, 512, 1, 40, 39, 1),        # 512 outputs, 9360 pixels
])
@pytest.mark.parametrize("rescale", ["plain", "clamped", "wide"])
def test_small_equals_separate_launches(B, C, O, stride, H, W, pad, rescale):
    from n2d2_amd import capi, runtime as rt
    from oracle.cells import ActSpec
    print("dw_pw_small", B, C, O, stride, H, W, pad, rescale, flush=True)
    rng = np.random.default_rng(C + O + H)
    x = rng.integers(0, 256, size=(B, C, H, W))
    wd, bd = rng.integers(-128, 128, size=(C, 1, 3, 3)), rng.integers(-2000, 2001, size=C)
    wp, bp = rng.integers(-128, 128, size=(O, C, 1, 1)), rng.integers(-20000, 20001, size=O)
    unsigned = dict(nb_bits=8, unsigned_out=True)
    if rescale == "plain":
        sd = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 11, 2 ** 12, size=C), frac_bits=18, **unsigned)
        sp = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 7, 2 ** 8, size=O), frac_bits=16, **unsigned)
    elif rescale == "clamped":         # a signed tensor between the cells
        sd = ActSpec("Linear", "FixedMult32", rng.integers(2 ** 13, 2 ** 14, size=C), frac_bits=21, nb_bits=8, unsigned_out=False)
        sp = ActSpec("Linear", "FixedMult32", rng.integers(2 ** 13, 2 ** 14, size=O), frac_bits=21, nb_bits=8, unsigned_out=False)
    else:                              # multipliers past 24 bits: 64-bit rescales
        sd = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 25, 2 ** 26, size=C), frac_bits=33, **unsigned)
        sp = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 25, 2 ** 26, size=O), frac_bits=35, **unsigned)
    dw = rt.Conv(wd, bd, rt.Act(C, **sd.kwargs()), capi.U8B, stride=(stride, stride), pad=(pad,) * 4, groups=C)
    pw = rt.Conv(wp, bp, rt.Act(O, **sp.kwargs()), capi.I8 if rescale == "clamped" else capi.U8B)
    xin = rt.DTensor.from_numpy(x, capi.U8B)
    want = pw.forward(dw.forward(xin))
    fused = rt.DwPwSmall.create(dw, pw)
    assert fused is not None
    out = rt.DTensor(B, O, want.H, want.W, want.dtype)
    launched = []
    for _ in range(2):                 # (the question whether it pays, between the two, changes nothing)
        with capi.launch_log() as log:
            assert np.array_equal(fused.forward(xin, out).to_numpy(), want.to_numpy())
        launched.append([e[0] for e in log.entries if e[0].startswith("dw_pw")])
        fused.pays(B, H, W)
    assert launched[0] == launched[1] and len(launched[0]) == 1


def test_small_takes_more_pixels_than_a_grid():
    """65535 work-groups of 16 pixels are one launch; 34 pixels more."""
    from n2d2_amd import capi, runtime as rt
    from oracle.cells import ActSpec
    rng = np.random.default_rng(7)
    H, W = 1023, 1025
    x = rng.integers(0, 256, size=(1, 32, H, W)).astype(np.int32)
    spec = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 11, 2 ** 12, size=32), frac_bits=18, nb_bits=8, unsigned_out=True)
    dw = rt.Conv(rng.integers(-128, 128, size=(32, 1, 3, 3)), None, rt.Act(32, **spec.kwargs()), capi.U8B, pad=(1,) * 4, groups=32)
    pw = rt.Conv(rng.integers(-128, 128, size=(32, 32, 1, 1)), None, rt.Act(32, **spec.kwargs()), capi.U8B)
    xin = rt.DTensor.from_numpy(x, capi.U8B)
    want = pw.forward(dw.forward(xin))
    out = rt.DTensor(1, 32, H, W, want.dtype)
    with capi.launch_log() as log:
        rt.DwPwSmall.create(dw, pw).forward(xin, out)
    assert [e[1] for e in log.entries] == [65535, 1]
    import torch
    assert torch.equal(out.buf, want.buf)


def test_small_declines_what_it_is_not_written_for():
    from n2d2_amd import capi, runtime as rt
    from oracle.cells import ActSpec
    rng = np.random.default_rng(5)
    act = lambda n: rt.Act(n, **ActSpec("Rectifier", "SingleShift", rng.integers(8, 12, size=n), nb_bits=8, unsigned_out=True).kwargs())
    conv = lambda O, C, k, g=1, **kw: rt.Conv(rng.integers(-9, 10, size=(O, C // g, k, k)), None, act(O), capi.U8B, groups=g, **kw)
    dw = conv(64, 64, 3, 64, pad=(1,) * 4)
    assert rt.DwPwSmall.create(dw, conv(32, 64, 1)) is not None
    assert rt.DwPwSmall.create(dw, conv(40, 64, 1)) is None                                  # outputs not in 32s
    assert rt.DwPwSmall.create(conv(48, 48, 3, 48, pad=(1,) * 4), conv(32, 48, 1)) is None   # channels not in 64s
    assert rt.DwPwSmall.create(conv(64, 64, 3, 64, pad=(2,) * 4, dil=(2, 2)), conv(32, 64, 1)) is None
    assert rt.DwPwSmall.create(dw, conv(32, 64, 3, pad=(1,) * 4)) is None
    # one pixel pays, a batch that does not fit the chip does not
    h = rt.DwPwSmall.create(conv(512, 512, 3, 512, pad=(1,) * 4), conv(512, 512, 1))
    assert h.pays(1, 14, 14) and not h.pays(8, 14, 14)


@pytest.mark.parametrize("batch,image", [(1, 224), (2, 96), (8, 160)])
def test_network_lays_out_only_the_pairs_it_launches(batch, image, monkeypatch):
    """The library says from the cells and sizes alone how a pair runs, so that no kernel's weights are laid out and thrown away."""
    from n2d2_amd import nets, runtime as rt
    made = []
    create = rt.DwPw.create.__func__           # (DwPwSmall inherits it)
    monkeypatch.setattr(rt.DwPw, "create", classmethod(lambda cls, dw, pw: made.append(cls) or create(cls, dw, pw)))
    net = nets.GpuNet(nets.mobilenet_v1(image=image), batch)
    fused = [cell for l, cell, fn in net.steps if isinstance(cell, rt.DwPw)]
    assert len(fused) == len(net.dw_pws) + len(net.dw_pws_small) >= 3
    assert made == [type(cell) for cell in fused]


@pytest.mark.parametrize("C,O,stride,sizes", [
    (32, 64, 1, {(1, 1): "tiles", (4, 28): "tiles"}),                                               # one chunk of channels: always ahead
    (64, 128, 1, {(1, 7): "small", (1, 50): "small", (1, 70): "tiles", (1, 200): "tiles"}),
    (128, 128, 2, {(1, 14): "small", (2, 56): "tiles", (16, 56): "tiles"}),
    (512, 128, 1, {(1, 14): "small", (1, 56): "apart", (2, 64): "apart", (1, 100): "tiles"}),        # many chunks: the launch is as long as they are
    (1024, 64, 1, {(1, 14): "small", (1, 100): "apart", (1, 128): "apart", (1, 140): "tiles"}),
    (256, 256, 1, {(1, 14): "small", (8, 28): "apart", (12, 28): "tiles", (33, 28): "tiles", (65, 28): "tiles"}),
    (512, 256, 1, {(1, 14): "small", (8, 28): "apart", (12, 28): "tiles", (32, 28): "tiles", (33, 28): "apart", (48, 28): "tiles"}),
    (512, 512, 1, {(1, 14): "small", (32, 14): "apart", (48, 14): "tiles", (64, 14): "tiles", (65, 14): "apart", (96, 14): "apart", (128, 14): "tiles", (112, 14): "tiles",
                   (192, 14): "apart", (96, 10): "apart"}),
    (1024, 512, 1, {(1, 7): "small", (64, 14): "apart"}),
    (512, 1024, 1, {(1, 7): "small", (64, 14): "apart"}),
])
def test_plan_follows_the_measured_lines(C, O, stride, sizes):
    """What the library plans on a chip of 256 compute units, (images, output rows and columns) by (images, rows and columns); the
    handles' own questions agree with it."""
    import torch
    from n2d2_amd import capi, runtime as rt
    from oracle.cells import ActSpec
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines were measured with 256 compute units")
    rng = np.random.default_rng(3)
    spec = lambda n: ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 7, 2 ** 8, size=n), frac_bits=16, nb_bits=8, unsigned_out=True)
    dw = rt.Conv(rng.integers(-128, 128, size=(C, 1, 3, 3)), None, rt.Act(C, **spec(C).kwargs()), capi.U8B, stride=(stride,) * 2, pad=(1,) * 4, groups=C)
    pw = rt.Conv(rng.integers(-128, 128, size=(O, C, 1, 1)), None, rt.Act(O, **spec(O).kwargs()), capi.U8B)
    tiles, small = rt.DwPw.create(dw, pw), rt.DwPwSmall.create(dw, pw)
    for (B, H), want in sizes.items():
        kind = rt.dw_pw_kind(dw, pw, B, H * stride, H * stride)
        assert {None: "apart", rt.DwPw: "tiles", rt.DwPwSmall: "small"}[kind] == want, (B, H)
        pays = tiles.pays(B, H * stride, H * stride), small.pays(B, H * stride, H * stride)
        assert any(pays) == (want != "apart") and (want != "tiles" or pays[0]) and (want != "small" or pays[1]), (B, H, pays)
    assert capi.lib.n2d2hip_dw_pw_plan(None, pw.handle, 1, 8, 8) == capi.lib.n2d2hip_dw_pw_plan(dw.handle, pw.handle, 0, 8, 8) == capi.DW_PW_APART
