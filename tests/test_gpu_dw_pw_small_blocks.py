"""The one-launch depthwise + 1x1 kernel with 32, 64 and 128 outputs a work-group: byte for byte the two separate launches, at the sizes where one
takes over from the other, with every rescale, several chunks of channels a wave, outputs that whole work-groups of 64 or 128 do not hold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# B, C, O, stride, H, W, blocks of 16 outputs (256 compute units: 512 channels from 257 work-groups on, 256 from 769, 192 from 1025)
CASES = [
    (1, 512, 512, 1, 14, 14, 2),       # 13 groups of pixels x 16
    (1, 512, 512, 1, 16, 16, 2),       # 256 work-groups
    (1, 512, 512, 1, 16, 17, 4),       # 272
    (2, 512, 512, 1, 16, 16, 4),       # 256 of 64 outputs
    (2, 512, 512, 1, 16, 17, 8),
    (4, 512, 512, 2, 31, 31, 8),
    (5, 512, 160, 1, 40, 13, 2),       # 815 work-groups, no whole ones of 64 outputs
    (3, 512, 192, 1, 21, 17, 4),       # 402, no whole ones of 128
    (1, 1024, 256, 1, 24, 23, 4),      # two chunks a wave
    (2, 1024, 256, 1, 24, 23, 8),
    (5, 512, 128, 1, 40, 13, 2),       # few outputs
    (9, 256, 192, 1, 25, 15, 4),
    (17, 192, 256, 1, 16, 16, 8),      # three waves
]


@pytest.mark.parametrize("B,C,O,stride,H,W,blocks", CASES)
@pytest.mark.parametrize("rescale", ["plain", "clamped", "wide"])
def test_equals_separate_launches(B, C, O, stride, H, W, blocks, rescale):
    import torch
    from n2d2_amd import capi, runtime as rt
    from oracle.cells import ActSpec
    print("dw_pw_small blocks", B, C, O, stride, H, W, blocks, rescale, flush=True)
    rng = np.random.default_rng(C + O + H)
    x = rng.integers(0, 256, size=(B, C, H, W))
    wd, bd = rng.integers(-128, 128, size=(C, 1, 3, 3)), rng.integers(-2000, 2001, size=C)
    wp, bp = rng.integers(-128, 128, size=(O, C, 1, 1)), rng.integers(-20000, 20001, size=O)
    unsigned = dict(nb_bits=8, unsigned_out=True)
    if rescale == "plain":
        sd = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 11, 2 ** 12, size=C), frac_bits=18, **unsigned)
        sp = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 7, 2 ** 8, size=O), frac_bits=16, **unsigned)
    elif rescale == "clamped":
        sd = ActSpec("Linear", "FixedMult32", rng.integers(2 ** 13, 2 ** 14, size=C), frac_bits=21, nb_bits=8, unsigned_out=False)
        sp = ActSpec("Linear", "FixedMult32", rng.integers(2 ** 13, 2 ** 14, size=O), frac_bits=21, nb_bits=8, unsigned_out=False)
    else:
        sd = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 25, 2 ** 26, size=C), frac_bits=33, **unsigned)
        sp = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 25, 2 ** 26, size=O), frac_bits=35, **unsigned)
    dw = rt.Conv(wd, bd, rt.Act(C, **sd.kwargs()), capi.U8B, stride=(stride, stride), pad=(1,) * 4, groups=C)
    pw = rt.Conv(wp, bp, rt.Act(O, **sp.kwargs()), capi.I8 if rescale == "clamped" else capi.U8B)
    xin = rt.DTensor.from_numpy(x, capi.U8B)
    want = pw.forward(dw.forward(xin))
    fused = rt.DwPwSmall.create(dw, pw)
    out = rt.DTensor(B, O, want.H, want.W, want.dtype)
    with capi.launch_log() as log:
        got = fused.forward(xin, out)
    assert np.array_equal(got.to_numpy(), want.to_numpy())
    small = [e[0] for e in log.entries if e[0].startswith("dw_pw_small_kernel")]
    if torch.cuda.get_device_properties(0).multi_processor_count == 256 and small:       # (few outputs: the kernel for many pixels takes some)
        assert small[0].endswith(" %d>" % blocks)
