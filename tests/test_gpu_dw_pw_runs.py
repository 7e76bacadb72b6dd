"""The one-launch depthwise + 1x1 kernel where a work-group runs over several tiles: against the two separate launches, byte for
byte.  (Single tiles, every channel count and the oracle are in test_gpu_int.py.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [
    (9, 32, 64, 1, 119, 161, 1),       # one chunk, 11 x 15 x 9 tiles: 186 an XCD for 160 work-groups, so runs of 1 and 2
    (13, 64, 128, 2, 113, 111, 1),     # stride 2, one chunk; 12 rows short of a tile
    (21, 128, 128, 1, 40, 43, 1),      # two chunks, more tiles than work-groups
    (9, 192, 64, 2, 95, 130, 0),       # three chunks (an odd number of steps a tile), no padding
    (11, 128, 256, 1, 49, 33, 1),      # 256 outputs, 16 waves
    (3, 128, 512, 1, 56, 57, 1),       # two work-groups of outputs
], ids=lambda c: "x".join(str(v) for v in c))
@pytest.mark.parametrize("small", [False, True], ids=["clamped", "plain"])
def test_runs_of_tiles_equal_separate_launches(case, small):
    from n2d2_amd import capi, runtime as rt
    from oracle.cells import ActSpec
    B, C, O, stride, H, W, pad = case
    print("dw_pw runs", case, small, flush=True)
    rng = np.random.default_rng(hash(case) % 1000 + small)
    x = rng.integers(0, 256, size=(B, C, H, W))
    wd, bd = rng.integers(-128, 128, size=(C, 1, 3, 3)), rng.integers(-2000, 2001, size=C)
    wp, bp = rng.integers(-128, 128, size=(O, C, 1, 1)), rng.integers(-20000, 20001, size=O)
    # multipliers that need no clamp before the multiply, or that do
    if small:
        sd = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 11, 2 ** 12, size=C), frac_bits=18, nb_bits=8, unsigned_out=True)
        sp = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 7, 2 ** 8, size=O), frac_bits=16, nb_bits=8, unsigned_out=True)
    else:
        sd = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 13, 2 ** 14, size=C), frac_bits=20, nb_bits=8, unsigned_out=True)
        sp = ActSpec("Linear", "FixedMult32", rng.integers(2 ** 13, 2 ** 14, size=O), frac_bits=21, nb_bits=8, unsigned_out=False)
    dw = rt.Conv(wd, bd, rt.Act(C, **sd.kwargs()), capi.U8B, stride=(stride, stride), pad=(pad,) * 4, groups=C)
    pw = rt.Conv(wp, bp, rt.Act(O, **sp.kwargs()), capi.U8B)
    xin = rt.DTensor.from_numpy(x, capi.U8B)
    want = pw.forward(dw.forward(xin))
    fused = rt.DwPw.create(dw, pw)
    assert fused is not None
    out = rt.DTensor(B, O, want.H, want.W, want.dtype)
    for _ in range(2):                 # (the second finds its buffers full of the first's bytes)
        assert np.array_equal(fused.forward(xin, out).to_numpy(), want.to_numpy())
