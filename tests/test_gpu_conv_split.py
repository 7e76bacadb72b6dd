"""The convolution kernel whose waves share K (layers of few output tiles): bit for bit the oracle's integers, and those of the
other kernels where a residual sum is folded in."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# B, C, H, W, O, kernel, stride, pad, halo of the input, weight bits: one K step, fewer steps than waves, steps that do not divide
# by the waves, ragged pixels and channels, every window form
CASES = [
    (1, 128, 1, 1, 16, 1, 1, 0, 0, 8),
    (3, 128, 5, 5, 48, 1, 1, 0, 0, 8),
    (2, 640, 7, 5, 40, 1, 2, 0, 0, 8),
    (5, 128, 7, 7, 130, 3, 1, 1, 0, 8),
    (2, 256, 9, 6, 96, 3, 2, 1, 0, 8),
    (2, 384, 6, 5, 64, 3, 1, 1, 1, 8),
    (1, 128, 11, 9, 33, 5, 1, 0, 0, 8),
    (33, 128, 4, 4, 32, 3, 1, 0, 0, 8),
    (2, 128, 8, 8, 64, 3, 1, 1, 1, 4),
    (3, 256, 7, 7, 128, 1, 1, 0, 0, 4),
    (2, 128, 5, 6, 40, 1, 1, 1, 0, 8),
    (2, 256, 9, 7, 72, 3, 2, 1, 0, 4),
]


def _conv(rt, capi, case, act, choice, rng_seed=3):
    B, C, H, W, O, k, s, p, halo, bits = case
    rng = np.random.default_rng(rng_seed)
    x = rng.integers(0, 256 if bits == 8 else 16, size=(B, C, H, W))
    w = rng.integers(-127, 128, size=(O, C, k, k)) if bits == 8 else rng.integers(-8, 8, size=(O, C, k, k))
    bias = rng.integers(-4096, 4097, size=O).astype(np.int32)
    conv = rt.Conv(w.astype(np.int32), bias, act, capi.U8B, stride=(s, s), pad=(p, p, p, p), weight_bits=bits, kernel_choice=choice)
    xd = rt.DTensor.from_numpy(x, capi.U8B)
    return x, w, bias, conv, xd.with_halo(halo) if halo else xd


# (4-bit weights without a rescale are another kernel's, whatever the choice)
@pytest.mark.parametrize("kind,case", [pytest.param(k, c, id="-".join(map(str, (k,) + c))) for k in ("shift", "clip", "raw") for c in CASES
                                       if k != "raw" or c[-1] == 8])
def test_waves_share_k_bit_exact(kind, case):
    from n2d2_amd import capi, runtime as rt
    from oracle import cells
    from oracle.cells import ActSpec
    B, C, H, W, O, k, s, p, halo, bits = case
    served = kind != "raw" or (k == 1 and p == 0 and bits == 8)        # (sums without a rescale: unpadded 1x1; the others go their way)
    rng = np.random.default_rng(C + O)
    spec = {"shift": ActSpec("Rectifier", "SingleShift", rng.integers(9, 14, size=O), nb_bits=8, unsigned_out=True),
            "clip": ActSpec("Linear", "FixedMult16", rng.integers(2 ** 8, 2 ** 10, size=O), frac_bits=20,
                            clipping=rng.uniform(2000.0, 90000.0, size=O).astype(np.float32), nb_bits=8, unsigned_out=False),
            "raw": ActSpec("Rectifier", "None")}[kind]
    print(case, kind, flush=True)
    x, w, bias, conv, xd = _conv(rt, capi, case, rt.Act(O, **spec.kwargs()), capi.KERNEL_SPLIT)
    with capi.launch_log() as log:
        got = conv.forward(xd)
    assert [e[0].startswith("conv_split_kernel") for e in log.entries] == [served]
    want = cells.conv_cell(x.astype(np.int32), w.astype(np.int32), bias, spec, stride=(s, s), pad=(p, p, p, p))
    assert np.array_equal(got.to_numpy(), want.astype(np.int64))


@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("case", [(2, 256, 7, 7, 128, 1, 1, 0, 0, 8), (5, 128, 5, 9, 192, 1, 1, 0, 0, 8), (2, 128, 8, 8, 128, 3, 1, 1, 1, 4)])
def test_folded_residual_sum(case, scaled):
    from n2d2_amd import capi, runtime as rt
    B, C, H, W, O, k, s, p, halo, bits = case
    rng = np.random.default_rng(9)
    other = rt.DTensor.from_numpy(rng.integers(0, 256, size=(B, O, H, W)), capi.U8B)
    outs = []
    for choice in (capi.KERNEL_SPLIT, capi.KERNEL_NO_SPLIT, capi.KERNEL_NO_SPLIT | capi.KERNEL_NO_SUM16):
        act = rt.Act(O, kind="Linear", mode="SingleShift", scaling=np.full(O, 11, np.uint8), nb_bits=8, unsigned_out=False)
        ew = rt.ElemWiseSum(2, O, rt.Act(O, kind="Rectifier", mode="SingleShift", scaling=np.full(O, 1, np.uint8), nb_bits=8, unsigned_out=True))
        if scaled:
            pre = rt.Act(O, kind="Linear", mode="FixedMult16", scaling=np.random.default_rng(4).integers(20, 60, size=O).astype(np.int32), frac_bits=6,
                         nb_bits=8, unsigned_out=False)
            assert ew.fold_input_scaling(1, pre)
        x, w, bias, conv, xd = _conv(rt, capi, case, act, choice)
        assert conv.fuse_sum(ew, 0, capi.U8B)
        out = rt.DTensor(B, O, H, W, capi.U8B, halo=1)
        conv.forward_sum(xd, other, out)
        outs.append(out.buf.cpu().numpy())
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
    assert len(np.unique(outs[0])) > 20
