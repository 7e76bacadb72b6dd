"""The 3x3 depthwise kernel at the edges of its strip rule: strips of 2, 4 and 8 rows, planes lower than a strip, of one row more and
one less than whole strips.  Against the general depthwise kernel, byte for byte (the oracle's comparisons are in test_gpu_int.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("B,C,H,W", [(1, 16, 1, 1), (1, 16, 2, 5), (1, 512, 7, 9), (1, 64, 9, 300), (3, 1024, 15, 16), (8, 512, 17, 14),
                                     (16, 512, 8, 15), (33, 256, 25, 20), (40, 512, 16, 7)])
def test_strips_equal_general_kernel(B, C, H, W, stride):
    from n2d2_amd import capi, runtime as rt
    from oracle.cells import ActSpec
    print("strips", B, C, H, W, stride, flush=True)
    rng = np.random.default_rng(B * H + W)
    w, bias = rng.integers(-128, 128, size=(C, 1, 3, 3)), rng.integers(-2000, 2001, size=C)
    spec = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 11, 2 ** 12, size=C), frac_bits=18, nb_bits=8, unsigned_out=True)
    x = rt.DTensor.from_numpy(rng.integers(0, 256, size=(B, C, H, W)), capi.U8B)
    got = {}
    for choice in (0, capi.KERNEL_NO_PIPE):
        conv = rt.Conv(w, bias, rt.Act(C, **spec.kwargs()), capi.U8B, stride=(stride, stride), pad=(1,) * 4, groups=C, kernel_choice=choice)
        got[choice] = conv.forward(x).to_numpy()
    assert np.array_equal(got[0], got[capi.KERNEL_NO_PIPE])


@pytest.mark.parametrize("B,C,H,W,stride,strips", [(40, 1024, 29, 20, 1, 2), (100, 1024, 13, 17, 1, 1), (110, 1024, 28, 16, 1, 1), (55, 512, 30, 33, 1, 2),
                                                   (170, 1024, 27, 20, 2, 1), (100, 512, 59, 40, 2, 3), (40, 1024, 59, 20, 2, 4)])
def test_long_strips_of_large_layers(B, C, H, W, stride, strips):
    """Layers that fill the chip several times over walk strips of up to 28 rows (14 with stride 2): how many a plane has, and the
    bytes of the general kernel."""
    import torch
    from n2d2_amd import capi, runtime as rt
    from oracle.cells import ActSpec
    print("long strips", B, C, H, W, stride, flush=True)
    rng = np.random.default_rng(B + H)
    w, bias = rng.integers(-128, 128, size=(C, 1, 3, 3)), rng.integers(-2000, 2001, size=C)
    spec = ActSpec("Rectifier", "FixedMult32", rng.integers(2 ** 11, 2 ** 12, size=C), frac_bits=18, nb_bits=8, unsigned_out=True)
    x = rt.DTensor(B, C, H, W, capi.U8B)
    x.buf.random_(-128, 128)
    outs = []
    for choice in (0, capi.KERNEL_NO_PIPE):
        conv = rt.Conv(w, bias, rt.Act(C, **spec.kwargs()), capi.U8B, stride=(stride, stride), pad=(1,) * 4, groups=C, kernel_choice=choice)
        with capi.launch_log() as log:
            outs.append(conv.forward(x))
        if choice == 0 and torch.cuda.get_device_properties(0).multi_processor_count == 256:          # (the lines were measured there)
            columns = B * outs[0].W * C // 4
            assert [e[0].startswith("depthwise3x3_kernel") for e in log.entries] == [True]
            assert 0 <= log.entries[0][1] * 256 - columns * strips < 8 * 256
    assert torch.equal(outs[0].buf, outs[1].buf)
