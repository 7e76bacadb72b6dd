"""The forward pass of a layer that spans its input against the same sum in float32 on the host, term for term: equal bits, at the
remainders of the kernel's steps of 128 terms, stages of 256, 8 images and 8 outputs, on both sides of the line between the two kernels."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ordered(B, K, O):
    """-> (the sum in the terms' order on the host, the call's, the launches)"""
    import torch
    from n2d2_amd import capi, runtime as rt
    rng = np.random.default_rng(K + O)
    x, w, bias, y0 = (rng.normal(size=s).astype(np.float32) for s in ((B, K), (O, K), (O,), (B, O)))
    want = np.zeros((B, O), np.float32)
    for k in range(K):
        want = want + w[None, :, k] * x[:, k, None]
    want = bias[None] + (want + np.float32(0.5) * y0)
    d = capi.ConvDesc(K // 4, O, 2, 2, 1, 1, 0, 0, 0, 0, 1, 1, 1, 0, capi.KERNEL_F32_DIRECT)
    dx, dw, db, dy = (torch.from_numpy(a).cuda() for a in (x, w, bias, y0))
    with capi.launch_log() as log:
        capi.check(capi.lib.n2d2hip_conv2d_f32_forward(C.byref(d), B, 2, 2, dx.data_ptr(), dw.data_ptr(), db.data_ptr(), 0.5, dy.data_ptr(), None, 0,
                                                       rt.stream_ptr()))
    torch.cuda.synchronize()
    return want, dy.cpu().numpy(), log.entries


@pytest.mark.parametrize("B,K,O", [(1, 60, 2), (2, 64, 1), (3, 68, 3), (1, 508, 1), (2, 512, 5), (5, 516, 2), (7, 1020, 10), (4, 1024, 9), (1, 1028, 3),
                                   (2, 2108, 2), (64, 200, 128), (65, 200, 128), (65, 516, 127), (91, 252, 91), (96, 772, 121), (128, 1028, 128)])
def test_four_sums_a_wave_and_sixty_four_a_work_group(B, K, O):
    """Up to two waves of four sums a SIMD, rings of 8 times 64 terms; past that work-groups of 64 sums: equal bits on either side of
    the line, at the remainders of both."""
    import torch
    print("chain forms", B, K, O, flush=True)
    want, got, log = _ordered(B, K, O)
    waves = -(-B // 2) * -(-O // 2)
    few = waves <= 8 * torch.cuda.get_device_properties(0).multi_processor_count
    assert [e[:3] for e in log] == [("conv_f32_chain_kernel", waves, 64) if few else ("conv_f32_chain_kernel", -(-B // 8) * -(-O // 8), 192)]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("B,K,O", [(1, 4, 1), (8, 124, 8), (9, 128, 7), (3, 132, 9), (8, 252, 16), (5, 256, 3), (2, 260, 8), (17, 384, 10), (8, 508, 8),
                                   (1, 768, 12), (8, 772, 1), (4, 1020, 8), (7, 1024, 5), (3, 2308, 11), (128, 132, 121),
                                   (137, 4, 121), (136, 124, 128), (131, 128, 127), (129, 772, 125), (2049, 260, 3), (130, 1028, 123)])
def test_equals_ordered_float32_sum(B, K, O):
    import torch
    from n2d2_amd import capi, runtime as rt
    print("chain", B, K, O, flush=True)
    rng = np.random.default_rng(K + O)
    x, w, bias, y0 = (rng.normal(size=s).astype(np.float32) for s in ((B, K), (O, K), (O,), (B, O)))
    want = np.zeros((B, O), np.float32)
    for k in range(K):
        want = want + w[None, :, k] * x[:, k, None]
    want = bias[None] + (want + np.float32(0.5) * y0)
    d = capi.ConvDesc(K // 4, O, 2, 2, 1, 1, 0, 0, 0, 0, 1, 1, 1, 0, capi.KERNEL_F32_DIRECT)
    dev = lambda a: torch.from_numpy(a).cuda()
    dx, dw, db, dy = dev(x), dev(w), dev(bias), dev(y0)
    with capi.launch_log() as log:
        capi.check(capi.lib.n2d2hip_conv2d_f32_forward(C.byref(d), B, 2, 2, dx.data_ptr(), dw.data_ptr(), db.data_ptr(), 0.5, dy.data_ptr(), None, 0,
                                                       rt.stream_ptr()))
    # a compute unit holds one work-group of 8 x 8 sums of the kernel whose waves share the work, and three of the other
    many = -(-B // 8) * -(-O // 8) > torch.cuda.get_device_properties(0).multi_processor_count
    assert [e[0] for e in log.entries] == ["conv_f32_chain_wave_kernel" if many else "conv_f32_chain_kernel"]
    torch.cuda.synchronize()
    assert np.array_equal(dy.cpu().numpy(), want)
