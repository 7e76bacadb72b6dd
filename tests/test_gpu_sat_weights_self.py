"""SAT weight levels where every block looks for the tensor's largest weight itself: at both ends of that range, from memory that 16-byte
loads do not fit, with the largest weight in the first, the last and the remainder's place, and over the weights themselves, which other blocks
must not be reading: bit-identical to levels computed in place or, with scaling, to a rounding of the scaling (its sums are in double)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _levels(n, offset, largest, scaling, in_place):
    import torch
    from n2d2_amd import capi, runtime
    host = np.random.default_rng(n).normal(0, 0.05, size=n).astype(np.float32)
    host[largest] = -0.75
    w = torch.zeros(n + 8, device="cuda")[offset:offset + n]
    w.copy_(torch.from_numpy(host))
    wq = w if in_place else torch.full((n + 8,), -7.0, device="cuda")[offset:offset + n]
    stats, ws = torch.empty(2, device="cuda"), torch.full((int(capi.lib.n2d2hip_quantizer_workspace_bytes(n)),), 0x7F, dtype=torch.uint8, device="cuda")
    capi.check(capi.lib.n2d2hip_sat_weight_forward(w.data_ptr(), wq.data_ptr(), n, 15.0, capi.SAT_DEFAULT, int(scaling), 10, stats.data_ptr(),
                                                   ws.data_ptr(), ws.numel(), runtime.stream_ptr()))
    torch.cuda.synchronize()
    return host, wq.cpu().numpy(), stats.cpu().numpy()


@pytest.mark.parametrize("scaling", [False, True])
@pytest.mark.parametrize("n", [1024, 1025, 8192, 8193, 8195, 65535, 65536, 65537])
def test_levels(n, scaling):
    from oracle import oracle as orc
    host, want, stats = _levels(n, 0, n // 2, scaling, True)
    ref, tmax, _ = orc.sat_weight_forward(host.astype(np.float64) if scaling else host, 15.0, "default", apply_scaling=scaling, outputs_size=10)
    assert abs(stats[0] - tmax) <= 1e-6 * tmax
    # (in 64 bits with scaling, as the sums of 65536 squares in 32 are off by 3e-4; a level moves where tanh's last bit lies on a tie)
    assert (np.abs(want - ref) > 1e-5 * np.abs(ref).max()).sum() <= max(2, int(2e-4 * n))
    for offset, largest in ((0, n // 2), (1, n // 2), (3, n // 2)):
        _, got, st = _levels(n, offset, largest, scaling, False)
        assert st[0] == stats[0]
        np.testing.assert_allclose(got, want, rtol=6e-7 if scaling else 0, atol=0)
    for offset, largest in ((0, 0), (0, n - 1), (2, n - 1)):
        _, got, st = _levels(n, offset, largest, scaling, False)
        assert st[0] == stats[0] and abs(got[largest] * st[1] + 1.0) <= 2.4e-7       # (the division's rounding and the product's)
