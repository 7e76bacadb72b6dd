"""The SAT weight quantizer where a tensor goes from one block to many, with and without scaling, and where its blocks grow: against
the CPU oracle, alone (n2d2hip_sat_weight_forward) and in one batch with tensors of other kinds (n2d2hip_sat_weight_forward_batch:
bit-identical to alone).  The scaling is sqrt of a float variance of n levels: a handful of roundings of 2^-24 (the sums are in
double), so 1e-6; a level moves where tanh's last bit lies on a tie, a handful in 10^4."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MODES = {"default": 1, "symrange": 3}


def _tensor(torch, lib, n, seed, given=None):
    w = np.random.default_rng(seed).normal(0, 0.05, size=n).astype(np.float32) if given is None else given
    ws = torch.full((int(lib.n2d2hip_quantizer_workspace_bytes(n)),), 0x7F, dtype=torch.uint8, device="cuda")
    return w, torch.from_numpy(w).cuda(), torch.full((n,), -7.0, device="cuda"), torch.full((2,), -7.0, device="cuda"), ws


def _forward(torch, capi, runtime, t, mode, scaling, outputs):
    _, dw, wq, stats, ws = t
    capi.check(capi.lib.n2d2hip_sat_weight_forward(dw.data_ptr(), wq.data_ptr(), dw.numel(), 15.0, MODES[mode], int(scaling), outputs,
                                                   stats.data_ptr(), ws.data_ptr(), ws.numel(), runtime.stream_ptr()))
    torch.cuda.synchronize()
    return wq.cpu().numpy(), stats.cpu().numpy()


@pytest.mark.parametrize("n,scaling", [(2, True), (1025, True), (8192, False), (8193, False), (12288, True), (12289, True), (114688, True), (114689, True),
                                       ((2 << 20) - 1, True), (2 << 20, True), ((4 << 20) + 13, True)])
@pytest.mark.parametrize("mode", sorted(MODES))
def test_one_block_to_many(n, scaling, mode):
    import torch
    from n2d2_amd import capi, runtime
    from oracle import oracle as orc
    t = _tensor(torch, capi.lib, n, n % 1000)
    got, st = _forward(torch, capi, runtime, t, mode, scaling, 84)
    ref, tmax, scal = orc.sat_weight_forward(t[0].astype(np.float64) if scaling else t[0], 15.0, mode, apply_scaling=scaling, outputs_size=84)
    assert abs(st[0] - tmax) <= 1e-6 * tmax and abs(st[1] - scal) <= max(1e-6, 4.0 / n) * scal, (st, tmax, scal)
    bad = np.abs(got.astype(np.float64) - ref) > 1e-5 * np.abs(ref).max()
    assert bad.sum() <= max(2, int(2e-4 * n)), int(bad.sum())
    # the scaling, of the levels that came out: in 64 bits
    if scaling and n > 2:
        levels = np.rint(got.astype(np.float64) * st[1] * 1e6) / 1e6
        assert abs(np.sqrt(levels.var(ddof=1) * 84) - st[1]) <= 2e-6 * st[1]


def test_batch_of_all_kinds_is_each_alone():
    import torch
    from n2d2_amd import capi, runtime
    kinds = [(150, 0), (9000, 0), (12289, 1), (840, 1), ((2 << 20) + 5, 1), (70000, 0), (20000, 1)]
    for some in (kinds, kinds[:4]):
        alone, items, keep = [], [], []
        for i, (n, scaling) in enumerate(some):
            t = _tensor(torch, capi.lib, n, i)
            alone.append(_forward(torch, capi, runtime, t, "default", scaling, 10))
            t = _tensor(torch, capi.lib, n, i)
            keep.append(t)
            items.append(capi.SatWeightItem(t[1].data_ptr(), t[2].data_ptr(), n, 15.0, 1, scaling, 10, t[3].data_ptr(), t[4].data_ptr(), t[4].numel()))
        arr = (capi.SatWeightItem * len(items))(*items)
        capi.check(capi.lib.n2d2hip_sat_weight_forward_batch(arr, len(items), runtime.stream_ptr()))
        torch.cuda.synchronize()
        for (wq, st), t in zip(alone, keep):
            # (a batch's blocks can be of another size, which adds the same sums in another order: a rounding of the scaling)
            np.testing.assert_allclose(t[3].cpu().numpy(), st, rtol=3e-7)
            np.testing.assert_allclose(t[2].cpu().numpy(), wq, rtol=6e-7, atol=0)


@pytest.mark.parametrize("n", [4096, 12289])
def test_equal_weights_and_nan(n):
    """No variance: a division by zero, as the formula has it; a NaN reaches the scaling and every level, but not the maximum."""
    import torch
    from n2d2_amd import capi, runtime
    got, st = _forward(torch, capi, runtime, _tensor(torch, capi.lib, n, 0, np.full(n, 0.25, np.float32)), "default", 1, 10)
    assert st[1] == 0.0 and np.isinf(got).all()
    for at in (0, n - 1):
        w = np.random.default_rng(1).normal(0, 0.05, size=n).astype(np.float32)
        w[at] = np.nan
        got, st = _forward(torch, capi, runtime, _tensor(torch, capi.lib, n, 0, w), "default", 1, 10)
        assert np.isfinite(st[0]) and np.isnan(st[1]) and np.isnan(got).all()
