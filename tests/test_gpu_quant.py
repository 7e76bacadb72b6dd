"""GPU parity of the SAT / LSQ fake-quant kernels against the CPU oracle:
1e-5 relative.  Elements whose pre-rounding value sits within 1e-5 of a rounding
tie may land on the neighbouring level (device tanh/division differ from libm in
the last bit); the tests bound how many and by how much."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(99)
TOL = 1e-5


@pytest.fixture(scope="module")
def q():
    import torch
    from n2d2_amd import capi, runtime

    class Q:
        lib, check, sp = capi.lib, staticmethod(capi.check), staticmethod(runtime.stream_ptr)

        @staticmethod
        def dev(a):
            return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()

        @staticmethod
        def ws(n):
            return torch.empty(int(capi.lib.n2d2hip_quantizer_workspace_bytes(n)), dtype=torch.uint8, device="cuda")

        @staticmethod
        def host(t):
            torch.cuda.synchronize()
            return t.cpu().numpy()
        empty = staticmethod(lambda n: torch.empty(n, dtype=torch.float32, device="cuda"))
        zeros = staticmethod(lambda n: torch.zeros(n, dtype=torch.float32, device="cuda"))
    return Q


def _close(got, want, scale=None):
    scale = np.maximum(np.abs(want), 1e-3) if scale is None else scale
    return np.abs(got.astype(np.float64) - want.astype(np.float64)) <= TOL * scale


MODES = {"none": 0, "default": 1, "fullrange": 2, "symrange": 3, "asymrange": 4, "none_asym": 5}


@pytest.mark.parametrize("mode,rng", [("symrange", 15.0), ("default", 15.0), ("fullrange", 15.0), ("asymrange", 15.0),
                                      ("none", 15.0), ("none_asym", 15.0), ("symrange", 255.0), ("default", 255.0)])
def test_sat_weight_forward_backward(q, mode, rng):
    from oracle import oracle as orc
    for shape in ((64, 64, 3, 3), (128, 64, 1, 1), (7, 3, 5, 5)):
        w = RNG.normal(0, 0.05, size=shape).astype(np.float32).reshape(-1)
        n = w.size
        want, tmax, _ = orc.sat_weight_forward(w, rng, mode)
        dw_, dwq_, dstats, ws = q.dev(w), q.empty(n), q.empty(2), q.ws(n)
        q.check(q.lib.n2d2hip_sat_weight_forward(dw_.data_ptr(), dwq_.data_ptr(), n, rng, MODES[mode], 0, 1, dstats.data_ptr(),
                                                 ws.data_ptr(), ws.numel(), q.sp()))
        got, stats = q.host(dwq_), q.host(dstats)
        assert abs(stats[0] - tmax) <= TOL * tmax
        ok = _close(got, want, scale=1.0)
        levels = {"symrange": np.floor(rng / 2), "asymrange": np.floor(rng / 2), "default": rng / 2, "fullrange": rng / 2}.get(mode)
        if levels is None:
            assert ok.all()
        else:
            # off-by-one-level only at rounding ties, and rarely
            bad = ~ok
            assert bad.sum() <= max(2, int(2e-4 * n)), (mode, bad.sum())
            assert np.all(np.abs(np.abs(got[bad] - want[bad]) * levels - 1.0) < 1e-3)
        # backward
        g = RNG.normal(size=n).astype(np.float32)
        want_b = orc.sat_weight_backward(g, w, rng, np.float32(tmax), mode if mode in ("fullrange", "asymrange") else "default")
        if mode == "none_asym":
            want_b = orc.sat_weight_backward(g, w, rng, np.float32(tmax), "asymrange")
        dg, dout = q.dev(g), q.empty(n)
        q.check(q.lib.n2d2hip_sat_weight_backward(dg.data_ptr(), dw_.data_ptr(), dout.data_ptr(), n, rng, MODES[mode], 0, dstats.data_ptr(), q.sp()))
        assert _close(q.host(dout), want_b, scale=np.maximum(np.abs(want_b), 1e-2)).all()


def test_sat_weight_scaling(q):
    from oracle import oracle as orc
    shape = (120, 400)                       # an FC layer, ApplyScaling = 1
    w = RNG.normal(0, 0.05, size=shape).astype(np.float32).reshape(-1)
    n = w.size
    want, tmax, scal = orc.sat_weight_forward(w.astype(np.float64), 15.0, "symrange", apply_scaling=True, outputs_size=120)
    dw_, dwq_, dstats, ws = q.dev(w), q.empty(n), q.empty(2), q.ws(n)
    q.check(q.lib.n2d2hip_sat_weight_forward(dw_.data_ptr(), dwq_.data_ptr(), n, 15.0, 3, 1, 120, dstats.data_ptr(), ws.data_ptr(), ws.numel(), q.sp()))
    got, stats = q.host(dwq_), q.host(dstats)
    assert abs(stats[1] - scal) <= TOL * scal
    ok = _close(got, want, scale=np.abs(want).max())
    assert (~ok).sum() <= 2
    # and against the float32 oracle, whose sequential float sums carry more rounding error than the tolerance allows at scale
    want32, _, scal32 = orc.sat_weight_forward(w, 15.0, "symrange", apply_scaling=True, outputs_size=120)
    assert abs(stats[1] - scal32) <= 5e-5 * scal32
    g = RNG.normal(size=n).astype(np.float32)
    want_b = orc.sat_weight_backward(g, w, 15.0, np.float32(stats[0]) * np.float32(stats[1]), "default")
    dg, dout = q.dev(g), q.empty(n)
    q.check(q.lib.n2d2hip_sat_weight_backward(dg.data_ptr(), dw_.data_ptr(), dout.data_ptr(), n, 15.0, 3, 1, dstats.data_ptr(), q.sp()))
    assert _close(q.host(dout), want_b, scale=np.maximum(np.abs(want_b), 1e-2)).all()


@pytest.mark.parametrize("alpha,rng", [(6.0, 15.0), (1.5, 255.0), (-2.0, 15.0)])
def test_sat_activation_forward_backward(q, alpha, rng):
    from oracle import oracle as orc
    n = 64 * 56 * 56 + 3
    x = RNG.normal(2.0, 3.0, size=n).astype(np.float32)
    x[:4] = [0.0, abs(alpha), -1.0, abs(alpha) * 2]
    want, fp = orc.sat_act_forward(x, rng, alpha, inference=False)
    dx, dfp, dalpha = q.dev(x), q.empty(n), q.dev([alpha])
    q.check(q.lib.n2d2hip_sat_act_forward(dx.data_ptr(), dfp.data_ptr(), n, rng, dalpha.data_ptr(), q.sp()))
    got = q.host(dx)
    assert np.array_equal(q.host(dfp), x)
    ok = _close(got, want, scale=abs(alpha))
    assert (~ok).sum() <= max(2, int(2e-5 * n))
    assert np.all(np.abs(np.abs(got[~ok] - want[~ok]) * rng / abs(alpha) - 1.0) < 1e-3)
    # inference flavour: no copy
    dx2 = q.dev(x)
    q.check(q.lib.n2d2hip_sat_act_forward(dx2.data_ptr(), None, n, rng, dalpha.data_ptr(), q.sp()))
    assert np.array_equal(q.host(dx2), got)
    # backward
    g = RNG.normal(size=n).astype(np.float32)
    want_dx, want_da, terms = orc.sat_act_backward(g.astype(np.float64), x.astype(np.float64), rng, alpha, beta=1.0, prev_diff_alpha=3.0)
    dg, ddx, dda, ws = q.dev(g), q.empty(n), q.dev([3.0]), q.ws(n)
    q.check(q.lib.n2d2hip_sat_act_backward(dg.data_ptr(), dfp.data_ptr(), ddx.data_ptr(), n, rng, dalpha.data_ptr(), 1.0, dda.data_ptr(),
                                           ws.data_ptr(), ws.numel(), q.sp()))
    assert np.array_equal(q.host(ddx), want_dx.astype(np.float32))          # pure masking: exact
    # the sum is order dependent: compare with the float64 oracle, relative to the magnitude summed
    assert abs(q.host(dda)[0] - want_da) <= TOL * np.abs(terms).sum()


@pytest.mark.parametrize("lo,hi", [(-8, 7), (0, 15), (-128, 127)])
def test_lsq_forward_backward(q, lo, hi):
    from oracle import oracle as orc
    n = 128 * 128 * 9 + 2
    step = np.float32(0.013)
    x = RNG.normal(0, 0.05, size=n).astype(np.float32)
    want = orc.lsq_forward(x, step, lo, hi)
    dx, dq_, dstep = q.dev(x), q.empty(n), q.dev([step])
    q.check(q.lib.n2d2hip_lsq_forward(dx.data_ptr(), dq_.data_ptr(), n, dstep.data_ptr(), lo, hi, q.sp()))
    got = q.host(dq_)
    ok = _close(got, want, scale=np.maximum(np.abs(want), float(step)))
    assert (~ok).sum() <= 2
    g = RNG.normal(size=n).astype(np.float32)
    want_dfp, want_sum = orc.lsq_backward(g.astype(np.float64), x.astype(np.float64), float(step), lo, hi)
    grad_scale = np.float32(1.0 / np.sqrt(n * hi))
    dg, ddfp, dds, ws = q.dev(g), q.empty(n), q.dev([0.5]), q.ws(n)
    q.check(q.lib.n2d2hip_lsq_backward(dg.data_ptr(), dx.data_ptr(), ddfp.data_ptr(), n, dstep.data_ptr(), lo, hi, float(grad_scale), 1.0,
                                       dds.data_ptr(), ws.data_ptr(), ws.numel(), q.sp()))
    assert np.array_equal(q.host(ddfp), want_dfp.astype(np.float32))
    # the sum is order dependent: held, like every other reduction, to TOL of the magnitude summed (float64 oracle)
    qv = x.astype(np.float64) / float(step)
    summed = np.abs(np.where(qv <= lo, lo, np.where(qv >= hi, hi, np.sign(qv) * np.floor(np.abs(qv) + 0.5) - qv)) * g).sum()
    want_ds = (want_sum + 0.5) * grad_scale
    assert abs(q.host(dds)[0] - want_ds) <= TOL * summed * grad_scale
    # new iteration: beta = 0 discards the previous value
    dds2 = q.dev([123.0])
    q.check(q.lib.n2d2hip_lsq_backward(dg.data_ptr(), dx.data_ptr(), ddfp.data_ptr(), n, dstep.data_ptr(), lo, hi, float(grad_scale), 0.0,
                                       dds2.data_ptr(), ws.data_ptr(), ws.numel(), q.sp()))
    assert abs(q.host(dds2)[0] - want_sum * grad_scale) <= TOL * summed * grad_scale


@pytest.mark.parametrize("n", [2, 1023, 1024, 1025, 10080, 16384, 16385])
@pytest.mark.parametrize("mode", ["default", "none"])
def test_sat_weights_around_the_one_launch_size(q, n, mode):
    """Up to 16 weights for each of 1024 threads run in one launch: both sides of that and of a thread's share, with scaling."""
    from oracle import oracle as orc
    w = np.random.default_rng(n).normal(0, 0.05, size=n).astype(np.float32)
    want, tmax, scal = orc.sat_weight_forward(w.astype(np.float64), 15.0, mode, apply_scaling=True, outputs_size=7)
    dw_, dwq_, dstats, ws = q.dev(w), q.empty(n), q.empty(2), q.ws(n)
    q.check(q.lib.n2d2hip_sat_weight_forward(dw_.data_ptr(), dwq_.data_ptr(), n, 15.0, MODES[mode], 1, 7, dstats.data_ptr(), ws.data_ptr(), ws.numel(),
                                             q.sp()))
    got, stats = q.host(dwq_), q.host(dstats)
    assert abs(stats[0] - tmax) <= TOL * tmax
    moved = ~_close(got * stats[1], want * scal, scale=1.0)
    # a weight on a rounding edge moves by a level, 2 / 15, and the variance (of order 0.05) by up to 2 * 2 / 15 / n
    assert moved.sum() <= 2 and np.all(np.abs(got[moved] * stats[1] - want[moved] * scal) <= 2.0 / 15.0 + 1e-4)
    assert abs(stats[1] - scal) <= (TOL + 3.0 * moved.sum() / n) * scal


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 4, 1027, 4096, 4097, 9002])
def test_quantizer_backward_sizes_and_alignments(q, n, shift):
    """Quads and what is left of them, one block and several, tensors that start beside a 16-byte boundary, in place."""
    from oracle import oracle as orc
    rng = np.random.default_rng(n)
    x, g = rng.normal(1.0, 2.0, size=n).astype(np.float32), rng.normal(size=n).astype(np.float32)
    at = lambda a: q.dev(np.concatenate([np.zeros(shift, dtype=np.float32), a]))[shift:]
    dx_, ws = at(x), q.ws(n)
    want_dx, want_da, terms = orc.sat_act_backward(g.astype(np.float64), x.astype(np.float64), 15.0, 1.5, beta=1.0, prev_diff_alpha=3.0)
    dg, dda, dalpha, dstep = at(g), q.dev([3.0]), q.dev([1.5]), q.dev([0.25])
    q.check(q.lib.n2d2hip_sat_act_backward(dg.data_ptr(), dx_.data_ptr(), dg.data_ptr(), n, 15.0, dalpha.data_ptr(), 1.0, dda.data_ptr(),
                                           ws.data_ptr(), ws.numel(), q.sp()))
    assert np.array_equal(q.host(dg), want_dx.astype(np.float32))
    assert abs(q.host(dda)[0] - want_da) <= TOL * (np.abs(terms).sum() + 3.0)
    want_dfp, want_sum = orc.lsq_backward(g.astype(np.float64), x.astype(np.float64), 0.25, -8, 7)
    dg, dds = at(g), q.dev([0.5])
    q.check(q.lib.n2d2hip_lsq_backward(dg.data_ptr(), dx_.data_ptr(), dg.data_ptr(), n, dstep.data_ptr(), -8, 7, 0.5, 1.0, dds.data_ptr(),
                                       ws.data_ptr(), ws.numel(), q.sp()))
    assert np.array_equal(q.host(dg), want_dfp.astype(np.float32))
    assert abs(q.host(dds)[0] - (want_sum + 0.5) * 0.5) <= TOL * (8 * np.abs(g).sum() + 1.0)
