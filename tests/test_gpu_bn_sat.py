"""Batch normalisation with the SAT quantizer applied on the way out against the two calls, bit for bit, and the sums of several
blocks finished by the launch that follows them against one block's: planes below and at the line between the two ways of
walking a tensor, of whole and broken quads, one and several blocks a channel, in place, learning and inference."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(3, 5, 1, 1), (2, 7, 9, 7), (40, 3, 7, 9), (2, 6, 8, 8), (5, 4, 10, 10), (32, 6, 10, 10), (3, 5, 9, 9), (130, 3, 9, 9), (140, 3, 7, 9), (33, 2, 16, 17), (20, 70, 32, 32)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("running", [0, 1])
@pytest.mark.parametrize("in_place", [False, True])
def test_quantized_on_the_way_out(shape, running, in_place):
    import torch
    from n2d2_amd import capi, runtime as rt
    print("bn sat", shape, running, in_place, flush=True)
    B, C, H, W = shape
    lib, rng = capi.lib, np.random.default_rng(B * C + H)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()
    x, scale, bias = dev(rng.normal(1, 2, shape)), dev(rng.normal(1, .3, C)), dev(rng.normal(0, .3, C))
    alpha, n = dev([1.7]), B * C * H * W
    ws = torch.empty(int(lib.n2d2hip_batchnorm_f32_workspace_bytes(B, C, H, W)), dtype=torch.uint8, device="cuda")
    out = {}
    for fused in (False, True):
        src = x.clone()
        y, fp = (src if in_place else torch.empty_like(x)), torch.empty_like(x)
        st = [dev(np.full(C, v)) for v in (0.2, 1.5, 9, 9)]
        args = [B, C, H, W, src.data_ptr(), scale.data_ptr(), bias.data_ptr()] + [s.data_ptr() for s in st] + [1e-4, 0.1, running, y.data_ptr()]
        if fused:
            capi.check(lib.n2d2hip_batchnorm_f32_forward_sat(*args, fp.data_ptr(), 15.0, alpha.data_ptr(), ws.data_ptr(), ws.numel(), rt.stream_ptr()))
        else:
            capi.check(lib.n2d2hip_batchnorm_f32_forward(*args, ws.data_ptr(), ws.numel(), rt.stream_ptr()))
            capi.check(lib.n2d2hip_sat_act_forward(y.data_ptr(), fp.data_ptr(), n, 15.0, alpha.data_ptr(), rt.stream_ptr()))
        out[fused] = [t.cpu().numpy() for t in (y, fp, *st)]
    for a, b in zip(out[False], out[True]):
        assert np.array_equal(a, b)
    if not running:                    # against 64 bits: x - mean over the root, its rounding errors and those of the statistics
        x64 = x.cpu().numpy().astype(np.float64)
        m, v = x64.mean((0, 2, 3)), x64.var((0, 2, 3))
        want = (x64 - m[:, None, None]) / np.sqrt(v + 1e-4)[:, None, None] * scale.cpu().numpy().astype(np.float64)[:, None, None] + bias.cpu().numpy()[:, None, None]
        assert np.max(np.abs(out[True][1] - want)) < 2e-5 * max(1.0, np.max(np.abs(want)))
        assert np.max(np.abs(out[True][4] - m)) < 1e-6 * np.max(np.abs(x64)) and np.max(np.abs(out[True][5] - v)) < 1e-5 * np.max(v)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("beta", [0.0, 0.5])
@pytest.mark.parametrize("to_input", [False, True])
def test_backward_finished_by_the_next_launch(shape, beta, to_input):
    """With the workspace (several blocks a channel, finished by the launch that writes diff_x) and without one (a block a channel)."""
    import torch
    from n2d2_amd import capi, runtime as rt
    print("bn backward", shape, beta, to_input, flush=True)
    B, C, H, W = shape
    lib, rng = capi.lib, np.random.default_rng(B * C + H)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()
    x, dy = dev(rng.normal(1, 2, shape)), dev(rng.normal(0, 1, shape))
    scale, m, v = dev(rng.normal(1, .3, C)), dev(rng.normal(1, .1, C)), dev(rng.uniform(3, 5, C))
    ws = torch.empty(int(lib.n2d2hip_batchnorm_f32_workspace_bytes(B, C, H, W)), dtype=torch.uint8, device="cuda")
    out = []
    for w in (None, ws):
        g = [dev(np.full(C, 0.25)) for _ in range(4)]
        dx = dy.clone()                # (diff_x over diff_y, as the cells use it)
        capi.check(lib.n2d2hip_batchnorm_f32_backward(B, C, H, W, x.data_ptr(), scale.data_ptr(), m.data_ptr(), v.data_ptr(), 1e-4, dx.data_ptr(), beta,
                                                      g[0].data_ptr(), beta, g[1].data_ptr(), g[2].data_ptr(), g[3].data_ptr(),
                                                      dx.data_ptr() if to_input else None, w.data_ptr() if w is not None else None,
                                                      w.numel() if w is not None else 0, rt.stream_ptr()))
        out.append([t.cpu().numpy() for t in (*g, dx)])
    # the sums are double on both sides and differ in their order only: one rounding to float apart
    for a, b in zip(*out):
        assert np.max(np.abs(a - b)) <= 4 * 2.0 ** -24 * max(1.0, np.max(np.abs(a)))


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("to_input", [False, True])
def test_quantizer_gradient_on_the_way_in(shape, beta, to_input):
    """The quantizer's gradient taken by the normalisation's sums against the two calls: the same bits but for alpha's gradient,
    whose double sum has another order."""
    import torch
    from n2d2_amd import capi, runtime as rt
    print("bn sat backward", shape, beta, to_input, flush=True)
    B, C, H, W = shape
    n = B * C * H * W
    lib, rng = capi.lib, np.random.default_rng(B * C + H)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()
    x, dy, fp, alpha = dev(rng.normal(1, 2, shape)), dev(rng.normal(0, 1, shape)), dev(rng.normal(0.8, 1, shape)), dev([1.7])
    scale, m, v = dev(rng.normal(1, .3, C)), dev(rng.normal(1, .1, C)), dev(rng.uniform(3, 5, C))
    ws = torch.empty(int(lib.n2d2hip_batchnorm_f32_backward_sat_workspace_bytes(B, C, H, W)), dtype=torch.uint8, device="cuda")
    qws = torch.empty(int(lib.n2d2hip_quantizer_workspace_bytes(n)), dtype=torch.uint8, device="cuda")
    out = []
    for fused in (False, True):
        g = [dev(np.full(C, 0.25)) for _ in range(4)]
        d, dx, da = dy.clone(), torch.full_like(dy, 9.0), dev([0.5])
        head = [B, C, H, W, x.data_ptr(), scale.data_ptr(), m.data_ptr(), v.data_ptr(), 1e-4]
        tail = [beta, g[0].data_ptr(), beta, g[1].data_ptr(), g[2].data_ptr(), g[3].data_ptr(), dx.data_ptr() if to_input else None, ws.data_ptr(), ws.numel(),
                rt.stream_ptr()]
        if fused:
            capi.check(lib.n2d2hip_batchnorm_f32_backward_sat(*head, fp.data_ptr(), 15.0, alpha.data_ptr(), beta, da.data_ptr(), d.data_ptr(), *tail))
        else:
            capi.check(lib.n2d2hip_sat_act_backward(d.data_ptr(), fp.data_ptr(), d.data_ptr(), n, 15.0, alpha.data_ptr(), beta, da.data_ptr(),
                                                    qws.data_ptr(), qws.numel(), rt.stream_ptr()))
            capi.check(lib.n2d2hip_batchnorm_f32_backward(*head, d.data_ptr(), *tail))
        out.append([t.cpu().numpy() for t in (*g, d, dx, da)])
    for a, b in zip(out[0][:-1], out[1][:-1]):
        assert np.array_equal(a, b)
    # one rounding to float apart (and one more where beta adds what was there)
    assert abs(out[0][-1][0] - out[1][-1][0]) <= 2 * 2.0 ** -23 * max(1.0, abs(out[0][-1][0]))
    assert lib.n2d2hip_batchnorm_f32_backward_sat(*head, fp.data_ptr(), 15.0, alpha.data_ptr(), beta, da.data_ptr(), d.data_ptr(), *tail[:-3], None, 0,
                                                  rt.stream_ptr()) == capi.ERR_WORKSPACE


@pytest.mark.parametrize("B,Cn,H,W,block", [(64, 300, 3, 3, 256), (16, 5, 8, 8, 256), (32, 2, 8, 8, 256), (27, 256, 1, 19, 512),
                                              (27, 257, 1, 19, 256), (16, 3, 8, 32, 512), (17, 3, 8, 32, 1024), (41, 7, 5, 5, 1024), (40, 7, 5, 5, 512)])
def test_a_channel_of_few_units_is_added_by_a_small_block(B, Cn, H, W, block):
    """A block of 1024 threads from 1025 units (values, or quads where the planes hold whole ones) a channel on, of 512 from 513 where
    256 compute units hold a channel each; mean and variance against 64 bits on either side of the lines."""
    import torch
    from n2d2_amd import capi, runtime as rt
    print("bn block", B, Cn, H, W, flush=True)
    x = torch.from_numpy(np.random.default_rng(B).normal(2.0, 3.0, (B, Cn, H, W)).astype(np.float32)).cuda()
    y, v = torch.empty_like(x), [torch.full((Cn,), float(i < 1 or i == 3), device="cuda") for i in range(6)]
    ws = torch.empty(int(capi.lib.n2d2hip_batchnorm_f32_workspace_bytes(B, Cn, H, W)), dtype=torch.uint8, device="cuda")
    with capi.launch_log() as log:
        capi.check(capi.lib.n2d2hip_batchnorm_f32_forward(B, Cn, H, W, x.data_ptr(), *(t.data_ptr() for t in v), 1e-5, 0.1, 0, y.data_ptr(), ws.data_ptr(),
                                                          ws.numel(), rt.stream_ptr()))
    assert [e[2] for e in log.entries if e[0].startswith("batchnorm_f32_stats_kernel")] == [block]
    x64 = x.double()
    m64, v64 = x64.mean((0, 2, 3)), x64.var((0, 2, 3), unbiased=False)
    assert float((v[4].double() - m64).abs().max()) <= float(m64.abs().max()) * 2.0 ** -23
    assert float(((v[5].double() - v64) / v64).abs().max()) <= 2.0 ** -22


@pytest.mark.parametrize("shape", SHAPES + [(64, 2, 64, 64)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("workspace", [False, True])
def test_backward_against_64_bits(shape, workspace):
    """A channel's sums are formed in double of x - mean as rounded to float (2^-24 of each) with 1 / sigma of a sigma rounded to float,
    and rounded once; dx then takes them as they were stored.  Bounds accordingly, twice 2^-24 for each rounding beside the sums."""
    import torch
    from n2d2_amd import capi, runtime as rt
    print("bn backward in 64 bits", shape, workspace, flush=True)
    B, C, H, W = shape
    lib, rng, u = capi.lib, np.random.default_rng(B + C * H), 2.0 ** -24
    x, dy = (rng.normal(k, 2 - k, shape).astype(np.float32) for k in (1, 0))
    scale, m, v = rng.normal(1, .3, C).astype(np.float32), rng.normal(1, .1, C).astype(np.float32), rng.uniform(.5, 5, C).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).cuda()
    X, D, S, M, V = map(dev, (x, dy, scale, m, v))
    ds, db, dm, dv, dx = (torch.empty(n, device="cuda") for n in (C, C, C, C, x.size))
    ws = torch.empty(int(lib.n2d2hip_batchnorm_f32_workspace_bytes(*shape)), dtype=torch.uint8, device="cuda")
    capi.check(lib.n2d2hip_batchnorm_f32_backward(*shape, X.data_ptr(), S.data_ptr(), M.data_ptr(), V.data_ptr(), 1e-5, D.data_ptr(), 0.0, ds.data_ptr(), 0.0,
                                                  db.data_ptr(), dm.data_ptr(), dv.data_ptr(), dx.data_ptr(), ws.data_ptr() if workspace else None,
                                                  ws.numel() if workspace else 0, rt.stream_ptr()))
    ds, db, dm, dv, dx = (t.cpu().numpy().astype(np.float64) for t in (ds, db, dm, dv, dx))
    d, n, at = dy.astype(np.float64), B * H * W, lambda a: a[:, None, None]
    c, g, sigma = x.astype(np.float64) - at(m.astype(np.float64)), scale.astype(np.float64), np.sqrt(v.astype(np.float64) + 1e-5)
    total = lambda a: a.sum((0, 2, 3))
    near = lambda got, want, terms: np.testing.assert_array_less(np.abs(got - want), u * terms + 1e-30)
    near(ds, total(d * c) / sigma, 4 * total(np.abs(d * c)) / sigma)
    near(db, total(d), total(np.abs(d)))
    near(dv, -.5 * g * total(d * c) / sigma ** 3, 4 * np.abs(g) * total(np.abs(d * c)) / sigma ** 3)
    near(dm, -g * total(d) / sigma - 2 * dv * total(c) / n, 8 * (np.abs(g) * total(np.abs(d)) / sigma + 2 * np.abs(dv) * total(np.abs(c)) / n))
    parts = [d * at(g / sigma), 2 * at(dv) * c / n, np.broadcast_to(at(dm) / n, shape)]
    near(dx.reshape(shape), sum(parts), 6 * sum(np.abs(p) for p in parts))
