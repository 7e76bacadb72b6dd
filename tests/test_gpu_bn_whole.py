"""Batch normalisation whose statistics and values come from one launch: at the edges of the rule that chooses it, with planes and outputs that
16-byte accesses do not fit, against 64 bits.  The statistics are sums in double (2^-24 relative for the one rounding of each, and of their
moving averages); a value takes four roundings from them: 4 x 2^-24 of its terms, which are below 6 sigma here, 2e-6 absolute."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,C,H,W", [(1, 3, 1, 2), (2, 5, 3, 5), (2, 5, 4, 4), (13, 7, 3, 5), (31, 6, 16, 16), (32, 6, 16, 16), (1, 3, 1, 8191),
                                     (128, 1024, 1, 1), (129, 1024, 1, 1), (42, 256, 14, 14), (8, 300, 13, 9)])
@pytest.mark.parametrize("sat", [False, True])
def test_forward(B, C, H, W, sat):
    import torch
    from n2d2_amd import capi, runtime
    rng = np.random.default_rng(B * C + H)
    x = rng.normal(1.5, 2.0, size=(B, C, H, W)).astype(np.float32)
    scale, bias = rng.uniform(0.5, 1.5, C).astype(np.float32), rng.normal(0, 0.3, C).astype(np.float32)
    n = B * H * W
    x64 = x.astype(np.float64)
    mean, var = x64.mean(axis=(0, 2, 3)), x64.var(axis=(0, 2, 3))
    per = lambda v: v.astype(np.float64)[:, None, None]  # noqa: E731
    want = per(scale) * (x64 - per(mean)) / np.sqrt(per(var) + 1e-5) + per(bias)
    for offset in (0, 1):                        # of the tensors that are written: their loads and stores by 16 bytes or by 4
        dev = lambda v: torch.from_numpy(v).cuda()  # noqa: E731
        dx, ds, db, rm, rv = dev(x), dev(scale), dev(bias), torch.zeros(C, device="cuda"), torch.ones(C, device="cuda")
        sm, sv = torch.empty(C, device="cuda"), torch.empty(C, device="cuda")
        y, fp = (torch.full((x.size + 1,), -7.0, device="cuda")[offset:offset + x.size] for _ in range(2))
        alpha = torch.full((1,), 1.25, device="cuda")
        ws = torch.empty(int(capi.lib.n2d2hip_batchnorm_f32_workspace_bytes(B, C, H, W)), dtype=torch.uint8, device="cuda")
        p = [t.data_ptr() for t in (dx, ds, db, rm, rv, sm, sv)]
        if sat:
            capi.check(capi.lib.n2d2hip_batchnorm_f32_forward_sat(B, C, H, W, *p, 1e-5, 0.25, 0, y.data_ptr(), fp.data_ptr(), 15.0, alpha.data_ptr(),
                                                                  ws.data_ptr(), ws.numel(), runtime.stream_ptr()))
        else:
            capi.check(capi.lib.n2d2hip_batchnorm_f32_forward(B, C, H, W, *p, 1e-5, 0.25, 0, y.data_ptr(), ws.data_ptr(), ws.numel(), runtime.stream_ptr()))
        torch.cuda.synchronize()
        got = (fp if sat else y).cpu().numpy().reshape(x.shape)
        tol = 2e-6 * max(1.0, np.abs(want).max())
        if n > 2:
            assert np.abs(got - want).max() <= tol
        np.testing.assert_allclose(sm.cpu().numpy(), mean, rtol=2e-7, atol=2e-7)
        np.testing.assert_allclose(sv.cpu().numpy(), var, rtol=1e-6)
        np.testing.assert_allclose(rm.cpu().numpy(), 0.25 * mean, rtol=4e-7, atol=2e-7)
        np.testing.assert_allclose(rv.cpu().numpy(), 0.25 * var * n / (n - 1) + 0.75, rtol=2e-6)
        if sat:                                  # the quantizer of the values that were kept, in 32 bits as the kernel has it
            c = np.clip(got, np.float32(0), np.float32(1.25))
            q = np.floor(np.float32(15) * (c / np.float32(1.25)) + np.float32(0.5)) / np.float32(15) * np.float32(1.25)
            z = y.cpu().numpy().reshape(x.shape)
            assert (np.abs(z - q) > 1e-6).sum() <= 2 + x.size // 100000      # (ties)


@pytest.mark.parametrize("B,C,H,W", [(1, 3, 1, 2), (2, 5, 3, 5), (2, 5, 4, 4), (13, 7, 3, 5), (31, 6, 16, 16), (32, 6, 16, 16), (1, 3, 1, 8191),
                                     (128, 1024, 1, 1), (129, 1024, 1, 1), (42, 256, 14, 14), (8, 300, 13, 9)])
@pytest.mark.parametrize("in_place", [False, True])
def test_backward(B, C, H, W, in_place):
    """The formulas in 64 bits on the statistics given; the sums are in double and rounded once, dx is worked out in double and rounded: 2^-24 of
    its terms, and of the terms of the statistics' gradients, which are sums of products of both inputs."""
    import torch
    from n2d2_amd import capi, runtime
    rng = np.random.default_rng(B * C + W)
    x, dy = rng.normal(1.5, 2.0, size=(B, C, H, W)).astype(np.float32), rng.normal(0.1, 1.0, size=(B, C, H, W)).astype(np.float32)
    scale = rng.uniform(0.5, 1.5, C).astype(np.float32)
    mean, var = x.astype(np.float64).mean(axis=(0, 2, 3)).astype(np.float32), (x.astype(np.float64).var(axis=(0, 2, 3)) + 0.1).astype(np.float32)
    n = B * H * W
    per = lambda v: v.astype(np.float64)[:, None, None]  # noqa: E731
    x64, d64, sigma = x.astype(np.float64), dy.astype(np.float64), np.sqrt(var.astype(np.float64) + 1e-5)
    centred = x64 - per(mean)
    total = lambda v: v.sum(axis=(0, 2, 3))  # noqa: E731
    dscale, dbias = total(d64 * centred) / sigma, total(d64)
    dvar = -0.5 * total(d64 * centred) * scale / sigma ** 3
    dmean = -total(d64) * scale / sigma + dvar * total(-2.0 * centred) / n
    want = d64 * per(scale) / per(sigma) + per(dvar) * 2.0 * centred / n + per(dmean) / n
    size = lambda v: np.abs(v).sum(axis=(0, 2, 3))  # noqa: E731
    for offset in (0, 1):
        dev = lambda v: torch.from_numpy(v).cuda()  # noqa: E731
        dx, s, m, v = dev(x), dev(scale), dev(mean), dev(var)
        g = torch.zeros(x.size + 1, device="cuda")[offset:offset + x.size]
        g.copy_(dev(dy).flatten())
        out = g if in_place else torch.full((x.size + 1,), -7.0, device="cuda")[offset:offset + x.size]
        ds, db = torch.ones(C, device="cuda"), torch.ones(C, device="cuda")
        dm, dv = torch.empty(C, device="cuda"), torch.empty(C, device="cuda")
        ws = torch.empty(int(capi.lib.n2d2hip_batchnorm_f32_workspace_bytes(B, C, H, W)), dtype=torch.uint8, device="cuda")
        capi.check(capi.lib.n2d2hip_batchnorm_f32_backward(B, C, H, W, dx.data_ptr(), s.data_ptr(), m.data_ptr(), v.data_ptr(), 1e-5, g.data_ptr(), 0.0,
                                                           ds.data_ptr(), 1.0, db.data_ptr(), dm.data_ptr(), dv.data_ptr(), out.data_ptr(), ws.data_ptr(),
                                                           ws.numel(), runtime.stream_ptr()))
        torch.cuda.synchronize()
        eps = 2.0 ** -23
        host = lambda t: t.cpu().numpy().astype(np.float64)  # noqa: E731
        terms = size(d64 * centred)
        # (x - mean is rounded before it is summed, sigma after its root)
        assert (np.abs(host(ds) - dscale) <= 4 * eps * terms / sigma).all()
        assert (np.abs(host(db) - 1.0 - dbias) <= 4 * eps * (size(d64) + 1.0)).all()
        assert (np.abs(host(dv) - dvar) <= 8 * eps * terms * scale / sigma ** 3).all()
        loose = size(d64) * scale / sigma + terms * scale / sigma ** 3 * size(centred) / n
        assert (np.abs(host(dm) - dmean) <= 8 * eps * loose).all()
        bound = 8 * eps * (np.abs(d64) * per(scale / sigma) + per(terms * scale / sigma ** 3) * np.abs(centred) / n + per(loose) / n)
        assert (np.abs(host(out).reshape(x.shape) - want) <= bound).all()
        if not in_place:
            assert np.array_equal(g.cpu().numpy(), dy.flatten())
