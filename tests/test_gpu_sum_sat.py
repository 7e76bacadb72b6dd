"""A float sum with the SAT quantizer behind it, forwards and backwards in one pass each, and the SAT weights' gradients in the launch that updates
the weights: bit for bit what the single calls leave (the same operations in the same order), over counts and addresses that 16-byte loads do
not fit, one and several blocks, an input that is there twice, gradients that are added to."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _floats(torch, rng, n, offset):
    t = torch.zeros(n + 4, device="cuda")[offset:offset + n]
    t.copy_(torch.from_numpy(rng.normal(0.4, 1.0, n).astype(np.float32)))
    return t


@pytest.mark.parametrize("inputs", [1, 2, 3, 8])
@pytest.mark.parametrize("n,offset", [(1, 0), (7, 0), (4096, 0), (4097, 0), (4100, 1), (300004, 0)])
def test_sum_and_quantizer(n, offset, inputs):
    import torch
    from n2d2_amd import capi, runtime as rt
    lib, st, rng = capi.lib, rt.stream_ptr(), np.random.default_rng(n + inputs)
    p = lambda ts: (C.c_void_p * len(ts))(*(t.data_ptr() for t in ts))  # noqa: E731
    f = lambda v: (C.c_float * len(v))(*v)  # noqa: E731
    xs = [_floats(torch, rng, n, offset) for _ in range(inputs)]
    w, s, alpha = f(rng.uniform(0.5, 1.5, inputs)), f(rng.uniform(-0.1, 0.1, inputs)), torch.tensor([1.7], device="cuda")
    y, fp, y1, fp1 = (_floats(torch, rng, n, offset) for _ in range(4))
    capi.check(lib.n2d2hip_elemwise_sum_f32_forward(inputs, p(xs), n, w, s, y.data_ptr(), st))
    capi.check(lib.n2d2hip_sat_act_forward(y.data_ptr(), fp.data_ptr(), n, 15.0, alpha.data_ptr(), st))
    capi.check(lib.n2d2hip_elemwise_sum_f32_forward_sat(inputs, p(xs), n, w, s, y1.data_ptr(), fp1.data_ptr(), 15.0, alpha.data_ptr(), st))
    assert torch.equal(y, y1) and torch.equal(fp, fp1)
    y1.fill_(-7.0)
    capi.check(lib.n2d2hip_elemwise_sum_f32_forward_sat(inputs, p(xs), n, w, s, y1.data_ptr(), None, 15.0, alpha.data_ptr(), st))
    assert torch.equal(y, y1)

    ws = torch.empty(int(lib.n2d2hip_quantizer_workspace_bytes(n)), dtype=torch.uint8, device="cuda")
    dy = _floats(torch, rng, n, offset)
    dxs = [_floats(torch, rng, n, offset) for _ in range(inputs)]
    betas = [float(k % 2) for k in range(inputs)]
    if inputs == 3:                                    # the first input once more: its second part is added to the first
        dxs[1], betas[1] = dxs[0], 1.0
    dy1 = dy.clone() if offset == 0 else _floats(torch, rng, n, offset).copy_(dy)
    dxs1 = [d.clone() for d in dxs]
    if inputs == 3:
        dxs1[1] = dxs1[0]
    da, da1 = torch.tensor([0.25], device="cuda"), torch.tensor([0.25], device="cuda")
    capi.check(lib.n2d2hip_sat_act_backward(dy.data_ptr(), fp.data_ptr(), dy.data_ptr(), n, 15.0, alpha.data_ptr(), 1.0, da.data_ptr(), ws.data_ptr(),
                                            ws.numel(), st))
    for k in range(inputs):
        capi.check(lib.n2d2hip_elemwise_sum_f32_backward(n, w[k], dy.data_ptr(), betas[k], dxs[k].data_ptr(), st))
    capi.check(lib.n2d2hip_elemwise_sum_f32_backward_sat(inputs, n, w, f(betas), p(dxs1), dy1.data_ptr(), fp.data_ptr(), 15.0, alpha.data_ptr(), 1.0,
                                                         da1.data_ptr(), ws.data_ptr(), ws.numel(), st))
    assert torch.equal(dy, dy1) and all(torch.equal(a, b) for a, b in zip(dxs, dxs1))
    # (the blocks' sums are in double; where addresses differ in what they allow, in another order)
    assert abs(float(da) - float(da1)) <= 1e-6 * max(1.0, abs(float(da)))


def test_weights_gradients_with_their_update():
    """40 tensors, more than a launch holds, 20 with gradients, two of which no item updates; momentum, decay, clamping."""
    import torch
    from n2d2_amd import capi, runtime as rt
    lib, st, rng = capi.lib, rt.stream_ptr(), np.random.default_rng(5)

    def run(together):
        rng = np.random.default_rng(5)
        keep, items, grads, out = [], [], [], []
        for k in range(40):
            n = [1, 255, 256, 257, 3000, 70001][k % 6]
            w, dq, dw, m = (_floats(torch, rng, n, 0) for _ in range(4))
            stats = torch.tensor([0.8, 1.3], device="cuda")
            keep.append((w, dq, dw, m, stats))
            if k % 2 == 0:
                grads.append(capi.SatWeightGradItem(dq.data_ptr(), w.data_ptr(), dw.data_ptr(), n, 15.0, [1, 2, 4][k % 3], k % 4 == 0, stats.data_ptr()))
            if k not in (8, 38):
                items.append(capi.SgdItem(w.data_ptr(), dw.data_ptr(), n, m.data_ptr() if k % 3 else None, 0.01, 0.9 if k % 3 else 0.0,
                                          1e-3 if k % 3 == 2 else 0.0, -0.5, 0.5, k % 5 == 0))
            out += [w, dw, m]
        ai, ag = (capi.SgdItem * len(items))(*items), (capi.SatWeightGradItem * len(grads))(*grads)
        if together:
            capi.check(lib.n2d2hip_sgd_update_f32_batch_sat(ai, len(items), ag, len(grads), st))
        else:
            capi.check(lib.n2d2hip_sat_weight_backward_batch(ag, len(grads), st))
            capi.check(lib.n2d2hip_sgd_update_f32_batch(ai, len(items), st))
        torch.cuda.synchronize()
        return [t.cpu().numpy() for t in out]
    for a, b in zip(run(False), run(True)):
        assert np.array_equal(a, b)
    bad = capi.SatWeightGradItem(None, None, None, 1, 15.0, 1, 0, None)
    w = torch.zeros(1, device="cuda")
    item = capi.SgdItem(w.data_ptr(), w.data_ptr(), 1, None, 0.01, 0.0, 0.0, 0.0, 0.0, 0)
    assert lib.n2d2hip_sgd_update_f32_batch_sat((capi.SgdItem * 1)(item), 1, (capi.SatWeightGradItem * 1)(bad), 1, st) == capi.ERR_INVALID
