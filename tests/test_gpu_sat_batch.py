"""The SAT weight quantizers of many tensors in one call: what one call for each tensor gives, bit for bit, at the sizes where a
tensor changes from one block of 1, 4, 8, 12 or 16 values a thread to many blocks, and past one launch's 16 tensors."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 1023, 1024, 1025, 4096, 4097, 16384, 16385, 16400, 70001, 300000, 5, 9, 333, 20000, 64, 17000]
MORE = [12288, 8192, 8193, 12289]          # (the first of them, the 19th tensor, is compared with the formula)


@pytest.mark.parametrize("count", [1, 3, 16, 18, 22])
def test_batch_equals_single_calls(count):
    import torch
    from n2d2_amd import capi, runtime as rt
    print("sat batch", count, flush=True)
    lib, rng = capi.lib, np.random.default_rng(count)
    sizes = SIZES[-count:] if count < 16 else (SIZES + MORE)[:count]
    ws = int(lib.n2d2hip_quantizer_workspace_bytes(max(sizes)))
    dev = lambda a: torch.from_numpy(a.astype(np.float32)).cuda()
    items, grads, one, keep = [], [], [], []
    for k, n in enumerate(sizes):
        w, dq = dev(rng.normal(0, 0.6, n)), dev(rng.normal(0, 1, n))
        wq, wq1, dw, dw1 = (torch.full((n,), 7.0, device="cuda") for _ in range(4))
        st, st1, space = torch.zeros(2, device="cuda"), torch.zeros(2, device="cuda"), torch.empty(ws, dtype=torch.uint8, device="cuda")
        mode, rng_, scale = k % 6, float([15, 255, 3][k % 3]), int(n > 1 and k % 2)
        items.append(capi.SatWeightItem(w.data_ptr(), wq.data_ptr(), n, rng_, mode, scale, 10 + k, st.data_ptr(), space.data_ptr(), ws))
        grads.append(capi.SatWeightGradItem(dq.data_ptr(), w.data_ptr(), dw.data_ptr(), n, rng_, mode, scale, st.data_ptr()))
        capi.check(lib.n2d2hip_sat_weight_forward(w.data_ptr(), wq1.data_ptr(), n, rng_, mode, scale, 10 + k, st1.data_ptr(), space.data_ptr(), ws,
                                                  rt.stream_ptr()))
        capi.check(lib.n2d2hip_sat_weight_backward(dq.data_ptr(), w.data_ptr(), dw1.data_ptr(), n, rng_, mode, scale, st1.data_ptr(), rt.stream_ptr()))
        one.append((wq, wq1, dw, dw1, st, st1))
        keep += [w, dq, space]
        # and against the formula in 64 bits (mode 0: tanh(w) / max |tanh(w)|): tanhf is good to 2 ulp, the quotient to half of one
        if mode == 0 and not scale:
            t = np.tanh(w.cpu().numpy().astype(np.float64))
            assert np.max(np.abs(wq1.cpu().numpy() - t / np.abs(t).max())) < 5 * 2.0 ** -24 * 2
    capi.check(lib.n2d2hip_sat_weight_forward_batch((capi.SatWeightItem * count)(*items), count, rt.stream_ptr()))
    capi.check(lib.n2d2hip_sat_weight_backward_batch((capi.SatWeightGradItem * count)(*grads), count, rt.stream_ptr()))
    torch.cuda.synchronize()
    for n, (wq, wq1, dw, dw1, st, st1) in zip(sizes, one):
        for a, b in ((wq, wq1), (dw, dw1), (st, st1)):
            assert torch.equal(a, b) and bool(torch.isfinite(a).all()), n


def test_batch_refuses_what_a_single_call_refuses():
    import torch
    from n2d2_amd import capi
    lib = capi.lib
    w, out, st, ws = torch.ones(8, device="cuda"), torch.empty(8, device="cuda"), torch.empty(2, device="cuda"), torch.empty(1 << 14, device="cuda")
    good = dict(w=w.data_ptr(), wq=out.data_ptr(), n=8, range=15.0, mode=1, apply_scaling=0, outputs_size=1, stats=st.data_ptr(), workspace=ws.data_ptr(),
                workspace_bytes=1 << 16)
    call = lambda **kw: lib.n2d2hip_sat_weight_forward_batch((capi.SatWeightItem * 2)(capi.SatWeightItem(**good), capi.SatWeightItem(**{**good, **kw})), 2, None)
    assert call(n=0) and call(w=None) and call(mode=9) and call(range=0.5) and call(workspace_bytes=8) and call(n=1, apply_scaling=1)
    assert lib.n2d2hip_sat_weight_forward_batch((capi.SatWeightItem * 1)(capi.SatWeightItem(**good)), 0, None)


@pytest.mark.parametrize("n", [16385, 262143, 262145, 2097153, 4194307])
def test_many_weights_fill_the_chip_and_equal_the_formula(n):
    """Tensors of many blocks, whose runs of 256 are dealt out by eights: every weight once, and the pass that writes them has as
    many threads as the chip holds (2048 a compute unit) as soon as there are as many weights."""
    import torch
    from n2d2_amd import capi, runtime as rt
    print("sat many", n, flush=True)
    ws = torch.empty(int(capi.lib.n2d2hip_quantizer_workspace_bytes(n)), dtype=torch.uint8, device="cuda")
    stats = torch.zeros(2, device="cuda")
    w = torch.from_numpy(np.random.default_rng(n).normal(0, 0.4, n).astype(np.float32)).cuda()
    for place in (0, n - 1, (n // 256 - 1) * 256 + 255, min(n - 1, 8 * 256 * 3 + 5)):          # the largest weight at either end and inside
        x = w.clone()
        x[place] = 2.5
        out = torch.full_like(x, 7.0)
        with capi.launch_log() as log:
            capi.check(capi.lib.n2d2hip_sat_weight_forward(x.data_ptr(), out.data_ptr(), n, 15.0, 0, 0, 1, stats.data_ptr(), ws.data_ptr(), ws.numel(),
                                                           rt.stream_ptr()))
        t = torch.tanh(x.double())
        assert abs(float(stats[0]) - float(np.tanh(2.5))) < 2.0 ** -23
        assert float((out.double() - t / t.abs().max()).abs().max()) < 5 * 2.0 ** -24 * 2         # (tanhf 2 ulp, the quotient half of one)
        (first, second) = log.entries
        cus = torch.cuda.get_device_properties(0).multi_processor_count
        assert first[0].startswith("sat_weight_first_kernel") and second[1] * second[2] >= min(n, 2048 * cus)
