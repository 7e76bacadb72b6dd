"""The first cells of a small network in one launch (n2d2hip_cell_run_*): every tensor against the cells launched one by one,
the outputs against the CPU oracle.  Integers: bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# name, input shape, input unsigned, rescale mode, cells: ("conv", outputs, kernel, stride, pad) / ("pool", kernel, stride, pad) / ("fc", outputs)
NETS = [
    ("lenet_like", (1, 28, 28), True, "FixedMult32", [("conv", 6, 5, 1, 0), ("pool", 2, 2, 0), ("conv", 16, 5, 1, 0), ("pool", 2, 2, 0),
                                                     ("fc", 120), ("fc", 84), ("fc", 10)]),
    # padded windows, 32 outputs (two blocks), overlapping padded pooling, sizes that fill no tile, signed input
    ("padded", (3, 13, 11), False, "SingleShift", [("conv", 16, 4, 2, 1), ("conv", 32, 3, 1, 1), ("pool", 3, 2, 1), ("fc", 128), ("fc", 7)]),
    # one pixel left, four channels all the way (channel stride 4), 8 x 8 kernel of 64 taps, float rescale
    ("four_channels", (4, 17, 19), True, "FloatMult", [("conv", 4, 8, 1, 0), ("conv", 3, 7, 3, 3), ("pool", 4, 4, 0), ("conv", 9, 1, 1, 0)]),
    # 16 input channels, the largest K, no fully-connected cell
    ("wide", (16, 9, 21), True, "DoubleShift", [("conv", 16, 7, 2, 3), ("conv", 17, 2, 1, 0), ("pool", 2, 1, 0)]),
    # a first fully-connected cell of 1024 inputs
    ("long_vector", (2, 10, 10), False, "FixedMult16", [("conv", 16, 3, 1, 0), ("pool", 1, 1, 0), ("conv", 16, 1, 1, 0), ("fc", 100), ("fc", 33)]),
]


@pytest.mark.parametrize("batch", [1, 3, 261])
@pytest.mark.parametrize("case", NETS, ids=[c[0] for c in NETS])
def test_cells_in_one_launch_bit_exact(case, batch):
    from n2d2_amd import capi, nets
    from oracle import cells
    name, shape, unsigned, mode, plan = case
    b = nets._Builder(name, shape, 5, mode, unsigned_data=unsigned)
    b.spec.input_unsigned = unsigned
    b.spec.unsigned["input"] = unsigned
    x = "input"
    for k, c in enumerate(plan):
        if c[0] == "conv":
            x = b.conv("c%d" % k, x, c[1], c[2], c[3], c[4])
        elif c[0] == "pool":
            x = b.pool("p%d" % k, x, "max", c[1], c[2], c[3])
        else:
            last = k + 1 == len(plan)
            x = b.fc("f%d" % k, x, c[1], kind="Linear" if last else "Rectifier", **({"mode": "None"} if last else {}))
    lo, hi = (0, 256) if unsigned else (-128, 128)
    img = np.random.default_rng(batch).integers(lo, hi, size=(batch,) + shape)
    print(name, batch, flush=True)
    run = nets.GpuNet(b.spec, batch)
    apart = nets.GpuNet(b.spec, batch, cell_runs=False)
    assert run.cell_run is not None and run._run_steps == len(run.steps)
    for net in (run, apart):
        net.set_input(img)
    with capi.launch_log() as log:
        run.forward()
    assert [e[0] for e in log.entries] and all("cell_run_kernel" in e[0] for e in log.entries) and len(log.entries) == 1
    apart.forward()
    for n, t in apart.tensors.items():
        used = t.cs if t.dtype != capi.I32 else t.C         # (channels past the last one: the stored 0, but not behind integers)
        a, b2 = (net.tensors[n].buf.cpu().numpy().reshape(-1, t.cs)[:, :used] for net in (run, apart))
        assert np.array_equal(a, b2), n
    got = run.tensors[b.spec.output].to_numpy()
    want = cells.run_net(b.spec, img[:3])[b.spec.output].astype(np.int64)
    assert np.array_equal(got[:3], want)
    # from the byte planes, replayed (from a graph where the conversion is a launch of its own) with other work between the replays
    edge_in_launch = run.cell_run.takes_edge(run.input_src)
    assert edge_in_launch == (shape[0] <= 4)
    replay = run.capture(1, with_input_conversion=True)
    for _ in range(3):
        for n in run.tensors:
            run.tensors[n].buf.fill_(7)
        assert np.array_equal(replay().to_numpy(), got)
        assert np.array_equal(run.input.buf.cpu().numpy(), apart.input.buf.cpu().numpy())


# Pairs of pixels a column of the matrix instruction: convolutions of 4 channels to at most 8 outputs, unpadded, rows of even length in and out
PAIRS = [
    # one tile and one pair behind it (17 pairs), 8 outputs, stride 1; then the same from a row of its own (1 x 2 pixels)
    ("eight_of_five", (4, 5, 38), True, "FixedMult32", [("conv", 8, 5, 1, 0), ("conv", 4, 1, 1, 0), ("conv", 3, 1, 1, 0)]),
    # three outputs (a channel stride of 4), float rescale, four K steps; a pair alone
    ("three_of_seven", (1, 7, 8), False, "FloatMult", [("conv", 3, 7, 1, 0), ("conv", 5, 1, 1, 0), ("fc", 12), ("fc", 6)]),
    # strides 2 and 3, 64-bit rescale; more tiles than two a wave
    ("stride_two", (3, 40, 42), True, "DoubleShift", [("conv", 4, 4, 2, 0), ("pool", 2, 2, 0), ("conv", 5, 3, 1, 0)]),
    ("stride_three", (2, 32, 50), True, "FixedMult16", [("conv", 6, 5, 3, 0), ("pool", 2, 2, 0), ("fc", 12), ("fc", 9)]),
    ("last_pair_of_two", (1, 37, 34), True, "SingleShift", [("conv", 6, 3, 1, 0), ("pool", 2, 2, 0), ("conv", 16, 3, 1, 0)]),
]


@pytest.mark.parametrize("batch", [1, 3])
@pytest.mark.parametrize("case", PAIRS, ids=[c[0] for c in PAIRS])
def test_pairs_of_pixels_bit_exact(case, batch):
    test_cells_in_one_launch_bit_exact(case, batch)


def test_run_is_planned_up_to_sixteen_images_a_compute_unit():
    import torch
    from n2d2_amd import nets, runtime as rt
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    spec = nets.lenet()
    assert nets.GpuNet(spec, 16 * cus).cell_run is not None and nets.GpuNet(spec, 16 * cus + 1).cell_run is None
    assert rt.CellRun.pays(1) and not rt.CellRun.pays(0)


def test_captured_forward_of_a_single_launch_is_that_launch():
    """One forward of a network that is one launch is replayed as the launch itself, two as a graph; both on the stream that is
    current at the call."""
    import torch
    from n2d2_amd import capi, nets
    net = nets.GpuNet(nets.lenet(), 2)
    net.set_input(np.random.default_rng(5).integers(0, 256, size=(2, 1, 32, 32)))
    want = net.forward().to_numpy()
    side = torch.cuda.Stream()
    for replay, launches in ((net.capture(), 1), (net.capture(1, with_input_conversion=True), 1), (net.capture(2), 0)):
        for stream in (torch.cuda.current_stream(), side):
            net.tensors[net.spec.output].buf.fill_(7)
            torch.cuda.synchronize()
            with torch.cuda.stream(stream), capi.launch_log() as log:
                replay()
            torch.cuda.synchronize()
            assert len(log.entries) == launches
            assert np.array_equal(net.tensors[net.spec.output].to_numpy(), want)


@pytest.mark.parametrize("shape", [(1, 1, 2, 2), (3, 1, 32, 32), (5, 3, 7, 4), (2, 4, 6, 10), (2, 2, 5, 5), (513, 3, 33, 36)])
@pytest.mark.parametrize("src,dst", [("U8", "U8B"), ("U8", "U8"), ("I8", "I8"), ("U8", "I8"), ("I8", "U8B")])
def test_byte_planes_to_pixels_of_four_channels(shape, src, dst):
    """The graph edge's conversion: every stored byte, from aligned planes, and from planes that begin at an odd address."""
    import torch
    from n2d2_amd import capi, runtime as rt
    B, C, H, W = shape
    x = np.random.default_rng(7).integers(*((0, 256) if src == "U8" else (-128, 128)), size=shape)
    lo, hi, off = {"U8B": (0, 255, -128), "U8": (0, 255, 0), "I8": (-128, 127, 0)}[dst]
    want = np.zeros((B, H, W, 4), np.int64)
    want[..., :C] = np.clip(x, lo, hi).transpose(0, 2, 3, 1)
    want = (want + off).astype(np.uint8).reshape(-1)
    flat = torch.from_numpy(x.astype(np.uint8 if src == "U8" else np.int8).reshape(-1))
    for shift in (0, 1):
        buf = torch.zeros(flat.numel() + 16, dtype=flat.dtype, device="cuda")[shift:shift + flat.numel()]
        buf.copy_(flat)
        t = rt.DTensor(B, C, H, W, getattr(capi, src), capi.NCHW, buf)
        out = rt.DTensor(B, C, H, W, getattr(capi, dst)).convert_from(t)
        assert np.array_equal(out.buf.cpu().numpy().view(np.uint8).reshape(-1), want), shift
