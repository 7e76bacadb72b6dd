"""Float convolutions on the bf16 matrix cores step by step of 32 products (conv_f32_taps_kernel): forward and data gradient against float64 in every
instance of the kernel, with infinities, NaN and the largest floats, and with workspaces that hold no partial results."""
import numpy as np
import pytest

from test_gpu_conv_parts import _inputs, _passes, _run

pytestmark = pytest.mark.gpu

# B, C, H, W, O, kH, kW, stride, pad; which result; the instance: waves along rows and pixels, 16 rows and 16 pixels of a wave, steps of one tap, sums in
# double.  Rows, pixels, channels and products left over, all residue classes of stride 2 (of 2 x 2, 1 x 1 and no taps), several ranges and one.
CASES = [((3, 16, 55, 115, 99, 5, 5, 1, 2), 1, "1, 4, 1, 2, false, false"), ((2, 129, 65, 112, 16, 5, 5, 1, 2), 0, "1, 4, 1, 2, false, false"),
         ((3, 16, 33, 63, 1149, 5, 5, 2, 2), 1, "1, 4, 1, 2, true, false"), ((2, 301, 35, 89, 16, 5, 5, 1, 2), 0, "1, 4, 1, 2, true, false"),
         ((3, 32, 51, 54, 133, 5, 5, 1, 0), 1, "1, 4, 2, 2, false, false"), ((1, 299, 32, 98, 32, 5, 5, 1, 2), 0, "1, 4, 2, 2, true, false"),
         ((1, 166, 17, 82, 131, 5, 5, 1, 2), 1, "2, 2, 2, 2, false, false"), ((33, 128, 27, 27, 256, 3, 3, 2, 1), 1, "2, 2, 2, 2, true, false"),
         ((5, 133, 25, 23, 133, 5, 5, 1, 0), 1, "2, 2, 2, 2, false, true"), ((1, 113, 49, 65, 130, 5, 5, 1, 0), 0, "2, 2, 2, 2, true, true"),
         ((1, 133, 9, 82, 1108, 5, 5, 2, 2), 0, "4, 1, 2, 4, false, false"), ((1, 453, 7, 33, 1045, 5, 5, 2, 2), 0, "4, 1, 2, 4, true, false"),
         ((23, 66, 60, 8, 102, 5, 5, 1, 0), 1, "4, 1, 2, 4, false, true"), ((15, 73, 9, 61, 108, 5, 5, 1, 0), 1, "4, 1, 2, 4, true, true"),
         ((11, 257, 33, 35, 300, 1, 1, 1, 0), 0, "2, 2, 2, 2, true, false"), ((47, 257, 33, 35, 300, 1, 1, 2, 0), 1, "2, 2, 2, 2, true, false")]


def _kernel(log, which):
    """The forward's (0) or the data gradient's (1): the launches of the two passes lay out weights first."""
    names = [e[0] for e in log.entries]
    start = [i for i, n in enumerate(names) if n.startswith("conv_f32_lay_taps_kernel")]
    kernels = [names[i + 1][len("conv_f32_taps_kernel<"):-1] for i in start]
    return kernels[-which] if kernels else None


@pytest.mark.parametrize("case,which,kernel", CASES, ids=str)
def test_against_float64(case, which, kernel):
    """A sum is rounded five times in 32 products, each time by 2.53e-8 of it in the root mean square; the i-th of L equal steps is sqrt(i / L) of
    the last; and no sum is off by a rounding a term."""
    from n2d2_amd import capi
    print("taps", case, which, flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 3)
    want, mag = _passes(x, w, dy, s, pad)[which], _passes(np.abs(x), np.abs(w), np.abs(dy), s, pad)[which]
    with capi.launch_log() as log:
        got = _run(x, w, dy, s, pad)[which]
    assert _kernel(log, which) == kernel
    k = w.shape[1 - which] * w.shape[2] * w.shape[3]
    assert (np.abs(got - want) <= 2.0 ** -24 * (np.abs(want) + (k + 4) * mag)).all()
    steps = -(-w.shape[1 - which] // 32) * w.shape[2] * w.shape[3]
    assert np.linalg.norm(got - want) <= 1.1 * 2.53e-8 * np.sqrt(1 + 5 * steps / 2) * np.linalg.norm(want)
    bias = rng.normal(size=w.shape[0]).astype(np.float32)
    more = _run(x, w, dy, s, pad, bias=bias, beta=0.5, start=3.0)[which] - np.float32(1.5)
    if which == 0:
        more = more - bias[None, :, None, None]
    assert np.abs(more - got).max() <= 2.0 ** -22 * (np.abs(got).max() + 5)
    # a workspace that holds the laid-out weights alone, half of it, and none: all of K
    for less in (4 * got.size + 16, lambda n: n // 2, lambda n: n):
        less_of_it = _run(x, w, dy, s, pad, less=less)[which]
        assert (np.abs(less_of_it - want) <= 2.0 ** -24 * (np.abs(want) + (k + 4) * mag)).all()


# Few rows, all of K in a block: sums in double
@pytest.mark.parametrize("case,which,kernel", [((2, 301, 35, 89, 16, 5, 5, 1, 2), 0, "1, 4, 1, 2, true, true"), ((2, 129, 65, 112, 16, 5, 5, 1, 2), 0, "1, 4, 1, 2, false, true"),
                                               ((1, 299, 32, 98, 32, 5, 5, 1, 2), 0, "1, 4, 2, 2, true, true"), ((3, 104, 31, 97, 32, 5, 5, 1, 2), 0, "1, 4, 2, 2, false, true")], ids=str)
def test_rows_of_16_and_32_in_one_range(case, which, kernel):
    from n2d2_amd import capi
    print("taps, one range", case, which, flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 3)
    want = _passes(x, w, dy, s, pad)[which]
    with capi.launch_log() as log:
        got = _run(x, w, dy, s, pad, less=4 * want.size + 16)[which]
    assert _kernel(log, which) == kernel
    steps = -(-w.shape[1 - which] // 32) * w.shape[2] * w.shape[3]
    assert np.linalg.norm(got - want) <= 1.1 * 2.53e-8 * np.sqrt(1 + 5 * steps / 2) * np.linalg.norm(want)


@pytest.mark.parametrize("case,which", [(c[0], c[1]) for c in CASES if c[2] in ("1, 4, 1, 2, false, false", "2, 2, 2, 2, true, false", "4, 1, 2, 4, true, true")], ids=str)
def test_infinities_nan_and_the_largest_floats(case, which):
    """An infinity gives infinities of the products' signs, NaN only against a zero or another infinity; a float that rounds to infinity in bf16 is finite."""
    print("taps, special values", case, which, flush=True)
    x, w, dy, s, pad, rng = _inputs(case, 4)
    big = np.float32(3.4e38)
    w *= np.float32(1e-3)
    w[np.abs(w) < 1e-5] = 1e-5
    w[3, 5, 0, 0] = 0.0
    t = dy if which else x
    flat = t.reshape(-1)
    flat[rng.permutation(flat.size)[:12]] = [np.inf, -np.inf, np.nan, big, -big, big, -big, big, np.inf, -big, 1e-42, -1e-42]
    clean = lambda a: np.where(np.isfinite(a), a, 0)        # noqa: E731
    got, want = _run(x, w, dy, s, pad)[which], _passes(x, w, dy, s, pad)[which]
    fin, mag = _passes(clean(x), w, clean(dy), s, pad)[which], _passes(np.abs(clean(x)), np.abs(w), np.abs(clean(dy)), s, pad)[which]
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got == np.inf, want == np.inf) and np.array_equal(got == -np.inf, want == -np.inf)
    ok = np.isfinite(want)
    assert (np.abs(got - fin)[ok] <= 2.0 ** -24 * (np.abs(fin) + (w.shape[1 - which] * w.shape[2] * w.shape[3] + 4) * mag)[ok]).all()
