"""The FP64 ramp filter by FFT on rows that are not ordinary: mixtures of
infinities and NaN against the plain FP64 sum, one or a few values that
dominate the row, the time that infinities cost, and batches with slices past
its length limit."""
import numpy as np
import pytest

from acumen_amd import ACU_IMG_FBP, Batch, _lib, synth
from helpers import HipBuffers

pytestmark = pytest.mark.gpu


def taps(N):
    """The reference's FP32 taps at distances -(N-1)..N-1 (tv_hpc.F90:53-56), one rounding per operation."""
    k = np.arange(-(N - 1), N)
    q = (4 * k * k - 1).astype(np.float32)
    pi = np.float32(np.pi)
    return np.float32(-(2.0 * N)) / ((pi * pi) * q)


def product(s):
    """The filter as the plain sum in FP64, unrounded."""
    T, N = s.shape
    h = taps(N).astype(np.float64)
    i = np.arange(N)
    with np.errstate(invalid="ignore"):
        return np.array([[np.sum(h[d - i + N - 1] * row) for d in i] for row in s.astype(np.float64)])


def ramp(ctx, s, reps=0):
    T, N = s.shape
    hb = HipBuffers()
    try:
        with Batch(ctx, [(N, T, 1, synth.angles(T))]) as b:
            d_s, d_o = hb.upload(s), hb.alloc(s.nbytes)
            b.ramp_dev(0, d_o, d_s)
            ctx.synchronize()
            if not reps:
                return hb.download(d_o, (T, N))
            best = np.inf
            for _ in range(reps):
                ctx.set_timing(True)
                b.ramp_dev(0, d_o, d_s)
                best = min(best, ctx.kernel_time(_lib.KIND_RAMP)[0])
            ctx.set_timing(False)
            return best
    finally:
        hb.close()


# threads per row 1, 2, 8, 16, 64 and 256: below a wave, one wave, several
@pytest.mark.parametrize("N", [4, 9, 17, 65, 130, 513, 2049])
def test_infinities_and_nan_together(ctx, N):
    print("[case] ramp rows, infinities", N, flush=True)
    rng = np.random.default_rng(N)
    inf, nan = np.inf, np.nan
    rows = [{0: inf}, {N - 1: -inf}, {N // 2: inf, 1: inf}, {0: -inf, N - 1: -inf}, {1: inf, N - 2: -inf},
            {0: inf, N // 2: -inf, N - 1: inf}, {N // 2: nan, 0: inf}, {N - 1: -nan}, {}]
    s = rng.normal(size=(len(rows) + 3, N)).astype(np.float32)
    for t, r in enumerate(rows):
        for j, v in r.items():
            s[t, j] = v
    s[-3] = inf
    s[-2] = np.where(rng.random(N) < 0.5, inf, -inf)
    s[-1] = 3e38  # finite, past FP32 in the result
    with np.errstate(over="ignore"):
        want = product(s).astype(np.float32)
    got = ramp(ctx, s)
    for t in range(len(s)):
        if not np.isfinite(s[t]).all():
            assert np.array_equal(got[t], want[t], equal_nan=True), t
    assert np.array_equal(np.isposinf(got[-1]), np.isposinf(want[-1]))


@pytest.mark.parametrize("N", [33, 1025, 4097])
def test_rows_with_dominating_values(ctx, N):
    """Every output within its own FP32 rounding (2^-24) of the product, and
    an FFT's error: 2^-53 of the root mean square of the row's outputs per
    rounding, of which 13 levels each way add up to 16 at five deviations."""
    print("[case] ramp rows, dominating values", N, flush=True)
    rng = np.random.default_rng(N)
    s = rng.random((4, N), dtype=np.float32)
    s[0, N // 3] = 1e6
    s[1, 0] = 1e12
    s[2, N - 1], s[2, N // 2] = 1e9, 1e4
    s[3, : N // 4] *= 1e8
    want = product(s)
    got = ramp(ctx, s).astype(np.float64)
    rms = np.sqrt(np.mean(want ** 2, axis=1, keepdims=True))
    bound = 2.0 ** -24 * np.abs(want) + 16 * 2.0 ** -53 * rms
    print("worst, in units of the bound:", np.max(np.abs(got - want) / bound, axis=1), flush=True)
    assert (np.abs(got - want) <= bound).all()


def test_infinities_cost_no_plain_sum(ctx):
    """A dead detector column (an infinity in every row) takes no more than a
    few times the finite rows' time."""
    print("[case] ramp rows, time", flush=True)
    s = np.random.default_rng(1).random((1500, 2049), dtype=np.float32)
    finite = ramp(ctx, s, 5)
    s[:, 700] = np.inf
    column = ramp(ctx, s, 5)
    print("ms:", finite, column, flush=True)
    assert column < 4 * finite


def fbp_images(ctx, spec, fs):
    with Batch(ctx, spec) as b:
        for i, f in enumerate(fs):
            b.set_sino(i, f)
        best = np.inf
        for _ in range(4):
            ctx.set_timing(True)
            b.fbp()
            best = min(best, ctx.kernel_time(_lib.KIND_RAMP)[0])
        ctx.set_timing(False)
        return [b.get_image(i, ACU_IMG_FBP) for i in range(len(fs))], best


def test_slices_past_the_fft_limit_share_a_launch(ctx):
    """Slices of N > 4097 (the FP64 matrix product) between slices within the
    limit equal single plans, and six of few angles take one launch's time: 71
    workgroups each, where the GPU runs several hundred at once."""
    print("[case] ramp past the FFT limit", flush=True)
    sizes = [(4099, 3), (65, 20), (4098, 70), (4500, 16), (33, 1), (4099, 3)]
    fs = [np.random.default_rng(i).random((T, N), np.float32) for i, (N, T) in enumerate(sizes)]
    spec = [(N, T, 4, synth.angles(T)) for N, T in sizes]
    got, _ = fbp_images(ctx, spec, fs)
    for i, f in enumerate(fs):
        want, _ = fbp_images(ctx, spec[i:i + 1], [f])
        assert np.array_equal(got[i], want[0]), i
    _, one = fbp_images(ctx, spec[3:4], fs[3:4])
    _, six = fbp_images(ctx, spec[3:4] * 6, fs[3:4] * 6)
    print("ms:", one, six, flush=True)
    assert six < 3 * one
