"""The FP64 ramp filter by FFT (every slice up to N = 4097): sizes around its
passes and its packing of rows into workgroups, rows that hold infinities or
NaN, and batches on both sides of its length limit."""
import numpy as np
import pytest

from acumen_amd import ACU_IMG_FBP, Batch, synth
from helpers import HipBuffers, rel
from oracle import ref

pytestmark = pytest.mark.gpu


def ramp(ctx, s):
    T, N = s.shape
    hb = HipBuffers()
    try:
        with Batch(ctx, [(N, T, 1, synth.angles(T))]) as b:
            d_s, d_o = hb.upload(s), hb.alloc(s.nbytes)
            b.ramp_dev(0, d_o, d_s)
            ctx.synchronize()
            return hb.download(d_o, (T, N))
    finally:
        hb.close()


# L = 4 and 8 (plain sums), 16 and 32 (one radix-8 pass, tails of 1 and 2
# points), 64 (tail of 4), and both sides of powers of two; T leaves the last
# workgroup partly filled
@pytest.mark.parametrize("N,T", [(3, 2), (5, 3), (6, 65), (9, 64), (10, 33), (17, 31), (18, 1), (33, 17), (65, 9),
                                 (129, 5), (258, 3), (514, 2), (1026, 3), (2049, 2), (2050, 1), (4097, 2)])
def test_fp64_fft_ramp_sizes(ctx, N, T):
    # the reference's FP32 taps are 6e-8 off the oracle's and the result's
    # rounding 3e-8: 2e-7 leaves a factor of two over both
    s = np.random.default_rng(10 * N + T).normal(size=(T, N)).astype(np.float32)
    want = ref.ramp(s.astype(np.float64), "f64")
    assert rel(ramp(ctx, s), want) < 2e-7


@pytest.mark.parametrize("N,T", [(7, 70), (65, 20), (1025, 3)])
def test_fp64_fft_ramp_nonfinite_rows(ctx, N, T):
    """A row of the product with an infinity at j is -inf but for +inf at j
    (every tap but the middle one is negative), with a NaN all NaN; the other
    rows are what they were."""
    s = np.random.default_rng(N).normal(size=(T, N)).astype(np.float32)
    clean = ramp(ctx, s)
    j = N // 3
    s[1, j] = np.inf
    s[2, N - 1] = np.nan
    got = ramp(ctx, s)
    want = np.full(N, -np.inf, np.float32)
    want[j] = np.inf
    assert np.array_equal(got[1], want)
    assert np.isnan(got[2]).all()
    keep = np.setdiff1d(np.arange(T), [1, 2])
    assert np.array_equal(got[keep], clean[keep])


def test_batch_past_the_length_limit_equals_single_plans(ctx):
    sizes = [(65, 20), (4099, 3), (129, 7), (1025, 2)]
    f = [np.random.default_rng(i).random((T, N), np.float32) for i, (N, T) in enumerate(sizes)]
    spec = [(N, T, 4, synth.angles(T)) for N, T in sizes]
    with Batch(ctx, spec) as b:
        for i, x in enumerate(f):
            b.set_sino(i, x)
        b.fbp()
        got = [b.get_image(i, ACU_IMG_FBP) for i in range(len(sizes))]
    for i, x in enumerate(f):
        with Batch(ctx, [spec[i]]) as b:
            b.set_sino(0, x)
            b.fbp()
            assert np.array_equal(got[i], b.get_image(0, ACU_IMG_FBP)), i
