"""Backprojection launches in which some slices are in pairs and others not, of
few tiles and of many, with slices that differ in their window (wpu) alone:
the bits of plans of one slice.  And a few pairs of long chains among single
slices cost no launch of their own."""
import numpy as np
import pytest

from acumen_amd import ACU_IMG_FBP, Batch, _lib, synth

pytestmark = pytest.mark.gpu


def spec(shapes):
    return [(N, T, synth.default_wpu(N) + w, synth.angles(T) + np.float32(0.25 * k)) for N, T, k, w in shapes]


def images(ctx, shapes, fs, ty):
    with Batch(ctx, spec(shapes)) as b:
        b.set_bp_tile(ty)
        for i, f in enumerate(fs):
            b.set_sino(i, f)
        b.fbp()
        return [b.get_image(i, ACU_IMG_FBP) for i in range(len(fs))]


# (N, T, k, w): k shifts the angles, w widens the window; each in 64 x 8 tiles
CASES = {
    "2720, pairs": [(257, 33, 0, 0)] * 16,
    "2040, too few": [(257, 33, 0, 0)] * 12,
    "3566, one window apart": [(513, 17, 0, 0)] * 5 + [(513, 17, 0, 9)],
    "windows in turn": [(513, 16, 0, i % 2) for i in range(10)],
    "pairs around single slices": [(513, 47, 0, 0), (300, 20, 1, 0), (513, 47, 0, 0), (65, 100, 2, 0), (513, 47, 0, 0),
                                   (129, 31, 3, 0), (513, 47, 0, 0), (513, 47, 0, 0)],
    "a quarter in pairs": [(513, 20, 0, 0)] * 2 + [(513, 20, k, 0) for k in range(1, 7)],
    "one tile more than the GPU holds at once": [(1025, 8, 0, 0)] * 6 + [(65, 9, 0, 0)],
}


@pytest.mark.parametrize("ty", [16, 32, 64])
@pytest.mark.parametrize("name", CASES)
def test_mixed_launches_equal_single_plans(ctx, name, ty):
    shapes = CASES[name]
    print("[case] bp mixed", name, ty, flush=True)
    rng = np.random.default_rng(9)
    fs = [rng.random((T, N), dtype=np.float32) for N, T, _, _ in shapes]
    got = images(ctx, shapes, fs, ty)
    for i in range(len(fs)):
        assert np.array_equal(got[i], images(ctx, shapes[i:i + 1], fs[i:i + 1], ty)[0]), i


def test_a_pair_of_long_chains_waits_for_nobody(ctx):
    """Two slices of 65^2 x 1500 beside three of 2049^2 x 300 take about the
    same time whether they are of one geometry or not."""
    print("[case] bp mixed, time", flush=True)
    ms = []
    for k in (0, 1):
        shapes = [(65, 1500, 0, 0), (65, 1500, k, 0)] + [(2049, 300, j, 0) for j in range(3)]
        with Batch(ctx, spec(shapes)) as b:
            best = np.inf
            for _ in range(5):
                ctx.set_timing(True)
                b.fbp()
                best = min(best, ctx.kernel_time(_lib.KIND_BP)[0])
            ctx.set_timing(False)
            ms.append(best)
    print("ms:", ms, flush=True)
    assert ms[0] < 1.4 * ms[1]
