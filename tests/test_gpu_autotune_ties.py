"""What the autotuner reports where candidates are one launch: the FFT ramp is
the FP64 ramp's within its size limit, and launches of few backprojection tiles
do not depend on the tile height.  And the tile height where it counts: batches
of more than 5200 tiles of 64 x 8, graph-replayed TV rebuilt at each height."""
import numpy as np
import pytest

from acumen_amd import ACU_IMG_FBP, ACU_IMG_TV, ACU_TV_GRAPH, ACU_TV_PLAIN, Batch, _lib, synth

pytestmark = pytest.mark.gpu


def batch(ctx, shapes):
    b = Batch(ctx, [(N, T, synth.default_wpu(N), synth.angles(T) + np.float32(0.25 * k)) for N, T, k in shapes])
    rng = np.random.default_rng(4)
    for i, (N, T, _) in enumerate(shapes):
        b.set_sino(i, rng.random((T, N), dtype=np.float32) / N)
    return b


# the split kernel, 16 rows, pairs at 16 rows
@pytest.mark.parametrize("shapes", [[(129, 100, 0)] * 2, [(257, 40, 0)] * 6, [(257, 40, 0)] * 24])
def test_one_launch_is_one_time(ctx, shapes):
    print("[case] autotune ties", shapes[0], len(shapes), flush=True)
    with batch(ctx, shapes) as b:
        b.fbp()
        before = [b.get_image(i, ACU_IMG_FBP) for i in range(len(shapes))]
        rep = b.autotune(reps=1)
        ms = rep["ramp"]["ms"]
        assert ms["fft"] == ms["fp64"] and rep["ramp"]["choice"] != "fft"
        assert b.ramp_variant() != _lib.RAMP_FFT
        assert len(set(rep["bp"]["ms"].values())) == 1
        assert b.bp_tile() == rep["bp"]["choice"]
        b.set_ramp_variant(_lib.RAMP_FP64)
        b.fbp()
        for i, v in enumerate(before):
            assert np.array_equal(b.get_image(i, ACU_IMG_FBP), v), i


def test_a_slice_past_the_fft_limit(ctx):
    print("[case] autotune past the FFT limit", flush=True)
    with batch(ctx, [(4099, 2, 0), (65, 20, 0)]) as b:
        rep = b.autotune(reps=1)
        assert set(rep["ramp"]["ms"]) == {"fp64", "fp32", "bf16x6"}
        assert len(set(rep["bp"]["ms"].values())) > 1  # 33670 tiles: the heights are launches of their own


# uneven slices (no pairs), and two in three in pairs
@pytest.mark.parametrize("shapes", [[(1025, 9, 0), (770, 20, 1), (1300, 5, 2)], [(1025, 17, 0)] * 4 + [(700, 33, 1)] * 2 + [(1030, 5, 2)]])
def test_heights_of_many_tiles_equal_single_plans(ctx, shapes):
    print("[case] heights of many tiles", shapes, flush=True)
    with batch(ctx, shapes) as b:
        for ty in (32, 64, 16):  # a graph captured at one height is rebuilt at the next
            b.set_bp_tile(ty)
            b.tvopt(0.05, 0.1, 2, 1, 2, ACU_TV_GRAPH)
            got = [b.get_image(i, ACU_IMG_TV) for i in range(len(shapes))]
            for i, (N, T, k) in enumerate(shapes):
                rng = np.random.default_rng(4)
                fs = [rng.random((t, n), dtype=np.float32) / n for n, t, _ in shapes]
                with Batch(ctx, [(N, T, synth.default_wpu(N), synth.angles(T) + np.float32(0.25 * k))]) as p:
                    p.set_sino(0, fs[i])
                    p.tvopt(0.05, 0.1, 2, 1, 2, ACU_TV_PLAIN)
                    assert np.array_equal(got[i], p.get_image(0, ACU_IMG_TV)), (ty, i)
