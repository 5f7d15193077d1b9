"""The TV solver's sums inside the kernels that use them, against the launches
of their own that the per-slice mode makes: the order of summation is the same,
so every result is the same bits.

Sides: one block of 1024 elements, one element more, one row more, and both
sides of the largest slice whose sums are added in place (640 blocks: 809^2
has 640, 810^2 has 641).
"""
import numpy as np
import pytest

from acumen_amd import ACU_IMG_TV, ACU_TV_BATCHED, ACU_TV_GRAPH, ACU_TV_PLAIN, Batch, _lib, synth

pytestmark = pytest.mark.gpu


def sinos(shapes):
    rng = np.random.default_rng(3)
    return [rng.random((T, N), dtype=np.float32) for N, T in shapes]


def run(ctx, shapes, fs, sched, mode, ninner, ncg):
    with Batch(ctx, [(N, T, synth.default_wpu(N), synth.angles(T)) for N, T in shapes]) as b:
        b.set_tv_schedule(sched)
        for i, f in enumerate(fs):
            b.set_sino(i, f)
        b.tvopt(0.05, 0.1, 3, ninner, ncg, mode)
        return [b.get_image(i, ACU_IMG_TV) for i in range(len(fs))] + [b.get_delta(i, 3) for i in range(len(fs))]


@pytest.mark.parametrize("sched", [_lib.ACU_TV_SCHED_REFERENCE, _lib.ACU_TV_SCHED_LINEAR])
@pytest.mark.parametrize("ninner,ncg", [(0, 3), (1, 0), (1, 1), (2, 3)])
@pytest.mark.parametrize("shapes", [((31, 9),), ((33, 40),), ((809, 6),), ((810, 6),), ((33, 7), (65, 48)),
                                    ((65, 20), (810, 6))])
def test_sums_in_place_equal_launched_sums(ctx, shapes, ninner, ncg, sched):
    print("[case] tv sums", shapes, ninner, ncg, sched, flush=True)
    fs = sinos(shapes)
    want = run(ctx, shapes, fs, sched, ACU_TV_PLAIN, ninner, ncg)
    for mode in (ACU_TV_BATCHED, ACU_TV_GRAPH):
        got = run(ctx, shapes, fs, sched, mode, ninner, ncg)
        for a, b in zip(got, want):
            assert np.isfinite(a).all()
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
