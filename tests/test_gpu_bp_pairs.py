"""Backprojection of slices of one geometry two to a workgroup, against plans
of one slice: the same arithmetic in the same order, so the same bits (the
sign of the zeros off the mask aside).

Launches are of more than 5200 tiles of 64 x 8, past those that smaller tiles
serve (and of more than 19000 where a slice has no partner), with odd counts,
geometries that alternate, and angle counts at the edges of the 16 angles staged at a time
and of the 32 summed as a block.
"""
import numpy as np
import pytest

from acumen_amd import ACU_IMG_FBP, ACU_IMG_TV, ACU_TV_GRAPH, Batch, _lib, synth

pytestmark = pytest.mark.gpu


def sinos(shapes):
    rng = np.random.default_rng(9)
    return [rng.random((T, N), dtype=np.float32) for N, T, _ in shapes]


def angles(T, k):
    return synth.angles(T) + np.float32(0.25 * k)


def single(ctx, N, T, k, f):
    with Batch(ctx, [(N, T, synth.default_wpu(N), angles(T, k))]) as p:
        p.set_sino(0, f)
        p.fbp()
        return p.get_image(0, ACU_IMG_FBP)


# (N, T, k): k shifts the angles, so slices of different k are not of one geometry
CASES = {
    "128, one block of 16 angles": [(128, 16, 0)] * 164,
    "65, 17 angles": [(65, 17, 0)] * 262,
    "257, 33 angles": [(257, 33, 0)] * 32,
    "257, two geometries in turn": [(257, 31, i % 2) for i in range(36)],
    "513, pairs and singles": [(513, 15, 0), (513, 15, 1), (513, 15, 0), (257, 47, 0), (513, 15, 2), (257, 47, 0),
                               (513, 48, 0), (513, 48, 3), (513, 48, 0), (2049, 9, 0), (2049, 9, 0), (2049, 1, 0)],
    "1025, 1 angle": [(1025, 1, 0)] * 4,
    "1026, 65 angles, odd count": [(1026, 65, 0)] * 9,
    "1025, too few tiles for an odd count": [(1025, 33, 0)] * 3,
    "257, few tiles": [(257, 33, 0)] * 5,
    "257, more than 64 angles, few tiles": [(257, 66, 0)] * 3,
}


@pytest.mark.parametrize("ty", [16, 32, 64])
@pytest.mark.parametrize("name", CASES)
def test_pairs_equal_single_plans(ctx, name, ty):
    shapes = CASES[name]
    print("[case] bp pairs", name, ty, flush=True)
    fs = sinos(shapes)
    with Batch(ctx, [(N, T, synth.default_wpu(N), angles(T, k)) for N, T, k in shapes]) as b:
        b.set_bp_tile(ty)
        for i, f in enumerate(fs):
            b.set_sino(i, f)
        b.fbp()
        got = [b.get_image(i, ACU_IMG_FBP) for i in range(len(fs))]
    for i in sorted(set(range(0, len(fs), max(1, len(fs) // 8))) | {len(fs) - 2, len(fs) - 1}):
        assert np.array_equal(got[i], single(ctx, *shapes[i], fs[i])), i


def test_new_angles_part_a_pair(ctx):
    shapes = [(513, 40, 0)] * 10
    fs = sinos(shapes)
    print("[case] bp pairs, new angles", flush=True)
    with Batch(ctx, [(N, T, synth.default_wpu(N), angles(T, k)) for N, T, k in shapes]) as b:
        for i, f in enumerate(fs):
            b.set_sino(i, f)
        b.tvopt(0.05, 0.1, 1, 1, 1, ACU_TV_GRAPH)
        for slots, k in (([1], 1), ([2, 5], 2), ([1], 0)):
            for i in slots:
                b.set_theta(i, angles(40, k))
                shapes[i] = (513, 40, k)
            b.tvopt(0.05, 0.1, 2, 1, 2, ACU_TV_GRAPH)
            for i, f in enumerate(fs):
                N, T, kk = shapes[i]
                with Batch(ctx, [(N, T, synth.default_wpu(N), angles(T, kk))]) as p:
                    p.set_sino(0, f)
                    p.tvopt(0.05, 0.1, 2, 1, 2, ACU_TV_GRAPH)
                    assert np.array_equal(b.get_image(i, ACU_IMG_FBP), p.get_image(0, ACU_IMG_FBP)), (k, i)
                    assert np.array_equal(b.get_image(i, ACU_IMG_TV), p.get_image(0, ACU_IMG_TV)), (k, i)


def test_tile_positions_keep_the_set_height(ctx):
    """Tile-relative positions round by the tile's height, so a small batch
    and a large one of the same slice agree at the height that is set."""
    N, T = 129, 40
    f = sinos([(N, T, 0)])[0]
    big = (1537, 1, synth.default_wpu(1537), synth.angles(1))
    print("[case] bp tile positions", flush=True)
    for ty in (16, 32):
        out = []
        for extra in ([], [big] * 2):
            with Batch(ctx, [(N, T, synth.default_wpu(N), synth.angles(T))] + extra) as b:
                b.set_bp_positions(_lib.ACU_BP_POS_TILE, _lib.ACU_BP_POS_TILE)
                b.set_bp_tile(ty)
                b.set_sino(0, f)
                b.fbp()
                out.append(b.get_image(0, ACU_IMG_FBP))
        assert np.array_equal(out[0], out[1])
