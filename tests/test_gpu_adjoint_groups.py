"""Gradients of slices of one geometry, which the adjoint takes 2, 4 or 8 to a
workgroup, against batches of one slice: the same arithmetic, the same bits.

Group sizes with full and partly filled tasks, geometries in turn, both sides
of the line between 4 and 8 together (2048 tiles of 16 x 16), and a slice with
an infinity beside finite ones.
"""
import numpy as np
import pytest

from acumen_amd import Batch, synth

pytestmark = pytest.mark.gpu


def run(ctx, shapes, xs, fs):
    with Batch(ctx, [(N, T, synth.default_wpu(N), synth.angles(T) + np.float32(0.5 * k)) for N, T, k in shapes]) as b:
        for i, f in enumerate(fs):
            b.set_sino(i, f)
        return b.loss_grad(xs)


def data(shapes):
    rng = np.random.default_rng(17)
    return ([rng.random((N, N), dtype=np.float32) for N, _, _ in shapes],
            [rng.random((T, N), dtype=np.float32) for N, T, _ in shapes])


CASES = {
    "2": [(33, 17, 0)] * 2,
    "3": [(48, 33, 0)] * 3,
    "9, small": [(65, 31, 0)] * 9,
    "two geometries in turn": [(65, 40, i % 2) for i in range(7)],
    "sizes mixed": [(65, 40, 0), (33, 40, 0), (65, 40, 0), (65, 41, 0), (33, 40, 0), (65, 40, 0), (16, 5, 0)],
    "8 together": [(257, 33, 0)] * 8,
    "8 and 3": [(225, 9, 0)] * 11,
}


@pytest.mark.parametrize("name", CASES)
def test_groups_equal_single_slices(ctx, name):
    shapes = CASES[name]
    print("[case] adjoint groups", name, flush=True)
    xs, fs = data(shapes)
    got = run(ctx, shapes, xs, fs)
    for i in range(len(shapes)):
        want = run(ctx, shapes[i:i + 1], xs[i:i + 1], fs[i:i + 1])
        assert np.array_equal(got[1][i], want[1][0]), i


def test_infinity_stays_in_its_slice(ctx):
    shapes = [(65, 40, 0)] * 3
    print("[case] adjoint groups, infinity", flush=True)
    xs, fs = data(shapes)
    fs[1][7, 30] = np.inf
    got = run(ctx, shapes, xs, fs)
    for i in (0, 1, 2):
        want = run(ctx, shapes[i:i + 1], xs[i:i + 1], fs[i:i + 1])
        assert np.array_equal(got[1][i], want[1][0], equal_nan=True), i
        assert np.isfinite(got[1][i]).all() == (i != 1)
