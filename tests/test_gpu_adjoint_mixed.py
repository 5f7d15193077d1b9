"""Gradients of batches in which some slices share a geometry and others do
not: every task of the adjoint's launch has its own width (1, 2, 4 or 8
slices), so its bits are those of single slices, and slices without a partner
cost what they do in a batch of different ones."""
import numpy as np
import pytest

from acumen_amd import Batch, _lib, synth

pytestmark = pytest.mark.gpu


def make(ctx, shapes):
    return Batch(ctx, [(N, T, synth.default_wpu(N), synth.angles(T) + np.float32(0.5 * k)) for N, T, k in shapes])


def run(ctx, shapes, xs, fs):
    with make(ctx, shapes) as b:
        for i, f in enumerate(fs):
            b.set_sino(i, f)
        return b.loss_grad(xs)[1]


CASES = {
    "widths 8, 4, 2 and 1": [(193, 9, 0)] * 8 + [(225, 9, 0), (225, 9, 1)] * 3 + [(225, 9, 2), (97, 9, 0), (225, 9, 2)],
    "5 and 6 different": [(209, 17, k) for k in (0, 1, 0, 2, 0, 3, 4, 0, 5, 0, 6)],
    "9, and one of another size": [(209, 8, 0)] * 9 + [(33, 200, 0)],
    "7 of few tiles": [(33, 33, 0)] * 7 + [(48, 7, 1)] * 2 + [(17, 64, 0)],
}


@pytest.mark.parametrize("name", CASES)
def test_mixed_widths_equal_single_slices(ctx, name):
    shapes = CASES[name]
    print("[case] adjoint mixed", name, flush=True)
    rng = np.random.default_rng(23)
    xs = [rng.random((N, N), dtype=np.float32) for N, _, _ in shapes]
    fs = [rng.random((T, N), dtype=np.float32) for N, T, _ in shapes]
    got = run(ctx, shapes, xs, fs)
    for i in range(len(shapes)):
        assert np.array_equal(got[i], run(ctx, shapes[i:i + 1], xs[i:i + 1], fs[i:i + 1])[0]), i


def test_single_slices_beside_a_group_keep_their_time(ctx):
    """The adjoint of 5 equal and 20 different slices takes no longer than of
    25 different ones."""
    print("[case] adjoint mixed, time", flush=True)
    ms = []
    for shapes in ([(513, 120, k) for k in range(25)], [(513, 120, 0)] * 5 + [(513, 120, k) for k in range(1, 21)]):
        xs = [np.zeros((N, N), np.float32) for N, _, _ in shapes]
        with make(ctx, shapes) as b:
            best = np.inf
            for _ in range(5):
                ctx.set_timing(True)
                b.loss_grad(xs, grad_s=False)
                best = min(best, ctx.kernel_time(_lib.KIND_ADJ)[0])
            ctx.set_timing(False)
            ms.append(best)
    print("ms:", ms, flush=True)
    assert ms[1] < 1.05 * ms[0]
