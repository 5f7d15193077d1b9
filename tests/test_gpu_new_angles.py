"""Changes of angles between launches over all slices: which slices share a
geometry is settled at the next launch, after any number of changes, of a new
tile height or of gradients in between, and the results are those of plans of
one slice."""
import numpy as np
import pytest

from acumen_amd import ACU_IMG_FBP, ACU_IMG_TV, ACU_TV_GRAPH, AcumenError, Batch, synth

pytestmark = pytest.mark.gpu

N, T, S = 257, 33, 24  # 4080 tiles of 64 x 8: pairs


def angles(k):
    return synth.angles(T) + np.float32(0.25 * k)


class Single:
    """Images and gradients of one slice at angles k, from plans of their own."""

    def __init__(self, ctx, fs, x):
        self.ctx, self.fs, self.x, self.seen = ctx, fs, x, {}

    def get(self, what, i, k):
        key = (what, i, k)
        if key not in self.seen:
            with Batch(self.ctx, [(N, T, synth.default_wpu(N), angles(k))]) as p:
                p.set_sino(0, self.fs[i])
                if what == "fbp":
                    p.fbp()
                    self.seen[key] = p.get_image(0, ACU_IMG_FBP)
                elif what == "tv":
                    p.tvopt(0.05, 0.1, 2, 1, 2, ACU_TV_GRAPH)
                    self.seen[key] = p.get_image(0, ACU_IMG_TV)
                else:
                    self.seen[key] = p.loss_grad([self.x])[1][0]
        return self.seen[key]


def test_launches_after_changes_of_angles(ctx):
    rng = np.random.default_rng(3)
    fs = [rng.random((T, N), dtype=np.float32) for _ in range(S)]
    x = rng.random((N, N), dtype=np.float32)
    one = Single(ctx, fs, x)
    look = (0, 1, 2, 7, S - 1)
    k = [0] * S
    with Batch(ctx, [(N, T, synth.default_wpu(N), angles(0))] * S) as b:
        def check(what):
            print("[case] new angles", what, k, flush=True)
            if what == "grad":
                got = b.loss_grad([x] * S)[1]
            elif what == "fbp":
                b.fbp()
                got = [b.get_image(i, ACU_IMG_FBP) for i in range(S)]
            else:
                b.tvopt(0.05, 0.1, 2, 1, 2, ACU_TV_GRAPH)
                got = [b.get_image(i, ACU_IMG_TV) for i in range(S)]
            for i in look:
                assert np.array_equal(got[i], one.get(what, i, k[i])), (what, i, k[i])

        def change(slots, v):
            for i in slots:
                k[i] = v
                b.set_theta(i, angles(v))

        for i, f in enumerate(fs):
            b.set_sino(i, f)
        check("fbp")
        change(range(S), 1)                # all, one by one: pairs part and join again
        check("fbp")
        change([1], 2)
        check("grad")                      # before any backprojection of the new pairs
        check("fbp")
        check("tv")
        change([0, 7], 2)
        b.set_bp_tile(64)                  # rebuilds the tasks while the pairs are unsettled
        check("tv")
        change(range(0, S, 2), 3)
        change(range(1, S, 2), 3)
        check("tv")
        change([0], 4)
        change([0], 3)                     # and back
        check("fbp")


def test_a_slice_without_angles_still_refuses(ctx):
    print("[case] new angles, one missing", flush=True)
    w = synth.default_wpu(N)
    with Batch(ctx, [(N, T, w, angles(0)), (N, T, w, None), (N, T, w, angles(0))]) as b:
        b.set_theta(0, angles(1))
        with pytest.raises(AcumenError):
            b.fbp()
        b.set_theta(1, angles(1))
        b.set_sino(1, np.ones((T, N), np.float32))
        b.fbp()
        got = b.get_image(1, ACU_IMG_FBP)
    with Batch(ctx, [(N, T, w, angles(1))]) as p:
        p.set_sino(0, np.ones((T, N), np.float32))
        p.fbp()
        assert np.array_equal(got, p.get_image(0, ACU_IMG_FBP))
