"""The adjoint projector around its 16 x 16 tiles (rim tiles and angles whose
samples leave the sweep take the checked loop) and its blocks of 32 angles,
and rays of infinity or NaN, which reach only the pixels they cover."""
import numpy as np
import pytest

from acumen_amd import Batch, synth
from helpers import rel
from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,T", [(3, 2), (15, 31), (16, 32), (17, 33), (32, 64), (34, 65), (49, 5), (112, 40)])
def test_adjoint_tile_edges(ctx, N, T):
    rng = np.random.default_rng(N + T)
    th = rng.uniform(-180.0, 360.0, T).astype(np.float32)
    y = rng.normal(size=(T, N)).astype(np.float32)
    with Batch(ctx, [(N, T, 4, th)]) as b:
        # the same positions and weights; FP32 sums in another order
        assert rel(b.radon_adjoint(y), ref.radon_adjoint(y, th, "f32")) < 5e-6


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_nonfinite_rays_reach_only_their_pixels(ctx, bad):
    N, T = 49, 40
    th = synth.angles(T)
    y = np.random.default_rng(3).normal(size=(T, N)).astype(np.float32)
    e = np.zeros((T, N), np.float32)
    for t, d in ((0, 20), (7, 3), (33, 40)):
        e[t, d] = 1.0
    with Batch(ctx, [(N, T, 4, th)]) as b:
        covered = b.radon_adjoint(e) > 0
        clean = b.radon_adjoint(y)
        got = b.radon_adjoint(np.where(e > 0, np.float32(bad), y))
    assert np.array_equal(np.isfinite(got), ~covered)
    assert rel(got[~covered], clean[~covered]) < 5e-6
