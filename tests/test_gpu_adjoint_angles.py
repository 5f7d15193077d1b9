"""The adjoint of angles that are not finite: such an angle has no samples, so
its rays reach no pixel, whatever they hold (the projector's own test of a
sample's cell fails for every one of them)."""
import numpy as np
import pytest

from acumen_amd import Batch, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("N,T", [(33, 40), (100, 7)])
def test_angles_that_are_not_finite(ctx, N, T, bad):
    print("[case] adjoint angles", N, T, bad, flush=True)
    th = synth.angles(T)
    y = np.random.default_rng(N).random((T, N), dtype=np.float32)
    gone = [0, 3, T - 1]
    z = y.copy()
    z[gone] = 0.0
    with Batch(ctx, [(N, T, synth.default_wpu(N), th)]) as b:
        want = b.radon_adjoint(z)
    th[gone] = bad
    y[3, N // 2] = np.inf
    with Batch(ctx, [(N, T, synth.default_wpu(N), th)]) as b:
        assert np.array_equal(b.radon_adjoint(y), want)
