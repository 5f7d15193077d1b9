"""The LDS projector of small launches (a block's angles over several
workgroups, boxes staged a chunk ahead) against the one of large launches,
bit for bit: one CG step of TV on one slice alone, and on the same slice in a
batch whose other slice makes the launches large ones.  Sizes around the ray
blocks of 64, the chunks of 32 steps and the angle blocks; coarse angles
whose boxes overflow into the global gathers."""
import numpy as np
import pytest

from acumen_amd import ACU_IMG_TV, ACU_TV_BATCHED, Batch, synth
from helpers import rel
from oracle import ref

pytestmark = pytest.mark.gpu

BIG = (1025, 400, 32, synth.angles(400))  # 1700 or more workgroups in every variant


@pytest.mark.parametrize("variant", [1, 2, 4])
@pytest.mark.parametrize("N,T", [(3, 1), (31, 5), (64, 17), (65, 48), (130, 33), (257, 180), (300, 7), (385, 15)])
def test_split_projection_equals_the_full_kernel(ctx, N, T, variant):
    rng = np.random.default_rng(N * T)
    spec = (N, T, max(1, N // 32), rng.uniform(0.0, 180.0, T).astype(np.float32) if N == 130 else synth.angles(T))
    f = rng.random((T, N), np.float32)

    def tv(slices, i):
        with Batch(ctx, slices) as b:
            for k in range(len(slices)):
                b.set_fp_variant(k, variant)
            b.set_sino(i, f)
            b.tvopt(0.05, 0.1, 1, 1, 1, ACU_TV_BATCHED)
            return b.get_image(i, ACU_IMG_TV)

    assert np.array_equal(tv([spec], 0), tv([BIG, spec], 1))


@pytest.mark.parametrize("N,T", [(65, 48), (129, 13), (300, 7)])
def test_border_and_gather_samples_match_oracle(ctx, N, T):
    """Images that are nonzero up to their edges: every edge decision is the
    reference's, so only rounding (1e-6) is left."""
    x = np.random.default_rng(N).random((N, N), np.float32) + np.float32(0.5)
    th = synth.angles(T)
    want = ref.radon(x, th, "f32")
    with Batch(ctx, [(N, T, 4, th)]) as b:
        for v in (1, 2, 4):
            b.set_fp_variant(0, v)
            assert rel(b.radon(x), want) < 1e-6, v
