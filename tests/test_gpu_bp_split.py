"""The backprojector of small launches (a workgroup's waves share out the
angle blocks) against the one of large launches, bit for bit: one slice
alone, and the same slice in a batch whose other slice makes the launch a
large one.  Sizes around its tiles (64 x 8 and 64 x 16), its angle blocks of
32 staged 8 at a time, and its rounds of 8 blocks."""
import numpy as np
import pytest

from acumen_amd import ACU_IMG_FBP, Batch, synth
from helpers import rel
from oracle import ref

pytestmark = pytest.mark.gpu

BIG = (1537, 1, 48, np.zeros(1, np.float32))  # its tiles take the launch past the split kernel's limit


@pytest.mark.parametrize("N,T", [(3, 1), (8, 9), (16, 33), (17, 31), (63, 257), (64, 8), (65, 300), (129, 64),
                                 (200, 513), (449, 40), (513, 65), (769, 33)])
def test_split_backprojection_equals_the_full_kernel(ctx, N, T):
    rng = np.random.default_rng(N * T)
    th = rng.uniform(-90.0, 270.0, T).astype(np.float32)
    f = rng.normal(size=(T, N)).astype(np.float32)
    spec = (N, T, max(1, N // 32), th)
    with Batch(ctx, [spec]) as b:
        b.set_sino(0, f)
        b.fbp()
        alone = b.get_image(0, ACU_IMG_FBP)
    with Batch(ctx, [BIG, spec]) as b:
        b.set_sino(1, f)
        b.fbp()
        assert np.array_equal(alone, b.get_image(1, ACU_IMG_FBP))
    # and the reference's own arithmetic (FP32 sums in another order: 1e-5)
    assert rel(alone, ref.iradon(f, th, spec[2], "f32")) < 1e-5
