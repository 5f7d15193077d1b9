"""The host-memory calls of a plan: angles set again, unchanged and changed,
the buffers and the task slot they keep between calls, and device-pointer
calls queued without a wait between them."""
import numpy as np
import pytest

from acumen_amd import ACU_IMG_FBP, ACU_IMG_TV, AcumenError, Batch, synth
from helpers import HipBuffers

pytestmark = pytest.mark.gpu
N, T, WPU = 65, 48, 4


def fresh(ctx, th, call):
    with Batch(ctx, [(N, T, WPU, th)]) as b:
        return call(b)


def test_angles_set_again(ctx):
    rng = np.random.default_rng(0)
    th1, th2 = synth.angles(T), rng.uniform(0, 180, T).astype(np.float32)
    x, f = rng.random((N, N), np.float32), rng.random((T, N), np.float32)
    with Batch(ctx, [(N, T, WPU, None)]) as b:
        for th in (th1, th1, th2, th2, th1):
            b.set_theta(0, th)
            b.set_sino(0, f)
            assert np.array_equal(b.radon(x), fresh(ctx, th, lambda p: p.radon(x)))
            b.tvopt(0.05, 0.1, 2)
            tv = b.get_image(0, ACU_IMG_TV)
            b.set_theta(0, th)  # unchanged angles still invalidate the slice's images
            for which in (ACU_IMG_TV, ACU_IMG_FBP):
                with pytest.raises(AcumenError):
                    b.get_image(0, which)

            def run(p):
                p.set_sino(0, f)
                p.tvopt(0.05, 0.1, 2)
                return p.get_image(0, ACU_IMG_TV)

            assert np.array_equal(tv, fresh(ctx, th, run))


def test_kept_buffers_hold_nothing_of_the_last_call(ctx):
    rng = np.random.default_rng(1)
    th = synth.angles(T)
    xs = [rng.random((N, N), np.float32) for _ in range(2)]
    fs = [rng.random((T, N), np.float32) for _ in range(2)]
    with Batch(ctx, [(N, T, WPU, th)]) as b:
        for x, f in zip(xs, fs):
            got = b.radon(x), b.iradon(f), b.radon_adjoint(f)
            want = fresh(ctx, th, lambda p: (p.radon(x), p.iradon(f), p.radon_adjoint(f)))
            for g, w in zip(got, want):
                assert np.array_equal(g, w)


def test_queued_device_calls_keep_their_own_tasks(ctx):
    """Calls on different pointers, queued back to back: each runs its own
    task though they share the batch's slot."""
    rng = np.random.default_rng(2)
    th = synth.angles(T)
    xs = [rng.random((N, N), np.float32) for _ in range(12)]
    hb = HipBuffers()
    try:
        with Batch(ctx, [(N, T, WPU, th)]) as b:
            want = [b.radon(x) for x in xs]
            src, dst = [hb.upload(x) for x in xs], [hb.alloc(4 * N * T) for _ in xs]
            for s, d in zip(src, dst):
                b.radon_dev(0, d, s)
            ctx.synchronize()
            for d, w in zip(dst, want):
                assert np.array_equal(hb.download(d, (T, N)), w)
    finally:
        hb.close()
