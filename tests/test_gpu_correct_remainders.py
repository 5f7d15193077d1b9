"""Corrections of every count of projections up to two groups of four and one
more, which the last workgroups take as 1, 2 or 3: each against the oracle,
and the rows of other projections untouched."""
import numpy as np
import pytest

from acumen_amd import _lib
from helpers import HipBuffers
from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [33, 300])
@pytest.mark.parametrize("count", range(1, 10))
def test_correct_remainders(ctx, n, count):
    print("[case] correct remainders", n, count, flush=True)
    th, sh, add, job0, nfiles = 0.011, -0.013, 1 - n % 2, 1, 11
    imgs = np.random.default_rng(count).normal(size=(count, n, n)).astype(np.float32)
    keep = np.full((n, nfiles, n + add), 7.0, np.float32)
    hb = HipBuffers()
    try:
        di, ds = hb.upload(imgs), hb.upload(keep)
        assert _lib.load().acu_prep_correct_dev(ctx.handle, n, add, th, sh, di, count, job0, nfiles, ds) == 0
        ctx.synchronize()
        got = hb.download(ds, keep.shape)
    finally:
        hb.close()
    for k in range(count):
        assert np.array_equal(got[:, job0 + k], ref.prep_correct(imgs[k], th, sh)), k
    rest = np.setdiff1d(np.arange(nfiles), job0 + np.arange(count))
    assert (got[:, rest] == 7.0).all()
