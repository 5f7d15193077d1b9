"""The median filter's strips of sorted rows (2 rows a wave for small images,
8 for large) around their edges, waves that hold a NaN, and corrections of
groups of projections."""
import numpy as np
import pytest

from acumen_amd import _lib
from helpers import HipBuffers
from oracle import ref
from test_median_net import network  # noqa: F401  (fixture: the comparator network)

pytestmark = pytest.mark.gpu


def median(ctx, l, c, r):
    n = c.shape[0]
    hb = HipBuffers()
    try:
        dl, dc, dr, do = hb.upload(l), hb.upload(c), hb.upload(r), hb.alloc(c.nbytes)
        assert _lib.load().acu_prep_median27_dev(ctx.handle, n, dl, dc, dr, do) == 0
        ctx.synchronize()
        return hb.download(do, (n, n))
    finally:
        hb.close()


@pytest.mark.parametrize("n", [1, 2, 3, 7, 61, 62, 63, 125, 1023])
def test_median_strip_edges(ctx, n):
    rng = np.random.default_rng(n)
    l, c, r = [np.round(rng.normal(size=(n, n)) * 4).astype(np.float32) for _ in range(3)]  # many ties
    l[0, 0], c[-1, -1] = np.inf, -np.inf
    assert np.array_equal(median(ctx, l, c, r), ref.prep_median27(l, c, r))


@pytest.mark.parametrize("n", [70, 1023])
def test_median_with_nans_is_the_networks(ctx, n, network):  # noqa: F811
    rng = np.random.default_rng(n)
    l, c, r = [rng.normal(size=(n, n)).astype(np.float32) for _ in range(3)]
    c[5, 66], l[n - 1, 0], r[n // 2, n // 2] = np.nan, np.nan, np.nan
    v = []
    for p in (l, c, r):
        q = np.pad(p, 1, mode="edge")
        v += [q[dy:dy + n, dx:dx + n].copy() for dy in range(3) for dx in range(3)]
    pairs, out = network
    for a, b in pairs:
        v[a], v[b] = np.fmin(v[a], v[b]), np.fmax(v[a], v[b])
    got = median(ctx, l, c, r)
    assert np.array_equal(got, v[out], equal_nan=True)


@pytest.mark.parametrize("count,job0,nfiles", [(1, 0, 1), (3, 2, 5), (4, 1, 6), (9, 0, 9)])
def test_correct_groups_of_projections(ctx, count, job0, nfiles):
    n, th, sh = 34, 0.011, -0.013
    nw = n + 1
    imgs = np.random.default_rng(count).normal(size=(count, n, n)).astype(np.float32)
    keep = np.full((n, nfiles, nw), 7.0, np.float32)
    hb = HipBuffers()
    try:
        di, ds = hb.upload(imgs), hb.upload(keep)
        assert _lib.load().acu_prep_correct_dev(ctx.handle, n, 1, th, sh, di, count, job0, nfiles, ds) == 0
        ctx.synchronize()
        got = hb.download(ds, keep.shape)
    finally:
        hb.close()
    for k in range(count):
        assert np.array_equal(got[:, job0 + k], ref.prep_correct(imgs[k], th, sh)), k
    rest = np.setdiff1d(np.arange(nfiles), job0 + np.arange(count))
    assert (got[:, rest] == 7.0).all()
