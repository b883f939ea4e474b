"""Long queues of rows that the screen's check cannot settle: the exact scans in
tiles. Crowds of equal and nearly equal centroids (data rows) put every row in
the queue; results equal the oracle's bit for bit."""

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from emeans_amd import HipDevice
    d = HipDevice()
    yield d
    d.close()


def _crowds(n, d, each, seed):
    """Groups of `each` rows within 1e-7 of one another, a third of them equal."""
    g = np.random.default_rng(seed)
    x = g.standard_normal((n, d)).astype(np.float32)
    x /= np.linalg.norm(x, axis=1, keepdims=True)
    base = x[np.arange(n) // each * each]
    y = base * (1 + 1e-7 * g.standard_normal((n, d)).astype(np.float32))
    y[::3] = base[::3]
    return np.ascontiguousarray(y.astype(np.float32))


@pytest.mark.parametrize("metric", ["ip", "l2"])
@pytest.mark.parametrize("n,d,k,off", [
    (5000, 32, 1000, 0),     # the last tiles part rows, part centroids
    (5000, 36, 1025, 1),     # four dimensions past the slabs, an unaligned matrix
    (2049, 100, 2100, 0),    # ranges of centroid tiles
    (40000, 64, 129, 0),     # more items than workgroups
    (4200, 388, 257, 3),
    (5000, 33, 1000, 0),     # odd widths
    (3000, 102, 700, 1),
])
def test_queued_tiles(dev, n, d, k, metric, off):
    from emeans_amd import Mat, Select
    g = np.random.default_rng(n + k)
    c = _crowds(k, d, 43, 1)
    x = g.standard_normal((n, d)).astype(np.float32)
    c[k // 2, 1] = np.nan
    x[7], x[8, 0], x[9, 1] = 0.0, np.nan, np.inf
    ids = g.permutation(n).astype(np.uint32)
    whole = dev.upload_f32(np.concatenate([np.zeros(off, np.float32), x.reshape(-1)]))
    xb = dev.wrap(whole.ptr + 4 * off, x.size, 0)
    cb, cn = dev.upload_f32(c), None
    if metric == "l2":
        cn = dev.zeros_f32(k)
        dev.row_norms(cb, k, d, cn)
    lab, sc = dev.zeros_u32(n), dev.zeros_f32(n)
    for i in (ids, None):
        f0 = dev.fallback_rows()
        dev.top1(Mat(xb, d), Select(None if i is None else dev.upload_u32(i), (3, n)), cb, cn, k,
                 metric, lab, sc)
        ol, os_ = np.zeros(n, np.uint32), np.zeros(n, np.float32)
        O.top1(x, d, c, metric, ids=i, rows=(3, n), labels=ol, scores=os_)
        gl, gs = dev.read_u32(lab), dev.read_f32(sc)
        assert (dev.fallback_rows() - f0) * k > 1 << 20  # the tiles ran
        assert np.array_equal(gl[3:], ol[3:])
        same = (gs[3:].view(np.uint32) == os_[3:].view(np.uint32)) | \
            (np.isnan(gs[3:]) & np.isnan(os_[3:]))
        assert same.all()
    del whole


@pytest.mark.parametrize("spherical", [False, True])
def test_queued_tiles_train(dev, spherical):
    """Tallied batches whose rows are queued (initial centroids in crowds)."""
    from emeans_amd import Config
    n, d, k = 20000, 48, 600
    x = _crowds(n, d, 2000, 2)
    cfg = Config(d=d, k=k, nepochs=2, batch_size=8192, spherical=spherical, seed=9)
    cent, info = dev.train_dev(dev.bind(x), n, cfg)
    assert info["fallback_rows"] * k > 1 << 21
    o = O.train(x, d, k, nepochs=cfg.nepochs, batch_size=cfg.batch_size, alpha0=cfg.alpha0,
                batch_law=cfg.batch_law, seed=cfg.seed, spherical=cfg.spherical,
                unused_threshold=cfg.unused_threshold)
    assert np.array_equal(info["labels"], o["labels"])
    assert info["positions"].tobytes() == o["positions"].tobytes()
    assert cent.tobytes() == o["centroids"].tobytes()


@pytest.mark.parametrize("m,n,d,kk,self_", [
    (700, 3000, 32, 10, False),    # parts of several tiles, the last a remainder
    (1, 5, 40, 16, False),         # fewer data rows than neighbours
    (33, 129, 20, 1, False),       # one past a query tile and a data tile; no screen
    (300, 20000, 33, 16, False),   # 64 parts
    (2900, 2900, 64, 16, True),
    (20000, 600, 36, 3, False),    # more query tiles than workgroups: one part
])
def test_queued_knn(dev, m, n, d, kk, self_):
    g = np.random.default_rng(m + n)
    x = _crowds(n, d, 97, 5)
    q = x if self_ else g.standard_normal((m, d)).astype(np.float32)
    if n > 500:
        x[n // 2, 1], x[n // 3, 2], x[11] = np.nan, np.inf, 0.0
        q[5 % m] = 0.0                       # every score +0 or -0
        x[20:60] *= np.where(g.random((40, 1)) < 0.5, -1, 1).astype(np.float32)
        q[6 % m, 0] = np.nan
    f0 = dev.fallback_rows()
    gi, gs = dev.topk(q, x, d, kk, self_)
    oi, os_ = O.knn(q, x, d, kk, self_)
    assert np.array_equal(gi, oi)
    assert gs.tobytes() == os_.tobytes()
    assert dev.fallback_rows() - f0 >= m // 2


@pytest.mark.parametrize("each,kk,queued", [
    (24, 12, False), (25, 12, True),   # lists of 24
    (33, 13, False), (40, 16, False), (41, 16, True),  # lists of 40
])
@pytest.mark.parametrize("n,d", [(600, 64), (9000, 33)])
def test_near_ties_within_the_lists(dev, n, d, each, kk, queued):
    """Near-ties that a list has room for beside the neighbours are settled from
    it; a list of more goes to the exact scan."""
    g = np.random.default_rng(n + each)
    x = _crowds(n, d, 1, 9)
    x[10:10 + each] = _crowds(each, d, each, 3)
    q = (x[10] + np.float32(0.01) * g.standard_normal((300, d))).astype(np.float32)
    f0 = dev.fallback_rows()
    gi, gs = dev.topk(q, x, d, kk, False)
    f1 = dev.fallback_rows() - f0
    oi, os_ = O.knn(q, x, d, kk, False)
    assert np.array_equal(gi, oi)
    assert gs.tobytes() == os_.tobytes()
    assert f1 == (len(q) if queued else 0)


def test_queued_knn_few(dev):
    """A few queued queries among many: the parts' lists and their ranking, call
    after call (the tickets are left at zero)."""
    g = np.random.default_rng(8)
    n, d, m = 9000, 48, 600
    x = _crowds(n, d, 1, 9)
    x[4000:4200] = x[4000]
    q = g.standard_normal((m, d)).astype(np.float32)
    q[::50] = x[4000] + np.float32(0.01) * q[::50]
    for kk in (1, 7, 16):
        gi, gs = dev.topk(q, x, d, kk, False)
        oi, os_ = O.knn(q, x, d, kk, False)
        assert np.array_equal(gi, oi)
        assert gs.tobytes() == os_.tobytes()
