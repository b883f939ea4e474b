"""Small selections against at most 64 centroids (one block holds all of them)
and training batches of up to 1,024 positions updated in one launch: the edges
of their row groups, centroid tiles, column phases and position words, with
NaN, infinities, ties and bad keys; bit-equal to the oracle."""

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


@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("n,d,k", [
    (1, 4, 1), (15, 36, 2), (16, 64, 16), (17, 1028, 16), (9, 60, 17), (1000, 768, 20),
    (33, 820, 32), (5, 100, 33), (700, 484, 64), (8192, 32, 7), (8193, 32, 7), (2100, 32, 64), (300, 64, 65),
])
def test_small_k(dev, n, d, k, metric):
    from emeans_amd import Mat, Select
    g = np.random.default_rng(n * 7 + k)
    x = g.standard_normal((n, d)).astype(np.float32)
    c = g.standard_normal((k, d)).astype(np.float32)
    c[k // 2] = c[0]  # ties go to the lower id
    if n > 8:
        x[3] = 0.0
        x[4, 1] = np.nan
        x[5, 2] = np.inf
        x[6] = 3e38
    if k > 3:
        c[1, 0] = np.nan
    ids = g.permutation(n).astype(np.uint32)
    lab, sc = dev.zeros_u32(n), dev.zeros_f32(n)
    cb, cn = dev.upload_f32(c), None
    if metric == "l2":
        cn = dev.zeros_f32(k)
        dev.row_norms(cb, k, d, cn)
    xb, idb = dev.bind(x), dev.upload_u32(ids)
    lo = n // 5
    for i, ib in ((ids, idb), (None, None)):
        dev.top1(Mat(xb, d), Select(ib, (lo, n)), cb, cn, k, metric, lab, sc)
        ol, osc = np.zeros(n, np.uint32), np.zeros(n, np.float32)
        O.top1(x, d, c, metric, ids=i, rows=(lo, n), labels=ol, scores=osc)
        gl, gs = dev.read_u32(lab), dev.read_f32(sc)
        assert np.array_equal(gl[lo:], ol[lo:])
        same = (gs[lo:].view(np.uint32) == osc[lo:].view(np.uint32)) | \
            (np.isnan(gs[lo:]) & np.isnan(osc[lo:]))
        assert same.all()


@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("n,d,k", [(8192, 32, 16), (8193, 32, 16), (4096, 36, 32), (4097, 36, 17),
                                   (2048, 64, 64), (2049, 64, 33)])
def test_small_k_row_limit(dev, n, d, k, metric):
    """The most rows of each centroid padding that one block's scan takes, and
    one more (the screen)."""
    from emeans_amd import Mat, Select
    g = np.random.default_rng(n + k)
    x = g.standard_normal((n, d)).astype(np.float32)
    c = g.standard_normal((k, d)).astype(np.float32)
    cb, cn = dev.upload_f32(c), None
    if metric == "l2":
        cn = dev.zeros_f32(k)
        dev.row_norms(cb, k, d, cn)
    lab, sc = dev.zeros_u32(n), dev.zeros_f32(n)
    dev.top1(Mat(dev.bind(x), d), Select(None, (0, n)), cb, cn, k, metric, lab, sc)
    ol, osc = O.top1(x, d, c, metric)
    assert np.array_equal(dev.read_u32(lab), ol)
    assert dev.read_f32(sc).tobytes() == osc.tobytes()


@pytest.mark.parametrize("spherical", [False, True])
@pytest.mark.parametrize("batch,k,d", [(8193, 10, 32), (4100, 20, 36), (2049, 50, 64)])
def test_small_k_train_over_limit(dev, batch, k, d, spherical):
    """Tallied batches just past the limit, their tails below it."""
    from emeans_amd import Config, Emeans
    g = np.random.default_rng(batch)
    n = 2 * batch + 301
    x = (g.standard_normal((n, d)) + 3 * g.standard_normal((k, d))[g.integers(0, k, n)])
    x = x.astype(np.float32)
    if spherical:
        x /= np.linalg.norm(x, axis=1, keepdims=True)
    cfg = Config(d=d, k=k, nepochs=2, batch_size=batch, spherical=spherical, seed=6)
    m = Emeans(cfg, dev)
    t = m.train_from(x, None)
    o = O.train(x, d, k, nepochs=cfg.nepochs, batch_size=cfg.batch_size, alpha0=cfg.alpha0,
                batch_law=cfg.batch_law, seed=cfg.seed, spherical=cfg.spherical,
                unused_threshold=cfg.unused_threshold)
    assert np.array_equal(t.labels, o["labels"])
    assert t.centroids.tobytes() == o["centroids"].tobytes()


def test_small_k_bad_id(dev):
    """A row id past the data is still reported."""
    from emeans_amd import Mat, Select
    x = np.ones((20, 16), np.float32)
    ids = np.arange(20, dtype=np.uint32)
    ids[11] = 20
    lab, sc = dev.zeros_u32(20), dev.zeros_f32(20)
    with pytest.raises(Exception):
        dev.top1(Mat(dev.bind(x), 16), Select(dev.upload_u32(ids), (0, 20)),
                 dev.upload_f32(x[:3].copy()), None, 3, "ip", lab, sc)
        dev.read_u32(lab)


@pytest.mark.parametrize("spherical", [False, True])
@pytest.mark.parametrize("batch,k,d", [(256, 6, 20), (257, 6, 20), (1000, 3, 64), (1024, 40, 32),
                                       (1025, 40, 32), (1024, 70, 1024), (700, 64, 100)])
def test_update_batches(dev, batch, k, d, spherical):
    from emeans_amd import Config, Emeans
    g = np.random.default_rng(batch + k)
    n = 3 * batch + 17
    x = (g.standard_normal((n, d)) + 3 * g.standard_normal((4, d))[g.integers(0, 4, n)])
    x = x.astype(np.float32)
    if spherical:
        x /= np.linalg.norm(x, axis=1, keepdims=True)
    cfg = Config(d=d, k=k, nepochs=3, batch_size=batch, spherical=spherical, seed=5)
    m = Emeans(cfg, dev)
    t = m.train_from(x, None)
    o = O.train(x, d, k, nepochs=cfg.nepochs, batch_size=cfg.batch_size, alpha0=cfg.alpha0,
                batch_law=cfg.batch_law, seed=cfg.seed, spherical=cfg.spherical,
                unused_threshold=cfg.unused_threshold)
    pos, usage = m.ema_state()
    assert np.array_equal(t.labels, o["labels"])
    assert pos.tobytes() == o["positions"].tobytes()
    assert usage.tobytes() == o["usage"].tobytes()
    assert t.centroids.tobytes() == o["centroids"].tobytes()
