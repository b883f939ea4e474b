"""The one-pass fp16 screen (k_screen5) at the sizes and inputs where its own
parts can go wrong: tile and slab remainders, parts, the append buffers' and
logs' overflows, and values around and beyond fp16's range. Results equal the
oracle's bit for bit: the screen only chooses what the exact chains score."""

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


def _rows(n, d, seed):
    x = np.random.default_rng(seed).standard_normal((n, d), dtype=np.float32)
    return (x / np.linalg.norm(x, axis=1, keepdims=True)).astype(np.float32)


def _knn(dev, q, x, kk, self_):
    d = x.shape[1]
    gi, gs = dev.topk(x if self_ else q, x, d, kk, self_)
    oi, os_ = O.knn(x if self_ else q, x, d, kk, self_)
    assert np.array_equal(gi, oi)
    assert gs.tobytes() == os_.tobytes()


@pytest.mark.parametrize("m,n,d,kk,self_", [
    (256, 512, 32, 1, False),    # the smallest call, one slab
    (257, 513, 33, 16, False),   # one past a tile of queries and of data
    (300, 9000, 99, 10, False),  # parts of several tiles, an odd width
    (700, 2100, 384, 16, False),
    (767, 767, 64, 10, True),
    (1025, 1025, 100, 16, True),
])
def test_knn_shapes(dev, m, n, d, kk, self_):
    _knn(dev, _rows(m, d, m + d), _rows(n, d, n + d), kk, self_)


def test_knn_bursts_and_crowds(dev):
    """Runs of 40 consecutive near-duplicates overflow a row's append buffer
    within a tile; 300 exact duplicates overflow the lists (the exact scan)."""
    n, d = 2000, 96
    x = _rows(n, d, 5)
    noise = np.random.default_rng(6).standard_normal((n, d), dtype=np.float32)
    for a in range(0, 1200, 40):
        x[a:a + 40] = x[a] + np.float32(1e-3) * noise[a:a + 40]
    x[1500:1800] = x[1500]
    _knn(dev, x, x, 10, True)
    _knn(dev, x[::5].copy(), x, 16, False)


def test_knn_rising_similarity(dev):
    """Data rows in order of rising similarity to every query: each one enters
    the lists when it comes, so the logs fill and are swept."""
    n, d, m = 8000, 64, 260
    base = _rows(1, d, 1)[0]
    t = np.linspace(2.0, 0.01, n, dtype=np.float32)[:, None]
    x = base + t * _rows(n, d, 2)
    x = (x / np.linalg.norm(x, axis=1, keepdims=True)).astype(np.float32)
    q = (base + np.float32(0.01) * _rows(m, d, 3)).astype(np.float32)
    _knn(dev, q, x, 16, False)


@pytest.mark.parametrize("case", ["large", "tiny", "mixed", "beyond", "special"])
def test_knn_ranges(dev, case):
    """Magnitudes that the scale brings into fp16's range, rows far below the
    others, elements that overflow fp16 (their residual is infinite: the exact
    scan), NaN and infinite elements."""
    m, n, d = 300, 1500, 128
    q, x = _rows(m, d, 11), _rows(n, d, 12)
    if case == "large":
        q, x = q * np.float32(1e9), x * np.float32(3e12)
    elif case == "tiny":
        q, x = q * np.float32(1e-15), x * np.float32(1e-12)
    elif case == "mixed":
        s = np.array([1.0, 1e-3, 1e-6, 1e-9], np.float32)
        q, x = q * s[np.arange(m) % 4][:, None], x * s[np.arange(n) % 4][:, None]
    elif case == "beyond":
        x[700] *= np.float32(1e7)
        q[5] *= np.float32(1e8)
    else:
        x[100, 3], x[200, 7], x[300] = np.nan, np.inf, 0.0
        q[7, 0], q[8, 1], q[9] = np.nan, -np.inf, 0.0
    _knn(dev, np.ascontiguousarray(q), np.ascontiguousarray(x), 10, False)


def _top1(dev, x, c, metric, ids=None):
    from emeans_amd import Mat, Select
    n, d = x.shape
    k = c.shape[0]
    m = n if ids is None else len(ids)
    cb, cn = dev.upload_f32(c), None
    if metric == "l2":
        cn = dev.zeros_f32(k)
        dev.row_norms(cb, k, d, cn)
    lab, sco = dev.zeros_u32(m), dev.zeros_f32(m)
    idb = None if ids is None else dev.upload_u32(ids)
    dev.top1(Mat(dev.bind(x), d), Select(idb, (0, m)), cb, cn, k, metric, lab, sco)
    gl, gs = dev.read_u32(lab), dev.read_f32(sco)
    ol, os_ = O.top1(x, d, c, metric, ids=ids)
    assert np.array_equal(gl, ol)
    assert gs.tobytes() == os_.tobytes()


@pytest.mark.parametrize("metric", ["ip", "l2"])
@pytest.mark.parametrize("n,d,k", [
    (33000, 32, 64),     # one tile per part, mostly padding; one slab
    (16384, 33, 512),
    (8191, 99, 1100),    # five tiles, the last a remainder
    (4097, 64, 2048),    # eight single-tile parts
    (4000, 100, 2049),   # nine tiles: parts of several
    (3000, 384, 5000),
])
def test_top1_shapes(dev, metric, n, d, k):
    ids = ((np.arange(n, dtype=np.uint64) * 7919 + 3) % n).astype(np.uint32)
    x, c = _rows(n, d, n + k), _rows(k, d, k)
    x[: n // 2] = c[np.arange(n // 2) % k] + np.float32(0.3) * x[: n // 2]
    _top1(dev, x, c, metric, ids)


@pytest.mark.parametrize("k", [1024, 3000])
@pytest.mark.parametrize("metric", ["ip", "l2"])
def test_top1_crowds(dev, metric, k):
    """Groups of 20 consecutive centroids within 1e-6, some exact duplicates:
    more near-ties than a part's list keeps, and than its buffers hold."""
    n, d = 8192, 128
    c = _rows(k, d, 21)
    noise = _rows(k, d, 22)
    for a in range(0, 400, 20):
        c[a:a + 20] = c[a] + np.float32(1e-6) * noise[a:a + 20]
        c[a + 7] = c[a + 3]
    x = c[np.arange(n) % k] + np.float32(0.2) * _rows(n, d, 23)
    _top1(dev, x, c, metric)


@pytest.mark.parametrize("case", ["large", "tiny", "mixed", "beyond", "special"])
@pytest.mark.parametrize("metric", ["ip", "l2"])
@pytest.mark.parametrize("k", [600, 2100])
def test_top1_ranges(dev, metric, case, k):
    """As test_knn_ranges."""
    n, d = 16384, 64
    x, c = _rows(n, d, 31), _rows(k, d, 32)
    if case == "large":
        x, c = x * np.float32(1e9), c * np.float32(3e12)
    elif case == "tiny":
        x, c = x * np.float32(1e-12), c * np.float32(1e-15)
    elif case == "mixed":
        s = np.array([1.0, 1e-3, 1e-6, 1e-9], np.float32)
        x, c = x * s[np.arange(n) % 4][:, None], c * s[np.arange(k) % 4][:, None]
    elif case == "beyond":
        x[5] *= np.float32(1e8)
        x[6, 9] = np.float32(1e6)
    else:
        x[7, 0], x[8, 1], x[9] = np.nan, -np.inf, 0.0
    _top1(dev, np.ascontiguousarray(x), np.ascontiguousarray(c), metric)


@pytest.mark.parametrize("k", [64, 2100])
@pytest.mark.parametrize("case", ["straddle", "overflow"])
def test_top1_largest_keys(dev, case, k):
    """L2 keys at the top of the f32 range. straddle: two centroids whose keys
    sweep across 3.0e38 from row to row, closer to each other than the screen's
    error. overflow: |c|^2 + 2 |x| |c| beyond the largest float, so no bound is
    finite and the exact scan decides."""
    n, d = 40000, 64
    g = np.random.default_rng(41)
    c = _rows(k, d, 42).astype(np.float64) * np.sqrt(3.3e38)
    if case == "straddle":
        u = _rows(2, d, 43).astype(np.float64)
        v = u[0] + 0.01 * (u[1] - (u[1] @ u[0]) * u[0])
        r = np.sqrt(3.2e38)
        c[k // 3], c[k // 2] = r * u[0], r * v / np.linalg.norm(v)
        # |c|^2 - 2 x.c sweeps 5e-6 of 3.0e38 around it
        t = (r * r - 3.0e38 * (1 + np.linspace(-5e-6, 5e-6, n))) / (2 * r)
        x = u[0] + 0.02 * _rows(n, d, 44)
        x *= (t / (x @ u[0]))[:, None]
    else:
        c[::k // 8] *= 0.8
        x = np.sqrt(3.0e38) * _rows(n, d, 45).astype(np.float64) * g.choice([0.3, 1.0], (n, 1))
    _top1(dev, x.astype(np.float32), c.astype(np.float32), "l2")


def test_top1_no_data_rows(dev):
    """Ids over an empty matrix are refused before any kernel reads a row."""
    from emeans_amd import Mat, Select
    n, d, k = 40000, 64, 300
    lab, sco = dev.zeros_u32(n), dev.zeros_f32(n)
    ids = dev.upload_u32(np.zeros(n, np.uint32))
    c = dev.upload_f32(_rows(k, d, 1))
    for m in (3, n):
        with pytest.raises(Exception, match="no data rows"):
            dev.top1(Mat(dev.zeros_f32(0), d), Select(ids, (0, m)), c, None, k, "ip", lab, sco)


@pytest.mark.parametrize("k,d", [(127, 200), (127, 300), (1016, 200), (64, 256), (2159, 320)])
def test_top1_large_columns(dev, k, d):
    """One column in units 3,000 times the others', wherever it lies: the
    screen still settles nearly every row."""
    n = 40000 if k < 1000 else 20000
    c, x = _rows(k, d, 51), _rows(n, d, 52)
    for t in (d // 3, d // 2, d - 40, d - 1):
        cc, xx = c.copy(), x.copy()
        cc[:, t] *= np.float32(3000)
        xx[:, t] *= np.float32(3000)
        f0 = dev.fallback_rows()
        _top1(dev, xx, cc, "ip")
        assert dev.fallback_rows() - f0 < n // 50


def test_top1_rows_outside_selection(dev):
    """Rows that are not selected say nothing of the selected ones' scale."""
    from emeans_amd import Mat, Select
    n, d, k = 60000, 64, 300
    x, c = _rows(n, d, 61), _rows(k, d, 62)
    x[20000:] *= np.float32(1e12)
    ids = np.random.default_rng(63).permutation(20000).astype(np.uint32)
    lab, sco = dev.zeros_u32(n), dev.zeros_f32(n)
    for i in (None, ids):
        f0 = dev.fallback_rows()
        dev.top1(Mat(dev.bind(x), d), Select(None if i is None else dev.upload_u32(i), (0, 20000)),
                 dev.upload_f32(c), None, k, "ip", lab, sco)
        ol, os_ = O.top1(x[:20000], d, c, "ip", ids=i)
        assert np.array_equal(dev.read_u32(lab)[:20000], ol)
        assert dev.read_f32(sco)[:20000].tobytes() == os_.tobytes()
        assert dev.fallback_rows() - f0 < 200


def _common(n, d, s, seed, unit=True):
    """Rows that share most of their length: a mean and noise s times it."""
    x = 1.0 + s * np.random.default_rng(seed).standard_normal((n, d))
    if unit:
        x /= np.linalg.norm(x, axis=1, keepdims=True)
    return x.astype(np.float32)


@pytest.mark.parametrize("metric", ["ip", "l2"])
@pytest.mark.parametrize("n,d,k", [(40000, 33, 256), (16384, 64, 1024), (16384, 128, 2500)])
def test_top1_common_mean(dev, metric, n, d, k):
    """The screen's error follows the centroids' distance from their mean, not
    their length: next to no row goes to the exact scan."""
    x, c = _common(n, d, 0.1, 71, metric == "ip"), _common(k, d, 0.1, 72, metric == "ip")
    f0 = dev.fallback_rows()
    _top1(dev, x, c, metric)
    assert dev.fallback_rows() - f0 < n // 20
    from emeans_amd import Mat, Select
    cb, cn = dev.upload_f32(c), None
    if metric == "l2":
        cn = dev.zeros_f32(k)
        dev.row_norms(cb, k, d, cn)
    r = dev.screen_margin(Mat(dev.bind(x), d), Select(None, (0, n)), cb, cn, k, metric)
    assert r["pairs"] > n // 2 and r["over"] == 0 and r["max_dot_ratio"] <= 0.5, r


@pytest.mark.parametrize("n,d,s", [(3000, 64, 0.2), (3001, 384, 0.3), (4000, 100, 0.1)])
def test_knn_common_mean(dev, n, d, s):
    x = _common(n, d, s, 73)
    f0 = dev.fallback_rows()
    _knn(dev, x, x, 10, True)
    _knn(dev, x[::7].copy(), x, 10, False)
    assert dev.fallback_rows() - f0 < n // 10
    _knn(dev, x[:2000].copy(), x, 60, False)
    r = dev.screen_margin_topk(dev.bind(x), n, dev.bind(x), n, d, True)
    assert r["pairs"] > n and r["over"] == 0 and r["max_dot_ratio"] <= 0.5, r


@pytest.mark.parametrize("spherical", [False, True])
@pytest.mark.parametrize("n,d,k,batch,s", [
    (40000, 64, 700, 16384, 0.15),   # the EMA's lines, revivals
    (30000, 36, 300, 16384, 3.0),
    (12000, 32, 8200, 1024, 0.2),    # the small batches' lines
])
def test_train_common_mean(dev, n, d, k, batch, s, spherical):
    from emeans_amd import Config
    x = _common(n, d, s, 74, spherical)
    x[: n // 2] += (0.3 * x[0]).astype(np.float32)  # two densities, so that some centroids die
    if spherical:
        x /= np.linalg.norm(x, axis=1, keepdims=True)
    cfg = Config(d=d, k=k, nepochs=2, batch_size=batch, spherical=spherical, seed=3)
    f0 = dev.fallback_rows()
    cent, info = dev.train_dev(dev.bind(x), n, cfg)
    o = O.train(x, d, k, nepochs=cfg.nepochs, batch_size=cfg.batch_size, alpha0=cfg.alpha0,
                batch_law=cfg.batch_law, seed=cfg.seed, spherical=cfg.spherical,
                unused_threshold=cfg.unused_threshold)
    assert np.array_equal(info["labels"], o["labels"])
    assert info["positions"].tobytes() == o["positions"].tobytes()
    assert cent.tobytes() == o["centroids"].tobytes()
    assert dev.fallback_rows() - f0 < n // 5


@pytest.mark.parametrize("d", [32, 36, 61, 64, 65, 96, 127, 128, 129])
def test_top1_narrow_rows(dev, d):
    """The lines of rows of up to 128 dimensions: one, two and four slabs a
    row, their remainders, and the first width past them."""
    n, k = 16411, 520
    x, c = _rows(n, d, 81), _rows(k, d, 82)
    ids = ((np.arange(n, dtype=np.uint64) * 7919 + 3) % n).astype(np.uint32)
    for i in (None, ids):
        f0 = dev.fallback_rows()
        _top1(dev, x, c, "ip", i)
        assert dev.fallback_rows() - f0 < n // 50


@pytest.mark.parametrize("metric", ["ip", "l2"])
def test_top1_pieces(dev, metric):
    """A selection of more rows than one piece, by ids and from an odd start."""
    from emeans_amd import Mat, Select
    n, d, k, lo = (1 << 20) + 70001, 32, 300, 5
    x, c = _rows(n, d, 91), _rows(k, d, 92)
    ids = ((np.arange(n, dtype=np.uint64) * 7919 + 3) % n).astype(np.uint32)
    cb, cn = dev.upload_f32(c), None
    if metric == "l2":
        cn = dev.zeros_f32(k)
        dev.row_norms(cb, k, d, cn)
    lab, sco = dev.zeros_u32(n), dev.zeros_f32(n)
    dev.top1(Mat(dev.bind(x), d), Select(dev.upload_u32(ids), (lo, n)), cb, cn, k, metric, lab, sco)
    ol, os_ = np.zeros(n, np.uint32), np.zeros(n, np.float32)
    O.top1(x, d, c, metric, ids=ids, rows=(lo, n), labels=ol, scores=os_)
    assert np.array_equal(dev.read_u32(lab), ol)
    assert dev.read_f32(sco).tobytes() == os_.tobytes()


@pytest.mark.parametrize("metric", ["ip", "l2"])
@pytest.mark.parametrize("n,d,k", [(300, 64, 2049), (2545, 100, 3000), (257, 33, 9000)])
def test_top1_few_rows_many_centroids(dev, metric, n, d, k):
    """A few row tiles against more than eight tiles of centroids."""
    x, c = _rows(n, d, n), _rows(k, d, k)
    x[: n // 2] = c[np.arange(n // 2) % k] + np.float32(0.3) * x[: n // 2]
    _top1(dev, x, c, metric)


@pytest.mark.parametrize("metric", ["ip", "l2"])
@pytest.mark.parametrize("n,d,k", [(16401, 35, 600), (32768, 33, 80), (32769, 34, 80)])
def test_top1_odd_width_check_blocks(dev, metric, n, d, k):
    """Odd widths: the check's blocks of 16 rows, up to the most that take them,
    and of 32, each with a remainder; near-ties and rows of NaN and zeros."""
    x, c = _rows(n, d, n), _rows(k, d, k)
    c[1:12] = c[0] * (1 + np.float32(1e-6) * np.arange(11, dtype=np.float32)[:, None])
    x[::3] = c[0] + np.float32(0.05) * x[::3]
    x[n - 1], x[n - 2, 1] = 0.0, np.nan
    _top1(dev, x, c, metric)
