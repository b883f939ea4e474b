"""Top-k past 16 neighbours from the one-pass screen's scores (k_screen5's
SCORES and k_select_screened, emh_topk_long.hip): ids and similarities equal
the oracle's bit for bit at the edges of its tiles and of its range, and where
queries fall back to the exact scan (more near-ties than it lists, a NaN row,
values beyond fp16's range)."""

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


def _rows(n, d, seed, centers=40, sigma=0.4):
    return O.contract_mixture(n, d, centers, sigma, True, seed).reshape(n, d)


def _same(g, o, what):
    bad = np.nonzero(g[0] != o[0])[0]
    assert bad.size == 0, f"{what}: {bad.size} ids differ, first at {bad[:4]}"
    assert g[1].tobytes() == o[1].tobytes(), f"{what}: sims differ"


@pytest.mark.parametrize("m,n,d,kk", [
    (2048, 16384, 32, 17),   # whole tiles, the fewest dimensions
    (513, 20001, 100, 128),  # one past a tile each way; a slab in part
    (257, 20737, 193, 512),  # the largest k of the screened selection; scalar loads
    (300, 20479, 164, 513),  # the first beyond it
    (16, 170001, 384, 129),  # the fewest queries
    (65, 4128, 3730, 129),   # the fewest rows a neighbour, many slabs
])
def test_screened_equals_oracle(dev, m, n, d, kk):
    x, q = _rows(n, d, m + n), _rows(m, d, 3 * m + n)
    q[::2] = x[: m : 2] + np.float32(0.01) * q[::2]
    _same(dev.topk(q, x, d, kk, False), O.knn(q, x, d, kk, False), "knn")


def test_screened_self_and_scaled(dev):
    """The rows themselves (exclude_self), and queries and data of other,
    different scales."""
    n, d, kk = 5601, 48, 30
    x = _rows(n, d, 5)
    _same(dev.topk(x, x, d, kk, True), O.knn(x, x, d, kk, True), "self")
    q = _rows(3800, d, 6) * np.float32(3e4)
    xs = x * np.float32(2e-6)
    _same(dev.topk(q, xs, d, kk, False), O.knn(q, xs, d, kk, False), "scaled")


@pytest.mark.parametrize("what", ["ties", "zeros", "nan", "inf", "range"])
def test_screened_falls_back(dev, what):
    n, d, m, kk = 9000, 40, 2800, 50
    x, q = _rows(n, d, 7), _rows(m, d, 8)
    if what == "ties":       # 5,000 equal rows, the best of ten queries
        x[2000:7000] = x[1999]
        q[20:30] = x[1999]
    elif what == "zeros":    # every score +0
        q[3] = 0.0
        q[4] = -0.0
    elif what == "nan":
        x[77] = np.nan
    elif what == "inf":      # +inf and NaN scores, never and always kept
        x[78] = np.inf
        x[79] = -np.inf
    else:                    # one row's element beyond fp16 at the others' scale
        x[80] *= np.float32(1e6)
        q[5] *= np.float32(1e7)
    _same(dev.topk(q, x, d, kk, False), O.knn(q, x, d, kk, False), what)
