"""A chain per row (k-means++'s dots, internal_scores' f64 squares) and the
exact dots of rows with cluster sums, at the edges of their 16-row groups,
256-column passes, 4-column loads and column tiles: bit-equal to the oracle."""

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


@pytest.mark.parametrize("n,d", [(2, 1), (15, 3), (16, 64), (17, 252), (17, 255), (18, 256), (33, 768), (50, 769),
                                 (100, 1536), (65, 1543)])
def test_row_chain(dev, n, d):
    g = np.random.default_rng(n + d)
    x = g.standard_normal((n, d)).astype(np.float32)
    x /= np.maximum(np.linalg.norm(x, axis=1, keepdims=True), 1e-6)
    xb = dev.bind(x)
    k = min(n, 6)
    assert np.array_equal(dev.kmeans_pp(xb, n, d, k, 7), O.kmeans_pp(x, d, k, 7))
    lab = (np.arange(n) % 3).astype(np.uint32)
    got = dev.internal_scores(xb, n, d, dev.upload_u32(lab), 3)
    want = O.internal_scores(x, d, lab, 3)
    for key in ("silhouette", "calinski_harabasz", "davies_bouldin", "objective"):
        assert got[key] == want[key], key


@pytest.mark.parametrize("nb", [1, 16, 17, 64, 65, 129])
@pytest.mark.parametrize("m,d", [(1, 5), (63, 16), (65, 33), (130, 100)])
def test_dots(dev, m, d, nb):
    g = np.random.default_rng(m + d + nb)
    a = g.standard_normal((m, d)).astype(np.float32)
    b = g.standard_normal((nb, d)).astype(np.float32)
    assert np.array_equal(dev.dots(a, b), O.dots(a, b))
