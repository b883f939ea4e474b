"""scatter_add past the small counting sort: more than 8,192 clusters
(positions dropped into their cluster's run in any order, then ranked, runs of
up to 512, or found by a walk) and more than 65,536 positions (chunks of several
rounds). Sums in selection order, so bit-equal to the oracle."""

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


@pytest.mark.parametrize("n,k,d,lo", [
    (20000, 9000, 36, 0),    # sizes around one register a lane and the ranked runs' end
    (20001, 16384, 33, 5),   # an odd width, positions that do not start at 0
    (70000, 100, 20, 3),     # many positions, few clusters
    (66000, 8193, 16, 0),
])
def test_scatter_order(dev, n, k, d, lo):
    from emeans_amd import Mat, Select
    g = np.random.default_rng(n + k)
    x = g.standard_normal((n, d)).astype(np.float32)
    labels = g.integers(0, k, n).astype(np.uint32)
    at = 0
    for j, c in enumerate((0, 1, 63, 64, 65, 511, 512, 513, 4000)):
        labels[labels == j] = k - 1
        labels[at:at + c] = j
        at += c
    labels = g.permutation(labels)
    ids = g.permutation(n).astype(np.uint32)
    sums, counts = dev.zeros_f32(k * d), dev.zeros_u32(k)
    acc0 = g.standard_normal(k * d).astype(np.float32)
    acc = dev.upload_f32(acc0)
    dev.scatter_add(Mat(dev.bind(x), d), Select(dev.upload_u32(ids), (lo, n)),
                    dev.upload_u32(labels), k, sums, counts, acc)
    oacc = acc0.copy()
    os_, oc = O.scatter_add(x, d, labels, k, ids=ids, rows=(lo, n), acc=oacc)
    assert np.array_equal(dev.read_u32(counts), oc)
    assert dev.read_f32(sums).tobytes() == os_.tobytes()
    assert dev.read_f32(acc).tobytes() == oacc.tobytes()


@pytest.mark.parametrize("n,k,d,lo,skew", [
    (65537, 1, 8, 0, 0),         # one past the one-round chunks
    (131072, 16, 12, 0, 1),      # two whole rounds
    (131079, 1024, 20, 6, 3),    # one position past them, from an odd start
    (200000, 8192, 8, 0, 1),
    (300001, 100, 33, 1, 2),     # a last chunk of a part of a round
])
def test_scatter_rounds(dev, n, k, d, lo, skew):
    from emeans_amd import Mat, Select
    g = np.random.default_rng(n + k)
    x = g.standard_normal((n, d)).astype(np.float32)
    labels = np.minimum((k * g.random(n) ** (1 + 2 * skew)), k - 1).astype(np.uint32)
    ids = g.integers(0, n, n).astype(np.uint32)
    sums, counts = dev.zeros_f32(k * d), dev.zeros_u32(k)
    lb, xb = dev.upload_u32(labels), dev.bind(x)
    for i in (None, ids):
        dev.scatter_add(Mat(xb, d), Select(None if i is None else dev.upload_u32(i), (lo, n)), lb,
                        k, sums, counts, None)
        os_, oc = O.scatter_add(x, d, labels, k, ids=i, rows=(lo, n))
        assert np.array_equal(dev.read_u32(counts), oc)
        assert dev.read_f32(sums).tobytes() == os_.tobytes()


def test_scatter_rounds_bad_label(dev):
    from emeans_amd import Mat, Select
    n, k, d = 140000, 50, 4
    labels = np.zeros(n, np.uint32)
    labels[131000] = k
    with pytest.raises(Exception):
        dev.scatter_add(Mat(dev.bind(np.ones((n, d), np.float32)), d), Select(None, (0, n)),
                        dev.upload_u32(labels), k, dev.zeros_f32(k * d), dev.zeros_u32(k), None)
        dev.read_u32(dev.zeros_u32(1))
