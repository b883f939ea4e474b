"""scatter_add past the chunked counting sort (more than 8,192 clusters, or
more than 65,536 positions): positions dropped into their cluster's run in any
order, then ranked (runs of up to 512) or found by a walk (longer ones). Sums
in selection order, so bit-equal to the oracle."""

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
    (70000, 100, 20, 3),     # many positions, few clusters: walks
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
