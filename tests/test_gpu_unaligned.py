"""Wrapped buffers that start at any float: rows and centroids 4, 8 and 12
bytes past a multiple of 16, on every route that copies 16 bytes a lane
(k_small1, k_queued1 as a direct selection and behind the screen's check, the
training batches that tally) and on those around them; bit-equal to the
oracle."""

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


def _at(dev, a, off):
    """a on the device, `off` floats past the start of its allocation (kept by
    the first of the two returned)."""
    whole = dev.upload_f32(np.concatenate([np.zeros(off, np.float32), a.reshape(-1)]))
    return whole, dev.wrap(whole.ptr + 4 * off, a.size, 0)


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("n,d,k", [
    (700, 36, 20),      # k_small1
    (5000, 100, 40),
    (9000, 32, 40),     # past its rows: the 128 x 128 screen
    (300, 772, 100),    # k_queued1, phases
    (4000, 64, 600),    # the screens, and the rows their checks queue
    (40000, 64, 80),
])
def test_unaligned_top1(dev, n, d, k, metric, off):
    from emeans_amd import Mat, Select
    g = np.random.default_rng(n + k + off)
    x = g.standard_normal((n, d)).astype(np.float32)
    c = g.standard_normal((k, d)).astype(np.float32)
    c[k // 2] = c[0]
    c[1:1 + k // 2:2] = c[0] * np.float32(1 + 1e-7)  # crowds: rows for the exact scan
    xw, xb = _at(dev, x, off)
    cw, cb = _at(dev, c, 4 - off)
    cn = None
    if metric == "l2":
        cn = dev.zeros_f32(k)
        dev.row_norms(cb, k, d, cn)
    lab, sc = dev.zeros_u32(n), dev.zeros_f32(n)
    dev.top1(Mat(xb, d), Select(None, (0, n)), cb, cn, k, metric, lab, sc)
    ol, os_ = O.top1(x, d, c, metric)
    assert np.array_equal(dev.read_u32(lab), ol)
    assert dev.read_f32(sc).tobytes() == os_.tobytes()
    del xw, cw


@pytest.mark.parametrize("spherical", [False, True])
@pytest.mark.parametrize("n,batch,k,d", [(3100, 1000, 12, 64), (5000, 2040, 64, 32),
                                         (9000, 4100, 40, 36)])
def test_unaligned_train(dev, n, batch, k, d, spherical):
    from emeans_amd import Config
    g = np.random.default_rng(n + k)
    x = g.standard_normal((n, d)).astype(np.float32)
    if spherical:
        x /= np.linalg.norm(x, axis=1, keepdims=True)
    cfg = Config(d=d, k=k, nepochs=3, batch_size=batch, spherical=spherical, seed=5)
    whole, xb = _at(dev, x, 1)
    cent, info = dev.train_dev(xb, n, cfg)
    o = O.train(x, d, k, nepochs=cfg.nepochs, batch_size=cfg.batch_size, alpha0=cfg.alpha0,
                batch_law=cfg.batch_law, seed=cfg.seed, spherical=cfg.spherical,
                unused_threshold=cfg.unused_threshold)
    assert np.array_equal(info["labels"], o["labels"])
    assert info["positions"].tobytes() == o["positions"].tobytes()
    assert cent.tobytes() == o["centroids"].tobytes()
    del whole
