"""The work that a user of this framework has it do, as timed cases.

One case is a dict; its "kind" says which public entry points run:

  assign  HipDevice.assign_dev: every row's nearest centroid, all resident
  train   HipDevice.train_dev: a whole training run on resident rows
  fit     Emeans.train, then Emeans.assign, from host arrays
  step    one batch as a caller of the Device ops queues it: the readout
          (row_norms or normalize_rows), top1, scatter_add, ema_update
  topk    HipDevice.topk_dev: exact neighbours, of the rows themselves or of
          other queries
  sweep   auto.sweep: automatic k's seedings, fits and scores

Labels, ids, centroids and scores follow one fixed float order (the fma chain
of each dot product, sums in row order), so two correct implementations give
the same bits; the tolerances of single calls are nevertheless those of 32-bit
sums, with a share of near-ties, and those of whole training runs, whose
trajectories have no meaning between equal and different, are "exact".
"""

import math

import numpy as np
import torch

from emeans_amd import Config, EmaStep, Emeans, HipDevice, Mat, Select
from emeans_amd import auto

_DEV = []


def _dev():
    """One handle, kept as a program keeps it."""
    if not _DEV:
        _DEV.append(HipDevice(0))
    return _DEV[0]


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # A few photos (or queries) against a coarse codebook: latency and launches.
        dict(name="assign_16x384_k256", kind="assign", n=16, d=384, k=256, metric="l2",
             data="mixture"),
        # An ordinary batch of word-vector-sized rows, no round size anywhere.
        dict(name="assign_10007x300_k1000", kind="assign", n=10007, d=300, k=1000, metric="l2",
             data="mixture"),
        # The benchmark's assignment at scale.
        dict(name="assign_2Mx1024_k16384", kind="assign", n=2_000_000, d=1024, k=16384,
             metric="ip", data="sphere"),
        # The smallest whole model, as the user class runs it from host arrays.
        dict(name="fit_20000x64_k32", kind="fit", n=20_000, d=64, k=32, metric="ip",
             data="blobs"),
        # The headline training run.
        dict(name="train_200kx768_k1024", kind="train", n=200_000, d=768, k=1024, metric="l2",
             data="mixture"),
        # Spherical training of sentence-embedding rows with a large codebook.
        dict(name="train_150001x384_k3000", kind="train", n=150_001, d=384, k=3000, metric="ip",
             data="blobs"),
        # One batch of the headline run, driven op by op from outside.
        dict(name="step_16384x768_k1024", kind="step", n=16384, d=768, k=1024, metric="l2",
             data="mixture"),
        # One large batch of an inverted-file codebook's training.
        dict(name="step_65536x1024_k16384", kind="step", n=65536, d=1024, k=16384, metric="ip",
             data="blobs"),
        # Duplicate search over a photo library: the benchmark's all-pairs kNN.
        dict(name="knn_self_500kx384_10", kind="topk", m=0, n=500_000, d=384, kk=10),
        # New photos against a library (the neighbours behind an incremental add).
        dict(name="knn_2000_100kx512_10", kind="topk", m=2000, n=100_000, d=512, kk=10),
        # A retrieval-sized neighbour list, past the screened sixteen.
        dict(name="knn_1000_50kx384_100", kind="topk", m=1000, n=50_000, d=384, kk=100),
        # Automatic k on one group of photos: many small fits and their scores.
        dict(name="sweep_12000x768", kind="sweep", n=12_000, d=768, ks="5,12,20", restarts=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng):
    """Mostly the widths that embeddings have, one in four any width."""
    if rng.random() < 0.25:
        return rng.randint(32, 1100)
    return rng.choice([64, 96, 100, 128, 200, 256, 300, 384, 512, 640, 768, 1024])


def draw(rng):
    kind = rng.choice(["assign", "assign", "train", "train", "step", "topk", "topk", "long",
                       "fit", "sweep"])
    d = _dim(rng)
    metric = rng.choice(["l2", "ip"])
    data = "mixture" if metric == "l2" else "blobs"
    if kind == "assign":
        return dict(kind=kind, n=_log(rng, 1, 400_000), d=d, k=_log(rng, 16, 16_384),
                    metric=metric, data=rng.choice([data, "sphere"]))
    if kind == "train":
        n = _log(rng, 20_000, 200_000)
        return dict(kind=kind, n=n, d=d, k=_log(rng, 16, min(4096, n // 30)), metric=metric,
                    data=data)
    if kind == "step":
        return dict(kind=kind, n=_log(rng, 1024, 65_536), d=d, k=_log(rng, 32, 16_384),
                    metric=metric, data=data)
    if kind == "topk":
        if rng.random() < 0.5:
            return dict(kind=kind, m=0, n=_log(rng, 2000, 150_000), d=d, kk=rng.randint(1, 16))
        return dict(kind=kind, m=_log(rng, 1, 20_000), n=_log(rng, 2000, 200_000), d=d,
                    kk=rng.randint(1, 16))
    if kind == "long":
        return dict(kind="topk", m=_log(rng, 1, 3000), n=_log(rng, 5000, 100_000), d=d,
                    kk=_log(rng, 17, 1000))
    if kind == "fit":
        return dict(kind=kind, n=_log(rng, 5000, 40_000), d=d, k=_log(rng, 8, 128),
                    metric="ip", data="blobs")
    k = rng.randint(4, 10)
    return dict(kind="sweep", n=_log(rng, 2000, 20_000), d=d, ks="%d,%d" % (k, 2 * k),
                restarts=rng.choice([2, 4]))


# ----------------------------------------------------------------- the inputs
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(1_000_003 * int(seed) + salt)
    return g


def _unit(x):
    return x.div_(x.norm(dim=1, keepdim=True).clamp_min_(1e-30))


def _rows(n, d, comps, data, seed):
    """(rows, component means), float32 on the GPU. mixture: a Gaussian mixture
    with Zipf(1.1) weights, means ~N(0, I), diagonal std ~U(0.2, 1); blobs:
    unit rows of equal-sized blobs, the rows' noise half as long as a mean;
    sphere: unit rows in no clusters (the means are unit rows too)."""
    g = _gen(seed, 1)
    means = torch.randn(comps, d, generator=g, device="cuda")
    if data == "sphere":
        x = torch.empty(n, d, device="cuda")
        for a in range(0, n, 262_144):
            x[a:a + 262_144] = _unit(torch.randn(min(n - a, 262_144), d, generator=g,
                                                 device="cuda"))
        return x, _unit(means)
    if data == "mixture":
        w = torch.arange(1, comps + 1, device="cuda", dtype=torch.float32).pow_(-1.1)
        lab = torch.multinomial(w, n, replacement=True, generator=g)
        std = torch.rand(comps, d, generator=g, device="cuda").mul_(0.8).add_(0.2)
        x = torch.randn(n, d, generator=g, device="cuda").mul_(std[lab]).add_(means[lab])
        return x, means
    _unit(means)
    lab = torch.randint(0, comps, (n,), generator=g, device="cuda")
    x = torch.randn(n, d, generator=g, device="cuda").mul_(0.5 / math.sqrt(d)).add_(means[lab])
    return _unit(x), means


def _near_duplicates(n, d, seed):
    """Unit rows, one in twenty a copy of another plus a little noise."""
    x, _ = _rows(n, d, 1, "sphere", seed)
    g = _gen(seed, 2)
    dst = torch.randperm(n, generator=g, device="cuda")[:n // 20]
    src = torch.randint(0, n, (dst.numel(),), generator=g, device="cuda")
    x[dst] = _unit(x[src] + 0.01 * torch.randn(dst.numel(), d, generator=g, device="cuda"))
    return x


def _inputs(case, seed):
    """The case's tensors, from the seed alone."""
    kind, d = case["kind"], case["d"]
    if kind == "topk":
        x = _near_duplicates(case["n"], d, seed)
        if case["m"] == 0:
            return dict(x=x)
        g = _gen(seed, 3)
        m = case["m"]
        # Half of the new rows are near a row of the library.
        src = torch.randint(0, case["n"], (m,), generator=g, device="cuda")
        q = _unit(torch.randn(m, d, generator=g, device="cuda"))
        q[::2] = _unit(x[src[::2]] + 0.02 * torch.randn(q[::2].shape, generator=g, device="cuda"))
        return dict(x=x, q=q)
    if kind == "sweep":
        x, _ = _rows(case["n"], d, 12, "blobs", seed)
        return dict(x=x)
    k = case["k"]
    comps = k
    x, means = _rows(case["n"], d, comps, case["data"], seed)
    if kind in ("train", "fit"):
        return dict(x=x)
    g = _gen(seed, 4)
    # Centroids part of the way through a training: a row of their cluster
    # mixed into its mean.
    noise = torch.randn(k, d, generator=g, device="cuda")
    if case["data"] == "sphere":
        c = means
    elif case["data"] == "mixture":
        c = means + 0.1 * noise
    else:
        c = _unit(means + (0.1 / math.sqrt(d)) * noise)
    return dict(x=x, c=c.contiguous())


def prepare(case, seed):
    case = dict(case)
    dev = _dev()
    t = _inputs(case, seed)
    kind, d = case["kind"], case["d"]
    s = dict(case=case, dev=dev, t=t)
    f = lambda *shape: torch.zeros(*shape, device="cuda")  # noqa: E731
    u = lambda *shape: torch.zeros(*shape, dtype=torch.int32, device="cuda")  # noqa: E731
    out = {}
    if kind == "assign":
        out = dict(labels=u(case["n"]), scores=f(case["n"]))
    elif kind == "train":
        s["config"] = Config(d=d, k=case["k"], spherical=case["metric"] == "ip", seed=int(seed))
        out = dict(centroids=f(case["k"], d))
    elif kind == "fit":
        s["config"] = Config(d=d, k=case["k"], spherical=True, seed=int(seed))
        s["x"] = t.pop("x").cpu().numpy()
    elif kind == "step":
        n, k = case["n"], case["k"]
        # The batch's rows in the order of a permutation, as an epoch draws them.
        t["ids"] = torch.randperm(n, generator=_gen(seed, 5), device="cuda").to(torch.int32)
        out = dict(labels=u(n), scores=f(n), sums=f(k, d), counts=u(k),
                   readout=f(k, d) if case["metric"] == "ip" else f(k), positions=t["c"].clone(),
                   usage=torch.full((k,), n / k, device="cuda"), acc=f(k, d))
        s["alpha"] = EmaStep.new(0.25)
    elif kind == "topk":
        m = case["m"] or case["n"]
        out = dict(ids=u(m, case["kk"]), sims=f(m, case["kk"]))
    elif kind == "sweep":
        s["x"] = t.pop("x").cpu().numpy()
        s["xb"] = dev.bind(s["x"])
        s["cfg"] = auto.AutoConfig(restarts=case["restarts"], seed=int(seed))
        s["ks"] = [int(v) for v in case["ks"].split(",")]
    torch.cuda.synchronize()
    # Views of the caller's own device memory.
    for name, v in list(t.items()) + list(out.items()):
        s["b_" + name] = dev.wrap(v.data_ptr(), v.numel(), int(v.dtype == torch.int32))
    s["out"] = out
    return s


# ---------------------------------------------------------------- the one pass
def run(s):
    case, dev, out = s["case"], s["dev"], s["out"]
    kind, d = case["kind"], case["d"]
    if kind == "assign":
        dev.assign_dev(s["b_x"], case["n"], d, s["b_c"], case["k"], case["metric"],
                       s["b_labels"], s["b_scores"])
        return out
    if kind == "train":
        cent, info = dev.train_dev(s["b_x"], case["n"], s["config"],
                                   centroids_out=s["b_centroids"])
        return dict(centroids=cent, positions=info["positions"], usage=info["usage"],
                    labels=info["labels"], objective=[e.obj for e in info["stats"]],
                    on_device=out["centroids"])
    if kind == "fit":
        model = Emeans(s["config"], dev)
        got = model.train(s["x"])
        a = model.assign(s["x"])
        return dict(centroids=got.centroids, train_labels=got.labels, labels=a.labels,
                    scores=a.scores)
    if kind == "step":
        n, k = case["n"], case["k"]
        x, sel = Mat(s["b_x"], d), Select(s["b_ids"], (0, n))
        if case["metric"] == "ip":
            dev.normalize_rows(s["b_positions"], k, d, s["b_readout"])
            cent, cnorm = s["b_readout"], None
        else:
            dev.row_norms(s["b_positions"], k, d, s["b_readout"])
            cent, cnorm = s["b_positions"], s["b_readout"]
        dev.top1(x, sel, cent, cnorm, k, case["metric"], s["b_labels"], s["b_scores"])
        dev.scatter_add(x, sel, s["b_labels"], k, s["b_sums"], s["b_counts"], s["b_acc"])
        dev.ema_update(s["b_positions"], s["b_usage"], s["b_sums"], s["b_counts"], k, d,
                       s["alpha"])
        return out
    if kind == "topk":
        q = s["b_x"] if case["m"] == 0 else s["b_q"]
        dev.topk_dev(q, case["m"] or case["n"], s["b_x"], case["n"], d, case["kk"],
                     case["m"] == 0, s["b_ids"], s["b_sims"])
        return out
    got, picks = auto.sweep(dev, s["x"], s["xb"], s["ks"], s["cfg"], 0)
    return dict(scores=[[v.k_eff, v.silhouette, v.calinski_harabasz, v.davies_bouldin,
                         v.objective] for v, _ in got],
                centroids=[f.centroids for _, f in got],
                labels=[dev.read_u32(f.labels) for _, f in got], picks=list(picks))


# ---------------------------------------------------- its size and its answer
def work(case):
    kind, d = case["kind"], case["d"]
    if kind == "topk":
        n, m = case["n"], case["m"] or case["n"]
        return {"bytes": 4 * n * d + (4 * m * d if case["m"] else 0) + 8 * m * case["kk"],
                "flops": 2 * m * n * d}
    if kind == "sweep":
        # Per fit five passes of training and one of assignment, per seeding
        # one row's dots with all rows for each pick, and the scores.
        n, r = case["n"], case["restarts"]
        ks = [int(v) for v in case["ks"].split(",")]
        flops = sum(6 * r * 2 * n * k * d + 4 * n * k * d for k in ks)
        return {"bytes": 4 * n * d * (1 + len(ks) * r),
                "flops": flops + r * max(ks) * 2 * n * d}
    n, k = case["n"], case["k"]
    if kind == "assign":
        return {"bytes": 4 * (n * d + k * d + 2 * n), "flops": 2 * n * k * d}
    if kind == "step":
        # Rows by id, labels and scores out; the moved state read and written.
        return {"bytes": 4 * (n * d + 3 * n + 5 * k * d + 4 * k), "flops": 2 * n * k * d + n * d}
    passes = 5 if kind == "train" else 6
    return {"bytes": 4 * (passes * n * d + 3 * k * d + n), "flops": passes * 2 * n * k * d}


def tolerance(case):
    if case["kind"] in ("train", "fit", "sweep"):
        return "exact"
    # Four times the largest seen against 64 bits over the listed cases and 30
    # drawn ones: 2.7e-6 on scores (chains of 901 products that cancel in the
    # squared distance), 1.4e-3 of the ids of long neighbour lists (two
    # neighbours in near-tie), 4.5e-6 of two million labels.
    if case["kind"] == "topk":
        return {"rel": 3e-6, "differ": 6e-3}
    return {"rel": 1.1e-5, "differ": 2e-5}


def _scores64(q, c, metric):
    s = q.double() @ c.double().t()
    if metric == "ip":
        return s
    c2 = c.double().square().sum(1)
    return s.mul_(2.0).sub_(c2[None, :])  # larger is nearer


def _top1_64(x, c, metric):
    labels = torch.empty(x.shape[0], dtype=torch.int64, device="cuda")
    scores = torch.empty(x.shape[0], dtype=torch.float64, device="cuda")
    rows = max(1, min(x.shape[0], (1 << 28) // c.shape[0]))
    for a in range(0, x.shape[0], rows):
        xa = x[a:a + rows]
        v, i = _scores64(xa, c, metric).max(1)
        labels[a:a + rows] = i
        if metric == "l2":
            v = (xa.double().square().sum(1) - v).clamp_min_(0.0)
        scores[a:a + rows] = v
    return labels, scores


def exact(case, seed):
    kind = case["kind"]
    if kind in ("train", "fit", "sweep"):
        # A training run's revivals and its choice of best fit follow the
        # float32 trajectory: in 64 bits it is another run.
        return None
    if work(case)["flops"] > 1.2e14:
        return None
    t = _inputs(case, seed)
    if kind == "assign":
        labels, scores = _top1_64(t["x"], t["c"], case["metric"])
        return dict(labels=labels, scores=scores)
    if kind == "topk":
        x = t["x"]
        q = t.get("q", x)
        ids, sims = [], []
        rows = max(1, min(q.shape[0], (1 << 27) // x.shape[0]))
        for a in range(0, q.shape[0], rows):
            s = _scores64(q[a:a + rows], x, "ip")
            if case["m"] == 0:
                r = torch.arange(s.shape[0], device="cuda")
                s[r, r + a] = -math.inf
            v, i = s.topk(case["kk"], dim=1)
            ids.append(i)
            sims.append(v)
        return dict(ids=torch.cat(ids), sims=torch.cat(sims))
    n, k, metric = case["n"], case["k"], case["metric"]
    x = t["x"][torch.randperm(n, generator=_gen(seed, 5), device="cuda")]
    c = t["c"].double()
    if metric == "ip":
        readout = c / c.norm(dim=1, keepdim=True)
        labels, scores = _top1_64(x, readout, metric)
    else:
        readout = c.square().sum(1)
        labels, scores = _top1_64(x, t["c"], metric)
    sums = torch.zeros(k, case["d"], dtype=torch.float64, device="cuda")
    for a in range(0, n, 16384):
        sums.index_add_(0, labels[a:a + 16384], x[a:a + 16384].double())
    counts = torch.bincount(labels, minlength=k).double()
    alpha = float(np.float32(0.25))
    usage0 = float(np.float32(n / k))
    usage = usage0 * (1.0 - alpha) + alpha * counts
    moved = (c * (usage0 * (1.0 - alpha)) + alpha * sums) / usage[:, None]
    positions = torch.where(counts[:, None] > 0, moved, c)
    return dict(labels=labels, scores=scores, sums=sums, counts=counts, readout=readout,
                positions=positions, usage=usage, acc=sums.clone())
