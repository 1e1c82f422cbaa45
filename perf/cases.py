"""Performance cases of the polygon-join library.

Each case is a dict of plain values.  "path" names what a user's program does:

  intersect     exact intersect of a resident set's candidate pairs
                (Device.intersect), bits on the host
  approx        intersect -a: the reference heuristic, or the MLP with an
                exact fallback band
  within        within-distance self-join of a resident -h set
  intersection  crossing counts and areas of A n B of the candidate pairs
  join          the whole query from host polygons: raster build, candidate
                pairs and intersect on the device
  join_within   the same for the within-distance self-join (-h raster build)
  train         Adam training of the 80-128-128-2 MLP on labelled pairs

and "data" the polygons: "star" (the plain intersect workload: 50..500
vertices, 2,000 per side and [0,100]^2 box, k boxes' worth in one larger box),
"lakes" (complex polygons of 1,000..200,000 vertices against lakes of
20..2,000, at the density of 20,000 x 500,000 in [0,40]^2), or one set of lakes
at the density of 300,000 in [0,20]^2 with a 10 km threshold.  Larger sets
keep the density and grow the box, so a case's work grows with its size alone.
A query takes its first _window(case) candidate pairs, the executables' batch
window (-b): the sets have a few more of them, a seed's number of its own.
"""
from __future__ import annotations

import numpy as np

from farm_amd import capi

NFEAT = 80
HIDDEN = 128
SHAPES = [(NFEAT, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (HIDDEN, 2), (2,)]


def listed() -> list[dict]:
    return [
        # one plain-workload query: 2,000 x 2,000 small polygons, ~3,900
        # pairs; what an interactive caller sends, bound by latency
        {"name": "intersect_star_1", "path": "intersect", "data": "star", "k": 1, "vpr": 10, "tile": 0},
        # a batch of the learned part's evaluation (~0.8 M pairs)
        {"name": "intersect_star_200", "path": "intersect", "data": "star", "k": 200, "vpr": 10, "tile": 0},
        # complex x lakes, an ordinary batch (~0.5 M pairs), with the
        # launch configuration the autotuner persists for this shape
        {"name": "intersect_lakes_mid", "path": "intersect", "data": "lakes", "na": 401, "nb": 9973, "vpr": 256,
         "tile": 8},
        # complex x lakes, a large batch (~6 M pairs): the headline workload
        {"name": "intersect_lakes_large", "path": "intersect", "data": "lakes", "na": 4000, "nb": 100000, "vpr": 256,
         "tile": 8},
        # -a with a network: features and inference for every pair, the
        # undecided band refined exactly
        {"name": "approx_learned_star_200", "path": "approx", "learned": True, "k": 200, "vpr": 10},
        # a small within-distance self-join (one town's lakes)
        {"name": "within_300", "path": "within", "n": 300, "vpr": 10},
        # an ordinary within-distance self-join (~6 M ordered pairs)
        {"name": "within_30000", "path": "within", "n": 30000, "vpr": 10},
        # areas of one plain-workload query's pairs
        {"name": "intersection_star_1", "path": "intersection", "data": "star", "k": 1, "vpr": 10},
        # areas of complex x lakes (~0.6 M pairs)
        {"name": "intersection_lakes", "path": "intersection", "data": "lakes", "na": 500, "nb": 10000, "vpr": 256},
        # new polygons: raster build, candidates and intersect in one go
        {"name": "join_lakes", "path": "join", "na": 400, "nb": 10000, "vpr": 256},
        # new lakes: -h raster build, candidates and within in one go
        {"name": "join_within_3000", "path": "join_within", "n": 3000, "vpr": 10},
        # two epochs of training on labelled pairs
        {"name": "train_65536", "path": "train", "rows": 65536, "batch": 2048, "epochs": 2},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng) -> dict:
    path = rng.choice(["intersect_star", "intersect_lakes", "approx", "within", "intersection_star",
                       "intersection_lakes", "join", "join_within", "train"])
    vpr = rng.choice([10, 10, 16, 33])
    if path == "intersect_star":
        return {"path": "intersect", "data": "star", "k": _log_int(rng, 1, 300), "vpr": vpr,
                "tile": rng.choice([0, 8])}
    if path == "intersect_lakes":
        na = _log_int(rng, 41, 2500)
        return {"path": "intersect", "data": "lakes", "na": na, "nb": na * 25 + rng.randrange(25),
                "vpr": rng.choice([64, 100, 256]), "tile": rng.choice([0, 8, 8])}
    if path == "approx":
        return {"path": "approx", "learned": rng.random() < 0.5, "k": _log_int(rng, 1, 300), "vpr": vpr}
    if path == "within":
        return {"path": "within", "n": _log_int(rng, 100, 25000), "vpr": vpr}
    if path == "intersection_star":
        return {"path": "intersection", "data": "star", "k": _log_int(rng, 1, 100), "vpr": vpr}
    if path == "intersection_lakes":
        na = _log_int(rng, 25, 400)
        return {"path": "intersection", "data": "lakes", "na": na, "nb": na * 20 + rng.randrange(20),
                "vpr": rng.choice([64, 100, 256])}
    if path == "join":
        na = _log_int(rng, 20, 1000)
        return {"path": "join", "na": na, "nb": na * 25 + rng.randrange(25), "vpr": rng.choice([64, 100, 256])}
    if path == "join_within":
        return {"path": "join_within", "n": _log_int(rng, 100, 9000), "vpr": vpr}
    batch = rng.choice([512, 1000, 2048, 4096])
    return {"path": "train", "rows": _log_int(rng, 6000, 130000), "batch": batch, "epochs": rng.choice([1, 2, 3])}


# ---------------------------------------------------------------- the data
def _star(k: int, seed: int):
    side = 100.0 * float(np.sqrt(k))
    kw = dict(nv_lo=50, nv_hi=500, r_mu=float(np.log(0.5)), r_sigma=0.5, amp=0.4)
    a = capi.HostSet.star_polygons(2 * seed + 1, 2000 * k, 0.0, side, **kw)
    b = capi.HostSet.star_polygons(2 * seed + 2, 2000 * k, 0.0, side, **kw)
    return a, b


def _lakes(na: int, nb: int, seed: int):
    side = 40.0 * float(np.sqrt(nb / 500000.0))
    return (capi.HostSet.complex_polygons(2 * seed + 1, na, 0.0, side),
            capi.HostSet.lake_polygons(2 * seed + 2, nb, 0.0, side))


def _lake_set(n: int, seed: int):
    return capi.HostSet.lake_polygons(2 * seed + 1, n, 0.0, 20.0 * float(np.sqrt(n / 300000.0)))


def _two_sets(case: dict, seed: int):
    if case.get("data", "star") == "star" and "k" in case:
        return _star(case["k"], seed)
    return _lakes(case["na"], case["nb"], seed)


def _overlapping(na: int, nb: int, reach: float, side: float) -> float:
    """Expected pairs of na and nb boxes whose centres, uniform in a box of
    this side, lie within reach of each other on both axes."""
    r = min(reach / side, 1.0)
    return na * nb * (2.0 * r - r * r) ** 2


def _window(case: dict) -> int:
    """Candidate pairs of one query: somewhat fewer than nearly every seed's
    sets have."""
    if "k" in case:
        return int(0.93 * 4240 * case["k"])
    if "n" in case:
        n = case["n"]
        return int(0.78 * _overlapping(n, n - 1, 0.304, 20.0 * float(np.sqrt(n / 300000.0))))
    na, nb = case["na"], case["nb"]
    return int(0.7 * _overlapping(na, nb, 1.35, 40.0 * float(np.sqrt(nb / 500000.0))))


def _whole(out: np.ndarray, n: int) -> np.ndarray:
    """out, with zeros for the pairs a seed's sets are short of n."""
    return out if len(out) == n else np.concatenate([out, np.zeros((n - len(out),) + out.shape[1:], out.dtype)])


def _weights(seed: int) -> np.ndarray:
    """He-uniform weights and zero biases, as one flat vector."""
    rng = np.random.default_rng(seed)
    parts = []
    for shape in SHAPES:
        if len(shape) == 2:
            lim = np.sqrt(6.0 / shape[0])
            parts.append(rng.uniform(-lim, lim, size=shape).astype(np.float32).reshape(-1))
        else:
            parts.append(np.zeros(shape, np.float32))
    return np.concatenate(parts)


def _training_data(case: dict, seed: int):
    """Normalised features, the bits and log costs of a noisy teacher."""
    rng = np.random.default_rng(seed)
    n = case["rows"]
    x = rng.standard_normal((n, NFEAT)).astype(np.float32)
    t = rng.standard_normal((NFEAT, 2)).astype(np.float32) / np.float32(np.sqrt(NFEAT))
    z = x @ t
    y = (z[:, 0] + 0.5 * rng.standard_normal(n) > 0).astype(np.float32)
    c = np.maximum(0.0, 10.0 + 3.0 * z[:, 1] + rng.standard_normal(n)).astype(np.float32)
    return x, y, c, _weights(seed + 1)


# ---------------------------------------------------------------- the calls
def prepare(case: dict, seed: int) -> dict:
    path = case["path"]
    st = {"case": case}
    dev = capi.Device(0)
    st["dev"] = dev
    if path == "train":
        st["x"], st["y"], st["c"], st["w"] = _training_data(case, seed)
        return st
    if path in ("within", "join_within"):
        s = _lake_set(case["n"], seed)
        st["set"] = s
        if path == "within":
            dev.rasterize_hostset(s, case["vpr"], 1)
            m = s.mbbs()
            dev.generate_pairs(m, m, expand_km=10.0, skip_self=True)
        return st
    a, b = _two_sets(case, seed)
    st["a"], st["b"] = a, b
    both = capi.HostSet.concat(a, b)
    st["set"] = both
    if path == "join":
        dev.set_tuning(8, 16, 4)
        return st
    dev.rasterize_hostset(both, case["vpr"])
    dev.generate_pairs(a.mbbs(), b.mbbs(), a_base=0, b_base=len(a))
    if case.get("tile"):
        dev.set_tuning(case["tile"], 16, 4)
    if case.get("learned"):
        feat, _ = dev.pair_features()
        mu, sd = feat.mean(0), feat.std(0)
        sd = np.where(sd > 1e-6, sd, 1.0)
        dev.mlp_set_params(_weights(seed + 1), np.concatenate([mu, 1.0 / sd]).astype(np.float32))
    return st


def run(st: dict):
    case, dev = st["case"], st["dev"]
    path = case["path"]
    if path == "train":
        dev.mlp_set_params(st["w"])
        losses = dev.mlp_train(st["x"], st["y"], st["c"], case["epochs"], case["batch"], 2e-3, 0.05, 1)
        return losses, dev.mlp_get_params()
    if path == "join":
        dev.rasterize_hostset(st["set"], case["vpr"])
        dev.generate_pairs(st["a"].mbbs(), st["b"].mbbs(), a_base=0, b_base=len(st["a"]))
    elif path == "join_within":
        dev.rasterize_hostset(st["set"], case["vpr"], 1)
        m = st["set"].mbbs()
        dev.generate_pairs(m, m, expand_km=10.0, skip_self=True)
    n = _window(case)
    end = min(n, dev.npairs)
    if path in ("intersect", "join"):
        return _whole(dev.intersect(0, end, mode=capi.MODE_EXACT_BATCHED).bits, n)
    if path == "approx":
        if case["learned"]:
            return _whole(dev.intersect(0, end, mode=capi.MODE_APPROX_LEARNED, accept=0.25, reject=-0.25).bits, n)
        return _whole(dev.intersect(0, end, mode=capi.MODE_APPROX_HEURISTIC).bits, n)
    if path == "intersection":
        counts, area, _ = dev.intersection_area(0, end)
        return _whole(counts, n), _whole(area, n)
    bits, dist, _ = dev.within(10.0, 0, end)
    return _whole(bits, n), _whole(dist, n)


# ---------------------------------------------------------------- the work
def work(case: dict) -> dict:
    """Each vertex, pair id and result moved once; one 42-operation segment
    test (22 double operations of a point-segment distance for within) per
    edge of either ring inside the other's box.  The counts are the
    distributions' means."""
    path = case["path"]
    if path == "train":
        steps = max(case["rows"] // case["batch"], 1) * case["epochs"]
        macs = NFEAT * HIDDEN + HIDDEN * HIDDEN + 2 * HIDDEN
        rows = steps * min(case["batch"], case["rows"])
        return {"bytes": 4.0 * case["rows"] * (NFEAT + 2), "flops": 6.0 * macs * rows}
    if path in ("within", "join_within"):
        n = case["n"]
        pairs = float(_window(case))
        # both rings' edges nearest the other ring: a tenth of them
        return {"bytes": 8.0 * 1011 * n + 17.0 * pairs, "flops": 22.0 * 202 * pairs}
    if "k" in case:
        k = case["k"]
        verts, edges = 2.0 * 2000 * k * 276, 140.0
    else:
        na, nb = case["na"], case["nb"]
        verts, edges = 4268.0 * na + 1011.0 * nb, 1400.0
    pairs = float(_window(case))
    out = 28.0 if path == "intersection" else 1.0
    if path == "approx":  # a pair is decided from its pixels
        return {"bytes": 2.0 * 2000 * case["k"] * (128 + 28) + 9.0 * pairs,
                "flops": (2.0 * (NFEAT * HIDDEN + HIDDEN * HIDDEN + 2 * HIDDEN) if case["learned"] else 20.0) * pairs}
    return {"bytes": 8.0 * verts + (8.0 + out) * pairs, "flops": 42.0 * edges * pairs}


# ---------------------------------------------------------------- 64 bits
def _shuffles(n: int, epochs: int, seed: int):
    """The training's row orders: Fisher-Yates over a 64-bit LCG."""
    mask = (1 << 64) - 1
    s = (seed * 6364136223846793005 + 1442695040888963407) & mask
    for _ in range(epochs):
        perm = list(range(n))
        for i in range(n - 1, 0, -1):
            s = (s * 6364136223846793005 + 1442695040888963407) & mask
            j = (s >> 33) % (i + 1)
            perm[i], perm[j] = perm[j], perm[i]
        yield np.asarray(perm)


def exact(case: dict, seed: int):
    """Training in float64.  The queries answer with whole numbers, or with
    distances and areas whose value is set by the binary32 predicates of the
    reference: those have no 64-bit counterpart."""
    if case["path"] != "train":
        return None
    x, y, c, w = _training_data(case, seed)
    x, y, c = x.astype(np.float64), y.astype(np.float64), c.astype(np.float64)
    w = w.astype(np.float64)
    off = np.cumsum([0] + [int(np.prod(s)) for s in SHAPES])
    view = lambda v, i: v[off[i]:off[i + 1]].reshape(SHAPES[i])  # noqa: E731
    lr, lam, b1, b2, eps = 2e-3, 0.05, 0.9, 0.999, 1e-8
    m, v, t = np.zeros_like(w), np.zeros_like(w), 0
    n, batch = case["rows"], min(case["batch"], case["rows"])
    losses = []
    for perm in _shuffles(n, case["epochs"], 1):
        total, nb = 0.0, 0
        for b0 in range(0, n - batch + 1, batch):
            ix = perm[b0:b0 + batch]
            X, Y, Cc = x[ix], y[ix], c[ix]
            h1 = np.maximum(X @ view(w, 0) + view(w, 1), 0)
            h2 = np.maximum(h1 @ view(w, 2) + view(w, 3), 0)
            z = h2 @ view(w, 4) + view(w, 5)
            e = z[:, 1] - Cc
            total += float(np.mean(np.maximum(z[:, 0], 0) - z[:, 0] * Y + np.log1p(np.exp(-np.abs(z[:, 0]))))
                           + lam * np.mean(e * e))
            nb += 1
            dz = np.stack([(1.0 / (1.0 + np.exp(-z[:, 0])) - Y) / batch, 2 * lam * e / batch], 1)
            d2 = (dz @ view(w, 4).T) * (h2 > 0)
            d1 = (d2 @ view(w, 2).T) * (h1 > 0)
            g = np.concatenate([(X.T @ d1).reshape(-1), d1.sum(0), (h1.T @ d2).reshape(-1), d2.sum(0),
                                (h2.T @ dz).reshape(-1), dz.sum(0)])
            t += 1
            m = b1 * m + (1 - b1) * g
            v = b2 * v + (1 - b2) * g * g
            w = w - lr * (m / (1 - b1 ** t)) / (np.sqrt(v / (1 - b2 ** t)) + eps)
        losses.append(total / max(nb, 1))
    return np.asarray(losses), w
