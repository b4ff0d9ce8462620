"""The work that users of lpa_amd have it do, as measurable cases.

A case is a dict of plain values with an "op":

  lp     a label-propagation run as the command-line drivers do it: start
         labels in, `iters` synchronous steps (20, the drivers' default),
         every step's changed count and the final labels out.  The graph is
         already uploaded and scheduled, as in a program that propagates
         several times over one graph.
  encode CGR encoding of a CSR held on the host, and the stream back
         (offline preparation of a file set on the device).
  bfs    BFS relabelling of a CSR held on the host, the step before encoding.
  train  training of the schedule's cost model on recorded samples.
  infer  the cost model's prediction for every vertex of a graph.

Graphs come from the generators that the benchmark and the tests use (R-MAT,
the lattice with dropped edges and shortcuts, the copying model).
"""
import random

import numpy as np

import lpa_amd as L

UNLABELLED = 0xFFFFFFFF
NPARAM = 1443
IN, HID, OUT = 8, 32, 3


def listed():
    return [
        # the smallest calls: a graph of a few thousand vertices, where the
        # number of launches and their latency decide (the smoke run's graph)
        dict(name="lp_rmat12", op="lp", gen="rmat", scale=12, ef=16, T=0, K=1, method="nova", graph=False, semi=False,
             cms_thresh=256, cms_depth=4, cms_width=512, iters=20),
        # a road-like graph: a million vertices of degree 4, almost no label
        # shared by neighbours at the start (the benchmark's lattice)
        dict(name="lp_lattice1024", op="lp", gen="lattice", side=1024, T=0, K=1, method="nova", graph=False, semi=False,
             cms_thresh=0, iters=20),
        # one label vector over a social graph, the drivers' plain use, with
        # the benchmark's sketch for the hubs
        dict(name="lp_rmat20", op="lp", gen="rmat", scale=20, ef=16, T=0, K=1, method="nova", graph=False, semi=False,
             cms_thresh=4096, cms_depth=4, cms_width=1024, iters=20),
        # the largest: eight label vectors at once over R-MAT 22, steps
        # replayed from a captured graph (the benchmark's second workload)
        dict(name="lp_rmat22_k8", op="lp", gen="rmat", scale=22, ef=16, T=0, K=8, method="nova", graph=True, semi=False,
             cms_thresh=4096, cms_depth=4, cms_width=1024, iters=20),
        # the two-kernel method: decode the stream, then propagate, each step
        dict(name="lp_cglp_rmat19", op="lp", gen="rmat", scale=19, ef=16, T=0, K=1, method="cglp", graph=False,
             semi=False, cms_thresh=0, iters=20),
        # semi-supervised labelling with many vectors: 1 % of the vertices
        # seeded from 100 classes, exact counts, replayed steps
        dict(name="lp_semi_rmat17_k64", op="lp", gen="rmat", scale=17, ef=16, T=0, K=64, method="nova", graph=True,
             semi=True, cms_thresh=0, iters=20),
        # a web-like directed graph whose small vertices stay uncompressed
        dict(name="lp_copying", op="lp", gen="copying", n=300_007, T=32, K=1, method="nova", graph=False, semi=False,
             cms_thresh=8192, cms_depth=4, cms_width=2048, iters=20),
        # an odd number of vectors over a ragged graph: rows of five labels
        # that no wide load fits
        dict(name="lp_copying_k5", op="lp", gen="copying", n=50_021, T=16, K=5, method="nova", graph=False, semi=False,
             cms_thresh=0, iters=20),
        # preparation: encoding and relabelling
        dict(name="encode_rmat19", op="encode", gen="rmat", scale=19, ef=16, T=0),
        dict(name="bfs_rmat19", op="bfs", gen="rmat", scale=19, ef=16),
        # the cost model: two epochs over the samples recorded on one graph
        # at the benchmark's batch size, and the prediction for a graph
        dict(name="train_200k", op="train", n=200_000, batch=2048, epochs=2),
        dict(name="infer_1m", op="infer", n=1 << 20),
    ]


def draw(rng: random.Random):
    """One more case of the same ranges; sizes are spread over their logarithm."""
    def log_int(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    op = rng.choice(["lp"] * 8 + ["encode", "bfs", "train", "infer"])
    if op == "train":
        return dict(op=op, n=log_int(2000, 200_000), batch=log_int(200, 4096), epochs=rng.randint(1, 2))
    if op == "infer":
        return dict(op=op, n=log_int(1000, 1 << 20))
    gen = rng.choice(["rmat", "rmat", "rmat", "lattice", "copying"])
    if gen == "rmat":
        c = dict(gen=gen, scale=rng.randint(10, 20), ef=rng.choice([4, 8, 16, 24]))
        verts = 1 << c["scale"]
        arcs = 2 * c["ef"] * verts
    elif gen == "lattice":
        c = dict(gen=gen, side=log_int(33, 1100))
        verts = c["side"] ** 2
        arcs = 4 * verts
    else:
        c = dict(gen=gen, n=log_int(5001, 300_000))
        verts = c["n"]
        arcs = 30 * verts
    if op == "bfs":
        return dict(c, op=op)
    c["T"] = rng.choice([0, 0, 16, 32])
    if op == "encode":
        return dict(c, op=op)
    # as many label vectors as keep the run below the largest listed one
    ks = [k for k in (1, 1, 2, 3, 4, 5, 7, 8, 8, 16, 17, 33, 64) if k * verts <= 1 << 24 and k * arcs <= 1 << 29]
    c["K"] = rng.choice(ks)
    cms = rng.choice([0, 0, 256, 1024, 4096, 8192])
    c.update(op=op, method=rng.choice(["nova"] * 5 + ["cglp", "csr"]), graph=rng.random() < 0.5,
             semi=rng.random() < (0.5 if c["K"] >= 16 else 0.15), cms_thresh=cms, iters=rng.choice([5, 10, 20]))
    if cms:
        c.update(cms_depth=rng.choice([3, 4]), cms_width=rng.choice([512, 1024, 2048]))
    return c


# ------------------------------------------------------------------ inputs

def _csr(case, seed, bfs):
    """the case's graph; R-MAT is BFS-relabelled like the benchmark's"""
    if case["gen"] == "rmat":
        if bfs:
            return L.gen_rmat_device_bfs(case["scale"], case["ef"], 0.57, 0.19, 0.19, seed=seed)
        return L.gen_rmat(case["scale"], case["ef"], 0.57, 0.19, 0.19, seed=seed, bfs=False)
    if case["gen"] == "lattice":
        return L.gen_lattice(case["side"], 0.10, 0.005, seed=seed)
    return L.gen_copying(case["n"], 30.0, 2.1, 100000, 0.7, 1000, seed=seed)


def _renamed(case, seed):
    """the case's graph with its vertices under other names, as a downloaded
    edge list has them: the same numbers of vertices and arcs for every seed"""
    g = _csr(case, 1, bfs=False)
    name = np.random.default_rng(seed).permutation(g.n).astype(np.uint32)
    return L.Csr.from_edges(g.n, np.repeat(name, g.degrees()), name[g.col], False)


def _semi_labels(n, K, seed):
    """in each vector 1 % of the vertices seeded with one of 100 classes"""
    rng = np.random.default_rng(seed)
    lab = np.full(n * K, UNLABELLED, np.uint32)
    idx = rng.choice(n * K, max(1, n * K // 100), replace=False)
    lab[idx] = rng.integers(0, 100, len(idx), dtype=np.uint32)
    return lab


def _features(rng, n):
    """vertex features as the engine gives them: log2(1 + x) of power-law
    degrees, interval and residual counts, bits and segments, the mean
    interval length, and the change flag"""
    deg = np.floor(np.minimum(rng.pareto(1.2, n) * 4 + 1, 1e5))
    itv = np.floor(deg * rng.uniform(0, 0.1, n))
    res = np.floor(deg * rng.uniform(0.5, 1, n))
    bits = 8 + res * rng.uniform(8, 20, n) + itv * rng.uniform(10, 24, n)
    si, sr = np.ceil((itv + 1) / 15), np.ceil((res + 1) / 18)
    mean = np.where(itv > 0, 4 + rng.exponential(2, n), 0)
    x = np.log2(1 + np.stack([deg, itv, res, bits, si, sr, mean], 1))
    return np.concatenate([x, (rng.random((n, 1)) < 0.3)], 1).astype(np.float32), deg


def _params(rng):
    p = np.zeros(NPARAM, np.float32)
    p[:256] = rng.normal(0, (2 / IN) ** 0.5, 256)
    p[288:1312] = rng.normal(0, (2 / HID) ** 0.5, 1024)
    p[1344:1440] = rng.normal(0, (2 / HID) ** 0.5, 96)
    return p


def _model_inputs(case, seed):
    """parameters, features, and for training the targets (log2 of a
    vertex's measured cost per kernel family) with the families measured"""
    rng = np.random.default_rng(seed)
    n = case["n"]
    p = _params(rng)
    x, deg = _features(rng, n)
    if case["op"] == "infer":
        return p, x, None, None
    cost = np.log2(1 + np.stack([200 + 40 * deg, 900 + 12 * deg, 4000 + 6 * deg], 1)) + rng.normal(0, 0.3, (n, 3))
    mask = np.stack([deg <= 1024, deg <= 2048, deg > 0], 1)
    return p, x, cost.astype(np.float32), mask.astype(np.uint8)


def prepare(case, seed):
    op = case["op"]
    if op in ("train", "infer"):
        p, x, t, mask = _model_inputs(case, seed)
        m = L.Mlp(0, seed=0)
        m.params = p
        return dict(case=case, model=m, p=p, x=x, t=t, mask=mask, seed=seed)
    if op in ("encode", "bfs"):
        g = _renamed(case, seed)
        e = L.Engine(0)
        if op == "bfs":
            return dict(case=case, engine=e, graph=g, row=g.row, col=g.col)
        row, col, _ = e.bfs_relabel(g.row, g.col, 0)
        # the stream goes into the program's own buffer: 3 bytes an arc and a
        # word a vertex hold it
        return dict(case=case, engine=e, row=row, col=col, buf=np.zeros(g.m * 3 // 8 + g.n + 16, np.int64))
    g = _csr(case, seed, bfs=True)
    e = L.Engine(0)
    e.upload(g.encode(case["T"], 128))
    cms = {}
    if case["cms_thresh"]:
        cms = dict(cms_thresh=case["cms_thresh"], cms_depth=case["cms_depth"], cms_width=case["cms_width"], cms_seed=0)
    e.config(K=case["K"], semi=case["semi"], **cms)
    e.schedule_degree()
    e.set_graph_mode(case["graph"])
    start = _semi_labels(g.n, case["K"], seed) if case["semi"] else None
    return dict(case=case, engine=e, start=start)


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "lp":
        e = state["engine"]
        e.labels_init(state["start"])
        step = {"nova": e.nova_iterate, "cglp": e.cglp_iterate, "csr": e.csr_iterate}[case["method"]]
        changed = [step() for _ in range(case["iters"])]
        return dict(labels=e.labels(), changed=np.array(changed, np.int64))
    if op == "encode":
        e = state["engine"]
        e.encode_csr(state["row"], state["col"], case["T"])
        words, offsets, vertices, nbits = e.stream()
        state["buf"][:len(words)] = words.view(np.int64)
        return dict(words=state["buf"], offsets=offsets.view(np.int64), vertices=vertices, nbits=nbits)
    if op == "bfs":
        row, col, perm = state["engine"].bfs_relabel(state["row"], state["col"], 0)
        return dict(row=row.view(np.int64), col=col, perm=perm)
    m = state["model"]
    if op == "infer":
        return m.forward(state["x"])
    m.params = state["p"]
    losses = m.train(state["x"], state["t"], state["mask"], epochs=case["epochs"], batch=case["batch"], lr=2e-3,
                     seed=state["seed"])
    return dict(losses=losses, params=m.params)


# ------------------------------------------------------------------- work

def _graph_size(case):
    """vertices, arcs and bits per arc of the stream, about (duplicate edges
    are dropped: more of them in small R-MAT graphs)"""
    if case["gen"] == "rmat":
        n = 1 << case["scale"]
        kept = 0.74 + 0.022 * (case["scale"] - 12)
        return n, 2 * case["ef"] * n * min(0.96, max(0.6, kept)), 13
    if case["gen"] == "lattice":
        n = case["side"] ** 2
        return n, 3.6 * n, 15
    return case["n"], 30 * case["n"], 12


def work(case):
    op = case["op"]
    if op == "infer":
        return dict(bytes=case["n"] * 4 * (IN + OUT), flops=case["n"] * 2 * (IN * HID + HID * HID + HID * OUT))
    if op == "train":
        samples = case["n"] * case["epochs"]
        return dict(bytes=samples * (4 * (IN + OUT) + OUT), flops=samples * 6 * (IN * HID + HID * HID + HID * OUT))
    n, m, bits = _graph_size(case)
    if op == "encode":
        return dict(bytes=8 * n + 4 * m + m * bits / 8 + 12 * n, flops=0)
    if op == "bfs":
        return dict(bytes=2 * (8 * n + 4 * m) + 4 * n, flops=0)
    # per step: the stream and an offset per vertex once, every label read
    # and written once; and the labels in and out of the run
    step = m * bits / 8 + 8 * n + 8 * n * case["K"]
    return dict(bytes=case["iters"] * step + 8 * n * case["K"], flops=0)


# ------------------------------------------------------------------ exact

def _unpack(p):
    return (p[:256].reshape(HID, IN), p[256:288], p[288:1312].reshape(HID, HID), p[1312:1344],
            p[1344:1440].reshape(OUT, HID), p[1440:])


def _forward64(p, x):
    w1, b1, w2, b2, w3, b3 = _unpack(p)
    h1 = np.maximum(x @ w1.T + b1, 0)
    h2 = np.maximum(h1 @ w2.T + b2, 0)
    return h1, h2, h2 @ w3.T + b3


def _shuffle(idx, state):
    """Fisher-Yates of idx in place with splitmix64 from `state`: value i of
    the stream swaps entry n - 1 - i"""
    n = len(idx)
    with np.errstate(over="ignore"):
        k = np.uint64(state) + np.arange(1, n, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        end = int(k[-1]) if n > 1 else state
        z = (k ^ (k >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z ^= z >> np.uint64(31)
        j = (z % np.arange(n, 1, -1, dtype=np.uint64)).tolist()
    a = idx.tolist()
    for i, q in zip(range(n - 1, 0, -1), j):
        a[i], a[q] = a[q], a[i]
    return np.array(a), end


def exact(case, seed):
    """training and prediction in 64 bits; every other result is whole numbers"""
    if case["op"] not in ("train", "infer"):
        return None
    p, x, t, mask = _model_inputs(case, seed)
    p, x = p.astype(np.float64), x.astype(np.float64)
    if case["op"] == "infer":
        return _forward64(p, x)[2]
    n, batch = case["n"], case["batch"]
    m1, m2 = np.zeros(NPARAM), np.zeros(NPARAM)
    idx, stream, step, losses = np.arange(n), seed, 0, []
    for _ in range(case["epochs"]):
        idx, stream = _shuffle(idx, stream)
        total, batches = 0.0, 0
        for b0 in range(0, n, batch):
            s = idx[b0:b0 + batch]
            xb = x[s]
            h1, h2, y = _forward64(p, xb)
            err = np.where(mask[s] != 0, y - t[s].astype(np.float64), 0.0)
            total += np.square(err).sum() / len(s)
            batches += 1
            dy = 2 * err / len(s)
            _, _, w2, _, w3, _ = _unpack(p)
            d2 = (dy @ w3) * (h2 > 0)
            d1 = (d2 @ w2) * (h1 > 0)
            g = np.concatenate([(d1.T @ xb).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0), (dy.T @ h2).ravel(),
                                dy.sum(0)])
            step += 1
            m1 = 0.9 * m1 + 0.1 * g
            m2 = 0.999 * m2 + 0.001 * g * g
            p = p - 2e-3 * (m1 / (1 - 0.9 ** step)) / (np.sqrt(m2 / (1 - 0.999 ** step)) + 1e-8)
        losses.append(total / batches)
    return dict(losses=np.array(losses), params=p)
