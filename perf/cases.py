"""Performance cases: label propagation as programs call it, over the range of
graphs, methods and calls the library serves.

A case is a dict of plain values.  `prepare` makes its graph from a seed and
the handle a program keeps (a graph, a session, a batch, a server), `run` is
one pass through the public entry points of glp_amd: propagation from L0 and
the labels (and other state the method has) copied to the host.

Graphs are the families the repository measures and tests with: R-MAT
(a, b, c = .57, .19, .19; scale 25 is the headline benchmark's), planted
partitions and LFR-style graphs.
"""
import math

import numpy as np
import torch

import glp_amd as G

METHODS = {"classic": G.CLASSIC, "layered": G.LAYERED, "slpa": G.SLPA, "countmin": G.COUNTMIN,
           "frequent": G.FREQUENT, "buffer": G.BUFFER, "seeded": G.SEEDED}

SERVED_STEPS = 10


def case(kind, graph, **kw):
    c = {"kind": kind, "graph": graph, "method": "classic", "steps": 10, "weighted": False}
    c.update(kw)
    return c


def listed():
    return [
        # the command line's shape: one call on a small graph, state made and
        # freed inside it (latency of allocation, planning, launches, copies)
        case("run", "lfr", name="run_lfr_2048", n=2048),
        # the smallest resident job: a thousand vertices in small communities,
        # where only launches count
        case("session", "planted", name="planted_1000", n=1000, k=20, deg_in=10.0, deg_out=2.0, steps=20),
        # the reference configuration of 65,536 vertices in 64 communities
        case("session", "planted", name="planted_65536", n=65536, k=64, deg_in=12.0, deg_out=4.0, steps=20),
        # an edge list as a .bin file holds it: ids unsorted, duplicates kept,
        # neighbours in file order
        case("session", "rmat", name="rmat18_file_order", scale=18, ef=16, sort=False, dedup=False),
        # the headline: a social-network-like graph, degree-sorted, with hubs
        case("session", "rmat", name="rmat25", scale=25, ef=16, sort=True, dedup=True),
        # the layered method where labels stay diverse
        case("session", "rmat", name="layered_rmat22", scale=22, ef=16, sort=True, dedup=True,
             method="layered", gamma_num=1, gamma_den=4),
        # a weighted graph run to convergence with the frontier
        case("session", "rmat", name="frontier_weighted_rmat21", scale=21, ef=16, sort=True, dedup=True,
             wmax=8, weighted=True, frontier=1, steps=25),
        # overlapping communities: the SLPA configuration with its post-processing
        case("session", "lfr", name="slpa_lfr_2e20", n=1 << 20, method="slpa", steps=20),
        # bounded-memory counting: a sketch and a heavy-hitter table
        case("session", "rmat", name="countmin_rmat21", scale=21, ef=16, sort=True, dedup=True,
             method="countmin", cm_rows=3, cm_width=200, steps=3),
        case("session", "rmat", name="frequent_rmat21", scale=21, ef=16, sort=True, dedup=True,
             method="frequent", cap=16, steps=3),
        # many graphs of uneven size stepped together
        case("batch", "planted", name="batch_96", graphs=96, nmin=1000, nmax=262144, steps=20),
        # a burst of weighted classic and layered jobs on resident graphs
        case("served", "rmat", name="served_48", jobs=48, resident=12, smin=12, smax=18, wmax=8,
             weighted=True, steps=SERVED_STEPS),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng, top_scale):
    g = rng.choice(["rmat", "rmat", "planted", "lfr"])
    if g == "rmat":
        return {"graph": g, "scale": rng.randint(10, top_scale), "ef": rng.randint(4, 24),
                "sort": rng.random() < 0.5, "dedup": rng.random() < 0.7}
    if g == "planted":
        n = _log_int(rng, 500, 1 << 20)
        d = rng.uniform(4.0, 48.0)
        out = rng.uniform(0.1, 0.4)
        return {"graph": g, "n": n, "k": max(4, n // rng.randint(100, 1000)), "deg_in": round(d * (1 - out), 3),
                "deg_out": round(d * out, 3)}
    return {"graph": g, "n": _log_int(rng, 2000, 1 << 20)}


def draw(rng):
    kind = rng.choice(["run", "session", "session", "session", "session", "session", "batch", "served"])
    if kind == "batch":
        return case(kind, "planted", graphs=_log_int(rng, 8, 96), nmin=1000, nmax=_log_int(rng, 4000, 262144),
                    steps=rng.randint(5, 20))
    if kind == "served":
        lo = rng.randint(11, 14)
        return case(kind, "rmat", jobs=_log_int(rng, 4, 48), resident=rng.randint(2, 12), smin=lo,
                    smax=rng.randint(lo + 1, 18), wmax=rng.randint(2, 9), weighted=True, steps=rng.randint(3, 10))
    if kind == "run":
        c = case(kind, **_draw_graph(rng, 16), steps=rng.randint(1, 20))
        c["method"] = rng.choice(["classic", "classic", "layered"])
    else:
        m = rng.choice(["classic", "classic", "classic", "layered", "layered", "slpa", "countmin", "frequent",
                        "buffer", "seeded"])
        c = case(kind, **_draw_graph(rng, {"classic": 22, "layered": 21}.get(m, 20)))
        c["method"] = m
        c["steps"] = rng.randint(1, 4) if m in ("countmin", "frequent", "buffer") else rng.randint(3, 24)
    if c["graph"] == "rmat" and rng.random() < 0.3:
        c["weighted"] = True
        c["wmax"] = rng.randint(2, 9)
    if c["method"] == "layered":
        c["gamma_num"], c["gamma_den"] = rng.choice([(0, 1), (1, 4), (1, 2), (1, 1)])
    if c["method"] == "classic":
        c["frontier"] = rng.choice([0, 0, 1])
    if c["method"] in ("classic", "layered", "seeded") and kind == "session":
        c["gather"] = rng.choice([0, 0, 0, 1])
        c["replay"] = rng.random() < 0.3
    if c["method"] == "countmin":
        c["cm_rows"], c["cm_width"] = rng.randint(1, 5), rng.randint(40, 600)
    if c["method"] in ("frequent", "buffer"):
        c["cap"] = rng.choice([4, 7, 16, 33, 64])
    if c["method"] == "seeded":
        c["frac"] = round(rng.uniform(0.001, 0.1), 4)
    return c


# ------------------------------------------------------------------ inputs ----

def _rmat(c, seed):
    """Symmetric R-MAT graph without self-loops, drawn on the GPU."""
    n = 1 << c["scale"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    parts = []
    total = n * c["ef"]
    for at in range(0, total, 1 << 25):
        k = min(1 << 25, total - at)
        u = torch.zeros(k, dtype=torch.int64, device="cuda")
        v = torch.zeros(k, dtype=torch.int64, device="cuda")
        for _ in range(c["scale"]):
            r = torch.rand(k, device="cuda", generator=gen)
            u.mul_(2).add_(r >= 0.76)                       # quadrants c, d
            v.mul_(2).add_(((r >= 0.57) & (r < 0.76)) | (r >= 0.95))  # b, d
        keep = u != v
        parts.append(torch.stack([u[keep], v[keep]]))
    u, v = torch.cat(parts, 1)
    del parts
    if c["dedup"]:
        key = torch.unique(torch.minimum(u, v) * n + torch.maximum(u, v))
        u, v = key // n, key % n
        del key
    if c["sort"]:
        deg = torch.bincount(u, minlength=n) + torch.bincount(v, minlength=n)
        rank = torch.empty(n, dtype=torch.int64, device="cuda")
        rank[torch.sort(deg, descending=True, stable=True).indices] = torch.arange(n, device="cuda")
        u, v = rank[u], rank[v]
        del deg, rank
    w = None
    if c.get("wmax"):
        w = torch.randint(1, c["wmax"] + 1, (len(u),), device="cuda", generator=gen)
    # both directions, in the order of the pairs (sorted lists when deduplicated)
    src, dst = torch.stack([u, v], 1).reshape(-1), torch.stack([v, u], 1).reshape(-1)
    del u, v
    if c["dedup"]:
        order = torch.sort(src * n + dst).indices
    else:
        order = torch.sort(src, stable=True).indices
    off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(torch.bincount(src, minlength=n), 0, out=off[1:])
    nbr = dst[order].to(torch.int32).cpu().numpy()
    ww = None if w is None else w.repeat_interleave(2)[order].to(torch.int32).cpu().numpy().astype(np.uint32)
    off = off.to(torch.int32).cpu().numpy()
    del src, dst, order
    torch.cuda.empty_cache()  # the graphs live in the library's memory, not in torch's
    return G.Graph.from_csr(off, nbr, ww)


def _graph(c, seed):
    if c["graph"] == "rmat":
        return _rmat(c, seed)
    if c["graph"] == "planted":
        return G.Graph.planted(c["n"], c["k"], c["deg_in"], c["deg_out"], seed=seed)
    return G.Graph.lfr(c["n"], seed=seed)


def _params(c):
    return G.make_params(method=METHODS[c["method"]], weighted=c["weighted"],
                         gamma=(c.get("gamma_num", 0), c.get("gamma_den", 1)), slpa_T=max(c["steps"], 1),
                         cm_rows=c.get("cm_rows", 3), cm_width=c.get("cm_width", 200), table_cap=c.get("cap", 16),
                         gather=c.get("gather", 0), frontier=c.get("frontier", 0))


def _seeds(c, n, seed):
    return np.random.default_rng(seed).random(n) < c["frac"]


def prepare(c, seed):
    if c["kind"] == "batch":
        graphs = []
        for i in range(c["graphs"]):  # the mix's sizes, graphs of this seed
            p = G.mix_params(1, i, c["nmin"], c["nmax"])
            graphs.append(G.Graph.planted(p["n"], p["k"], p["deg_in"], p["deg_out"], seed=seed * 1000 + i))
        return {"case": c, "batch": G.Batch(graphs, method=METHODS[c["method"]])}
    if c["kind"] == "served":
        rng = np.random.default_rng(1)  # the mix's sizes and jobs, graphs of this seed
        sv = G.Server(budget_bytes=16 << 30, max_slots=64)
        pool = []
        for i in range(c["resident"]):
            scale = c["smin"] + i % (c["smax"] - c["smin"] + 1)
            pool.append((sv.add_rmat(scale, int(rng.integers(8, 33)), seed=seed * 100 + i, wmax=c["wmax"]), 1 << scale))
        jobs = [(pool[int(rng.integers(len(pool)))], bool(rng.integers(2))) for _ in range(c["jobs"])]
        return {"case": c, "server": sv, "jobs": jobs,
                "classic": G.make_params(method=G.CLASSIC, weighted=True),
                "layered": G.make_params(method=G.LAYERED, gamma=(1, 4), weighted=True)}
    g = _graph(c, seed)
    if c["kind"] == "run":
        return {"case": c, "graph": g, "params": _params(c)}
    s = G.Session(g, _params(c))
    if c["method"] == "seeded":
        s.set_seeds(_seeds(c, g.n, seed))
    return {"case": c, "graph": g, "session": s}


def run(state):
    c = state["case"]
    if c["kind"] == "run":
        return G.run(state["graph"], c["steps"], state["params"])[0]
    if c["kind"] == "batch":
        b = state["batch"]
        b.reset()
        b.run(c["steps"], mode=1)
        return np.concatenate([b.labels(i) for i in range(c["graphs"])])
    if c["kind"] == "served":
        sv = state["server"]
        ids = [(sv.submit_resident(gid, c["steps"], state["layered" if lay else "classic"]), n)
               for (gid, n), lay in state["jobs"]]
        labels = [sv.wait(j, n)[0] for j, n in ids]
        for j, _ in ids:
            sv.release(j)
        return np.concatenate(labels)
    s = state["session"]
    s.reset()
    s.step(c["steps"], graph=bool(c.get("replay")))
    if c["method"] == "slpa":
        dominant, nsets, sets = s.slpa_post(kmax=4)
        return {"dominant": dominant, "nsets": nsets, "sets": sets}
    if c["method"] == "layered":
        return {"labels": s.labels(), "volume": s.volume()}
    if c.get("frontier"):
        return {"labels": s.labels(), "changes": s.changes()}
    return s.labels()


# -------------------------------------------------------------------- work ----

def _size(c):
    """Vertices and directed edges (their expectation)."""
    if c["graph"] == "rmat":
        n = 1 << c["scale"]
        lost = min(0.5, 0.093 * 0.829 ** (c["scale"] - 18) * c["ef"] / 16) if c["dedup"] else 0.0
        return n, 2 * c["ef"] * n * (1 - lost)
    if c["graph"] == "planted":
        return c["n"], c["n"] * (c["deg_in"] + c["deg_out"])
    return c["n"], c["n"] * 19.6


def _step_bytes(c, n, m):
    """CSR once, each vertex's label in and out; a layered step also reads and
    writes a volume per label, an SLPA step reads a memory word per vertex."""
    b = 4 * m * (2 if c["weighted"] else 1) + 12 * n
    if c["method"] == "layered":
        b += 8 * n
    if c["method"] == "slpa":
        b += 4 * n
    return b


def work(c):
    if c["kind"] == "batch":
        mean = (c["nmax"] - c["nmin"]) / math.log(c["nmax"] / c["nmin"])
        n = c["graphs"] * mean
        return {"bytes": c["steps"] * _step_bytes(c, n, 34 * n), "flops": 0}
    if c["kind"] == "served":
        scales = [c["smin"] + i % (c["smax"] - c["smin"] + 1) for i in range(c["resident"])]
        total = 0
        for s in scales:
            n, m = _size({"graph": "rmat", "scale": s, "ef": 20, "dedup": True})
            total += _step_bytes(c, n, m)
        return {"bytes": c["steps"] * c["jobs"] * total / len(scales), "flops": 0}
    n, m = _size(c)
    # with the frontier, steps after the first few touch few vertices
    b = (min(c["steps"], 5) if c.get("frontier") else c["steps"]) * _step_bytes(c, n, m)
    if c["method"] == "slpa":
        b += 4 * n * (c["steps"] + 1) + 4 * n * 6  # post-processing: the memory in, six words a vertex out
    return {"bytes": b, "flops": 0}


# ------------------------------------------------------------------- exact ----

def exact(c, seed):
    """Labels (and volumes) by sorting each step's (vertex, label) pairs, in
    whole 64-bit numbers: classic, layered and seeded propagation on graphs of
    up to a few tens of millions of edge visits.  Every output is a whole
    number, so this says what is right, not how near a rounding comes."""
    if c["kind"] not in ("run", "session") or c["method"] not in ("classic", "layered", "seeded"):
        return None
    if _size(c)[1] * c["steps"] > 4e8:
        return None
    off, nbr, w = _graph(c, seed).csr()
    n = len(off) - 1
    d = "cuda" if torch.cuda.is_available() else "cpu"
    deg = torch.from_numpy(np.diff(off).astype(np.int64)).to(d)
    src = torch.repeat_interleave(torch.arange(n, device=d), deg)
    dst = torch.from_numpy(nbr.astype(np.int64)).to(d)
    f = torch.from_numpy(w.astype(np.int64)).to(d) if c["weighted"] else torch.ones_like(src)
    lab = torch.arange(n, device=d)
    fixed = torch.zeros(n, dtype=torch.bool, device=d)
    if c["method"] == "seeded":
        fixed = torch.from_numpy(_seeds(c, n, seed)).to(d)
        lab = torch.where(fixed, lab, -1)
    p, q = c.get("gamma_num", 0), c.get("gamma_den", 1)
    if c["method"] != "layered":
        p, q = 0, 1
    changes = []
    for _ in range(c["steps"]):
        vol = torch.bincount(lab.clamp(min=0), minlength=n)
        show = lab[dst]
        on = show >= 0
        pair, inv = torch.unique(src[on] * n + show[on], return_inverse=True)
        cnt = torch.zeros(len(pair), dtype=torch.int64, device=d).scatter_add_(0, inv, f[on])
        v, l = pair // n, pair % n
        word = ((q + p) * cnt - p * vol[l] + (1 << 31)) * (1 << 31) + l
        best = torch.full((n,), -1, dtype=torch.int64, device=d).scatter_reduce_(0, v, word, "amax")
        new = torch.where((best >= 0) & ~fixed, best % (1 << 31), lab)
        changes.append(int((new != lab).sum()))
        lab = new
    labels = lab.to(torch.int32).cpu().numpy()
    if c["method"] == "layered" and c["kind"] == "session":
        return {"labels": labels, "volume": torch.bincount(lab, minlength=n).to(torch.int32).cpu().numpy()}
    if c.get("frontier") and c["kind"] == "session":
        return {"labels": labels, "changes": np.array(changes, dtype=np.int64)}
    return labels
