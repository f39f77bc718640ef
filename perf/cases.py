"""The counting calls that programs make, as cases to be timed.

Every way into the counter is here: graphs handed over from host memory (a CSR,
an edge list, a device CSR in the reference launcher's layout), graphs resident
in HBM that are counted again and again, one rank's share of a vertex split,
batches of many small graphs, and requests to the server.  Sizes run from a
graph of 256 vertices, where launches and copies are all there is, to R-MAT
scale 26 (two thousand million entries).

A context, and the server, are made once per process and kept, as a program
that counts many graphs keeps them; a graph, a batch or a list of requests is
made from the seed for each state.
"""
import math

import numpy as np

import xxtric_amd

_KEPT = {}


def _ctx():
    if "ctx" not in _KEPT:
        _KEPT["ctx"] = xxtric_amd.Context(0)
    return _KEPT["ctx"]


def _server():
    if "server" not in _KEPT:
        _KEPT["server"] = xxtric_amd.Server(_ctx(), hbm_budget_bytes=2 << 30, max_batch_graphs=1024, max_inflight=2)
    return _KEPT["server"]


# ---- the cases ---------------------------------------------------------------
def listed():
    return [
        # The smallest call: a host CSR (int64, as Graph::edge_list_ holds it) with
        # per-vertex counts -- a unit test's or an interactive user's graph.
        {"name": "csr_rgg_256_pv", "kind": "csr_rgg", "n": 256, "orient": "degree", "per_vertex": True},
        # A mid-sized host CSR with the reference's id orientation and per-vertex counts.
        {"name": "csr_er_20000_id_pv", "kind": "csr_er", "n": 20001, "degree": 32, "orient": "id", "per_vertex": True},
        # An edge list as read from a file (amazon0302's size): built into a CSR and counted.
        {"name": "edges_262111", "kind": "edges", "n": 262111, "m": 899792},
        # The reference launcher's call: an int64 CSR already in device memory.
        {"name": "ffi_rmat_s16", "kind": "ffi", "scale": 16, "edgefactor": 16},
        # The reference's own test graph (tric -n 100000 -l), resident, counted again and again.
        {"name": "rgg_1e5", "kind": "rgg", "n": 100000, "connect": False, "orient": "degree", "per_vertex": False},
        # A skewed graph of the size that a large serving request has.
        {"name": "rmat_s18", "kind": "rmat", "scale": 18, "edgefactor": 16, "permute": True, "per_vertex": False},
        # The benchmark's middle size.
        {"name": "rmat_s22", "kind": "rmat", "scale": 22, "edgefactor": 16, "permute": True, "per_vertex": False},
        # The same with the generator's own labels (hubs at low ids), per vertex.
        {"name": "rmat_s22_raw_pv", "kind": "rmat", "scale": 22, "edgefactor": 16, "permute": False, "per_vertex": True},
        # The headline benchmark: R-MAT scale 26, the whole graph.
        {"name": "rmat_s26", "kind": "rmat", "scale": 26, "edgefactor": 16, "permute": True, "per_vertex": False},
        # One rank of an 8-way vertex split: its slice of the graph, its owned triangles.
        {"name": "owned_rmat_s23_0of8", "kind": "owned", "scale": 23, "edgefactor": 16, "parts": 8, "rank": 0},
        # Many small graphs (half geometric, half random), resident, one pipeline over all.
        {"name": "batch_1024", "kind": "batch", "count": 1024, "nmax": 20000},
        # Requests of that mix handed to the server from host memory, results polled.
        {"name": "serve_256", "kind": "serve", "count": 256, "nmax": 20000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["csr_rgg", "csr_er", "edges", "ffi", "rgg", "rgg", "rmat", "rmat", "rmat", "owned", "batch",
                       "serve"])
    c = {"kind": kind}
    if kind in ("csr_rgg", "csr_er"):
        c["n"] = _log(rng, 64, 70000 if kind == "csr_rgg" else 30000)
        if kind == "csr_er":
            c["degree"] = rng.randint(4, 64)
        c["orient"] = rng.choice(["degree", "id"])
        c["per_vertex"] = rng.random() < 0.5
    elif kind == "edges":
        c["n"] = _log(rng, 500, 400000)
        c["m"] = int(c["n"] * rng.uniform(1.5, 8.0))
    elif kind == "ffi":
        c["scale"] = rng.randint(9, 19)
        c["edgefactor"] = rng.randint(5, 24)
    elif kind == "rgg":
        c["n"] = _log(rng, 1000, 400000)
        c["connect"] = rng.random() < 0.5
        c["orient"] = rng.choice(["degree", "degree", "id"])
        c["per_vertex"] = rng.random() < 0.3
    elif kind == "rmat":
        c["scale"] = rng.randint(10, 24)
        c["edgefactor"] = rng.randint(6, 24)
        c["permute"] = rng.random() < 0.7
        c["per_vertex"] = rng.random() < 0.3
    elif kind == "owned":
        c["scale"] = rng.randint(12, 23)
        c["edgefactor"] = rng.randint(6, 20)
        c["parts"] = rng.randint(2, 16)
        c["rank"] = rng.randrange(c["parts"])
    elif kind == "batch":
        c["count"] = _log(rng, 8, 1200)
        c["nmax"] = _log(rng, 500, 20000)
    else:
        c["count"] = _log(rng, 4, 400)
        c["nmax"] = _log(rng, 500, 20000)
    return c


# ---- inputs ------------------------------------------------------------------
def _er_edges(n, degree, seed):
    """Uniform random pairs with about `degree` neighbours a vertex."""
    r = np.random.default_rng([seed, n, degree])
    return r.integers(0, n, n * degree // 2), r.integers(0, n, n * degree // 2)


def _mixed_edges(n, m, seed):
    """Half the edges to nearby ids, half to a skewed choice of vertices, in any
    order and direction, some of them repeated -- as a file of pairs has them."""
    r = np.random.default_rng([seed, n, m])
    near = m // 2
    u = r.integers(0, n, m)
    v = np.empty(m, np.int64)
    v[:near] = (u[:near] + r.geometric(0.15, near)) % n
    v[near:] = (n * r.random(m - near) ** 3).astype(np.int64)
    p = r.permutation(m)
    flip = r.random(m) < 0.5
    u, v = u[p], v[p]
    return np.where(flip, v, u), np.where(flip, u, v)


def _simple_csr(n, u, v):
    """Symmetric CSR without self-loops or repeated entries (int64)."""
    keep = u != v
    a, b = np.concatenate([u[keep], v[keep]]), np.concatenate([v[keep], u[keep]])
    key = np.unique(a * n + b)
    off = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(key // n, minlength=n), out=off[1:])
    return off, key % n


def _seed32(seed):
    return int(seed) % 2000003 + 1


def prepare(case, seed):
    k = case["kind"]
    s = {"case": case, "ctx": _ctx()}
    if k == "csr_rgg":
        s["off"], s["tails"] = xxtric_amd.rgg_generate(case["n"], seed=_seed32(seed))
    elif k == "csr_er":
        s["off"], s["tails"] = _simple_csr(case["n"], *_er_edges(case["n"], case["degree"], seed))
    elif k == "edges":
        s["src"], s["dst"] = _mixed_edges(case["n"], case["m"], seed)
    elif k == "ffi":
        g = s["ctx"].rmat(case["scale"], case["edgefactor"], seed=int(seed))
        off, tails = g.download()
        g.close()
        s["nv"] = len(off) - 1
        s["d_off"] = s["ctx"].to_device(off)
        s["d_tails"] = s["ctx"].to_device(tails.astype(np.int64))
        s["d_count"] = s["ctx"].to_device(np.zeros(1, np.int64))
        s["zero"] = np.zeros(1, np.int64)
    elif k == "rgg":
        off, tails = xxtric_amd.rgg_generate(case["n"], seed=_seed32(seed), connect=case["connect"],
                                             strict=case["connect"])
        s["g"] = s["ctx"].graph(off, tails)
    elif k == "rmat":
        s["g"] = s["ctx"].rmat(case["scale"], case["edgefactor"], seed=int(seed), permute=case["permute"])
    elif k == "owned":
        g = s["ctx"].rmat(case["scale"], case["edgefactor"], seed=int(seed))
        s["lo"] = g.nv * case["rank"] // case["parts"]
        s["hi"] = g.nv * (case["rank"] + 1) // case["parts"]
        s["g"] = g.slice(s["lo"], s["hi"])
        g.close()
    elif k == "batch":
        size = [xxtric_amd.batch_params(int(seed), i, 200, case["nmax"])[0] for i in range(case["count"])]
        nv = sum(size)
        s["b"] = xxtric_amd.Batch(s["ctx"], nv, 72 * nv + 4096, case["count"])
        s["b"].add_generated(int(seed), 0, case["count"], 200, case["nmax"])
    else:
        s["server"] = _server()
        s["graphs"] = [xxtric_amd.batch_graph_csr(int(seed), i, 200, case["nmax"]) for i in range(case["count"])]
    return s


def run(state):
    c, k = state["case"], state["case"]["kind"]
    if k in ("csr_rgg", "csr_er"):
        return state["ctx"].count_csr(state["off"], state["tails"], per_vertex=c["per_vertex"], orient=c["orient"])
    if k == "edges":
        return state["ctx"].count_edges(c["n"], state["src"], state["dst"])
    if k == "ffi":
        state["d_count"].upload(state["zero"])
        state["ctx"].single_gpu_count(state["nv"], state["d_off"].ptr, state["d_tails"].ptr, state["d_count"].ptr)
        return state["d_count"].download(np.int64, 1)
    if k == "rgg":
        return state["g"].count(per_vertex=c["per_vertex"], orient=c["orient"])
    if k == "rmat":
        return state["g"].count(per_vertex=c["per_vertex"])
    if k == "owned":
        return state["g"].count_owned(state["lo"], state["hi"], total=False)[:2]
    if k == "batch":
        state["b"].run()
        return state["b"].results()
    tickets = [state["server"].submit(off, tails) for off, tails in state["graphs"]]
    state["server"].drain()
    return np.array([state["server"].poll(t)[0] for t in tickets], np.uint64)


# ---- what a pass cannot do without -------------------------------------------
def _csr_bytes(n, entries, id_bytes):
    return 8 * (n + 1) + id_bytes * entries


def work(case):
    """Input bytes read once and results written once (entries as expected from
    the generators); the count has no arithmetic that a matrix unit would do."""
    k = case["kind"]
    if k in ("csr_rgg", "rgg"):
        n = case["n"]
        r = xxtric_amd.rgg_radius_connect(n) if case.get("connect") else xxtric_amd.rgg_radius(n)
        b = _csr_bytes(n, n * n * math.pi * r * r, 8 if k == "csr_rgg" else 4)
    elif k == "csr_er":
        n = case["n"]
        b = _csr_bytes(n, n * case["degree"], 8)
    elif k == "edges":
        n, b = case["n"], 16 * case["m"]
    elif k in ("ffi", "rmat", "owned"):
        n = 1 << case["scale"]
        b = _csr_bytes(n, 1.9 * case["edgefactor"] * n, 8 if k == "ffi" else 4)
    else:
        # n log-uniform in [200, nmax], mean degree about 9 (geometric) or 34 (random)
        n = case["count"] * (case["nmax"] - 200) / math.log(case["nmax"] / 200.0)
        b = _csr_bytes(n, 21.5 * n, 4) + 8 * case["count"]
    if case.get("per_vertex"):
        b += 8 * n
    return {"bytes": float(b + 8), "flops": 0.0}


# ---- the counts in plain numpy ------------------------------------------------
def _count(n, off, tails):
    """Total and per-vertex counts (each triangle at its smallest id): every pair
    of higher neighbours of a vertex is looked up among the edges."""
    u = np.repeat(np.arange(n), np.diff(off))
    up = tails > u
    a, b = u[up], tails[up]
    key = a * n + b  # ascending
    deg = np.bincount(a, minlength=n)
    first = np.concatenate([[0], np.cumsum(deg)])
    rest = first[a + 1] - np.arange(len(a)) - 1  # later neighbours of the same vertex
    pv = np.zeros(n, np.int64)
    step = max(1, int(2e7 // max(1, rest.max(initial=1))))
    for i in range(0, len(a), step):
        r = rest[i:i + step]
        e = np.repeat(np.arange(i, i + len(r)), r)
        j = np.arange(len(e)) - np.repeat(np.cumsum(r) - r, r) + e + 1
        want = b[e] * n + b[j]
        at = np.minimum(np.searchsorted(key, want), len(key) - 1)
        pv += np.bincount(a[e[key[at] == want]], minlength=n)
    return int(pv.sum()), pv.astype(np.uint64)


def exact(case, seed):
    """The counts of the inputs that are made here; None where the library's own
    generators make them."""
    if case["kind"] == "csr_er":
        off, tails = _simple_csr(case["n"], *_er_edges(case["n"], case["degree"], seed))
    elif case["kind"] == "edges":
        off, tails = _simple_csr(case["n"], *_mixed_edges(case["n"], case["m"], seed))
    else:
        return None
    total, pv = _count(case["n"], off, tails)
    return (total, pv) if case.get("per_vertex") else total
