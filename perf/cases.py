"""The work that a user has this library do, as measurable cases.

Every case is a plain dict with a "kind", the path that it takes through the
public entry points:

run          A graph in host arrays to its communities: GraphGPU on the CSR,
             LouvainGPU.run, the clustering back (what the command line does).
phase        One phase on a resident graph: singleton partition, modularity,
             iterations until they gain no more than the threshold, the
             communities and their totals (the benchmark's iterations).
steps        The same with the single GraphGPU calls of the reference's driver:
             update, weights and ids batch by batch, then the modularity.
batch        Many planted-partition graphs of mixed sizes in one handle, run
             to completion together.
serve        Requests of mixed sizes handed to a running server, all awaited.
window       A graph whose arcs stream through a device window, run to the end.
modularity   The modularity of a given partition of a graph that is on the
             device, without an allocation, on the caller's stream.

Graphs are R-MAT (0.57, 0.19, 0.19, 0.05), Chung-Lu with Pareto(2.1) degrees,
or planted partitions in blocks of 64, symmetric, without self arcs or
duplicates, with unit or U(0, 1] weights.  "stream": the program keeps a
stream of its own and gives it to its handles, as one that makes large
handles one after another does; otherwise a handle makes its own.
"""
import numpy as np
import torch

import nido_amd as na

TOL = 1e-6
DEV = "cuda"


def listed():
    return [
        # the smallest: the 1,024-vertex planted partition at the command line's defaults
        dict(name="run-sbm-1k", kind="run", graph="sbm", n=1024, inner=19.0, outer=4.8, weighted=False, nb=2),
        # an ordinary request: a small power-law graph
        dict(name="run-rmat-s14", kind="run", graph="rmat", n=1 << 14, ef=16, weighted=False, nb=2),
        # an odd size, weighted: a mid-size graph of an analysis job
        dict(name="run-chunglu-300k", kind="run", graph="chunglu", n=300007, mean=32.0, dmax=5000.0, weighted=True, nb=8),
        # the largest graph of the benchmark's request stream
        dict(name="run-rmat-s20", kind="run", graph="rmat", n=1 << 20, ef=32, weighted=False, nb=32, stream=True),
        # the benchmark's graph: iterations of its first phase
        dict(name="phase-rmat-s22", kind="phase", graph="rmat", n=1 << 22, ef=16, weighted=True, nb=32, stream=True),
        # a flatter degree distribution, ragged size, unit weights
        dict(name="phase-chunglu-2m", kind="phase", graph="chunglu", n=2100001, mean=32.0, dmax=50000.0, weighted=False, nb=32,
             stream=True),
        # a driver that makes the single calls itself
        dict(name="steps-rmat-s17", kind="steps", graph="rmat", n=1 << 17, ef=16, weighted=True, nb=8),
        # many graphs at once, an eighth of the benchmark's 4,096
        dict(name="batch-512-sbm", kind="batch", graphs=512, nmin=256, nmax=65536, inner=12.0, outer=2.0, weighted=True, nb=32,
             stream=True),
        # a handful of small graphs at once
        dict(name="batch-40-small", kind="batch", graphs=40, nmin=200, nmax=5000, inner=12.0, outer=2.0, weighted=False, nb=2),
        # a burst of requests
        dict(name="serve-24-mixed", kind="serve", requests=24, smin=10, smax=17, weighted=False, nb=32),
        # a graph of five windows
        dict(name="window-rmat-s19", kind="window", graph="rmat", n=1 << 19, ef=16, weighted=True, nb=32, parts=5),
        # a given partition scored on the device
        dict(name="modularity-1m", kind="modularity", graph="sbm", n=1 << 20, inner=12.0, outer=2.0, weighted=True),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["run", "run", "phase", "phase", "steps", "batch", "serve", "window", "modularity"])
    weighted = rng.random() < 0.5
    nb = rng.choice([2, 8, 32])
    if kind == "batch":
        graphs = _log(rng, 8, 512)
        return dict(kind=kind, graphs=graphs, nmin=256, nmax=_log(rng, 1024, 65536), inner=12.0, outer=2.0, weighted=weighted,
                    nb=nb, stream=graphs > 64 or rng.random() < 0.5)
    if kind == "serve":
        smin = rng.randint(10, 13)
        return dict(kind=kind, requests=rng.randint(4, 24), smin=smin, smax=rng.randint(smin, 16), weighted=weighted, nb=nb)
    hi = {"run": 1 << 20, "phase": 1 << 21, "steps": 1 << 19, "window": 1 << 19, "modularity": 1 << 21}[kind]
    lo = {"run": 1 << 10, "phase": 1 << 16, "steps": 1 << 12, "window": 1 << 15, "modularity": 1 << 10}[kind]
    n = _log(rng, lo, hi)
    graph = rng.choice(["rmat", "chunglu", "sbm"]) if kind != "modularity" else "sbm"
    c = dict(kind=kind, graph=graph, n=n, weighted=weighted)
    if kind != "modularity":
        c |= dict(nb=nb, stream=n > 1 << 18 or rng.random() < 0.5)
    if graph == "rmat":
        c["ef"] = rng.choice([8, 16])
    elif graph == "chunglu":
        c |= dict(mean=rng.choice([8.0, 32.0]), dmax=float(min(50000, max(64, n // 60))))
    else:
        c |= dict(inner=12.0, outer=2.0)
    if kind == "window":
        c |= dict(nb=32, parts=rng.randint(2, 6))
    return c


# ---- inputs ------------------------------------------------------------------
def _csr(n, u, v, weighted, gen):
    """The symmetric CSR of the edges (u, v) (duplicates and self arcs dropped)
    as device tensors; both arcs of an edge have its weight."""
    key = torch.minimum(u, v) * n + torch.maximum(u, v)
    key = torch.unique(key[u != v])
    lo, hi = key // n, key % n
    del key, u, v
    m = lo.numel()
    w = 1.0 - torch.rand(m, generator=gen, device=DEV, dtype=torch.float64) if weighted else \
        torch.ones(m, device=DEV, dtype=torch.float64)
    key, order = torch.sort(torch.cat([lo * n + hi, hi * n + lo]))
    del lo, hi
    off = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(torch.bincount(key // n, minlength=n), 0)
    return off, key % n, w[order % m] if m else w


def _rmat(n, ef, gen):
    scale = max(1, (n - 1).bit_length())
    m = n * ef
    u = torch.zeros(m, dtype=torch.int64, device=DEV)
    v = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(scale):
        r = torch.rand(m, generator=gen, device=DEV)
        u = 2 * u + (r >= 0.76)
        v = 2 * v + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    return u % n, v % n


def _chunglu(n, mean, dmax, gen):
    d = (2.0 * (1.0 - torch.rand(n, generator=gen, device=DEV, dtype=torch.float64)) ** (-1.0 / 1.1)).clamp_(max=dmax)
    cum = torch.cumsum(d, 0)
    m = int(n * mean / 2)

    def ends():
        return torch.searchsorted(cum, torch.rand(m, generator=gen, device=DEV, dtype=torch.float64) * cum[-1]).clamp_(max=n - 1)
    return ends(), ends()


def _sbm(sizes, inner, outer, gen):
    """Planted partitions of the given sizes side by side, blocks of 64."""
    sizes = torch.tensor(sizes, device=DEV)
    n = int(sizes.sum())
    first = torch.cumsum(sizes, 0) - sizes
    graph = torch.repeat_interleave(torch.arange(len(sizes), device=DEV), sizes)
    us, vs = [], []
    for degree, within in ((inner, True), (outer, False)):
        u = torch.randint(n, (int(n * degree / 2),), generator=gen, device=DEV)
        g = graph[u]
        base, size = first[g], sizes[g]
        if within:
            block = (u - base) // 64 * 64
            base, size = base + block, torch.clamp(size - block, max=64)
        us.append(u)
        vs.append(base + (torch.rand(u.numel(), generator=gen, device=DEV, dtype=torch.float64) * size).long())
    return torch.cat(us), torch.cat(vs)


def _graph(case, gen):
    n = case["n"]
    if case["graph"] == "rmat":
        u, v = _rmat(n, case["ef"], gen)
    elif case["graph"] == "chunglu":
        u, v = _chunglu(n, case["mean"], case["dmax"], gen)
    else:
        u, v = _sbm([n], case["inner"], case["outer"], gen)
    return _csr(n, u, v, case["weighted"], gen)


def _host(csr):
    return tuple(x.cpu().numpy() for x in csr)


def _sizes(case):
    """Vertex counts log-uniform in [nmin, nmax], the same for every seed, so
    that a pass on other inputs is as much work."""
    k, ratio = case["graphs"], case["nmax"] / case["nmin"]
    return [int(case["nmin"] * ratio ** (((i * 0.6180339887498949) % 1.0))) for i in range(1, k + 1)]


def _requests(case):
    """(scale, edge factor) of every request: all scales, all edge factors."""
    span = case["smax"] - case["smin"] + 1
    return [(case["smin"] + i % span, (8, 16, 32)[i // span % 3]) for i in range(case["requests"])]


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed) + 1)
    kind = case["kind"]
    if kind == "modularity":
        off, col, w = _graph(case, gen)
        n = case["n"]
        # the planted blocks with a tenth of the vertices elsewhere
        comm = torch.arange(n, device=DEV) // 64
        move = torch.rand(n, generator=gen, device=DEV) < 0.1
        comm = torch.where(move, torch.randint(n, (n,), generator=gen, device=DEV) // 64, comm)
        return dict(case=case, off=off, col=col, w=w, comm=comm, q=torch.zeros(1, dtype=torch.float64, device=DEV))
    if kind == "batch":
        sizes = _sizes(case)
        u, v = _sbm(sizes, case["inner"], case["outer"], gen)
        csr = _host(_csr(sum(sizes), u, v, case["weighted"], gen))
        return dict(case=case, csr=(np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64),) + csr, stream=_stream(case))
    if kind == "serve":
        graphs = [_host(_csr(1 << s, *_rmat(1 << s, ef, gen), case["weighted"], gen)) for s, ef in _requests(case)]
        return dict(case=case, graphs=graphs, server=na.Server(slots=8, nbatches=case["nb"], tol=TOL, group=64))
    csr = _host(_graph(case, gen))
    s = dict(case=case, csr=csr, stream=_stream(case))
    if kind in ("phase", "steps"):
        s["handle"] = na.GraphGPU(csr, case["nb"], stream=_handle(s["stream"]))
    return s


def _stream(case):
    return torch.cuda.Stream() if case.get("stream") else None


def _handle(stream):
    return stream.cuda_stream if stream else None


# ---- one pass ----------------------------------------------------------------
def _run_whole(csr, nb, stream, window=0):
    g = na.GraphGPU(csr, nb, stream=_handle(stream), window=window)
    st = na.LouvainGPU(tol=TOL, nbatches=nb).run(g)
    out = dict(clustering=g.clustering(), q=st.q, phases=st.phases, loops=st.total_loops)
    g.close()
    return out


def _run_phase(g):
    g.singleton_partition()
    q0 = q = g.compute_modularity()
    dq, loops = 1.0, 0
    while dq > TOL and loops < na.DEFAULT_ITERATIONS:
        q, dq, _ = g.louvain_iteration(q)
        loops += 1
    return dict(q0=q0, q=q, loops=loops, communities=g.communities(), totals=g.community_weights())


def _run_steps(g, nb):
    g.singleton_partition()
    q0 = q = g.compute_modularity()
    dq, loops = 1.0, 0
    while dq > TOL and loops < na.DEFAULT_ITERATIONS:
        for b in range(nb):
            g.louvain_update(b)
            g.update_community_weights(b)
            g.update_community_ids(b)
        now = g.compute_modularity()
        dq = now - q
        loops += 1
        if dq < 0:
            g.restore_community()
        else:
            q = now
    return dict(q0=q0, q=q, loops=loops, communities=g.communities(), totals=g.community_weights())


def _run_batch(csr, nb, stream):
    b = na.BatchGPU(csr=csr, nbatches=nb, stream=_handle(stream))
    b.run(tol=TOL)
    q = np.array([b.graph_stats(i).q for i in range(b.ngraphs)])
    out = dict(clustering=np.concatenate([b.clustering(i) for i in range(b.ngraphs)]), q=q)
    b.close()
    return out


def _run_serve(server, graphs):
    ids = [server.submit(g, borrow=True) for g in graphs]
    q, parts = [], []
    for i in ids:
        st, _ = server.wait(i)
        q.append(st.q)
        parts.append(server.clustering(i))
        server.release(i)
    return dict(clustering=np.concatenate(parts), q=np.array(q))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        return _run_whole(state["csr"], case["nb"], state["stream"])
    if kind == "window":
        return _run_whole(state["csr"], case["nb"], state["stream"], window=_window(state["csr"][0], case["parts"]))
    if kind == "phase":
        return _run_phase(state["handle"])
    if kind == "steps":
        return _run_steps(state["handle"], case["nb"])
    if kind == "batch":
        return _run_batch(state["csr"], case["nb"], state["stream"])
    if kind == "serve":
        return _run_serve(state["server"], state["graphs"])
    s = state
    na.modularity_noalloc(case["n"], s["col"].numel(), s["off"].data_ptr(), s["col"].data_ptr(), s["w"].data_ptr(),
                          s["comm"].data_ptr(), s["q"].data_ptr(), torch.cuda.current_stream().cuda_stream)
    return s["q"]


def _window(off, parts):
    """Arcs of a window that holds 1/parts of the graph, and any one row."""
    return max(int(off[-1]) // parts + 1, int(np.max(np.diff(off))))


# ---- the least that a pass reads and writes, and its values in 64 bits -----------
def _shape(case):
    """(vertices, arcs) of one input, about."""
    if case["kind"] == "batch":
        n = sum(_sizes(case))
    elif case["kind"] == "serve":
        r = _requests(case)
        return sum(1 << s for s, _ in r), sum(2 * ef << s for s, ef in r)
    else:
        n = case["n"]
    degree = 2 * case["ef"] if case.get("graph") == "rmat" else case["mean"] if "mean" in case else case["inner"] + case["outer"]
    return n, int(n * degree)


def work(case):
    """The CSR read once (int64 offsets and ids, FP64 weights), one int64 per
    vertex written; one addition per arc."""
    n, m = _shape(case)
    per_vertex = 24 if case["kind"] in ("phase", "steps") else 16
    return {"bytes": 16 * m + per_vertex * n, "flops": m}


def exact(case, seed):
    """Modularities that follow from the input alone; the partitions a run
    finds, and theirs, are its own."""
    kind = case["kind"]
    if kind not in ("phase", "steps", "modularity"):
        return None
    gen = torch.Generator(device=DEV).manual_seed(int(seed) + 1)
    if kind == "modularity":
        s = prepare(case, seed)
        off, col, w, comm = (s[k].cpu().numpy() for k in ("off", "col", "w", "comm"))
    else:
        off, col, w = _host(_graph(case, gen))
        comm = np.arange(case["n"])
    src = np.repeat(np.arange(case["n"]), np.diff(off))
    twom = w.sum()
    totals = np.bincount(comm[src], weights=w, minlength=case["n"])
    q = w[comm[src] == comm[col]].sum() / twom - np.square(totals / twom).sum()
    if kind == "modularity":
        return np.array([q])
    return dict(q0=float(q), q=None, loops=None, communities=None, totals=None)
