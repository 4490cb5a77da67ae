"""Performance cases: the calls that a user of the framework makes, over the
sizes and options they are made with.

Graphs are the two families that the benchmark and the tests run: R-MAT
(a, b, c = .57, .19, .19, duplicate arcs and self-loops removed, weights
[1, 100]; here also with a vertex count that is no power of two) and
4-neighbour grids, both arc directions, with or without random shortcut edges
(weights [1, 1000]).  They are made on the GPU from the seed and handed to the
framework as host CSR arrays, the form in which its constructor takes them.

A case's "out" says where the program wants the result: "host" (the array that
the call returns), "device" (left in the graph's device buffer, read in place)
or "caller" (the caller's own device buffer).
"""
import ctypes
import math

import numpy as np
import torch

import gpugraphalgo_amd as gga
from gpugraphalgo_amd import _lib
from gpugraphalgo_amd.serve import TRACE_DTYPE, Server

DEVICE = "cuda"
INF = 0xFFFFFFFF


def listed():
    return [
        # A small mesh (a city's streets) asked one route table at a time: each
        # call is hundreds of thin steps, so latency is everything.
        {"name": "sssp_mesh_small", "do": "sssp", "family": "grid", "rows": 100, "cols": 77, "cut": 0.0,
         "level": 0, "mda": 0, "out": "host"},
        # The smallest R-MAT configuration of the tests: BFS on 2^14 vertices.
        {"name": "bfs_rmat14", "do": "bfs", "family": "rmat", "n": 1 << 14, "ef": 16, "level": 0, "mda": 32,
         "out": "host"},
        # A mid-size social graph, odd vertex count, split by the histogram
        # rule, distances into the caller's own buffer (no allocation).
        {"name": "sssp_rmat17_caller", "do": "sssp", "family": "rmat", "n": 131071, "ef": 16, "level": -1, "mda": 0,
         "out": "caller"},
        # BFS levels of a sparser graph of 1.5 M vertices, unsplit (hubs whole),
        # as an array on the host.
        {"name": "bfs_rmat1500k_host", "do": "bfs", "family": "rmat", "n": 1500001, "ef": 8, "level": 0, "mda": 0,
         "out": "host"},
        # The headline configuration: SSSP on R-MAT s22, ef 16, T = 128, the
        # result left on the device; and BFS on the same graph.
        {"name": "sssp_rmat22", "do": "sssp", "family": "rmat", "n": 1 << 22, "ef": 16, "level": 0, "mda": 128,
         "out": "device"},
        {"name": "bfs_rmat22", "do": "bfs", "family": "rmat", "n": 1 << 22, "ef": 16, "level": 0, "mda": 128,
         "out": "device"},
        # A road-like mesh without shortcuts: thousands of hops across.
        {"name": "sssp_mesh_1m", "do": "sssp", "family": "grid", "rows": 1024, "cols": 1024, "cut": 0.0, "level": 0,
         "mda": 0, "out": "device"},
        # The large grid with 0.5% shortcuts of the benchmark's second leg.
        {"name": "sssp_grid4096_shortcuts", "do": "sssp", "family": "grid", "rows": 4096, "cols": 4096,
         "cut": 0.005, "level": 0, "mda": 0, "out": "device"},
        # All-pairs style work: levels from 256 sources of a small graph at
        # once, as one host array.
        {"name": "multi_bfs_rmat16", "do": "multi_bfs", "family": "rmat", "n": 1 << 16, "ef": 16, "level": 0,
         "mda": 64, "lanes": 256, "out": "host"},
        # 32 SSSP lanes of one engine on R-MAT s20 (steps replayed from
        # captured graphs), the distances fetched into device buffers.
        {"name": "engine_sssp32_rmat20", "do": "engine", "family": "rmat", "n": 1 << 20, "ef": 16, "level": 0,
         "mda": 16, "lanes": 32, "bfs": 0, "out": "device"},
        # Serving: a burst of mixed BFS / SSSP queries on two R-MAT graphs and
        # two grids, each answer into a device buffer.
        {"name": "serve_burst", "do": "serve", "family": "mixed", "scale": 16, "side": 512, "queries": 48,
         "out": "device"},
        # Node splitting of a resident graph by level, the chunk table read
        # back (the preprocessing that the reference does on the host).
        {"name": "split_rmat20", "do": "split", "family": "rmat", "n": 1 << 20, "ef": 16, "level": 512, "mda": 0,
         "out": "host"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    do = rng.choice(["bfs", "bfs", "sssp", "sssp", "sssp", "multi_bfs", "engine", "serve", "split"])
    if do == "serve":
        return {"do": do, "family": "mixed", "scale": rng.randint(13, 16), "side": rng.randint(64, 512),
                "queries": rng.randint(4, 48), "out": "device"}
    c = {"do": do, "level": 0, "mda": rng.choice([0, 16, 32, 64, 128, 256, 1024])}
    if do in ("bfs", "sssp") and rng.random() < 0.45:
        c.update(family="grid", mda=0, cut=rng.choice([0.0, 0.005]))
        top = 1024 if c["cut"] == 0.0 else 4096
        c.update(rows=_log_int(rng, 16, top), cols=_log_int(rng, 16, top))
    else:
        c.update(family="rmat", ef=rng.randint(4, 20))
        top = {"multi_bfs": 1 << 18, "engine": 1 << 20}.get(do, 1 << 22)
        c["n"] = min(_log_int(rng, 1 << 10, top), (1 << 26) // c["ef"])
        if c["mda"] == 0 and rng.random() < 0.7:
            c["level"] = rng.choice([-1, 8, 64, 512])
    c["out"] = "host"
    if do in ("bfs", "sssp"):
        c["out"] = rng.choice(["host", "device"])
        # the allocation-free form is for split graphs within its fixed workspace
        if do == "sssp" and rng.random() < 0.3 and c.get("n", c.get("rows", 0) * c.get("cols", 0)) <= 1 << 20:
            c["out"] = "caller"
    elif do == "multi_bfs":
        c["lanes"] = min(256, max(1, (1 << 24) // c["n"]), _log_int(rng, 1, 256))
    elif do == "engine":
        c.update(lanes=rng.randint(2, 32), out="device")
        c["bfs"] = rng.choice([0, c["lanes"] // 2])
    return c


# ------------------------------------------------------------------ inputs
def _csr(n, u, v, w):
    row = torch.zeros(n + 1, dtype=torch.int64, device=DEVICE)
    row[1:] = torch.cumsum(torch.bincount(u, minlength=n), 0)
    return [x.to(torch.int32).cpu().numpy().view(np.uint32) for x in (row, v, w)]


def _rmat(n, ef, gen):
    """Arcs (u, v, w) of an R-MAT graph, sorted by (u, v); ids >= n are left out."""
    arcs = n * ef
    u = torch.zeros(arcs, dtype=torch.int64, device=DEVICE)
    v = torch.zeros(arcs, dtype=torch.int64, device=DEVICE)
    for _ in range(max(1, (n - 1).bit_length())):
        r = torch.rand(arcs, device=DEVICE, generator=gen)
        u = 2 * u + (r >= 0.76)
        v = 2 * v + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    key = torch.unique((u * n + v)[(u < n) & (v < n) & (u != v)])
    u, v = key // n, key % n
    w = torch.randint(1, 101, (u.numel(),), device=DEVICE, generator=gen)
    return u, v, w


def _grid(rows, cols, cut, gen):
    n = rows * cols
    i = torch.arange(n, device=DEVICE)
    a = torch.cat([i[i % cols != cols - 1], i[i < n - cols]])
    b = torch.cat([i[i % cols != cols - 1] + 1, i[i < n - cols] + cols])
    extra = int(round(cut * a.numel()))
    if extra:
        x = torch.randint(0, n, (extra,), device=DEVICE, generator=gen)
        y = torch.randint(0, n, (extra,), device=DEVICE, generator=gen)
        x, y = x[x != y], y[x != y]
        a, b = torch.cat([a, torch.minimum(x, y)]), torch.cat([b, torch.maximum(x, y)])
    key = torch.unique(a * n + b)
    a, b = key // n, key % n
    w = torch.randint(1, 1001, (a.numel(),), device=DEVICE, generator=gen)
    u, v, w = torch.cat([a, b]), torch.cat([b, a]), torch.cat([w, w])
    order = torch.argsort(u * n + v)
    return u[order], v[order], w[order]


def _graph(case, gen):
    """(n, u, v, w) on the GPU."""
    if case["family"] == "grid":
        return (case["rows"] * case["cols"],) + _grid(case["rows"], case["cols"], case["cut"], gen)
    return (case["n"],) + _rmat(case["n"], case["ef"], gen)


def _sources(n, u, k, gen):
    """k sources among the vertices with out-edges (distinct where there are k)."""
    cand = torch.unique_consecutive(u)
    at = torch.randperm(cand.numel(), device=DEVICE, generator=gen)[:k]
    at = at.repeat(-(-k // at.numel()))[:k]
    return [int(x) for x in cand[at].cpu()]


def _resident(n, u, v, w, mda=0, level=0):
    dg = gga.DeviceGraph(gga.csr_from_arrays(*_csr(n, u, v, w)))
    dg.split(mda=mda, level=level)
    return dg


def _mixed(case, gen):
    """The served graphs: two R-MAT, two grids."""
    s, a = case["scale"], case["side"]
    return [(1 << s,) + _rmat(1 << s, 16, gen), (3 << (s - 2),) + _rmat(3 << (s - 2), 16, gen),
            (a * a,) + _grid(a, a, 0.0, gen), ((a // 2) * a,) + _grid(a // 2, a, 0.005, gen)]


def _trace(case, graphs, gen):
    """(graph, source, bfs) of each query: the graphs in turn, half of them BFS."""
    k = case["queries"]
    which = [i % len(graphs) for i in range(k)]
    bfs = torch.randint(0, 2, (k,), device=DEVICE, generator=gen).tolist()
    pool = [_sources(n, u, k, gen) for n, u, _, _ in graphs]
    return [(g, pool[g][i], bfs[i]) for i, g in enumerate(which)]


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def prepare(case, seed):
    gen = _generator(seed)
    if case["do"] == "serve":
        graphs = _mixed(case, gen)
        queries = _trace(case, graphs, gen)
        dgs = [_resident(*g, mda=64 if i < 2 else 0) for i, g in enumerate(graphs)]
        srv = Server(use_graph=True)
        for dg in dgs:
            srv.add_graph(dg)
        trace = np.zeros(len(queries), dtype=TRACE_DTYPE)
        for i, (g, src, bfs) in enumerate(queries):
            trace[i] = (g, src, bfs, 0.0)
        out = [torch.empty(graphs[g][0], dtype=torch.int32, device=DEVICE) for g, _, _ in queries]
        return {"case": case, "dgs": dgs, "srv": srv, "trace": trace, "out": out}
    n, u, v, w = _graph(case, gen)
    lanes = case.get("lanes", 1)
    srcs = _sources(n, u, lanes, gen)
    s = {"case": case, "n": n, "src": srcs}
    s["dg"] = _resident(n, u, v, w, mda=case["mda"], level=case["level"])
    if case["do"] == "engine":
        s["eng"] = gga.MultiSourceEngine(s["dg"])
        s["bfs"] = set(range(case["bfs"]))
        s["out"] = torch.empty((lanes, n), dtype=torch.int32, device=DEVICE)
        s["ptrs"] = (ctypes.c_void_p * gga.MultiSourceEngine.LANES)()
        for i in range(lanes):
            s["ptrs"][i] = s["out"][i].data_ptr()
    elif case["out"] == "caller":
        s["out"] = torch.empty(n, dtype=torch.int32, device=DEVICE)
        s["opts"], s["stats"] = _lib.Opts(), _lib.Stats()
        s["opts"].mode, s["opts"].inf = _lib.MODES["auto"], INF
    elif case["do"] == "split":
        # host arrays for a chunk table of any threshold (at most n + m chunks)
        s["begin"], s["own"] = (np.zeros(n * (1 + case["ef"]) + 1, dtype=np.int32) for _ in range(2))
    return s


# -------------------------------------------------------------------- calls
class _InPlace:
    """The graph's device result as torch reads foreign device memory (the
    tensor made from it keeps the graph alive)."""

    def __init__(self, dg):
        self.dg = dg
        ptr = int(_lib.load().gga_graph_dist_device(dg._h))
        self.__cuda_array_interface__ = {"shape": (dg.n,), "typestr": "<i4", "data": (ptr, False), "version": 2}


def run(s):
    case = s["case"]
    do = case["do"]
    if do == "serve":
        s["srv"].replay(s["trace"], outs=[(t.data_ptr(),) for t in s["out"]])
        return s["out"]
    dg = s["dg"]
    if do in ("bfs", "sssp"):
        if case["out"] == "caller":
            _lib.check(_lib.load().gga_sssp_noalloc(dg._h, s["src"][0], s["out"].data_ptr(), ctypes.byref(s["opts"]),
                                                    ctypes.byref(s["stats"])), "gga_sssp_noalloc")
            return s["out"]
        call = dg.bfs if do == "bfs" else dg.sssp
        if case["out"] == "host":
            return call(s["src"][0])[0].view(np.int32)
        call(s["src"][0], keep_on_device=True)
        return torch.as_tensor(_InPlace(dg), device=DEVICE)
    if do == "multi_bfs":
        return dg.multi_bfs(s["src"])[0].view(np.int32)
    if do == "engine":
        eng, k = s["eng"], case["lanes"]
        eng.start(dict(enumerate(s["src"])), bfs=s["bfs"])
        eng.run(use_graph=1)
        _lib.check(_lib.load().gga_ms_fetch(eng._h, (1 << k) - 1, s["ptrs"], 1), "gga_ms_fetch")
        return s["out"]
    dg.split(mda=case["mda"], level=case["level"])
    _lib.check(_lib.load().gga_graph_chunks(dg._h, s["begin"].ctypes.data, s["own"].ctypes.data), "gga_graph_chunks")
    return [s["begin"], s["own"]]


# ------------------------------------------------------- what a pass needs
def _size(case):
    """(vertices, arcs) up to the few duplicate arcs."""
    if case["family"] == "grid":
        n = case["rows"] * case["cols"]
        return n, int(4 * n * (1 + case["cut"]))
    return case["n"], case["n"] * case["ef"]


def work(case):
    """Offsets, destinations and (SSSP) weights read once, results written once."""
    if case["do"] == "serve":
        per = [((1 << case["scale"]) * k // 4, 16) for k in (4, 3)]
        per += [(case["side"] ** 2 * k // 2, 4) for k in (2, 1)]
        n = sum(x for x, _ in per) / 4
        m = sum(x * d for x, d in per) / 4
        return {"bytes": case["queries"] * (8 * n + 6 * m), "flops": case["queries"] * m}
    n, m = _size(case)
    k = case.get("lanes", 1)
    if case["do"] == "split":
        return {"bytes": 4 * n + 4 * n + 8 * n, "flops": n}
    edge = 4 if case["do"] in ("bfs", "multi_bfs") else 8
    return {"bytes": 4 * n + edge * m + 4 * n * k, "flops": m * k}


# ----------------------------------------------------------- plain results
def _distances(n, u, v, w, srcs, hops):
    """Bellman-Ford in 64 bits, one source after another."""
    got = []
    for src, hop in zip(srcs, hops):
        d = torch.full((n,), 1 << 62, dtype=torch.int64, device=DEVICE)
        d[src] = 0
        step = torch.ones_like(w) if hop else w
        while True:
            before = d.clone()
            for _ in range(8):
                d = d.scatter_reduce(0, v, d[u] + step, "amin")
            if torch.equal(before, d):
                break
        got.append(torch.where(d >= INF, torch.tensor(INF, device=DEVICE), d).to(torch.int32))
    return got


def exact(case, seed):
    gen = _generator(seed)
    if case["do"] == "serve":
        graphs = _mixed(case, gen)
        return [_distances(*graphs[g], [src], [bfs])[0] for g, src, bfs in _trace(case, graphs, gen)]
    n, u, v, w = _graph(case, gen)
    srcs = _sources(n, u, case.get("lanes", 1), gen)
    if case["do"] == "split":
        deg = torch.bincount(u, minlength=n)
        most = int(deg.max())
        if case["mda"]:
            mda = case["mda"]
        elif case["level"] >= 0:
            mda = -(-most // case["level"]) if case["level"] else most
        else:
            return None   # the histogram rule works in 32-bit floats
        count = torch.clamp((deg + mda - 1) // mda, min=1)
        size = (deg + count - 1) // count
        own = torch.repeat_interleave(torch.arange(n, device=DEVICE), count)
        rank = torch.arange(own.numel(), device=DEVICE) - (torch.cumsum(count, 0) - count)[own]
        begin = (torch.cumsum(deg, 0) - deg)[own] + rank * size[own]
        table = torch.zeros((2, n * (1 + case["ef"]) + 1), dtype=torch.int32, device=DEVICE)
        table[0, : own.numel() + 1] = torch.cat([begin, deg.sum()[None]])
        table[1, : own.numel()] = own
        return list(table)
    if case["do"] in ("bfs", "multi_bfs"):
        hops = [True] * len(srcs)
    else:
        hops = [i < case.get("bfs", 0) for i in range(len(srcs))]
    got = _distances(n, u, v, w, srcs, hops)
    return torch.stack(got) if "lanes" in case else got[0]
