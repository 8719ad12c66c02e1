"""Performance cases: the work users have the partitioner do, each through a public entry point.

Whole calls (most of what a program does with the library):
  host      gk_partition           host CSR in, host partition out, copies included
  device    gk_partition_device    CSR already on the GPU, partition stays there
  packed    gk_partition_packed    many graphs in one packed CSR, with the launch options the batched form is run with
  serve     gk_serve_*             a burst of requests submitted together, every result waited for
Single stages, as a program calls them that drives its own multilevel loop:
  coarsen   gk_k_match, gk_k_group, gk_k_cluster, gk_k_contract: one coarsening level
  refine    gk_k_project, gk_k_gain, gk_k_round, gk_k_cut: one uncoarsening level
  cut       gk_k_cut_noalloc       cut and part weights of a given partition, no allocation and no synchronisation

Graph families are the ones the library is tested and benchmarked on: 2-D Delaunay meshes (uniform points numbered in
drawing order, or along a Hilbert curve), road networks, layered circuit-like DAGs with weights, and triangulated grids
(the same degrees as a Delaunay mesh, made on the GPU, numbered row by row or at random).
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The package (its folder's name is no identifier), loaded once."""
    if "gkway_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location("gkway_amd", os.path.join(ROOT, "dac_g-kway_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules["gkway_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["gkway_amd"]


gk = _package()
_held = {}


def _context():
    """One context for the whole program, as a program keeps it."""
    if "context" not in _held:
        _held["context"] = gk.Context(0)
    return _held["context"]


def _server():
    """One request loop for the whole program."""
    if "server" not in _held:
        _held["server"] = gk.Server(0)
    return _held["server"]


def listed():
    return [
        # A partition's quality looked up inside a loop that may not allocate: launches and latency count.
        {"name": "cut_small", "what": "cut", "graph": "grid", "n": 20011, "k": 16, "weighted": False, "shuffled": False},
        # The size of the reference's sample graph (delaunay_n11), a few parts: the smallest whole call.
        {"name": "host_small", "what": "host", "graph": "delaunay", "n": 2048, "k": 4},
        # An ordinary mesh from a program that holds it in host memory.
        {"name": "host_mesh", "what": "host", "graph": "hilbert", "n": 100003, "k": 32},
        # An ordinary mesh already on the GPU, vertices numbered without locality.
        {"name": "device_mesh", "what": "device", "graph": "delaunay", "n": 400009, "k": 64},
        # The headline single graph's size: 2^22 vertices, 12.6 M edges, 64 parts, numbered without locality.
        {"name": "device_mesh_large", "what": "device", "graph": "grid", "n": 4194304, "k": 64, "weighted": False,
         "shuffled": True},
        # A road network: degree 2.1, long chains, many parts.
        {"name": "device_road", "what": "device", "graph": "road", "n": 600011, "k": 256},
        # A circuit-like DAG, weighted, hubs, many parts: hundreds to thousands of refinement rounds.
        {"name": "device_dag", "what": "device", "graph": "dag", "n": 300007, "k": 256},
        # Many small graphs at once, as the batched benchmark draws them.
        {"name": "packed_batch", "what": "packed", "count": 160, "lo": 500, "hi": 50000},
        # A burst of requests to the serving loop.
        {"name": "serve_burst", "what": "serve", "count": 24, "lo": 1000, "hi": 60000},
        # One level of coarsening: the first and largest of the headline mesh, and of a weighted DAG with hubs.
        {"name": "coarsen_mesh", "what": "coarsen", "graph": "grid", "n": 4194304, "weighted": False, "shuffled": True},
        {"name": "coarsen_dag", "what": "coarsen", "graph": "dag", "n": 1000003},
        # One level of uncoarsening: projection, gains, eight refinement rounds, the cut.
        {"name": "refine_mesh", "what": "refine", "graph": "grid", "n": 2000003, "k": 64, "weighted": True,
         "shuffled": False, "rounds": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges: sizes spread over their logarithm, odd ones among them."""
    what = rng.choice(["host", "device", "device", "packed", "serve", "coarsen", "coarsen", "refine", "refine", "cut"])
    ks = [2, 4, 8, 16, 32, 64, 128, 256]
    if what == "packed":
        return {"what": what, "count": _log_int(rng, 8, 160), "lo": 500, "hi": _log_int(rng, 2000, 50000)}
    if what == "serve":
        return {"what": what, "count": _log_int(rng, 2, 24), "lo": 1000, "hi": _log_int(rng, 3000, 60000)}
    grid = {"graph": "grid", "weighted": rng.random() < 0.5, "shuffled": rng.random() < 0.5}
    if what == "cut":
        return {"what": what, "n": _log_int(rng, 2000, 4194304), "k": rng.choice(ks), **grid}
    if what == "refine":
        return {"what": what, "n": _log_int(rng, 20000, 2000003), "k": rng.choice(ks), "rounds": rng.randint(2, 8), **grid}
    graph = rng.choice(["delaunay", "hilbert", "road", "dag", "grid"])
    if what == "coarsen":
        case = {"what": what, "n": _log_int(rng, 4000, 4194304 if graph == "grid" else 600000)}
    else:
        most = {"delaunay": 400000, "hilbert": 300000, "road": 400000, "dag": 200000, "grid": 3000000}[graph]
        case = {"what": what, "n": _log_int(rng, 2000, most if what == "device" else min(most, 200000))}
        case["k"] = rng.choice([k for k in ks if k * 200 <= case["n"]])
    return {**case, **(grid if graph == "grid" else {"graph": graph})}


# ---------------------------------------------------------------- graphs
def _grid(n, seed, weighted, shuffled):
    """Triangulated grid of n vertices, one diagonal of each cell at random, as device tensors (xadj, adj, w, vw) and the
    row and column of every vertex.  Row by row numbering, or a random one."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    cols = max(2, int(math.sqrt(n)))
    v = torch.arange(n, device="cuda")
    row, col = v // cols, v % cols
    turn = torch.randint(0, 2, (n,), generator=gen, device="cuda").bool()
    inner = col < cols - 1
    ends = [(v, v + 1, inner), (v, v + cols, torch.ones_like(inner)), (v, v + cols + 1, inner & turn),
            (v + 1, v + cols, inner & ~turn)]
    a = torch.cat([x[keep] for x, _, keep in ends])
    b = torch.cat([y[keep] for _, y, keep in ends])
    inside = (a < n) & (b < n)
    a, b = a[inside], b[inside]
    if shuffled:
        name = torch.randperm(n, generator=gen, device="cuda")
        a, b = name[a], name[b]
        back = torch.empty_like(name)
        back[name] = v
        row, col = row[back], col[back]
    if weighted:
        w = torch.randint(1, 101, (len(a),), generator=gen, device="cuda", dtype=torch.int32)
        vw = torch.randint(1, 5, (n,), generator=gen, device="cuda", dtype=torch.int32)
    else:
        w = torch.ones(len(a), dtype=torch.int32, device="cuda")
        vw = torch.ones(n, dtype=torch.int32, device="cuda")
    key, at = torch.sort(torch.cat([a * n + b, b * n + a]))
    xadj = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    xadj[1:] = torch.cumsum(torch.bincount(key // n, minlength=n), 0)
    return (xadj.int(), (key % n).int(), torch.cat([w, w])[at].contiguous(), vw), row, col


def _family(graph, n, seed):
    """A graph of the library's generators, in host memory."""
    if graph == "delaunay":
        return gk.delaunay(n, seed)
    if graph == "hilbert":
        return gk.delaunay_hilbert(n, seed)
    if graph == "road":
        return gk.road(n, seed)
    return gk.dag(n, int(min(200, max(2, round(math.sqrt(n))))), seed)


def _host_graph(case, seed):
    if case["graph"] != "grid":
        return _family(case["graph"], case["n"], seed)
    arrays, _, _ = _grid(case["n"], seed, case["weighted"], case["shuffled"])
    return gk.Graph(*(t.cpu().numpy() for t in arrays))


def _device_graph(case, seed):
    if case["graph"] == "grid":
        return _grid(case["n"], seed, case["weighted"], case["shuffled"])[0]
    g = _family(case["graph"], case["n"], seed)
    return tuple(torch.from_numpy(x).cuda() for x in (g.xadj, g.adjncy, g.adjwgt, g.vwgt))


def _set(case, seed):
    """Graphs of a batch or a burst: vertex counts spread evenly over the logarithm of [lo, hi] (the same for every
    seed), meshes and DAGs in turn; and their part counts."""
    count, lo, hi = case["count"], case["lo"], case["hi"]
    ks = [2, 4, 8, 16, 32] if case["what"] == "packed" else [8, 16, 64]
    graphs, parts = [], []
    for i in range(count):
        n = int(lo * (hi / lo) ** ((i * 0.6180339887) % 1.0))
        graphs.append(_family("delaunay" if i % 2 == 0 else "dag", n, seed * 1000003 + i))
        parts.append(ks[(i * 7 + seed) % len(ks)])
    return graphs, parts


def _ptr(t):
    return ctypes.cast(t.data_ptr(), gk.I32P)


def _csr(arrays):
    c = gk.Csr()
    c.n, c.nnz = len(arrays[0]) - 1, len(arrays[1])
    c.xadj, c.adjncy, c.adjwgt, c.vwgt = (_ptr(t) for t in arrays)
    return c


def _room(case, nnz):
    """Coarse entries a coarsening level's buffers hold: the fine level's, and the same for every graph of a case."""
    return max(nnz, 8 * case["n"])


def _ints(n):
    return torch.zeros(max(1, n), dtype=torch.int32, device="cuda")


# ---------------------------------------------------------------- inputs
def prepare(case, seed):
    what = case["what"]
    state = {"what": what}
    if what == "host":
        state.update(ctx=_context(), graph=_host_graph(case, seed), k=case["k"])
    elif what == "device":
        arrays = _device_graph(case, seed)
        state.update(ctx=_context(), arrays=arrays, csr=_csr(arrays), params=gk.params(case["k"]),
                     part=_ints(len(arrays[3])))
    elif what == "packed":
        graphs, ks = _set(case, seed)
        pack, v_off, e_off = gk.pack_graphs(graphs)
        arrays = tuple(torch.from_numpy(x).cuda() for x in (pack.xadj, pack.adjncy, pack.adjwgt, pack.vwgt))
        p = gk.PackedCsr()
        p.ngraphs, p.n, p.nnz = len(graphs), pack.n, pack.nnz
        p.xadj, p.adjncy, p.adjwgt, p.vwgt = (_ptr(t) for t in arrays)
        p.v_off, p.e_off = v_off.ctypes.data_as(gk.I32P), e_off.ctypes.data_as(gk.I32P)
        flags = gk.GK_FLAG_PERSISTENT | gk.GK_FLAG_GRAPH_ROUNDS | gk.GK_FLAG_AUTOTUNE
        state.update(ctx=_context(), arrays=arrays, offsets=(v_off, e_off), pack=p, part=_ints(pack.n),
                     params=(gk.Params * len(ks))(*[gk.params(k, flags=flags) for k in ks]),
                     stats=(gk.Stats * len(ks))())
    elif what == "serve":
        graphs, ks = _set(case, seed)
        state.update(server=_server(), graphs=graphs, ks=ks)
    elif what == "coarsen":
        arrays = _device_graph(case, seed)
        n, nnz = len(arrays[3]), _room(case, len(arrays[1]))
        state.update(ctx=_context(), arrays=arrays, csr=_csr(arrays))
        state.update({name: _ints(n) for name in ("cand", "label", "stamp", "order", "cmap", "cvwgt")})
        state.update(cxadj=_ints(n + 1), cadjncy=_ints(nnz), cadjwgt=_ints(nnz))
    elif what == "refine":
        state.update(_refine_inputs(case, seed))
    else:
        arrays, row, col = _grid(case["n"], seed, case["weighted"], case["shuffled"])
        state.update(ctx=_context(), arrays=arrays, csr=_csr(arrays), k=case["k"], part=_blocks(row, col, case["k"], seed),
                     cut=torch.zeros(1, dtype=torch.int64, device="cuda"),
                     weights=torch.zeros(case["k"], dtype=torch.int64, device="cuda"), stream=torch.cuda.Stream())
    torch.cuda.synchronize()
    return state


def _blocks(row, col, k, seed):
    """A partition of the grid into k blocks with ragged borders, as a coarser level leaves it."""
    gen = torch.Generator(device="cuda").manual_seed(seed + 17)
    down = 2 ** (int(math.log2(k)) // 2)
    across = k // down
    rows, cols = int(row.max()) + 1, int(col.max()) + 1
    sway = 3.0
    noise = torch.rand(2, len(row), generator=gen, device="cuda", dtype=torch.float64) - 0.5
    r = (row.double() + sway * noise[0]).clamp(0, rows - 1)
    c = (col.double() + sway * noise[1]).clamp(0, cols - 1)
    return ((r * down / rows).long().clamp(max=down - 1) * across + (c * across / cols).long().clamp(max=across - 1)).int()


def _refine_inputs(case, seed):
    """A level to refine: the fine graph, its map onto coarse vertices of two by two cells, and their partition."""
    arrays, row, col = _grid(case["n"], seed, case["weighted"], case["shuffled"])
    k, n = case["k"], case["n"]
    cell = (row // 2) * (int(col.max()) // 2 + 1) + col // 2
    _, cmap = torch.unique(cell, return_inverse=True)
    nc = int(cmap.max()) + 1
    crow = torch.zeros(nc, dtype=torch.int64, device="cuda").index_copy_(0, cmap, row // 2)
    ccol = torch.zeros(nc, dtype=torch.int64, device="cuda").index_copy_(0, cmap, col // 2)
    cpart = _blocks(crow, ccol, k, seed)
    xadj, adj, _, vw = arrays
    src = torch.repeat_interleave(torch.arange(n, device="cuda"), (xadj[1:] - xadj[:-1]).long())
    part = cpart[cmap]
    differs = part[src] != part[adj.long()]
    cbnd = torch.zeros(nc, dtype=torch.int32, device="cuda")
    cbnd[cmap[src[differs]]] = 1
    pw = torch.bincount(part.long(), weights=vw.double(), minlength=k).int()
    # Blocks of one partition differ in weight by their share of the ragged rows: the cap leaves 3% above the heaviest.
    cap = int(int(pw.max()) * 1.03)
    state = dict(ctx=_context(), arrays=arrays, csr=_csr(arrays), k=k, rounds=case["rounds"], cap=cap, cmap=cmap.int(),
                 cpart=cpart, cbnd=cbnd, pw0=pw, pw=torch.empty_like(pw), stream=torch.cuda.Stream(),
                 nmoves=np.zeros(case["rounds"], np.int32), pos=np.zeros(case["rounds"], np.int32))
    state.update({name: _ints(n) for name in ("part", "bnd", "gain", "dest", "updated")})
    return state


# ---------------------------------------------------------------- passes
def _ok(status):
    if status != gk.GK_OK:
        raise RuntimeError(f"{gk.lib().gk_strerror(status).decode()}: {gk.lib().gk_last_error().decode()}")


def run(state):
    return _RUNS[state["what"]](state)


def _run_host(s):
    part, stats = s["ctx"].partition(s["graph"], s["k"])
    return {"part": part, "cut": stats.cut}


def _run_device(s):
    stats = gk.Stats()
    _ok(gk.lib().gk_partition_device(s["ctx"].handle, ctypes.byref(s["csr"]), ctypes.byref(s["params"]), _ptr(s["part"]),
                                     ctypes.byref(stats), None))
    return {"part": s["part"], "cut": stats.cut}


def _run_packed(s):
    _ok(gk.lib().gk_partition_packed(s["ctx"].handle, ctypes.byref(s["pack"]), s["params"], _ptr(s["part"]), s["stats"], None))
    return {"part": s["part"], "cuts": np.array([x.cut for x in s["stats"]], np.int64)}


def _run_serve(s):
    ids = s["server"].submit_many(s["graphs"], s["ks"])
    done = [s["server"].wait(i) for i in ids]
    return {"part": np.concatenate([part for part, _ in done]), "cuts": np.array([st.cut for _, st in done], np.int64)}


def _run_coarsen(s):
    L, h, c = gk.lib(), s["ctx"].handle, ctypes.byref(s["csr"])
    n = s["csr"].n
    sweeps, nc, nnz = ctypes.c_int32(), ctypes.c_int32(), ctypes.c_int32()
    p = {name: _ptr(s[name]) for name in ("cand", "label", "stamp", "order", "cmap", "cvwgt", "cxadj", "cadjncy", "cadjwgt")}
    _ok(L.gk_k_match(h, c, p["cand"], None))
    _ok(L.gk_k_group(h, n, p["cand"], p["label"], p["stamp"], ctypes.byref(sweeps), None))
    _ok(L.gk_k_cluster(h, n, p["label"], p["stamp"], s["csr"].vwgt, 6, p["order"], p["cmap"], p["cvwgt"], ctypes.byref(nc), None))
    _ok(L.gk_k_contract(h, c, p["cmap"], nc, p["cxadj"], p["cadjncy"], p["cadjwgt"], ctypes.byref(nnz), None))
    out = {name: s[name] for name in p}
    out.update(sweeps=sweeps.value, vertices=nc.value, entries=nnz.value)
    return out


def _run_refine(s):
    L, h, c, stream = gk.lib(), s["ctx"].handle, ctypes.byref(s["csr"]), ctypes.c_void_p(s["stream"].cuda_stream)
    p = {name: _ptr(s[name]) for name in ("cmap", "cpart", "cbnd", "part", "bnd", "gain", "dest", "updated", "pw")}
    with torch.cuda.stream(s["stream"]):
        s["pw"].copy_(s["pw0"])
    _ok(L.gk_k_project(h, s["csr"].n, p["cmap"], p["cpart"], p["cbnd"], p["part"], p["bnd"], p["gain"], p["dest"],
                       p["updated"], stream))
    _ok(L.gk_k_gain(h, c, s["k"], p["part"], p["updated"], p["bnd"], p["gain"], p["dest"], stream))
    gained, cut = ctypes.c_int64(), ctypes.c_int64()
    _ok(L.gk_k_round(h, c, s["k"], s["cap"], 1024, s["rounds"], p["part"], p["bnd"], p["gain"], p["dest"], p["pw"],
                     s["nmoves"].ctypes.data_as(gk.I32P), s["pos"].ctypes.data_as(gk.I32P), ctypes.byref(gained), None, None,
                     stream))
    _ok(L.gk_k_cut(h, c, s["k"], p["part"], ctypes.byref(cut), None, stream))
    out = {name: s[name] for name in ("part", "bnd", "gain", "dest", "pw")}
    out.update(nmoves=s["nmoves"], pos=s["pos"], gained=gained.value, cut=cut.value)
    return out


def _run_cut(s):
    _ok(gk.lib().gk_k_cut_noalloc(s["ctx"].handle, ctypes.byref(s["csr"]), s["k"], _ptr(s["part"]), s["cut"].data_ptr(),
                                  s["weights"].data_ptr(), s["stream"].cuda_stream))
    return {"cut": s["cut"], "weights": s["weights"]}


_RUNS = {"host": _run_host, "device": _run_device, "packed": _run_packed, "serve": _run_serve, "coarsen": _run_coarsen,
         "refine": _run_refine, "cut": _run_cut}


# ---------------------------------------------------------------- sizes and values
# Entries of a row, on average, by family (both directions of an edge counted).
_DEGREE = {"delaunay": 6.0, "hilbert": 6.0, "grid": 6.0, "road": 2.1, "dag": 3.5}


def work(case):
    """Bytes of one pass: the CSR (row bounds, neighbours, edge and vertex weights) read once, the results written once.
    All arithmetic is integer comparison and addition: one for each entry."""
    what = case["what"]
    if what in ("packed", "serve"):
        sizes = [int(case["lo"] * (case["hi"] / case["lo"]) ** ((i * 0.6180339887) % 1.0)) for i in range(case["count"])]
        n = sum(sizes)
        nnz = sum(x * _DEGREE["delaunay" if i % 2 == 0 else "dag"] for i, x in enumerate(sizes))
    else:
        n = case["n"]
        nnz = n * _DEGREE[case["graph"]]
    csr = 8 * n + 8 * nnz
    if what == "coarsen":
        # Five arrays per vertex, and a coarse graph of about a quarter of the vertices and half of the entries.
        return {"bytes": csr + 20 * n + 8 * (n / 4) + 8 * (nnz / 2), "flops": nnz}
    if what == "refine":
        # The map read, and four arrays of state per vertex written.
        return {"bytes": csr + 20 * n, "flops": nnz}
    return {"bytes": csr + 4 * n, "flops": nnz}


def exact(case, seed):
    """Cut and part weights, and a coarsening level, in plain torch with 64-bit integers.  The other cases' results
    come from a sequence of greedy decisions, for which there is no formula."""
    if case["what"] == "cut":
        s = prepare(case, seed)
        xadj, adj, w, vw = (t.long() for t in s["arrays"])
        part = s["part"].long()
        src = torch.repeat_interleave(torch.arange(len(vw), device="cuda"), xadj[1:] - xadj[:-1])
        cut = (w * (part[src] != part[adj])).sum().reshape(1) // 2
        return {"cut": cut, "weights": torch.zeros(case["k"], dtype=torch.int64, device="cuda").index_add_(0, part, vw)}
    if case["what"] == "coarsen":
        arrays = tuple(t.long() for t in _device_graph(case, seed))
        out = _exact_coarsen(*arrays)
        room = {"cvwgt": case["n"], "cxadj": case["n"] + 1, "cadjncy": _room(case, len(arrays[1]))}
        room["cadjwgt"] = room["cadjncy"]
        # What a level leaves unused of its buffers stays zero.
        out.update({name: torch.nn.functional.pad(out[name], (0, size - len(out[name]))) for name, size in room.items()})
        return out
    return None


def _exact_coarsen(xadj, adj, w, vw):
    n = len(vw)
    v = torch.arange(n, device="cuda")
    deg = xadj[1:] - xadj[:-1]
    src = torch.repeat_interleave(v, deg)
    # The neighbour of the heaviest edge, then of the lowest degree, then of the lowest number; none: itself.
    top = torch.zeros(n, dtype=torch.int64, device="cuda").scatter_reduce_(0, src, w, "amax")
    key = torch.where(w == top[src], deg[adj] * n + adj, torch.iinfo(torch.int64).max)
    best = torch.full((n,), torch.iinfo(torch.int64).max, device="cuda").scatter_reduce_(0, src, key, "amin")
    cand = torch.where(deg > 0, best % n, v)
    # Hops to the pair of vertices that chose each other, and the largest number in the component.
    root = cand[cand] == v
    to = torch.where(root, v, cand)
    stamp = (~root).long()
    sweeps = 0
    while not torch.equal(to[to], to):
        stamp = stamp + stamp[to]
        to = to[to]
        sweeps += 1
    pair = torch.maximum(to, cand[to])
    label = torch.zeros(n, dtype=torch.int64, device="cuda").scatter_reduce_(0, pair, v, "amax")[pair]
    # Groups in order of (label, stamp, number), cut into coarse vertices of at most six.
    order = torch.argsort(label * (int(stamp.max()) + 1) + stamp, stable=True)
    first = torch.full((n,), n, dtype=torch.int64, device="cuda").scatter_reduce_(0, label[order], v, "amin")
    chunk = torch.cumsum(((v - first[label[order]]) % 6 == 0).long(), 0) - 1
    cmap = torch.empty_like(chunk)
    cmap[order] = chunk
    nc = int(chunk[-1]) + 1
    cvwgt = torch.zeros(nc, dtype=torch.int64, device="cuda").index_add_(0, cmap, vw)
    a, b = cmap[src], cmap[adj]
    pairs, which = torch.unique((a * nc + b)[a != b], return_inverse=True)
    cw = torch.zeros(len(pairs), dtype=torch.int64, device="cuda").index_add_(0, which, w[a != b])
    cxadj = torch.zeros(nc + 1, dtype=torch.int64, device="cuda")
    cxadj[1:] = torch.cumsum(torch.bincount(pairs // nc, minlength=nc), 0)
    return {"cand": cand, "label": label, "stamp": stamp, "order": order, "cmap": cmap, "cvwgt": cvwgt, "cxadj": cxadj,
            "cadjncy": pairs % nc, "cadjwgt": cw, "sweeps": sweeps, "vertices": nc, "entries": len(pairs)}
