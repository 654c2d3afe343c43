"""The task programs of this framework as a user's program runs them, for timing.

Every case goes through the public entry points (gtap_amd, include/gtap.h) on device memory
that the caller owns, on the default configuration:

  fib, nqueens    fork-join recursion, one task per call or placement, a short sweep of sizes
  nqueens_cutoff  n-queens at the reference's benchmark settings (tasks to row 7)
  sort            cilksort of uint32 keys (block mode)
  bfs             asynchronous BFS with one queue or four EPAQ queues
  spmv            CSR float64 matrix-vector product, a task per row
  tree            the binary-tree workload, float64
  stream          a mixed job stream in one resident launch
  lowered_sort    a user's own `#pragma gtap` program, built by the lowering tool (a four-way
                  merge sort in thread mode, gtap_amd/lower/examples/csort.gtap.cu), its
                  variables set and its entry kernel launched by the host

Device buffers are torch tensors; their addresses go to the C ABI.
"""
import ctypes
import math

import numpy as np
import torch

import gtap_amd as G

DEV = "cuda"
INF = G.INF_DEPTH

# nodes of the n-queens search tree (the root included): one task each
NQ_TASKS = {1: 2, 2: 3, 3: 6, 4: 17, 5: 54, 6: 153, 7: 552, 8: 2057, 9: 8394, 10: 35539, 11: 166926, 12: 856189,
            13: 4674890, 14: 27358553, 15: 171129072}


def listed():
    return [
        # The smallest calls: a recursion of some ten thousand tasks, where launch latency and
        # the depth of the spawn tree count (the sizes below the reference's scaling plots).
        {"name": "fib 18", "kind": "fib", "n": 18, "count": 3},
        # The reference's fib evaluation at its ordinary size (millions of empty tasks: pure
        # scheduling cost).
        {"name": "fib 30", "kind": "fib", "n": 30, "count": 3},
        # The headline workload: n-queens with one task per placement, irregular fan-out.
        {"name": "n-queens 14", "kind": "nqueens", "n": 14, "count": 3},
        # The reference's n-queens benchmark: tasks for the first rows, sequential search below.
        {"name": "n-queens cutoff 15", "kind": "nqueens_cutoff", "n": 15, "count": 3, "cutoff": 7},
        # The cilksort benchmark's size.
        {"name": "cilksort 64M", "kind": "sort", "n": 1 << 26, "few": False},
        # A small ragged sort inside a larger program: a few leaves and merges.
        {"name": "cilksort 20011", "kind": "sort", "n": 20011, "few": False},
        # The BFS benchmark graph's size and shape, with EPAQ by out-degree.
        {"name": "bfs rmat 22 epaq", "kind": "bfs", "graph": "rmat", "scale": 22, "edge_factor": 16, "queues": 4, "split": 64},
        # A medium graph with one queue.
        {"name": "bfs rmat 18", "kind": "bfs", "graph": "rmat", "scale": 18, "edge_factor": 16, "queues": 1, "split": 64},
        # The SpMV example's default size: a million rows of about 300 entries.
        {"name": "spmv 1M x 300", "kind": "spmv", "rows": 1 << 20, "avg": 300, "cutoff": 16},
        # The binary-tree example's default size: memory and arithmetic work in every node.
        {"name": "tree 15", "kind": "tree", "height": 15, "mem_ops": 64, "iters": 512, "input_n": 1 << 20},
        # A batch of mixed jobs (fib, n-queens, sorts) replayed as one launch.
        {"name": "stream 1024 jobs", "kind": "stream", "jobs": 1024},
        # A user's own program from `#pragma gtap` source.
        {"name": "lowered csort 500009", "kind": "lowered_sort", "n": 500009},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fib", "nqueens", "nqueens_cutoff", "sort", "sort", "bfs", "bfs", "spmv", "spmv", "tree", "stream",
                       "lowered_sort"])
    if kind == "fib":
        return {"kind": kind, "n": rng.randint(8, 30), "count": rng.randint(2, 4)}
    if kind == "nqueens":
        return {"kind": kind, "n": rng.randint(8, 14), "count": rng.randint(2, 4)}
    if kind == "nqueens_cutoff":
        return {"kind": kind, "n": rng.randint(10, 15), "count": rng.randint(2, 3), "cutoff": rng.randint(5, 8)}
    if kind == "sort":
        return {"kind": kind, "n": _log(rng, 1000, 1 << 26), "few": rng.random() < 0.25}
    if kind == "bfs":
        queues, split = rng.choice([1, 4]), rng.choice([32, 64])
        if rng.random() < 0.7:
            return {"kind": kind, "graph": "rmat", "scale": rng.randint(10, 22), "edge_factor": rng.randint(6, 16),
                    "queues": queues, "split": split}
        return {"kind": kind, "graph": "uniform", "nv": _log(rng, 1000, 4 << 20), "edge_factor": rng.randint(4, 16),
                "queues": queues, "split": split}
    if kind == "spmv":
        rows = _log(rng, 500, 1 << 20)
        return {"kind": kind, "rows": rows, "avg": _log(rng, 3, 300), "cutoff": rng.choice([8, 16, 16, 32])}
    if kind == "tree":
        return {"kind": kind, "height": rng.randint(8, 15), "mem_ops": rng.randint(0, 64), "iters": rng.randint(16, 512),
                "input_n": 1 << rng.randint(12, 20)}
    if kind == "stream":
        return {"kind": kind, "jobs": _log(rng, 16, 1024)}
    return {"kind": kind, "n": _log(rng, 1000, 500009)}


# ---------------------------------------------------------------- inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _keys(case, seed):
    """uint32 keys (as int32 bit patterns): uniform, or few distinct values."""
    g, n = _gen(seed), case["n"]
    if case.get("few"):
        return torch.randint(0, 100, (n,), device=DEV, dtype=torch.int32, generator=g)
    return torch.randint(-(1 << 31), 1 << 31, (n,), device=DEV, dtype=torch.int64, generator=g).to(torch.int32)


def _graph(case, seed):
    """(row offsets, columns) of an R-MAT (a, b, c = .57, .19, .19) or a uniform random graph."""
    g = _gen(seed)
    nv = 1 << case["scale"] if case["graph"] == "rmat" else case["nv"]
    ne = nv * case["edge_factor"]
    if case["graph"] == "rmat":
        src = torch.zeros(ne, device=DEV, dtype=torch.int32)
        dst = torch.zeros(ne, device=DEV, dtype=torch.int32)
        for _ in range(case["scale"]):
            r = torch.rand(ne, device=DEV, generator=g)
            src.mul_(2).add_((r >= 0.76).to(torch.int32))
            dst.mul_(2).add_((((r >= 0.57) & (r < 0.76)) | (r >= 0.95)).to(torch.int32))
    else:
        src = torch.randint(0, nv, (ne,), device=DEV, dtype=torch.int32, generator=g)
        dst = torch.randint(0, nv, (ne,), device=DEV, dtype=torch.int32, generator=g)
    src, order = torch.sort(src, stable=True)
    col = dst[order].contiguous()
    row = torch.searchsorted(src, torch.arange(nv + 1, device=DEV, dtype=torch.int32)).to(torch.int32)
    return row.contiguous(), col


def _matrix(case, seed):
    """A square CSR matrix: 1 .. 2 avg - 1 entries a row, ascending columns spread over the
    row, values in [-1, 1); and a vector."""
    g, rows, avg = _gen(seed), case["rows"], case["avg"]
    counts = torch.randint(1, 2 * avg, (rows,), device=DEV, generator=g).clamp_(max=rows)
    row_ptr = torch.zeros(rows + 1, device=DEV, dtype=torch.int64)
    torch.cumsum(counts, 0, out=row_ptr[1:])
    nnz = int(row_ptr[-1])
    k = torch.arange(nnz, device=DEV) - torch.repeat_interleave(row_ptr[:-1], counts)
    length = torch.repeat_interleave(counts, counts).to(torch.float32)
    at = (k + torch.rand(nnz, device=DEV, generator=g)) / length
    del k, length
    col = (at * rows).to(torch.int32).clamp_(max=rows - 1)
    del at
    val = torch.rand(nnz, device=DEV, dtype=torch.float64, generator=g).mul_(2).sub_(1)
    x = torch.rand(rows, device=DEV, dtype=torch.float64, generator=g).mul_(4).sub_(2)
    return row_ptr.to(torch.int32), col, val, x


def _sweep(case, seed):
    """The sizes n - count + 1 .. n, in an order that starts at another one for each seed."""
    ns = list(range(case["n"] - case["count"] + 1, case["n"] + 1))
    at = seed % len(ns)
    return ns[at:] + ns[:at]


_ready = False
_modules = {}


def _runtime():
    global _ready
    if not _ready:
        if G.gtap_initialize() != 0:
            raise RuntimeError("gtap_initialize failed")
        _ready = True


def _module(name):
    if name not in _modules:
        from gtap_amd import build
        _modules[name] = G.EntryModule(build.lowered_lib(name), name)
    return _modules[name]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "lowered_sort":
        _module("csort")
    _runtime()
    s = {"case": case, "stats": G.RunStats()}
    if kind in ("fib", "nqueens", "nqueens_cutoff"):
        s["sizes"] = _sweep(case, seed)
    elif kind in ("sort", "lowered_sort"):
        s["keys"] = _keys(case, seed)
        s["work"] = torch.empty_like(s["keys"])
        s["tmp"] = torch.empty_like(s["keys"])
    elif kind == "bfs":
        s["row"], s["col"] = _graph(case, seed)
        s["depth"] = torch.empty(s["row"].numel() - 1, device=DEV, dtype=torch.int32)
    elif kind == "spmv":
        s["row"], s["col"], s["val"], s["x"] = _matrix(case, seed)
        s["y"] = torch.empty(case["rows"], device=DEV, dtype=torch.float64)
    elif kind == "tree":
        s["input"] = torch.rand(case["input_n"], device=DEV, dtype=torch.float64, generator=_gen(seed)).mul_(2).sub_(1)
        # values above 1 too, so that the sums that seed the arithmetic are not all negative or small
        s["input"] *= 1000.0
        s["out"] = torch.empty((2 << case["height"]) - 1, device=DEV, dtype=torch.float64)
    elif kind == "stream":
        s["stream"] = _Stream(seed, case["jobs"])
    torch.cuda.synchronize()
    return s


class _Stream(G.Stream):
    """A job stream that is given back with its state."""

    def __del__(self):
        self.close()


def _check(status, what):
    if status != 0:
        raise RuntimeError(f"{what}: status {status}")


def run(state):
    case, L, st = state["case"], G.lib(), ctypes.byref(state["stats"])
    kind = case["kind"]
    if kind == "fib":
        return [G.fib(n)[0] for n in state["sizes"]]
    if kind == "nqueens":
        return [G.nqueens(n)[0] for n in state["sizes"]]
    if kind == "nqueens_cutoff":
        return [G.nqueens_cutoff(n, case["cutoff"])[0] for n in state["sizes"]]
    if kind == "sort":
        k, w, t = state["keys"], state["work"], state["tmp"]
        _check(L.gtap_memcpy_dtod(w.data_ptr(), k.data_ptr(), 4 * case["n"]), "copy")
        _check(L.gtap_cilksort(w.data_ptr(), t.data_ptr(), case["n"], 0, 0, st), "cilksort")
        return w
    if kind == "lowered_sort":
        k, w, t = state["keys"], state["work"], state["tmp"]
        m = _module("csort")
        _check(L.gtap_memcpy_dtod(w.data_ptr(), k.data_ptr(), 4 * case["n"]), "copy")
        m.set_symbol("g_keys", w.data_ptr(), ctypes.c_uint64)
        m.set_symbol("g_tmp", t.data_ptr(), ctypes.c_uint64)
        _check(m.launch("csort_kernel", [ctypes.c_int], case["n"]), "csort")
        return w
    if kind == "bfs":
        row, col, depth = state["row"], state["col"], state["depth"]
        _check(L.gtap_bfs(row.data_ptr(), col.data_ptr(), row.numel() - 1, col.numel(), 0, depth.data_ptr(),
                          case["queues"], case["split"], st), "bfs")
        return depth
    if kind == "spmv":
        _check(L.gtap_spmv(state["row"].data_ptr(), state["col"].data_ptr(), state["val"].data_ptr(),
                           state["x"].data_ptr(), state["y"].data_ptr(), case["rows"], case["rows"], case["cutoff"], st),
               "spmv")
        return state["y"]
    if kind == "tree":
        _check(L.gtap_tree(case["height"], case["mem_ops"], case["iters"], state["input"].data_ptr(), case["input_n"],
                           state["out"].data_ptr(), st), "tree")
        return state["out"]
    return state["stream"].run_batched()[0]


# ---------------------------------------------------------------- work and correctness


def _fib(n):
    a, b = 0, 1
    for _ in range(n):
        a, b = b, a + b
    return a


def work(case):
    kind = case["kind"]
    if kind == "fib":
        # per task: its frame written and read, its result, its id, its join
        return {"bytes": sum(48 * (2 * _fib(n + 1) - 1) for n in _sweep(case, 0)), "flops": 0}
    if kind == "nqueens":
        return {"bytes": sum(72 * NQ_TASKS[n] for n in _sweep(case, 0)), "flops": 0}
    if kind == "nqueens_cutoff":
        # about ten bit operations per placement; the search below the cutoff needs no memory
        return {"bytes": 0, "flops": sum(10 * NQ_TASKS[n] for n in _sweep(case, 0))}
    if kind in ("sort", "lowered_sort"):
        return {"bytes": 8 * case["n"], "flops": 0}
    if kind == "bfs":
        nv = 1 << case["scale"] if case["graph"] == "rmat" else case["nv"]
        return {"bytes": 8 * nv + 4 * nv * case["edge_factor"], "flops": 0}
    if kind == "spmv":
        rows, nnz = case["rows"], case["rows"] * min(case["avg"], case["rows"])
        return {"bytes": 12 * nnz + 20 * rows, "flops": 2 * nnz}
    if kind == "tree":
        nodes = (2 << case["height"]) - 1
        return {"bytes": 8 * nodes + 8 * min(case["input_n"], nodes * case["mem_ops"]),
                "flops": nodes * (case["mem_ops"] + 2 * case["iters"])}
    # 40 % fib in [18, 28], 30 % n-queens in [8, 12], 30 % sorts of 2^10 .. 2^20 keys
    fib = 48 * sum(2 * _fib(n + 1) - 1 for n in range(18, 29)) / 11
    nq = 72 * sum(NQ_TASKS[n] for n in range(8, 13)) / 5
    keys = ((1 << 20) - (1 << 10)) / math.log(1 << 10)
    return {"bytes": int(case["jobs"] * (0.4 * fib + 0.3 * nq + 0.3 * 8 * keys)), "flops": 0}


def tolerance(case):
    """Whole numbers throughout, except spmv and tree. Those two promise the bits: a row of
    spmv is one fused multiply-add chain in column order, a node of tree sums its reads in order."""
    return "exact"


def _xs32(x):
    m = 0xFFFFFFFF
    x = x ^ (x << 13) & m
    x = x ^ (x >> 17)
    return x ^ (x << 5) & m


def _nqueens(n):
    """Placements of n queens, row by row over all partial boards."""
    mask = (1 << n) - 1
    cols = diag = anti = torch.zeros(1, device=DEV, dtype=torch.int64)
    for _ in range(n):
        free = mask & ~(cols | diag | anti)
        parts = []
        for c in range(n):
            at = torch.nonzero(free & (1 << c)).reshape(-1)
            parts.append((cols[at] | 1 << c, (diag[at] | 1 << c) << 1 & mask, (anti[at] | 1 << c) >> 1))
        cols, diag, anti = (torch.cat([p[i] for p in parts]) for i in range(3))
    return cols.numel()


def _exact_bfs(row, col):
    nv = row.numel() - 1
    depth = torch.full((nv,), INF, device=DEV, dtype=torch.int32)
    depth[0] = 0
    src = torch.repeat_interleave(torch.arange(nv, device=DEV, dtype=torch.int32), (row[1:] - row[:-1]).to(torch.int64))
    level = 0
    while True:
        hit = col[depth[src] == level]
        hit = hit[depth[hit] == INF]
        if hit.numel() == 0:
            return depth
        level += 1
        depth[hit] = level


def _exact_tree(case, inp):
    m32 = 0xFFFFFFFF
    node = torch.arange((2 << case["height"]) - 1, device=DEV, dtype=torch.int64)
    seed = _xs32(node ^ 0x9E3779B9)
    acc = torch.zeros(node.numel(), device=DEV, dtype=torch.float64)
    for m in range(case["mem_ops"]):
        acc += inp[_xs32((seed + m * 747796405) & m32) & (case["input_n"] - 1)]
    mix = ((0x9E3779B9 ^ node) + acc.clamp(0.0, 4294967295.0).to(torch.int64)) & m32
    for it in range(case["iters"]):
        # fma(x, 1 + 2^-23, 1 - 2^-24) in whole multiples of 2^-24, rounded once
        x = _xs32((seed + it * 747796405) & m32)
        y = ((x << 24) + 2 * x + (1 << 24) - 1).to(torch.float64)
        mix ^= y.view(torch.int64) & m32
    return mix.to(torch.float64)


def exact(case, seed):
    kind = case["kind"]
    if kind == "fib":
        return [_fib(n) for n in _sweep(case, seed)]
    if kind in ("nqueens", "nqueens_cutoff"):
        return [_nqueens(n) for n in _sweep(case, seed)]
    if kind in ("sort", "lowered_sort"):
        u = torch.sort(_keys(case, seed).to(torch.int64) & 0xFFFFFFFF)[0]
        return u.to(torch.int32)
    if kind == "bfs":
        return _exact_bfs(*_graph(case, seed))
    if kind == "spmv":
        row, col, val, x = _matrix(case, seed)
        prod = torch.zeros(val.numel() + 1, device=DEV, dtype=torch.float64)
        prod[:-1] = val * x[col]
        rows = torch.repeat_interleave(torch.arange(case["rows"], device=DEV), (row[1:] - row[:-1]).to(torch.int64))
        return torch.zeros(case["rows"], device=DEV, dtype=torch.float64).index_add_(0, rows, prod[:-1])
    if kind == "tree":
        inp = torch.rand(case["input_n"], device=DEV, dtype=torch.float64, generator=_gen(seed)).mul_(2).sub_(1)
        return _exact_tree(case, inp * 1000.0)
    return None  # the job stream's keys come from the framework's own generator
