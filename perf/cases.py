"""What this repository's kernels are timed on: SpMV, SpMM, SDDMM and the solver step
around SpMV (fused_spmv_axpy, axpy), fp64 CSR with int64 indices, each through the entry
point a program calls (``Variant.launch_async``, ``launch_spmv_noalloc``) on arrays that
already live in device memory.

The matrices are the four families of ``tilegen_amd.matrices`` (uniform random, banded,
power law, dense rows) and its 4x4 blocks, drawn on the GPU from the seed; values and dense
operands are U(-1, 1).  A case's schedule is the one this repository ships for that kernel
and family (``tilegen_amd.schedules``).

A case is {"name", "op", "pattern", "rows", "K"}:
  op       spmv | noalloc | step | spmm | sddmm
  pattern  uniform (16 per row) | banded (7 diagonals) | power_law (P(len) ~ len^-2.03, up to
           5000) | dense_rows (1% of 2000, the rest 4) | blocks4 / blocks25 (that many dense
           4x4 blocks per block row)
  rows     rows = columns
  K        dense columns (spmm, sddmm), 0 otherwise
"""

import ctypes
import math

import torch

from tilegen_amd import runtime
from tilegen_amd.codegen import Config
from tilegen_amd.schedules import TUNED
from tilegen_amd.variant import Variant, operand_order

# one of the wide schedules that every kernel is tested on (schedules.TEST_SCHEDULES); on
# skewed rows the tuner picks tiles of 128 rows on 512 lanes for SpMM
WIDE = Config(tile_size=128, threads_per_row=8, unroll=2, vector_width=2, block_size=512)
SPMV_SCHEDULE = {"uniform": "c1", "banded": "c2", "power_law": "c3a", "dense_rows": "c3b"}

ALPHA, BETA = -1.0, 1.0     # residual b - A x
OMEGA = 0.7                 # relaxation of the step x + omega r


def listed():
    return [
        # a matrix of a test or a coarse grid level: one launch of a few workgroups
        {"name": "spmv_small", "op": "spmv", "pattern": "uniform", "rows": 2000, "K": 0},
        # the benchmark's headline matrix
        {"name": "spmv_uniform", "op": "spmv", "pattern": "uniform", "rows": 100000, "K": 0},
        # a stencil operator of a large grid, odd row count: bound by its streams
        {"name": "spmv_banded_large", "op": "spmv", "pattern": "banded", "rows": 3200001, "K": 0},
        # a graph's adjacency matrix, ten times the benchmark's
        {"name": "spmv_power_law_large", "op": "spmv", "pattern": "power_law", "rows": 1000003,
         "K": 0},
        # a few dense rows among short ones (constraints, hubs)
        {"name": "spmv_dense_rows", "op": "spmv", "pattern": "dense_rows", "rows": 20000, "K": 0},
        # the entry point for callers that may not allocate, on the benchmark's graph
        {"name": "noalloc_power_law", "op": "noalloc", "pattern": "power_law", "rows": 100000,
         "K": 0},
        # one relaxation step of an iterative solver: r = b - A x, then x + omega r
        {"name": "step_banded", "op": "step", "pattern": "banded", "rows": 200000, "K": 0},
        # the benchmark's SpMM: a feature matrix of 64 columns
        {"name": "spmm_uniform_k64", "op": "spmm", "pattern": "uniform", "rows": 100000, "K": 64},
        # graph features of an odd width on skewed rows
        {"name": "spmm_power_law_k63", "op": "spmm", "pattern": "power_law", "rows": 100000,
         "K": 63},
        # a stencil on many right-hand sides, wider than one pass of the lanes
        {"name": "spmm_banded_k130", "op": "spmm", "pattern": "banded", "rows": 200000, "K": 130},
        # the benchmark's larger SDDMM: block-sparse scores, 10 M nonzeros
        {"name": "sddmm_blocks25_k64", "op": "sddmm", "pattern": "blocks25", "rows": 100000,
         "K": 64},
        # edge scores of a graph with wide features
        {"name": "sddmm_power_law_k130", "op": "sddmm", "pattern": "power_law", "rows": 100000,
         "K": 130},
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["spmv", "spmv", "spmm", "spmm", "sddmm", "sddmm", "step", "noalloc"])
    if op in ("spmv", "step", "noalloc"):
        pattern = rng.choice(["uniform", "banded", "power_law", "dense_rows"])
        top = {"uniform": 400000, "banded": 3200000, "power_law": 1000000, "dense_rows": 100000}
        if op == "noalloc":
            top.update(power_law=400000, dense_rows=50000)
        rows = _between(rng, 2000, top[pattern])
        return {"op": op, "pattern": pattern, "rows": rows, "K": 0}
    pattern = rng.choice(["uniform", "banded", "power_law", "dense_rows"] if op == "spmm" else
                         ["blocks4", "blocks25", "uniform", "power_law"])
    K = _between(rng, 4, 256)
    per_row = {"uniform": 16, "banded": 7, "power_law": 8, "dense_rows": 24, "blocks4": 16,
               "blocks25": 100}[pattern]
    most = 1e8 / (per_row * K)               # nonzeros x K of the benchmark's SpMM
    rows = _between(rng, 2000, max(2500, min(200000, most)))
    return {"op": op, "pattern": pattern, "rows": rows, "K": K}


# --------------------------------------------------------------------------- #
# inputs
# --------------------------------------------------------------------------- #
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _power_law_lengths(n):
    """min(5000, floor(u^(-1/1.03))) at n evenly spaced u, no row over half the columns."""
    u = (torch.arange(n, dtype=torch.float64) + 0.5) / n
    return u.pow(-1.0 / 1.03).floor().clamp(1, min(5000, n // 2)).long()


def _dense_lengths(n):
    counts = torch.full((n,), 4)
    counts[:max(1, n // 100)] = min(2000, n // 2)
    return counts


def _block_lengths(n, per):
    """``per`` blocks of 4 columns; rows past the last whole block row are empty."""
    counts = torch.full((n,), per * 4)
    counts[n // 4 * 4:] = 0
    return counts


def _distinct(g, counts, ncols):
    """Ascending distinct uniform columns, counts[i] of them for row i: drawn with repeats,
    repeats dropped, and the rows that came out short drawn again for what they lack."""
    dev = counts.device
    key = torch.empty(0, dtype=torch.int64, device=dev)
    lack = counts
    while int(lack.sum()):
        rows = torch.repeat_interleave(torch.arange(counts.numel(), device=dev), lack)
        cols = torch.randint(ncols, (rows.numel(),), generator=g, device=dev)
        key = torch.unique(torch.cat([key, rows * ncols + cols]))
        lack = counts - torch.bincount(key // ncols, minlength=counts.numel())
    return key % ncols


def _structure(pattern, n, g, dev):
    """(indptr, indices) of an n x n matrix, columns ascending within each row.  The same
    case has the same row lengths, in another order for another seed."""
    if pattern == "banded":
        cols = torch.arange(n, device=dev)[:, None] + torch.arange(-3, 4, device=dev)
        keep = (cols >= 0) & (cols < n)
        counts, cols = keep.sum(1), cols[keep]
    elif pattern.startswith("blocks"):
        per, nb = int(pattern[6:]), n // 4
        b = _distinct(g, torch.full((nb,), per, device=dev), nb)
        cols = (b.reshape(nb, per, 1) * 4 + torch.arange(4, device=dev)).reshape(nb, 1, per * 4)
        cols = cols.expand(nb, 4, per * 4).reshape(-1)
        counts = _block_lengths(n, per).to(dev)
    elif pattern == "uniform":
        counts = torch.full((n,), 16, device=dev)
        cols = _distinct(g, counts, n)
    else:
        lengths = _power_law_lengths(n) if pattern == "power_law" else _dense_lengths(n)
        counts = lengths.to(dev)[torch.randperm(n, generator=g, device=dev)]
        cols = _distinct(g, counts, n)
    indptr = torch.zeros(n + 1, dtype=torch.int64, device=dev)
    indptr[1:] = counts.cumsum(0)
    return indptr, cols.contiguous()


def _inputs(case, seed):
    dev, n, K = _device(), case["rows"], case["K"]
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    indptr, indices = _structure(case["pattern"], n, g, dev)

    def u(*shape):
        return torch.rand(*shape, generator=g, device=dev, dtype=torch.float64) * 2 - 1

    a = {"indptr": indptr, "indices": indices, "data": u(indices.numel())}
    if case["op"] == "spmm":
        a["B"] = u(n, K)
    elif case["op"] == "sddmm":
        a["U"], a["V"] = u(n, K), u(n, K)
    else:
        a["x"] = u(n)
        if case["op"] == "step":
            a["w"] = u(n)
    return a


# --------------------------------------------------------------------------- #
# the calls
# --------------------------------------------------------------------------- #
class _Call:
    """A variant bound to device arrays: what a program keeps between calls."""

    def __init__(self, kernel, config, arrays, out, scalars, M, N, K, nnz):
        self.variant = Variant(kernel, config)
        names = dict(arrays)
        names["y" if kernel == "spmv" else "C" if kernel in ("spmm", "sddmm") else "z"] = out
        values = self.variant.abi_values(None, names, scalars, M, N, K, nnz)
        self.values = [ctypes.cast(v.data_ptr(), t) if isinstance(v, torch.Tensor) else v
                       for v, t in zip(values, self.variant.launch.argtypes)]
        self.keep = (arrays, out)

    def __call__(self):
        self.variant.launch_async(self.values, None)


def _schedule(op, pattern):
    if op == "spmm":
        return WIDE if pattern in ("power_law", "dense_rows") else TUNED["c4"]
    if op == "sddmm":
        return TUNED["c5x25"] if pattern == "blocks25" else TUNED["c5"]
    return TUNED[SPMV_SCHEDULE[pattern]]


def prepare(case, seed):
    op, n, K = case["op"], case["rows"], case["K"]
    a = _inputs(case, seed)
    nnz = a["indices"].numel()
    dev = a["data"].device
    state = {"op": op, "arrays": a}
    if op == "spmm":
        out = torch.zeros(n, K, dtype=torch.float64, device=dev)
    elif op == "sddmm":
        out = torch.zeros(nnz, dtype=torch.float64, device=dev)
    else:
        out = torch.zeros(n, dtype=torch.float64, device=dev)
    if op == "noalloc":
        state["fn"] = runtime.noalloc_lib().launch_spmv_noalloc
        state["args"] = [a[k].data_ptr() for k in ("indptr", "indices", "data", "x")] + \
            [out.data_ptr(), n, n, nnz, None]
        state["out"] = out
        return state
    config = _schedule(op, case["pattern"])
    if op == "step":
        new = torch.zeros_like(out)
        state["calls"] = [
            _Call("fused_spmv_axpy", config, a, out, {"alpha": ALPHA, "beta": BETA}, n, n, 0, nnz),
            _Call("axpy", WIDE, {"x": a["x"], "w": out}, new, {"alpha": 1.0, "beta": OMEGA},
                  n, n, 0, nnz)]
        state["out"] = {"residual": out, "x": new}
        return state
    dense = operand_order(op)[0]
    arrays = {k: a[k] for k in ["indptr", "indices", "data"] + dense}
    state["calls"] = [_Call(op, config, arrays, out, {}, n, n, K, nnz)]
    state["out"] = out
    return state


def run(state):
    if state["op"] == "noalloc":
        runtime.check(state["fn"](*state["args"]), "launch_spmv_noalloc")
    else:
        for call in state["calls"]:
            call()
    return state["out"]


# --------------------------------------------------------------------------- #
# what a pass needs, and what it should give
# --------------------------------------------------------------------------- #
def _nnz(case):
    n, pattern = case["rows"], case["pattern"]
    if pattern == "banded":
        return 7 * n - 12
    if pattern == "uniform":
        return 16 * n
    if pattern == "power_law":
        return int(_power_law_lengths(n).sum())
    if pattern == "dense_rows":
        return int(_dense_lengths(n).sum())
    return int(_block_lengths(n, int(pattern[6:])).sum())


def work(case):
    op, n, K, nnz = case["op"], case["rows"], case["K"], _nnz(case)
    structure = 8 * (n + 1) + 16 * nnz
    if op == "spmm":
        return {"bytes": structure + 16 * n * K, "flops": 2 * nnz * K}
    if op == "sddmm":
        return {"bytes": structure + 16 * n * K + 8 * nnz, "flops": 2 * nnz * K}
    if op == "step":                 # A, x, b read; r written; x + omega r written
        return {"bytes": structure + 32 * n, "flops": 2 * nnz + 5 * n}
    return {"bytes": structure + 16 * n, "flops": 2 * nnz}


def tolerance(case):
    """fp64 sums in another order: about four times what ``run`` and ``exact`` differ by
    (2e-16 with short rows, 1.0e-15 to 1.5e-15 where rows of thousands are summed)."""
    skewed = case["pattern"] in ("power_law", "dense_rows") and case["op"] != "sddmm"
    return {"rel": 6e-15 if skewed else 1e-15}


def exact(case, seed):
    a = _inputs(case, seed)
    n, op = case["rows"], case["op"]
    rows = torch.repeat_interleave(torch.arange(n, device=a["data"].device),
                                   a["indptr"][1:] - a["indptr"][:-1])
    cols, data = a["indices"], a["data"]
    step = max(1, (1 << 27) // max(1, case["K"]))     # 1 GiB of products at a time
    if op == "sddmm":
        return torch.cat([(a["U"][rows[s:s + step]] * a["V"][cols[s:s + step]]).sum(1)
                          * data[s:s + step] for s in range(0, data.numel(), step)])
    if op == "spmm":
        C = torch.zeros(n, case["K"], dtype=torch.float64, device=data.device)
        for s in range(0, data.numel(), step):
            C.index_add_(0, rows[s:s + step], a["B"][cols[s:s + step]] * data[s:s + step, None])
        return C
    y = torch.zeros(n, dtype=torch.float64, device=data.device)
    y.index_add_(0, rows, data * a["x"][cols])
    if op == "step":
        r = ALPHA * y + BETA * a["w"]
        return {"residual": r, "x": a["x"] + OMEGA * r}
    return y
