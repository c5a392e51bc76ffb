"""SDDMM's sample of neighbouring rows: dense blocks pass for blocks, hubs and short rows do not
(on the CPU, with the kernel's own test); matrices of both kinds match the oracle past 64 columns
(on the GPU), with fewer rows than pairs are sampled and with empty rows."""

from __future__ import annotations

import numpy as np
import pytest

from tests.test_gpu_parity import _check
from tests.util import csr
from tilegen_amd.codegen import generate
from tilegen_amd.dsl import standard_kernels
from tilegen_amd.matrices import make_baseline
from tilegen_amd.schedules import TUNED

CFG = TUNED["c5"]


def _rows(cols, n):
    ip = np.r_[0, np.cumsum([len(c) for c in cols])].astype(np.int64)
    ind = np.concatenate([np.asarray(c, dtype=np.int64) for c in cols]) if ip[-1] else []
    return csr(len(cols), n, ip, ind, np.random.default_rng(2).uniform(-1, 1, int(ip[-1])))


def _matrix(kind, M, n=700):
    rng = np.random.default_rng(8)
    if kind == "hub in every row":       # half of the rows are the hub alone
        return _rows([np.r_[0, np.sort(rng.choice(n - 1, rng.integers(0, 9) // 2, False)) + 1]
                      for _ in range(M)], n)
    if kind == "hubs at both ends":
        return _rows([np.r_[0, np.sort(rng.choice(n - 2, 3 + r % 3, False)) + 1, n - 1]
                      for r in range(M)], n)
    if kind == "arrow":
        return _rows([np.r_[0, min(r + 1, n - 1)] for r in range(M)], n)
    if kind == "empty":
        return _rows([[] for _ in range(M)], n)
    per = {"blocks of 4": 4, "blocks of 2": 2}[kind]
    cols = [np.sort(rng.choice(n // per, 3, False)) for _ in range(-(-M // per))]
    return _rows([(cols[r // per][:, None] * per + np.arange(per)).ravel() for r in range(M)], n)


def _passes(A):
    """tg_blocked on the CPU."""
    src = generate(standard_kernels()["sddmm"], CFG, "hip", write=False).source
    for text in ("tg_i64 r = R * i / 8 + (i & 3);", "const bool in = i < 8 && r + 2 <= R;",
                 "bool same = in && p1 - p0 > 1 && p2 - p1 > 1;",
                 "indices[p0 + (p1 - p0) / 2] == indices[p1 + (p2 - p1) / 2];",
                 "(__ballot(same))) >= 3;"):
        assert text in src
    R, n = A.shape[0], 0
    for i in range(8):
        r = R * i // 8 + (i & 3)
        if r + 2 <= R:
            a, b = (A.indices[A.indptr[q]:A.indptr[q + 1]] for q in (r, r + 1))
            n += len(a) > 1 and len(b) > 1 and a[0] == b[0] and a[len(a) // 2] == b[len(b) // 2]
    return n >= 3


@pytest.mark.parametrize("kind,want", [("hub in every row", False), ("hubs at both ends", False),
                                       ("arrow", False), ("empty", False), ("blocks of 4", True),
                                       ("blocks of 2", True)])
def test_what_passes_for_blocks(kind, want):
    assert _passes(_matrix(kind, 640)) == want


def test_the_benchmarks_blocks_pass():
    assert _passes(make_baseline("c5", scale=0.02))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["hub in every row", "hubs at both ends", "arrow", "empty",
                                  "blocks of 4", "blocks of 2"])
def test_parity(kind, hip_ready):
    for M in (1, 2, 3, 9, 640):
        A = _matrix(kind, M)
        for K in (65, 96, 129, 193, 257):
            print("[gpu] sddmm %s rows=%d K=%d" % (kind, M, K), flush=True)
            _check("sddmm", CFG, A, K=K, label="%s rows=%d K=%d" % (kind, M, K))
