"""SpMM's tiles in contiguous eighths per XCD: only where the eighths hold like shares of the
nonzeros (on the CPU, with the kernel's own test), each tile once either way (on the GPU, at tile
counts that are and are not multiples of 8, with empty eighths and rows ordered by length)."""

from __future__ import annotations

import re

import numpy as np
import pytest

from tests.test_gpu_parity import _check
from tests.util import csr
from tilegen_amd.codegen import generate
from tilegen_amd.dsl import standard_kernels
from tilegen_amd.schedules import TUNED

CFG = TUNED["c4"]
T = CFG.tile_size


def _lengths(kind, M):
    if kind == "alike":
        return np.full(M, 5)
    if kind == "first eighth":
        return np.where(np.arange(M) < M // 8, 36, 4)
    if kind == "by length":
        return np.sort(np.random.default_rng(3).geometric(0.2, M).clip(0, 60))[::-1]
    return np.where(np.arange(M) < M // 2, 8, 0)       # empty half


def _dealt_in_turn(ip, M):
    """The kernel's test on the row pointers at the edges of the eighths of its tiles."""
    src = generate(standard_kernels()["spmm"], CFG, "hip", write=False).source
    assert re.search(r"const tg_i64 off = 8 \* \(ev - e0\) - l \* all;\s+"
                     r"if \(__ballot\(16 \* \(off < 0 \? -off : off\) > all\)\)", src)
    tn, l = (M + T - 1) // T, np.arange(9)
    ev = ip[np.minimum((l * (tn // 8) + np.minimum(l, tn % 8)) * T, M)]
    off = 8 * (ev - ev[0]) - l * (ev[8] - ev[0])
    return bool((16 * abs(off) > ev[8] - ev[0]).any())


@pytest.mark.parametrize("kind,in_turn", [("alike", False), ("first eighth", True),
                                          ("by length", True), ("empty half", True)])
@pytest.mark.parametrize("M", [100000, 99991])
def test_only_like_shares_are_dealt_in_eighths(kind, in_turn, M):
    ip = np.r_[0, np.cumsum(_lengths(kind, M))]
    assert _dealt_in_turn(ip, M) == in_turn


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["alike", "first eighth", "by length", "empty half"])
def test_every_tile_once(kind, hip_ready):
    for M in (1, T, 7 * T, 8 * T + 1, 64 * T, 67 * T - 3, 2053 * T + 5):
        lengths = _lengths(kind, M)
        rng = np.random.default_rng(M)
        ip = np.r_[0, np.cumsum(lengths)].astype(np.int64)
        A = csr(M, 300, ip, rng.integers(0, 300, ip[-1]), rng.uniform(-1, 1, ip[-1]))
        for K in (17, 33, 64):
            print("[gpu] spmm %s rows=%d K=%d" % (kind, M, K), flush=True)
            _check("spmm", CFG, A, K=K, label="%s rows=%d K=%d" % (kind, M, K))
