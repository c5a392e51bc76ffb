"""Stream ranges dealt to the XCDs in contiguous eighths: the dealing gives every range to one
workgroup (on the CPU), and SpMV and fused_spmv_axpy match the oracle at the grids on both
sides of the lines where the dealing starts and stops (on the GPU), with grids that are and
are not multiples of 8 and rows cut across the edges of the eighths."""

from __future__ import annotations

import re

import numpy as np
import pytest

from tests.test_gpu_parity import _check
from tests.util import csr
from tilegen_amd.codegen import STREAM_XCD, generate
from tilegen_amd.dsl import standard_kernels
from tilegen_amd.schedules import STREAM_TEST_SCHEDULES, TUNED

CFG = STREAM_TEST_SCHEDULES[1]      # ranges of 64: the most workgroups per nonzero
CH = CFG.block_size * CFG.unroll
LOW, HIGH = STREAM_XCD
GRIDS = (1, 2, 7, 8, 9, LOW - 1, LOW, LOW + 1, HIGH, HIGH + 1, HIGH + 2, HIGH + 8)


def test_every_range_has_one_workgroup():
    src = generate(standard_kernels()["spmv"], CFG, "hip", write=False).source
    expr = re.search(r"const tg_i64 e = gridDim.x <= (\d+)u \|\| gridDim.x > (\d+)u \?\s+"
                     r"xc \* xq \+ \(xc < xr \? xc : xr\) \+ blockIdx.x / 8 : blockIdx.x;", src)
    assert expr and (int(expr[1]), int(expr[2])) == STREAM_XCD
    for G in list(range(1, 70)) + list(GRIDS):
        b = np.arange(G)
        e = b % 8 * (G // 8) + np.minimum(b % 8, G % 8) + b // 8
        assert np.array_equal(np.sort(e), b), G


def test_the_upper_line_counts_nonzeros():
    for cfg in STREAM_TEST_SCHEDULES + [TUNED["c3a"], TUNED["c3b"]]:
        ch = cfg.block_size * cfg.unroll
        src = generate(standard_kernels()["spmv"], cfg, "hip", write=False).source
        assert "gridDim.x > %du ?" % ((1 << 22) // ch) in src, cfg.short()


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["c3a", "c3b"])
def test_wider_ranges_at_the_upper_line(case, hip_ready):
    ch = TUNED[case].block_size * TUNED[case].unroll
    for G in ((1 << 22) // ch, (1 << 22) // ch + 1, (1 << 22) // ch + 7):
        nnz, rng = (G - 1) * ch + 5, np.random.default_rng(G)
        ip = np.r_[0, np.sort(rng.integers(0, nnz + 1, nnz // 8)), nnz].astype(np.int64)
        A = csr(ip.size - 1, 700, ip, rng.integers(0, 700, nnz), rng.uniform(-1, 1, nnz))
        print("[gpu] spmv %s stream grid %d" % (case, G), flush=True)
        _check("spmv", TUNED[case], A, K=1, label="%s grid %d" % (case, G))


@pytest.mark.gpu
@pytest.mark.parametrize("G", GRIDS)
def test_stream_grids_at_the_lines(G, hip_ready):
    nnz = (G - 1) * CH + CH // 2               # floor(nnz / CH) + 1 = G ranges
    rng = np.random.default_rng(G)
    M, N = max(1, nnz // 9), 500
    cuts = np.sort(rng.integers(0, nnz + 1, M - 1))
    if M > 20:
        cuts[M // 3:M // 3 + 4] = cuts[M // 3]   # a row over many ranges, empty rows before it
        cuts[M // 3 + 4:M // 3 + 9] = cuts[min(M - 2, M // 3 + 60)]
        cuts = np.sort(cuts)
    ip = np.r_[0, cuts, nnz].astype(np.int64)
    A = csr(M, N, ip, rng.integers(0, N, nnz), rng.uniform(-1, 1, nnz))
    for kernel in ("spmv", "fused_spmv_axpy"):
        print("[gpu] %s stream grid %d rows=%d nnz=%d" % (kernel, G, M, nnz), flush=True)
        _check(kernel, CFG, A, K=1, label="grid %d" % G)
