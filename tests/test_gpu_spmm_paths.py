"""GPU parity of SpMM's paths over staged row pointers, at the edges of the rule that
chooses them: K up to 16 (lane groups alone), 17 to 32 (two column slices per lane group),
over 32 (one wave per nonzero, 64, 128 or 256 columns a pass, with one to three columns
left over), whole 128-byte lines (lane groups again, unless the tile is skewed or its
columns lie close together); rows that dwarf their tile (the helper workgroups) alone, side
by side, first and last, and rows cut between the waves of a tile."""

from __future__ import annotations

import numpy as np
import pytest

from tests.test_gpu_parity import _check, _operands
from tests.util import csr, ragged
from tilegen_amd.codegen import Config
from tilegen_amd.matrices import make_baseline
from tilegen_amd.schedules import TUNED, schedule_id
from tilegen_amd.variant import Variant

pytestmark = pytest.mark.gpu

CFGS = [
    TUNED["c4"],                                                     # one wave per tile
    Config(tile_size=128, threads_per_row=8, unroll=2, vector_width=2, block_size=512),
    Config(tile_size=12, threads_per_row=64, unroll=1, vector_width=1, block_size=192),
    Config(tile_size=1024, threads_per_row=8, unroll=2, vector_width=2, block_size=1024),
    Config(tile_size=2, threads_per_row=32, unroll=16, vector_width=2, block_size=64),
]
KS = (16, 17, 31, 32, 33, 48, 64, 65, 127, 128, 129, 130, 256, 257, 259)


def _unsorted(A):
    """The same matrix with every row's columns descending."""
    ind, dat = A.indices.copy(), A.data.copy()
    for r in range(A.shape[0]):
        s = slice(A.indptr[r], A.indptr[r + 1])
        ind[s], dat[s] = ind[s][::-1].copy(), dat[s][::-1].copy()
    return csr(A.shape[0], A.shape[1], A.indptr, ind, dat)


def _matrices():
    dwarf = ragged(41, 700, 6000, 9, empty_every=6,
                   long_rows=[(0, 5000), (40, 3000), (41, 2600), (300, 1100), (301, 900),
                              (302, 130), (699, 4000)])
    return {
        "dwarfing rows": dwarf,
        "dwarfing rows, columns descending": _unsorted(dwarf),
        "every row long": ragged(42, 70, 3000, 0, long_rows=[(r, 300 + 7 * r) for r in range(70)]),
        "one row": ragged(43, 1, 4000, 0, long_rows=[(0, 3500)]),
        "banded": make_baseline("c2", scale=0.004),
        "uniform": make_baseline("c1", scale=0.008),
        "no nonzeros": csr(90, 50, np.zeros(91, dtype=np.int64), [], []),
    }


@pytest.mark.parametrize("cfg", CFGS, ids=[schedule_id(c) for c in CFGS])
def test_spmm_paths(cfg, hip_ready):
    for label, A in _matrices().items():
        for K in KS:
            print("[gpu] spmm %s %s K=%d" % (cfg.short(), label, K), flush=True)
            _check("spmm", cfg, A, K=K, label="%s K=%d" % (label, K))


@pytest.mark.parametrize("K", [20, 63, 64, 130])
def test_spmm_again_onto_nan_gives_the_same_bits(K, hip_ready):
    """Cut rows and helper sums are added in a fixed order, and every element of C is
    written, rows without nonzeros included."""
    A = _matrices()["dwarfing rows"]
    for cfg in CFGS[:2]:
        v, ops = Variant("spmm", cfg), _operands("spmm", A, K)
        first = v.run(A, **ops)
        assert np.array_equal(v.run(A, out=np.full((A.shape[0], K), np.nan), **ops), first)


@pytest.mark.parametrize("K", [20, 33, 64, 65, 200])
def test_spmm_rows_of_b_that_no_nonzero_names_stay_out(K, hip_ready):
    """Masked lanes load a row that the tile names, so infinities and NaNs elsewhere in B
    (its first and last rows among them) cannot reach a sum."""
    A = _matrices()["dwarfing rows"]
    A = csr(A.shape[0], A.shape[1] + 2, A.indptr, A.indices + 1, A.data)
    B = np.random.default_rng(5).uniform(-1, 1, size=(A.shape[1], K))
    B[0], B[-1] = np.inf, np.nan
    want = A[:, 1:-1] @ B[1:-1]
    for cfg in CFGS[:3]:
        out = Variant("spmm", cfg).run(A, B=B)
        # sums of at most 5000 products of numbers in (-1, 1): 5000 eps each at most
        assert np.abs(out - want).max() <= 5000 * np.finfo(float).eps * 5000 ** 0.5
