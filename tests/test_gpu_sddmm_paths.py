"""GPU parity of SDDMM's paths at the edges of the rule that chooses them: the chunked path
with rows that dwarf their tile (the helper workgroups at position boundaries) and the runs of
equal nonzeros per wave (K odd, over the chunked path's registers, or an unaligned base), for
each width of the runs' lane groups; runs that begin and end inside rows, rows without
nonzeros by the hundred between two nonzeros, one row alone, and neighbouring rows that share
their columns (the wave-per-row path)."""

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
    TUNED["c5"],
    Config(tile_size=128, threads_per_row=8, unroll=2, vector_width=2, block_size=512),
    Config(tile_size=12, threads_per_row=64, unroll=1, vector_width=1, block_size=192),
    Config(tile_size=32, threads_per_row=1, unroll=1, vector_width=1, block_size=128),
    Config(tile_size=1, threads_per_row=4, unroll=1, vector_width=1, block_size=64),  # untiled
]
KS = (1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 130, 255, 256, 257, 259)


def _sparse_rows():
    """3000 rows, nonzeros in every 701st alone: hundreds of empty rows inside one run."""
    return ragged(52, 3000, 400, 0, long_rows=[(r, 3 + r % 90) for r in range(5, 3000, 701)])


def _matrices():
    return {
        "dwarfing rows": ragged(51, 700, 6000, 9, empty_every=6,
                                long_rows=[(0, 5000), (40, 3000), (41, 2600), (300, 1100),
                                           (302, 257), (699, 4000)]),
        "rows far apart": _sparse_rows(),
        "one row": ragged(53, 1, 4000, 0, long_rows=[(0, 3500)]),
        "one nonzero": csr(400, 5, np.r_[np.zeros(200, dtype=np.int64), np.ones(201, dtype=np.int64)],
                           [3], [2.5]),
        "blocks": make_baseline("c5", scale=0.01),
        "no nonzeros": csr(90, 50, np.zeros(91, dtype=np.int64), [], []),
    }


@pytest.mark.parametrize("cfg", CFGS, ids=[schedule_id(c) for c in CFGS])
def test_sddmm_paths(cfg, hip_ready):
    for label, A in _matrices().items():
        for K in KS:
            print("[gpu] sddmm %s %s K=%d" % (cfg.short(), label, K), flush=True)
            _check("sddmm", cfg, A, K=K, label="%s K=%d" % (label, K))


@pytest.mark.parametrize("K", [7, 33, 64, 65, 130, 300])
def test_sddmm_rows_that_no_nonzero_names_stay_out(K, hip_ready):
    """Lanes past K and past a run load what others own and add none of it: infinities and
    NaNs in rows of U and V that no nonzero names cannot reach a result, and every output
    is written."""
    A = _matrices()["dwarfing rows"]
    A = csr(A.shape[0], A.shape[1] + 2, A.indptr, A.indices + 1, A.data)
    ops = _operands("sddmm", A, K)
    U, V = np.array(ops["U"]), np.array(ops["V"])
    V[0], V[-1] = np.inf, np.nan
    U[np.diff(A.indptr) == 0] = np.nan
    rows = np.repeat(np.arange(A.shape[0]), np.diff(A.indptr))
    want = A.data * np.einsum("ik,ik->i", U[rows], V[A.indices])
    scale = np.abs(A.data) * np.einsum("ik,ik->i", np.abs(U[rows]), np.abs(V[A.indices]))
    for cfg in CFGS[:3]:
        out = Variant("sddmm", cfg).run(A, U=U, V=V, out=np.full(A.nnz, np.nan))
        # a sum of K products in any order: K + 2 roundings of its terms' size
        assert (np.abs(out - want) <= (K + 2) * np.finfo(float).eps * scale).all()
