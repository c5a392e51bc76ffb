"""GPU parity of SpMM's band path (B rows staged in LDS) at its edges: tiles whose columns span
exactly the staged rows and one more, rows of eight nonzeros and of nine, empty rows, a last tile
of one row, columns out of order, K with and without columns left over 16; and B rows inside a
tile's span that no nonzero names stay out of the sums, non-finite or not."""

from __future__ import annotations

import numpy as np
import pytest

from tests.test_gpu_parity import _check, _operands
from tests.util import csr
from tilegen_amd.codegen import SPMM_BAND
from tilegen_amd.schedules import TUNED
from tilegen_amd.variant import Variant

pytestmark = pytest.mark.gpu

CFG = TUNED["c4"]
T = CFG.tile_size
M = 2048 * T + 1        # the path is for grids of at least 2048 one-wave tiles
KS = (33, 34, 47, 48, 49, 64, 65, 130)


def _band(span, longest, skip=0):
    """Tile t's columns lie in [t T, t T + span), both ends used; every ``skip``-th row empty,
    the others of 1 to ``longest`` columns in random order."""
    rng = np.random.default_rng(span * 100 + longest)
    N, ip, ind = M + span, [0], []
    for r in range(M):
        base, n = r // T * T, int(rng.integers(1, longest + 1))
        if r % T == 0:
            cols = [base + span - 1, base]
        elif r % T == T - 1:
            cols = base + rng.permutation(span)[:longest]
        elif skip and r % skip == 0:
            cols = []
        else:
            cols = base + rng.permutation(span)[:n]
        ind.extend(cols)
        ip.append(len(ind))
    return csr(M, N, ip, ind, rng.uniform(-1, 1, len(ind)))


@pytest.mark.parametrize("span,longest,skip", [(SPMM_BAND, 8, 3), (SPMM_BAND + 1, 8, 0),
                                               (SPMM_BAND, 9, 5), (9, 8, 0)])
def test_spmm_band_edges(span, longest, skip, hip_ready):
    A = _band(span, longest, skip)
    for K in KS:
        print("[gpu] spmm band span=%d longest=%d K=%d" % (span, longest, K), flush=True)
        _check("spmm", CFG, A, K=K, label="span %d, rows of %d, K=%d" % (span, longest, K))


@pytest.mark.parametrize("K", [33, 64, 130])
def test_spmm_band_rows_of_b_that_no_nonzero_names(K, hip_ready):
    A = _band(SPMM_BAND, 5)
    A.data[:] = np.where(A.indices % 3 == 1, 0.0, A.data)
    keep = A.indices % 3 != 1
    ip = np.r_[0, np.cumsum(np.add.reduceat(keep, A.indptr[:-1]))]
    A = csr(A.shape[0], A.shape[1], ip, A.indices[keep], A.data[keep])
    Bm = _operands("spmm", A, K)["B"]
    bad = Bm.copy()
    bad[1::3] = np.nan
    v = Variant("spmm", CFG)
    assert np.array_equal(v.run(A, B=bad), v.run(A, B=Bm))
