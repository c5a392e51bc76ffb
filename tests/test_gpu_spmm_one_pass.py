"""GPU parity of SpMM where a lane group's columns just cover K, just miss it and are twice too
many, on rows alike, rows that dwarf their tile and a band; and of the two column slices past 64
columns, which small grids take on whole 128-byte lines and on bands."""

from __future__ import annotations

import pytest

from tests.test_gpu_parity import _check
from tests.util import ragged
from tilegen_amd.matrices import make_baseline
from tilegen_amd.schedules import TEST_SCHEDULES, TUNED, schedule_id

pytestmark = pytest.mark.gpu

CFGS = [TUNED["c4"], TEST_SCHEDULES[4], TEST_SCHEDULES[5], TEST_SCHEDULES[6]]


@pytest.mark.parametrize("cfg", CFGS, ids=[schedule_id(c) for c in CFGS])
def test_spmm_lane_groups_that_cover_k(cfg, hip_ready):
    lanes, pairs = cfg.threads_per_row, 2 * cfg.threads_per_row
    mats = {"alike": make_baseline("c1", scale=0.01), "band": make_baseline("c2", scale=0.01),
            "dwarfing": ragged(91, 600, 3000, 9, empty_every=5,
                               long_rows=[(0, 2900), (300, 1500), (599, 1000)])}
    for label, A in mats.items():
        for K in sorted({17, 20, lanes - 1, lanes, lanes + 1, pairs - 2, pairs, pairs + 1, pairs + 2,
                         80, 96, 112, 144, 272}):
            print("[gpu] spmm %s %s K=%d" % (cfg.short(), label, K), flush=True)
            _check("spmm", cfg, A, K=K, label="%s K=%d" % (label, K))
