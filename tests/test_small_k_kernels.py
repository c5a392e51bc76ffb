"""SpMM and SDDMM's two code objects: no schedule that is shipped or tested spills to scratch in
either; on the GPU the one of few columns gives the bits of the whole kernel at every K that
takes it, and a program that has launched at one K captures a launch at the other."""

from __future__ import annotations

import os
import re
import subprocess

import numpy as np
import pytest

from tests.test_gpu_parity import _operands
from tests.util import ragged
from tilegen_amd.codegen import Config, generate
from tilegen_amd.dsl import standard_kernels
from tilegen_amd.schedules import ODD_BLOCK_SCHEDULES, TEST_SCHEDULES, TUNED
from tilegen_amd.variant import Variant
from tilegen_amd.verify import compile_generated

WIDE = Config(tile_size=128, threads_per_row=8, unroll=2, vector_width=2, block_size=512)
NARROW = Config()      # one lane per row, single columns
BATCH32 = Config(tile_size=2, threads_per_row=32, unroll=16, vector_width=2, block_size=64)


@pytest.mark.parametrize("kernel,most", [("spmm", 64), ("sddmm", 130)])
def test_no_schedule_uses_scratch(kernel, most, tmp_path):
    readelf = "/opt/rocm/llvm/bin/llvm-readelf"
    if not os.path.exists(readelf):
        pytest.skip("llvm-readelf not available")
    for cfg in [TUNED["c4"], TUNED["c5"], NARROW, BATCH32] + TEST_SCHEDULES + ODD_BLOCK_SCHEDULES:
        gen = generate(standard_kernels()[kernel], cfg, "hip", outdir=str(tmp_path))
        co = compile_generated(gen, "hip", str(tmp_path))[0][:-3]
        for path in (co + ".co", co + "_small.co"):
            if not os.path.exists(path):
                assert cfg.tile_size <= 1 and kernel == "spmm"   # one path, one code object
                continue
            notes = subprocess.run([readelf, "--notes", path], capture_output=True,
                                   text=True).stdout
            meta = dict(re.findall(r"\.(private_segment_fixed_size|vgpr_spill_count|vgpr_count):"
                                   r"\s+(\d+)", notes))
            assert meta["private_segment_fixed_size"] == "0", (cfg.short(), path, meta)
            assert meta["vgpr_spill_count"] == "0", (cfg.short(), path, meta)
            # light schedules (a batch of at most 8 doubles) stay light at few columns
            if cfg.unroll * cfg.vector_width * (cfg.threads_per_row <= 8) in range(1, 9) \
                    and path.endswith("_small.co"):
                assert int(meta["vgpr_count"]) <= most, (cfg.short(), path, meta)


def _bufs(kernel, A, K):
    from tilegen_amd import runtime as rt
    ops = _operands(kernel, A, K)
    host = {"indptr": A.indptr.astype(np.int64), "indices": A.indices.astype(np.int64),
            "data": np.asarray(A.data, dtype=np.float64), **ops,
            "C": np.full((A.shape[0], K) if kernel == "spmm" else A.nnz, np.nan)}
    return {k: rt.DeviceBuffer(v) for k, v in host.items()}


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", ["spmm", "sddmm"])
@pytest.mark.parametrize("cfg", [TUNED["c4"], TUNED["c5"], WIDE, NARROW, TEST_SCHEDULES[6]],
                         ids=["c4", "c5", "wide", "narrow", "64 lanes"])
def test_small_kernel_gives_the_whole_kernels_bits(kernel, cfg, hip_ready):
    from tilegen_amd import runtime as rt
    A = ragged(81, 700, 900, 12, empty_every=6, long_rows=[(0, 880), (300, 700), (301, 60)])
    v = Variant(kernel, cfg)
    for K in (1, 2, 8, 15, 16, 17, 32, 64):
        print("[gpu] %s %s K=%d" % (kernel, cfg.short(), K), flush=True)
        bufs = _bufs(kernel, A, K)
        try:
            vals = v.abi_values(A, bufs, {}, *A.shape, K, A.nnz)
            v.device_call(vals)
            got = bufs["C"].to_host()
            bufs["C"].upload(np.full_like(got, np.nan))
            g, b, l = v.geometry(*A.shape, K, A.nnz)
            rt.time_launches(v.function(), g, b, l, [vals], 0, 1)
            assert np.array_equal(bufs["C"].to_host(), got), K
        finally:
            for d in bufs.values():
                d.free()


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", ["spmm", "sddmm"])
@pytest.mark.parametrize("first,then", [(130, 8), (8, 130)])
def test_capture_at_another_k(kernel, first, then, tmp_path, hip_ready):
    from tilegen_amd import runtime as rt
    A = ragged(82, 500, 600, 12)
    # a schedule of its own per case, so that neither code object is loaded yet
    v = Variant(kernel, Config(tile_size=16, threads_per_row=8, unroll=1, vector_width=1,
                               block_size=128 if first < then else 256))
    sets = {K: _bufs(kernel, A, K) for K in (first, then)}
    vals = {K: v.abi_values(A, b, {}, *A.shape, K, A.nnz) for K, b in sets.items()}
    s, exec_ = rt.stream_create(), None
    try:
        v.launch_async(vals[first], s)
        rt.stream_synchronize(s)
        print("[gpu] graph %s K=%d after K=%d" % (kernel, then, first), flush=True)
        exec_ = rt.graph_capture(s, lambda: v.launch_async(vals[then], s))
        y = sets[then]["C"]
        v.device_call(vals[then])
        want = y.to_host()
        for _ in range(4):
            y.upload(np.full_like(want, np.nan))
            rt.graph_launch(exec_, s, sync=True)
            assert np.array_equal(y.to_host(), want)
            v.device_call(vals[first])
    finally:
        if exec_:
            rt.graph_destroy(exec_)
        rt.stream_destroy(s)
        for b in sets.values():
            for d in b.values():
                d.free()
