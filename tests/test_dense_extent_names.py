"""SpMM and SDDMM whose dense extent is not called "K": the launcher asks for the grid of the
extent the kernel compares, and a launch on the grid that is given for no K in particular writes
every tile."""

from __future__ import annotations

import ctypes
import re

import numpy as np
import pytest

from tests.util import ragged
from tilegen_amd.codegen import Config, generate
from tilegen_amd.dsl import CSR, assign, dense_tensor, i, j, k, kernel, reduce_sum, sparse_tensor
from tilegen_amd.schedules import TUNED

WIDE = Config(tile_size=128, threads_per_row=8, unroll=2, vector_width=2, block_size=512)


def _spmm(F):
    A, B = sparse_tensor("A", CSR, shape=("M", "N")), dense_tensor("B", shape=("N", F))
    C = dense_tensor("C", shape=("M", F))
    return kernel("spmm", [assign(C[i, k], reduce_sum(j, A[i, j] * B[j, k]))])


def _sddmm(F):
    A, C = sparse_tensor("A", CSR, shape=("M", "N")), sparse_tensor("C", CSR, shape=("M", "N"))
    U, V = dense_tensor("U", shape=("M", F)), dense_tensor("V", shape=("N", F))
    return kernel("sddmm", [assign(C[i, j], A[i, j] * reduce_sum(k, U[i, k] * V[j, k]))])


@pytest.mark.parametrize("make", [_spmm, _sddmm], ids=["spmm", "sddmm"])
@pytest.mark.parametrize("F", ["K", "F", "N"])
def test_launcher_passes_the_kernels_dense_extent(make, F):
    host = generate(make(F), WIDE, "hip", write=False).host_source
    assert re.search(r"tgv_geometry\(M, N, %s, nnz, &grid" % F, host)


@pytest.mark.parametrize("make", [_spmm, _sddmm], ids=["spmm", "sddmm"])
def test_grid_is_tgv_geometrys(make, tmp_path):
    from tilegen_amd.verify import compile_generated
    for cfg in (WIDE, TUNED["c4"], TUNED["c5"], Config()):
        gen = generate(make("K"), cfg, "hip", outdir=str(tmp_path))
        lib = ctypes.CDLL(compile_generated(gen, "hip", str(tmp_path))[0])
        lib.tgv_geometry.argtypes = [ctypes.c_int64] * 4 + [ctypes.c_void_p] * 3
        g, b, l = ctypes.c_int64(), ctypes.c_int32(), ctypes.c_int32()
        for M in (0, 1, 63, 700, 100003, 1 << 31):
            for nnz in (0, 1, 5000, 16 * M):
                for K in (0, 1, 16, 17, 32, 33, 64, 65):
                    lib.tgv_geometry(M, 9, K, nnz, ctypes.byref(g), ctypes.byref(b),
                                     ctypes.byref(l))
                    assert gen.geometry.grid(M, nnz, K) == g.value, (cfg.short(), M, nnz, K)
        assert gen.geometry.grid(700, 5000) == gen.geometry.grid(700, 5000, 0)


def _operands(A, F, out):
    rng = np.random.default_rng(4)
    M, N = A.shape
    mats = {"spmm": [(N, F)], "sddmm": [(M, F), (N, F)]}[out]
    return [rng.uniform(-1, 1, s) for s in mats]


def _run(name, cfg, A, F, outdir, raw_grid=None):
    """The launch_<name> of a library whose extent is "F" or its kernel on tgv_geometry's
    grid for ``raw_grid`` columns."""
    from tilegen_amd import runtime as rt
    from tilegen_amd.verify import compile_generated
    gen = generate((_spmm if name == "spmm" else _sddmm)("F"), cfg, "hip", outdir=str(outdir))
    lib = ctypes.CDLL(compile_generated(gen, "hip", str(outdir))[0])
    dense = _operands(A, F, name)
    out = np.full((A.shape[0], F) if name == "spmm" else A.nnz, np.nan)
    bufs = [rt.DeviceBuffer(np.ascontiguousarray(v)) for v in
            [A.indptr.astype(np.int64), A.indices.astype(np.int64), A.data] + dense + [out]]
    dims = {"M": A.shape[0], "N": A.shape[1], "F": F, "nnz": A.nnz}
    vals = list(bufs) + [int(dims[n]) for t, n in gen.abi_args if t == "int64_t"]
    try:
        if raw_grid is None:
            rt.lib().tg_clear_error()
            getattr(lib, "launch_" + name)(*[ctypes.c_void_p(int(v.ptr)) if v in bufs else
                                             ctypes.c_int64(v) for v in vals])
            rt.check_status("launch")
        else:
            g, b, l = ctypes.c_int64(), ctypes.c_int32(), ctypes.c_int32()
            lib.tgv_geometry.argtypes = [ctypes.c_int64] * 4 + [ctypes.c_void_p] * 3
            lib.tgv_geometry(A.shape[0], A.shape[1], raw_grid, 0, ctypes.byref(g),
                             ctypes.byref(b), ctypes.byref(l))
            lib.tgv_function.restype = ctypes.c_void_p
            rt.time_launches(lib.tgv_function(), g.value, b.value, l.value, [vals], 0, 1)
        return bufs[-1].to_host(), dense
    finally:
        for d in bufs:
            d.free()


@pytest.mark.gpu
@pytest.mark.parametrize("raw_grid", [None, 0])
@pytest.mark.parametrize("cfg", [TUNED["c4"], WIDE, TUNED["c5"]], ids=["c4", "wide", "c5"])
def test_every_tile_is_written(cfg, raw_grid, tmp_path, hip_ready):
    A = ragged(61, 900, 700, 12, empty_every=7, long_rows=[(0, 690), (400, 650), (899, 600)])
    rows = np.repeat(np.arange(A.shape[0]), np.diff(A.indptr))
    for F in (16, 33, 64, 130):
        for name in ("spmm", "sddmm"):
            print("[gpu] %s %s F=%d grid %s" % (name, cfg.short(), F, raw_grid), flush=True)
            got, dense = _run(name, cfg, A, F, tmp_path, raw_grid)
            if name == "spmm":
                want, size = A @ dense[0], abs(A) @ np.abs(dense[0])
            else:
                U, V = dense[0][rows], dense[1][A.indices]
                want, size = A.data * (U * V).sum(1), np.abs(A.data) * np.abs(U * V).sum(1)
            # sums of at most 700 products in any order: a rounding each, of the terms' size
            assert (np.abs(got - want) <= 702 * np.finfo(float).eps * size).all(), (name, F)
