"""SDDMM kernels whose output reads more than the sparse value and the dot product: a scalar
factor, a row vector, both.  They compile for gfx950 under every schedule form, and match on
the GPU at K on both sides of the chunked path's limit, over rows that dwarf their tile and
runs that cross rows."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from tests.util import ragged
from tilegen_amd.codegen import Config, generate
from tilegen_amd.dsl import (CSR, assign, dense_tensor, i, j, k, kernel, reduce_sum,
                             scalar_tensor, sparse_tensor)
from tilegen_amd.schedules import TUNED
from tilegen_amd.verify import compile_generated

CFGS = [TUNED["c5"], Config(tile_size=32, threads_per_row=1, unroll=1, vector_width=1),
        Config(tile_size=1, threads_per_row=4, unroll=1, vector_width=1, block_size=64)]
FORMS = ["scalar", "vector", "both"]


def _kernel(form):
    A, C = sparse_tensor("A", CSR, shape=("M", "N")), sparse_tensor("C", CSR, shape=("M", "N"))
    U, V = dense_tensor("U", shape=("M", "K")), dense_tensor("V", shape=("N", "K"))
    d, per = dense_tensor("d", shape=("M",)), scalar_tensor("per")
    out = A[i, j] * reduce_sum(k, U[i, k] * V[j, k])
    if form != "scalar":
        out = A[i, j] * d[i] * reduce_sum(k, U[i, k] * V[j, k])
    return kernel("sddmm", [assign(C[i, j], out if form == "vector" else per * out)])


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("cfg", CFGS, ids=["c5", "narrow", "untiled"])
def test_output_expression_compiles(form, cfg, tmp_path):
    compile_generated(generate(_kernel(form), cfg, "hip", outdir=str(tmp_path)), "hip",
                      str(tmp_path))


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("cfg", CFGS, ids=["c5", "narrow", "untiled"])
def test_output_expression(form, cfg, tmp_path, hip_ready):
    from tilegen_amd import runtime as rt
    A = ragged(71, 900, 700, 12, empty_every=7, long_rows=[(0, 690), (400, 650), (899, 600)])
    rows, rng = np.repeat(np.arange(A.shape[0]), np.diff(A.indptr)), np.random.default_rng(6)
    gen = generate(_kernel(form), cfg, "hip", outdir=str(tmp_path))
    lib = ctypes.CDLL(compile_generated(gen, "hip", str(tmp_path))[0])
    for K in (1, 2, 63, 64, 65, 130):
        arrays = {"indptr": A.indptr.astype(np.int64), "indices": A.indices.astype(np.int64),
                  "data": A.data, "d": rng.uniform(-1, 1, A.shape[0]),
                  "U": rng.uniform(-1, 1, (A.shape[0], K)),
                  "V": rng.uniform(-1, 1, (A.shape[1], K)), "C": np.full(A.nnz, np.nan)}
        per, dims = 1.75, {"M": A.shape[0], "N": A.shape[1], "K": K, "nnz": A.nnz}
        bufs = {n: rt.DeviceBuffer(v) for n, v in arrays.items()}
        args = [ctypes.c_void_p(bufs[n].ptr) if t.endswith("*") else
                ctypes.c_double(per) if t == "double" else ctypes.c_int64(dims[n])
                for t, n in gen.abi_args]
        print("[gpu] sddmm %s %s K=%d" % (form, cfg.short(), K), flush=True)
        rt.lib().tg_clear_error()
        lib.launch_sddmm(*args)
        rt.check_status("launch_sddmm")
        got = bufs["C"].to_host()
        for b in bufs.values():
            b.free()
        f = A.data * (arrays["d"][rows] if form != "scalar" else 1.0) * \
            (per if form != "vector" else 1.0)
        terms = arrays["U"][rows] * arrays["V"][A.indices]
        # K products and sums and the output's factors, a rounding each of the terms' size
        err = (K + 4) * np.finfo(float).eps * np.abs(f) * np.abs(terms).sum(1)
        assert (np.abs(got - f * terms.sum(1)) <= err).all(), (form, cfg.short(), K)
