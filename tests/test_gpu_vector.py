"""GrB_vxm / GrB_mxv (vectors as 1 x n rows on GrB_mxm's kernels) on the GPU
against the oracle."""
import ctypes

import numpy as np
import pytest

import pyoracle as O
from graphblas_amd import capi
from graphblas_amd import workloads as W
from helpers import SR, ZT, DevCsr, assert_csr_equal, download, rand_csr

pytestmark = pytest.mark.gpu


def _row(idx, vals, n):
    """1 x n CSR of a sparse vector."""
    order = np.argsort(idx)
    return W.Csr(1, n, np.array([0, len(idx)], dtype=np.int64), np.asarray(idx, dtype=np.int64)[order],
                 None if vals is None else np.asarray(vals)[order])


def _got(w, n):
    I, X = w.to_arrays()
    return W.Csr(1, n, np.array([0, len(I)], dtype=np.int64), I, X)


def test_vxm_bfs_step(grb):
    """q'<!v'> = q'*A with ANY_SECONDI (the BFS step; GrB_DESC_RSC)."""
    G = W.rmat_sym(12, 16, seed=3)
    n = G.nrows
    Gd = capi.Matrix.from_csr(G, "bool")
    rng = np.random.default_rng(1)
    src = np.sort(rng.choice(n, 20, replace=False))
    q = capi.Vector.from_arrays(src, np.ones(20, dtype=np.int64), "int64", n)
    vis = np.union1d(src, rng.choice(n, 200, replace=False))
    v = capi.Vector.from_arrays(vis, np.ones(len(vis), dtype=bool), "bool", n)
    w = capi.Vector("int64", n)
    assert capi.vxm(w, v, "GxB_ANY_SECONDI_INT64", q, Gd, "RSC") == 0, capi.last_error()
    F = _row(src, np.ones(20, dtype=np.int64), n)
    V = _row(vis, None, n)
    ref = O.saxpy3("any_secondi_int64", F, G, M=V, mask_comp=True)
    assert_csr_equal(_got(w, n), ref, what="vxm bfs")


@pytest.mark.parametrize("desc", [None, "T0"])
def test_mxv_plus_times(grb, desc):
    rng = np.random.default_rng(7)
    A = rand_csr(120, 90, 0.05, rng, "fp64")
    Ad = capi.Matrix.from_csr(A, "fp64")
    ulen = 90 if desc is None else 120
    idx = np.sort(rng.choice(ulen, 30, replace=False))
    vals = rng.random(30)
    u = capi.Vector.from_arrays(idx, vals, "fp64", ulen)
    wlen = 120 if desc is None else 90
    w = capi.Vector("fp64", wlen)
    assert capi.mxv(w, None, "GrB_PLUS_TIMES_SEMIRING_FP64", Ad, u, desc) == 0, capi.last_error()
    U = _row(idx, vals, ulen)
    # w' = u' * A'  (A*u), or u' * A (A'*u)
    B = O.transpose(A) if desc is None else A
    ref = O.saxpy3("plus_times_fp64", U, B)
    assert_csr_equal(_got(w, wlen), ref, fp_tol=1e-12, what=f"mxv {desc}")
    # the dense product agrees too
    dense = A.to_scipy().toarray()
    uu = np.zeros(ulen)
    uu[idx] = vals
    dw = dense @ uu if desc is None else dense.T @ uu
    I, X = w.to_arrays()
    assert np.allclose(dw[I], X, rtol=1e-12, atol=0)


def test_vxm_transposed_with_accum_and_mask(grb):
    rng = np.random.default_rng(9)
    A = rand_csr(80, 60, 0.08, rng, "int64")
    Ad = capi.Matrix.from_csr(A, "int64")
    idx = np.sort(rng.choice(60, 25, replace=False))
    vals = rng.integers(-5, 6, 25)
    u = capi.Vector.from_arrays(idx, vals, "int64", 60)
    w0i = np.sort(rng.choice(80, 30, replace=False))
    w0x = rng.integers(-5, 6, 30)
    w = capi.Vector.from_arrays(w0i, w0x, "int64", 80)
    mi = np.sort(rng.choice(80, 40, replace=False))
    m = capi.Vector.from_arrays(mi, np.ones(40, dtype=bool), "bool", 80)
    # w'<m'> += u' * A'   (GrB_INP1 = TRAN)
    assert capi.vxm(w, m, "GrB_PLUS_TIMES_SEMIRING_INT64", u, Ad, "T1", accum="GrB_PLUS_INT64") == 0, \
        capi.last_error()
    U = _row(idx, vals.astype(np.int64), 60)
    M = _row(mi, None, 80)
    T = O.saxpy3("plus_times_int64", U, O.transpose(A), M=M)
    C0 = _row(w0i, w0x.astype(np.int64), 80)
    ref = O.accum_mask(C0, M, T, op=1, dtype=np.int64)
    assert_csr_equal(_got(w, 80), ref, what="w<m> += u'A'")


def _mostly_empty(rng):
    """Row lengths: 70001 rows, 1 to 3 entries in 2400 of them, some long ones,
    one longer than a chunk, the last row empty."""
    lens = np.zeros(70001, dtype=np.int64)
    lens[rng.choice(70000, 2400, replace=False)] = rng.integers(1, 4, 2400)
    lens[[0, 17, 30000, 50000, 60000, 69999]] = [1, 65, 3000, 64, 100, 200]
    return lens


@pytest.mark.parametrize("comp", [False, True])
@pytest.mark.parametrize("shape", ["one row", "short", "hub", "chunk", "empty rows"])
@pytest.mark.parametrize("handle", ["GxB_PLUS_PAIR_INT64", "GxB_PLUS_PAIR_INT32", "GxB_ANY_PAIR_BOOL",
                                    "GxB_ANY_SECONDI_INT64", "GrB_PLUS_TIMES_SEMIRING_INT64",
                                    "GrB_MIN_PLUS_SEMIRING_INT32", "GrB_MAX_PLUS_SEMIRING_INT32",
                                    "GrB_MIN_PLUS_SEMIRING_FP64", "GrB_PLUS_TIMES_SEMIRING_FP64"])
def test_vxm_bt(grb, handle, shape, comp):
    """u'*B' without a transpose: one row, many short and empty rows, rows that
    span several chunks of 2048 entries, rows that end where a chunk ends, and
    chunks that span more empty rows than a workgroup walks."""
    print(f"[vector] vxm_bt {handle} {shape} comp={comp}", flush=True)
    rng = np.random.default_rng(len(handle) + len(shape))
    K = 9000
    lens = {"one row": [4096], "short": rng.integers(0, 9, 3000), "chunk": [2048, 0, 1, 2047, 64, 65, 1919, 2048],
            "empty rows": _mostly_empty(rng), "hub": np.where(np.arange(300) % 97 == 5, 8500, rng.integers(0, 40, 300))}[shape]
    p = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    j = np.concatenate([np.sort(rng.choice(K, size=int(l), replace=False)) for l in lens]).astype(np.int64)
    n, name = len(lens), SR[handle][0]
    vt = {"INT64": "int64", "INT32": "int32", "FP64": "fp64", "BOOL": "bool"}[handle.split("_")[-1]]

    def vals(k):
        return (rng.random(k) if vt == "fp64" else rng.integers(1, 100, k)).astype(
            {"int64": np.int64, "int32": np.int32, "fp64": np.float64, "bool": np.uint8}[vt])
    B = W.Csr(n, K, p, j, vals(len(j)))
    ui = np.sort(rng.choice(K, size=K // 2, replace=False)).astype(np.int64)
    U = _row(ui, vals(len(ui)), K)
    M = _row(np.arange(0, n, 3), rng.integers(0, 2, len(range(0, n, 3))).astype(np.int64), n) if comp else None
    code = SR[handle][1][2]
    dU, dB = DevCsr(U, code), DevCsr(B, code)
    dM = DevCsr(M, 8) if comp else None
    out, sr = capi.GmCsrOut(), capi.GmSemiring(*SR[handle][1])
    rc = capi.lib().gm_vxm_bt(ctypes.byref(out), ctypes.byref(dM.view) if comp else None, False,
                              ctypes.byref(dU.view), ctypes.byref(dB.view), len(j), ctypes.byref(sr))
    assert rc == 0, capi.last_error()
    got = download(out, ZT[vt])
    kw = {"M": M, "mask_comp": True, "mask_struct": False} if comp else {}
    ref = O.saxpy3(name, U, O.transpose(B), **kw)
    # tree sums of at most 8500 positive products against sequential ones
    assert_csr_equal(got, ref, fp_tol=1e-12 if "PLUS_TIMES_SEMIRING_FP64" in handle else None, what=shape)
    for d in (dU, dB, dM):
        if d:
            d.free()


def test_vxm_nan_products_both_ways(grb):
    """min_plus_fp64 over NaN products: u'*B' read as held and u'*C with C = B'
    held by rows agree, an entry whose products are all NaN is NaN."""
    rng = np.random.default_rng(17)
    B = rand_csr(400, 3000, 0.05, rng, "fp64")
    B.x[rng.random(B.nnz) < 0.7] = np.nan
    rows = np.repeat(np.arange(400), np.diff(B.p))
    B.x[rows % 3 == 0] = np.nan
    ui = np.sort(rng.choice(3000, 2000, replace=False))
    ux = rng.random(2000)
    u = capi.Vector.from_arrays(ui, ux, "fp64", 3000)
    ref = O.saxpy3("min_plus_fp64", _row(ui, ux, 3000), O.transpose(B))
    assert np.isnan(ref.x).any() and (~np.isnan(ref.x)).any()
    Bd, Bt = capi.Matrix.from_csr(B, "fp64"), capi.Matrix.from_csr(O.transpose(B), "fp64")
    for what, call in (("mxv", lambda w: capi.mxv(w, None, "GrB_MIN_PLUS_SEMIRING_FP64", Bd, u)),
                       ("vxm", lambda w: capi.vxm(w, None, "GrB_MIN_PLUS_SEMIRING_FP64", u, Bt))):
        w = capi.Vector("fp64", 400)
        assert call(w) == 0, capi.last_error()
        got = _got(w, 400)
        assert np.array_equal(got.j, ref.j), what
        assert np.array_equal(got.x, ref.x, equal_nan=True), what


def test_mxv_without_room_for_dense_vectors(grb):
    """An allocation forced to fail anywhere in the product that reads B as
    held: B is transposed instead and the result is the same."""
    rng = np.random.default_rng(23)
    B = rand_csr(300, 500, 0.05, rng, "int64")
    Bd = capi.Matrix.from_csr(B, "int64")
    ui = np.sort(rng.choice(500, 200, replace=False))
    ux = rng.integers(-9, 10, 200)
    u = capi.Vector.from_arrays(ui, ux, "int64", 500)
    ref = O.saxpy3("plus_times_int64", _row(ui, ux, 500), O.transpose(B))
    L = capi.lib()
    for n in range(8):
        w = capi.Vector("int64", 300)
        L.gm_debug_fail_after(n)
        try:
            rc = capi.mxv(w, None, "GrB_PLUS_TIMES_SEMIRING_INT64", Bd, u)
        finally:
            L.gm_debug_fail_after(-1)
        assert rc == 0, f"allocation {n}: {capi.last_error()}"
        assert_csr_equal(_got(w, 300), ref, what=f"allocation {n}")


def test_mxv_empty_rows_cost(grb):
    """Empty rows are not walked one workgroup at a time: 2000 entries in 2^24
    rows take at most 10 times a call on 2^12 rows (2.3 times as measured)."""
    import time
    best = {}
    for lg in (12, 24):
        n, rng = 1 << lg, np.random.default_rng(lg)
        key = np.sort(rng.choice(n, 2000, replace=False))
        B = W.Csr(n, n, np.searchsorted(key, np.arange(n + 1)).astype(np.int64), rng.permutation(key), rng.random(2000))
        Bd = capi.Matrix.from_csr(B, "fp64")
        u = capi.Vector.from_arrays(key, np.ones(2000), "fp64", n)
        w = capi.Vector("fp64", n)
        ts = []
        for _ in range(8):
            t = time.perf_counter()
            assert capi.mxv(w, None, "GrB_PLUS_TIMES_SEMIRING_FP64", Bd, u) == 0, capi.last_error()
            ts.append(time.perf_counter() - t)
        best[lg] = min(ts)
        got = _got(w, n)
        assert np.array_equal(got.j, key) and np.array_equal(got.x, B.x)
    assert best[24] <= 10 * best[12], best


@pytest.mark.parametrize("handle", ["GrB_PLUS_TIMES_SEMIRING_FP64", "GxB_ANY_PAIR_BOOL"])
@pytest.mark.parametrize("lg", [18, 22, 23])
def test_mxv_result_memory(grb, lg, handle):
    """A sparse result of a long one-row product keeps about its entries'
    memory, below and above the size that is written at its bound (2^22 fp64
    entries), also as the product of a spread row."""
    n, L = 1 << lg, capi.lib()
    rng = np.random.default_rng(lg)
    vt = "fp64" if "FP64" in handle else "bool"
    key = np.sort(rng.choice(n, 2000, replace=False))
    one = np.ones(2000, dtype=np.float64 if vt == "fp64" else bool)
    B = W.Csr(n, n, np.searchsorted(key, np.arange(n + 1)).astype(np.int64), rng.permutation(key),
              rng.random(2000) if vt == "fp64" else one.astype(np.uint8))
    Bd = capi.Matrix.from_csr(B, vt)
    u = capi.Vector.from_arrays(key, one, vt, n)
    w = capi.Vector(vt, n)
    before = L.gm_arena_bytes_in_use()
    assert capi.mxv(w, None, handle, Bd, u) == 0, capi.last_error()
    held = L.gm_arena_bytes_in_use() - before
    got = _got(w, n)
    assert np.array_equal(got.j, key) and (vt == "bool" or np.array_equal(got.x, B.x))
    assert held <= 5 << 20, f"{held} bytes for 2000 entries"
    # 50000 rows with the same 40 columns: 2 million products, 40 entries
    D = W.Csr(50000, n, np.arange(50001) * 40, np.tile(np.arange(40) * (n // 40), 50000),
              rng.random(2000000) if vt == "fp64" else np.ones(2000000, dtype=np.uint8))
    Dd = capi.Matrix.from_csr(D, vt)
    v = capi.Vector.from_arrays(np.arange(50000), np.ones(50000, dtype=one.dtype), vt, 50000)
    w = capi.Vector(vt, n)
    before = L.gm_arena_bytes_in_use()
    assert capi.vxm(w, None, handle, v, Dd) == 0, capi.last_error()
    held = L.gm_arena_bytes_in_use() - before
    assert np.array_equal(_got(w, n).j, np.arange(40) * (n // 40))
    assert held <= 5 << 20, f"{held} bytes for 40 entries"
