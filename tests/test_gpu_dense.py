"""Bitmap and full matrices and the products with a bitmap or full result
(saxbit, saxpy4, saxpy5) on the GPU against the oracle.

The oracle computes every product in CSR (its saxpy3 restatement, which sums
each entry's terms for k ascending and keeps the last writer for ANY, like
the dense-result kernel), and C += A*B as accum(C, A*B) (its accum_mask
restatement).  Bar: bit-exact for bool/integer semirings and ANY; plus_times
fp64 within 1e-12 relative per entry (both sum in k order, so it is
bit-exact in practice).
"""
import numpy as np
import pytest

import pyoracle as O
from graphblas_amd import capi
from graphblas_amd.workloads import Csr
from helpers import SR, assert_csr_equal, rand_csr

pytestmark = pytest.mark.gpu

FP_TOL = 1e-12
VT = {"GrB_PLUS_TIMES_SEMIRING_FP64": "fp64", "GrB_MIN_PLUS_SEMIRING_INT32": "int32",
      "GrB_PLUS_TIMES_SEMIRING_INT64": "int64", "GrB_MIN_PLUS_SEMIRING_INT64": "int64",
      "GrB_MAX_PLUS_SEMIRING_INT32": "int32", "GrB_MIN_PLUS_SEMIRING_FP64": "fp64"}
TN = {"fp64": "fp64", "int32": "int32", "int64": "int64", None: "bool"}
ZT = {"plus_pair_int64": "int64", "plus_pair_int32": "int32", "any_pair_bool": "bool",
      "plus_times_fp64": "fp64", "min_plus_int32": "int32", "any_secondi_int64": "int64",
      "plus_times_int64": "int64", "min_plus_int64": "int64", "max_plus_int32": "int32",
      "min_plus_fp64": "fp64"}


def _dense_of(A: Csr, dtype):
    """(values, present) of a host CSR."""
    x = np.zeros((A.nrows, A.ncols), dtype=dtype)
    b = np.zeros((A.nrows, A.ncols), dtype=bool)
    rows = np.repeat(np.arange(A.nrows), np.diff(A.p))
    b[rows, A.j] = True
    if A.x is not None:
        x[rows, A.j] = A.x
    else:
        x[rows, A.j] = 1
    return x, b


def _csr_of(x, b):
    rows, cols = np.nonzero(b)
    p = np.zeros(x.shape[0] + 1, dtype=np.int64)
    np.add.at(p, rows + 1, 1)
    p = np.cumsum(p)
    return Csr(x.shape[0], x.shape[1], p, cols.astype(np.int64), x[rows, cols].copy())


def _matrix(A: Csr, fmt: str, tname: str):
    """A GrB_Matrix holding A as 'sparse', 'bitmap' or 'full' (full: A is dense)."""
    if fmt == "sparse":
        return capi.Matrix.from_csr(A, tname)
    x, b = _dense_of(A, capi.NP_TYPES[tname])
    if fmt == "full":
        assert b.all()
        return capi.Matrix.from_dense(x, None, tname)
    return capi.Matrix.from_dense(x, b, tname)


def test_pack_unpack_and_conform(grb):
    rng = np.random.default_rng(5)
    A = rand_csr(70, 90, 0.2, rng, "fp64")
    x, b = _dense_of(A, np.float64)
    M = capi.Matrix.from_dense(x, b, "fp64")
    assert M.sparsity == capi.Matrix.BITMAP and M.nvals == A.nnz
    assert_csr_equal(M.to_csr(), A, what="bitmap -> CSR")
    gx, gb = M.to_dense()
    assert np.array_equal(gb, b) and np.array_equal(gx[b], x[b])
    # sparse only, then bitmap only, then full only (entries missing: stays bitmap)
    M.set_sparsity_control(capi.Matrix.SPARSE)
    assert M.sparsity == capi.Matrix.SPARSE
    assert_csr_equal(M.to_csr(), A, what="conform to sparse")
    M.set_sparsity_control(capi.Matrix.BITMAP)
    assert M.sparsity == capi.Matrix.BITMAP
    assert_csr_equal(M.to_csr(), A, what="conform to bitmap")
    M.set_sparsity_control(capi.Matrix.FULL)
    assert M.sparsity == capi.Matrix.BITMAP
    # a full matrix
    F = capi.Matrix.from_dense(x, None, "fp64")
    assert F.sparsity == capi.Matrix.FULL and F.nvals == 70 * 90
    fx, fb = F.to_dense()
    assert fb.all() and np.array_equal(fx, x)
    F.set_sparsity_control(capi.Matrix.SPARSE)
    assert F.sparsity == capi.Matrix.SPARSE and F.nvals == 70 * 90
    F.set_sparsity_control(capi.Matrix.FULL)
    assert F.sparsity == capi.Matrix.FULL
    assert np.array_equal(F.to_dense()[0], x)
    # reduce and dup of a bitmap matrix
    assert abs(capi.reduce_sum_fp64(M) - float(A.x.sum())) <= 1e-12 * max(1.0, abs(float(A.x.sum())))


CASES = [("sparse", "bitmap"), ("bitmap", "sparse"), ("full", "full"), ("bitmap", "bitmap"),
         ("sparse", "full")]


@pytest.mark.parametrize("handle", list(SR))
@pytest.mark.parametrize("fa,fb", CASES)
def test_saxbit_semirings(grb, handle, fa, fb):
    """C = A*B with a bitmap or full operand: C bitmap (saxbit)."""
    print(f"[dense] saxbit {handle} A {fa} B {fb}", flush=True)
    rng = np.random.default_rng(hash((handle, fa, fb)) % (2 ** 32))
    vt = VT.get(handle)
    name, _ = SR[handle]
    tn = TN[vt] if vt else ("bool" if "pair" in name or "secondi" in name else "int64")
    m, k, n = 120, 100, 2500          # two column tiles of C
    A = rand_csr(m, k, 1.0 if fa == "full" else 0.3, rng, vt)
    B = rand_csr(k, n, 1.0 if fb == "full" else (0.02 if fb == "sparse" else 0.3), rng, vt)
    Ad, Bd = _matrix(A, fa, tn), _matrix(B, fb, tn)
    C = capi.Matrix(ZT[name], m, n)
    capi.mxm_checked(C, None, handle, Ad, Bd)
    assert C.sparsity == capi.Matrix.BITMAP, "saxbit gives a bitmap C"
    ref = O.saxpy3(name, A, B)
    assert_csr_equal(C.to_csr(), ref, fp_tol=FP_TOL if "fp64" in name else None, what=handle)


@pytest.mark.parametrize("mask", ["bitmap", "bitmap_comp", "sparse_comp", "full_valued"])
@pytest.mark.parametrize("handle", ["GrB_PLUS_TIMES_SEMIRING_FP64", "GxB_PLUS_PAIR_INT64",
                                    "GxB_ANY_SECONDI_INT64", "GrB_MIN_PLUS_SEMIRING_INT32"])
def test_saxbit_masks(grb, handle, mask):
    print(f"[dense] saxbit mask {mask} {handle}", flush=True)
    rng = np.random.default_rng(hash((handle, mask)) % (2 ** 32))
    vt = VT.get(handle)
    name, _ = SR[handle]
    tn = TN[vt] if vt else "bool"
    m, k, n = 90, 60, 300
    A = rand_csr(m, k, 0.3, rng, vt)
    B = rand_csr(k, n, 0.3, rng, vt)
    Mk = rand_csr(m, n, 0.4, rng, "int32")
    comp = mask.endswith("comp")
    struct = mask in ("bitmap", "bitmap_comp", "sparse_comp")
    if mask == "full_valued":
        # a full mask whose zero values exclude their entries
        xm = rng.integers(0, 2, (m, n)).astype(np.int32)
        Md = capi.Matrix.from_dense(xm, None, "int32")
        Mref = _csr_of(xm, np.ones((m, n), dtype=bool))
    else:
        Mref = Mk
        Md = _matrix(Mk, "sparse" if mask.startswith("sparse") else "bitmap", "int32")
    Ad, Bd = capi.Matrix.from_csr(A, tn), _matrix(B, "bitmap", tn)
    C = capi.Matrix(ZT[name], m, n)
    desc = {(True, True): "RSC", (True, False): "RC", (False, True): "S", (False, False): None}[(comp, struct)]
    capi.mxm_checked(C, Md, handle, Ad, Bd, desc)
    ref = O.saxpy3(name, A, B, M=Mref, mask_comp=comp, mask_struct=struct)
    assert_csr_equal(C.to_csr(), ref, fp_tol=FP_TOL if "fp64" in name else None, what=mask)


@pytest.mark.parametrize("which", ["saxpy4", "saxpy5"])
@pytest.mark.parametrize("handle,accum", [("GrB_PLUS_TIMES_SEMIRING_FP64", "GrB_PLUS_FP64"),
                                          ("GrB_MIN_PLUS_SEMIRING_INT32", "GrB_MIN_INT32"),
                                          ("GrB_PLUS_TIMES_SEMIRING_INT64", "GrB_PLUS_INT64")])
def test_saxpy45_full_accumulate(grb, which, handle, accum):
    """C += A*B with C full and the monoid as accum: saxpy4 (A sparse, B full)
    and saxpy5 (A full, B sparse); C stays full and equals accum(C, A*B)."""
    print(f"[dense] {which} {handle}", flush=True)
    rng = np.random.default_rng(hash((which, handle)) % (2 ** 32))
    vt = VT[handle]
    name, _ = SR[handle]
    dt = capi.NP_TYPES[vt]
    m, k, n = 80, 70, 2200
    if which == "saxpy4":
        A = rand_csr(m, k, 0.1, rng, vt)
        B = rand_csr(k, n, 1.0, rng, vt)
        Ad, Bd = capi.Matrix.from_csr(A, vt), _matrix(B, "full", vt)
    else:
        A = rand_csr(m, k, 1.0, rng, vt)
        B = rand_csr(k, n, 0.05, rng, vt)
        Ad, Bd = _matrix(A, "full", vt), capi.Matrix.from_csr(B, vt)
    cx = (rng.random((m, n)) if vt == "fp64" else rng.integers(-50, 50, (m, n))).astype(dt)
    C = capi.Matrix.from_dense(cx, None, vt)
    capi.mxm_checked(C, None, handle, Ad, Bd, None, accum)
    assert C.sparsity == capi.Matrix.FULL, "C += A*B keeps C full"
    T = O.saxpy3(name, A, B)
    Cin = _csr_of(cx, np.ones((m, n), dtype=bool))
    op = {"GrB_PLUS_FP64": 1, "GrB_PLUS_INT64": 1, "GrB_MIN_INT32": 4}[accum]
    ref = O.accum_mask(Cin, None, T, op=op, dtype=dt)
    assert_csr_equal(C.to_csr(), ref, fp_tol=FP_TOL if vt == "fp64" else None, what=which)


def test_dense_operands_through_sparse_paths(grb):
    """A transposed bitmap operand and a sparse-enough case take the CSR form
    of the dense matrix (dot3 / saxpy3) and give the same result."""
    rng = np.random.default_rng(9)
    A = rand_csr(150, 120, 0.1, rng, "fp64")
    B = rand_csr(150, 200, 0.1, rng, "fp64")
    Ad = _matrix(A, "bitmap", "fp64")
    Bd = _matrix(B, "bitmap", "fp64")
    C = capi.Matrix("fp64", 120, 200)
    capi.mxm_checked(C, None, "GrB_PLUS_TIMES_SEMIRING_FP64", Ad, Bd, "T0")   # C = A'*B
    ref = O.saxpy3("plus_times_fp64", O.transpose(A), B)
    assert_csr_equal(C.to_csr(), ref, fp_tol=FP_TOL, what="A' * B bitmap")
    # {S} * {B} with few nonempty rows of A: C sparse (saxpy3 on B's CSR form)
    A2 = rand_csr(400, 150, 0.1, rng, "fp64", empty_rows=0.9)
    C2 = capi.Matrix("fp64", 400, 200)
    capi.mxm_checked(C2, None, "GrB_PLUS_TIMES_SEMIRING_FP64", capi.Matrix.from_csr(A2, "fp64"), Bd)
    assert C2.sparsity == capi.Matrix.SPARSE
    assert_csr_equal(C2.to_csr(), O.saxpy3("plus_times_fp64", A2, B), fp_tol=FP_TOL, what="S*B")
    # C's sparsity control applies to the result: bitmap result held sparse
    C3 = capi.Matrix("fp64", 150, 200)
    C3.set_sparsity_control(capi.Matrix.SPARSE)
    Ad2 = _matrix(rand_csr(150, 150, 0.3, rng, "fp64"), "bitmap", "fp64")
    capi.mxm_checked(C3, None, "GrB_PLUS_TIMES_SEMIRING_FP64", Ad2, Bd)
    assert C3.sparsity == capi.Matrix.SPARSE


def test_saxbit_cabi_errors(grb):
    L = capi.lib()
    out = capi.GmDenseOut()
    sr = capi.GmSemiring(1, 1, 11)
    # both forms of A given: invalid
    a = capi.GmCsr()
    d = capi.GmDense()
    import ctypes
    rc = L.gm_saxbit(ctypes.byref(out), None, None, False, True, ctypes.byref(a), ctypes.byref(d),
                     ctypes.byref(a), None, ctypes.byref(sr), None)
    assert rc == capi.GrB_INVALID_VALUE


@pytest.mark.parametrize("fa,fb", [("sparse", "full"), ("sparse", "bitmap"), ("bitmap", "full")])
@pytest.mark.parametrize("n", [1, 2, 3, 31, 32, 33, 64, 65, 130])
@pytest.mark.parametrize("handle", ["GrB_PLUS_TIMES_SEMIRING_FP64", "GrB_MIN_PLUS_SEMIRING_INT32",
                                    "GxB_ANY_SECONDI_INT64", "GxB_ANY_PAIR_BOOL"])
def test_saxbit_widths(grb, handle, n, fa, fb):
    """Few dense columns: every team width and its remainders, rows without
    entries, one entry, and more entries than a team reads at a time."""
    print(f"[dense] saxbit width {n} {handle} A {fa} B {fb}", flush=True)
    rng = np.random.default_rng(n + len(handle))
    vt = VT.get(handle)
    name, _ = SR[handle]
    tn = TN[vt] if vt else "bool"
    m, k = 77, 150
    A = rand_csr(m, k, 0.3, rng, vt, empty_rows=0.2)
    B = rand_csr(k, n, 1.0 if fb == "full" else 0.6, rng, vt)
    Ad, Bd = _matrix(A, fa, tn), _matrix(B, fb, tn)
    C = capi.Matrix(ZT[name], m, n)
    capi.mxm_checked(C, None, handle, Ad, Bd)
    ref = O.saxpy3(name, A, B)
    # terms are added for k ascending: the same bits as the oracle
    assert_csr_equal(C.to_csr(), ref, what=f"{handle} n={n}")


@pytest.mark.parametrize("n", [1, 5, 64, 100])
@pytest.mark.parametrize("handle", ["GrB_PLUS_TIMES_SEMIRING_FP64", "GrB_MIN_PLUS_SEMIRING_INT32"])
def test_saxbit_hub_rows(grb, handle, n):
    """Rows of A on both sides of the hub length and of a stage's end (8192
    products: 128 entries for 64 columns, 8192 for one)."""
    print(f"[dense] saxbit hubs {handle} n={n}", flush=True)
    rng = np.random.default_rng(n)
    vt = VT[handle]
    name, _ = SR[handle]
    k = 9000
    lens = [0, 511, 512, 513, 640, 641, 8192, 8193, 9000, 3]
    p = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    j = np.concatenate([np.sort(rng.choice(k, size=l, replace=False)) for l in lens]).astype(np.int64)
    x = rng.random(len(j)) if vt == "fp64" else rng.integers(-50, 50, len(j)).astype(np.int32)
    A = Csr(len(lens), k, p, j, x)
    for fb in ("full", "bitmap"):
        B = rand_csr(k, n, 1.0 if fb == "full" else 0.5, rng, vt)
        C = capi.Matrix(ZT[name], len(lens), n)
        capi.mxm_checked(C, None, handle, capi.Matrix.from_csr(A, vt), _matrix(B, fb, vt))
        assert_csr_equal(C.to_csr(), O.saxpy3(name, A, B), what=f"{handle} n={n} {fb}")


def test_saxbit_hub_row_past_32_bits(grb):
    """A hub row whose number needs 33 bits, with one bool column (34 GB of row
    pointers): it is computed, and no row that its low bits name."""
    import ctypes
    print("[dense] hub row 2^32", flush=True)
    L = capi.lib()
    m, nz = (1 << 32) + 1, 600
    p, j, x = L.gm_malloc(8 * (m + 1)), L.gm_malloc(8 * nz), L.gm_malloc(nz)
    out = capi.GmDenseOut()
    try:
        if not (p and j and x):
            pytest.skip("34 GB of device memory are not free")
        tail, cols, ones = np.array([0, nz], dtype=np.int64), np.arange(nz, dtype=np.int64), np.ones(nz, dtype=np.uint8)
        assert L.gm_memset(p, 0, 8 * (m + 1)) == 0
        assert L.gm_memcpy_h2d(p + 8 * (m - 1), tail.ctypes.data, 16) == 0
        assert L.gm_memcpy_h2d(j, cols.ctypes.data, cols.nbytes) == 0
        assert L.gm_memcpy_h2d(x, ones.ctypes.data, nz) == 0
        A, B = capi.GmCsr(), capi.GmDense(nz, 1, None, x, 0, 1)
        A.nrows, A.ncols, A.p, A.j, A.x, A.iso, A.type = m, nz, p, j, x, 1, 1
        sr = capi.GmSemiring(*SR["GxB_ANY_PAIR_BOOL"][1])
        rc = L.gm_saxbit(ctypes.byref(out), None, None, False, True, ctypes.byref(A), None, None,
                         ctypes.byref(B), ctypes.byref(sr), None)
        assert rc == 0, capi.last_error()
        got = np.zeros(2, dtype=np.int8)
        assert L.gm_memcpy_d2h(got[:1].ctypes.data, out.b, 1) == 0
        assert L.gm_memcpy_d2h(got[1:].ctypes.data, out.b + m - 1, 1) == 0
        assert out.nvals == 1 and got.tolist() == [0, 1]
    finally:
        for q in (p, j, x, out.b, out.x):
            if q:
                L.gm_free(q)
        L.gm_arena_trim()


@pytest.mark.parametrize("fa", ["sparse", "bitmap"])
def test_saxbit_few_long_rows_cost(grb, fa):
    """16 long rows of A spread over the device: at most four times one row's
    time (1.0 times as measured, 16 on one workgroup), and the same values."""
    import time
    rng = np.random.default_rng(3)
    k, n = (100000, 64) if fa == "sparse" else (20000, 64)
    x = rng.random(k)
    B = capi.Matrix.from_dense(rng.random((k, n)), None, "fp64")
    best, rows = {}, {}
    for m in (1, 16):
        if fa == "sparse":
            A = capi.Matrix.from_csr(Csr(m, k, np.arange(m + 1, dtype=np.int64) * k, np.tile(np.arange(k), m),
                                         np.tile(x, m)), "fp64")
        else:
            A = capi.Matrix.from_dense(np.tile(x, (m, 1)), np.ones((m, k), dtype=bool), "fp64")
        C, ts = capi.Matrix("fp64", m, n), []
        for _ in range(5):
            t = time.perf_counter()
            capi.mxm_checked(C, None, "GrB_PLUS_TIMES_SEMIRING_FP64", A, B)
            ts.append(time.perf_counter() - t)
        best[m], rows[m] = min(ts), C.to_dense()[0]
    assert np.array_equal(rows[16], np.tile(rows[1], (16, 1)))
    assert best[16] <= 4 * best[1], best


def _hub_csr(rng, k, lens, vt):
    p = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    j = np.concatenate([np.sort(rng.choice(k, size=l, replace=False)) for l in lens]).astype(np.int64)
    x = rng.random(len(j)) if vt == "fp64" else rng.integers(-50, 50, len(j)).astype(np.int32)
    return Csr(len(lens), k, p, j, x)


@pytest.mark.parametrize("mask", ["bitmap", "bitmap_comp", "sparse_comp", "valued"])
@pytest.mark.parametrize("n", [1, 5, 64, 130])
@pytest.mark.parametrize("fa", ["sparse", "bitmap"])
@pytest.mark.parametrize("handle", ["GrB_PLUS_TIMES_SEMIRING_FP64", "GxB_ANY_SECONDI_INT64"])
def test_saxbit_masked_rows(grb, handle, fa, n, mask):
    """Masks over a full B's columns: rows whose columns are all excluded, some
    or none, among short rows, empty rows and hub rows of A."""
    print(f"[dense] masked rows {handle} A {fa} n={n} {mask}", flush=True)
    rng = np.random.default_rng(n + len(mask))
    vt = VT.get(handle)
    name, _ = SR[handle]
    tn = TN[vt] if vt else "bool"
    k = 2000
    A = _hub_csr(rng, k, [0, 3, 513, 700, 1300, 40, 513, 90, 17, 1, 700], "fp64")
    if not vt:
        A.x = None
    B = rand_csr(k, n, 1.0, rng, vt)
    m = A.nrows
    xm = rng.integers(0, 2, (m, n)).astype(np.int32)
    bm = rng.random((m, n)) < 0.5
    for r in (2, 5, 9):                                  # all allowed / excluded: one way or the other
        xm[r], bm[r] = 1, True
    for r in (3, 7, 10):
        xm[r], bm[r] = 0, False
    comp, struct = mask.endswith("comp"), mask != "valued"
    Mref = _csr_of(xm if not struct else np.ones((m, n), dtype=np.int32), bm if struct else np.ones((m, n), dtype=bool))
    Md = capi.Matrix.from_csr(Mref, "int32") if mask.startswith("sparse") else \
        capi.Matrix.from_dense(xm if not struct else np.ones((m, n), dtype=np.int32), bm if struct else None, "int32")
    C = capi.Matrix(ZT[name], m, n)
    desc = {(True, True): "RSC", (False, True): "S", (False, False): None}[(comp, struct)]
    capi.mxm_checked(C, Md, handle, _matrix(A, fa, tn), _matrix(B, "full", tn), desc)
    assert_csr_equal(C.to_csr(), O.saxpy3(name, A, B, M=Mref, mask_comp=comp, mask_struct=struct), what=mask)


@pytest.mark.parametrize("n", [1, 64, 100])
@pytest.mark.parametrize("handle,accum", [("GrB_PLUS_TIMES_SEMIRING_FP64", "GrB_PLUS_FP64"),
                                          ("GrB_MIN_PLUS_SEMIRING_INT32", "GrB_MIN_INT32")])
def test_saxpy4_hub_rows(grb, handle, accum, n):
    """C += A*B, C and B full, with hub rows of A."""
    rng = np.random.default_rng(n)
    vt = VT[handle]
    name, _ = SR[handle]
    dt = capi.NP_TYPES[vt]
    A = _hub_csr(rng, 1500, [0, 513, 3, 1500, 512, 700], vt)
    B = rand_csr(1500, n, 1.0, rng, vt)
    cx = (rng.random((6, n)) if vt == "fp64" else rng.integers(-50, 50, (6, n))).astype(dt)
    C = capi.Matrix.from_dense(cx, None, vt)
    capi.mxm_checked(C, None, handle, capi.Matrix.from_csr(A, vt), _matrix(B, "full", vt), None, accum)
    ref = O.accum_mask(_csr_of(cx, np.ones((6, n), dtype=bool)), None, O.saxpy3(name, A, B),
                       op={"GrB_PLUS_FP64": 1, "GrB_MIN_INT32": 4}[accum], dtype=dt)
    assert_csr_equal(C.to_csr(), ref, fp_tol=FP_TOL if vt == "fp64" else None, what="saxpy4 hubs")


def test_saxbit_excluded_columns_cost(grb):
    """Columns that a bitmap mask excludes are not gathered: with none allowed,
    at most 0.6 of the unmasked product's time (0.2 as measured)."""
    import time
    rng = np.random.default_rng(4)
    m, n = 60000, 1000
    p = np.arange(m + 1, dtype=np.int64) * 30
    A = Csr(m, m, p, np.sort(rng.integers(0, m // 30, (m, 30)) + np.arange(30) * (m // 30), axis=1).ravel(), rng.random(30 * m))
    Ad = capi.Matrix.from_csr(A, "fp64")
    Bd = capi.Matrix.from_dense(rng.random((m, n)), None, "fp64")
    none = capi.Matrix.from_dense(np.ones((m, n), dtype=bool), np.zeros((m, n), dtype=bool), "bool")
    best = {}
    for what, M in (("all", None), ("none", none)):
        C, ts = capi.Matrix("fp64", m, n), []
        for _ in range(4):
            t = time.perf_counter()
            capi.mxm_checked(C, M, "GrB_PLUS_TIMES_SEMIRING_FP64", Ad, Bd, None if M is None else "RS")
            ts.append(time.perf_counter() - t)
        best[what] = min(ts)
        assert C.nvals == (m * n if M is None else 0)
    assert best["none"] <= 0.6 * best["all"], best


def test_saxbit_without_room_for_hub_list(grb):
    """The hub rows' list (the fourth allocation) forced not to fit: one of the
    size that A's entries allow takes its place."""
    import ctypes
    rng = np.random.default_rng(8)
    A = _hub_csr(rng, 1500, [0, 513, 3, 1500, 512, 700], "fp64")
    B = rand_csr(1500, 65, 1.0, rng, "fp64")
    L = capi.lib()
    dA, dB = capi.DeviceCsr(A, 11), L.gm_malloc(8 * 1500 * 65)
    x = np.ascontiguousarray(_dense_of(B, np.float64)[0])
    assert L.gm_memcpy_h2d(dB, x.ctypes.data, x.nbytes) == 0
    out, sr = capi.GmDenseOut(), capi.GmSemiring(*SR["GrB_PLUS_TIMES_SEMIRING_FP64"][1])
    bd = capi.GmDense(1500, 65, None, dB, 0, 11)
    L.gm_debug_fail_after(3)
    try:
        rc = L.gm_saxbit(ctypes.byref(out), None, None, False, True, ctypes.byref(dA.view), None, None,
                         ctypes.byref(bd), ctypes.byref(sr), None)
    finally:
        L.gm_debug_fail_after(-1)
    assert rc == 0, capi.last_error()
    got, b = np.zeros((6, 65)), np.zeros((6, 65), dtype=np.int8)
    assert L.gm_memcpy_d2h(got.ctypes.data, out.x, got.nbytes) == 0
    assert L.gm_memcpy_d2h(b.ctypes.data, out.b, b.nbytes) == 0
    assert_csr_equal(_csr_of(got, b != 0), O.saxpy3("plus_times_fp64", A, B), what="without a hub list")
    for q in (dB, out.x, out.b):
        L.gm_free(q)
    dA.free()
