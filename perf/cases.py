"""Workloads that the library's speed is measured on, each through its public
entry points: the C API (graphblas_amd.capi: GrB_mxv / GrB_vxm on vectors, the
request server) and the device C ABI of include/gm_kernels.h (gm_dot3,
gm_saxpy3, gm_saxbit, gm_batch_dot3), whose operands and results stay in HBM.

A case is a dict of plain values.  Its "kind" says what it stands for:

  tri      triangle count C<L> = L*U' (masked dot3, pattern semirings) on an
           RMAT graph: interactive sizes up to the RMAT scale 22 benchmark
  similar  scores of given pairs C<M> = A*B' (masked dot3 with values): sparse
           feature rows compared along the edges of a graph
  batch    many small graphs at once, C<A> = A*A' each (gm_batch_dot3), half
           plus_pair int32 and half min_plus int32
  er       C = A*B of Erdos-Renyi matrices (saxpy3, rows of similar length)
  square   C = A*A of an RMAT graph (saxpy3, rows of very uneven length)
  bfs      second level of many breadth-first searches, C<!V> = F*A with
           any_secondi int64 (saxpy3 with a complemented mask)
  sssp     hops of d min= d min.+ A from one source (GrB_vxm with an accumulator)
  power    steps of y = A*x (GrB_mxv), x starting full
  served   a burst of one-level BFS requests to the request server, results
           fetched to the host
  spmm     sparse matrix times full matrix of few columns, C = A*B (bitmap
           result) or C += A*B (full result)

Inputs are made on the GPU from the case and the seed: the case fixes a matrix
up to the order of its vertices, the seed shuffles the vertices (inside small
windows for an RMAT graph, which keeps its hubs together) and gives the values.
So every seed has other inputs and results of the same sizes.
"""
import ctypes

import numpy as np
import torch

from graphblas_amd import capi
from graphblas_amd import workloads as W

# semiring -> (add, multiply, type) codes, values' dtype (None: pattern only),
# result dtype
SEMIRINGS = {
    "plus_pair_int64": ((1, 3, 8), None, torch.int64),
    "plus_pair_int32": ((1, 3, 6), None, torch.int32),
    "any_pair_bool": ((4, 3, 1), None, torch.uint8),
    "any_secondi_int64": ((4, 4, 8), None, torch.int64),
    "plus_times_fp64": ((1, 1, 11), torch.float64, torch.float64),
    "plus_times_int64": ((1, 1, 8), torch.int64, torch.int64),
    "min_plus_int32": ((2, 2, 6), torch.int32, torch.int32),
    "min_plus_int64": ((2, 2, 8), torch.int64, torch.int64),
    "min_plus_fp64": ((2, 2, 11), torch.float64, torch.float64),
    "max_plus_int32": ((3, 2, 6), torch.int32, torch.int32),
}
GRB = {"plus_times_fp64": ("GrB_PLUS_TIMES_SEMIRING_FP64", "fp64"),
       "plus_times_int64": ("GrB_PLUS_TIMES_SEMIRING_INT64", "int64"),
       "min_plus_int32": ("GrB_MIN_PLUS_SEMIRING_INT32", "int32"),
       "min_plus_int64": ("GrB_MIN_PLUS_SEMIRING_INT64", "int64"),
       "min_plus_fp64": ("GrB_MIN_PLUS_SEMIRING_FP64", "fp64")}
TYPESTR = {torch.int64: "<i8", torch.int32: "<i4", torch.int8: "|i1", torch.uint8: "|u1",
           torch.float64: "<f8"}
GB_CODE = {torch.int64: 8, torch.int32: 6, torch.uint8: 1, torch.float64: 11}
DEV = "cuda"


def listed():
    return [
        # a small interactive graph: latency of one call, n not a power of two
        {"name": "tri small", "kind": "tri", "n": 1000, "ef": 16, "semiring": "plus_pair_int64"},
        # the scale-14 triangle count of the benchmark
        {"name": "tri scale 14", "kind": "tri", "n": 1 << 14, "ef": 16, "semiring": "plus_pair_int64"},
        # the benchmark's default: scale 22, hub rows of 100k and more entries
        {"name": "tri scale 22", "kind": "tri", "n": 1 << 22, "ef": 16, "semiring": "plus_pair_int64"},
        # similarity of sparse feature rows along a graph's edges, valued mask
        {"name": "similar", "kind": "similar", "n": 30011, "f": 4096, "row": 40, "deg": 24,
         "semiring": "plus_times_fp64", "valued_mask": True},
        # a sixteenth of the 4096-graph batch benchmark, the same size ranges
        {"name": "batch", "kind": "batch", "graphs": 256, "n_hi": 65536},
        # the Erdos-Renyi product of the benchmark
        {"name": "er scale 20", "kind": "er", "n": 1 << 20, "row": 8, "semiring": "plus_times_fp64"},
        # paths of length two in a power-law graph, ragged n
        {"name": "square", "kind": "square", "n": 40009, "ef": 8, "semiring": "plus_times_fp64"},
        # 64 searches at their second level on the served benchmark's graph
        {"name": "bfs level", "kind": "bfs", "n": 1 << 20, "ef": 16, "rows": 64},
        # shortest paths by hops from one source
        {"name": "sssp hops", "kind": "sssp", "n": 60013, "ef": 16, "steps": 4,
         "semiring": "min_plus_int32"},
        # power iteration / PageRank-like propagation
        {"name": "power steps", "kind": "power", "n": 1 << 16, "ef": 16, "steps": 3,
         "semiring": "plus_times_fp64"},
        # a burst of requests to a resident graph (the served benchmark's)
        {"name": "served burst", "kind": "served", "n": 1 << 20, "ef": 16, "requests": 64},
        # graph times a block of vectors (features, many right-hand sides)
        {"name": "spmm", "kind": "spmm", "n": 1 << 16, "ef": 16, "width": 64,
         "semiring": "plus_times_fp64", "accum": False},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["tri", "tri", "similar", "batch", "er", "square", "bfs", "sssp", "power",
                       "served", "spmm"])
    if kind == "tri":
        n = _log(rng, 256, 1 << 21)
        return {"kind": kind, "n": n, "ef": rng.randint(4, 32 if n < (1 << 20) else 16),
                "semiring": rng.choice(["plus_pair_int64", "plus_pair_int32", "any_pair_bool"])}
    if kind == "similar":
        return {"kind": kind, "n": _log(rng, 500, 60000), "f": _log(rng, 256, 16384),
                "row": rng.randint(8, 64), "deg": rng.randint(4, 32),
                "semiring": rng.choice(["plus_times_fp64", "plus_times_int64", "min_plus_int32",
                                        "max_plus_int32", "min_plus_fp64"]),
                "valued_mask": rng.random() < 0.5}
    if kind == "batch":
        return {"kind": kind, "graphs": _log(rng, 16, 256), "n_hi": _log(rng, 2048, 65536)}
    if kind == "er":
        return {"kind": kind, "n": _log(rng, 1024, 1 << 20), "row": rng.randint(2, 12),
                "semiring": rng.choice(["plus_times_fp64", "plus_times_int64", "min_plus_int64",
                                        "min_plus_int32", "any_pair_bool"])}
    if kind == "square":
        return {"kind": kind, "n": _log(rng, 512, 50000), "ef": rng.randint(4, 8),
                "semiring": rng.choice(["plus_times_fp64", "plus_times_int64", "min_plus_int32",
                                        "any_pair_bool", "plus_pair_int64"])}
    if kind == "bfs":
        return {"kind": kind, "n": _log(rng, 4096, 1 << 20), "ef": rng.randint(8, 16),
                "rows": _log(rng, 1, 128)}
    if kind == "sssp":
        return {"kind": kind, "n": _log(rng, 1024, 70000), "ef": rng.randint(8, 16),
                "steps": rng.randint(2, 5),
                "semiring": rng.choice(["min_plus_int32", "min_plus_int64", "min_plus_fp64"])}
    if kind == "power":
        return {"kind": kind, "n": _log(rng, 1024, 70000), "ef": rng.randint(8, 16),
                "steps": rng.randint(1, 4),
                "semiring": rng.choice(["plus_times_fp64", "plus_times_fp64", "plus_times_int64"])}
    if kind == "served":
        return {"kind": kind, "n": _log(rng, 1 << 14, 1 << 20), "ef": 16,
                "requests": _log(rng, 4, 128)}
    return {"kind": "spmm", "n": _log(rng, 1024, 1 << 17), "ef": rng.randint(4, 16),
            "width": _log(rng, 1, 128),
            "semiring": rng.choice(["plus_times_fp64", "plus_times_int64", "min_plus_int32"]),
            "accum": rng.random() < 0.5}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

class Operand:
    """A CSR matrix in torch tensors and its gm_csr view."""

    def __init__(self, nrows, ncols, p, j, x=None):
        self.nrows, self.ncols, self.p, self.j, self.x = nrows, ncols, p, j, x

    def view(self):
        return capi.GmCsr(self.nrows, self.ncols, self.p.data_ptr(), self.j.data_ptr(),
                          None if self.x is None else self.x.data_ptr(), 0,
                          1 if self.x is None else GB_CODE[self.x.dtype])

    def rows(self):
        return torch.repeat_interleave(torch.arange(self.nrows, device=DEV), torch.diff(self.p))

    def host(self):
        return W.Csr(self.nrows, self.ncols, self.p.cpu().numpy(), self.j.cpu().numpy(),
                     None if self.x is None else self.x.cpu().numpy())


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7fffffffffff)
    return g


def _from_keys(key, nrows, ncols):
    """CSR of sorted distinct row*ncols + column keys."""
    row = torch.div(key, ncols, rounding_mode="floor")
    p = torch.searchsorted(row, torch.arange(nrows + 1, device=DEV))
    return Operand(nrows, ncols, p, key - row * ncols)


def _rmat_keys(n, ef, g):
    """Symmetric, loop-free, deduplicated RMAT(0.57, 0.19, 0.19) on n vertices."""
    r = torch.zeros(n * ef, dtype=torch.int64, device=DEV)
    c = torch.zeros_like(r)
    for _ in range(max(1, (n - 1).bit_length())):
        u = torch.rand(n * ef, generator=g, device=DEV)
        r = 2 * r + (u >= 0.76)
        c = 2 * c + (((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
    keep = (r < n) & (c < n) & (r != c)
    r, c = r[keep], c[keep]
    return torch.unique(torch.cat([r * n + c, c * n + r]))


def _rmat(n, ef, g):
    return _from_keys(_rmat_keys(n, ef, g), n, n)


def _uniform(nrows, ncols, per_row, g):
    """per_row distinct uniform columns in every row."""
    per_row = min(per_row, ncols)
    j = torch.randint(ncols, (nrows, per_row), generator=g, device=DEV).sort(1).values
    while True:
        dup = (j[:, 1:] == j[:, :-1]).any(1).nonzero().flatten()
        if dup.numel() == 0:
            break
        j[dup] = torch.randint(ncols, (dup.numel(), per_row), generator=g, device=DEV).sort(1).values
    p = torch.arange(nrows + 1, device=DEV) * per_row
    return Operand(nrows, ncols, p, j.reshape(-1).contiguous())


def _values(n, dtype, g):
    if dtype is None:
        return None
    if dtype == torch.float64:
        return torch.rand(n, generator=g, device=DEV, dtype=dtype)
    return torch.randint(1, 101, (n,), generator=g, device=DEV).to(dtype)


def _shuffle(n, g, window=None):
    """A permutation of n that moves an index inside its window (default: anywhere)."""
    w = n if window is None else window
    at = torch.div(torch.arange(n, device=DEV), w, rounding_mode="floor")
    to = torch.empty(n, dtype=torch.int64, device=DEV)
    to[torch.argsort(at + torch.rand(n, generator=g, device=DEV, dtype=torch.float64))] = \
        torch.arange(n, device=DEV)
    return to


def _relabel(o, prow, pcol):
    """Row i becomes prow[i] and column j pcol[j]; values move along."""
    key, order = torch.sort(prow[o.rows()] * o.ncols + pcol[o.j])
    r = _from_keys(key, o.nrows, o.ncols)
    r.x = None if o.x is None else o.x[order]
    return r


WINDOW = 64                       # of an RMAT graph's vertex shuffle


def _graph(c, g):
    """The case's RMAT graph, shuffled: (graph, the shuffle, the graph before)."""
    base = _rmat(c["n"], c["ef"], _gen(1))
    to = _shuffle(c["n"], g, WINDOW)
    return _relabel(base, to, to), to, base


# ---------------------------------------------------------------------------
# results: tensors over the library's device arrays, released with them
# ---------------------------------------------------------------------------

class _Owned:
    def __init__(self, ptr, n, dtype):
        self.ptr = ptr
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": TYPESTR[dtype],
                                         "data": (ptr, False), "version": 3}

    def __del__(self):
        capi.lib().gm_free(self.ptr)


def _take(ptr, n, dtype):
    if not ptr:
        return torch.empty(0, dtype=dtype, device=DEV)
    if n == 0:
        capi.lib().gm_free(ptr)
        return torch.empty(0, dtype=dtype, device=DEV)
    return torch.as_tensor(_Owned(ptr, n, dtype), device=DEV)


def _csr(C, dtype):
    return (_take(C.p, C.nrows + 1, torch.int64), _take(C.j, C.nvals, torch.int64),
            _take(C.x, 1 if C.iso else C.nvals, dtype))


def _check(rc):
    if rc != 0:
        raise capi.GrBError(rc, capi.last_error())


class State:
    """What a program keeps between calls; close() releases library objects."""

    def __init__(self, case):
        self.case = case
        self.sr = capi.GmSemiring(*SEMIRINGS[case["semiring"]][0]) if "semiring" in case else None
        self.dtype = SEMIRINGS[case["semiring"]][2] if "semiring" in case else None
        self.aux = self.server = None

    def __del__(self):
        if self.aux:
            capi.lib().gm_csr_aux_free(self.aux)
        if self.server:
            self.server.close()


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------

def _prepare_tri(s, c, g):
    n = c["n"]
    base = _rmat(n, c["ef"], _gen(1))
    key = base.rows() * n + base.j
    low = base.j < base.rows()
    to = _shuffle(n, g, WINDOW)
    s.L, s.U = (_relabel(_from_keys(k, n, n), to, to) for k in (key[low], key[~low]))
    s.args = (s.L.view(), s.U.view())


def _prepare_similar(s, c, g):
    vt = SEMIRINGS[c["semiring"]][1]
    n, f, h = c["n"], c["f"], _gen(1)
    s.A, s.B, s.M = _uniform(n, f, c["row"], h), _uniform(n, f, c["row"], h), _uniform(n, n, c["deg"], h)
    if c["valued_mask"]:
        s.M.x = (torch.rand(s.M.j.numel(), generator=h, device=DEV) < 0.8).to(torch.uint8)
    pi, pj, pk = _shuffle(n, g), _shuffle(n, g), _shuffle(f, g)
    s.A, s.B, s.M = _relabel(s.A, pi, pk), _relabel(s.B, pj, pk), _relabel(s.M, pi, pj)
    s.A.x, s.B.x = (_values(o.j.numel(), vt, g) for o in (s.A, s.B))
    s.args = (s.M.view(), s.A.view(), s.B.view())


def _prepare_batch(s, c, g):
    k, lo, hi = c["graphs"], 512, c["n_hi"]
    s.graphs, s.groups = [], []
    for t in range(k):
        # sizes and edge factors spread evenly over their ranges
        u, v = (t * 0.6180339887498949) % 1.0, (t * 0.7548776662466927) % 1.0
        n = int(round(lo * (hi / lo) ** u))
        to = _shuffle(n, g, WINDOW)
        A = _relabel(_rmat(n, 4 + int(29 * v), _gen(1 + t)), to, to)
        A.x = _values(A.j.numel(), torch.int32, g)
        s.graphs.append(A)
    for q, name in enumerate(("plus_pair_int32", "min_plus_int32")):
        views = [A.view() for A in s.graphs[q::2]]
        reqs = (capi.GmDot3Request * max(len(views), 1))()
        for t, v in enumerate(views):
            reqs[t] = capi.GmDot3Request(v, v, v)
        base = np.zeros((2, len(views) + 1), dtype=np.int64)
        s.groups.append((reqs, len(views), base, capi.GmSemiring(*SEMIRINGS[name][0])))


def _prepare_spgemm(s, c, g):
    vt = SEMIRINGS[c["semiring"]][1]
    n, h = c["n"], _gen(1)
    if c["kind"] == "er":
        pi, pk, pj = (_shuffle(n, g) for _ in range(3))
        s.A, s.B = (_uniform(n, n, c["row"], h) for _ in range(2))
        s.A, s.B = _relabel(s.A, pi, pk), _relabel(s.B, pk, pj)
        s.A.x, s.B.x = (_values(o.j.numel(), vt, g) for o in (s.A, s.B))
    else:
        s.A, _, _ = _graph(c, g)
        s.A.x = _values(s.A.j.numel(), vt, g)
        s.B = s.A
    a, b = s.A.view(), s.B.view()
    # B's derived forms, kept with B while it does not change
    aux = ctypes.c_void_p()
    torch.cuda.synchronize()
    _check(capi.lib().gm_csr_aux_build(ctypes.byref(aux), ctypes.byref(b)))
    s.aux = aux.value
    b.aux = s.aux
    s.args = (a, b)


def _prepare_bfs(s, c, g):
    n, k, h = c["n"], c["rows"], _gen(2)
    s.A, to, base = _graph(c, g)
    deg = torch.diff(base.p)
    live = deg.nonzero().flatten()
    src = live[torch.randint(live.numel(), (k,), generator=h, device=DEV)]
    # frontier: the sources' neighbours; visited: frontier and source
    at = torch.repeat_interleave(torch.arange(k, device=DEV), deg[src])
    off = torch.arange(at.numel(), device=DEV) - (torch.cumsum(deg[src], 0) - deg[src])[at]
    fkey = at * n + to[base.j[base.p[src][at] + off]]
    vkey = torch.cat([fkey, torch.arange(k, device=DEV) * n + to[src]])
    s.F, s.V = (_from_keys(torch.sort(x).values, k, n) for x in (fkey, vkey))
    s.sr, s.dtype = capi.GmSemiring(*SEMIRINGS["any_secondi_int64"][0]), torch.int64
    s.args = (s.V.view(), s.F.view(), s.A.view())


def _prepare_vector(s, c, g):
    A, to, base = _graph(c, g)
    vt = SEMIRINGS[c["semiring"]][1]
    A.x = _values(A.j.numel(), vt, g)
    name = GRB[c["semiring"]][1]
    if c["kind"] == "power":
        if vt == torch.float64:
            A.x = A.x * 2.0 / torch.diff(A.p).to(vt).clamp(min=1)[A.rows()]
        s.x0 = _values(c["n"], vt, g)
        s.x = capi.Vector.from_arrays(np.arange(c["n"]), s.x0.cpu().numpy(), name, c["n"])
        s.y = [capi.Vector(name, c["n"]) for _ in range(2)]
    else:
        s.source = int(to[base.j[base.j.numel() // 3]])
    s.T = A
    s.A = capi.Matrix.from_csr(A.host(), name)


def _prepare_served(s, c, g):
    s.A, to, _ = _graph(c, g)
    to, rng = to.cpu().numpy(), np.random.default_rng(1)
    s.reqs = []
    for r in range(c["requests"]):
        # sizes log-uniform in [1, 256]
        k = int(round(256 ** ((r * 0.6180339887498949 + 0.5) % 1.0)))
        s.reqs.append(np.sort(to[rng.choice(c["n"], size=k, replace=False)]).astype(np.int64))
    torch.cuda.synchronize()
    s.server = capi.Server(s.A.view(), SEMIRINGS["any_secondi_int64"][0], workers=2,
                           max_batch_reqs=256, flop_budget=1 << 22)


def _prepare_spmm(s, c, g):
    vt = SEMIRINGS[c["semiring"]][1]
    s.A, _, _ = _graph(c, g)
    s.A.x = _values(s.A.j.numel(), vt, g)
    s.B = _values(c["n"] * c["width"], vt, g)
    s.C = _values(c["n"] * c["width"], vt, g) if c["accum"] else None

    def full(x):
        return capi.GmDense(c["n"], c["width"], None, x.data_ptr(), 0, GB_CODE[x.dtype])
    s.args = (s.A.view(), full(s.B), full(s.C) if c["accum"] else None)


def prepare(case, seed):
    capi.init()
    s, g, kind = State(case), _gen(seed), case["kind"]
    if kind == "tri":
        _prepare_tri(s, case, g)
    elif kind == "similar":
        _prepare_similar(s, case, g)
    elif kind == "batch":
        _prepare_batch(s, case, g)
    elif kind in ("er", "square"):
        _prepare_spgemm(s, case, g)
    elif kind == "bfs":
        _prepare_bfs(s, case, g)
    elif kind in ("sssp", "power"):
        _prepare_vector(s, case, g)
    elif kind == "served":
        _prepare_served(s, case, g)
    else:
        _prepare_spmm(s, case, g)
    torch.cuda.synchronize()      # the library's stream reads the inputs next
    return s


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------

_ref = ctypes.byref


def _run_batch(s):
    out = []
    for reqs, k, base, sr in s.groups:
        if k == 0:
            continue
        C = capi.GmCsrOut()
        _check(capi.lib().gm_batch_dot3(_ref(C), base[0].ctypes.data, base[1].ctypes.data, reqs, k,
                                        True, _ref(sr), None))
        out += _csr(C, torch.int32)
    return out


def _run_sssp(s):
    c = s.case
    sr, t = GRB[c["semiring"]]
    d = capi.Vector.from_arrays([s.source], [0], t, c["n"])
    for _ in range(c["steps"]):
        _check(capi.vxm(d, None, sr, d, s.A, accum="GrB_MIN_" + t.upper()))
    return d.to_arrays()


def _run_power(s):
    x = s.x
    for t in range(s.case["steps"]):
        y = s.y[t & 1]
        _check(capi.mxv(y, None, GRB[s.case["semiring"]][0], s.A, x))
        x = y
    return x.to_arrays()


def _run_served(s):
    ids = [s.server.submit(r) for r in s.reqs]
    rows = []
    for i in ids:
        rows.append(s.server.fetch(i, s.server.wait(i)))
        s.server.release(i)
    return [np.concatenate([r[t] for r in rows]) for t in range(3)]


def run(state):
    s, L = state, capi.lib()
    kind = s.case["kind"]
    if kind == "batch":
        return _run_batch(s)
    if kind == "sssp":
        return _run_sssp(s)
    if kind == "power":
        return _run_power(s)
    if kind == "served":
        return _run_served(s)
    if kind == "spmm":
        a, b, cin = s.args
        D = capi.GmDenseOut()
        _check(L.gm_saxbit(_ref(D), None, None, False, False, _ref(a), None, None, _ref(b), _ref(s.sr),
                           _ref(cin) if cin is not None else None))
        return _take(D.b, D.nrows * D.ncols, torch.int8), _take(D.x, D.nrows * D.ncols, s.dtype)
    C = capi.GmCsrOut()
    if kind == "tri":
        l, u = s.args
        _check(L.gm_dot3(_ref(C), _ref(l), True, _ref(l), _ref(u), _ref(s.sr), None))
    elif kind == "similar":
        m, a, b = s.args
        _check(L.gm_dot3(_ref(C), _ref(m), not s.case["valued_mask"], _ref(a), _ref(b), _ref(s.sr), None))
    elif kind == "bfs":
        v, f, a = s.args
        _check(L.gm_saxpy3(_ref(C), _ref(v), True, True, _ref(f), _ref(a), _ref(s.sr), None))
    else:
        a, b = s.args
        _check(L.gm_saxpy3(_ref(C), None, False, False, _ref(a), _ref(b), _ref(s.sr), None))
    return _csr(C, s.dtype)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and the exact results
# ---------------------------------------------------------------------------

def work(case):
    """Inputs read once, outputs written once (8-byte indices); multiplies and
    additions by the expected number of matching pairs.  The RMAT figures are
    estimates from these generators (deduplication leaves about 0.96 of the
    edges at these sizes)."""
    c, kind = case, case["kind"]
    n = c.get("n", 0)
    vt = SEMIRINGS[c["semiring"]][1] if "semiring" in c else None
    vs = 0 if vt is None else torch.tensor([], dtype=vt).element_size()
    zs = torch.tensor([], dtype=SEMIRINGS[c["semiring"]][2]).element_size() if "semiring" in c else 8
    nnz = 2 * 0.96 * n * c.get("ef", 0)
    if kind == "tri":
        return {"bytes": 24.0 * (n + 1) + 8 * nnz + (8 + zs) * 0.33 * nnz, "flops": 2 * 16 * nnz}
    if kind == "similar":
        mnz, anz, hits = n * c["deg"], n * c["row"], n * c["deg"] * c["row"] ** 2 / c["f"]
        return {"bytes": 32.0 * (n + 1) + 9 * mnz + 2 * (8 + vs) * anz + (8 + zs) * min(mnz, hits),
                "flops": 2.0 * hits}
    if kind == "batch":
        nnz = sum(2 * 0.8 * 512 * (c["n_hi"] / 512) ** ((t + 0.5) / c["graphs"]) * 18
                  for t in range(c["graphs"]))
        return {"bytes": (8 + 2 + 12) * nnz, "flops": 2 * 16 * nnz}
    if kind == "er":
        nnz, fl = n * c["row"], n * c["row"] ** 2
        return {"bytes": 24.0 * (n + 1) + 2 * (8 + vs) * nnz + (8 + zs) * fl, "flops": 2.0 * fl}
    if kind == "square":
        return {"bytes": 16.0 * (n + 1) + (8 + vs) * nnz + (8 + zs) * 40 * nnz, "flops": 2 * 120 * nnz}
    if kind == "bfs":
        rows = 30000.0 * c["rows"] * n / (1 << 20)
        return {"bytes": 8.0 * n + 16 * rows + 8 * 2 * rows, "flops": 2 * rows}
    if kind in ("sssp", "power"):
        return {"bytes": c["steps"] * ((8.0 + vs) * nnz + 24 * n), "flops": 2 * c["steps"] * nnz}
    if kind == "served":
        ks = 46.0 * c["requests"]
        return {"bytes": ks * (8 * 2 * c["ef"] + 16 * 2 * c["ef"] + 40), "flops": ks * 2 * c["ef"]}
    w = c["width"]
    return {"bytes": 8.0 * n + (8 + vs) * nnz + n * w * (vs + zs + (zs if c["accum"] else 1)),
            "flops": 2 * nnz * w}


def _exact_spgemm(A, B):
    ln = torch.diff(B.p)[A.j]
    e = torch.repeat_interleave(torch.arange(A.j.numel(), device=DEV), ln)
    q = B.p[A.j][e] + torch.arange(e.numel(), device=DEV) - (torch.cumsum(ln, 0) - ln)[e]
    key, at = torch.unique(A.rows()[e] * B.ncols + B.j[q], return_inverse=True)
    return torch.zeros(key.numel(), dtype=torch.float64, device=DEV).index_add_(0, at, A.x[e] * B.x[q])


def exact(case, seed):
    if case.get("semiring") != "plus_times_fp64":
        return None               # integers, or sums of two numbers: one rounding
    s = prepare(case, seed)
    kind, n = case["kind"], case["n"]
    if kind in ("er", "square"):
        return None, None, _exact_spgemm(s.A, s.B)
    if kind == "similar":
        dense = [torch.zeros((n, case["f"]), dtype=torch.float64, device=DEV) for _ in range(2)]
        for o, d in zip((s.A, s.B), dense):
            d[o.rows(), o.j] = o.x
        rows, out = s.M.rows(), []
        for t in range(0, rows.numel(), 8192):
            i, j = rows[t:t + 8192], s.M.j[t:t + 8192]
            a, b = dense[0][i], dense[1][j]
            hit = ((a != 0) & (b != 0)).any(1)
            if s.M.x is not None:
                hit &= s.M.x[t:t + 8192] != 0
            out.append((a * b).sum(1)[hit])
        return None, None, torch.cat(out)
    if kind == "power":
        A, rows = s.T, s.T.rows()
        x, has = s.x0, torch.ones(n, dtype=torch.bool, device=DEV)
        for _ in range(case["steps"]):
            live = has[A.j]
            y = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, rows[live], A.x[live] * x[A.j[live]])
            has = torch.zeros(n, dtype=torch.bool, device=DEV)
            has[rows[live]] = True
            x = y
        return None, x[has]
    B = s.B.view(n, case["width"])
    C = s.C.view(n, case["width"]).clone() if case["accum"] else torch.zeros_like(B)
    rows = s.A.rows()
    for t in range(0, rows.numel(), 1 << 20):
        k = slice(t, t + (1 << 20))
        C.index_add_(0, rows[k], s.A.x[k, None] * B[s.A.j[k]])
    return (C.reshape(-1),) if case["accum"] else (None, C.reshape(-1))
