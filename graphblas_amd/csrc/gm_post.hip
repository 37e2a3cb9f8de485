// gm_post.hip: the steps around the product kernels that GrB_mxm needs for
// its full contract, kept on the device:
//
//   gm_transpose    CSR of A' from the CSR of A (the reference's
//                   GB_transpose, Source/transpose/GB_transpose.c, used when
//                   the orientation rules of GB_AxB_meta.c:683-694,718-723
//                   leave an explicit transpose).  Entries are keyed
//                   (column << 32 | row) and stably radix-sorted (rocPRIM)
//                   on the column bits with their positions: the entries
//                   enter in row order, so the rows of A' come out sorted; row
//                   pointers by binary search of each row's first key, then
//                   a gather of the values.
//   gm_accum_mask   C<M, replace> = accum (C, T): the reference's
//                   GB_accum_mask (Source/mask/GB_accum_mask.c) for sparse
//                   C, M and T of one type.  Work is per entry of C and of
//                   T, never per row: an entry finds its place in the other
//                   operand's row and in the mask row by binary search.

#include <cstring>
#include <rocprim/device/device_radix_sort.hpp>
#include "gm_internal.h"
#include "gm_block.h"

namespace gm
{

static inline unsigned post_grid(int64_t n, int nt, int64_t cap)
{
    int64_t g = (n + nt - 1) / nt;
    if (g > cap) g = cap;
    return (unsigned) (g > 0 ? g : 1);
}

__global__ void k_post_zero(int64_t *x, int64_t n)
{
    const int64_t stride = (int64_t) gridDim.x * blockDim.x;
    for (int64_t t = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; t < n; t += stride) x[t] = 0;
}

//------------------------------------------------------------------------------
// transpose
//------------------------------------------------------------------------------

// key of entry p: (column << 32) | row; pos[p] = p.  A workgroup takes
// TR_TILE consecutive entries: the rows holding its first and last entry are
// found once, and each entry searches only between them.
constexpr int TR_TILE = 256 * 16;

__device__ __forceinline__ int64_t tr_row_of(const int64_t *__restrict__ Ap, int64_t lo, int64_t hi, int64_t p)
{
    // last i in [lo, hi] with Ap[i] <= p
    while (lo < hi)
    {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (Ap[mid] <= p) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__global__ void k_tr_keys(const int64_t *__restrict__ Ap, const int64_t *__restrict__ Aj, int64_t m,
                          int64_t nnz, uint64_t *__restrict__ keys, int64_t *__restrict__ pos)
{
    __shared__ int64_t s_r[2];
    for (int64_t t0 = (int64_t) blockIdx.x * TR_TILE; t0 < nnz; t0 += (int64_t) gridDim.x * TR_TILE)
    {
        const int64_t t1 = (t0 + TR_TILE < nnz) ? t0 + TR_TILE : nnz;
        if (threadIdx.x < 2) s_r[threadIdx.x] = tr_row_of(Ap, 0, m - 1, threadIdx.x == 0 ? t0 : t1 - 1);
        __syncthreads();
        const int64_t r0 = s_r[0], r1 = s_r[1];
        __syncthreads();
        for (int64_t p = t0 + threadIdx.x; p < t1; p += blockDim.x)
        {
            const int64_t i = tr_row_of(Ap, r0, r1, p);
            keys[p] = ((uint64_t) Aj[p] << 32) | (uint64_t) i;
            pos[p] = p;
        }
    }
}

__device__ __forceinline__ int64_t lb_u64(const uint64_t *a, int64_t n, uint64_t v)
{
    int64_t lo = 0, hi = n;
    while (lo < hi)
    {
        const int64_t mid = (lo + hi) >> 1;
        if (a[mid] < v) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// T.p[r] = first sorted key of column r; T.j = row; T.x = A.x[pos]
__global__ void k_tr_rows(const uint64_t *__restrict__ keys, int64_t nnz, int64_t n,
                          int64_t *__restrict__ Tp)
{
    const int64_t stride = (int64_t) gridDim.x * blockDim.x;
    for (int64_t r = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; r <= n; r += stride)
        Tp[r] = (r == n) ? nnz : lb_u64(keys, nnz, (uint64_t) r << 32);
}

__global__ void k_tr_fill(const uint64_t *__restrict__ keys, const int64_t *__restrict__ pos,
                          int64_t nnz, const uint8_t *__restrict__ Ax, int32_t xsize,
                          int64_t *__restrict__ Tj, uint8_t *__restrict__ Tx)
{
    const int64_t stride = (int64_t) gridDim.x * blockDim.x;
    for (int64_t q = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; q < nnz; q += stride)
    {
        Tj[q] = (int64_t) (keys[q] & 0xffffffffull);
        if (Tx)
        {
            const int64_t p = pos[q];
            for (int b = 0; b < xsize; b++) Tx[q * xsize + b] = Ax[p * xsize + b];
        }
    }
}

//------------------------------------------------------------------------------
// accum + mask
//------------------------------------------------------------------------------

template <class Z>
__device__ __forceinline__ Z accum_apply(int op, Z c, Z t)
{
    if constexpr (std::is_same<Z, double>::value)
    {
        switch (op)
        {
            case 1: return __dadd_rn(c, t);
            case 2: return __dsub_rn(c, t);
            case 3: return __dmul_rn(c, t);
            case 4: return fmin(c, t);
            case 5: return fmax(c, t);
            case 6: return c;
            case 9: return 1.0;
            case 10: return (c != 0.0 || t != 0.0) ? 1.0 : 0.0;
            case 11: return (c != 0.0 && t != 0.0) ? 1.0 : 0.0;
            default: return t;          // SECOND, ANY
        }
    }
    else if constexpr (std::is_same<Z, uint8_t>::value)
    {
        // bool: PLUS and MAX and LOR are "or"; TIMES, MIN and LAND are "and";
        // MINUS is "xor" (GrB's bool arithmetic)
        const bool a = c != 0, b = t != 0;
        switch (op)
        {
            case 1: case 5: case 10: return (uint8_t) (a || b);
            case 2: return (uint8_t) (a != b);
            case 3: case 4: case 11: return (uint8_t) (a && b);
            case 6: return (uint8_t) a;
            case 9: return 1;
            default: return (uint8_t) b;
        }
    }
    else
    {
        using U = typename std::make_unsigned<Z>::type;   // wrap-around arithmetic
        switch (op)
        {
            case 1: return (Z) ((U) c + (U) t);
            case 2: return (Z) ((U) c - (U) t);
            case 3: return (Z) ((U) c * (U) t);
            case 4: return c < t ? c : t;
            case 5: return c > t ? c : t;
            case 6: return c;
            case 9: return 1;
            case 10: return (Z) ((c != 0) || (t != 0));
            case 11: return (Z) ((c != 0) && (t != 0));
            default: return t;
        }
    }
}

struct AccArgs
{
    int64_t m, nc, nt;
    const int64_t *Cp, *Cj; const void *Cx; int32_t c_iso;
    const int64_t *Tp, *Tj; const void *Tx; int32_t t_iso;
    const int64_t *Mp, *Mj; const void *Mx; int32_t m_iso, msize;
    int32_t has_mask, mask_comp, mask_struct, replace, op;
    int64_t ntc, ntt;     // tiles of C's and T's entries (one entry past the end included)
    uint64_t *bits;       // LEAN: a bit per entry (C's tiles, then T's), set for an output entry
    uint32_t *rank;       // per entry (the same order): output entries before it in its tile
    uint8_t *state;       // per entry: AC_*
    int64_t *other;       // per entry: its place in the other operand
    int64_t *toff;        // ntc + ntt + 1: output entries before each tile
    int64_t *Op;
    int64_t *Oj;
    void *Ox;
};

// what becomes of an entry: nothing, its own value, both values through the
// accumulator, the other operand's value.  An index that C and T share is
// put out by C's entry alone.
enum { AC_NONE = 0, AC_OWN = 1, AC_BOTH = 2, AC_OTHER = 3 };

// One tile per workgroup: the fate of AC_NT * IPT entries of C or of T and their
// ranks among the tile's output entries.  A row may hold all the entries (a
// vector is one row), so the unit is the entry: the rows of a tile's ends are
// searched once, each entry searches only between them.  Bound by the searches'
// dependent reads.  C and T of 2^20 rows with 8 entries each, int64, PLUS: 1043
// us with a thread per row walking it twice, 685 us here; four hops of a
// shortest-path vector that grows to 44000 entries (one row): 66 ms and 1.1
// ms with their products.
// IPT is AC_IPT, or 1 for a merge of at most AC_FEW such tiles, which would leave
// most CUs idle: a thread's eight searches follow one another.
// LEAN, for merges whose 13 bytes of state an entry do not fit: a bit an entry
// is kept, and the writing pass searches again.
constexpr int AC_NT = 256;
constexpr int AC_IPT = 8;
constexpr int AC_FEW = 4 * AC_NT;

// what becomes of entry e of C (of T), in row i; y: its place in the other operand
__device__ __forceinline__ int ac_fate(const AccArgs &g, bool isC, int64_t i, int64_t e, int64_t &y)
{
    const int64_t *Yp = isC ? g.Tp : g.Cp, *Yj = isC ? g.Tj : g.Cj;
    const int64_t j = isC ? g.Cj[e] : g.Tj[e];
    bool both = false;
    y = 0;
    if (Yp)
    {
        const int64_t y1 = Yp[i + 1];
        y = lower_bound(Yj, Yp[i], y1, j);
        both = y < y1 && Yj[y] == j;
    }
    bool allow = true;
    if (g.has_mask)
    {
        const int64_t m1 = g.Mp[i + 1], q = lower_bound(g.Mj, g.Mp[i], m1, j);
        const bool in = q < m1 && g.Mj[q] == j && (g.mask_struct || mask_true(g.Mx, q, g.msize, g.m_iso));
        allow = g.mask_comp ? !in : in;
    }
    if (!isC) return (allow && !both) ? AC_OWN : AC_NONE;
    if (!allow) return g.replace ? AC_NONE : AC_OWN;
    if (g.op) return both ? AC_BOTH : AC_OWN;
    return both ? AC_OTHER : AC_NONE;
}

template <bool LEAN, int IPT>
__global__ __launch_bounds__(AC_NT) void k_accum_state(AccArgs g)
{
    constexpr int NW = AC_NT / 64, TILE = AC_NT * IPT;
    __shared__ int64_t s_r[2];
    __shared__ int s_cnt[IPT * NW];
    const bool isC = (int64_t) blockIdx.x < g.ntc;
    const int64_t t0 = ((int64_t) blockIdx.x - (isC ? 0 : g.ntc)) * TILE;
    const int64_t n = isC ? g.nc : g.nt;
    const int64_t *Xp = isC ? g.Cp : g.Tp;
    const int64_t t1 = t0 + TILE < n ? t0 + TILE : n;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const size_t slot = (size_t) blockIdx.x * TILE;
    if (threadIdx.x < 2 && t0 < t1) s_r[threadIdx.x] = tr_row_of(Xp, 0, g.m - 1, threadIdx.x == 0 ? t0 : t1 - 1);
    __syncthreads();
    unsigned long long bal[IPT];
    #pragma unroll
    for (int t = 0; t < IPT; t++)
    {
        const int64_t e = t0 + t * AC_NT + threadIdx.x;
        int st = AC_NONE;
        int64_t y = 0;
        if (e < t1)
        {
            const int64_t i = tr_row_of(Xp, s_r[0], s_r[1], e);
            st = ac_fate(g, isC, i, e, y);
        }
        if (!LEAN && e <= n)
        {
            g.state[slot + t * AC_NT + threadIdx.x] = (uint8_t) st;
            g.other[slot + t * AC_NT + threadIdx.x] = y;
        }
        bal[t] = __ballot(st != AC_NONE);
        if (lane == 0) s_cnt[t * NW + wv] = __popcll(bal[t]);
        if (LEAN && lane == 0) g.bits[(slot >> 6) + t * NW + wv] = bal[t];
    }
    __syncthreads();
    int run = 0, total = 0;
    for (int q = 0; q < IPT * NW; q++)
    {
        if (q < wv) run += s_cnt[q];
        total += s_cnt[q];
    }
    #pragma unroll
    for (int t = 0; t < IPT && !LEAN; t++)
    {
        if (t0 + t * AC_NT + threadIdx.x <= n)
            g.rank[slot + t * AC_NT + threadIdx.x] = (uint32_t) (run + __popcll(bal[t] & ((1ull << lane) - 1ull)));
        for (int q = 0; q < NW; q++)
            if (t * NW + wv + q < IPT * NW) run += s_cnt[t * NW + wv + q];
    }
    if (threadIdx.x == 0) g.toff[blockIdx.x] = total;
}

// output entries in slot s's tile before s
template <bool LEAN, int IPT>
__device__ __forceinline__ int64_t ac_rank(const AccArgs &g, int64_t s)
{
    if constexpr (!LEAN) return (int64_t) g.rank[s];
    int64_t r = 0;
    for (int64_t w = s / (AC_NT * IPT) * ((AC_NT * IPT) / 64); w < s >> 6; w++) r += __popcll(g.bits[w]);
    return r + __popcll(g.bits[s >> 6] & ((1ull << (s & 63)) - 1ull));
}

// output entries of C (T) before its entry p, p up to the entry count
template <bool LEAN, int IPT>
__device__ __forceinline__ int64_t ac_before_c(const AccArgs &g, const int64_t *toff, int64_t p)
{
    return toff[p / (AC_NT * IPT)] + ac_rank<LEAN, IPT>(g, p);
}
template <bool LEAN, int IPT>
__device__ __forceinline__ int64_t ac_before_t(const AccArgs &g, const int64_t *toff, int64_t p)
{
    return toff[g.ntc + p / (AC_NT * IPT)] - toff[g.ntc] + ac_rank<LEAN, IPT>(g, g.ntc * (AC_NT * IPT) + p);
}

// the fate of entry p of C (of T) as k_accum_state found it
template <bool LEAN, int IPT>
__device__ __forceinline__ int ac_again(const AccArgs &g, bool isC, int64_t p, int64_t &y)
{
    const int64_t s = isC ? p : g.ntc * (AC_NT * IPT) + p;
    if constexpr (!LEAN)
    {
        y = g.other[s];
        return g.state[s];
    }
    if (!((g.bits[s >> 6] >> (s & 63)) & 1ull)) return AC_NONE;
    return ac_fate(g, isC, tr_row_of(isC ? g.Cp : g.Tp, 0, g.m - 1, p), p, y);
}

// Every output entry to its place: the entries of both operands before it.
// IPT = 1: toff holds the tiles' counts, which every workgroup scans for itself,
// as a scan's launch costs a small merge more.  The total is left in host[0].
// 1000 rows of 8 entries in C and T, sizes unknown: 56.9 us with a thread a row
// counting and filling, 68.9 with large tiles, a scan and the sizes and the
// total copied, 50.5 here.
template <class Z, bool LEAN, int IPT>
__global__ __launch_bounds__(AC_NT) void k_accum_write(AccArgs g, int64_t *host)
{
    constexpr bool FEW = IPT == 1;
    constexpr int PER = AC_FEW / AC_NT;
    __shared__ int64_t s_toff[FEW ? AC_FEW + 1 : 1], s_scan[AC_NT / 64 + 1];
    const int64_t tiles = g.ntc + g.ntt;
    const int64_t *toff = g.toff;
    if constexpr (FEW)
    {
        int64_t c[PER], sum = 0, total;
        #pragma unroll
        for (int u = 0; u < PER; u++)
        {
            const int t = (int) threadIdx.x * PER + u;
            c[u] = t < tiles ? g.toff[t] : 0;
            sum += c[u];
        }
        int64_t run = block_exclusive_scan<int64_t, AC_NT>(sum, s_scan, &total);
        #pragma unroll
        for (int u = 0; u < PER; u++)
        {
            s_toff[(int) threadIdx.x * PER + u] = run;
            run += c[u];
        }
        if (threadIdx.x == 0) s_toff[AC_FEW] = total;
        __syncthreads();
        toff = s_toff;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) host[0] = toff[tiles];
    const Z *Cx = (const Z *) g.Cx, *Tx = (const Z *) g.Tx;
    Z *Ox = (Z *) g.Ox;
    const int64_t stride = (int64_t) gridDim.x * AC_NT, t0 = (int64_t) blockIdx.x * AC_NT + threadIdx.x;
    for (int64_t p = t0; p < g.nc; p += stride)
    {
        int64_t q;
        const int st = ac_again<LEAN, IPT>(g, true, p, q);
        if (st == AC_NONE) continue;
        const int64_t o = ac_before_c<LEAN, IPT>(g, toff, p) + ac_before_t<LEAN, IPT>(g, toff, q);
        g.Oj[o] = g.Cj[p];
        if (st == AC_OTHER) Ox[o] = Tx[g.t_iso ? 0 : q];
        else
        {
            const Z c = Cx[g.c_iso ? 0 : p];
            Ox[o] = st == AC_BOTH ? accum_apply<Z>(g.op, c, Tx[g.t_iso ? 0 : q]) : c;
        }
    }
    for (int64_t q = t0; q < g.nt; q += stride)
    {
        int64_t p;
        if (ac_again<LEAN, IPT>(g, false, q, p) == AC_NONE) continue;
        const int64_t o = ac_before_t<LEAN, IPT>(g, toff, q) + ac_before_c<LEAN, IPT>(g, toff, p);
        g.Oj[o] = g.Tj[q];
        Ox[o] = Tx[g.t_iso ? 0 : q];
    }
    for (int64_t i = t0; i <= g.m; i += stride)
        g.Op[i] = ac_before_c<LEAN, IPT>(g, toff, g.Cp ? g.Cp[i] : 0) + ac_before_t<LEAN, IPT>(g, toff, g.Tp[i]);
}

// nnz(C) and nnz(T) to the host
__global__ void k_accum_sizes(const int64_t *Cp, const int64_t *Tp, int64_t m, int64_t *host)
{
    if (threadIdx.x == 0) host[0] = Cp ? Cp[m] : 0;
    if (threadIdx.x == 1) host[1] = Tp[m];
}

// the merge of operands whose entry counts are known; hp: pinned
template <class Z, bool LEAN, int IPT>
static int accum_try(gm_csr_out *O, AccArgs g, const gm_csr *T, int64_t *hp)
{
    hipStream_t st = stream();
    const int64_t m = g.m;
    constexpr int64_t TILE = AC_NT * IPT;
    g.ntc = g.nc / TILE + 1;
    g.ntt = g.nt / TILE + 1;
    const int64_t tiles = g.ntc + g.ntt;
    const size_t slots = (size_t) tiles * TILE;
    DevBuf Op, Oj, Ox, work;
    auto output = [&](int64_t entries) {
        if (!Oj.alloc(sizeof(int64_t) * (size_t) (entries > 0 ? entries : 1)) ||
            !Ox.alloc(sizeof(Z) * (size_t) (entries > 0 ? entries : 1)))
            return set_error(GM_OUT_OF_MEMORY, "accum: output (%lld entries)", (long long) entries);
        g.Oj = Oj.as<int64_t>();
        g.Ox = Ox.ptr;
        return GM_SUCCESS;
    };
    // a small output at its bound, so that its size needs no wait of its own
    const int64_t most = g.nc + g.nt;
    const bool bound = most * (int64_t) (sizeof(int64_t) + sizeof(Z)) <= OUT_BOUND_MAX;
    if (bound) GM_TRY(output(most));
    const size_t tbytes = sizeof(int64_t) * (size_t) (tiles + 1);
    if (!Op.alloc(sizeof(int64_t) * (m + 1))) return set_error(GM_OUT_OF_MEMORY, "accum: row pointers");
    if (!work.alloc(tbytes + (LEAN ? slots / 8 : slots * 13))) return set_error(GM_OUT_OF_MEMORY, "accum: workspace");
    g.toff = work.as<int64_t>();
    g.bits = (uint64_t *) (g.toff + tiles + 1);
    g.other = g.toff + tiles + 1;
    g.rank = (uint32_t *) (g.other + slots);
    g.state = (uint8_t *) (g.rank + slots);
    g.Op = Op.as<int64_t>();
    {
        ProfScope ps("accum_mask_state");
        k_accum_state<LEAN, IPT><<<(unsigned) tiles, AC_NT, 0, st>>>(g);
        GM_HIP(hipGetLastError(), "k_accum_state");
    }
    if (IPT != 1) GM_TRY(scan_exclusive_i64(g.toff, g.toff, tiles));
    if (!bound)
    {
        GM_HIP(hipMemcpyAsync(hp, g.toff + tiles, sizeof(int64_t), hipMemcpyDeviceToHost, st), "accum nnz");
        GM_HIP(hipStreamSynchronize(st), "accum nnz sync");
        GM_TRY(output(hp[0]));
    }
    {
        ProfScope ps("accum_mask_write");
        int64_t items = g.nc > g.nt ? g.nc : g.nt;
        if (m + 1 > items) items = m + 1;
        k_accum_write<Z, LEAN, IPT><<<post_grid(items, AC_NT, (int64_t) cu_count() * 16), AC_NT, 0, st>>>(g, hp);
        GM_HIP(hipGetLastError(), "k_accum_write");
    }
    GM_HIP(hipStreamSynchronize(st), "accum sync");
    const int64_t nz = hp[0];
    if (bound)
    {
        bool moved = fit_block(Oj, sizeof(int64_t) * nz, sizeof(int64_t) * most);
        moved |= fit_block(Ox, sizeof(Z) * nz, sizeof(Z) * most);
        if (moved) GM_HIP(hipStreamSynchronize(st), "accum fit sync");
    }
    O->nrows = m;
    O->ncols = T->ncols;
    O->nvals = nz;
    O->p = (int64_t *) Op.release();
    O->j = (int64_t *) Oj.release();
    O->x = Ox.release();
    O->iso = 0;
    O->type = T->type;
    return GM_SUCCESS;
}

template <class Z>
static int accum_mask_run(gm_csr_out *O, const gm_csr *C, const gm_csr *M, bool mask_comp,
                          bool mask_struct, bool replace, const gm_csr *T, int32_t op, int64_t nc, int64_t nt)
{
    hipStream_t st = stream();
    const int64_t m = T->nrows;
    AccArgs g;
    memset(&g, 0, sizeof(g));
    g.m = m;
    if (C && C->p) { g.Cp = C->p; g.Cj = C->j; g.Cx = C->x; g.c_iso = C->iso; }
    g.Tp = T->p; g.Tj = T->j; g.Tx = T->x; g.t_iso = T->iso;
    if (M && M->p)
    {
        g.has_mask = 1;
        g.Mp = M->p; g.Mj = M->j; g.Mx = mask_struct ? nullptr : M->x;
        g.m_iso = M->iso; g.msize = (int32_t) type_size(M->type);
    }
    g.mask_comp = mask_comp ? 1 : 0;
    g.mask_struct = (mask_struct || !M || !M->x) ? 1 : 0;
    g.replace = replace ? 1 : 0;
    g.op = op;
    int64_t *hp = (int64_t *) pinned_scratch(2 * sizeof(int64_t));
    if (!hp) return set_error(GM_OUT_OF_MEMORY, "pinned scratch");
    const bool known = nc >= 0 && nt >= 0;
    hp[0] = g.Cp && known ? nc : 0;
    hp[1] = nt;
    if (!known)
    {
        k_accum_sizes<<<1, 64, 0, st>>>(g.Cp, g.Tp, m, hp);
        GM_HIP(hipGetLastError(), "k_accum_sizes");
        GM_HIP(hipStreamSynchronize(st), "accum sizes sync");
    }
    g.nc = hp[0];
    g.nt = hp[1];
    // (a merge of few tiles is below OUT_BOUND_MAX)
    const bool few = g.nc / AC_NT + g.nt / AC_NT + 2 <= AC_FEW;
    int rc = few ? accum_try<Z, false, 1>(O, g, T, hp) : accum_try<Z, false, AC_IPT>(O, g, T, hp);
    if (rc == GM_OUT_OF_MEMORY) rc = accum_try<Z, true, AC_IPT>(O, g, T, hp);
    return rc;
}

} // namespace gm

using namespace gm;

extern "C" int gm_transpose(gm_csr_out *T, const gm_csr *A)
{
    if (!T || !A || !A->p) return set_error(GM_INVALID_VALUE, "gm_transpose: NULL argument");
    if (A->nrows >= ((int64_t) 1 << 32) || A->ncols >= ((int64_t) 1 << 32))
        return set_error(GM_NO_VALUE, "gm_transpose: dimensions beyond 2^32");
    GM_TRY(ensure_init());
    hipStream_t st = stream();
    const int64_t m = A->nrows, n = A->ncols;
    int64_t nnz = 0;
    {
        int64_t *hp = (int64_t *) pinned_scratch(sizeof(int64_t));
        if (!hp) return set_error(GM_OUT_OF_MEMORY, "pinned scratch");
        GM_HIP(hipMemcpyAsync(hp, A->p + m, sizeof(int64_t), hipMemcpyDeviceToHost, st), "nnz(A)");
        GM_HIP(hipStreamSynchronize(st), "nnz(A) sync");
        nnz = *hp;
    }
    const size_t xs = A->x ? type_size(A->type) : 0;
    const bool iso = A->iso != 0;
    DevBuf Tp, Tj, Tx, k0, k1, p0, p1, tmp;
    if (!Tp.alloc(sizeof(int64_t) * (n + 1)) || !Tj.alloc(sizeof(int64_t) * (nnz > 0 ? nnz : 1)) ||
        (xs && !Tx.alloc(iso ? xs : xs * (nnz > 0 ? nnz : 1))))
        return set_error(GM_OUT_OF_MEMORY, "gm_transpose: output");
    if (nnz > 0)
    {
        if (!k0.alloc(8 * nnz) || !k1.alloc(8 * nnz) || !p0.alloc(8 * nnz) || !p1.alloc(8 * nnz))
            return set_error(GM_OUT_OF_MEMORY, "gm_transpose: sort buffers");
        const unsigned grid = post_grid(nnz, 256, (int64_t) cu_count() * 16);
        {
            ProfScope ps("transpose_keys");
            k_tr_keys<<<post_grid(nnz, TR_TILE, (int64_t) cu_count() * 16), 256, 0, st>>>(
                A->p, A->j, m, nnz, k0.as<uint64_t>(), p0.as<int64_t>());
            GM_HIP(hipGetLastError(), "k_tr_keys");
        }
        // the keys enter in row order and the radix sort is stable, so
        // sorting by the column bits alone leaves each column's rows ascending
        int cbits = 1;
        while (cbits < 32 && ((int64_t) 1 << cbits) < n) cbits++;
        const unsigned begin_bit = 32u, end_bit = 32u + (unsigned) cbits;
        size_t tb = 0;
        GM_HIP(rocprim::radix_sort_pairs(nullptr, tb, k0.as<uint64_t>(), k1.as<uint64_t>(),
                                         p0.as<int64_t>(), p1.as<int64_t>(), (size_t) nnz, begin_bit, end_bit,
                                         st), "transpose sort size");
        if (!tmp.alloc(tb)) return set_error(GM_OUT_OF_MEMORY, "gm_transpose: sort storage");
        {
            ProfScope ps("transpose_sort");
            GM_HIP(rocprim::radix_sort_pairs(tmp.ptr, tb, k0.as<uint64_t>(), k1.as<uint64_t>(),
                                             p0.as<int64_t>(), p1.as<int64_t>(), (size_t) nnz, begin_bit,
                                             end_bit, st), "transpose sort");
        }
        {
            ProfScope ps("transpose_fill");
            k_tr_rows<<<post_grid(n + 1, 256, (int64_t) cu_count() * 16), 256, 0, st>>>(
                k1.as<uint64_t>(), nnz, n, Tp.as<int64_t>());
            GM_HIP(hipGetLastError(), "k_tr_rows");
            k_tr_fill<<<grid, 256, 0, st>>>(k1.as<uint64_t>(), p1.as<int64_t>(), nnz,
                                            (const uint8_t *) A->x, (int32_t) xs, Tj.as<int64_t>(),
                                            (xs && !iso) ? Tx.as<uint8_t>() : nullptr);
            GM_HIP(hipGetLastError(), "k_tr_fill");
        }
    }
    else
    {
        k_post_zero<<<post_grid(n + 1, 256, 1024), 256, 0, st>>>(Tp.as<int64_t>(), n + 1);
        GM_HIP(hipGetLastError(), "k_post_zero");
    }
    if (xs && iso) GM_HIP(hipMemcpyAsync(Tx.ptr, A->x, xs, hipMemcpyDeviceToDevice, st), "iso value");
    GM_HIP(hipStreamSynchronize(st), "transpose sync");
    T->nrows = n;
    T->ncols = m;
    T->nvals = nnz;
    T->p = (int64_t *) Tp.release();
    T->j = (int64_t *) Tj.release();
    T->x = xs ? Tx.release() : nullptr;
    T->iso = iso ? 1 : 0;
    T->type = A->type;
    return GM_SUCCESS;
}

extern "C" int gm_accum_mask(gm_csr_out *O, const gm_csr *C, const gm_csr *M, bool mask_comp,
                             bool mask_struct, bool replace, const gm_csr *T, int32_t accum_op)
{
    return gm_accum_mask_sized(O, C, -1, M, mask_comp, mask_struct, replace, T, -1, accum_op);
}

extern "C" int gm_accum_mask_sized(gm_csr_out *O, const gm_csr *C, int64_t nc, const gm_csr *M, bool mask_comp,
                                   bool mask_struct, bool replace, const gm_csr *T, int64_t nt, int32_t accum_op)
{
    if (!O || !T || !T->p) return set_error(GM_INVALID_VALUE, "gm_accum_mask: NULL argument");
    if (C && C->p && (C->nrows != T->nrows || C->ncols != T->ncols || C->type != T->type))
        return set_error(GM_INVALID_VALUE, "gm_accum_mask: C and T differ in shape or type");
    if (M && M->p && (M->nrows != T->nrows || M->ncols != T->ncols))
        return set_error(GM_INVALID_VALUE, "gm_accum_mask: mask shape");
    if (accum_op < 0 || accum_op > 11)
        return set_error(GM_INVALID_VALUE, "gm_accum_mask: accumulator %d", accum_op);
    if ((C && C->p && !C->x) || !T->x)
        return set_error(GM_INVALID_VALUE, "gm_accum_mask: C and T need values");
    GM_TRY(ensure_init());
    switch (T->type)
    {
        case GM_BOOL: return accum_mask_run<uint8_t>(O, C, M, mask_comp, mask_struct, replace, T, accum_op, nc, nt);
        case GM_INT32: return accum_mask_run<int32_t>(O, C, M, mask_comp, mask_struct, replace, T, accum_op, nc, nt);
        case GM_INT64: return accum_mask_run<int64_t>(O, C, M, mask_comp, mask_struct, replace, T, accum_op, nc, nt);
        case GM_FP64: return accum_mask_run<double>(O, C, M, mask_comp, mask_struct, replace, T, accum_op, nc, nt);
        default: return set_error(GM_NO_VALUE, "gm_accum_mask: type %d not supported", T->type);
    }
}
