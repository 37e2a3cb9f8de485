// gm_sx_push.h: saxpy3 rows whose products are spread over the whole device.
//
// A row of C with very many products (a frontier that has reached the hubs, a
// vector times a matrix) keeps one workgroup of the hash kernels busy for
// milliseconds while the rest of the device idles.  For semirings whose
// updates may come in any order (SX_ANY_ORDER) such a row gets a dense table
// in HBM instead, one cell per column of C, and its products are cut into
// items of PU_CH that any workgroup takes:
//
//   pre      running sum of |B(k,:)| over A's entries (device scan)
//   items    (row, chunk) -> the A entry that holds the chunk's first product
//   push     256 A entries at a time in LDS; every product finds its entry by
//            a search there, tests the mask's bit and updates its cell with an
//            atomic, after a plain read that skips what would change nothing
//            (MIN, MAX, ANY: a stale read only costs an atomic)
//   count    present cells per segment of PU_SEG columns, scan -> Cp[i]
//   write    the cells in column order, so nothing is sorted
//
// Cells hold the largest inner index + 1 (ANY), a count (PLUS_PAIR), or the
// value with sx_cell0 for "none"; a bit per column says present where the cell
// cannot (PLUS_TIMES, ANY_PAIR, an integer product equal to the identity, a
// NaN).
//
// What bounds it: the atomics at L2 / memory, the gathers of B, and for few
// rows the launches.  Second level of 64 searches on RMAT scale 20
// (any_secondi, 1.9M entries of C): 53.6 ms with one workgroup per row, 0.90
// ms for the call here.
#pragma once

namespace gm
{

constexpr int PU_CH = 4096;            // products per item
constexpr int PU_SEG = 2048;           // columns per compaction segment
constexpr int PU_NT = 256;

// cells: 32-bit inner index + 1 or count, else the semiring's values
template <class S>
constexpr bool PU_U32 = S::any_min_k || (S::add == GM_ADD_PLUS && S::mult == GM_MULT_PAIR);
template <class S>
constexpr bool PU_BITS = !PU_U32<S>;   // a presence bit per column
template <class S>
using PuCell = std::conditional_t<PU_U32<S>, uint32_t, typename S::Z>;

struct PushArgs
{
    uint32_t *drow;                    // the dense rows
    int64_t *dflops;
    int64_t D, nw;                     // rows; 32-bit words of a bit row
    const int64_t *pre;                // nnz(A) + 1 running products
    int64_t *coff;                     // D + 1: first item of row d
    uint32_t *it_d;                    // per item: its row's index d
    int64_t *it_e;                     //           its first product's A entry
    void *tab;                         // D x n cells
    uint32_t *bits, *mbits;            // D x nw presence / mask bits
    int32_t all_bits;                  // every present cell has its bit (absent cells hold anything)
    int64_t nseg;
    int64_t *seg;                      // D x nseg + 1: scanned segment counts
};

// products of every row of a few-row A, each row over gridDim.x workgroups
__global__ __launch_bounds__(PU_NT) void k_sx_rowflops(SxArgs g, unsigned long long *rowf)
{
    __shared__ unsigned long long s[PU_NT / 64 + 1];
    const int64_t i = blockIdx.y;
    unsigned long long f = 0;
    for (int64_t e = g.Ap[i] + (int64_t) blockIdx.x * PU_NT + threadIdx.x; e < g.Ap[i + 1];
         e += (int64_t) gridDim.x * PU_NT)
    {
        const int64_t k = g.Aj[e];
        f += (unsigned long long) (g.Bp[k + 1] - g.Bp[k]);
    }
    const unsigned long long tot = block_sum<unsigned long long, PU_NT>(f, s);
    if (threadIdx.x == 0 && tot) atomicAdd(&rowf[i], tot);
}

// |B(k,:)| of every entry of A
__global__ __launch_bounds__(PU_NT) void k_sx_elen(SxArgs g, int64_t nnz, int64_t *len)
{
    for (int64_t e = (int64_t) blockIdx.x * PU_NT + threadIdx.x; e < nnz; e += (int64_t) gridDim.x * PU_NT)
    {
        const int64_t k = g.Aj[e];
        len[e] = g.Bp[k + 1] - g.Bp[k];
    }
}

__global__ __launch_bounds__(PU_NT) void k_sx_push_chunks(PushArgs h)
{
    for (int64_t d = (int64_t) blockIdx.x * PU_NT + threadIdx.x; d < h.D; d += (int64_t) gridDim.x * PU_NT)
        h.coff[d] = (h.dflops[d] + PU_CH - 1) / PU_CH;
}

// last index in [lo, hi] with a[index] <= v
__device__ __forceinline__ int64_t pu_last_le(const int64_t *a, int64_t lo, int64_t hi, int64_t v)
{
    while (lo < hi)
    {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (a[mid] <= v) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(PU_NT) void k_sx_push_items(SxArgs g, PushArgs h)
{
    const int64_t n = h.coff[h.D];
    for (int64_t it = (int64_t) blockIdx.x * PU_NT + threadIdx.x; it < n; it += (int64_t) gridDim.x * PU_NT)
    {
        const int64_t d = pu_last_le(h.coff, 0, h.D - 1, it);
        const int64_t i = h.drow[d], a0 = g.Ap[i], a1 = g.Ap[i + 1];
        h.it_d[it] = (uint32_t) d;
        h.it_e[it] = pu_last_le(h.pre, a0, a1 - 1, h.pre[a0] + (it - h.coff[d]) * PU_CH);
    }
}

template <class S>
__global__ __launch_bounds__(PU_NT) void k_sx_push_init(PushArgs h, int64_t cells, int64_t words, int mask)
{
    const int64_t stride = (int64_t) gridDim.x * PU_NT, t0 = (int64_t) blockIdx.x * PU_NT + threadIdx.x;
    if constexpr (!S::iso_out)
    {
        PuCell<S> *tab = (PuCell<S> *) h.tab;
        const PuCell<S> id = PU_U32<S> ? (PuCell<S>) 0 : (PuCell<S>) sx_cell0<S>();
        for (int64_t t = t0; t < cells; t += stride) tab[t] = id;
    }
    if constexpr (PU_BITS<S>)
        for (int64_t t = t0; t < words; t += stride) h.bits[t] = 0;
    if (mask)
        for (int64_t t = t0; t < words; t += stride) h.mbits[t] = 0;
}

// the mask's true entries of the dense rows as bits (gridDim.x workgroups a row)
__global__ __launch_bounds__(PU_NT) void k_sx_push_mask(SxArgs g, PushArgs h)
{
    for (int64_t d = blockIdx.y; d < h.D; d += gridDim.y)
    {
        const int64_t i = h.drow[d];
        for (int64_t q = g.Mp[i] + (int64_t) blockIdx.x * PU_NT + threadIdx.x; q < g.Mp[i + 1];
             q += (int64_t) gridDim.x * PU_NT)
        {
            if (!g.mask_struct && !mask_true(g.Mx, q, g.msize, g.m_iso)) continue;
            const int64_t j = g.Mj[q];
            atomicOr(&h.mbits[d * h.nw + (j >> 5)], 1u << (j & 31));
        }
    }
}

template <class S>
__device__ __forceinline__ void pu_update(const PushArgs &h, int64_t n, int64_t d, int64_t j, typename S::Z t)
{
    using Z = typename S::Z;
    uint32_t *bw = h.bits + d * h.nw + (j >> 5);
    const uint32_t bit = 1u << (j & 31);
    if constexpr (S::iso_out)
    {
        if (!(*bw & bit)) atomicOr(bw, bit);
    }
    else if constexpr (S::any_min_k)
    {
        uint32_t *c = (uint32_t *) h.tab + d * n + j;
        const uint32_t v = (uint32_t) t + 1u;
        if (*c < v) atomicMax(c, v);
    }
    else if constexpr (PU_U32<S>)
    {
        atomicAdd((uint32_t *) h.tab + d * n + j, 1u);
    }
    else
    {
        Z *c = (Z *) h.tab + d * n + j;
        if constexpr (S::add == GM_ADD_PLUS)
        {
            if (!(*bw & bit)) atomicOr(bw, bit);
            if constexpr (SX_ANY_ORDER<S>) sx_atomic_upd<S>(c, t);
        }
        else
        {
            // a NaN, or an integer equal to the identity, leaves the cell as it is
            const Z cur = *c;
            if (t != t || t == sx_cell0<S>())
            {
                if (!(*bw & bit)) atomicOr(bw, bit);
            }
            else if (sx_changes<S>(cur, t)) sx_atomic_upd<S>(c, t);
        }
    }
}

template <class S>
__global__ __launch_bounds__(PU_NT) void k_sx_push(SxArgs g, PushArgs h)
{
    using Z = typename S::Z;
    __shared__ int64_t s_pre[PU_NT + 1], s_bs[PU_NT], s_k[PU_NT];
    __shared__ Z s_av[PU_NT];
    const int tid = threadIdx.x;
    const int64_t nitems = h.coff[h.D];
    for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x)
    {
        const int64_t d = h.it_d[it], i = h.drow[d];
        const int64_t a0 = g.Ap[i], a1 = g.Ap[i + 1];
        int64_t f = h.pre[a0] + (it - h.coff[d]) * PU_CH;
        const int64_t fe = h.pre[a1] < f + PU_CH ? h.pre[a1] : f + PU_CH;
        for (int64_t e = h.it_e[it]; f < fe; e += PU_NT)
        {
            __syncthreads();
            const int64_t q = e + tid;
            s_pre[tid] = q < a1 ? h.pre[q] : INT64_MAX;
            if (q < a1)
            {
                const int64_t k = g.Aj[q];
                s_k[tid] = k;
                s_bs[tid] = g.Bp[k];
                s_av[tid] = S::geta((const Z *) g.Ax, q, g.a_iso);
            }
            if (tid == 0) s_pre[PU_NT] = h.pre[e + PU_NT < a1 ? e + PU_NT : a1];
            __syncthreads();
            const int64_t we = s_pre[PU_NT] < fe ? s_pre[PU_NT] : fe;
            // four products per thread and step, their gathers together (past
            // the window's end: its last product again, not applied)
            constexpr int UN = 4;
            for (int64_t f0 = f + tid; f0 < we; f0 += UN * PU_NT)
            {
                int lo[UN];
                int64_t pb[UN], j[UN];
                #pragma unroll
                for (int u = 0; u < UN; u++)
                {
                    const int64_t ff = f0 + u * PU_NT < we ? f0 + u * PU_NT : we - 1;
                    int l = 0, r = PU_NT - 1;
                    #pragma unroll
                    for (int s = 0; s < 8; s++)
                    {
                        const int mid = (l + r + 1) >> 1;
                        const bool le = s_pre[mid] <= ff;
                        l = le ? mid : l;
                        r = le ? r : (mid > l ? mid - 1 : l);
                    }
                    lo[u] = l;
                    pb[u] = s_bs[l] + (ff - s_pre[l]);
                }
                #pragma unroll
                for (int u = 0; u < UN; u++) j[u] = g.Bj[pb[u]];
                #pragma unroll
                for (int u = 0; u < UN; u++)
                {
                    if (f0 + u * PU_NT >= we) continue;
                    if (g.mode != MODE_NONE)
                    {
                        const bool in = (h.mbits[d * h.nw + (j[u] >> 5)] >> (j[u] & 31)) & 1u;
                        if (in != (g.mode == MODE_MASK)) continue;
                    }
                    pu_update<S>(h, g.n, d, j[u],
                                 S::mul(s_av[lo[u]], S::geta((const Z *) g.Bx, pb[u], g.b_iso), s_k[lo[u]]));
                }
            }
            f = we;
        }
        __syncthreads();
    }
}

// is column j of dense row d present; its value
template <class S>
__device__ __forceinline__ bool pu_present(const PushArgs &h, int64_t n, int64_t d, int64_t j, typename S::Z &z)
{
    using Z = typename S::Z;
    if constexpr (PU_U32<S>)
    {
        const uint32_t c = ((const uint32_t *) h.tab)[d * n + j];
        z = S::any_min_k ? (Z) ((int64_t) c - 1) : (Z) c;
        return c != 0;
    }
    else
    {
        const bool bit = (h.bits[d * h.nw + (j >> 5)] >> (j & 31)) & 1u;
        if constexpr (S::iso_out) return bit;
        else
        {
            z = ((const Z *) h.tab)[d * n + j];
            if constexpr (std::is_same<Z, double>::value) return bit || (S::add != GM_ADD_PLUS && !h.all_bits && z == z);
            else return bit || (S::add != GM_ADD_PLUS && !h.all_bits && z != sx_cell0<S>());
        }
    }
}

template <class S>
__global__ __launch_bounds__(PU_NT) void k_sx_push_count(SxArgs g, PushArgs h)
{
    __shared__ int s[PU_NT / 64 + 1];
    for (int64_t w = blockIdx.x; w < h.D * h.nseg; w += gridDim.x)
    {
        const int64_t d = w / h.nseg, c0 = (w - d * h.nseg) * PU_SEG;
        int c = 0;
        #pragma unroll
        for (int t = 0; t < PU_SEG / PU_NT; t++)
        {
            const int64_t j = c0 + t * PU_NT + threadIdx.x;
            typename S::Z z;
            if (j < g.n && pu_present<S>(h, g.n, d, j, z)) c++;
        }
        const int tot = block_sum<int, PU_NT>(c, s);
        if (threadIdx.x == 0) h.seg[w] = tot;
    }
}

__global__ __launch_bounds__(PU_NT) void k_sx_push_rows(SxArgs g, PushArgs h)
{
    for (int64_t d = (int64_t) blockIdx.x * PU_NT + threadIdx.x; d < h.D; d += (int64_t) gridDim.x * PU_NT)
        g.Cp[h.drow[d]] = h.seg[(d + 1) * h.nseg] - h.seg[d * h.nseg];
}

template <class S>
__global__ __launch_bounds__(PU_NT) void k_sx_push_write(SxArgs g, PushArgs h)
{
    using Z = typename S::Z;
    constexpr int NIT = PU_SEG / PU_NT, NW = PU_NT / 64;
    __shared__ int s_cnt[NIT * NW];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int64_t w = blockIdx.x; w < h.D * h.nseg; w += gridDim.x)
    {
        const int64_t d = w / h.nseg, c0 = (w - d * h.nseg) * PU_SEG;
        const int64_t base = g.Cp[h.drow[d]] + (h.seg[w] - h.seg[d * h.nseg]);
        if (h.seg[w + 1] == h.seg[w]) continue;          // uniform across the workgroup
        unsigned long long bal[NIT];
        Z z[NIT];
        #pragma unroll
        for (int t = 0; t < NIT; t++)
        {
            const int64_t j = c0 + t * PU_NT + threadIdx.x;
            z[t] = Z(0);
            bal[t] = __ballot(j < g.n && pu_present<S>(h, g.n, d, j, z[t]));
            if (lane == 0) s_cnt[t * NW + wv] = __popcll(bal[t]);
        }
        __syncthreads();
        int run = 0;
        for (int q = 0; q < wv; q++) run += s_cnt[q];
        #pragma unroll
        for (int t = 0; t < NIT; t++)
        {
            if ((bal[t] >> lane) & 1ull)
            {
                const int64_t pos = base + run + __popcll(bal[t] & ((1ull << lane) - 1ull));
                g.Ci[pos] = c0 + t * PU_NT + threadIdx.x;
                if constexpr (!S::iso_out) ((Z *) g.Cx)[pos] = z[t];
            }
            for (int q = 0; q < NW; q++)
                if (t * NW + wv + q < NIT * NW) run += s_cnt[t * NW + wv + q];
        }
        __syncthreads();
    }
}

} // namespace gm
