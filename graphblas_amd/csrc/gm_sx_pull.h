// gm_sx_pull.h: a one-row A times B', C = A*B' and C<!M> = A*B' (GrB_mxv, and
// GrB_vxm with a transposed matrix), without transposing B.
//
// A is spread out as a dense vector with a presence bit per index; then
//   pull   a workgroup takes PL_CH consecutive entries of B, whatever rows
//          they belong to (a hub row is cut into many pieces, a thousand
//          short rows share one), forms the products in LDS and sums each
//          row's piece there: short pieces by a thread, long ones by a
//          wavefront.  Rows inside the chunk are done; the pieces of rows
//          that cross a chunk's ends are kept
//   fix    one wavefront per such row joins its pieces in order
// and the result is compacted as the spread rows' tables are (gm_sx_push.h).
// The cuts depend on B alone, so fp64 sums are the same from run to run; they
// are tree sums, as in dot3.  ANY with the inner index keeps the largest k, the
// last writer of the saxpy methods.
//
// Bound by the entries of B, read once, the gathers of A's values (L2) and,
// at a few million entries, by its ten launches.  Three products with an RMAT
// matrix of n = 65536, 1.82M entries, fp64, and the last vector's copy to the
// host: 350 ms with the transpose and one workgroup for the row, 0.53 ms here.
#pragma once

namespace gm
{

constexpr int PL_NT = 256;
constexpr int PL_IPT = 8;
constexpr int PL_CH = PL_NT * PL_IPT;      // entries of B per workgroup
constexpr int PL_LONG = 64;                // longer pieces: a wavefront
// A chunk over more rows than this, mostly empty ones, searches its entries'
// rows.  2000 entries over 2^13 rows: 113 us a GrB_mxv either way; over 2^14
// 128 walked and 113 searched, over 2^24 21.0 ms and 0.196 ms.
constexpr int64_t PL_WALK = 4 * PL_CH;

struct PullArgs
{
    int64_t nnz, nch;
    uint32_t *ubits;            // A's presence bits over the inner index
    void *uval;                 // A's values there
    void *pz;                   // 2 x nch: the chunks' pieces of a row begun before, of a row that goes on
    uint8_t *pe;
    int64_t *lrow;              // nch: the chunk's row that begins in it and goes on, or -1
};

// the products of one lane or piece, combined in any grouping: ANY with the
// inner index keeps the largest
template <class S>
__device__ __forceinline__ void pl_join(bool &e, typename S::Z &z, bool e2, typename S::Z z2)
{
    if (!e2) return;
    if (!e) { e = true; z = z2; }
    else if constexpr (S::any_min_k) z = z2 > z ? z2 : z;
    else z = S::upd(z, z2);
}

template <class S>
__device__ __forceinline__ void pl_wave_join(bool &e, typename S::Z &z)
{
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1)
    {
        const int e2 = __shfl_down((int) e, off, 64);
        const typename S::Z z2 = shfl_down<typename S::Z>(z, off, 64);
        pl_join<S>(e, z, e2 != 0, z2);
    }
}

template <class S>
__global__ __launch_bounds__(PL_NT) void k_pull_scatter(SxArgs g, PullArgs p)
{
    using Z = typename S::Z;
    const int64_t nz = g.Ap[1] - g.Ap[0];
    for (int64_t t = (int64_t) blockIdx.x * PL_NT + threadIdx.x; t < nz; t += (int64_t) gridDim.x * PL_NT)
    {
        const int64_t q = g.Ap[0] + t, k = g.Aj[q];
        atomicOr(&p.ubits[k >> 5], 1u << (k & 31));
        if constexpr (!S::pattern) ((Z *) p.uval)[k] = S::geta((const Z *) g.Ax, q, g.a_iso);
    }
}

// last row r in [0, n) with Bp[r] <= v, by the lanes of a wavefront together
__device__ __forceinline__ int64_t pl_row_of(const int64_t *Bp, int64_t n, int64_t v)
{
    const int lane = threadIdx.x & 63;
    int64_t lo = 0, hi = n;                 // Bp[lo] <= v < Bp[hi]
    while (hi - lo > 1)
    {
        const int64_t step = (hi - lo + 63) / 64;
        const int64_t at = lo + (int64_t) lane * step;
        const int c = __popcll(__ballot(at < hi && Bp[at] <= v));
        const int64_t nlo = lo + (int64_t) (c - 1) * step, nhi = lo + (int64_t) c * step;
        lo = nlo;
        hi = nhi < hi ? nhi : hi;
    }
    return lo;
}

// row j's result: its cell and presence bit, unless the mask holds j
template <class S>
__device__ __forceinline__ void pl_store(const SxArgs &g, const PushArgs &h, int64_t j, bool e, typename S::Z z)
{
    if (!e) return;
    if (g.mode != MODE_NONE && ((h.mbits[j >> 5] >> (j & 31)) & 1u)) return;
    if constexpr (PU_U32<S>) ((uint32_t *) h.tab)[j] = S::any_min_k ? (uint32_t) z + 1u : (uint32_t) z;
    else
    {
        if constexpr (!S::iso_out) ((typename S::Z *) h.tab)[j] = z;
        atomicOr(&h.bits[j >> 5], 1u << (j & 31));
    }
}

template <class S>
__global__ __launch_bounds__(PL_NT) void k_pull(SxArgs g, PushArgs h, PullArgs p)
{
    using Z = typename S::Z;
    __shared__ Z s_z[PL_CH];
    __shared__ unsigned long long s_has[PL_CH / 64];
    __shared__ int64_t s_row[2];
    __shared__ int s_list[PL_CH / PL_LONG + 2], s_nlist;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int64_t nrows = g.n;
    for (int64_t c = blockIdx.x; c < p.nch; c += gridDim.x)
    {
        const int64_t e0 = c * PL_CH, e1 = e0 + PL_CH < p.nnz ? e0 + PL_CH : p.nnz;
        if (tid == 0) { s_nlist = 0; p.lrow[c] = -1; }
        if (wv < 2)
        {
            const int64_t r = pl_row_of(g.Bp, nrows, wv == 0 ? e0 : e1 - 1);
            if (lane == 0) s_row[wv] = r;
        }
        int64_t k[PL_IPT];
        #pragma unroll
        for (int t = 0; t < PL_IPT; t++)
        {
            const int64_t e = e0 + t * PL_NT + tid;
            k[t] = e < e1 ? g.Bj[e] : -1;
        }
        #pragma unroll
        for (int t = 0; t < PL_IPT; t++)
        {
            const int64_t e = e0 + t * PL_NT + tid;
            const bool in = k[t] >= 0 && ((p.ubits[k[t] >> 5] >> (k[t] & 31)) & 1u);
            if (in)
            {
                Z a = Z(0);
                if constexpr (!S::pattern) a = ((const Z *) p.uval)[k[t]];
                s_z[t * PL_NT + tid] = S::mul(a, S::geta((const Z *) g.Bx, e, g.b_iso), k[t]);
            }
            const unsigned long long b = __ballot(in);
            if (lane == 0) s_has[(t * PL_NT + tid) >> 6] = b;
        }
        __syncthreads();
        const int64_t r0 = s_row[0], r1 = s_row[1];
        // a piece's result: the whole row's, or one of the chunk's two kept pieces
        auto put = [&](int64_t r, bool e, Z z) {
            const bool before = g.Bp[r] < e0, after = g.Bp[r + 1] > e1;
            if (!before && !after) { pl_store<S>(g, h, r, e, z); return; }
            const int64_t s = before ? 2 * c : 2 * c + 1;
            ((Z *) p.pz)[s] = z;
            p.pe[s] = e ? 1 : 0;
            if (!before) p.lrow[c] = r;
        };
        // entries [b0, b1) of row r
        auto piece = [&](int64_t r, int64_t b0, int64_t b1) {
            if (b1 - b0 > PL_LONG) { s_list[atomicAdd(&s_nlist, 1)] = (int) (r - r0); return; }
            bool e = false;
            Z z = S::identity();
            for (int q = (int) (b0 - e0); q < (int) (b1 - e0); q++)
                if ((s_has[q >> 6] >> (q & 63)) & 1ull) pl_join<S>(e, z, true, s_z[q]);
            put(r, e, z);
        };
        if (r1 - r0 <= PL_WALK)
            for (int64_t r = r0 + tid; r <= r1; r += PL_NT)
            {
                const int64_t b0 = g.Bp[r] > e0 ? g.Bp[r] : e0, b1 = g.Bp[r + 1] < e1 ? g.Bp[r + 1] : e1;
                if (b0 < b1) piece(r, b0, b1);
            }
        else
        {
            // mostly empty rows: a thread searches its entries' rows, in step,
            // and takes those that begin with one of them
            int64_t lo[PL_IPT], hi[PL_IPT];
            #pragma unroll
            for (int t = 0; t < PL_IPT; t++) { lo[t] = r0; hi[t] = r1; }
            for (int64_t w = r1 - r0; w > 0; w >>= 1)
            {
                #pragma unroll
                for (int t = 0; t < PL_IPT; t++)
                {
                    const int64_t mid = (lo[t] + hi[t] + 1) >> 1;
                    if (g.Bp[mid] <= e0 + t * PL_NT + tid) lo[t] = mid;
                    else hi[t] = mid - 1;
                }
            }
            #pragma unroll
            for (int t = 0; t < PL_IPT; t++)
            {
                const int64_t e = e0 + t * PL_NT + tid, b1 = g.Bp[lo[t] + 1];
                if (e < e1 && (e == e0 || g.Bp[lo[t]] == e)) piece(lo[t], e, b1 < e1 ? b1 : e1);
            }
        }
        __syncthreads();
        for (int l = wv; l < s_nlist; l += PL_NT / 64)
        {
            const int64_t r = r0 + s_list[l];
            const int64_t b0 = g.Bp[r] > e0 ? g.Bp[r] : e0, b1 = g.Bp[r + 1] < e1 ? g.Bp[r + 1] : e1;
            bool e = false;
            Z z = S::identity();
            for (int q = (int) (b0 - e0) + lane; q < (int) (b1 - e0); q += 64)
                if ((s_has[q >> 6] >> (q & 63)) & 1ull) pl_join<S>(e, z, true, s_z[q]);
            pl_wave_join<S>(e, z);
            if (lane == 0) put(r, e, z);
        }
        __syncthreads();
    }
}

// rows that cross chunk ends: one wavefront per chunk in which such a row begins
template <class S>
__global__ __launch_bounds__(PL_NT) void k_pull_fix(SxArgs g, PushArgs h, PullArgs p)
{
    using Z = typename S::Z;
    const int lane = threadIdx.x & 63;
    for (int64_t c = (int64_t) blockIdx.x * (PL_NT / 64) + (threadIdx.x >> 6); c < p.nch;
         c += (int64_t) gridDim.x * (PL_NT / 64))
    {
        const int64_t r = p.lrow[c];
        if (r < 0) continue;
        const int64_t last = (g.Bp[r + 1] - 1) / PL_CH;
        bool e = false;
        Z z = S::identity();
        if (lane == 0 && p.pe[2 * c + 1]) { e = true; z = ((const Z *) p.pz)[2 * c + 1]; }
        for (int64_t q = c + 1 + lane; q <= last; q += 64)
            if (p.pe[2 * q]) pl_join<S>(e, z, true, ((const Z *) p.pz)[2 * q]);
        pl_wave_join<S>(e, z);
        if (lane == 0) pl_store<S>(g, h, r, e, z);
    }
}

__global__ void k_pull_ptr(int64_t *Cp, const int64_t *seg, int64_t nseg)
{
    if (threadIdx.x == 0) { Cp[0] = 0; Cp[1] = seg[nseg]; }
}

} // namespace gm
