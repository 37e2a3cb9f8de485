// gm_sx_tile.h: saxpy3 rows of C that are dense enough to be cut into tiles of
// TL_W columns.
//
// One wavefront computes one tile of one row with its accumulators in LDS, so
// no two wavefronts share a column: a row's work spreads over n / TL_W
// wavefronts, nothing is hashed or sorted, and there is no barrier.  The
// wavefront reads A(i,:) 64 entries at a time, finds each B(k,:)'s part inside
// the tile (from per-tile offsets of B's rows when enough rows use them, else
// by binary search), and takes the parts' products 64 at a time in flop order.
// Columns of a B row are distinct, and lanes that meet in a column go lowest
// first (sx_ordered_upd), so fp64 sums are the reference's sequential sums;
// any-order semirings update with LDS atomics.
//
//   phase 0  the tile's presence bits, the mask applied to them, and their
//            count; the counts' scan gives Cp[i] and every tile's place
//   phase 1  the values, written in column order at the bits' ranks
//
// Bound by the latency of its dependent steps (A entry, offsets, products,
// LDS), covered by 16 wavefronts per CU.  RMAT square, n = 40009, 0.47M entries,
// 59.8M entries of C, fp64: 30.3 ms with a workgroup and a table in HBM per
// row, 4.3 ms here for the call.
#pragma once

namespace gm
{

constexpr int TL_W = 1024;             // columns of a tile
constexpr int TL_NT = 256;
constexpr int TL_RUN = 4;              // tiles a wavefront takes at once (1 of a very heavy row)
constexpr int TL_UN = 4;               // windows of 64 products read ahead

struct TileArgs
{
    const uint32_t *front, *back;      // very heavy rows: front[q]; the others: back[-(q - nf)]
    int64_t nf, T, nt;                 // very heavy rows, all rows, tiles of a row
    const uint32_t *tpos;              // NULL, or nrows(B) x (nt + 1) offsets of B's rows
    uint64_t *bits;                    // T x nt x (TL_W / 64)
    int64_t *seg;                      // T x nt + 1: scanned tile counts
    unsigned long long *next;          // eight counters, 128 bytes apart
};

__device__ __forceinline__ int64_t tl_row(const TileArgs &t, int64_t q)
{
    return q < t.nf ? t.front[q] : *(t.back - (q - t.nf));
}

// offsets of every row of B at the tile boundaries
__global__ __launch_bounds__(TL_NT) void k_sx_tile_pos(const int64_t *__restrict__ Bp, const int64_t *__restrict__ Bj,
                                                       int64_t nrows, int64_t nt, uint32_t *__restrict__ pos)
{
    const int64_t total = nrows * (nt + 1);
    for (int64_t x = (int64_t) blockIdx.x * TL_NT + threadIdx.x; x < total; x += (int64_t) gridDim.x * TL_NT)
    {
        const int64_t r = x / (nt + 1), c = x - r * (nt + 1);
        const int64_t p0 = Bp[r], p1 = Bp[r + 1];
        pos[x] = (uint32_t) ((c == nt ? p1 : lower_bound(Bj, p0, p1, c * TL_W)) - p0);
    }
}

template <class S, int PHASE>
__global__ __launch_bounds__(TL_NT) void k_sx_tile(SxArgs g, TileArgs t)
{
    using Z = typename S::Z;
    constexpr int NWV = TL_NT / 64, NW = TL_W / 32;
    constexpr bool VALS = PHASE == 1 && !S::iso_out;
    __shared__ Z s_acc[NWV][VALS ? TL_W : 1];
    __shared__ uint32_t s_bits[NWV][PHASE == 0 ? NW : 1], s_mask[NWV][PHASE == 0 ? NW : 1];
    __shared__ uint32_t s_own[NWV][VALS ? SX_OWN : 1];
    __shared__ int32_t s_pre[NWV][64];
    __shared__ int64_t s_lo[NWV][64], s_k[NWV][S::mult == GM_MULT_K ? 64 : 1];
    __shared__ Z s_av[NWV][VALS ? 64 : 1];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t nt4 = (t.nt + TL_RUN - 1) / TL_RUN;
    const int64_t hunits = t.nf * t.nt, units = hunits + (t.T - t.nf) * nt4;
    if constexpr (VALS && !SX_ANY_ORDER<S>)
        for (int x = lane; x < SX_OWN; x += 64) s_own[wv][x] = 0xffffffffu;
    wave_sync();
    // The symbolic phase's units are dealt out by stride (80000 units from one
    // counter: 1.74 ms, 1.03 ms by stride); the numeric phase's, whose work
    // varies more (by stride 3.06 ms, one counter 2.52 ms), from eight counters,
    // one for the units of each remainder by 8, a workgroup's own first.
    int64_t su = (int64_t) blockIdx.x + (int64_t) wv * gridDim.x;
    int rem = (int) (blockIdx.x & 7), left = 8;
    while (true)
    {
        int64_t u = su;
        if constexpr (PHASE == 0) su += (int64_t) gridDim.x * NWV;
        else
        {
            u = units;
            while (left > 0)
            {
                int64_t k = 0;
                if (lane == 0) k = (int64_t) atomicAdd(&t.next[16 * rem], 1ull);
                u = __shfl(k, 0, 64) * 8 + rem;
                if (u < units) break;
                rem = (rem + 1) & 7;
                left--;
            }
        }
        if (u >= units) break;
        const bool heavy = u < hunits;
        const int64_t v = u - hunits;
        const int64_t q = heavy ? u / t.nt : t.nf + v / nt4;
        const int64_t cb = heavy ? u - q * t.nt : (v - (q - t.nf) * nt4) * TL_RUN;
        const int64_t ce = heavy ? cb + 1 : (cb + TL_RUN < t.nt ? cb + TL_RUN : t.nt);
        const int64_t i = tl_row(t, q), a0 = g.Ap[i], a1 = g.Ap[i + 1];
        for (int64_t c = cb; c < ce; c++)
        {
            const int64_t at = q * t.nt + c, c0 = c * TL_W;
            if (PHASE == 1 && t.seg[at + 1] == t.seg[at]) continue;
            if constexpr (PHASE == 0)
                for (int x = lane; x < NW; x += 64) { s_bits[wv][x] = 0; s_mask[wv][x] = 0; }
            if constexpr (VALS)
                for (int x = lane; x < TL_W; x += 64) s_acc[wv][x] = SX_ANY_ORDER<S> ? sx_cell0<S>() : S::identity();
            wave_sync();
            for (int64_t ea = a0; (PHASE == 0 || VALS) && ea < a1; ea += 64)
            {
                const int64_t e = ea + lane;
                int64_t k = 0, lo = 0;
                int32_t len = 0;
                Z av = Z(0);
                if (e < a1)
                {
                    k = g.Aj[e];
                    lo = g.Bp[k];
                    if (t.tpos)
                    {
                        const uint32_t *tp = t.tpos + k * (t.nt + 1) + c;
                        const uint32_t l = tp[0];
                        len = (int32_t) (tp[1] - l);
                        lo += l;
                    }
                    else
                    {
                        const int64_t b1 = g.Bp[k + 1];
                        lo = lower_bound(g.Bj, lo, b1, c0);
                        len = (int32_t) (lower_bound(g.Bj, lo, b1 < lo + TL_W ? b1 : lo + TL_W, c0 + TL_W) - lo);
                    }
                    if constexpr (VALS) av = S::geta((const Z *) g.Ax, e, g.a_iso);
                }
                const int32_t inc = wave_inclusive_scan<int32_t>(len);
                const int32_t tot = __shfl(inc, 63, 64);
                if (tot == 0) continue;
                s_pre[wv][lane] = inc - len;
                s_lo[wv][lane] = lo;
                if constexpr (VALS) s_av[wv][lane] = av;
                if constexpr (S::mult == GM_MULT_K) s_k[wv][lane] = k;
                wave_sync();
                for (int32_t f0 = 0; f0 < tot; f0 += 64 * TL_UN)
                {
                    int own[TL_UN];
                    int64_t pb[TL_UN];
                    int32_t slot[TL_UN];
                    Z b[TL_UN];
                    #pragma unroll
                    for (int w = 0; w < TL_UN; w++)
                    {
                        // the entry a product belongs to: the last whose offset is <= it
                        const int32_t f = f0 + w * 64 + lane, fc = f < tot ? f : tot - 1;
                        int l = 0;
                        #pragma unroll
                        for (int s = 32; s > 0; s >>= 1)
                            if (s_pre[wv][l + s] <= fc) l += s;
                        own[w] = l;
                        pb[w] = s_lo[wv][l] + (fc - s_pre[wv][l]);
                    }
                    #pragma unroll
                    for (int w = 0; w < TL_UN; w++)
                    {
                        slot[w] = (int32_t) (g.Bj[pb[w]] - c0);
                        if constexpr (VALS) b[w] = S::geta((const Z *) g.Bx, pb[w], g.b_iso);
                    }
                    #pragma unroll
                    for (int w = 0; w < TL_UN; w++)
                    {
                        if (f0 + w * 64 >= tot) break;
                        const bool in = f0 + w * 64 + lane < tot;
                        if constexpr (PHASE == 0)
                        {
                            const uint32_t bit = 1u << (slot[w] & 31);
                            if (in && !(s_bits[wv][slot[w] >> 5] & bit)) atomicOr(&s_bits[wv][slot[w] >> 5], bit);
                        }
                        else if constexpr (VALS)
                        {
                            int64_t kk = 0;
                            if constexpr (S::mult == GM_MULT_K) kk = s_k[wv][own[w]];
                            const Z tv = S::mul(s_av[wv][own[w]], b[w], kk);
                            if constexpr (SX_ANY_ORDER<S>)
                            {
                                if (in) sx_atomic_upd<S>(&s_acc[wv][slot[w]], tv);
                            }
                            else sx_ordered_upd<S>(s_acc[wv], in ? slot[w] : -1, tv, s_own[wv]);
                        }
                    }
                }
                wave_sync();
            }
            if constexpr (PHASE == 0)
            {
                if (g.mode != MODE_NONE)
                {
                    // the mask row's true entries inside the tile
                    const int64_t m1 = g.Mp[i + 1], mlo = lower_bound(g.Mj, g.Mp[i], m1, c0);
                    for (int64_t p = mlo + lane; p < m1 && g.Mj[p] < c0 + TL_W; p += 64)
                        if (g.mask_struct || mask_true(g.Mx, p, g.msize, g.m_iso))
                            atomicOr(&s_mask[wv][(g.Mj[p] - c0) >> 5], 1u << ((g.Mj[p] - c0) & 31));
                }
                wave_sync();
                int cnt = 0;
                if (lane < NW)
                {
                    uint32_t w = s_bits[wv][lane];
                    if (g.mode == MODE_MASK) w &= s_mask[wv][lane];
                    else if (g.mode == MODE_NOTMASK) w &= ~s_mask[wv][lane];
                    ((uint32_t *) t.bits)[at * NW + lane] = w;
                    cnt = __popc(w);
                }
                #pragma unroll
                for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
                if (lane == 0) t.seg[at] = cnt;
            }
            else
            {
                int64_t pos = g.Cp[i] + (t.seg[at] - t.seg[q * t.nt]);
                for (int x = 0; x < TL_W / 64; x++)
                {
                    const unsigned long long w = t.bits[at * (TL_W / 64) + x];
                    if ((w >> lane) & 1ull)
                    {
                        const int64_t p = pos + __popcll(w & ((1ull << lane) - 1ull));
                        g.Ci[p] = c0 + x * 64 + lane;
                        if constexpr (VALS) ((Z *) g.Cx)[p] = s_acc[wv][x * 64 + lane];
                    }
                    pos += __popcll(w);
                }
            }
            wave_sync();
        }
    }
}

__global__ __launch_bounds__(TL_NT) void k_sx_tile_rows(SxArgs g, TileArgs t)
{
    for (int64_t q = (int64_t) blockIdx.x * TL_NT + threadIdx.x; q < t.T; q += (int64_t) gridDim.x * TL_NT)
        g.Cp[tl_row(t, q)] = t.seg[(q + 1) * t.nt] - t.seg[q * t.nt];
}

} // namespace gm
