// gm_saxpy3.hip: row-wise Gustavson/hash SpGEMM, C = A*B, C<M> = A*B,
// C<!M> = A*B (the reference's saxpy3 method).
//
// Reference: Source/mxm/GB_AxB_saxpy3.c:119-700 (driver: flop count, tasks,
// symbolic, numeric), GB_AxB_saxpy3_flopcount.c:81-478,
// GB_AxB_saxpy3_symbolic.c + factory/GB_AxB_saxpy3_symbolic_template.c
// (phase1 counts), template/GB_AxB_saxpy3_template.c (numeric), coarse hash
// phase5 (GB_AxB_saxpy3_coarseHash_phase5.c:22-93) for the accumulation order.
//
// Layout: all operands CSR in HBM.  C(i,:) = (+)_k A(i,k) (x) B(k,:).
//
//  flops   eight lanes per row (the workgroup for a long row of A, the device
//          for few rows): f = sum |B(k,:)|, table size t = f (or
//          min(f, |M(i,:)|) for C<M>, and <= ncols).  Rows are binned:
//            single  |A(i,:)| == 1: C(i,:) is B(k,:) filtered by the mask,
//                    already sorted; no hash table at all
//            wave S  t <= 64   : one wavefront, 128-slot LDS table
//            wave L  t <= 512  : one wavefront, 1024-slot LDS table
//            block   t <= 2048 : one 256-thread workgroup, 4096-slot table
//            heavy   larger    : dealt out by k_sx_classify to tiles of C's
//                    columns in LDS (gm_sx_tile.h), to dense HBM tables that
//                    the whole device updates (gm_sx_push.h), or to one
//                    workgroup with a table of 2^ceil(log2 2t) slots in HBM
//                    (sub-allocated by an atomic bump)
//  symbolic  per row, hash-insert the allowed column indices, count new keys
//            -> Cp[i]; device exclusive scan -> row pointers, nnz(C).
//  numeric   the same inserts plus values; flops are enumerated in the
//            reference's sequential order (k ascending over A(i,:), then j
//            ascending over B(k,:)).  fp64 sums apply them in that order (lanes
//            that meet in a column go lowest first, wavefronts in turn), so
//            they equal the reference's coarse-task sums bit for bit; where
//            any order gives the same result (SX_ANY_ORDER) updates are
//            atomics, and ANY keeps the largest k, the last writer, as
//            GB_HX_UPDATE "z = t" does.
//            Rows are then sorted in LDS (rank count / bitonic) and written
//            to C: C is returned with sorted rows.
//  Masks     M(i,j) is tested by binary search in the sorted row M(i,:).
//
// Hash: multiplicative (Fibonacci) hashing of the 31-bit column index,
// linear probing, EMPTY = 0xffffffff.  Column indices are < 2^31-1.

#include "gm_internal.h"
#include "gm_block.h"
#include <cstring>

namespace gm
{

constexpr int SX_NT = 256;
constexpr uint32_t SX_EMPTY = 0xffffffffu;
// BIN_HVY collects the rows beyond the LDS tables; k_sx_classify deals them out
// to BIN_GLB (a hash table each), BIN_DNS (products spread over the device) and
// BIN_TIL (tiles of columns)
enum { BIN_SINGLE = 0, BIN_WS = 1, BIN_WL = 2, BIN_BLK = 3, BIN_GLB = 4, BIN_DNS = 5, BIN_HVY = 6, BIN_TIL = 7,
       SX_NBINS = 8 };
// counters: the bins, then
enum { CNT_SLOTS = 8,       // table slots of BIN_GLB
       CNT_BIGSUM = 9,      // entries of the big rows (symbolic)
       CNT_SMALL = 10,      // flops of the small rows
       CNT_HFLOPS = 11,     // flops of BIN_HVY
       CNT_NNZA = 12,       // nnz(A)
       CNT_BIGT = 13,       // most entries the big rows can have
       CNT_TILF = 14,       // BIN_TIL's very heavy rows (at the list's front; the others from its back)
       CNT_TILA = 15,       // A's entries in BIN_TIL's rows
       CNT_TILB = 22,       // BIN_TIL's other rows
       CNT_MAXLEN = 16,     // k_sx_maxlen's six results
       SX_NCNT = 32 };
enum { MODE_NONE = 0, MODE_MASK = 1, MODE_NOTMASK = 2 };

struct SxArgs
{
    int64_t m, n;
    const int64_t *Ap, *Aj;
    const void *Ax;
    int32_t a_iso;
    const int64_t *Bp, *Bj;
    const void *Bx;
    int32_t b_iso;
    const int64_t *Mp, *Mj;
    const void *Mx;
    int32_t msize, m_iso, mask_struct, mode;
    int64_t *Cp;
    int64_t *Ci;
    void *Cx;
    uint32_t *rows;               // SX_NBINS x ls row ids, or NULL: rows are only counted
    int64_t ls;
    unsigned long long *cnt;      // bin counters and totals (CNT_*)
    int64_t *hflops;              // per BIN_HVY row: its flops
    const unsigned long long *rowf;   // NULL, or the rows' flops (few-row A)
    int64_t *gtab_off;            // per global-bin row: offset of its table
    int32_t *gtab_log2;           // per global-bin row: log2 of its table size
    uint32_t *gkeys;
    void *gvals;
    uint64_t *glist;
    int64_t ws_max, wl_max, blk_max;
    // B's entries as 16-byte (column, value bits) pairs, or null: one B row
    // of the gather then spans one contiguous range instead of two.  With
    // rec_lg >= 0 they are B's row records instead (row k at k << rec_lg,
    // its length in the top byte of the first record's column)
    const int64_t *Bjx;
    int32_t rec_lg;
    // row tables: 0 the reference's rule (a table that holds every column of
    // C is indexed by the column itself, Gustavson's dense workspace; a
    // global-bin row whose hash table would be at least ncols/12 slots, or
    // whose flops reach ncols/2, gets such a table), 1 always hash
    // (GxB_AxB_HASH), 2 dense wherever a table holds every column or a
    // global-bin row's dense table is at most 16 times its hash table
    // (GxB_AxB_GUSTAVSON)
    int32_t table;
};

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint32_t sx_hash(uint32_t key, int logT)
{
    return (key * 0x9E3779B1u) >> (32 - logT);
}

// Is column j allowed by the mask for row i?  M(i,:) is [pm0, pm1).
__device__ __forceinline__ bool sx_mask_ok(const SxArgs &g, int64_t pm0, int64_t pm1, int64_t j)
{
    if (g.mode == MODE_NONE) return true;
    const int64_t q = lower_bound(g.Mj, pm0, pm1, j);
    bool in = (q < pm1) && (g.Mj[q] == j);
    if (in && !g.mask_struct) in = mask_true(g.Mx, q, g.msize, g.m_iso);
    return (g.mode == MODE_MASK) ? in : !in;
}

// insert key; returns its slot and whether this call created it.  dense: the
// table has a slot for every column, the key's own (no probing happens)
__device__ __forceinline__ int32_t sx_insert(uint32_t *keys, int logT, uint32_t key, bool &created,
                                             bool dense)
{
    const uint32_t mask = (1u << logT) - 1u;
    uint32_t h = dense ? key : sx_hash(key, logT);
    created = false;
    while (true)
    {
        uint32_t k = keys[h];
        if (k == key) return (int32_t) h;
        if (k == SX_EMPTY)
        {
            uint32_t prev = atomicCAS(&keys[h], SX_EMPTY, key);
            if (prev == SX_EMPTY) { created = true; return (int32_t) h; }
            if (prev == key) return (int32_t) h;
        }
        h = (h + 1) & mask;
    }
}

// Semirings whose updates of one entry may come in any order with the same
// bits: integer sums, MIN, MAX, and ANY with the inner index, whose last
// writer is the largest k.  fp64 sums keep the flop order.
template <class S>
constexpr bool SX_ANY_ORDER = S::add == GM_ADD_MIN || S::add == GM_ADD_MAX || S::any_min_k || S::iso_out ||
                              (S::add == GM_ADD_PLUS && !std::is_same<typename S::Z, double>::value);

// what an accumulator of the any-order updates holds before its first product:
// the identity, or for fp64 MIN / MAX the NaN that the updates below replace
// with any number, so that products which are all NaN leave a NaN and not an
// infinity (as an entry's first product does elsewhere, which fmin / fmax
// then keep only among NaNs)
template <class S>
__device__ __forceinline__ typename S::Z sx_cell0()
{
    if constexpr (std::is_same<typename S::Z, double>::value && (S::add == GM_ADD_MIN || S::add == GM_ADD_MAX))
        return __builtin_bit_cast(double, S::add == GM_ADD_MIN ? 0x7ff8000000000000ull : 0xfff8000000000000ull);
    else return S::identity();
}

// can t change a cell that holds cur?  A plain read of the cell may be stale:
// it is then an earlier value, which t may seem to change and does not.  The
// zeros are told apart by their bits, so that -0 is the smaller one whichever
// comes first.
template <class S>
__device__ __forceinline__ bool sx_changes(typename S::Z cur, typename S::Z t)
{
    if constexpr (std::is_same<typename S::Z, double>::value)
    {
        if (S::add == GM_ADD_MIN ? cur < t : cur > t) return false;
        return __builtin_bit_cast(uint64_t, cur) != __builtin_bit_cast(uint64_t, t);
    }
    else return S::upd(cur, t) != cur;
}

// *p = *p (+) t, atomically (SX_ANY_ORDER semirings; *p starts at sx_cell0)
template <class S>
__device__ __forceinline__ void sx_atomic_upd(typename S::Z *p, typename S::Z t)
{
    using Z = typename S::Z;
    static_assert(SX_ANY_ORDER<S>, "fp64 sums are ordered");
    if constexpr (S::iso_out) return;
    else if constexpr (std::is_same<Z, double>::value)
    {
        // fmin / fmax of the bits: a NaN changes nothing; doubles of one sign
        // order as their bits do (negative ones in reverse), with sx_cell0
        // beyond the infinity of its sign
        if (t != t) return;
        const long long b = __builtin_bit_cast(long long, t);
        const bool neg = b < 0;
        if ((S::add == GM_ADD_MIN) != neg)
        {
            if (S::add == GM_ADD_MIN) atomicMin((long long *) p, b);
            else atomicMin((unsigned long long *) p, (unsigned long long) b);
        }
        else
        {
            if (S::add == GM_ADD_MIN) atomicMax((unsigned long long *) p, (unsigned long long) b);
            else atomicMax((long long *) p, b);
        }
    }
    else if constexpr (S::add == GM_ADD_PLUS)
    {
        if constexpr (sizeof(Z) == 8) atomicAdd((unsigned long long *) p, (unsigned long long) t);
        else atomicAdd((unsigned int *) p, (unsigned int) t);
    }
    else if constexpr (S::add == GM_ADD_MIN)
    {
        if constexpr (sizeof(Z) == 8) atomicMin((long long *) p, (long long) t);
        else atomicMin((int *) p, (int) t);
    }
    else
    {
        if constexpr (sizeof(Z) == 8) atomicMax((long long *) p, (long long) t);
        else atomicMax((int *) p, (int) t);
    }
}

// vals[slot] = vals[slot] (+) t for the wavefront's lanes with slot >= 0, in
// lane order where lanes share a slot.  Each round the lowest lane of every
// owner cell (OWN cells, all ones between calls) applies its term, so a
// wavefront takes as many rounds as lanes meet in one cell, two or three
// mostly, where a walk over all 64 lanes always pays 64 steps (a row of 65536
// entries times 1.8M entries, fp64: 117 -> 49 ms on one workgroup).
constexpr int SX_OWN = 128;
template <class S>
__device__ __forceinline__ void sx_ordered_upd(typename S::Z *vals, int32_t slot, typename S::Z t, uint32_t *own)
{
    const uint32_t lane = threadIdx.x & 63;
    uint32_t *o = own + ((uint32_t) slot & (SX_OWN - 1));
    bool pend = slot >= 0;
    while (__ballot(pend))
    {
        if (pend) atomicMin(o, lane);
        wave_sync();
        const bool win = pend && *(volatile uint32_t *) o == lane;
        wave_sync();
        if (win)
        {
            vals[slot] = S::upd(vals[slot], t);
            *o = 0xffffffffu;
            pend = false;
        }
        wave_sync();
    }
}

} // namespace gm

#include "gm_sx_push.h"
#include "gm_sx_pull.h"
#include "gm_sx_tile.h"

namespace gm
{

//------------------------------------------------------------------------------
// team-of-TG helpers (TG lanes of one wavefront work on one row)
//------------------------------------------------------------------------------

constexpr int TG = 8;          // lanes per row in the flop-count and fused kernels
constexpr int FEW_ROWS = 256;             // A with at most this many rows: k_sx_rowflops
constexpr int64_t FLOPS_TEAM_MAX = 256;   // longer rows of A: counted by the workgroup
constexpr int FMAX = 64;       // largest flop count of a "small" row

template <class T>
__device__ __forceinline__ T team_incl_scan(T v)
{
    const int sub = threadIdx.x & (TG - 1);
    #pragma unroll
    for (int off = 1; off < TG; off <<= 1)
    {
        T u = __shfl_up(v, off, TG);
        if (sub >= off) v += u;
    }
    return v;
}

template <class T>
__device__ __forceinline__ T team_sum(T v)
{
    #pragma unroll
    for (int off = 1; off < TG; off <<= 1) v += __shfl_xor(v, off, TG);
    return v;
}

//------------------------------------------------------------------------------
// max row lengths of A and B (decides whether every row is "small"):
// out[0] / out[1]; and nnz(A) / nnz(B) in out[2] / out[5], so that one copy
// brings all four to the host
//------------------------------------------------------------------------------

__global__ __launch_bounds__(SX_NT) void k_sx_maxlen(const int64_t *__restrict__ Ap, int64_t m,
                                                     const int64_t *__restrict__ Bp, int64_t kb,
                                                     unsigned long long *out)
{
    __shared__ unsigned long long s[2][SX_NT / 64];
    unsigned long long ma = 0, mb = 0;
    const int64_t lim = m > kb ? m : kb;
    if (blockIdx.x == 0 && threadIdx.x == 0)
    {
        out[2] = (unsigned long long) Ap[m];
        out[5] = (unsigned long long) Bp[kb];
    }
    // four consecutive rows per thread and pass, so that one pass of a
    // modest grid has all of its loads in flight together
    for (int64_t i0 = ((int64_t) blockIdx.x * SX_NT + threadIdx.x) * 4; i0 < lim;
         i0 += (int64_t) gridDim.x * SX_NT * 4)
    {
        #pragma unroll
        for (int u = 0; u < 4; u++)
        {
            const int64_t i = i0 + u;
            if (i < m) { unsigned long long l = (unsigned long long) (Ap[i + 1] - Ap[i]); ma = l > ma ? l : ma; }
            if (i < kb) { unsigned long long l = (unsigned long long) (Bp[i + 1] - Bp[i]); mb = l > mb ? l : mb; }
        }
    }
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1)
    {
        unsigned long long ua = __shfl_xor(ma, off, 64), ub = __shfl_xor(mb, off, 64);
        ma = ua > ma ? ua : ma;
        mb = ub > mb ? ub : mb;
    }
    if ((threadIdx.x & 63) == 0) { s[0][threadIdx.x >> 6] = ma; s[1][threadIdx.x >> 6] = mb; }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        for (int w = 1; w < SX_NT / 64; w++)
        {
            ma = s[0][w] > ma ? s[0][w] : ma;
            mb = s[1][w] > mb ? s[1][w] : mb;
        }
        // an atomic only where this block raises the maximum seen so far
        // (a stale read only costs an atomic that was not needed)
        const unsigned long long ca = __hip_atomic_load(&out[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long cb = __hip_atomic_load(&out[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (ma > ca) atomicMax(&out[0], ma);
        if (mb > cb) atomicMax(&out[1], mb);
    }
}

//------------------------------------------------------------------------------
// flops + binning: TG lanes per row (coalesced reads of A(i,:) and of the
// B row pointers it names).  Rows with f <= fs are "small"; their flops are
// summed into cnt[CNT_SMALL] (capacity for the fused kernel) and they are listed in
// BIN_WS (used only when the fused kernel is not).  Larger rows go to the
// single / wave1024 / block4096 / global bins.
//------------------------------------------------------------------------------

// A row of f flops from la entries of A is cut into tiles (gm_sx_tile.h) when
// finding the parts of B's rows costs less than a hash table's inserts and sort:
// la * (n / TL_W) <= 4 f (n = 40009: rows whose B rows hold 10 entries or more
// on average), with 16 flops per tile at least.
__device__ __forceinline__ bool sx_tiled(const SxArgs &g, int64_t f, int64_t la)
{
    const int64_t nt = (g.n + TL_W - 1) / TL_W;
    return g.table != 1 && f >= 16 * nt && (double) la * (double) nt <= 4.0 * (double) f;
}

__global__ __launch_bounds__(SX_NT) void k_sx_flops(SxArgs g, int64_t fs, int list_small)
{
    __shared__ unsigned int s_bc[SX_NBINS];
    __shared__ unsigned long long s_base[SX_NBINS];
    __shared__ unsigned long long s_red[SX_NT / 64 + 1];
    __shared__ int s_long[SX_NT / TG], s_nlong;
    const int sub = threadIdx.x & (TG - 1);
    unsigned long long fsum = 0;          // flops of this thread's small rows
    unsigned long long bsum = 0;          // size bounds of its big rows
    if (blockIdx.x == 0 && threadIdx.x == 0) g.cnt[CNT_NNZA] = (unsigned long long) g.Ap[g.m];
    for (int64_t base = (int64_t) blockIdx.x * (SX_NT / TG); base < g.m;
         base += (int64_t) gridDim.x * (SX_NT / TG))
    {
        const int64_t i = base + threadIdx.x / TG;
        int64_t f = 0, a0 = 0, a1 = 0;
        if (threadIdx.x == 0) s_nlong = 0;
        __syncthreads();
        if (i < g.m)
        {
            a0 = g.Ap[i];
            a1 = g.Ap[i + 1];
            if (g.rowf) f = sub == 0 ? (int64_t) g.rowf[i] : 0;
            else if (a1 - a0 > FLOPS_TEAM_MAX)
            {
                if (sub == 0) s_long[atomicAdd(&s_nlong, 1)] = threadIdx.x / TG;
            }
            else
                for (int64_t e = a0 + sub; e < a1; e += TG)
                {
                    const int64_t k = g.Aj[e];
                    f += g.Bp[k + 1] - g.Bp[k];
                }
        }
        __syncthreads();
        // the workgroup takes the tile's long rows together
        for (int q = 0; q < s_nlong; q++)
        {
            const int64_t r = base + s_long[q], r1 = g.Ap[r + 1];
            unsigned long long fl = 0;
            #pragma unroll 4
            for (int64_t e = g.Ap[r] + threadIdx.x; e < r1; e += SX_NT)
            {
                const int64_t k = g.Aj[e];
                fl += (unsigned long long) (g.Bp[k + 1] - g.Bp[k]);
            }
            const unsigned long long tot = block_sum<unsigned long long, SX_NT>(fl, s_red);
            if (r == i && sub == 0) f = (int64_t) tot;
        }
        f = team_sum<int64_t>(f);
        int bin = -1;
        int64_t t = f;
        if (threadIdx.x < SX_NBINS) s_bc[threadIdx.x] = 0;
        if (i < g.m && sub == 0)
        {
            if (g.mode == MODE_MASK)
            {
                const int64_t mi = g.Mp[i + 1] - g.Mp[i];
                if (mi < t) t = mi;
            }
            if (t > g.n) t = g.n;
            if (f == 0 || t == 0) g.Cp[i] = 0;
            else if (f <= fs) { bin = list_small ? BIN_WS : -1; fsum += (unsigned long long) f; }
            else if (a1 - a0 == 1) bin = BIN_SINGLE;
            else if (t <= g.wl_max) bin = BIN_WL;
            else if (t <= g.blk_max && !sx_tiled(g, f, a1 - a0)) bin = BIN_BLK;
            else bin = BIN_HVY;
            if (f > fs && t > 0) bsum += (unsigned long long) t;
        }
        __syncthreads();
        // block-aggregated appends: LDS counters, one global atomic per bin
        unsigned int local = 0;
        if (bin >= 0) local = atomicAdd(&s_bc[bin], 1u);
        __syncthreads();
        if (threadIdx.x < SX_NBINS && s_bc[threadIdx.x] > 0)
            s_base[threadIdx.x] = atomicAdd(&g.cnt[threadIdx.x], (unsigned long long) s_bc[threadIdx.x]);
        __syncthreads();
        if (bin >= 0)
        {
            const unsigned long long slot = s_base[bin] + local;
            if (g.rows) g.rows[(int64_t) bin * g.ls + (int64_t) slot] = (uint32_t) i;
            if (bin == BIN_HVY)
            {
                if (g.rows) g.hflops[slot] = f;
                atomicAdd(&g.cnt[CNT_HFLOPS], (unsigned long long) f);
            }
        }
        __syncthreads();
    }
    // one atomic per workgroup for each sum
    fsum = block_sum<unsigned long long, SX_NT>(fsum, s_red);
    bsum = block_sum<unsigned long long, SX_NT>(bsum, s_red);
    if (threadIdx.x == 0)
    {
        if (fsum) atomicAdd(&g.cnt[CNT_SMALL], fsum);
        if (bsum) atomicAdd(&g.cnt[CNT_BIGT], bsum);
    }
}

// Deals the heavy rows out, by flops f, entries la of A(i,:) and the columns n:
//   dense table (BIN_DNS; the semiring allows any order, dmax rows at most): a
//     row with more than 1/512 of all heavy flops, on which one workgroup
//     would outlast the others, and at least n/128 flops, so that the table's
//     clearing and compaction stay below its updates; or a row whose own
//     workgroup (50 ns a flop) would take longer than tables for all the
//     heavy rows (2.5e-6 us a column): 20000 f >= heavy rows * n (second BFS
//     level of 64 searches, RMAT 20: 1.34 -> 0.90 ms)
//   tiles (BIN_TIL, tmax rows at most): sx_tiled, or for a very heavy fp64 row,
//     whose order the dense table does not keep, la * (n / TL_W) <= 64 f
//   dense table again: at least n/4 flops
//   else a hash table of 2^ceil(log2(2t)) slots, load factor <= 1/2, or a
//     dense one of 2^ceil(log2(ncols)) slots (SxArgs::table)
__global__ __launch_bounds__(SX_NT) void k_sx_classify(SxArgs g, int64_t *dflops, int64_t dmax, int64_t tmax)
{
    const int64_t count = (int64_t) g.cnt[BIN_HVY];
    const double total = (double) g.cnt[CNT_HFLOPS];
    const int64_t nt = (g.n + TL_W - 1) / TL_W;
    for (int64_t q = (int64_t) blockIdx.x * SX_NT + threadIdx.x; q < count; q += (int64_t) gridDim.x * SX_NT)
    {
        const uint32_t i = g.rows[(int64_t) BIN_HVY * g.ls + q];
        const int64_t f = g.hflops[q], la = g.Ap[i + 1] - g.Ap[i];
        const bool most = (double) f * 512 > total;
        const bool push = dmax > 0 && g.table != 1;
        const bool tile = tmax > 0 && g.table != 1 &&
                          (sx_tiled(g, f, la) ||
                           (!push && most && f >= 16 * nt && (double) la * (double) nt <= 64.0 * (double) f));
        if (push && ((most && f >= g.n / 128) || (!tile && f >= g.n / 4) ||
                     20000.0 * (double) f >= (double) count * (double) g.n))
        {
            const int64_t d = (int64_t) atomicAdd(&g.cnt[BIN_DNS], 1ull);
            if (d < dmax)
            {
                g.rows[(int64_t) BIN_DNS * g.ls + d] = i;
                dflops[d] = f;
                continue;
            }
        }
        else if (tile)
        {
            if ((int64_t) atomicAdd(&g.cnt[BIN_TIL], 1ull) < tmax)
            {
                if (most) g.rows[(int64_t) BIN_TIL * g.ls + atomicAdd(&g.cnt[CNT_TILF], 1ull)] = i;
                else g.rows[(int64_t) (BIN_TIL + 1) * g.ls - 1 - atomicAdd(&g.cnt[CNT_TILB], 1ull)] = i;
                atomicAdd(&g.cnt[CNT_TILA], (unsigned long long) la);
                continue;
            }
        }
        int64_t t = f;
        if (g.mode == MODE_MASK && g.Mp[i + 1] - g.Mp[i] < t) t = g.Mp[i + 1] - g.Mp[i];
        if (t > g.n) t = g.n;
        int lg = ilog2_ceil(2 * t);
        const int lgd = ilog2_ceil(g.n);
        const bool dn = (g.table == 0 && (((int64_t) 1 << lg) >= g.n / 12 || t >= g.n / 2)) ||
                        (g.table == 2 && lgd <= lg + 4);
        if (dn && lgd > lg) lg = lgd;
        const int64_t slot = (int64_t) atomicAdd(&g.cnt[BIN_GLB], 1ull);
        g.rows[(int64_t) BIN_GLB * g.ls + slot] = i;
        g.gtab_off[slot] = (int64_t) atomicAdd(&g.cnt[CNT_SLOTS], 1ull << lg);
        g.gtab_log2[slot] = lg;
    }
}

// sum of the symbolic counts of the rows in the big bins -> cnt[CNT_BIGSUM]
__global__ __launch_bounds__(SX_NT) void k_sx_sum_big(SxArgs g, int64_t dmax)
{
    __shared__ unsigned long long s_red[SX_NT / 64];
    unsigned long long sum = 0;
    // (the tiled rows' two lists: from the front and from the back)
    const int bins[7] = {BIN_SINGLE, BIN_WL, BIN_BLK, BIN_GLB, BIN_DNS, BIN_TIL, BIN_TIL};
    for (int b = 0; b < 7; b++)
    {
        int64_t count = (int64_t) g.cnt[b < 5 ? bins[b] : b == 5 ? CNT_TILF : CNT_TILB];
        if (bins[b] == BIN_DNS && count > dmax) count = dmax;
        const uint32_t *list = g.rows + (int64_t) bins[b] * g.ls;
        if (b == 6) list += g.ls - count;
        for (int64_t q = (int64_t) blockIdx.x * SX_NT + threadIdx.x; q < count;
             q += (int64_t) gridDim.x * SX_NT)
            sum += (unsigned long long) g.Cp[list[q]];
    }
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        unsigned long long tsum = 0;
        for (int w = 0; w < SX_NT / 64; w++) tsum += s_red[w];
        if (tsum) atomicAdd(&g.cnt[CNT_BIGSUM], tsum);
    }
}

//------------------------------------------------------------------------------
// single-entry rows: C(i,:) = A(i,k) (x) B(k,:) filtered by the mask
//------------------------------------------------------------------------------

constexpr int SINGLE_UN = 8;
template <class S, int PHASE>
__global__ __launch_bounds__(SX_NT) void k_sx_single(SxArgs g)
{
    using Z = typename S::Z;
    const int lane = threadIdx.x & 63;
    const int64_t count = (int64_t) g.cnt[BIN_SINGLE];
    const uint32_t *list = g.rows + (int64_t) BIN_SINGLE * g.ls;
    for (int64_t q = (int64_t) blockIdx.x * 4 + (threadIdx.x >> 6); q < count;
         q += (int64_t) gridDim.x * 4)
    {
        const int64_t i = list[q];
        const int64_t e = g.Ap[i];
        const int64_t k = g.Aj[e];
        const int64_t b0 = g.Bp[k], b1 = g.Bp[k + 1];
        const int64_t pm0 = g.Mp ? g.Mp[i] : 0, pm1 = g.Mp ? g.Mp[i + 1] : 0;
        if (PHASE == 0 && g.mode == MODE_NONE)
        {
            if (lane == 0) g.Cp[i] = b1 - b0;
            continue;
        }
        const Z av = S::geta((const Z *) g.Ax, e, g.a_iso);
        const int64_t cbase = PHASE ? g.Cp[i] : 0;
        const int64_t cend = PHASE ? g.Cp[i + 1] : 0;
        int64_t run = 0;
        // SINGLE_UN windows of 64 entries, their reads out together
        for (int64_t c0 = b0; c0 < b1; c0 += 64 * SINGLE_UN)
        {
            int64_t j[SINGLE_UN];
            Z x[SINGLE_UN];
            bool ok[SINGLE_UN];
            #pragma unroll
            for (int u = 0; u < SINGLE_UN; u++)
            {
                const int64_t pb = c0 + u * 64 + lane;
                ok[u] = pb < b1;
                j[u] = g.Bj[ok[u] ? pb : b1 - 1];
                x[u] = Z(0);
                if constexpr (PHASE == 1 && !S::iso_out) x[u] = S::geta((const Z *) g.Bx, ok[u] ? pb : b1 - 1, g.b_iso);
            }
            #pragma unroll
            for (int u = 0; u < SINGLE_UN; u++) ok[u] = ok[u] && sx_mask_ok(g, pm0, pm1, j[u]);
            #pragma unroll
            for (int u = 0; u < SINGLE_UN; u++)
            {
                const unsigned long long bal = __ballot(ok[u]);
                if (PHASE == 1 && ok[u])
                {
                    const int64_t pos = cbase + run + __popcll(bal & ((1ull << lane) - 1ull));
                    if (pos < cend)
                    {
                        g.Ci[pos] = j[u];
                        if constexpr (!S::iso_out) ((Z *) g.Cx)[pos] = S::mul(av, x[u], k);
                    }
                }
                run += __popcll(bal);
            }
        }
        if (PHASE == 0 && lane == 0) g.Cp[i] = run;
    }
}

//------------------------------------------------------------------------------
// one row on a team of NT lanes (NT = 64: one wavefront; NT = 256: one
// workgroup).  keys/vals/list are the row's table (LDS or HBM), logT its size.
//------------------------------------------------------------------------------

template <int NT>
__device__ __forceinline__ void team_sync()
{
    if constexpr (NT == 64) wave_sync(); else __syncthreads();
}

// bitonic sort of list[0..P) (P a power of two), ascending
template <int NT>
__device__ void team_bitonic(uint64_t *list, int64_t P, int tid)
{
    for (int64_t k = 2; k <= P; k <<= 1)
    {
        for (int64_t jj = k >> 1; jj > 0; jj >>= 1)
        {
            for (int64_t t = tid; t < P / 2; t += NT)
            {
                const int64_t lo = 2 * t - (t & (jj - 1));
                const int64_t hi = lo + jj;
                const bool asc = (lo & k) == 0;
                const uint64_t a = list[lo], b = list[hi];
                if ((a > b) == asc) { list[lo] = b; list[hi] = a; }
            }
            team_sync<NT>();
        }
    }
}

template <class S, int NT, int PHASE>
__device__ void sx_row(const SxArgs &g, int64_t i, uint32_t *keys, typename S::Z *vals,
                       uint64_t *list, int logT, int64_t *s_pre, int64_t *s_k, int64_t *s_bs,
                       typename S::Z *s_av, uint32_t *own, int64_t *s_red)
{
    using Z = typename S::Z;
    constexpr int NWV = NT / 64;
    const int tid = (NT == 64) ? (threadIdx.x & 63) : threadIdx.x;
    const int lane = threadIdx.x & 63;
    const int wv = (NT == 64) ? 0 : (threadIdx.x >> 6);
    const int64_t T = (int64_t) 1 << logT;
    const bool dense = g.table != 1 && T >= g.n;    // Gustavson: index by column

    for (int64_t t = tid; t < T; t += NT)
    {
        keys[t] = SX_EMPTY;
        if (PHASE) vals[t] = SX_ANY_ORDER<S> ? sx_cell0<S>() : S::identity();
    }
    if constexpr (PHASE == 1 && !SX_ANY_ORDER<S>)
        for (int t = lane; t < SX_OWN; t += 64) own[t] = 0xffffffffu;
    team_sync<NT>();

    const int64_t a0 = g.Ap[i], a1 = g.Ap[i + 1];
    const int64_t pm0 = g.Mp ? g.Mp[i] : 0, pm1 = g.Mp ? g.Mp[i + 1] : 0;
    int64_t nnew = 0;

    for (int64_t ea = a0; ea < a1; ea += NT)
    {
        // stage up to NT entries of A(i,:) with their B-row extents
        const int64_t e = ea + tid;
        int64_t len = 0;
        if (e < a1)
        {
            const int64_t k = g.Aj[e];
            const int64_t bs = g.Bp[k];
            len = g.Bp[k + 1] - bs;
            s_k[tid] = k;
            s_bs[tid] = bs;
            if (PHASE) s_av[tid] = S::geta((const Z *) g.Ax, e, g.a_iso);
        }
        int64_t total;
        int64_t pre;
        if constexpr (NT == 64)
        {
            const int64_t inc = wave_inclusive_scan<int64_t>(len);
            pre = inc - len;
            total = __shfl(inc, 63, 64);
        }
        else
        {
            pre = block_exclusive_scan<int64_t, NT>(len, s_red, &total);
        }
        s_pre[tid] = pre;
        const int64_t nA = (a1 - ea) < NT ? (a1 - ea) : NT;
        team_sync<NT>();

        for (int64_t f0 = 0; f0 < total; f0 += NT)
        {
            const int64_t f = f0 + tid;
            int32_t slot = -1;
            bool created = false;
            Z tv = S::identity();
            if (f < total)
            {
                // owning A entry: last index with s_pre <= f
                int lo = 0, hi = (int) nA - 1;
                while (lo < hi)
                {
                    const int mid = (lo + hi + 1) >> 1;
                    if (s_pre[mid] <= f) lo = mid; else hi = mid - 1;
                }
                const int64_t pb = s_bs[lo] + (f - s_pre[lo]);
                const int64_t j = g.Bj[pb];
                if (sx_mask_ok(g, pm0, pm1, j))
                {
                    if (PHASE)
                        tv = S::mul(s_av[lo], S::geta((const Z *) g.Bx, pb, g.b_iso), s_k[lo]);
                    slot = sx_insert(keys, logT, (uint32_t) j, created, dense);
                }
            }
            if (PHASE == 0)
            {
                nnew += created ? 1 : 0;
            }
            else
            {
                // updates in any order need no turns and no barrier; fp64
                // sums apply in flop order: wavefront by wavefront
                if constexpr (SX_ANY_ORDER<S>)
                {
                    if (slot >= 0) sx_atomic_upd<S>(&vals[slot], tv);
                }
                else
                {
                    for (int w = 0; w < NWV; w++)
                    {
                        if (w == wv) sx_ordered_upd<S>(vals, slot, tv, own);
                        team_sync<NT>();
                    }
                }
            }
        }
        team_sync<NT>();
    }

    if (PHASE == 0)
    {
        int64_t tot;
        if constexpr (NT == 64)
        {
            tot = wave_inclusive_scan<int64_t>(nnew);
            tot = __shfl(tot, 63, 64);
        }
        else
        {
            tot = block_sum<int64_t, NT>(nnew, s_red);
        }
        if (tid == 0) g.Cp[i] = tot;
        return;
    }

    // numeric: gather the row's keys, sort, write C(i,:)
    const int64_t cbase = g.Cp[i], c = g.Cp[i + 1] - cbase;
    int64_t run = 0;
    for (int64_t t0 = 0; t0 < T; t0 += NT)
    {
        const int64_t t = t0 + tid;
        const uint32_t k = (t < T) ? keys[t] : SX_EMPTY;
        const bool v = (k != SX_EMPTY);
        int64_t pos, cnt;
        if constexpr (NT == 64)
        {
            const unsigned long long bal = __ballot(v);
            pos = __popcll(bal & ((1ull << lane) - 1ull));
            cnt = __popcll(bal);
        }
        else
        {
            pos = block_exclusive_scan<int64_t, NT>(v ? 1 : 0, s_red, &cnt);
        }
        if (v && run + pos < c) list[run + pos] = ((uint64_t) k << 32) | (uint64_t) t;
        run += cnt;
    }
    team_sync<NT>();
    if (c <= 64 && NT == 64)
    {
        // rank by counting: keys in a row are distinct
        if (lane < c)
        {
            const uint64_t my = list[lane];
            int r = 0;
            for (int t = 0; t < c; t++) r += (list[t] < my) ? 1 : 0;
            g.Ci[cbase + r] = (int64_t) (my >> 32);
            if constexpr (!S::iso_out) ((Z *) g.Cx)[cbase + r] = vals[(uint32_t) my & (uint32_t) (T - 1)];
        }
        team_sync<NT>();
        return;
    }
    int64_t P = 1;
    while (P < c) P <<= 1;
    for (int64_t t = c + tid; t < P; t += NT) list[t] = ~0ull;
    team_sync<NT>();
    team_bitonic<NT>(list, P, tid);
    for (int64_t t = tid; t < c; t += NT)
    {
        const uint64_t w = list[t];
        g.Ci[cbase + t] = (int64_t) (w >> 32);
        if constexpr (!S::iso_out) ((Z *) g.Cx)[cbase + t] = vals[(uint32_t) w & (uint32_t) (T - 1)];
    }
    team_sync<NT>();
}

// one wavefront per row, LDS table of 2^LOGT slots; 4 rows per workgroup
template <class S, int LOGT, int PHASE>
__global__ __launch_bounds__(SX_NT) void k_sx_wave(SxArgs g, int bin)
{
    using Z = typename S::Z;
    constexpr int T = 1 << LOGT;
    constexpr int NWV = SX_NT / 64;
    __shared__ uint32_t s_keys[NWV][T];
    __shared__ Z s_vals[NWV][PHASE ? T : 1];
    __shared__ uint64_t s_list[NWV][PHASE ? T / 2 : 1];
    __shared__ int64_t s_pre[NWV][64], s_k[NWV][64], s_bs[NWV][64];
    __shared__ Z s_av[NWV][64];
    __shared__ uint32_t s_own[NWV][SX_OWN];
    const int wv = threadIdx.x >> 6;
    const int64_t count = (int64_t) g.cnt[bin];
    const uint32_t *list = g.rows + (int64_t) bin * g.ls;
    for (int64_t q = (int64_t) blockIdx.x * NWV + wv; q < count; q += (int64_t) gridDim.x * NWV)
    {
        sx_row<S, 64, PHASE>(g, (int64_t) list[q], s_keys[wv], s_vals[wv], s_list[wv], LOGT,
                             s_pre[wv], s_k[wv], s_bs[wv], s_av[wv], s_own[wv], nullptr);
    }
}

// one workgroup per row, LDS table of 2^LOGT slots
template <class S, int LOGT, int PHASE>
__global__ __launch_bounds__(SX_NT) void k_sx_block(SxArgs g)
{
    using Z = typename S::Z;
    constexpr int T = 1 << LOGT;
    __shared__ uint32_t s_keys[T];
    __shared__ Z s_vals[PHASE ? T : 1];
    __shared__ uint64_t s_list[PHASE ? T / 2 : 1];
    __shared__ int64_t s_pre[SX_NT], s_k[SX_NT], s_bs[SX_NT];
    __shared__ Z s_av[SX_NT];
    __shared__ uint32_t s_own[SX_NT / 64][SX_OWN];
    __shared__ int64_t s_red[SX_NT / 64 + 1];
    const int64_t count = (int64_t) g.cnt[BIN_BLK];
    const uint32_t *list = g.rows + (int64_t) BIN_BLK * g.ls;
    for (int64_t q = blockIdx.x; q < count; q += gridDim.x)
    {
        sx_row<S, SX_NT, PHASE>(g, (int64_t) list[q], s_keys, s_vals, s_list, LOGT,
                                s_pre, s_k, s_bs, s_av, s_own[threadIdx.x >> 6], s_red);
    }
}

// one workgroup per row, table in HBM
template <class S, int PHASE>
__global__ __launch_bounds__(SX_NT) void k_sx_global(SxArgs g)
{
    using Z = typename S::Z;
    __shared__ int64_t s_pre[SX_NT], s_k[SX_NT], s_bs[SX_NT];
    __shared__ Z s_av[SX_NT];
    __shared__ uint32_t s_own[SX_NT / 64][SX_OWN];
    __shared__ int64_t s_red[SX_NT / 64 + 1];
    const int64_t count = (int64_t) g.cnt[BIN_GLB];
    const uint32_t *list = g.rows + (int64_t) BIN_GLB * g.ls;
    for (int64_t q = blockIdx.x; q < count; q += gridDim.x)
    {
        const int64_t off = g.gtab_off[q];
        const int lg = g.gtab_log2[q];
        sx_row<S, SX_NT, PHASE>(g, (int64_t) list[q], g.gkeys + off, ((Z *) g.gvals) + off,
                                g.glist + off, lg, s_pre, s_k, s_bs, s_av, s_own[threadIdx.x >> 6], s_red);
    }
}

__global__ void k_sx_zero(unsigned long long *x, int n)
{
    if ((int) threadIdx.x < n) x[threadIdx.x] = 0;
}

__global__ void k_sx_iso_one(void *x, int size)
{
    if (threadIdx.x == 0 && blockIdx.x == 0)
    {
        uint8_t *b = (uint8_t *) x;
        for (int t = 0; t < size; t++) b[t] = 0;
        b[0] = 1;
    }
}

//------------------------------------------------------------------------------
// single-pass fused kernel for small rows (f <= fs <= 64)
//------------------------------------------------------------------------------
//
// A persistent grid takes tiles of FUSED_NT/TG = 64 consecutive rows in ticket
// order.  One team of TG = 8 lanes per row:
//   expand   the row's flops, in the reference's order (A(i,:) in chunks of
//            TG entries, B(k,:) in order), into LDS as sort keys
//            (j << 6 | flop index) plus values; masked-out flops stay at the
//            all-ones key
//   sort     bitonic sort of the keys (the flop index makes them unique and
//            keeps equal columns in flop order)
//   compress runs of one column are reduced in flop order, so fp64 sums are
//            the reference's sequential ascending-k sums and ANY keeps the
//            last writer
// Rows with f > fs ("big") were counted beforehand by the hash kernels; the
// tile only adds their counts to the scan.  The tile's output offset comes
// from a decoupled look-back over the previous tiles' published counts
// (status word: 2-bit flag | 62-bit count); then C(tile rows) is written with
// contiguous, coalesced stores, together with Cp.  Ticket order means a tile
// only waits on tiles already running; a bounded spin turns a lost
// predecessor into an error flag instead of a hang.

// B packed as (column, value bits) pairs for the fused kernel's gathers: for
// 8-byte values that the semiring reads
template <class S>
constexpr bool SX_PACK_OK = sizeof(typename S::Z) == 8 && !S::pattern;

__global__ __launch_bounds__(256) void k_sx_pack(const int64_t *__restrict__ Bj,
                                                 const int64_t *__restrict__ Bx, int64_t nnz,
                                                 longlong2 *__restrict__ out)
{
    for (int64_t e = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; e < nnz;
         e += (int64_t) gridDim.x * blockDim.x)
        out[e] = make_longlong2(Bj[e], Bx[e]);
}

// Row records of B (gm_csr_aux): slot s of row k at (k << lg) + s holds
// (column, value bits) of the row's s-th entry, or (0, 0) past its end; slot
// 0's column carries the row length in its top byte (columns < 2^56)
constexpr long long SX_REC_COL = (1ll << 56) - 1;
constexpr int SX_REC_MAX_LG = 4;          // rows of at most 16 entries

__global__ __launch_bounds__(256) void k_sx_rec_build(const int64_t *__restrict__ Bp,
                                                      const int64_t *__restrict__ Bj,
                                                      const int64_t *__restrict__ Bx, int64_t nrows,
                                                      int lg, longlong2 *__restrict__ out)
{
    const int64_t total = nrows << lg;
    const int64_t smask = ((int64_t) 1 << lg) - 1;
    for (int64_t t = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; t < total;
         t += (int64_t) gridDim.x * blockDim.x)
    {
        const int64_t k = t >> lg, sl = t & smask;
        const int64_t p0 = Bp[k], len = Bp[k + 1] - p0;
        long long c = 0, v = 0;
        if (sl < len) { c = Bj[p0 + sl]; v = Bx[p0 + sl]; }
        if (sl == 0) c |= (long long) ((unsigned long long) len << 56);
        out[t] = make_longlong2(c, v);
    }
}

// threads of a fused-kernel workgroup: 64-row tiles halve the look-backs of
// 32-row ones (ER 2^20: 0.861 against 0.899 ms; 16-row tiles 1.32 ms)
constexpr int FUSED_NT = 512;
constexpr int SX_FUSED_WAVES = 4;
constexpr int FUSED_ROWS = FUSED_NT / TG;  // rows of a tile
constexpr unsigned long long LB_AGG = 1ull << 62;
constexpr unsigned long long LB_PRE = 2ull << 62;
constexpr unsigned long long LB_MASK = (1ull << 62) - 1;
constexpr int LB_SPIN_LIMIT = 1 << 22;
constexpr int LB_WIN = 1;            // look-back window: LB_WIN x 64 predecessors (one wavefront's loads per step measured fastest)

// K: the sort key type, (j << 6 | flop).  32-bit keys (columns < 2^26) halve
// the key LDS and the sort's shuffles and registers.
// The bound's second argument is the wavefronts per SIMD asked for; with
// 32-bit keys SX_FUSED_WAVES, so that a workgroup waiting in its look-back
// is covered by the others on the CU; 64-bit keys double the key LDS and ask
// for three.
// PK: 0 B read from Bp/Bj/Bx, 1 from the packed pairs, 2 from the row records
template <class S, class K, int NT, int PK>
__global__ __launch_bounds__(NT, sizeof(K) == 4 ? SX_FUSED_WAVES : 3)
void k_sx_fused(SxArgs g, int64_t fs, unsigned long long *status, int64_t ntiles, int64_t *host)
{
    using Z = typename S::Z;
    constexpr int FUSED_ROWS = NT / TG;
    static_assert(FUSED_ROWS <= 64, "the tile's row offsets are scanned by one wavefront");
    // per-team rows padded by one element so the 8 teams of a wavefront
    // start on different LDS banks
    __shared__ K s_key[FUSED_ROWS][FMAX + 1];         // sort keys, then output columns (int32)
    __shared__ Z s_val[FUSED_ROWS][FMAX + 1];         // flop values, then output values
    __shared__ int64_t s_cnt[FUSED_ROWS], s_off[FUSED_ROWS + 1];
    __shared__ int s_big[FUSED_ROWS];
    __shared__ int64_t s_tile, s_prefix;

    const int team = threadIdx.x / TG, sub = threadIdx.x & (TG - 1);
    K *key = s_key[team];
    Z *val = s_val[team];
    int32_t *outj = (int32_t *) s_key[team];
    unsigned long long *ticket = status + ntiles;

    while (true)
    {
        if (threadIdx.x == 0) s_tile = (int64_t) atomicAdd(ticket, 1ull);
        __syncthreads();
        const int64_t tile = s_tile;
        if (tile >= ntiles) break;
        const int64_t i = tile * FUSED_ROWS + team;

        #pragma unroll
        for (int u = 0; u < FMAX / TG; u++) key[sub * (FMAX / TG) + u] = (K) ~(K) 0;
        int64_t f = 0, cnt = 0;
        int big = 0, nallow = 0;
        if (i < g.m)
        {
            const int64_t a0 = g.Ap[i], a1 = g.Ap[i + 1];
            const int64_t pm0 = g.Mp ? g.Mp[i] : 0, pm1 = g.Mp ? g.Mp[i + 1] : 0;
            wave_sync();
            for (int64_t e0 = a0; e0 < a1; e0 += TG)
            {
                const int64_t e = e0 + sub;
                int64_t k = 0, bs = 0, len = 0;
                Z av = S::identity();
                if (e < a1)
                {
                    k = g.Aj[e];
                    if constexpr (PK == 2)
                    {
                        // the row's run of records; its length rides in the
                        // first record, whose line the team reads next anyway
                        bs = k << g.rec_lg;
                        len = (int64_t) ((unsigned long long) g.Bjx[2 * bs] >> 56);
                    }
                    else
                    {
                        bs = g.Bp[k];
                        len = g.Bp[k + 1] - bs;
                    }
                    av = S::geta((const Z *) g.Ax, e, g.a_iso);
                }
                const int64_t inc = team_incl_scan<int64_t>(len);
                const int64_t tot = __shfl(inc, TG - 1, TG);
                if (f + tot > fs) { big = 1; break; }
                // the chunk's flop offsets in every lane's registers; flop q
                // belongs to the last A entry whose offset is <= q (entries
                // past the row's end have offset tot, never <= q)
                const int32_t pre = (int32_t) (inc - len);
                int32_t pres[TG];
                #pragma unroll
                for (int m = 0; m < TG; m++) pres[m] = __shfl(pre, m, TG);
                // the chunk's flops in three passes, so that the B gathers of
                // all FMAX/TG flops of a lane are in flight together: owners
                // and B positions (a lane past the chunk's flops takes its
                // last flop's, a valid position), the gathers, then the keys
                if (tot > 0)
                {
                    constexpr int NIT = FMAX / TG;
                    int los[NIT];
                    int64_t pbs[NIT];
                    #pragma unroll
                    for (int it = 0; it < NIT; it++)
                    {
                        const int64_t q = (int64_t) it * TG + sub;
                        const int32_t qc = (int32_t) (q < tot ? q : tot - 1);
                        int lo = -1;
                        #pragma unroll
                        for (int m = 0; m < TG; m++) lo += (pres[m] <= qc) ? 1 : 0;
                        // shuffled by every lane of the team (a lane outside a
                        // branch would return zeros)
                        los[it] = lo;
                        pbs[it] = __shfl(bs, lo, TG) + (qc - __shfl(pre, lo, TG));
                    }
                    int64_t js[NIT];
                    uint64_t xb[NIT];
                    #pragma unroll
                    for (int it = 0; it < NIT; it++)
                    {
                        if constexpr (PK != 0)
                        {
                            const longlong2 jx = *(const longlong2 *) (g.Bjx + 2 * pbs[it]);
                            js[it] = (PK == 2) ? (jx.x & SX_REC_COL) : jx.x;
                            xb[it] = (uint64_t) jx.y;
                        }
                        else
                        {
                            js[it] = g.Bj[pbs[it]];
                            xb[it] = 0;
                        }
                    }
                    #pragma unroll
                    for (int it = 0; it < NIT; it++)
                    {
                        const int64_t q = (int64_t) it * TG + sub;
                        const Z avl = shfl_any<Z>(av, los[it], TG);
                        const int64_t kl = (S::mult == GM_MULT_K) ? __shfl(k, los[it], TG) : 0;
                        if (q < tot && sx_mask_ok(g, pm0, pm1, js[it]))
                        {
                            const int64_t fq = f + q;
                            key[fq] = (K) (((K) js[it] << 6) | (K) fq);
                            if constexpr (!S::iso_out)
                            {
                                Z bv;
                                if constexpr (PK != 0) bv = __builtin_bit_cast(Z, xb[it]);
                                else bv = S::geta((const Z *) g.Bx, pbs[it], g.b_iso);
                                val[fq] = S::mul(avl, bv, kl);
                            }
                            nallow++;
                        }
                    }
                }
                f += tot;
                wave_sync();
            }
            if (big) cnt = g.Cp[i];
        }
        nallow = team_sum<int>(nallow);
        if (!big && nallow > 0)
        {
            // bitonic sort of the 64 keys: lane sub holds positions
            // sub*8 .. sub*8+7 in registers; distances < 8 are register
            // compare-exchanges, distances >= 8 are width-8 shuffles
            constexpr int PER_L = FMAX / TG;
            K kr[PER_L];
            #pragma unroll
            for (int r = 0; r < PER_L; r++) kr[r] = key[sub * PER_L + r];
            #pragma unroll
            for (int kk = 2; kk <= FMAX; kk <<= 1)
            {
                #pragma unroll
                for (int jj = kk >> 1; jj > 0; jj >>= 1)
                {
                    if (jj >= PER_L)
                    {
                        const int lmask = jj / PER_L;
                        const bool lower = (sub & lmask) == 0;
                        #pragma unroll
                        for (int r = 0; r < PER_L; r++)
                        {
                            const int idx = sub * PER_L + r;
                            const bool asc = (idx & kk) == 0;
                            K o;
                            if constexpr (sizeof(K) == 4)
                                o = (K) __shfl_xor((unsigned int) kr[r], lmask, TG);
                            else
                                o = (K) __shfl_xor((unsigned long long) kr[r], lmask, TG);
                            const K mn = kr[r] < o ? kr[r] : o, mx = kr[r] < o ? o : kr[r];
                            kr[r] = (lower == asc) ? mn : mx;
                        }
                    }
                    else
                    {
                        #pragma unroll
                        for (int r = 0; r < PER_L; r++)
                        {
                            const int partner = r ^ jj;
                            if (partner > r)
                            {
                                const int idx = sub * PER_L + r;
                                const bool asc = (idx & kk) == 0;
                                const K a = kr[r], b = kr[partner];
                                if ((a > b) == asc) { kr[r] = b; kr[partner] = a; }
                            }
                        }
                    }
                }
            }
            #pragma unroll
            for (int r = 0; r < PER_L; r++) key[sub * PER_L + r] = kr[r];
            wave_sync();
            // compress: lane owns sorted positions sub*8 .. sub*8+7, whose
            // keys are still in kr[]; a run's head sums its values in flop
            // order from registers, and from LDS only past the lane's end
            constexpr int PER = FMAX / TG;
            const K kprev = (K) shfl_any<K>(kr[PER - 1], sub > 0 ? sub - 1 : 0, TG);
            Z vv[PER];
            #pragma unroll
            for (int u = 0; u < PER; u++)
            {
                vv[u] = S::identity();
                if constexpr (!S::iso_out)
                    if (sub * PER + u < nallow) vv[u] = val[kr[u] & 63];
            }
            int32_t hj[PER];
            Z hz[PER];
            int nh = 0;
            #pragma unroll
            for (int u = 0; u < PER; u++)
            {
                const int p = sub * PER + u;
                hj[u] = -1;
                if (p < nallow)
                {
                    const int64_t jp = (int64_t) (kr[u] >> 6);
                    const K kb = (u == 0) ? kprev : kr[u > 0 ? u - 1 : 0];
                    if (p == 0 || (int64_t) (kb >> 6) != jp)
                    {
                        Z z = vv[u];
                        bool open = true;
                        #pragma unroll
                        for (int u2 = u + 1; u2 < PER; u2++)
                        {
                            if (open && sub * PER + u2 < nallow && (int64_t) (kr[u2] >> 6) == jp)
                            {
                                if constexpr (!S::iso_out) z = S::upd(z, vv[u2]);
                            }
                            else open = false;
                        }
                        if (open)
                        {
                            for (int p2 = sub * PER + PER; p2 < nallow; p2++)
                            {
                                const K k2 = key[p2];
                                if ((int64_t) (k2 >> 6) != jp) break;
                                if constexpr (!S::iso_out) z = S::upd(z, val[k2 & 63]);
                            }
                        }
                        hj[u] = (int32_t) jp;
                        hz[u] = z;
                        nh++;
                    }
                }
            }
            const int inc = team_incl_scan<int>(nh);
            int r = inc - nh;
            cnt = __shfl(inc, TG - 1, TG);
            wave_sync();
            #pragma unroll
            for (int u = 0; u < PER; u++)
            {
                if (hj[u] >= 0)
                {
                    outj[r] = hj[u];
                    if constexpr (!S::iso_out) val[r] = hz[u];
                    r++;
                }
            }
        }
        if (sub == 0)
        {
            s_cnt[team] = cnt;
            s_big[team] = big;
        }
        __syncthreads();
        if (threadIdx.x < 64)
        {
            // wavefront 0: tile offsets, then a look-back over up to 64
            // predecessors per step (lane l reads tile - 1 - l)
            const int lane = threadIdx.x;
            // row offsets of the tile: inclusive scan of the row counts
            // across the wavefront's lanes
            const int64_t c = lane < FUSED_ROWS ? s_cnt[lane] : 0;
            int64_t incl = c;
            #pragma unroll
            for (int off = 1; off < FUSED_ROWS; off <<= 1)
            {
                const int64_t o = __shfl_up(incl, off, 64);
                if (lane >= off) incl += o;
            }
            const int64_t run = __shfl(incl, FUSED_ROWS - 1, 64);
            if (lane == 0)
                __hip_atomic_store(&status[tile], (tile == 0 ? LB_PRE : LB_AGG) | (unsigned long long) run,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (lane < FUSED_ROWS) s_off[lane] = incl - c;
            if (lane == 0) s_off[FUSED_ROWS] = run;
            int64_t prefix = 0;
            if (tile > 0)
            {
                // window of LB_WIN*64 predecessors, position u*64 + lane =
                // distance - 1; all loads are independent (relaxed: the
                // counts travel inside the status words themselves)
                int64_t end = tile - 1;
                int spins = 0;
                while (true)
                {
                    unsigned long long w[LB_WIN];
                    #pragma unroll
                    for (int u = 0; u < LB_WIN; u++)
                    {
                        const int64_t idx = end - (int64_t) u * 64 - lane;
                        w[u] = (idx >= 0) ? __hip_atomic_load(&status[idx], __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_AGENT)
                                          : LB_PRE;
                    }
                    int firstp = LB_WIN * 64;
                    bool zero_before = false;
                    #pragma unroll
                    for (int u = 0; u < LB_WIN; u++)
                    {
                        const unsigned long long flag = w[u] & ~LB_MASK;
                        const unsigned long long bp = __ballot(flag == LB_PRE);
                        const unsigned long long b0 = __ballot(flag == 0);
                        if (firstp == LB_WIN * 64)
                        {
                            const int fp = bp ? (__ffsll((long long) bp) - 1) : 64;
                            const unsigned long long upto =
                                (fp >= 63) ? ~0ull : ((2ull << fp) - 1ull);
                            if (b0 & upto) zero_before = true;
                            if (fp < 64) firstp = u * 64 + fp;
                        }
                    }
                    if (zero_before)
                    {
                        // a predecessor has not published yet
                        if (++spins > LB_SPIN_LIMIT)
                        {
                            if (lane == 0)
                                __hip_atomic_store(&host[1], (int64_t) 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                        continue;
                    }
                    int64_t v = 0;
                    #pragma unroll
                    for (int u = 0; u < LB_WIN; u++)
                        if (u * 64 + lane <= firstp) v += (int64_t) (w[u] & LB_MASK);
                    #pragma unroll
                    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
                    prefix += v;
                    if (firstp < LB_WIN * 64) break;
                    end -= LB_WIN * 64;
                }
                if (lane == 0)
                    __hip_atomic_store(&status[tile], LB_PRE | (unsigned long long) (prefix + run),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (lane == 0) s_prefix = prefix;
        }
        __syncthreads();
        const int64_t prefix = s_prefix;
        const int64_t total = s_off[FUSED_ROWS];
        if (sub == 0 && i < g.m) g.Cp[i] = prefix + s_off[team];
        if (tile == ntiles - 1 && threadIdx.x == 0)
        {
            // the host reads nnz(C) there after its wait: no copy to queue
            g.Cp[g.m] = prefix + total;
            host[0] = prefix + total;
        }
        // each team copies its own small row: the row's entries are
        // contiguous in C, its lanes store consecutive ones
        if (!big && i < g.m)
        {
            const int64_t r0 = prefix + s_off[team];
            for (int pos = sub; pos < (int) cnt; pos += TG)
            {
                g.Ci[r0 + pos] = (int64_t) outj[pos];
                if constexpr (!S::iso_out) ((Z *) g.Cx)[r0 + pos] = val[pos];
            }
        }
        __syncthreads();
    }
}

__global__ void k_sx_fill_u64(unsigned long long *x, int64_t n)
{
    for (int64_t t = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (int64_t) gridDim.x * blockDim.x)
        x[t] = 0;
}

static inline unsigned sx_grid(int64_t items, int64_t per_block, int64_t cap)
{
    int64_t g = (items + per_block - 1) / per_block;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (unsigned) g;
}

// the dense rows' device arrays between their build and the writing of C
struct SxPush
{
    PushArgs h;
    DevBuf pre, coff, it_d, it_e, tab, bits, mbits, seg;
    void drop()
    {
        pre.drop(); coff.drop(); it_d.drop(); it_e.drop(); tab.drop(); bits.drop(); mbits.drop(); seg.drop();
    }
};

// bytes of one dense row
template <class S>
static double sx_push_row_bytes(int64_t n, bool masked)
{
    return (S::iso_out ? 0.0 : (double) sizeof(PuCell<S>) * (double) n) + (masked ? 0.25 : 0.125) * (double) n +
           8.0 * (double) (n / PU_SEG + 1);
}

// tables, products and counts of the dense rows (their Cp entries)
template <class S>
static int sx_push_build(SxArgs &g, SxPush &p, int64_t D, int64_t nnzA, int64_t hflops)
{
    hipStream_t st = stream();
    const int64_t cap = (int64_t) cu_count() * 8;
    PushArgs &h = p.h;
    h.D = D;
    h.drow = g.rows + (int64_t) BIN_DNS * g.ls;
    h.nw = (g.n + 31) >> 5;
    h.nseg = (g.n + PU_SEG - 1) / PU_SEG;
    const int64_t items = hflops / PU_CH + D + 1;
    const bool masked = g.mode != MODE_NONE;
    if (!p.pre.alloc(sizeof(int64_t) * (nnzA + 1)) || !p.coff.alloc(sizeof(int64_t) * (D + 1)) ||
        !p.it_d.alloc(sizeof(uint32_t) * items) || !p.it_e.alloc(sizeof(int64_t) * items) ||
        (!S::iso_out && !p.tab.alloc(sizeof(PuCell<S>) * (size_t) (D * g.n))) ||
        (PU_BITS<S> && !p.bits.alloc(sizeof(uint32_t) * (size_t) (D * h.nw))) ||
        (masked && !p.mbits.alloc(sizeof(uint32_t) * (size_t) (D * h.nw))) ||
        !p.seg.alloc(sizeof(int64_t) * (size_t) (D * h.nseg + 1)))
        return set_error(GM_OUT_OF_MEMORY, "saxpy3: dense rows (%lld)", (long long) D);
    h.pre = p.pre.as<int64_t>(); h.coff = p.coff.as<int64_t>();
    h.it_d = p.it_d.as<uint32_t>(); h.it_e = p.it_e.as<int64_t>();
    h.tab = p.tab.ptr; h.bits = p.bits.as<uint32_t>(); h.mbits = p.mbits.as<uint32_t>();
    h.seg = p.seg.as<int64_t>();
    ProfScope ps("sx_push");
    k_sx_elen<<<sx_grid(nnzA, PU_NT, cap), PU_NT, 0, st>>>(g, nnzA, p.pre.as<int64_t>());
    GM_TRY(scan_exclusive_i64(p.pre.as<int64_t>(), p.pre.as<int64_t>(), nnzA));
    k_sx_push_chunks<<<sx_grid(D, PU_NT, cap), PU_NT, 0, st>>>(h);
    GM_TRY(scan_exclusive_i64(h.coff, h.coff, D));
    k_sx_push_items<<<sx_grid(items, PU_NT, cap), PU_NT, 0, st>>>(g, h);
    k_sx_push_init<S><<<sx_grid(D * g.n, PU_NT * 8, cap * 2), PU_NT, 0, st>>>(h, D * g.n, D * h.nw, masked);
    if (masked)
    {
        const dim3 grid(sx_grid(cap, D, 64), (unsigned) (D < 32768 ? D : 32768));
        k_sx_push_mask<<<grid, PU_NT, 0, st>>>(g, h);
    }
    k_sx_push<S><<<sx_grid(items, 1, cap), PU_NT, 0, st>>>(g, h);
    k_sx_push_count<S><<<sx_grid(D * h.nseg, 1, cap * 2), PU_NT, 0, st>>>(g, h);
    GM_TRY(scan_exclusive_i64(h.seg, h.seg, D * h.nseg));
    k_sx_push_rows<<<sx_grid(D, PU_NT, cap), PU_NT, 0, st>>>(g, h);
    GM_HIP(hipGetLastError(), "sx_push");
    return GM_SUCCESS;
}

template <class S>
static int sx_push_write(SxArgs &g, SxPush &p)
{
    ProfScope ps("sx_push_write");
    k_sx_push_write<S><<<sx_grid(p.h.D * p.h.nseg, 1, (int64_t) cu_count() * 16), PU_NT, 0, stream()>>>(g, p.h);
    return check_hip(hipGetLastError(), "k_sx_push_write");
}

// the tiled rows' device arrays
struct SxTile
{
    TileArgs t;
    DevBuf tpos, bits, seg, next;
    void drop() { tpos.drop(); bits.drop(); seg.drop(); next.drop(); }
};

static int64_t sx_tile_row_bytes(int64_t n) { return (n + TL_W - 1) / TL_W * (TL_W / 8 + 8); }

template <class S, int PHASE>
static int sx_tile_run(SxArgs &g, TileArgs &t)
{
    hipStream_t st = stream();
    ProfScope ps(PHASE == 0 ? "sx_tile_sym" : "sx_tile_num");
    if (PHASE == 1) k_sx_zero<<<1, 128, 0, st>>>(t.next, 128);
    const int64_t units = t.nf * t.nt + (t.T - t.nf) * ((t.nt + TL_RUN - 1) / TL_RUN);
    k_sx_tile<S, PHASE><<<sx_grid(units, TL_NT / 64, (int64_t) cu_count() * 8), TL_NT, 0, st>>>(g, t);
    return check_hip(hipGetLastError(), "k_sx_tile");
}

// bits and counts of the tiled rows (their Cp entries); kb: rows of B
static int sx_tile_build(SxArgs &g, SxTile &x, const int64_t *hc, int64_t kb)
{
    hipStream_t st = stream();
    const int64_t cap = (int64_t) cu_count() * 8;
    TileArgs &t = x.t;
    t.nf = hc[CNT_TILF];
    t.T = hc[BIN_TIL];
    t.nt = (g.n + TL_W - 1) / TL_W;
    t.front = g.rows + (int64_t) BIN_TIL * g.ls;
    t.back = t.front + g.ls - 1;
    if (!x.bits.alloc((size_t) (t.T * t.nt) * (TL_W / 8)) || !x.seg.alloc(sizeof(int64_t) * (size_t) (t.T * t.nt + 1)) ||
        !x.next.alloc(128 * sizeof(unsigned long long)))
        return set_error(GM_OUT_OF_MEMORY, "saxpy3: tiled rows (%lld)", (long long) t.T);
    t.bits = x.bits.as<uint64_t>();
    t.seg = x.seg.as<int64_t>();
    t.next = x.next.as<unsigned long long>();
    t.tpos = nullptr;
    // B's offsets at the tile ends, when the rows look up at least a quarter as
    // many as there are and they fit 1 GB
    if (4 * hc[CNT_TILA] >= kb && (double) kb * (double) (t.nt + 1) <= (double) (1 << 28) &&
        x.tpos.alloc(sizeof(uint32_t) * (size_t) (kb * (t.nt + 1))))
    {
        ProfScope ps("sx_tile_pos");
        k_sx_tile_pos<<<sx_grid(kb * (t.nt + 1), TL_NT, cap * 4), TL_NT, 0, st>>>(g.Bp, g.Bj, kb, t.nt,
                                                                               x.tpos.as<uint32_t>());
        GM_HIP(hipGetLastError(), "k_sx_tile_pos");
        t.tpos = x.tpos.as<uint32_t>();
    }
    GM_TRY((sx_tile_run<SR<GM_ADD_ANY, GM_MULT_PAIR, uint8_t>, 0>(g, t)));
    GM_TRY(scan_exclusive_i64(t.seg, t.seg, t.T * t.nt));
    k_sx_tile_rows<<<sx_grid(t.T, TL_NT, cap), TL_NT, 0, st>>>(g, t);
    return check_hip(hipGetLastError(), "k_sx_tile_rows");
}

// flop count, binning and the dealing out of the heavy rows; hc receives the
// counters
static int sx_count(SxArgs &g, int64_t fs, int list_small, int64_t dmax, int64_t tmax, int64_t *dflops, int64_t *hc,
                    unsigned long long *hp)
{
    hipStream_t st = stream();
    DevBuf rowf;
    {
        ProfScope ps("sx_flops");
        if (g.m <= FEW_ROWS)
        {
            // a few rows may be very long: each one over many workgroups
            if (!rowf.alloc(sizeof(unsigned long long) * g.m)) return set_error(GM_OUT_OF_MEMORY, "saxpy3: flops");
            k_sx_zero<<<1, FEW_ROWS, 0, st>>>(rowf.as<unsigned long long>(), (int) g.m);
            const dim3 grid((unsigned) ((cu_count() * 4 + g.m - 1) / g.m), (unsigned) g.m);
            k_sx_rowflops<<<grid, PU_NT, 0, st>>>(g, rowf.as<unsigned long long>());
            g.rowf = rowf.as<unsigned long long>();
        }
        k_sx_flops<<<sx_grid(g.m, SX_NT / TG, (int64_t) cu_count() * 16), SX_NT, 0, st>>>(g, fs, list_small);
        g.rowf = nullptr;
        if (g.rows) k_sx_classify<<<sx_grid(g.m, SX_NT, (int64_t) cu_count()), SX_NT, 0, st>>>(g, dflops, dmax, tmax);
        GM_HIP(hipGetLastError(), "k_sx_flops");
    }
    GM_HIP(hipMemcpyAsync(hp, g.cnt, SX_NCNT * sizeof(unsigned long long), hipMemcpyDeviceToHost, st), "bin counts");
    GM_HIP(hipStreamSynchronize(st), "bin counts sync");
    for (int t = 0; t < SX_NCNT; t++) hc[t] = (int64_t) hp[t];
    if (hc[BIN_DNS] > dmax) hc[BIN_DNS] = dmax;
    hc[BIN_TIL] = hc[CNT_TILF] + hc[CNT_TILB];
    return GM_SUCCESS;
}

// pattern-only instance used by the symbolic phase of every semiring
using SxSym = SR<GM_ADD_ANY, GM_MULT_PAIR, uint8_t>;

template <class S, int PHASE>
static int sx_launch_phase(SxArgs &g, const int64_t *cnt, bool skip_ws)
{
    hipStream_t st = stream();
    const int64_t cap = (int64_t) cu_count() * 32;
    const char *names[2][5] = {
        {"sx_sym_single", "sx_sym_wave128", "sx_sym_wave1024", "sx_sym_block4096", "sx_sym_global"},
        {"sx_num_single", "sx_num_wave128", "sx_num_wave1024", "sx_num_block4096", "sx_num_global"}};
    if (cnt[BIN_SINGLE] > 0)
    {
        ProfScope ps(names[PHASE][0]);
        k_sx_single<S, PHASE><<<sx_grid(cnt[BIN_SINGLE], 4, cap), SX_NT, 0, st>>>(g);
        GM_HIP(hipGetLastError(), "k_sx_single");
    }
    if (cnt[BIN_WS] > 0 && !skip_ws)
    {
        ProfScope ps(names[PHASE][1]);
        k_sx_wave<S, 7, PHASE><<<sx_grid(cnt[BIN_WS], 4, cap), SX_NT, 0, st>>>(g, BIN_WS);
        GM_HIP(hipGetLastError(), "k_sx_wave128");
    }
    if (cnt[BIN_WL] > 0)
    {
        ProfScope ps(names[PHASE][2]);
        k_sx_wave<S, 10, PHASE><<<sx_grid(cnt[BIN_WL], 4, cap), SX_NT, 0, st>>>(g, BIN_WL);
        GM_HIP(hipGetLastError(), "k_sx_wave1024");
    }
    if (cnt[BIN_BLK] > 0)
    {
        ProfScope ps(names[PHASE][3]);
        k_sx_block<S, 12, PHASE><<<sx_grid(cnt[BIN_BLK], 1, cap), SX_NT, 0, st>>>(g);
        GM_HIP(hipGetLastError(), "k_sx_block4096");
    }
    if (cnt[BIN_GLB] > 0)
    {
        ProfScope ps(names[PHASE][4]);
        k_sx_global<S, PHASE><<<sx_grid(cnt[BIN_GLB], 1, cap), SX_NT, 0, st>>>(g);
        GM_HIP(hipGetLastError(), "k_sx_global");
    }
    return GM_SUCCESS;
}

template <class S>
static int saxpy3_run(gm_csr_out *C, const gm_csr *M, bool mask_comp, bool mask_struct,
                      const gm_csr *A, const gm_csr *B, const gm_saxpy3_params *prm)
{
    using Z = typename S::Z;
    hipStream_t st = stream();
    const int64_t m = A->nrows, n = B->ncols;
    const size_t zs = sizeof(Z);
    const size_t entry_bytes = sizeof(int64_t) + (S::iso_out ? 0 : zs);

    DevBuf Cp, cnt, lists;
    // the counters and the fused kernel's tile status words, cleared together
    const int64_t ntiles = (m + FUSED_ROWS - 1) / FUSED_ROWS;
    if (!Cp.alloc(sizeof(int64_t) * (m + 1)) ||
        !cnt.alloc(sizeof(unsigned long long) * (size_t) (SX_NCNT + ntiles + 1)))
        return set_error(GM_OUT_OF_MEMORY, "saxpy3: workspace");

    SxArgs g;
    g.m = m; g.n = n;
    g.Ap = A->p; g.Aj = A->j; g.Ax = A->x; g.a_iso = A->iso;
    g.Bp = B->p; g.Bj = B->j; g.Bx = B->x; g.b_iso = B->iso;
    g.Mp = M ? M->p : nullptr; g.Mj = M ? M->j : nullptr;
    g.Mx = (M && !mask_struct) ? M->x : nullptr;
    g.msize = M ? (int32_t) type_size(M->type) : 0;
    g.m_iso = M ? M->iso : 0;
    g.mask_struct = (mask_struct || !M || !M->x) ? 1 : 0;
    g.mode = !M ? MODE_NONE : (mask_comp ? MODE_NOTMASK : MODE_MASK);
    g.Cp = Cp.as<int64_t>(); g.Ci = nullptr; g.Cx = nullptr;
    g.rows = nullptr; g.ls = 0; g.cnt = cnt.as<unsigned long long>();
    g.hflops = nullptr; g.rowf = nullptr;
    g.gtab_off = nullptr; g.gtab_log2 = nullptr;
    g.gkeys = nullptr; g.gvals = nullptr; g.glist = nullptr;
    g.Bjx = nullptr;
    g.rec_lg = -1;
    g.table = prm ? (int32_t) prm->table : 0;
    if (g.table < 0 || g.table > 2) return set_error(GM_INVALID_VALUE, "saxpy3: table %d", (int) g.table);
    const gm_saxpy3_params tu = saxpy3_tuned();
    g.ws_max = pick_param(prm ? prm->wave_small_max : 0, tu.wave_small_max, 64);
    g.wl_max = pick_param(prm ? prm->wave_large_max : 0, tu.wave_large_max, 512);
    g.blk_max = pick_param(prm ? prm->block_max : 0, tu.block_max, 2048);
    if (g.ws_max > FMAX) g.ws_max = FMAX;
    if (g.wl_max > 512) g.wl_max = 512;
    if (g.blk_max > 2048) g.blk_max = 2048;
    const int64_t fs = g.ws_max;        // flops bound of a "small" row
    const int mode = (prm && prm->mode) ? (int) prm->mode : (int) tu.mode;
    // the fused kernel holds C's small rows at their flop bound until the
    // scan; it is used while that bound stays within a third of HBM
    const double budget = (double) device_hbm_bytes() / 3.0;

    // dense rows at most: their tables within 1/32 of HBM
    int64_t dmax = 0;
    if (SX_ANY_ORDER<S> && B->nrows < (int64_t) 0xffffffff)
        dmax = (int64_t) ((double) device_hbm_bytes() / 32.0 / (sx_push_row_bytes<S>(n, M != nullptr) + 1.0));
    // tiled rows at most: their bits within 1/64 of HBM
    const int64_t tmax = n > 0 ? device_hbm_bytes() / 64 / sx_tile_row_bytes(n) : 0;
    int64_t hc[SX_NCNT] = {0};
    unsigned long long *hp = (unsigned long long *) pinned_scratch(SX_NCNT * sizeof(unsigned long long));
    if (!hp) return set_error(GM_OUT_OF_MEMORY, "pinned scratch");
    if (m == 0)
    {
        k_sx_fill_u64<<<1, 64, 0, st>>>((unsigned long long *) g.Cp, 1);
        GM_HIP(hipGetLastError(), "k_sx_fill_u64");
        C->nrows = m; C->ncols = n; C->nvals = 0;
        if (!Cp.ptr) return GM_OUT_OF_MEMORY;
        DevBuf Ci, Cx;
        if (!Ci.alloc(8) || !Cx.alloc(zs)) return set_error(GM_OUT_OF_MEMORY, "saxpy3: output");
        GM_HIP(hipStreamSynchronize(st), "saxpy3 sync");
        C->p = (int64_t *) Cp.release(); C->j = (int64_t *) Ci.release(); C->x = Cx.release();
        C->iso = S::iso_out ? 1 : 0;
        return GM_SUCCESS;
    }

    // 1. max row lengths of A and B, and nnz(A), for the all-small shortcut.
    // When A has far fewer rows than B (a few frontier rows against a large
    // graph) the flop pass below is as cheap as this one, so it is skipped
    // together with its synchronisation.
    int64_t maxA = 0, maxB = 0, nnzA = 0, nnzB = -1;
    const bool probe_small = m * 8 >= B->nrows;
    k_sx_fill_u64<<<sx_grid(SX_NCNT + ntiles + 1, 256, 1024), 256, 0, st>>>(g.cnt, SX_NCNT + ntiles + 1);
    GM_HIP(hipGetLastError(), "k_sx_fill_u64");
    if (probe_small)
    {
        {
            ProfScope ps("sx_maxlen");
            const int64_t lim = m > B->nrows ? m : B->nrows;
            k_sx_maxlen<<<sx_grid((lim + 3) / 4, SX_NT, (int64_t) cu_count() * 8), SX_NT, 0, st>>>(
                A->p, m, B->p, B->nrows, g.cnt + CNT_MAXLEN);
            GM_HIP(hipGetLastError(), "k_sx_maxlen");
        }
        // max |A(i,:)|, max |B(k,:)|, nnz(A), -, -, nnz(B)
        GM_HIP(hipMemcpyAsync(hp, g.cnt + CNT_MAXLEN, 6 * sizeof(unsigned long long), hipMemcpyDeviceToHost, st),
               "maxlen d2h");
        GM_HIP(hipStreamSynchronize(st), "maxlen sync");
        maxA = (int64_t) hp[0];
        maxB = (int64_t) hp[1];
        nnzA = (int64_t) hp[2];
        nnzB = (int64_t) hp[5];
    }

    bool fused = (mode != 2);
    bool all_small = fused && probe_small && (double) maxA * (double) maxB <= (double) fs &&
                     (double) nnzA * (double) maxB * (double) entry_bytes <= budget;
    int64_t cap_small = all_small ? nnzA * maxB : 0;

    // 2. flop count and binning (skipped when every row is small)
    int64_t *dflops = nullptr;
    if (!all_small)
    {
        // the bins' row lists and the heavy rows' records, in one block
        auto place = [&](int64_t ls) {
            if (!lists.alloc((size_t) ls * (3 * sizeof(int64_t) + (SX_NBINS + 1) * sizeof(uint32_t)))) return false;
            g.ls = ls;
            g.gtab_off = lists.as<int64_t>();
            g.hflops = g.gtab_off + ls;
            dflops = g.hflops + ls;
            g.rows = (uint32_t *) (dflops + ls);
            g.gtab_log2 = (int32_t *) (g.rows + SX_NBINS * ls);
            return true;
        };
        if (!place(m))
        {
            // without room for every row in every bin the rows are counted first
            GM_TRY(sx_count(g, fs, fused ? 0 : 1, dmax, tmax, nullptr, hc, hp));
            if (fused && (double) hc[CNT_SMALL] * (double) entry_bytes > budget)
            {
                fused = false;
                k_sx_fill_u64<<<1, 64, 0, st>>>(g.cnt, SX_NCNT);
                GM_TRY(sx_count(g, fs, 1, dmax, tmax, nullptr, hc, hp));
            }
            int64_t ls = 1;
            for (int bin : {BIN_SINGLE, BIN_WS, BIN_WL, BIN_BLK, BIN_HVY}) ls = hc[bin] > ls ? hc[bin] : ls;
            k_sx_fill_u64<<<1, 64, 0, st>>>(g.cnt, SX_NCNT);
            if (!place(ls)) return set_error(GM_OUT_OF_MEMORY, "saxpy3: row lists");
        }
        GM_TRY(sx_count(g, fs, fused ? 0 : 1, dmax, tmax, dflops, hc, hp));
        cap_small = hc[CNT_SMALL];
        if (fused && (double) cap_small * (double) entry_bytes > budget)
        {
            // too large to hold at the flop bound: redo the binning with the
            // small rows listed for the symbolic + numeric path
            fused = false;
            k_sx_fill_u64<<<1, 64, 0, st>>>(g.cnt, SX_NCNT);
            GM_TRY(sx_count(g, fs, 1, dmax, tmax, dflops, hc, hp));
        }
    }

    DevBuf gkeys, gvals, glist;
    SxTile tiles;
    SxPush push;
    memset(&push.h, 0, sizeof(push.h));
    push.h.dflops = dflops;
    // the heavy rows' tables, and the counts of the tiled and dense ones
    auto tables = [&]() -> int {
        const int64_t gslots = hc[CNT_SLOTS];
        if (gslots > 0)
        {
            if (!gkeys.alloc(sizeof(uint32_t) * gslots) || !gvals.alloc(zs * gslots) ||
                !glist.alloc(sizeof(uint64_t) * gslots))
                return set_error(GM_OUT_OF_MEMORY, "saxpy3: global hash tables (%lld slots)",
                                 (long long) gslots);
            g.gkeys = gkeys.as<uint32_t>(); g.gvals = gvals.ptr; g.glist = glist.as<uint64_t>();
        }
        if (hc[BIN_TIL] > 0) GM_TRY(sx_tile_build(g, tiles, hc, B->nrows));
        if constexpr (SX_ANY_ORDER<S>)
            if (hc[BIN_DNS] > 0) GM_TRY(sx_push_build<S>(g, push, hc[BIN_DNS], hc[CNT_NNZA], hc[CNT_HFLOPS]));
        return GM_SUCCESS;
    };
    int trc = tables();
    if (trc == GM_OUT_OF_MEMORY && hc[BIN_TIL] + hc[BIN_DNS] > 0)
    {
        // no room for the tiles' bits or the dense tables: a hash table for
        // every heavy row, which is as large as its own products
        gkeys.drop(); gvals.drop(); glist.drop();
        tiles.drop();
        push.drop();
        k_sx_fill_u64<<<1, 64, 0, st>>>(g.cnt, SX_NCNT);
        GM_TRY(sx_count(g, fs, fused ? 0 : 1, 0, 0, dflops, hc, hp));
        trc = tables();
    }
    GM_TRY(trc);
    const int64_t nbig = hc[BIN_SINGLE] + hc[BIN_WL] + hc[BIN_BLK] + hc[BIN_GLB] + hc[BIN_DNS] +
                         hc[BIN_TIL];
    const bool have_big = nbig > 0;
    int64_t nvals = 0, held = 0;        // held: entries C has room for, if at the big rows' bound and small
    DevBuf Ci, Cx;
    if (fused)
    {
        // 3. symbolic phase of the big rows only
        int64_t big_total = 0;
        if (have_big)
        {
            GM_TRY((sx_launch_phase<SxSym, 0>(g, hc, true)));
            // the output's room for them: their bound while that is small, else
            // their exact sum, at the price of a kernel and a wait (about 20 us a
            // call; with the sizes accum_mask need not fetch, four hops of one
            // source over 60000 vertices went from 1258 to 1157 us)
            big_total = hc[CNT_BIGT];
        }
        const bool at_bound = have_big && (double) big_total * (double) entry_bytes <= (double) OUT_BOUND_MAX;
        if (have_big && !at_bound)
        {
            k_sx_sum_big<<<sx_grid(nbig, SX_NT, 512), SX_NT, 0, st>>>(g, dmax);
            GM_HIP(hipGetLastError(), "k_sx_sum_big");
            GM_HIP(hipMemcpyAsync(hp, g.cnt + CNT_BIGSUM, sizeof(unsigned long long),
                                  hipMemcpyDeviceToHost, st), "big total");
            GM_HIP(hipStreamSynchronize(st), "big total sync");
            big_total = (int64_t) hp[0];
        }
        const int64_t cap = cap_small + big_total;
        if (at_bound && (double) cap * (double) entry_bytes <= 2.0 * (double) OUT_BOUND_MAX) held = cap;
        if (!Ci.alloc(sizeof(int64_t) * (cap > 0 ? cap : 1)) ||
            !Cx.alloc(S::iso_out ? zs : zs * (cap > 0 ? cap : 1)))
            return set_error(GM_OUT_OF_MEMORY, "saxpy3: output (%lld entries)", (long long) cap);
        g.Ci = Ci.as<int64_t>();
        g.Cx = Cx.ptr;
        // 4. fused small-row kernel with the look-back scan over all rows
        // B's rows: from its row records when the operand carries them (one
        // aligned run per gathered row, no row pointers); else as 16-byte
        // (column, value) pairs when its rows are gathered at least about once
        // each on average (the pack reads and writes B once)
        DevBuf bjx;
        int pk = 0;
        if constexpr (SX_PACK_OK<S>)
        {
            const gm_csr_aux *ax = B->aux;
            if (!B->iso && B->x && ax && ax->rec && ax->rec_lg >= 0 && ax->nrows == B->nrows)
            {
                g.Bjx = (const int64_t *) ax->rec;
                g.rec_lg = ax->rec_lg;
                pk = 2;
            }
            else if (!B->iso && B->x && nnzB > 0 && 2 * nnzA >= B->nrows &&
                     bjx.alloc(sizeof(longlong2) * nnzB))
            {
                ProfScope ps("sx_pack");
                k_sx_pack<<<sx_grid(nnzB, 256, (int64_t) cu_count() * 16), 256, 0, st>>>(
                    B->j, (const int64_t *) B->x, nnzB, bjx.as<longlong2>());
                GM_HIP(hipGetLastError(), "k_sx_pack");
                g.Bjx = bjx.as<int64_t>();
                pk = 1;
            }
        }
        {
            ProfScope ps("sx_fused");
            const int64_t gcap = (int64_t) cu_count() * 8 * 256 / FUSED_NT;
            const int64_t grid = ntiles < gcap ? ntiles : gcap;
            unsigned long long *stp = g.cnt + SX_NCNT;
            int64_t *host = (int64_t *) hp;         // nnz(C), look-back error
            host[0] = 0;
            host[1] = 0;
            const bool k32 = B->ncols <= ((int64_t) 1 << 26);
#define GM_SX_FUSED(K, PKV) \
    k_sx_fused<S, K, FUSED_NT, PKV><<<(unsigned) grid, FUSED_NT, 0, st>>>(g, fs, stp, ntiles, host)
            if constexpr (SX_PACK_OK<S>)
            {
                if (pk == 2 && k32) GM_SX_FUSED(uint32_t, 2);
                else if (pk == 2) GM_SX_FUSED(uint64_t, 2);
                else if (pk == 1 && k32) GM_SX_FUSED(uint32_t, 1);
                else if (pk == 1) GM_SX_FUSED(uint64_t, 1);
            }
            if (pk == 0 && k32) GM_SX_FUSED(uint32_t, 0);
            else if (pk == 0) GM_SX_FUSED(uint64_t, 0);
#undef GM_SX_FUSED
            GM_HIP(hipGetLastError(), "k_sx_fused");
        }
        GM_HIP(hipStreamSynchronize(st), "fused sync");
        if (hp[1] != 0) return set_error(GM_PANIC, "saxpy3: look-back scan did not complete");
        nvals = (int64_t) hp[0];
        // 5. numeric phase of the big rows
        if (have_big && nvals > 0) GM_TRY((sx_launch_phase<S, 1>(g, hc, true)));
        if (hc[BIN_TIL] > 0 && nvals > 0) GM_TRY((sx_tile_run<S, 1>(g, tiles.t)));
        if constexpr (SX_ANY_ORDER<S>)
            if (hc[BIN_DNS] > 0 && nvals > 0) GM_TRY(sx_push_write<S>(g, push));
    }
    else
    {
        // symbolic + scan + numeric for every row
        GM_TRY((sx_launch_phase<SxSym, 0>(g, hc, false)));
        GM_TRY(scan_exclusive_i64(g.Cp, g.Cp, m));
        GM_HIP(hipMemcpyAsync(hp + 11, g.Cp + m, sizeof(int64_t), hipMemcpyDeviceToHost, st), "nnz(C)");
        GM_HIP(hipStreamSynchronize(st), "nnz(C) sync");
        nvals = (int64_t) hp[11];
        if (!Ci.alloc(sizeof(int64_t) * (nvals > 0 ? nvals : 1)) ||
            !Cx.alloc(S::iso_out ? zs : zs * (nvals > 0 ? nvals : 1)))
            return set_error(GM_OUT_OF_MEMORY, "saxpy3: output (%lld entries)", (long long) nvals);
        g.Ci = Ci.as<int64_t>();
        g.Cx = Cx.ptr;
        if (nvals > 0) GM_TRY((sx_launch_phase<S, 1>(g, hc, false)));
        if (hc[BIN_TIL] > 0 && nvals > 0) GM_TRY((sx_tile_run<S, 1>(g, tiles.t)));
        if constexpr (SX_ANY_ORDER<S>)
            if (hc[BIN_DNS] > 0 && nvals > 0) GM_TRY(sx_push_write<S>(g, push));
    }
    if (S::iso_out)
    {
        k_sx_iso_one<<<1, 1, 0, st>>>(Cx.ptr, (int) zs);
        GM_HIP(hipGetLastError(), "k_sx_iso_one");
    }
    if (held > 0)
    {
        (void) fit_block(Ci, sizeof(int64_t) * nvals, sizeof(int64_t) * held);
        if (!S::iso_out) (void) fit_block(Cx, zs * nvals, zs * held);
    }
    GM_HIP(hipStreamSynchronize(st), "saxpy3 sync");
    C->nrows = m;
    C->ncols = n;
    C->nvals = nvals;
    C->p = (int64_t *) Cp.release();
    C->j = (int64_t *) Ci.release();
    C->x = Cx.release();
    C->iso = S::iso_out ? 1 : 0;
    return GM_SUCCESS;
}

// C = A*B' or C<!M> = A*B' for a one-row A (gm_sx_pull.h)
template <class S>
static int vxm_bt_run(gm_csr_out *C, const gm_csr *M, bool mask_struct, const gm_csr *A, const gm_csr *B,
                      int64_t nnz)
{
    using Z = typename S::Z;
    hipStream_t st = stream();
    const int64_t n = B->nrows, k = A->ncols, cap = (int64_t) cu_count() * 8;
    const int64_t nw = (n + 31) >> 5, kw = (k + 31) >> 5;
    SxArgs g;
    memset(&g, 0, sizeof(g));
    g.m = 1; g.n = n;
    g.Ap = A->p; g.Aj = A->j; g.Ax = A->x; g.a_iso = A->iso;
    g.Bp = B->p; g.Bj = B->j; g.Bx = B->x; g.b_iso = B->iso;
    if (M)
    {
        g.Mp = M->p; g.Mj = M->j; g.Mx = mask_struct ? nullptr : M->x;
        g.msize = (int32_t) type_size(M->type); g.m_iso = M->iso;
        g.mask_struct = (mask_struct || !M->x) ? 1 : 0;
        g.mode = MODE_NOTMASK;
    }
    PushArgs h;
    PullArgs p;
    memset(&h, 0, sizeof(h));
    memset(&p, 0, sizeof(p));
    p.nnz = nnz;
    p.nch = (nnz + PL_CH - 1) / PL_CH;
    h.D = 1; h.nw = nw; h.all_bits = 1;
    h.nseg = (n + PU_SEG - 1) / PU_SEG;
    // cleared words: the row id, A's bits, the mask's, the result's bits or
    // its 32-bit cells
    const int64_t words = 2 + kw + (M ? nw : 0) + (PU_U32<S> ? n : nw);
    DevBuf Cp, Ci, Cx, zero, val, tab, part, seg;
    // the result at its bound of n entries, or once they are counted
    const size_t xs = S::iso_out ? 0 : sizeof(Z);
    const bool bound = n * (int64_t) (sizeof(int64_t) + xs) <= OUT_BOUND_MAX;
    auto result = [&](int64_t entries) {
        if (!Ci.alloc(sizeof(int64_t) * entries) || !Cx.alloc(S::iso_out ? sizeof(Z) : sizeof(Z) * entries)) return false;
        g.Ci = Ci.as<int64_t>();
        g.Cx = Cx.ptr;
        return true;
    };
    if (!Cp.alloc(2 * sizeof(int64_t)) || (bound && !result(n)) || !zero.alloc(sizeof(uint32_t) * (words + 1)) ||
        (!S::pattern && !val.alloc(sizeof(Z) * k)) || (!PU_U32<S> && !S::iso_out && !tab.alloc(sizeof(Z) * n)) ||
        !part.alloc((size_t) p.nch * (2 * sizeof(Z) + sizeof(int64_t) + 2) + 8) ||
        !seg.alloc(sizeof(int64_t) * (h.nseg + 1)))
        return set_error(GM_OUT_OF_MEMORY, "one-row product: workspace");
    g.Cp = Cp.as<int64_t>();
    uint32_t *w = zero.as<uint32_t>();
    h.drow = w;
    p.ubits = w + 2;
    h.mbits = p.ubits + kw;
    h.bits = h.mbits + (M ? nw : 0);
    h.tab = PU_U32<S> ? (void *) h.bits : tab.ptr;
    h.seg = seg.as<int64_t>();
    p.uval = val.ptr;
    p.lrow = part.as<int64_t>();
    p.pz = p.lrow + p.nch;
    p.pe = (uint8_t *) p.pz + 2 * sizeof(Z) * p.nch;
    int64_t *hp = (int64_t *) pinned_scratch(sizeof(int64_t));
    if (!hp) return set_error(GM_OUT_OF_MEMORY, "pinned scratch");
    {
        ProfScope ps("sx_pull");
        const int64_t zw = (words + 1) / 2;
        k_sx_fill_u64<<<sx_grid(zw, 256, cap), 256, 0, st>>>(zero.as<unsigned long long>(), zw);
        k_pull_scatter<S><<<sx_grid(k, PL_NT, cap), PL_NT, 0, st>>>(g, p);
        if (M) k_sx_push_mask<<<dim3((unsigned) cu_count(), 1), PU_NT, 0, st>>>(g, h);
        if (p.nch > 0)
        {
            k_pull<S><<<sx_grid(p.nch, 1, cap), PL_NT, 0, st>>>(g, h, p);
            k_pull_fix<S><<<sx_grid(p.nch, PL_NT / 64, cap), PL_NT, 0, st>>>(g, h, p);
        }
        k_sx_push_count<S><<<sx_grid(h.nseg, 1, cap), PU_NT, 0, st>>>(g, h);
        GM_TRY(scan_exclusive_i64(h.seg, h.seg, h.nseg));
        k_pull_ptr<<<1, 64, 0, st>>>(g.Cp, h.seg, h.nseg);
        if (!bound)
        {
            GM_HIP(hipMemcpyAsync(hp, g.Cp + 1, sizeof(int64_t), hipMemcpyDeviceToHost, st), "nnz(C)");
            GM_HIP(hipStreamSynchronize(st), "one-row product nnz sync");
            if (!result(hp[0]))
                return set_error(GM_OUT_OF_MEMORY, "one-row product: output (%lld entries)", (long long) hp[0]);
        }
        k_sx_push_write<S><<<sx_grid(h.nseg, 1, cap), PU_NT, 0, st>>>(g, h);
        if (S::iso_out) k_sx_iso_one<<<1, 1, 0, st>>>(Cx.ptr, (int) sizeof(Z));
        GM_HIP(hipGetLastError(), "one-row product");
    }
    GM_HIP(hipMemcpyAsync(hp, g.Cp + 1, sizeof(int64_t), hipMemcpyDeviceToHost, st), "nnz(C)");
    GM_HIP(hipStreamSynchronize(st), "one-row product sync");
    if (bound)
    {
        bool moved = fit_block(Ci, sizeof(int64_t) * hp[0], sizeof(int64_t) * n);
        moved |= fit_block(Cx, xs * hp[0], xs * n);
        if (moved) GM_HIP(hipStreamSynchronize(st), "one-row product fit sync");
    }
    C->nrows = 1;
    C->ncols = n;
    C->nvals = hp[0];
    C->p = (int64_t *) Cp.release();
    C->j = (int64_t *) Ci.release();
    C->x = Cx.release();
    C->iso = S::iso_out ? 1 : 0;
    return GM_SUCCESS;
}

} // namespace gm

using namespace gm;

extern "C" int gm_vxm_bt(gm_csr_out *C, const gm_csr *M, bool mask_struct, const gm_csr *A, const gm_csr *B,
                         int64_t nnz_b, const gm_semiring *sr)
{
    if (!C || !A || !B || !sr) return set_error(GM_INVALID_VALUE, "gm_vxm_bt: NULL argument");
    if (!semiring_supported(sr) || !operand_ok(sr, A) || !operand_ok(sr, B))
        return set_error(GM_NO_VALUE, "gm_vxm_bt: case not handled by the GPU kernels");
    // cells and counts are 32-bit; the dense vector is as long as the inner index
    if (A->nrows != 1 || A->ncols != B->ncols || nnz_b < 0 || B->nrows < 1 || A->ncols < 1 ||
        A->ncols >= (int64_t) 0xffffffff || B->nrows >= (int64_t) 0x7fffffff ||
        (M && (M->nrows != 1 || M->ncols != B->nrows)))
        return set_error(GM_NO_VALUE, "gm_vxm_bt: shape not handled");
    GM_TRY(ensure_init());
#define GM_VBT_CASE(ADD, MULT, ZC, Z)                                             \
    if (sr->add_op == ADD && sr->mult_op == MULT && sr->ztype == ZC)              \
    {                                                                             \
        int rc = vxm_bt_run<SR<ADD, MULT, Z>>(C, M, mask_struct, A, B, nnz_b);    \
        if (rc == GM_SUCCESS) C->type = ZC;                                       \
        return rc;                                                                \
    }
    GM_SEMIRING_LIST(GM_VBT_CASE)
#undef GM_VBT_CASE
    return set_error(GM_NO_VALUE, "gm_vxm_bt: semiring not instantiated");
}

//------------------------------------------------------------------------------
// total multiplies of C=A*B: the sum over A's entries (i,k) of |B(k,:)|.
// Partial sums per workgroup, then one workgroup adds them (no atomics).
//------------------------------------------------------------------------------

constexpr int FLOPS_NT = 256;
constexpr int FLOPS_MAXG = 2048;

__global__ __launch_bounds__(FLOPS_NT) void k_flopcount(const int64_t *__restrict__ Aj, int64_t nnz,
                                                        const int64_t *__restrict__ Bp,
                                                        unsigned long long *part)
{
    __shared__ unsigned long long s[FLOPS_NT / 64];
    unsigned long long f = 0;
    for (int64_t e = (int64_t) blockIdx.x * FLOPS_NT + threadIdx.x; e < nnz;
         e += (int64_t) gridDim.x * FLOPS_NT)
    {
        const int64_t k = Aj[e];
        f += (unsigned long long) (Bp[k + 1] - Bp[k]);
    }
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) f += __shfl_xor(f, off, 64);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = f;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        for (int w = 1; w < FLOPS_NT / 64; w++) f += s[w];
        part[blockIdx.x] = f;
    }
}

__global__ __launch_bounds__(FLOPS_NT) void k_flopcount_sum(unsigned long long *part, int n)
{
    __shared__ unsigned long long s[FLOPS_NT / 64];
    unsigned long long f = 0;
    for (int t = threadIdx.x; t < n; t += FLOPS_NT) f += part[t];
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) f += __shfl_xor(f, off, 64);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = f;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        for (int w = 1; w < FLOPS_NT / 64; w++) f += s[w];
        part[FLOPS_MAXG] = f;
    }
}

extern "C" int gm_flopcount(int64_t *flops, const gm_csr *A, const gm_csr *B)
{
    if (!flops || !A || !B) return set_error(GM_INVALID_VALUE, "gm_flopcount: NULL argument");
    if (A->ncols != B->nrows)
        return set_error(GM_INVALID_VALUE, "gm_flopcount: A is %lld x %lld, B is %lld x %lld",
                         (long long) A->nrows, (long long) A->ncols, (long long) B->nrows,
                         (long long) B->ncols);
    *flops = 0;
    if (A->nrows == 0 || B->nrows == 0) return GM_SUCCESS;
    if (!A->p || !B->p) return set_error(GM_INVALID_VALUE, "gm_flopcount: NULL row pointers");
    GM_TRY(ensure_init());
    hipStream_t st = stream();
    unsigned long long *hp = (unsigned long long *) pinned_scratch(16 * sizeof(unsigned long long));
    if (!hp) return set_error(GM_OUT_OF_MEMORY, "pinned scratch");
    GM_HIP(hipMemcpyAsync(hp, A->p + A->nrows, sizeof(int64_t), hipMemcpyDeviceToHost, st), "nnz(A)");
    GM_HIP(hipStreamSynchronize(st), "nnz(A) sync");
    const int64_t nnz = (int64_t) hp[0];
    if (nnz <= 0) return GM_SUCCESS;
    if (!A->j) return set_error(GM_INVALID_VALUE, "gm_flopcount: NULL column indices");
    DevBuf part;
    if (!part.alloc(sizeof(unsigned long long) * (FLOPS_MAXG + 1)))
        return set_error(GM_OUT_OF_MEMORY, "gm_flopcount: workspace");
    const unsigned grid = sx_grid(nnz, FLOPS_NT * 4, FLOPS_MAXG);
    k_flopcount<<<grid, FLOPS_NT, 0, st>>>(A->j, nnz, B->p, part.as<unsigned long long>());
    GM_HIP(hipGetLastError(), "k_flopcount");
    k_flopcount_sum<<<1, FLOPS_NT, 0, st>>>(part.as<unsigned long long>(), (int) grid);
    GM_HIP(hipGetLastError(), "k_flopcount_sum");
    GM_HIP(hipMemcpyAsync(hp, part.as<unsigned long long>() + FLOPS_MAXG, sizeof(unsigned long long),
                          hipMemcpyDeviceToHost, st), "flops d2h");
    GM_HIP(hipStreamSynchronize(st), "flops sync");
    *flops = (int64_t) hp[0];
    return GM_SUCCESS;
}

extern "C" bool gm_saxpy3_branch(const gm_csr *M, bool mask_comp, bool mask_struct,
                                 const gm_csr *A, const gm_csr *B, const gm_semiring *sr)
{
    (void) mask_comp;
    (void) mask_struct;
    if (!A || !B || !sr) return false;
    if (!semiring_supported(sr)) return false;
    if (!operand_ok(sr, A) || !operand_ok(sr, B)) return false;
    if (A->ncols != B->nrows) return false;
    if (M && (M->nrows != A->nrows || M->ncols != B->ncols)) return false;
    // column indices are hashed as 31-bit keys; row ids are 32-bit
    if (B->ncols >= (int64_t) 0x7fffffff || A->nrows >= ((int64_t) 1 << 32)) return false;
    return true;
}

extern "C" int gm_saxpy3(gm_csr_out *C, const gm_csr *M, bool mask_comp, bool mask_struct,
                         const gm_csr *A, const gm_csr *B, const gm_semiring *sr,
                         const gm_saxpy3_params *params)
{
    if (!C || !A || !B || !sr) return set_error(GM_INVALID_VALUE, "gm_saxpy3: NULL argument");
    if (!gm_saxpy3_branch(M, mask_comp, mask_struct, A, B, sr))
        return set_error(GM_NO_VALUE, "gm_saxpy3: case not handled by the GPU kernels");
    GM_TRY(ensure_init());
#define GM_SX_CASE(ADD, MULT, ZC, Z)                                                      \
    if (sr->add_op == ADD && sr->mult_op == MULT && sr->ztype == ZC)                      \
    {                                                                                     \
        int rc = saxpy3_run<SR<ADD, MULT, Z>>(C, M, mask_comp, mask_struct, A, B, params); \
        if (rc == GM_SUCCESS) C->type = ZC;                                               \
        return rc;                                                                        \
    }
    GM_SEMIRING_LIST(GM_SX_CASE)
#undef GM_SX_CASE
    return set_error(GM_NO_VALUE, "gm_saxpy3: semiring not instantiated");
}

//------------------------------------------------------------------------------
// derived forms of an operand (gm_csr_aux)
//------------------------------------------------------------------------------

extern "C" int gm_csr_aux_build(gm_csr_aux **aux, const gm_csr *X)
{
    if (!aux || !X) return set_error(GM_INVALID_VALUE, "gm_csr_aux_build: NULL argument");
    *aux = nullptr;
    // row records need 8-byte values, one per entry, and columns below 2^56
    if (!X->p || X->nrows <= 0 || !X->x || X->iso || type_size(X->type) != 8 ||
        X->ncols >= ((int64_t) 1 << 56))
        return GM_SUCCESS;
    GM_TRY(ensure_init());
    hipStream_t st = stream();
    DevBuf cnt;
    if (!cnt.alloc(8 * sizeof(unsigned long long))) return set_error(GM_OUT_OF_MEMORY, "aux: workspace");
    unsigned long long *hp = (unsigned long long *) pinned_scratch(8 * sizeof(unsigned long long));
    if (!hp) return set_error(GM_OUT_OF_MEMORY, "pinned scratch");
    k_sx_fill_u64<<<1, 64, 0, st>>>(cnt.as<unsigned long long>(), 8);
    k_sx_maxlen<<<sx_grid(X->nrows, SX_NT * 4, (int64_t) cu_count() * 4), SX_NT, 0, st>>>(
        X->p, X->nrows, X->p, 0, cnt.as<unsigned long long>());
    GM_HIP(hipGetLastError(), "aux: k_sx_maxlen");
    GM_HIP(hipMemcpyAsync(hp, cnt.ptr, 8 * sizeof(unsigned long long), hipMemcpyDeviceToHost, st),
           "aux: lengths");
    GM_HIP(hipStreamSynchronize(st), "aux: sync");
    const int64_t maxlen = (int64_t) hp[0], nnz = (int64_t) hp[2];
    int lg = 0;
    while (((int64_t) 1 << lg) < maxlen) lg++;
    if (nnz <= 0 || lg > SX_REC_MAX_LG || (X->nrows << lg) > nnz + nnz / 2 + 1024) return GM_SUCCESS;
    gm_csr_aux *a = (gm_csr_aux *) calloc(1, sizeof(gm_csr_aux));
    if (!a) return set_error(GM_OUT_OF_MEMORY, "aux: header");
    a->nrows = X->nrows;
    a->rec_lg = lg;
    a->rec = gm_malloc(sizeof(longlong2) * (size_t) (X->nrows << lg));
    if (!a->rec)
    {
        free(a);
        return set_error(GM_OUT_OF_MEMORY, "aux: row records");
    }
    k_sx_rec_build<<<sx_grid(X->nrows << lg, 256, (int64_t) cu_count() * 16), 256, 0, st>>>(
        X->p, X->j, (const int64_t *) X->x, X->nrows, lg, (longlong2 *) a->rec);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess)
    {
        gm_free(a->rec);
        free(a);
        return check_hip(e, "aux: k_sx_rec_build");
    }
    *aux = a;
    return GM_SUCCESS;
}

extern "C" void gm_csr_aux_free(gm_csr_aux *aux)
{
    if (!aux) return;
    gm_free(aux->rec);
    free(aux);
}
