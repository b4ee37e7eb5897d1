// Batched multi-source semiring SpMM (k sources as k dense columns, row-major n x k) for gfx950.
//
// Same merge-path tiles as the SpMV of g1/spmv_merge.hpp (same coordinates, kMergeThreads "virtual
// threads" of kMergeItems merge steps per tile); here each virtual thread is executed by a group of K
// lanes, lane j owning column j, so the K lanes walk the same steps in lockstep and load the K values of
// a source row with one coalesced access. A workgroup runs its tile's virtual threads in K rounds of
// G = 256/K. Every value a round needs from global memory (the x values of its nonzeros and, for the
// min-plus apply, the old values of the rows it closes) is loaded one round ahead into registers, with
// a fixed count of loads per round, so that the loads of round r+1 are in flight while round r walks.
//
// Fold order: a row's value is the fold, left to right, of the virtual threads' partial folds, exactly
// as in spmv_merge_tile_kernel: a closing virtual thread merges the tails since the last closing
// virtual thread (across rounds through the open carry), then its head; the tile's open row leaves as
// the tile carry. A batched plus-times column therefore equals the single-source SpMV of that column,
// bit for bit.
//
// Rows are finished by a policy (row_done) called together by the K lanes of a group, with the row's
// K column values; the policy fuses the engine's apply step. Rows that cross tiles are finished by the
// fixup kernel with the same policy.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "g1/device.hpp"
#include "g1/semiring.hpp"
#include "g1/spmv_merge.hpp"

namespace g1 {

constexpr int kSpmmMaxK = 64;

// Per-tile record of the SpMM: K carries and K deferred heads, then flags.
template <typename S, int K>
struct SpmmTileRec {
    typename S::acc_t carry[K];
    typename S::acc_t head[K];
    uint32_t flags;
};

template <typename S, int K>
inline size_t spmm_records_bytes(uint32_t n_rows, uint32_t nnz) {
    return static_cast<size_t>(merge_num_tiles(n_rows, nnz)) * sizeof(SpmmTileRec<S, K>);
}

// Lanes of the calling thread's K-lane group as a mask of the group's ballot bits.
template <int K>
__device__ __forceinline__ uint64_t group_bits(uint64_t wave_ballot) {
    if constexpr (K == 64) {
        return wave_ballot;
    } else {
        const uint32_t shift = (lane_id() / K) * K;
        return (wave_ballot >> shift) & ((1ull << K) - 1ull);
    }
}

template <typename S, int K, typename P>
__global__ void __launch_bounds__(256)
spmm_tile_kernel(uint32_t n_rows, uint32_t nnz, const uint32_t* __restrict__ row_offsets,
                 const uint32_t* __restrict__ col, const typename S::value_t* __restrict__ vals,
                 const MergeCoord* __restrict__ coords, SpmmTileRec<S, K>* __restrict__ recs, P pol,
                 unsigned long long* __restrict__ changed) {
    using acc_t = typename S::acc_t;
    using value_t = typename S::value_t;
    using x_t = typename S::x_t;
    using aux_t = typename P::aux_t;
    constexpr int G = 256 / K;                  // virtual threads per round
    constexpr int kRounds = kMergeThreads / G;  // = K: a quarter of the virtual threads is K / 4 rounds
    constexpr int kWavesG = kWave / K;          // groups per wave
    __shared__ uint32_t s_rowend[kMergeTile + 1];
    __shared__ uint32_t s_col[kMergeTile];
    __shared__ value_t s_w[kMergeTile];
    __shared__ aux_t s_aux[P::kHasAux ? kMergeTile : 1];
    __shared__ uint32_t s_vi[kMergeThreads + 1];  // first row (tile-relative) of each virtual thread
    __shared__ uint32_t s_vj[kMergeThreads + 1];  // first nonzero (tile-relative) of each virtual thread
    __shared__ acc_t s_tail[2][G][K];
    __shared__ acc_t s_carry[2][K];  // the open row since the quarter's start (a quarter: 64 virtual threads)
    __shared__ acc_t s_outer[2][K];  // ... and in the quarters before it
    __shared__ uint32_t s_hm[2][256 / kWave];  // closing groups of the round, one word per wave
    __shared__ unsigned long long s_or;

    const uint32_t tile = blockIdx.x;
    const uint32_t tid = threadIdx.x;
    const MergeCoord c0 = coords[tile];
    const MergeCoord c1 = coords[tile + 1];
    const uint32_t rows = c1.x - c0.x;
    const uint32_t nzs = c1.y - c0.y;
    const uint32_t total = rows + nzs;
    {
        uint32_t re[kMergeItems], ci[kMergeItems];
        value_t wv[kMergeItems];
#pragma unroll
        for (int r = 0; r < kMergeItems; ++r) {
            const uint32_t k = r * 256 + tid;
            if (k < rows) re[r] = row_offsets[c0.x + 1 + k];
            if (k < nzs) {
                ci[r] = col[c0.y + k];
                wv[r] = vals ? vals[c0.y + k] : value_t(1);
            }
        }
        if constexpr (P::kHasAux) {
            aux_t ax[kMergeItems];
#pragma unroll
            for (int r = 0; r < kMergeItems; ++r) {
                const uint32_t k = r * 256 + tid;
                if (k < nzs) ax[r] = pol.aux(ci[r]);
            }
#pragma unroll
            for (int r = 0; r < kMergeItems; ++r) {
                const uint32_t k = r * 256 + tid;
                if (k < nzs) s_aux[k] = ax[r];
            }
        }
#pragma unroll
        for (int r = 0; r < kMergeItems; ++r) {
            const uint32_t k = r * 256 + tid;
            if (k < rows) s_rowend[k] = re[r];
            if (k < nzs) {
                s_col[k] = ci[r];
                s_w[k] = wv[r];
            }
        }
        if (tid == 0) s_rowend[rows] = kInf;
    }
    __syncthreads();
    {
        // start coordinate of virtual thread tid (the SpMV thread's search)
        uint32_t d = tid * kMergeItems;
        if (d > total) d = total;
        uint32_t lo = d > nzs ? d - nzs : 0u;
        uint32_t hi = d < rows ? d : rows;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (static_cast<uint64_t>(s_rowend[mid]) + 1 <= static_cast<uint64_t>(c0.y) + (d - mid)) lo = mid + 1;
            else hi = mid;
        }
        s_vi[tid] = lo;
        s_vj[tid] = d - lo;
        if (tid == 0) {
            s_vi[kMergeThreads] = rows;
            s_vj[kMergeThreads] = nzs;
        }
        if (tid < static_cast<uint32_t>(K)) s_carry[0][tid] = s_outer[0][tid] = S::identity();
    }
    __syncthreads();

    const uint32_t j = tid % K;  // column of this lane
    const uint32_t g = tid / K;  // virtual thread slot within a round
    const uint32_t wave = tid / kWave;
    // The tile's first closed row is deferred to the fixup when it began in an earlier tile.
    const bool first_started_before = (rows > 0) && (row_offsets[c0.x] < c0.y);
    bool seen = false;     // some row closed in an earlier round
    bool seen_q = false;   // ... of this quarter
    uint64_t counted = 0;  // OR of the changed-column masks this lane's policy calls reported

    // Loads of round r: x values of its nonzeros, old values of the rows it closes (fixed count).
    auto fetch = [&](int r, x_t (&xs)[kMergeItems], x_t (&ds)[kMergeItems]) {
        const uint32_t vt = r * G + g;
        const uint32_t j0 = s_vj[vt], j1 = s_vj[vt + 1];
        const uint32_t i0 = s_vi[vt], i1 = s_vi[vt + 1];
#pragma unroll
        for (int t = 0; t < kMergeItems; ++t) {
            const bool has = j0 + t < j1;
            const uint32_t q = has ? j0 + t : 0u;
            const uint32_t u = has ? s_col[q] : 0u;
            xs[t] = pol.x(u, has ? s_aux[P::kHasAux ? q : 0u] : aux_t(0), j, has);
            if constexpr (P::kRowOld) {
                const bool hr = i0 + t < i1;
                ds[t] = pol.row_old(hr ? c0.x + i0 + t : 0u, j);
            }
        }
    };

    // One round: walk, then the closing virtual threads. xc/dc hold the round's loads.
    auto round = [&](int r, x_t (&xc)[kMergeItems], x_t (&dc)[kMergeItems]) {

        // ---- walk of virtual thread vt (the SpMV thread's loop, over this lane's column)
        const uint32_t vt = r * G + g;
        uint32_t d = vt * kMergeItems;
        if (d > total) d = total;
        uint32_t d_end = d + kMergeItems;
        if (d_end > total) d_end = total;
        uint32_t i = s_vi[vt];
        uint32_t jn = s_vj[vt];
        x_t p[kMergeItems];
#pragma unroll
        for (int t = 0; t < kMergeItems; ++t) {
            uint32_t q = jn + t;
            if (q >= static_cast<uint32_t>(kMergeTile)) q = kMergeTile - 1;
            p[t] = S::combine(s_w[q], xc[t]);
        }
        acc_t acc = S::identity();
        acc_t head = S::identity();
        bool hasend = false;
        uint32_t first_row = 0;
        x_t head_old = x_t(0);
        uint32_t re = s_rowend[i];
#pragma unroll
        for (int k = 0; k < kMergeItems; ++k) {
            if (d + k < d_end) {
                if (c0.y + jn < re) {
                    S::add(acc, p[0]);
#pragma unroll
                    for (int t = 0; t + 1 < kMergeItems; ++t) p[t] = p[t + 1];
                    ++jn;
                } else {
                    if (!hasend) {
                        head = acc;
                        hasend = true;
                        first_row = c0.x + i;
                        head_old = dc[0];
                    } else {
                        counted |= pol.row_done(c0.x + i, j, S::finalize(acc), dc[0]);
                    }
#pragma unroll
                    for (int t = 0; t + 1 < kMergeItems; ++t) dc[t] = dc[t + 1];
                    acc = S::identity();
                    ++i;
                    re = s_rowend[i];
                }
            }
        }
        const int par = r & 1;
        s_tail[par][g][j] = acc;
        {
            const uint64_t b = ballot(j == 0 && hasend);
            if (lane_id() == 0) {
                uint32_t hw = 0;
#pragma unroll
                for (int q = 0; q < kWavesG; ++q) hw |= static_cast<uint32_t>((b >> (q * K)) & 1ull) << q;
                s_hm[par][wave] = hw << (wave * kWavesG);
            }
        }
        __syncthreads();

        // ---- closing virtual threads: fold the tails since the last closer, then the head
        uint32_t hm = 0;
#pragma unroll
        for (int q = 0; q < 256 / kWave; ++q) hm |= s_hm[par][q];
        const acc_t open = s_carry[par][j];
        const acc_t outer = s_outer[par][j];
        if (hasend) {
            const uint32_t below = hm & ((g == 31) ? 0x7fffffffu : ((1u << g) - 1u));
            acc_t chain;
            uint32_t v0;
            if (below) {
                v0 = 31u - __clz(below);
                chain = S::identity();
            } else {
                v0 = 0;
                chain = open;
            }
            for (uint32_t v = v0; v < g; ++v) chain = S::merge(chain, s_tail[par][v][j]);
            acc_t whole = S::merge(chain, head);
            if (!below && !seen_q) whole = S::merge(outer, whole);  // the quarter's first closed row
            if (!below && !seen && first_started_before) {
                recs[tile].head[j] = whole;
            } else {
                counted |= pol.row_done(first_row, j, S::finalize(whole), head_old);
            }
        }
        const bool quarter_end = (r + 1) % (kRounds / 4) == 0;
        if (g == static_cast<uint32_t>(G - 1)) {
            acc_t c;
            uint32_t v0;
            if (hm) {
                v0 = 31u - __clz(hm);
                c = S::identity();
            } else {
                v0 = 0;
                c = open;
            }
            for (uint32_t v = v0; v < static_cast<uint32_t>(G); ++v) c = S::merge(c, s_tail[par][v][j]);
            acc_t o = outer;
            if (quarter_end) {
                o = (seen_q || hm != 0) ? S::merge(S::identity(), c) : S::merge(outer, c);
                c = S::identity();
            }
            s_carry[par ^ 1][j] = c;
            s_outer[par ^ 1][j] = o;
            if (r + 1 == kRounds) {
                recs[tile].carry[j] = o;
                if (j == 0) {
                    const bool any = seen || hm != 0;
                    uint32_t flags = any ? kTileHasEnd : 0u;
                    if (any && first_started_before) flags |= kTileDeferred;
                    recs[tile].flags = flags;
                }
            }
        }
        seen_q = !quarter_end && (seen_q || hm != 0);
        seen = seen || hm != 0;
    };

    // Two register buffers in turn (no copies, so the loads of the next round stay in flight while a
    // round walks); every fetch issues the same number of loads (the last ones repeat the final round).
    x_t xa[kMergeItems], da[kMergeItems], xb[kMergeItems], db[kMergeItems];
    fetch(0, xa, da);
    for (int r = 0; r < kRounds; r += 2) {
        fetch(r + 1, xb, db);
        round(r, xa, da);
        fetch(r + 2 < kRounds ? r + 2 : kRounds - 1, xa, da);
        round(r + 1, xb, db);
    }
    // Columns with a changed row: OR them into *changed, with an atomic only when this tile adds bits
    // that are not set yet (a device-wide word hit by every tile would serialize them).
    if (changed) {
        if (tid == 0) s_or = 0ull;
        __syncthreads();
        if (counted) atomicOr(&s_or, static_cast<unsigned long long>(counted));
        __syncthreads();
        if (tid == 0 && s_or) {
            const unsigned long long cur = *reinterpret_cast<volatile unsigned long long*>(changed);
            if (s_or & ~cur) atomicOr(changed, s_or);
        }
    }
}

// Min-plus variant of the tile kernel for order-free semirings (min is exact, so any fold order gives
// the same bits): group g of K lanes walks the contiguous run of K virtual threads g*K .. g*K+K-1 (8K
// merge items) alone, with its running minimum in registers and no workgroup barrier inside the walk;
// the loads of the next virtual thread are in flight while one walks (two register buffers). The
// group's first closed row and its open tail are combined across groups once, after one barrier,
// in group order. Tile records and the fixup are those of spmm_tile_kernel.
template <int K, typename P>
__global__ void __launch_bounds__(256)
spmm_minplus_kernel(uint32_t n_rows, uint32_t nnz, const uint32_t* __restrict__ row_offsets,
                    const uint32_t* __restrict__ col, const uint32_t* __restrict__ vals,
                    const MergeCoord* __restrict__ coords, SpmmTileRec<MinPlusU32, K>* __restrict__ recs, P pol,
                    unsigned long long* __restrict__ changed) {
    using S = MinPlusU32;
    using acc_t = S::acc_t;
    using aux_t = typename P::aux_t;
    constexpr int G = 256 / K;  // groups
    __shared__ uint32_t s_rowend[kMergeTile + 1];
    __shared__ uint32_t s_col[kMergeTile];
    __shared__ uint32_t s_w[kMergeTile];
    __shared__ aux_t s_aux[kMergeTile];
    __shared__ uint32_t s_vi[kMergeThreads + 1];
    __shared__ uint32_t s_vj[kMergeThreads + 1];
    __shared__ uint32_t s_ghead[G][K];
    __shared__ uint32_t s_gtail[G][K];
    __shared__ uint32_t s_gold[G][K];
    __shared__ uint32_t s_grow[G];
    __shared__ uint32_t s_gend[G];
    __shared__ unsigned long long s_or;

    const uint32_t tile = blockIdx.x;
    const uint32_t tid = threadIdx.x;
    const MergeCoord c0 = coords[tile];
    const MergeCoord c1 = coords[tile + 1];
    const uint32_t rows = c1.x - c0.x;
    const uint32_t nzs = c1.y - c0.y;
    const uint32_t total = rows + nzs;
    {
        uint32_t re[kMergeItems], ci[kMergeItems], wv[kMergeItems];
        aux_t ax[kMergeItems];
#pragma unroll
        for (int r = 0; r < kMergeItems; ++r) {
            const uint32_t k = r * 256 + tid;
            if (k < rows) re[r] = row_offsets[c0.x + 1 + k];
            if (k < nzs) {
                ci[r] = col[c0.y + k];
                wv[r] = vals ? vals[c0.y + k] : 1u;
            }
        }
#pragma unroll
        for (int r = 0; r < kMergeItems; ++r) {
            const uint32_t k = r * 256 + tid;
            if (k < nzs) ax[r] = pol.aux(ci[r]);
        }
#pragma unroll
        for (int r = 0; r < kMergeItems; ++r) {
            const uint32_t k = r * 256 + tid;
            if (k < rows) s_rowend[k] = re[r];
            if (k < nzs) {
                s_col[k] = ci[r];
                s_w[k] = wv[r];
                s_aux[k] = ax[r];
            }
        }
        if (tid == 0) {
            s_rowend[rows] = kInf;
            s_or = 0ull;
        }
    }
    __syncthreads();
    {
        uint32_t d = tid * kMergeItems;
        if (d > total) d = total;
        uint32_t lo = d > nzs ? d - nzs : 0u;
        uint32_t hi = d < rows ? d : rows;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (static_cast<uint64_t>(s_rowend[mid]) + 1 <= static_cast<uint64_t>(c0.y) + (d - mid)) lo = mid + 1;
            else hi = mid;
        }
        s_vi[tid] = lo;
        s_vj[tid] = d - lo;
        if (tid == 0) {
            s_vi[kMergeThreads] = rows;
            s_vj[kMergeThreads] = nzs;
        }
    }
    __syncthreads();

    const uint32_t j = tid % K;
    const uint32_t g = tid / K;
    uint64_t counted = 0;

    auto fetch = [&](uint32_t vt, uint32_t (&xs)[kMergeItems], uint32_t (&ds)[kMergeItems]) {
        const uint32_t j0 = s_vj[vt], j1 = s_vj[vt + 1];
        const uint32_t i0 = s_vi[vt], i1 = s_vi[vt + 1];
#pragma unroll
        for (int t = 0; t < kMergeItems; ++t) {
            const bool has = j0 + t < j1;
            const uint32_t q = has ? j0 + t : 0u;
            const uint32_t u = has ? s_col[q] : 0u;
            xs[t] = pol.x(u, has ? s_aux[q] : aux_t(0), j, has);
            const bool hr = i0 + t < i1;
            ds[t] = pol.row_old(hr ? c0.x + i0 + t : 0u, j);
        }
    };

    uint32_t acc = kInf;       // running minimum of the open row
    bool gend = false;         // the group closed a row
    uint32_t grow = 0, ghead = kInf, gold = 0;
    uint32_t i = s_vi[g * K];  // current row (tile-relative)
    uint32_t jn = s_vj[g * K];
    uint32_t re = s_rowend[i];
    auto walk = [&](uint32_t vt, uint32_t (&xc)[kMergeItems], uint32_t (&dc)[kMergeItems]) {
        uint32_t d = vt * kMergeItems;
        if (d > total) d = total;
        uint32_t d_end = d + kMergeItems;
        if (d_end > total) d_end = total;
        uint32_t p[kMergeItems];
#pragma unroll
        for (int t = 0; t < kMergeItems; ++t) {
            uint32_t q = jn + t;
            if (q >= static_cast<uint32_t>(kMergeTile)) q = kMergeTile - 1;
            p[t] = S::combine(s_w[q], xc[t]);
        }
#pragma unroll
        for (int k = 0; k < kMergeItems; ++k) {
            if (d + k < d_end) {
                if (c0.y + jn < re) {
                    acc = p[0] < acc ? p[0] : acc;
#pragma unroll
                    for (int t = 0; t + 1 < kMergeItems; ++t) p[t] = p[t + 1];
                    ++jn;
                } else {
                    if (!gend) {
                        gend = true;
                        grow = c0.x + i;
                        ghead = acc;
                        gold = dc[0];
                    } else {
                        counted |= pol.row_done(c0.x + i, j, acc, dc[0]);
                    }
#pragma unroll
                    for (int t = 0; t + 1 < kMergeItems; ++t) dc[t] = dc[t + 1];
                    acc = kInf;
                    ++i;
                    re = s_rowend[i];
                }
            }
        }
    };

    uint32_t xa[kMergeItems], da[kMergeItems], xb[kMergeItems], db[kMergeItems];
    const uint32_t v0 = g * K;
    fetch(v0, xa, da);
    for (uint32_t r = 0; r < static_cast<uint32_t>(K); r += 2) {
        fetch(v0 + r + 1, xb, db);
        walk(v0 + r, xa, da);
        fetch(v0 + (r + 2 < static_cast<uint32_t>(K) ? r + 2 : K - 1), xa, da);
        walk(v0 + r + 1, xb, db);
    }
    s_ghead[g][j] = ghead;
    s_gtail[g][j] = acc;
    s_gold[g][j] = gold;
    if (j == 0) {
        s_grow[g] = grow;
        s_gend[g] = gend ? 1u : 0u;
    }
    __syncthreads();
    // Groups in order (lanes of group 0): a group's first closed row gets the open minimum carried
    // from the groups before it; the tile's first closed row is deferred when it began before the tile.
    const bool first_started_before = (rows > 0) && (row_offsets[c0.x] < c0.y);
    if (g == 0) {
        uint32_t carry = kInf;
        bool seen = false;
        for (int q = 0; q < G; ++q) {
            if (s_gend[q]) {
                const uint32_t h = s_ghead[q][j];
                const uint32_t whole = h < carry ? h : carry;
                if (!seen && first_started_before) {
                    recs[tile].head[j] = acc_t{whole};
                } else {
                    counted |= pol.row_done(s_grow[q], j, whole, s_gold[q][j]);
                }
                seen = true;
                carry = s_gtail[q][j];
            } else {
                const uint32_t t = s_gtail[q][j];
                carry = t < carry ? t : carry;
            }
        }
        recs[tile].carry[j] = acc_t{carry};
        if (j == 0) {
            uint32_t flags = seen ? kTileHasEnd : 0u;
            if (seen && first_started_before) flags |= kTileDeferred;
            recs[tile].flags = flags;
        }
    }
    if (changed) {
        if (counted) atomicOr(&s_or, static_cast<unsigned long long>(counted));
        __syncthreads();
        if (tid == 0 && s_or) {
            const unsigned long long cur = *reinterpret_cast<volatile unsigned long long*>(changed);
            if (s_or & ~cur) atomicOr(changed, s_or);
        }
    }
}

// One group of K lanes per tile: finish the deferred first row of each tile (carries of the tiles it
// crosses, left to right, then the tile's head), as spmv_merge_fixup_kernel does per column.
template <typename S, int K, typename P>
__global__ void __launch_bounds__(256) spmm_fixup_kernel(uint32_t num_tiles, const MergeCoord* __restrict__ coords,
                                                        const SpmmTileRec<S, K>* __restrict__ recs, P pol,
                                                        unsigned long long* __restrict__ changed) {
    using acc_t = typename S::acc_t;
    const uint32_t t = (blockIdx.x * 256 + threadIdx.x) / K;
    const uint32_t j = threadIdx.x % K;
    const bool live = t < num_tiles && t > 0 && (recs[t].flags & kTileDeferred) != 0u;
    // Whole groups agree on `live` (t is uniform within a group), so row_done is called by full groups.
    if (!live) return;
    // The nearest tile u < t that closes a row (or tile 0): the group's K lanes test K tiles per step.
    uint32_t u = t - 1;
    for (;;) {
        const bool has_end = j <= u && (recs[u - j].flags & kTileHasEnd) != 0u;
        const uint64_t hits = group_bits<K>(ballot(has_end));
        if (hits) {
            u -= static_cast<uint32_t>(__builtin_ctzll(hits));
            break;
        }
        if (u < static_cast<uint32_t>(K)) {
            u = 0;
            break;
        }
        u -= K;
    }
    // Carries left to right (the fold order of spmv_merge_fixup_kernel), loaded eight at a time.
    acc_t acc = S::identity();
    uint32_t v = u;
    for (; v + 8 <= t; v += 8) {
        acc_t cv[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) cv[i] = recs[v + i].carry[j];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc = S::merge(acc, cv[i]);
    }
    for (; v < t; ++v) acc = S::merge(acc, recs[v].carry[j]);
    acc = S::merge(acc, recs[t].head[j]);
    const uint32_t row = coords[t].x;
    typename S::x_t old = typename S::x_t(0);
    if constexpr (P::kRowOld) old = pol.row_old(row, j);
    const uint64_t c = pol.row_done(row, j, S::finalize(acc), old);
    // Thousands of tiles may report changed columns; the shared word is only written with new bits.
    if (c && changed) {
        const unsigned long long cur = *reinterpret_cast<volatile unsigned long long*>(changed);
        if (c & ~cur) atomicOr(changed, static_cast<unsigned long long>(c));
    }
}

// ------------------------------------------------------------------------------------------------
// x rows that a wave of the 64-column kernels below keeps in flight.
constexpr uint32_t kWaveChunk = 16;
// Merge steps of a quarter of a merge tile: what a wave of spmv_merge_tile_kernel folds.
constexpr uint32_t kQuarter = kMergeTile / kMergeWaves;
static_assert(64 % kWaveChunk == 0, "a block of 64 indices holds whole chunks");

// The number of rows of [lo, hi) that end before merge step `diag`: row r does when row_offsets[r + 1] + r + 1 <=
// diag (merge_path_search with 64 rows tested at a time). Every lane of the wave calls it and gets lo plus that.
__device__ __forceinline__ uint32_t wave_merge_search(const uint32_t* __restrict__ row_offsets, uint32_t lo, uint32_t hi,
                                                      uint64_t diag) {
    const uint32_t lane = lane_id();
    while (lo < hi) {
        const uint32_t stride = (hi - lo + kWave - 1) / kWave;
        const uint32_t r = lo + lane * stride;
        const bool ended = lane * stride < hi - lo && static_cast<uint64_t>(row_offsets[r + 1]) + r + 1 <= diag;
        const uint32_t k = static_cast<uint32_t>(__popcll(ballot(ended)));  // the first k lanes
        if (k == 0) break;
        lo += (k - 1) * stride + 1;                  // row lo - 1 ended
        if (hi - lo >= stride) hi = lo + stride - 1;  // and row lo - 1 + stride, if tested, did not
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// Min-plus SpMM at k = 64: a workgroup of four waves takes a merge-path tile, a wave a quarter of its merge
// steps, lane j owns column j.
//
// A wave takes its merge steps (nonzeros and row ends, in merge order) 64 at a time, a lane each: the lane of a
// nonzero holds its source and weight, the lane of a row end holds the row. The steps that are row ends are one
// 64-bit mask: the ends of the next 64 rows, loaded a lane each, say which lanes they fall on. A source that
// did not change last iteration is replaced by row n, which is never reached, and so is a row none of whose
// nonzeros in the block can lower it; a block without any is stepped over. The distances of a nonzero's
// source and the old distances of a row end are then the same load of 64 columns, sixteen in flight while the
// sixteen before them fold: a nonzero adds its weight and takes the minimum, a row end (weight 0) compares the
// minimum with its old distances, stores what improved and starts the next row. So a step costs two reads of
// a lane, an address, an add and a minimum, and two scalar instructions; what bounds it is the 128 bytes of
// distances it loads, and where next to no source is active the chain from a block's row ends to its sources to
// their activity. Three blocks of that chain are under way at a time, a block's weights load when it turns out to have
// an active source, the quarters' starts come from a partition of their own, and with kMany (more tiles than the chip
// holds at once, built for eight waves a SIMD) a quarter whose first block is idle is looked over as a whole.
// Measured on 2.1 M vertices, 33 M edges, 16-bit distances: a dense iteration 1.25 -> 0.69 ms (6.6 TB/s of
// distance rows, the old ones with them), the batch 15.9 -> 9.2 ms, against a wave per tile that loaded 64
// sources' rows, folded them around a bitmap of row starts and then loaded the old rows of what it closed; with the
// above 8.3 ms, and an iteration with one active source 0.11 ms (0.18 before it, 0.26 the wave per tile), on as many
// edges between random vertices 0.12 (0.23, 0.16).
//
// Min is order-free, so the result does not depend on how rows are cut into tiles, quarters or blocks; rows that
// cross tiles leave head / carry records in the SpmmTileRec layout and are finished by spmm_fixup_kernel
// with MinPlusBatchPolicy<64>, as for the other min-plus kernels. Distances are updated in place (a
// source row read during the iteration may already hold this iteration's smaller value): each column
// still decreases monotonically to the same fixed point, and an iteration with no change ends the run.
// Every column of an active source is relaxed: a column whose distance did not change last iteration was
// relaxed through this edge when it last changed, so it cannot improve the row now, and the result (a fixed
// point of min) is the same.
//
// Distances are stored as DT: uint32_t, or int16_t when every finite distance of the run is below
// kCompactLimit (then a source row is one 128-byte line instead of two). 16-bit storage is exact or
// void: -1 is the unreached distance, so a sign-extending load yields G1_INF for it and the distance
// itself otherwise; a relaxation that would store a finite value >= kCompactLimit sets *overflow instead and
// counts as no change (the run then still ends, and the caller reruns the batch with 32-bit storage). With 16-bit
// storage the weight is added with unsigned saturation, which equals the semiring's combine because x + w cannot wrap (the caller only
// picks 16-bit storage when every weight is <= 0xFFFF0000).
constexpr uint32_t kCompactLimit = 0x7FFFu;

template <typename DT>
__device__ __forceinline__ uint32_t widen_dist(DT raw) {
    if constexpr (sizeof(DT) == 2) return static_cast<uint32_t>(static_cast<int32_t>(raw));
    return static_cast<uint32_t>(raw);
}

// act[v >> 5] bit (v & 31): mask[v] != 0 (the vertex changed in the last iteration); some[v >> 11] bit ((v >> 6) & 31):
// any of the 64 vertices of v's group did. A wave takes eight groups (16 words of act, a byte of some), their masks
// loaded together.
static __global__ void __launch_bounds__(256) act_bits_kernel(uint32_t n, const unsigned long long* __restrict__ mask,
                                                       uint32_t* __restrict__ act, uint8_t* __restrict__ some) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wi = blockIdx.x * 4u + threadIdx.x / 64u;
    const uint32_t v0 = wi * 512u;
    if (v0 >= n) return;
    unsigned long long c[8];
#pragma unroll
    for (uint32_t t = 0; t < 8; ++t) {
        const uint32_t v = v0 + t * 64u + lane;
        c[t] = mask[v < n ? v : n - 1];
    }
    uint32_t mine = 0;  // bit t: vertex `lane` of group t
#pragma unroll
    for (uint32_t t = 0; t < 8; ++t)
        if (c[t] != 0ull && v0 + t * 64u + lane < n) mine |= 1u << t;
    uint32_t word = 0, groups = 0;
#pragma unroll
    for (uint32_t t = 0; t < 8; ++t) {
        const uint64_t b = ballot((mine >> t) & 1u);
        if (lane / 2 == t) word = static_cast<uint32_t>(b >> (32 * (lane & 1u)));
        groups |= (b != 0ull ? 1u : 0u) << t;
    }
    if (lane < 16) act[wi * 16u + lane] = word;
    if (lane == 0) some[wi] = static_cast<uint8_t>(groups);
}

template <bool kWeighted, bool kMany, typename DT>
__global__ void __launch_bounds__(256, kMany ? 8 : 1)
spmm_minplus_wave_kernel(uint32_t n_rows, uint32_t num_quarters, const uint32_t* __restrict__ row_offsets,
                         const uint32_t* __restrict__ col, const uint32_t* __restrict__ vals,
                         const MergeCoord* __restrict__ quarters, SpmmTileRec<MinPlusU32, 64>* __restrict__ recs,
                         DT* __restrict__ D, const uint32_t* __restrict__ act_prev, const uint32_t* __restrict__ some_prev,
                         unsigned long long* __restrict__ mask_next, unsigned long long* __restrict__ changed,
                         uint32_t* __restrict__ overflow) {
    __shared__ uint32_t s_mark[kMergeWaves][64];
    __shared__ uint32_t s_carry[kMergeWaves][64];
    __shared__ uint32_t s_ends[kMergeWaves];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile = blockIdx.x;
    auto start = [&](uint32_t w) { return quarters[tile * kMergeWaves + w < num_quarters ? tile * kMergeWaves + w : num_quarters]; };
    const MergeCoord c0 = start(0), begin = start(wave), end = start(wave + 1);
    const uint32_t r0 = begin.x, r_last = end.x, q0 = begin.y;
    const uint32_t steps = r_last - r0 + (end.y - q0);
    const bool continued = r0 < r_last && row_offsets[r0] < q0;  // its first row end closes an earlier quarter's row

    uint32_t acc = kInf;   // running minimum of the open row
    uint32_t part = kInf;  // the continued row's, once closed
    uint64_t counted = 0;
    // Row r's distances become min(old, val); the columns that improved go to mask_next (cleared before the launch).
    auto apply = [&](uint32_t r, uint32_t val, uint32_t old) {
        bool improved = val < old;
        if (sizeof(DT) == 2 && improved && val >= kCompactLimit) {
            *overflow = 1u;
            improved = false;  // nothing is stored: a change reported here would be reported again for ever
        }
        if (improved) D[static_cast<size_t>(r) * 64 + lane] = static_cast<DT>(val);
        const uint64_t bits = ballot(improved);
        if (lane == 0 && bits) mask_next[r] = bits;
        counted |= bits;
    };
    auto dist = [&](uint32_t u) -> uint32_t {
        // 16-bit storage: 32-bit byte offsets, the caller keeps (n_rows + 1) * 128 below 2^32
        if constexpr (sizeof(DT) == 2)
            return widen_dist<DT>(*reinterpret_cast<const DT*>(reinterpret_cast<const char*>(D) + ((u << 7) + (lane << 1))));
        return D[static_cast<size_t>(u) * 64 + lane];
    };

    // One block of 64 merge steps from row i, nonzero j on: the row-end mask, and the lane's row (a row end) or source
    // (a nonzero; a lane past the last step is a nonzero that `live` leaves out).
    struct Block {
        uint64_t ends, live;
        uint32_t id;
    };
    uint32_t* mark = s_mark[wave];
    // the ends of the 64 rows from row i on, a lane each: they say which steps of the block are row ends
    auto load_ends = [&](uint32_t i) -> uint32_t { return i + lane < r_last ? row_offsets[i + 1 + lane] : kInf; };
    auto load_block = [&](uint32_t i, uint32_t j, uint32_t left, uint32_t end) -> Block {
        Block b;
        const uint32_t at = i + lane < r_last ? end - j + lane : 64u;  // the step its end falls on
        // (a wave's LDS operations run in program order, which the compiler must keep too)
        mark[lane] = 0u;
        asm volatile("" ::: "memory");
        if (at < 64) mark[at] = 1u;
        asm volatile("" ::: "memory");
        const bool is_end = mark[lane] != 0u;
        b.ends = ballot(is_end);
        const uint32_t before = mask_prefix(b.ends);
        b.live = ballot(lane < left && !is_end);
        b.id = i + before;
        if (lane < left && !is_end) b.id = __builtin_nontemporal_load(col + (j + lane - before));
        return b;
    };
    auto activity = [&](const Block& b) -> uint32_t { return (b.live >> lane) & 1ull ? act_prev[b.id >> 5] : 0u; };

    // Three blocks are under way: the one that folds, whose sources' activity is there or on its way; the next, whose
    // sources are; and the one after it, whose row ends are.
    uint64_t pending = 0;  // 1: the open row has an active nonzero in an earlier block
    uint32_t i = r0, j = q0;
    Block cur = load_block(i, j, steps, load_ends(i));
    uint32_t j_cur = j;
    auto pass = [&](const Block& b) {
        const uint32_t rows = static_cast<uint32_t>(__popcll(b.ends));
        i += rows;
        j += 64 - rows;
    };
    pass(cur);
    Block next{0, 0, 0};
    uint32_t j_next = j, ends2 = 0;
    if (steps > 64) {
        next = load_block(i, j, steps - 64, load_ends(i));
        pass(next);
        if (steps > 128) ends2 = load_ends(i);
    }
    uint32_t word = activity(cur);
    for (uint32_t s = 0; s < steps; s += 64) {
        Block next2{0, 0, 0};
        const uint32_t j_next2 = j;
        uint32_t next_word = 0;
        if (s + 128 < steps) {
            next2 = load_block(i, j, steps - s - 128, ends2);
            pass(next2);
            if (s + 192 < steps) ends2 = load_ends(i);
        }
        if (s + 64 < steps) next_word = activity(next);
        const uint64_t active = ballot((word >> (cur.id & 31u)) & 1u) & cur.live;
        // A row end needs its row when a nonzero since the row end before it is active (or the row is pending):
        // adding the active bits to the runs of ones between the row ends carries into exactly those.
        const uint64_t runs = ~cur.ends;
        const uint64_t sum = runs + active;
        const uint64_t all = sum + pending;
        const uint64_t need = all & cur.ends;
        pending = (sum < runs ? 1u : 0u) | (all < sum ? 1u : 0u);
        const bool idle = (active | need) == 0ull;
        const uint32_t id = ((active | need) >> lane) & 1ull ? cur.id : n_rows;
        if (kMany && idle && s == 0 && steps > 128) {
            // Where the first block is idle, the rest mostly is: the sources past the next block are looked at without
            // their row ends, by their groups' activity first (a table that the L1 holds), and a quarter without an
            // active one is done.
            bool hit = ((next_word >> (next.id & 31u)) & 1u) != 0u;
            const uint32_t left = end.y - j_next2;
            for (uint32_t q = 0; q < left; q += 8 * 64) {
                uint32_t id[8], group[8];
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k) {
                    const uint32_t at = q + k * 64 + lane;
                    id[k] = at < left ? __builtin_nontemporal_load(col + j_next2 + at) : 0u;
                }
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k) group[k] = q + k * 64 + lane < left ? some_prev[id[k] >> 11] : 0u;
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k)
                    if ((group[k] >> ((id[k] >> 6) & 31u)) & 1u) hit |= ((act_prev[id[k] >> 5] >> (id[k] & 31u)) & 1u) != 0u;
            }
            if (ballot(hit) == 0ull) break;
        }
        if (!idle) {
            uint32_t w = 1;  // (a row end's: 0)
            if (kWeighted) w = (active >> lane) & 1ull ? __builtin_nontemporal_load(vals + (j_cur + lane - mask_prefix(cur.ends))) : 0u;
            else if ((cur.ends >> lane) & 1ull) w = 0;
            uint32_t x[kWaveChunk];
#pragma unroll
            for (uint32_t t = 0; t < kWaveChunk; ++t) x[t] = dist(__builtin_amdgcn_readlane(id, t));
            for (uint32_t c = 0; c < 64; c += kWaveChunk) {
                uint32_t p[kWaveChunk];
#pragma unroll
                for (uint32_t t = 0; t < kWaveChunk; ++t) {
                    const uint32_t wt = __builtin_amdgcn_readlane(w, c + t);
                    p[t] = sizeof(DT) == 2 ? __builtin_elementwise_add_sat(x[t], wt) : MinPlusU32::combine(wt, x[t]);
                }
                if (c + kWaveChunk < 64) {
#pragma unroll
                    for (uint32_t t = 0; t < kWaveChunk; ++t) x[t] = dist(__builtin_amdgcn_readlane(id, c + kWaveChunk + t));
                }
                const uint32_t ends = static_cast<uint32_t>(need >> c);
#pragma unroll
                for (uint32_t t = 0; t < kWaveChunk; ++t) {
                    if ((ends >> t) & 1u) {
                        const uint32_t r = __builtin_amdgcn_readlane(id, c + t);
                        if (continued && r == r0) part = acc;
                        else apply(r, acc, p[t]);
                        acc = kInf;
                    } else {
                        acc = p[t] < acc ? p[t] : acc;
                    }
                }
            }
        }
        cur = next;
        next = next2;
        j_cur = j_next;
        j_next = j_next2;
        word = next_word;
    }

    s_carry[wave][lane] = acc;
    if (lane == 0) s_ends[wave] = r_last > r0;
    __syncthreads();
    // The minimum of the quarters' open rows before w since the last one that closed a row.
    auto outer = [&](int w, bool& any) {
        int u = w - 1;
        while (u > 0 && !s_ends[u]) --u;
        any = u >= 0 && s_ends[u] != 0u;
        uint32_t m = kInf;
        for (int v = u > 0 ? u : 0; v < w; ++v) m = s_carry[v][lane] < m ? s_carry[v][lane] : m;
        return m;
    };
    bool before;
    if (continued) {
        const uint32_t o = outer(static_cast<int>(wave), before);
        const uint32_t whole = part < o ? part : o;
        if (!before && row_offsets[r0] < c0.y) recs[tile].head[lane] = MinPlusU32::acc_t{whole};
        else if (ballot(whole != kInf)) apply(r0, whole, dist(r0));
    }
    if (wave == kMergeWaves - 1) {
        recs[tile].carry[lane] = MinPlusU32::acc_t{outer(kMergeWaves, before)};
        if (lane == 0) recs[tile].flags = (before ? kTileHasEnd : 0u) | (before && row_offsets[c0.x] < c0.y ? kTileDeferred : 0u);
    }
    if (counted && lane == 0) {
        const unsigned long long seen = *reinterpret_cast<volatile unsigned long long*>(changed);
        if (counted & ~seen) atomicOr(changed, static_cast<unsigned long long>(counted));
    }
}

// ------------------------------------------------------------------------------------------------
// Batched SSSP / BFS (min-plus). Per vertex: D[v*K + j] the distance of column j, and a mask of the
// columns whose distance changed in the last iteration (mask_prev[v] bit j). A source contributes to
// column j only when that bit is set, so inactive sources cost one 8-byte mask read per nonzero. The
// row's owner applies the result: d = min(D, y); changed bits go to mask_next[v] (written once per row
// per iteration, so the masks need no atomics and no clearing). The columns that changed are ORed into a
// per-iteration word, so each column's convergence is known.
template <int K>
struct MinPlusBatchPolicy {
    using aux_t = unsigned long long;
    static constexpr bool kHasAux = true;   // the source's change mask, staged per nonzero
    static constexpr bool kRowOld = true;   // the apply needs the row's old distance
    uint32_t* D;
    const unsigned long long* mask_prev;
    unsigned long long* mask_next;
    __device__ __forceinline__ aux_t aux(uint32_t u) const { return mask_prev[u]; }
    // Always one load (a resident dummy row for inactive entries) so every round issues the same count.
    __device__ __forceinline__ uint32_t x(uint32_t u, aux_t m, uint32_t j, bool has) const {
        const bool on = has && ((m >> j) & 1ull);
        const uint32_t v = D[on ? static_cast<size_t>(u) * K + j : j];
        return on ? v : kInf;
    }
    __device__ __forceinline__ uint32_t row_old(uint32_t row, uint32_t j) const {
        return D[static_cast<size_t>(row) * K + j];
    }
    // Called by the K lanes of a group together (lane j = column j); returns 1 on lane 0 of the group
    // with the columns of the row that changed (0 on the other lanes).
    __device__ __forceinline__ uint64_t row_done(uint32_t row, uint32_t j, uint32_t y, uint32_t old) const {
        const bool improved = y < old;
        if (improved) D[static_cast<size_t>(row) * K + j] = y;
        const uint64_t bits = group_bits<K>(ballot(improved));
        if (j == 0) mask_next[row] = bits;
        return (j == 0) ? bits : 0ull;
    }
};

// The fixup side of spmm_minplus_wave_kernel with 16-bit distance storage (row_old / row_done only).
struct MinPlusBatchPolicy16 {
    using aux_t = unsigned long long;
    static constexpr bool kHasAux = true;
    static constexpr bool kRowOld = true;
    int16_t* D;
    const unsigned long long* mask_prev;
    unsigned long long* mask_next;
    uint32_t* overflow;
    __device__ __forceinline__ uint32_t row_old(uint32_t row, uint32_t j) const {
        return widen_dist<int16_t>(D[static_cast<size_t>(row) * 64 + j]);
    }
    __device__ __forceinline__ uint64_t row_done(uint32_t row, uint32_t j, uint32_t y, uint32_t old) const {
        bool improved = y < old;
        if (improved && y >= kCompactLimit) {
            *overflow = 1u;
            improved = false;  // as in the kernel
        }
        if (improved) D[static_cast<size_t>(row) * 64 + j] = static_cast<int16_t>(y);
        const uint64_t bits = ballot(improved);
        if (j == 0) mask_next[row] = bits;
        return (j == 0) ? bits : 0ull;
    }
};

// Batched plus-times: writes y row-major; the PageRank-style apply runs as its own kernel.
template <int K>
struct PlusTimesBatchPolicy {
    using aux_t = uint32_t;
    static constexpr bool kHasAux = false;
    static constexpr bool kRowOld = false;
    const float* X;
    float* Y;
    static constexpr bool kScale = false;
    __device__ __forceinline__ void init(uint32_t) {}
    template <bool kWide>
    __device__ __forceinline__ float x(uint32_t u, uint32_t j) const {
        if constexpr (kWide) return X[static_cast<size_t>(u) * K + j];
        return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(X) + (u * (K * 4u) + j * 4u));
    }
    __device__ __forceinline__ void store(uint32_t row, uint32_t j, float y) const {
        Y[static_cast<size_t>(row) * K + j] = y;
    }
    __device__ __forceinline__ aux_t aux(uint32_t) const { return 0u; }
    __device__ __forceinline__ float x(uint32_t u, aux_t, uint32_t j, bool) const {
        return X[static_cast<size_t>(u) * K + j];
    }
    __device__ __forceinline__ float row_old(uint32_t, uint32_t) const { return 0.0f; }
    __device__ __forceinline__ uint64_t row_done(uint32_t row, uint32_t j, float y, float) const {
        Y[static_cast<size_t>(row) * K + j] = y;
        return 0ull;
    }
};

// ------------------------------------------------------------------------------------------------
// One iteration of batched personalized PageRank over 64 columns without x and y arrays: a source's x is its old
// rank times its out-weight's inverse (the product rank_apply_batch_kernel would have stored, so the same bits),
// and a row's sum goes straight to its new rank. Columns in state[0] (converged, or padding) are not stored:
// rank_delta_batch_kernel carries their ranks over. Saves y written and read and x written, 12 of 20 bytes an element
// beside the gathers, for a multiplication a nonzero and its source's scale (which streams beside the weights on
// large graphs, see scales_stream in batch.hip): 0.7 M vertices x 64 columns 0.38 (product) + 0.17 ms (apply) an
// iteration before, 0.40 + 0.06 (L1 partials) here. Small graphs keep the two (ppr_fused).
struct RankBatchPolicy {
    using aux_t = uint32_t;
    static constexpr bool kHasAux = false;
    static constexpr bool kRowOld = false;
    static constexpr bool kScale = true;
    const float* R_old;
    float* R_new;
    const float* iw;
    const float* iw_nz;  // iw of each nonzero's source, in the nonzeros' order (null: gathered from iw)
    const uint32_t* seeds;
    float base_seed;
    const unsigned long long* state;
    uint32_t seed = 0;
    bool running = false;
    __device__ __forceinline__ void init(uint32_t j) {
        seed = seeds[j];
        running = !((state[0] >> j) & 1ull);
    }
    template <bool kWide>
    __device__ __forceinline__ float x(uint32_t u, uint32_t j) const {
        if constexpr (kWide) return R_old[static_cast<size_t>(u) * 64 + j];
        return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(R_old) + (u * 256u + j * 4u));
    }
    __device__ __forceinline__ bool scale_streams() const { return iw_nz != nullptr; }
    __device__ __forceinline__ float scale_at(uint32_t e) const { return __builtin_nontemporal_load(iw_nz + e); }
    __device__ __forceinline__ float scale(uint32_t u) const { return iw[u]; }
    __device__ __forceinline__ void store(uint32_t row, uint32_t j, float y) const {
        const float rn = (row == seed ? base_seed : 0.0f) + y;
        if (running) R_new[static_cast<size_t>(row) * 64 + j] = rn;
    }
    __device__ __forceinline__ uint64_t row_done(uint32_t row, uint32_t j, float y, float) {
        init(j);
        store(row, j, y);
        return 0ull;
    }
};

// SpMM over 64 columns: a workgroup of four waves takes a merge-path tile, a wave a quarter of its merge
// steps, lane j = column j, the walk on the scalar unit. It reproduces the fold of spmv_merge_tile_kernel
// exactly, per column: a quarter's 512 steps are cut into the same 64 runs of 8 that the threads of one of
// its waves take; inside a run a row's products are added left to right; a run that closes a row finishes
// its first closed row by merging, left to right, the tails of the runs since the last run that closed a
// row and then its own head; the quarters' carries are merged in front of the first row a quarter closes,
// the tile's open row leaves as the carry, a first row that began before the tile as the deferred head
// (finished by spmm_fixup_kernel). Batched personalized PageRank columns therefore stay bit-identical to the
// single-source runs.
//
// Quarters, because a wave per tile left too few waves: 11 M rows and nonzeros are 5,300 tiles for 8,192
// resident waves, and each wave's chain of loads is then as long as the launch. Where quarters are too few as well
// (small matrices, see spmm_split in step.hip) a workgroup of kParts waves takes one quarter: the order of the sums is
// that of the quarter's 64 runs, so a wave keeps the tails of its runs in LDS up to the first that closes a row, and
// what a row holds in the waves before it is folded in front of them once all are done (32 KB of LDS at eight waves
// of eight runs, 32 waves a CU). The records are then the quarters', and spmm_quarter_fixup_kernel folds them.
//
// What bounds it is the x rows, 256 bytes per nonzero, as long as the walk keeps out of their way; the walk is
// one wave-uniform stream, so its scalar instructions are what it is made of. The x rows go to registers
// kWaveChunk at a time: a chunk's products are formed from the rows loaded during the chunk before, the next
// chunk's loads are issued, and the products are folded while those fly. The fold is unrolled over the chunk
// and its next event (a row's end or a run's end, whichever comes first) is kept as a position in the chunk,
// so a nonzero without an event costs a compare, a branch and its add; a source's row is a 32-bit offset
// (kWide: 64-bit, for x arrays of 4 GB and more), one vector instruction. Column indices and values come 64 at
// a time, a block ahead, and are read out of their lanes. Measured: 16 M nonzeros x 64 columns
// 1.03 ms with the round-based tile kernel, 0.66 ms here (6.5 TB/s of x rows; 0.88 ms with a wave per tile, 0.85 ms
// with the run counter and the 64-bit row addresses on the scalar unit as well, 19 scalar instructions a
// nonzero against 8); 11 M nonzeros of a PPR batch 0.72 ms with x parked in LDS and a wave per tile, 0.38 ms.

// P: init(lane) once per wave; x<kWide>(u, lane) the lane's value of source u, loaded unconditionally (a
// column the policy leaves out may read any valid element: its products are never stored), times scale(u) where
// kScale says so (scale_at(e) of nonzero e instead where scale_streams() does, uniform); store(row, lane, y).
template <typename S, bool kValues, bool kWide, uint32_t kParts, typename P>
__global__ void __launch_bounds__(kParts == 1 ? 256 : kParts * kWave)
spmm_wave_kernel(uint32_t n_rows, uint32_t nnz, bool find, const uint32_t* __restrict__ row_offsets,
                 const uint32_t* __restrict__ col, const typename S::value_t* __restrict__ vals,
                 MergeCoord* __restrict__ coords, SpmmTileRec<S, 64>* __restrict__ recs, P pol) {
    using acc_t = typename S::acc_t;
    using value_t = typename S::value_t;
    using x_t = typename S::x_t;
    using y_t = typename S::y_t;
    static_assert(sizeof(value_t) == 4, "values travel through readlane");
    constexpr bool kSplit = kParts > 1;
    constexpr uint32_t kWaves = kSplit ? kParts : kMergeWaves;
    constexpr uint32_t kSteps = kQuarter / kParts;      // merge steps of a wave
    constexpr uint32_t kRuns = kSteps / kMergeItems;
    constexpr uint64_t kTileSteps = kWaves * kSteps;
    __shared__ acc_t s_carry[kWaves][64];
    __shared__ acc_t s_tail[kSplit ? kWaves : 1][kSplit ? kRuns : 1][64];  // the runs before the first that closes a row
    __shared__ uint32_t s_tails[kWaves];                                   // ... and their number
    __shared__ uint32_t s_ends[kWaves];
    __shared__ uint32_t s_row[kWaves + 1];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile = blockIdx.x;
    pol.init(lane);

    // The waves' bounds: the merge-path search of the wave's first step, 64 rows at a time, within the tile's rows
    // or, when the caller has no partition, in all of them (the tile's start then goes to coords for the fixup).
    MergeCoord c0{0, 0}, c1{n_rows, nnz};
    const uint64_t total = static_cast<uint64_t>(n_rows) + nnz;
    const uint64_t step0 = tile * kTileSteps;
    const uint64_t step1 = step0 + kTileSteps < total ? step0 + kTileSteps : total;
    auto part_start = [&](uint32_t w) { return step0 + w * kSteps < step1 ? step0 + w * kSteps : step1; };
    if (!find) {
        c0 = coords[tile];
        c1 = coords[tile + 1];
    }
    const uint32_t first = wave_merge_search(row_offsets, c0.x, c1.x, part_start(wave));
    if (find && wave == kWaves - 1) c1.x = wave_merge_search(row_offsets, first, n_rows, step1);
    if (lane == 0) {
        s_row[wave] = first;
        if (wave == kWaves - 1) s_row[kWaves] = c1.x;
    }
    __syncthreads();
    if (find) {
        c0.x = __builtin_amdgcn_readfirstlane(s_row[0]);
        c0.y = static_cast<uint32_t>(step0 - c0.x);
        if (threadIdx.x == 0) {
            coords[tile] = c0;
            if (tile == gridDim.x - 1) coords[tile + 1] = MergeCoord{n_rows, nnz};
        }
    }
    const uint32_t r0 = first, r_last = __builtin_amdgcn_readfirstlane(s_row[wave + 1]);
    // Nonzeros are counted from `base` on, the block of 64 that holds the wave's first one, so that no sum of a
    // position and a chunk or a run passes 32 bits, however many nonzeros the matrix has (up to 2^32 - 2).
    const uint32_t first_nz = static_cast<uint32_t>(part_start(wave) - r0);
    const uint32_t base = first_nz & ~63u;
    col += base;
    if (kValues) vals += base;
    const uint32_t q0 = first_nz - base, q1 = static_cast<uint32_t>(part_start(wave + 1) - r_last) - base;

    // row ends of 64 consecutive rows, one per lane, read out with readlane
    uint32_t rbase = r0;
    uint32_t rwin = row_offsets[lane < n_rows - rbase ? rbase + 1 + lane : n_rows] - base;
    auto row_end = [&](uint32_t r) -> uint32_t {
        if (r - rbase >= 64u) {
            rbase = r;
            rwin = row_offsets[lane < n_rows - rbase ? rbase + 1 + lane : n_rows] - base;
        }
        return __builtin_amdgcn_readlane(rwin, r - rbase);
    };

    uint32_t r = r0;                                 // next row to close
    uint32_t re = r0 < r_last ? row_end(r0) : kInf;  // its end (kInf: no further row end in the tile)
    // The nonzero before which the run ends unless a row closes first (each row closed is a step too).
    uint32_t run = q0 + kMergeItems;
    acc_t acc = S::identity(), head = S::identity(), chain = S::identity();
    bool hasend = false, any_end = false;
    uint32_t first_row = 0;

    acc_t part = S::identity();  // the first row the wave closes, as far as the wave (kSplit: its run) holds it
    uint32_t part_row = 0;
    uint32_t tails = 0;

    // End of a run of 8 steps (the same folds as merge_walk's, per column). What is folded in front of a split
    // quarter's first closed row waits in LDS until the waves before this one are done.
    auto run_end = [&]() {
        if (hasend) {
            if (any_end) {
                pol.store(first_row, lane, S::finalize(S::merge(chain, head)));
            } else {
                part = kSplit ? head : S::merge(chain, head);
                part_row = first_row;
            }
            chain = acc;
            any_end = true;
            hasend = false;
        } else if (!kSplit || any_end) {
            chain = S::merge(chain, acc);
        } else if (tails < kRuns) {  // (a run past the last step holds nothing)
            s_tail[kSplit ? wave : 0][kSplit ? tails : 0][lane] = acc;
            ++tails;
        }
        acc = S::identity();
    };
    // Every run and row that ends before nonzero q is added.
    auto events = [&](uint32_t q) {
        if (run == q) {
            run_end();
            run = q + kMergeItems;
        }
        while (re <= q) {
            if (!hasend) {
                head = acc;
                hasend = true;
                first_row = r;
            } else {
                pol.store(r, lane, S::finalize(acc));
            }
            acc = S::identity();
            ++r;
            re = r < r_last ? row_end(r) : kInf;
            if (--run == q) {
                run_end();
                run = q + kMergeItems;
            }
        }
    };

    if (q0 < q1) {
        constexpr uint32_t kPer = 64 / kWaveChunk;  // chunks per block of indices
        const uint32_t c_end = (q1 + kWaveChunk - 1) / kWaveChunk;
        uint32_t c = q0 / kWaveChunk;
        // a lane outside the tile's nonzeros holds source 0 (never folded)
        uint32_t sB = 0;  // the scales of the block loaded last, if they stream
        auto load_block = [&](uint32_t b, uint32_t& cv, uint32_t& wv) {
            const uint32_t q = b * 64u + lane;
            cv = 0;
            wv = 0;
            if constexpr (P::kScale) sB = 0;
            if (q >= q0 && q < q1) {
                cv = __builtin_nontemporal_load(col + q);
                if (kValues) wv = __builtin_bit_cast(uint32_t, __builtin_nontemporal_load(vals + q));
                if constexpr (P::kScale) {
                    if (pol.scale_streams()) sB = __builtin_bit_cast(uint32_t, pol.scale_at(base + q));
                }
            }
        };
        // the scales of the block whose sources are cv: s if they stream
        auto scales = [&](uint32_t cv, uint32_t s) {
            if constexpr (P::kScale) {
                if (!pol.scale_streams()) s = __builtin_bit_cast(uint32_t, pol.scale(cv));
            }
            return s;
        };
        x_t xn[kWaveChunk];
        auto load_x = [&](uint32_t cv, uint32_t at) {
#pragma unroll
            for (uint32_t t = 0; t < kWaveChunk; ++t)
                xn[t] = pol.template x<kWide>(__builtin_amdgcn_readlane(cv, at + t), lane);
        };
        uint32_t cA, wA, cB, wB;
        load_block(c / kPer, cA, wA);
        uint32_t sA = scales(cA, sB);  // the block's scales, a lane each
        load_block(c / kPer + 1, cB, wB);
        load_x(cA, (c % kPer) * kWaveChunk);
        for (; c < c_end; ++c) {
            const uint32_t at = (c % kPer) * kWaveChunk;
            y_t p[kWaveChunk];
#pragma unroll
            for (uint32_t t = 0; t < kWaveChunk; ++t) {
                value_t w = value_t(1);
                if (kValues) w = __builtin_bit_cast(value_t, static_cast<uint32_t>(__builtin_amdgcn_readlane(wA, at + t)));
                x_t x = xn[t];
                if constexpr (P::kScale) x *= __builtin_bit_cast(float, static_cast<uint32_t>(__builtin_amdgcn_readlane(sA, at + t)));
                p[t] = S::combine(w, x);
            }
            if (at + kWaveChunk == 64u) {
                cA = cB;
                wA = wB;
                sA = scales(cA, sB);
                load_x(cA, 0);
                load_block((c + 1) / kPer + 1, cB, wB);
            } else {
                load_x(cA, at + kWaveChunk);  // past the tile's end: source 0's row, unused
            }
            const uint32_t qc = c * kWaveChunk;
            if (qc < q0 || q1 - qc < kWaveChunk) {
                // the tile's first or last chunk: products outside the tile fold as nothing
                const uint32_t ta = q0 > qc ? q0 - qc : 0u;
#pragma unroll
                for (uint32_t t = 0; t < kWaveChunk; ++t)
                    if (t < ta || qc + t >= q1) p[t] = S::nothing();
            }
            // next: the position of the first event in the chunk (none before q0; past q1 only ends of runs that
            // add nothing)
            auto upcoming = [&]() { return (re < run ? re : run) - qc; };
            uint32_t next = upcoming();
#pragma unroll
            for (uint32_t t = 0; t < kWaveChunk; ++t) {
                if (next <= t) {
                    events(qc + t);
                    next = upcoming();
                }
                S::add(acc, p[t]);
            }
        }
    }
    events(q1);  // the rows left end at q1
    run_end();

    s_carry[wave][lane] = chain;
    if (lane == 0) {
        s_ends[wave] = any_end;
        s_tails[wave] = tails;
    }
    __syncthreads();
    // The fold in front of wave w since the last wave before it that closed a row: the quarters' carries
    // (merge_wave_chain), or in a split quarter that wave's carry and the tails of the runs after it.
    auto outer = [&](int w, bool& any) {
        int u = w - 1;
        while (u > 0 && !s_ends[u]) --u;
        any = u >= 0 && s_ends[u] != 0u;
        acc_t sum = S::identity();
        int v = u > 0 ? u : 0;
        if constexpr (kSplit) {
            if (any) sum = s_carry[v++][lane];
            for (; v < w; ++v)
                for (uint32_t k = 0; k < s_tails[v]; ++k) sum = S::merge(sum, s_tail[v][k][lane]);
        } else {
            for (; v < w; ++v) sum = S::merge(sum, s_carry[v][lane]);
        }
        return sum;
    };
    bool before;
    if (any_end) {
        acc_t chain = outer(static_cast<int>(wave), before);
        if constexpr (kSplit)
            for (uint32_t k = 0; k < tails; ++k) chain = S::merge(chain, s_tail[wave][k][lane]);
        const acc_t whole = S::merge(chain, part);
        if (!before && row_offsets[part_row] < c0.y) recs[tile].head[lane] = whole;
        else pol.store(part_row, lane, S::finalize(whole));
    }
    if (wave == kWaves - 1) {
        recs[tile].carry[lane] = outer(kWaves, before);
        if (lane == 0) {
            uint32_t flags = before ? kTileHasEnd : 0u;
            if (before && row_offsets[c0.x] < c0.y) flags |= kTileDeferred;
            recs[tile].flags = flags;
        }
    }
}

// spmm_fixup_kernel for records of quarters: a wave per quarter finishes its deferred first row. The carries of
// the quarters that the row crosses are folded tile by tile, and the tiles' sums left to right in front of the
// last tile's, as the merge kernels fold them.
template <typename S, typename P>
__global__ void __launch_bounds__(256) spmm_quarter_fixup_kernel(uint32_t quarters, const MergeCoord* __restrict__ coords,
                                                                 const SpmmTileRec<S, 64>* __restrict__ recs, P pol) {
    using acc_t = typename S::acc_t;
    const uint32_t t = (blockIdx.x * 256 + threadIdx.x) / 64;
    const uint32_t j = threadIdx.x % 64;
    if (t == 0 || t >= quarters || (recs[t].flags & kTileDeferred) == 0u) return;
    uint32_t u = t - 1;  // the nearest quarter before t that closes a row, or the first: 64 tested at a time
    for (;;) {
        const uint64_t hits = ballot(j <= u && (recs[u - (j <= u ? j : 0u)].flags & kTileHasEnd) != 0u);
        if (hits) {
            u -= static_cast<uint32_t>(__builtin_ctzll(hits));
            break;
        }
        if (u < 64) {
            u = 0;
            break;
        }
        u -= 64;
    }
    acc_t tiles = S::identity(), tile = S::identity();
    bool crossed = false;
    auto add = [&](uint32_t v, acc_t carry) {
        tile = S::merge(tile, carry);
        if (v % kMergeWaves == kMergeWaves - 1) {
            tiles = S::merge(tiles, tile);
            tile = S::identity();
            crossed = true;
        }
    };
    uint32_t v = u;
    for (; v + 8 <= t; v += 8) {
        acc_t cv[8];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) cv[i] = recs[v + i].carry[j];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) add(v + i, cv[i]);
    }
    for (; v < t; ++v) add(v, recs[v].carry[j]);
    const acc_t last = S::merge(tile, recs[t].head[j]);
    pol.row_done(coords[t].x, j, S::finalize(crossed ? S::merge(tiles, last) : last), typename S::x_t(0));
}

// One pass of the wave kernel, over tiles of kMergeTile steps or (kParts > 1) quarters of them; x_bytes is the size of
// the x array the policy reads. With `find` the waves search the whole matrix for their bounds and leave the tiles'
// (quarters') starts in coords, otherwise coords holds the partition.
template <typename S, uint32_t kParts = 1, typename P>
inline void launch_spmm_wave(uint32_t n_rows, uint32_t nnz, bool find, const uint32_t* row_off, const uint32_t* col,
                             const typename S::value_t* vals, MergeCoord* coords, SpmmTileRec<S, 64>* recs, const P& pol,
                             uint64_t x_bytes, hipStream_t s) {
    const bool wide = x_bytes >= (1ull << 32);
    constexpr bool kSplit = kParts > 1;
    const uint32_t blocks = merge_num_tiles_for(n_rows, nnz, kSplit ? kQuarter : kMergeTile);
    auto go = [&](auto kernel) {
        kernel<<<blocks, kSplit ? kParts * kWave : 256, 0, s>>>(n_rows, nnz, find, row_off, col, vals, coords, recs, pol);
    };
    if (vals) {
        if (wide) go(spmm_wave_kernel<S, true, true, kParts, P>);
        else go(spmm_wave_kernel<S, true, false, kParts, P>);
    } else {
        if (wide) go(spmm_wave_kernel<S, false, true, kParts, P>);
        else go(spmm_wave_kernel<S, false, false, kParts, P>);
    }
}

}  // namespace g1
