// Whole queries on high-diameter, low-degree graphs (road networks, grids): one workgroup of 1024
// threads runs one single-source BFS or SSSP from start to end, with workgroup barriers between
// iterations. Such a graph needs thousands of iterations of a few thousand edges each; as separate
// launches of the 2048-workgroup advance kernel each iteration would cost its launch and its chain of
// dependent loads, and a Bellman-Ford frontier re-relaxes every vertex about a hundred times on a
// weighted grid. Here an iteration costs a handful of dependent memory round trips, and SSSP runs
// near-far (Davidson et al., "Work-efficient parallel GPU methods for single-source shortest paths",
// IPDPS 2014): only vertices below a threshold T are expanded; the others wait in a far list until the
// near frontier is empty, then T grows by delta and the far list is split. One launch runs any number of
// independent queries, one per workgroup (the batched road-graph engine of the query server).
//
// The relaxations are the push engine's (SsspPush / BfsPush: 64-bit (dist, stamp) atomicMin, depth CAS),
// so results are bit-identical to every other engine's. What bounds an iteration is its chain of dependent
// steps, not its few hundred edges, so the chain is kept to two global round trips and one barrier:
//   1. a near entry carries its row's start and end (loaded by the relaxation that filed it, beside its
//      atomic), four lanes take it, one edge each, and the edge's target and weight and the source's
//      distance load together: no row-offset trip, no degree prefix, no search for an edge's source;
//   2. the atomics, with the targets' row offsets beside them.
// Three rotating counters leave one barrier per iteration. The query's state belongs to its workgroup, so
// its atomics have workgroup scope. Measured against reading the row offsets at the start of an iteration, a
// prefix sum over the chunk and a binary search per edge: grid 213 x 213 (distances in LDS, 550 iterations)
// 2.9 -> 1.5 us an iteration, 1.68 -> 0.83 ms a run; 48 queries on a 610 x 377 grid (distances in memory, 1390
// iterations) 5.8 -> 2.9 us, 8.0 -> 4.1 ms; one SSSP on 2048 x 2048 68 -> 53 ms, BFS 44 -> 34 ms.

#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "g1/device.hpp"
#include "g1/push.hpp"

namespace g1 {

constexpr int kRoadThreads = 1024;
constexpr uint32_t kRoadChunk = 4096;     // near entries kept in LDS, per frontier
constexpr uint32_t kRoadLanes = 4;        // lanes per near entry: most road and grid vertices have at most four edges
constexpr uint32_t kRoadGroups = kRoadThreads / kRoadLanes;

// Per-query device state. dstamp (SSSP) or depth (BFS) must be initialized by the caller (source set).
struct RoadQuery {
    uint32_t sssp;               // 1: SSSP (dstamp), 0: BFS (depth)
    unsigned long long* dstamp;  // SSSP: (dist << 32 | stamp), n words
    uint32_t* depth;             // BFS: n words; road_lds_kernel: the result of either kind
    uint32_t* q[2];              // near frontier buffers, q_cap (>= n) entries each
    uint32_t* far[2];            // far lists (SSSP), far_cap entries each
    uint32_t src;
    uint32_t status;             // out: 0 done, 2 far list overflow (run the query elsewhere)
    uint32_t iterations;         // out: expanded iterations
    uint32_t splits;             // out: far-list splits
    unsigned long long frontier_sum;  // out: vertices expanded
    unsigned long long edges_sum;     // out: relaxations
};

// A pointer read from a query record, as a pointer to global memory: through a generic one the compiler issues flat
// accesses, whose completion the LDS counter waits for as well, so that every LDS read after a store to a far list
// waited for that store.
template <typename T>
using road_global = __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ road_global<T> to_global(T* p) {
    return (road_global<T>)p;
}

// The start and end of v's row in one 8-byte load (any u32 alignment).
struct RoadRow {
    uint32_t beg, end;
};
__device__ __forceinline__ RoadRow road_row(const uint32_t* __restrict__ row_off, uint32_t v) {
    typedef uint32_t pair_t __attribute__((ext_vector_type(2), aligned(4)));
    const pair_t p = *reinterpret_cast<const pair_t*>(row_off + v);
    return RoadRow{p.x, p.y};
}

// The threads' sums of v folded over the workgroup (every thread calls it once, after a barrier).
__device__ __forceinline__ unsigned long long road_block_sum(unsigned long long v, unsigned long long* s) {
    v = wave_sum(v);
    if (lane_id() == 0) s[threadIdx.x / kWave] = v;
    __syncthreads();
    unsigned long long t = 0;
    for (int w = 0; w < kRoadThreads / kWave; ++w) t += s[w];
    return t;
}

static __global__ void __launch_bounds__(kRoadThreads)
road_query_kernel(const uint32_t* __restrict__ row_off, const uint32_t* __restrict__ col,
                  const uint32_t* __restrict__ wts, RoadQuery* queries, uint32_t delta, uint32_t far_cap,
                  uint32_t q_cap, uint32_t it_limit) {
    __shared__ uint32_t s_q[2][kRoadChunk];  // entries 0 .. kRoadChunk-1 of the two near frontiers:
    __shared__ uint32_t s_rb[2][kRoadChunk];  // vertex, row start, row end
    __shared__ uint32_t s_re[2][kRoadChunk];
    __shared__ unsigned long long s_sum[kRoadThreads / kWave];
    __shared__ uint32_t s_n[3];
    __shared__ uint32_t s_far[2];
    __shared__ uint32_t s_bad[3];  // raised beside the counter of the same index
    RoadQuery& Q = queries[blockIdx.x];
    const uint32_t tid = threadIdx.x;
    const uint32_t sub = tid % kRoadLanes, grp = tid / kRoadLanes;
    const bool kSssp = Q.sssp != 0;  // uniform per workgroup
    const uint32_t src = Q.src;
    const road_global<unsigned long long> ds = to_global(Q.dstamp);
    const road_global<uint32_t> depth = to_global(Q.depth);
    const road_global<uint32_t> gq[2] = {to_global(Q.q[0]), to_global(Q.q[1])};
    const road_global<uint32_t> far[2] = {to_global(Q.far[0]), to_global(Q.far[1])};
    // Appends v to near frontier b (counter c): LDS for the first kRoadChunk entries, the query's buffer
    // after them.
    auto push_near = [&](uint32_t b, uint32_t c, uint32_t v, RoadRow r) {
        const uint32_t pos = atomicAdd(&s_n[c], 1u);
        if (pos >= q_cap) {
            s_bad[c] = 1;
        } else if (pos < kRoadChunk) {
            s_q[b][pos] = v;
            s_rb[b][pos] = r.beg;
            s_re[b][pos] = r.end;
        } else {
            gq[b][pos] = v;
        }
    };
    auto push_far = [&](uint32_t f, uint32_t c, uint32_t v) {
        const uint32_t pos = atomicAdd(&s_far[f], 1u);
        if (pos < far_cap) far[f][pos] = v;
        else s_bad[c] = 1;
    };
    auto dist_of = [&](uint32_t v) -> uint32_t {
        return static_cast<uint32_t>(__hip_atomic_load(&ds[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >> 32);
    };
    // SSSP: a relaxation that wins (the vertex's first improvement of the iteration) files the vertex by
    // its new distance: near frontier (out) below T, far list above. A later improvement in the same
    // iteration does not win, except one that crosses T from above (the vertex was filed far, or not at
    // all, by a value >= T): it files the vertex near as well. A near entry is expanded with the distance it
    // has when its edges are loaded (an improvement in that iteration re-files it for the next). BFS:
    // plain alternating frontiers.
    if (tid == 0) {
        const RoadRow r = road_row(row_off, src);
        s_q[0][0] = src;
        s_rb[0][0] = r.beg;
        s_re[0][0] = r.end;
        s_n[0] = 1;
        s_n[1] = 0;
        s_n[2] = 0;
        s_far[0] = 0;
        s_far[1] = 0;
        s_bad[0] = s_bad[1] = s_bad[2] = 0;
    }
    __syncthreads();
    uint32_t cur = 0, cc = 0, fcur = 0, it = 0, splits = 0;  // near buffer, near counter, far list
    uint32_t T = delta;  // near-far threshold (SSSP)
    unsigned long long fsum = 0, esum = 0;  // esum: this thread's share
    for (;;) {
        const uint32_t n = s_n[cc];
        if (n == 0) {
            const uint32_t nfar = kSssp ? s_far[fcur] : 0u;
            if (nfar == 0) break;
            __syncthreads();  // every thread has read both counts
            // Split: raise T. A far entry whose distance is now in [T_old, T) becomes a candidate; one
            // below T_old was already expanded (every improvement made it a candidate, and a candidate
            // below the threshold of its time is expanded, while one above it was filed far again and
            // released by the split that passed it); the rest stay far. Copies of one vertex may be
            // expanded twice: that only repeats relaxations that cannot win.
            const uint32_t t_old = T;
            T = (T > 0xFFFFFFFFu - delta) ? 0xFFFFFFFFu : T + delta;
            for (uint32_t i = tid; i < nfar; i += kRoadThreads) {
                const uint32_t v = far[fcur][i];
                const uint32_t d = dist_of(v);
                const RoadRow r = road_row(row_off, v);
                if (d < t_old) continue;
                if (d < T) push_near(cur, cc, v, r);
                else push_far(fcur ^ 1, cc, v);
            }
            __syncthreads();
            if (tid == 0) {
                s_far[fcur] = 0;
                if (s_n[cc] > q_cap) s_n[cc] = q_cap;  // (flagged above; the run is abandoned)
            }
            fcur ^= 1;
            ++splits;
            __syncthreads();
            if (s_bad[cc]) break;
            continue;
        }
        if (it >= it_limit) {
            if (tid == 0) s_bad[cc] = 1;
            break;
        }
        const uint32_t out = cur ^ 1;
        const uint32_t oc = cc == 2 ? 0 : cc + 1;
        if (tid == 0) s_n[oc == 2 ? 0 : oc + 1] = 0;  // the last iteration's input counter: next iteration's output
        fsum += n;
        // R x kRoadGroups entries from entry base on, all of a thread's loads in flight together (an idle
        // lane reads the row of entry 0's vertex and uses nothing).
        auto expand = [&](auto rounds, uint32_t base) {
            constexpr uint32_t R = decltype(rounds)::value;
            uint32_t u[R], k[R], re[R];
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                const uint32_t i = base + r * kRoadGroups + grp;
                const bool have = i < n;
                const bool in_lds = !have || i < kRoadChunk;
                const uint32_t j = have && in_lds ? i : 0u;
                u[r] = s_q[cur][j];
                uint32_t rb = s_rb[cur][j];
                re[r] = s_re[cur][j];
                if (!in_lds) {
                    u[r] = gq[cur][i];
                    const RoadRow row = road_row(row_off, u[r]);
                    rb = row.beg;
                    re[r] = row.end;
                }
                if (!have) re[r] = rb;
                if (sub == 0) esum += re[r] - rb;
                k[r] = rb + sub;
            }
            for (;;) {  // one pass unless an entry has more than kRoadLanes edges
                uint32_t v[R], w[R];
                unsigned long long dw[R];
                bool on[R], any = false;
#pragma unroll
                for (uint32_t r = 0; r < R; ++r) {
                    on[r] = k[r] < re[r];
                    any |= on[r];
                }
                if (!any) break;
#pragma unroll
                for (uint32_t r = 0; r < R; ++r) {
                    const uint32_t e = on[r] ? k[r] : 0u;
                    v[r] = col[e];
                    if (kSssp) {
                        w[r] = wts[e];
                        dw[r] = __hip_atomic_load(&ds[u[r]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                }
                RoadRow row[R];
#pragma unroll
                for (uint32_t r = 0; r < R; ++r) row[r] = road_row(row_off, v[r]);
                if (kSssp) {
                    unsigned long long old[R];
                    uint32_t nd[R];
#pragma unroll
                    for (uint32_t r = 0; r < R; ++r) {
                        nd[r] = static_cast<uint32_t>(dw[r] >> 32) + w[r];
                        old[r] = 0ull;
                        if (on[r])
                            old[r] = __hip_atomic_fetch_min(
                                &ds[v[r]], (static_cast<unsigned long long>(nd[r]) << 32) | (it + 1), __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
#pragma unroll
                    for (uint32_t r = 0; r < R; ++r) {
                        const uint32_t od = static_cast<uint32_t>(old[r] >> 32);
                        if (!on[r] || nd[r] >= od) continue;
                        const bool first = static_cast<uint32_t>(old[r]) < it + 1;
                        if (nd[r] < T && (first || od >= T)) push_near(out, oc, v[r], row[r]);
                        else if (nd[r] >= T && first) push_far(fcur, oc, v[r]);
                    }
                } else {
                    uint32_t old[R];
#pragma unroll
                    for (uint32_t r = 0; r < R; ++r) {
                        old[r] = 0u;
                        uint32_t none = kInf;
                        if (on[r]) {
                            __hip_atomic_compare_exchange_strong(&depth[v[r]], &none, it + 1, __ATOMIC_RELAXED,
                                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                            old[r] = none;  // kInf where the exchange took place
                        }
                    }
#pragma unroll
                    for (uint32_t r = 0; r < R; ++r)
                        if (on[r] && old[r] == kInf) push_near(out, oc, v[r], row[r]);
                }
#pragma unroll
                for (uint32_t r = 0; r < R; ++r) k[r] += kRoadLanes;
            }
        };
        uint32_t base = 0;
        while (n - base > 2 * kRoadGroups) {
            expand(std::integral_constant<uint32_t, 4>{}, base);
            base += 4 * kRoadGroups;
            if (base >= n) break;
        }
        if (base < n) {
            if (n - base > kRoadGroups) expand(std::integral_constant<uint32_t, 2>{}, base);
            else expand(std::integral_constant<uint32_t, 1>{}, base);
        }
        cur = out;
        cc = oc;
        ++it;
        __syncthreads();
        if (s_bad[cc]) break;  // the next iteration raises another flag, so every thread sees the same here
    }
    __syncthreads();
    const bool bad = (s_bad[0] | s_bad[1] | s_bad[2]) != 0;
    const unsigned long long edges = road_block_sum(esum, s_sum);
    if (tid == 0) {
        Q.status = bad ? 2u : 0u;
        Q.iterations = it;
        Q.splits = splits;
        Q.frontier_sum = fsum;  // uniform: every thread saw the same n
        Q.edges_sum = edges;
    }
}

// BFS and SSSP queries on small road-like graphs (n <= kRoadLdsMaxN): the same near-far iteration with the
// distances kept in LDS as 16-bit values (vertex v in half v & 1 of word v >> 1, 0xFFFF = unreached), so a
// relaxation is an LDS compare-and-swap instead of an atomic on a distance word in memory and one global
// round trip is left: an edge's target and weight, with the target's row offsets beside the compare-and-swap.
// Two LDS bitmaps say which vertices wait in a near frontier and in the far list, so each list holds a vertex
// once: a relaxation files its target unless it already waits there, an entry leaves its bitmap before its
// distance is read (an improvement that comes later files it again). BFS is the same with unit weights and
// every distance near. Distances are exact while they stay below 0xFFFF; a relaxation that would reach it
// ends the query with status 2, as does a far-list overflow, leaving its result unwritten so the caller can
// run the query on road_query_kernel instead. On success the distances go to Q.depth. Same results, bit for
// bit, as every engine.
constexpr uint32_t kRoadLdsMaxN = 46080;  // 16-bit distances: 90 KB of LDS
constexpr uint32_t kRoadLdsChunk = 2048;

static __global__ void __launch_bounds__(kRoadThreads)
road_lds_kernel(uint32_t n, const uint32_t* __restrict__ row_off, const uint32_t* __restrict__ col,
                const uint32_t* __restrict__ wts, RoadQuery* queries, uint32_t delta, uint32_t far_cap,
                uint32_t q_cap, uint32_t it_limit) {
    __shared__ uint32_t s_d[kRoadLdsMaxN / 2];
    __shared__ uint32_t s_near[kRoadLdsMaxN / 32];
    __shared__ uint32_t s_wait[kRoadLdsMaxN / 32];
    __shared__ uint32_t s_q[2][kRoadLdsChunk];
    __shared__ uint32_t s_rb[2][kRoadLdsChunk];
    __shared__ uint32_t s_re[2][kRoadLdsChunk];
    __shared__ unsigned long long s_sum[kRoadThreads / kWave];
    __shared__ uint32_t s_n[3];
    __shared__ uint32_t s_far[2];
    __shared__ uint32_t s_bad[3];  // raised beside the counter of the same index
    RoadQuery& Q = queries[blockIdx.x];
    const uint32_t tid = threadIdx.x;
    const uint32_t sub = tid % kRoadLanes, grp = tid / kRoadLanes;
    const bool kSssp = Q.sssp != 0;  // uniform per workgroup
    const uint32_t src = Q.src;
    const road_global<uint32_t> gq[2] = {to_global(Q.q[0]), to_global(Q.q[1])};
    const road_global<uint32_t> far[2] = {to_global(Q.far[0]), to_global(Q.far[1])};
    // The second load of an edge: its weight, or (BFS) its target again. Without a branch between them the two are in
    // flight together (30 sources of a 150x200 grid 642 -> 629 us with the pointers above). road_query_kernel keeps its
    // branch: its second load comes with the distance, which a BFS has no use for (48 sources of a 610x377 grid: 4.07
    // against 4.19 ms).
    const uint32_t* const second = kSssp ? wts : col;
    const uint32_t words = (n + 1) / 2, fwords = (n + 31) / 32;
    for (uint32_t i = tid; i < words; i += kRoadThreads) s_d[i] = 0xFFFFFFFFu;
    for (uint32_t i = tid; i < fwords; i += kRoadThreads) {
        s_near[i] = 0u;
        s_wait[i] = 0u;
    }
    __syncthreads();
    if (tid == 0) {
        const RoadRow r = road_row(row_off, src);
        s_d[src >> 1] &= ~(0xFFFFu << (16u * (src & 1u)));  // distance 0
        s_q[0][0] = src;
        s_rb[0][0] = r.beg;
        s_re[0][0] = r.end;
        s_n[0] = 1;
        s_n[1] = 0;
        s_n[2] = 0;
        s_far[0] = 0;
        s_far[1] = 0;
        s_bad[0] = s_bad[1] = s_bad[2] = 0;
    }
    __syncthreads();
    auto dist = [&](uint32_t v) -> uint32_t { return (s_d[v >> 1] >> (16u * (v & 1u))) & 0xFFFFu; };
    auto push_near = [&](uint32_t b, uint32_t c, uint32_t v, RoadRow r) {
        const uint32_t pos = atomicAdd(&s_n[c], 1u);
        if (pos >= q_cap) {
            s_bad[c] = 1;
        } else if (pos < kRoadLdsChunk) {
            s_q[b][pos] = v;
            s_rb[b][pos] = r.beg;
            s_re[b][pos] = r.end;
        } else {
            gq[b][pos] = v;
        }
    };
    auto push_far = [&](uint32_t f, uint32_t c, uint32_t v) {
        const uint32_t pos = atomicAdd(&s_far[f], 1u);
        if (pos < far_cap) far[f][pos] = v;
        else s_bad[c] = 1;
    };
    uint32_t cur = 0, cc = 0, fcur = 0, it = 0, splits = 0;
    uint32_t T = kSssp ? delta : 0xFFFFFFFFu;
    unsigned long long fsum = 0, esum = 0;
    for (;;) {
        const uint32_t nn = s_n[cc];
        if (nn == 0) {
            const uint32_t nfar = s_far[fcur];
            if (nfar == 0) break;
            __syncthreads();  // every thread has read both counts
            const uint32_t t_old = T;
            T = (T > 0xFFFFFFFFu - delta) ? 0xFFFFFFFFu : T + delta;
            for (uint32_t i = tid; i < nfar; i += kRoadThreads) {
                const uint32_t v = far[fcur][i];
                const uint32_t bit = 1u << (v & 31u);
                const uint32_t d = dist(v);
                const RoadRow r = road_row(row_off, v);
                if (d >= T) {
                    push_far(fcur ^ 1, cc, v);  // still waits
                    continue;
                }
                atomicAnd(&s_wait[v >> 5], ~bit);
                if (d < t_old) continue;  // was expanded
                atomicOr(&s_near[v >> 5], bit);
                push_near(cur, cc, v, r);
            }
            __syncthreads();
            if (tid == 0) {
                s_far[fcur] = 0;
                if (s_n[cc] > q_cap) s_n[cc] = q_cap;
            }
            fcur ^= 1;
            ++splits;
            __syncthreads();
            if (s_bad[cc]) break;
            continue;
        }
        if (it >= it_limit) {
            if (tid == 0) s_bad[cc] = 1;
            break;
        }
        const uint32_t out = cur ^ 1;
        const uint32_t oc = cc == 2 ? 0 : cc + 1;
        if (tid == 0) s_n[oc == 2 ? 0 : oc + 1] = 0;
        fsum += nn;
        auto expand = [&](auto rounds, uint32_t base) {
            constexpr uint32_t R = decltype(rounds)::value;
            uint32_t u[R], k[R], re[R], du[R];
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                const uint32_t i = base + r * kRoadGroups + grp;
                const bool have = i < nn;
                const bool in_lds = !have || i < kRoadLdsChunk;
                const uint32_t j = have && in_lds ? i : 0u;
                u[r] = s_q[cur][j];
                uint32_t rb = s_rb[cur][j];
                re[r] = s_re[cur][j];
                if (!in_lds) {
                    u[r] = gq[cur][i];
                    const RoadRow row = road_row(row_off, u[r]);
                    rb = row.beg;
                    re[r] = row.end;
                }
                if (!have) re[r] = rb;
                if (have && sub == 0) {
                    atomicAnd(&s_near[u[r] >> 5], ~(1u << (u[r] & 31u)));  // before the distance is read
                    esum += re[r] - rb;
                }
                k[r] = rb + sub;
            }
            // The bits before the distances: a wave's LDS operations run in its program order, which the
            // compiler must keep too.
            asm volatile("" ::: "memory");
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) du[r] = dist(u[r]);
            for (;;) {
                uint32_t v[R], w[R];
                bool on[R], any = false;
#pragma unroll
                for (uint32_t r = 0; r < R; ++r) {
                    on[r] = k[r] < re[r];
                    any |= on[r];
                }
                if (!any) break;
#pragma unroll
                for (uint32_t r = 0; r < R; ++r) {
                    const uint32_t e = on[r] ? k[r] : 0u;
                    v[r] = col[e];
                    w[r] = second[e];
                }
                RoadRow row[R];
#pragma unroll
                for (uint32_t r = 0; r < R; ++r) {
                    row[r] = road_row(row_off, v[r]);
                    if (!kSssp) w[r] = 1u;
                }
#pragma unroll
                for (uint32_t r = 0; r < R; ++r) {
                    if (!on[r]) continue;
                    if (w[r] >= 0xFFFFu - du[r]) {  // du + w would reach 0xFFFF: not representable here
                        s_bad[oc] = 1;
                        continue;
                    }
                    const uint32_t nd = du[r] + w[r];
                    uint32_t* word = &s_d[v[r] >> 1];
                    const uint32_t sh = 16u * (v[r] & 1u);
                    uint32_t old = *word;
                    bool improved = false;
                    while (nd < ((old >> sh) & 0xFFFFu)) {
                        const uint32_t prev = atomicCAS(word, old, (old & ~(0xFFFFu << sh)) | (nd << sh));
                        if (prev == old) {
                            improved = true;
                            break;
                        }
                        old = prev;
                    }
                    if (!improved) continue;
                    const uint32_t bit = 1u << (v[r] & 31u);
                    if (nd < T) {
                        if ((atomicOr(&s_near[v[r] >> 5], bit) & bit) == 0u) push_near(out, oc, v[r], row[r]);
                    } else if ((atomicOr(&s_wait[v[r] >> 5], bit) & bit) == 0u) {
                        push_far(fcur, oc, v[r]);
                    }
                }
#pragma unroll
                for (uint32_t r = 0; r < R; ++r) k[r] += kRoadLanes;
            }
        };
        uint32_t base = 0;
        while (nn - base > 2 * kRoadGroups) {
            expand(std::integral_constant<uint32_t, 4>{}, base);
            base += 4 * kRoadGroups;
            if (base >= nn) break;
        }
        if (base < nn) {
            if (nn - base > kRoadGroups) expand(std::integral_constant<uint32_t, 2>{}, base);
            else expand(std::integral_constant<uint32_t, 1>{}, base);
        }
        cur = out;
        cc = oc;
        ++it;
        __syncthreads();
        if (s_bad[cc]) break;  // the next iteration raises another flag, so every thread sees the same here
    }
    __syncthreads();
    const bool bad = (s_bad[0] | s_bad[1] | s_bad[2]) != 0;
    if (!bad) {
        for (uint32_t v = tid; v < n; v += kRoadThreads) {
            const uint32_t d = dist(v);
            to_global(Q.depth)[v] = d == 0xFFFFu ? kInf : d;
        }
    }
    const unsigned long long edges = road_block_sum(esum, s_sum);
    if (tid == 0) {
        Q.status = bad ? 2u : 0u;
        Q.iterations = it;
        Q.splits = splits;
        Q.frontier_sum = fsum;
        Q.edges_sum = edges;
    }
}

}  // namespace g1
