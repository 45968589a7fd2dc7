// egs_bins.h -- dense rounds of large games in two streaming kernels: every edge's candidate
// value from LDS-resident slices of the values, then every vertex's fold in LDS.
//
// A dense round gathers the value of every edge's successor.  Gathered from memory, each is an
// L2 request and a cache line through a compute unit's L1: 33.5M of them took 200 us on the
// 2^22-vertex game, 8M of them 73 us on a 10^6-vertex one, three to six times what the bytes
// take.  Here no gather leaves a compute unit:
//   * the edges are cut into chunks and the successors into slices of at most kBinSlice; the
//     layout (k_bin_build) groups a chunk's edges by slice into runs, as 32-bit words
//     (w << 15) | place in slice, with each edge's vertex in the chunk as 16 bits beside it.
//     Runs are padded to 16 edges, a cache sector, since neighbouring runs are written from
//     different compute units; padding belongs to a vertex past the chunk's last;
//   * k_bin_gather: a workgroup loads a slice of the values into LDS and walks its runs in
//     all chunks (of its part), storing a - w for every edge at the edge's own place;
//   * k_bin_reduce: a workgroup per chunk streams its candidates and vertex numbers, folds
//     them into LDS words and applies the lifts.
// Both stream: 4 + 4 bytes an edge read and written, then 4 + 2 read.  OMINUS(a, w) is a
// monotone clamp of a - w, so the folds run over the raw differences (saturated; a TOP value
// stays past MG since mg + 2 wmax < 2^31 - 1) and the clamp is applied once per vertex.
//
// Chunks cut a line on which a vertex takes kBinHead places and then one per edge, at even
// distances, through vertices too: at most the first and the last vertex of a chunk have edges
// in others.  Each chunk folds its part of such a vertex into the vertex's word in memory and
// counts itself; the last one applies the lift.  So hubs need no kernels of their own here.
// Rounds are synchronous.
#pragma once

#include <climits>

#include "egs_device.h"
#include "egs_internal.h"

namespace egs {

// Workgroup i of a gather: its slice and its part of the chunks.  Workgroups of one XCD (i mod
// 8) take neighbouring slices, whose runs in a chunk share cache lines.
__device__ __forceinline__ void bin_place(const DevGame &g, int i, int &slice, int &part) {
    const int per = g.bins >> 3;                 // bins is a multiple of 8
    const int x = i & 7, k = i >> 3;
    slice = x * per + k % per;
    part = k / per;
}

// Every run of a slice in the chunks of a part: run(put) calls put(edge index, two words) for
// each pair of edges, the workgroup's waves on separate chunks.  A wave has eight runs in
// flight, a lane two edges of each (runs are about 100 edges: bin_share), and the next eight
// loading while these are used: with four runs and no loads ahead the gather of the
// 2^22-vertex game took 100 us.
struct BinWalk {
    static constexpr int kRuns = 8;
    int w_lo, w_hi;                              // the wave's chunks
    const int *beg, *end;
    const uint32_t *edges;
    int b, e, c0;                                // 64 runs' ends, from chunk c0 on
    unsigned long long x[kRuns];                 // the next eight runs' words

    bool once;                                   // the edges outgrow the memory-side cache

    __device__ __forceinline__ unsigned long long load(int k) const {
        const unsigned long long *p = (const unsigned long long *)(edges + k);
        return once ? __builtin_nontemporal_load(p) : *p;
    }
    __device__ __forceinline__ void ends() {
        const int lane = threadIdx.x & 63;
        b = e = 0;
        if (c0 + lane < w_hi) {
            b = beg[c0 + lane];
            e = end[c0 + lane];
        }
    }
    __device__ __forceinline__ void fetch(int i, int count) {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int q = 0; q < kRuns; q++) {
            x[q] = 0;
            if (i + q < count) {
                const int k = __builtin_amdgcn_readlane(b, i + q) + 2 * lane;
                if (k < __builtin_amdgcn_readlane(e, i + q))
                    x[q] = load(k);
            }
        }
    }
    // The first loads, issued before the slice is in LDS.
    __device__ __forceinline__ void start(const DevGame &g, int slice, int part, int parts) {
        const int waves = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int nc = g.nchunks;
        const int c_lo = (int)((int64_t)nc * part / parts), c_hi = (int)((int64_t)nc * (part + 1) / parts);
        const int span = c_hi - c_lo;
        w_lo = c_lo + (int)((int64_t)span * wave / waves);
        w_hi = c_lo + (int)((int64_t)span * (wave + 1) / waves);
        beg = g.boff + (size_t)slice * nc;
        end = beg + nc;
        edges = g.bedges;
        once = g.bin_once;
        c0 = w_lo;
        ends();
        fetch(0, min(64, w_hi - c0));
    }
    template <class F>
    __device__ __forceinline__ void run(F put) {
        const int lane = threadIdx.x & 63;
        while (c0 < w_hi) {
            const int count = min(64, w_hi - c0);
            for (int i = 0; i < count; i += kRuns) {
                unsigned long long y[kRuns];
#pragma unroll
                for (int q = 0; q < kRuns; q++) y[q] = x[q];
                if (i + kRuns < count) fetch(i + kRuns, count);
#pragma unroll
                for (int q = 0; q < kRuns; q++) {
                    if (i + q >= count) break;
                    const int rb = __builtin_amdgcn_readlane(b, i + q), re = __builtin_amdgcn_readlane(e, i + q);
                    const int k = rb + 2 * lane;
                    if (k < re) put(k, (uint32_t)y[q], (uint32_t)(y[q] >> 32));
                    for (int k0 = rb + 128; k0 < re; k0 += 256) {      // a longer run's rest
                        unsigned long long z[2];
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const int kk = k0 + 128 * h + 2 * lane;
                            z[h] = kk < re ? load(kk) : 0;
                        }
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const int kk = k0 + 128 * h + 2 * lane;
                            if (kk < re) put(kk, (uint32_t)z[h], (uint32_t)(z[h] >> 32));
                        }
                    }
                }
            }
            c0 += 64;
            if (c0 < w_hi) {
                ends();
                fetch(0, min(64, w_hi - c0));
            }
        }
    }
};

// A slice of n-long `src` into LDS through f(value, index), 1,024 threads.
template <class T, class S, class F>
__device__ __forceinline__ void bin_load(const DevGame &g, int slice, const S *src, T *lds, F f) {
    const int first = slice * g.bin_w, count = max(0, min(g.bin_w, g.n - first));
    for (int i = threadIdx.x; i < count; i += 4 * blockDim.x) {
        S x[4];
#pragma unroll
        for (int k = 0; k < 4; k++) x[k] = i + k * (int)blockDim.x < count ? src[first + i + k * (int)blockDim.x] : S(0);
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (i + k * (int)blockDim.x < count) lds[i + k * (int)blockDim.x] = f(x[k], first + i + k * (int)blockDim.x);
    }
}

// A chunk: its edges [e0, e1), its vertices from v0 on, and which of them have edges elsewhere.
struct BinChunk {
    int v0, nv, e0, e1;
    bool split_first, split_last;
};
__device__ __forceinline__ BinChunk bin_chunk(const DevGame &g, int c) {
    BinChunk k{};
    k.e0 = g.bchunk[2 * c];
    k.v0 = g.bchunk[2 * c + 1];
    k.e1 = g.bchunk[2 * c + 2];
    if (k.e1 <= k.e0) return k;
    const int vn = g.bchunk[2 * c + 3];                      // vertex of edge e1 (n past the last)
    const bool into = g.ptr[vn] < k.e1;                      // its first edges are in this chunk
    k.nv = vn - k.v0 + (into ? 1 : 0);
    k.split_first = g.ptr[k.v0] < k.e0 || (k.nv == 1 && into);
    k.split_last = into;
    return k;
}
// Chunks that hold edges of vertex v.
__device__ __forceinline__ int bin_holders(const DevGame &g, int v) {
    const int64_t at = (int64_t)kBinHead * (v + 1);
    return (int)((at + g.ptr[v + 1] - 1) / g.bin_share - (at + g.ptr[v]) / g.bin_share) + 1;
}

// The fold of a chunk's candidates [b, e) into LDS words: key[vertex] = min of candidate ^ mask, the
// mask complementing the owner's whose fold is a maximum (owner 1 in the rounds, MAX1, owner 0
// in the longest-path passes).  key starts at the largest T.
// Neighbours in a run are often of one vertex (all of them in a hub's chunks): a thread folds
// equal neighbours before its LDS atomics, and a chunk of one vertex is folded in registers.
template <class T, class V4, bool MAX1 = true>
__device__ __forceinline__ void bin_fold(const DevGame &g, const T *cand, int b, int e, int n0l, int nv, T *key) {
    const bool mixed = n0l > 0 && n0l < nv;
    const T mask0 = MAX1 ? T(0) : T(-1), mask1 = MAX1 ? T(-1) : T(0), mask = n0l <= 0 ? mask1 : mask0;
    constexpr int U = sizeof(T) == 4 ? 4 : 2;
    constexpr int N = sizeof(V4) / sizeof(T);    // candidates per load
    T lone = key[nv];                            // the neutral value
    for (int k0 = b + 4 * (int)threadIdx.x; k0 < e; k0 += 4 * U * (int)blockDim.x) {
        V4 c[U][4 / N];
        ushort4 v[U];
#pragma unroll
        for (int q = 0; q < U; q++) {
            const int k = k0 + 4 * q * (int)blockDim.x;
            if (k < e) {
#pragma unroll
                for (int h = 0; h < 4 / N; h++) c[q][h] = *(const V4 *)(cand + k + N * h);
                v[q] = *(const ushort4 *)(g.bids + k);
            }
        }
#pragma unroll
        for (int q = 0; q < U; q++) {
            if (k0 + 4 * q * (int)blockDim.x >= e) break;
            const int vs[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
            T cs[4];
#pragma unroll
            for (int h = 0; h < 4; h++)
                cs[h] = ((const T *)&c[q][h / N])[h % N] ^ (mixed ? (vs[h] >= n0l ? mask1 : mask0) : mask);
            if (nv == 1) {
#pragma unroll
                for (int h = 0; h < 4; h++)
                    if (vs[h] == 0) lone = cs[h] < lone ? cs[h] : lone;
                continue;
            }
#pragma unroll
            for (int h = 0; h < 4; h++) {
                if (h < 3 && vs[h] == vs[h + 1]) cs[h + 1] = cs[h] < cs[h + 1] ? cs[h] : cs[h + 1];
                else atomicMin(&key[vs[h]], cs[h]);
            }
        }
    }
    if (nv == 1) {
        for (int d = 32; d >= 1; d >>= 1) {
            const T o = __shfl_xor(lone, d, 64);
            lone = o < lone ? o : lone;
        }
        if ((threadIdx.x & 63) == 0) atomicMin(&key[0], lone);
    }
}

// This chunk's fold of vertex v, shared with other chunks, into hacc[v]: true for the chunk
// that completes it, which gets the whole fold and leaves the words neutral again.  Only
// atomics touch the words, and each is complete (its result used) before the next.
__device__ __forceinline__ bool bin_share_fold(const DevGame &g, int v, int &fold) {
    egs_complete(atomicMin(&g.hacc[v], fold));
    if (atomicAdd(&g.hcnt[v], 1) != bin_holders(g, v) - 1) return false;
    fold = atomicExch(&g.hacc[v], INT_MAX);
    g.hcnt[v] = 0;
    return true;
}

// The same for a longest-path candidate in hbest[v], kept as the workgroup-per-vertex passes
// keep it (owner 0 a maximum, owner 1 a minimum).
__device__ __forceinline__ bool bin_share_best(const DevGame &g, int v, bool owner1, long long &best) {
    egs_complete(owner1 ? atomicMin(&g.hbest[v], best) : atomicMax(&g.hbest[v], best));
    if (atomicAdd(&g.hcnt[v], 1) != bin_holders(g, v) - 1) return false;
    best = (long long)atomicExch((unsigned long long *)&g.hbest[v],
                                 (unsigned long long)(owner1 ? LLONG_MAX : LLONG_MIN));
    g.hcnt[v] = 0;
    return true;
}

}  // namespace egs
