// egs_games.h -- the many-games kernel shared by the batched solver (egs_batch.hip) and
// the serving loop (egs_serve.hip).
//
// A launch runs over a list of game descriptors.  A persistent workgroup claims one whole
// game at a time from a device counter and runs in-place (Gauss-Seidel) sweeps over its
// vertices until a complete sweep changes nothing (a block-wide vote), the launch's sweep
// cap for that game is reached, or the workgroup's edge budget for the launch is spent.
// A sweep may stop part-way at a chunk boundary: the game's GameState keeps the vertex
// cursor and whether the sweep has changed anything so far, so a later launch resumes it.
// A sweep that changed nothing proves the fixpoint even when it spanned launches: no value
// moved while it ran, so every vertex was checked against the final values.
// A game's values sit in the workgroup's LDS, 32 or 16 bits each; of a game past that the
// first ones do and the rest are in global memory (game_layout).
// Every `every` sweeps (doubling while proofs fail) the workgroup tries the certified TOP
// proof of egs_accel.hip on its game.
#pragma once

#include <climits>

#include "egs_device.h"

namespace egs {

struct GameState {
    int64_t sweeps;        // sweeps done so far
    int64_t edges;         // edges relaxed so far
    int64_t lifted;
    int64_t cert_passes;
    int64_t next_cert;     // sweep count of the next proof attempt
    int32_t gap;           // current attempt spacing
    int32_t converged;     // 1 once a sweep changed nothing
    int32_t certificates;
    int32_t started;       // values initialised
    int32_t bf_cap;        // longest-path passes per candidate threshold (doubles while attempts run out)
    int32_t cursor;        // first vertex of the current sweep not yet visited
    int32_t dirty;         // the current sweep has changed a value
    int32_t reserved;
};

struct GameDesc {
    const int *ptr;        // n+1 local CSR offsets
    const void *edges;     // m edges: uint32 (w << shift) | succ, or int2 {succ, w} when shift == 0
    int *values;           // n
    int *rise;             // n: number of the sweep in which each vertex last rose (proof candidates)
    int *h;                // n scratch (proofs: potentials above the warm start)
    GameState *state;
    int64_t m;
    int n, n0, mg, wmax;
    int shift, group;
};

constexpr int kGameFirstCap = 32;      // longest-path passes per candidate at a game's first attempt
constexpr int kGameCandidates = 8;     // gap thresholds tried per attempt (plus the last-rise set)
constexpr int kGameCertifyEvery = 4;   // default sweeps before the first proof attempt

struct CertArgs {
    int every;             // sweeps between proof attempts; <= 0 = no proofs
    int max_passes;        // ceiling of the longest-path passes per candidate threshold
    int first_cap;         // passes per candidate at a game's first attempt
    int candidates;        // thresholds tried per attempt
};

// Pointers read from a descriptor are generic to the compiler, whose flat loads go through
// both memory paths and wait for both: a sweep of the batch of 1,024 games took 444 us with
// them.  They are cast to the global address space where they are used, and LDS is named
// directly.
template <class T>
using InGlobal = __attribute__((address_space(1))) T;
template <class T>
__device__ __forceinline__ InGlobal<T> *in_global(T *p) { return (InGlobal<T> *)p; }
extern __shared__ __align__(16) int game_lds[];

// A game's values in the workgroup's LDS.  WHOLE and SPLIT: the first `split` values as they
// are, the rest (none when WHOLE) in the game's global array hi.  SHORT: 16 bits a value, with
// kShortTop for TOP and kShortFar for a value past them, which hi holds.
enum : int { GAME_WHOLE = 0, GAME_SHORT = 1, GAME_SPLIT = 2 };
constexpr int kShortTop = 0xfffe, kShortFar = 0xffff;
struct GameVals {
    int *hi;
    int split;
    int lay;
    int d_at;              // where potentials of their own lie in LDS, or 0: in the game's global array
    __device__ __forceinline__ static int low16(int v) { return ((const uint16_t *)game_lds)[v]; }
    __device__ __forceinline__ int far(int c, int v) const {
        return c < kShortTop ? c : c == kShortTop ? EGS_TOP : in_global(hi)[v];
    }
    __device__ __forceinline__ int get(int v) const {
        if (lay == GAME_SHORT) return far(low16(v), v);
        return v < split ? game_lds[v] : in_global(hi)[v];
    }
    __device__ __forceinline__ void set_short(int v, int x) const {
        const int c = x == EGS_TOP ? kShortTop : min(x, kShortFar);
        if (x >= kShortTop && x != EGS_TOP) {
            in_global(hi)[v] = x;
            __threadfence_block();               // there before anyone is sent to it
        }
        ((uint16_t *)game_lds)[v] = (uint16_t)(x >= kShortTop && x != EGS_TOP ? kShortFar : c);
    }
    __device__ __forceinline__ void set(int v, int x) const {
        if (lay == GAME_SHORT) set_short(v, x);
        else if (v < split) game_lds[v] = x;
        else in_global(hi)[v] = x;
    }
};

template <int LAY>
__device__ __forceinline__ int gv(const GameVals &V, int v) {
    if (LAY == GAME_WHOLE) return game_lds[v];
    if (LAY == GAME_SHORT) return V.far(V.low16(v), v);
    return v < V.split ? game_lds[v] : in_global(V.hi)[v];
}
template <int LAY>
__device__ __forceinline__ void gv_set(const GameVals &V, int v, int x) {
    if (LAY == GAME_WHOLE) game_lds[v] = x;
    else if (LAY == GAME_SHORT) V.set_short(v, x);
    else V.set(v, x);
}
// The values of N vertices, all loads in flight together.
template <int LAY, int N>
__device__ __forceinline__ void gv_gather(const GameVals &V, const int (&v)[N], int (&x)[N]) {
    if (LAY == GAME_WHOLE) {
#pragma unroll
        for (int j = 0; j < N; j++) x[j] = game_lds[v[j]];
    } else if (LAY == GAME_SHORT) {
        bool away = false;
#pragma unroll
        for (int j = 0; j < N; j++) x[j] = V.low16(v[j]);
#pragma unroll
        for (int j = 0; j < N; j++) {
            away |= x[j] == kShortFar;
            x[j] = x[j] == kShortTop ? EGS_TOP : x[j];
        }
        if (away) {
#pragma unroll
            for (int j = 0; j < N; j++)
                if (x[j] == kShortFar) x[j] = in_global(V.hi)[v[j]];
        }
    } else {
        int c[N];
#pragma unroll
        for (int j = 0; j < N; j++) {            // split < n: no branch on where a value lies
            x[j] = game_lds[min(v[j], V.split - 1)];
            c[j] = in_global(V.hi)[max(v[j], V.split)];
        }
#pragma unroll
        for (int j = 0; j < N; j++) x[j] = v[j] < V.split ? x[j] : c[j];
    }
}

__device__ __forceinline__ void game_edge(const GameDesc &b, int64_t k, int &succ, int &w) {
    if (b.shift) {
        const uint32_t e = in_global((const uint32_t *)b.edges)[k];
        succ = (int)(e & ((1u << b.shift) - 1u));
        w = ((int)e) >> b.shift;
    } else {
        const InGlobal<const int> *e = in_global((const int *)b.edges) + 2 * k;
        succ = e[0];
        w = e[1];
    }
}

// Edge loads in flight per lane: a lane's edges are read one after another from global
// memory, and one load at a time leaves the loops latency-bound.  Slots past a vertex's
// last edge read vertex 0 and are not used.
constexpr int kGameU = 4;

// Part of a sweep by groups of G lanes, from vertex `cursor`, chunk by chunk (a chunk is
// one vertex per group) while `spent` < `budget`; returns the next cursor.  `spent` adds
// the chunk's edge count, read from the offsets by every lane, so it stays block-uniform
// and the loop keeps waves whole for the DPP reductions.
template <int G, int LAY>
__device__ __forceinline__ int game_sweep_part(const GameDesc &b, const GameVals &V, int cursor, int64_t budget, int sweep_no,
                                               int64_t &spent, int64_t &edges_done, int &lifted, bool &changed) {
    const int gl = threadIdx.x % G;
    const int gid = threadIdx.x / G;
    const int ngroups = blockDim.x / G;
    int base = cursor;
    // the next chunk's offsets load while this chunk runs (they never change)
    int s_n = 0, e_n = 0, c0_n = 0, c1_n = 0;
    auto fetch = [&](int at) {
        const int u = at + gid;
        if (u < b.n) {
            s_n = in_global(b.ptr)[u];
            e_n = in_global(b.ptr)[u + 1];
        }
        c0_n = in_global(b.ptr)[at];
        c1_n = in_global(b.ptr)[min(at + ngroups, b.n)];
    };
    if (base < b.n) fetch(base);
    while (base < b.n && spent < budget) {
        spent += c1_n - c0_n;
        const int v = base + gid;
        const bool valid = v < b.n;
        int s = 0, e = 0, old = 0;
        if (valid) {
            s = s_n;
            e = e_n;
        }
        if (base + ngroups < b.n) fetch(base + ngroups);
        if (valid) {
            old = gv<LAY>(V, v);
            if (old == EGS_TOP) e = s;          // TOP is final: nothing to gather
        }
        const bool owner1 = v >= b.n0;
        int key = EGS_TOP;
        for (int k0 = s + gl; k0 < e; k0 += G * kGameU) {
            int su[kGameU], wv[kGameU], a[kGameU];
#pragma unroll
            for (int j = 0; j < kGameU; j++) {
                su[j] = 0;
                wv[j] = 0;
                if (k0 + j * G < e) game_edge(b, k0 + j * G, su[j], wv[j]);
            }
#pragma unroll
            for (int j = 0; j < kGameU; j++) a[j] = gv<LAY>(V, su[j]);
#pragma unroll
            for (int j = 0; j < kGameU; j++)
                if (k0 + j * G < e) key = min(key, egs_key(egs_ominus(a[j], wv[j], b.mg), owner1));
        }
        key = egs_group_min<G>(key);
        const int t = egs_unkey(key, owner1);
        if (valid && gl == 0) {
            edges_done += e - s;
            if (old < t) {
                gv_set<LAY>(V, v, t);
                in_global(b.rise)[v] = sweep_no;
                changed = true;
                lifted++;
            }
        }
        base += ngroups;
    }
    return min(base, b.n);
}

constexpr int kGameDOut = -1;          // potential of a vertex outside a proof's candidate

// ---- packed edges: eight slots a lane, one chunk ahead -----------------------------------
//
// Latency bounds the loops above: a chunk's edges are loaded, four words a lane, once its
// offsets are there, and a compute unit's 16 waves (one workgroup takes all of its LDS) cover
// little of that.  Games with 32-bit edges whose values and weights leave room in 31 bits
// (game_wide) take these instead: a lane holds eight edge words of its vertex, two 16-byte
// loads, and loads the next chunk's while it folds this one's; the folds run over the raw
// differences a - w (saturated; OMINUS is a monotone clamp of them, applied once a vertex).
// Bound now by VALU issue (some 200 operations a wave and chunk) beside random LDS reads.  A
// sweep of 256 games of 19,000 vertices and degree 2-16, one to a compute unit: 458 edges/ns
// before, 969 now; of 2,000 vertices: 487 and 710; of complete games of 400: 506 and 1,268.
constexpr int kWideSlots = 8;
typedef uint32_t GameWords __attribute__((ext_vector_type(4), aligned(4)));

// mg + 2 wmax < TOP: a TOP value less a weight stays past every member's difference.
__device__ __forceinline__ bool game_wide(const GameDesc &b) {
    return b.shift > 0 && (int64_t)b.mg + 2 * (int64_t)b.wmax < EGS_TOP;
}

// A lane's words of the first G * kWideSlots edges of a row [s, e): the quads gl and gl + G.
// Quads past the row read the game's first, so no load passes the game's edges by more than
// three words (values or stamps follow them).  own: what the fetch read of the vertex.
struct GameRow {
    int s, e, own;
    GameWords x[2];
};
template <int G>
__device__ __forceinline__ void game_row_load(const InGlobal<const uint32_t> *edges, GameRow &r, int at) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int k = at + 4 * (int)(threadIdx.x % G + G * i);
        r.x[i] = *(const InGlobal<const GameWords> *)(edges + (k < r.e ? k : 0));
    }
}
// The lane's slots of the words at `at`: f(words, which are there); the others are word 0.
template <int G, class F>
__device__ __forceinline__ void game_row_slots(const GameRow &r, int at, F f) {
    uint32_t word[kWideSlots];
    bool there[kWideSlots];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int left = r.e - at - 4 * (int)(threadIdx.x % G + G * i);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            there[4 * i + j] = j < left;
            word[4 * i + j] = j < left ? r.x[i][j] : 0u;
        }
    }
    f(word, there);
}

// Rows of the vertices from `cursor` on, a chunk of one vertex per group at a time while a
// chunk begins below `end`: want(v, own) reads the vertex and tells whether its edges are
// needed (if not the row is empty), visit(v, row, slots) folds it, slots(f) giving the lane's
// slots.  Every lane of a vertex's group calls.  Returns the next cursor.
template <int G, class W, class V>
__device__ __forceinline__ int game_rows(const GameDesc &b, int cursor, int end, W want, V visit) {
    const int gid = threadIdx.x / G, ng = blockDim.x / G;
    const InGlobal<const uint32_t> *edges = in_global((const uint32_t *)b.edges);
    int s_n, e_n;
    auto offsets = [&](int base) {
        s_n = e_n = 0;
        if (base < end && base + gid < b.n) {
            s_n = in_global(b.ptr)[base + gid];
            e_n = in_global(b.ptr)[base + gid + 1];
        }
    };
    auto fetch = [&](int base, GameRow &r) {
        r.s = s_n;
        r.own = 0;
        r.e = e_n > s_n && want(base + gid, r.own) ? e_n : s_n;
        game_row_load<G>(edges, r, r.s);
    };
    GameRow now, next;
    int base = cursor;
    offsets(base);
    fetch(base, now);
    offsets(base + ng);
    for (; base < end; base += ng) {
        fetch(base + ng, next);
        offsets(base + 2 * ng);
        visit(base + gid, now, [&](auto f) {
            game_row_slots<G>(now, now.s, f);
            for (int at = now.s + G * kWideSlots; at < now.e; at += G * kWideSlots) {   // a longer row's rest
                game_row_load<G>(edges, now, at);
                game_row_slots<G>(now, at, f);
            }
        });
        now = next;
    }
    return min(base, b.n);
}

// game_sweep_part for such games.
template <int G, int LAY>
__device__ __forceinline__ int game_sweep_wide(const GameDesc &b, const GameVals &V, int cursor, int64_t budget, int sweep_no,
                                               int64_t &spent, int64_t &edges_done, int &lifted, bool &changed) {
    const int p0 = in_global(b.ptr)[cursor], shift = b.shift;
    const uint32_t smask = (1u << shift) - 1u;
    int end = b.n;                               // chunks begin while the budget is not spent
    if (b.m - p0 >= budget - spent) {
        int lo = cursor;                         // the first vertex at or past the budget's end
        while (lo < end) {
            const int mid = lo + (end - lo) / 2;
            if (b.ptr[mid] - p0 >= budget - spent) end = mid;
            else lo = mid + 1;
        }
    }
    const int next = game_rows<G>(
        b, cursor, end,
        [&](int v, int &own) {
            own = gv<LAY>(V, v);
            return own != EGS_TOP;               // TOP is final: nothing to gather
        },
        [&](int v, const GameRow &r, auto slots) {
            const int m = v >= b.n0 ? -1 : 0;
            int key = EGS_TOP;
            slots([&](const uint32_t (&word)[kWideSlots], const bool (&there)[kWideSlots]) {
                int u[kWideSlots], a[kWideSlots];
#pragma unroll
                for (int j = 0; j < kWideSlots; j++) u[j] = (int)(word[j] & smask);
                gv_gather<LAY>(V, u, a);
#pragma unroll
                for (int j = 0; j < kWideSlots; j++) {
                    const int d = __builtin_elementwise_sub_sat(a[j], (int)word[j] >> shift) ^ m;
                    key = there[j] ? min(key, d) : key;
                }
            });
            key = egs_group_min<G>(key);
            const int d = key ^ m, t = d > b.mg ? EGS_TOP : max(d, 0);
            if (threadIdx.x % G == 0 && r.e > r.s) {
                edges_done += r.e - r.s;
                if (r.own < t) {
                    gv_set<LAY>(V, v, t);
                    in_global(b.rise)[v] = sweep_no;
                    changed = true;
                    lifted++;
                }
            }
        });
    spent += in_global(b.ptr)[next] - p0;
    return next;
}

// A proof's potentials in the place of the values (game_certify): H(v) = S (F - f(v)) + 1 + d(v)
// on the candidate, F the largest value, kPotTop at TOP and kPotOut elsewhere.  One number a
// vertex holds both what an edge's candidate S w + 1 + H(u) takes, so a pass gathers once an
// edge, as a sweep does, and needs no more LDS.  (Value and potential apart are two gathers, and
// past 20,000 vertices the potentials of 32 bits were gathered from L2: an attempt took 2.0 ms on
// games of 39,000 vertices, degree 2-16, one to a compute unit, and takes 0.64.)
// Any S >= 1 is sound: a cycle of S W + L <= 0 has W < 0.  A smaller S than n + 1 only proves
// fewer cycles, those of average -1 / S or below.  S (F + wmax) stays within a quarter of the
// range, 2^28 or (16 bits) 32,000; a potential past kPotMax ends the passes.  What a smaller
// scale does not settle (past the range, or out of passes) is tried again with n + 1 and
// potentials of their own in 64 bits, so that every proof of theirs is found in the same attempt
// (a ring of 300 vertices that loses one unit a turn under values of 5 10^6 was never proved
// without; 1,024 games of the batched family need the second try too rarely to show: 4.00 ms
// with it, 4.03 without).
constexpr int kPotOut = 0x60000000, kPotTop = -kPotOut, kPotGone = 0x48000000;
constexpr int kPotRange = 1 << 28, kPotMax = 0x30000000, kShortRange = 32000, kShortMax = 65000;
template <bool SHORT>
__device__ __forceinline__ int pot_get(int v) {
    if (!SHORT) return game_lds[v];
    const int c = ((const uint16_t *)game_lds)[v];
    return c == 0 ? kPotTop : c == kShortFar ? kPotOut : c;
}
template <bool SHORT>
__device__ __forceinline__ void pot_set(int v, int h) {
    if (SHORT) ((uint16_t *)game_lds)[v] = (uint16_t)(h == kPotTop ? 0 : h == kPotOut ? kShortFar : h);
    else game_lds[v] = h;
}
__device__ __forceinline__ bool pot_member(int h) { return (unsigned)h < (unsigned)kPotOut; }

template <int G, bool SHORT>
__device__ __forceinline__ void game_pass(const GameDesc &b, int scale, bool &ch, bool &over) {
    const int shift = b.shift;
    const uint32_t smask = (1u << shift) - 1u;
    constexpr int most = SHORT ? kShortMax : kPotMax;
    game_rows<G>(
        b, 0, b.n,
        [&](int v, int &own) {
            own = pot_get<SHORT>(v);
            return pot_member(own);
        },
        [&](int v, const GameRow &r, auto slots) {
            const int m = v >= b.n0 ? 0 : -1;    // owner 0's maximum as a minimum of complements
            int key = INT_MAX;
            slots([&](const uint32_t (&word)[kWideSlots], const bool (&there)[kWideSlots]) {
                int h[kWideSlots];
#pragma unroll
                for (int j = 0; j < kWideSlots; j++) h[j] = pot_get<SHORT>((int)(word[j] & smask));
#pragma unroll
                for (int j = 0; j < kWideSlots; j++) {
                    const int c = (__mul24(scale, (int)word[j] >> shift) + 1 + h[j]) ^ m;
                    key = there[j] ? min(key, c) : key;
                }
            });
            const int best = egs_group_min<G>(key) ^ m;
            if (threadIdx.x % G == 0 && r.e > r.s) {
                // owner 1 breaks closure when no edge stays in D or reaches TOP, owner 0 when any leaves
                if (best >= kPotGone) {
                    pot_set<SHORT>(v, kPotOut);
                    ch = true;
                } else if (best > r.own) {
                    pot_set<SHORT>(v, min(best, most));
                    ch = true;
                    over |= best > most;
                }
            }
        });
}

// The certified TOP proof inside the workgroup (the steps of egs_accel.hip).  Candidate
// sets D, tried in turn until one yields a non-empty proven set:
//   * every admissible gap threshold B, smallest first: D = {v : B < f(v) < TOP};
//   * the vertices that rose in the last sweep (`last`): D = {v : rise(v) == last, f(v) < TOP}.
// When no window is empty, the smallest threshold whose window holds only a few values
// takes the place of the gap thresholds.
// Check 1 (closure): an owner-0 vertex of D has every successor in D or TOP, an owner-1
// vertex at least one; vertices that break it are removed until it holds (the greatest
// closed subset), during the passes of check 2: the longest-path game on D with w' = (n+1) w + 1,
//   h(v) <- max(h(v), max_{u in D} w'(v,u) + h(u))           (owner 0)
//   h(v) <- max(h(v), min_{u in D or TOP} w'(v,u) + h(u))    (owner 1; a TOP successor ends the path)
// reaches a fixpoint within `cap` passes.  At a fixpoint the minimising successors form a
// strategy sigma of player 1 under which every cycle inside D has weight <= -1, which is
// the proof; any fixpoint will do, so the iteration starts from h = (n+1) (MG - f): the
// lifting keeps f(u) - f(v) >= w(v,u) along such edges, so this start is already close.
// Returns the vertices set to TOP; `cap_hit` tells whether some candidate ran out of passes.
// Potentials are kept as d(v) = h(v) - (n+1) (MG - f(v)) >= 0, 4 bytes next to the values;
// kGameDOut marks a vertex outside D (TOP is read off the value).  A d past INT_MAX ends the
// attempt as if it diverged: it only gives up a proof.
__device__ __forceinline__ bool game_in_d_x(const GameDesc &b, int x, int v, int B, int last) {
    return x != EGS_TOP && (B >= 0 ? x > B : in_global(b.rise)[v] == last);
}

// One candidate on potentials in the values' place, the values read from the game's global
// array: 1 after a fixpoint (members: what is left of it), 0 when out of passes, kPotNone
// without members, kPotPast when a potential left the range.
constexpr int kPotNone = -1, kPotPast = -2;
template <bool SHORT>
__device__ __forceinline__ int game_pot_proof(const GameDesc &b, int scale, int top, int B, int last, int cap,
                                              int64_t &passes_done) {
    int members = 0;
    for (int v = threadIdx.x; v < b.n; v += blockDim.x) {
        const int x = in_global(b.values)[v];
        const bool in = game_in_d_x(b, x, v, B, last);
        pot_set<SHORT>(v, x == EGS_TOP ? kPotTop : in ? scale * (top - x) + 1 : kPotOut);
        members += in;
    }
    if (__syncthreads_count(members > 0) == 0) return kPotNone;
    for (int p = 0; p < cap; p++) {
        bool ch = false, over = false;
        if (b.group > 8) game_pass<64, SHORT>(b, scale, ch, over);
        else game_pass<2, SHORT>(b, scale, ch, over);
        passes_done++;
        if (__syncthreads_or(over)) return kPotPast;
        if (!__syncthreads_or(ch)) return 1;
    }
    return 0;
}

__device__ __forceinline__ int game_certify(const GameDesc &b, const GameVals &V, int last, int cap, int max_cands,
                            int64_t &passes_done,
                            bool &cap_hit) {
    auto d_get = [&](int v) { return V.d_at ? game_lds[V.d_at + v] : in_global(b.h)[v]; };
    auto d_set = [&](int v, int d) {
        if (V.d_at) game_lds[V.d_at + v] = d;
        else in_global(b.h)[v] = d;
    };
    __shared__ int win[64], flo[64];
    __shared__ unsigned long long s_cand;
    __shared__ int s_marked, s_top;
    const int wmax = b.wmax;
    if (wmax <= 0) return 0;
    const long long scale = (long long)b.n + 1;
    // divergence bound: at a fixpoint h <= max start + (n - 1) max w'; 2x headroom in int64
    const double bound_d = (double)scale * b.mg + (double)b.n * ((double)scale * wmax + 1);
    if (bound_d > 4.0e18) return 0;
    const long long bound = (long long)scale * b.mg + (long long)b.n * (scale * wmax + 1);
    for (int i = threadIdx.x; i < 64; i += blockDim.x) { win[i] = 0; flo[i] = 0; }
    if (threadIdx.x == 0) s_top = 0;
    int most = 0;                             // the largest value below TOP
    __syncthreads();
    for (int v = threadIdx.x; v < b.n; v += blockDim.x) {
        const int x = V.get(v);
        if (x == EGS_TOP || x <= 0) continue;
        most = max(most, x);
        const unsigned below = ((unsigned)x - 1u) / (unsigned)wmax, q = below + 1u;      // q = ceil(x / W)
        if ((q & (q - 1u)) == 0) atomicAdd(&win[31 - __clz(q)], 1);
        if (below > 0) atomicAdd(&flo[31 - __clz(below)], 1);
    }
    most = -egs_group_min<64>(-most);
    if ((threadIdx.x & 63) == 0) atomicMax(&s_top, most);
    __syncthreads();
    if (threadIdx.x == 0) {
        // bit j set: B_j = W * 2^j has an empty window, non-TOP values above it, B_j <= MG - W
        unsigned long long mask = 0, near = 0;
        int64_t above = 0;                    // #{non-TOP values > W * 2^j} while j descends
        for (int k = 63; k >= 40; k--) above += flo[k];
        for (int j = 39; j >= 1; j--) {
            above += flo[j];
            if (((int64_t)wmax << j) > (int64_t)b.mg - wmax || above == 0) continue;
            if (win[j] == 0) mask |= 1ull << j;
            else if (win[j] <= max((int64_t)64, above / 256)) near = 1ull << j;   // ends as the smallest
        }
        // no empty window: the smallest threshold whose window holds a few stragglers (the
        // members whose edges reach them are pruned)
        if (mask == 0) mask = near;
        unsigned long long keep = 0;          // the lowest max_cands thresholds
        for (int k = 0; k < max_cands && mask; k++) {
            keep |= mask & (~mask + 1);
            mask &= mask - 1;
        }
        s_cand = keep | 1ull;                 // bit 0: the vertices that rose in the last sweep
        s_marked = 0;
    }
    __syncthreads();
    unsigned long long cand = s_cand;
    // potentials in the values' place where the values are whole or 16 bits: the values go to
    // the game's global array, which every candidate's membership is read from
    const int range = V.lay == GAME_SHORT ? kShortRange : kPotRange;
    const int pot = game_wide(b) && V.lay != GAME_SPLIT && wmax < 1 << 23
                        ? (int)min((long long)range / (s_top + (long long)wmax), scale) : 0;
    auto restore = [&]() {
        __syncthreads();
        for (int v = threadIdx.x; v < b.n; v += blockDim.x) V.set(v, in_global(b.values)[v]);
        __syncthreads();
    };
    if (pot > 0) {
        for (int v = threadIdx.x; v < b.n; v += blockDim.x) in_global(b.values)[v] = V.get(v);
        __syncthreads();
    }
    int B = -1;
    while (cand) {
        // gap thresholds first, smallest first; the last-rise set after them
        const bool recent = (cand & ~1ull) == 0;
        if (recent) {
            B = -1;
            cand = 0;
        } else {
            const int j = __ffsll(cand & ~1ull) - 1;
            cand &= ~(1ull << j);
            B = (int)((int64_t)wmax << j);
        }
        if (pot > 0) {
            const int got = V.lay == GAME_SHORT ? game_pot_proof<true>(b, pot, s_top, B, last, cap, passes_done)
                                                : game_pot_proof<false>(b, pot, s_top, B, last, cap, passes_done);
            if (got > 0) {
                int mine = 0;
                for (int v = threadIdx.x; v < b.n; v += blockDim.x)
                    if (pot_member(V.lay == GAME_SHORT ? pot_get<true>(v) : pot_get<false>(v))) {
                        in_global(b.values)[v] = EGS_TOP;
                        mine++;
                    }
                if (mine) atomicAdd(&s_marked, mine);
                __syncthreads();
                if (s_marked > 0) break;
                __syncthreads();              // pruning emptied the candidate: try the next
            }
            // the same candidate with n + 1 after a potential past the range, and where a
            // smaller scale ran out of passes: n + 1 may need fewer
            if (got == 0 && pot == scale) cap_hit = true;
            if (got != kPotPast && (got != 0 || pot == scale)) continue;
            restore();
        }
        // pass 0: membership, closure and the first longest-path step, from the values alone
        // (the warm start of a successor is (n+1) (MG - f)).  A member that breaks closure
        // leaves D (h = kGameHOut); later passes check it again against the removals, so the
        // passes compute the greatest closed subset of the candidate along with h.
        bool ch = false, over = false;
        int members = 0;
        for (int v = threadIdx.x; v < b.n; v += blockDim.x) {
            const int x = V.get(v);
            if (!game_in_d_x(b, x, v, B, last)) { d_set(v, kGameDOut); continue; }
            members++;
            const long long h0 = scale * ((long long)b.mg - x);
            const bool owner1 = v >= b.n0;
            long long best = owner1 ? LLONG_MAX : LLONG_MIN;
            bool any = false, all = true;
            const int s = in_global(b.ptr)[v], e = in_global(b.ptr)[v + 1];
            for (int k0 = s; k0 < e; k0 += kGameU) {
                int uu[kGameU], ww[kGameU], xu[kGameU];
#pragma unroll
                for (int j = 0; j < kGameU; j++) {
                    uu[j] = 0;
                    ww[j] = 0;
                    if (k0 + j < e) game_edge(b, k0 + j, uu[j], ww[j]);
                }
#pragma unroll
                for (int j = 0; j < kGameU; j++) xu[j] = V.get(uu[j]);
#pragma unroll
                for (int j = 0; j < kGameU; j++) {
                    if (k0 + j >= e) break;
                    if (xu[j] == EGS_TOP) {
                        any = true;
                        if (owner1) best = LLONG_MIN;
                    } else if (game_in_d_x(b, xu[j], uu[j], B, last)) {
                        any = true;
                        const long long c = scale * ww[j] + 1 + scale * ((long long)b.mg - xu[j]);
                        best = owner1 ? min(best, c) : max(best, c);
                    } else {
                        all = false;
                    }
                }
            }
            if (owner1 ? !any : !all) {
                d_set(v, kGameDOut);
                ch = true;
            } else if (best > h0) {
                d_set(v, (int)min(best - h0, (long long)INT_MAX));
                ch = true;
                over |= best > bound || best - h0 >= INT_MAX;
            } else {
                d_set(v, 0);
            }
        }
        if (__syncthreads_count(members > 0) == 0) continue;
        passes_done++;
        bool converged = __syncthreads_count(ch) == 0, diverged = __syncthreads_or(over) != 0;
        for (int p = 1; p < cap && !converged && !diverged; p++) {
            ch = false;
            over = false;
            for (int v = threadIdx.x; v < b.n; v += blockDim.x) {
                const int dv = d_get(v);
                if (dv < 0) continue;
                const long long h0 = scale * ((long long)b.mg - V.get(v));
                const long long hv = h0 + dv;
                const bool owner1 = v >= b.n0;
                long long best = owner1 ? LLONG_MAX : LLONG_MIN;
                bool out = false;
                const int s = in_global(b.ptr)[v], e = in_global(b.ptr)[v + 1];
                for (int k0 = s; k0 < e; k0 += kGameU) {
                    int uu[kGameU], ww[kGameU], xu[kGameU], du[kGameU];
#pragma unroll
                    for (int j = 0; j < kGameU; j++) {
                        uu[j] = 0;
                        ww[j] = 0;
                        if (k0 + j < e) game_edge(b, k0 + j, uu[j], ww[j]);
                    }
#pragma unroll
                    for (int j = 0; j < kGameU; j++) {
                        xu[j] = V.get(uu[j]);
                        du[j] = d_get(uu[j]);
                    }
#pragma unroll
                    for (int j = 0; j < kGameU; j++) {
                        if (k0 + j >= e) break;
                        if (xu[j] == EGS_TOP) {       // ends the path: -infinity for the game
                            if (owner1) best = LLONG_MIN;
                            continue;
                        }
                        if (du[j] < 0) { out = true; continue; }
                        const long long c = scale * ww[j] + 1 + scale * ((long long)b.mg - xu[j]) + du[j];
                        best = owner1 ? min(best, c) : max(best, c);
                    }
                }
                // owner 1 breaks closure when no edge reaches D or TOP, owner 0 when any leaves
                if (owner1 ? best == LLONG_MAX : out) {
                    d_set(v, kGameDOut);
                    ch = true;
                } else if (best > hv) {
                    d_set(v, (int)min(best - h0, (long long)INT_MAX));
                    ch = true;
                    over |= best > bound || best - h0 >= INT_MAX;
                }
            }
            passes_done++;
            converged = __syncthreads_count(ch) == 0;
            diverged = __syncthreads_or(over) != 0;
        }
        if (diverged || !converged) {
            if (!diverged) cap_hit = true;
            continue;
        }
        int mine = 0;
        for (int v = threadIdx.x; v < b.n; v += blockDim.x)
            if (d_get(v) >= 0) { V.set(v, EGS_TOP); mine++; }
        if (mine) atomicAdd(&s_marked, mine);
        __syncthreads();
        if (s_marked > 0) return s_marked;
        __syncthreads();                      // pruning emptied the candidate: try the next
    }
    if (pot > 0) restore();
    return s_marked;
}

// Advance one game until its fixpoint, a due proof attempt, `max_sweeps` more complete
// sweeps, or `budget` edges (checked per chunk).  `sst` is the workgroup's shared copy of
// the game's state; the proof itself runs in game_prove, outside the lane-width variants,
// so the kernel carries one copy of it.  Adds the edges charged to the budget to `spent`
// and the complete sweeps to `sweeps` (both block-uniform); returns whether it stopped
// because a proof attempt is due.
template <int G>
__device__ __forceinline__ bool game_run(const GameDesc &b, const GameVals &V, GameState &sst, int64_t budget, int64_t max_sweeps,
                         const CertArgs &ca, int64_t &spent, int64_t &sweeps) {
    // the fields the loop changes, as scalars (a whole-struct copy ends up in scratch)
    int cursor = sst.cursor;
    bool converged = sst.converged != 0, dirty = sst.dirty != 0;
    const int64_t sweeps0 = sst.sweeps, next_cert = sst.next_cert;
    const bool wide = game_wide(b);
    __syncthreads();
    int64_t edges_done = 0, used = 0, done = 0;
    int lifted = 0;
    bool proof_due = false;
    while (!converged && used < budget && done < max_sweeps) {
        bool ch = false;
        const int no = (int)(sweeps0 + done + 1);
#define EGS_SWEEP(F, LAY) cursor = F<G, LAY>(b, V, cursor, budget, no, used, edges_done, lifted, ch)
        if (wide && V.lay == GAME_WHOLE) EGS_SWEEP(game_sweep_wide, GAME_WHOLE);
        else if (wide && V.lay == GAME_SHORT) EGS_SWEEP(game_sweep_wide, GAME_SHORT);
        else if (wide) EGS_SWEEP(game_sweep_wide, GAME_SPLIT);
        else if (V.lay == GAME_WHOLE) EGS_SWEEP(game_sweep_part, GAME_WHOLE);
        else EGS_SWEEP(game_sweep_part, GAME_SPLIT);
#undef EGS_SWEEP
        dirty = __syncthreads_or(ch || dirty) != 0;
        if (cursor < b.n) break;                    // budget spent part-way through the sweep
        done++;
        cursor = 0;
        if (!dirty) {
            converged = true;
            break;
        }
        dirty = false;
        if (ca.every > 0 && sweeps0 + done >= next_cert) {
            proof_due = true;
            break;
        }
    }
    spent += used;
    sweeps += done;
    __shared__ unsigned long long red[2];
    if (threadIdx.x == 0) { red[0] = 0; red[1] = 0; }
    __syncthreads();
    if (edges_done) atomicAdd(&red[0], (unsigned long long)edges_done);
    if (lifted) atomicAdd(&red[1], (unsigned long long)lifted);
    __syncthreads();
    if (threadIdx.x == 0) {
        sst.edges += (int64_t)red[0];
        sst.lifted += (int64_t)red[1];
        sst.sweeps = sweeps0 + done;
        sst.cursor = cursor;
        sst.converged = converged ? 1 : 0;
        sst.dirty = dirty ? 1 : 0;
    }
    __syncthreads();
    return proof_due;
}

// One proof attempt at a sweep boundary; schedules the next one (spacing back to `every`
// after a proof, doubled after a failure, pass cap doubled when a candidate ran out).
__device__ __forceinline__ void game_prove(const GameDesc &b, const GameVals &V, GameState &sst, const CertArgs &ca) {
    const int cap = sst.bf_cap;
    __syncthreads();
    int64_t passes = 0;
    bool cap_hit = false;
    const int marked = game_certify(b, V, (int)sst.sweeps, cap, ca.candidates, passes, cap_hit);
    const bool hit = __syncthreads_or(cap_hit) != 0;
    if (threadIdx.x == 0) {
        sst.cert_passes += passes;
        if (marked > 0) {
            sst.certificates++;
            sst.gap = ca.every;
        } else {
            sst.gap = min(sst.gap * 2, 1 << 16);
            if (hit) sst.bf_cap = min(sst.bf_cap * 2, ca.max_passes);
        }
        sst.next_cert = sst.sweeps + sst.gap;
    }
    __syncthreads();
}

// Where a game's values and proof potentials go in lds_cap ints of LDS: whole while they fit,
// 16 bits each up to twice that, else split.  256 games of 49,900 vertices and degree 2-16, one
// to a compute unit: 8.1 ms split, 2.3 with 16 bits.
__device__ __forceinline__ GameVals game_layout(const GameDesc &b, int lds_cap) {
    const int64_t n = b.n, behind = (n + 3) & ~3ll;
    GameVals V{b.values, b.n, GAME_WHOLE, behind + n <= lds_cap ? (int)behind : 0};
    if (n <= lds_cap) return V;
    if (game_wide(b) && n <= 2 * (int64_t)lds_cap) {
        V.lay = GAME_SHORT;
        return V;
    }
    V.lay = GAME_SPLIT;
    V.split = lds_cap;
    return V;
}

// The persistent many-games kernel (internal linkage: each including unit keeps a copy).
// Each workgroup claims games in `order` until they run out or its `wg_budget` edges for
// this launch are spent; a game gets at most `max_sweeps` complete sweeps per launch.
static __global__ __launch_bounds__(1024) void k_games(const GameDesc *__restrict__ games, const int *__restrict__ order,
                                                int ngames, int *counter, int lds_cap, int64_t wg_budget,
                                                int64_t max_sweeps, CertArgs ca) {
    __shared__ int s_idx;
    __shared__ GameState s_st;
    int64_t left = wg_budget;
    while (left > 0) {
        if (threadIdx.x == 0) s_idx = atomicAdd(counter, 1);
        __syncthreads();
        const int idx = s_idx;
        __syncthreads();
        if (idx >= ngames) break;          // every workgroup leaves once the games run out
        const GameDesc b = games[order[idx]];
        const GameVals V = game_layout(b, lds_cap);
        if (threadIdx.x == 0) {
            s_st = *b.state;
            if (!s_st.started) {
                s_st.started = 1;
                s_st.gap = ca.every;
                s_st.next_cert = ca.every > 0 ? ca.every : INT64_MAX;
                s_st.bf_cap = min(ca.first_cap, ca.max_passes);
                s_st.cursor = 0;
                s_st.dirty = 0;
                s_idx = -1;                // marks a fresh game for the value set-up below
            }
        }
        __syncthreads();
        const bool fresh = s_idx < 0;
        if (fresh) {
            for (int v = threadIdx.x; v < b.n; v += blockDim.x) {
                V.set(v, 0);
                in_global(b.rise)[v] = 0;
            }
        } else {
            for (int v = threadIdx.x; v < V.split; v += blockDim.x) V.set(v, in_global(b.values)[v]);
        }
        __syncthreads();
        int64_t sweeps_left = max_sweeps;
        for (;;) {
            int64_t spent = 0, sweeps = 0;
            bool due;
            switch (b.group) {
            case 1: due = game_run<1>(b, V, s_st, left, sweeps_left, ca, spent, sweeps); break;
            case 2: due = game_run<2>(b, V, s_st, left, sweeps_left, ca, spent, sweeps); break;
            case 4: due = game_run<4>(b, V, s_st, left, sweeps_left, ca, spent, sweeps); break;
            case 8: due = game_run<8>(b, V, s_st, left, sweeps_left, ca, spent, sweeps); break;
            case 16: due = game_run<16>(b, V, s_st, left, sweeps_left, ca, spent, sweeps); break;
            case 32: due = game_run<32>(b, V, s_st, left, sweeps_left, ca, spent, sweeps); break;
            default: due = game_run<64>(b, V, s_st, left, sweeps_left, ca, spent, sweeps); break;
            }
            left -= spent;
            sweeps_left -= sweeps;
            if (!due) break;
            game_prove(b, V, s_st, ca);
            if (left <= 0 || sweeps_left <= 0) break;
        }
        for (int v = threadIdx.x; v < V.split; v += blockDim.x) in_global(b.values)[v] = V.get(v);
        if (threadIdx.x == 0) *b.state = s_st;
        __syncthreads();
    }
}

}  // namespace egs
