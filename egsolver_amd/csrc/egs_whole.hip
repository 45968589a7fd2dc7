// egs_whole.hip -- a whole solve in one launch, for games whose rounds are shorter than the
// launches and read-backs between them.
//
// Replaces, for such games, the reference's host-driven round loop (src/dev_EG_alg.cu:307-381).
// The round kernels (egs_rounds.hip) cost a launch and a fixed chain of loads per round and
// the proof schedule (egs_accel.hip) several host round trips per attempt: a 2,000-vertex
// game spent 420-480 us on 2 us of memory traffic.  Here the workgroups of one launch keep
// their share of the game on chip for the whole solve and meet at a barrier in memory:
//   * workgroup b owns consecutive vertices, cut so that vertices plus edges are even
//     (k_whole_prep); their values, partial keys and proof potentials live in LDS;
//   * a thread owns up to R consecutive edges, in registers (with R = 16, 70 to 111 of them
//     spill to scratch), whatever the degrees: it folds them into its vertices' LDS keys with
//     one LDS atomic per vertex it touches;
//   * a round gathers the successors' values (LDS in the one-workgroup form, else global
//     memory), folds, applies the lifts of its own vertices and votes on the risers.
// Rounds are synchronous; values only rise and never pass the least fixpoint, and a round that
// began with every value visible and in which nothing rose ends the run at lift(val) == val.
// The TOP proofs are those of egs_accel.hip (same candidates, same passes, evaluated on every
// member).
//
// Bound: the barrier (1.9 us for the arrivals and their answer, and an agent release and
// acquire per workgroup, 0.7 us in all with 64 workgroups and 3.4 us with 256) and one
// gather latency per round.  Whole solves with one proof, device time, against the round
// kernels: n = 9,973, degree 2..16: 74 us (244); n = 30,011: 96 us (275); n = 87,148:
// 161 us (346); n = 140,000: 219 us (394).
//
// The barrier needs every workgroup resident.  A workgroup that waits past its limit raises
// the abort flag and leaves; the others see the flag in their own waits and leave too, and
// the host goes on with the round kernels from the values reached (any prefix of the rounds
// is a valid start of theirs, and so is a partly marked proven set; only a run with a round cap
// begins again, since the rounds of a launch that gave up are not counted).
#include <climits>

#include "egs_device.h"
#include "egs_internal.h"

namespace egs {

// Potentials: a successor outside D (and not at TOP) counts as +inf, one at TOP as -inf.  They
// are finite and far past every potential, so that an edge's candidate w' + h needs no test:
// a fold above kWInf / 2 has met +inf, one below -kWInf / 2 only -inf.
constexpr long long kWInf = 1ll << 62;
__device__ __forceinline__ bool w_member(long long h) { return h >= 0 && h < kWInf / 2; }

// A vote's 64-bit word: sum of per-thread counts, waves that changed something, waves past
// the divergence bound, arrivals.  A wave field has room for every wave of the largest launch:
// with one bit less, a pass in which all 4,096 waves changed something read as one past the
// bound, and a game whose vertices all climb (312,926 of degree 2) was never proved.
constexpr int kVoteChanged = 22, kVoteOver = 35, kVoteArrive = 48, kVoteWaves = (1 << 13) - 1;
static_assert(kWholeMaxNb * (int64_t)kWholeShareMax < 1 << kVoteChanged && kWholeMaxNb * 16 <= kVoteWaves &&
              kVoteChanged + 13 == kVoteOver && kVoteOver + 13 == kVoteArrive, "the fields of a vote hold their sums");

__device__ __forceinline__ unsigned long long ctl_load(const unsigned long long *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void ctl_store(unsigned long long *p, unsigned long long x) {
    __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long ctl_add(unsigned long long *p, unsigned long long x) {
    return __hip_atomic_fetch_add(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Zero the control block and (fresh) the values, and cut the vertices into nb workgroup
// shares: bound[b] is the first v with ptr[v] + v >= b * share.
__global__ __launch_bounds__(256) void k_whole_prep(const int *__restrict__ ptr, int n, int nb, int64_t share, int fresh,
                                                    int *__restrict__ val, WholeCtl *__restrict__ ctl) {
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < (int)(offsetof(WholeCtl, bound) / 4); i += blockDim.x) ((int *)ctl)[i] = 0;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v <= n; v += (int64_t)gridDim.x * blockDim.x) {
        if (fresh && v < n) val[v] = 0;
        if (nb > 1) {
            const int64_t lo = v > 0 ? (ptr[v - 1] + v - 1) / share + 1 : 0;
            const int64_t hi = v < n ? (ptr[v] + v) / share : nb;    // the shares past the last vertex are empty
            for (int64_t b = lo; b <= hi && b <= nb; b++) ctl->bound[b] = (int)v;
        }
    }
}

// The candidates of gap_candidates (egs_accel.hip) from the histograms in LDS (64 windows, 64
// floors), then -1, the last round's risers.  Returns how many.
__device__ int whole_candidates(const int *bins, int wmax, int mg, int max_cands, long long *out) {
    int c = 0, near_j = 0;
    int64_t above = 0;
    unsigned long long mask = 0;
    for (int j = 31; j >= 1; j--) {                 // values have 31 bits
        above += bins[64 + j];
        if (((int64_t)wmax << j) > (int64_t)mg - wmax || above == 0) continue;
        if (bins[j] == 0) mask |= 1ull << j;
        else if (bins[j] <= max((int64_t)64, above / 256)) near_j = j;   // ends as the smallest
    }
    for (; mask && c < max_cands; mask &= mask - 1) out[c++] = (int64_t)wmax << (__ffsll(mask) - 1);
    if (near_j && c < max_cands) out[c++] = (int64_t)wmax << near_j;
    out[c++] = -1;
    return c;
}

template <int R, bool ONE>
__global__ __launch_bounds__(1024) void k_whole(WholeArgs a) {
    extern __shared__ __align__(16) long long dyn[];
    __shared__ unsigned long long s_acc[2], s_total;
    __shared__ int s_ok, s_ncand;
    __shared__ int s_bins[128];
    __shared__ long long s_cand[16];
    __shared__ unsigned long long s_sum[2];
    const int tid = threadIdx.x, T = blockDim.x, lane = tid & 63;
    const bool lead = ONE || blockIdx.x == 0;
    const long long tick0 = wall_clock64();
    int v0 = 0, nb = a.n;
    if (!ONE) {
        v0 = a.ctl->bound[blockIdx.x];
        nb = a.ctl->bound[blockIdx.x + 1] - v0;
    }
    long long *hown = dyn, *hk = dyn + a.nbmax;     // own potentials, partial candidates
    int *own = (int *)(hk + a.nbmax), *key = own + a.nbmax;
    int *row = (int *)hk;                           // set-up only: own row offsets
    const int n0l = a.n0 - v0;                      // own vertices from n0l on belong to owner 1
    const bool fresh = a.round0 == 0;
    for (int i = tid; i <= nb; i += T) row[i] = a.ptr[v0 + i];
    for (int i = tid; i < nb; i += T) {
        own[i] = fresh ? 0 : a.val[v0 + i];
        key[i] = INT_MAX;
        if (fresh && a.rise) a.rise[v0 + i] = 0;
    }
    if (tid == 0) { s_acc[0] = 0; s_acc[1] = 0; s_sum[0] = 0; s_sum[1] = 0; s_ncand = 0; }
    __syncthreads();
    // this thread's edges [elo, elo + cnt), the local vertex of the first one, and the slots
    // after which its fold goes to the vertex's key (a row's last edge, the thread's last)
    const int e0 = row[0], mb = row[nb] - e0, per = (mb + T - 1) / T;
    const int elo = e0 + tid * per, cnt = max(0, min(per, e0 + mb - elo));
    int vl0 = 0;
    if (cnt > 0) {
        int lo = 0, hi = nb;                        // largest i with row[i] <= elo
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (row[mid] <= elo) lo = mid; else hi = mid;
        }
        vl0 = lo;
    }
    unsigned su[R];                                 // byte offset of the successor's value
    int w[R];
    unsigned flush = 0;
    int vl1 = vl0;                                  // the thread's last vertex
    {
        int vl = vl0;
#pragma unroll
        for (int j = 0; j < R; j++) {
            su[j] = 0;
            w[j] = 0;
            if (j < cnt) {
                const int2 e = a.edges[elo + j];
                su[j] = 4u * (unsigned)e.x;
                w[j] = e.y;
                vl1 = vl;
                if (elo + j + 1 == row[vl + 1]) {
                    flush |= 1u << j;
                    vl++;
                }
            }
        }
        if (cnt > 0) flush |= 1u << (cnt - 1);
    }
    __syncthreads();                                // row's space becomes hk
    // A wave whose vertices all belong to one owner folds with that owner's mask in a scalar
    // register.  OMINUS(a, w) = clamp(a - w) for a monotone clamp (> mg: TOP, < 0: 0), so the
    // folds run over a - w, saturated (a TOP value stays past mg: mg + wmax < TOP), and the
    // clamp is applied once per vertex; owner 1's maximum is a minimum of complements.
    const bool any0 = __any(cnt > 0 && vl0 < n0l), any1 = __any(cnt > 0 && vl1 >= n0l);
    const bool mixed = any0 && any1;
    unsigned live = (1u << cnt) - 1u;               // edges of vertices not yet seen at TOP
    // edges of vertices at TOP need no gather: they are pointed at the first value
    auto drop_top = [&]() {
        int vl = vl0;
#pragma unroll
        for (int j = 0; j < R; j++) {
            if (j < cnt && own[vl] == EGS_TOP) {
                live &= ~(1u << j);
                su[j] = 0;
            }
            if ((flush >> j) & 1u) vl++;
        }
    };
    if (!fresh) drop_top();

    // ---- the vote: a sum over all workgroups and, past it, their stores visible ------------
    unsigned gen = 0;
    int par = 0;
    auto vote = [&](int count, bool changed, bool over, unsigned long long &total) -> bool {
        const int sum = egs_wave_sum(count);
        const unsigned long long mine = (unsigned long long)(unsigned)sum |
                                        ((unsigned long long)(__any(changed) ? 1 : 0) << kVoteChanged) |
                                        ((unsigned long long)(__any(over) ? 1 : 0) << kVoteOver);
        if (lane == 0 && mine) atomicAdd(&s_acc[par], mine);
        if (!ONE) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's stores have left the CU
        __syncthreads();
        if (ONE) {
            total = s_acc[par];
            if (tid == 0) s_acc[par ^ 1] = 0;
            par ^= 1;
            __syncthreads();
            return true;
        }
        if (tid == 0) {
            // arrivals by group of workgroups, the last of a group adds the group's sum to the
            // root, the last there hands the total to every group's release word: one counter
            // for all costs 15 ns a workgroup (3.8 us at 256; this way 1.9 us at any number)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            const unsigned q = gen & 3, nx = (gen + 2) & 3;
            const int ng = min((int)gridDim.x, kWholeGroups), gi = blockIdx.x % ng;
            const int size = ((int)gridDim.x - gi + ng - 1) / ng;
            const unsigned long long one = 1ull << kVoteArrive;
            unsigned long long add = s_acc[par] + one;
            unsigned long long x = ctl_add(&a.ctl->group[q][gi][0], add) + add;
            if ((int)(x >> kVoteArrive) == size) {
                ctl_store(&a.ctl->group[nx][gi][0], 0);     // free: everyone has left the vote before this one
                ctl_store(&a.ctl->release[nx][gi][0], 0);
                add = (x & (one - 1)) + one;
                x = ctl_add(&a.ctl->root[q][0], add) + add;
                if ((int)(x >> kVoteArrive) == ng) {
                    ctl_store(&a.ctl->root[nx][0], 0);
                    for (int k = 0; k < ng; k++) ctl_store(&a.ctl->release[q][k][0], x);
                }
            }
            const unsigned long long *p = &a.ctl->release[q][gi][0];
            int ok = 1;
            const long long t0 = wall_clock64();
            x = ctl_load(p);
            for (int spin = 1; x == 0; spin++) {
                __builtin_amdgcn_s_sleep(1);
                x = ctl_load(p);
                if (((spin & 63) == 0 || a.wait == 0) && x == 0) {
                    const bool late = wall_clock64() - t0 > a.wait;
                    if (late) ctl_store(&a.ctl->abort_flag, 1);
                    if (late || ctl_load(&a.ctl->abort_flag)) {
                        ok = 0;
                        break;
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            s_total = x;
            s_ok = ok;
            s_acc[par ^ 1] = 0;
        }
        gen++;
        par ^= 1;
        __syncthreads();
        total = s_total;
        return s_ok != 0;
    };
    auto vcount = [](unsigned long long x) { return (int64_t)(x & ((1ull << kVoteChanged) - 1)); };

    // ---- one round ---------------------------------------------------------------------
    unsigned long long edges_done = 0;
    unsigned lifted = 0;
    // A thread's slot masks are kept as bits and tested where they are used: left to itself
    // the compiler turns them into a scalar register pair per slot and spills those.
    auto opaque = [](unsigned x) {
        asm volatile("" : "+v"(x));
        return x;
    };
    auto fold = [&](const int (&x)[R], bool mix, int mask) {
        const unsigned fl = opaque(flush);
        int vl = vl0, kk = INT_MAX;
#pragma unroll
        for (int j = 0; j < R; j++) {
            if (j >= per) break;
            const int m = mix ? (vl >= n0l ? -1 : 0) : mask;
            kk = min(kk, __builtin_elementwise_sub_sat(x[j], w[j]) ^ m);
            if ((fl >> j) & 1u) {
                atomicMin(&key[vl], kk);
                vl++;
                kk = INT_MAX;
            }
        }
    };
    auto sweep = [&](bool first, int r) -> int {
        int x[R];
        const char *vals = ONE ? (const char *)own : (const char *)a.val;
#pragma unroll
        for (int j = 0; j < R; j++) {
            x[j] = 0;
            if (j < per && !first) x[j] = *(const int *)(vals + su[j]);
        }
        if (mixed) fold(x, true, 0);
        else fold(x, false, any1 ? -1 : 0);
        edges_done += __popc(live);
        __syncthreads();
        int up = 0;
        for (int i = tid; i < nb; i += T) {
            const int d = key[i] ^ (i >= n0l ? -1 : 0);
            const int t = d > a.mg ? EGS_TOP : max(d, 0), old = own[i];
            key[i] = INT_MAX;
            if (old < t) {
                own[i] = t;
                if (!ONE) a.val[v0 + i] = t;
                if (a.rise) a.rise[v0 + i] = r;
                up++;
            }
        }
        lifted += up;
        return up;
    };

    // ---- one TOP proof attempt after round r; false: the launch was aborted ----------------
    int64_t marked = 0;
    int passes = 0, pruned = 0, cap_hit = 0, attempts = 0;
    long long marked_sum = 0;
    const int iscale = a.n + 1;
    const long long scale = iscale;
    const long long bound = scale * a.mg + (long long)a.n * (scale * a.wmax + 1);
    auto prove = [&](int r, int cap) -> bool {
        marked = 0;
        cap_hit = 0;
        unsigned long long tot;
        if (a.wmax <= 0 || !a.rise) return true;
        // histograms of the values against B_j = W 2^j, as k_gap_hist: windows, then floors
        for (int i = tid; i < 128; i += T) s_bins[i] = 0;
        __syncthreads();
        const unsigned W = (unsigned)a.wmax;
        for (int i = tid; i < nb; i += T) {
            const int x = own[i];
            if (x == EGS_TOP || x <= 0) continue;
            const unsigned below = ((unsigned)x - 1u) / W, q = below + 1u;      // q = ceil(x / W)
            if ((q & (q - 1u)) == 0) atomicAdd(&s_bins[31 - __clz(q)], 1);
            if (below > 0) atomicAdd(&s_bins[64 + 31 - __clz(below)], 1);
        }
        __syncthreads();
        if (!ONE) {
            int *gh = a.ctl->hist[attempts & 1], *other = a.ctl->hist[(attempts + 1) & 1];
            for (int i = tid; i < 128; i += T)
                if (s_bins[i])
                    __hip_atomic_fetch_add(&gh[i], s_bins[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (!vote(0, false, false, tot)) return false;
            for (int i = tid; i < 128; i += T) {
                s_bins[i] = __hip_atomic_load(&gh[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (blockIdx.x == 0) __hip_atomic_store(&other[i], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
        }
        if (tid == 0) s_ncand = whole_candidates(s_bins, a.wmax, a.mg, a.max_cands, s_cand);
        __syncthreads();
        const int ncand = s_ncand;
        for (int c = 0; c < ncand; c++) {
            const long long B = s_cand[c];
            int members = 0;
            for (int i = tid; i < nb; i += T) {
                const int x = own[i];
                const bool in = x != EGS_TOP && (B >= 0 ? x > B : a.rise[v0 + i] == r);
                const long long hv = x == EGS_TOP ? -kWInf : in ? scale * ((long long)a.mg - x) : kWInf;
                hown[i] = hv;
                if (!ONE) a.h[v0 + i] = hv;
                hk[i] = LLONG_MAX;
                members += in;
            }
            if (!vote(members, false, false, tot)) return false;
            const int64_t m0 = vcount(tot);
            if (m0 == 0) continue;
            unsigned mem = 0;                       // edges of the candidate's members
            {
                int vl = vl0;
#pragma unroll
                for (int j = 0; j < R; j++) {
                    if (j < cnt && w_member(hown[vl])) mem |= 1u << j;
                    if ((flush >> j) & 1u) vl++;
                }
            }
            bool converged = false, diverged = false;
            for (int p = 0; p < cap && !converged && !diverged; p++) {
                // owner 0 takes the maximum of w' + h over its edges (+inf: one leaves D, so
                // it breaks closure; -inf edges, to TOP, do not count), owner 1 the minimum
                // (+inf: none stays in D or reaches TOP, so it breaks closure)
                const unsigned fl = opaque(flush), mm = opaque(mem);
                int vl = vl0;
                long long best = LLONG_MAX;         // a minimum, of complements for owner 0
                constexpr int H = R < 8 ? R : 8;    // gathers in flight
                const char *hs = ONE ? (const char *)hown : (const char *)a.h;
#pragma unroll
                for (int j0 = 0; j0 < R; j0 += H) {
                    if (j0 >= per) break;
                    long long hu[H];
#pragma unroll
                    for (int j = 0; j < H; j++) {
                        hu[j] = 0;
                        if ((mm >> (j0 + j)) & 1u) hu[j] = *(const long long *)(hs + 2u * su[j0 + j]);
                    }
#pragma unroll
                    for (int j = 0; j < H; j++) {
                        const long long c = (long long)iscale * w[j0 + j] + hu[j];   // w' = iscale w + 1: the 1 below
                        best = min(best, c ^ (vl >= n0l ? 0ll : -1ll));
                        if ((fl >> (j0 + j)) & 1u) {
                            if ((mm >> (j0 + j)) & 1u) atomicMin(&hk[vl], best);
                            vl++;
                            best = LLONG_MAX;
                        }
                    }
                }
                __syncthreads();
                int alive = 0;
                bool ch = false, over = false;
                for (int i = tid; i < nb; i += T) {
                    const long long hv = hown[i];
                    if (!w_member(hv)) continue;
                    const long long b = (hk[i] ^ (i >= n0l ? 0ll : -1ll)) + 1;
                    hk[i] = LLONG_MAX;
                    long long nv = hv;
                    if (b > kWInf / 2) nv = kWInf;
                    else if (b > hv) {
                        nv = b;
                        over |= b > bound;
                    }
                    alive += nv < kWInf / 2;
                    if (nv != hv) {
                        hown[i] = nv;
                        if (!ONE) a.h[v0 + i] = nv;
                        ch = true;
                    }
                }
                if (!vote(alive, ch, over, tot)) return false;
                passes++;
                converged = ((tot >> kVoteChanged) & kVoteWaves) == 0;
                diverged = ((tot >> kVoteOver) & kVoteWaves) != 0;
            }
            const int64_t left = vcount(tot);
            pruned += left < m0;
            if (diverged || !converged) {
                cap_hit |= !diverged;
                continue;
            }
            if (left == 0) continue;
            for (int i = tid; i < nb; i += T)
                if (w_member(hown[i])) {
                    own[i] = EGS_TOP;
                    if (!ONE) a.val[v0 + i] = EGS_TOP;
                }
            __syncthreads();
            drop_top();
            marked = left;
            marked_sum += left;
            return true;
        }
        return true;
    };

    // ---- the run -----------------------------------------------------------------------
    unsigned long long tot = 0;
    int64_t r = a.round0, next_cert = a.next_cert;
    int gap = a.gap, cap = a.cap, certs = 0, wants = 0, status = kWholeLimit;
    int64_t initial = 0;
    const long long tick1 = wall_clock64();
    // a launch that goes on has rounds behind it whose risers are not known: it sweeps first
    bool known = false;
    // The round after a proof may read values from before it: the vertices marked TOP are stored
    // with no barrier behind them.  A quiet one says nothing.
    bool marks = false;
    for (;;) {
        if (known && !marks && vcount(tot) == 0) { status = kWholeDone; break; }
        if (r - a.round0 >= a.limit) break;
        marks = false;
        if (a.every > 0 && known && r >= next_cert) {
            const int before = passes;
            if (!prove((int)r, cap)) return;
            attempts++;
            if (marked > 0) {
                certs++;
                marks = !ONE;
            } else {
                gap = cert_next_gap(gap, a.every, passes - before + 2 * s_ncand);
                if (cap_hit) cap = min(cap * 2, a.max_passes);
            }
            next_cert = r + gap;
        }
        const bool first = r == 0;
        r++;
        const int up = sweep(first, (int)r);
        if (!vote(up, false, false, tot)) return;
        known = true;
        if (first) {
            initial = vcount(tot);
            if (initial == 0) r = 0;                // nothing is active: no round counts
        } else if (a.sparse_exit && vcount(tot) * a.m / a.n < a.dense_min && vcount(tot) > 0 &&
                   ++wants >= a.sparse_exit) {
            status = kWholeSparse;
            break;
        }
    }
    if (ONE)
        for (int i = tid; i < nb; i += T) {
            a.val[i] = own[i];
            if (a.mirror) a.mirror[i] = own[i];
        }
    // statistics: edges and lifts of the launch (processed = vertices times its rounds)
    {
        const unsigned long long lf = lifted;
        unsigned long long e = edges_done, l = lf;
        for (int d = 32; d >= 1; d >>= 1) {
            e += __shfl_xor(e, d, 64);
            l += __shfl_xor(l, d, 64);
        }
        if (lane == 0) {
            atomicAdd(&s_sum[0], e);
            atomicAdd(&s_sum[1], l);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (!ONE && tid < 2)
            __hip_atomic_fetch_add(&a.ctl->sum[tid], s_sum[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned long long dummy;
        if (!ONE && !vote(0, false, false, dummy)) return;
        if (lead && tid == 0) {
            WholeResult *o = a.out;
            o->status = status;
            o->rounds = r;
            o->initial = initial;
            o->attempts = attempts;
            o->certs = certs;
            o->pruned = pruned;
            o->passes = passes;
            o->marked = marked_sum;
            o->edges = initial == 0 && fresh && r == 0 ? 0 : (long long)(ONE ? s_sum[0] : ctl_load(&a.ctl->sum[0]));
            o->lifted = (long long)(ONE ? s_sum[1] : ctl_load(&a.ctl->sum[1]));
            o->next_cert = next_cert;
            o->gap = gap;
            o->cap = cap;
            o->ticks_setup = tick1 - tick0;
            o->ticks = wall_clock64() - tick0;
            __threadfence_system();
            __hip_atomic_store(&o->done, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// ---------------------------------------------------------------------------------------
// The smallest games: one workgroup, a thread per vertex (or V of them), no LDS atomics
// ---------------------------------------------------------------------------------------
//
// For games of out-degree at most D with n <= 1024 V: a thread keeps its vertices' edges,
// values, rise stamps and potentials in registers and LDS holds what others gather.  A round
// is D V gathers, three VALU operations each, and one workgroup barrier, in place; the form
// above spends its time on the folds' LDS atomics and its second phase (1.8 us a round at
// n = 1,499, degree 4, against 0.5 here).
template <int D, int V>
__global__ __launch_bounds__(1024) void k_whole_small(WholeArgs a) {
    extern __shared__ __align__(16) long long dyn[];
    __shared__ int s_flag[3];
    __shared__ int s_bins[128], s_ncand;
    __shared__ long long s_cand[16];
    __shared__ unsigned long long s_acc[2], s_sum[2];
    const int tid = threadIdx.x, T = blockDim.x, lane = tid & 63;
    const long long tick0 = wall_clock64();
    long long *hp = dyn;                            // potentials
    int *own = (int *)(dyn + a.nbmax);              // values
    const bool fresh = a.round0 == 0;
    // padding slots are neutral: below every candidate of a maximum (which the clamp cuts at
    // 0), past every candidate of a minimum
    unsigned su[V][D];                              // byte offset of the successor's value
    int w[V][D], val[V], rise[V], deg[V];
#pragma unroll
    for (int q = 0; q < V; q++) {
        const int v = q * T + tid;
        int s = 0, e = 0;
        if (v < a.n) {
            s = a.ptr[v];
            e = a.ptr[v + 1];
        }
        deg[q] = e - s;
        val[q] = v >= a.n || fresh ? 0 : a.val[v];
        rise[q] = v >= a.n || fresh || !a.rise ? 0 : a.rise[v];
        if (v < a.n) own[v] = val[q];
#pragma unroll
        for (int j = 0; j < D; j++) {
            su[q][j] = 0;
            w[q][j] = v >= a.n0 ? INT_MAX : INT_MIN;
            if (j < deg[q]) {
                const int2 x = a.edges[s + j];
                su[q][j] = 4u * (unsigned)x.x;
                w[q][j] = x.y;
            }
        }
    }
    if (tid < 3) s_flag[tid] = 0;
    if (tid < 2) { s_acc[tid] = 0; s_sum[tid] = 0; }
    __syncthreads();
    int slot = 0, par = 0;
    // whether any thread says so; one barrier (a flag is cleared two votes before its next use)
    auto any_vote = [&](bool x) -> bool {
        if (__any(x) && lane == 0) s_flag[slot] = 1;
        __syncthreads();
        const bool got = s_flag[slot] != 0;
        const int next = slot == 2 ? 0 : slot + 1;
        if (tid == 0) s_flag[next == 2 ? 0 : next + 1] = 0;
        slot = next;
        return got;
    };
    auto sum_vote = [&](int count, bool changed, bool over) -> unsigned long long {
        const int sum = egs_wave_sum(count);
        const unsigned long long mine = (unsigned long long)(unsigned)sum |
                                        ((unsigned long long)(__any(changed) ? 1 : 0) << kVoteChanged) |
                                        ((unsigned long long)(__any(over) ? 1 : 0) << kVoteOver);
        if (lane == 0 && mine) atomicAdd(&s_acc[par], mine);
        __syncthreads();
        const unsigned long long total = s_acc[par];
        if (tid == 0) s_acc[par ^ 1] = 0;
        par ^= 1;
        __syncthreads();
        return total;
    };
    auto vcount = [](unsigned long long x) { return (int64_t)(x & ((1ull << kVoteChanged) - 1)); };
    unsigned edges_done = 0, lifted = 0;            // of one launch: at most 8,192 rounds of 64 edges
    // a round; returns this thread's risers
    auto sweep = [&](bool first, int r) -> int {
        int up = 0;
#pragma unroll
        for (int q = 0; q < V; q++) {
            const int v = q * T + tid;
            const int m = v >= a.n0 ? -1 : 0;
            int x[D], kk = INT_MAX;
#pragma unroll
            for (int j = 0; j < D; j++) x[j] = first ? 0 : *(const int *)((const char *)own + su[q][j]);
#pragma unroll
            for (int j = 0; j < D; j++) kk = min(kk, __builtin_elementwise_sub_sat(x[j], w[q][j]) ^ m);
            const int d = kk ^ m;
            const int t = d > a.mg ? EGS_TOP : max(d, 0);
            if (val[q] != EGS_TOP) edges_done += deg[q];
            if (v < a.n && val[q] < t) {
                val[q] = t;
                own[v] = t;
                rise[q] = r;
                up++;
            }
        }
        lifted += up;
        return up;
    };

    int64_t marked = 0;
    int passes = 0, pruned = 0, cap_hit = 0, attempts = 0;
    long long marked_sum = 0;
    const int iscale = a.n + 1;
    const long long scale = iscale;
    const long long bound = scale * a.mg + (long long)a.n * (scale * a.wmax + 1);
    // one TOP proof attempt after round r, as in k_whole (every thread enters and leaves together)
    auto prove = [&](int r, int cap) {
        marked = 0;
        cap_hit = 0;
        if (a.wmax <= 0) return;
        for (int i = tid; i < 128; i += T) s_bins[i] = 0;
        __syncthreads();
        const unsigned W = (unsigned)a.wmax;
#pragma unroll
        for (int q = 0; q < V; q++) {
            const int x = val[q];
            if (q * T + tid >= a.n || x == EGS_TOP || x <= 0) continue;
            const unsigned below = ((unsigned)x - 1u) / W, c = below + 1u;      // c = ceil(x / W)
            if ((c & (c - 1u)) == 0) atomicAdd(&s_bins[31 - __clz(c)], 1);
            if (below > 0) atomicAdd(&s_bins[64 + 31 - __clz(below)], 1);
        }
        __syncthreads();
        if (tid == 0) s_ncand = whole_candidates(s_bins, a.wmax, a.mg, a.max_cands, s_cand);
        __syncthreads();
        const int ncand = s_ncand;
        for (int c = 0; c < ncand; c++) {
            const long long B = s_cand[c];
            int members = 0;
            long long h[V];
#pragma unroll
            for (int q = 0; q < V; q++) {
                const int v = q * T + tid, x = val[q];
                const bool in = v < a.n && x != EGS_TOP && (B >= 0 ? x > B : rise[q] == r);
                h[q] = x == EGS_TOP ? -kWInf : in ? scale * ((long long)a.mg - x) : kWInf;
                if (v < a.n) hp[v] = h[q];
                members += in;
            }
            unsigned long long tot = sum_vote(members, false, false);
            const int64_t m0 = vcount(tot);
            if (m0 == 0) continue;
            bool converged = false, diverged = false;
            for (int p = 0; p < cap && !converged && !diverged; p++) {
                int alive = 0;
                bool ch = false, over = false;
#pragma unroll
                for (int q = 0; q < V; q++) {
                    const int v = q * T + tid;
                    if (!w_member(h[q])) continue;
                    const bool owner1 = v >= a.n0;
                    long long best = owner1 ? LLONG_MAX : LLONG_MIN;
#pragma unroll
                    for (int j = 0; j < D; j++) {
                        if (j >= deg[q]) break;
                        const long long cnd =
                            (long long)iscale * w[q][j] + *(const long long *)((const char *)hp + 2u * su[q][j]);
                        best = owner1 ? min(best, cnd) : max(best, cnd);
                    }
                    best += 1;
                    if (best > kWInf / 2) {         // breaks closure (see k_whole)
                        h[q] = kWInf;
                        hp[v] = kWInf;
                        ch = true;
                        continue;
                    }
                    alive++;
                    if (best > h[q]) {
                        h[q] = best;
                        hp[v] = best;
                        ch = true;
                        over |= best > bound;
                    }
                }
                tot = sum_vote(alive, ch, over);
                passes++;
                converged = ((tot >> kVoteChanged) & kVoteWaves) == 0;
                diverged = ((tot >> kVoteOver) & kVoteWaves) != 0;
            }
            const int64_t left = vcount(tot);
            pruned += left < m0;
            if (diverged || !converged) {
                cap_hit |= !diverged;
                continue;
            }
            if (left == 0) continue;
#pragma unroll
            for (int q = 0; q < V; q++)
                if (w_member(h[q])) {
                    val[q] = EGS_TOP;
                    own[q * T + tid] = EGS_TOP;
                }
            __syncthreads();
            marked = left;
            marked_sum += left;
            return;
        }
    };

    int64_t r = a.round0, next_cert = a.next_cert, initial = 0;
    int gap = a.gap, cap = a.cap, certs = 0, status = kWholeLimit;
    const long long tick1 = wall_clock64();
    bool known = false, up = true;
    for (;;) {
        if (known && !up) { status = kWholeDone; break; }
        if (r - a.round0 >= a.limit) break;
        if (a.every > 0 && known && r >= next_cert) {
            prove((int)r, cap);
            attempts++;
            if (marked > 0) {
                certs++;
            } else {
                // without cert_next_gap's bound: its registers cost every round 4% (plain value
                // iteration at n = 1,499: 690 us against 660)
                gap = min(gap * 2, 1 << 16);
                if (cap_hit) cap = min(cap * 2, a.max_passes);
            }
            next_cert = r + gap;
        }
        r++;
        if (r == 1) {
            initial = vcount(sum_vote(sweep(true, 1), false, false));
            up = initial > 0;
            if (!up) r = 0;                         // nothing is active: no round counts
        } else {
            up = any_vote(sweep(false, (int)r) > 0);
        }
        known = true;
    }
#pragma unroll
    for (int q = 0; q < V; q++) {
        const int v = q * T + tid;
        if (v < a.n) {
            a.val[v] = val[q];
            if (a.mirror) a.mirror[v] = val[q];
            if (a.rise) a.rise[v] = rise[q];
        }
    }
    unsigned long long e = edges_done, l = lifted;
    for (int d = 32; d >= 1; d >>= 1) {
        e += __shfl_xor(e, d, 64);
        l += __shfl_xor(l, d, 64);
    }
    if (lane == 0) {
        atomicAdd(&s_sum[0], e);
        atomicAdd(&s_sum[1], l);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
        WholeResult *o = a.out;
        o->status = status;
        o->rounds = r;
        o->initial = initial;
        o->attempts = attempts;
        o->certs = certs;
        o->pruned = pruned;
        o->passes = passes;
        o->marked = marked_sum;
        o->edges = fresh && r == 0 ? 0 : (long long)s_sum[0];
        o->lifted = (long long)s_sum[1];
        o->next_cert = next_cert;
        o->gap = gap;
        o->cap = cap;
        o->ticks_setup = tick1 - tick0;
        o->ticks = wall_clock64() - tick0;
        __threadfence_system();
        __hip_atomic_store(&o->done, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ---------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------

// The share of the game one workgroup takes and the launch shape, or nb == 0 when the game
// does not suit a single launch.
WholePlan whole_plan(int n, int64_t m, int mg, int wmax, int max_outdeg, int max_nb) {
    WholePlan p{};
    // a TOP value less a weight stays past MG; potentials stay far below kWInf
    if ((int64_t)mg + wmax >= EGS_TOP) return p;
    if (((double)n + 1) * mg + (double)n * (((double)n + 1) * wmax + 1) > 0.5e18) return p;
    // at most 16 slots a thread, of which 8 to 16 registers (of 128 a thread has) spill already
    const int D = max_outdeg <= 4 ? 4 : max_outdeg <= 8 ? 8 : 16;
    const int V = n <= 1024 ? 1 : 2;
    if (max_outdeg <= 16 && n <= 2048 && D * V <= 16) {
        p.small_d = D;
        p.small_v = V;
        p.nb = 1;
        p.nbmax = n;
        p.threads = ((n + V - 1) / V + 63) / 64 * 64;
        return p;
    }
    if (n <= kWholeOneN && m <= kWholeOneM) {
        p.nb = 1;
        p.nbmax = n + 1;
        p.threads = 64;
        while (p.threads < 1024 && p.threads * 4 < m) p.threads *= 2;
        p.per = (int)((m + p.threads - 1) / p.threads);
        p.share = m + n;
        return p;
    }
    const int64_t weight = m + n;
    const int64_t most = std::min(kWholeMaxNb, max_nb);
    const int64_t nb = std::min<int64_t>(most, std::max<int64_t>(8, (weight + kWholeShare - 1) / kWholeShare));
    if (nb < 2) return p;
    const int64_t share = (weight + nb - 1) / nb;
    // a share ends past its last vertex: up to share + max_outdeg edges, share / 2 + 1 vertices
    if (share > kWholeShareMax || share + max_outdeg > 1024 * 16) return p;
    p.nb = (int)nb;
    p.nbmax = (int)(share / 2 + 2);
    p.threads = 1024;
    p.per = (int)((share + max_outdeg + 1023) / 1024);
    p.share = share;
    return p;
}

hipError_t launch_whole_prep(const WholePlan &p, const DevGame &g, WholeCtl *ctl, bool fresh, hipStream_t st) {
    hipLaunchKernelGGL(k_whole_prep, dim3(grid_for((int64_t)g.n + 1, 256, 1024)), dim3(256), 0, st, g.ptr, g.n, p.nb,
                       p.share, fresh ? 1 : 0, g.val, ctl);
    return hipGetLastError();
}

// LDS bytes of a workgroup.
size_t whole_lds(const WholePlan &p) { return (size_t)p.nbmax * (p.small_d ? 12 : 24) + 16; }

hipError_t launch_whole(const WholePlan &p, const WholeArgs &a, hipStream_t st) {
    const size_t lds = whole_lds(p);
    if (p.small_d) {
#define EGS_SMALL(DD, VV)                                                                   \
    if (p.small_d == DD && p.small_v == VV)                                                 \
        hipLaunchKernelGGL((k_whole_small<DD, VV>), dim3(1), dim3(p.threads), lds, st, a);
        EGS_SMALL(4, 1) EGS_SMALL(4, 2) EGS_SMALL(8, 1) EGS_SMALL(8, 2) EGS_SMALL(16, 1)
#undef EGS_SMALL
        return hipGetLastError();
    }
    const dim3 grid(p.nb), threads(p.threads);
#define EGS_WHOLE(RR)                                                                       \
    if (p.nb == 1) hipLaunchKernelGGL((k_whole<RR, true>), grid, threads, lds, st, a);     \
    else hipLaunchKernelGGL((k_whole<RR, false>), grid, threads, lds, st, a);
    if (p.per <= 4) { EGS_WHOLE(4) }
    else if (p.per <= 8) { EGS_WHOLE(8) }
    else { EGS_WHOLE(16) }
#undef EGS_WHOLE
    return hipGetLastError();
}

}  // namespace egs
