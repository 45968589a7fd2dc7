// egs_internal.h -- structures shared between the HIP translation units of libegs.so.
#pragma once

#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdint.h>

#include <atomic>

struct egs_solver;

namespace egs {

// Workgroups of a solver's single launches (egs_whole.hip) at most.
void solver_limit_whole(egs_solver *s, int max_nb);

// Compute units of a device held by this process's launches under way: single launches, whose
// workgroups wait for one another, and the many-games kernel, whose workgroups stay for long.
// A workgroup of either takes a unit (1,024 threads of 87 to 128 registers; all of its LDS).
// A launch's workgroups go to the eight XCDs in turn and stay with their XCD, full or not:
// every launch holds as many units of each, and the many-games kernel has a workgroup per game
// at most (with 256 for 100 games the first to come took them, whole XCDs at a time, and a solve
// beside them waited for their end; 200 games with a workgroup each leave it its 0.6 ms).
inline int units_of(int workgroups, int cus) { return workgroups > cus ? cus : (workgroups + 7) / 8 * 8; }
struct DeviceUnits {
    std::atomic<int> single{0}, games{0};
};
DeviceUnits &device_units(int device);
struct UnitsHeld {
    std::atomic<int> &held;
    int n;
    UnitsHeld(std::atomic<int> &h, int units) : held(h), n(units) { held.fetch_add(n); }
    ~UnitsHeld() { held.fetch_sub(n); }
    UnitsHeld(const UnitsHeld &) = delete;
};

// Frontier lists are split into kSub sub-queues of sub_cap slots plus one overflow region
// of n slots; a workgroup appends to sub-queue (blockIdx.x % kSub), so no counter sees
// more than a few dozen workgroups' atomics per round.
constexpr int kSub = 64;
constexpr int kListCounters = kSub + 1;     // kSub sub-queue counters + overflow counter
constexpr int kLdsCap = 2048;               // per-workgroup LDS staging of appends
constexpr int kStatSlots = 8192;            // upper bound on any round kernel's grid

// Round modes, decided on the device at the start of every round from the previous
// round's mode and output-list size (see decide_mode in egs_rounds.hip).
enum : int { MODE_QUEUE = 0, MODE_LIFTED = 1, MODE_DENSE = 2, MODE_DONE = 3 };

// One game resident on the device, passed by value to every kernel.
struct DevGame {
    int n, n0, mg;
    int64_t m;
    const int *ptr;       // n+1 CSR offsets (internal numbering, owner-0 first)
    const int2 *edges;    // m packed {successor, weight}
    const int *cptr;      // n+1 CSC offsets
    const int *cpred;     // m predecessors
    const int *cweight;   // the weights of their edges (null: the transpose does not hold them)
    int *val;             // n values
    int *stamp;           // n: last round a vertex was claimed for / queued for
    int *list[2];         // output lists, ping-pong: kSub*sub_cap + n slots each
    int sub_cap;
    int *lcnt;            // 3 slots x kListCounters
    int *mode;            // [0..2] mode of round r at r % 3; [3] a round whose input list
                          // holds its count but no items (a phased dense round before the transpose)
    int *dbig, *dhuge;    // per-round deferral lists (sparse modes)
    int *ring;            // [3..5] dbig counters, [6..8] dhuge counters, [9] nsbig, [10] nshuge,
                          // [11] a round that must sweep all vertices (after a TOP proof),
                          // [12] 1 once the transpose exists (sparse rounds allowed),
                          // [13] rounds that would have gone sparse without it,
                          // [14] the absolute number of the next batch's first round,
                          // [15] nonzero once any vertex has been set to TOP
    const int *sbig;      // static: vertices with big_deg < deg <= huge_deg
    const int *shuge;     // static: vertices with deg > huge_deg
    int big_deg, huge_deg;
    int64_t dense_min;    // estimated work (vertices) at or above which a round sweeps all
    unsigned long long *stats;  // per-workgroup slots of {processed, edges, lifted, preds}
    int *rounds_done;     // last round that was not MODE_DONE
    int *rise;            // n: round in which each vertex last rose (TOP proof candidates);
                          // null when proofs are off
    // Dense rounds in successor-range phases (phases > 1): in phase s a vertex folds its
    // edges whose successor lies in slice s = [s << slice_shift, (s + 1) << slice_shift), so
    // the value gathers of the whole grid come from one slice small enough to stay in L2.
    int phases;           // 1 = one in-place sweep (body_dense)
    int slice_shift;
    // Slice layout in tiles of kSliceTile vertices: tile T's low-degree edges lie in its own
    // CSR range from ptr[T * kSliceTile], grouped by (slice, vertex).  For tile T and slice
    // s, slen[(T * phases + s) * kSliceTile + j] is the number of edges of vertex
    // T * kSliceTile + j into slice s (0 above big_deg and past n) and
    // sbase[(T * phases + s) * kSliceWaves + w] is where the edges of wave w's 64 vertices
    // start; a vertex's edges follow those of the lower lanes of its wave.
    const uint8_t *slen;
    const int *sbase;
    const void *sedges;   // uint32 (w << sshift) | succ when sshift > 0, else int2 {succ, w}
    int sshift;
    const unsigned long long *bigmask;   // bit v: vertex v is above big_deg (lifted by the wave/block kernels)
    // Dense rounds over binned edges (egs_bins.h; bins > 0): slices of the successors, successors
    // per slice with floor(2^32 / bin_w) + 1, parts of the chunks per slice, chunks.
    int bins, bin_w, bin_parts, nchunks;
    unsigned bin_magic;
    uint32_t *bedges;     // (w << 15) | place in slice, per chunk grouped by slice
    uint16_t *bids;       // the edge's vertex in the chunk
    int *cand;            // a - w of each edge (8 bytes of room: the proof passes keep w' + h)
    int *boff;            // [bins + 1][nchunks]: where a chunk's run of a slice starts
    int *bchunk;          // nchunks + 1 pairs: a chunk's first edge and that edge's vertex
    int4 *bdesc;          // nchunks: first vertex, vertices and split flags, first and last padded edge
    int bin_share;        // places of the chunks' line per chunk
    int bin_once;         // 1: words, vertex numbers and candidates outgrow the memory-side cache
    int hubs;             // some vertex is above huge_deg
    int round_grid;       // workgroups of k_round's low-degree part
    int hub_fused;        // 1: k_round's grid continues with the hub part in dense rounds
    int wave_grid, block_grid;   // workgroups of the wave and workgroup-per-vertex hub bodies
    int phase_grid;       // workgroups of the phased kernels (about what the device holds at once)
    int phase_tiles;      // tiles of the slice layout per workgroup, at most 32 (96 KB of LDS
                          // at 12 bytes per vertex; the dense kernel keeps a 32-bit mask of them)
    int *hacc, *hcnt;     // n each: partial keys and finished chunks of the vertices above
                          // huge_deg (TOP and 0 between rounds)
    long long *hbest;     // n: partial longest-path candidates of the vertices above huge_deg
                          // in proof passes (each owner's identity between passes)
    int *hflag;           // n: bit 0 a successor changed, bit 1 an edge leaves D (0 between passes)
};

constexpr int kMaxPhases = 16;             // successor slices of a phased dense round, at most
constexpr int kDefaultPhases = 8;          // slices of 2 MB of values on the 2^22-vertex game
constexpr int kPhaseMinN = 1 << 20;        // up to this many vertices the values (4 MB) fit one XCD's L2
constexpr int kSliceTile = 256;            // vertices per tile of the slice layout
constexpr int kSliceWaves = kSliceTile / 64;
constexpr int kMaxSliceDeg = 255;          // a vertex's edges into one slice fit a byte

// Binned games: successors of a slice at most (128 KB of values; half of that up to kBinHalfN
// vertices), slices at most, the largest |w| of a packed edge.
constexpr int kBinSlice = 1 << 15;
constexpr int kBinHalfN = 1 << 21;
constexpr int kBinMax = 512;
constexpr int kBinWmax = 65535;
constexpr int kBinHead = 4;                // places of a vertex on the chunks' line, before its edges
constexpr int kBinShareMin = 4096, kBinShareMax = 16384;   // places of a chunk
constexpr int kBinSplitFirst = 1 << 29, kBinSplitLast = 1 << 30, kBinNv = (1 << 29) - 1;   // bdesc's second word
constexpr int kBinPad = 16;                // runs are padded to this many edges
constexpr int kBinMinN = 400000;             // the rule on degrees and both sides' times: bins_pay

// Edge k of the slice layout: successor and weight.
template <bool PACK>
__device__ __forceinline__ void slice_edge(const DevGame &g, int k, int &succ, int &w) {
    if (PACK) {
        const uint32_t e = ((const uint32_t *)g.sedges)[k];
        succ = (int)(e & ((1u << g.sshift) - 1u));
        w = ((int)e) >> g.sshift;
    } else {
        const int2 e = ((const int2 *)g.sedges)[k];
        succ = e.x;
        w = e.y;
    }
}

// Launch shape of one round.
struct LaunchShape {
    int group;       // lanes per vertex in k_round (1..64)
    int grid;        // workgroups of k_round
    int use_wave, use_block;
    int wave_grid, block_grid;
};

// Rounds to the next proof attempt after one that proved nothing and cost as much as `cost`
// rounds: twice as many as to this one, while attempts would take less than a sixteenth of the
// rounds.  Doubled without end, a long run whose vertices could be proved at round r went on to
// the next power of two: games of degree 2 with 485,000 vertices took 61, 135 and 368 ms, with
// at most eight times the cost between attempts 34, 91 and 256; runs that no proof helps took
// 2 to 8% longer then, which sixteen halves.
__host__ __device__ inline int cert_next_gap(int gap, int every, int cost) {
    const int64_t twice = 2 * (int64_t)gap, most = 16 * (int64_t)cost, g = twice < most ? twice : most;
    return (int)(g > every ? g : every);
}

// A whole solve in one launch (egs_whole.hip).
constexpr int kWholeMaxNb = 256;           // workgroups at most
constexpr int kWholeGroups = 8;            // groups of workgroups in a vote
constexpr int64_t kWholeWait = 400000;     // barrier wait limit (4 ms) before a launch gives up
constexpr int kWholeOneN = 5999, kWholeOneM = 8192;    // one workgroup up to this size (8 edges a thread; with
                                           // 16 it spills: n = 4,000, degree 4: 160 us against 120 on 8 workgroups)
// Vertices + edges per workgroup while workgroups are left.  Device time of a solve (degree
// 2..16, us) at shares of 1,536 / 2,304 / 3,072 / 4,608 / 6,144: n = 9,973: 71 / 71 / 74 / 85 / 93;
// n = 30,011: 113 / 100 / 96 / 102 / 101; n = 87,148: 166 / 166 / 166 / 170 / 161.
constexpr int kWholeShare = 3072;
constexpr int kWholeShareMax = 7168;       // past this (all workgroups in use) the round kernels win:
                                           // n = 262,147, degree 8: 444 us against 353
enum : int { kWholeNone = 0, kWholeDone = 1, kWholeLimit = 2, kWholeSparse = 3 };

struct WholeCtl {
    unsigned long long root[4][16];        // vote words, a cache line each: all groups,
    unsigned long long group[4][kWholeGroups][16];    // the workgroups of a group,
    unsigned long long release[4][kWholeGroups][16];  // the total, handed to a group
    unsigned long long abort_flag, pad0[15];
    unsigned long long sum[16];            // edges relaxed, lifts
    int hist[2][128];                      // value histograms of the proof attempts, in turn
    int bound[kWholeMaxNb + 1];            // first vertex of each workgroup
};
struct WholeResult {
    int status, attempts, certs, pruned, gap, cap;
    long long rounds, initial, passes, marked, edges, lifted, next_cert, ticks_setup, ticks;
    unsigned done;                         // the launch's seq, stored last
};
struct WholeArgs {
    int n, n0, mg, wmax;
    int64_t m;
    const int *ptr;
    const int2 *edges;
    int *val, *rise;                       // rise: null without proofs
    long long *h;
    WholeCtl *ctl;
    WholeResult *out;
    int *mirror;                           // a copy of the values for the host (one workgroup; may be null)
    int nbmax;                             // vertices of a workgroup at most (LDS)
    int64_t limit;                         // rounds of this launch at most
    int64_t round0, next_cert;             // rounds already run; the round of the next attempt
    int every, gap, cap, max_passes, max_cands;
    int sparse_exit;                       // leave after this many rounds below dense_min (0: never)
    int64_t dense_min;
    int64_t wait;                          // barrier wait limit in 100 MHz ticks
    unsigned seq;
};
struct WholePlan {
    int nb, nbmax, threads, per;           // workgroups (0: not for this game), LDS vertices, threads, edges a thread
    int64_t share;                         // vertices + edges per workgroup
    int small_d, small_v;                  // a thread per vertex: edge slots, vertices a thread (0: not)
};
WholePlan whole_plan(int n, int64_t m, int mg, int wmax, int max_outdeg, int max_nb);
size_t whole_lds(const WholePlan &p);
hipError_t launch_whole_prep(const WholePlan &p, const DevGame &g, WholeCtl *ctl, bool fresh, hipStream_t st);
hipError_t launch_whole(const WholePlan &p, const WholeArgs &a, hipStream_t st);

// What a load has to know of its game, reduced on the device: one partial per workgroup, then
// launch_load_finish adds them up and stores the record (`done`, its number, last).
struct LoadPartial {
    unsigned long long mg;                 // sum over the workgroup's rows of max(0, max -w)
    int dmax, wmax;                        // largest out-degree and |w|
};
struct LoadResult {
    unsigned long long mg;
    int dmax, wmax, n0, bad;
    unsigned done;
};
constexpr int kLoadGrid = 1024;            // workgroups (and partials) at most
// Workgroup maxima and the sum of x, d and w to *out, by thread 0 (256 threads).
__device__ __forceinline__ void load_partial(unsigned long long x, int d, int w, LoadPartial *out) {
    __shared__ unsigned long long sx[4];
    __shared__ int sd[4], sw[4];
    for (int k = 32; k >= 1; k >>= 1) {
        x += __shfl_xor(x, k, 64);
        d = max(d, __shfl_xor(d, k, 64));
        w = max(w, __shfl_xor(w, k, 64));
    }
    const int wid = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sx[wid] = x;
        sd[wid] = d;
        sw[wid] = w;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        *out = LoadPartial{sx[0] + sx[1] + sx[2] + sx[3], max(max(sd[0], sd[1]), max(sd[2], sd[3])),
                           max(max(sw[0], sw[1]), max(sw[2], sw[3]))};
}

// |w| as the host checks take it (INT_MIN counts as INT_MAX).
__device__ __forceinline__ int load_abs(int w) { return w < 0 ? (w == INT_MIN ? INT_MAX : -w) : w; }
// Device arrays into the solver's ptr and edges, with the statistics (mg is not summed).
hipError_t launch_load_device(const int *ptr, const int *succ, const int *w, int n, int64_t m, int *ptr_out,
                              int2 *edges, LoadPartial *part, int *nparts, hipStream_t st);
hipError_t launch_load_finish(const LoadPartial *part, int nparts, const int *n0, const int *bad, unsigned seq,
                              LoadResult *out, hipStream_t st);

hipError_t launch_unpack(const uint32_t *packed, int shift, int2 *edges, int64_t m, hipStream_t st);
hipError_t launch_transpose(const DevGame &g, int *tile_sum, int *fill, hipStream_t st);
// The transpose as a two-level stable counting sort (egs_transpose.hip): cpred in ascending
// source order per column.  Buffers: counts and offs of transpose_counts_len + 1 ints each,
// scan_tiles of transpose_counts_len / 4096 + 2 ints, items[m].  transpose_sorted_fits
// says whether a game's sizes fit the buffers.
int transpose_bshift(int n);
int64_t transpose_counts_len(int n, int64_t m);
bool transpose_sorted_fits(int n, int64_t m, int64_t counts_cap, int64_t items_cap);
// cweight (may be null, for games that transpose_weights_fit): the weights of cpred's edges.
bool transpose_weights_fit(int n, int wmax);
hipError_t launch_transpose_sorted(const DevGame &g, int *counts, int *offs, int *scan_tiles, int2 *items, int *cweight,
                                   hipStream_t st);
// bad (may be null): a non-zero word makes the kernels return at once.
hipError_t launch_exclusive_scan(const int *in, int n, int *tile_sum, int *out, hipStream_t st,
                                 const int *bad = nullptr);
constexpr int kTrTileEdges = 1 << 14;        // edges per tile of the sorted transpose

// A game in read order on the device and the work arrays of its renaming (egs_ingest.hip).
struct ReadOrderBuffers {
    const uint8_t *owner;                      // n: 0 = owner 0 (token MAX), else owner 1
    const int *rptr, *rsucc, *rw;              // read-order CSR, successors as read indices
    int *flag0, *pre0, *rev, *ext_of_int, *deg, *scan_tiles;   // n (+1) each; scan_tiles n/4096 + 1
};
hipError_t launch_read_order_check(const int *rptr, const int *rsucc, int n, int64_t m, int *bad, hipStream_t st);
// bad (may be null): a non-zero word makes every kernel return at once.  The partials take the
// place of flag0; their number goes to *nparts.
hipError_t launch_internalise(const ReadOrderBuffers &b, int n, const int *bad, int *ptr, int2 *edges,
                              LoadPartial **part, int *nparts, hipStream_t st);
hipError_t launch_classify(const DevGame &g, int *counts, hipStream_t st);
// in_slices: the slice set-up (init) already stored the initial state of the vertices up to
// big_deg and counted, without listing, the active ones (no transpose: round 1 sweeps densely)
hipError_t launch_init(const DevGame &g, hipStream_t st, bool in_slices);
hipError_t launch_slices(const DevGame &g, hipStream_t st, bool init);
// Binned games: values to 0 and the chunk bounds; then the layout, with round 1 done on the
// way (`first`: what follows is round 2) or not.
int bin_share(int n, int64_t m, int bins);
inline size_t bin_key_slots(const DevGame &g) { return (size_t)(g.bin_share / (kBinHead + 1) + 4); }   // vertex words of a chunk, with the padding's
hipError_t launch_bin_prep(const DevGame &g, hipStream_t st);
hipError_t launch_bin_build(const DevGame &g, bool first, hipStream_t st);
int pack_shift(int n, int wmax);
// Round j of a batch (absolute round ring[14] + j); launch_advance ends the batch.
hipError_t launch_round(const DevGame &g, const LaunchShape &sh, int j, hipStream_t st);
hipError_t launch_advance(const DevGame &g, int rounds, hipStream_t st);
// Rounds in one workgroup from the next one on, `limit` at most, while each is sparse and its
// list short; ring[14] tells the round reached.  For lists of up to tail_items(sh).
constexpr int kTailLanes = 2048;           // items times lanes a vertex: two turns of the workgroup
int tail_items(const LaunchShape &sh);
hipError_t launch_tail(const DevGame &g, const LaunchShape &sh, int limit, hipStream_t st);
// Round `next` is the first of the round kernels on values reached otherwise (after
// launch_prepare_reset): a full sweep, or none when they have converged.
hipError_t launch_resume(const DevGame &g, int next, bool converged, hipStream_t st);
hipError_t launch_prepare_reset(const DevGame &g, hipStream_t st);
hipError_t launch_sum_stats(const DevGame &g, int nslots, unsigned long long *out, hipStream_t st);
hipError_t launch_violations(const DevGame &g, unsigned long long *out, hipStream_t st);
hipError_t launch_winning(const int *val, int n, unsigned *out, hipStream_t st);
hipError_t launch_hbest_reset(const DevGame &g, hipStream_t st);
int grid_for(int64_t work, int threads, int cap);

// Certified TOP detection (egs_accel.hip).
struct CertBuffers {
    int *hist;        // device: 2 x 64 histogram bins + 8 flags
    long long *h;     // device: n longest-path potentials
    int *bfcnt;       // device: ring of 64 pass counters
    unsigned *bits;   // device: 3 two-level bitmaps (ceil(n/32) words + a bit-per-word summary)
    int *pinned;      // host pinned: 2 x 64 + 4 + 64 ints
    hipEvent_t ev = nullptr;   // waits on read-backs go through this event when set (else the stream)
};
// Wait for everything queued on `st` so far: through `ev` (recorded, then waited on) when
// given, else the whole stream.
inline hipError_t wait_queued(hipEvent_t ev, hipStream_t st) {
    if (!ev) return hipStreamSynchronize(st);
    hipError_t e = hipEventRecord(ev, st);
    return e == hipSuccess ? hipEventSynchronize(ev) : e;
}
struct CertResult {
    int threshold;       // last threshold tried
    int tried;           // candidates tried
    int passes;          // longest-path passes over all candidates
    int marked;          // vertices set to TOP
    int closure_failed;  // candidates that lost vertices to the closure check
    int cap_hit;         // some candidate ran out of passes (neither converged nor diverged)
    int last_passes;     // passes of the last candidate that converged (0: none did)
};
int gap_candidates(const int *win, const int *flo, int wmax, int mg, int64_t *out, int max_out);
// The value histogram of the next attempt, queued with its read-back into the pinned area.
hipError_t certify_prefetch(const DevGame &g, const CertBuffers &cb, int wmax, hipStream_t st);
// stop (may be null): polled before each candidate and each chunk of passes; a set flag
// abandons the attempt with nothing marked.  pass_hint: passes an earlier attempt of the
// same run needed (0: none yet), which sizes the first chunk queued before a read-back.
int certify_top(const DevGame &g, const CertBuffers &cb, int wmax, int last, int cap, int max_cands, bool has_big,
                bool hist_ready, const volatile uint32_t *stop, int pass_hint, hipStream_t st, CertResult &res);
// Potentials certifying that every TOP vertex of the current values is won by player 1
// (cb.h: >= 0 on the certified set, -1 elsewhere).  Returns 1 when the whole TOP set is
// certified, 0 when not (closure failed, divergence or the pass cap; see res), -1 on a HIP
// error, -2 when the potentials could overflow 64 bits.
int certify_all_top(const DevGame &g, const CertBuffers &cb, int wmax, int max_passes, bool has_big,
                    hipStream_t st, CertResult &res);

}  // namespace egs
