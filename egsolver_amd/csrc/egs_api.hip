// egs_api.hip -- C-ABI of libegs.so: device queries and the one-game solver object.
//
// The solver object owns one device workspace.  The round loop keeps the frontier size
// on the device: rounds are enqueued in batches and the host reads one counter per
// batch through pinned memory, one batch behind, so the GPU never waits for the host
// between rounds (the reference blocks on thrust::remove's count twice per round,
// src/dev_EG_alg.cu:346-373).
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <chrono>

#include "../../include/egs.h"
#include "egs_device.h"
#include "egs_internal.h"
#include "egs_pack.h"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

#define HIP_TRY(expr)                                                                       \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess)                                                               \
            return fail(EGS_E_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_),   \
                        __FILE__, __LINE__);                                                \
    } while (0)

int check_gfx950(int device) {
    hipDeviceProp_t p;
    HIP_TRY(hipGetDeviceProperties(&p, device));
    if (strncmp(p.gcnArchName, "gfx950", 6) != 0)
        return fail(EGS_E_HIP, "device %d is %s; libegs.so is built for gfx950 only", device,
                    p.gcnArchName);
    return EGS_OK;
}

// Loop bound of src/egsolver.c:64-90: a negative request means n*m*MG+1, saturated to
// LONG_MAX-1 on overflow.
int64_t egs_max_loop_c(int64_t m, int64_t n, int64_t mg, int64_t maxloop) {
    if (maxloop >= 0) return maxloop;
    if (mg > (INT64_MAX - 1) / (n * m)) return INT64_MAX - 1;
    return n * m * mg + 1;
}

// Offsets (in ints) inside the solver's pinned readback block.
constexpr int kPinProbe = 2048;   // 2 x kProbeStride: per-batch counter probes
constexpr int kProbeStride = 512;
constexpr int kPinInit = 320;     // kListCounters ints
constexpr int kPinConv = 448;     // kListCounters ints
constexpr int kPinStats = 640;    // 6 x u64
constexpr int kPinViol = 704;     // 1 x u64
constexpr int kPinCert = 1024;    // certification readbacks (2 x 64 + 4 + 64 ints)
constexpr int kPinOne = 1281;     // the constant 1 (raises ring[12])
constexpr int kPinLoad = 768;     // a LoadResult
constexpr int kPinWhole = 1344;   // a WholeResult
static_assert(kPinWhole * 4 + sizeof(egs::WholeResult) <= 4 * 2048, "the read-back area holds a WholeResult");
constexpr int kProbeWant = 100;   // offset in a probe slot of ring[13] when it needs a copy of its own
// The transpose costs about ten dense rounds to build, and a sparse round saves at most one
// dense round: build it once this many rounds have wanted it (a proof usually leaves only a
// round or two, which do not pay for it).
constexpr int kSparseWantRounds = 6;
// A binned dense round costs a third to a half of a sweep: more of them before the transpose.
constexpr int kSparseWantBinned = 16;
constexpr int kCertFirstCap = 64;     // longest-path passes per candidate at the first attempt
constexpr int kCertCandidates = 8;    // gap thresholds tried per attempt (plus the last-round rise set)
constexpr int kCertTryRounds = 12;    // a candidate's launches and read-back, in rounds
constexpr int kCertEvery = 7;         // default rounds before the first proof attempt
// ... of a binned game, whose rounds all start from the round before's values and cost less: a
// first attempt after 7 or 8 rounds more often fails (with 9 the solve of 10^6 vertices of
// degree 2-12 took 979 us against 1323-1345, that of 1.6 10^6 of degree 3 4.9 ms against 6.4;
// where 8 is enough, 9 costs 1 to 6%)
constexpr int kCertEveryBinned = 9;
constexpr int kGraphSizes = 6;        // captured batches of 1, 2, 4, ..., 32 rounds
constexpr int kWholeDenseN = 1 << 16; // single launches sweep every round densely; above this size a run of
                                     // sparse rounds goes to the round kernels
constexpr int64_t kMemorySideCache = 256 << 20;
constexpr int kBinDensePart = 128;    // a binned round wants the transpose below 1/128 of the vertices
constexpr int kTailRounds = 4096;     // rounds of a one-workgroup launch at most (tens of milliseconds)
constexpr int kStopBatch = 4;         // rounds queued ahead of the host when a stop flag is polled

double egs_now_ms() {
    return 1e-6 * (double)std::chrono::duration_cast<std::chrono::nanoseconds>(
                      std::chrono::steady_clock::now().time_since_epoch()).count();
}

int pow2ceil(int x) {
    int p = 1;
    while (p < x) p <<= 1;
    return p;
}

// Byte offsets of every array in a solver's device workspace (one block), for games up to
// n_cap vertices and m_cap edges.  constexpr so that the size of the no-allocation
// workspace below is known at compile time.
struct Layout {
    size_t ptr, edges, cptr, cpred, cweight, val, stamp, l0, l1, dbig, dhuge, sbig, shuge, lcnt, mode, ring, rounds, misc,
        tile, fill, stats, statsum, sigma, h, hist, bfcnt, bits, hacc, hcnt, hbest, hflag, tcounts, toffs, tscan,
        titems, slen, sbase, sedges, bigmask, bedges, bcand, boff, bchunk, bdesc, whole, total;
    int64_t tcounts_cap, bin_cap, boff_cap;
    int sub_cap;
    bool phased, binned, weights;
};

constexpr size_t align256c(size_t x) { return (x + 255) & ~(size_t)255; }

// lean: without the arrays that only make rounds faster (the binned layout, the transpose's weights).
constexpr Layout make_layout(int32_t n_cap, int64_t m_cap, bool lean = false) {
    Layout L{};
    const size_t n1 = (size_t)n_cap + 1, m = (size_t)m_cap;
    const size_t tiles = (size_t)(n_cap + 4095) / 4096 + 1;
    const int64_t sc = (2 * (int64_t)n_cap + egs::kSub - 1) / egs::kSub;
    L.sub_cap = sc > 256 ? (int)sc : 256;
    const size_t list_ints = (size_t)egs::kSub * (size_t)L.sub_cap + n1;
    size_t off = 0;
    auto take = [&off](size_t bytes) {
        const size_t o = off;
        off += align256c(bytes);
        return o;
    };
    L.ptr = take(4 * n1);
    L.edges = take(8 * m);
    L.cptr = take(4 * n1);
    L.cpred = take(4 * m);
    L.val = take(4 * n1);
    L.stamp = take(4 * n1);
    L.l0 = take(4 * list_ints);
    L.l1 = take(4 * list_ints);
    L.dbig = take(4 * n1);
    L.dhuge = take(4 * n1);
    L.sbig = take(4 * n1);
    L.shuge = take(4 * n1);
    L.lcnt = take(4 * 3 * egs::kListCounters);
    L.mode = take(4 * 4);
    L.ring = take(4 * 16);
    L.rounds = take(4 * 16);
    L.misc = take(8 * 16);
    L.tile = take(4 * tiles);
    L.fill = take(4 * n1);
    L.stats = take(8 * 4 * (size_t)egs::kStatSlots);
    L.statsum = take(8 * 8);
    L.sigma = take(4 * n1);
    L.h = take(8 * n1);
    L.hist = take(4 * 256);
    L.bfcnt = take(4 * 64);
    L.bits = take(4 * 3 * (n1 / 32 + n1 / 1024 + 4));
    L.hacc = take(4 * n1);
    L.hcnt = take(4 * n1);
    L.hbest = take(8 * n1);
    L.hflag = take(4 * n1);
    // sorted transpose: per (edge tile, destination bucket) counts, bucket sizes and starts,
    // and the edges as (source, destination) items grouped by bucket
    const int64_t nb_cap = std::min<int64_t>(4096, ((int64_t)n_cap + 2047) / 2048);
    L.tcounts_cap = ((m_cap + egs::kTrTileEdges - 1) / egs::kTrTileEdges) * nb_cap;
    L.tcounts = take(4 * ((size_t)L.tcounts_cap + 1));
    L.toffs = take(4 * ((size_t)L.tcounts_cap + 1));
    L.tscan = take(4 * ((size_t)L.tcounts_cap / 4096 + 2));
    L.titems = take(8 * m);
    // phased dense rounds (large games): per tile and slice the vertices' edge counts (a
    // byte each) and the wave bases, and the edges in (tile, slice, vertex) order
    L.phased = n_cap >= egs::kPhaseMinN;
    const size_t ptiles = (size_t)n_cap / egs::kSliceTile + 1;
    L.slen = L.phased ? take(ptiles * egs::kMaxPhases * egs::kSliceTile) : 0;
    L.sbase = L.phased ? take(4 * ptiles * egs::kMaxPhases * egs::kSliceWaves) : 0;
    L.sedges = L.phased ? take(8 * m) : 0;
    // binned dense rounds: words, vertex numbers and candidates of the padded edges, in whole
    // cache lines (the vertex numbers follow the words and are read four at a time) and with
    // room for a step past the last index in 31 bits
    L.binned = n_cap >= egs::kBinMinN && !lean;
    L.bin_cap = L.binned ? m_cap + m_cap / 2 + (1 << 20) : 0;
    if (L.bin_cap > 0x7fff0000) L.bin_cap = 0x7fff0000;
    L.bin_cap &= ~(int64_t)63;
    L.bedges = L.binned ? take(6 * (size_t)L.bin_cap + 256) : 0;
    L.bcand = L.binned ? take(8 * (size_t)L.bin_cap) : 0;
    L.weights = !lean;
    L.cweight = L.binned ? L.bcand : L.weights ? take(4 * m) : 0;   // a game leaves the bins with its transpose
    const size_t chunks = ((size_t)egs::kBinHead * n1 + m) / egs::kBinShareMin + 2;
    L.boff_cap = L.binned ? (int64_t)((size_t)L.bin_cap / egs::kBinPad + chunks) : 0;
    L.boff = L.binned ? take(4 * (size_t)L.boff_cap) : 0;
    L.bchunk = L.binned ? take(8 * (chunks + 1)) : 0;
    L.bdesc = L.binned ? take(16 * chunks) : 0;
    L.bigmask = L.phased ? take(8 * ((size_t)n_cap / 64 + 2)) : 0;
    L.whole = take(sizeof(egs::WholeCtl));
    L.total = off;
    return L;
}
static_assert(make_layout(egs::kBinMinN, 2000001).bin_cap % 64 == 0 && make_layout(1 << 23, 0x7fffffff).bin_cap % 64 == 0,
              "vertex numbers behind the words are aligned at every capacity");

}  // namespace

struct egs_solver {
    int device = 0;
    int cus = 0;                      // compute units of the device
    hipStream_t stream = nullptr;
    bool csc_built = false;           // the transpose exists for the loaded game (ring[12] raised)
    int32_t n_cap = 0;
    int64_t m_cap = 0;
    void *block = nullptr;
    size_t block_bytes = 0;
    int *d_ptr = nullptr, *d_cptr = nullptr, *d_cpred = nullptr, *d_cweight = nullptr, *d_val = nullptr;
    int *d_stamp = nullptr, *d_list[2] = {nullptr, nullptr}, *d_dbig = nullptr, *d_dhuge = nullptr;
    int *d_sbig = nullptr, *d_shuge = nullptr, *d_lcnt = nullptr, *d_mode = nullptr;
    int *d_ring = nullptr, *d_rounds = nullptr, *d_misc = nullptr, *d_tile = nullptr, *d_fill = nullptr;
    int sub_cap = 0;
    int *d_sigma = nullptr, *d_hist = nullptr, *d_bfcnt = nullptr;   // d_sigma: rise stamps
    unsigned *d_bits = nullptr;     // three bitmaps of raised potentials (proof passes)
    int *d_hacc = nullptr, *d_hcnt = nullptr;   // shared lifts of the vertices above huge_deg
    long long *d_hbest = nullptr;               // shared proof passes of the same vertices
    int *d_hflag = nullptr;
    int *d_tcounts = nullptr, *d_toffs = nullptr, *d_tscan = nullptr;   // sorted transpose
    int2 *d_titems = nullptr;
    int64_t tcounts_cap = 0;
    uint8_t *d_slen = nullptr;                  // phased dense rounds (large n_cap)
    int *d_sbase = nullptr;
    int2 *d_sedges = nullptr;
    unsigned long long *d_bigmask = nullptr;
    uint32_t *d_bedges = nullptr;               // binned dense rounds (large n_cap)
    int *d_bcand = nullptr, *d_boff = nullptr, *d_bchunk = nullptr;
    int4 *d_bdesc = nullptr;
    int64_t bin_cap = 0, boff_cap = 0;          // padded edges and run starts there is room for
    bool bins_open = false;                     // the binned layout of this prepare is still to be built
    long long *d_h = nullptr;
    egs::WholeCtl *d_whole = nullptr;
    egs::WholePlan whole{};           // nb > 0: iterate() runs the game in single launches (egs_whole.hip)
    unsigned load_seq = 0;            // loads whose record was asked for
    unsigned whole_seq = 0;           // launches so far
    int whole_max_nb = 0;             // workgroups of such a launch at most
    int64_t whole_wait = egs::kWholeWait;
    int64_t whole_rounds = 0;         // rounds of the run they have done
    bool whole_gave_up = false;       // the last of them gave up: the values are past those rounds
    egs_stats whole_st{};             // what those rounds counted
    int wmax = 0;
    int cert_every = 32, cert_gap = 32, cert_max_passes = 1024;
    int cert_cap = 64;        // longest-path passes per candidate; doubles while attempts run out of passes
    int cert_pass_hint = 0;   // passes the run's last converged candidate needed
    int64_t next_cert = 0;
    int2 *d_edges = nullptr;
    unsigned long long *d_stats = nullptr, *d_statsum = nullptr;
    int *h_probe = nullptr;   // pinned: per-batch counter probes + misc readbacks
    char *h_small = nullptr;  // behind them, out_small bytes for small read-backs
    size_t out_small = 0;
    char *h_out = nullptr;    // pinned, 2 x out_half bytes, made at the first larger read-back
    size_t out_half = 0;
    bool mirrored = false;    // h_small holds the values of the run that has just converged
    bool values_set = false;  // the run's values were replaced (egs_solver_set_values)
    bool values_out = false;  // their device address was handed out: read-backs go to the device
    int probe_want[2] = {kProbeWant, kProbeWant};   // where each probe slot holds ring[13]
    hipEvent_t ev_probe[2] = {nullptr, nullptr};
    hipEvent_t ev_a = nullptr, ev_b = nullptr;
    hipEvent_t ev_pa = nullptr, ev_pb = nullptr;   // prepare's span, read after a later wait
    bool prep_open = false;   // prepare's time and initial frontier not read yet

    egs::DevGame g{};
    egs::LaunchShape sh{};
    // batches of 2^k rounds (k < kGraphSizes) captured once per prepare and replayed
    hipGraphExec_t graph[kGraphSizes] = {};
    egs::DevGame graph_g{};           // the game and shape the graphs were captured with
    egs::LaunchShape graph_sh{};
    bool use_graphs = false;
    bool no_alloc = false;            // the no-allocation entry point's solver: never graphs
    bool loaded = false, prepared = false;
    int max_outdeg = 0;
    int64_t next_round = 1;
    int64_t phase_cap = 0;
    bool capped = false;              // by the options, not by the reference's bound
    int batch_rounds = 32;
    const volatile uint32_t *stop_flag = nullptr;
    egs_stats st{};
};

// Point the solver's arrays into a workspace laid out by make_layout.
static void bind_layout(egs_solver *s, char *b, const Layout &L) {
    s->sub_cap = L.sub_cap;
    s->d_ptr = (int *)(b + L.ptr);
    s->d_edges = (int2 *)(b + L.edges);
    s->d_cptr = (int *)(b + L.cptr);
    s->d_cpred = (int *)(b + L.cpred);
    s->d_cweight = L.weights ? (int *)(b + L.cweight) : nullptr;
    s->d_val = (int *)(b + L.val);
    s->d_stamp = (int *)(b + L.stamp);
    s->d_list[0] = (int *)(b + L.l0);
    s->d_list[1] = (int *)(b + L.l1);
    s->d_dbig = (int *)(b + L.dbig);
    s->d_dhuge = (int *)(b + L.dhuge);
    s->d_sbig = (int *)(b + L.sbig);
    s->d_shuge = (int *)(b + L.shuge);
    s->d_lcnt = (int *)(b + L.lcnt);
    s->d_mode = (int *)(b + L.mode);
    s->d_ring = (int *)(b + L.ring);
    s->d_rounds = (int *)(b + L.rounds);
    s->d_misc = (int *)(b + L.misc);
    s->d_tile = (int *)(b + L.tile);
    s->d_fill = (int *)(b + L.fill);
    s->d_stats = (unsigned long long *)(b + L.stats);
    s->d_statsum = (unsigned long long *)(b + L.statsum);
    s->d_sigma = (int *)(b + L.sigma);
    s->d_h = (long long *)(b + L.h);
    s->d_hist = (int *)(b + L.hist);
    s->d_bfcnt = (int *)(b + L.bfcnt);
    s->d_bits = (unsigned *)(b + L.bits);
    s->d_hacc = (int *)(b + L.hacc);
    s->d_hcnt = (int *)(b + L.hcnt);
    s->d_hbest = (long long *)(b + L.hbest);
    s->d_hflag = (int *)(b + L.hflag);
    s->d_tcounts = (int *)(b + L.tcounts);
    s->d_toffs = (int *)(b + L.toffs);
    s->d_tscan = (int *)(b + L.tscan);
    s->d_titems = (int2 *)(b + L.titems);
    s->tcounts_cap = L.tcounts_cap;
    s->d_whole = (egs::WholeCtl *)(b + L.whole);
    if (L.binned) {
        s->d_bedges = (uint32_t *)(b + L.bedges);
        s->d_bcand = (int *)(b + L.bcand);
        s->bin_cap = L.bin_cap;
        s->boff_cap = L.boff_cap;
        s->d_boff = (int *)(b + L.boff);
        s->d_bchunk = (int *)(b + L.bchunk);
        s->d_bdesc = (int4 *)(b + L.bdesc);
    }
    if (L.phased) {
        s->d_slen = (uint8_t *)(b + L.slen);
        s->d_sbase = (int *)(b + L.sbase);
        s->d_sedges = (int2 *)(b + L.sedges);
        s->d_bigmask = (unsigned long long *)(b + L.bigmask);
    }
}

// Timing and probes use events when the solver owns them; a solver without events (the
// no-allocation entry point) times on the host and waits on the whole stream instead.
static hipError_t mark_start(egs_solver *s, double *host_t0) {
    if (s->ev_a) return hipEventRecord(s->ev_a, s->stream);
    *host_t0 = egs_now_ms();
    return hipSuccess;
}
static hipError_t mark_stop(egs_solver *s, double host_t0, float *ms) {
    if (s->ev_b) {
        hipError_t e = hipEventRecord(s->ev_b, s->stream);
        if (e == hipSuccess) e = hipEventSynchronize(s->ev_b);
        if (e == hipSuccess) e = hipEventElapsedTime(ms, s->ev_a, s->ev_b);
        return e;
    }
    hipError_t e = hipStreamSynchronize(s->stream);
    *ms = (float)(egs_now_ms() - host_t0);
    return e;
}
static hipError_t probe_mark(egs_solver *s, int slot) {
    return s->ev_probe[slot] ? hipEventRecord(s->ev_probe[slot], s->stream) : hipSuccess;
}
static hipError_t probe_wait(egs_solver *s, int slot) {
    return s->ev_probe[slot] ? hipEventSynchronize(s->ev_probe[slot]) : hipStreamSynchronize(s->stream);
}

// Wait for the word `done`, stored last by queued work that ends, to become seq: a spin on the
// pinned word that asks the stream now and then, so that work that ended without storing it is
// noticed (false).  On return the work's stores to pinned memory are visible.
static hipError_t wait_word(egs_solver *s, const unsigned *done, unsigned seq, bool *got) {
    hipError_t q = hipErrorNotReady;
    for (;;) {
        for (int k = 0; k < 4096 && __atomic_load_n(done, __ATOMIC_ACQUIRE) != seq; k++) __builtin_ia32_pause();
        *got = __atomic_load_n(done, __ATOMIC_ACQUIRE) == seq;
        if (*got) return hipSuccess;
        if (q != hipErrorNotReady) return q;         // the stream was done before this last look
        q = hipStreamQuery(s->stream);
    }
}

// `bytes` of device memory to a pageable host buffer, after the work queued so far.  A copy
// into pageable memory runs at 2-4 GB/s up to about 1 MB and 16 GB/s beyond (350 KB took
// 154 us, 16 MB 1.02 ms); into pinned memory it takes 14 us and 0.30 ms.  So it goes through
// pinned memory: the small area made with the solver, or two halves of a buffer made at the
// first larger read, one filling while the other is copied out by the packing threads.
constexpr size_t kOutSmall = 128 << 10;    // the small area at most
constexpr size_t kOutHalf = 1 << 20;       // a half of the large buffer at most
static hipError_t read_back(egs_solver *s, void *dst, const void *src, size_t bytes) {
    hipError_t e;
    if (bytes <= s->out_small) {
        e = hipMemcpyAsync(s->h_small, src, bytes, hipMemcpyDeviceToHost, s->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
        if (e == hipSuccess) memcpy(dst, s->h_small, bytes);
        return e;
    }
    const size_t half = std::min(bytes, kOutHalf);
    if (!s->no_alloc && s->out_half < half) {
        if (s->h_out) (void)hipHostFree(s->h_out);
        s->h_out = nullptr;
        s->out_half = 0;
        if (hipHostMalloc((void **)&s->h_out, 2 * half, hipHostMallocDefault) == hipSuccess) s->out_half = half;
        else (void)hipGetLastError();      // the plain copy below needs no buffer
    }
    if (s->out_half < half) {
        e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s->stream);
        return e == hipSuccess ? hipStreamSynchronize(s->stream) : e;
    }
    const int64_t chunks = (int64_t)((bytes + half - 1) / half);
    auto len = [&](int64_t c) { return std::min(half, bytes - (size_t)c * half); };
    for (int64_t c = 0; c <= chunks; c++) {
        if (c > 0) {                       // chunk c - 1 has arrived before chunk c is queued behind it
            e = hipStreamSynchronize(s->stream);
            if (e != hipSuccess) return e;
        }
        if (c < chunks) {
            e = hipMemcpyAsync(s->h_out + (size_t)(c & 1) * half, (const char *)src + (size_t)c * half, len(c),
                               hipMemcpyDeviceToHost, s->stream);
            if (e != hipSuccess) return e;
        }
        if (c > 0) egs_pk_copy((char *)dst + (size_t)(c - 1) * half, s->h_out + (size_t)((c - 1) & 1) * half, len(c - 1));
    }
    return hipSuccess;
}

// The record of a load (launch_load_finish last on the stream), on the host.  The no-allocation
// solver has no pinned block and copies it from device memory.
static hipError_t read_load(egs_solver *s, const egs::LoadPartial *part, int nparts, const int *n0, const int *bad,
                            egs::LoadResult **out) {
    egs::LoadResult *res = (egs::LoadResult *)(s->h_probe + kPinLoad);
    *out = res;
    const unsigned seq = ++s->load_seq;
    __atomic_store_n(&res->done, 0u, __ATOMIC_RELEASE);
    egs::LoadResult *to = s->no_alloc ? (egs::LoadResult *)s->d_misc : res;
    hipError_t e = egs::launch_load_finish(part, nparts, n0, bad, seq, to, s->stream);
    if (e != hipSuccess) return e;
    if (s->no_alloc) {
        e = hipMemcpyAsync(res, to, sizeof(*res), hipMemcpyDeviceToHost, s->stream);
        return e == hipSuccess ? hipStreamSynchronize(s->stream) : e;
    }
    bool got = false;
    e = wait_word(s, &res->done, seq, &got);
    return got ? hipSuccess : e != hipSuccess ? e : hipErrorUnknown;
}

// Items in a list from its counters (sub-queues clamp at sub_cap; the rest overflowed).
static int64_t list_total(const egs_solver *s, const int *c) {
    int64_t t = 0;
    for (int k = 0; k < egs::kSub; k++) t += std::min(c[k], s->sub_cap);
    return t + c[egs::kSub];
}

// prepare's time and initial frontier size, once its closing event has passed
static hipError_t close_prepare(egs_solver *s) {
    if (!s->prep_open) return hipSuccess;
    float ms = 0.f;
    hipError_t e = hipEventSynchronize(s->ev_pb);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, s->ev_pa, s->ev_pb);
    if (e != hipSuccess) return e;
    s->st.ms_prepare = ms;
    s->st.initial_active = (int32_t)list_total(s, s->h_probe + kPinInit);
    s->prep_open = false;
    return hipSuccess;
}

static void drop_graphs(egs_solver *s) {
    for (auto &x : s->graph)
        if (x) {
            (void)hipGraphExecDestroy(x);
            x = nullptr;
        }
}

// One batch of `rounds` rounds (k_advance last) on the solver stream.
static hipError_t launch_batch(egs_solver *s, int rounds) {
    for (int j = 0; j < rounds; j++) {
        hipError_t e = egs::launch_round(s->g, s->sh, j, s->stream);
        if (e != hipSuccess) return e;
    }
    return egs::launch_advance(s->g, rounds, s->stream);
}

// The same batch as a graph of 2^k rounds, captured on first use after a prepare.
static hipError_t replay_batch(egs_solver *s, int k) {
    if (!s->graph[k]) {
        hipGraph_t gr = nullptr;
        hipError_t e = hipStreamBeginCapture(s->stream, hipStreamCaptureModeThreadLocal);
        if (e != hipSuccess) return e;
        const hipError_t le = launch_batch(s, 1 << k);
        e = hipStreamEndCapture(s->stream, &gr);
        if (le != hipSuccess) e = le;
        if (e == hipSuccess) e = hipGraphInstantiate(&s->graph[k], gr, nullptr, nullptr, 0);
        if (gr) (void)hipGraphDestroy(gr);
        if (e != hipSuccess) {
            s->graph[k] = nullptr;
            return e;
        }
    }
    return hipGraphLaunch(s->graph[k], s->stream);
}

egs::DeviceUnits &egs::device_units(int device) {
    static DeviceUnits units[64];
    return units[(unsigned)device % 64];
}

// The large-route workers of a server share the compute units a slice leaves free.
void egs::solver_limit_whole(egs_solver *s, int max_nb) { s->whole_max_nb = std::min(s->cus, max_nb); }

extern "C" {

const char *egs_last_error(void) { return g_err; }

void egs_solver_whole_wait(egs_solver *s, int64_t us) { s->whole_wait = us * 100; }

int egs_device_query(int device, egs_device_info *out) {
    if (!out) return fail(EGS_E_ARG, "egs_device_query: null output");
    memset(out, 0, sizeof(*out));
    int count = 0;
    HIP_TRY(hipGetDeviceCount(&count));
    out->device_count = count;
    if (device < 0 || device >= count)
        return fail(EGS_E_ARG, "device %d not available (%d devices)", device, count);
    hipDeviceProp_t p;
    HIP_TRY(hipGetDeviceProperties(&p, device));
    snprintf(out->name, sizeof(out->name), "%s", p.name);
    snprintf(out->arch, sizeof(out->arch), "%s", p.gcnArchName);
    out->warp_size = p.warpSize;
    out->max_threads_per_block = p.maxThreadsPerBlock;
    out->multiprocessors = p.multiProcessorCount;
    out->total_mem = (int64_t)p.totalGlobalMem;
    out->shared_mem_per_block = (int64_t)p.sharedMemPerBlock;
    out->clock_khz = p.clockRate;
    out->ecc = p.ECCEnabled;
    int dv = 0, rv = 0;
    HIP_TRY(hipDriverGetVersion(&dv));
    HIP_TRY(hipRuntimeGetVersion(&rv));
    out->driver_version = dv;
    out->runtime_version = rv;
    out->cap_major = p.major;
    out->cap_minor = p.minor;
    return EGS_OK;
}

int egs_host_alloc(void **p, size_t bytes) {
    if (!p) return fail(EGS_E_ARG, "egs_host_alloc: null output");
    *p = nullptr;
    if (hipHostMalloc(p, bytes ? bytes : 1, hipHostMallocDefault) != hipSuccess)
        return fail(EGS_E_NOMEM, "hipHostMalloc of %zu bytes failed", bytes);
    return EGS_OK;
}

int egs_host_free(void *p) {
    if (p) HIP_TRY(hipHostFree(p));
    return EGS_OK;
}

int egs_runtime_error(char *buf, int len) {
    hipError_t e = hipGetLastError();
    if (buf && len > 0) snprintf(buf, (size_t)len, "%s", e == hipSuccess ? "" : hipGetErrorString(e));
    return (int)e;
}

int egs_device_reset(int device) {
    HIP_TRY(hipSetDevice(device));
    HIP_TRY(hipDeviceReset());
    return EGS_OK;
}

int egs_solver_destroy(egs_solver *s) {
    if (!s) return EGS_OK;
    (void)hipSetDevice(s->device);
    if (s->stream) (void)hipStreamSynchronize(s->stream);
    drop_graphs(s);
    if (s->block) (void)hipFree(s->block);
    if (s->h_probe) (void)hipHostFree(s->h_probe);
    if (s->h_out) (void)hipHostFree(s->h_out);
    for (auto &e : s->ev_probe) if (e) (void)hipEventDestroy(e);
    if (s->ev_a) (void)hipEventDestroy(s->ev_a);
    if (s->ev_b) (void)hipEventDestroy(s->ev_b);
    if (s->ev_pa) (void)hipEventDestroy(s->ev_pa);
    if (s->ev_pb) (void)hipEventDestroy(s->ev_pb);
    if (s->stream) (void)hipStreamDestroy(s->stream);
    delete s;
    return EGS_OK;
}

int egs_solver_create(int device, int32_t n_cap, int64_t m_cap, egs_solver **out) {
    if (!out) return fail(EGS_E_ARG, "egs_solver_create: null output");
    *out = nullptr;
    if (n_cap < 1 || m_cap < 1 || m_cap > 0x7fffffffLL)
        return fail(EGS_E_ARG, "egs_solver_create: need 1 <= n_cap and 1 <= m_cap < 2^31 (got %d, %lld)",
                    n_cap, (long long)m_cap);
    int rc = check_gfx950(device);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(device));
    egs_solver *s = new egs_solver();
    s->device = device;
    if (hipDeviceGetAttribute(&s->cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) s->cus = 256;
    s->whole_max_nb = s->cus;
    s->n_cap = n_cap;
    s->m_cap = m_cap;
    Layout L = make_layout(n_cap, m_cap);
    if (hipMalloc(&s->block, L.total) != hipSuccess) {
        // 28 bytes an edge where there is no room for 49 (32 below kBinMinN vertices)
        (void)hipGetLastError();
        L = make_layout(n_cap, m_cap, true);
        s->block = nullptr;
    }
    s->block_bytes = L.total;
    if (!s->block && hipMalloc(&s->block, L.total) != hipSuccess) {
        egs_solver_destroy(s);
        return fail(EGS_E_NOMEM, "hipMalloc of %zu bytes failed", L.total);
    }
    bind_layout(s, (char *)s->block, L);
    constexpr size_t kProbeBytes = 4 * (kPinProbe + 2 * kProbeStride);
    s->out_small = std::min(kOutSmall, 4 * ((size_t)n_cap + 32));
    if (hipHostMalloc((void **)&s->h_probe, kProbeBytes + s->out_small, hipHostMallocDefault) != hipSuccess) {
        egs_solver_destroy(s);
        return fail(EGS_E_NOMEM, "hipHostMalloc failed");
    }
    s->h_small = (char *)s->h_probe + kProbeBytes;
    s->h_probe[kPinOne] = 1;
    if (hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&s->ev_probe[0]) != hipSuccess || hipEventCreate(&s->ev_probe[1]) != hipSuccess ||
        hipEventCreate(&s->ev_a) != hipSuccess || hipEventCreate(&s->ev_b) != hipSuccess ||
        hipEventCreate(&s->ev_pa) != hipSuccess || hipEventCreate(&s->ev_pb) != hipSuccess) {
        egs_solver_destroy(s);
        return fail(EGS_E_HIP, "stream/event creation failed");
    }
    *out = s;
    return EGS_OK;
}

static void bind_game(egs_solver *s, int32_t n, int32_t n0, int64_t m, int32_t mg);

int egs_solver_load(egs_solver *s, int mem, int32_t n, int32_t n0, int64_t m, int32_t mg,
                    const int32_t *ptr, const int32_t *succ, const int32_t *w) {
    if (!s) return fail(EGS_E_ARG, "null solver");
    if (n < 1 || n0 < 0 || n0 > n || m < 1 || mg < 0 || !ptr || !succ || !w)
        return fail(EGS_E_ARG, "egs_solver_load: bad game (n=%d n0=%d m=%lld mg=%d)", n, n0,
                    (long long)m, mg);
    if (n > s->n_cap || m > s->m_cap)
        return fail(EGS_E_CAPACITY, "game (n=%d, m=%lld) exceeds solver capacity (%d, %lld)", n,
                    (long long)m, s->n_cap, (long long)s->m_cap);
    HIP_TRY(hipSetDevice(s->device));
    if (mem == EGS_MEM_HOST) {
        // validate the CSR on the host (fused with the int2 packing) before anything reaches
        // the device
        int2 *packed = (int2 *)malloc(sizeof(int2) * (size_t)m);
        if (!packed) return fail(EGS_E_NOMEM, "host staging allocation failed");
        int32_t wm = 0, mx = 0;
        int64_t bad = -1;
        const int chk = egs_pk_check_pack64(n, m, ptr, succ, w, (int32_t *)packed, &wm, &mx, &bad);
        if (chk) free(packed);
        switch (chk) {
        case EGS_PK_BAD_OFFSETS:
            return fail(EGS_E_ARG, "CSR offsets must run from 0 to m (got %d..%d)", ptr[0], ptr[n]);
        case EGS_PK_NO_EDGE: return fail(EGS_E_ARG, "vertex %lld has no out-edge", (long long)bad);
        case EGS_PK_BAD_SUCC:
            return fail(EGS_E_ARG, "edge %lld: successor %d out of range", (long long)bad, succ[bad]);
        default: break;
        }
        s->max_outdeg = mx;
        s->wmax = wm;
        // what a prepare of the game before has queued still reads the arrays
        const hipError_t e0 = hipStreamSynchronize(s->stream);
        hipError_t e1 = e0 != hipSuccess ? e0 : hipMemcpy(s->d_ptr, ptr, sizeof(int) * ((size_t)n + 1), hipMemcpyHostToDevice);
        hipError_t e2 = e1 != hipSuccess ? e1 : hipMemcpy(s->d_edges, packed, sizeof(int2) * (size_t)m, hipMemcpyHostToDevice);
        free(packed);
        HIP_TRY(e1);
        HIP_TRY(e2);
    } else if (mem == EGS_MEM_DEVICE) {
        // device inputs are trusted to be a valid CSR of this shape (the caller owns them)
        egs::LoadPartial *part = (egs::LoadPartial *)s->d_stats;     // prepare clears it later
        egs::LoadResult *res;
        int nparts = 0;
        HIP_TRY(egs::launch_load_device(ptr, succ, w, n, m, s->d_ptr, s->d_edges, part, &nparts, s->stream));
        HIP_TRY(read_load(s, part, nparts, nullptr, nullptr, &res));
        s->max_outdeg = res->dmax;
        s->wmax = res->wmax;
    } else {
        return fail(EGS_E_ARG, "mem must be EGS_MEM_HOST or EGS_MEM_DEVICE");
    }
    bind_game(s, n, n0, m, mg);
    return EGS_OK;
}

int egs_solver_load_packed(egs_solver *s, int32_t n, int32_t n0, int64_t m, int32_t mg, const int32_t *d_ptr,
                           const uint32_t *d_edges, int32_t shift, int32_t wmax, int32_t max_outdeg) {
    if (!s) return fail(EGS_E_ARG, "null solver");
    if (n < 1 || n0 < 0 || n0 > n || m < 1 || mg < 0 || !d_ptr || !d_edges || shift < 1 || shift > 30 || wmax < 0 ||
        max_outdeg < 1)
        return fail(EGS_E_ARG, "egs_solver_load_packed: bad game (n=%d n0=%d m=%lld mg=%d shift=%d)", n, n0,
                    (long long)m, mg, shift);
    if (n > s->n_cap || m > s->m_cap)
        return fail(EGS_E_CAPACITY, "game (n=%d, m=%lld) exceeds solver capacity (%d, %lld)", n,
                    (long long)m, s->n_cap, (long long)s->m_cap);
    HIP_TRY(hipSetDevice(s->device));
    // device inputs are trusted to be a checked CSR of this shape (the caller owns them)
    HIP_TRY(hipMemcpyAsync(s->d_ptr, d_ptr, sizeof(int) * ((size_t)n + 1), hipMemcpyDeviceToDevice, s->stream));
    HIP_TRY(egs::launch_unpack(d_edges, shift, s->d_edges, m, s->stream));
    s->max_outdeg = max_outdeg;
    s->wmax = wmax;
    bind_game(s, n, n0, m, mg);
    return EGS_OK;
}

int egs_solver_load_read_order(egs_solver *s, int mem, int32_t n, int64_t m, const uint8_t *owner,
                               const int32_t *rptr, const int32_t *rsucc, const int32_t *rw, int32_t *n0_out,
                               int32_t *mg_out, int32_t *ext_of_int) {
    if (!s) return fail(EGS_E_ARG, "null solver");
    if (n < 1 || m < 1 || !owner || !rptr || !rsucc || !rw || (mem != EGS_MEM_HOST && mem != EGS_MEM_DEVICE))
        return fail(EGS_E_ARG, "egs_solver_load_read_order: bad game (n=%d m=%lld)", n, (long long)m);
    if (n > s->n_cap || m > s->m_cap)
        return fail(EGS_E_CAPACITY, "game (n=%d, m=%lld) exceeds solver capacity (%d, %lld)", n, (long long)m,
                    s->n_cap, (long long)s->m_cap);
    HIP_TRY(hipSetDevice(s->device));
    egs::ReadOrderBuffers b{};
    if (mem == EGS_MEM_HOST) {
        // one upload into work space that prepare and the rounds rewrite later
        uint8_t *d_owner = (uint8_t *)s->d_stamp;
        int *d_rsucc = (int *)s->d_titems, *d_rw = (int *)s->d_titems + m;
        HIP_TRY(hipMemcpyAsync(d_owner, owner, (size_t)n, hipMemcpyHostToDevice, s->stream));
        HIP_TRY(hipMemcpyAsync(s->d_cptr, rptr, sizeof(int) * ((size_t)n + 1), hipMemcpyHostToDevice, s->stream));
        HIP_TRY(hipMemcpyAsync(d_rsucc, rsucc, sizeof(int) * (size_t)m, hipMemcpyHostToDevice, s->stream));
        HIP_TRY(hipMemcpyAsync(d_rw, rw, sizeof(int) * (size_t)m, hipMemcpyHostToDevice, s->stream));
        b.owner = d_owner;
        b.rptr = s->d_cptr;
        b.rsucc = d_rsucc;
        b.rw = d_rw;
    } else {
        b.owner = owner;
        b.rptr = rptr;
        b.rsucc = rsucc;
        b.rw = rw;
    }
    // the check's verdict stays on the device: the kernels after it return at once on a bad
    // game, and the host reads it with the result
    int *d_bad = s->d_misc + 24;
    HIP_TRY(egs::launch_read_order_check(b.rptr, b.rsucc, n, m, d_bad, s->stream));
    b.flag0 = s->d_sigma;
    b.pre0 = s->d_fill;
    b.rev = s->d_dbig;
    b.ext_of_int = s->d_sbig;
    b.deg = s->d_dhuge;
    b.scan_tiles = s->d_tile;
    egs::LoadPartial *part = nullptr;
    egs::LoadResult *res;
    int nparts = 0;
    HIP_TRY(egs::launch_internalise(b, n, d_bad, s->d_ptr, s->d_edges, &part, &nparts, s->stream));
    HIP_TRY(read_load(s, part, nparts, s->d_fill + n, d_bad, &res));
    if (res->bad & 1) return fail(EGS_E_ARG, "read-order offsets must run from 0 to m");
    if (res->bad & 2) return fail(EGS_E_ARG, "a vertex has no out-edge");
    if (res->bad & 4) return fail(EGS_E_ARG, "a successor is out of range");
    if (res->mg > 0x7fffffffULL) return fail(EGS_E_ARG, "Error too high weights --> overflow (MG past INT32_MAX)");
    if (ext_of_int) {
        s->mirrored = false;
        HIP_TRY(read_back(s, ext_of_int, s->d_sbig, sizeof(int) * (size_t)n));
    }
    const int32_t n0 = res->n0, mg = (int32_t)res->mg;
    s->max_outdeg = res->dmax;
    s->wmax = res->wmax;
    bind_game(s, n, n0, m, mg);
    if (n0_out) *n0_out = n0;
    if (mg_out) *mg_out = mg;
    return EGS_OK;
}

int egs_solver_read_game(egs_solver *s, int32_t *ptr, int32_t *succ, int32_t *w) {
    if (!s || !s->loaded || !ptr || !succ || !w) return fail(EGS_E_STATE, "egs_solver_read_game: nothing loaded");
    HIP_TRY(hipSetDevice(s->device));
    const int64_t m = s->g.m;
    int2 *tmp = (int2 *)malloc(sizeof(int2) * (size_t)m);
    if (!tmp) return fail(EGS_E_NOMEM, "host buffer of %lld edges", (long long)m);
    hipError_t e1 = hipMemcpyAsync(ptr, s->d_ptr, sizeof(int) * ((size_t)s->g.n + 1), hipMemcpyDeviceToHost, s->stream);
    hipError_t e2 = hipMemcpyAsync(tmp, s->d_edges, sizeof(int2) * (size_t)m, hipMemcpyDeviceToHost, s->stream);
    hipError_t e3 = hipStreamSynchronize(s->stream);
    if (e1 == hipSuccess && e2 == hipSuccess && e3 == hipSuccess)
        for (int64_t k = 0; k < m; k++) {
            succ[k] = tmp[k].x;
            w[k] = tmp[k].y;
        }
    free(tmp);
    HIP_TRY(e1);
    HIP_TRY(e2);
    HIP_TRY(e3);
    return EGS_OK;
}

// Point the device-game view at the solver's arrays for a freshly loaded game.
static void bind_game(egs_solver *s, int32_t n, int32_t n0, int64_t m, int32_t mg) {
    egs::DevGame &g = s->g;
    g.n = n;
    g.n0 = n0;
    g.mg = mg;
    g.m = m;
    g.ptr = s->d_ptr;
    g.edges = s->d_edges;
    g.cptr = s->d_cptr;
    g.cpred = s->d_cpred;
    g.val = s->d_val;
    g.stamp = s->d_stamp;
    g.list[0] = s->d_list[0];
    g.list[1] = s->d_list[1];
    g.sub_cap = s->sub_cap;
    g.lcnt = s->d_lcnt;
    g.mode = s->d_mode;
    g.dbig = s->d_dbig;
    g.dhuge = s->d_dhuge;
    g.sbig = s->d_sbig;
    g.shuge = s->d_shuge;
    g.ring = s->d_ring;
    g.stats = s->d_stats;
    g.rounds_done = s->d_rounds;
    s->loaded = true;
    s->prepared = false;
    s->whole = egs::WholePlan{};
    s->mirrored = false;
    s->bins_open = false;
}

// Binned dense rounds (egs_bins.h) where the packed word holds the weights, the options leave
// the dense rounds' form open, and they win: a binned round starts from the round before's
// values only, so it needs a quarter more rounds than sweeps in place, and two launches.  Solves,
// binned against sweeps (phases above 2^20 vertices): 741 us against 810 at 400,003 vertices of
// degree 2-16, 1360 against 1677 at 10^6 of degree 3-6, 2.9 ms against 3.7 at 3 10^6 of degree
// 3-6, 5.5 against 10.8 at 4 10^6 of degree 2-5; skewed degrees 4.8 ms against 5.9 at 450,003
// and 13.6 against 20.0 at 10^6 of average degree 2.2.  Low even degrees lose (5.2 ms against
// 4.0 at 2 10^6 of degree 2-5, 6.4 against 4.1 at 1.6 10^6 of degree 3, 9.9 against 8.3 at
// 4 10^6 of degree 3): their long runs of sparse rounds need the transpose sooner.
static bool bins_pay(const egs_solver *s) {
    const egs::DevGame &g = s->g;
    if (g.n < egs::kBinMinN) return false;
    if (s->max_outdeg > g.big_deg) return true;
    return g.n <= egs::kBinHalfN ? g.m >= 4 * (int64_t)g.n : 2 * g.m >= 7 * (int64_t)g.n;
}

// whole: the game runs in single launches, which need none of this; what takes such a run over
// (leave_whole) finds no layout built for it, so it gets sweeps.
static void pick_bins(egs_solver *s, const egs_options *o, bool whole) {
    egs::DevGame &g = s->g;
    g.cweight = nullptr;
    g.bins = 0;
    g.bin_w = g.bin_parts = g.nchunks = g.bin_share = 0;
    g.bin_magic = 0;
    g.bin_once = 0;
    g.bedges = s->d_bedges;
    g.bids = (uint16_t *)(s->d_bedges + s->bin_cap);
    g.cand = s->d_bcand;
    g.boff = s->d_boff;
    g.bchunk = s->d_bchunk;
    g.bdesc = s->d_bdesc;
    g.hubs = s->max_outdeg > g.huge_deg;
    if (whole || o->graphs > 0 || o->slices != 0 || !s->d_boff || !bins_pay(s) || g.dense_min > g.n || s->wmax > egs::kBinWmax ||
        (int64_t)g.mg + 2 * (int64_t)s->wmax >= EGS_TOP || g.n > (int64_t)egs::kBinMax * egs::kBinSlice)
        return;
    // slices and parts that fill the device evenly: 512 workgroups with half slices (two to a
    // compute unit), else 256
    const bool half = g.n <= egs::kBinHalfN;
    const int wide = half ? egs::kBinSlice / 2 : egs::kBinSlice, wgs = half ? 512 : 256;
    const int least = (g.n + wide - 1) / wide;
    g.bin_parts = std::max(1, wgs / least);
    const int bins = (std::max(wgs / g.bin_parts, least) + 7) & ~7;
    g.bin_w = (g.n + bins - 1) / bins;
    g.bin_magic = (unsigned)((1ull << 32) / (unsigned)g.bin_w + 1);
    g.bin_share = egs::bin_share(g.n, g.m, bins);
    const int64_t places = g.m + (int64_t)egs::kBinHead * g.n;
    g.nchunks = (int)((places + g.bin_share - 1) / g.bin_share);
    const int64_t padded = g.m + (int64_t)g.nchunks * egs::kBinPad * bins + egs::kBinPad;
    if (bins > egs::kBinMax || padded > s->bin_cap || (int64_t)(bins + 1) * g.nchunks > s->boff_cap)
        return;
    g.bins = bins;
    g.bin_once = 10 * padded > kMemorySideCache * 3 / 4;
    // sparse rounds need the transpose, after which the run leaves the bins (build_csc): worth
    // it only for long tails
    if (o->dense_pct == 0) g.dense_min = std::max<int64_t>(1, g.n / kBinDensePart);
}

// Whether one-sweep games lift their static hub lists in the same launch as the sweep.
static void pick_hub_fused(egs_solver *s) {
    egs::DevGame &g = s->g;
    const egs::LaunchShape &sh = s->sh;
    g.hub_fused = g.phases == 1 && !g.bins && (sh.use_wave || sh.use_block) &&
                  g.round_grid + g.wave_grid + g.block_grid <= egs::kStatSlots;     // a statistics slot per workgroup
}

static int pick_shape(egs_solver *s, const egs_options *o, bool whole) {
    egs::DevGame &g = s->g;
    egs::LaunchShape &sh = s->sh;
    egs_options def{};
    if (!o) o = &def;
    const double avg = (double)g.m / (double)g.n;
    int G = o->group;
    if (G == 0) G = std::min(16, pow2ceil((int)(avg + 0.999)));
    if (G < 1 || G > 64 || (G & (G - 1)))
        return fail(EGS_E_ARG, "group must be a power of two in 1..64 (got %d)", G);
    sh.group = G;
    g.big_deg = o->big_deg > 0 ? o->big_deg : std::max(64, 8 * G);
    g.huge_deg = o->huge_deg > 0 ? o->huge_deg : 4096;
    if (g.huge_deg < g.big_deg) g.huge_deg = g.big_deg;
    const int pct = o->dense_pct > 0 ? o->dense_pct : 12;
    g.dense_min = pct > 100 ? INT64_MAX : std::max<int64_t>(1, (int64_t)g.n * pct / 100);
    sh.grid = o->grid > 0 ? o->grid : 1024;
    if (sh.grid > egs::kStatSlots) sh.grid = egs::kStatSlots;
    sh.use_wave = s->max_outdeg > g.big_deg;
    sh.use_block = s->max_outdeg > g.huge_deg;
    sh.wave_grid = 1024;
    sh.block_grid = 1024;
    s->batch_rounds = o->batch_rounds > 0 ? o->batch_rounds : 32;
    // with a stop flag at most kStopBatch rounds are queued ahead of the host, so a stop
    // takes effect within a few rounds
    if (o->stop_flag) s->batch_rounds = std::min(s->batch_rounds, kStopBatch);
    if (o->graphs < -1 || o->graphs > 1) return fail(EGS_E_ARG, "graphs must be -1, 0 or 1 (got %d)", o->graphs);
    s->use_graphs = o->graphs > 0 && !o->stop_flag && !s->no_alloc;
    s->phase_cap = egs_max_loop_c(g.m, g.n, g.mg, o->max_phases);
    s->capped = o->max_phases >= 0;
    s->stop_flag = o->stop_flag;
    s->cert_every = o->certify_every == 0 ? kCertEvery : (o->certify_every < 0 ? 0 : o->certify_every);
    s->cert_max_passes = o->cert_max_passes > 0 ? o->cert_max_passes : 1024;
    g.rise = s->cert_every > 0 ? s->d_sigma : nullptr;    // rise stamps only when proofs run
    // phased dense rounds where the value array outgrows the L2 (and the buffers exist):
    // slices of 2^slice_shift successors, at most kMaxPhases of them
    // auto: phases once the value array outgrows 4 MB (at 2^20 vertices one in-place sweep
    // wins: the skewed 2^20 game solved in 13.6 ms in 81 rounds, against 15.8-16.3 ms in 98-99
    // rounds with 2-8 phases)
    int want = o->slices == 0 ? (g.n > egs::kPhaseMinN ? egs::kDefaultPhases : 1) : o->slices;
    if (want < 1 || want > egs::kMaxPhases)
        return fail(EGS_E_ARG, "slices must be 0 (auto) or 1..%d (got %d)", egs::kMaxPhases, o->slices);
    g.phases = 1;
    g.slice_shift = 31;
    pick_bins(s, o, whole);
    if (g.bins && o->certify_every == 0) s->cert_every = kCertEveryBinned;
    if (want > 1 && s->d_slen && !g.bins) {
        int shift = 0;
        while (((int64_t)(want) << shift) < g.n) shift++;          // want slices of 2^shift cover n
        g.slice_shift = shift;
        g.phases = (int)(((int64_t)g.n + (1LL << shift) - 1) >> shift);
        if (g.big_deg > egs::kMaxSliceDeg) g.big_deg = egs::kMaxSliceDeg;   // lengths are bytes
        if (g.huge_deg < g.big_deg) g.huge_deg = g.big_deg;
        sh.use_wave = s->max_outdeg > g.big_deg;
        sh.use_block = s->max_outdeg > g.huge_deg;
    }
    g.slen = s->d_slen;
    g.sbase = s->d_sbase;
    g.sedges = s->d_sedges;
    g.sshift = g.phases > 1 ? egs::pack_shift(g.n, s->wmax) : 0;   // 32-bit slice edges when they fit
    g.hacc = s->d_hacc;
    g.hcnt = s->d_hcnt;
    g.hbest = s->d_hbest;
    g.hflag = s->d_hflag;
    g.bigmask = s->d_bigmask;
    // The phased kernels run about as many workgroups as the device holds at once (eight of
    // 256 threads per CU), each over a fixed set of tiles whose partial results sit in LDS.
    const int64_t tiles = ((int64_t)g.n + egs::kSliceTile - 1) / egs::kSliceTile;
    const int wpc = o->phase_wgs_per_cu > 0 ? std::min(o->phase_wgs_per_cu, 32) : 8;
    g.phase_grid = (int)std::min<int64_t>(tiles, wpc * (int64_t)std::max(1, s->cus));
    g.phase_tiles = (int)((tiles + g.phase_grid - 1) / g.phase_grid);
    if (g.phases > 1 && g.phase_tiles * egs::kSliceTile * 12 > 96 * 1024) {
        // keep the closure kernel's partial state (12 bytes a vertex) within 96 KB of LDS
        g.phase_tiles = 96 * 1024 / (egs::kSliceTile * 12);
        g.phase_grid = (int)((tiles + g.phase_tiles - 1) / g.phase_tiles);
    }
    g.round_grid = sh.grid;
    g.wave_grid = sh.use_wave ? sh.wave_grid : 0;
    g.block_grid = sh.use_block ? sh.block_grid : 0;
    pick_hub_fused(s);
    return EGS_OK;
}

// Transpose on the solver stream, then open the sparse round modes (ring[12] = 1).
static hipError_t build_csc(egs_solver *s) {
    const bool sorted = egs::transpose_sorted_fits(s->g.n, s->g.m, s->tcounts_cap, s->m_cap);
    // with the weights where there are hubs to keep out of the rounds (pred_can_rise; without,
    // the look at them costs a round 1.5 us of 13 and saves nothing: 2-regular games took 13%
    // longer); in the place of a binned game's candidates.  Graphs keep the arguments they were
    // captured with, so not there.
    // A vertex that replaced values leave below its lift is in no round's work, which the look at
    // the weights (pred_can_rise) rests on: not there either.
    int *cweight = sorted && !s->values_set && s->sh.use_wave && !s->use_graphs && egs::transpose_weights_fit(s->g.n, s->wmax) ? s->d_cweight : nullptr;
    s->g.cweight = cweight;
    hipError_t e = sorted
                       ? egs::launch_transpose_sorted(s->g, s->d_tcounts, s->d_toffs, s->d_tscan, s->d_titems, cweight,
                                                      s->stream)
                       : egs::launch_transpose(s->g, s->d_tile, s->d_fill, s->stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(s->d_ring + 12, s->h_probe + kPinOne, sizeof(int), hipMemcpyHostToDevice, s->stream);
    if (e == hipSuccess) s->csc_built = true;
    if (s->g.bins) {
        // sparse rounds from here on, dense ones as sweeps in place
        s->g.bins = 0;
        pick_hub_fused(s);
    }
    return e;
}

// Set-up of the round kernels: counters, static hub lists, slice layout, initial frontier.
// A binned game's first round is done with its layout (`first`).
static int prepare_rounds(egs_solver *s, bool first = false) {
    // graphs hold the launch arguments they were captured with: kept while those stay the same
    if (memcmp(&s->graph_g, &s->g, sizeof(s->g)) != 0 || memcmp(&s->graph_sh, &s->sh, sizeof(s->sh)) != 0) {
        drop_graphs(s);
        memcpy(&s->graph_g, &s->g, sizeof(s->g));
        memcpy(&s->graph_sh, &s->sh, sizeof(s->sh));
    }
    // The set-up is timed by its own events and not waited for: the first round queues
    // behind it at once, and its time and the initial frontier are read after a later wait.
    // (The no-allocation solver has no events: it times on the host and waits here.)
    const bool lazy = s->ev_pa && s->ev_pb;
    double t0 = 0;
    if (lazy) HIP_TRY(hipEventRecord(s->ev_pa, s->stream));
    else HIP_TRY(mark_start(s, &t0));
    HIP_TRY(egs::launch_prepare_reset(s->g, s->stream));   // statistics, counters, modes, ring slots
    // The transpose only feeds the sparse round modes, and many solves never need them
    // (config-2-like games sweep densely until a proof ends them).  Rounds stay dense while
    // it is missing; a round that would have gone sparse raises ring[13], and the host
    // builds the transpose at its next probe and opens sparse rounds (ring[12]).
    if (s->g.dense_min > s->g.n) HIP_TRY(build_csc(s));     // dense sweeps switched off
    if (s->sh.use_block)             // shared lifts of the vertices above huge_deg start empty
        HIP_TRY(egs::launch_hbest_reset(s->g, s->stream));
    HIP_TRY(egs::launch_classify(s->g, s->d_ring + 9, s->stream));
    if (s->g.bins) {
        s->bins_open = false;
        HIP_TRY(egs::launch_bin_build(s->g, first, s->stream));
    } else {
        // with slices and no transpose the slice set-up also stores the initial state
        const bool init_in_slices = s->g.phases > 1 && !s->csc_built;
        HIP_TRY(egs::launch_slices(s->g, s->stream, init_in_slices));
        HIP_TRY(egs::launch_init(s->g, s->stream, init_in_slices));
    }
    // the initial frontier's counters ride on the same wait as the timing
    HIP_TRY(hipMemcpyAsync(s->h_probe + kPinInit, s->d_lcnt + 1 * egs::kListCounters,
                           sizeof(int) * egs::kListCounters, hipMemcpyDeviceToHost, s->stream));
    if (lazy) {
        HIP_TRY(hipEventRecord(s->ev_pb, s->stream));
        memset(&s->st, 0, sizeof(s->st));
        s->prep_open = true;
    } else {
        float ms = 0.f;
        HIP_TRY(mark_stop(s, t0, &ms));
        memset(&s->st, 0, sizeof(s->st));
        s->st.ms_prepare = ms;
        s->st.initial_active = (int32_t)list_total(s, s->h_probe + kPinInit);
    }
    return EGS_OK;
}

// Single launches suit a solve whose options leave the round kernels' shape open and that
// nothing has to stop part-way (the stop flag is polled between rounds on the host).
static bool takes_whole(const egs_options *o) {
    return !o || (o->group == 0 && o->big_deg == 0 && o->huge_deg == 0 && o->grid == 0 && o->batch_rounds == 0 &&
                  o->dense_pct == 0 && o->slices == 0 && o->phase_wgs_per_cu == 0 && o->graphs == 0 && !o->stop_flag);
}

// Vertices of g with lift(val)(v) != val(v).
static int count_violations(egs_solver *s, const egs::DevGame &g, int64_t *violations) {
    HIP_TRY(egs::launch_violations(g, (unsigned long long *)s->d_misc, s->stream));
    unsigned long long *h = (unsigned long long *)(s->h_probe + kPinViol);
    HIP_TRY(hipMemcpyAsync(h, s->d_misc, sizeof(unsigned long long), hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    *violations = (int64_t)*h;
    return EGS_OK;
}

// Hand a run over from single launches to the round kernels: their whole set-up when it has
// not begun, else the counters and lists, with the values reached and the next round a full
// sweep (none when the run has converged).
static int leave_whole(egs_solver *s) {
    s->mirrored = false;
    if (s->bins_open) return prepare_rounds(s);
    if (s->whole.nb == 0) return EGS_OK;
    s->whole.nb = 0;
    const bool reached = s->whole_gave_up && !s->capped;
    if (s->whole_rounds == 0 && !s->st.converged && !reached) return prepare_rounds(s);
    HIP_TRY(egs::launch_prepare_reset(s->g, s->stream));
    if (s->sh.use_block) HIP_TRY(egs::launch_hbest_reset(s->g, s->stream));
    HIP_TRY(egs::launch_classify(s->g, s->d_ring + 9, s->stream));
    HIP_TRY(egs::launch_resume(s->g, (int)s->next_round, s->st.converged != 0, s->stream));
    if (s->whole_rounds == 0 && !s->st.converged) {
        // the initial frontier: the vertices that a lift of zeros changes (the stamps are zeros now)
        egs::DevGame zero = s->g;
        zero.val = s->d_stamp;
        int64_t active = 0;
        if (int rc = count_violations(s, zero, &active)) return rc;
        s->st.initial_active = (int32_t)active;
    }
    return EGS_OK;
}

// A single launch whose workgroups would not all fit beside other launches is not made (they
// would wait for each other until their limit); the round kernels take the game.
struct WholeRoom {
    egs::DeviceUnits &u;
    int want;
    bool ok;
    WholeRoom(const egs_solver *s) : u(egs::device_units(s->device)), want(s->whole.nb > 1 ? egs::units_of(s->whole.nb, s->cus) : 0) {
        ok = want == 0 ||                                      // one workgroup waits for nobody
             u.single.fetch_add(want) + want + u.games.load() <= s->cus;
    }
    ~WholeRoom() { u.single.fetch_sub(want); }
};

// Rounds in single launches until the fixpoint, `limit` more rounds, or a state that the
// round kernels serve better; *status tells which (kWholeNone: the launch gave up waiting for
// its workgroups, and the values are some state between its start and the fixpoint).
static int run_whole(egs_solver *s, int64_t limit, int *status) {
    // a launch of this many rounds ends within tens of milliseconds
    constexpr int64_t kRoundsPerLaunch = 8192;
    egs::WholeArgs a{};
    const egs::DevGame &g = s->g;
    a.n = g.n;
    a.n0 = g.n0;
    a.mg = g.mg;
    a.wmax = s->wmax;
    a.m = g.m;
    a.ptr = g.ptr;
    a.edges = g.edges;
    a.val = g.val;
    a.rise = g.rise;
    a.h = s->d_h;
    a.ctl = s->d_whole;
    a.nbmax = s->whole.nbmax;
    a.wait = s->whole_wait;
    a.every = s->cert_every;
    a.max_passes = s->cert_max_passes;
    a.max_cands = kCertCandidates;
    a.sparse_exit = g.n > kWholeDenseN ? kSparseWantRounds : 0;
    a.dense_min = g.dense_min;
    // the result comes back through the pinned block, which the kernel stores into; the
    // no-allocation solver has none and copies it from device memory
    egs::WholeResult *res = (egs::WholeResult *)(s->h_probe + kPinWhole);
    // one workgroup stores its values into the small read-back area on its way out
    a.mirror = s->whole.nb == 1 && !s->values_out && 4 * (size_t)g.n <= s->out_small ? (int *)s->h_small : nullptr;
    a.out = s->no_alloc ? (egs::WholeResult *)s->d_misc : res;
    *status = egs::kWholeNone;
    WholeRoom room(s);
    if (!room.ok) return EGS_OK;
    *status = egs::kWholeLimit;
    while (*status == egs::kWholeLimit && limit > 0) {
        a.limit = std::min(limit, kRoundsPerLaunch);
        a.round0 = s->whole_rounds;
        a.next_cert = s->next_cert;
        a.gap = (int)s->cert_gap;
        a.cap = s->cert_cap;
        a.seq = ++s->whole_seq;
        __atomic_store_n(&res->done, 0u, __ATOMIC_RELEASE);     // no launch of this solver is running
        if (s->whole_rounds > 0) HIP_TRY(egs::launch_whole_prep(s->whole, g, s->d_whole, false, s->stream));
        HIP_TRY(egs::launch_whole(s->whole, a, s->stream));
        bool got = false;
        if (s->no_alloc) {
            HIP_TRY(hipMemcpyAsync(res, a.out, sizeof(*res), hipMemcpyDeviceToHost, s->stream));
            HIP_TRY(hipStreamSynchronize(s->stream));
            got = res->done == a.seq;
        } else {
            HIP_TRY(wait_word(s, &res->done, a.seq, &got));
        }
        if (!got) {
            *status = egs::kWholeNone;
            s->whole_gave_up = true;
            break;
        }
        const int64_t ran = res->rounds - s->whole_rounds;
        if (s->whole_rounds == 0) {
            s->st.initial_active = (int32_t)res->initial;
            s->st.ms_prepare += 1e-5 * (double)res->ticks_setup;
        } else {
            s->st.ms_iterate += 1e-5 * (double)res->ticks_setup;
        }
        s->st.ms_iterate += 1e-5 * (double)(res->ticks - res->ticks_setup);
        s->whole_st.processed += ran * g.n;
        s->whole_st.edges_relaxed += res->edges;
        s->whole_st.lifted += res->lifted;
        s->st.cert_attempts += res->attempts;
        s->st.certificates += res->certs;
        s->st.cert_passes += res->passes;
        s->st.top_marked += res->marked;
        s->st.cert_pruned += res->pruned;
        s->whole_rounds = res->rounds;
        s->next_round = res->rounds + 1;
        s->next_cert = res->next_cert;
        s->cert_gap = res->gap;
        s->cert_cap = res->cap;
        limit -= ran;
        *status = res->status;
        s->mirrored = a.mirror != nullptr;
    }
    s->st.phases = s->whole_rounds;
    s->st.processed = s->whole_st.processed;
    s->st.edges_relaxed = s->whole_st.edges_relaxed;
    s->st.lifted = s->whole_st.lifted;
    s->st.converged = *status == egs::kWholeDone;
    return EGS_OK;
}

int egs_solver_prepare(egs_solver *s, const egs_options *opt) {
    if (!s || !s->loaded) return fail(EGS_E_STATE, "egs_solver_prepare: no game loaded");
    HIP_TRY(hipSetDevice(s->device));
    const egs::WholePlan plan = takes_whole(opt) ? egs::whole_plan(s->g.n, s->g.m, s->g.mg, s->wmax, s->max_outdeg, s->whole_max_nb) : egs::WholePlan{};
    int rc = pick_shape(s, opt, plan.nb > 0);
    if (rc) return rc;
    HIP_TRY(close_prepare(s));
    s->csc_built = false;
    s->next_round = 1;
    s->cert_gap = s->cert_every;
    s->next_cert = s->cert_every;
    s->cert_cap = std::min(kCertFirstCap, s->cert_max_passes);
    s->cert_pass_hint = 0;
    s->whole_rounds = 0;
    s->whole_gave_up = false;
    s->whole_st = egs_stats{};
    s->mirrored = false;
    s->values_set = false;
    s->bins_open = false;
    s->whole = plan;
    if (s->whole.nb > 0) {
        HIP_TRY(egs::launch_whole_prep(s->whole, s->g, s->d_whole, true, s->stream));
        memset(&s->st, 0, sizeof(s->st));
    } else if (s->g.bins) {
        // the values and chunks now; the layout with the first round, in iterate()
        HIP_TRY(egs::launch_bin_prep(s->g, s->stream));
        memset(&s->st, 0, sizeof(s->st));
        s->bins_open = true;
    } else {
        rc = prepare_rounds(s);
        if (rc) return rc;
    }
    s->prepared = true;
    return EGS_OK;
}

// The run's statistics: queued on the stream before the run's closing wait, read after it.
static int queue_stats(egs_solver *s) {
    HIP_TRY(egs::launch_sum_stats(s->g, egs::kStatSlots, s->d_statsum, s->stream));
    unsigned long long *h = (unsigned long long *)(s->h_probe + kPinStats);
    // statistics, last round and the next round's input size in one read-back
    HIP_TRY(hipMemcpyAsync(h, s->d_statsum, sizeof(unsigned long long) * 6, hipMemcpyDeviceToHost, s->stream));
    return EGS_OK;
}

static int collect_stats(egs_solver *s) {
    const unsigned long long *h = (const unsigned long long *)(s->h_probe + kPinStats);
    // on top of the rounds done in single launches
    s->st.processed = (int64_t)h[0] + s->whole_st.processed;
    s->st.edges_relaxed = (int64_t)h[1] + s->whole_st.edges_relaxed;
    s->st.lifted = (int64_t)h[2] + s->whole_st.lifted;
    s->st.pred_visits = (int64_t)h[3];
    s->st.phases = (int32_t)h[4];
    s->st.csc_built = s->csc_built ? 1 : 0;
    s->st.converged = h[5] == 0;
    return EGS_OK;
}

int egs_solver_iterate(egs_solver *s, int64_t max_phases, egs_stats *st) {
    if (!s || !s->prepared) return fail(EGS_E_STATE, "egs_solver_iterate: call egs_solver_prepare first");
    HIP_TRY(hipSetDevice(s->device));
    int64_t limit = s->phase_cap - (s->next_round - 1);
    if (max_phases >= 0 && max_phases < limit) limit = max_phases;
    if (s->next_round + limit > 0x7ffffff0LL) limit = 0x7ffffff0LL - s->next_round;
    if (s->whole.nb > 0) {
        int status = egs::kWholeNone, rc = EGS_OK;
        // (no launch where no round is allowed: the round kernels' set-up tells the frontier's size)
        if (max_phases < 0 && !s->st.converged && (limit > 0 || s->whole_rounds > 0)) {
            const int64_t before = s->whole_rounds;
            rc = run_whole(s, limit, &status);
            if (rc) return rc;
            limit -= s->whole_rounds - before;
        }
        if (status == egs::kWholeDone || status == egs::kWholeLimit || s->st.converged) {
            if (st) *st = s->st;
            return s->st.converged ? 1 : 0;
        }
        rc = leave_whole(s);
        if (rc) return rc;
        if (status == egs::kWholeSparse) HIP_TRY(build_csc(s));
    }
    int64_t launched = 0;
    if (s->bins_open) {
        const bool first = limit > 0 && !(s->stop_flag && *s->stop_flag);
        const int rc = prepare_rounds(s, first);
        if (rc) return rc;
        if (first) {
            s->next_round = 2;
            launched = 1;
        }
    }
    double t0 = 0;
    HIP_TRY(mark_start(s, &t0));
    int pending = -1;     // probe slot in flight
    bool done = false;
    int batch = 4;        // grow towards batch_rounds so short solves do not overshoot much
    int64_t listed = -1;  // items of the latest list read back (-1: not known)
    while (!done && launched < limit) {
        int nb = (int)std::min<int64_t>(batch, limit - launched);
        const bool accel = s->cert_every > 0;
        if (accel && s->next_round - 1 >= s->next_cert) {
            // pause: converged already?  else try to prove a climbing set is TOP
            HIP_TRY(hipMemcpyAsync(s->h_probe + kPinConv, s->d_lcnt + (s->next_round % 3) * egs::kListCounters,
                                   sizeof(int) * egs::kListCounters, hipMemcpyDeviceToHost, s->stream));
            // the attempt's value histogram rides on the same wait
            // waits through an event: a busy wait on it wakes the host sooner than a stream
            // synchronisation (small games solved 4-8% faster)
            egs::CertBuffers cb{s->d_hist, s->d_h, s->d_bfcnt, s->d_bits, s->h_probe + kPinCert, s->ev_b};
            const bool hist = s->wmax > 0;
            if (hist) HIP_TRY(egs::certify_prefetch(s->g, cb, s->wmax, s->stream));
            // from the run's second attempt on, one more round runs while the host waits for
            // these read-backs (a no-op when the frontier was already empty) and the attempt
            // starts after it; any candidate set is proved or refused exactly, so the
            // histogram may be a round old.  Not before the first attempt: its proof usually
            // marks many vertices TOP, after which the same round costs less.
            const bool ahead = s->st.cert_attempts > 0 && launched < limit && !(s->stop_flag && *s->stop_flag) &&
                               s->ev_b;
            if (ahead) {
                HIP_TRY(hipEventRecord(s->ev_b, s->stream));
                HIP_TRY(egs::launch_round(s->g, s->sh, 0, s->stream));
                HIP_TRY(egs::launch_advance(s->g, 1, s->stream));
                s->next_round++;
                launched++;
                HIP_TRY(hipEventSynchronize(s->ev_b));
            } else {
                HIP_TRY(egs::wait_queued(cb.ev, s->stream));
            }
            if (list_total(s, s->h_probe + kPinConv) == 0) break;
            if (s->stop_flag && *s->stop_flag) break;
            egs::CertResult cr;
            const int got = egs::certify_top(s->g, cb, s->wmax, (int)(s->next_round - 1), s->cert_cap,
                                             kCertCandidates, s->sh.use_wave != 0, hist, s->stop_flag,
                                             s->cert_pass_hint, s->stream, cr);
            if (got < 0) return fail(EGS_E_HIP, "certification: %s", hipGetErrorString(hipGetLastError()));
            if (cr.last_passes > 0) s->cert_pass_hint = cr.last_passes;
            s->st.cert_attempts++;
            s->st.cert_passes += cr.passes;
            s->st.cert_pruned += cr.closure_failed;
            if (got > 0) {
                s->st.certificates++;
                s->st.top_marked += cr.marked;
                // the marking kernel has named the next round (ring[11]) a full sweep
                // the spacing stays as the failures before left it (cert_next_gap): a long run
                // that keeps proving small sets does not pay an attempt every few rounds
                batch = 1;        // the fixpoint often follows at once: probe again early
                nb = 1;
                listed = -1;
            } else {
                s->cert_gap = egs::cert_next_gap(s->cert_gap, s->cert_every, cr.passes + kCertTryRounds * cr.tried);
                if (cr.cap_hit) s->cert_cap = std::min(s->cert_cap * 2, s->cert_max_passes);
            }
            s->next_cert = s->next_round - 1 + s->cert_gap;
            pending = -1;
        }
        if (accel) nb = (int)std::max<int64_t>(1, std::min<int64_t>(nb, s->next_cert - (s->next_round - 1)));
        // a short list after the transpose: the sparse tail, in launches of as many rounds as are
        // left before the next proof attempt (not with a stop flag, which is polled every round)
        if (listed > 0 && listed <= egs::tail_items(s->sh) && s->csc_built && !s->use_graphs && !s->stop_flag) {
            int64_t most = std::min<int64_t>(limit - launched, kTailRounds);
            if (accel) most = std::max<int64_t>(1, std::min(most, s->next_cert - (s->next_round - 1)));
            HIP_TRY(egs::launch_tail(s->g, s->sh, (int)most, s->stream));
            // the counters of all three lists, the modes and the ring lie in this order
            int *hp = s->h_probe + kPinProbe;
            HIP_TRY(hipMemcpyAsync(hp, s->d_lcnt, sizeof(int) * (size_t)(s->d_ring + 16 - s->d_lcnt), hipMemcpyDeviceToHost,
                                   s->stream));
            HIP_TRY(probe_mark(s, 0));
            HIP_TRY(probe_wait(s, 0));
            pending = -1;
            const int reached = hp[s->d_ring + 14 - s->d_lcnt];
            const int ran = reached - (int)s->next_round;
            listed = -1;
            if (ran > 0) {
                s->next_round = reached;
                launched += ran;
                listed = list_total(s, hp + (reached % 3) * egs::kListCounters);
                if (listed == 0) done = true;
                continue;
            }
        }
        int k = 0;
        if (s->use_graphs) {
            for (int b = kGraphSizes - 1; b >= 0; b--)
                while (nb - k >= (1 << b)) {
                    HIP_TRY(replay_batch(s, b));
                    k += 1 << b;
                }
        } else {
            for (; k < nb; k++) {
                // the stop flag is polled before every round, as the reference polls
                // timeout_expired once per round (src/dev_EG_alg.cu:376)
                if (s->stop_flag && *s->stop_flag) break;
                HIP_TRY(egs::launch_round(s->g, s->sh, k, s->stream));
            }
            if (k > 0) HIP_TRY(egs::launch_advance(s->g, k, s->stream));
        }
        if (k == 0) break;
        s->next_round += k;
        launched += k;
        const int slot = (pending + 1) & 1;
        int *hp = s->h_probe + kPinProbe + slot * kProbeStride;
        const int *src = s->d_lcnt + (s->next_round % 3) * egs::kListCounters;
        // Until the transpose exists the probe also reads ring[13].  The list counters, the
        // round modes and the ring lie in that order in the device arena, so one copy of the
        // span from this slot's counters to ring[13] reads both.
        const ptrdiff_t span = s->d_ring + 14 - src;
        if (s->csc_built) {
            HIP_TRY(hipMemcpyAsync(hp, src, sizeof(int) * egs::kListCounters, hipMemcpyDeviceToHost, s->stream));
        } else if (span > egs::kListCounters && span <= kProbeStride) {
            HIP_TRY(hipMemcpyAsync(hp, src, sizeof(int) * (size_t)span, hipMemcpyDeviceToHost, s->stream));
            s->probe_want[slot] = (int)span - 1;
        } else {
            HIP_TRY(hipMemcpyAsync(hp, src, sizeof(int) * egs::kListCounters, hipMemcpyDeviceToHost, s->stream));
            HIP_TRY(hipMemcpyAsync(hp + kProbeWant, s->d_ring + 13, sizeof(int), hipMemcpyDeviceToHost, s->stream));
            s->probe_want[slot] = kProbeWant;
        }
        HIP_TRY(probe_mark(s, slot));
        if (pending >= 0) {
            HIP_TRY(probe_wait(s, pending));
            listed = list_total(s, s->h_probe + kPinProbe + pending * kProbeStride);
            if (listed == 0) done = true;
            // enough rounds wanted to go sparse: build the transpose now
            if (!done && !s->csc_built && s->h_probe[kPinProbe + pending * kProbeStride + s->probe_want[pending]] >= (s->g.bins ? kSparseWantBinned : kSparseWantRounds))
                HIP_TRY(build_csc(s));
        }
        pending = slot;
        if (s->stop_flag && *s->stop_flag) break;
        if (batch < s->batch_rounds) batch = std::min(s->batch_rounds, batch * 2);
    }
    int rc = queue_stats(s);
    if (rc) return rc;
    float ms = 0.f;
    HIP_TRY(mark_stop(s, t0, &ms));                  // also the wait for the statistics
    HIP_TRY(close_prepare(s));
    rc = collect_stats(s);
    if (rc) return rc;
    s->st.ms_iterate += ms;
    if (st) *st = s->st;
    return s->st.converged ? 1 : 0;
}

int egs_solver_stats(egs_solver *s, egs_stats *st) {
    if (!s || !st) return fail(EGS_E_ARG, "null argument");
    // asked between prepare and the first round, where the first launch of the run would make the
    // initial frontier: it is counted here (with every value 0 the vertices that a lift changes)
    // and the run left as it is
    const bool unborn = s->prepared && (s->bins_open || (s->whole.nb > 0 && s->whole_rounds == 0 && !s->st.converged));
    if (unborn) {
        HIP_TRY(hipSetDevice(s->device));
        double t0 = 0;
        float ms = 0.f;
        int64_t active = 0;
        HIP_TRY(mark_start(s, &t0));
        if (int rc = egs_solver_count_violations(s, &active)) return rc;
        HIP_TRY(mark_stop(s, t0, &ms));
        s->st.initial_active = (int32_t)active;
        s->st.ms_prepare = ms;
    }
    HIP_TRY(close_prepare(s));
    *st = s->st;
    return EGS_OK;
}

int egs_solver_read_values(egs_solver *s, int32_t *host_values) {
    if (!s || !s->loaded || !host_values) return fail(EGS_E_STATE, "egs_solver_read_values: nothing to read");
    const size_t bytes = sizeof(int) * (size_t)s->g.n;
    if (s->mirrored) {
        memcpy(host_values, s->h_small, bytes);
        return EGS_OK;
    }
    HIP_TRY(hipSetDevice(s->device));
    HIP_TRY(read_back(s, host_values, s->d_val, bytes));
    return EGS_OK;
}

int egs_solver_read_winning(egs_solver *s, uint32_t *host_bits) {
    if (!s || !s->loaded || !host_bits) return fail(EGS_E_STATE, "egs_solver_read_winning: nothing to read");
    HIP_TRY(hipSetDevice(s->device));
    // the proof bitmaps are idle outside an attempt: the first holds ceil(n/32) words
    HIP_TRY(egs::launch_winning(s->d_val, s->g.n, s->d_bits, s->stream));
    s->mirrored = false;                     // the small read-back area is used
    HIP_TRY(read_back(s, host_bits, s->d_bits, sizeof(uint32_t) * (((size_t)s->g.n + 31) / 32)));
    return EGS_OK;
}

const int32_t *egs_solver_device_values(egs_solver *s) {
    if (!s) return nullptr;
    s->values_out = true;
    s->mirrored = false;
    return s->d_val;
}

void *egs_solver_stream(egs_solver *s) { return s ? (void *)s->stream : nullptr; }

int egs_solver_read_csc(egs_solver *s, int32_t *cptr, int32_t *cpred) {
    if (!s || !s->prepared) return fail(EGS_E_STATE, "egs_solver_read_csc: not prepared");
    HIP_TRY(hipSetDevice(s->device));
    if (int rc = leave_whole(s)) return rc;
    if (!s->csc_built) HIP_TRY(build_csc(s));
    HIP_TRY(hipMemcpyAsync(cptr, s->d_cptr, sizeof(int) * ((size_t)s->g.n + 1), hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipMemcpyAsync(cpred, s->d_cpred, sizeof(int) * (size_t)s->g.m, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return EGS_OK;
}

int egs_solver_count_violations(egs_solver *s, int64_t *violations) {
    if (!s || !s->loaded || !violations) return fail(EGS_E_STATE, "egs_solver_count_violations: nothing loaded");
    HIP_TRY(hipSetDevice(s->device));
    return count_violations(s, s->g, violations);
}

int egs_solver_set_values(egs_solver *s, const int32_t *host_values) {
    if (!s || !s->prepared || !host_values) return fail(EGS_E_STATE, "egs_solver_set_values: call egs_solver_prepare first");
    HIP_TRY(hipSetDevice(s->device));
    if (int rc = leave_whole(s)) return rc;
    s->values_set = true;
    s->g.cweight = nullptr;
    HIP_TRY(hipMemcpyAsync(s->d_val, host_values, sizeof(int) * (size_t)s->g.n, hipMemcpyHostToDevice, s->stream));
    // the values may hold TOP: the phased rounds then read their TOP masks (ring[15])
    HIP_TRY(hipMemcpyAsync(s->d_ring + 15, s->h_probe + kPinOne, sizeof(int), hipMemcpyHostToDevice, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return EGS_OK;
}

int egs_solver_top_certificate(egs_solver *s, int32_t max_passes, int64_t *host_h, int32_t *passes) {
    if (!s || !s->prepared || !host_h) return fail(EGS_E_STATE, "egs_solver_top_certificate: call egs_solver_prepare first");
    HIP_TRY(hipSetDevice(s->device));
    if (int rc = leave_whole(s)) return rc;
    egs::CertBuffers cb{s->d_hist, s->d_h, s->d_bfcnt, s->d_bits, s->h_probe + kPinCert};
    egs::CertResult cr;
    const int got = egs::certify_all_top(s->g, cb, s->wmax, max_passes > 0 ? max_passes : (1 << 16),
                                         s->sh.use_wave != 0, s->stream, cr);
    if (got == -1) return fail(EGS_E_HIP, "certificate: %s", hipGetErrorString(hipGetLastError()));
    if (got == -2) return fail(EGS_E_ARG, "certificate: potentials of this game could overflow 64 bits");
    HIP_TRY(read_back(s, host_h, s->d_h, sizeof(int64_t) * (size_t)s->g.n));
    if (passes) *passes = cr.passes;
    return got;
}

int egs_solve(int device, int32_t n, int32_t n0, int64_t m, int32_t mg, const int32_t *ptr,
              const int32_t *succ, const int32_t *w, int32_t *values, const egs_options *opt,
              egs_stats *st) {
    egs_solver *s = nullptr;
    int rc = egs_solver_create(device, n, m, &s);
    if (rc) return rc;
    rc = egs_solver_load(s, EGS_MEM_HOST, n, n0, m, mg, ptr, succ, w);
    if (!rc) rc = egs_solver_prepare(s, opt);
    if (!rc) {
        rc = egs_solver_iterate(s, -1, st);
        if (rc >= 0) rc = egs_solver_read_values(s, values) ? EGS_E_HIP : EGS_OK;
    }
    egs_solver_destroy(s);
    return rc;
}

// ---------------------------------------------------------------------------------------
// Solve without allocating: for callers that cannot allocate device memory (code under HIP
// graph capture, tight serving loops, harnesses that forbid hipMalloc).  The workspace of
// the one-game solver for games up to kNoAllocN vertices and kNoAllocM edges is a
// file-scope device array; each device that runs it holds its own copy until the process
// ends, found once per device with hipGetSymbolAddress (the array's name is not a device
// address in host code).  The host side of the solver is a static object per device.
// Calls that overlap on one device share both and race.
// ---------------------------------------------------------------------------------------

namespace {

constexpr int32_t kNoAllocN = 1 << 16;
constexpr int64_t kNoAllocM = 1 << 20;
constexpr size_t kScratchBytes = make_layout(kNoAllocN, kNoAllocM).total;
constexpr int kNoAllocDevices = 64;

struct NoAllocSlot {
    egs_solver s;
    int probe[kPinProbe + 2 * kProbeStride];   // the solver's read-back area (pageable; every read waits on the stream)
    bool ready = false;
};
NoAllocSlot g_noalloc[kNoAllocDevices];

}  // namespace

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

static int noalloc_setup(int dev) {
    NoAllocSlot &sl = g_noalloc[dev];
    if (sl.ready) return EGS_OK;
    int rc = check_gfx950(dev);
    if (rc) return rc;
    char *ptr = nullptr;
    hipError_t e = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
        return fail(EGS_E_HIP, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
    egs_solver &s = sl.s;
    s.device = dev;
    s.no_alloc = true;
    if (hipDeviceGetAttribute(&s.cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) s.cus = 256;
    s.whole_max_nb = s.cus;
    s.n_cap = kNoAllocN;
    s.m_cap = kNoAllocM;
    s.block = nullptr;                 // not owned: never freed
    s.block_bytes = kScratchBytes;
    bind_layout(&s, ptr, make_layout(kNoAllocN, kNoAllocM));
    s.h_probe = sl.probe;
    s.h_probe[kPinOne] = 1;
    sl.ready = true;
    return EGS_OK;
}

int egs_solve_noalloc(int32_t n, int32_t n0, int64_t m, int32_t mg, const int32_t *d_ptr, const int32_t *d_succ,
                      const int32_t *d_w, int32_t *d_values, const egs_options *opt, egs_stats *st, void *stream) {
    if (n < 1 || n0 < 0 || n0 > n || m < 1 || mg < 0 || !d_ptr || !d_succ || !d_w || !d_values)
        return fail(EGS_E_ARG, "egs_solve_noalloc: bad game (n=%d n0=%d m=%lld mg=%d)", n, n0, (long long)m, mg);
    if (n > kNoAllocN || m > kNoAllocM)
        return fail(EGS_E_CAPACITY,
                    "egs_solve_noalloc: game (n=%d, m=%lld) exceeds the fixed workspace (%d vertices, %lld edges)", n,
                    (long long)m, kNoAllocN, (long long)kNoAllocM);
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kNoAllocDevices) return fail(EGS_E_ARG, "egs_solve_noalloc: device %d out of range", dev);
    int rc = noalloc_setup(dev);
    if (rc) return rc;
    egs_solver *s = &g_noalloc[dev].s;
    s->stream = (hipStream_t)stream;
    s->stop_flag = nullptr;
    rc = egs_solver_load(s, EGS_MEM_DEVICE, n, n0, m, mg, d_ptr, d_succ, d_w);
    if (!rc) rc = egs_solver_prepare(s, opt);
    if (rc) return rc;
    rc = egs_solver_iterate(s, -1, st);
    if (rc < 0) return rc;
    HIP_TRY(hipMemcpyAsync(d_values, s->d_val, sizeof(int32_t) * (size_t)n, hipMemcpyDeviceToDevice, s->stream));
    HIP_TRY(hipStreamSynchronize(s->stream));
    return rc;
}

}  // extern "C"
