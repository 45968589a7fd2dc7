// egs_ingest.hip -- a game in read order turned into the solver's internal game on the device.
//
// The reference's host driver renames vertices so that owner-0 vertices (token MAX) come
// first and owner-1 vertices follow, each block in read order (qsort with the default
// comparator, src/egsolver.c:146-214, stable under glibc), builds the internal CSR
// (src/egsolver.c:253-281) and sums MG = sum_v max(0, max_e -w_e) (src/egsolver.c:283-304).
// Here all three run as kernels after one upload of the read-order arrays:
//   check    offsets from 0 to m with an edge per vertex, successors in range;
//   rename   a scan of the owner-0 flags gives every read index its internal id (owner 0:
//            the owner-0 vertices before it; owner 1: n0 plus the owner-1 vertices before it);
//   rows     a scan of the renamed degrees gives the internal offsets, and each read row is
//            copied to its internal place with renamed successors; on the way MG is summed in
//            64 bits (refused past INT32_MAX as the reference refuses it) and the largest
//            degree and |w| taken.
// The kernels after the check return at once when it found fault, so that the host asks once.
#include "egs_device.h"
#include "egs_internal.h"

namespace egs {

__global__ __launch_bounds__(256) void k_rd_check(const int *__restrict__ rptr, const int *__restrict__ rsucc, int n,
                                                  int64_t m, int *__restrict__ bad) {
    int b = 0;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x)
        if (rptr[r + 1] <= rptr[r]) b |= 2;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < m; e += (int64_t)gridDim.x * blockDim.x)
        if ((unsigned)rsucc[e] >= (unsigned)n) b |= 4;
    if (blockIdx.x == 0 && threadIdx.x == 0 && (rptr[0] != 0 || rptr[n] != m)) b |= 1;
    for (int d = 32; d >= 1; d >>= 1) b |= __shfl_xor(b, d, 64);
    if ((threadIdx.x & 63) == 0 && b) atomicOr(bad, b);
}

__global__ __launch_bounds__(256) void k_rd_flags(const uint8_t *__restrict__ owner, int n, int *__restrict__ flag0,
                                                  const int *bad) {
    if (bad && *bad) return;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x)
        flag0[r] = owner[r] == 0;
}

// pre0[r] = owner-0 vertices before read index r (pre0[n] = n0).
__global__ __launch_bounds__(256) void k_rd_rename(const uint8_t *__restrict__ owner, const int *__restrict__ rptr,
                                                   const int *__restrict__ pre0, int n, int *__restrict__ rev,
                                                   int *__restrict__ ext_of_int, int *__restrict__ deg,
                                                   const int *bad) {
    if (bad && *bad) return;
    const int n0 = pre0[n];
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x) {
        const int i = owner[r] == 0 ? pre0[r] : n0 + (int)r - pre0[r];
        rev[r] = i;
        ext_of_int[i] = (int)r;
        deg[i] = rptr[r + 1] - rptr[r];
    }
}

// Read row r -> internal row rev[r], and the rows' share of MG, the largest degree and |w|.  A
// workgroup takes 256 rows at a time: their edges are consecutive in read order, so it reads
// them with consecutive threads whatever the degrees, finds an edge's row among the 257
// offsets in LDS, and folds max(0, -w) into the row's LDS word.  Bound by the random reads of
// rev and HBM (16 bytes an edge).  A lane per row, with MG, degrees and weights as three more
// passes that ended in thousands of same-address atomics, took 240 us at n = 262,147, m =
// 2.1M (42 + 55 + 48 + 95); this takes 17 us.
__global__ __launch_bounds__(256) void k_rd_rows(const int *__restrict__ rptr, const int *__restrict__ rsucc,
                                                 const int *__restrict__ rw, const int *__restrict__ rev,
                                                 const int *__restrict__ ptr, int n, int2 *__restrict__ edges,
                                                 LoadPartial *__restrict__ part, const int *bad) {
    if (bad && *bad) return;
    __shared__ int s_row[257], s_at[256];
    __shared__ unsigned s_worst[256];
    const int t = threadIdx.x;
    unsigned long long mg = 0;
    int dmax = 0, wmax = 0;
    for (int64_t r0 = (int64_t)blockIdx.x * 256; r0 < n; r0 += (int64_t)gridDim.x * 256) {
        const int rows = (int)min((int64_t)256, n - r0);
        if (t < rows) {
            const int s = rptr[r0 + t];
            s_row[t] = s;
            s_at[t] = ptr[rev[r0 + t]] - s;          // internal place less read place
            dmax = max(dmax, rptr[r0 + t + 1] - s);
        }
        if (t == 0) s_row[rows] = rptr[r0 + rows];
        s_worst[t] = 0;
        __syncthreads();
        const unsigned e1 = (unsigned)s_row[rows];
        for (unsigned at = (unsigned)s_row[0] + t; at < e1; at += 256) {   // past 2^31 in the last step
            const int e = (int)at;
            int lo = 0, hi = rows;                   // largest row starting at or before e
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (s_row[mid] <= e) lo = mid; else hi = mid;
            }
            const int w = rw[e];
            edges[e + s_at[lo]] = make_int2(rev[rsucc[e]], w);
            if (w < 0) atomicMax(&s_worst[lo], 0u - (unsigned)w);
            wmax = max(wmax, load_abs(w));
        }
        __syncthreads();
        mg += s_worst[t];
        __syncthreads();
    }
    load_partial(mg, dmax, wmax, part + blockIdx.x);
}

hipError_t launch_read_order_check(const int *rptr, const int *rsucc, int n, int64_t m, int *bad, hipStream_t st) {
    hipError_t e = hipMemsetAsync(bad, 0, sizeof(int), st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_rd_check, dim3(grid_for(std::max<int64_t>(n, m), 256, 4096)), dim3(256), 0, st, rptr, rsucc, n,
                       m, bad);
    return hipGetLastError();
}

hipError_t launch_internalise(const ReadOrderBuffers &b, int n, const int *bad, int *ptr, int2 *edges,
                              LoadPartial **part, int *nparts, hipStream_t st) {
    const int grid = grid_for(n, 256, 4096);
    hipLaunchKernelGGL(k_rd_flags, dim3(grid), dim3(256), 0, st, b.owner, n, b.flag0, bad);
    hipError_t e = launch_exclusive_scan(b.flag0, n, b.scan_tiles, b.pre0, st, bad);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_rd_rename, dim3(grid), dim3(256), 0, st, b.owner, b.rptr, (const int *)b.pre0, n, b.rev,
                       b.ext_of_int, b.deg, bad);
    e = launch_exclusive_scan(b.deg, n, b.scan_tiles, ptr, st, bad);
    if (e != hipSuccess) return e;
    // a partial per 256 rows at most: 16 bytes, in place of 1,024 bytes of flags
    *part = (LoadPartial *)b.flag0;
    *nparts = grid_for(n, 256, kLoadGrid);
    hipLaunchKernelGGL(k_rd_rows, dim3(*nparts), dim3(256), 0, st, b.rptr, b.rsucc, b.rw, (const int *)b.rev,
                       (const int *)ptr, n, edges, *part, bad);
    return hipGetLastError();
}

}  // namespace egs
