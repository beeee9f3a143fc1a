// mbh_histogram_noalloc: the quantized histogram of mbh_histogram for callers
// that cannot allocate device memory (code under HIP graph capture, serving
// loops, harnesses that forbid hipMalloc). Inputs and the output are the
// caller's device buffers; the block partials live in `scratch`, a static
// device array of kScratchBytes that each GPU the library runs on holds until
// the process ends. No hipMalloc, hipFree, hipMemset or allocating library
// routine is called on this path.
//
// In host code `scratch` names a host-side stand-in, not a device address:
// the address of each device's copy is taken once per device with
// hipGetSymbolAddress (with that device current) and only that address is
// handed to kernels.
//
// Calls on one GPU share its scratch: two calls that overlap on one GPU (on
// different streams, or from different host threads) race. Every partial cell
// a call reads is written by the same call first, so nothing is carried over
// from an earlier call.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <mutex>

#include "../../include/mojoboost_hip.h"
#include "../../include/mojotrees.h"

namespace {

constexpr size_t kScratchBytes = (size_t)MBH_NOALLOC_SCRATCH_BYTES;
constexpr int kMaxDevices = 64;
constexpr int kThreads = 512;          // of a histogram block
constexpr int kMaxBlocks = 2048;       // row chunks of one call, at most
// Features a histogram block takes (its LDS histogram: 8 bytes per cell,
// 16 KB at 256 bins, so four blocks share a CU), and at most this many
// feature tiles (then a tile holds more features of fewer bins).
constexpr int kTileFeatures = 8;
constexpr int kMaxTiles = 1024;
// A call's rows are spread over about kTargetBlocks (row chunk, feature tile)
// blocks, in chunks of at least kMinChunk rows. Fewer chunks leave fewer
// partials to store and merge.
constexpr int kTargetBlocks = 1024;
constexpr int kMinChunk = 1024;
constexpr int kOldMinChunk = 2048;     // rows per chunk behind the size limit's wording (below)
constexpr int kMergeThreads = 256;
// Cells of a merge block, of kMergeThreads / kMergeCells threads each.
constexpr int kMergeCells = 32;
// From this many cells on, fewer partials than those threads are summed by a
// thread a cell (k_na_merge has both sides' figures).
constexpr int kMergeMany = 1 << 16;

__device__ __align__(256) unsigned char scratch[kScratchBytes];

std::mutex g_mu;
void *g_scratch[kMaxDevices] = {};

void set_err(char *err, int32_t len, const char *m) {
    if (err && len > 0) std::snprintf(err, (size_t)len, "%s", m);
}

// The device address of the current device's scratch, looked up once per
// device (hipGetSymbolAddress with that device current).
hipError_t device_scratch(void **out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_mu);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch[dev] = p;
    }
    *out = g_scratch[dev];
    return hipSuccess;
}

// Rows a block may pack into its 64-bit LDS counters (count in bits [0, 20),
// hessian sum in [20, 42), signed gradient sum in [42, 64)) before a field
// overflows, for |q_grad| <= B/2 + 1 and 0 <= q_hess <= B + 1.
int64_t chunk_limit(int B) {
    int64_t lim = (1 << 20) - 1;
    const int64_t h = ((1 << 22) - 1) / (B + 1);
    const int64_t g = ((1 << 21) - 1) / (B / 2 + 1);
    if (h < lim) lim = h;
    if (g < lim) lim = g;
    return lim;
}

__global__ void k_na_clear(int32_t *status) {
    if (status && threadIdx.x == 0 && blockIdx.x == 0) *status = 0;
}

// Block (x, y): rows [x * chunk, ...) of the selection, features
// [y * ft, y * ft + ft). A thread takes kU rows at a time: their ids and
// pairs first, then the bins of kG features of all of them, kU x kG loads in
// flight before the first is added (a load per feature and row, each waited
// for, bound this kernel by latency: 75 us for 500K of 1M rows x 28 at
// 255 bins, 16 us this way). Each bin adds a packed (grad, hess, 1) counter into
// the block's LDS histogram, whose every cell the block then writes as
// partial x. Entries that are out of range (a row id outside [0, n), a
// quantized pair outside the lattice, a bin id >= n_bins) are not added and
// flag *status.
template <bool kList>
__global__ __launch_bounds__(kThreads) void k_na_hist(const uint8_t *__restrict__ bins_cm, int64_t n, int F, int nb,
                                                     const int8_t *__restrict__ qg, const int8_t *__restrict__ qh,
                                                     const int32_t *__restrict__ rows, int64_t m, int64_t chunk,
                                                     int ft, int gmax, int hmax,
                                                     unsigned long long *__restrict__ part, int32_t *status) {
    constexpr int kU = 4, kG = 4;
    extern __shared__ unsigned long long lds[];
    const int f0 = (int)blockIdx.y * ft;
    const int nf = min(ft, F - f0);
    for (int i = threadIdx.x; i < nf * nb; i += kThreads) lds[i] = 0ULL;
    __syncthreads();
    const int64_t c0 = (int64_t)blockIdx.x * chunk;
    const int64_t c1 = c0 + chunk < m ? c0 + chunk : m;
    bool bad = false;
    for (int64_t i0 = c0 + threadIdx.x; i0 < c1; i0 += (int64_t)kU * kThreads) {
        int64_t r[kU];
        bool in[kU];
        unsigned long long packed[kU];
        // loads past the chunk repeat its last entry and are not added
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int64_t i = i0 + (int64_t)u * kThreads;
            in[u] = i < c1;
            const int64_t at = in[u] ? i : c1 - 1;
            r[u] = kList ? (int64_t)rows[at] : at;
        }
        int g[kU], h[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const bool ok = r[u] >= 0 && r[u] < n;
            bad |= in[u] && !ok;
            in[u] = in[u] && ok;
            r[u] = ok ? r[u] : 0;
            g[u] = qg[r[u]];
            h[u] = qh[r[u]];
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const bool ok = g[u] >= -gmax && g[u] <= gmax && h[u] >= 0 && h[u] <= hmax;
            bad |= in[u] && !ok;
            in[u] = in[u] && ok;
            packed[u] = (unsigned long long)(((long long)g[u] << 42) + ((long long)h[u] << 20) + 1LL);
        }
        for (int fg = 0; fg < nf; fg += kG) {
            int b[kG][kU];
#pragma unroll
            for (int k = 0; k < kG; ++k) {
                const int f = fg + k < nf ? fg + k : nf - 1;
                const uint8_t *col = bins_cm + (size_t)(f0 + f) * n;
#pragma unroll
                for (int u = 0; u < kU; ++u) b[k][u] = col[r[u]];
            }
#pragma unroll
            for (int k = 0; k < kG; ++k) {
                if (fg + k >= nf) break;
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    const bool ok = b[k][u] < nb;
                    bad |= in[u] && !ok;
                    if (in[u] && ok) atomicAdd(&lds[(fg + k) * nb + b[k][u]], packed[u]);
                }
            }
        }
    }
    if (bad && status) atomicOr(status, 1);
    __syncthreads();
    unsigned long long *out = part + ((size_t)blockIdx.x * F + f0) * nb;
    for (int i = threadIdx.x; i < nf * nb; i += kThreads) out[i] = lds[i];
}

// kCells (feature, bin) cells per block, each summed by several threads
// (thread t takes the partials t / kCells, + threads per cell, ..., four
// loads in flight), then over LDS: int32 {grad, hess, count}. One thread per
// cell walked every partial alone, 28 blocks in all for 28 x 255 cells
// (68 us; 5 us this way). Where the cells alone fill the chip and the
// partials are fewer than the threads, most of which would idle, a thread a
// cell: 2.05M cells, 1 partial: 25.7 -> 8.6 us; 1.02M, 2: 14.2 -> 7.0; 510K,
// 4: 8.4 -> 5.8 (7.7K cells, 6 partials: 2.3 against 3.2 us).
template <int kCells>
__global__ __launch_bounds__(kMergeThreads) void k_na_merge(const unsigned long long *__restrict__ part, int blocks,
                                                           int cells, int32_t *__restrict__ out) {
    constexpr int kPer = kMergeThreads / kCells;
    __shared__ int sum[3][kPer][kCells];
    const int lc = threadIdx.x % kCells, p = threadIdx.x / kCells;
    const int c = (int)blockIdx.x * kCells + lc;
    // int32 sums: the caller's rows x (B + 1) stay below 2^31
    int g = 0, h = 0, cnt = 0;
    auto add = [&](unsigned long long v) {
        cnt += (int)(v & 0xFFFFFULL);
        h += (int)((v >> 20) & 0x3FFFFFULL);
        g += (int)((long long)v >> 42);
    };
    if (c < cells) {
        int b = p;
        for (; b + 3 * kPer < blocks; b += 4 * kPer) {
            unsigned long long v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = part[(size_t)(b + u * kPer) * cells + c];
#pragma unroll
            for (int u = 0; u < 4; ++u) add(v[u]);
        }
        for (; b < blocks; b += kPer) add(part[(size_t)b * cells + c]);
    }
    sum[0][p][lc] = g;
    sum[1][p][lc] = h;
    sum[2][p][lc] = cnt;
    __syncthreads();
    // the block's 3 x kCells outputs, consecutive in memory
    for (int i = threadIdx.x; i < 3 * kCells; i += kMergeThreads) {
        const int cell = i / 3, k = i - 3 * cell;
        if ((int)blockIdx.x * kCells + cell >= cells) break;
        int v = 0;
        for (int q = 0; q < kPer; ++q) v += sum[k][q][cell];
        out[(size_t)3 * blockIdx.x * kCells + i] = v;
    }
}

}  // namespace

extern "C" int32_t mbh_histogram_noalloc(const uint8_t *bins_cm, int64_t n_rows, int32_t n_features,
                                         int32_t n_bins, const int8_t *q_grad, const int8_t *q_hess,
                                         const int32_t *rows, int64_t n_sel, int32_t B, int32_t *out,
                                         int32_t *status, void *stream, char *err, int32_t err_len) {
    if (!bins_cm || !q_grad || !q_hess || !out || n_rows <= 0 || n_features <= 0 || n_bins < 2 ||
        n_bins > 256 || (rows && n_sel <= 0)) {
        set_err(err, err_len, "invalid arguments");
        return MOJOTREES_ERROR_INVALID_ARGUMENT;
    }
    if (n_rows >= ((int64_t)1 << 31)) {
        set_err(err, err_len, "n_rows must be below 2^31");
        return MOJOTREES_ERROR_INVALID_ARGUMENT;
    }
    if (B < 2 || B > 126 || B % 2 != 0) {
        set_err(err, err_len, "num_grad_quant_bins must be even and in [2, 126]");
        return MOJOTREES_ERROR_INVALID_ARGUMENT;
    }
    const int64_t m = rows ? n_sel : n_rows;
    if ((double)m * (double)(B + 1) >= 2147483647.0) {
        set_err(err, err_len, "rows * (num_grad_quant_bins + 1) must stay below 2^31 for int32 histogram cells");
        return MOJOTREES_ERROR_INVALID_ARGUMENT;
    }
    // one partial in 64-bit arithmetic, checked before anything divides by
    // it or narrows the cell count (n_features * n_bins may exceed int)
    const int64_t cells64 = (int64_t)n_features * (int64_t)n_bins;
    const uint64_t partial_bytes = (uint64_t)cells64 * sizeof(unsigned long long);
    if (partial_bytes > (uint64_t)kScratchBytes) {
        set_err(err, err_len,
                "n_features * n_bins exceeds the no-alloc scratch (one partial of 8 bytes per cell must fit "
                "MBH_NOALLOC_SCRATCH_BYTES)");
        return MOJOTREES_ERROR_INVALID_ARGUMENT;
    }
    const int cells = (int)cells64;  // at most kScratchBytes / 8 after the check
    int max_blocks = (int)(kScratchBytes / partial_bytes);
    if (max_blocks > kMaxBlocks) max_blocks = kMaxBlocks;
    const int64_t limit = chunk_limit(B);
    // refused when even max_blocks chunks (no fewer rows each than the size
    // rule has always granted) pack more rows than the counters hold
    const int64_t most = (m + kOldMinChunk - 1) / kOldMinChunk < max_blocks ? (m + kOldMinChunk - 1) / kOldMinChunk
                                                                            : (int64_t)max_blocks;
    if ((m + most - 1) / most > limit) {
        set_err(err, err_len,
                "selection too large for the no-alloc scratch at this n_features * n_bins "
                "(the packed block counters would overflow)");
        return MOJOTREES_ERROR_INVALID_ARGUMENT;
    }
    int tiles = (n_features + kTileFeatures - 1) / kTileFeatures;
    if (tiles > kMaxTiles) tiles = kMaxTiles;
    const int ft = (n_features + tiles - 1) / tiles;
    tiles = (n_features + ft - 1) / ft;
    const int64_t want = kTargetBlocks / tiles > 1 ? kTargetBlocks / tiles : 1;
    int64_t chunk = (m + want - 1) / want;
    if (chunk < kMinChunk) chunk = kMinChunk;
    if (chunk < (m + max_blocks - 1) / max_blocks) chunk = (m + max_blocks - 1) / max_blocks;
    if (chunk > limit) chunk = limit;  // never below m / max_blocks: refused above
    const int64_t blocks = (m + chunk - 1) / chunk;
    void *sp = nullptr;
    hipError_t e = device_scratch(&sp);
    if (e != hipSuccess) {
        set_err(err, err_len, hipGetErrorString(e));
        return MOJOTREES_ERROR_TRAINING;
    }
    auto *part = (unsigned long long *)sp;
    hipStream_t st = (hipStream_t)stream;
    if (status) hipLaunchKernelGGL(k_na_clear, dim3(1), dim3(64), 0, st, status);
    hipLaunchKernelGGL(rows ? k_na_hist<true> : k_na_hist<false>, dim3((unsigned)blocks, (unsigned)tiles),
                       dim3(kThreads), (size_t)ft * n_bins * sizeof(unsigned long long), st, bins_cm, n_rows,
                       (int)n_features, (int)n_bins, q_grad, q_hess, rows, m, chunk, ft, B / 2 + 1, B + 1, part,
                       status);
    const bool single = cells >= kMergeMany && blocks < kMergeThreads / kMergeCells;
    const int mc = single ? kMergeThreads : kMergeCells;
    hipLaunchKernelGGL(single ? k_na_merge<kMergeThreads> : k_na_merge<kMergeCells>,
                       dim3((unsigned)((cells + mc - 1) / mc)), dim3(kMergeThreads), 0, st,
                       (const unsigned long long *)part, (int)blocks, cells, out);
    e = hipGetLastError();
    if (e != hipSuccess) {
        set_err(err, err_len, hipGetErrorString(e));
        return MOJOTREES_ERROR_TRAINING;
    }
    return MOJOTREES_OK;
}
