// Launchers for the kernels in mb_kernels.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "mb_state.h"

namespace mb {

hipError_t launch_objective(const DevState &s, int grid, hipStream_t st);
hipError_t launch_softmax(const DevState &s, int grid, hipStream_t st);
// The GOSS selection of the round (no-ops before the warmup ends).
hipError_t launch_goss(const DevState &s, int grid, hipStream_t st);
// max |g|, |h| of the round's weighted GOSS sample (quantized gradients,
// between launch_goss and launch_quantize).
hipError_t launch_goss_stats(const DevState &s, int grid, hipStream_t st);
// The magnitude-sum lattice's reduction and scales (before launch_quantize).
hipError_t launch_magnitude(const DevState &s, hipStream_t st);
// write_pairs = false leaves the max-abs int8 pairs to launch_hist(quantize).
hipError_t launch_quantize(const DevState &s, int grid, hipStream_t st, bool write_pairs = true);
// Raises the dynamic LDS limits of the kernels that need more than 64 KB.
hipError_t prepare_kernels(const DevState &s);
size_t hist_lds_bytes(const DevState &s);
// histogram accumulators: packed int8-lattice counters, fp64 sums of fp32
// gradients, int32 sums of the magnitude-sum lattice
enum AccKind { kAccQuant = 0, kAccFloat = 1, kAccWide = 2 };
inline int acc_kind(const HyperParams &hp) { return hp.wide ? kAccWide : hp.quantized ? kAccQuant : kAccFloat; }
// accumulation LDS of a tile of tile_f features
size_t pb_lds_bytes_for(int tile_f, int lds_stride, int kind);
size_t plan_lds_bytes(const DevState &s);
// Whether the planner can grow s's trees (its dynamic and own LDS, its slots).
hipError_t planner_fits(const DevState &s, bool *fits);
size_t score_lds_bytes(const DevState &s);
size_t rank_lds_bytes(const DevState &s);
// With both events given, the runtime records them at the kernel's own start
// and end (for timing without queue gaps).
// quantize: the root build quantizes the rows it reads and writes their
// pairs into the records (max-abs lattice only; other kinds ignore it).
hipError_t launch_hist(const DevState &s, hipStream_t st, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr,
                       bool quantize = false);
hipError_t launch_partition(const DevState &s, hipStream_t st, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr,
                            bool root = false);
hipError_t launch_accum(const DevState &s, hipStream_t st, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);
hipError_t launch_scan(const DevState &s, int root_mode, hipStream_t st);
hipError_t launch_plan(const DevState &s, int root_mode, hipStream_t st, Batch *host = nullptr);
hipError_t launch_score(const DevState &s, int grid, hipStream_t st);
// The score update fused with the next round's objective (single-output L2
// and binary): after it, the next tree skips launch_objective.
hipError_t launch_score_objective(const DevState &s, int grid, hipStream_t st);
hipError_t launch_round_end(const DevState &s, hipStream_t st);
hipError_t launch_round_end_quantize(const DevState &s, hipStream_t st);
hipError_t launch_round_combine(const RoundStates &rs, int sampling, hipStream_t st);
// Grid of a grid-stride rows kernel: as many blocks per CU as its registers
// and LDS let stay resident (at most 8), times n_cu, so that every block runs
// from the start instead of a partial second round of blocks following the
// first.
enum RowsKernel { kRowsScore = 0, kRowsScoreObjective = 1, kRowsSoftmax = 2 };
int rows_grid(const DevState &s, RowsKernel k, int n_cu);
hipError_t launch_build_records(const uint8_t *bins_cm, uint8_t *records, int64_t n, int F, int rec,
                                int tile_f, int n_tiles, int grid, hipStream_t st);
// n x K row-major from class-major scores.
hipError_t launch_row_major(const double *in, double *out, int64_t n, int K, hipStream_t st);
// Buffers of an arena (aligned, and padded to 256 bytes) that a call's start
// zeroes, in one launch: a hipMemset each took 12 us of the host in a slab,
// 12 of them a call.
struct ZeroList {
    static constexpr int kMost = 24;
    uint4 *p[kMost];
    uint64_t words[kMost];  // of 16 bytes
    int n = 0;
    void add(void *at, size_t bytes) {
        if (n < kMost) {
            p[n] = (uint4 *)at;
            words[n] = (bytes + 15) / 16;
        }
        ++n;  // past kMost: the launch is refused
    }
};
hipError_t launch_zero(const ZeroList &z, int n_cu, hipStream_t st);
hipError_t launch_fill_f64(double *p, int64_t n, int K, const double *base, int grid, hipStream_t st);
hipError_t launch_exp_sigmoid(const double *x, double *e, double *sg, int64_t n, hipStream_t st);

}  // namespace mb
