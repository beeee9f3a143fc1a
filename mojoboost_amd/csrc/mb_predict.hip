// mbh_predict_binned: raw scores of a flat ensemble from column-major bins
// (Tree.predict_row, src/mojotrees/tree.mojo:483-505; Booster.predict_raw_row,
// src/mojotrees/boosting.mojo:1722-1760). A row's bin for a node's feature:
// the missing bin follows the default direction, otherwise bin <= threshold
// goes left. The class's trees are added in ascending order as
// fma(learning_rate, value, score), the host predictor's fused update, so the
// scores are its bits.
//
// Blocks of 512 threads walk trees held in LDS over rows whose bins are held
// in LDS. A block takes RB rows of one class (a power of two) and goes through
// the class's trees a chunk of at most kChunkWords words at a time. A node is
// one 64-bit word (below) that names the byte its split reads and its left
// child's place, the right child next to it, so a step of a walk is two LDS
// reads and about a dozen vector instructions.
//   k_predict_rows (large inputs): a row per thread, taken through the chunk's
//     trees on its own -- a leaf names the next tree's root -- so lanes wait for
//     one another once per chunk and not once per tree, and adds each leaf as
//     it reaches it. Bound by instruction issue.
//   k_predict_wide (fewer rows): RB rows x 512 / RB trees walked side by
//     side, kU trees per thread in step; the leaves go to LDS and one thread
//     per row adds them in tree order, so the sums are the same bits.
// A thread per row chasing 16-byte nodes and record bytes through the caches,
// as before, was bound by that chain's latency (two blocks on the whole chip
// for 501 rows): 1M rows x 200 trees of 255 leaves 6525 us, now 1080;
// 501 rows x 100 trees of 31 leaves 488 us, now 27.
//
// Trees of more words than a chunk, trees that reach a node twice (files may
// hold both) and more features than a word names take k_predict, the plain walk
// over global memory.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/mojoboost_hip.h"
#include "../../include/mojotrees.h"
#include "mb_memory.h"
#include "mb_trees.h"

namespace {

using namespace mb::trees;

constexpr int kThreads = 512;
constexpr int kU = 4;            // trees a thread of k_predict_wide walks at once
constexpr int kTreeCap = 256;    // trees of a chunk
constexpr int kLeafCap = 4096;   // k_predict_wide: rows x trees of leaf values in LDS (32 KB)
constexpr size_t kBinBudget = 64 * 1024;  // LDS of a block's bins
constexpr int kMinRows = 4;      // rows of a block, at least
// k_predict_rows needs this many blocks to fill the chip; below, rows are
// split until about as many blocks of k_predict_wide share the work (each
// stages every tree of its class once, so not more).
constexpr int kBlocksTarget = 512;
// Of a matrix in several batches, columns of at least kLongColumn rows are
// copied each on its own, shorter ones gathered kStageBytes at a time: a copy
// costs some 9 us beside its bytes. 200K rows x 20,000 (columns of 107K and
// 93K) 441 ms on their own, 213 gathered; 24K x 100,000 1900 and 141; 2.2M x
// 1,000 89 and 150.
constexpr int64_t kLongColumn = 1 << 18;
constexpr int64_t kStageBytes = (int64_t)16 << 20;

struct PredictArgs {
    const uint8_t *bins;  // F x n, column-major
    int64_t n;
    int32_t F, K;
    double learning_rate;
    const double *base;   // K scores, or null
    double *out;          // n x K
    const unsigned long long *cat;  // 4 words per node, or null
    // the chunks' words, per tree (class-major) its root's byte offset in
    // its chunk, the chunks, those of class k at [chunk_of[k], chunk_of[k + 1])
    const unsigned long long *words;
    const uint32_t *tree;
    const Chunk *chunk;
    const int32_t *chunk_of;
    int32_t log_rows;     // log2 RB
    // k_predict
    const int4 *nodes;    // {feature (-1: leaf), threshold, left, right}, absolute
    const int32_t *md;    // missing_bin * 2 + default_left
    const double *value;
    const int32_t *root;  // per tree
    int64_t n_trees;
    int32_t max_steps;    // nodes of the largest tree: no walk is longer
};

__global__ __launch_bounds__(256) void k_predict(PredictArgs a) {
    const int k = blockIdx.y;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < a.n; r += stride) {
        double acc = a.base ? a.base[k] : 0.0;
        for (int64_t t = k; t < a.n_trees; t += a.K) {
            int node = a.root[t];
            int4 nd = a.nodes[node];
            // children have larger indices than their parent (host-checked),
            // so a walk ends within the tree's node count
            for (int d = 0; nd.x >= 0 && d < a.max_steps; ++d) {
                const int b = a.bins[(size_t)nd.x * a.n + r];
                const int md = a.md[node];
                const bool left = nd.y < 0 ? ((a.cat[(size_t)node * 4 + (b >> 6)] >> (b & 63)) & 1ULL) != 0
                                           : (b == (md >> 1)) ? (md & 1) : (b <= nd.y);
                node = left ? nd.z : nd.w;
                nd = a.nodes[node];
            }
            acc = fma(a.learning_rate, a.value[node], acc);
        }
        a.out[r * a.K + k] = acc;
    }
}

// The block's bins: four features of a row in a 32-bit word, rows
// consecutive, so a wave's reads fall on the lanes' own banks whatever the
// features. Rows past the end repeat the last one.
__device__ __forceinline__ void stage_bins(const PredictArgs &a, uint32_t *bins, int64_t r0, int lg) {
    const int FD = (a.F + 3) >> 2;
    for (int i = threadIdx.x; i < FD << lg; i += kThreads) {
        const int q = i >> lg, l = i & ((1 << lg) - 1);
        const int64_t r = r0 + l < a.n ? r0 + l : a.n - 1;
        uint32_t w = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int f = 4 * q + j < a.F ? 4 * q + j : a.F - 1;
            w |= (uint32_t)a.bins[(size_t)f * a.n + r] << (8 * j);
        }
        bins[i] = w;
    }
}

__device__ __forceinline__ void stage_words(const PredictArgs &a, const Chunk &ch, unsigned long long *words) {
    __syncthreads();  // the chunk before is done with
    for (int i = threadIdx.x; i < ch.n_words; i += kThreads) words[i] = a.words[(size_t)ch.word0 + i];
    __syncthreads();
}

// One step from inner node w at byte offset `at` of the chunk: the child's
// offset. row4: 4 x the row's place in the block (bins in LDS); row: its
// place in the matrix (bins in global memory).
template <bool kLdsBins, bool kMiss, bool kCat>
__device__ __forceinline__ uint32_t step(const PredictArgs &a, const unsigned char *bins, const Chunk &ch,
                                         unsigned long long w, uint32_t at, uint32_t row4, int64_t row) {
    const uint32_t lo = (uint32_t)w, hi = (uint32_t)(w >> 32);
    uint32_t b;
    if constexpr (kLdsBins) b = bins[(lo >> 16) + row4];
    else b = a.bins[(size_t)(lo >> 16) * a.n + row];
    bool left = b <= (hi & 255u);
    if constexpr (kMiss) left = b == ((hi >> 8) & 511u) ? (hi & kDefLeft) != 0 : left;
    if constexpr (kCat)
        if (hi & kCatNode)
            left = ((a.cat[((size_t)ch.node0 + (at >> 3)) * 4 + (b >> 6)] >> (b & 63u)) & 1ULL) != 0;
    return (lo & 0xFFFFu) + (left ? 0u : 8u);
}

// kLdsBins: the rows' bins are staged in LDS (else more features than
// kBinBudget takes: read from global memory). kMiss: some node has a
// missing bin. kCat: the ensemble has category sets.
template <bool kLdsBins, bool kMiss, bool kCat>
__global__ __launch_bounds__(kThreads) void k_predict_rows(PredictArgs a) {
    extern __shared__ unsigned long long lds[];
    const int tid = threadIdx.x, k = blockIdx.y, lg = a.log_rows;  // 2^lg == kThreads
    const int64_t r0 = (int64_t)blockIdx.x << lg;
    const int64_t row = r0 + tid < a.n ? r0 + tid : a.n - 1;
    const unsigned char *wb = (const unsigned char *)lds;
    unsigned char *bins = (unsigned char *)(lds + kChunkWords);
    if constexpr (kLdsBins) stage_bins(a, (uint32_t *)bins, r0, lg);
    double acc = a.base ? a.base[k] : 0.0;
    for (int c = a.chunk_of[k]; c < a.chunk_of[k + 1]; ++c) {
        const Chunk ch = a.chunk[c];
        stage_words(a, ch, lds);
        uint32_t at = 0;  // the first tree's root
        while (at != kEnd) {
            const unsigned long long w = *(const unsigned long long *)(wb + at);
            const uint32_t lo = (uint32_t)w;
            if ((uint32_t)(w >> 32) & kLeaf) {
                acc = fma(a.learning_rate, *(const double *)(wb + (lo >> 16)), acc);
                at = lo & 0xFFFFu;
            } else {
                at = step<kLdsBins, kMiss, kCat>(a, bins, ch, w, at, 4u * tid, row);
            }
        }
    }
    if (r0 + tid < a.n) a.out[row * a.K + k] = acc;
}

template <bool kLdsBins, bool kMiss, bool kCat>
__global__ __launch_bounds__(kThreads) void k_predict_wide(PredictArgs a) {
    extern __shared__ unsigned long long lds[];
    __shared__ uint32_t s_tree[kTreeCap];
    const int tid = threadIdx.x, k = blockIdx.y;
    const int lg = a.log_rows, TG = kThreads >> lg;
    const int lr = tid & ((1 << lg) - 1), tg = tid >> lg;
    const int64_t r0 = (int64_t)blockIdx.x << lg;
    const int64_t row = r0 + lr < a.n ? r0 + lr : a.n - 1;
    const unsigned char *wb = (const unsigned char *)lds;
    double *leafs = (double *)(lds + kChunkWords);
    unsigned char *bins = (unsigned char *)(lds + kChunkWords + kLeafCap);
    if constexpr (kLdsBins) stage_bins(a, (uint32_t *)bins, r0, lg);
    double acc = a.base ? a.base[k] : 0.0;
    for (int c = a.chunk_of[k]; c < a.chunk_of[k + 1]; ++c) {
        const Chunk ch = a.chunk[c];
        stage_words(a, ch, lds);
        for (int i = tid; i < ch.n_trees; i += kThreads) s_tree[i] = a.tree[ch.tree0 + i];
        __syncthreads();
        for (int t0 = tg; t0 < ch.n_trees; t0 += kU * TG) {
            uint32_t at[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) at[u] = s_tree[t0 + u * TG < ch.n_trees ? t0 + u * TG : t0];
            unsigned long long w[kU];
            for (;;) {
                bool all = true;
#pragma unroll
                for (int u = 0; u < kU; ++u) w[u] = *(const unsigned long long *)(wb + at[u]);
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    if ((uint32_t)(w[u] >> 32) & kLeaf) continue;
                    all = false;
                    at[u] = step<kLdsBins, kMiss, kCat>(a, bins, ch, w[u], at[u], 4u * lr, row);
                }
                if (all) break;
            }
#pragma unroll
            for (int u = 0; u < kU; ++u)
                if (t0 + u * TG < ch.n_trees)
                    leafs[((t0 + u * TG) << lg) + lr] = *(const double *)(wb + ((uint32_t)w[u] >> 16));
        }
        __syncthreads();
        if (tg == 0) {
            int t = 0;
            for (; t + 8 <= ch.n_trees; t += 8) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = leafs[((t + u) << lg) + lr];
#pragma unroll
                for (int u = 0; u < 8; ++u) acc = fma(a.learning_rate, v[u], acc);
            }
            for (; t < ch.n_trees; ++t) acc = fma(a.learning_rate, leafs[(t << lg) + lr], acc);
        }
    }
    if (tg == 0 && r0 + lr < a.n) a.out[(r0 + lr) * a.K + k] = acc;
}

struct Error {
    int32_t code;
    std::string msg;
};

#define HIPP(expr)                                                                           \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess)                                                                \
            throw Error{MOJOTREES_ERROR_TRAINING,                                            \
                        std::string("HIP error in ") + #expr + ": " + hipGetErrorString(e_)}; \
    } while (0)

struct DeviceBlock {
    uint8_t *p = nullptr;
    ~DeviceBlock() {
        if (p) (void)hipFree(p);
    }
};

size_t up(size_t b) { return (b + 255) & ~(size_t)255; }

// The host's image of everything but the bins and the scores, uploaded as
// one copy; parts are placed at 256-byte offsets and written in place (memory
// of a call's own: zeroing it and copying the parts together cost a few
// milliseconds per million nodes).
struct Image {
    std::unique_ptr<uint8_t[]> bytes;
    size_t size = 0, room = 0;
    // at most `total` bytes in `parts` parts
    Image(size_t total, int parts) : bytes(new uint8_t[total + (size_t)parts * 256]), room(total + (size_t)parts * 256) {}
    template <class T>
    T *part(size_t count, size_t &at) {
        at = up(size);
        size = at + count * sizeof(T);
        if (size > room) throw Error{MOJOTREES_ERROR_TRAINING, "internal: prediction image"};
        return (T *)(bytes.get() + at);
    }
    template <class T>
    size_t put(const T *src, size_t count) {
        size_t at;
        T *to = part<T>(count, at);
        if (count) std::memcpy(to, src, count * sizeof(T));
        return at;
    }
};

using Kernel = void (*)(PredictArgs);

template <bool kLdsBins, bool kMiss, bool kCat>
Kernel pick(bool rows) {
    return rows ? k_predict_rows<kLdsBins, kMiss, kCat> : k_predict_wide<kLdsBins, kMiss, kCat>;
}

// The matrix in global memory and category sets are rare enough to share
// the form that also looks for missing bins.
Kernel pick_kernel(bool rows, bool lds_bins, bool miss, bool cat) {
    if (!lds_bins) return cat ? pick<false, true, true>(rows) : pick<false, true, false>(rows);
    if (cat) return pick<true, true, true>(rows);
    return miss ? pick<true, true, false>(rows) : pick<true, false, false>(rows);
}

}  // namespace

extern "C" int32_t mbh_predict_binned(const uint8_t *bins_cm, int64_t n, int32_t F, int32_t num_class,
                                      double learning_rate, const double *base, const int64_t *node_offset,
                                      int64_t tree_begin, int64_t tree_end, const int32_t *feature,
                                      const int32_t *threshold, const int32_t *left, const int32_t *right,
                                      const double *value, const int32_t *default_left, const int32_t *missing_bin,
                                      const uint64_t *cat_bits, double *out, char *err, int32_t err_len) {
    auto fail = [&](int32_t code, const char *m) {
        if (err && err_len > 0) std::snprintf(err, (size_t)err_len, "%s", m);
        return code;
    };
    if (!bins_cm || !node_offset || !feature || !threshold || !left || !right || !value || !default_left ||
        !missing_bin || !out || n <= 0 || F <= 0 || num_class <= 0 || tree_begin < 0 || tree_end < tree_begin ||
        tree_begin % num_class != 0)
        return fail(MOJOTREES_ERROR_INVALID_ARGUMENT, "invalid prediction arguments");
    if (mbh_device_count() == 0)
        return fail(MOJOTREES_ERROR_UNSUPPORTED, "no gfx950 (MI355X) device is available to this process");
    try {
        const int K = num_class;
        const Trees e{node_offset, tree_begin, tree_end, feature, threshold, left, right, value, default_left,
                      missing_bin, cat_bits};
        const Shapes shapes = check_trees(e, F);
        // row batches bound the device copy of the matrix
        const int64_t per_row = (int64_t)F + 8 * K;
        const int64_t batch = std::max<int64_t>(4096, std::min<int64_t>(n, ((int64_t)1 << 31) / per_row));
        const int64_t m0 = std::min(batch, n);
        // a row per thread where that fills the chip; else the block's rows
        // are halved until about kBlocksTarget blocks share a batch; then
        // until their bins fit the LDS budget
        static_assert(kThreads == 512 && kMinRows == 4, "log2 of a block's rows: 9 .. 2");
        const size_t row_bytes = (size_t)((F + 3) / 4) * 4;
        const bool lds_bins = row_bytes * kMinRows <= kBinBudget;
        auto blocks = [&](int l) { return ((m0 + ((int64_t)1 << l) - 1) >> l) * K; };
        int lg = 9;
        const bool rows = blocks(lg) >= kBlocksTarget && (!lds_bins || (row_bytes << lg) <= kBinBudget);
        if (!rows)
            do --lg;
            while (lg > 2 && (blocks(lg) < kBlocksTarget || (lds_bins && (row_bytes << lg) > kBinBudget)));
        PredictArgs a{};
        a.F = F;
        a.K = K;
        a.learning_rate = learning_rate;
        a.log_rows = lg;
        const int64_t T = tree_end - tree_begin, o0 = node_offset[tree_begin], nn = node_offset[tree_end] - o0;
        const size_t cat_words = cat_bits ? (size_t)nn * 4 : 0;
        size_t o_base = 0, o_cat = 0, o_words = 0, o_tree = 0, o_chunk = 0, o_of = 0, o_nodes = 0, o_md = 0,
               o_value = 0, o_root = 0;
        auto place = [&](int32_t f) { return lds_bins ? (uint32_t)(((f >> 2) << (lg + 2)) + (f & 3)) : (uint32_t)f; };
        std::unique_ptr<Image> im;
        Packed p;
        bool packed = false;
        if (F <= 65536 && chunks_hold(shapes)) {
            im.reset(new Image((size_t)shapes.words * 8 + cat_words * 8 + (size_t)T * (4 + sizeof(Chunk)) +
                                   (size_t)K * 12 + 4, 6));
            unsigned long long *words = im->part<unsigned long long>((size_t)shapes.words, o_words);
            unsigned long long *cat = cat_bits ? im->part<unsigned long long>(cat_words, o_cat) : nullptr;
            packed = pack_trees(e, shapes, K, rows ? kTreeCap : std::min(kTreeCap, kLeafCap >> lg), place, words, cat, p);
        }
        if (packed) {
            o_tree = im->put(p.tree.data(), p.tree.size());
            o_chunk = im->put(p.chunk.data(), p.chunk.size());
            o_of = im->put(p.chunk_of.data(), p.chunk_of.size());
        } else {
            im.reset(new Image((size_t)nn * (sizeof(int4) + 4 + 8) + cat_words * 8 + (size_t)T * 4 + (size_t)K * 8, 6));
            int4 *nodes = im->part<int4>((size_t)nn, o_nodes);
            int32_t *md = im->part<int32_t>((size_t)nn, o_md), *root = im->part<int32_t>((size_t)T, o_root);
            for (int64_t t = tree_begin; t < tree_end; ++t) {
                const int64_t first = node_offset[t] - o0;
                root[t - tree_begin] = (int32_t)first;
                for (int64_t i = node_offset[t]; i < node_offset[t + 1]; ++i) {
                    nodes[i - o0] = make_int4(feature[i] >= 0 ? feature[i] : -1, threshold[i],
                                              (int32_t)(first + left[i]), (int32_t)(first + right[i]));
                    md[i - o0] = missing_bin[i] * 2 + (default_left[i] ? 1 : 0);
                }
            }
            o_value = im->put(value + o0, (size_t)nn);
            if (cat_bits) o_cat = im->put(cat_bits + (size_t)o0 * 4, cat_words);
        }
        if (base) o_base = im->put(base, (size_t)K);
        const size_t at_bins = up(im->size), at_out = at_bins + up((size_t)F * m0);
        DeviceBlock d;
        HIPP(mb::device_malloc((void **)&d.p, at_out + (size_t)m0 * K * sizeof(double)));
        if (im->size) HIPP(hipMemcpyAsync(d.p, im->bytes.get(), im->size, hipMemcpyHostToDevice, 0));
        a.bins = d.p + at_bins;
        a.out = (double *)(d.p + at_out);
        a.base = base ? (const double *)(d.p + o_base) : nullptr;
        a.cat = cat_bits ? (const unsigned long long *)(d.p + o_cat) : nullptr;
        a.words = (const unsigned long long *)(d.p + o_words);
        a.tree = (const uint32_t *)(d.p + o_tree);
        a.chunk = (const Chunk *)(d.p + o_chunk);
        a.chunk_of = (const int32_t *)(d.p + o_of);
        a.nodes = (const int4 *)(d.p + o_nodes);
        a.md = (const int32_t *)(d.p + o_md);
        a.value = (const double *)(d.p + o_value);
        a.root = (const int32_t *)(d.p + o_root);
        a.n_trees = T;
        a.max_steps = shapes.largest;
        const size_t lds = (size_t)kChunkWords * 8 + (rows ? 0 : (size_t)kLeafCap * 8) + (lds_bins ? row_bytes << lg : 0);
        const Kernel kernel = pick_kernel(rows, lds_bins, p.missing, cat_bits != nullptr);
        if (packed)
            HIPP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        std::unique_ptr<uint8_t[]> stage;
        for (int64_t r0 = 0; r0 < n; r0 += batch) {
            const int64_t m = std::min(batch, n - r0);
            a.n = m;
            // one batch is the caller's matrix as it lies; of several, each
            // column's part
            if (m == n) {
                HIPP(hipMemcpyAsync(d.p + at_bins, bins_cm, (size_t)F * m, hipMemcpyHostToDevice, 0));
            } else if (m >= kLongColumn) {
                HIPP(hipMemcpy2DAsync(d.p + at_bins, m, bins_cm + r0, n, m, F, hipMemcpyHostToDevice, 0));
            } else {
                const int64_t cols = std::max<int64_t>(1, std::min<int64_t>(F, kStageBytes / m));
                if (!stage) stage.reset(new uint8_t[(size_t)std::max<int64_t>(kStageBytes, m)]);
                for (int64_t f0 = 0; f0 < F; f0 += cols) {
                    const int64_t nf = std::min<int64_t>(cols, F - f0);
                    for (int64_t f = 0; f < nf; ++f)
                        std::memcpy(stage.get() + f * m, bins_cm + (size_t)(f0 + f) * n + r0, (size_t)m);
                    HIPP(hipMemcpy(d.p + at_bins + (size_t)f0 * m, stage.get(), (size_t)(nf * m), hipMemcpyHostToDevice));
                }
            }
            if (!packed) {
                const int grid = (int)std::min<int64_t>((m + 255) / 256, 4096);
                hipLaunchKernelGGL(k_predict, dim3(grid, K), dim3(256), 0, 0, a);
            } else {
                const int64_t gx = (m + ((int64_t)1 << lg) - 1) >> lg;
                hipLaunchKernelGGL(kernel, dim3((unsigned)gx, (unsigned)K), dim3(kThreads), lds, 0, a);
            }
            HIPP(hipGetLastError());
            HIPP(hipMemcpy(out + r0 * K, a.out, (size_t)m * K * sizeof(double), hipMemcpyDeviceToHost));
        }
    } catch (const Error &e) {
        return fail(e.code, e.msg.c_str());
    } catch (const BadTrees &e) {
        return fail(MOJOTREES_ERROR_INVALID_ARGUMENT, e.what());
    } catch (const std::exception &e) {
        return fail(MOJOTREES_ERROR_TRAINING, e.what());
    }
    return MOJOTREES_OK;
}
