// The host side of batch prediction: the trees of a flat ensemble, checked and
// packed into the chunks that mb_predict.hip's kernels walk.
#pragma once

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <stdexcept>
#include <vector>

namespace mb {
namespace trees {

// Words of a chunk: nodes, then leaf values (24 KB of LDS, and room for a
// tree of 1024 leaves: 2047 nodes and 1024 values).
constexpr int kChunkWords = 3072;

// A node's word. Low half: bits 0-15 the left child's byte offset in the
// chunk (the right child's is 8 more), 16-31 the feature's place: the byte
// offset of its bin for the block's row 0 (bins in LDS), or the feature
// itself (bins in global memory). High half: bits 0-7 the threshold (a bin <=
// it goes left), 8-16 the missing bin (kNoBin: none), then the flags. A leaf:
// kLeaf, bits 16-31 its value's byte offset in the chunk, 0-15 the next
// tree's root (kEnd: none in the chunk).
constexpr uint32_t kNoBin = 256;
constexpr uint32_t kDefLeft = 1u << 17;
constexpr uint32_t kCatNode = 1u << 18;    // routes by its category set
constexpr uint32_t kLeaf = 1u << 31;
constexpr uint32_t kEnd = 0xFFFF;

struct Chunk {
    int32_t tree0, n_trees;
    int32_t word0, n_words;  // its words, nodes first
    int32_t node0, pad_;     // its first node among all nodes (category sets)
};

struct BadTrees : std::invalid_argument {
    using std::invalid_argument::invalid_argument;
};

// The ensemble as the caller laid it out (include/mojoboost_hip.h).
struct Trees {
    const int64_t *off;
    int64_t t0, t1;
    const int32_t *feature, *threshold, *left, *right;
    const double *value;
    const int32_t *default_left, *missing_bin;
    const uint64_t *cat_bits;
};

// What one pass over the trees finds: the nodes of the largest one, the words
// of the largest and of all (a word a node and one a leaf), and of each its
// leaves and whether every right child follows its left one (the trainer's
// order, which the chunks keep).
struct Shapes {
    int32_t largest = 1;
    int64_t most_words = 0, words = 0;
    std::vector<int32_t> leaves;
    std::vector<uint8_t> paired;
};

// Node offsets in order, children after their parents and within their
// tree (so that every walk ends), features in range, sets where needed.
inline Shapes check_trees(const Trees &e, int32_t F) {
    const int64_t o0 = e.off[e.t0], o1 = e.off[e.t1], nn = o1 - o0;
    if (nn < 0 || nn >= ((int64_t)1 << 31)) throw BadTrees("invalid node offsets");
    Shapes s;
    s.leaves.resize((size_t)(e.t1 - e.t0));
    s.paired.resize((size_t)(e.t1 - e.t0));
    for (int64_t t = e.t0; t < e.t1; ++t) {
        const int64_t a = e.off[t], b = e.off[t + 1];
        if (b <= a || a < o0 || b > o1) throw BadTrees("invalid node offsets");
        s.largest = std::max<int32_t>(s.largest, (int32_t)(b - a));
        int32_t leaves = 0;
        bool paired = true;
        for (int64_t i = a; i < b; ++i) {
            if (e.feature[i] < 0) {
                ++leaves;
                continue;
            }
            const int64_t loc = i - a;
            if (e.feature[i] >= F || e.left[i] <= loc || e.right[i] <= loc || e.left[i] >= b - a ||
                e.right[i] >= b - a)
                throw BadTrees("malformed tree: a child index must exceed its parent's");
            // a node without a threshold is categorical and routes by its set
            if (e.threshold[i] < 0 && !e.cat_bits) throw BadTrees("a categorical node needs its category set (cat_bits)");
            paired = paired && e.right[i] == e.left[i] + 1;
        }
        s.leaves[(size_t)(t - e.t0)] = leaves;
        s.paired[(size_t)(t - e.t0)] = paired;
        s.most_words = std::max(s.most_words, b - a + leaves);
        s.words += b - a + leaves;
    }
    return s;
}

// Whether every tree fits a chunk (and a word's place its 32 bits).
inline bool chunks_hold(const Shapes &s) { return s.most_words <= kChunkWords && s.words < ((int64_t)1 << 31); }

// The ensemble in chunks, beside their words.
struct Packed {
    std::vector<uint32_t> tree;
    std::vector<Chunk> chunk;
    std::vector<int32_t> chunk_of;
    bool missing = false;
};

// Packs trees that chunks_hold into sh.words words and, with category sets,
// four words a node of `cat`; `place` gives a feature's place. False for a
// tree that reaches a node twice, siblings not next to each other: its words
// have no second place.
template <class Place>
bool pack_trees(const Trees &e, const Shapes &sh, int K, int max_chunk_trees, Place place, unsigned long long *packed,
                unsigned long long *cat, Packed &p) {
    std::vector<int32_t> order, index;  // a tree's nodes, siblings next to each other
    std::vector<uint8_t> seen;
    p.tree.reserve((size_t)(e.t1 - e.t0));
    p.chunk_of.push_back(0);
    int32_t word0 = 0, node0 = 0;
    for (int k = 0; k < K; ++k) {
        for (int64_t t = e.t0 + k; t < e.t1;) {
            // the trees from t on that share a chunk, and their nodes
            int32_t trees = 0, nodes = 0, words = 0;
            for (int64_t q = t; q < e.t1 && trees < max_chunk_trees; q += K, ++trees) {
                const int32_t c = (int32_t)(e.off[q + 1] - e.off[q]), w = c + sh.leaves[(size_t)(q - e.t0)];
                if (words + w > kChunkWords) break;
                nodes += c;
                words += w;
            }
            p.chunk.push_back(Chunk{(int32_t)p.tree.size(), trees, word0, words, node0, 0});
            unsigned long long *nw = packed + word0, *values = nw + nodes;
            uint32_t n0 = 0, v = 0;
            for (int j = 0; j < trees; ++j, t += K) {
                const int64_t a = e.off[t];
                const int32_t count = (int32_t)(e.off[t + 1] - a);
                const bool paired = sh.paired[(size_t)(t - e.t0)] != 0;
                if (!paired) {
                    order.assign(1, 0);
                    index.assign((size_t)count, 0);  // an inner node's left child in `order`
                    seen.assign((size_t)count, 0);
                    for (size_t i = 0; i < order.size(); ++i) {
                        const int64_t nd = a + order[i];
                        if (e.feature[nd] < 0) continue;
                        for (const int32_t child : {e.left[nd], e.right[nd]})
                            if (seen[(size_t)child]++) return false;
                        index[i] = (int32_t)order.size();
                        order.push_back(e.left[nd]);
                        order.push_back(e.right[nd]);
                    }
                }
                p.tree.push_back(8 * n0);
                const uint32_t next = j + 1 < trees ? 8 * (n0 + (uint32_t)count) : kEnd;
                const int32_t used = paired ? count : (int32_t)order.size();
                for (int32_t i = 0; i < used; ++i) {
                    const int64_t nd = a + (paired ? i : order[(size_t)i]);
                    uint32_t lo, hi;
                    if (e.feature[nd] < 0) {
                        lo = (8 * ((uint32_t)nodes + v)) << 16 | next;
                        hi = kLeaf;
                        std::memcpy(&values[v++], &e.value[nd], 8);
                    } else {
                        const int32_t th = e.threshold[nd], mb = e.missing_bin[nd];
                        const int32_t child = paired ? e.left[nd] : index[(size_t)i];
                        lo = 8 * (n0 + (uint32_t)child) | (place(e.feature[nd]) << 16);
                        hi = kNoBin << 8;
                        if (th < 0) {
                            hi |= kCatNode;
                        } else {
                            hi |= (uint32_t)std::min(th, 255);
                            if (mb >= 0 && mb < 256) {
                                hi = (hi & 255u) | (uint32_t)mb << 8 | (e.default_left[nd] ? kDefLeft : 0u);
                                p.missing = true;
                            }
                        }
                    }
                    nw[n0 + (uint32_t)i] = ((unsigned long long)hi << 32) | lo;
                    if (cat)
                        std::memcpy(&cat[((size_t)node0 + n0 + (uint32_t)i) * 4], &e.cat_bits[(size_t)nd * 4], 32);
                }
                for (int32_t i = used; i < count; ++i) nw[n0 + (uint32_t)i] = 0;  // not reached
                n0 += (uint32_t)count;
            }
            for (int32_t i = (int32_t)v; i < words - nodes; ++i) values[i] = 0;
            word0 += words;
            node0 += nodes;
        }
        p.chunk_of.push_back((int32_t)p.chunk.size());
    }
    return true;
}

}  // namespace trees
}  // namespace mb
