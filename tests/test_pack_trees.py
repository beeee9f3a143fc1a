"""The packing of an ensemble for the prediction kernels (mb_trees.h),
compiled for the host with AddressSanitizer: random trees whose nodes are
shared or unreached, siblings neighbours or not, in one class and several.
A packed ensemble walks to the same leaves, in the same order, as the trees
do; one with a node reached twice, siblings apart, is not packed."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <random>
#include "mb_trees.h"
using namespace mb::trees;

struct Forest {
    std::vector<int64_t> off{0};
    std::vector<int32_t> feature, threshold, left, right, dl, mb;
    std::vector<double> value;
    Trees view() const {
        return Trees{off.data(), 0, (int64_t)off.size() - 1, feature.data(), threshold.data(), left.data(),
                     right.data(), value.data(), dl.data(), mb.data(), nullptr};
    }
    void node(int32_t f, int32_t t, int32_t l, int32_t r) {
        feature.push_back(f), threshold.push_back(t), left.push_back(l), right.push_back(r);
        dl.push_back(0), mb.push_back(-1), value.push_back((double)value.size());
    }
    void end() { off.push_back((int64_t)feature.size()); }
};

constexpr int kF = 5;

double leaf_of(const Forest &fo, int64_t t, const uint8_t *row) {
    int64_t at = fo.off[t];
    while (fo.feature[at] >= 0)
        at = fo.off[t] + (row[fo.feature[at]] <= fo.threshold[at] ? fo.left[at] : fo.right[at]);
    return fo.value[at];
}

struct Pack : Packed {
    std::vector<unsigned long long> words;  // their end is guarded
};

// the packed walk of class k, as the kernels do it; its leaf values in order
std::vector<double> packed_walk(const Pack &p, int k, const uint8_t *row) {
    std::vector<double> got;
    for (int c = p.chunk_of[k]; c < p.chunk_of[k + 1]; ++c) {
        const Chunk &ch = p.chunk[c];
        const unsigned long long *w = p.words.data() + ch.word0;
        auto word = [&](uint32_t at) {
            if (at % 8 || (int32_t)(at / 8) >= ch.n_words) std::printf("offset %u outside the chunk\n", at), std::exit(1);
            return w[at / 8];
        };
        uint32_t at = 0;
        while (at != kEnd) {
            const uint32_t lo = (uint32_t)word(at), hi = (uint32_t)(word(at) >> 32);
            if (hi & kLeaf) {
                double v;
                const unsigned long long bits = word(lo >> 16);
                std::memcpy(&v, &bits, 8);
                got.push_back(v);
                at = lo & 0xFFFFu;
            } else {
                at = (lo & 0xFFFFu) + (row[lo >> 16] <= (hi & 255u) ? 0u : 8u);
            }
        }
    }
    return got;
}

bool pack(const Forest &fo, int K, Pack &p) {
    const Trees e = fo.view();
    const Shapes sh = check_trees(e, kF);
    if (!chunks_hold(sh)) std::printf("a tree past a chunk\n"), std::exit(1);
    p.words.resize((size_t)sh.words);
    return pack_trees(e, sh, K, 256, [](int32_t f) { return (uint32_t)f; }, p.words.data(), nullptr, p);
}

int main(int argc, char **argv) {
    std::mt19937_64 r(std::atoi(argv[1]));
    auto below = [&](int n) { return (int)(r() % (uint64_t)n); };
    long packed = 0, refused = 0;
    for (int round = 0; round < 3000; ++round) {
        const int K = 1 + below(3), T = K * (1 + below(6));
        Forest fo;
        bool must_pack = true;
        for (int t = 0; t < T; ++t) {
            const int n = 1 + below(round % 50 == 0 ? 900 : 12), kind = below(3);
            // kind 0: siblings neighbours, nodes shared and unreached at will;
            // kind 1: any two later children; kind 2: a proper tree, siblings apart
            if (kind == 2) {
                // depth-first numbering: the left child next, the right one
                // after the left's subtree
                std::vector<int32_t> f, l, rr;
                struct Grow {
                    std::vector<int32_t> &f, &l, &r;
                    std::mt19937_64 &g;
                    int32_t make(int depth) {
                        const int32_t at = (int32_t)f.size();
                        f.push_back(-1), l.push_back(-1), r.push_back(-1);
                        if (depth > 0 && g() % 4 != 0) {
                            f[at] = (int32_t)(g() % kF);
                            const int32_t a = make(depth - 1);
                            const int32_t b = make(depth - 1);
                            l[at] = a, r[at] = b;
                        }
                        return at;
                    }
                } grow{f, l, rr, r};
                grow.make(6);
                for (size_t i = 0; i < f.size(); ++i) fo.node(f[i], below(8), l[i], rr[i]);
            } else {
                for (int i = 0; i < n; ++i) {
                    const bool inner = i + 2 < n && below(4) != 0;
                    int a = 0, b = 0;
                    if (inner && kind == 0) {
                        a = i + 1 + below(n - i - 2);
                        b = a + 1;
                    } else if (inner) {
                        a = i + 1 + below(n - i - 1);
                        b = i + 1 + below(n - i - 1);
                    }
                    fo.node(inner ? below(kF) : -1, below(8), inner ? a : -1, inner ? b : -1);
                }
                must_pack = must_pack && kind == 0;
            }
            fo.end();
        }
        Pack p;
        if (!pack(fo, K, p)) {
            if (must_pack) return std::printf("round %d: not packed\n", round), 1;
            ++refused;
            continue;
        }
        ++packed;
        for (int s = 0; s < 20; ++s) {
            uint8_t row[kF];
            for (auto &b : row) b = (uint8_t)below(8);
            for (int k = 0; k < K; ++k) {
                std::vector<double> want;
                for (int t = k; t < T; t += K) want.push_back(leaf_of(fo, t, row));
                if (packed_walk(p, k, row) != want) return std::printf("round %d: other leaves\n", round), 1;
            }
        }
    }
    if (packed < 300 || refused < 300) return std::printf("%ld packed, %ld not\n", packed, refused), 1;

    // as many visits as nodes, four of them leaves of a tree of two
    for (int more = 0; more < 2; ++more) {
        Forest fo;
        fo.node(0, 3, 3, 4), fo.node(1, 3, 2, 5), fo.node(1, 3, 5, 6), fo.node(1, 3, 5, 6), fo.node(2, 3, 6, 5);
        fo.node(-1, 0, -1, -1), fo.node(-1, 0, -1, -1), fo.end();
        if (more) fo.node(-1, 0, -1, -1), fo.end();
        Pack p;
        if (pack(fo, 1, p)) return std::printf("a node reached twice was packed\n"), 1;
    }
    // one leaf for every split
    Forest fo;
    for (int i = 0; i < 3; ++i) fo.node(0, 3, 3, 3);
    fo.node(-1, 0, -1, -1), fo.end();
    Pack p;
    if (pack(fo, 1, p)) return std::printf("a leaf reached twice was packed\n"), 1;
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    at = tmp_path_factory.mktemp("pack")
    (at / "pack.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-g", "-O1", "-std=c++17", "-fsanitize=address", f"-I{ROOT / 'mojoboost_amd' / 'csrc'}",
                    str(at / "pack.cpp"), "-o", str(at / "pack")], check=True)
    return at / "pack"


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_packing_of_shared_and_unreached_nodes(program, seed):
    out = subprocess.run([str(program), str(seed)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr[:2000]
