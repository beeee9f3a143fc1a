// LDS layout of the planning kernel (k_plan), shared by the kernel and the
// host's check that it fits.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace mb {

// Frontier slots that the replay holds in registers: more leaves would lose
// the ones above.
constexpr int kPlanSlots = 512;
constexpr size_t kPlanLdsMost = 160 * 1024;  // of a workgroup

// The fields of a selected leaf's explored node the batch setup needs.
struct SelNode {
    int64_t begin, end, n_left;
    int32_t buf, hist, depth, feature, bin, default_left, cat, pad_;
};

// Byte offsets in the planner's dynamic LDS.
struct PlanLayout {
    size_t sn, mbin;
    size_t wg, eg, cb, kr, wf, el, ep, rw, fr, ci, sl_e, sl_fid, cm_e, cm_fid, cm_lf, sel_e, pcnt, poff, qcnt, qoff;
    size_t total;
};

__host__ __device__ inline PlanLayout plan_layout(int L, int E, int K, int F) {
    PlanLayout p;
    size_t o = 0;
    auto take = [&o](size_t bytes, size_t align) {
        o = (o + align - 1) & ~(align - 1);
        const size_t at = o;
        o += bytes;
        return at;
    };
    p.wg = take((size_t)8 * 2 * K, 8);       // pair's best gain
    p.eg = take((size_t)8 * E, 8);           // explored node's gain view
    p.cb = take((size_t)8 * E, 8);           // replay: explored node's bar; selection: bottleneck values
    p.kr = take((size_t)8 * E, 8);           // replay: a step's right children; selection: fr, ci
    p.fr = p.kr;                             // in the committed frontier
    p.ci = p.kr + (size_t)4 * E;             // jump pointers, then candidates' node ids
    p.wf = take((size_t)4 * 2 * K, 4);       // pair's best feature
    p.el = take((size_t)4 * E, 4);           // explored node's left child
    p.ep = take((size_t)4 * E, 4);           // explored node's parent
    p.rw = take((size_t)4 * E, 4);           // explored node's rows
    p.sl_e = take((size_t)4 * L, 4);
    p.sl_fid = take((size_t)4 * L, 4);
    p.cm_e = take((size_t)4 * L, 4);
    p.cm_fid = take((size_t)4 * L, 4);
    p.cm_lf = take((size_t)4 * L, 4);
    p.sel_e = take((size_t)4 * K, 4);
    p.pcnt = take((size_t)4 * K, 4);
    p.poff = take((size_t)4 * (K + 1), 4);
    p.qcnt = take((size_t)4 * K, 4);
    p.qoff = take((size_t)4 * (K + 1), 4);
    p.sn = take(sizeof(SelNode) * K, 16);    // the selected leaves' nodes
    p.mbin = take((size_t)4 * F, 4);         // missing bin per feature
    p.total = o;
    return p;
}

// Whether the planner runs num_leaves leaves, in `dynamic` bytes of LDS beside
// the kernel's own arrays (some 9 KB).
inline bool plan_fits(int num_leaves, size_t dynamic, size_t own) {
    return num_leaves <= kPlanSlots && dynamic + own <= kPlanLdsMost;
}

}  // namespace mb
