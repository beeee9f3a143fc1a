"""The planner's LDS layout and the host's check of it (mb_plan.h), compiled
for the host: over 2 to 1024 leaves and 1 to 40,000 features, what is accepted
fits a workgroup's 160 KiB beside the kernel's own arrays and the replay's
slots, its arrays are apart, and less is accepted where more is."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include <vector>
#define __host__
#define __device__
#include "mb_plan.h"
using namespace mb;
int main() {
    const int K = 32;
    const size_t own = 9000;
    for (int F : {1, 6, 28, 126, 1000, 5000, 20000, 40000}) {
        bool before = true;
        int most = 0;
        for (int L = 2; L <= 1024; ++L) {
            const int E = 1 + 2 * std::min(4 * L - 1, 2047);  // as the trainer sets it
            const PlanLayout p = plan_layout(L, E, K, F);
            const bool fits = plan_fits(L, p.total, own);
            if (fits && !before) return std::printf("%d leaves, not one less\n", L), 1;
            before = fits;
            if (!fits) continue;
            most = L;
            if (p.total + own > 160 * 1024 || L > kPlanSlots) return std::printf("%d x %d does not fit\n", L, F), 1;
            struct Part { size_t at, bytes; };
            std::vector<Part> v{{p.wg, 16u * K}, {p.eg, 8u * E}, {p.cb, 8u * E}, {p.fr, 4u * E}, {p.ci, 4u * E},
                                {p.wf, 8u * K}, {p.el, 4u * E}, {p.ep, 4u * E}, {p.rw, 4u * E}, {p.sl_e, 4u * L},
                                {p.sl_fid, 4u * L}, {p.cm_e, 4u * L}, {p.cm_fid, 4u * L}, {p.cm_lf, 4u * L},
                                {p.sel_e, 4u * K}, {p.pcnt, 4u * K}, {p.poff, 4u * (K + 1)}, {p.qcnt, 4u * K},
                                {p.qoff, 4u * (K + 1)}, {p.sn, sizeof(SelNode) * K}, {p.mbin, 4u * F}};
            std::sort(v.begin(), v.end(), [](Part a, Part b) { return a.at < b.at; });
            for (size_t i = 0; i < v.size(); ++i)
                if (v[i].at + v[i].bytes > (i + 1 < v.size() ? v[i + 1].at : p.total))
                    return std::printf("%d x %d: arrays overlap\n", L, F), 1;
            // a replay step's right children: two words each, a lane of 64 or a leaf each
            if (16u * std::min(64, L - 1) > 8u * E) return std::printf("%d leaves: right children\n", L), 1;
        }
        if (F <= 28 && (most < 473 || most > kPlanSlots)) return std::printf("%d features: %d leaves\n", F, most), 1;
        if (F == 40000 && most != 0) return std::printf("40000 features: %d leaves\n", most), 1;
    }
    // the slots bound the leaves whatever the LDS
    return plan_fits(kPlanSlots, 0, 0) && !plan_fits(kPlanSlots + 1, 0, 0) ? 0 : 1;
}
"""


def test_accepted_leaves_fit(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text("")
    (tmp_path / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{tmp_path}", f"-I{ROOT / 'mojoboost_amd' / 'csrc'}",
                    str(tmp_path / "plan.cpp"), "-o", str(tmp_path / "plan")], check=True)
    out = subprocess.run([str(tmp_path / "plan")], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
