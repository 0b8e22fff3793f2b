// The waves of the near field (near_tasks, elfmm_plan.cpp) over the near lists of
// a tree, for CPU tests.
#include <vector>

#include "../../elfmmlib3d_amd/csrc/elfmm_internal.h"

using namespace elfmm;

// Waves of the near field, 0 if each point's lanes do not meet a lane exactly once
// or a box's lanes per point are not one power of two up to 64.
extern "C" int near_tasks_check(const double *src, int n, const double *tgt, int nt, int nbox, int src_eval)
{
    Tree T;
    Plan P;
    std::vector<int> tasks = {7, 7, 7};              // an earlier call's
    if (build_tree(src, n, tgt, nt, nbox, 0, T)) return 0;
    plan_reset(P);
    build_plan_near(T, src_eval, false, false, P);
    near_tasks(T, P, src_eval, tasks);
    if (tasks.size() % 3) return 0;
    size_t k = 0;
    for (size_t q = 0; q < P.nf_boxes.size(); q++) {
        int b = P.nf_boxes[q], ntri = 0, split = k < tasks.size() ? tasks[k + 2] : 0;
        for (int e = P.nf_start[q]; e < P.nf_start[q + 1]; e++) ntri += T.src_count[P.nf_items[e]];
        if (ntri != P.nf_ntri[q] || split < 1 || split > 64 || (split & (split - 1))) return 0;
        int64_t lanes = (int64_t)((src_eval ? T.src_count[b] : 0) + T.tgt_count[b]) * split;
        for (int64_t l0 = 0; l0 < lanes; l0 += 64, k += 3)
            if (k >= tasks.size() || tasks[k] != (int)q || tasks[k + 1] != l0 || tasks[k + 2] != split) return 0;
    }
    return k == tasks.size() ? (int)(k / 3) : 0;
}
