// Host build of the near-field kernel's pair code (elfmm_near.h) beside the
// direct sum's (elfmm_math.h), for CPU tests.
#include "../../elfmmlib3d_amd/csrc/elfmm_near.h"

extern "C" void near_host_pair(const double *tri, const double *ssl, const double *sdl, const double *P, int iself,
                               double rlam, double rmu, int sl, int dl, int st, double *out9)
{
    double rec[elfmm::NF_REC];
    elfmm::nf_make_record(tri, ssl, sdl, rec);
    for (int i = 0; i < 9; i++) out9[i] = 0.0;
    double c1 = (rlam + rmu) / (rlam + 2 * rmu);
    auto f = sl && dl ? (st ? elfmm::near_pair<true, true, true> : elfmm::near_pair<true, true, false>)
             : dl     ? (st ? elfmm::near_pair<false, true, true> : elfmm::near_pair<false, true, false>)
                      : (st ? elfmm::near_pair<true, false, true> : elfmm::near_pair<true, false, false>);
    f(rec, P, iself, rlam, rmu, c1, out9);
    for (int i = 0; i < 9; i++) out9[i] *= 0.5 / rmu;
}

extern "C" void near_host_old(const double *tri, const double *ssl, const double *sdl, const double *P, int iself,
                              double rlam, double rmu, int sl, int dl, double *out9)
{
    double rec[elfmm::NF_REC];
    elfmm::nf_make_record(tri, ssl, sdl, rec);
    for (int i = 0; i < 9; i++) out9[i] = 0.0;
    elfmm::nf_pair(rec, P, iself, rlam, rmu, (rlam + rmu) / (rlam + 2 * rmu), sl, dl, out9);
}
