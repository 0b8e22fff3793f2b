// The pair code of the direct sum (elfmm_math.h) in long double: every double of
// the header is one, the interface stays double.
#include <cmath>
#include <math.h>
#include <cstdint>

using std::atan2;
using std::fabs;
using std::log;
using std::sqrt;
#define double long double
#include "../../elfmmlib3d_amd/csrc/elfmm_math.h"
#undef double

extern "C" void near_long(const double *tri, const double *ssl, const double *sdl, const double *P, int iself,
                          double rlam, double rmu, int sl, int dl, double *out9)
{
    long double rec[elfmm::NF_REC], t[9], a[3], b[3], p[3], o[9] = {}, l = rlam, m = rmu;
    for (int i = 0; i < 9; i++) t[i] = tri[i];
    for (int i = 0; i < 3; i++) a[i] = ssl[i], b[i] = sdl[i], p[i] = P[i];
    elfmm::nf_make_record(t, a, b, rec);
    elfmm::nf_pair(rec, p, iself, l, m, (l + m) / (l + 2 * m), sl, dl, o);
    for (int i = 0; i < 9; i++) out9[i] = (double)o[i];
}
