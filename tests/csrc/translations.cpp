// The operators of build_operators (records: rotate, shift along z, rotate
// back, in the matrix cores' layout; dense matrices for M2L of the lower orders)
// applied on the host, against the addition theorems summed over all degrees
// and orders in long double.
#include <cmath>
#include <complex>
#include <random>
#include <vector>

#include "../../elfmmlib3d_amd/csrc/elfmm_internal.h"

using namespace elfmm;
typedef long double LD;
typedef std::complex<LD> CL;

namespace {
LD fact(int n)
{
    LD f = 1;
    for (int i = 2; i <= n; i++) f *= i;
    return f;
}
LD binom(int n, int k) { return k < 0 || k > n ? 0 : fact(n) / fact(k) / fact(n - k); }

// R_l^m (irr 0) or I_l^m (irr 1) at x, all 0 <= m <= l <= p
std::vector<CL> harmonics(int p, const LD *x, int irr)
{
    std::vector<CL> v((p + 1) * (p + 2) / 2);
    LD r = std::sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]), ct = x[2] / r, phi = std::atan2(x[1], x[0]);
    LD st = std::sqrt(x[0] * x[0] + x[1] * x[1]) / r, pmm = 1;
    for (int m = 0; m <= p; m++) {
        if (m) pmm *= -(2 * m - 1) * st;
        LD a = 0, b = pmm;
        for (int l = m; l <= p; l++) {
            v[l * (l + 1) / 2 + m] = std::sqrt(fact(l - m) / fact(l + m)) * (irr ? std::pow(r, -l - 1) : std::pow(r, l)) * b *
                                     std::polar((LD)1, m * phi);
            LD c = ((2 * l + 1) * ct * b - (l + m) * a) / (l - m + 1);
            a = b;
            b = c;
        }
    }
    return v;
}
CL at(const std::vector<CL> &v, int l, int m)
{
    if (m >= 0) return v[l * (l + 1) / 2 + m];
    CL c = std::conj(v[l * (l + 1) / 2 - m]);
    return m & 1 ? -c : c;
}

// the record on the real or imaginary parts x of the turned coefficients
void apply(int p, const double *rec, int im, std::vector<double> &x)
{
    const size_t Z = trans_blocks(p + 2);
    for (int stage = 0; stage < 3; stage++) {
        const double *A = rec + Z * (stage == 0 ? im : stage == 1 ? 2 : 3 + im);
        std::vector<double> y(x.size());
        for (int n = 1; n <= p + 1; n++) {
            const double *B = A + trans_blocks(n);
            int ks = (n + 3) / 4, m = p + 1 - n;
            auto row = [&](int k) { return stage == 1 ? (m + k) * (m + k + 1) / 2 + m : n * (n - 1) / 2 + k; };
            for (int r = 0; r < n; r++)
                for (int c = 0; c < n; c++)
                    y[row(r)] += B[((size_t)(r / 16) * ks + c / 4) * 64 + c % 4 * 16 + r % 16] * x[row(c)];
        }
        x = y;
    }
}
}  // namespace

// Worst difference of the translations of order p relative to the result's
// norm per degree: kind 0 M2M, 1 L2L (index = octant), 2 M2L (index = offset;
// *order its order, -1 where it has no operator).
extern "C" double translation_error(int iprec, int p, int kind, int index, int seed, int *order)
{
    static Operators ops;
    static int built = -99, builtp = -1;
    if (built != iprec || builtp != p) {
        int itable[343];
        list2_orders(iprec_eps(iprec), itable);
        build_operators(p, itable, ops);
        built = iprec;
        builtp = p;
    }
    int pt = kind == 2 ? ops.m2l_pt[index] : p;
    *order = pt;
    if (pt < 0) return 0;
    const double phi = kind == 2 ? ops.m2l_phi[index] : ops.oct_phi[index];
    const double *rec = kind == 2 ? &ops.m2l[ops.m2l_off[index]]
                                  : (kind ? ops.l2l : ops.m2m).data() + index * trans_doubles(p);
    const int refl = kind == 2 ? ops.m2l_refl[index] : 0, h = (pt + 1) * (pt + 2) / 2;
    LD t[3];
    if (kind == 2) t[0] = -(index / 49 - 3), t[1] = -(index / 7 % 7 - 3), t[2] = -(index % 7 - 3);
    else for (int d = 0; d < 3; d++) t[d] = index >> d & 1 ? 0.25 : -0.25;
    std::mt19937 g(seed);
    std::uniform_real_distribution<double> U(-1, 1);
    std::vector<CL> in(h), out(h);
    for (int l = 0; l <= pt; l++)
        for (int m = 0; m <= l; m++) in[l * (l + 1) / 2 + m] = CL(U(g), m ? U(g) : 0.0) * (LD)std::pow(0.6, l);
    std::vector<double> re(h), im(h);
    auto turn = [&](int l, int m) { return std::polar((LD)1, m * (LD)phi) * (LD)(refl && (l + m) & 1 ? -1 : 1); };
    for (int l = 0; l <= pt; l++)
        for (int m = 0; m <= l; m++) {
            CL v = in[l * (l + 1) / 2 + m] * turn(l, m);
            re[l * (l + 1) / 2 + m] = (double)v.real();
            im[l * (l + 1) / 2 + m] = (double)v.imag();
        }
    if (kind == 2 && h < m2l_turned_h(p)) {
        std::vector<double> r(h), i(h);
        for (int a = 0; a < h; a++)
            for (int b = 0; b < h; b++) {
                r[a] += rec[(size_t)a * h + b] * re[b];
                i[a] += rec[(size_t)(h + a) * h + b] * im[b];
            }
        re = r;
        im = i;
    } else {
        apply(pt, rec, 0, re);
        apply(pt, rec, 1, im);
    }
    std::vector<CL> H = harmonics(kind == 2 ? 2 * pt : pt, t, kind == 2);
    LD worst = 0;
    for (int j = 0; j <= pt; j++) {
        LD num = 0, den = 0;
        for (int k = 0; k <= j; k++) {
            CL s = 0;
            for (int l = 0; l <= pt; l++)
                for (int m = -l; m <= l; m++) {
                    if (kind == 2)
                        s += (LD)((j + k) & 1 ? -1 : 1) * std::sqrt(binom(l + j - m + k, j + k) * binom(l + j + m - k, j - k)) *
                             at(H, l + j, m - k) * at(in, l, m);
                    else if (kind == 0 && l <= j && std::abs(k - m) <= j - l)
                        s += std::sqrt(binom(j + k, l + m) * binom(j - k, l - m)) * std::ldexp((LD)1, -l) *
                             std::conj(at(H, j - l, k - m)) * at(in, l, m);
                    else if (kind == 1 && l >= j && std::abs(m - k) <= l - j)
                        s += std::sqrt(binom(l + m, j + k) * binom(l - m, j - k)) * std::ldexp((LD)1, -j) * at(H, l - j, m - k) *
                             at(in, l, m);
                }
            int q = j * (j + 1) / 2 + k;
            CL got = CL(re[q], im[q]) * std::conj(std::polar((LD)1, k * (LD)phi)) * (LD)(refl && (j + k) & 1 ? -1 : 1);
            num += std::norm(got - s);
            den += std::norm(s);
        }
        worst = std::max(worst, std::sqrt(num / den));
    }
    return (double)worst;
}
