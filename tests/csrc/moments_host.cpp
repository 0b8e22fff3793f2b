// Host build of the P2M / P2L moment kernels' body (elfmm_moments.h): one
// thread per lane of a workgroup, barriers and wave operations (shuffle, the
// 16 x 16 x 4 product in its operand layout) emulated, LDS an array of exactly
// the size the launch asks for, filled with NaN. Checked against the node sums
// of the same sources in long double, charge and dipole columns through the
// harmonics' ladders.
#include <pthread.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <random>
#include <thread>
#include <vector>

using std::max;
using std::min;

#define __global__
#define __device__
#define __constant__ static
#define __shared__
#define __forceinline__ inline

#include "../../elfmmlib3d_amd/csrc/elfmm_math.h"

namespace {
struct Dim {
    int x;
};
thread_local Dim threadIdx;
Dim blockIdx{0}, blockDim{1};
struct double2 {
    double x, y;
};
struct gemm_d4 {
    double v[4];
    double &operator[](int i) { return v[i]; }
};
constexpr int PMAX = 44, NRHS = 4;
double g_fact[2 * PMAX + 8], g_sdfact[PMAX + 4];
double *emu_lds;
pthread_barrier_t g_bar, g_wave[16];
int g_si[16][64];
double g_a[16][64], g_b[16][64];

void __syncthreads() { pthread_barrier_wait(&g_bar); }

int __shfl_up(int v, int off)
{
    int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    g_si[w][l] = v;
    pthread_barrier_wait(&g_wave[w]);
    int r = l >= off ? g_si[w][l - off] : v;
    pthread_barrier_wait(&g_wave[w]);
    return r;
}

// lane l holds A[row l % 16][k l / 16], B[k l / 16][col l % 16] and, in register
// i, D[row l / 16 + 4 i][col l % 16]
gemm_d4 mfma(double a, double b, gemm_d4 c)
{
    int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    g_a[w][l] = a;
    g_b[w][l] = b;
    pthread_barrier_wait(&g_wave[w]);
    for (int i = 0; i < 4; i++)
        for (int k = 0; k < 4; k++) c[i] += g_a[w][k * 16 + (l >> 4) + 4 * i] * g_b[w][k * 16 + (l & 15)];
    pthread_barrier_wait(&g_wave[w]);
    return c;
}

#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, x, y, z) mfma(a, b, c)
void unsafeAtomicAdd(double *p, double v) { *p += v; }    // no two lanes share a coefficient
#include "../../elfmmlib3d_amd/csrc/elfmm_moments.h"

template <bool IRR, class Z, bool MIND = false>
void launch(int p, const std::vector<int> &boxes, const std::vector<int> &ls, const std::vector<int> &li,
            const double *cen, const double *sides, const int *ss, const int *sc, const double *tri, const double *tc,
            int nc, double *ex, const std::vector<int> &parts = {}, MindMoments mind = {})
{
    size_t nl = (size_t)Z::lds(IRR ? p + 1 : p), nwg = parts.empty() ? boxes.size() : parts.size() / 3;
    for (size_t b = 0; b < nwg; b++) {
        blockIdx.x = (int)b;
        emu_lds = (double *)std::aligned_alloc(16, (nl * 8 + 15) / 16 * 16);
        std::fill(emu_lds, emu_lds + nl, NAN);
        pthread_barrier_init(&g_bar, nullptr, Z::NT);
        for (int w = 0; w < Z::WB; w++) pthread_barrier_init(&g_wave[w], nullptr, 64);
        std::vector<std::thread> th;
        for (int t = 0; t < Z::NT; t++)
            th.emplace_back([&, t] {
                threadIdx.x = t;
                p2t_body<IRR, Z, MIND>(p, boxes.data(), parts.empty() ? nullptr : parts.data(), mind, ls.data(),
                                       li.data(), cen, sides, ss, sc, tri, tc, nc, ex, emu_lds);
            });
        for (auto &t : th) t.join();
        pthread_barrier_destroy(&g_bar);
        for (int w = 0; w < Z::WB; w++) pthread_barrier_destroy(&g_wave[w]);
        std::free(emu_lds);
    }
}

typedef long double LD;
const double RULE[18][3] = {ELFMM_RULE4, ELFMM_RULE6};
}  // namespace

// The worst relative difference, over boxes, right-hand sides and degrees, of
// the expansions of order p (nq nodes a triangle); irr 0: multipoles of four
// leaves of counts[4] triangles; 1: locals of two boxes, one from nlist source
// boxes, one from a single one. Negative: no shape takes the order.
extern "C" double moments_host(int p, int nq, int irr, const int *counts, int nlist, int seed)
{
    double f = 1, d = 1;
    for (int k = 0; k < 2 * PMAX + 8; k++) g_fact[k] = f, f *= k + 1;
    for (int m = 0; m < PMAX + 4; m++) g_sdfact[m] = d, d *= -(2.0 * m + 1);
    const int ph = irr ? p + 1 : p, nc = (p + 1) * (p + 2), shape = p2t_shape(ph, nq);
    if (shape < 0) return -1;
    std::mt19937 g(seed);
    std::uniform_real_distribution<double> U(-1, 1);
    int nb = std::max(4, nlist + 1);
    std::vector<int> sc(nb), ss(nb);
    int n = 0;
    for (int b = 0; b < nb; b++) sc[b] = counts[b % 4], ss[b] = n, n += sc[b];
    std::vector<double> tri(9 * n), nrm(3 * n), sl(3 * n), dl(3 * n), tc(48 * n), cen(3 * nb), sides(nb, 1.3);
    for (int i = 0; i < n; i++) {
        double c[3] = {0.4 * U(g) + (irr ? 3.0 : 0.0), 0.4 * U(g), 0.4 * U(g)};
        for (int k = 0; k < 9; k++) tri[9 * i + k] = c[k % 3] + 0.1 * U(g);
        for (int k = 0; k < 3; k++) nrm[3 * i + k] = U(g), sl[3 * i + k] = U(g), dl[3 * i + k] = U(g);
    }
    for (double &c : cen) c = 0.1 * U(g);
    const double mu = 0.7, c1 = 0.6, c2 = 0.4, dls = -1.0;
    blockDim.x = 1;
    threadIdx.x = 0;
    for (int i = 0; i < n; i++) {
        blockIdx.x = i;
        k_tcoef(n, tri.data(), nrm.data(), sl.data(), dl.data(), 1, 1, mu, c1, c2, dls, tc.data());
    }
    std::vector<int> boxes, ls, li;
    if (irr) {
        boxes = {0, 2};
        ls = {0, nlist, nlist + 1};
        for (int k = 1; k <= nlist; k++) li.push_back(k);
        li.push_back(0);
    } else {
        boxes = {0, 1, 2, 3};
    }
    std::vector<double> ex((size_t)nb * NRHS * nc, 0.0);
    auto go = [&](auto z) {
        using Z = decltype(z);
        if (irr) launch<true, Z>(p, boxes, ls, li, cen.data(), sides.data(), ss.data(), sc.data(), tri.data(), tc.data(), nc, ex.data());
        else launch<false, Z>(p, boxes, ls, li, cen.data(), sides.data(), ss.data(), sc.data(), tri.data(), tc.data(), nc, ex.data());
    };
    if (shape == 0) go(P2TShape0{});
    else if (shape == 1) go(P2TShape1{});
    else if (shape == 2) go(P2TShape2{});
    else go(P2TShape3{});

    double worst = 0;
    for (size_t b = 0; b < boxes.size(); b++) {
        int bx = boxes[b];
        std::vector<int> src;
        if (irr) src.assign(li.begin() + ls[b], li.begin() + ls[b + 1]);
        else src.push_back(bx);
        const size_t P1 = ph + 1;
        std::vector<LD> M(16 * P1 * P1 * 2, 0);
        for (int sb : src)
            for (int i = ss[sb]; i < ss[sb] + sc[sb]; i++)
                for (int q = 0; q < nq; q++) {
                    const double *r = RULE[(nq == 12 ? 6 : 0) + q], *t = &tri[9 * i], *nv = &nrm[3 * i], *s1 = &sl[3 * i];
                    LD u = r[0], v = r[1], X[3], a[3], e[3], b3[3] = {dls * dl[3 * i], dls * dl[3 * i + 1], dls * dl[3 * i + 2]};
                    for (int k = 0; k < 3; k++) {
                        a[k] = (LD)t[3 + k] - t[k], e[k] = (LD)t[6 + k] - t[k];
                        X[k] = t[k] + u * a[k] + v * e[k];
                    }
                    LD cx = a[1] * e[2] - a[2] * e[1], cy = a[2] * e[0] - a[0] * e[2], cz = a[0] * e[1] - a[1] * e[0];
                    LD w = r[2] * sqrtl(cx * cx + cy * cy + cz * cz), col[16];
                    LD sX = 0, bX = 0, nX = 0, bn = 0;
                    for (int k = 0; k < 3; k++) sX += s1[k] * X[k], bX += b3[k] * X[k], nX += nv[k] * X[k], bn += b3[k] * nv[k];
                    for (int j = 0; j < 3; j++) {
                        col[j] = w * s1[j] / (2 * mu);
                        for (int k = 0; k < 3; k++) col[4 + 3 * j + k] = w * (nv[k] * b3[j] + b3[k] * nv[j]) / 2;
                        col[13 + j] = w * c1 * (nv[j] * bX + b3[j] * nX) / 2;
                    }
                    col[3] = w * (sX * c1 / (2 * mu) + bn * c2);
                    LD x = (X[0] - cen[3 * bx]) / sides[bx], y = (X[1] - cen[3 * bx + 1]) / sides[bx], z = (X[2] - cen[3 * bx + 2]) / sides[bx];
                    LD r2 = x * x + y * y + z * z, i2 = irr ? 1 / r2 : 1, dr = irr ? sqrtl(i2) : 1, di = 0, zz = z * i2, rr = irr ? i2 : r2;
                    for (int m = 0; m <= ph; m++) {
                        if (m) {
                            LD c = -(LD)(2 * m - 1) * i2, nr = c * (x * dr - y * di), ni = c * (x * di + y * dr);
                            dr = nr, di = ni;
                        }
                        LD ar = 0, ai = 0, br = dr, bi = di;
                        for (int l = m; l <= ph; l++) {
                            for (int c = 0; c < 16; c++) {
                                M[((c * P1 + l) * P1 + m) * 2] += col[c] * br;
                                M[((c * P1 + l) * P1 + m) * 2 + 1] += col[c] * bi;
                            }
                            LD k1 = (2 * l + 1) * zz, k2 = (LD)(l + m) * (l - m) * rr, nr = k1 * br - k2 * ar, ni = k1 * bi - k2 * ai;
                            ar = br, ai = bi, br = nr, bi = ni;
                        }
                    }
                }
        auto hn = [&](int l, int m) { return 1 / sqrtl((LD)g_fact[l + std::abs(m)] * g_fact[l - std::abs(m)]); };
        auto get = [&](int col, int l, int m, LD &re, LD &im) {
            int am = std::abs(m);
            re = im = 0;
            if (l < 0 || l > ph || am > l) return;
            re = M[((col * P1 + l) * P1 + am) * 2], im = M[((col * P1 + l) * P1 + am) * 2 + 1];
            if (m < 0) re = -re;                      // -conj of order 1
        };
        LD is = 1 / (LD)sides[bx], f0 = irr ? is : 1, f1 = irr ? is * is : is;
        for (int r = 0; r < NRHS; r++)
            for (int l = 0; l <= p; l++) {
                LD num = 0, den = 0;
                for (int m = 0; m <= l; m++) {
                    int ld = irr ? l + 1 : l - 1, c0 = 4 + 3 * r;
                    auto at = [&](LD v, int mm) { return ld >= 0 && std::abs(mm) <= ld ? v * hn(ld, mm) : (LD)0; };
                    LD fp = irr ? at(sqrtl((LD)(l + m + 1) * (l + m + 2)), m + 1) : at(sqrtl((LD)(l - m) * (l - m - 1)), m + 1);
                    LD fm = irr ? at(sqrtl((LD)(l - m + 1) * (l - m + 2)), m - 1) : at(sqrtl((LD)(l + m) * (l + m - 1)), m - 1);
                    LD fz = irr ? -at(sqrtl((LD)(l - m + 1) * (l + m + 1)), m) : at(sqrtl((LD)(l - m) * (l + m)), m);
                    LD qr, qi, xpr, xpi, ypr, ypi, xmr, xmi, ymr, ymi, zr, zi;
                    get(r, l, m, qr, qi);
                    get(c0, ld, m + 1, xpr, xpi);
                    get(c0 + 1, ld, m + 1, ypr, ypi);
                    get(c0, ld, m - 1, xmr, xmi);
                    get(c0 + 1, ld, m - 1, ymr, ymi);
                    get(c0 + 2, ld, m, zr, zi);
                    LD fh = hn(l, m) * f0, re = fh * qr + f1 * (fp * (xpr + ypi) / 2 + fm * (ymi - xmr) / 2 + fz * zr);
                    LD im = -fh * qi + f1 * (fp * (ypr - xpi) / 2 + fm * (xmi + ymr) / 2 - fz * zi);
                    const double *e = &ex[((size_t)bx * NRHS + r) * nc + l * (l + 1) + 2 * m];
                    num += (e[0] - re) * (e[0] - re) + (e[1] - im) * (e[1] - im);
                    den += re * re + im * im;
                }
                double rel = (double)sqrtl(num / den);
                if (!(rel <= worst)) worst = rel;     // NaN stays
            }
    }
    return worst;
}

// One box of `count` triangles in `nparts` parts beside a whole one: the worst
// relative difference, over degrees, of the parts' multipole from the whole
// box's, and of the Mindlin moments (both layers, in parts) from the node sums
// in long double of the Racah-normalised harmonics (Condon-Shortley phase).
extern "C" double moment_parts_host(int p, int nq, int count, int nparts, int seed)
{
    double f = 1, d = 1;
    for (int k = 0; k < 2 * PMAX + 8; k++) g_fact[k] = f, f *= k + 1;
    for (int m = 0; m < PMAX + 4; m++) g_sdfact[m] = d, d *= -(2.0 * m + 1);
    const int nc = (p + 1) * (p + 2), nown = nc / 2, shape = p2t_shape(p, nq), n = count;
    std::mt19937 g(seed);
    std::uniform_real_distribution<double> U(-1, 1);
    std::vector<double> tri(9 * n), nrm(3 * n), sl(3 * n), dl(3 * n), tc(48 * n), cen = {0.1, -0.05, -0.2}, sides = {1.3};
    for (int i = 0; i < n; i++) {
        double c[3] = {0.4 * U(g), 0.4 * U(g), 0.4 * U(g)};
        for (int k = 0; k < 9; k++) tri[9 * i + k] = c[k % 3] + 0.1 * U(g);
        for (int k = 0; k < 3; k++) nrm[3 * i + k] = U(g), sl[3 * i + k] = U(g), dl[3 * i + k] = U(g);
    }
    std::vector<int> boxes = {0}, none, ss = {0}, sc = {n}, parts;
    for (int j = 0; j < nparts; j++) parts.insert(parts.end(), {0, n * j / nparts, n * (j + 1) / nparts - n * j / nparts});
    auto each = [&](auto fn) {
        blockDim.x = 1;
        threadIdx.x = 0;
        for (int i = 0; i < n; i++) blockIdx.x = i, fn();
    };
    auto shaped = [&](auto fn) {
        shape == 0 ? fn(P2TShape0{}) : shape == 1 ? fn(P2TShape1{}) : shape == 2 ? fn(P2TShape2{}) : fn(P2TShape3{});
    };
    double worst = 0;
    auto note = [&](LD num, LD den) {
        double rel = (double)sqrtl(num / den);
        if (!(rel <= worst)) worst = rel;             // NaN stays
    };
    std::vector<double> whole(NRHS * nc, 0.0), cut(NRHS * nc, 0.0), G((size_t)2 * MindMoments::MCOLS * nown, 0.0);
    each([&] { k_tcoef(n, tri.data(), nrm.data(), sl.data(), dl.data(), 1, 1, 0.7, 0.6, 0.4, -1.0, tc.data()); });
    shaped([&](auto z) {
        using Z = decltype(z);
        launch<false, Z>(p, boxes, none, none, cen.data(), sides.data(), ss.data(), sc.data(), tri.data(), tc.data(), nc, whole.data());
        launch<false, Z>(p, boxes, none, none, cen.data(), sides.data(), ss.data(), sc.data(), tri.data(), tc.data(), nc, cut.data(), parts);
    });
    for (int r = 0; r < NRHS; r++)
        for (int l = 0; l <= p; l++) {
            LD num = 0, den = 0;
            for (int k = l * (l + 1); k < (l + 1) * (l + 2); k++) {
                LD w = whole[r * nc + k], e = cut[r * nc + k] - w;
                num += e * e;
                den += w * w;
            }
            if (den > 0) note(num, den);
        }
    for (int layer = 0; layer < 2; layer++) {
        each([&] { k_mind_tcoef(n, layer, tri.data(), nrm.data(), layer ? dl.data() : sl.data(), tc.data()); });
        MindMoments mm;
        for (int c = 0; c < 16; c++) mm.col[c] = layer ? (c < 12 ? 6 + c : -1) : (c < 6 ? c : -1);
        mm.G = (double2 *)G.data();
        shaped([&](auto z) {
            using Z = decltype(z);
            launch<false, Z, true>(p, boxes, none, none, cen.data(), sides.data(), ss.data(), sc.data(), tri.data(), tc.data(), nc, nullptr, parts, mm);
        });
    }
    std::vector<LD> want((size_t)2 * MindMoments::MCOLS * nown, 0);
    for (int i = 0; i < n; i++)
        for (int q = 0; q < nq; q++) {
            const double *r = RULE[(nq == 12 ? 6 : 0) + q], *t = &tri[9 * i], *nv = &nrm[3 * i], *b = &dl[3 * i];
            LD X[3], a[3], e[3], v[18];
            for (int k = 0; k < 3; k++) {
                a[k] = (LD)t[3 + k] - t[k], e[k] = (LD)t[6 + k] - t[k];
                X[k] = t[k] + r[0] * a[k] + r[1] * e[k];
            }
            LD cx = a[1] * e[2] - a[2] * e[1], cy = a[2] * e[0] - a[0] * e[2], cz = a[0] * e[1] - a[1] * e[0];
            LD w = r[2] * sqrtl(cx * cx + cy * cy + cz * cz);
            for (int k = 0; k < 3; k++) v[k] = w * sl[3 * i + k], v[6 + k] = w * (LD)b[k] * nv[k];
            v[9] = w * ((LD)b[0] * nv[1] + (LD)b[1] * nv[0]);
            v[10] = w * ((LD)b[0] * nv[2] + (LD)b[2] * nv[0]);
            v[11] = w * ((LD)b[1] * nv[2] + (LD)b[2] * nv[1]);
            for (int k = 0; k < 3; k++) v[3 + k] = v[k] * X[2];
            for (int k = 0; k < 6; k++) v[12 + k] = v[6 + k] * X[2];
            LD x = X[0] - cen[0], y = X[1] - cen[1], z = X[2] - cen[2], r2 = x * x + y * y + z * z, dr = 1, di = 0;
            for (int m = 0; m <= p; m++) {
                if (m) {
                    LD c = -sqrtl((2 * m - 1) / (LD)(2 * m)), nr = c * (x * dr - y * di);
                    di = c * (x * di + y * dr), dr = nr;
                }
                LD ar = 0, ai = 0, br = dr, bi = di;
                for (int l = m; l <= p; l++) {
                    for (int c = 0; c < 18; c++) {
                        LD *o = &want[2 * ((size_t)c * nown + l * (l + 1) / 2 + m)];
                        o[0] += v[c] * br;
                        o[1] += v[c] * bi;
                    }
                    LD dn = sqrtl((LD)(l + 1 + m) * (l + 1 - m)), k1 = (2 * l + 1) * z / dn, k2 = sqrtl((LD)(l + m) * (l - m)) * r2 / dn;
                    LD nr = k1 * br - k2 * ar, ni = k1 * bi - k2 * ai;
                    ar = br, ai = bi, br = nr, bi = ni;
                }
            }
        }
    for (int c = 0; c < 18; c++)
        for (int l = 0; l <= p; l++) {
            LD num = 0, den = 0;
            for (size_t k = (size_t)c * 2 * nown + l * (l + 1); k < (size_t)c * 2 * nown + (l + 1) * (l + 2); k++) {
                num += (G[k] - want[k]) * (G[k] - want[k]);
                den += want[k] * want[k];
            }
            note(num, den);
        }
    return worst;
}
