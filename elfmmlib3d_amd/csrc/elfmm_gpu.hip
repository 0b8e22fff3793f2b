// gfx950 kernels and host orchestration for the elastostatic triangle FMM.
//
// One apply of elfmm3dtriatarg (src/elfmm3dtria.f:162) runs as:
//   host:   octree + lists (bit-exact with the reference), interaction plan
//   device: gather into tree order -> per-triangle near-field records and
//           quadrature-node sources for the four Laplace problems
//           far field:  P2M -> M2M (per level) -> M2L -> P2L -> L2L (per
//                       level) -> L2T and M2T
//           near field: pair quadratures over self + list 1 (second stream)
//           assembly:   elastic combination + near field, scatter to the
//                       caller's order
// The four Laplace problems of elfmm3dtriatargmain_fast
// (src/elfmm3dtria.f:437-566) share one tree and run as four right-hand
// sides of every translation, so each operator matrix is applied to four
// vectors at once. All arithmetic is FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>
#include <utility>
#include <vector>

#include "../../include/elfmm_gfx950.h"
#include "elfmm_half.h"
#include "elfmm_internal.h"
#include "elfmm_math.h"
#include "elfmm_mindlin.h"
#include "elfmm_near.h"
#include "elfmm_octree.h"

namespace elfmm {
struct MindPlan;                                     // plan of the Mindlin far field (below)

// ------------------------------------------------------------------------
// constants and tables
// ------------------------------------------------------------------------

constexpr int PMAX = 44;                     // largest supported order
constexpr int SQN = (2 * PMAX + 6) * (2 * PMAX + 6);
constexpr int NRHS = 4;                      // Laplace problems per apply
constexpr int NODE_STRIDE = 20;              // X[3], q[4], d[4][3], pad

__device__ double g_sq[SQN];                 // sqrt(k)
__device__ double g_isq[SQN];                // 1/sqrt(k), 0 at k=0
__device__ double g_fact[2 * PMAX + 8];       // k!
__device__ double g_sdfact[PMAX + 4];         // (-1)^m (2m-1)!!
__device__ int g_coef_m[(PMAX + 1) * (PMAX + 2) / 2];   // order m of packed coefficient c

// D3-symmetric triangle rules on (0,0),(1,0),(0,1) as generated by the
// reference's triasymq (src/triasymq.f:26): (u, v, weight). The FMM forms
// expansions from the rule of order 1, 2, 3 or 6 by precision
// (src/lfmm3dtrilhess.f:619-640): 1, 3, 6 or 12 nodes, stored back to back.
__constant__ double c_qrule[22][3] = {
    // order 1
    {3.33333333333333259e-01, 3.33333333333333426e-01, 5.00000000000000000e-01},
    // order 2
    {1.66666666666666796e-01, 1.66666666666666657e-01, 1.66666666666666657e-01},
    {6.66666666666666630e-01, 1.66666666666666796e-01, 1.66666666666666657e-01},
    {1.66666666666666630e-01, 6.66666666666666741e-01, 1.66666666666666657e-01},
    // order 3
    {4.45948490915964835e-01, 1.08103018168070289e-01, 1.11690794839005750e-01},
    {4.45948490915964890e-01, 4.45948490915964946e-01, 1.11690794839005750e-01},
    {1.08103018168070192e-01, 4.45948490915965057e-01, 1.11690794839005750e-01},
    {9.15762135097709234e-02, 9.15762135097707153e-02, 5.49758718276609423e-02},
    {8.16847572980458403e-01, 9.15762135097709096e-02, 5.49758718276609423e-02},
    {9.15762135097707430e-02, 8.16847572980458514e-01, 5.49758718276609423e-02},
    // order 6 (src/triasymq.f:53-55)
    ELFMM_RULE6};

// Nodes per triangle and first row of c_qrule for a precision flag.
inline void quad_rule(int iprec, int &nq, int &q0)
{
    if (iprec <= -2) {
        nq = 1;
        q0 = 0;
    } else if (iprec == -1) {
        nq = 3;
        q0 = 1;
    } else if (iprec == 0) {
        nq = 6;
        q0 = 4;
    } else {
        nq = 12;
        q0 = 10;
    }
}

#define HIPOK(expr)                                                                      \
    do {                                                                                 \
        hipError_t e_ = (expr);                                                          \
        if (e_ != hipSuccess) {                                                          \
            std::fprintf(stderr, "elfmm_gfx950: %s failed: %s (%s:%d)\n", #expr,         \
                         hipGetErrorString(e_), __FILE__, __LINE__);                     \
            throw HipFailure{e_};                                                        \
        }                                                                                \
    } while (0)

struct HipFailure {
    hipError_t err;
};

// accumulator of one v_mfma_f64_16x16x4f64 (four doubles per lane)
typedef double gemm_d4 __attribute__((ext_vector_type(4)));

#include "elfmm_moments.h"

// order m of packed coefficient index c = l*(l+1)/2 + m (c < 2^20), from
// a float square root and one correction each way: no table load
__device__ __forceinline__ int coef_m(int c)
{
    int l = (int)((sqrtf(8.0f * (float)c + 1.0f) - 1.0f) * 0.5f);
    if ((l + 1) * (l + 2) / 2 <= c) l++;
    if (l * (l + 1) / 2 > c) l--;
    return c - l * (l + 1) / 2;
}


// Stream the integer-coefficient harmonics V_l^m = sqrt((l+m)!(l-m)!) R_l^m
// (IRR=false) or sqrt((l+m)!(l-m)!) I_l^m (IRR=true), 0 <= m <= l <= p,
// m-outer. Legendre recurrences with integer coefficients:
//   V_m^m = -(2m-1) (x+iy) V_{m-1}^{m-1} / r^{2 IRR},   V_0^0 = r^{-IRR}
//   V_l^m = ((2l-1) z V_{l-1}^m - (l+m-1)(l-m-1) r^{2(1-IRR)} V_{l-2}^m) / r^{2 IRR}
// so the dependent chain has no table loads; the normalisation
// 1/sqrt((l+m)!(l-m)!) is folded into whatever the values multiply.
template <bool IRR, class F>
__device__ __forceinline__ void stream_harm_u(int p, double x, double y, double z, F &&f)
{
    double r2 = x * x + y * y + z * z;
    double ir2 = IRR ? 1.0 / r2 : 1.0;
    double dr = IRR ? sqrt(ir2) : 1.0, di = 0.0;
    double zz = z * ir2, rr = IRR ? ir2 : r2;
    for (int m = 0; m <= p; m++) {
        if (m > 0) {
            double c = -(double)(2 * m - 1) * ir2;
            double nr = c * (x * dr - y * di), ni = c * (x * di + y * dr);
            dr = nr;
            di = ni;
        }
        double ar = dr, ai = di;
        f(m, m, ar, ai);
        if (m + 1 > p) continue;
        double cz = (double)(2 * m + 1) * zz;
        double br = cz * ar, bi = cz * ai;
        f(m + 1, m, br, bi);
        for (int l = m + 2; l <= p; l++) {
            double k1 = (double)(2 * l - 1) * zz;
            double k2 = (double)((l + m - 1) * (l - m - 1)) * rr;
            double cr = k1 * br - k2 * ar, ci = k1 * bi - k2 * ai;
            f(l, m, cr, ci);
            ar = br;
            ai = bi;
            br = cr;
            bi = ci;
        }
    }
}

// ------------------------------------------------------------------------
// setup kernels
// ------------------------------------------------------------------------

__global__ void k_tables()
{
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < SQN; k += gridDim.x * blockDim.x) {
        g_sq[k] = sqrt((double)k);
        g_isq[k] = k ? 1.0 / sqrt((double)k) : 0.0;
    }
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < (PMAX + 1) * (PMAX + 2) / 2;
         c += gridDim.x * blockDim.x) {
        int l = 0;
        while ((l + 1) * (l + 2) / 2 <= c) l++;
        g_coef_m[c] = c - l * (l + 1) / 2;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        double d = 1.0;
        for (int m = 0; m < PMAX + 4; m++) {
            g_sdfact[m] = d;
            d *= -(double)(2 * m + 1);
        }
        double f = 1.0;
        for (int k = 0; k < 2 * PMAX + 8; k++) {
            g_fact[k] = f;
            f *= (double)(k + 1);
        }
    }
}

// Gather inputs into tree order; per-triangle near-field records.
__global__ void k_gather(int n, int nt, const int *__restrict__ iz, const int *__restrict__ izt,
                         const double *__restrict__ tri, const double *__restrict__ nrm,
                         const double *__restrict__ src, int ifsl, const double *__restrict__ ssl,
                         int ifdl, const double *__restrict__ sdl, const double *__restrict__ tgt,
                         double *__restrict__ tri_s, double *__restrict__ nrm_s,
                         double *__restrict__ ssl_s, double *__restrict__ sdl_s,
                         double *__restrict__ pts, double *__restrict__ rec)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        int o = iz[i];
        double t[9], s1[3], s2[3];
        for (int d = 0; d < 9; d++) t[d] = tri[9 * (size_t)o + d];
        for (int d = 0; d < 3; d++) {
            s1[d] = ifsl ? ssl[3 * (size_t)o + d] : 0.0;
            s2[d] = ifdl ? sdl[3 * (size_t)o + d] : 0.0;
            nrm_s[3 * (size_t)i + d] = nrm[3 * (size_t)o + d];
            ssl_s[3 * (size_t)i + d] = s1[d];
            sdl_s[3 * (size_t)i + d] = s2[d];
            pts[3 * (size_t)i + d] = src[3 * (size_t)o + d];
        }
        for (int d = 0; d < 9; d++) tri_s[9 * (size_t)i + d] = t[d];
        nf_make_record(t, s1, s2, rec + (size_t)i * NF_REC);
    } else if (i < n + nt) {
        int j = i - n;
        int o = izt[j];
        for (int d = 0; d < 3; d++) pts[3 * (size_t)i + d] = tgt[3 * (size_t)o + d];
    }
}

// Quadrature-node sources of the four Laplace problems
// (src/elfmm3dtria.f:449-492 constant densities j=1..3 and :508-547 the
// vertex-linear problem), interpolated with the reference's node formula
// (src/lfmm3dtrilhess.f:1340-1364) and weight*2*area.
__global__ void k_nodes(int n, int nq, int q0, const double *__restrict__ tri_s, const double *__restrict__ nrm_s,
                        const double *__restrict__ ssl_s, const double *__restrict__ sdl_s,
                        int ifsl, int ifdl, double rmu, double c1, double c2, double dls,
                        double *__restrict__ nodes)
{
    int gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= nq * n) return;
    int i = gid / nq, qn = q0 + gid % nq;
    const double *t = tri_s + 9 * (size_t)i;
    double u = c_qrule[qn][0], v = c_qrule[qn][1];
    double X[3];
    for (int d = 0; d < 3; d++) X[d] = t[d] + u * (t[3 + d] - t[d]) + v * (t[6 + d] - t[d]);
    double ax = t[3] - t[0], ay = t[4] - t[1], az = t[5] - t[2];
    double bx = t[6] - t[0], by = t[7] - t[1], bz = t[8] - t[2];
    double cx = ay * bz - az * by, cy = az * bx - ax * bz, cz = ax * by - ay * bx;
    double area = 0.5 * sqrt(cx * cx + cy * cy + cz * cz);
    double w = c_qrule[qn][2] * (area * 2);
    const double *nv = nrm_s + 3 * (size_t)i, *sl = ssl_s + 3 * (size_t)i;
    const double dl[3] = {dls * sdl_s[3 * (size_t)i], dls * sdl_s[3 * (size_t)i + 1], dls * sdl_s[3 * (size_t)i + 2]};
    double *o = nodes + (size_t)gid * NODE_STRIDE;
    o[0] = X[0];
    o[1] = X[1];
    o[2] = X[2];
    for (int j = 0; j < 3; j++) {
        o[3 + j] = ifsl ? w * (sl[j] / (2 * rmu)) : 0.0;
        for (int d = 0; d < 3; d++)
            o[7 + 3 * j + d] = ifdl ? w * ((nv[d] * dl[j] + dl[d] * nv[j]) / 2) : 0.0;
    }
    double cv[3], dv[3][3];
    for (int m = 0; m < 3; m++) {
        const double *V = t + 3 * m;
        cv[m] = 0.0;
        if (ifsl) cv[m] = (sl[0] * V[0] + sl[1] * V[1] + sl[2] * V[2]) * c1 / (2 * rmu);
        if (ifdl) cv[m] += (dl[0] * nv[0] + dl[1] * nv[1] + dl[2] * nv[2]) * c2;
        double sv = dl[0] * V[0] + dl[1] * V[1] + dl[2] * V[2];
        double nvv = nv[0] * V[0] + nv[1] * V[1] + nv[2] * V[2];
        for (int d = 0; d < 3; d++) dv[m][d] = ifdl ? (c1 * nv[d] * sv + c1 * dl[d] * nvv) / 2 : 0.0;
    }
    o[6] = w * (cv[0] + u * (cv[1] - cv[0]) + v * (cv[2] - cv[0]));
    for (int d = 0; d < 3; d++) o[16 + d] = w * (dv[0][d] + u * (dv[1][d] - dv[0][d]) + v * (dv[2][d] - dv[0][d]));
    o[19] = 0.0;
}

// ------------------------------------------------------------------------
// P2M and P2L: quadrature nodes -> expansion, one workgroup per box
// ------------------------------------------------------------------------

// Column m of the unnormalised harmonics of one point, stored in stream
// order: V_l^m at doubles 2*pos and 2*pos + 1, pos = m*(ph+1) - m*(m-1)/2
// + (l - m); sdf = (-1)^m (2m-1)!!. The diagonal term in closed form,
//   V_m^m = (-1)^m (2m-1)!! (x+iy)^m / r^(2m IRR) * r^(-IRR),
// by binary powering, then up the column (l = m..ph) with the integer
// Legendre recurrence of stream_harm_u,
//   V_l^m = ((2l-1) z V_{l-1}^m - (l+m-1)(l-m-1) r^{2(1-IRR)} V_{l-2}^m) / r^{2 IRR}.
template <bool IRR>
__device__ __forceinline__ void harm_column_stream(int ph, int m, double sdf, double x, double y, double z,
                                                   double *H)
{
    double r2 = x * x + y * y + z * z;
    double ir2 = IRR ? 1.0 / r2 : 1.0;
    double zz = z * ir2, rr = IRR ? ir2 : r2;
    double ur = x * ir2, ui = y * ir2;                 // (x+iy) / r^(2 IRR)
    double dr = sdf * (IRR ? sqrt(ir2) : 1.0), di = 0.0;
    for (int e = m; e; e >>= 1) {
        if (e & 1) {
            double t = dr * ur - di * ui;
            di = dr * ui + di * ur;
            dr = t;
        }
        double t = ur * ur - ui * ui;
        ui = 2.0 * ur * ui;
        ur = t;
    }
    double2 *o = (double2 *)(H + 2 * (m * (ph + 1) - m * (m - 1) / 2));
    double ar = dr, ai = di;
    o[0] = double2{ar, ai};
    if (m + 1 > ph) return;
    double k1 = (double)(2 * m + 1);
    double br = k1 * zz * ar, bi = k1 * zz * ai;
    o[1] = double2{br, bi};
    // l = m+2..ph: (2l-1) and (l+m-1)(l-m-1), each step adding 2 and (2l-1)
    double k1c = (double)(2 * m + 3), k2c = (double)(2 * m + 1);
    for (int t = 2; t <= ph - m; t++) {
        double f1 = k1c * zz, f2 = k2c * rr;
        double cr = f1 * br - f2 * ar, ci = f1 * bi - f2 * ai;
        o[t] = double2{cr, ci};
        ar = br;
        ai = bi;
        br = cr;
        bi = ci;
        k2c += k1c;
        k1c += 2.0;
    }
}

// P2M (IRR=false: multipole of a leaf from its own quadrature nodes,
// overwrite) and P2L (IRR=true: local expansion of a box from the nodes of
// its list-4 boxes, add) on the FP64 matrix cores. The node sums are
// formed first as moments
//   M[c16][row] = sum_nodes w_c16(node) V_row(node),
// c16 = the 16 node weights (charge of rhs 0-3, then the dipole of rhs 0-3,
// x y z each) and row = 2*pos + part over the harmonics V up to degree ph
// (p, or p + 1 for P2L) in stream order: one 16 x 16 x 4 product per four
// nodes and 16 rows. Wave w of the WB waves accumulates row tiles w, w+WB,
// ... (TW of them; the LDS rows are padded with zeros to WB * TW tiles and
// the products of tiles past the last are dropped). The harmonics of NK nodes at a time are built in LDS, one
// (node, order) column per thread. The expansion coefficients then follow from the
// moments: charge term from V_l^m, dipole term through the gradient
// ladders from degree l - 1 (l + 1 for P2L), orders m, m +- 1.
template <bool IRR, int WB, int TW, int NK>
__device__ __forceinline__ void p2x_body(
    int p, int nq, int stride, const int *__restrict__ boxes, const int *__restrict__ lstart,
    const int *__restrict__ litems, const double *__restrict__ centers,
    const double *__restrict__ sides, const int *__restrict__ src_start,
    const int *__restrict__ src_count, const double *__restrict__ nodes, int nc,
    double *__restrict__ expn)
{
    extern __shared__ double lds[];
    int ph = IRR ? p + 1 : p;
    int ntiles = ((ph + 1) * (ph + 2) + 15) / 16;
    int box = boxes[blockIdx.x];
    double s = sides[box], is = 1.0 / s;
    double cx = centers[3 * box], cy = centers[3 * box + 1], cz = centers[3 * box + 2];
    int lane = threadIdx.x & 63;
    int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int kq = lane >> 4, n16 = lane & 15;
    for (int e = threadIdx.x; e < NK * stride; e += blockDim.x) lds[e] = 0.0;   // padding rows stay zero
    gemm_d4 acc[TW];
#pragma unroll
    for (int j = 0; j < TW; j++) acc[j] = gemm_d4{0.0, 0.0, 0.0, 0.0};
    // this thread's harmonic column for every chunk: node gk, order gm
    int gk = threadIdx.x / (ph + 1), gm = threadIdx.x - gk * (ph + 1);
    double gsdf = g_sdfact[min(gm, PMAX + 3)];        // loaded once: no table load inside the chunk loop
    int ns = IRR ? lstart[blockIdx.x + 1] - lstart[blockIdx.x] : 1;
    // chunks (source box sb, first node n0) in order; the node record of
    // this thread's column and the node weights of its operand lanes are
    // loaded one chunk ahead
    auto box_nodes = [&](int sb_, int &nn_) {
        int sbox = IRR ? litems[lstart[blockIdx.x] + sb_] : box;
        nn_ = nq * src_count[sbox];
        return nodes + (size_t)nq * src_start[sbox] * NODE_STRIDE;
    };
    int sb = 0, n0 = 0, nn = 0;
    const double *nd = ns > 0 ? box_nodes(0, nn) : nullptr;
    while (sb < ns && nn == 0) {
        sb++;
        if (sb < ns) nd = box_nodes(sb, nn);
    }
    double gx = 0.0, gy = 0.0, gz = 0.0, wa[NK / 4];
    auto fetch = [&](const double *nd_, int n0_, int cnt_) {
        if (gk < cnt_) {
            const double *X = nd_ + (size_t)(n0_ + gk) * NODE_STRIDE;
            gx = X[0];                                // raw: no wait on the load here
            gy = X[1];
            gz = X[2];
        }
#pragma unroll
        for (int ks = 0; ks < NK / 4; ks++) {
            int k = 4 * ks + kq;
            wa[ks] = k < cnt_ ? nd_[(size_t)(n0_ + k) * NODE_STRIDE + 3 + n16] : 0.0;
        }
    };
    if (sb < ns) fetch(nd, 0, min(NK, nn));
    while (sb < ns) {
        int cnt = min(NK, nn - n0);
        double cxg = gx, cyg = gy, czg = gz, cwa[NK / 4];
#pragma unroll
        for (int ks = 0; ks < NK / 4; ks++) cwa[ks] = wa[ks];
        // advance to the next chunk and start its loads
        {
            int nsb = sb, nn0 = n0 + NK, nnn = nn;
            const double *nnd = nd;
            while (nsb < ns && nn0 >= nnn) {
                nsb++;
                nn0 = 0;
                if (nsb < ns) nnd = box_nodes(nsb, nnn);
            }
            if (nsb < ns) fetch(nnd, nn0, min(NK, nnn - nn0));
            __syncthreads();                          // previous chunk's products done
            if (gk < NK) {
                double *H = lds + (size_t)gk * stride;
                if (gk < cnt) {
                    harm_column_stream<IRR>(ph, gm, gsdf, (cxg - cx) * is, (cyg - cy) * is, (czg - cz) * is, H);
                } else {
                    int b0 = 2 * (gm * (ph + 1) - gm * (gm - 1) / 2);
                    for (int t = 0; t <= 2 * (ph - gm) + 1; t++) H[b0 + t] = 0.0;
                }
            }
            sb = nsb;
            n0 = nn0;
            nn = nnn;
            nd = nnd;
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < NK / 4; ks++) {
            const double *Hk = lds + (size_t)(4 * ks + kq) * stride + 16 * w + n16;
            double b[TW];
#pragma unroll
            for (int j = 0; j < TW; j++) b[j] = Hk[16 * WB * j];
#pragma unroll
            for (int j = 0; j < TW; j++) acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(cwa[ks], b[j], acc[j], 0, 0, 0);
        }
    }
    // coefficients, one right-hand side at a time: its four moment columns
    // (charge, dipole x y z) go to LDS, then one thread per coefficient
    int nco = (p + 1) * (p + 2) / 2;
    double f0s = IRR ? is : 1.0;
    double f1s = IRR ? is * is : is;
    double *Ms = lds;                                 // 4 x stride
    for (int r = 0; r < NRHS; r++) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < TW; j++) {
            int T = w + WB * j;
            if (T >= ntiles) continue;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                int c16 = kq + 4 * i;
                int col = c16 == r ? 0 : (c16 >= 4 && (c16 - 4) / 3 == r ? 1 + (c16 - 4) % 3 : -1);
                if (col >= 0) Ms[col * stride + 16 * T + n16] = acc[j][i];
            }
        }
        __syncthreads();
        // moment (column col, degree ll, order mm >= -1); order -1 = -conj(order 1)
        auto mget = [&](int col, int ll, int mm, double &re, double &im) {
            int am = mm < 0 ? -mm : mm;
            if (ll < 0 || ll > ph || am > ll) {
                re = 0.0;
                im = 0.0;
                return;
            }
            int row = 2 * (am * (ph + 1) - am * (am - 1) / 2 + (ll - am));
            re = Ms[col * stride + row];
            im = Ms[col * stride + row + 1];
            if (mm < 0) re = -re;
        };
        for (int c = threadIdx.x; c < nco; c += blockDim.x) {
            int l, m;
            coef_nk(c, l, m);
            int ld = IRR ? l + 1 : l - 1;
            double fh = hnorm(l, m) * f0s, fp, fm, fz;
            if (!IRR) {
                bool vp = ld >= 0 && m + 1 <= ld, vm = ld >= 0 && m - 1 <= ld && m + ld > 0, vz = ld >= 0 && m <= ld;
                fp = vp ? sqrt((double)((l - m) * (l - m - 1))) * hnorm(ld, m + 1) : 0.0;
                fm = vm ? sqrt((double)((l + m) * (l + m - 1))) * hnorm(ld, m - 1) : 0.0;
                fz = vz ? sqrt((double)((l - m) * (l + m))) * hnorm(ld, m) : 0.0;
            } else {
                fp = sqrt((double)((l + m + 1) * (l + m + 2))) * hnorm(l + 1, m + 1);
                fm = sqrt((double)((l - m + 1) * (l - m + 2))) * hnorm(l + 1, m - 1);
                fz = -sqrt((double)((l - m + 1) * (l + m + 1))) * hnorm(l + 1, m);
            }
            fp *= 0.5 * f1s;
            fm *= 0.5 * f1s;
            fz *= f1s;
            double qr, qi, xpr, xpi, ypr, ypi, xmr, xmi, ymr, ymi, zr, zi;
            mget(0, l, m, qr, qi);
            mget(1, ld, m + 1, xpr, xpi);
            mget(2, ld, m + 1, ypr, ypi);
            mget(1, ld, m - 1, xmr, xmi);
            mget(2, ld, m - 1, ymr, ymi);
            mget(3, ld, m, zr, zi);
            // conj(q V + d.grad V), d.grad V through the ladders
            double re = fh * qr + fp * (xpr + ypi) + fm * (ymi - xmr) + fz * zr;
            double im = -fh * qi + fp * (ypr - xpi) + fm * (xmi + ymr) - fz * zi;
            double *e = expn + ((size_t)box * NRHS + r) * nc + 2 * c;
            if (IRR) {
                e[0] += re;
                e[1] += im;
            } else {
                e[0] = re;
                e[1] = im;
            }
        }
    }
}

template <int WB, int TW, int NK>
__global__ __launch_bounds__(64 * WB, TW <= 7 ? 4 : 2) void k_p2m(
    int p, int nq, int stride, const int *__restrict__ boxes, const int *__restrict__ lstart,
    const int *__restrict__ litems, const double *__restrict__ centers,
    const double *__restrict__ sides, const int *__restrict__ src_start,
    const int *__restrict__ src_count, const double *__restrict__ nodes, int nc,
    double *__restrict__ expn)
{
    p2x_body<false, WB, TW, NK>(p, nq, stride, boxes, lstart, litems, centers, sides, src_start, src_count, nodes, nc, expn);
}

template <int WB, int TW, int NK>
__global__ __launch_bounds__(64 * WB, TW <= 7 ? 4 : 2) void k_p2l(
    int p, int nq, int stride, const int *__restrict__ boxes, const int *__restrict__ lstart,
    const int *__restrict__ litems, const double *__restrict__ centers,
    const double *__restrict__ sides, const int *__restrict__ src_start,
    const int *__restrict__ src_count, const double *__restrict__ nodes, int nc,
    double *__restrict__ expn)
{
    p2x_body<true, WB, TW, NK>(p, nq, stride, boxes, lstart, litems, centers, sides, src_start, src_count, nodes, nc, expn);
}



// P2M and P2L of triangles through their moments (elfmm_moments.h)
template <class Z, bool MIND>
__global__ __launch_bounds__(Z::NT, 2) void k_p2m_tri(
    int p, const int *__restrict__ boxes, const int *__restrict__ parts, MindMoments mind,
    const double *__restrict__ centers, const double *__restrict__ sides, const int *__restrict__ src_start,
    const int *__restrict__ src_count, const double *__restrict__ tri_s, const double *__restrict__ tcoef, int nc,
    double *__restrict__ expn)
{
    extern __shared__ double lds[];                  // no static LDS beside it: it starts at 0
    p2t_body<false, Z, MIND>(p, boxes, parts, mind, nullptr, nullptr, centers, sides, src_start, src_count, tri_s,
                             tcoef, nc, expn, lds);
}

template <class Z>
__global__ __launch_bounds__(Z::NT, 2) void k_p2l_tri(
    int p, const int *__restrict__ boxes, const int *__restrict__ lstart, const int *__restrict__ litems,
    const double *__restrict__ centers, const double *__restrict__ sides, const int *__restrict__ src_start,
    const int *__restrict__ src_count, const double *__restrict__ tri_s, const double *__restrict__ tcoef, int nc,
    double *__restrict__ expn)
{
    extern __shared__ double lds[];                  // no static LDS beside it: it starts at 0
    p2t_body<true, Z, false>(p, boxes, nullptr, MindMoments{}, lstart, litems, centers, sides, src_start, src_count,
                             tri_s, tcoef, nc, expn, lds);
}

// ------------------------------------------------------------------------
// Translations (M2L, M2M, L2L) on the matrix cores
// ------------------------------------------------------------------------

// M2L of the lower orders (tiles with h < h_turned), with the translation
// rotated into the xz-plane: per pair, x' = e^{i m phi} x (coefficient-wise), y'_re = R x'_re,
// y'_im = I x'_im with the operator's two real h x h matrices, then
// y = e^{-i k phi} y', scaled (1/s of the target box) and added to the
// destination expansion. A tile is ML_M = 64 output coefficients for ML_P = 32
// pairs x NRHS right-hand sides (128 columns). Wave w owns coefficients
// 16*(w/2) .. +16 and columns 64*(w%2) .. +64: 4 column blocks of 16 x 16
// accumulators for the real parts and 4 for the imaginary parts, so the
// output rotation pairs values held by the same lane.
constexpr int ML_THREADS = 512;
constexpr int ML_K = 8;
constexpr int MA_LD = ML_K + 1;
constexpr int MB_LD = ML_P * NRHS + 2;
constexpr int ML_ST_LD = 2 * ML_M + 2;               // doubles per staged output column (padded)
constexpr int ML_OPER = 2 * ML_M * MA_LD + 2 * ML_K * MB_LD;
constexpr int ML_SMEM = 2 * ML_OPER > 32 * ML_ST_LD ? 2 * ML_OPER : 32 * ML_ST_LD;   // two operand buffers
constexpr int ML_APER = ML_M * ML_K / ML_THREADS;    // operator entries per thread and matrix
constexpr int ML_BPER = ML_P * NRHS * ML_K / ML_THREADS;   // source entries per thread
static_assert(ML_APER >= 1 && ML_BPER >= 1 && ML_K % 4 == 0, "loader shapes");

__global__ __launch_bounds__(ML_THREADS, 4) void k_m2l(const M2LTile *__restrict__ tiles, int ntiles, int h_turned,
                                                    const double *__restrict__ A_all,
                                                    const int *__restrict__ psrc,
                                                    const int *__restrict__ pdst,
                                                    const double *__restrict__ pscale,
                                                    const double *__restrict__ X, double *__restrict__ Y,
                                                    int nc)
{
    // operand tiles during the products (two buffers: step k0 + ML_K is
    // written while step k0 is multiplied); the output staging afterwards
    __shared__ double smem[ML_SMEM];
    // (cos m phi, sin m phi) of each packed coefficient k = l(l+1)/2 + m,
    // zero past h up to the next multiple of ML_M (rows and K steps of the
    // last tile read there)
    constexpr int CSK_N = ((PMAX + 1) * (PMAX + 2) / 2 + ML_M - 1) / ML_M * ML_M;
    __shared__ double2 csk[CSK_N];
    // the tiles come in launch order (workgroup b on XCD b % 8); empty
    // tiles fill the slots past an XCD's last one
    int tix = blockIdx.x;
    if (tix >= ntiles) return;
    M2LTile t = tiles[tix];
    if (t.npair <= 0 || t.h >= h_turned) return;
    const double *Rm = A_all + t.a_off, *Im = Rm + (size_t)t.h * t.h;
    int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int wr = (wave >> 1) * 16, wc = (wave & 1) * 64;
    // a wave whose 16 rows all lie past the operator's last row (h is not a
    // multiple of ML_M) only helps load: its products would be zero
    const bool rows_on = t.row0 + wr < t.h;
    for (int k = tid; k < (t.h + ML_M - 1) / ML_M * ML_M; k += ML_THREADS) {
        double sn = 0.0, c = 0.0;
        if (k < t.h) {
            int l, m;
            coef_nk(k, l, m);
            sincos(m * t.phi, &sn, &c);
            // the operator of the z-mirrored offset: (-1)^(l+m) on input and output
            if (t.refl && ((l + m) & 1)) {
                sn = -sn;
                c = -c;
            }
        }
        csk[k] = double2{c, sn};
    }
    // loaders: A ML_M rows x ML_K k (ML_APER per thread per matrix); B
    // ML_P * NRHS columns x ML_K coefficients (ML_BPER per thread, real and
    // imaginary part each)
    int ar = tid / (ML_K / ML_APER), ak = (tid % (ML_K / ML_APER)) * ML_APER;
    int arow = t.row0 + ar;
    bool arow_ok = arow < t.h;
    int bc = tid / (ML_K / ML_BPER), bk = (tid % (ML_K / ML_BPER)) * ML_BPER;
    int bpair = bc / NRHS, brhs = bc % NRHS;
    int bsrc = bpair < t.npair ? psrc[t.pair0 + bpair] : -1;
    const double *Xc = bsrc >= 0 ? X + ((size_t)bsrc * NRHS + brhs) * nc : nullptr;
    gemm_d4 accr[4], acci[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        accr[j] = gemm_d4{0.0, 0.0, 0.0, 0.0};
        acci[j] = gemm_d4{0.0, 0.0, 0.0, 0.0};
    }
    int li = lane & 15, lq = lane >> 4;
    // operands of K chunk k0 into registers: operator rows as stored, the
    // source coefficients raw (rotated when written to LDS)
    double a_r[ML_APER], a_i[ML_APER], x_r[ML_BPER], x_i[ML_BPER];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int q = 0; q < ML_APER; q++) {
            int k = k0 + ak + q;
            bool ok = arow_ok && k < t.h;
            a_r[q] = ok ? Rm[(size_t)arow * t.h + k] : 0.0;
            a_i[q] = ok ? Im[(size_t)arow * t.h + k] : 0.0;
        }
#pragma unroll
        for (int q = 0; q < ML_BPER; q++) {
            int k = k0 + bk + q;
            bool ok = Xc && k < t.h;
            x_r[q] = ok ? Xc[2 * k] : 0.0;
            x_i[q] = ok ? Xc[2 * k + 1] : 0.0;
        }
    };
    // registers -> LDS buffer b (the source coefficients rotated on the way)
    auto store = [&](int b, int k0) {
        double *Ar = smem + b * ML_OPER, *Ai = Ar + ML_M * MA_LD;
        double *Br = Ar + 2 * ML_M * MA_LD, *Bi = Br + ML_K * MB_LD;
#pragma unroll
        for (int q = 0; q < ML_APER; q++) {
            Ar[ar * MA_LD + ak + q] = a_r[q];
            Ai[ar * MA_LD + ak + q] = a_i[q];
        }
#pragma unroll
        for (int q = 0; q < ML_BPER; q++) {
            double2 e = csk[k0 + bk + q];
            Br[(bk + q) * MB_LD + bc] = e.x * x_r[q] - e.y * x_i[q];
            Bi[(bk + q) * MB_LD + bc] = e.y * x_r[q] + e.x * x_i[q];
        }
    };
    fetch(0);
    __syncthreads();                                  // rotation table ready
    store(0, 0);
    if (ML_K < t.h) fetch(ML_K);
    __syncthreads();
    int b = 0;
    for (int k0 = 0; k0 < t.h; k0 += ML_K, b ^= 1) {
        // buffer b holds step k0; buffer b ^ 1 was last read before the
        // previous barrier, so it takes step k0 + ML_K during the products
        if (rows_on) {
            const double *Ar = smem + b * ML_OPER, *Ai = Ar + ML_M * MA_LD;
            const double *Br = Ar + 2 * ML_M * MA_LD, *Bi = Br + ML_K * MB_LD;
#pragma unroll
            for (int ks = 0; ks < ML_K; ks += 4) {
                double a0 = Ar[(wr + li) * MA_LD + ks + lq];
                double a1 = Ai[(wr + li) * MA_LD + ks + lq];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    double br = Br[(ks + lq) * MB_LD + wc + j * 16 + li];
                    double bi = Bi[(ks + lq) * MB_LD + wc + j * 16 + li];
                    accr[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, br, accr[j], 0, 0, 0);
                    acci[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, bi, acci[j], 0, 0, 0);
                }
            }
        }
        if (k0 + ML_K < t.h) {
            store(b ^ 1, k0 + ML_K);
            if (k0 + 2 * ML_K < t.h) fetch(k0 + 2 * ML_K);   // in flight during the next products
        }
        __syncthreads();                              // buffer b ^ 1 written, buffer b free
    }
    // Output in four passes of 32 columns (column block j of both column
    // halves): the rotated, scaled results go to LDS, then each wave adds
    // 64 consecutive doubles of one destination expansion (FP64 atomics:
    // several source boxes feed one destination).
    constexpr int ST_LD = ML_ST_LD;
    static_assert(32 * ST_LD <= ML_SMEM, "staging fits the operand LDS");
    for (int j = 0; j < 4; j++) {
        __syncthreads();                              // products (or previous pass) done with LDS
        int cidx = (wc >> 6) * 16 + li;               // staged column of this lane
        int col = wc + j * 16 + li;
        int pair = col / NRHS;
        double sc = pair < t.npair ? pscale[t.pair0 + pair] : 0.0;
        // lane holds coefficients lane/16 + 4 r of its 16-row block, column lane % 16
#pragma unroll
        for (int rr = 0; rr < 4; rr++) {
            int rl = wr + lq + 4 * rr;
            double2 e = csk[t.row0 + rl];
            double yr = accr[j][rr], yi = acci[j][rr];
            smem[cidx * ST_LD + 2 * rl] = (e.x * yr + e.y * yi) * sc;
            smem[cidx * ST_LD + 2 * rl + 1] = (e.x * yi - e.y * yr) * sc;
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < 32 * 2 * ML_M / ML_THREADS; it++) {
            int g = it * ML_THREADS + tid;
            int cc = g / (2 * ML_M), o = g - cc * (2 * ML_M);
            int gcol = (cc >> 4) * 64 + j * 16 + (cc & 15);
            int gp = gcol / NRHS, r = gcol % NRHS;
            int co = t.row0 + (o >> 1);
            if (gp >= t.npair || co >= t.h) continue;
            double *y = Y + ((size_t)pdst[t.pair0 + gp] * NRHS + r) * nc;
            unsafeAtomicAdd(&y[2 * t.row0 + o], smem[cc * ST_LD + o]);
        }
    }
}

// M2M, L2L and M2L of the higher orders: a translation is rotated about z (e^{i m
// phi} per coefficient), then about y so that it points along z, applied there,
// and rotated back: the rotations mix
// the orders of one degree, the shift the degrees of one order, and real and
// imaginary parts stay apart, so a part goes through three block-diagonal
// products of (p+1)^3 / 3 multiplications each instead of one dense product of
// (p+1)^4 / 4 (order 26: 0.08 M to 0.29 M a pair and right-hand side, both
// parts). M2M and L2L of 16,400 pairs at order 26: 0.89 ms, dense 1.49; the
// M2L orders of 22 and more of 303,000 pairs 2.9 ms, dense 4.2; what is left is
// the address arithmetic, the barriers and the adds, not the matrix cores. The
// result is scaled (1/s of the target box for M2L, 1 for M2M and L2L) and added
// to the destination expansion (FP64 atomics: several sources feed one).
//
// A workgroup takes TR_P = 4 pairs x NRHS right-hand sides, the 16 columns of a
// matrix-core tile: the tile list is that of the dense products, the 8 parts
// of a tile's 32 pairs are dealt to the group's row blocks (grid: tiles x
// most parts of a row block). One part's coefficients stay in LDS, [coefficient][column],
// through its three products, the other part's in registers. A unit of work is
// 16 rows of one block: its operand comes from L2 as the matrix cores read it
// (build_operators), the next unit's in flight during the products of this
// one; the units, longest first, go to the W waves to and fro, and a product is
// written back once all waves have read its operands. U units a wave, EJ
// coefficients a lane and column, KM steps a unit at most.
constexpr int TR_P = 4, TR_LD = TR_P * NRHS + 1;
static_assert(TR_P * NRHS == 16, "columns of a matrix-core tile");
struct TransTab {
    int v[PMAX + 3];
};
constexpr TransTab make_trans_tab()
{
    TransTab t{};
    for (int n = 0; n < PMAX + 3; n++) t.v[n] = (int)trans_blocks(n);
    return t;
}
__constant__ const TransTab c_trans = make_trans_tab();

// rows of LDS at order p: three degrees of zeros past the last
__host__ __device__ constexpr int tr_rows(int p) { return (p + 4) * (p + 5) / 2; }
inline size_t trans_lds(int p) { return (size_t)tr_rows(p) * TR_LD * 8; }

template <int W, int U, int EJ, int KM>
__device__ __forceinline__ void trans_tile(const M2LTile *__restrict__ tiles, int ntiles, int h_turned,
                                           const double *__restrict__ A_all, const int *__restrict__ psrc,
                                           const int *__restrict__ pdst, const double *__restrict__ pscale,
                                           const double *__restrict__ X, double *__restrict__ Y, int nc, double *S)
{
    constexpr int C = 16 / W;                         // columns of a wave
    __shared__ double2 cs[PMAX + 1];                  // (cos m phi, sin m phi)
    // the tiles come in launch order (workgroup b on XCD b % 8); empty
    // tiles fill the slots past an XCD's last one
    if ((int)blockIdx.x >= ntiles) return;
    const M2LTile t = tiles[blockIdx.x];
    if (t.npair <= 0 || t.h < h_turned) return;
    const int nrb = (t.h + ML_M - 1) / ML_M, rb = t.row0 / ML_M, parts = ML_P / TR_P;
    const int sub = (parts * rb + nrb - 1) / nrb + (int)blockIdx.y;
    if (sub >= (parts * (rb + 1) + nrb - 1) / nrb || sub * TR_P >= t.npair) return;
    const int pair0 = t.pair0 + sub * TR_P, npair = min(TR_P, t.npair - sub * TR_P);
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = t.h, N = (int)((sqrtf(8.0f * h + 1.0f) - 1.0f) * 0.5f + 0.5f);   // p + 1
    if (tid < N) {
        double sn, c;
        sincos(tid * t.phi, &sn, &c);
        cs[tid] = double2{c, sn};
    }
    // the wave's columns, lane = coefficient
    double2 x[C][EJ];
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int col = wave + W * c, pair = col / NRHS;
        const bool on = pair < npair;
        const double2 *Xc =
            reinterpret_cast<const double2 *>(X + ((size_t)(on ? psrc[pair0 + pair] : 0) * NRHS + col % NRHS) * nc);
#pragma unroll
        for (int j = 0; j < EJ; j++) x[c][j] = on && lane + 64 * j < h ? Xc[lane + 64 * j] : double2{0.0, 0.0};
    }
    __syncthreads();
    auto phase = [&](int k) {                         // and the signs (-1)^(l+m) of a z-mirrored operator
        int l, m;
        coef_nk(k, l, m);
        double2 e = cs[m];
        return t.refl && ((l + m) & 1) ? double2{-e.x, -e.y} : e;
    };
    for (int k = h * TR_LD + tid; k < tr_rows(N - 1) * TR_LD; k += 64 * W) S[k] = 0.0;
    double keep[C][EJ];
#pragma unroll
    for (int j = 0; j < EJ; j++) {
        const int k = lane + 64 * j;
        if (k >= h) continue;
        const double2 e = phase(k);
#pragma unroll
        for (int c = 0; c < C; c++) {
            S[k * TR_LD + wave + W * c] = e.x * x[c][j].x - e.y * x[c][j].y;
            keep[c][j] = e.y * x[c][j].x + e.x * x[c][j].y;
        }
    }
    // unit s of the wave: size n of its block (0: none) and row tile rt
    auto unit = [&](int s, int &n, int &rt) {
        int u = W * s + (s & 1 ? W - 1 - wave : wave), c3 = max(N - 32, 0) * 3;
        if (u < c3) {
            n = N - u / 3;
            rt = u % 3;
            return;
        }
        u -= c3;
        int top = min(N, 32), c2 = max(top - 16, 0) * 2;
        if (u < c2) {
            n = top - u / 2;
            rt = u & 1;
            return;
        }
        n = max(min(top, 16) - (u - c2), 0);
        rt = 0;
    };
    const double *rec = A_all + t.a_off + lane;
    const int Z = c_trans.v[N + 1];
    // One product of a part. SHIFT: blocks of an order, whose coefficients lie j
    // apart at degree j; else of a degree, one after the other. Columns past a
    // block meet zeros of the operand: they read what follows (the rows past the
    // last coefficient are zero).
    auto product = [&](auto shift, const double *B) {
        constexpr bool SHIFT = decltype(shift)::value;
        double a[KM];
        auto load = [&](int s) {
            int n, rt;
            unit(s, n, rt);
            const int ks = (n + 3) >> 2;
            const double *Ap = B + c_trans.v[n] + rt * ks * 64;
#pragma unroll
            for (int q = 0; q < KM; q++) a[q] = q < ks ? Ap[q * 64] : 0.0;
        };
        // coefficient of row k of a block of size n
        auto coef = [&](int n, int k) {
            return SHIFT ? (N - n + k) * (N - n + k + 1) / 2 + N - n : n * (n - 1) / 2 + k;
        };
        gemm_d4 acc[U];
        load(0);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < U; s++) {
            int n, rt;
            unit(s, n, rt);
            acc[s] = gemm_d4{0.0, 0.0, 0.0, 0.0};
            const int ks = (n + 3) >> 2;
            const double *row = S + coef(n, lq) * TR_LD + li;
            int step = (4 * (N - n + lq) + 10) * TR_LD;
#pragma unroll
            for (int q = 0; q < KM; q++)
                if (q < ks) {
                    double b = SHIFT ? *row : row[4 * q * TR_LD];
                    acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], b, acc[s], 0, 0, 0);
                    if (SHIFT) {
                        row += step;
                        step += 16 * TR_LD;
                    }
                }
            if (s + 1 < U) load(s + 1);
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < U; s++) {
            int n, rt;
            unit(s, n, rt);
            const int k0 = 16 * rt + lq;              // lane holds rows lane/16 + 4 i of the tile, column lane % 16
            double *row = S + coef(n, k0) * TR_LD + li;
            int step = (4 * (N - n + k0) + 10) * TR_LD;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (k0 + 4 * i < n) *(SHIFT ? row : row + 4 * i * TR_LD) = acc[s][i];
                if (SHIFT) {
                    row += step;
                    step += 16 * TR_LD;
                }
            }
        }
    };
#pragma unroll 1
    for (int part = 0; part < 2; part++) {
        product(std::false_type{}, rec + (size_t)Z * part);
        product(std::true_type{}, rec + (size_t)Z * 2);
        product(std::false_type{}, rec + (size_t)Z * (3 + part));
        __syncthreads();
        if (part == 0)
#pragma unroll
            for (int j = 0; j < EJ; j++) {
                const int k = lane + 64 * j;
                if (k >= h) continue;
#pragma unroll
                for (int c = 0; c < C; c++) {
                    double v = S[k * TR_LD + wave + W * c];
                    S[k * TR_LD + wave + W * c] = keep[c][j];
                    keep[c][j] = v;
                }
            }
    }
    // rotated back about z, scaled and added: 64 consecutive doubles of the
    // destination per step
    double sc[C];
    double *y[C];
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int col = wave + W * c, pair = col / NRHS;
        const bool on = pair < npair;
        sc[c] = on ? pscale[pair0 + pair] : 0.0;
        y[c] = on ? Y + ((size_t)pdst[pair0 + pair] * NRHS + col % NRHS) * nc : nullptr;
    }
#pragma unroll
    for (int j = 0; j < EJ; j++) {
        if (64 * j >= h) break;
        const int k = lane + 64 * j;
        const double2 e = k < h ? phase(k) : double2{0.0, 0.0};
#pragma unroll
        for (int c = 0; c < C; c++) {
            if (!y[c]) continue;
            double yr = k < h ? keep[c][j] : 0.0, yi = k < h ? S[k * TR_LD + wave + W * c] : 0.0;
            double re = (e.x * yr + e.y * yi) * sc[c], im = (e.x * yi - e.y * yr) * sc[c];
#pragma unroll
            for (int half = 0; half < 2; half++) {
                int src = 32 * half + (lane >> 1);
                double vr = __shfl(re, src), vi = __shfl(im, src);
                if (64 * j + src < h) unsafeAtomicAdd(y[c] + 128 * j + 64 * half + lane, lane & 1 ? vi : vr);
            }
        }
    }
}

template <int W, int U, int EJ, int KM>
__global__ __launch_bounds__(64 * W, 4) void k_m2l_turned(const M2LTile *__restrict__ tiles, int ntiles, int h_turned,
                                                    const double *__restrict__ A_all,
                                                    const int *__restrict__ psrc,
                                                    const int *__restrict__ pdst,
                                                    const double *__restrict__ pscale,
                                                    const double *__restrict__ X, double *__restrict__ Y,
                                                    int nc)
{
    extern __shared__ double lds[];
    trans_tile<W, U, EJ, KM>(tiles, ntiles, h_turned, A_all, psrc, pdst, pscale, X, Y, nc, lds);
}

// M2M / L2L of one level: the same body with the octants' operators
template <int W, int U, int EJ, int KM>
__global__ __launch_bounds__(64 * W, 4) void k_m2m_l2l(const M2LTile *__restrict__ tiles, int ntiles, int h_turned,
                                                    const double *__restrict__ A_all,
                                                    const int *__restrict__ psrc,
                                                    const int *__restrict__ pdst,
                                                    const double *__restrict__ pscale,
                                                    const double *__restrict__ X, double *__restrict__ Y,
                                                    int nc)
{
    extern __shared__ double lds[];
    trans_tile<W, U, EJ, KM>(tiles, ntiles, h_turned, A_all, psrc, pdst, pscale, X, Y, nc, lds);
}

// The kernels: 8 waves to order 26 (38 units, 378 coefficients: two workgroups
// a CU), 16 to PMAX (87 and 1035).
static_assert(PMAX <= 44, "units and coefficients of the largest order");
// (Order 39, M2M and L2L: 0.71 ms with 16 waves, 0.83 with 8, dense 1.20.)
constexpr auto k_m2l_turned_26 = k_m2l_turned<8, 5, 6, 7>, k_m2l_turned_max = k_m2l_turned<16, 6, 17, 12>;
constexpr auto k_m2m_l2l_26 = k_m2m_l2l<8, 5, 6, 7>, k_m2m_l2l_max = k_m2m_l2l<16, 6, 17, 12>;
static_assert(tr_rows(PMAX) * TR_LD * 8 + (PMAX + 1) * 16 <= 160 * 1024, "LDS of a CU");
inline auto m2m_l2l_kernel(int p) { return p <= 26 ? k_m2m_l2l_26 : k_m2m_l2l_max; }
inline int trans_threads(int p) { return p <= 26 ? 512 : 1024; }
// h: the fewest coefficients among the tiles (a row block then has most parts)
inline dim3 trans_grid(int ntiles, int h)
{
    int nrb = (h + ML_M - 1) / ML_M;
    return dim3(ntiles, (ML_P / TR_P + nrb - 1) / nrb);
}


// ------------------------------------------------------------------------
// Evaluation of expansions at points: L2T (local) and M2T (list 4)
// ------------------------------------------------------------------------

// ---- L2T / M2T on the FP64 matrix cores ----------------------------------
// For one expansion (slot) the nine fields of all four right-hand sides at
// a set of points are one product F (36 x K) * H (K x npts): K runs over the
// real and imaginary parts of the harmonics V_l^m (0 <= m <= l <= ph, ph = p
// for a local expansion, p + 2 for a multipole), in the order the harmonic
// recurrence produces them (m outer, l inner). Step s of the product covers
// stream positions 2s and 2s+1: K index 4s + kk is the real (kk even) or
// imaginary (kk odd) part of position 2s + kk/2. The 36 rows sit in three
// 16-row tiles: row 4*(q%4) + r of tile q/4 is field q of right-hand side r,
// so that in the v_mfma_f64_16x16x4f64 output (lane l, register i holds row
// l/16 + 4i) one lane ends up with all nine fields of one right-hand side;
// tile 2 keeps only field 8 (rows 0-3) and is stored compactly. Per step the
// slot's operand takes EA_STEP doubles: tiles 0 and 1 (64 each), tile 2
// rows 0-3 (16). The entries carry the weights of the real
// field sum (1 for m = 0, 2 otherwise), the minus sign of the imaginary
// part and the normalisation 1/sqrt((l+m)!(l-m)!).
constexpr int EA_STEP = 144;

// Operand entries of steps [s0, s0 + sn) of one slot into dst (step s0 at
// dst[0]) from the slot's expansions E (NRHS x nc doubles) and the field
// table; threads tid, tid + nthr, ... of the caller. Every operand double
// is a gather of at most three expansion entries (build_field_table); a
// thread forms one table entry for the four right-hand sides, 32
// contiguous bytes. A step's tiles 0 and 1 are [kk][q%4][rhs] (64 doubles
// each; the operand lane (kk, row) reads kk*16 + row) and tile 2 is
// [kk][rhs].
__device__ __forceinline__ void build_operand(int s0, int sn, double *dst, const double *__restrict__ E,
                                              int nc, const FieldTerm *__restrict__ tab, int tid, int nthr)
{
#pragma unroll 1
    for (int it = tid; it < sn * 36; it += nthr) {
        int sl = it / 36, e = it - sl * 36;
        int st = s0 + sl, kk, q, off;
        if (e < 32) {
            kk = (e >> 2) & 3;
            q = 4 * (e >> 4) + (e & 3);
            off = sl * EA_STEP + (e >> 4) * 64 + kk * 16 + (e & 3) * 4;
        } else {
            kk = e - 32;
            q = 8;
            off = sl * EA_STEP + 128 + kk * 4;
        }
        const FieldTerm &f = tab[((2 * st + (kk >> 1)) * 2 + (kk & 1)) * 9 + q];
        int4 ix = *reinterpret_cast<const int4 *>(f.idx);
        double2 c01 = *reinterpret_cast<const double2 *>(f.c);
        double c2 = f.c[2];
        double v[NRHS];
#pragma unroll
        for (int r = 0; r < NRHS; r++) {
            const double *Er = E + r * nc;
            v[r] = c01.x * Er[ix.x] + c01.y * Er[ix.y] + c2 * Er[ix.z];
        }
        static_assert(NRHS == 4, "one 32-byte store per entry");
        double2 *o = reinterpret_cast<double2 *>(dst + off);
        o[0] = double2{v[0], v[1]};
        o[1] = double2{v[2], v[3]};
    }
}

constexpr int EW_WAVES = 4;         // wave tasks per workgroup
constexpr int EW_TILES = EW_PTS / 16;

// Evaluate the field operand of a slot at up to EW_PTS points per wave.
// A wave task is (slot, first point task, count); lane (kk, j) generates,
// for point j of each 16-point tile, the K entries 4s + kk of the harmonics
// by the integer-coefficient Legendre recurrence (two stream positions per
// step), and the matrix cores form the 36 x 16 field blocks. A lane carries its
// own part only, real or imaginary (the recurrence along a column is real): a
// third less arithmetic than both, and registers for a fourth wave per SIMD,
// which the gathers of the operand wait for (order 26, 182,000 points: L2T 0.83
// ms, 1.25 with both; M2T of 38,400 pairs 2.1, 2.4). IRR=false:
// local expansion at a leaf's own points (plain adds: one slot per point);
// IRR=true: multipole of a list-3 box at the points of the boxes listing it
// (atomic adds). The operand never goes to memory: it is formed in LDS
// from the expansion through the field table, EB_CHUNK steps at a time.
// SH=true: workgroup b takes wave tasks [bt[b], bt[b+1]), all of one slot
// (at most EW_WAVES); the slot's expansions are staged in LDS once and the
// workgroup forms each chunk for all its waves (double-buffered: the next
// chunk is formed while slower waves finish the current one); waves
// without a task only help form it. SH=false: wave task blockIdx.x *
// EB_WAVES + wave, each wave forming its own operand in its part of LDS
// (L2T leaves mostly have one wave task).
constexpr int EB_CHUNK = 8;
constexpr int EB_WAVES = 1;         // wave tasks per workgroup without SH (2 measured slower)

template <bool IRR, bool SH>
__device__ __forceinline__ void meval_body(int p, int nwt, const int *__restrict__ wt,
                                                        const int *__restrict__ bt,
                                                        const int *__restrict__ t_pt,
                                                        const int *__restrict__ slot_box,
                                                        const double *__restrict__ centers,
                                                        const double *__restrict__ sides,
                                                        const double *__restrict__ pts,
                                                        const double *__restrict__ expn, int nc,
                                                        const FieldTerm *__restrict__ tab, int nsteps,
                                                        double *__restrict__ lap)
{
    __shared__ __align__(16) double As[SH ? 2 * EB_CHUNK * EA_STEP : EB_WAVES * EB_CHUNK * EA_STEP];
    extern __shared__ double Es[];                 // SH: the slot's expansions (NRHS x nc)
    int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int w = SH ? bt[blockIdx.x] + wv : (int)blockIdx.x * EB_WAVES + wv;
    // every wave reaches the workgroup barriers; one without a task runs on
    // a valid slot with no points
    bool act = SH ? w < bt[blockIdx.x + 1] : w < nwt;
    if (!act) w = SH ? bt[blockIdx.x] : nwt - 1;
    int lane = threadIdx.x & 63, j = lane & 15, kk = lane >> 4;
    int slot = __builtin_amdgcn_readfirstlane(wt[3 * w]);
    int t0 = __builtin_amdgcn_readfirstlane(wt[3 * w + 1]);
    int cnt = act ? __builtin_amdgcn_readfirstlane(wt[3 * w + 2]) : 0;
    const bool im = kk & 1;
    int ebox = slot_box[slot];
    double is = 1.0 / sides[ebox];
    double cx = centers[3 * ebox], cy = centers[3 * ebox + 1], cz = centers[3 * ebox + 2];
    int ph = IRR ? p + 2 : p;

    double hx[EW_TILES], hy[EW_TILES], zz[EW_TILES], rr[EW_TILES], ir2[EW_TILES];
    // column starts (complex) and the lane's part (real for even kk, imaginary for
    // odd) of the last two harmonics of the column: the recurrence is real
    double dr[EW_TILES], di[EW_TILES], pv[EW_TILES], cv[EW_TILES];
    int gp[EW_TILES];
#pragma unroll
    for (int i = 0; i < EW_TILES; i++) {
        int k = 16 * i + j;
        double x = 1.0, y = 0.0, z = 0.0;       // a finite stand-in for an empty column
        gp[i] = -1;
        if (k < cnt) {
            gp[i] = t_pt[t0 + k];
            x = (pts[3 * (size_t)gp[i]] - cx) * is;
            y = (pts[3 * (size_t)gp[i] + 1] - cy) * is;
            z = (pts[3 * (size_t)gp[i] + 2] - cz) * is;
        }
        double r2 = x * x + y * y + z * z;
        ir2[i] = IRR ? 1.0 / r2 : 1.0;
        hx[i] = x;
        hy[i] = y;
        zz[i] = z * ir2[i];
        rr[i] = IRR ? ir2[i] : r2;
        dr[i] = IRR ? sqrt(ir2[i]) : 1.0;
        di[i] = 0.0;
        cv[i] = im ? 0.0 : dr[i];
        pv[i] = 0.0;
    }
    int ntile = (cnt + 15) >> 4;
    gemm_d4 acc[3][EW_TILES];
#pragma unroll
    for (int t = 0; t < 3; t++)
#pragma unroll
        for (int i = 0; i < EW_TILES; i++) acc[t][i] = gemm_d4{0.0, 0.0, 0.0, 0.0};

    int l = 0, m = 0;                        // stream position of cv
    // advance cv to the next stream position
    auto advance = [&]() {
        l++;
        if (l > ph) {
            m++;
            l = m;
            double c = -(double)(2 * m - 1);
#pragma unroll
            for (int i = 0; i < EW_TILES; i++) {
                double ci2 = c * ir2[i];
                double nr = ci2 * (hx[i] * dr[i] - hy[i] * di[i]);
                double ni = ci2 * (hx[i] * di[i] + hy[i] * dr[i]);
                dr[i] = nr;
                di[i] = ni;
                cv[i] = im ? ni : nr;
                pv[i] = 0.0;
            }
        } else {
            double k1c = (double)(2 * l - 1), k2c = (double)((l + m - 1) * (l - m - 1));
#pragma unroll
            for (int i = 0; i < EW_TILES; i++) {
                double k1 = k1c * zz[i], k2 = k2c * rr[i];
                double nv = k1 * cv[i] - k2 * pv[i];
                pv[i] = cv[i];
                cv[i] = nv;
            }
        }
    };
    int lo = kk * 16 + j;                          // operand row j = 4*(q%4) + rhs
    // one step: B entries at stream positions 2s (kk 0, 1) and 2s+1 (kk 2, 3)
    auto step = [&](double a0, double a1, double a2) {
        double b[EW_TILES];
        bool live0 = m <= ph;
#pragma unroll
        for (int i = 0; i < EW_TILES; i++) b[i] = live0 ? cv[i] : 0.0;
        advance();
        bool live1 = m <= ph;
#pragma unroll
        for (int i = 0; i < EW_TILES; i++)
            if (kk >= 2) b[i] = live1 ? cv[i] : 0.0;
        advance();
#pragma unroll
        for (int i = 0; i < EW_TILES; i++) {
            if (i < ntile) {
                acc[0][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b[i], acc[0][i], 0, 0, 0);
                acc[1][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b[i], acc[1][i], 0, 0, 0);
                acc[2][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a2, b[i], acc[2][i], 0, 0, 0);
            }
        }
    };
    const double *E = expn + (size_t)ebox * NRHS * nc;
    if (SH) {
        constexpr int CH = EB_CHUNK * EA_STEP;       // doubles per chunk
        constexpr int NT = 64 * EW_WAVES;
        int nchunk = (nsteps + EB_CHUNK - 1) / EB_CHUNK;
        for (int e = threadIdx.x; e < NRHS * nc; e += NT) Es[e] = E[e];
        __syncthreads();
        build_operand(0, min(EB_CHUNK, nsteps), As, Es, nc, tab, threadIdx.x, NT);
        __syncthreads();
        for (int c = 0; c < nchunk; c++) {
            int s0 = c * EB_CHUNK, sn = min(EB_CHUNK, nsteps - s0);
            int nsn = c + 1 < nchunk ? min(EB_CHUNK, nsteps - s0 - EB_CHUNK) : 0;
            const double *Ac = As + (c & 1) * CH;
            for (int ss = 0; ss < sn; ss++) {
                const double *a = Ac + ss * EA_STEP;
                step(a[lo], a[64 + lo], j < 4 ? a[128 + kk * 4 + j] : 0.0);
            }
            if (nsn > 0) build_operand(s0 + EB_CHUNK, nsn, As + ((c + 1) & 1) * CH, Es, nc, tab, threadIdx.x, NT);
            __syncthreads();
        }
    } else {
        double *Bw = As + wv * (EB_CHUNK * EA_STEP);
        for (int s0 = 0; s0 < nsteps; s0 += EB_CHUNK) {
            int sn = min(EB_CHUNK, nsteps - s0);
            __syncthreads();                           // the previous chunk has been read
            build_operand(s0, sn, Bw, E, nc, tab, lane, 64);
            __syncthreads();
            for (int ss = 0; ss < sn; ss++) {
                const double *a = Bw + ss * EA_STEP;
                step(a[lo], a[64 + lo], j < 4 ? a[128 + kk * 4 + j] : 0.0);
            }
        }
    }
    double s1 = IRR ? is : 1.0;
    double g1 = s1 * is, g2 = g1 * is;
#pragma unroll
    for (int i = 0; i < EW_TILES; i++) {
        if (gp[i] < 0) continue;
        // lane (kk, j), register e of tile t: field 4t + e of rhs kk at point j
        double f0 = acc[0][i][0], f1 = acc[0][i][1], f2 = acc[0][i][2], f3 = acc[0][i][3];
        double f4 = acc[1][i][0], f5 = acc[1][i][1], f6 = acc[1][i][2], f7 = acc[1][i][3];
        double f8 = acc[2][i][0];
        double v[10] = {s1 * f0, g1 * f1, g1 * f2, g1 * f3, g2 * f4, g2 * f5, -g2 * (f4 + f5),
                        g2 * f6, g2 * f7, g2 * f8};
        double *o = lap + (size_t)gp[i] * 40 + kk * 10;
#pragma unroll
        for (int q = 0; q < 10; q++) {
            if (IRR)
                unsafeAtomicAdd(o + q, v[q]);
            else
                o[q] += v[q];
        }
    }
}

// L2T (local expansions at the leaves' own points, one wave per wave task
// forming its operand in LDS) and M2T (multipoles of list-3 boxes, operand
// shared in LDS)
__global__ __launch_bounds__(64 * EB_WAVES, 4) void k_l2t(int p, int nwt, const int *__restrict__ wt,
                                            const int *__restrict__ t_pt, const int *__restrict__ slot_box,
                                            const double *__restrict__ centers,
                                            const double *__restrict__ sides, const double *__restrict__ pts,
                                            const double *__restrict__ expn, int nc,
                                            const FieldTerm *__restrict__ tab, int nsteps,
                                            double *__restrict__ lap)
{
    meval_body<false, false>(p, nwt, wt, nullptr, t_pt, slot_box, centers, sides, pts, expn, nc, tab, nsteps,
                             lap);
}

__global__ __launch_bounds__(64 * EW_WAVES, 3) void k_m2t(int p, int nwt, const int *__restrict__ wt,
                                                        const int *__restrict__ bt,
                                                        const int *__restrict__ t_pt,
                                                        const int *__restrict__ slot_box,
                                                        const double *__restrict__ centers,
                                                        const double *__restrict__ sides,
                                                        const double *__restrict__ pts,
                                                        const double *__restrict__ expn, int nc,
                                                        const FieldTerm *__restrict__ tab, int nsteps,
                                                        double *__restrict__ lap)
{
    meval_body<true, true>(p, nwt, wt, bt, t_pt, slot_box, centers, sides, pts, expn, nc, tab, nsteps, lap);
}


// ------------------------------------------------------------------------
// Near field: self + list 1 pair quadratures, one wave per workgroup
// ------------------------------------------------------------------------

constexpr int NF_THREADS = 256;

// Wave b takes lanes [l0, l0 + 64) of leaf q's (point, lane) pairs, (q, l0, split)
// = tasks[3b..]: each point's near triangles (the lists of its boxes one after
// another) are dealt to `split` lanes, a power of two chosen per leaf
// (near_tasks), so every lane has a triangle in every step but the last. Up
// to 64 boxes of the near list at a time: their first triangles and running
// counts are scanned across the wave into LDS, and a lane finds the box of
// its next triangle by walking those counts. Bound by FP64 vector issue (pair
// code: elfmm_near.h). 81,920 triangles + 100,000 targets, iprec 2 (25.0e6
// pairs, both layers, strain): 4.25 ms with two passes over the edges
// and a 256-thread workgroup per leaf whose lanes idled in boxes of fewer
// triangles than lanes per point, 1.32 ms in this form; 217 points against 180
// triangles: 0.23 and 0.014 ms.
template <bool SL, bool DL, bool ST>
__global__ __launch_bounds__(64) void k_near(
    int n, int n_src_eval, const int *__restrict__ boxes, const int *__restrict__ lstart,
    const int *__restrict__ litems, const int *__restrict__ src_start,
    const int *__restrict__ src_count, const int *__restrict__ tgt_start,
    const int *__restrict__ tgt_count, const int *__restrict__ tasks, const double *__restrict__ pts,
    const double *__restrict__ rec, double rlam, double rmu, double c1, double *__restrict__ nf)
{
    __shared__ int pre[65], first[64];               // triangles before each box of the pass; its first triangle
    int lane = threadIdx.x;
    int q = tasks[3 * blockIdx.x], l0 = tasks[3 * blockIdx.x + 1], split = tasks[3 * blockIdx.x + 2];
    int tbox = boxes[q];
    int ns_eval = n_src_eval ? src_count[tbox] : 0;
    int npts = ns_eval + tgt_count[tbox];
    int k = (l0 + lane) / split, sub = lane & (split - 1);
    bool has = k < npts;
    int selfidx = has && k < ns_eval ? src_start[tbox] + k : -1;
    int gp = !has ? -1 : (k < ns_eval ? selfidx : n + tgt_start[tbox] + (k - ns_eval));
    double P[3] = {0.0, 0.0, 0.0};
    if (has)
        for (int d = 0; d < 3; d++) P[d] = pts[3 * (size_t)gp + d];
    double acc[9];
#pragma unroll
    for (int c = 0; c < 9; c++) acc[c] = 0.0;
    for (int b0 = lstart[q], b1 = lstart[q + 1]; b0 < b1; b0 += 64) {
        int cnt = 0, s0 = 0;
        if (b0 + lane < b1) {
            int sbox = litems[b0 + lane];
            s0 = src_start[sbox];
            cnt = src_count[sbox];
        }
        int end = cnt;
        for (int off = 1; off < 64; off <<= 1) {
            int v = __shfl_up(end, off);
            if (lane >= off) end += v;
        }
        __syncthreads();                              // the previous pass has been walked
        if (lane == 0) pre[0] = 0;
        pre[lane + 1] = end;
        first[lane] = s0;
        __syncthreads();
        int total = pre[64], bi = 0;
        for (int t = has ? sub : total; t < total; t += split) {
            while (t >= pre[bi + 1]) bi++;
            int i = first[bi] + t - pre[bi];
            near_pair<SL, DL, ST>(rec + (size_t)i * NF_REC, P, i == selfidx, rlam, rmu, c1, acc);
        }
    }
    constexpr int NO = ST ? 9 : 3;
    for (int off = split >> 1; off > 0; off >>= 1)
#pragma unroll
        for (int c = 0; c < NO; c++) acc[c] += __shfl_xor(acc[c], off);
    if (!has || sub) return;
    const double sc = 0.5 / rmu;
#pragma unroll
    for (int c = 0; c < 9; c++) nf[(size_t)gp * 9 + c] = sc * acc[c];
}

// The variant for the layers and outputs of a call.
inline auto near_kernel(bool sl, bool dl, bool strain)
{
    return sl && dl ? (strain ? k_near<true, true, true> : k_near<true, true, false>)
           : dl     ? (strain ? k_near<false, true, true> : k_near<false, true, false>)
                    : (strain ? k_near<true, false, true> : k_near<true, false, false>);
}

// Stored near-field interactions (iter mode). For near box q with npts
// points and ntri triangles (its near list concatenated), pair slot
// s = point * ntri + triangle holds W words at store[sbase[q] +
// store_idx(k, t, w, ntri, W)] (point k, triangle t). Words per pair: for each
// layer present (single, then double) and k = 0..2, the fields of the unit
// density e_k: the displacement (3) if fd, the strain xx yy zz xy xz yz (6)
// if fs.
struct StoreLayout {
    int W, fd, fs, ifsl, ifdl;
};

// Each point's ntri slots in tiles of 64 triangles, a tile holding its W
// words one after another (64 doubles each, fewer in the point's last
// tile): the wave that reads triangles 64j .. 64j + 63 of a point reads one
// tile, W x 64 consecutive doubles, for each word 64 of them.
__device__ __forceinline__ int64_t store_idx(int k, int t, int w, int ntri, int W)
{
    int t0 = t & ~63;
    int tw = ntri - t0 < 64 ? ntri - t0 : 64;
    return ((int64_t)k * ntri + t0) * W + (int64_t)w * tw + (t - t0);
}

// Walk of one lane over its share of a point's near triangles: the
// concatenated list is dealt round-robin to the point's tpp lanes.
template <class F>
__device__ __forceinline__ void near_walk(int b0, int b1, const int *__restrict__ litems,
                                          const int *__restrict__ src_start, const int *__restrict__ src_count,
                                          int sub, int tpp, F &&f)
{
    int j0 = sub, cum = 0;
    for (int bb = b0; bb < b1; bb++) {
        int sbox = litems[bb];
        int s0 = src_start[sbox], sn = src_count[sbox];
        for (; j0 < sn; j0 += tpp) f(s0 + j0, cum + j0);
        j0 -= sn;
        cum += sn;
    }
}

// icomp 2: evaluate every pair for the unit densities, store the fields,
// and accumulate the pair's contribution for the current densities.
// Workgroup b takes points [p0, p0 + ST_CHUNK) of near box qb, (qb, p0) =
// chunk[2b], chunk[2b + 1]: the iter leaves are large and few, and one
// workgroup per leaf left most of the device idle behind the largest.
constexpr int ST_CHUNK = 16;
__global__ __launch_bounds__(NF_THREADS) void k_near_store(
    int n, int n_src_eval, const int *__restrict__ boxes, const int *__restrict__ lstart,
    const int *__restrict__ litems, const int *__restrict__ src_start,
    const int *__restrict__ src_count, const int *__restrict__ tgt_start,
    const int *__restrict__ tgt_count, const int64_t *__restrict__ sbase, const int *__restrict__ ntri_q,
    const int *__restrict__ chunk, const double *__restrict__ pts, const double *__restrict__ rec,
    const double *__restrict__ ssl_s, const double *__restrict__ sdl_s, double rlam, double rmu, double c1,
    StoreLayout L, double *__restrict__ store, double *__restrict__ nf)
{
    __shared__ double red[NF_THREADS][9];
    int qb = chunk[2 * blockIdx.x], p0 = chunk[2 * blockIdx.x + 1];
    int tbox = boxes[qb];
    int ns_eval = n_src_eval ? src_count[tbox] : 0;
    int npts = ns_eval + tgt_count[tbox];
    int b0 = lstart[qb], b1 = lstart[qb + 1];
    int ntri = ntri_q[qb];
    double *S = store + sbase[qb];
    {
        int ip0 = p0;
        int cnt = min(ST_CHUNK, npts - ip0);
        int tpp = max(1, NF_THREADS / cnt);
        int ip = threadIdx.x / tpp, sub = threadIdx.x % tpp;
        double acc[9];
#pragma unroll
        for (int q = 0; q < 9; q++) acc[q] = 0.0;
        int gp = -1, selfidx = -1;
        if (ip < cnt) {
            int k = ip0 + ip;
            if (k < ns_eval) {
                gp = src_start[tbox] + k;
                selfidx = gp;
            } else {
                gp = n + tgt_start[tbox] + (k - ns_eval);
            }
            double P[3] = {pts[3 * (size_t)gp], pts[3 * (size_t)gp + 1], pts[3 * (size_t)gp + 2]};
            near_walk(b0, b1, litems, src_start, src_count, sub, tpp, [&](int i, int t) {
                double sg[2][3] = {{ssl_s[3 * (size_t)i], ssl_s[3 * (size_t)i + 1], ssl_s[3 * (size_t)i + 2]},
                                   {sdl_s[3 * (size_t)i], sdl_s[3 * (size_t)i + 1], sdl_s[3 * (size_t)i + 2]}};
                nf_pair_basis(rec + (size_t)i * NF_REC, P, i == selfidx, rlam, rmu, c1, L.ifsl, L.ifdl,
                              [&](int layer, int kk, const double *v) {
                                  int w = ((L.ifsl && layer ? 3 : 0) + kk) * (3 * L.fd + 6 * L.fs);
                                  double c = sg[layer][kk];
                                  if (L.fd)
                                      for (int q = 0; q < 3; q++, w++) S[store_idx(k, t, w, ntri, L.W)] = v[q];
                                  if (L.fs)
                                      for (int q = 3; q < 9; q++, w++) S[store_idx(k, t, w, ntri, L.W)] = v[q];
#pragma unroll
                                  for (int q = 0; q < 9; q++) acc[q] += c * v[q];
                              });
            });
        }
#pragma unroll
        for (int q = 0; q < 9; q++) red[threadIdx.x][q] = acc[q];
        __syncthreads();
        if (ip < cnt && sub == 0) {
            for (int t = 1; t < tpp; t++)
#pragma unroll
                for (int q = 0; q < 9; q++) acc[q] += red[threadIdx.x + t][q];
#pragma unroll
            for (int q = 0; q < 9; q++) nf[(size_t)gp * 9 + q] = acc[q];
        }
        __syncthreads();
    }
}

// icomp 3: near field from the stored fields and nr <= RB density sets; bound
// by the read of the store. A task is PTS points of a near box (part
// b % (ST_CHUNK / PTS) of chunk b / (ST_CHUNK / PTS)); the 4 waves take
// its tiles of 64 triangles in turn: a lane finds its slot's triangle in the
// box's list (first slots in LDS, RP_LIST boxes at a time), loads the
// triangle's densities once and then streams that slot of every point, one
// tile of the store (store_idx) per point and load. The layers present (NL:
// d0, then d1) and the fields stored (FD displacement, FS strain) are
// compile-time, so all words of a slot are loaded before the first is used.
// Densities d0/d1: [set][triangle][3] in tree order (stride dstride doubles
// per set); output nf: [set][point][9] (stride nstride).
constexpr int RP_LIST = 512;
constexpr int replay_pts(int nl, bool fd, bool fs, int rb)
{
    int w = nl * 3 * (3 * fd + 6 * fs);
    return rb > 1 ? 1 : w <= 18 ? 4 : w <= 27 ? 2 : 1;
}

template <int NL, bool FD, bool FS, int RB>
__global__ __launch_bounds__(NF_THREADS, 2) void k_near_replay(
    int n, int n_src_eval, const int *__restrict__ boxes, const int *__restrict__ lstart,
    const int *__restrict__ litems, const int *__restrict__ src_start,
    const int *__restrict__ src_count, const int *__restrict__ tgt_start,
    const int64_t *__restrict__ sbase, const int *__restrict__ ntri_q,
    const int *__restrict__ pstart, const int *__restrict__ chunk, int ntask, const double *__restrict__ d0,
    const double *__restrict__ d1, size_t dstride, int nr, const double *__restrict__ store,
    double *__restrict__ nf, size_t nstride)
{
    constexpr int NF = 3 * FD + 6 * FS;                 // fields per unit density
    constexpr int W = NL * 3 * NF;                      // words per slot
    constexpr int Q0 = FD ? 0 : 3;                      // first output component
    constexpr int PTS = replay_pts(NL, FD, FS, RB);
    constexpr int NWAVE = NF_THREADS / 64;
    __shared__ int first[RP_LIST + 1], start[RP_LIST];  // first slot, first triangle of each box of the list
    __shared__ double red[NWAVE][RB * PTS * NF];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (int task = blockIdx.x; task < ntask; task += gridDim.x) {
        const int *ch = chunk + 2 * (task / (ST_CHUNK / PTS));
        const int qb = ch[0], k0 = ch[1] + task % (ST_CHUNK / PTS) * PTS;
        const int np = min(PTS, pstart[qb + 1] - pstart[qb] - k0);
        if (np <= 0) continue;
        const int ntri = ntri_q[qb], b0 = lstart[qb], b1 = lstart[qb + 1];
        const double *S = store + sbase[qb] + (int64_t)k0 * ntri * W;
        double acc[RB][PTS][NF];
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
            for (int k = 0; k < PTS; k++)
#pragma unroll
                for (int q = 0; q < NF; q++) acc[r][k][q] = 0.0;
        int done = 0;                                   // slots of the list's earlier boxes
        for (int c0 = b0; c0 < b1; c0 += RP_LIST) {
            const int nb = min(RP_LIST, b1 - c0);
            __syncthreads();
            if (wave == 0) {
                int cum = done;
                for (int e = 0; e < nb; e += 64) {
                    int cnt = 0;
                    if (e + lane < nb) {
                        int box = litems[c0 + e + lane];
                        start[e + lane] = src_start[box];
                        cnt = src_count[box];
                    }
                    int end = cnt;
                    for (int off = 1; off < 64; off <<= 1) {
                        int v = __shfl_up(end, off);
                        if (lane >= off) end += v;
                    }
                    if (e + lane < nb) first[e + lane] = cum + end - cnt;
                    cum += __shfl(end, 63);
                }
                if (lane == 0) first[nb] = cum;
            }
            __syncthreads();
            const int last = first[nb];
            // tiles that hold slots of these boxes
            for (int t0 = (done / 64 + ((wave - done / 64) & (NWAVE - 1))) * 64; t0 < last; t0 += 64 * NWAVE) {
                const int t = t0 + lane, tw = min(64, ntri - t0);
                if (t < done || t >= last) continue;
                int lo = 0, hi = nb - 1;                // first[lo] <= t < first[lo + 1]
                while (lo < hi) {
                    int mid = (lo + hi + 1) >> 1;
                    if (first[mid] <= t) lo = mid;
                    else hi = mid - 1;
                }
                const size_t i = start[lo] + (t - first[lo]);
                double c[NL][3];
                auto dens = [&](int r) {
#pragma unroll
                    for (int a = 0; a < NL; a++)
#pragma unroll
                        for (int kk = 0; kk < 3; kk++) c[a][kk] = (a ? d1 : d0)[r * dstride + 3 * i + kk];
                };
                if (RB == 1) dens(0);
                const double *Sx = S + (int64_t)t0 * W + lane;   // word w at Sx[w * tw]
#pragma unroll
                for (int k = 0; k < PTS; k++) {
                    if (k >= np) break;
                    double v[W];
#pragma unroll
                    for (int w = 0; w < W; w++) v[w] = Sx[(int64_t)k * ntri * W + w * tw];
#pragma unroll
                    for (int r = 0; r < RB; r++) {
                        if (r >= nr) break;
                        if (RB > 1) dens(r);
#pragma unroll
                        for (int a = 0; a < NL; a++)
#pragma unroll
                            for (int kk = 0; kk < 3; kk++)
#pragma unroll
                                for (int q = 0; q < NF; q++) acc[r][k][q] += c[a][kk] * v[(a * 3 + kk) * NF + q];
                    }
                }
            }
            done = last;
        }
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
            for (int k = 0; k < PTS; k++)
#pragma unroll
                for (int q = 0; q < NF; q++) {
                    double v = acc[r][k][q];
                    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
                    if (lane == 0) red[wave][(r * PTS + k) * NF + q] = v;
                }
        __syncthreads();
        const int tbox = boxes[qb], ns_eval = n_src_eval ? src_count[tbox] : 0;
        for (int e = threadIdx.x; e < min(nr, RB) * np * 9; e += NF_THREADS) {
            int r = e / (np * 9), k = e / 9 % np, q = e % 9;
            double v = 0.0;
            if (q >= Q0 && q < Q0 + NF)
                for (int w = 0; w < NWAVE; w++) v += red[w][(r * PTS + k) * NF + q - Q0];
            int kp = k0 + k, gp = kp < ns_eval ? src_start[tbox] + kp : n + tgt_start[tbox] + (kp - ns_eval);
            nf[r * nstride + (size_t)gp * 9 + q] = v;
        }
    }
}

// Densities of one more right-hand side into tree order (the geometry and
// the first set go through k_gather).
__global__ void k_gather_dens(int n, const int *__restrict__ iz, int ifsl, const double *__restrict__ ssl, int ifdl,
                              const double *__restrict__ sdl, double *__restrict__ ssl_s, double *__restrict__ sdl_s)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int o = iz[i];
    for (int d = 0; d < 3; d++) {
        ssl_s[3 * (size_t)i + d] = ifsl ? ssl[3 * (size_t)o + d] : 0.0;
        sdl_s[3 * (size_t)i + d] = ifdl ? sdl[3 * (size_t)o + d] : 0.0;
    }
}

// Zero fill of a device array. A kernel rather than hipMemsetAsync, so that
// the sequences that use it can be captured into a graph and replayed.
__global__ void k_fill0(double *__restrict__ a, size_t n)
{
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) a[i] = 0.0;
}

inline hipError_t launch_fill0(double *a, size_t n, hipStream_t s)
{
    if (!n) return hipSuccess;
    size_t blocks = std::min<size_t>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(k_fill0, dim3((unsigned)blocks), dim3(256), 0, s, a, n);
    return hipGetLastError();
}

// Where a sequence of kernels goes: a stream (launched at once), or a graph
// under construction (one kernel node per launch, depending on the lane's
// previous node and on what after() added). Cross-lane order: after(o)
// makes the lane's next kernel wait for o's last one (an event between the
// streams, or a graph edge).
struct Lane {
    hipStream_t stream = nullptr;
    hipEvent_t ev = nullptr;                         // stream lanes: marks this lane's last launch for after()
    hipGraph_t graph = nullptr;
    hipGraphNode_t last = nullptr;
    std::vector<hipGraphNode_t> deps;                // graph lanes: extra dependencies of the next node

    template <class... KA, class... A>
    void launch(void (*k)(KA...), dim3 grid, dim3 block, size_t sh, A... args)
    {
        static_assert(sizeof...(KA) == sizeof...(A), "kernel arguments");
        if (!graph) {
            hipLaunchKernelGGL(k, grid, block, sh, stream, args...);
            HIPOK(hipGetLastError());
            return;
        }
        std::tuple<KA...> vals(static_cast<KA>(args)...);
        add_node((void *)k, grid, block, sh, vals, std::index_sequence_for<KA...>{});
    }
    void fill0(double *a, size_t n)
    {
        if (!n) return;
        size_t blocks = std::min<size_t>((n + 255) / 256, 8192);
        launch(k_fill0, dim3((unsigned)blocks), dim3(256), 0, a, n);
    }
    void after(Lane &o)
    {
        if (graph) {
            if (o.last) deps.push_back(o.last);
        } else {
            HIPOK(hipEventRecord(o.ev, o.stream));
            HIPOK(hipStreamWaitEvent(stream, o.ev, 0));
        }
    }

  private:
    template <class Tup, size_t... I>
    void add_node(void *fn, dim3 grid, dim3 block, size_t sh, Tup &vals, std::index_sequence<I...>)
    {
        void *ptrs[sizeof...(I) + 1] = {(void *)&std::get<I>(vals)...};
        hipKernelNodeParams p{};
        p.func = fn;
        p.gridDim = grid;
        p.blockDim = block;
        p.sharedMemBytes = (unsigned)sh;
        p.kernelParams = ptrs;
        p.extra = nullptr;
        if (last) deps.push_back(last);
        hipGraphNode_t node = nullptr;
        HIPOK(hipGraphAddKernelNode(&node, graph, deps.empty() ? nullptr : deps.data(), deps.size(), &p));
        deps.clear();
        last = node;
    }
};

// Direct sum (el3dtriadirecttarg): every triangle at every point.
__global__ __launch_bounds__(NF_THREADS) void k_direct(int n, int npts_eval, int n_src_eval,
                                                      const double *__restrict__ pts,
                                                      const double *__restrict__ rec, double rlam,
                                                      double rmu, double c1, int ifsl, int ifdl,
                                                      double *__restrict__ nf)
{
    // one wave-sized group of threads per point, split over triangles
    constexpr int TPP = 64;
    __shared__ double red[NF_THREADS][9];
    int ip = blockIdx.x * (NF_THREADS / TPP) + threadIdx.x / TPP;
    int sub = threadIdx.x % TPP;
    double acc[9];
#pragma unroll
    for (int q = 0; q < 9; q++) acc[q] = 0.0;
    int gp = -1;
    if (ip < npts_eval) {
        gp = ip < n_src_eval ? ip : n + (ip - n_src_eval);
        int selfidx = ip < n_src_eval ? ip : -1;
        double P[3] = {pts[3 * (size_t)gp], pts[3 * (size_t)gp + 1], pts[3 * (size_t)gp + 2]};
        for (int i = sub; i < n; i += TPP)
            nf_pair(rec + (size_t)i * NF_REC, P, i == selfidx, rlam, rmu, c1, ifsl, ifdl, acc);
    }
#pragma unroll
    for (int q = 0; q < 9; q++) red[threadIdx.x][q] = acc[q];
    __syncthreads();
    if (ip < npts_eval && sub == 0) {
        for (int t = 1; t < TPP; t++)
#pragma unroll
            for (int q = 0; q < 9; q++) acc[q] += red[threadIdx.x + t][q];
#pragma unroll
        for (int q = 0; q < 9; q++) nf[(size_t)gp * 9 + q] = acc[q];
    }
}

// Inputs of the direct sum in the caller's order: near-field records of the
// triangles and the evaluation points (sources, then targets).
__global__ void k_direct_prep(int n, int nt, const double *__restrict__ tri, const double *__restrict__ src,
                              int ifsl, const double *__restrict__ ssl, int ifdl, const double *__restrict__ sdl,
                              const double *__restrict__ tgt, double *__restrict__ pts, double *__restrict__ rec)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        double t[9], s1[3], s2[3];
        for (int d = 0; d < 9; d++) t[d] = tri[9 * (size_t)i + d];
        for (int d = 0; d < 3; d++) {
            s1[d] = ifsl ? ssl[3 * (size_t)i + d] : 0.0;
            s2[d] = ifdl ? sdl[3 * (size_t)i + d] : 0.0;
            pts[3 * (size_t)i + d] = src[3 * (size_t)i + d];
        }
        nf_make_record(t, s1, s2, rec + (size_t)i * NF_REC);
    } else if (i < n + nt) {
        for (int d = 0; d < 3; d++) pts[3 * (size_t)i + d] = tgt[3 * (size_t)(i - n) + d];
    }
}

// ------------------------------------------------------------------------
// Assembly: elastic combination of the four Laplace problems
// (elfmm3dlap1/elfmm3dlap2, src/el3routs.f:1392-1500, then strain =
// sym(hessmatr), src/elfmm3dtria.f:586-606) plus the near field, scattered
// to the caller's order.
// ------------------------------------------------------------------------

// Displacement u and displacement gradient hm (added to) from the four
// Laplace fields at point X (10 values per problem: potential, gradient,
// Hessian xx yy zz xy xz yz): problems 0-2 by elfmm3dlap1, problem 3 by
// elfmm3dlap2 (src/el3routs.f:1392-1500).
__device__ __forceinline__ void lap_to_elastic(const double *__restrict__ o, const double *X, double c1,
                                               double u[3], double hm[3][3])
{
    for (int j = 0; j < 3; j++) {
        const double *f = o + 10 * j;
        double pot = f[0], fld[3] = {-f[1], -f[2], -f[3]};
        double h[3][3] = {{f[4], f[7], f[8]}, {f[7], f[5], f[9]}, {f[8], f[9], f[6]}};
        u[j] += (2 - c1) * pot;
        for (int d = 0; d < 3; d++) u[d] += c1 * X[j] * fld[d];
        for (int d = 0; d < 3; d++) {
            hm[j][d] -= (2 - c1) * fld[d];
            hm[d][j] += fld[d] * c1;
        }
        for (int a = 0; a < 3; a++)
            for (int b = 0; b < 3; b++) hm[a][b] -= X[j] * h[a][b] * c1;
    }
    const double *f = o + 30;
    double h[3][3] = {{f[4], f[7], f[8]}, {f[7], f[5], f[9]}, {f[8], f[9], f[6]}};
    for (int d = 0; d < 3; d++) u[d] += f[1 + d];
    for (int a = 0; a < 3; a++)
        for (int b = 0; b < 3; b++) hm[a][b] += h[a][b];
}

__global__ void k_assemble(int n, int nt, int src_eval, const int *__restrict__ iz,
                           const int *__restrict__ izt, const double *__restrict__ pts,
                           const double *__restrict__ lap, const double *__restrict__ nf,
                           double c1, int usefar, int accumulate, int half, int ifpt, double *__restrict__ ptfrc,
                           int ifst, double *__restrict__ strain, int ifptt, double *__restrict__ ptfrct,
                           int ifstt, double *__restrict__ straint)
{
    int ip = blockIdx.x * blockDim.x + threadIdx.x;
    if (ip >= n + nt) return;
    bool is_src = ip < n;
    if (is_src && !src_eval) return;
    const double *X = pts + 3 * (size_t)ip;
    double u[3] = {0, 0, 0}, hm[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    if (usefar) lap_to_elastic(lap + (size_t)ip * 40, X, c1, u, hm);
    // half space: the far field is the anti-image (src/elhfmm3dtria_iter.f:
    // 1344-1372: third column of the gradient flipped before the strain is
    // formed), subtracted from the result (:761-777)
    if (half)
        for (int a = 0; a < 3; a++) hm[a][2] = -hm[a][2];
    const double *g = nf + (size_t)ip * 9;
    double st[3][3];
    for (int a = 0; a < 3; a++)
        for (int b = 0; b < 3; b++) st[a][b] = half ? -(hm[a][b] + hm[b][a]) / 2 : (hm[a][b] + hm[b][a]) / 2;
    if (half)
        for (int d = 0; d < 3; d++) u[d] = -u[d];
    st[0][0] += g[3];
    st[1][1] += g[4];
    st[2][2] += g[5];
    st[0][1] += g[6];
    st[1][0] += g[6];
    st[0][2] += g[7];
    st[2][0] += g[7];
    st[1][2] += g[8];
    st[2][1] += g[8];
    for (int d = 0; d < 3; d++) u[d] += g[d];
    // iz == nullptr: points are in the caller's order
    int o = is_src ? (iz ? iz[ip] : ip) : (izt ? izt[ip - n] : ip - n);
    double *po = is_src ? (ifpt ? ptfrc + 3 * (size_t)o : nullptr) : (ifptt ? ptfrct + 3 * (size_t)o : nullptr);
    double *so = is_src ? (ifst ? strain + 9 * (size_t)o : nullptr) : (ifstt ? straint + 9 * (size_t)o : nullptr);
    // accumulate: add to the caller's values (the iter engine's near-field-only
    // mode adds its result, src/elfmm3dtria_iter_1.f:960-971)
    if (po)
        for (int d = 0; d < 3; d++) po[d] = accumulate ? po[d] + u[d] : u[d];
    if (so)
        for (int a = 0; a < 3; a++)
            for (int b = 0; b < 3; b++) so[3 * b + a] = accumulate ? so[3 * b + a] + st[a][b] : st[a][b];
}

// ------------------------------------------------------------------------
// Point sources (elfmm3dparttarg, src/elfmm3dpart.f:104-500)
// ------------------------------------------------------------------------

// Point sources into tree order as node records of the four Laplace
// problems (src/elfmm3dpart.f:336-444), weight 1: charges sigma_sl/(2 mu)
// and dipoles sym(sigma_dv x sigma_dl) for problems 0-2; problem 3 with
// charge (sigma_sl . x) c1/(2 mu) + (sigma_dl . sigma_dv) c2 and dipole
// c1 (sigma_dv (sigma_dl . x) + sigma_dl (sigma_dv . x)) / 2. The
// evaluation points (sources, then targets) in tree order.
__global__ void k_pgather(int n, int nt, const int *__restrict__ iz, const int *__restrict__ izt,
                          const double *__restrict__ src, int ifsl, const double *__restrict__ ssl, int ifdl,
                          const double *__restrict__ sdl, const double *__restrict__ sdv,
                          const double *__restrict__ tgt, double rmu, double c1, double c2,
                          double *__restrict__ pts, double *__restrict__ nodes)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        size_t o = (size_t)iz[i];
        double X[3], sl[3], dl[3], dv[3];
        for (int d = 0; d < 3; d++) {
            X[d] = src[3 * o + d];
            sl[d] = ifsl ? ssl[3 * o + d] : 0.0;
            dl[d] = ifdl ? sdl[3 * o + d] : 0.0;
            dv[d] = ifdl ? sdv[3 * o + d] : 0.0;
            pts[3 * (size_t)i + d] = X[d];
        }
        double *r = nodes + (size_t)i * NODE_STRIDE;
        r[0] = X[0];
        r[1] = X[1];
        r[2] = X[2];
        for (int j = 0; j < 3; j++) {
            r[3 + j] = ifsl ? sl[j] / (2 * rmu) : 0.0;
            for (int d = 0; d < 3; d++) r[7 + 3 * j + d] = ifdl ? (dv[d] * dl[j] + dl[d] * dv[j]) / 2 : 0.0;
        }
        double q = 0.0;
        if (ifsl) q = (sl[0] * X[0] + sl[1] * X[1] + sl[2] * X[2]) * c1 / (2 * rmu);
        if (ifdl) q += (dl[0] * dv[0] + dl[1] * dv[1] + dl[2] * dv[2]) * c2;
        r[6] = q;
        double dlx = dl[0] * X[0] + dl[1] * X[1] + dl[2] * X[2], dvx = dv[0] * X[0] + dv[1] * X[1] + dv[2] * X[2];
        for (int d = 0; d < 3; d++) r[16 + d] = ifdl ? (c1 * dv[d] * dlx + c1 * dl[d] * dvx) / 2 : 0.0;
        r[19] = 0.0;
    } else if (i < n + nt) {
        size_t o = (size_t)izt[i - n];
        for (int d = 0; d < 3; d++) pts[3 * (size_t)i + d] = tgt[3 * o + d];
    }
}

constexpr int PN_THREADS = 256;     // lanes per workgroup
constexpr int PN_TILE = 256;        // source records per LDS tile
constexpr int PN_REC = 14;          // x y z, f[3], D xx xy xz yy yz zz, c2 tr D, pad

// Near field of point sources: each point of a leaf (its sources, then its
// targets) against the sources of the leaf's near boxes (self + list 1),
// without the self pair (lfmm3dparthess_direct_self / _direct,
// src/lfmm3dparthess.f:1150-1470). A pair is evaluated as the elastic fields
// themselves, not as the four Laplace problems the reference splits them
// into: with R = x - y, f = sigma_sl / (2 mu), D = sym(sigma_dl x sigma_dv),
// v = D R, c1 + c2 = 1,
//   u      = R along + (2 - c1) f / r + 2 c2 v / r^3
//   strain = I along + sym(R P) + 2 c2 D / r^3
//   along  = (c1 f.R - c2 tr D + 3 c1 R.v / r^2) / r^3
//   P      = -(3 (c1 f.R - c2 tr D) + 15 c1 R.v / r^2) R / r^5
//            + (2 c1 - 2) f / r^3 + 6 (c1 - c2) v / r^5
// about 80 operations a pair (both layers, strain) with 10 sums to hold,
// against 290 and 40 for the Laplace fields. Bound by FP64 vector issue.
// A point's sources are dealt to S lanes (a power of two, chosen per leaf by
// point_chunks), added across them at the end; a workgroup takes PN_THREADS
// consecutive (point, lane) pairs of one leaf, chunk = (near box, first
// pair, S), and the source records go through LDS in tiles.
// 1,000,000 points at iprec 2 (5.8e9 pairs): 53.4 ms as Laplace fields, 19.1
// in this form (beside the far field); 3,704 points at iprec 1: 0.80 and 0.03.
template <bool SL, bool DL, bool ST>
__global__ __launch_bounds__(PN_THREADS) void k_pnear(int n, int src_eval, const int *__restrict__ nfb,
                                                     const int *__restrict__ nfs, const int *__restrict__ nfi,
                                                     const int *__restrict__ ss, const int *__restrict__ sc,
                                                     const int *__restrict__ ts, const int *__restrict__ tc,
                                                     const int *__restrict__ chunks,
                                                     const double *__restrict__ pts,
                                                     const double *__restrict__ nodes, double c1,
                                                     double *__restrict__ nf)
{
    __shared__ __align__(16) double S[PN_TILE * PN_REC];
    int q = chunks[3 * blockIdx.x], l0 = chunks[3 * blockIdx.x + 1], split = chunks[3 * blockIdx.x + 2];
    int b = nfb[q];
    int nsb = src_eval ? sc[b] : 0;
    int loc = (l0 + (int)threadIdx.x) / split, sub = (int)threadIdx.x & (split - 1);
    bool has = loc < nsb + tc[b];
    int ip = has ? (loc < nsb ? ss[b] + loc : n + ts[b] + (loc - nsb)) : -1;
    double x = has ? pts[3 * (size_t)ip] : 0.0, y = has ? pts[3 * (size_t)ip + 1] : 0.0,
           z = has ? pts[3 * (size_t)ip + 2] : 0.0;
    const double c2 = 1.0 - c1;
    double u0 = 0.0, u1 = 0.0, u2 = 0.0, al = 0.0;
    double hxx = 0.0, hyy = 0.0, hzz = 0.0, hxy = 0.0, hxz = 0.0, hyz = 0.0;   // off-diagonal sums doubled
    auto pair = [&](const double *r, bool self) {
        double Rx = x - r[0], Ry = y - r[1], Rz = z - r[2];
        double r2 = Rx * Rx + Ry * Ry + Rz * Rz;
        // 1/sqrt(r2) from the hardware estimate and one third-order step
        double i1 = __builtin_amdgcn_rsq(r2);
        double e = fma(-r2 * i1, i1, 1.0);
        i1 = fma(i1 * e, fma(0.375, e, 0.5), i1);
        if (self) i1 = 0.0;
        double i2 = i1 * i1, i3 = i1 * i2, i5 = i3 * i2;
        double t = 0.0, w = 0.0, vx = 0.0, vy = 0.0, vz = 0.0;
        if (SL) t = c1 * (r[3] * Rx + r[4] * Ry + r[5] * Rz);
        if (DL) {
            vx = r[6] * Rx + r[7] * Ry + r[8] * Rz;
            vy = r[7] * Rx + r[9] * Ry + r[10] * Rz;
            vz = r[8] * Rx + r[10] * Ry + r[11] * Rz;
            w = (vx * Rx + vy * Ry + vz * Rz) * i2;
            t -= r[12];
        }
        double along = i3 * (DL ? fma(3.0 * c1, w, t) : t);
        u0 = fma(along, Rx, u0);
        u1 = fma(along, Ry, u1);
        u2 = fma(along, Rz, u2);
        double g3 = 2.0 * c2 * i3;
        if (SL) {
            double g1 = (2.0 - c1) * i1;
            u0 = fma(g1, r[3], u0);
            u1 = fma(g1, r[4], u1);
            u2 = fma(g1, r[5], u2);
        }
        if (DL) {
            u0 = fma(g3, vx, u0);
            u1 = fma(g3, vy, u1);
            u2 = fma(g3, vz, u2);
        }
        if (ST) {
            double ga = i5 * (DL ? fma(-15.0 * c1, w, -3.0 * t) : -3.0 * t);
            double px = ga * Rx, py = ga * Ry, pz = ga * Rz;
            if (SL) {
                double a3 = -g3;                      // 2 c1 - 2 = -2 c2
                px = fma(a3, r[3], px);
                py = fma(a3, r[4], py);
                pz = fma(a3, r[5], pz);
            }
            if (DL) {
                double b5 = 6.0 * (c1 - c2) * i5;
                px = fma(b5, vx, px);
                py = fma(b5, vy, py);
                pz = fma(b5, vz, pz);
            }
            al += along;
            hxx = fma(Rx, px, hxx);
            hyy = fma(Ry, py, hyy);
            hzz = fma(Rz, pz, hzz);
            hxy = fma(Rx, py, fma(Ry, px, hxy));
            hxz = fma(Rx, pz, fma(Rz, px, hxz));
            hyz = fma(Ry, pz, fma(Rz, py, hyz));
            if (DL) {
                double g6 = 2.0 * g3;
                hxx = fma(g3, r[6], hxx);
                hxy = fma(g6, r[7], hxy);
                hxz = fma(g6, r[8], hxz);
                hyy = fma(g3, r[9], hyy);
                hyz = fma(g6, r[10], hyz);
                hzz = fma(g3, r[11], hzz);
            }
        }
    };
    for (int k = nfs[q]; k < nfs[q + 1]; k++) {
        int jb = nfi[k], j0 = ss[jb], cnt = sc[jb];
        for (int t0 = 0; t0 < cnt; t0 += PN_TILE) {
            int m = min(PN_TILE, cnt - t0);
            __syncthreads();                          // previous tile done
            for (int sj = threadIdx.x; sj < m; sj += PN_THREADS) {
                const double *o = nodes + (size_t)(j0 + t0 + sj) * NODE_STRIDE;
                double *d = S + sj * PN_REC;
                for (int c = 0; c < 6; c++) d[c] = o[c];
                d[6] = o[7];
                d[7] = o[8];
                d[8] = o[9];
                d[9] = o[11];
                d[10] = o[12];
                d[11] = o[15];
                d[12] = c2 * (o[7] + o[11] + o[15]);
            }
            __syncthreads();
            if (!has) continue;
            if (jb == b && src_eval) {                // the self pair is in this box
                for (int sj = sub; sj < m; sj += split) pair(S + sj * PN_REC, j0 + t0 + sj == ip);
            } else {
                for (int sj = sub; sj < m; sj += split) pair(S + sj * PN_REC, false);
            }
        }
    }
    double g[9] = {u0, u1, u2, hxx + al, hyy + al, hzz + al, 0.5 * hxy, 0.5 * hxz, 0.5 * hyz};
    for (int off = split >> 1; off > 0; off >>= 1)
#pragma unroll
        for (int c = 0; c < 9; c++) g[c] += __shfl_xor(g[c], off);
    if (!has || sub) return;
    double *o = nf + (size_t)ip * 9;
#pragma unroll
    for (int c = 0; c < 9; c++) o[c] = g[c];
}

// ------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------

namespace {

struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
    ~DevBuf()
    {
        if (p) (void)hipFree(p);
    }
    template <class T>
    T *get()
    {
        return (T *)p;
    }
    void ensure(size_t b)
    {
        if (b <= bytes) return;
        if (p) HIPOK(hipFree(p));
        p = nullptr;
        bytes = 0;
        HIPOK(hipMalloc(&p, std::max<size_t>(b, 256)));
        bytes = std::max<size_t>(b, 256);
    }
};

struct OpsCache {
    int p = -1;
    double eps = -1;
    Operators ops;
    DevBuf m2m, l2l, m2l;
    DevBuf ft_loc, ft_mp;                            // field tables of L2T / M2T
    // Mindlin harmonic far field: full-order operators of the near list-2
    // offsets (|dz| <= 1) and the plane-wave / proxy tables
    bool mind_ready = false;
    Operators mind_ops;
    DevBuf mind_m2l, mind_tab, mind_px, mind_pxo;    // ..., proxy matrices and their offsets
    MindPw mind_pw{};
    int mind_nq = 0;
    size_t mind_off[8] = {};                         // ycst, gl, ytab, eph, wl, pw tab, pw ints
};

constexpr int NPHASE = 12;

// Per-device state shared by all host threads (created and read under g_mu;
// an OpsCache is immutable once built).
struct DeviceState {
    bool tables = false;
    int cus = 256;                                   // compute units
    bool p2x_wide = false;                           // 16-wave P2M/P2L for orders above 26
    std::map<int, std::unique_ptr<OpsCache>> ops;   // by iprec
};

// P2M/P2L launch shapes: 8 waves x 7 row tiles with 8-node chunks up to 56
// tiles (p <= 26); above, 16 waves x 7 tiles with 8-node chunks (116 KB of
// LDS, where the device allows it), else 8 waves x 14 tiles with 4-node chunks
constexpr int P2X_WIDE_STRIDE = 16 * 16 * 7 + 16;   // rows of 112 tiles, padded off a bank multiple

std::mutex g_mu;
std::map<int, DeviceState *> *g_dev = new std::map<int, DeviceState *>();
thread_local double g_times[16];
// half-space parts evaluated (bit 0 image near field, bit 1 anti-image far
// field, bit 2 Mindlin harmonic far field): a diagnostic for tests that
// compare each part with the reference's routine of that part
std::atomic<int> g_half_parts{7};
thread_local double g_stats[16];

DeviceState &device_state()
{
    int dev = 0;
    HIPOK(hipGetDevice(&dev));
    auto &ds = (*g_dev)[dev];
    if (!ds) ds = new DeviceState();
    if (!ds->tables) {
        hipLaunchKernelGGL(k_tables, dim3(64), dim3(256), 0, 0);
        HIPOK(hipGetLastError());
        HIPOK(hipDeviceSynchronize());
        // M2T stages the four expansions of a slot (order up to PMAX) in LDS
        int mf = NRHS * (PMAX + 1) * (PMAX + 2) * 8;
        HIPOK(hipFuncSetAttribute((const void *)k_m2t, hipFuncAttributeMaxDynamicSharedMemorySize, mf));
        for (auto *k : {k_m2l_turned_max, k_m2m_l2l_max})
            HIPOK(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)trans_lds(PMAX)));
        for (auto *k : {k_m2l_turned_26, k_m2m_l2l_26})
            HIPOK(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)trans_lds(26)));
        int wide = 8 * P2X_WIDE_STRIDE * 8;
        ds->p2x_wide =
            hipFuncSetAttribute((const void *)k_p2m<16, 7, 8>, hipFuncAttributeMaxDynamicSharedMemorySize, wide) ==
                hipSuccess &&
            hipFuncSetAttribute((const void *)k_p2l<16, 7, 8>, hipFuncAttributeMaxDynamicSharedMemorySize, wide) ==
                hipSuccess;
        (void)hipGetLastError();                     // a refused size leaves the narrow shape in use
        auto tri_lds = [](auto z) {                  // 154 KB for the largest shape
            using Z = decltype(z);
            int ph = 0;
            while (Z::fits(ph + 1)) ph++;
            int b = Z::lds(ph) * 8;
            for (const void *k : {(const void *)k_p2m_tri<Z, false>, (const void *)k_p2m_tri<Z, true>, (const void *)k_p2l_tri<Z>})
                HIPOK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, b));
        };
        tri_lds(P2TShape0{});
        tri_lds(P2TShape1{});
        tri_lds(P2TShape2{});
        tri_lds(P2TShape3{});
        HIPOK(hipDeviceGetAttribute(&ds->cus, hipDeviceAttributeMultiprocessorCount, dev));
        ds->tables = true;
    }
    return *ds;
}

OpsCache &operators_for(DeviceState &ds, int iprec)
{
    auto &oc = ds.ops[iprec];
    if (!oc) {
        oc.reset(new OpsCache());
        double eps = iprec_eps(iprec);
        oc->eps = eps;
        oc->p = expansion_order(eps);
        int itab[343];
        list2_orders(eps, itab);
        try {
            build_operators(oc->p, itab, oc->ops);
        } catch (const std::exception &) {
            throw HipFailure{hipErrorInvalidValue};
        }
        oc->m2m.ensure(oc->ops.m2m.size() * 8);
        oc->l2l.ensure(oc->ops.l2l.size() * 8);
        oc->m2l.ensure(oc->ops.m2l.size() * 8);
        HIPOK(hipMemcpy(oc->m2m.p, oc->ops.m2m.data(), oc->ops.m2m.size() * 8, hipMemcpyHostToDevice));
        HIPOK(hipMemcpy(oc->l2l.p, oc->ops.l2l.data(), oc->ops.l2l.size() * 8, hipMemcpyHostToDevice));
        HIPOK(hipMemcpy(oc->m2l.p, oc->ops.m2l.data(), oc->ops.m2l.size() * 8, hipMemcpyHostToDevice));
        for (int irr = 0; irr < 2; irr++) {
            std::vector<FieldTerm> ft;
            build_field_table(oc->p, irr != 0, ft);
            DevBuf &d = irr ? oc->ft_mp : oc->ft_loc;
            d.ensure(ft.size() * sizeof(FieldTerm));
            HIPOK(hipMemcpy(d.p, ft.data(), ft.size() * sizeof(FieldTerm), hipMemcpyHostToDevice));
        }
    }
    return *oc;
}

// Packed upload of many host arrays into one device buffer: offsets are
// assigned first (256-byte aligned), then the arrays are copied into a
// pinned staging buffer by the host pool and sent in one transfer. The
// arrays must stay unchanged until pack() has run.
struct Packer {
    struct Item {
        const void *src;
        size_t bytes, off;
    };
    std::vector<Item> items;
    size_t size = 0;
    template <class T>
    size_t add(const std::vector<T> &v)
    {
        size_t off = (size + 255) & ~(size_t)255;
        items.push_back({v.data(), v.size() * sizeof(T), off});
        size = off + v.size() * sizeof(T);
        return off;
    }
    void pack(char *dst) const
    {
        constexpr size_t PIECE = 1 << 20;
        std::vector<std::pair<int, size_t>> work;     // (item, piece start)
        for (size_t i = 0; i < items.size(); i++)
            for (size_t a = 0; a < items[i].bytes; a += PIECE) work.push_back({(int)i, a});
        parallel_chunks((int)work.size(), [&](int w, int) {
            const Item &it = items[work[w].first];
            size_t a = work[w].second, e = std::min(it.bytes, a + PIECE);
            std::memcpy(dst + it.off + a, (const char *)it.src + a, e - a);
        });
    }
};

// Grow-only pinned host buffer (hipHostMalloc).
struct PinnedBuf {
    char *p = nullptr;
    size_t bytes = 0;
    void ensure(size_t b)
    {
        if (b <= bytes) return;
        if (p) HIPOK(hipHostFree(p));
        p = nullptr;
        bytes = 0;
        size_t nb = b + b / 4 + 4096;
        HIPOK(hipHostMalloc((void **)&p, nb, hipHostMallocDefault));
        bytes = nb;
    }
};

constexpr int SET_LANES = 8;

// Device buffers of one Mindlin far field.
struct MindScratch {
    DevBuf exps, pts, lap, inp, rec, pw, skel, gm, tcoef;
    std::shared_ptr<elfmm::MindPlan> plan;           // of the last far field (for a later assembly)
};

// Per-host-thread state: device buffers, the near-field stream and the
// events of one apply. Applies on different host threads (each on its own
// stream) run concurrently: host planning of one overlaps device work of
// the others.
struct Workspace {
    DevBuf plan, inp, exps, pts, lap, nf, nodes, rec;
    DevBuf part[3];                                  // far-field lists of a plan sent in parts
    DevBuf tgtm, htmp, hq;                           // half space: mirrored targets, icomp-1 pairs, queue
    MindScratch mind[SET_LANES];                     // Mindlin far field, one per set lane
    DevBuf dmulti, nfm;                           // several density sets: densities, near fields
    std::vector<double> hsrc, htgt;
    std::unique_ptr<OctreeWork> oct;                 // device octree buffers
    Plan planh;
    Tree treeh;
    std::vector<int> near_waves;
    PinnedBuf stage, part_stage[3];   // plan staging; the call that filled them has completed before reuse
    hipStream_t near_stream = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr, ev_done = nullptr;
    hipEvent_t ev[2 * NPHASE] = {};
    // several density sets: far fields of SET_LANES sets at a time, each on
    // its own stream with its own scratch
    hipStream_t set_stream[SET_LANES] = {};
    hipEvent_t set_ev[SET_LANES] = {};
    hipEvent_t ev_mind[2] = {};                      // device time of a Mindlin far field beside the anti-image
    DevBuf set_exps[SET_LANES], set_lap[SET_LANES], set_nodes[SET_LANES];
    void init_set_lanes()
    {
        if (set_stream[0]) return;
        for (int j = 0; j < SET_LANES; j++) {
            HIPOK(hipStreamCreateWithFlags(&set_stream[j], hipStreamNonBlocking));
            HIPOK(hipEventCreateWithFlags(&set_ev[j], hipEventDisableTiming));
        }
        HIPOK(hipEventCreate(&ev_mind[0]));
        HIPOK(hipEventCreate(&ev_mind[1]));
    }
    void init_streams()
    {
        if (near_stream) return;
        HIPOK(hipStreamCreateWithFlags(&near_stream, hipStreamNonBlocking));
        HIPOK(hipEventCreateWithFlags(&ev_fork, hipEventDisableTiming));
        HIPOK(hipEventCreateWithFlags(&ev_join, hipEventDisableTiming));
        HIPOK(hipEventCreateWithFlags(&ev_done, hipEventDisableTiming));
        for (int i = 0; i < 2 * NPHASE; i++) HIPOK(hipEventCreate(&ev[i]));
    }
};
thread_local Workspace *g_ws = nullptr;   // lives until process exit
thread_local Tree *g_oct_tree = nullptr;  // the last elfmm_gfx950_octree_dev tree of this thread

// The far fields of different applies take a device in the order the
// applies finish planning: an apply's first far-field kernel waits for the
// last far-field kernel of the apply before it (from any host thread, on
// any stream). Without the order, two applies in flight share the GPU,
// finish together and then plan their next requests together while the GPU
// idles; with it, one request's host planning overlaps the kernels of the
// request ahead of it. Near fields (their own stream, their own buffers)
// are not ordered: the next apply's near field fills what the current far
// field leaves idle. The tail event belongs to a workspace, and workspaces
// live until process exit.
// Applies plan (octree, lists, task lists) one at a time: the planner's
// parallel regions share one worker pool, so applies planning together
// interleave their regions and all finish late; in turn, the first one
// reaches the GPU after one planning time instead of several.
std::mutex g_plan_mu;

// Applies in progress in this process (all devices), and the others an
// apply saw when it started.
std::atomic<int> g_inflight{0};
struct InFlight {
    int others;
    InFlight() : others(g_inflight.fetch_add(1)) {}
    ~InFlight() { g_inflight.fetch_sub(1); }
};

constexpr int ORDER_DEVICES = 64;
std::mutex g_order_mu;
hipEvent_t g_order_tail[ORDER_DEVICES] = {};

double now_ms()
{
    return std::chrono::duration<double, std::milli>(
               std::chrono::steady_clock::now().time_since_epoch())
        .count();
}

int max_lds()
{
    static int v = 0;
    if (!v) {
        int dev = 0;
        (void)hipGetDevice(&dev);
        hipDeviceProp_t pr;
        if (hipGetDeviceProperties(&pr, dev) == hipSuccess)
            v = (int)std::min<size_t>(pr.sharedMemPerBlock, 65536);
        else
            v = 65536;
    }
    return v;
}

// Offsets of the arrays of a tree and its plan, each in the packed device
// buffer of its part (FarLaunch), which may be one and the same.
struct PlanOffsets {
    size_t iz, izt, cen, side, ss, sc, ts, tc, p2m, p2mp, p2lb, p2ls, p2li, l2t, l2tp, m2tsb, m2tp, l2tw, m2tw, m2tbt;
    size_t nfb, nfs, nfi, m2lt;
    size_t nfw, near_waves = 0;                      // near_tasks, where the near field is integrated
    std::vector<LaunchOff> m2m, l2l;
    LaunchOff m2l;
};

// Points and near field: what the gather, the near field and the assembly
// read, and the boxes' sources.
void pack_near(Packer &pk, const Tree &T, const Plan &PL, PlanOffsets &o)
{
    o.iz = pk.add(T.iz);
    o.izt = pk.add(T.iztarg);
    o.ss = pk.add(T.src_start);
    o.sc = pk.add(T.src_count);
    o.ts = pk.add(T.tgt_start);
    o.tc = pk.add(T.tgt_count);
    o.nfb = pk.add(PL.nf_boxes);
    o.nfs = pk.add(PL.nf_start);
    o.nfi = pk.add(PL.nf_items);
}

void pack_near_tasks(Packer &pk, const std::vector<int> &tasks, PlanOffsets &o)
{
    o.nfw = pk.add(tasks);
    o.near_waves = tasks.size() / 3;
}

LaunchOff pack_launch(Packer &pk, const GemmLaunch &g)
{
    LaunchOff l;
    l.tiles = pk.add(g.tiles);
    l.src = pk.add(g.src);
    l.dst = pk.add(g.dst);
    l.sc = pk.add(g.scale);
    return l;
}

// The three parts of the far-field lists (build_plan_up, _m2l, _eval)
void pack_up(Packer &pk, const Tree &T, const Plan &PL, PlanOffsets &o)
{
    o.cen = pk.add(T.centers);
    o.side = pk.add(PL.sides);
    o.p2m = pk.add(PL.p2m_boxes);
    o.p2mp = pk.add(PL.p2m_parts);
    o.p2lb = pk.add(PL.p2l_boxes);
    o.p2ls = pk.add(PL.p2l_start);
    o.p2li = pk.add(PL.p2l_items);
    o.m2m.clear();
    for (auto &g : PL.m2m_l) o.m2m.push_back(pack_launch(pk, g));
}

void pack_m2l(Packer &pk, const Plan &PL, PlanOffsets &o)
{
    o.l2l.clear();
    for (auto &g : PL.l2l_l) o.l2l.push_back(pack_launch(pk, g));
    o.m2l = pack_launch(pk, PL.m2l);
    o.m2lt = pk.add(PL.m2l_tiles);
}

void pack_eval(Packer &pk, const Plan &PL, PlanOffsets &o)
{
    o.l2t = pk.add(PL.l2t_boxes);
    o.l2tp = pk.add(PL.l2t_tpt);
    o.m2tsb = pk.add(PL.m2t_slot_box);
    o.m2tp = pk.add(PL.m2t_tpt);
    o.l2tw = pk.add(PL.l2t_wt);
    o.m2tw = pk.add(PL.m2t_wt);
    o.m2tbt = pk.add(PL.m2t_bt);
}

void pack_plan(Packer &pk, const Tree &T, const Plan &PL, PlanOffsets &o)
{
    pack_near(pk, T, PL, o);
    pack_up(pk, T, PL, o);
    pack_m2l(pk, PL, o);
    pack_eval(pk, PL, o);
}

// One far field of the free-space (or anti-image) FMM: the four Laplace
// problems from quadrature nodes to 40 fields per point (potential,
// gradient, Hessian of each problem), src/lfmm3dtrilhess.f steps 1-7.
struct FarLaunch {
    const DeviceState *ds;
    const OpsCache *oc;
    const Plan *PL;
    const PlanOffsets *o;
    // the packed plan on the device: points and near field, then the parts of
    // the far field
    const char *P, *PU, *PM, *PE;
    int iprec, n, nb;
    const double *tri_s, *nrm_s, *ssl, *sdl;         // tree order
    int ifsl, ifdl;
    double mu, c1, c2, dls;                          // k_nodes coefficients and double-layer sign
    const double *pts;
    double *nodes, *exps, *lap;                      // scratch of far_scratch() doubles each
    bool points = false;                             // nodes already hold point sources (one per source)
};

// Doubles of FarLaunch scratch: nodes, expansions (multipoles then
// locals), fields.
void far_scratch(int iprec, int n, int np, int nb, int p, size_t &nodes, size_t &exps, size_t &lap)
{
    int nq, q0;
    quad_rule(iprec, nq, q0);
    nodes = (size_t)n * nq * NODE_STRIDE;            // or 48 coefficients per triangle (k_tcoef), nq >= 6
    exps = (size_t)2 * nb * NRHS * ncoef(p);
    lap = (size_t)np * 40;
}

// M2M / L2L of one level (unit scale)
void enqueue_trans(const GemmLaunch &g, const LaunchOff &l, const char *P, const DevBuf &A, const double *X, double *Y,
                   int nc, Lane &ln)
{
    if (g.tiles.empty()) return;
    int ntiles = (int)g.tiles.size(), p = (int)(std::sqrt(nc + 0.25) - 1.0);   // nc = (p + 1)(p + 2)
    ln.launch(m2m_l2l_kernel(p), trans_grid(ntiles, nc / 2), dim3(trans_threads(p)), trans_lds(p), (const M2LTile *)(P + l.tiles),
              ntiles, 0, (const double *)A.p, (const int *)(P + l.src), (const int *)(P + l.dst),
              (const double *)(P + l.sc), X, Y, nc);
}

// M2L: the turned orders (the list's first tiles, xcd_order), then the others
void enqueue_m2l_tiles(const std::vector<M2LTile> &list, size_t at, const LaunchOff &l, const char *P, const double *A,
                       int p, const double *X, double *Y, Lane &ln)
{
    const int nc = ncoef(p), ht = m2l_turned_h(p);
    auto turned = [&](const M2LTile &t) { return t.npair > 0 && t.h >= ht; };
    int n1 = (int)list.size(), n0 = 0;
    while (n1 && !turned(list[n1 - 1])) n1--;
    while (n0 < (int)list.size() && (turned(list[n0]) || list[n0].npair <= 0)) n0++;
    n0 = n0 / 8 * 8;                                  // XCD of a workgroup: index % 8
    const M2LTile *tiles = (const M2LTile *)(P + at);
    const int *src = (const int *)(P + l.src), *dst = (const int *)(P + l.dst);
    const double *sc = (const double *)(P + l.sc);
    if (n1)
        ln.launch(p <= 26 ? k_m2l_turned_26 : k_m2l_turned_max, trans_grid(n1, ht), dim3(trans_threads(p)), trans_lds(p), tiles, n1, ht, A, src, dst, sc, X, Y,
                  nc);
    const int nd = (int)list.size() - n0;
    if (nd > 0)
        ln.launch(k_m2l, dim3(nd), dim3(ML_THREADS), 0, tiles + n0, nd, ht, A, src, dst, sc, X, Y, nc);
}

// P2M, M2M and P2L (build_plan_up)
template <class Mark>
void enqueue_up(const FarLaunch &a, size_t np, Lane &ln, Mark mark)
{
    const Plan &PL = *a.PL;
    const PlanOffsets &o = *a.o;
    const OpsCache &oc = *a.oc;
    const int *ss = (const int *)(a.P + o.ss), *sc = (const int *)(a.P + o.sc);
    auto I = [&](size_t off) { return (const int *)(a.PU + off); };
    auto D = [&](size_t off) { return (const double *)(a.PU + off); };
    const int p = oc.p, nc = ncoef(p), n = a.n;
    int nq, q0;
    quad_rule(a.iprec, nq, q0);
    if (a.points) nq = 1;
    double *mp = a.exps, *lo = mp + (size_t)a.nb * NRHS * nc;
    mark(2, true);
    ln.fill0(a.exps, (size_t)2 * a.nb * NRHS * nc);
    ln.fill0(a.lap, np * 40);
    // triangles with 6 or 12 nodes go through three moments each; rules of 1 and
    // 3 nodes and point sources through one product per node
    const bool tri = !a.points && nq >= 6;
    if (tri)
        ln.launch(k_tcoef, dim3((n + 255) / 256), dim3(256), 0, n, a.tri_s, a.nrm_s, a.ssl, a.sdl, a.ifsl, a.ifdl,
                  a.mu, a.c1, a.c2, a.dls, a.nodes);
    else if (!a.points)
        ln.launch(k_nodes, dim3((nq * n + 255) / 256), dim3(256), 0, n, nq, q0, a.tri_s, a.nrm_s, a.ssl, a.sdl,
                  a.ifsl, a.ifdl, a.mu, a.c1, a.c2, a.dls, a.nodes);
    auto p2t = [&](auto z, bool irr, size_t nbx, const int *bx, const int *ls, const int *li, double *out) {
        using Z = decltype(z);
        size_t sh = (size_t)Z::lds(irr ? p + 1 : p) * 8;
        if (irr)
            ln.launch(k_p2l_tri<Z>, dim3(nbx), dim3(Z::NT), sh, p, bx, ls, li, D(o.cen), D(o.side), ss, sc,
                      a.tri_s, (const double *)a.nodes, nc, out);
        else
            ln.launch(k_p2m_tri<Z, false>, dim3(PL.p2m_parts.size() / 3), dim3(Z::NT), sh, p, bx, I(o.p2mp),
                      MindMoments{}, D(o.cen), D(o.side), ss, sc, a.tri_s, (const double *)a.nodes, nc, out);
    };
    // P2M / P2L: moments on the matrix cores (shapes at P2X_WIDE_STRIDE)
    auto p2x = [&](bool irr, size_t nbx, const int *bx, const int *ls, const int *li, double *out) {
        int ph = irr ? p + 1 : p;
        int ntiles = ((ph + 1) * (ph + 2) + 15) / 16;
        int shape = ntiles <= 8 * 7 ? 0 : (a.ds->p2x_wide ? 1 : 2);
        int wb = shape == 1 ? 16 : 8, tw = shape == 2 ? 14 : 7, nk = shape == 2 ? 4 : 8;
        int rows = 16 * wb * tw;                            // WB * TW tiles, zero-padded
        int stride = rows + (rows % 32 == 0 ? 16 : 0);
        size_t sh = (size_t)nk * stride * 8;                // nk nodes of harmonics
        if (ntiles > wb * tw || (shape != 1 && (int)sh > max_lds()) || nk * (ph + 1) > 64 * wb)
            HIPOK(hipErrorInvalidValue);
        auto kern = irr ? (shape == 0 ? k_p2l<8, 7, 8> : shape == 1 ? k_p2l<16, 7, 8> : k_p2l<8, 14, 4>)
                        : (shape == 0 ? k_p2m<8, 7, 8> : shape == 1 ? k_p2m<16, 7, 8> : k_p2m<8, 14, 4>);
        ln.launch(kern, dim3(nbx), dim3(64 * wb), sh, p, nq, stride, bx, ls, li, D(o.cen), D(o.side), ss,
                  sc, (const double *)a.nodes, nc, out);
    };
    auto p2 = [&](bool irr, size_t nbx, const int *bx, const int *ls, const int *li, double *out) {
        if (!tri) return p2x(irr, nbx, bx, ls, li, out);
        switch (p2t_shape(irr ? p + 1 : p, nq)) {
        case 0: return p2t(P2TShape0{}, irr, nbx, bx, ls, li, out);
        case 1: return p2t(P2TShape1{}, irr, nbx, bx, ls, li, out);
        case 2: return p2t(P2TShape2{}, irr, nbx, bx, ls, li, out);
        case 3: return p2t(P2TShape3{}, irr, nbx, bx, ls, li, out);
        default: HIPOK(hipErrorInvalidValue);
        }
    };
    if (!PL.p2m_boxes.empty()) p2(false, PL.p2m_boxes.size(), I(o.p2m), nullptr, nullptr, mp);
    mark(2, false);
    mark(3, true);
    for (size_t k = 0; k < PL.m2m_l.size(); k++) enqueue_trans(PL.m2m_l[k], o.m2m[k], a.PU, oc.m2m, mp, mp, nc, ln);
    mark(3, false);
    mark(5, true);
    if (!PL.p2l_boxes.empty()) p2(true, PL.p2l_boxes.size(), I(o.p2lb), I(o.p2ls), I(o.p2li), lo);
    mark(5, false);
}

// M2L and L2L (build_plan_m2l)
template <class Mark>
void enqueue_m2l(const FarLaunch &a, Lane &ln, Mark mark)
{
    const Plan &PL = *a.PL;
    const PlanOffsets &o = *a.o;
    const OpsCache &oc = *a.oc;
    const char *P = a.PM;
    const int nc = ncoef(oc.p);
    double *mp = a.exps, *lo = mp + (size_t)a.nb * NRHS * nc;
    mark(4, true);
    enqueue_m2l_tiles(PL.m2l_tiles, o.m2lt, o.m2l, P, (const double *)oc.m2l.p, oc.p, mp,
                      lo, ln);
    mark(4, false);
    mark(6, true);
    for (size_t k = 0; k < PL.l2l_l.size(); k++) enqueue_trans(PL.l2l_l[k], o.l2l[k], P, oc.l2l, lo, lo, nc, ln);
    mark(6, false);
}

// L2T and M2T (build_plan_eval)
template <class Mark>
void enqueue_eval(const FarLaunch &a, Lane &ln, Mark mark)
{
    const Plan &PL = *a.PL;
    const PlanOffsets &o = *a.o;
    const OpsCache &oc = *a.oc;
    const double *cen = (const double *)(a.PU + o.cen), *side = (const double *)(a.PU + o.side);
    auto I = [&](size_t off) { return (const int *)(a.PE + off); };
    const int p = oc.p, nc = ncoef(p);
    double *mp = a.exps, *lo = mp + (size_t)a.nb * NRHS * nc;
    auto meval = [&](bool irr, size_t o_sb, size_t o_wt, int nwt, size_t o_bt, int nbt, size_t o_tp, const double *ex) {
        int ph = irr ? p + 2 : p;
        int nsteps = ((ph + 1) * (ph + 2) / 2 + 1) / 2;
        if (irr) {   // M2T: several wave tasks per slot sharing the operand, formed in LDS
            size_t sh = (size_t)NRHS * nc * 8;
            ln.launch(k_m2t, dim3(nbt), dim3(64 * EW_WAVES), sh, p, nwt, I(o_wt), I(o_bt), I(o_tp), I(o_sb),
                      cen, side, a.pts, ex, nc, (const FieldTerm *)oc.ft_mp.p, nsteps, a.lap);
        } else {     // L2T: mostly one wave task per leaf; each wave forms its operand
            ln.launch(k_l2t, dim3((nwt + EB_WAVES - 1) / EB_WAVES), dim3(64 * EB_WAVES), 0, p, nwt, I(o_wt),
                      I(o_tp), I(o_sb), cen, side, a.pts, ex, nc, (const FieldTerm *)oc.ft_loc.p, nsteps,
                      a.lap);
        }
    };
    mark(7, true);
    if (!PL.l2t_tpt.empty()) meval(false, o.l2t, o.l2tw, (int)PL.l2t_wt.size() / 3, 0, 0, o.l2tp, lo);
    mark(7, false);
    mark(8, true);
    if (!PL.m2t_tpt.empty())
        meval(true, o.m2tsb, o.m2tw, (int)PL.m2t_wt.size() / 3, o.m2tbt, (int)PL.m2t_bt.size() - 1, o.m2tp, mp);
    mark(8, false);
}

// Enqueues the far field on one stream with kernel launches only (no
// memsets, copies or host waits), so that it can be captured into a graph.
// mark(k, begin) brackets phase k (2 nodes and P2M, 3 M2M, 4 M2L, 5 P2L, 6
// L2L, 7 L2T, 8 M2T) for the caller's timing events.
template <class Mark>
void enqueue_far(const FarLaunch &a, size_t np, Lane &ln, Mark mark)
{
    enqueue_up(a, np, ln, mark);
    enqueue_m2l(a, ln, mark);
    enqueue_eval(a, ln, mark);
}

// The far-field lists of a plan in three parts, each packed, sent and started
// before the next is built, so that the host builds M2L's lists beside P2M, M2M
// and P2L and the evaluation's beside M2L (81,920 triangles + 100,000 targets:
// the lists take 3 ms of host time, the kernels before M2L 3.3 ms; apply 19.8 ->
// 16.2 ms). Only for an apply that is alone: its far field would hold up the
// others' while the host builds (far fields run in order).
template <class Mark>
void run_far_parts(FarLaunch a, const Tree &T, Plan &PL, PlanOffsets &o, bool src_eval, size_t np, Workspace &W,
                   Lane &ln, Mark mark)
{
    auto send = [&](int part, auto &&pack) {
        Packer pk;
        pack(pk);
        W.part[part].ensure(pk.size);
        W.part_stage[part].ensure(pk.size);
        pk.pack(W.part_stage[part].p);
        HIPOK(hipMemcpyAsync(W.part[part].p, W.part_stage[part].p, pk.size, hipMemcpyHostToDevice, ln.stream));
        return (const char *)W.part[part].p;
    };
    const Operators *ops = &a.oc->ops;
    build_plan_up(T, ops, PL, false);
    a.PU = send(0, [&](Packer &pk) { pack_up(pk, T, PL, o); });
    enqueue_up(a, np, ln, mark);
    build_plan_m2l(T, ops, src_eval, NRHS, PL);
    a.PM = send(1, [&](Packer &pk) { pack_m2l(pk, PL, o); });
    enqueue_m2l(a, ln, mark);
    build_plan_eval(T, a.n, ops, src_eval, PL, false);
    a.PE = send(2, [&](Packer &pk) { pack_eval(pk, PL, o); });
    enqueue_eval(a, ln, mark);
}

}  // namespace

// Whether an octree of np points, nbox per leaf, is built on the host although
// the device is free: the device build is a chain of about 20 launches and a
// round trip per level (0.34 ms for 217 points, 0.69 for 3,880, 0.82 for 9,200),
// the host's costs about 0.02 us a point and 1 us a box (0.005, 0.43 and 1.0
// ms for the same points at 40 to a leaf). With larger leaves the boxes are
// fewer (host and device, ms: 12,000 points at 400 to a leaf 0.26 and 0.46,
// 20,000 0.36 and 0.51; 20,000 in a cluster of many levels 1.29 and 1.69; 14,580
// at 240 0.42 and 0.60).
bool small_tree(int np, int nbox) { return np <= 6000 || (np <= 20000 && np / 64 <= nbox); }

// The apply: device pointers in, device pointers out.
// Stored near-field interactions of the iter entry points, owned by the
// library and named in the caller's wsave by a handle:
// wsave[0] = ITER_MAGIC, wsave[1] = id, wsave[2] = n, wsave[3] = nt.
constexpr int ITER_HANDLE_WORDS = 4;
constexpr double ITER_MAGIC = 1178879565.0;
struct MindPlan;

// A device-resident iter store with what later products of its geometry
// reuse. Held by shared_ptr: the registry owns one reference, every call
// using the store another, so a release (or a new store on the same wsave)
// during a call frees it only when that call has finished.
struct NearStore {
    DevBuf data;
    int64_t words = 0;
    int n = 0, nt = 0, iprec = 0;
    int flags = 0;                 // ifsl | ifdl<<1 | ifpt<<2 | ifst<<3 | ifptt<<4 | ifstt<<5
    int64_t nslots = 0;            // signature of the near lists the store was built for
    size_t nboxes = 0, nitems = 0;
    // the octree and task lists of the apply that built the store and the
    // coordinates they were built on (sources, targets as the tree saw
    // them): later products of the same coordinates use them instead of
    // planning again
    std::vector<double> xs, xt;
    std::unique_ptr<Tree> tree;
    std::unique_ptr<Plan> plan;
    // half space: the Mindlin far field's octree and plan (built by the
    // first product that needs it)
    std::mutex mind_mu;
    std::shared_ptr<MindPlan> mind;
};

std::map<long, std::shared_ptr<NearStore>> g_stores;
long g_next_store = 1;

// the store named by wsave (caller holds g_mu)
std::shared_ptr<NearStore> find_store(const double *wsave, int lwsave)
{
    if (!wsave || lwsave < ITER_HANDLE_WORDS || wsave[0] != ITER_MAGIC) return nullptr;
    auto it = g_stores.find((long)wsave[1]);
    return it == g_stores.end() ? nullptr : it->second;
}

bool same_coords(const std::vector<double> &v, const double *x, size_t nx)
{
    return v.size() == nx && (nx == 0 || std::memcmp(v.data(), x, nx * 8) == 0);
}

// One apply. it == nullptr: elfmm3dtriatarg. Otherwise the iter engine
// (elfmm3dtriatargiter, src/elfmm3dtria_iter_1.f:160): leaf size of the
// iter FMM, half-space root rule (the reference builds its iter entry
// points only in the half-space link set, with d3tstrcr_mindlin.f), lists 3
// and 4 in the near field, and icomp_type 1 (compute), 2 (compute and
// store), 3 (replay the store), 4 (plan only), 5 (store, near field only).
struct IterCall {
    int icomp;
    double *wsave;
    int lwsave;
    int status = 0;                // 64: icomp 3 found no matching store (computed directly)
    // replays of several density sets (icomp 3 only): densities and outputs
    // are nrhs consecutive blocks of the single-set layout
    int nrhs = 1;
    std::shared_ptr<NearStore> store;   // the store this call used or made
    // half space (elhfmm3dtriatargiter, src/elhfmm3dtria_iter.f:46-272):
    // tree on the sources and the mirrored targets; far field = the
    // anti-image FMM (src/elhfmm3dtria_iter.f:937-1381) with (lam + 4 mu,
    // -mu), -sigma_dl and the (c2 + 2) charge term, subtracted; near field =
    // the adaptive image integrals of lists 1, 3, 4 and self
    // (src/elhfmm3dtria_iter.f:1387-2602). Source outputs are not evaluated.
    int half = 0;
};

int triatarg_dev(int iprec, double rlam, double rmu, int n, const double *d_tri,
                 const double *d_nrm, const double *d_src, int ifsl, const double *d_ssl,
                 int ifdl, const double *d_sdl, int ifpt, double *d_pt, int ifst, double *d_st,
                 int nt, const double *d_tgt, int ifptt, double *d_ptt, int ifstt, double *d_stt,
                 hipStream_t stream, bool direct_only, IterCall *it = nullptr)
{
    for (int i = 0; i < 16; i++) g_times[i] = 0;
    double t_start = now_ms();
    if (n < 1) return 0;
    if (!direct_only && (iprec > 3 || iprec < -2)) return 16;
    InFlight inflight;
    DeviceState *dsp;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        dsp = &device_state();
    }
    DeviceState &ds = *dsp;
    if (!g_ws) g_ws = new Workspace();
    Workspace &W = *g_ws;
    W.init_streams();
    int src_eval = (ifpt || ifst) ? 1 : 0;
    int tgt_eval = (ifptt || ifstt) ? 1 : 0;
    if (!tgt_eval) nt = 0;
    double c1 = (rlam + rmu) / (rlam + 2 * rmu), c2 = rmu / (rlam + 2 * rmu);
    // Lame constants and combination coefficients of the far field: the
    // anti-image FMM in the half space (src/elhfmm3dtria_iter.f:747-750,
    // :1289)
    const bool half_far = it && it->half;
    const double lamF = half_far ? rlam + 4 * rmu : rlam, muF = half_far ? -rmu : rmu;
    const double c1F = (lamF + muF) / (lamF + 2 * muF), c2F = muF / (lamF + 2 * muF) + (half_far ? 2.0 : 0.0);

    // ---- host copies of the coordinates: iter calls compare them with a
    // kept store's; the host octree (ELFMM_HOST_TREE=1, or a tree deeper
    // than the device build holds) is built from them
    const bool half = it && it->half;
    const double *d_tgt_in = d_tgt;                  // before the half space mirrors it
    // the octree is built on the device when this is the only apply in
    // flight and the points are not few; beside other applies it is built on
    // the host, where it overlaps their kernels instead of queueing behind
    // them (ELFMM_HOST_TREE=1: always on the host, =0: always on the device)
    const char *ht_env = std::getenv("ELFMM_HOST_TREE");
    bool host_tree = direct_only || (ht_env && ht_env[0] == '1');
    const int nbox =
        direct_only ? n + nt : (it ? iprec_nbox_iter(iprec, n + nt) : iprec_nbox(iprec, n + nt));
    if (!host_tree && !(ht_env && ht_env[0] == '0')) host_tree = inflight.others > 0 || small_tree(n + nt, nbox);
    bool have_host = false;
    auto host_coords = [&]() {
        if (have_host) return;
        W.hsrc.resize(3 * (size_t)n);
        W.htgt.resize(3 * (size_t)std::max(nt, 1));
        HIPOK(hipMemcpyAsync(W.hsrc.data(), d_src, 3 * (size_t)n * 8, hipMemcpyDeviceToHost, stream));
        if (nt) HIPOK(hipMemcpyAsync(W.htgt.data(), d_tgt_in, 3 * (size_t)nt * 8, hipMemcpyDeviceToHost, stream));
        HIPOK(hipStreamSynchronize(stream));
        // the half-space tree and far field see the mirrored targets
        if (half)
            for (int j = 0; j < nt; j++) W.htgt[3 * (size_t)j + 2] = -W.htgt[3 * (size_t)j + 2];
        have_host = true;
    };
    if (it || host_tree) host_coords();
    if (half) {
        W.tgtm.ensure(3 * (size_t)std::max(nt, 1) * 8);
        HIPOK(launch_mirror(nt, d_tgt, W.tgtm.get<double>(), stream));
        d_tgt = W.tgtm.get<double>();
    }
    // one apply plans at a time, with the whole worker pool (see g_plan_mu)
    std::unique_lock<std::mutex> plan_lk(g_plan_mu);
    double t0 = now_ms();

    bool iter = it != nullptr;
    // iter products of one geometry (icomp 3 on the wsave of an icomp-2
    // apply) take the octree and task lists kept with the near-field store
    int flags0 = ifsl | ifdl << 1 | ifpt << 2 | ifst << 3 | ifptt << 4 | ifstt << 5 | (half ? 1 << 6 : 0);
    std::shared_ptr<NearStore> kept;
    if (iter && it->icomp == 3) {
        std::shared_ptr<NearStore> st;
        {
            std::lock_guard<std::mutex> lk(g_mu);
            st = find_store(it->wsave, it->lwsave);
        }
        if (st && st->tree && st->plan && st->n == n && st->nt == nt && st->iprec == iprec && st->flags == flags0 &&
            same_coords(st->xs, W.hsrc.data(), 3 * (size_t)n) && same_coords(st->xt, W.htgt.data(), 3 * (size_t)nt))
            kept = st;
    }
    Tree &Tnew = W.treeh;
    if (!kept) {
        bool deep = host_tree;
        if (!host_tree) {
            if (!W.oct) W.oct.reset(new OctreeWork());
            HIPOK(build_tree_dev(d_src, n, d_tgt, nt, nbox, iter ? 1 : 0, Tnew, *W.oct, stream, deep));
        }
        if (deep) {
            host_coords();
            if (build_tree(W.hsrc.data(), n, W.htgt.data(), nt, nbox, iter ? 1 : 0, Tnew)) return 4;
        }
    }
    const Tree &T = kept ? *kept->tree : Tnew;
    double t_tree = now_ms();
    g_times[12] = t_tree - t0;
    int nb = T.nboxes;
    OpsCache *oc = nullptr;
    if (!direct_only) {
        std::lock_guard<std::mutex> lk(g_mu);
        oc = &operators_for(ds, iprec);
    }
    int p = oc ? oc->p : 0;

    // ---- plan
    // A plain apply (no iter store, no half space) plans its near field
    // first, launches it, and builds the far-field lists while it runs
    // (ELFMM_SPLIT_PLAN=0: one plan before any launch).
    Plan &PL = kept ? *kept->plan : W.planh;
    const char *sp_env = std::getenv("ELFMM_SPLIT_PLAN");
    const bool split = !iter && !direct_only && !kept && oc && !(sp_env && sp_env[0] == '0');
    if (split) {
        plan_reset(PL);
        build_plan_near(T, src_eval, false, false, PL);
    } else {
        if (!kept) build_plan(T, n, oc ? &oc->ops : nullptr, src_eval, direct_only, NRHS, PL, iter);
        plan_lk.unlock();
        for (int i = 0; i < 16; i++) g_stats[i] = PL.stats[i];
    }
    // iter: near-store layout and the reference's store size in words
    // (elfmm3dtriaiter_count, src/elfmm3dtria_iter_1.f:1468-1515)
    std::vector<int64_t> nf_sbase;
    std::vector<int> nf_ntri, nf_pstart(1, 0);     // nf_pstart: first point of each near box
    std::vector<int> nf_chunk;                      // (near box, first point) per store workgroup
    StoreLayout SL{0, (ifpt || ifptt) ? 1 : 0, (ifst || ifstt) ? 1 : 0, ifsl ? 1 : 0, ifdl ? 1 : 0};
    SL.W = (SL.ifsl + SL.ifdl) * 3 * (3 * SL.fd + 6 * SL.fs);
    int64_t store_words = 0;
    std::shared_ptr<NearStore> store;
    int icomp = iter ? it->icomp : 1;
    if (iter) {
        double refw = 0;
        int nl = ifsl + ifdl;
        int64_t nslots = 0;
        for (size_t q = 0; q < PL.nf_boxes.size(); q++) {
            int b = PL.nf_boxes[q];
            int ntri = 0;
            for (int k = PL.nf_start[q]; k < PL.nf_start[q + 1]; k++) ntri += T.src_count[PL.nf_items[k]];
            int npt = (src_eval ? T.src_count[b] : 0) + T.tgt_count[b];
            nf_ntri.push_back(ntri);
            nf_sbase.push_back(store_words);
            nf_pstart.push_back(nf_pstart.back() + npt);
            for (int p0 = 0; p0 < npt; p0 += ST_CHUNK) {
                nf_chunk.push_back((int)q);
                nf_chunk.push_back(p0);
            }
            store_words += (int64_t)npt * ntri * SL.W;
            nslots += (int64_t)npt * ntri;
            refw += (double)nl * ntri *
                    ((src_eval ? T.src_count[b] : 0) * 3.0 * (3 * ifpt + 9 * ifst) +
                     T.tgt_count[b] * 3.0 * (3 * ifptt + 9 * ifstt));
        }
        g_stats[14] = refw;
        g_stats[15] = (double)store_words;
        int flags = flags0;
        if (icomp == 4) {
            g_times[0] = now_ms() - t0;
            g_times[11] = now_ms() - t_start;
            return 0;
        }
        // the store registry is shared by all threads (under g_mu); a call
        // holds its store by shared_ptr until it returns
        std::lock_guard<std::mutex> lk(g_mu);
        if (icomp == 3) {
            // only a store built on these coordinates is replayed
            store = kept;
            if (store && !(store->n == n && store->nt == nt && store->iprec == iprec && store->flags == flags &&
                           store->nslots == nslots && store->nboxes == PL.nf_boxes.size() &&
                           store->nitems == PL.nf_items.size()))
                store = nullptr;
            if (!store) {
                icomp = 1;
                it->status = 64;
            }
        }
        if (icomp == 2 || icomp == 5) {
            if (it->lwsave < ITER_HANDLE_WORDS || !it->wsave) {
                icomp = icomp == 5 ? 6 : 1;          // no room for a handle: compute directly
            } else {
                if (std::shared_ptr<NearStore> old = find_store(it->wsave, it->lwsave)) {
                    for (auto e = g_stores.begin(); e != g_stores.end(); ++e)
                        if (e->second == old) {
                            g_stores.erase(e);
                            break;
                        }
                }
                size_t freeb = 0, totalb = 0;
                bool fits = hipMemGetInfo(&freeb, &totalb) == hipSuccess &&
                            (size_t)store_words * 8 + ((size_t)1 << 30) < freeb;
                if (!fits) {
                    icomp = icomp == 5 ? 6 : 1;
                } else {
                    auto ns = std::make_shared<NearStore>();
                    ns->data.ensure((size_t)std::max<int64_t>(store_words, 1) * 8);
                    ns->words = store_words;
                    ns->n = n;
                    ns->nt = nt;
                    ns->iprec = iprec;
                    ns->flags = flags;
                    ns->nslots = nslots;
                    ns->nboxes = PL.nf_boxes.size();
                    ns->nitems = PL.nf_items.size();
                    ns->xs.assign(W.hsrc.begin(), W.hsrc.begin() + 3 * (size_t)n);
                    ns->xt.assign(W.htgt.begin(), W.htgt.begin() + 3 * (size_t)nt);
                    ns->tree = std::make_unique<Tree>(T);
                    ns->plan = std::make_unique<Plan>(PL);
                    long id = g_next_store++;
                    store = ns;
                    g_stores[id] = std::move(ns);
                    it->wsave[0] = ITER_MAGIC;
                    it->wsave[1] = (double)id;
                    it->wsave[2] = n;
                    it->wsave[3] = nt;
                }
            }
        }
    }
    if (iter) it->store = store;
    // icomp 5 and its no-store fallback (6) skip the far field
    bool near_only = iter && (icomp == 5 || icomp == 6);
    auto &nf_boxes = PL.nf_boxes;

    // half space: integrals of the image near field per near box (units: 3
    // unit densities when storing, else the caller's densities) and, for
    // icomp 1, the per-pair results' bases
    std::vector<int64_t> h_tb(1, 0), h_tbase(1, 0);
    int h_units = (icomp == 2 || icomp == 5) ? 3 : 1;
    if (half && !direct_only) {
        int nl = ifsl + ifdl;
        for (size_t q = 0; q < PL.nf_boxes.size(); q++) {
            int64_t np_q = T.tgt_count[PL.nf_boxes[q]];
            h_tb.push_back(h_tb.back() + np_q * nf_ntri[q] * nl * h_units);
            h_tbase.push_back(h_tbase.back() + np_q * nf_ntri[q] * nl * 9);
        }
    }

    // ---- upload plan
    Packer pk;
    PlanOffsets po;
    if (split) {
        pack_near(pk, T, PL, po);                    // the far field gets its own buffers once its lists exist
    } else {
        pack_plan(pk, T, PL, po);
    }
    // no store, no half space, a layer: the near field is integrated (k_near)
    if (!direct_only && !half && !store && (ifsl || ifdl)) {
        near_tasks(T, PL, src_eval, W.near_waves);
        pack_near_tasks(pk, W.near_waves, po);
    }
    const size_t o_iz = po.iz, o_izt = po.izt, o_ss = po.ss, o_sc = po.sc, o_ts = po.ts, o_tc = po.tc;
    const size_t o_nfb = po.nfb, o_nfs = po.nfs, o_nfi = po.nfi;
    size_t o_sbase = pk.add(nf_sbase), o_ntri = pk.add(nf_ntri), o_pst = pk.add(nf_pstart);
    size_t o_nfc = pk.add(nf_chunk);
    size_t o_htb = pk.add(h_tb), o_htbase = pk.add(h_tbase);
    W.plan.ensure(pk.size);
    W.stage.ensure(pk.size);
    pk.pack(W.stage.p);
    double t1 = now_ms();
    g_times[0] = t1 - t0;
    g_times[13] = t1 - t_tree;
    // phase k runs between events ev[2k] and ev[2k+1] on its stream
    bool ran[NPHASE] = {};
    auto ev_begin = [&](int k, hipStream_t st) { HIPOK(hipEventRecord(W.ev[2 * k], st)); };
    auto ev_end = [&](int k, hipStream_t st) {
        HIPOK(hipEventRecord(W.ev[2 * k + 1], st));
        ran[k] = true;
    };
    ev_begin(1, stream);
    HIPOK(hipMemcpyAsync(W.plan.p, W.stage.p, pk.size, hipMemcpyHostToDevice, stream));
    char *P = W.plan.get<char>();
    auto I = [&](size_t off) { return (const int *)(P + off); };
    auto D = [&](size_t off) { return (const double *)(P + off); };

    // ---- device buffers
    int np = n + nt;
    W.pts.ensure(3 * (size_t)np * 8);
    W.rec.ensure((size_t)n * NF_REC * 8);
    W.inp.ensure((size_t)n * 18 * 8);
    W.nf.ensure((size_t)np * 9 * 8);
    double *tri_s = W.inp.get<double>(), *nrm_s = tri_s + 9 * (size_t)n, *ssl_s = nrm_s + 3 * (size_t)n,
           *sdl_s = ssl_s + 3 * (size_t)n;
    hipLaunchKernelGGL(k_gather, dim3((np + 255) / 256), dim3(256), 0, stream, n, nt, I(o_iz), I(o_izt),
                       d_tri, d_nrm, d_src, ifsl, d_ssl, ifdl, d_sdl, d_tgt, tri_s, nrm_s, ssl_s, sdl_s,
                       W.pts.get<double>(), W.rec.get<double>());
    HIPOK(hipGetLastError());
    HIPOK(hipMemsetAsync(W.nf.p, 0, (size_t)np * 9 * 8, stream));
    // several density sets: all of them in tree order, [layer][set][triangle][3]
    const int nrhs = it ? it->nrhs : 1;
    double *dm0 = nullptr, *dm1 = nullptr;
    if (nrhs > 1) {
        W.dmulti.ensure((size_t)2 * nrhs * n * 3 * 8);
        dm0 = W.dmulti.get<double>();
        dm1 = dm0 + (size_t)nrhs * n * 3;
        for (int r = 0; r < nrhs; r++)
            hipLaunchKernelGGL(k_gather_dens, dim3((n + 255) / 256), dim3(256), 0, stream, n, I(o_iz), ifsl,
                               ifsl ? d_ssl + (size_t)r * n * 3 : nullptr, ifdl, ifdl ? d_sdl + (size_t)r * n * 3 : nullptr,
                               dm0 + (size_t)r * n * 3, dm1 + (size_t)r * n * 3);
        HIPOK(hipGetLastError());
        W.nfm.ensure((size_t)nrhs * np * 9 * 8);
        HIPOK(hipMemsetAsync(W.nfm.p, 0, (size_t)nrhs * np * 9 * 8, stream));
    }
    ev_end(1, stream);

    // ---- near field on its own stream, overlapping the far field
    // ELFMM_SERIAL_NEAR=1 (read at every apply) runs the near field on the
    // caller's stream ahead of the far field: no overlap, so the per-phase
    // times are those of each kernel alone
    const char *sne = std::getenv("ELFMM_SERIAL_NEAR");
    bool serial_near = sne && sne[0] == '1';
    hipStream_t ns = serial_near ? stream : W.near_stream;
    // replay of the stored near field for this store layout (layers present,
    // fields stored); with SL.W == 0 nothing is stored and the near field
    // stays zero
    auto run_replay = [&](hipStream_t rs) -> hipError_t {
        if (!(SL.W > 0 && !nf_chunk.empty())) return hipSuccess;
        const double *d0 = nrhs > 1 ? (SL.ifsl ? dm0 : dm1) : (SL.ifsl ? ssl_s : sdl_s), *d1 = nrhs > 1 ? dm1 : sdl_s;
        double *out = nrhs > 1 ? W.nfm.get<double>() : W.nf.get<double>();
        size_t dstr = (size_t)n * 3, nstr = (size_t)np * 9;
        // One set beside its far field: a few workgroups per CU, each taking
        // every grid-th task, which leaves registers to the far field; launched
        // whole, the replay holds every CU and P2M, half a CU's registers a
        // workgroup, waits for its end. By the bytes to read, at order 26 one per
        // CU up to 16 GB (15.1 GB of both layers' displacements, 46,080 triangles:
        // 3.71 ms a product, 4.04 with three, 4.24 whole; 9.7 GB of both layers
        // with strain, 11,520 triangles: 2.20, 2.40, 2.46) and three above, where
        // one reads too slowly (21 GB: 6.22 ms, 6.90 with one, 6.34 whole; 109 GB:
        // 27.6, 39.3, 27.4; between 16 and 21 GB not measured). Two at order 14
        // and below, whose far field is short (8 GB: 2.93, 3.37 with one, 3.14
        // whole; 14.6 GB: 3.53, 3.62, 3.93; 44 GB: 8.81, 9.51, 8.62). Whole:
        // order 39, where a workgroup of P2M takes
        // a whole CU (2.15, limited 2.31), several sets, whose far fields
        // outweigh the replay (16 sets of 32,000 triangles: 16.0, limited
        // 18.4), and no far field.
        const bool beside = nrhs == 1 && oc && !near_only && T.nlev >= 2 && p <= 30;
        const int per_cu = !beside ? 0 : p <= 14 ? 2 : store_words <= 2000000000 ? 1 : 3;
        auto run = [&](auto rk, int rb) {
            int ntask = (int)nf_chunk.size() / 2 * (ST_CHUNK / replay_pts(SL.ifsl + SL.ifdl, SL.fd, SL.fs, rb));
            for (int r0 = 0; r0 < nrhs; r0 += rb)
                hipLaunchKernelGGL(rk, dim3(per_cu ? std::min(ntask, per_cu * ds.cus) : ntask), dim3(NF_THREADS), 0, rs, n, src_eval, I(o_nfb), I(o_nfs),
                                   I(o_nfi), I(o_ss), I(o_sc), I(o_ts), (const int64_t *)(P + o_sbase), I(o_ntri),
                                   I(o_pst), I(o_nfc), ntask, d0 + r0 * dstr, d1 + r0 * dstr, dstr, std::min(rb, nrhs - r0),
                                   store->data.get<double>(), out + r0 * nstr, nstr);
        };
        auto layers = [&](auto nl) {
            constexpr int NL = decltype(nl)::value, RB = NL == 2 ? 4 : 8;   // sets per pass over the store
            if (nrhs > 1)
                SL.fd && SL.fs ? run(k_near_replay<NL, true, true, RB>, RB)
                               : SL.fd ? run(k_near_replay<NL, true, false, RB>, RB) : run(k_near_replay<NL, false, true, RB>, RB);
            else
                SL.fd && SL.fs ? run(k_near_replay<NL, true, true, 1>, 1)
                               : SL.fd ? run(k_near_replay<NL, true, false, 1>, 1) : run(k_near_replay<NL, false, true, 1>, 1);
        };
        SL.ifsl + SL.ifdl == 2 ? layers(std::integral_constant<int, 2>{}) : layers(std::integral_constant<int, 1>{});
        return hipGetLastError();
    };
    if (nrhs > 1 && !(store && icomp == 3)) return it->status == 64 ? 64 : 16;   // several sets: replays only
    HIPOK(hipEventRecord(W.ev_fork, stream));
    HIPOK(hipStreamWaitEvent(ns, W.ev_fork, 0));
    ev_begin(9, ns);
    if (direct_only) {
        int npe = (src_eval ? n : 0) + nt;
        int per = NF_THREADS / 64;
        if (npe)
            hipLaunchKernelGGL(k_direct, dim3((npe + per - 1) / per), dim3(NF_THREADS), 0, ns, n, npe,
                               src_eval ? n : 0, W.pts.get<double>(), W.rec.get<double>(), rlam, rmu, c1, ifsl,
                               ifdl, W.nf.get<double>());
    } else if (half) {
        int nqb = (int)nf_boxes.size(), nl = ifsl + ifdl;
        if (!(g_half_parts.load() & 1)) nqb = 0;
        HalfNearArgs ha{(const int64_t *)(P + o_htb), nqb, I(o_nfb), I(o_nfs), I(o_nfi), I(o_ss), I(o_sc),
                        I(o_ts), I(o_ntri), nullptr, W.pts.get<double>(), tri_s, nrm_s, ssl_s, sdl_s,
                        n, ifsl, ifdl, SL.fd, SL.fs, h_units, 0, rlam, rmu};
        int64_t ntask = h_tb.back();
        if (nqb && nl && (SL.fd || SL.fs) && ntask > 0) {
            W.hq.ensure(adap_stack_bytes(ntask));
            if (store && (icomp == 2 || icomp == 5)) {
                ha.sbase = (const int64_t *)(P + o_sbase);
                ha.W = SL.W;
                HIPOK(launch_hnear(ha, ntask, W.hq.p, store->data.get<double>(), ns));
                HIPOK(run_replay(ns));
            } else if (store && icomp == 3) {
                HIPOK(run_replay(ns));
            } else {
                W.htmp.ensure((size_t)h_tbase.back() * 8);
                ha.sbase = (const int64_t *)(P + o_htbase);
                ha.W = 9 * nl;
                HIPOK(launch_hnear(ha, ntask, W.hq.p, W.htmp.get<double>(), ns));
                HIPOK(launch_hnear_sum(n, I(o_nfb), I(o_ts), (const int64_t *)(P + o_htbase), I(o_ntri), I(o_pst),
                                       nqb, nf_pstart.back(), nl, W.htmp.get<double>(), W.nf.get<double>(), ns));
            }
        }
    } else if (!nf_boxes.empty() && store && (icomp == 2 || icomp == 5)) {
        hipLaunchKernelGGL(k_near_store, dim3(nf_chunk.size() / 2), dim3(NF_THREADS), 0, ns, n, src_eval,
                           I(o_nfb), I(o_nfs), I(o_nfi), I(o_ss), I(o_sc), I(o_ts), I(o_tc),
                           (const int64_t *)(P + o_sbase), I(o_ntri), I(o_nfc), W.pts.get<double>(),
                           W.rec.get<double>(), ssl_s, sdl_s, rlam, rmu, c1, SL, store->data.get<double>(),
                           W.nf.get<double>());
    } else if (!nf_boxes.empty() && store && icomp == 3) {
        HIPOK(run_replay(ns));
    } else if (po.near_waves) {                      // no layer: the near field stays zero
        hipLaunchKernelGGL(near_kernel(ifsl, ifdl, ifst || ifstt), dim3(po.near_waves), dim3(64), 0, ns, n,
                           src_eval, I(o_nfb), I(o_nfs), I(o_nfi), I(o_ss), I(o_sc), I(o_ts), I(o_tc), I(po.nfw),
                           W.pts.get<double>(), W.rec.get<double>(), rlam, rmu, c1, W.nf.get<double>());
    }
    HIPOK(hipGetLastError());
    ev_end(9, ns);
    HIPOK(hipEventRecord(W.ev_join, ns));

    // split plan: the far-field lists, built while the near field runs; in
    // parts while the far field runs too when no other apply is in flight
    const bool usefar = oc && T.nlev >= 2 && !near_only && !(half && !(g_half_parts.load() & 2));
    const bool parts = split && usefar && inflight.others == 0;
    const char *PF = P;
    double tf0 = now_ms();
    auto planned = [&]() {
        plan_lk.unlock();
        for (int i = 0; i < 16; i++) g_stats[i] = PL.stats[i];
        double tf1 = now_ms();
        g_times[13] += tf1 - tf0;
        g_times[0] += tf1 - tf0;
    };
    if (split && !usefar) {
        build_plan_up(T, &oc->ops, PL, false);       // its counts (no far field below level 2)
        planned();
    } else if (split && !parts) {
        build_plan_far(T, n, &oc->ops, src_eval, NRHS, PL, false);
        Packer pkf;
        pack_up(pkf, T, PL, po);
        pack_m2l(pkf, PL, po);
        pack_eval(pkf, PL, po);
        W.part[0].ensure(pkf.size);
        W.part_stage[0].ensure(pkf.size);
        pkf.pack(W.part_stage[0].p);
        HIPOK(hipMemcpyAsync(W.part[0].p, W.part_stage[0].p, pkf.size, hipMemcpyHostToDevice, stream));
        PF = W.part[0].get<char>();
        planned();
    }

    // far fields of different applies run in order (see g_order_mu)
    int dev = 0;
    HIPOK(hipGetDevice(&dev));
    std::unique_lock<std::mutex> order(g_order_mu);
    if (dev < ORDER_DEVICES && g_order_tail[dev]) HIPOK(hipStreamWaitEvent(stream, g_order_tail[dev], 0));

    // ---- far field (and assembly) of each density set
    if (nrhs > 1) {
        // several sets: their far fields SET_LANES at a time on streams of
        // their own (one set's far field leaves much of the device idle),
        // each lane with its own scratch; a lane assembles its set once the
        // near field of all sets is done
        W.init_set_lanes();
        int L = std::min(nrhs, SET_LANES);
        size_t n_nodes, n_exps, n_lap;
        far_scratch(iprec, n, np, nb, p, n_nodes, n_exps, n_lap);
        HIPOK(hipEventRecord(W.ev_fork, stream));
        for (int j = 0; j < L; j++) {
            HIPOK(hipStreamWaitEvent(W.set_stream[j], W.ev_fork, 0));
            if (usefar) {
                W.set_exps[j].ensure(n_exps * 8);
                W.set_lap[j].ensure(n_lap * 8);
                W.set_nodes[j].ensure(n_nodes * 8);
            }
        }
        for (int r = 0; r < nrhs; r++) {
            int j = r % L;
            hipStream_t sj = W.set_stream[j];
            const double *ssl_r = dm0 + (size_t)r * n * 3, *sdl_r = dm1 + (size_t)r * n * 3;
            double *lap_j = usefar ? W.set_lap[j].get<double>() : nullptr;
            if (usefar) {
                FarLaunch fl{&ds, oc, &PL, &po, P, PF, PF, PF, iprec, n, nb, tri_s, nrm_s, ssl_r, sdl_r, ifsl, ifdl,
                             muF, c1F, c2F, half ? -1.0 : 1.0, W.pts.get<double>(), W.set_nodes[j].get<double>(),
                             W.set_exps[j].get<double>(), lap_j};
                Lane ln;
                ln.stream = sj;
                enqueue_far(fl, (size_t)np, ln, [](int, bool) {});
            }
            if (r < L) HIPOK(hipStreamWaitEvent(sj, W.ev_join, 0));
            hipLaunchKernelGGL(k_assemble, dim3((np + 255) / 256), dim3(256), 0, sj, n, nt, src_eval, I(o_iz),
                               I(o_izt), W.pts.get<double>(), lap_j, W.nfm.get<double>() + (size_t)r * np * 9,
                               c1F, usefar ? 1 : 0, (near_only && !half) ? 1 : 0, half ? 1 : 0,
                               ifpt, ifpt ? d_pt + (size_t)r * n * 3 : nullptr, ifst,
                               ifst ? d_st + (size_t)r * n * 9 : nullptr, ifptt,
                               ifptt ? d_ptt + (size_t)r * nt * 3 : nullptr, ifstt,
                               ifstt ? d_stt + (size_t)r * nt * 9 : nullptr);
            HIPOK(hipGetLastError());
        }
        for (int j = 0; j < L; j++) {
            HIPOK(hipEventRecord(W.set_ev[j], W.set_stream[j]));
            HIPOK(hipStreamWaitEvent(stream, W.set_ev[j], 0));
        }
        HIPOK(hipEventRecord(W.ev_done, stream));
        if (dev < ORDER_DEVICES) g_order_tail[dev] = W.ev_done;
        order.unlock();
        HIPOK(hipStreamSynchronize(stream));
        g_times[11] = now_ms() - t_start;
        return 0;
    }
    for (int r = 0; r < nrhs; r++) {
        const double *ssl_r = nrhs > 1 ? dm0 + (size_t)r * n * 3 : ssl_s;
        const double *sdl_r = nrhs > 1 ? dm1 + (size_t)r * n * 3 : sdl_s;
        if (usefar) {
            size_t n_nodes, n_exps, n_lap;
            far_scratch(iprec, n, np, nb, p, n_nodes, n_exps, n_lap);
            W.exps.ensure(n_exps * 8);
            W.lap.ensure(n_lap * 8);
            W.nodes.ensure(n_nodes * 8);
            FarLaunch fl{&ds, oc, &PL, &po, P, PF, PF, PF, iprec, n, nb, tri_s, nrm_s, ssl_r, sdl_r, ifsl, ifdl,
                         muF, c1F, c2F, half ? -1.0 : 1.0, W.pts.get<double>(), W.nodes.get<double>(),
                         W.exps.get<double>(), W.lap.get<double>()};
            Lane ln;
            ln.stream = stream;
            auto mark = [&](int k, bool begin) {
                if (begin)
                    ev_begin(k, stream);
                else
                    ev_end(k, stream);
            };
            if (parts) {
                run_far_parts(fl, T, PL, po, src_eval, (size_t)np, W, ln, mark);
                planned();
            } else {
                enqueue_far(fl, (size_t)np, ln, mark);
            }
        }
        if (r + 1 == nrhs) {
            HIPOK(hipEventRecord(W.ev_done, stream));
            if (dev < ORDER_DEVICES) g_order_tail[dev] = W.ev_done;
            order.unlock();
        }
        if (r == 0) HIPOK(hipStreamWaitEvent(stream, W.ev_join, 0));
        ev_begin(10, stream);
        hipLaunchKernelGGL(k_assemble, dim3((np + 255) / 256), dim3(256), 0, stream, n, nt, src_eval, I(o_iz),
                           I(o_izt), W.pts.get<double>(), usefar ? W.lap.get<double>() : nullptr,
                           nrhs > 1 ? W.nfm.get<double>() + (size_t)r * np * 9 : W.nf.get<double>(),
                           c1F, usefar ? 1 : 0, (near_only && !half) ? 1 : 0, half ? 1 : 0,
                           ifpt, ifpt ? d_pt + (size_t)r * n * 3 : nullptr, ifst, ifst ? d_st + (size_t)r * n * 9 : nullptr,
                           ifptt, ifptt ? d_ptt + (size_t)r * nt * 3 : nullptr,
                           ifstt, ifstt ? d_stt + (size_t)r * nt * 9 : nullptr);
        HIPOK(hipGetLastError());
        ev_end(10, stream);
    }
    HIPOK(hipStreamSynchronize(stream));
    for (int k = 1; k <= 10; k++) {
        float ms = 0.0f;
        if (ran[k] && hipEventElapsedTime(&ms, W.ev[2 * k], W.ev[2 * k + 1]) == hipSuccess) g_times[k] = ms;
    }
    g_times[11] = now_ms() - t_start;
    return 0;
}

// Workgroups of the point near field (k_pnear): (near box, first (point,
// lane) pair, lanes per point). Lanes per point: at least as many as give
// the device PN_WAVES waves (a small call has few points: at 3,704 points and
// one lane each 58 waves would run 256 CUs), then per box up to four times
// that, the one that leaves the fewest lanes of its last wave idle (195
// points fill 3.05 waves at one lane each, 12.2 at four).
std::vector<int> point_chunks(const Tree &T, const Plan &PL, int src_eval)
{
    constexpr int64_t PN_WAVES = 4096;               // 256 CUs x 4 SIMDs x 4
    auto npts = [&](int b) { return (src_eval ? T.src_count[b] : 0) + T.tgt_count[b]; };
    int64_t total = 0;
    for (int b : PL.nf_boxes) total += npts(b);
    int low = 1;
    while (low < 64 && total * low < PN_WAVES * 64) low *= 2;
    std::vector<int> chunks;
    for (size_t q = 0; q < PL.nf_boxes.size(); q++) {
        int64_t np = npts(PL.nf_boxes[q]);
        int best = low;
        auto waves = [&](int s) { return (double)((np * s + 63) / 64) / s; };   // lane-time of the box
        for (int s = 2 * low; s <= std::min(64, 4 * low); s *= 2)
            if (waves(s) < 0.95 * waves(best)) best = s;
        for (int64_t l0 = 0; l0 < np * best; l0 += PN_THREADS) {
            chunks.push_back((int)q);
            chunks.push_back((int)l0);
            chunks.push_back(best);
        }
    }
    return chunks;
}

// The point-source apply (elfmm3dparttarg, src/elfmm3dpart.f:104-500):
// the octree of the points with the particle FMM's leaf size, the far
// field of the triangle apply with one node per point (k_pgather), the
// point near field beside it (k_pnear) and the same assembly. direct: one
// box holding every point, so the near field is the whole O(N^2) sum
// without self pairs (el3dpartdirecttarg, :506-712).
int parttarg_dev(int iprec, double rlam, double rmu, int n, const double *d_src, int ifsl, const double *d_ssl,
                 int ifdl, const double *d_sdl, const double *d_sdv, int ifpt, double *d_pt, int ifst, double *d_st,
                 int nt, const double *d_tgt, int ifptt, double *d_ptt, int ifstt, double *d_stt, hipStream_t stream,
                 bool direct)
{
    for (int i = 0; i < 16; i++) g_times[i] = 0;
    double t_start = now_ms();
    if (n < 1) return 0;
    if (!direct && (iprec > 3 || iprec < -2)) return 16;
    InFlight inflight;
    DeviceState *dsp;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        dsp = &device_state();
    }
    DeviceState &ds = *dsp;
    if (!g_ws) g_ws = new Workspace();
    Workspace &W = *g_ws;
    W.init_streams();
    int src_eval = (ifpt || ifst) ? 1 : 0;
    if (!(ifptt || ifstt)) nt = 0;
    double c1 = (rlam + rmu) / (rlam + 2 * rmu), c2 = rmu / (rlam + 2 * rmu);
    // octree on the device unless another apply is in flight or the points
    // are few (as the triangle apply); the one-box tree of the direct sum on the host
    const char *ht_env = std::getenv("ELFMM_HOST_TREE");
    bool host_tree = direct || (ht_env && ht_env[0] == '1');
    const int nbox = direct ? n + nt : iprec_nbox_part(iprec, n + nt);
    if (!host_tree && !(ht_env && ht_env[0] == '0')) host_tree = inflight.others > 0 || small_tree(n + nt, nbox);

    std::unique_lock<std::mutex> plan_lk(g_plan_mu);
    double t0 = now_ms();
    Tree &T = W.treeh;
    bool deep = host_tree;
    if (!host_tree) {
        if (!W.oct) W.oct.reset(new OctreeWork());
        HIPOK(build_tree_dev(d_src, n, d_tgt, nt, nbox, 0, T, *W.oct, stream, deep));
    }
    if (deep) {
        W.hsrc.resize(3 * (size_t)n);
        W.htgt.resize(3 * (size_t)std::max(nt, 1));
        HIPOK(hipMemcpyAsync(W.hsrc.data(), d_src, 3 * (size_t)n * 8, hipMemcpyDeviceToHost, stream));
        if (nt) HIPOK(hipMemcpyAsync(W.htgt.data(), d_tgt, 3 * (size_t)nt * 8, hipMemcpyDeviceToHost, stream));
        HIPOK(hipStreamSynchronize(stream));
        if (build_tree(W.hsrc.data(), n, W.htgt.data(), nt, nbox, 0, T)) return 4;
    }
    g_times[12] = now_ms() - t0;
    OpsCache *oc = nullptr;
    if (!direct) {
        std::lock_guard<std::mutex> lk(g_mu);
        oc = &operators_for(ds, iprec);
    }
    int p = oc ? oc->p : 0;
    Plan &PL = W.planh;
    plan_reset(PL);
    build_plan_near(T, src_eval, false, false, PL);
    const std::vector<int> chunks = point_chunks(T, PL, src_eval);
    Packer pk;
    PlanOffsets po;
    pack_near(pk, T, PL, po);
    size_t o_ch = pk.add(chunks);
    W.plan.ensure(pk.size);
    W.stage.ensure(pk.size);
    pk.pack(W.stage.p);
    HIPOK(hipMemcpyAsync(W.plan.p, W.stage.p, pk.size, hipMemcpyHostToDevice, stream));
    g_times[0] = now_ms() - t0;
    const char *P = W.plan.get<char>();
    auto I = [&](size_t off) { return (const int *)(P + off); };

    int np = n + nt, nb = T.nboxes;
    bool usefar = oc && T.nlev >= 2;
    size_t n_nodes = (size_t)n * NODE_STRIDE;
    if (usefar) {
        size_t f_nodes, f_exps, f_lap;
        far_scratch(iprec, n, np, nb, p, f_nodes, f_exps, f_lap);
        n_nodes = std::max(n_nodes, f_nodes);
        W.exps.ensure(f_exps * 8);
        W.lap.ensure(f_lap * 8);
    }
    W.nodes.ensure(n_nodes * 8);
    W.pts.ensure(3 * (size_t)np * 8);
    W.nf.ensure((size_t)np * 9 * 8);
    hipLaunchKernelGGL(k_pgather, dim3((np + 255) / 256), dim3(256), 0, stream, n, nt, I(po.iz), I(po.izt), d_src,
                       ifsl, d_ssl, ifdl, d_sdl, d_sdv, d_tgt, rmu, c1, c2, W.pts.get<double>(),
                       W.nodes.get<double>());
    HIPOK(hipGetLastError());
    HIPOK(launch_fill0(W.nf.get<double>(), (size_t)np * 9, stream));
    // near field on its own stream, beside the far field
    hipStream_t ns = W.near_stream;
    HIPOK(hipEventRecord(W.ev_fork, stream));
    HIPOK(hipStreamWaitEvent(ns, W.ev_fork, 0));
    bool strain = ifst || ifstt;
    auto pnear = ifsl && ifdl ? (strain ? k_pnear<true, true, true> : k_pnear<true, true, false>)
                 : ifdl       ? (strain ? k_pnear<false, true, true> : k_pnear<false, true, false>)
                              : (strain ? k_pnear<true, false, true> : k_pnear<true, false, false>);
    if (!chunks.empty() && (ifsl || ifdl))            // no layer: the near field stays zero
        hipLaunchKernelGGL(pnear, dim3(chunks.size() / 3), dim3(PN_THREADS), 0, ns, n, src_eval, I(po.nfb),
                           I(po.nfs), I(po.nfi), I(po.ss), I(po.sc), I(po.ts), I(po.tc), I(o_ch),
                           W.pts.get<double>(), W.nodes.get<double>(), c1, W.nf.get<double>());
    HIPOK(hipGetLastError());
    HIPOK(hipEventRecord(W.ev_join, ns));
    // far-field lists, as the triangle apply
    const bool parts = usefar && inflight.others == 0;
    const char *PF = P;
    double tf0 = now_ms();
    auto planned = [&]() {
        plan_lk.unlock();
        for (int i = 0; i < 16; i++) g_stats[i] = PL.stats[i];
        g_times[0] += now_ms() - tf0;
    };
    if (!usefar) {
        build_plan_up(T, oc ? &oc->ops : nullptr, PL, false);
        planned();
    } else if (!parts) {
        build_plan_far(T, n, &oc->ops, src_eval, NRHS, PL, false);
        Packer pkf;
        pack_up(pkf, T, PL, po);
        pack_m2l(pkf, PL, po);
        pack_eval(pkf, PL, po);
        W.part[0].ensure(pkf.size);
        W.part_stage[0].ensure(pkf.size);
        pkf.pack(W.part_stage[0].p);
        HIPOK(hipMemcpyAsync(W.part[0].p, W.part_stage[0].p, pkf.size, hipMemcpyHostToDevice, stream));
        PF = W.part[0].get<char>();
        planned();
    }
    // far fields of different applies run in order (see g_order_mu)
    int dev = 0;
    HIPOK(hipGetDevice(&dev));
    std::unique_lock<std::mutex> order(g_order_mu);
    if (dev < ORDER_DEVICES && g_order_tail[dev]) HIPOK(hipStreamWaitEvent(stream, g_order_tail[dev], 0));
    if (usefar) {
        FarLaunch fl{&ds, oc, &PL, &po, P, PF, PF, PF, iprec, n, nb, nullptr, nullptr, nullptr, nullptr, ifsl, ifdl,
                     rmu, c1, c2, 1.0, W.pts.get<double>(), W.nodes.get<double>(), W.exps.get<double>(),
                     W.lap.get<double>(), true};
        Lane ln;
        ln.stream = stream;
        auto mark = [](int, bool) {};
        if (parts) {
            run_far_parts(fl, T, PL, po, src_eval, (size_t)np, W, ln, mark);
            planned();
        } else {
            enqueue_far(fl, (size_t)np, ln, mark);
        }
    }
    HIPOK(hipEventRecord(W.ev_done, stream));
    if (dev < ORDER_DEVICES) g_order_tail[dev] = W.ev_done;
    order.unlock();
    HIPOK(hipStreamWaitEvent(stream, W.ev_join, 0));
    hipLaunchKernelGGL(k_assemble, dim3((np + 255) / 256), dim3(256), 0, stream, n, nt, src_eval, I(po.iz),
                       I(po.izt), W.pts.get<double>(), usefar ? W.lap.get<double>() : nullptr, W.nf.get<double>(),
                       c1, usefar ? 1 : 0, 0, 0, ifpt, d_pt, ifst, d_st, ifptt, d_ptt, ifstt, d_stt);
    HIPOK(hipGetLastError());
    HIPOK(hipStreamSynchronize(stream));
    g_times[11] = now_ms() - t_start;
    return 0;
}

namespace {
// Tables of the Mindlin far field for one precision flag, built once.
void mindlin_tables(OpsCache &oc, int iprec)
{
    if (oc.mind_ready) return;
    int p = oc.p;
    // operators of full order for the near offsets (the reference translates
    // them with l3dmplocquadu at order p, src/lfmm3droutsmindlin.f:347-361)
    int itab[343];
    for (int o = 0; o < 343; o++) {
        int k = o % 7 - 3;
        itab[o] = std::abs(k) <= 1 ? p : 0;
    }
    build_operators(p, itab, oc.mind_ops);
    oc.mind_m2l.ensure(oc.mind_ops.m2l.size() * 8);
    HIPOK(hipMemcpy(oc.mind_m2l.p, oc.mind_ops.m2l.data(), oc.mind_ops.m2l.size() * 8, hipMemcpyHostToDevice));
    const PwTable &T = pw_table(iprec);
    int nl = T.nlams;
    std::vector<int> foff(nl + 1, 0), poff(nl + 1, 0), nf(nl), np(nl);
    for (int i = 0; i < nl; i++) {
        nf[i] = pw_nfour(T, i);
        np[i] = pw_nphys(T, i);
        foff[i + 1] = foff[i] + nf[i];
        poff[i + 1] = poff[i] + np[i];
    }
    int ntp = poff[nl];
    std::vector<double> tab(4 * (size_t)ntp), rl(T.rlams, T.rlams + nl), wt(T.whts, T.whts + nl);
    std::vector<int> jnl(ntp);
    for (int i = 0; i < nl; i++)
        for (int j = 0; j < np[i]; j++) {
            double u = j * (2 * M_PI / np[i]);
            int k = poff[i] + j;
            tab[4 * k] = T.rlams[i];
            tab[4 * k + 1] = std::cos(u);
            tab[4 * k + 2] = std::sin(u);
            tab[4 * k + 3] = 1.0 / np[i];
            jnl[k] = i;
        }
    int nq = 2 * p, nquad = 2 * p;
    std::vector<double> ycst((p + 1) * (p + 1)), gl(2 * nquad), ytab((size_t)nquad * (p + 1) * (p + 1)),
        eph(2 * (size_t)(p + 1) * nquad), wl((size_t)nl * (p + 1));
    ylg(p, 1.0 / std::sqrt(3.0), ycst.data());
    gauss_legendre(nquad, gl.data(), gl.data() + nquad);
    for (int jj = 0; jj < nquad; jj++) ylg(p, gl[jj], ytab.data() + (size_t)jj * (p + 1) * (p + 1));
    for (int m = 0; m <= p; m++)
        for (int k = 0; k < nquad; k++) {
            double ph = 2 * M_PI * (k + 1) / nquad;
            eph[2 * ((size_t)m * nquad + k)] = std::cos(m * ph);
            eph[2 * ((size_t)m * nquad + k) + 1] = -std::sin(m * ph);
        }
    for (int i = 0; i < nl; i++)
        for (int l = 0; l <= p; l++) wl[(size_t)i * (p + 1) + l] = T.whts[i] * std::pow(T.rlams[i], (double)l);
    // one device buffer: doubles first, then ints
    std::vector<const std::vector<double> *> dv = {&ycst, &gl, &ytab, &eph, &wl, &tab, &rl, &wt};
    size_t off = 0;
    std::vector<size_t> doff;
    for (auto *v : dv) {
        doff.push_back(off);
        off += (v->size() * 8 + 255) & ~(size_t)255;
    }
    std::vector<const std::vector<int> *> iv = {&jnl, &foff, &poff, &nf, &np};
    std::vector<size_t> ioff;
    for (auto *v : iv) {
        ioff.push_back(off);
        off += (v->size() * 4 + 255) & ~(size_t)255;
    }
    oc.mind_tab.ensure(off);
    char *base = oc.mind_tab.get<char>();
    for (size_t i = 0; i < dv.size(); i++) HIPOK(hipMemcpy(base + doff[i], dv[i]->data(), dv[i]->size() * 8, hipMemcpyHostToDevice));
    for (size_t i = 0; i < iv.size(); i++) HIPOK(hipMemcpy(base + ioff[i], iv[i]->data(), iv[i]->size() * 4, hipMemcpyHostToDevice));
    for (int i = 0; i < 5; i++) oc.mind_off[i] = doff[i];
    MindPw &pw = oc.mind_pw;
    pw.nlams = nl;
    pw.nexptot = foff[nl];
    pw.nexptotp = ntp;
    pw.tab = (const double *)(base + doff[5]);
    pw.rlams = (const double *)(base + doff[6]);
    pw.whts = (const double *)(base + doff[7]);
    pw.jnl = (const int *)(base + ioff[0]);
    pw.foff = (const int *)(base + ioff[1]);
    pw.poff = (const int *)(base + ioff[2]);
    pw.nfour = (const int *)(base + ioff[3]);
    pw.nphys = (const int *)(base + ioff[4]);
    oc.mind_nq = nq;
    mind_set_lds_limits(mind_far_lds(ntp, foff[nl]));
    // proxy matrices of the near offsets
    int index[343];
    std::vector<int> offs = mind_proxy_offsets(index);
    int noff = (int)offs.size() / 3;
    oc.mind_pxo.ensure(offs.size() * 4);
    HIPOK(hipMemcpy(oc.mind_pxo.p, offs.data(), offs.size() * 4, hipMemcpyHostToDevice));
    oc.mind_px.ensure(mind_proxy_op_doubles(p, nq, noff) * 8);
    HIPOK(launch_mind_proxy_op(p, nq, nquad, noff, oc.mind_pxo.get<int>(), (const double *)(base + doff[1]),
                               (const double *)(base + doff[2]), (const double *)(base + doff[3]),
                               oc.mind_px.get<double>(), nullptr));
    HIPOK(hipStreamSynchronize(nullptr));
    oc.mind_ready = true;
}

}  // namespace

// The Mindlin far field's octree, task lists and their device copy for one
// geometry (mirrored centroids, targets, precision).
struct MindPlan {
    int iprec = 0, n = 0, nt = 0;
    Tree T;
    Plan PL;
    MindlinPlan MP;
    std::vector<std::vector<int>> bsc;        // per M2M launch: boxes whose B is rescaled after it
    DevBuf dev;                               // packed plan
    size_t o_iz, o_izt, o_cen, o_side, o_lev, o_ss, o_sc, o_p2m, o_l2t, o_l2tp, o_l2tw, o_src, o_slot, o_fb, o_fs,
        o_fi, o_px, o_parts;
    std::vector<size_t> o_bsc;
    std::vector<LaunchOff> off_m2m, off_l2l;
    LaunchOff off_m2l;
};

// Builds the plan (host octree on the mirrored centroids and the targets,
// lists, upload). Returns 4 if the octree cannot be built; *out stays null
// when the tree has fewer than three levels (no far field).
int build_mind_plan(OpsCache &oc, int iprec, int n, const double *d_src, int nt, const double *d_tgt,
                    hipStream_t stream, std::shared_ptr<MindPlan> &out)
{
    out.reset();
    std::vector<double> hs(3 * (size_t)n), ht(3 * (size_t)nt);
    HIPOK(hipMemcpyAsync(hs.data(), d_src, hs.size() * 8, hipMemcpyDeviceToHost, stream));
    HIPOK(hipMemcpyAsync(ht.data(), d_tgt, ht.size() * 8, hipMemcpyDeviceToHost, stream));
    HIPOK(hipStreamSynchronize(stream));
    for (int i = 0; i < n; i++) hs[3 * (size_t)i + 2] = -hs[3 * (size_t)i + 2];
    auto mp = std::make_shared<MindPlan>();
    MindPlan &M = *mp;
    M.iprec = iprec;
    M.n = n;
    M.nt = nt;
    Tree &T = M.T;
    if (build_tree(hs.data(), n, ht.data(), nt, iprec_nbox_iter(iprec, n + nt), 1, T)) return 4;
    if (T.nlev < 2) return 0;
    Plan &PL = M.PL;
    build_plan(T, n, &oc.ops, false, false, NRHS, PL, true);
    MindlinPlan &MP = M.MP;
    build_mindlin_plan(T, oc.mind_ops, MP);
    // far targets also take a box's own outgoing waves when it has sources
    {
        std::vector<int> fb, fs(1, 0), fi;
        size_t q = 0;
        for (int b = 0; b < T.nboxes; b++) {
            if (T.level[b] < 2 || !T.tgt_count[b]) continue;
            bool listed = q < MP.far_boxes.size() && MP.far_boxes[q] == b;
            if (!listed && !T.src_count[b]) continue;
            fb.push_back(b);
            if (listed) {
                fi.insert(fi.end(), MP.far_items.begin() + MP.far_start[q], MP.far_items.begin() + MP.far_start[q + 1]);
                q++;
            }
            fs.push_back((int)fi.size());
        }
        MP.far_boxes.swap(fb);
        MP.far_start.swap(fs);
        MP.far_items.swap(fi);
    }
    std::vector<int> levels(T.level.begin(), T.level.end());
    for (auto &g : PL.m2m_l) {
        int lev = g.dst.empty() ? -1 : T.level[g.dst[0]];
        M.bsc.push_back(lev >= 0 && lev < 64 ? MP.b_scale_boxes[lev] : std::vector<int>());
    }
    Packer pk;
    M.o_iz = pk.add(T.iz);
    M.o_izt = pk.add(T.iztarg);
    M.o_cen = pk.add(T.centers);
    M.o_side = pk.add(PL.sides);
    M.o_lev = pk.add(levels);
    M.o_ss = pk.add(T.src_start);
    M.o_sc = pk.add(T.src_count);
    M.o_p2m = pk.add(PL.p2m_boxes);
    M.o_l2t = pk.add(PL.l2t_boxes);
    M.o_l2tp = pk.add(PL.l2t_tpt);
    M.o_l2tw = pk.add(PL.l2t_wt);
    M.o_src = pk.add(MP.src_boxes);
    M.o_slot = pk.add(MP.pw_slot);
    M.o_fb = pk.add(MP.far_boxes);
    M.o_fs = pk.add(MP.far_start);
    M.o_fi = pk.add(MP.far_items);
    M.o_px = pk.add(MP.px_tasks);
    M.o_parts = pk.add(PL.p2m_parts);
    for (auto &v : M.bsc) M.o_bsc.push_back(pk.add(v));
    auto add_launch = [&](const GemmLaunch &g) {
        LaunchOff o;
        o.tiles = pk.add(g.tiles);
        o.src = pk.add(g.src);
        o.dst = pk.add(g.dst);
        o.sc = pk.add(g.scale);
        return o;
    };
    for (auto &g : PL.m2m_l) M.off_m2m.push_back(add_launch(g));
    for (auto &g : PL.l2l_l) M.off_l2l.push_back(add_launch(g));
    M.off_m2l = add_launch(MP.m2l);
    M.dev.ensure(pk.size);
    std::vector<char> stage(pk.size);
    pk.pack(stage.data());
    HIPOK(hipMemcpyAsync(M.dev.p, stage.data(), pk.size, hipMemcpyHostToDevice, stream));
    HIPOK(hipStreamSynchronize(stream));
    out = mp;
    return 0;
}

// Mindlin harmonic-image far field (lfmm3dmindlintriatarg,
// src/lfmm3dtriamindlin_iter_1.f:41, on the mirrored triangles with the
// original normals as dipole directions, src/elhfmm3dtria_iter.f:795-804),
// added to the target outputs: its own octree on the mirrored centroids
// and the targets (leaf size of the iter engine, half-space root rule), B,
// C1 and C2 as three right-hand sides of the Laplace translation kernels,
// the plane-wave and proxy-charge steps in elfmm_mindlin.hip. The near
// hooks of the reference engine are empty
// (src/lfmm3dtriamindlin_iter_1.f:1366-1368): the image near field covers
// lists 1, 3 and 4. With an iter store, the plan is built once and kept
// with the store for the later products of its geometry.
int mindlin_far_dev(int iprec, double rlam, double rmu, int n, const double *d_tri, const double *d_nrm,
                    const double *d_src, int ifsl, const double *d_ssl, int ifdl, const double *d_sdl, int nt,
                    const double *d_tgt, int ifptt, double *d_ptt, int ifstt, double *d_stt, hipStream_t stream,
                    NearStore *store, int lane, bool sync, bool assemble)
{
    if (g_ws) g_ws->mind[lane].plan = nullptr;      // set again when the far field runs
    if (n < 1 || nt < 1 || !(ifptt || ifstt) || !(ifsl || ifdl)) return 0;
    DeviceState *dsp;
    OpsCache *oc;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        dsp = &device_state();
        oc = &operators_for(*dsp, iprec);
        mindlin_tables(*oc, iprec);
    }
    if (oc->p > 39 || oc->mind_pw.nexptot > 544) return 16;
    if (!g_ws) g_ws = new Workspace();
    Workspace &W = *g_ws;
    MindScratch &S = W.mind[lane];
    int p = oc->p, nc = ncoef(p), np = n + nt;
    std::shared_ptr<MindPlan> mpl;
    if (store) {
        std::lock_guard<std::mutex> lk(store->mind_mu);
        if (store->mind && store->mind->iprec == iprec && store->mind->n == n && store->mind->nt == nt)
            mpl = store->mind;
    }
    if (!mpl) {
        int ier = build_mind_plan(*oc, iprec, n, d_src, nt, d_tgt, stream, mpl);
        if (ier) return ier;
        if (!mpl) return 0;
        if (store) {
            std::lock_guard<std::mutex> lk(store->mind_mu);
            store->mind = mpl;
        }
    }
    const MindPlan &M = *mpl;
    const Tree &T = M.T;
    const Plan &PL = M.PL;
    const MindlinPlan &MP = M.MP;
    const char *P = (const char *)M.dev.p;
    auto I = [&](size_t off) { return (const int *)(P + off); };
    auto D = [&](size_t off) { return (const double *)(P + off); };
    // inputs in tree order: mirrored triangles and centroids, original normals
    S.inp.ensure(((size_t)9 * n + 3 * (size_t)n + 18 * (size_t)n) * 8);
    double *trim = S.inp.get<double>(), *srcm = trim + 9 * (size_t)n, *tri_s = srcm + 3 * (size_t)n,
           *nrm_s = tri_s + 9 * (size_t)n, *ssl_s = nrm_s + 3 * (size_t)n, *sdl_s = ssl_s + 3 * (size_t)n;
    S.pts.ensure(3 * (size_t)np * 8);
    S.rec.ensure((size_t)n * NF_REC * 8);
    HIPOK(launch_mirror(3 * n, d_tri, trim, stream));
    HIPOK(launch_mirror(n, d_src, srcm, stream));
    hipLaunchKernelGGL(k_gather, dim3((np + 255) / 256), dim3(256), 0, stream, n, nt, I(M.o_iz), I(M.o_izt), trim,
                       d_nrm, srcm, ifsl, d_ssl, ifdl, d_sdl, d_tgt, tri_s, nrm_s, ssl_s, sdl_s, S.pts.get<double>(),
                       S.rec.get<double>());
    HIPOK(hipGetLastError());
    int nb = T.nboxes;
    S.exps.ensure((size_t)2 * nb * NRHS * nc * 8);
    double *mp = S.exps.get<double>(), *lo = mp + (size_t)nb * NRHS * nc;
    HIPOK(hipMemsetAsync(S.exps.p, 0, (size_t)2 * nb * NRHS * nc * 8, stream));
    S.pw.ensure((size_t)std::max(MP.npw, 1) * 3 * 2 * oc->mind_pw.nexptotp * 8);
    S.skel.ensure((size_t)std::max(MP.npw, 1) * 2 * oc->mind_nq * 4 * 8);
    char *tb = oc->mind_tab.get<char>();
    MindDev md;
    md.args = MindArgs{p, ifsl, ifdl, rlam, rmu, T.size, I(M.o_lev), I(M.o_ss), I(M.o_sc), D(M.o_cen), tri_s, nrm_s,
                       ssl_s, sdl_s, nc, mp, lo};
    md.pw = oc->mind_pw;
    md.slot = I(M.o_slot);
    md.ycst = (const double *)(tb + oc->mind_off[0]);
    md.nq = oc->mind_nq;
    md.pwo = S.pw.get<double>();
    md.skel = S.skel.get<double>();
    md.pxoffs = oc->mind_pxo.get<int>();
    md.pxop = oc->mind_px.get<double>();
    md.wl = (const double *)(tb + oc->mind_off[4]);
    S.gm.ensure(mind_p2m_scratch_bytes(p, (int)PL.p2m_boxes.size()));
    md.gmom = S.gm.get<double>();
    // upward pass
    const int nbx = (int)PL.p2m_boxes.size(), nown = nc / 2;
    if (nbx && iprec >= 0) {
        const int shape = p2t_shape(p, iprec >= 1 ? 12 : 6);
        if (shape < 0) HIPOK(hipErrorInvalidValue);
        // triangle moments (elfmm_moments.h), one layer at a time: 6 or 12 columns
        HIPOK(launch_fill0(S.gm.get<double>(), (size_t)2 * nbx * MindMoments::MCOLS * nown, stream));
        S.tcoef.ensure((size_t)48 * n * 8);
        for (int dl = 0; dl < 2; dl++) {
            if (!(dl ? ifdl : ifsl)) continue;
            hipLaunchKernelGGL(k_mind_tcoef, dim3((n + 255) / 256), dim3(256), 0, stream, n, dl, tri_s, nrm_s,
                               dl ? sdl_s : ssl_s, S.tcoef.get<double>());
            HIPOK(hipGetLastError());
            MindMoments mm;
            for (int c = 0; c < 16; c++) mm.col[c] = dl ? (c < 12 ? 6 + c : -1) : (c < 6 ? c : -1);
            mm.G = S.gm.get<double2>();
            auto run = [&](auto z) {
                using Z = decltype(z);
                hipLaunchKernelGGL((k_p2m_tri<Z, true>), dim3(PL.p2m_parts.size() / 3), dim3(Z::NT),
                                   (size_t)Z::lds(p) * 8, stream, p, I(M.o_p2m), I(M.o_parts), mm, D(M.o_cen),
                                   D(M.o_side), I(M.o_ss), I(M.o_sc), tri_s, S.tcoef.get<double>(), nc,
                                   (double *)nullptr);
                HIPOK(hipGetLastError());
            };
            shape == 0 ? run(P2TShape0{}) : shape == 1 ? run(P2TShape1{}) : shape == 2 ? run(P2TShape2{}) : run(P2TShape3{});
        }
        HIPOK(launch_mind_combine(md, I(M.o_p2m), nbx, stream));
    } else {
        HIPOK(launch_mind_p2m(md, I(M.o_p2m), nbx, stream));
    }
    Lane ln;
    ln.stream = stream;
    for (size_t k = 0; k < PL.m2m_l.size(); k++) {
        enqueue_trans(PL.m2m_l[k], M.off_m2m[k], P, oc->m2m, mp, mp, nc, ln);
        HIPOK(launch_mind_bscale(md, I(M.o_bsc[k]), (int)M.bsc[k].size(), stream));
    }
    // plane waves, proxy rings and B's remainder of every sourced box
    HIPOK(launch_mind_bmod(md, I(M.o_src), (int)MP.src_boxes.size(), stream));
    // list 2: near pairs (exact M2L of the remainder of B, and of C1, C2;
    // the proxies' field), far pairs (plane waves)
    enqueue_m2l_tiles(MP.m2l.tiles, M.off_m2l.tiles, M.off_m2l, P,
                      oc->mind_m2l.get<double>(), p, mp, lo, ln);
    HIPOK(launch_mind_proxy(md, I(M.o_px), (int)MP.px_tasks.size() / 3, I(M.off_m2l.src), I(M.off_m2l.dst), stream));
    HIPOK(launch_mind_far(md, I(M.o_fb), I(M.o_fs), I(M.o_fi), (int)MP.far_boxes.size(), stream));
    // downward pass and evaluation
    for (size_t k = 0; k < PL.l2l_l.size(); k++)
        enqueue_trans(PL.l2l_l[k], M.off_l2l[k], P, oc->l2l, lo, lo, nc, ln);
    S.lap.ensure((size_t)np * 40 * 8);
    HIPOK(hipMemsetAsync(S.lap.p, 0, (size_t)np * 40 * 8, stream));
    if (!PL.l2t_tpt.empty()) {
        int nwt = (int)PL.l2t_wt.size() / 3;
        int nsteps = ((p + 1) * (p + 2) / 2 + 1) / 2;
        hipLaunchKernelGGL(k_l2t, dim3((nwt + EB_WAVES - 1) / EB_WAVES), dim3(64 * EB_WAVES), 0, stream, p, nwt,
                           I(M.o_l2tw), I(M.o_l2tp), I(M.o_l2t), D(M.o_cen), D(M.o_side), S.pts.get<double>(), lo,
                           nc, oc->ft_loc.get<FieldTerm>(), nsteps, S.lap.get<double>());
        HIPOK(hipGetLastError());
    }
    S.plan = mpl;
    if (assemble)
        HIPOK(launch_mind_assemble(n, nt, I(M.o_izt), S.pts.get<double>(), S.lap.get<double>(), rmu, ifptt, d_ptt,
                                   ifstt, d_stt, stream));
    if (sync) HIPOK(hipStreamSynchronize(stream));
    return 0;
}

// The Mindlin fields of lane's last far field added to the outputs (after
// a mindlin_far_dev call with assemble = false on the same lane and stream).
void mindlin_assemble_dev(int lane, int n, int nt, double rmu, int ifptt, double *d_ptt, int ifstt, double *d_stt,
                          hipStream_t stream)
{
    MindScratch &S = g_ws->mind[lane];
    if (!S.plan) return;                             // no far field ran
    const char *P = (const char *)S.plan->dev.p;
    HIPOK(launch_mind_assemble(n, nt, (const int *)(P + S.plan->o_izt), S.pts.get<double>(), S.lap.get<double>(),
                               rmu, ifptt, d_ptt, ifstt, d_stt, stream));
}

// Half-space apply (elhfmm3dtriatargiter, src/elhfmm3dtria_iter.f:46-272):
// targets only. icomp 1-3: the anti-image far field and the image near field
// (one iter apply on the sources and the mirrored targets), then the
// Mindlin harmonic far field added; icomp 5: the image near field only
// (stored); icomp 4: plan only; icomp 0: outputs zero.
int htriatargiter_dev(int iprec, double rlam, double rmu, int n, const double *d_tri, const double *d_nrm,
                      const double *d_src, int ifsl, const double *d_ssl, int ifdl, const double *d_sdl, int nt,
                      const double *d_tgt, int ifptt, double *d_ptt, int ifstt, double *d_stt, hipStream_t stream,
                      IterCall &it)
{
    if (!(ifptt || ifstt) || nt < 1 || n < 1) return 0;
    if (it.icomp == 0 || it.icomp < 0 || it.icomp > 5) {
        if (ifptt) HIPOK(hipMemsetAsync(d_ptt, 0, 3 * (size_t)nt * 8, stream));
        if (ifstt) HIPOK(hipMemsetAsync(d_stt, 0, 9 * (size_t)nt * 8, stream));
        HIPOK(hipStreamSynchronize(stream));
        return 0;
    }
    it.half = 1;
    double t0 = now_ms();
    // a replay (icomp 3) of one set whose store holds its Mindlin plan: the
    // Mindlin far field runs on a stream of its own beside the anti-image
    // far field and the image near field, and its fields are added once
    // those have been written
    if (it.icomp == 3 && it.nrhs == 1 && (g_half_parts.load() & 4)) {
        std::shared_ptr<NearStore> st;
        {
            std::lock_guard<std::mutex> lk(g_mu);
            st = find_store(it.wsave, it.lwsave);
        }
        bool have_plan = false;
        if (st) {
            std::lock_guard<std::mutex> lk(st->mind_mu);
            have_plan = st->mind && st->mind->iprec == iprec && st->mind->n == n && st->mind->nt == nt;
        }
        if (have_plan) {
            if (!g_ws) g_ws = new Workspace();
            Workspace &W = *g_ws;
            W.init_streams();
            W.init_set_lanes();
            hipStream_t ms = W.set_stream[0];
            HIPOK(hipEventRecord(W.ev_fork, stream));
            HIPOK(hipStreamWaitEvent(ms, W.ev_fork, 0));
            HIPOK(hipEventRecord(W.ev_mind[0], ms));
            int ier = mindlin_far_dev(iprec, rlam, rmu, n, d_tri, d_nrm, d_src, ifsl, d_ssl, ifdl, d_sdl, nt, d_tgt,
                                      ifptt, d_ptt, ifstt, d_stt, ms, st.get(), 0, false, false);
            HIPOK(hipEventRecord(W.ev_mind[1], ms));
            if (!ier)
                ier = triatarg_dev(iprec, rlam, rmu, n, d_tri, d_nrm, d_src, ifsl, d_ssl, ifdl, d_sdl, 0, nullptr, 0,
                                   nullptr, nt, d_tgt, ifptt, d_ptt, ifstt, d_stt, stream, false, &it);
            // the anti-image apply has completed (it synchronizes its stream)
            if (!ier && it.status != 64) mindlin_assemble_dev(0, n, nt, rmu, ifptt, d_ptt, ifstt, d_stt, ms);
            HIPOK(hipStreamSynchronize(ms));
            if (!ier && it.status == 64)          // no store after all: the Mindlin fields of a fresh plan
                ier = mindlin_far_dev(iprec, rlam, rmu, n, d_tri, d_nrm, d_src, ifsl, d_ssl, ifdl, d_sdl, nt,
                                      d_tgt, ifptt, d_ptt, ifstt, d_stt, stream, nullptr, 0, true, true);
            double t2 = now_ms();
            float mms = 0.0f;
            if (hipEventElapsedTime(&mms, W.ev_mind[0], W.ev_mind[1]) == hipSuccess) g_times[14] = mms;
            g_times[15] = t2 - t0;
            return ier;
        }
    }
    int ier = triatarg_dev(iprec, rlam, rmu, n, d_tri, d_nrm, d_src, ifsl, d_ssl, ifdl, d_sdl, 0, nullptr, 0,
                           nullptr, nt, d_tgt, ifptt, d_ptt, ifstt, d_stt, stream, false, &it);
    if (ier || it.icomp == 4 || it.icomp == 5) return ier;
    double t1 = now_ms();
    if (g_half_parts.load() & 4) {
        // several sets: SET_LANES Mindlin far fields at a time, on streams
        // of their own with their own scratch
        Workspace &W = *g_ws;
        int L = it.nrhs > 1 ? std::min(it.nrhs, SET_LANES) : 0;
        if (L) {
            W.init_set_lanes();
            HIPOK(hipEventRecord(W.ev_fork, stream));
            for (int j = 0; j < L; j++) HIPOK(hipStreamWaitEvent(W.set_stream[j], W.ev_fork, 0));
        }
        for (int r = 0; r < it.nrhs && !ier; r++)
            ier = mindlin_far_dev(iprec, rlam, rmu, n, d_tri, d_nrm, d_src, ifsl,
                                  ifsl ? d_ssl + (size_t)r * n * 3 : nullptr, ifdl,
                                  ifdl ? d_sdl + (size_t)r * n * 3 : nullptr, nt, d_tgt, ifptt,
                                  ifptt ? d_ptt + (size_t)r * nt * 3 : nullptr, ifstt,
                                  ifstt ? d_stt + (size_t)r * nt * 9 : nullptr, L ? W.set_stream[r % L] : stream,
                                  it.store.get(), L ? r % L : 0, L == 0, true);
        for (int j = 0; j < L; j++) {
            HIPOK(hipEventRecord(W.set_ev[j], W.set_stream[j]));
            HIPOK(hipStreamWaitEvent(stream, W.set_ev[j], 0));
        }
        if (L) HIPOK(hipStreamSynchronize(stream));
    }
    double t2 = now_ms();
    g_times[14] = t2 - t1;
    g_times[15] = t2 - t0;
    return ier;
}

// Direct half-space sum (elh3dtriadirecttarg, src/elh3dtria.f:53): the
// free-space direct sum plus the adaptive image integral of every (point,
// triangle) pair with the caller's densities.
int hdirect_dev(double rlam, double rmu, int n, const double *d_tri, const double *d_nrm, const double *d_src,
                int ifsl, const double *d_ssl, int ifdl, const double *d_sdl, int ifpt, double *d_pt, int ifst,
                double *d_st, int nt, const double *d_tgt, int ifptt, double *d_ptt, int ifstt, double *d_stt,
                hipStream_t stream)
{
    int ier = triatarg_dev(0, rlam, rmu, n, d_tri, d_nrm, d_src, ifsl, d_ssl, ifdl, d_sdl, ifpt, d_pt, ifst, d_st,
                           nt, d_tgt, ifptt, d_ptt, ifstt, d_stt, stream, true);
    if (ier) return ier;
    if (!g_ws) g_ws = new Workspace();
    Workspace &W = *g_ws;
    auto part = [&](int np, const double *pts, int fp, double *op, int fs, double *os) {
        if (np < 1 || !(fp || fs)) return;
        W.hq.ensure(hdirect_scratch_bytes(np, n));
        HIPOK(launch_hdirect(np, pts, n, d_tri, d_nrm, d_ssl, d_sdl, ifsl, ifdl, fp, fs, rlam, rmu, W.hq.p, op, os,
                             stream));
        HIPOK(hipStreamSynchronize(stream));
    };
    part(n, d_src, ifpt, d_pt, ifst, d_st);
    part(nt, d_tgt, ifptt, d_ptt, ifstt, d_stt);
    return 0;
}


// ------------------------------------------------------------------------
// Batch of meshes: many independent free-space applies (elfmm3dtriatarg on
// each mesh) on geometries fixed at creation. Trees, task lists and device
// buffers are built once; an apply gathers the densities, runs every mesh's
// near and far field and scatters the outputs, as one graph replay (or as
// direct launches, when the tuner finds those faster). Meshes are spread
// over branches (stream pairs: far field, near field), largest planned work
// first onto the least loaded branch; meshes of one branch run in turn and
// share its scratch buffers.
// ------------------------------------------------------------------------
namespace {

constexpr int BATCH_MAX_WIDTH = 16;
constexpr int BATCH_FOREST = 100;                   // width argument of the forest schedule

struct BatchMesh {
    int n = 0, nt = 0;
    size_t off = 0, offt = 0;                        // first triangle, first target in the packed arrays
    Tree T;
    Plan PL;
    PlanOffsets po;
    DevBuf plan, inp, pts, rec;
    bool usefar = false;
    double cost = 0;                                 // planned work (flop-like units) for the schedule
    size_t n_nodes = 0, n_exps = 0, n_lap = 0;
};

struct BatchBranch {
    hipStream_t far = nullptr, near = nullptr;       // direct launches
    hipEvent_t ev_far = nullptr, ev_near = nullptr, ev_out = nullptr;
    DevBuf nodes, exps, lap, nf;
    std::vector<int> meshes;
};

// All meshes' octrees as one forest, planned and applied as one FMM (its
// task lists never cross from one tree to another).
struct BatchForest {
    Tree T;
    Plan PL;
    PlanOffsets po;
    DevBuf plan, inp, pts, rec, nf, nodes, exps, lap;
    bool usefar = false;
};

struct Batch {
    BatchForest forest;
    int dev = 0, iprec = 0;
    double rlam = 1, rmu = 1;
    int ifsl = 0, ifdl = 0, ifpt = 0, ifst = 0, ifptt = 0, ifstt = 0, src_eval = 0;
    size_t ntri = 0, ntgt = 0;
    DeviceState *ds = nullptr;
    OpsCache *oc = nullptr;
    std::vector<std::unique_ptr<BatchMesh>> mesh;
    DevBuf geo, dens, out;
    double *tri = nullptr, *nrm = nullptr, *src = nullptr, *tgt = nullptr;
    double *ssl = nullptr, *sdl = nullptr, *pt = nullptr, *st = nullptr, *ptt = nullptr, *stt = nullptr;
    BatchBranch br[BATCH_MAX_WIDTH];
    hipStream_t tstream = nullptr;                   // the tuner's stream
    hipEvent_t ev_start = nullptr, ev_t0 = nullptr, ev_t1 = nullptr;
    int width = 0, graph_mode = 1;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<double> tune;                        // (graph, width, ms) of each schedule tried
    std::mutex mu;
    ~Batch()
    {
        (void)hipDeviceSynchronize();
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        for (auto &b : br) {
            if (b.far) (void)hipStreamDestroy(b.far);
            if (b.near) (void)hipStreamDestroy(b.near);
            for (hipEvent_t e : {b.ev_far, b.ev_near, b.ev_out})
                if (e) (void)hipEventDestroy(e);
        }
        if (tstream) (void)hipStreamDestroy(tstream);
        for (hipEvent_t e : {ev_start, ev_t0, ev_t1})
            if (e) (void)hipEventDestroy(e);
    }
};

// Longest-processing-time assignment of the meshes to w branches, and the
// branches' scratch sized for their largest mesh.
void batch_schedule(Batch &B, int w)
{
    if (w == 0) return;                              // the forest has its own buffers
    std::vector<int> order(B.mesh.size());
    for (size_t i = 0; i < order.size(); i++) order[i] = (int)i;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return B.mesh[a]->cost > B.mesh[b]->cost; });
    std::vector<double> load(w, 0.0);
    for (int b = 0; b < BATCH_MAX_WIDTH; b++) B.br[b].meshes.clear();
    for (int m : order) {
        int b = (int)(std::min_element(load.begin(), load.end()) - load.begin());
        load[b] += B.mesh[m]->cost;
        B.br[b].meshes.push_back(m);
    }
    for (int b = 0; b < w; b++) {
        BatchBranch &R = B.br[b];
        size_t nn = 0, ne = 0, nl = 0, nf = 0;
        for (int m : R.meshes) {
            const BatchMesh &M = *B.mesh[m];
            nn = std::max(nn, M.n_nodes);
            ne = std::max(ne, M.n_exps);
            nl = std::max(nl, M.n_lap);
            nf = std::max(nf, (size_t)(M.n + M.nt) * 9);
        }
        R.nodes.ensure(nn * 8);
        R.exps.ensure(ne * 8);
        R.lap.ensure(nl * 8);
        R.nf.ensure(nf * 8);
    }
}

// What one apply of the batch runs on: a mesh (its plan, tree-order
// buffers and its branch's scratch) or the forest of all meshes.
struct BatchView {
    int n, nt, nb;
    size_t off, offt;                                // first triangle / target in the packed arrays
    const char *P;                                   // packed plan on the device
    const Plan *PL;
    const PlanOffsets *po;
    double *inp, *pts, *rec, *nf, *nodes, *exps, *lap;
    bool usefar;
};

// One apply on two lanes: f runs the gather, the far field and the
// assembly, q the near field between them.
void batch_enqueue_view(Batch &B, const BatchView &V, Lane &f, Lane &q)
{
    const char *P = V.P;
    auto I = [&](size_t off) { return (const int *)(P + off); };
    const int n = V.n, nt = V.nt, np = n + nt;
    const PlanOffsets &po = *V.po;
    double *tri_s = V.inp, *nrm_s = tri_s + 9 * (size_t)n, *ssl_s = nrm_s + 3 * (size_t)n, *sdl_s = ssl_s + 3 * (size_t)n;
    const double c1 = (B.rlam + B.rmu) / (B.rlam + 2 * B.rmu), c2 = B.rmu / (B.rlam + 2 * B.rmu);
    const double *none = nullptr;
    f.launch(k_gather, dim3((np + 255) / 256), dim3(256), 0, n, nt, I(po.iz), I(po.izt),
             (const double *)(B.tri + 9 * V.off), (const double *)(B.nrm + 3 * V.off),
             (const double *)(B.src + 3 * V.off), B.ifsl, B.ifsl ? (const double *)(B.ssl + 3 * V.off) : none,
             B.ifdl, B.ifdl ? (const double *)(B.sdl + 3 * V.off) : none,
             nt ? (const double *)(B.tgt + 3 * V.offt) : none, tri_s, nrm_s, ssl_s, sdl_s, V.pts, V.rec);
    f.fill0(V.nf, (size_t)np * 9);
    bool near = po.near_waves && (B.ifsl || B.ifdl);
    if (near) {
        q.after(f);
        q.launch(near_kernel(B.ifsl, B.ifdl, B.ifst || B.ifstt), dim3(po.near_waves), dim3(64), 0, n,
                 B.src_eval, I(po.nfb), I(po.nfs), I(po.nfi), I(po.ss), I(po.sc), I(po.ts), I(po.tc), I(po.nfw),
                 (const double *)V.pts, (const double *)V.rec, B.rlam, B.rmu, c1, V.nf);
    }
    if (V.usefar) {
        FarLaunch fl{B.ds, B.oc, V.PL, V.po, P, P, P, P, B.iprec, n, V.nb, tri_s, nrm_s, ssl_s, sdl_s, B.ifsl, B.ifdl,
                     B.rmu, c1, c2, 1.0, V.pts, V.nodes, V.exps, V.lap};
        enqueue_far(fl, (size_t)np, f, [](int, bool) {});
    }
    if (near) f.after(q);
    double *nul = nullptr;
    f.launch(k_assemble, dim3((np + 255) / 256), dim3(256), 0, n, nt, B.src_eval, I(po.iz), I(po.izt),
             (const double *)V.pts, V.usefar ? (const double *)V.lap : none, (const double *)V.nf, c1,
             V.usefar ? 1 : 0, 0, 0, B.ifpt, B.ifpt ? B.pt + 3 * V.off : nul, B.ifst, B.ifst ? B.st + 9 * V.off : nul,
             B.ifptt, B.ifptt && nt ? B.ptt + 3 * V.offt : nul, B.ifstt, B.ifstt && nt ? B.stt + 9 * V.offt : nul);
}

void batch_enqueue_mesh(Batch &B, BatchMesh &M, BatchBranch &R, Lane &f, Lane &q)
{
    BatchView V{M.n, M.nt, M.T.nboxes, M.off, M.offt, M.plan.get<char>(), &M.PL, &M.po, M.inp.get<double>(),
                M.pts.get<double>(), M.rec.get<double>(), R.nf.get<double>(), R.nodes.get<double>(),
                R.exps.get<double>(), R.lap.get<double>(), M.usefar};
    batch_enqueue_view(B, V, f, q);
}

void batch_enqueue_forest(Batch &B, Lane &f, Lane &q)
{
    BatchForest &F = B.forest;
    BatchView V{(int)B.ntri, (int)B.ntgt, F.T.nboxes, 0, 0, F.plan.get<char>(), &F.PL, &F.po, F.inp.get<double>(),
                F.pts.get<double>(), F.rec.get<double>(), F.nf.get<double>(), F.nodes.get<double>(),
                F.exps.get<double>(), F.lap.get<double>(), F.usefar};
    batch_enqueue_view(B, V, f, q);
}

// Every mesh's apply over w branches; meshes are issued round-robin over
// the branches. Direct launches fork from s0 and join back into it; a graph
// (g != nullptr) gets one independent chain of nodes per branch.
void batch_enqueue(Batch &B, int w, hipStream_t s0, hipGraph_t g)
{
    if (w == 0) {                                    // the forest: one apply over all meshes
        Lane f, q;
        f.graph = q.graph = g;
        f.stream = B.br[0].far;
        f.ev = B.br[0].ev_far;
        q.stream = B.br[0].near;
        q.ev = B.br[0].ev_near;
        if (!g) {
            HIPOK(hipEventRecord(B.ev_start, s0));
            HIPOK(hipStreamWaitEvent(f.stream, B.ev_start, 0));
        }
        batch_enqueue_forest(B, f, q);
        if (!g) {
            HIPOK(hipEventRecord(B.br[0].ev_out, f.stream));
            HIPOK(hipStreamWaitEvent(s0, B.br[0].ev_out, 0));
        }
        return;
    }
    Lane fl[BATCH_MAX_WIDTH], ql[BATCH_MAX_WIDTH];
    for (int b = 0; b < w; b++) {
        BatchBranch &R = B.br[b];
        fl[b].graph = ql[b].graph = g;
        fl[b].stream = R.far;
        fl[b].ev = R.ev_far;
        ql[b].stream = R.near;
        ql[b].ev = R.ev_near;
    }
    if (!g) {
        HIPOK(hipEventRecord(B.ev_start, s0));
        for (int b = 0; b < w; b++) HIPOK(hipStreamWaitEvent(B.br[b].far, B.ev_start, 0));
    }
    size_t depth = 0;
    for (int b = 0; b < w; b++) depth = std::max(depth, B.br[b].meshes.size());
    for (size_t k = 0; k < depth; k++)
        for (int b = 0; b < w; b++)
            if (k < B.br[b].meshes.size()) batch_enqueue_mesh(B, *B.mesh[B.br[b].meshes[k]], B.br[b], fl[b], ql[b]);
    if (!g)
        for (int b = 0; b < w; b++) {
            HIPOK(hipEventRecord(B.br[b].ev_out, B.br[b].far));
            HIPOK(hipStreamWaitEvent(s0, B.br[b].ev_out, 0));
        }
}

void batch_drop_graph(Batch &B)
{
    if (B.exec) HIPOK(hipGraphExecDestroy(B.exec));
    if (B.graph) HIPOK(hipGraphDestroy(B.graph));
    B.exec = nullptr;
    B.graph = nullptr;
}

// The graph of the current schedule, built node by node (no stream capture).
void batch_build_graph(Batch &B, int w)
{
    batch_drop_graph(B);
    HIPOK(hipGraphCreate(&B.graph, 0));
    batch_enqueue(B, w, nullptr, B.graph);
    HIPOK(hipGraphInstantiate(&B.exec, B.graph, nullptr, nullptr, 0));
}

void batch_launch(Batch &B, hipStream_t s)
{
    if (B.graph_mode)
        HIPOK(hipGraphLaunch(B.exec, s));
    else
        batch_enqueue(B, B.width, s, nullptr);
}

// Milliseconds of one apply under the current schedule: the best of reps
// after one warm-up (of one, when the warm-up alone took over 50 ms).
double batch_time(Batch &B, int reps)
{
    HIPOK(hipEventRecord(B.ev_t0, B.tstream));
    batch_launch(B, B.tstream);
    HIPOK(hipEventRecord(B.ev_t1, B.tstream));
    HIPOK(hipEventSynchronize(B.ev_t1));
    float best = 1e30f;
    HIPOK(hipEventElapsedTime(&best, B.ev_t0, B.ev_t1));
    if (best > 50.0f) reps = 1;
    best = 1e30f;
    for (int r = 0; r < reps; r++) {
        HIPOK(hipEventRecord(B.ev_t0, B.tstream));
        batch_launch(B, B.tstream);
        HIPOK(hipEventRecord(B.ev_t1, B.tstream));
        HIPOK(hipEventSynchronize(B.ev_t1));
        float ms = 0;
        HIPOK(hipEventElapsedTime(&ms, B.ev_t0, B.ev_t1));
        best = std::min(best, ms);
    }
    return best;
}

// The tuner: the forest (width 0) and each width (1, 2, 4, 8, 16 up to the
// mesh count), as direct launches and as a graph replay, timed on the
// batch's current densities; the fastest is kept (built last, so its
// graph's buffers stay fixed) and the buffers of the other kind released.
// width > 0 times only that width as a graph, width < 0 only -width as
// direct launches; +-BATCH_FOREST the forest.
void batch_tune(Batch &B, int width)
{
    int nm = (int)B.mesh.size();
    std::vector<int> widths;
    if (width == BATCH_FOREST || width == -BATCH_FOREST)
        widths.push_back(0);
    else if (width != 0)
        widths.push_back(std::min({std::abs(width), BATCH_MAX_WIDTH, nm}));
    else {
        widths.push_back(0);
        for (int w = 1; w <= BATCH_MAX_WIDTH; w *= 2)
            if (w == 1 || w <= nm) widths.push_back(w);
    }
    int best_w = widths[0], best_g = 1;
    double best_ms = 1e300;
    B.tune.clear();
    for (int w : widths)
        for (int g = (width > 0 ? 1 : 0); g <= (width < 0 ? 0 : 1); g++) {
            batch_drop_graph(B);
            batch_schedule(B, w);
            B.width = w;
            B.graph_mode = g;
            if (g) batch_build_graph(B, w);
            double ms = batch_time(B, 3);
            B.tune.insert(B.tune.end(), {(double)g, (double)w, ms});
            if (ms < best_ms) {
                best_ms = ms;
                best_w = w;
                best_g = g;
            }
        }
    // every branch beyond the chosen width is released, then the chosen
    // schedule is set up again (its scratch is already large enough)
    batch_drop_graph(B);
    batch_schedule(B, best_w);
    if (best_w == 0) {
        // the forest won: the per-mesh tree-order buffers go
        for (auto &M : B.mesh)
            for (DevBuf *d : {&M->inp, &M->pts, &M->rec}) {
                if (d->p) HIPOK(hipFree(d->p));
                d->p = nullptr;
                d->bytes = 0;
            }
    } else {
        BatchForest &F = B.forest;
        for (DevBuf *d : {&F.inp, &F.pts, &F.rec, &F.nf, &F.nodes, &F.exps, &F.lap}) {
            if (d->p) HIPOK(hipFree(d->p));
            d->p = nullptr;
            d->bytes = 0;
        }
    }
    for (int b = best_w; b < BATCH_MAX_WIDTH; b++) {
        BatchBranch &R = B.br[b];
        for (DevBuf *d : {&R.nodes, &R.exps, &R.lap, &R.nf}) {
            if (d->p) HIPOK(hipFree(d->p));
            d->p = nullptr;
            d->bytes = 0;
        }
    }
    B.width = best_w;
    B.graph_mode = best_g;
    if (best_g) batch_build_graph(B, best_w);
}

int batch_create(int iprec, double rlam, double rmu, int nmesh, const int *nparts, const double *d_tri,
                 const double *d_nrm, const double *d_src, int ifsl, int ifdl, int ifpt, int ifst,
                 const int *ntarget, const double *d_tgt, int ifptt, int ifstt, int width, Batch **out)
{
    *out = nullptr;
    if (iprec > 3 || iprec < -2 || nmesh < 1 || !nparts ||
        ((width < -BATCH_MAX_WIDTH || width > BATCH_MAX_WIDTH) && std::abs(width) != BATCH_FOREST))
        return 16;
    auto B = std::make_unique<Batch>();
    HIPOK(hipGetDevice(&B->dev));
    B->iprec = iprec;
    B->rlam = rlam;
    B->rmu = rmu;
    B->ifsl = ifsl;
    B->ifdl = ifdl;
    B->ifpt = ifpt;
    B->ifst = ifst;
    B->ifptt = ifptt;
    B->ifstt = ifstt;
    B->src_eval = (ifpt || ifst) ? 1 : 0;
    std::vector<size_t> off(nmesh + 1, 0), offt(nmesh + 1, 0);
    for (int m = 0; m < nmesh; m++) {
        int nm = nparts[m], ntm = (ntarget && (ifptt || ifstt)) ? ntarget[m] : 0;
        if (nm < 1 || ntm < 0) return 16;
        off[m + 1] = off[m] + nm;
        offt[m + 1] = offt[m] + ntm;
    }
    B->ntri = off[nmesh];
    B->ntgt = offt[nmesh];
    if (B->ntgt && !d_tgt) return 16;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        B->ds = &device_state();
        B->oc = &operators_for(*B->ds, iprec);
    }
    // geometry, densities and outputs in the caller's order, mesh after mesh
    size_t nT = B->ntri, nG = B->ntgt;
    B->geo.ensure((15 * nT + 3 * nG) * 8);
    B->tri = B->geo.get<double>();
    B->nrm = B->tri + 9 * nT;
    B->src = B->nrm + 3 * nT;
    B->tgt = B->src + 3 * nT;
    HIPOK(hipMemcpy(B->tri, d_tri, 9 * nT * 8, hipMemcpyDeviceToDevice));
    HIPOK(hipMemcpy(B->nrm, d_nrm, 3 * nT * 8, hipMemcpyDeviceToDevice));
    HIPOK(hipMemcpy(B->src, d_src, 3 * nT * 8, hipMemcpyDeviceToDevice));
    if (nG) HIPOK(hipMemcpy(B->tgt, d_tgt, 3 * nG * 8, hipMemcpyDeviceToDevice));
    B->dens.ensure(6 * nT * 8);
    B->ssl = B->dens.get<double>();
    B->sdl = B->ssl + 3 * nT;
    size_t no = (ifpt ? 3 * nT : 0) + (ifst ? 9 * nT : 0) + (ifptt ? 3 * nG : 0) + (ifstt ? 9 * nG : 0);
    B->out.ensure(no * 8);
    double *o = B->out.get<double>();
    B->pt = ifpt ? o : nullptr;
    o += ifpt ? 3 * nT : 0;
    B->st = ifst ? o : nullptr;
    o += ifst ? 9 * nT : 0;
    B->ptt = ifptt ? o : nullptr;
    o += ifptt ? 3 * nG : 0;
    B->stt = ifstt ? o : nullptr;
    HIPOK(launch_fill0(B->ssl, 6 * nT, nullptr));
    HIPOK(hipDeviceSynchronize());
    std::vector<double> hs(3 * nT), ht(3 * std::max<size_t>(nG, 1));
    HIPOK(hipMemcpy(hs.data(), d_src, 3 * nT * 8, hipMemcpyDeviceToHost));
    if (nG) HIPOK(hipMemcpy(ht.data(), d_tgt, 3 * nG * 8, hipMemcpyDeviceToHost));
    // per mesh: octree, task lists, the packed plan and the tree-order buffers
    const OpsCache &oc = *B->oc;
    std::vector<int> waves;
    for (int m = 0; m < nmesh; m++) {
        auto M = std::make_unique<BatchMesh>();
        M->n = nparts[m];
        M->nt = (int)(offt[m + 1] - offt[m]);
        M->off = off[m];
        M->offt = offt[m];
        int np = M->n + M->nt;
        {
            std::lock_guard<std::mutex> lk(g_plan_mu);
            if (build_tree(hs.data() + 3 * M->off, M->n, ht.data() + 3 * M->offt, M->nt, iprec_nbox(iprec, np), 0,
                           M->T))
                return 4;
            build_plan(M->T, M->n, &oc.ops, B->src_eval != 0, false, NRHS, M->PL, false);
        }
        M->usefar = M->T.nlev >= 2;
        far_scratch(iprec, M->n, np, M->T.nboxes, oc.p, M->n_nodes, M->n_exps, M->n_lap);
        if (!M->usefar) M->n_nodes = M->n_exps = M->n_lap = 0;
        const double *st = M->PL.stats;
        M->cost = 2400.0 * st[6] + (M->usefar ? st[4] : 0.0) + 2.0e4 * np + 1.0e9;
        Packer pk;
        pack_plan(pk, M->T, M->PL, M->po);
        near_tasks(M->T, M->PL, B->src_eval != 0, waves);
        pack_near_tasks(pk, waves, M->po);
        std::vector<char> stage(pk.size);
        pk.pack(stage.data());
        M->plan.ensure(pk.size);
        HIPOK(hipMemcpy(M->plan.p, stage.data(), pk.size, hipMemcpyHostToDevice));
        M->inp.ensure((size_t)M->n * 18 * 8);
        M->pts.ensure((size_t)np * 3 * 8);
        M->rec.ensure((size_t)M->n * NF_REC * 8);
        B->mesh.push_back(std::move(M));
    }
    // the forest of all trees, one plan
    {
        BatchForest &F = B->forest;
        std::vector<const Tree *> ts;
        std::vector<int> so, to;
        for (int m = 0; m < nmesh; m++) {
            ts.push_back(&B->mesh[m]->T);
            so.push_back((int)off[m]);
            to.push_back((int)offt[m]);
        }
        int np = (int)(nT + nG);
        {
            std::lock_guard<std::mutex> lk(g_plan_mu);
            build_forest(ts, so, to, F.T);
            build_plan(F.T, (int)nT, &oc.ops, B->src_eval != 0, false, NRHS, F.PL, false);
        }
        F.usefar = F.T.nlev >= 2;
        Packer pk;
        pack_plan(pk, F.T, F.PL, F.po);
        near_tasks(F.T, F.PL, B->src_eval != 0, waves);
        pack_near_tasks(pk, waves, F.po);
        std::vector<char> stage(pk.size);
        pk.pack(stage.data());
        F.plan.ensure(pk.size);
        HIPOK(hipMemcpy(F.plan.p, stage.data(), pk.size, hipMemcpyHostToDevice));
        F.inp.ensure(nT * 18 * 8);
        F.pts.ensure((size_t)np * 3 * 8);
        F.rec.ensure(nT * NF_REC * 8);
        F.nf.ensure((size_t)np * 9 * 8);
        if (F.usefar) {
            size_t a, e, l;
            far_scratch(iprec, (int)nT, np, F.T.nboxes, oc.p, a, e, l);
            F.nodes.ensure(a * 8);
            F.exps.ensure(e * 8);
            F.lap.ensure(l * 8);
        }
    }
    HIPOK(hipStreamCreateWithFlags(&B->tstream, hipStreamNonBlocking));
    HIPOK(hipEventCreateWithFlags(&B->ev_start, hipEventDisableTiming));
    HIPOK(hipEventCreate(&B->ev_t0));
    HIPOK(hipEventCreate(&B->ev_t1));
    for (auto &R : B->br) {
        HIPOK(hipStreamCreateWithFlags(&R.far, hipStreamNonBlocking));
        HIPOK(hipStreamCreateWithFlags(&R.near, hipStreamNonBlocking));
        HIPOK(hipEventCreateWithFlags(&R.ev_far, hipEventDisableTiming));
        HIPOK(hipEventCreateWithFlags(&R.ev_near, hipEventDisableTiming));
        HIPOK(hipEventCreateWithFlags(&R.ev_out, hipEventDisableTiming));
    }
    batch_tune(*B, width);
    HIPOK(hipStreamSynchronize(B->tstream));
    *out = B.release();
    return 0;
}

}  // namespace

// ------------------------------------------------------------------------
// Direct sum without allocation. The workspace of el3dtriadirecttarg (the
// triangles' near-field records, the points, the per-point fields) lives in
// `scratch`, a file-scope device array of NOALLOC_BYTES on every device the
// library runs on, held until the process ends. Its device address is taken
// once per device (hipGetSymbolAddress) and only that address is passed to
// kernels. Calls on one device share the array: calls that overlap on one
// device race, and each call overwrites what the last one left.
// ------------------------------------------------------------------------
constexpr int64_t NOALLOC_MAX_TRI = 131072;        // n
constexpr int64_t NOALLOC_MAX_PTS = 262144;        // n + nt
constexpr size_t NOALLOC_BYTES = (size_t)(NOALLOC_MAX_TRI * NF_REC + NOALLOC_MAX_PTS * 12) * 8;   // 46 MiB
static __device__ __align__(256) double scratch[NOALLOC_BYTES / 8];

namespace {
constexpr int NOALLOC_DEVICES = 64;
std::mutex g_noalloc_mu;
double *g_noalloc_ptr[NOALLOC_DEVICES] = {};

// this device's address of `scratch` (nullptr if it cannot be had)
double *noalloc_scratch()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NOALLOC_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        double *p = nullptr;
        if (hipGetSymbolAddress((void **)&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        g_noalloc_ptr[dev] = p;
    }
    return g_noalloc_ptr[dev];
}
}  // namespace

}  // namespace elfmm

// ------------------------------------------------------------------------
// C-ABI
// ------------------------------------------------------------------------

using namespace elfmm;

namespace {

struct HostCall {
    std::vector<void *> bufs;
    ~HostCall()
    {
        for (void *p : bufs) (void)hipFree(p);
    }
    double *up(const double *h, size_t count)
    {
        void *d = nullptr;
        HIPOK(hipMalloc(&d, std::max<size_t>(count, 1) * 8));
        bufs.push_back(d);
        if (h && count) HIPOK(hipMemcpy(d, h, count * 8, hipMemcpyHostToDevice));
        return (double *)d;
    }
    double *out(size_t count)
    {
        void *d = nullptr;
        HIPOK(hipMalloc(&d, std::max<size_t>(count, 1) * 8));
        bufs.push_back(d);
        return (double *)d;
    }
};

int host_apply(int iprec, double rlam, double rmu, int n, const double *tri, const double *nrm,
               const double *src, int ifsl, const double *ssl, int ifdl, const double *sdl, int ifpt,
               double *pt, int ifst, double *st, int nt, const double *tgt, int ifptt, double *ptt,
               int ifstt, double *stt, bool direct)
{
    try {
        HostCall hc;
        if (!(ifpt || ifst)) {
            ifpt = ifst = 0;
        }
        if (!(ifptt || ifstt)) nt = 0;
        double *d_tri = hc.up(tri, 9 * (size_t)n), *d_nrm = hc.up(nrm, 3 * (size_t)n),
               *d_src = hc.up(src, 3 * (size_t)n);
        double *d_ssl = ifsl ? hc.up(ssl, 3 * (size_t)n) : nullptr;
        double *d_sdl = ifdl ? hc.up(sdl, 3 * (size_t)n) : nullptr;
        double *d_tgt = hc.up(nt ? tgt : nullptr, 3 * (size_t)nt);
        double *d_pt = ifpt ? hc.out(3 * (size_t)n) : nullptr, *d_st = ifst ? hc.out(9 * (size_t)n) : nullptr;
        double *d_ptt = ifptt && nt ? hc.out(3 * (size_t)nt) : nullptr;
        double *d_stt = ifstt && nt ? hc.out(9 * (size_t)nt) : nullptr;
        int ier = triatarg_dev(iprec, rlam, rmu, n, d_tri, d_nrm, d_src, ifsl, d_ssl, ifdl, d_sdl, ifpt, d_pt,
                               ifst, d_st, nt, d_tgt, ifptt, d_ptt, ifstt, d_stt, nullptr, direct);
        if (ier) return ier;
        if (ifpt) HIPOK(hipMemcpy(pt, d_pt, 3 * (size_t)n * 8, hipMemcpyDeviceToHost));
        if (ifst) HIPOK(hipMemcpy(st, d_st, 9 * (size_t)n * 8, hipMemcpyDeviceToHost));
        if (d_ptt) HIPOK(hipMemcpy(ptt, d_ptt, 3 * (size_t)nt * 8, hipMemcpyDeviceToHost));
        if (d_stt) HIPOK(hipMemcpy(stt, d_stt, 9 * (size_t)nt * 8, hipMemcpyDeviceToHost));
        return 0;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

// Host-array iter apply: icomp 0 computes nothing (the reference's
// icomp 0 skips both passes, src/elfmm3dtria_iter_1.f:311-319) and reports
// the reference's work-array size; icomp 4 plans only and leaves the
// outputs untouched; icomp 5 adds the near field to the caller's values.
int host_apply_iter(int iprec, double rlam, double rmu, int n, const double *tri, const double *nrm,
                    const double *src, int ifsl, const double *ssl, int ifdl, const double *sdl, int ifpt,
                    double *pt, int ifst, double *st, int nt, const double *tgt, int ifptt, double *ptt,
                    int ifstt, double *stt, int icomp, double *wsave, int lwsave, int *lused)
{
    if (icomp == 0 || icomp < 0 || icomp > 5) {
        // the reference's lused after its work-array bookkeeping
        // (src/elfmm3dtria_iter_1.f:254-296)
        *lused = 50 * n + 29 * nt;
        return 0;
    }
    try {
        HostCall hc;
        if (!(ifpt || ifst)) ifpt = ifst = 0;
        if (!(ifptt || ifstt)) nt = 0;
        bool add = icomp == 5;
        double *d_tri = hc.up(tri, 9 * (size_t)n), *d_nrm = hc.up(nrm, 3 * (size_t)n),
               *d_src = hc.up(src, 3 * (size_t)n);
        double *d_ssl = ifsl ? hc.up(ssl, 3 * (size_t)n) : nullptr;
        double *d_sdl = ifdl ? hc.up(sdl, 3 * (size_t)n) : nullptr;
        double *d_tgt = hc.up(nt ? tgt : nullptr, 3 * (size_t)nt);
        auto outbuf = [&](int flag, double *h, size_t count) -> double * {
            if (!flag) return nullptr;
            return add ? hc.up(h, count) : hc.out(count);
        };
        double *d_pt = outbuf(ifpt, pt, 3 * (size_t)n), *d_st = outbuf(ifst, st, 9 * (size_t)n);
        double *d_ptt = outbuf(ifptt && nt, ptt, 3 * (size_t)nt), *d_stt = outbuf(ifstt && nt, stt, 9 * (size_t)nt);
        IterCall it{icomp, wsave, lwsave};
        int ier = triatarg_dev(iprec, rlam, rmu, n, d_tri, d_nrm, d_src, ifsl, d_ssl, ifdl, d_sdl, ifpt, d_pt,
                               ifst, d_st, nt, d_tgt, ifptt, d_ptt, ifstt, d_stt, nullptr, false, &it);
        *lused = ITER_HANDLE_WORDS;
        if (ier) return ier;
        if (icomp == 4) return 0;
        if (ifpt) HIPOK(hipMemcpy(pt, d_pt, 3 * (size_t)n * 8, hipMemcpyDeviceToHost));
        if (ifst) HIPOK(hipMemcpy(st, d_st, 9 * (size_t)n * 8, hipMemcpyDeviceToHost));
        if (d_ptt) HIPOK(hipMemcpy(ptt, d_ptt, 3 * (size_t)nt * 8, hipMemcpyDeviceToHost));
        if (d_stt) HIPOK(hipMemcpy(stt, d_stt, 9 * (size_t)nt * 8, hipMemcpyDeviceToHost));
        return it.status;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

// Host-array half-space apply (targets only): icomp 4 plans only and leaves
// the outputs untouched; icomp 0 zeroes the outputs (the reference zeroes
// them on entry and computes nothing, src/elhfmm3dtria_iter.f:178-228).
int host_apply_h(int iprec, double rlam, double rmu, int n, const double *tri, const double *nrm, const double *src,
                 int ifsl, const double *ssl, int ifdl, const double *sdl, int nt, const double *tgt, int ifptt,
                 double *ptt, int ifstt, double *stt, int icomp, double *wsave, int lwsave, int *lused)
{
    if (!(ifptt || ifstt) || nt < 1) return 0;
    try {
        HostCall hc;
        double *d_tri = hc.up(tri, 9 * (size_t)n), *d_nrm = hc.up(nrm, 3 * (size_t)n),
               *d_src = hc.up(src, 3 * (size_t)n);
        double *d_ssl = ifsl ? hc.up(ssl, 3 * (size_t)n) : nullptr;
        double *d_sdl = ifdl ? hc.up(sdl, 3 * (size_t)n) : nullptr;
        double *d_tgt = hc.up(tgt, 3 * (size_t)nt);
        double *d_ptt = ifptt ? hc.out(3 * (size_t)nt) : nullptr, *d_stt = ifstt ? hc.out(9 * (size_t)nt) : nullptr;
        IterCall it{icomp, wsave, lwsave};
        int ier = htriatargiter_dev(iprec, rlam, rmu, n, d_tri, d_nrm, d_src, ifsl, d_ssl, ifdl, d_sdl, nt, d_tgt,
                                    ifptt, d_ptt, ifstt, d_stt, nullptr, it);
        *lused = ITER_HANDLE_WORDS;
        if (ier) return ier;
        if (icomp == 4) return 0;
        if (d_ptt) HIPOK(hipMemcpy(ptt, d_ptt, 3 * (size_t)nt * 8, hipMemcpyDeviceToHost));
        if (d_stt) HIPOK(hipMemcpy(stt, d_stt, 9 * (size_t)nt * 8, hipMemcpyDeviceToHost));
        return it.status;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

// Host-array point apply: inputs copied to the device, outputs back.
// half (with direct): the Mindlin half-space direct sum, the free-space
// sum plus the image part of every source (elh3dpartdirecttarg).
int host_apply_part(int iprec, double rlam, double rmu, int n, const double *src, int ifsl, const double *ssl,
                    int ifdl, const double *sdl, const double *sdv, int ifpt, double *pt, int ifst, double *st,
                    int nt, const double *tgt, int ifptt, double *ptt, int ifstt, double *stt, bool direct,
                    bool half = false)
{
    try {
        HostCall hc;
        if (!(ifptt || ifstt)) nt = 0;
        double *d_src = hc.up(src, 3 * (size_t)n);
        double *d_ssl = ifsl ? hc.up(ssl, 3 * (size_t)n) : nullptr;
        double *d_sdl = ifdl ? hc.up(sdl, 3 * (size_t)n) : nullptr;
        double *d_sdv = ifdl ? hc.up(sdv, 3 * (size_t)n) : nullptr;
        double *d_tgt = hc.up(nt ? tgt : nullptr, 3 * (size_t)nt);
        double *d_pt = ifpt ? hc.out(3 * (size_t)n) : nullptr, *d_st = ifst ? hc.out(9 * (size_t)n) : nullptr;
        double *d_ptt = ifptt && nt ? hc.out(3 * (size_t)nt) : nullptr;
        double *d_stt = ifstt && nt ? hc.out(9 * (size_t)nt) : nullptr;
        int ier = parttarg_dev(iprec, rlam, rmu, n, d_src, ifsl, d_ssl, ifdl, d_sdl, d_sdv, ifpt, d_pt, ifst, d_st,
                               nt, d_tgt, ifptt, d_ptt, ifstt, d_stt, nullptr, direct);
        if (ier) return ier;
        if (half) {
            HIPOK(launch_pimage((ifpt || ifst) ? n : 0, n, nt, d_src, d_tgt, d_ssl, d_sdl, d_sdv, ifsl, ifdl, rlam,
                                rmu, ifpt, d_pt, ifst, d_st, ifptt && nt, d_ptt, ifstt && nt, d_stt, nullptr));
            HIPOK(hipStreamSynchronize(nullptr));
        }
        if (ifpt) HIPOK(hipMemcpy(pt, d_pt, 3 * (size_t)n * 8, hipMemcpyDeviceToHost));
        if (ifst) HIPOK(hipMemcpy(st, d_st, 9 * (size_t)n * 8, hipMemcpyDeviceToHost));
        if (d_ptt) HIPOK(hipMemcpy(ptt, d_ptt, 3 * (size_t)nt * 8, hipMemcpyDeviceToHost));
        if (d_stt) HIPOK(hipMemcpy(stt, d_stt, 9 * (size_t)nt * 8, hipMemcpyDeviceToHost));
        return 0;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

int host_apply_hdirect(double rlam, double rmu, int n, const double *tri, const double *nrm, const double *src,
                       int ifsl, const double *ssl, int ifdl, const double *sdl, int ifpt, double *pt, int ifst,
                       double *st, int nt, const double *tgt, int ifptt, double *ptt, int ifstt, double *stt)
{
    try {
        HostCall hc;
        if (!(ifptt || ifstt)) nt = 0;
        double *d_tri = hc.up(tri, 9 * (size_t)n), *d_nrm = hc.up(nrm, 3 * (size_t)n),
               *d_src = hc.up(src, 3 * (size_t)n);
        double *d_ssl = ifsl ? hc.up(ssl, 3 * (size_t)n) : nullptr;
        double *d_sdl = ifdl ? hc.up(sdl, 3 * (size_t)n) : nullptr;
        double *d_tgt = hc.up(nt ? tgt : nullptr, 3 * (size_t)nt);
        double *d_pt = ifpt ? hc.out(3 * (size_t)n) : nullptr, *d_st = ifst ? hc.out(9 * (size_t)n) : nullptr;
        double *d_ptt = ifptt && nt ? hc.out(3 * (size_t)nt) : nullptr;
        double *d_stt = ifstt && nt ? hc.out(9 * (size_t)nt) : nullptr;
        int ier = hdirect_dev(rlam, rmu, n, d_tri, d_nrm, d_src, ifsl, d_ssl, ifdl, d_sdl, ifpt, d_pt, ifst, d_st,
                              nt, d_tgt, ifptt, d_ptt, ifstt, d_stt, nullptr);
        if (ier) return ier;
        if (ifpt) HIPOK(hipMemcpy(pt, d_pt, 3 * (size_t)n * 8, hipMemcpyDeviceToHost));
        if (ifst) HIPOK(hipMemcpy(st, d_st, 9 * (size_t)n * 8, hipMemcpyDeviceToHost));
        if (d_ptt) HIPOK(hipMemcpy(ptt, d_ptt, 3 * (size_t)nt * 8, hipMemcpyDeviceToHost));
        if (d_stt) HIPOK(hipMemcpy(stt, d_stt, 9 * (size_t)nt * 8, hipMemcpyDeviceToHost));
        return 0;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

}  // namespace

extern "C" {

void elfmm3dtriatargiter_(int *ier, const int *iprec, const double *rlam, const double *rmu,
                          const double *triangle, const double *trinorm, const int *nparts,
                          const double *source, const int *ifsingle, const double *sigma_sl,
                          const int *ifdouble, const double *sigma_dl, const int *ifptfrc, double *ptfrc,
                          const int *ifstrain, double *strain, const int *ntargs, const double *target,
                          const int *ifptfrctarg, double *ptfrctarg, const int *ifstraintarg,
                          double *straintarg, const int *icomp_type, double *wsave, const int *lwsave,
                          int *lused)
{
    *ier = host_apply_iter(*iprec, *rlam, *rmu, *nparts, triangle, trinorm, source, *ifsingle == 1, sigma_sl,
                           *ifdouble == 1, sigma_dl, *ifptfrc == 1, ptfrc, *ifstrain == 1, strain, *ntargs,
                           target, *ifptfrctarg == 1, ptfrctarg, *ifstraintarg == 1, straintarg, *icomp_type,
                           wsave, *lwsave, lused);
}

void elfmm3dtriaiter_(int *ier, const int *iprec, const double *rlam, const double *rmu,
                      const double *triangle, const double *trinorm, const int *nparts, const double *source,
                      const int *ifsingle, const double *sigma_sl, const int *ifdouble,
                      const double *sigma_dl, const int *ifptfrc, double *ptfrc, const int *ifstrain,
                      double *strain, const int *icomp_type, double *wsave, const int *lwsave, int *lused)
{
    *ier = host_apply_iter(*iprec, *rlam, *rmu, *nparts, triangle, trinorm, source, *ifsingle == 1, sigma_sl,
                           *ifdouble == 1, sigma_dl, *ifptfrc == 1, ptfrc, *ifstrain == 1, strain, 0, nullptr, 0,
                           nullptr, 0, nullptr, *icomp_type, wsave, *lwsave, lused);
}

int elfmm_gfx950_triatargiter_dev(int iprec, double rlam, double rmu, int nparts, const double *d_triangle,
                                  const double *d_trinorm, const double *d_source, int ifsingle,
                                  const double *d_sigma_sl, int ifdouble, const double *d_sigma_dl,
                                  int ifptfrc, double *d_ptfrc, int ifstrain, double *d_strain, int ntargs,
                                  const double *d_target, int ifptfrctarg, double *d_ptfrctarg,
                                  int ifstraintarg, double *d_straintarg, int icomp_type, double *wsave,
                                  int lwsave, int *lused, void *stream)
{
    if (icomp_type < 1 || icomp_type > 5) {
        *lused = 50 * nparts + 29 * ntargs;
        return 0;
    }
    try {
        IterCall it{icomp_type, wsave, lwsave};
        int ier = triatarg_dev(iprec, rlam, rmu, nparts, d_triangle, d_trinorm, d_source, ifsingle == 1,
                               d_sigma_sl, ifdouble == 1, d_sigma_dl, ifptfrc == 1, d_ptfrc, ifstrain == 1,
                               d_strain, ntargs, d_target, ifptfrctarg == 1, d_ptfrctarg, ifstraintarg == 1,
                               d_straintarg, (hipStream_t)stream, false, &it);
        *lused = ITER_HANDLE_WORDS;
        return ier ? ier : it.status;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

int elfmm_gfx950_triatargiter_multi_dev(int iprec, double rlam, double rmu, int nparts, const double *d_triangle,
                                        const double *d_trinorm, const double *d_source, int nrhs, int ifsingle,
                                        const double *d_sigma_sl, int ifdouble, const double *d_sigma_dl,
                                        int ifptfrc, double *d_ptfrc, int ifstrain, double *d_strain, int ntargs,
                                        const double *d_target, int ifptfrctarg, double *d_ptfrctarg,
                                        int ifstraintarg, double *d_straintarg, double *wsave, int lwsave,
                                        void *stream)
{
    if (nrhs < 1) return 0;
    try {
        IterCall it{3, wsave, lwsave};
        it.nrhs = nrhs;
        int ier = triatarg_dev(iprec, rlam, rmu, nparts, d_triangle, d_trinorm, d_source, ifsingle == 1,
                               d_sigma_sl, ifdouble == 1, d_sigma_dl, ifptfrc == 1, d_ptfrc, ifstrain == 1,
                               d_strain, ntargs, d_target, ifptfrctarg == 1, d_ptfrctarg, ifstraintarg == 1,
                               d_straintarg, (hipStream_t)stream, false, &it);
        return ier ? ier : it.status;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

int elfmm_gfx950_htriatargiter_multi_dev(int iprec, double rlam, double rmu, int nparts, const double *d_triangle,
                                         const double *d_trinorm, const double *d_source, int nrhs, int ifsingle,
                                         const double *d_sigma_sl, int ifdouble, const double *d_sigma_dl,
                                         int ntargs, const double *d_target, int ifptfrctarg, double *d_ptfrctarg,
                                         int ifstraintarg, double *d_straintarg, double *wsave, int lwsave,
                                         void *stream)
{
    if (nrhs < 1) return 0;
    try {
        IterCall it{3, wsave, lwsave};
        it.nrhs = nrhs;
        int ier = htriatargiter_dev(iprec, rlam, rmu, nparts, d_triangle, d_trinorm, d_source, ifsingle == 1,
                                    d_sigma_sl, ifdouble == 1, d_sigma_dl, ntargs, d_target, ifptfrctarg == 1,
                                    d_ptfrctarg, ifstraintarg == 1, d_straintarg, (hipStream_t)stream, it);
        return ier ? ier : it.status;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

int elfmm_gfx950_iter_release(const double *wsave, int lwsave)
{
    std::shared_ptr<NearStore> s;          // freed here unless a running call still holds it
    std::lock_guard<std::mutex> lk(g_mu);
    s = find_store(wsave, lwsave);
    if (!s) return 0;
    for (auto e = g_stores.begin(); e != g_stores.end(); ++e)
        if (e->second == s) {
            g_stores.erase(e);
            return 1;
        }
    return 0;
}

void elhfmm3dtriatargiter_(int *ier, const int *iprec, const double *rlam, const double *rmu,
                           const double *triangle, const double *trinorm, const int *nparts, const double *source,
                           const int *ifsingle, const double *sigma_sl, const int *ifdouble, const double *sigma_dl,
                           const int *ntargs, const double *target, const int *ifptfrctarg, double *ptfrctarg,
                           const int *ifstraintarg, double *straintarg, const int *icomp_type, double *wsave,
                           const int *lwsave, int *lused)
{
    *ier = host_apply_h(*iprec, *rlam, *rmu, *nparts, triangle, trinorm, source, *ifsingle == 1, sigma_sl,
                        *ifdouble == 1, sigma_dl, *ntargs, target, *ifptfrctarg == 1, ptfrctarg, *ifstraintarg == 1,
                        straintarg, *icomp_type, wsave, *lwsave, lused);
}

int elfmm_gfx950_htriatargiter_dev(int iprec, double rlam, double rmu, int nparts, const double *d_triangle,
                                   const double *d_trinorm, const double *d_source, int ifsingle,
                                   const double *d_sigma_sl, int ifdouble, const double *d_sigma_dl, int ntargs,
                                   const double *d_target, int ifptfrctarg, double *d_ptfrctarg, int ifstraintarg,
                                   double *d_straintarg, int icomp_type, double *wsave, int lwsave, int *lused,
                                   void *stream)
{
    try {
        IterCall it{icomp_type, wsave, lwsave};
        int ier = htriatargiter_dev(iprec, rlam, rmu, nparts, d_triangle, d_trinorm, d_source, ifsingle == 1,
                                    d_sigma_sl, ifdouble == 1, d_sigma_dl, ntargs, d_target, ifptfrctarg == 1,
                                    d_ptfrctarg, ifstraintarg == 1, d_straintarg, (hipStream_t)stream, it);
        if (lused) *lused = ITER_HANDLE_WORDS;
        return ier ? ier : it.status;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

void elh3dtriadirecttarg_(const double *rlam, const double *rmu, const double *triangle, const double *trinorm,
                          const int *nsource, const double *source, const int *ifsingle, const double *sigma_sl,
                          const int *ifdouble, const double *sigma_dl, const int *ifptfrc, double *ptfrc,
                          const int *ifstrain, double *strain, const int *ntarget, const double *target,
                          const int *ifptfrctarg, double *ptfrctarg, const int *ifstraintarg, double *straintarg)
{
    (void)host_apply_hdirect(*rlam, *rmu, *nsource, triangle, trinorm, source, *ifsingle == 1, sigma_sl,
                             *ifdouble == 1, sigma_dl, *ifptfrc == 1, ptfrc, *ifstrain == 1, strain, *ntarget,
                             target, *ifptfrctarg == 1, ptfrctarg, *ifstraintarg == 1, straintarg);
}

void elfmm_gfx950_half_parts(int mask) { g_half_parts.store(mask & 7); }

int elfmm_gfx950_el3dtriadirecttarg_noalloc(double rlam, double rmu, int nsource, const double *d_triangle,
                                            const double *d_trinorm, const double *d_source, int ifsingle,
                                            const double *d_sigma_sl, int ifdouble, const double *d_sigma_dl,
                                            int ifptfrc, double *d_ptfrc, int ifstrain, double *d_strain,
                                            int ntarget, const double *d_target, int ifptfrctarg,
                                            double *d_ptfrctarg, int ifstraintarg, double *d_straintarg,
                                            void *stream)
{
    (void)d_trinorm;   // the double layer's orientation is the triangle's own normal
    int n = nsource;
    int ifpt = ifptfrc == 1, ifst = ifstrain == 1, ifptt = ifptfrctarg == 1, ifstt = ifstraintarg == 1;
    int nt = (ifptt || ifstt) ? ntarget : 0;
    if (n < 1) return 0;
    if (nt < 0 || (int64_t)n > NOALLOC_MAX_TRI || (int64_t)n + nt > NOALLOC_MAX_PTS) return 128;
    double *base = noalloc_scratch();
    if (!base) return 32;
    double *rec = base, *pts = rec + NOALLOC_MAX_TRI * NF_REC, *nf = pts + 3 * NOALLOC_MAX_PTS;
    hipStream_t st = (hipStream_t)stream;
    int ifsl = ifsingle == 1, ifdl = ifdouble == 1;
    int src_eval = (ifpt || ifst) ? 1 : 0;
    int npe = (src_eval ? n : 0) + nt;
    double c1 = (rlam + rmu) / (rlam + 2 * rmu);
    hipLaunchKernelGGL(k_direct_prep, dim3((n + nt + 255) / 256), dim3(256), 0, st, n, nt, d_triangle, d_source,
                       ifsl, d_sigma_sl, ifdl, d_sigma_dl, d_target, pts, rec);
    int per = NF_THREADS / 64;
    if (npe)
        hipLaunchKernelGGL(k_direct, dim3((npe + per - 1) / per), dim3(NF_THREADS), 0, st, n, npe,
                           src_eval ? n : 0, pts, rec, rlam, rmu, c1, ifsl, ifdl, nf);
    hipLaunchKernelGGL(k_assemble, dim3((n + nt + 255) / 256), dim3(256), 0, st, n, nt, src_eval, nullptr, nullptr,
                       pts, nullptr, nf, c1, 0, 0, 0, ifpt, d_ptfrc, ifst, d_strain, ifptt, d_ptfrctarg, ifstt,
                       d_straintarg);
    return hipGetLastError() == hipSuccess ? 0 : 32;
}

void elfmm3dtriatarg_(int *ier, const int *iprec, const double *rlam, const double *rmu,
                      const double *triangle, const double *trinorm, const int *nparts,
                      const double *source, const int *ifsingle, const double *sigma_sl,
                      const int *ifdouble, const double *sigma_dl, const int *ifptfrc, double *ptfrc,
                      const int *ifstrain, double *strain, const int *ntargs, const double *target,
                      const int *ifptfrctarg, double *ptfrctarg, const int *ifstraintarg,
                      double *straintarg)
{
    *ier = host_apply(*iprec, *rlam, *rmu, *nparts, triangle, trinorm, source, *ifsingle == 1, sigma_sl,
                      *ifdouble == 1, sigma_dl, *ifptfrc == 1, ptfrc, *ifstrain == 1, strain, *ntargs, target,
                      *ifptfrctarg == 1, ptfrctarg, *ifstraintarg == 1, straintarg, false);
}

void elfmm3dtria_(int *ier, const int *iprec, const double *rlam, const double *rmu,
                  const double *triangle, const double *trinorm, const int *nparts, const double *source,
                  const int *ifsingle, const double *sigma_sl, const int *ifdouble,
                  const double *sigma_dl, const int *ifptfrc, double *ptfrc, const int *ifstrain,
                  double *strain)
{
    *ier = host_apply(*iprec, *rlam, *rmu, *nparts, triangle, trinorm, source, *ifsingle == 1, sigma_sl,
                      *ifdouble == 1, sigma_dl, *ifptfrc == 1, ptfrc, *ifstrain == 1, strain, 0, nullptr, 0,
                      nullptr, 0, nullptr, false);
}

void el3dtriadirecttarg_(const double *rlam, const double *rmu, const double *triangle,
                         const double *trinorm, const int *nsource, const double *source,
                         const int *ifsingle, const double *sigma_sl, const int *ifdouble,
                         const double *sigma_dl, const int *ifptfrc, double *ptfrc, const int *ifstrain,
                         double *strain, const int *ntarget, const double *target,
                         const int *ifptfrctarg, double *ptfrctarg, const int *ifstraintarg,
                         double *straintarg)
{
    (void)host_apply(0, *rlam, *rmu, *nsource, triangle, trinorm, source, *ifsingle == 1, sigma_sl,
                     *ifdouble == 1, sigma_dl, *ifptfrc == 1, ptfrc, *ifstrain == 1, strain, *ntarget, target,
                     *ifptfrctarg == 1, ptfrctarg, *ifstraintarg == 1, straintarg, true);
}

void elfmm3dparttarg_(int *ier, const int *iprec, const double *rlam, const double *rmu, const int *nparts,
                      const double *source, const int *ifsingle, const double *sigma_sl, const int *ifdouble,
                      const double *sigma_dl, const double *sigma_dv, const int *ifptfrc, double *ptfrc,
                      const int *ifstrain, double *strain, const int *ntargs, const double *target,
                      const int *ifptfrctarg, double *ptfrctarg, const int *ifstraintarg, double *straintarg)
{
    *ier = host_apply_part(*iprec, *rlam, *rmu, *nparts, source, *ifsingle == 1, sigma_sl, *ifdouble == 1, sigma_dl,
                           sigma_dv, *ifptfrc == 1, ptfrc, *ifstrain == 1, strain, *ntargs, target,
                           *ifptfrctarg == 1, ptfrctarg, *ifstraintarg == 1, straintarg, false);
}

void elfmm3dpart_(int *ier, const int *iprec, const double *rlam, const double *rmu, const int *nparts,
                  const double *source, const int *ifsingle, const double *sigma_sl, const int *ifdouble,
                  const double *sigma_dl, const double *sigma_dv, const int *ifptfrc, double *ptfrc,
                  const int *ifstrain, double *strain)
{
    *ier = host_apply_part(*iprec, *rlam, *rmu, *nparts, source, *ifsingle == 1, sigma_sl, *ifdouble == 1, sigma_dl,
                           sigma_dv, *ifptfrc == 1, ptfrc, *ifstrain == 1, strain, 0, nullptr, 0, nullptr, 0, nullptr,
                           false);
}

void el3dpartdirecttarg_(const double *rlam, const double *rmu, const int *nsource, const double *source,
                         const int *ifsingle, const double *sigma_sl, const int *ifdouble, const double *sigma_dl,
                         const double *sigma_dv, const int *ifptfrc, double *ptfrc, const int *ifstrain,
                         double *strain, const int *ntarget, const double *target, const int *ifptfrctarg,
                         double *ptfrctarg, const int *ifstraintarg, double *straintarg)
{
    (void)host_apply_part(0, *rlam, *rmu, *nsource, source, *ifsingle == 1, sigma_sl, *ifdouble == 1, sigma_dl,
                          sigma_dv, *ifptfrc == 1, ptfrc, *ifstrain == 1, strain, *ntarget, target,
                          *ifptfrctarg == 1, ptfrctarg, *ifstraintarg == 1, straintarg, true);
}

void elh3dpartdirecttarg_(const double *rlam, const double *rmu, const int *nsource, const double *source,
                          const int *ifsingle, const double *sigma_sl, const int *ifdouble, const double *sigma_dl,
                          const double *sigma_dv, const int *ifptfrc, double *ptfrc, const int *ifstrain,
                          double *strain, const int *ntarget, const double *target, const int *ifptfrctarg,
                          double *ptfrctarg, const int *ifstraintarg, double *straintarg)
{
    (void)host_apply_part(0, *rlam, *rmu, *nsource, source, *ifsingle == 1, sigma_sl, *ifdouble == 1, sigma_dl,
                          sigma_dv, *ifptfrc == 1, ptfrc, *ifstrain == 1, strain, *ntarget, target,
                          *ifptfrctarg == 1, ptfrctarg, *ifstraintarg == 1, straintarg, true, true);
}

int elfmm_gfx950_parttarg_dev(int iprec, double rlam, double rmu, int nparts, const double *d_source, int ifsingle,
                              const double *d_sigma_sl, int ifdouble, const double *d_sigma_dl,
                              const double *d_sigma_dv, int ifptfrc, double *d_ptfrc, int ifstrain, double *d_strain,
                              int ntargs, const double *d_target, int ifptfrctarg, double *d_ptfrctarg,
                              int ifstraintarg, double *d_straintarg, void *stream)
{
    try {
        return parttarg_dev(iprec, rlam, rmu, nparts, d_source, ifsingle == 1, d_sigma_sl, ifdouble == 1,
                            d_sigma_dl, d_sigma_dv, ifptfrc == 1, d_ptfrc, ifstrain == 1, d_strain, ntargs, d_target,
                            ifptfrctarg == 1, d_ptfrctarg, ifstraintarg == 1, d_straintarg, (hipStream_t)stream,
                            false);
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

int elfmm_gfx950_triatarg_dev(int iprec, double rlam, double rmu, int nparts, const double *d_triangle,
                              const double *d_trinorm, const double *d_source, int ifsingle,
                              const double *d_sigma_sl, int ifdouble, const double *d_sigma_dl, int ifptfrc,
                              double *d_ptfrc, int ifstrain, double *d_strain, int ntargs,
                              const double *d_target, int ifptfrctarg, double *d_ptfrctarg, int ifstraintarg,
                              double *d_straintarg, void *stream)
{
    try {
        return triatarg_dev(iprec, rlam, rmu, nparts, d_triangle, d_trinorm, d_source, ifsingle == 1, d_sigma_sl,
                            ifdouble == 1, d_sigma_dl, ifptfrc == 1, d_ptfrc, ifstrain == 1, d_strain, ntargs,
                            d_target, ifptfrctarg == 1, d_ptfrctarg, ifstraintarg == 1, d_straintarg,
                            (hipStream_t)stream, false);
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

int elfmm_gfx950_batch_create(int iprec, double rlam, double rmu, int nmesh, const int *nparts,
                              const double *d_triangle, const double *d_trinorm, const double *d_source,
                              int ifsingle, int ifdouble, int ifptfrc, int ifstrain, const int *ntargs,
                              const double *d_target, int ifptfrctarg, int ifstraintarg, int width, void **batch)
{
    if (!batch) return 16;
    *batch = nullptr;
    try {
        Batch *B = nullptr;
        int ier = batch_create(iprec, rlam, rmu, nmesh, nparts, d_triangle, d_trinorm, d_source, ifsingle == 1,
                               ifdouble == 1, ifptfrc == 1, ifstrain == 1, ntargs, d_target, ifptfrctarg == 1,
                               ifstraintarg == 1, width, &B);
        *batch = B;
        return ier;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

int elfmm_gfx950_batch_buffers(void *batch, double **d_sigma_sl, double **d_sigma_dl, double **d_ptfrc,
                               double **d_strain, double **d_ptfrctarg, double **d_straintarg)
{
    if (!batch) return 16;
    Batch &B = *(Batch *)batch;
    if (d_sigma_sl) *d_sigma_sl = B.ssl;
    if (d_sigma_dl) *d_sigma_dl = B.sdl;
    if (d_ptfrc) *d_ptfrc = B.pt;
    if (d_strain) *d_strain = B.st;
    if (d_ptfrctarg) *d_ptfrctarg = B.ptt;
    if (d_straintarg) *d_straintarg = B.stt;
    return 0;
}

int elfmm_gfx950_batch_apply(void *batch, const double *d_sigma_sl, const double *d_sigma_dl, double *d_ptfrc,
                             double *d_strain, double *d_ptfrctarg, double *d_straintarg, void *stream)
{
    if (!batch) return 16;
    Batch &B = *(Batch *)batch;
    int cur = 0;
    if (hipGetDevice(&cur) != hipSuccess || cur != B.dev) return 16;
    try {
        std::lock_guard<std::mutex> lk(B.mu);
        hipStream_t s = (hipStream_t)stream;
        size_t nT = B.ntri, nG = B.ntgt;
        auto in = [&](double *dst, const double *src, size_t cnt) {
            if (dst && src && src != dst) HIPOK(hipMemcpyAsync(dst, src, cnt * 8, hipMemcpyDeviceToDevice, s));
        };
        auto outc = [&](double *dst, const double *src, size_t cnt) {
            if (dst && src && src != dst && cnt) HIPOK(hipMemcpyAsync(dst, src, cnt * 8, hipMemcpyDeviceToDevice, s));
        };
        if (B.ifsl) in(B.ssl, d_sigma_sl, 3 * nT);
        if (B.ifdl) in(B.sdl, d_sigma_dl, 3 * nT);
        batch_launch(B, s);
        outc(d_ptfrc, B.pt, 3 * nT);
        outc(d_strain, B.st, 9 * nT);
        outc(d_ptfrctarg, B.ptt, 3 * nG);
        outc(d_straintarg, B.stt, 9 * nG);
        return 0;
    } catch (const HipFailure &) {
        return 32;
    } catch (const std::bad_alloc &) {
        return 8;
    }
}

int elfmm_gfx950_batch_schedule(void *batch, int *width, int *graph, int ntune, double *tune)
{
    if (!batch) return -1;
    Batch &B = *(Batch *)batch;
    std::lock_guard<std::mutex> lk(B.mu);
    if (width) *width = B.width;
    if (graph) *graph = B.graph_mode;
    int nt = (int)B.tune.size() / 3;
    if (tune)
        for (int i = 0; i < std::min(nt, ntune) * 3; i++) tune[i] = B.tune[i];
    return nt;
}

int elfmm_gfx950_batch_destroy(void *batch)
{
    if (!batch) return 0;
    Batch *B = (Batch *)batch;
    int cur = 0;
    if (hipGetDevice(&cur) != hipSuccess || cur != B->dev) return 16;
    delete B;
    return 0;
}

void elfmm_gfx950_last_timings(double *ms16)
{
    for (int i = 0; i < 16; i++) ms16[i] = g_times[i];
}

void elfmm_gfx950_last_stats(double *st16)
{
    for (int i = 0; i < 16; i++) st16[i] = g_stats[i];
}

int elfmm_gfx950_octree_dev(const double *d_source, int n, const double *d_target, int nt, int nbox, int imindlin,
                            int *sizes, void *stream)
{
    try {
        if (n < 1 || nt < 0 || nbox < 1 || (nt && !d_target)) return -16;
        if (!g_ws) g_ws = new Workspace();
        Workspace &W = *g_ws;
        if (!W.oct) W.oct.reset(new OctreeWork());
        if (!g_oct_tree) g_oct_tree = new Tree();
        bool deep = false;
        HIPOK(build_tree_dev(d_source, n, d_target, nt, nbox, imindlin ? 1 : 0, *g_oct_tree, *W.oct,
                             (hipStream_t)stream, deep));
        if (deep) return -4;
        const Tree &T = *g_oct_tree;
        if (sizes) {
            sizes[0] = T.nboxes;
            sizes[1] = T.nlev;
            for (int t = 1; t <= 5; t++) sizes[1 + t] = (int)T.litems[t].size();
        }
        return T.nboxes;
    } catch (const HipFailure &) {
        return -32;
    } catch (const std::bad_alloc &) {
        return -8;
    }
}

void elfmm_gfx950_octree_get(int *boxes, double *centers, int *iz, int *iztarg, int *lstart, int *litems)
{
    if (!g_oct_tree) return;
    const Tree &T = *g_oct_tree;
    for (int b = 0; b < T.nboxes; b++) {
        int *o = boxes + 18 * b;
        o[0] = T.level[b];
        for (int d = 0; d < 3; d++) o[1 + d] = T.ijk[3 * b + d];
        o[4] = T.parent[b];
        o[5] = T.nkids[b];
        o[6] = T.src_start[b];
        o[7] = T.src_count[b];
        o[8] = T.tgt_start[b];
        o[9] = T.tgt_count[b];
        for (int q = 0; q < 8; q++) o[10 + q] = T.kids[8 * b + q];
    }
    std::memcpy(centers, T.centers.data(), 3 * sizeof(double) * T.nboxes);
    std::memcpy(iz, T.iz.data(), sizeof(int) * T.iz.size());
    if (!T.iztarg.empty()) std::memcpy(iztarg, T.iztarg.data(), sizeof(int) * T.iztarg.size());
    for (int t = 1; t <= 5; t++) {
        std::memcpy(lstart, T.lstart[t].data(), sizeof(int) * (T.nboxes + 1));
        lstart += T.nboxes + 1;
        if (!T.litems[t].empty()) std::memcpy(litems, T.litems[t].data(), sizeof(int) * T.litems[t].size());
        litems += T.litems[t].size();
    }
}

int elfmm_gfx950_expansion_order(int iprec)
{
    if (iprec < -2 || iprec > 3) return -1;
    return expansion_order(iprec_eps(iprec));
}

const char *elfmm_gfx950_version(void) { return "elfmm_gfx950 0.1 (gfx950, FP64)"; }

}  // extern "C"
