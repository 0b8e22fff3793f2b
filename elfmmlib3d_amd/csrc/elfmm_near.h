// One near-field (point, triangle) pair in one pass over the three edges:
// the pair code of the near-field kernel (also compiled for the host, where
// tests compare it with nf_pair of elfmm_math.h, which the direct sum keeps).
//
// Same integrals as nf_pair (src/elfmm3dtria.f:1689-2009, 2368-2905), less
// work:
//   - the distances to the three vertices are computed once (each edge's
//     primitives and the solid angle use them), 3 square roots a pair, and
//     the edges' tangents come from the record;
//   - the primitives int t^m / (t^2 + rho^2)^(q/2) of an edge follow from the
//     two distances without a branch on the foot point's side: with
//     A = r + |t| at both ends and opp = foot point inside the edge,
//       K01 = log(A1 A2 / rho^2)             (opp), log(max A / min A) (else),
//             as log(1 + x), x a sum of terms of one sign: A1 A2 - rho^2 =
//             r1 |t2| + r2 |t1| + |t1 t2| + (r1^2 r2^2 - rho^4) / (r1 r2 + rho^2),
//             max A - min A = L + |t1 + t2| L / (r1 + r2), so K01 ~ L/R keeps its digits
//             at distances R >> L (the sums over the edges lose R/L of them, not
//             (R/L)^2: 6.0e-15 of a single layer's displacement at R = 8 L, 2.0e-14
//             from the ratio's logarithm, measured against long double)
//       K03 = 2 L (r1 + r2) A1 A2 / (r1 r2 E),
//             E = rho^2 (A1 + A2)^2 (opp), (A1 A2 + rho^2)^2 (else)
//       3 K25 = K03 (u1^2 + u1 u2 + u2^2),  u = t / r
//       3 K05 = K03 (1/r1^2 + 1/r2^2 + (1 - u1 u2) / rho^2),
//             (1 - u1 u2) / rho^2 = P / (rho^2 r1 r2) (opp),
//             (t1^2 + t2^2 + rho^2) / (r1 r2 P) (else),  P = r1 r2 + |t1 t2|
//     (K03 = (u2 - u1) / rho^2 by the half-angle form of the difference of
//     two sines), every term of one sign, so a point near an edge's line
//     keeps its digits;
//   - of the integral tensors only the entries that the densities meet are
//     formed, the others from Laplace(1/r) = 0 and Laplace(r) = 2/r, e.g.
//     sum_l int d_l d_l d_a r = 2 int d_a (1/r);
//   - the layers and the strain are template parameters.
#pragma once

#include "elfmm_math.h"

namespace elfmm {

// 1/x and 1/sqrt(x) for x > 0: the hardware estimate and one third-order step
// (to the last bit or two) on the device.
ELFMM_HD double nf_rcp(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double y = __builtin_amdgcn_rcp(x);
    double e = fma(-x, y, 1.0);
    return fma(y, fma(e, e, e), y);
#else
    return 1.0 / x;
#endif
}
ELFMM_HD double nf_rsqrt(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double y = __builtin_amdgcn_rsq(x);
    double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
#else
    return 1.0 / sqrt(x);
#endif
}

// log(1 + x), x >= 0: the rounding of 1 + x given back to first order.
ELFMM_HD double nf_log1p(double x)
{
    double u = 1.0 + x;
    return log(u) + (x - (u - 1.0)) * nf_rcp(u);
}

// Sums over the edges, in the triangle's frame (z normal), w = -z0.
struct NearSums {
    double F, r1x, r1y;                              // K01: del, n_x, n_y
    double b2xx, b2xy, b2yy;                         // int d_i d_j r
    double xxx, xxy, xyy, yyy, xxz, xyz, yyz;        // int d_i d_j d_k r (xxz, xyz, yyz without the factor w)
    double k3x, k3y, k3d, qxx, qxy;                  // K03: n_x, n_y, del; -int d_x d_x, d_x d_y of 1/r
    double x4xx, x4xy, x4yy, y4yy;                   // int d_i d_j d_k d_z r over w, jk in the plane
    double x4xz, x4yz, y4yz;                         // int d_i d_j d_z d_z r
};

template <bool SL, bool DL, bool ST>
ELFMM_HD void near_edge(double sx, double sy, double L, double t1, double del, double w, double w2, double r1,
                        double ir1, double r2, double ir2, NearSums &S)
{
    const double nx = sy, ny = -sx, p = sx * sy, sy2 = sy * sy, sx2 = sx * sx;
    double t2 = t1 + L, del2 = del * del, rho2 = del2 + w2;
    bool opp = t1 < 0.0 && t2 > 0.0;
    double a1 = t1 < 0.0 ? -t1 : t1, a2 = t2 < 0.0 ? -t2 : t2;
    double A1 = r1 + a1, A2 = r2 + a2, A12 = A1 * A2, sum = r1 + r2, i12 = ir1 * ir2;
    double k11 = L * (t1 + t2) * nf_rcp(sum);
    // K01
    double r12 = r1 * r2, a12 = a1 * a2;
    double x1 = (rho2 * (a1 * a1 + a2 * a2) + a12 * a12) * nf_rcp(r12 + rho2) + (r1 * a2 + r2 * a1 + a12);
    double x2 = L + (k11 < 0.0 ? -k11 : k11);
    double irho2 = nf_rcp(opp ? rho2 : (A1 > A2 ? A2 : A1));
    double k01 = nf_log1p((opp ? x1 : x2) * irho2);
    double nxk = nx * k01, dk = del * k01;
    S.F += dk;
    S.r1x += nxk;
    S.r1y += ny * k01;
    if (SL) {
        S.b2xx += p * k11 + sy2 * dk;
        S.b2xy += sy2 * k11 - p * dk;
        S.b2yy += sx2 * dk - p * k11;
    }
    if (!ST && !DL) return;
    // orders 3 of r and 2 of 1/r: K03, K13
    double k13 = k11 * i12;
    double e = opp ? A1 + A2 : A12 + rho2;
    e = e * e * (opp ? rho2 : 1.0);
    double k03 = 2.0 * L * sum * A12 * i12 * nf_rcp(e);
    double k3n = nx * k03, k3y = ny * k03, g3 = del * k03;
    {
        // D_ij = delta_ij K01 - int u_i u_j / r^3 in the edge's frame (s, n, z)
        double ss = rho2 * k03, sn = del * k13, nn = k01 - del * g3, d = ss - nn;
        double xx = sx2 * d + nn - 2.0 * p * sn;
        double yy = ss + nn - xx;
        S.xxx += nx * xx;
        S.xyy += nx * yy;
        double xy = p * d - (sy2 - sx2) * sn;
        S.xxy += nx * xy;
        S.yyy += ny * yy;
        double xz = -sx * k13 - nx * g3, yz = -sy * k13 - ny * g3;
        S.xxz += nx * xz;
        S.xyz += nx * yz;
        S.yyz += ny * yz;
    }
    if (!DL || !ST) return;
    S.k3x += k3n;
    S.k3y += k3y;
    S.k3d += g3;
    S.qxx += p * k13 + sy2 * g3;
    S.qxy += sy2 * k13 - p * g3;
    // order 4 of r: 3 K25 - K03, 3 K15, 3 K05
    double u1 = t1 * ir1, u2 = t2 * ir2, g1 = ir1 * ir1, g2 = ir2 * ir2;
    double P = r12 + a12;
    double M = t1 * t1 + t2 * t2 + rho2;
    double W = opp ? P * irho2 : M * nf_rcp(P);
    double y5 = g1 + g2 + W * i12;                                          // 3 K05 / K03
    double k15 = k13 * (g1 + g2 + i12);                                     // 3 K15
    double ss = k03 * (u1 * u1 + u1 * u2 + u2 * u2 - 1.0), sn = del * k15, nn = k03 * (del2 * y5 - 1.0);
    double d = ss - nn, xx = sx2 * d + nn + 2.0 * p * sn, yy = ss + nn - xx;
    double xy = p * d + (sy2 - sx2) * sn;
    S.x4xx += nx * xx;
    S.x4xy += nx * xy;
    S.x4yy += nx * yy;
    S.y4yy += ny * yy;
    double sz = w2 * k15 - k13, nz = g3 * (w2 * y5 - 1.0);
    double xz = sx * sz + nx * nz, yz = sy * sz + ny * nz;
    S.x4xz += nx * xz;
    S.x4yz += nx * yz;
    S.y4yz += ny * yz;
}

// Accumulates into out: displacement (3) and, with ST, strain (xx yy zz xy xz
// yz) of one pair, global coordinates, times 2 mu (the caller scales the sum).
// rec: NF_REC words of nf_make_record.
template <bool SL, bool DL, bool ST>
ELFMM_HD void near_pair(const double *rec, const double *P, int iself, double rlam, double rmu, double c1, double *out)
{
    double x0, y0, z0;
    nf_local_point(rec, P, x0, y0, z0);
    z0 = iself ? 0.0 : z0;                            // the principal value at the triangle's own centroid
    const double a = rec[12], b = rec[13], c = rec[14], w = -z0, w2 = z0 * z0;
    double xb = x0 - a, xc = x0 - b, yc = y0 - c;
    double yz2 = y0 * y0 + w2;
    double qa = x0 * x0 + yz2, qb = xb * xb + yz2, qc = xc * xc + yc * yc + w2;
    double ia = nf_rsqrt(qa), ib = nf_rsqrt(qb), ic = nf_rsqrt(qc);
    double la = qa * ia, lb = qb * ib, lc = qc * ic;
    NearSums S = {};
    near_edge<SL, DL, ST>(1.0, 0.0, a, -x0, y0, w, w2, la, ia, lb, ib, S);
    {
        double iL = rec[21], sx = (b - a) * iL, sy = c * iL;
        near_edge<SL, DL, ST>(sx, sy, (b - a) * sx + c * sy, -(xb * sx + y0 * sy), y0 * sx - xb * sy, w, w2, lb, ib,
                              lc, ic, S);
    }
    {
        double iL = rec[22], sx = -b * iL, sy = -c * iL;
        near_edge<SL, DL, ST>(sx, sy, -(b * sx + c * sy), -(xc * sx + yc * sy), yc * sx - xc * sy, w, w2, lc, ic,
                              la, ia, S);
    }
    double wz = 0.0;                                  // the signed solid angle
    if (z0 != 0.0) {
        double ab = x0 * xb + yz2, ac = x0 * xc + y0 * yc + w2, bc = xb * xc + y0 * yc + w2;
        wz = 2.0 * atan2(z0 * a * c, (la * lb + ab) * lc + ac * lb + bc * la);
    }
    const double F = S.F - z0 * wz, r1x = S.r1x, r1y = S.r1y;
    double d0 = 0.0, d1 = 0.0, d2 = 0.0;
    double hxx = 0.0, hxy = 0.0, hxz = 0.0, hyy = 0.0, hyz = 0.0, hzz = 0.0;
    const double xxz = w * S.xxz, xyz = w * S.xyz, yyz = w * S.yyz;
    const double xzz = 2.0 * r1x - S.xxx - S.xyy, yzz = 2.0 * r1y - S.xxy - S.yyy, zzz = 2.0 * wz - xxz - yyz;
    if (SL) {
        const double s0 = rec[15], s1 = rec[16], s2 = rec[17];
        double xz = w * r1x, yz = w * r1y, zz = 2.0 * F - S.b2xx - S.b2yy;
        d0 = 2.0 * s0 * F - c1 * (s0 * S.b2xx + s1 * S.b2xy + s2 * xz);
        d1 = 2.0 * s1 * F - c1 * (s0 * S.b2xy + s1 * S.b2yy + s2 * yz);
        d2 = 2.0 * s2 * F - c1 * (s0 * xz + s1 * yz + s2 * zz);
        if (ST) {
            hxx = c1 * (s0 * S.xxx + s1 * S.xxy + s2 * xxz) - 2.0 * s0 * r1x;
            hxy = c1 * (s0 * S.xxy + s1 * S.xyy + s2 * xyz) - s0 * r1y - s1 * r1x;
            hxz = c1 * (s0 * xxz + s1 * xyz + s2 * xzz) - s0 * wz - s2 * r1x;
            hyy = c1 * (s0 * S.xyy + s1 * S.yyy + s2 * yyz) - 2.0 * s1 * r1y;
            hyz = c1 * (s0 * xyz + s1 * yyz + s2 * yzz) - s1 * wz - s2 * r1y;
            hzz = c1 * (s0 * xzz + s1 * yzz + s2 * zzz) - 2.0 * s2 * wz;
        }
    }
    if (DL) {
        const double s0 = rec[18], s1 = rec[19], s2 = rec[20];
        const double l = (2.0 - 2.0 * c1) * rlam * s2, m = 2.0 * rmu, mc = -2.0 * c1 * rmu;
        double sr = s0 * r1x + s1 * r1y + s2 * wz;
        d0 += l * r1x + mc * (s0 * xxz + s1 * xyz + s2 * xzz) + m * s0 * wz;
        d1 += l * r1y + mc * (s0 * xyz + s1 * yyz + s2 * yzz) + m * s1 * wz;
        d2 += l * wz + mc * (s0 * xzz + s1 * yzz + s2 * zzz) + m * (s2 * wz + sr);
        if (ST) {
            // r: int d_i d_j (1/r); f: int d_i d_j d_k d_z r
            double rxx = -S.qxx, rxy = -S.qxy, rzz = S.k3d, ryy = -rzz - rxx, rxz = -w * S.k3x, ryz = -w * S.k3y;
            double fxxx = w * S.x4xx, fxxy = w * S.x4xy, fxyy = w * S.x4yy, fyyy = w * S.y4yy;
            double fxxz = S.x4xz, fxyz = S.x4yz, fyyz = S.y4yz;
            double fxzz = 2.0 * rxz - fxxx - fxyy, fyzz = 2.0 * ryz - fxxy - fyyy, fzzz = 2.0 * rzz - fxxz - fyyz;
            double vx = s0 * rxx + s1 * rxy + s2 * rxz, vy = s0 * rxy + s1 * ryy + s2 * ryz,
                   vz = s0 * rxz + s1 * ryz + s2 * rzz;
            hxx -= l * rxx + mc * (s0 * fxxx + s1 * fxxy + s2 * fxxz) + m * s0 * rxz;
            hxy -= l * rxy + mc * (s0 * fxxy + s1 * fxyy + s2 * fxyz) + rmu * (s0 * ryz + s1 * rxz);
            hxz -= l * rxz + mc * (s0 * fxxz + s1 * fxyz + s2 * fxzz) + rmu * (s0 * rzz + s2 * rxz + vx);
            hyy -= l * ryy + mc * (s0 * fxyy + s1 * fyyy + s2 * fyyz) + m * s1 * ryz;
            hyz -= l * ryz + mc * (s0 * fxyz + s1 * fyyz + s2 * fyzz) + rmu * (s1 * rzz + s2 * ryz + vy);
            hzz -= l * rzz + mc * (s0 * fxzz + s1 * fyzz + s2 * fzzz) + m * (s2 * rzz + vz);
        }
    }
    const double *U = rec;
    out[0] += U[0] * d0 + U[3] * d1 + U[6] * d2;
    out[1] += U[1] * d0 + U[4] * d1 + U[7] * d2;
    out[2] += U[2] * d0 + U[5] * d1 + U[8] * d2;
    if (ST) {
        // U H U^T, row by row
        double p0 = U[0] * hxx + U[3] * hxy + U[6] * hxz, p1 = U[0] * hxy + U[3] * hyy + U[6] * hyz,
               p2 = U[0] * hxz + U[3] * hyz + U[6] * hzz;
        out[3] += p0 * U[0] + p1 * U[3] + p2 * U[6];
        out[6] += p0 * U[1] + p1 * U[4] + p2 * U[7];
        out[7] += p0 * U[2] + p1 * U[5] + p2 * U[8];
        p0 = U[1] * hxx + U[4] * hxy + U[7] * hxz;
        p1 = U[1] * hxy + U[4] * hyy + U[7] * hyz;
        p2 = U[1] * hxz + U[4] * hyz + U[7] * hzz;
        out[4] += p0 * U[1] + p1 * U[4] + p2 * U[7];
        out[8] += p0 * U[2] + p1 * U[5] + p2 * U[8];
        p0 = U[2] * hxx + U[5] * hxy + U[8] * hxz;
        p1 = U[2] * hxy + U[5] * hyy + U[8] * hyz;
        p2 = U[2] * hxz + U[5] * hyz + U[8] * hzz;
        out[5] += p0 * U[2] + p1 * U[5] + p2 * U[8];
    }
}

}  // namespace elfmm
