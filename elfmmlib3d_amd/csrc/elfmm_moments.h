// P2M and P2L of triangles: device code of elfmm_gpu.hip, which includes this
// file inside its namespace after the tables it reads (g_fact, g_sdfact), NRHS
// and gemm_d4. Tests build it for the host, a thread per lane, with the wave
// operations emulated.
#pragma once

// degree and order of packed coefficient index c = l*(l+1)/2 + m
__device__ __forceinline__ void coef_nk(int c, int &n, int &k)
{
    n = (int)((sqrt(8.0 * c + 1.0) - 1.0) * 0.5);
    while ((n + 1) * (n + 2) / 2 <= c) n++;
    while (n * (n + 1) / 2 > c) n--;
    k = c - n * (n + 1) / 2;
}


// 1/sqrt((l+m)! (l-m)!): the factor between the integer-coefficient
// harmonics V below and the normalised R_l^m / I_l^m.
__device__ __forceinline__ double hnorm(int l, int m)
{
    m = m < 0 ? -m : m;
    return 1.0 / sqrt(g_fact[l + m] * g_fact[l - m]);
}


// The rules of 6 and 12 nodes, one after the other: w (1, u, v) and (u, v) of
// each node.
struct QMom {
    double m[18][5];
};
constexpr QMom make_qmom()
{
    constexpr double rule[18][3] = {ELFMM_RULE4, ELFMM_RULE6};
    QMom q{};
    for (int i = 0; i < 18; i++) {
        q.m[i][0] = rule[i][2];
        q.m[i][1] = rule[i][2] * rule[i][0];
        q.m[i][2] = rule[i][2] * rule[i][1];
        q.m[i][3] = rule[i][0];
        q.m[i][4] = rule[i][1];
    }
    return q;
}
__constant__ QMom c_qmom = make_qmom();

// ---- P2M and P2L of triangles ---------------------------------------------
// The 12 (or 6) nodes of a triangle carry densities that are linear over it,
// so the node sums go through three moments of the triangle per harmonic,
//   U_j = sum_nodes omega (1, u, v)_j B(node),
// and the 16 moment columns of p2x_body are sums of coefficient x U_j over the
// triangles (k_tcoef: problems 0-2 take U_0 alone, problem 3 all three): per
// triangle and coefficient 12 x 11 + 3 x 32 operations instead of
// 12 x (8 + 32). B is V without the factor (-1)^m (2l-1)!!:
//   B_m^m = ((x + iy) / r^(2 IRR))^m r^(-IRR),
//   B_l   = zz B_{l-1} - beta rr B_{l-2},
//   beta  = (l+m-1)(l-m-1) / ((2l-1)(2l-3)).
// A lane holds the recurrences of half a triangle's nodes (NH) for the column
// pair c: order m = c (degrees c..ph), then m = ph - c (degrees ph - c..ph),
// ph + 2 steps for every c, so all lanes are busy throughout; the half is that
// of the wave, so that its rule's constants are scalars. tc triangles at a
// time, S steps at a time: the lanes write their partial moments to LDS, then
// the waves take 16-row tiles of the slice, K = 3 tc moments (the halves are
// added on the way in), 16 columns, accumulators in registers for all slices
// (NS slices x RT tiles per wave). The start values of all columns come from
// one table of powers per node. Bound by FP64 issue (11 operations per node,
// step and lane) and the two barriers of a slice. Against one product per node
// (which point sources and rules of 1 and 3 nodes keep: three moments are no
// fewer than their nodes): 81,920 triangles + 100,000 targets, iprec 2, P2L
// 3.71 -> 1.89 ms, nodes and P2M 1.36 -> 0.83 ms; 20,480 + 20,480 at iprec 3, P2L
// 5.03 -> 2.17 ms; 27,380 + 20,011 at iprec 1, P2L 1.36 -> 0.32 ms.

// Coefficients of the 16 columns and 3 moments of every triangle,
// [triangle][moment][column], 2 x area folded in: the densities of k_nodes.
__global__ void k_tcoef(int n, const double *__restrict__ tri_s, const double *__restrict__ nrm_s,
                        const double *__restrict__ ssl_s, const double *__restrict__ sdl_s, int ifsl, int ifdl,
                        double rmu, double c1, double c2, double dls, double *__restrict__ tcoef)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double t[9], nv[3], sl[3], dl[3];
    for (int d = 0; d < 9; d++) t[d] = tri_s[9 * (size_t)i + d];
    for (int d = 0; d < 3; d++) {
        nv[d] = nrm_s[3 * (size_t)i + d];
        sl[d] = ifsl ? ssl_s[3 * (size_t)i + d] : 0.0;
        dl[d] = ifdl ? dls * sdl_s[3 * (size_t)i + d] : 0.0;
    }
    double ax = t[3] - t[0], ay = t[4] - t[1], az = t[5] - t[2];
    double bx = t[6] - t[0], by = t[7] - t[1], bz = t[8] - t[2];
    double cx = ay * bz - az * by, cy = az * bx - ax * bz, cz = ax * by - ay * bx;
    double w = sqrt(cx * cx + cy * cy + cz * cz);    // 2 x area
    double *o = tcoef + (size_t)i * 48;
    for (int j = 0; j < 3; j++) {
        o[j] = w * (sl[j] / (2 * rmu));
        for (int d = 0; d < 3; d++) o[4 + 3 * j + d] = w * ((nv[d] * dl[j] + dl[d] * nv[j]) / 2);
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
    o[3] = w * cv[0];
    for (int d = 0; d < 3; d++) o[13 + d] = w * dv[0][d];
    for (int j = 1; j < 3; j++) {
        for (int q = 0; q < 13; q++) o[16 * j + q] = 0.0;
        o[16 * j + 3] = w * (cv[j] - cv[0]);
        for (int d = 0; d < 3; d++) o[16 * j + 13 + d] = w * (dv[j][d] - dv[0][d]);
    }
}

// The same for the Mindlin moments of one layer, whose sums are the same with
// other columns (the 20,020-triangle fault mesh: 0.33 ms for both layers, 1.38
// from the 12 nodes' harmonics per triangle; the densities of
// elfmm_mindlin.hip, k_mind_moments): values v (single layer: sigma_sl; double:
// the six sym-pairs of sigma_dl and the normal) in columns 0.., y3 v behind
// them, y3 = the node's height, linear over the triangle.
__global__ void k_mind_tcoef(int n, int dl, const double *__restrict__ tri_s, const double *__restrict__ nrm_s,
                             const double *__restrict__ den_s, double *__restrict__ tcoef)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double *t = tri_s + 9 * (size_t)i, *b = den_s + 3 * (size_t)i, *nv = nrm_s + 3 * (size_t)i;
    double ax = t[3] - t[0], ay = t[4] - t[1], az = t[5] - t[2];
    double bx = t[6] - t[0], by = t[7] - t[1], bz = t[8] - t[2];
    double cx = ay * bz - az * by, cy = az * bx - ax * bz, cz = ax * by - ay * bx;
    double w = sqrt(cx * cx + cy * cy + cz * cz);    // 2 x area
    double v[6] = {b[0], b[1], b[2], 0.0, 0.0, 0.0};
    if (dl) {
        v[0] = b[0] * nv[0];
        v[1] = b[1] * nv[1];
        v[2] = b[2] * nv[2];
        v[3] = b[0] * nv[1] + b[1] * nv[0];
        v[4] = b[0] * nv[2] + b[2] * nv[0];
        v[5] = b[1] * nv[2] + b[2] * nv[1];
    }
    const double y3[3] = {t[2], t[5] - t[2], t[8] - t[2]};
    double *o = tcoef + (size_t)i * 48;
    const int nv_ = dl ? 6 : 3;
    for (int j = 0; j < 3; j++)
        for (int q = 0; q < 16; q++)
            o[16 * j + q] = q < nv_ ? (j ? 0.0 : w * v[q]) : (q < 2 * nv_ ? w * y3[j] * v[q - nv_] : 0.0);
}

// Shape of a launch: waves per workgroup, steps per slice, most slices, most
// column pairs, nodes per half triangle; the row tiles of a slice go to the
// waves in RT rounds (in the last of NS slices one step is left at most where
// RT > 1: one round). TC triangles per chunk are KS K-steps. The padded row
// count of a moment in LDS is twice an odd number, so that the lanes' 16-byte
// writes of different triangles meet different banks.
template <int WB_, int S_, int NS_, int NP_, int NH_>
struct P2TShape {
    static constexpr int WB = WB_, S = S_, NS = NS_, NP = NP_, NH = NH_;
    static constexpr int ROWS = (NP * S * 2 + 15) / 16 * 16, STRIDE = ROWS + 2, RT = (ROWS / 16 + WB - 1) / WB;
    static constexpr int TC = 32 * WB / NP, KS = (3 * TC + 3) / 4, HS = 4 * KS * STRIDE, NT = 64 * WB;
    static constexpr bool fits(int ph) { return (ph + 2) / 2 <= NP && ph + 2 <= (NS - 1) * S + (RT > 1 ? 1 : S); }
    // doubles of dynamic LDS: U (before it the powers, at the end the
    // moments), second columns' start values, zz and rr of the nodes,
    // recurrence constants, source boxes and triangles
    static constexpr int imax(int a, int b) { return a > b ? a : b; }
    static constexpr int ubuf(int ph) { return imax(imax(2 * HS, TC * 2 * NH * (ph + 1) * 2), 4 * NS * ROWS); }
    static constexpr int lds(int ph) { return ubuf(ph) + 2 * NH * NT + 4 * TC * NH + (ph + 2) * NP + (65 + 64 + TC + 1) / 2; }
};
// iprec 0 (order 9, 6 nodes), 1 (14), 2 (26), 3 (39): the least waves whose
// accumulators fit 256 registers a lane, so that the small leaves of the low
// orders do not leave lanes idle
using P2TShape0 = P2TShape<2, 4, 4, 6, 3>;
using P2TShape1 = P2TShape<2, 4, 5, 8, 6>;
using P2TShape2 = P2TShape<4, 4, 8, 14, 6>;
using P2TShape3 = P2TShape<8, 3, 14, 21, 6>;
static_assert(P2TShape0::fits(10) && P2TShape1::fits(15) && P2TShape2::fits(27) && P2TShape3::fits(40), "P2L's degrees");
// The shape for degree ph and nq nodes, -1 if none fits.
inline int p2t_shape(int ph, int nq)
{
    if (nq == 6) return P2TShape0::fits(ph) ? 0 : -1;
    if (nq != 12) return -1;
    return P2TShape1::fits(ph) ? 1 : (P2TShape2::fits(ph) ? 2 : (P2TShape3::fits(ph) ? 3 : -1));
}

// Where the moments themselves are wanted (MIND, the Mindlin P2M): column c16
// to col[c16] of G, [box of the list][MCOLS][coefficient], harmonics
// Racah-normalised and unscaled, added with atomics; -1: column not wanted.
struct MindMoments {
    int col[16];
    double2 *G;
    static constexpr int MCOLS = 18;
};

// Workgroup b of P2M takes part b, (box of the list, its first triangle,
// triangles), the whole of box b of the list if there are no parts; a part of
// a box adds its coefficients with atomics.
// lds: Z::lds() doubles, 16-byte aligned (16-byte accesses)
template <bool IRR, class Z, bool MIND>
__device__ __forceinline__ void p2t_body(int p, const int *__restrict__ boxes, const int *__restrict__ parts,
                                         MindMoments mind, const int *__restrict__ lstart,
                                         const int *__restrict__ litems, const double *__restrict__ centers,
                                         const double *__restrict__ sides, const int *__restrict__ src_start,
                                         const int *__restrict__ src_count, const double *__restrict__ tri_s,
                                         const double *__restrict__ tcoef, int nc, double *__restrict__ expn, double *lds)
{
    constexpr int WB = Z::WB, S = Z::S, NS = Z::NS, NP = Z::NP, NH = Z::NH, RT = Z::RT, TC = Z::TC, KS = Z::KS;
    constexpr int ROWS = Z::ROWS, STRIDE = Z::STRIDE, HS = Z::HS, NT = Z::NT;
    constexpr int NQ = 2 * NH, Q0 = NH == 6 ? 6 : 0;
    const int ph = IRR ? p + 1 : p, nst = ph + 2, npair = (ph + 2) / 2, ubuf = Z::ubuf(ph);
    double *U = lds;                                  // [half][moment k][row]; before it the powers; at the end the moments
    double2 *st2 = reinterpret_cast<double2 *>(lds + ubuf);                 // [node][thread]: second column's start
    double2 *zr = st2 + NH * NT;                      // [triangle][node]: zz, rr
    double *beta = reinterpret_cast<double *>(zr + TC * NQ);                // [step][c]: recurrence constant after the step
    // triangles before each source box of a pass, its first triangle, the chunk's triangles
    int *pre = reinterpret_cast<int *>(beta + nst * NP), *first = pre + 65, *tidx = first + 64;
    int tid = threadIdx.x, lane = tid & 63;
    int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int kq = lane >> 4, n16 = lane & 15;
    int half = 2 * wave / WB;                         // of the triangle's nodes
    int hl = tid - half * 32 * WB, c = hl / TC, mt = hl - c * TC;
    int len1 = ph + 1 - c;
    const int bi = !IRR && parts ? parts[3 * blockIdx.x] : (int)blockIdx.x, box = boxes[bi];
    const int part0 = !IRR && parts ? parts[3 * blockIdx.x + 1] : 0;
    const int partn = !IRR && parts ? parts[3 * blockIdx.x + 2] : src_count[box];
    const bool whole = IRR || partn == src_count[box];
    double side = sides[box], is = 1.0 / side;
    double cx = centers[3 * box], cy = centers[3 * box + 1], cz = centers[3 * box + 2];
    for (int e = tid; e < ubuf; e += NT) lds[e] = 0.0;   // rows that no lane writes stay finite
    for (int e = tid; e < nst * NP; e += NT) {
        int s = e / NP, cc = min(e - s * NP, npair - 1), l1 = ph + 1 - cc;
        int m = s < l1 ? cc : ph - cc, l = s < l1 ? cc + s : m + s - l1;
        beta[e] = (double)((l + m) * (l - m)) / (double)((2 * l + 1) * (2 * l - 1));
    }
    gemm_d4 acc[NS][RT];
#pragma unroll
    for (int i = 0; i < NS; i++)
#pragma unroll
        for (int r = 0; r < RT; r++) acc[i][r] = gemm_d4{0.0, 0.0, 0.0, 0.0};
    int b0 = IRR ? lstart[blockIdx.x] : 0, b1 = IRR ? lstart[blockIdx.x + 1] : 1;
    for (; b0 < b1; b0 += 64) {
        __syncthreads();                              // the previous pass is done with pre, first
        if (wave == 0) {
            int cnt = 0, s0 = 0;
            if (b0 + lane < b1) {
                int sbox = IRR ? litems[b0 + lane] : box;
                s0 = src_start[sbox] + part0;
                cnt = IRR ? src_count[sbox] : partn;
            }
            int end = cnt;
            for (int off = 1; off < 64; off <<= 1) {
                int v = __shfl_up(end, off);
                if (lane >= off) end += v;
            }
            if (lane == 0) pre[0] = 0;
            pre[lane + 1] = end;
            first[lane] = s0;
        }
        __syncthreads();
        int total = pre[64];
        for (int t0 = 0; t0 < total; t0 += TC) {
            int cnt = min(TC, total - t0), ks_n = (3 * cnt + 3) / 4;
            // start values: the powers of every node, one node per thread
            for (int e = tid; e < cnt * NQ; e += NT) {
                int tt = e / NQ, q = e - tt * NQ, t = t0 + tt;
                int lo = 0, hi = 63;                  // pre[lo] <= t < pre[lo + 1]
                while (lo < hi) {
                    int mid = (lo + hi + 1) >> 1;
                    if (pre[mid] <= t) lo = mid;
                    else hi = mid - 1;
                }
                int i = first[lo] + t - pre[lo];
                if (q == 0) tidx[tt] = i;
                const double *v = tri_s + 9 * (size_t)i;
                double uu = c_qmom.m[Q0 + q][3], vv = c_qmom.m[Q0 + q][4];
                double x = (v[0] + uu * (v[3] - v[0]) + vv * (v[6] - v[0]) - cx) * is;
                double y = (v[1] + uu * (v[4] - v[1]) + vv * (v[7] - v[1]) - cy) * is;
                double zc = (v[2] + uu * (v[5] - v[2]) + vv * (v[8] - v[2]) - cz) * is;
                double r2 = x * x + y * y + zc * zc, ir2 = IRR ? 1.0 / r2 : 1.0;
                double ur = x * ir2, ui = y * ir2, dr = IRR ? sqrt(ir2) : 1.0, di = 0.0;
                zr[e] = double2{zc * ir2, IRR ? ir2 : r2};
                double2 *pw = reinterpret_cast<double2 *>(U) + (size_t)e * (ph + 1);
                for (int m = 0; m <= ph; m++) {
                    pw[m] = double2{dr, di};
                    double t2 = dr * ur - di * ui;
                    di = dr * ui + di * ur;
                    dr = t2;
                }
            }
            __syncthreads();
            bool on = c < npair && mt < cnt;
            double r1r[NH], r1i[NH], r2r[NH], r2i[NH], zz[NH], rr[NH];
#pragma unroll
            for (int q = 0; q < NH; q++) {
                r1r[q] = r1i[q] = r2r[q] = r2i[q] = zz[q] = rr[q] = 0.0;
                if (on) {
                    int e = mt * NQ + half * NH + q;
                    const double2 *pw = reinterpret_cast<const double2 *>(U) + (size_t)e * (ph + 1);
                    double2 a = pw[c], g = zr[e];
                    r1r[q] = a.x;
                    r1i[q] = a.y;
                    zz[q] = g.x;
                    rr[q] = g.y;
                    st2[q * NT + tid] = pw[ph - c];
                }
            }
            double a[KS];                         // coefficients: column n16, moment 4 ks + kq
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                int k = 4 * ks + kq, tt = k / 3;
                a[ks] = tt < cnt ? tcoef[((size_t)tidx[tt] * 3 + (k - 3 * tt)) * 16 + n16] : 0.0;
            }
            __syncthreads();                          // the powers have been read
            double *Uw = U + half * HS + 3 * mt * STRIDE + 2 * c;
            // one step: moments of the current terms (xr, xi) to LDS, the next
            // terms over the previous ones (yr, yi)
            auto gen_step = [&](int s, int st, double (&xr)[NH], double (&xi)[NH], double (&yr)[NH], double (&yi)[NH]) {
                if (s == len1) {
#pragma unroll
                    for (int q = 0; q < NH; q++) {
                        double2 b = st2[q * NT + tid];
                        xr[q] = b.x;
                        xi[q] = b.y;
                    }
                }
                double be = beta[s * NP + c];
                double m0r = 0.0, m0i = 0.0, m1r = 0.0, m1i = 0.0, m2r = 0.0, m2i = 0.0;
#pragma unroll
                for (int q = 0; q < NH; q++) {
                    const double *wm = c_qmom.m[Q0 + half * NH + q];
                    double w = wm[0], wu = wm[1], wv = wm[2];
                    m0r = fma(w, xr[q], m0r);
                    m0i = fma(w, xi[q], m0i);
                    m1r = fma(wu, xr[q], m1r);
                    m1i = fma(wu, xi[q], m1i);
                    m2r = fma(wv, xr[q], m2r);
                    m2i = fma(wv, xi[q], m2i);
                    double g = be * rr[q];
                    yr[q] = fma(zz[q], xr[q], -g * yr[q]);
                    yi[q] = fma(zz[q], xi[q], -g * yi[q]);
                }
                double *o = Uw + st * 2 * NP;
                *reinterpret_cast<double2 *>(o) = double2{m0r, m0i};
                *reinterpret_cast<double2 *>(o + STRIDE) = double2{m1r, m1i};
                *reinterpret_cast<double2 *>(o + 2 * STRIDE) = double2{m2r, m2i};
            };
#pragma unroll
            for (int sl = 0; sl < NS; sl++) {
                int s0 = sl * S, sn = min(S, nst - s0);
                if (sn <= 0) continue;
                if (on) {
#pragma unroll
                    for (int st = 0; st < S; st++) {
                        if (st >= sn) break;
                        // the current terms sit in r1 at even steps, in r2 at odd ones
                        if ((sl * S + st) & 1) gen_step(s0 + st, st, r2r, r2i, r1r, r1i);
                        else gen_step(s0 + st, st, r1r, r1i, r2r, r2i);
                    }
                }
                __syncthreads();
                int nt = (2 * NP * sn + 15) / 16;
#pragma unroll
                for (int r = 0; r < (sl == NS - 1 ? 1 : RT); r++) {
                    int tile = wave + WB * r;
                    if (tile >= nt) continue;
                    const double *b = U + 16 * tile + n16 + kq * STRIDE;
#pragma unroll
                    for (int ks = 0; ks < KS; ks++) {
                        if (ks >= ks_n) break;
                        const double *bk = b + 4 * ks * STRIDE;
                        acc[sl][r] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ks], bk[0] + bk[HS], acc[sl][r], 0, 0, 0);
                    }
                }
                __syncthreads();
            }
        }
    }
    if (MIND) {
        const int nown = (p + 1) * (p + 2) / 2;
#pragma unroll
        for (int sl = 0; sl < NS; sl++)
#pragma unroll
            for (int rt = 0; rt < (sl == NS - 1 ? 1 : RT); rt++) {
                int row = 16 * (wave + WB * rt) + n16, st = row / (2 * NP), rem = row - st * 2 * NP, cc = rem >> 1;
                int s = sl * S + st, l1 = ph + 1 - cc;
                bool second = s >= l1;
                if (row >= ROWS || st >= S || s >= nst || cc >= npair || (second && 2 * cc == ph)) continue;
                int m = second ? ph - cc : cc, l = second ? m + s - l1 : cc + s;
                double f = pow(side, (double)l) * hnorm(l, m) * g_sdfact[l] * ((l + m) & 1 ? -1.0 : 1.0);
                double *o = (double *)(mind.G + (size_t)bi * MindMoments::MCOLS * nown + l * (l + 1) / 2 + m) + (rem & 1);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    int col = mind.col[kq + 4 * i];
                    if (col >= 0) unsafeAtomicAdd(o + (size_t)2 * col * nown, f * acc[sl][rt][i]);
                }
            }
        return;
    }
    // coefficients, one right-hand side at a time, as p2x_body; moment (col,
    // degree ll, order mm) at slice s / S, step s % S, column pair c
    int nco = (p + 1) * (p + 2) / 2;
    double f0s = IRR ? is : 1.0;
    double f1s = IRR ? is * is : is;
    double *Ms = lds;
    constexpr int MSZ = NS * ROWS;
    for (int r = 0; r < NRHS; r++) {
        __syncthreads();
#pragma unroll
        for (int sl = 0; sl < NS; sl++)
#pragma unroll
            for (int rt = 0; rt < (sl == NS - 1 ? 1 : RT); rt++) {
                int tile = wave + WB * rt;
                if (16 * tile >= ROWS) continue;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    int c16 = kq + 4 * i;
                    int col = c16 == r ? 0 : (c16 >= 4 && (c16 - 4) / 3 == r ? 1 + (c16 - 4) % 3 : -1);
                    if (col >= 0) Ms[col * MSZ + sl * ROWS + 16 * tile + n16] = acc[sl][rt][i];
                }
            }
        __syncthreads();
        auto mget = [&](int col, int ll, int mm, double &re, double &im) {
            int am = mm < 0 ? -mm : mm;
            if (ll < 0 || ll > ph || am > ll) {
                re = 0.0;
                im = 0.0;
                return;
            }
            int cc = min(am, ph - am), s = am == cc ? ll - am : ph + 1 - cc + ll - am;
            const double *o = Ms + col * MSZ + s / S * ROWS + s % S * 2 * NP + 2 * cc;
            re = o[0];
            im = o[1];
            if (mm < 0) re = -re;
        };
        for (int cf = tid; cf < nco; cf += NT) {
            int l, m;
            coef_nk(cf, l, m);
            int ld = IRR ? l + 1 : l - 1;
            // (-1)^m (2l-1)!! of the moments' degree: V = that x B; orders m +- 1 carry the other sign
            double sg = ((l + m) & 1) ? -1.0 : 1.0;
            double v0 = sg * g_sdfact[l], v1 = ld >= 0 ? ((ld + l) & 1 ? -sg : sg) * g_sdfact[ld] : 0.0;
            double fh = hnorm(l, m) * f0s * v0, fp, fm, fz;
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
            fp *= -0.5 * f1s * v1;
            fm *= -0.5 * f1s * v1;
            fz *= f1s * v1;
            double qr, qi, xpr, xpi, ypr, ypi, xmr, xmi, ymr, ymi, zr_, zi_;
            mget(0, l, m, qr, qi);
            mget(1, ld, m + 1, xpr, xpi);
            mget(2, ld, m + 1, ypr, ypi);
            mget(1, ld, m - 1, xmr, xmi);
            mget(2, ld, m - 1, ymr, ymi);
            mget(3, ld, m, zr_, zi_);
            double re = fh * qr + fp * (xpr + ypi) + fm * (ymi - xmr) + fz * zr_;
            double im = -fh * qi + fp * (ypr - xpi) + fm * (xmi + ymr) - fz * zi_;
            double *e = expn + ((size_t)box * NRHS + r) * nc + 2 * cf;
            if (IRR) {
                e[0] += re;
                e[1] += im;
            } else if (whole) {
                e[0] = re;
                e[1] = im;
            } else {
                unsafeAtomicAdd(e, re);
                unsafeAtomicAdd(e + 1, im);
            }
        }
    }
}
