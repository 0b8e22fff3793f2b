// Host planner, part 2: the task lists of one apply, built from the octree
// on the host worker pool.
//
// Which boxes take part in each step follows the reference's
// lfmm3dtrilhesstargmain (src/lfmm3dtrilhess.f:517-1215) and lfmm3d_list2
// (src/lfmm3drouts.f:297-496): multipoles of sourced leaves at level >= 2,
// M2M/L2L between sourced boxes, M2L over list 2 from level 2 down (target
// boxes without targets pruned when no source outputs are requested), P2L
// over list 4, M2T over list 3, L2T at leaves of level >= 2, near field over
// self + list 1. Each translation step is grouped by operator so that one
// dense matrix serves many (source, destination) pairs.
#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "elfmm_internal.h"

namespace elfmm {
namespace {

void add_pairs(GemmLaunch &g, int64_t a_off, int h, double phi, const int *src, const int *dst, const double *scale,
               int np, int refl = 0)
{
    int base = (int)g.src.size();
    g.src.insert(g.src.end(), src, src + np);
    g.dst.insert(g.dst.end(), dst, dst + np);
    g.scale.insert(g.scale.end(), scale, scale + np);
    for (int p0 = 0; p0 < np; p0 += ML_P)
        for (int r0 = 0; r0 < h; r0 += ML_M)
            g.tiles.push_back({a_off, h, r0, base + p0, std::min(ML_P, np - p0), phi, refl});
}

// Launch order of translation tiles: workgroup b of a launch runs on XCD
// b % 8 and takes tiles[b]. Tiles of one operator are cut into runs, the
// runs go heaviest first to the least loaded XCD (work of a tile: its K
// extent h plus the output adds, worth about 40 coefficients), and each
// XCD takes its runs highest order first, so every XCD ends at about the
// same time and an operator's tiles stay together in one XCD's L2.
// Slots past an XCD's last tile hold empty tiles (npair = 0).
void xcd_order(std::vector<M2LTile> &tiles)
{
    constexpr int NX = 8;
    if (tiles.size() < 2 * NX) return;
    auto work = [](const M2LTile &t) { return t.h + 40.0; };
    double total = 0;
    for (auto &t : tiles) total += work(t);
    double cap = total / (NX * 16);
    struct Run {
        size_t b, e;
        double w;
        int h;
    };
    std::vector<Run> runs;
    for (size_t i = 0; i < tiles.size(); i++) {
        if (runs.empty() || tiles[i].a_off != tiles[runs.back().b].a_off || runs.back().w >= cap)
            runs.push_back({i, i, 0.0, tiles[i].h});
        runs.back().e = i + 1;
        runs.back().w += work(tiles[i]);
    }
    std::vector<int> by_w(runs.size());
    for (size_t r = 0; r < runs.size(); r++) by_w[r] = (int)r;
    std::stable_sort(by_w.begin(), by_w.end(), [&](int a, int b) { return runs[a].w > runs[b].w; });
    std::vector<int> bin[NX];
    double load[NX] = {0};
    for (int r : by_w) {
        int x = (int)(std::min_element(load, load + NX) - load);
        load[x] += runs[r].w;
        bin[x].push_back(r);
    }
    size_t nmax = 0;
    std::vector<M2LTile> seq[NX];
    for (int x = 0; x < NX; x++) {
        std::stable_sort(bin[x].begin(), bin[x].end(), [&](int a, int b) {
            return runs[a].h != runs[b].h ? runs[a].h > runs[b].h : a < b;
        });
        for (int r : bin[x]) seq[x].insert(seq[x].end(), tiles.begin() + runs[r].b, tiles.begin() + runs[r].e);
        nmax = std::max(nmax, seq[x].size());
    }
    M2LTile empty{0, 0, 0, 0, 0, 0.0};
    tiles.assign(nmax * NX, empty);
    for (int x = 0; x < NX; x++)
        for (size_t i = 0; i < seq[x].size(); i++) tiles[i * NX + x] = seq[x][i];
}

// octant of child c in parent b: bit d set when c is the upper half in d
inline int octant(const Tree &T, int c, int b)
{
    int o = 0;
    for (int d = 0; d < 3; d++)
        if (T.ijk[3 * c + d] != 2 * (T.ijk[3 * b + d] - 1) + 1) o |= 1 << d;
    return o;
}

inline int offset_index(const Tree &T, int j, int b)
{
    return (T.ijk[3 * j] - T.ijk[3 * b] + 3) * 49 + (T.ijk[3 * j + 1] - T.ijk[3 * b + 1] + 3) * 7 +
           (T.ijk[3 * j + 2] - T.ijk[3 * b + 2] + 3);
}

// M2M (up) or L2L (down) launch for one level: pairs grouped by octant.
GemmLaunch tree_pass(const Tree &T, int lev, int nc, const double *oct_phi, bool up)
{
    int h = nc / 2, p = 0;
    while (ncoef(p) < nc) p++;
    const int64_t oper = (int64_t)trans_doubles(p);
    GemmLaunch g;
    std::vector<int> s[8], d[8];
    for (int b = T.laddr[2 * lev]; b < T.laddr[2 * lev] + T.laddr[2 * lev + 1]; b++) {
        if (!T.nkids[b] || (up && T.src_count[b] == 0)) continue;
        for (int q = 0; q < T.nkids[b]; q++) {
            int c = T.kids[8 * b + q];
            if (up && T.src_count[c] == 0) continue;
            int o = octant(T, c, b);
            s[o].push_back(up ? c : b);
            d[o].push_back(up ? b : c);
        }
    }
    for (int o = 0; o < 8; o++)
        if (!s[o].empty()) {
            std::vector<double> one(s[o].size(), 1.0);
            add_pairs(g, o * oper, h, oct_phi[o], s[o].data(), d[o].data(), one.data(),
                      (int)s[o].size());
        }
    xcd_order(g.tiles);
    return g;
}

constexpr int CHUNK = 64;

// Split each slot's task range [off[s], off[s+1]) into evaluation wave tasks
// of at most EW_PTS points: (slot, first task, count) triples.
template <class I>
void wave_tasks(const std::vector<I> &off, std::vector<int> &wt)
{
    wt.clear();
    for (size_t s = 0; s + 1 < off.size(); s++)
        for (I t = off[s]; t < off[s + 1]; t += EW_PTS) {
            wt.push_back((int)s);
            wt.push_back((int)t);
            wt.push_back((int)std::min<I>(EW_PTS, off[s + 1] - t));
        }
}

// P2M workgroups: a box's triangles are a chain of chunks of 8 to 12, so where
// the boxes are too few to fill the device (iter leaves hold up to 240
// triangles) they are cut into equal parts, about P2M_WG of them, none under
// P2M_MIN triangles (a part's coefficients cost about as much as three
// triangles). A fault mesh of 20,020 triangles: the whole half-space product
// 5.15 ms, 6.2 with a workgroup per box and the Mindlin moments per node.
void p2m_parts(const Tree &T, Plan &P)
{
    constexpr int64_t P2M_WG = 1024, P2M_MIN = 18;
    int64_t total = 0;
    for (int b : P.p2m_boxes) total += T.src_count[b];
    const int64_t per = std::max(P2M_MIN, (total + P2M_WG - 1) / P2M_WG);
    for (size_t i = 0; i < P.p2m_boxes.size(); i++) {
        int64_t c = T.src_count[P.p2m_boxes[i]], k = (int64_t)P.p2m_boxes.size() >= P2M_WG ? 1 : (c + per - 1) / per;
        for (int64_t j = 0; j < k; j++) {
            int a = (int)(c * j / k), e = (int)(c * (j + 1) / k);
            for (int v : {(int)i, a, e - a}) P.p2m_parts.push_back(v);
        }
    }
}

// Order of n entries by decreasing weight, equal weights in their order.
std::vector<int> heaviest_first(const std::vector<double> &w)
{
    std::vector<std::pair<double, int>> k(w.size());
    for (size_t i = 0; i < w.size(); i++) k[i] = {-w[i], (int)i};
    std::sort(k.begin(), k.end());
    std::vector<int> o(w.size());
    for (size_t i = 0; i < w.size(); i++) o[i] = k[i].second;
    return o;
}

}  // namespace

void build_plan_near(const Tree &T, bool src_eval, bool direct_only, bool iter, Plan &P)
{
    int nb = T.nboxes;
    auto npts = [&](int b) { return (src_eval ? T.src_count[b] : 0) + T.tgt_count[b]; };
    P.nf_boxes.clear();
    P.nf_start.assign(1, 0);
    P.nf_items.clear();
    P.nf_ntri.clear();
    P.stats[6] = 0;
    if (direct_only) return;
    // leaves: near field over self + list 1. With iter, lists 3 and 4 join
    // the near field; the reference evaluates a box's list 4 at every point
    // below it, so a leaf also takes the list 4 of each of its ancestors and
    // every point is handled once, by its leaf.
    auto each = [&](int b, auto &&f) {
        for (int q = T.lstart[1][b]; q < T.lstart[1][b + 1]; q++)
            if (int j = T.litems[1][q]; T.src_count[j]) f(j);
        if (T.src_count[b]) f(b);
        if (!iter) return;
        for (int q = T.lstart[3][b]; q < T.lstart[3][b + 1]; q++)
            if (int j = T.litems[3][q]; T.src_count[j]) f(j);
        for (int a = b; a >= 0; a = T.parent[a])
            for (int q = T.lstart[4][a]; q < T.lstart[4][a + 1]; q++)
                if (int j = T.litems[4][q]; T.src_count[j]) f(j);
    };
    // entries and triangles of every box's list, by chunks of boxes
    std::vector<int> items(nb, 0), tris(nb, 0);
    int nchunk = (nb + CHUNK - 1) / CHUNK;
    parallel_chunks(nchunk, [&](int ch, int) {
        for (int b = ch * CHUNK; b < std::min(nb, (ch + 1) * CHUNK); b++)
            if (!T.nkids[b] && npts(b))
                each(b, [&](int j) {
                    items[b]++;
                    tris[b] += T.src_count[j];
                });
    });
    std::vector<int> box;
    std::vector<double> w;
    for (int b = 0; b < nb; b++)
        if (items[b]) {
            box.push_back(b);
            w.push_back((double)tris[b] * npts(b));
        }
    // heaviest (points x triangles) first, so the long boxes do not start last
    std::vector<int> ord = heaviest_first(w);
    int nq = (int)box.size();
    P.nf_boxes.resize(nq);
    P.nf_start.resize(nq + 1);
    P.nf_ntri.resize(nq);
    double npair_near = 0;
    for (int q = 0; q < nq; q++) {
        int b = P.nf_boxes[q] = box[ord[q]];
        P.nf_start[q + 1] = P.nf_start[q] + items[b];
        P.nf_ntri[q] = tris[b];
        npair_near += w[ord[q]];
    }
    P.nf_items.resize(P.nf_start[nq]);
    parallel_chunks((nq + CHUNK - 1) / CHUNK, [&](int ch, int) {
        for (int q = ch * CHUNK; q < std::min(nq, (ch + 1) * CHUNK); q++) {
            int k = P.nf_start[q];
            each(P.nf_boxes[q], [&](int j) { P.nf_items[k++] = j; });
        }
    });
    P.stats[6] = npair_near;
}

// Lanes per point of each near box: the power of two that costs the box the
// least time, waves x (steps per wave + 1): the last step and the last wave
// of a box run partly idle, and setting a wave up and adding its lanes costs
// about a step (20 points, 135 triangles: 2 waves x 35 at 4 lanes, 3 x 18 at
// 8, 5 x 10 at 16, 10 x 6 at 32). A call too small to give the device
// NF_WAVES waves that way starts from more lanes per point: 217 points
// against 180 triangles took 205 us as one workgroup per leaf.
void near_tasks(const Tree &T, const Plan &P, bool src_eval, std::vector<int> &tasks)
{
    constexpr int NF_WAVES = 2048;                   // 256 CUs x 4 SIMDs x 2
    auto npts = [&](int b) { return (src_eval ? T.src_count[b] : 0) + T.tgt_count[b]; };
    int nq = (int)P.nf_boxes.size();
    double total = 0;
    for (int b : P.nf_boxes) total += npts(b);
    int low = 0;                                     // log2 of the lanes per point
    while (low < 6 && total * (1 << low) < NF_WAVES * 64.0) low++;
    std::vector<int> start(nq + 1, 0);
    std::vector<unsigned char> lanes(nq);
    for (int q = 0; q < nq; q++) {
        int64_t np = npts(P.nf_boxes[q]), cost = 0;
        for (int k = low; k <= 6; k++) {
            int64_t c = (((np << k) + 63) >> 6) * (((P.nf_ntri[q] + (1 << k) - 1) >> k) + 1);
            if (!cost || c < cost) lanes[q] = (unsigned char)k, cost = c;
        }
        start[q + 1] = start[q] + (int)(((np << lanes[q]) + 63) >> 6);
    }
    tasks.resize(3 * (size_t)start[nq]);
    for (int q = 0; q < nq; q++)
        for (int k = 0; k < start[q + 1] - start[q]; k++) {
            int *t = &tasks[3 * (size_t)(start[q] + k)];
            t[0] = q;
            t[1] = 64 * k;
            t[2] = 1 << lanes[q];
        }
}

void plan_reset(Plan &P)
{
    for (std::vector<int> *v : {&P.p2m_boxes, &P.p2m_parts, &P.p2l_boxes, &P.p2l_start, &P.p2l_items, &P.m2t_items, &P.l2t_boxes,
                                &P.nf_boxes, &P.nf_start, &P.nf_items, &P.nf_ntri, &P.l2t_tpt, &P.m2t_slot_box,
                                &P.m2t_tpt, &P.l2t_wt, &P.m2t_wt, &P.m2t_bt})
        v->clear();
    P.sides.clear();
    P.m2m_l.clear();
    P.l2l_l.clear();
    P.m2l.tiles.clear();
    P.m2l_tiles.clear();
    for (double &v : P.stats) v = 0;
}

void build_plan(const Tree &T, int n, const Operators *ops, bool src_eval, bool direct_only, int nrhs,
                Plan &P, bool iter)
{
    plan_reset(P);
    build_plan_near(T, src_eval, direct_only, iter, P);
    build_plan_far(T, n, ops, src_eval, nrhs, P, iter);
}

void build_plan_far(const Tree &T, int n, const Operators *ops, bool src_eval, int nrhs, Plan &P, bool iter)
{
    build_plan_up(T, ops, P, iter);
    build_plan_m2l(T, ops, src_eval, nrhs, P);
    build_plan_eval(T, n, ops, src_eval, P, iter);
}

void build_plan_up(const Tree &T, const Operators *ops, Plan &P, bool iter)
{
    int nb = T.nboxes;
    P.sides.resize(nb);
    for (int b = 0; b < nb; b++) P.sides[b] = T.box_side.empty() ? T.size / (double)(1 << T.level[b]) : T.box_side[b];
    P.stats[0] = nb;
    P.stats[1] = T.nlev;
    P.stats[2] = ops ? ops->p : 0;
    P.p2l_start.assign(1, 0);
    if (!ops) return;
    // M2M children at lev+1 -> parents at lev, for lev = nlev-1 .. 2, the P2M
    // leaves and the P2L lists side by side
    int nup = std::max(0, T.nlev - 2);
    std::vector<GemmLaunch> up(nup);
    parallel_chunks(nup + 2, [&](int task, int) {
        if (task >= 2) {
            up[task - 2] = tree_pass(T, T.nlev - 1 - (task - 2), ncoef(ops->p), ops->oct_phi, true);
        } else if (task == 1) {
            std::vector<int> bx;
            std::vector<double> w;
            for (int b = 0; b < nb; b++)
                if (!T.nkids[b] && T.level[b] >= 2 && T.src_count[b] > 0) {
                    bx.push_back(b);
                    w.push_back(T.src_count[b]);
                }
            // one workgroup per box, most sources first
            for (int q : heaviest_first(w)) P.p2m_boxes.push_back(bx[q]);
            p2m_parts(T, P);
        } else if (!iter) {
            // P2L: local of box j from the sources of i with j in list3(i)
            // (src/lfmm3dtrilhess.f:760-829); owner j, sources list4(j).
            // Heaviest first: one workgroup per box, so the longest ones
            // start first and the launch ends evenly.
            std::vector<int> bx;
            std::vector<double> w;
            for (int j = 0; j < nb; j++) {
                double n4 = 0;
                for (int q = T.lstart[4][j]; q < T.lstart[4][j + 1]; q++) n4 += T.src_count[T.litems[4][q]];
                if (n4 > 0) {
                    bx.push_back(j);
                    w.push_back(n4);
                }
            }
            for (int q : heaviest_first(w)) {
                int j = bx[q];
                P.p2l_boxes.push_back(j);
                for (int k = T.lstart[4][j]; k < T.lstart[4][j + 1]; k++)
                    if (T.src_count[T.litems[4][k]]) P.p2l_items.push_back(T.litems[4][k]);
                P.p2l_start.push_back((int)P.p2l_items.size());
            }
        }
    });
    double m2m_pairs = 0;
    for (GemmLaunch &g : up) {
        if (g.tiles.empty()) continue;
        m2m_pairs += g.src.size();
        P.m2m_l.push_back(std::move(g));
    }
    P.stats[8] = m2m_pairs;
    P.stats[10] = (double)P.p2m_boxes.size();
    P.stats[11] = (double)P.p2l_items.size();
}

void build_plan_m2l(const Tree &T, const Operators *ops, bool src_eval, int nrhs, Plan &P)
{
    int nb = T.nboxes;
    int p = ops ? ops->p : 0;
    int nchunk = (nb + CHUNK - 1) / CHUNK;
    if (!ops) {
        P.m2l.src.clear();
        P.m2l.dst.clear();
        P.m2l.scale.clear();
        return;
    }
    {
        // M2L over list 2, grouped by offset: per-chunk counts by offset,
        // then every chunk fills its slice of each offset's run, so the
        // pairs of one offset stay in increasing target-box order.
        std::vector<int> cnt(343 * (size_t)nchunk, 0);
        auto m2l_target = [&](int b) { return T.level[b] >= 2 && (src_eval || T.tgt_count[b] > 0); };
        parallel_chunks(nchunk, [&](int ch, int) {
            int *c = &cnt[343 * (size_t)ch];
            for (int b = ch * CHUNK; b < std::min(nb, (ch + 1) * CHUNK); b++) {
                if (!m2l_target(b)) continue;
                for (int q = T.lstart[2][b]; q < T.lstart[2][b + 1]; q++) {
                    int j = T.litems[2][q];
                    if (T.src_count[j]) c[offset_index(T, j, b)]++;
                }
            }
        });
        std::vector<int> ostart(344, 0);
        for (int o = 0; o < 343; o++) {
            int run = ostart[o];
            for (int ch = 0; ch < nchunk; ch++) {
                int v = cnt[343 * (size_t)ch + o];
                cnt[343 * (size_t)ch + o] = run;
                run += v;
            }
            ostart[o + 1] = run;
        }
        int npair = ostart[343];
        // the pair arrays keep the previous plan's memory (plan_reset): the
        // fill below writes every entry, so no allocation or clearing here
        std::vector<int> &ps = P.m2l.src, &pd = P.m2l.dst;
        std::vector<double> &psc = P.m2l.scale;
        ps.resize(npair);
        pd.resize(npair);
        psc.resize(npair);
        parallel_chunks(nchunk, [&](int ch, int) {
            int *pos = &cnt[343 * (size_t)ch];
            for (int b = ch * CHUNK; b < std::min(nb, (ch + 1) * CHUNK); b++) {
                if (!m2l_target(b)) continue;
                double isb = 1.0 / P.sides[b];
                for (int q = T.lstart[2][b]; q < T.lstart[2][b + 1]; q++) {
                    int j = T.litems[2][q];
                    if (!T.src_count[j]) continue;
                    int k = pos[offset_index(T, j, b)]++;
                    ps[k] = j;
                    pd[k] = b;
                    psc[k] = isb;
                }
            }
        });
        // work counts: the flops of dense operators (what orders below
        // m2l_turned_h execute) and the reference's point-and-shoot count per
        // pair and right-hand side, two rotations
        // R(p) = 4 sum (2n+1)^2 and a z-shift Z(p) = 6 sum_j sum_k (p+1-|k|)
        std::vector<double> alg_m2l(p + 1, 0.0);
        for (int pt = 0; pt <= p; pt++) {
            double R = 0, Z = 0;
            for (int a = 0; a <= pt; a++) R += 4.0 * (2 * a + 1) * (2 * a + 1);
            for (int jj = 0; jj <= pt; jj++)
                for (int kk = -jj; kk <= jj; kk++) Z += 6.0 * (pt + 1 - std::abs(kk));
            alg_m2l[pt] = 2 * R + Z;
        }
        double dense = 0, alg = 0;
        // the pairs are already in offset order; tiles per offset cover
        // ML_P pairs by ML_M coefficients of that offset's rotated operator.
        // Offsets sharing an operator lay out their tiles together (tile
        // slot order: offsets by operator), so that xcd_order keeps them in
        // one run.
        std::vector<int> oord(343);
        for (int o = 0; o < 343; o++) oord[o] = o;
        std::stable_sort(oord.begin(), oord.end(), [&](int a, int b) { return ops->m2l_off[a] < ops->m2l_off[b]; });
        std::vector<int64_t> tstart(343, 0);
        int64_t ntile = 0;
        for (int q = 0; q < 343; q++) {
            int o = oord[q];
            int m = ostart[o + 1] - ostart[o];
            int h = ncoef(ops->m2l_pt[o]) / 2;
            tstart[o] = ntile;
            ntile += m ? (int64_t)((m + ML_P - 1) / ML_P) * ((h + ML_M - 1) / ML_M) : 0;
            if (!m) continue;
            // two real h x h products per pair and right-hand side
            dense += m * 2.0 * 2.0 * h * (double)h * nrhs;
            alg += m * alg_m2l[ops->m2l_pt[o]] * nrhs;
        }
        P.m2l_tiles.resize(ntile);
        parallel_chunks(343, [&](int o, int) {
            int m = ostart[o + 1] - ostart[o];
            if (!m) return;
            int h = ncoef(ops->m2l_pt[o]) / 2;
            M2LTile *t = &P.m2l_tiles[tstart[o]];
            for (int p0 = 0; p0 < m; p0 += ML_P)
                for (int r0 = 0; r0 < h; r0 += ML_M)
                    *t++ = M2LTile{ops->m2l_off[o], h, r0, ostart[o] + p0, std::min(ML_P, m - p0), ops->m2l_phi[o],
                                   ops->m2l_refl[o]};
        });
        // L2L parents at lev -> children, for lev = 2 .. nlev-1, beside the
        // launch order of the M2L tiles
        int ndown = std::max(0, T.nlev - 2);
        std::vector<GemmLaunch> down(ndown);
        parallel_chunks(ndown + 1, [&](int task, int) {
            if (task) down[task - 1] = tree_pass(T, 1 + task, ncoef(p), ops->oct_phi, false);
            else xcd_order(P.m2l_tiles);
        });
        double l2l_pairs = 0;
        for (GemmLaunch &g : down) {
            if (g.tiles.empty()) continue;
            l2l_pairs += g.src.size();
            P.l2l_l.push_back(std::move(g));
        }
        P.stats[3] = npair;
        P.stats[4] = dense;
        P.stats[5] = alg;
        P.stats[7] = (double)std::count_if(P.m2l_tiles.begin(), P.m2l_tiles.end(), [](const M2LTile &t) { return t.npair > 0; });
        P.stats[9] = l2l_pairs;
    }
}

void build_plan_eval(const Tree &T, int n, const Operators *ops, bool src_eval, Plan &P, bool iter)
{
    int nb = T.nboxes;
    auto npts = [&](int b) { return (src_eval ? T.src_count[b] : 0) + T.tgt_count[b]; };
    // L2T: the leaves with points at level >= 2
    for (int b = 0; b < nb; b++)
        if (!T.nkids[b] && npts(b) && ops && T.level[b] >= 2) P.l2t_boxes.push_back(b);

    // evaluation tasks: L2T one per point of each leaf; M2T one per (point,
    // list-3 box), grouped by the box whose field operand is read
    auto fill_points = [&](int b, int *tp) {
        int k = 0;
        if (src_eval)
            for (int i = T.src_start[b]; i < T.src_start[b] + T.src_count[b]; i++, k++) tp[k] = i;
        for (int i = T.tgt_start[b]; i < T.tgt_start[b] + T.tgt_count[b]; i++, k++) tp[k] = n + i;
    };
    {
        int nl = (int)P.l2t_boxes.size();
        std::vector<int> off(nl + 1, 0);
        for (int q = 0; q < nl; q++) off[q + 1] = off[q] + npts(P.l2t_boxes[q]);
        P.l2t_tpt.resize(off[nl]);
        parallel_chunks((nl + CHUNK - 1) / CHUNK, [&](int ch, int) {
            for (int q = ch * CHUNK; q < std::min(nl, (ch + 1) * CHUNK); q++)
                fill_points(P.l2t_boxes[q], &P.l2t_tpt[off[q]]);
        });
        wave_tasks(off, P.l2t_wt);
    }
    // M2T: multipole of i at the points of j with j in list4(i)
    // (src/lfmm3dtrilhess.f:864-981): a slot per sourced box i, its owners the
    // boxes with points of list 4, the dual of list 3
    if (ops && !iter) {
        std::vector<int> ostart(1, 0);
        std::vector<int64_t> toff(1, 0);
        for (int i = 0; i < nb; i++) {
            if (!T.src_count[i]) continue;
            int64_t t = 0;
            for (int q = T.lstart[4][i]; q < T.lstart[4][i + 1]; q++) {
                int j = T.litems[4][q];
                if (!npts(j)) continue;
                P.m2t_items.push_back(j);
                t += npts(j);
            }
            if (!t) continue;
            P.m2t_slot_box.push_back(i);
            ostart.push_back((int)P.m2t_items.size());
            toff.push_back(toff.back() + t);
        }
        int ns = (int)P.m2t_slot_box.size();
        const std::vector<int> &owners = P.m2t_items;
        P.m2t_tpt.resize(toff[ns]);
        parallel_chunks((ns + CHUNK - 1) / CHUNK, [&](int ch, int) {
            for (int sl = ch * CHUNK; sl < std::min(ns, (ch + 1) * CHUNK); sl++) {
                int64_t at = toff[sl];
                for (int k = ostart[sl]; k < ostart[sl + 1]; k++) {
                    fill_points(owners[k], &P.m2t_tpt[at]);
                    at += npts(owners[k]);
                }
            }
        });
        wave_tasks(toff, P.m2t_wt);
        // workgroups of up to 4 consecutive wave tasks of one slot
        int nw = (int)P.m2t_wt.size() / 3;
        for (int w = 0; w < nw; w++)
            if (w == 0 || P.m2t_wt[3 * w] != P.m2t_wt[3 * (w - 1)] || w - P.m2t_bt.back() == 4) P.m2t_bt.push_back(w);
        if (nw) P.m2t_bt.push_back(nw);
    }
    P.stats[12] = (double)P.m2t_items.size();
    P.stats[13] = (double)P.l2t_boxes.size();
}

std::vector<int> mind_proxy_offsets(int *index)
{
    std::vector<int> v;
    for (int o = 0; o < 343; o++) {
        int i = o / 49 - 3, j = o / 7 % 7 - 3, k = o % 7 - 3;
        bool near = std::abs(k) <= 1 && (std::abs(i) > 1 || std::abs(j) > 1);
        index[o] = near ? (int)v.size() / 3 : -1;
        if (near) v.insert(v.end(), {i, j, k});
    }
    return v;
}

void build_mindlin_plan(const Tree &T, const Operators &ops, MindlinPlan &MP)
{
    int px[343];
    mind_proxy_offsets(px);
    MP = MindlinPlan();
    int nb = T.nboxes;
    MP.pw_slot.assign(nb, -1);
    for (int b = 0; b < nb; b++) {
        if (T.level[b] < 2 || !T.src_count[b]) continue;
        MP.src_boxes.push_back(b);
        MP.pw_slot[b] = MP.npw++;
        if (T.nkids[b] && T.level[b] < 64) MP.b_scale_boxes[T.level[b]].push_back(b);
    }
    std::vector<int> cnt(343, 0);
    std::vector<std::pair<int, int>> near_pairs;   // (offset, pair index)
    std::vector<int> ns, nd;
    MP.far_start.push_back(0);
    for (int b = 0; b < nb; b++) {
        if (T.level[b] < 2 || !T.tgt_count[b]) continue;
        int nfar = 0;
        for (int q = T.lstart[2][b]; q < T.lstart[2][b + 1]; q++) {
            int j = T.litems[2][q];
            if (!T.src_count[j]) continue;
            // z offset of target and source centres in box sides (src/lfmm3droutsmindlin.f:329-333)
            double side = T.size / (double)(1 << T.level[j]);
            double zdis = (T.centers[3 * b + 2] - T.centers[3 * j + 2]) / side;
            if (std::fabs(zdis) < 1.5) {
                int o = offset_index(T, j, b);
                near_pairs.push_back({o, (int)ns.size()});
                ns.push_back(j);
                nd.push_back(b);
            } else {
                MP.far_items.push_back(j);
                nfar++;
            }
        }
        if (nfar) {
            MP.far_boxes.push_back(b);
            MP.far_start.push_back((int)MP.far_items.size());
        }
    }
    // near pairs grouped by offset, tiles of the full-order operators
    std::stable_sort(near_pairs.begin(), near_pairs.end(),
                     [](const std::pair<int, int> &a, const std::pair<int, int> &b) { return a.first < b.first; });
    GemmLaunch &g = MP.m2l;
    for (size_t k = 0; k < near_pairs.size();) {
        size_t e = k;
        while (e < near_pairs.size() && near_pairs[e].first == near_pairs[k].first) e++;
        int o = near_pairs[k].first;
        std::vector<int> s(e - k), d(e - k);
        std::vector<double> sc(e - k);
        for (size_t i = k; i < e; i++) {
            s[i - k] = ns[near_pairs[i].second];
            d[i - k] = nd[near_pairs[i].second];
            sc[i - k] = (double)(1 << T.level[d[i - k]]) / T.size;
        }
        int h = ncoef(ops.m2l_pt[o]) / 2;
        for (size_t i = k; i < e; i += MIND_PX)
            for (int v : {px[o], (int)i, (int)std::min<size_t>(MIND_PX, e - i)}) MP.px_tasks.push_back(v);
        add_pairs(g, ops.m2l_off[o], h, ops.m2l_phi[o], s.data(), d.data(), sc.data(), (int)(e - k), ops.m2l_refl[o]);
        k = e;
    }
    MP.m2l_tiles = g.tiles;
}

void build_forest(const std::vector<const Tree *> &trees, const std::vector<int> &soff, const std::vector<int> &toff,
                  Tree &F)
{
    F = Tree();
    int nt = (int)trees.size();
    int L = 0;
    for (const Tree *t : trees) L = std::max(L, t->nlev);
    // new id of box b of tree k: level-major, trees in order within a level
    std::vector<std::vector<int>> nid(nt);
    std::vector<std::pair<int, int>> order;                 // (tree, box) by new id
    F.laddr.clear();
    for (int lev = 0; lev <= L; lev++) {
        int first = (int)order.size();
        for (int k = 0; k < nt; k++) {
            const Tree &T = *trees[k];
            if (nid[k].empty()) nid[k].assign(T.nboxes, -1);
            if (lev > T.nlev) continue;
            for (int b = T.laddr[2 * lev]; b < T.laddr[2 * lev] + T.laddr[2 * lev + 1]; b++) {
                nid[k][b] = (int)order.size();
                order.push_back({k, b});
            }
        }
        F.laddr.push_back(first);
        F.laddr.push_back((int)order.size() - first);
    }
    int nb = (int)order.size();
    F.nboxes = nb;
    F.nlev = L;
    F.level.resize(nb);
    F.ijk.resize(3 * (size_t)nb);
    F.parent.resize(nb);
    F.kids.assign(8 * (size_t)nb, -1);
    F.nkids.resize(nb);
    F.src_start.resize(nb);
    F.src_count.resize(nb);
    F.tgt_start.resize(nb);
    F.tgt_count.resize(nb);
    F.centers.resize(3 * (size_t)nb);
    F.box_side.resize(nb);
    for (int t = 1; t <= 5; t++) F.lstart[t].assign(nb + 1, 0);
    for (int q = 0; q < nb; q++) {
        int k = order[q].first, b = order[q].second;
        const Tree &T = *trees[k];
        F.level[q] = T.level[b];
        for (int d = 0; d < 3; d++) {
            F.ijk[3 * q + d] = T.ijk[3 * b + d];
            F.centers[3 * q + d] = T.centers[3 * b + d];
        }
        F.parent[q] = T.parent[b] < 0 ? -1 : nid[k][T.parent[b]];
        F.nkids[q] = T.nkids[b];
        for (int c = 0; c < T.nkids[b]; c++) F.kids[8 * q + c] = nid[k][T.kids[8 * b + c]];
        F.src_start[q] = soff[k] + T.src_start[b];
        F.src_count[q] = T.src_count[b];
        F.tgt_start[q] = toff[k] + T.tgt_start[b];
        F.tgt_count[q] = T.tgt_count[b];
        F.box_side[q] = T.size / (double)(1 << T.level[b]);
        for (int t = 1; t <= 5; t++) F.lstart[t][q + 1] = F.lstart[t][q] + T.lstart[t][b + 1] - T.lstart[t][b];
    }
    for (int t = 1; t <= 5; t++) {
        F.litems[t].resize(F.lstart[t][nb]);
        parallel_chunks((nb + 255) / 256, [&](int ch, int) {
            for (int q = ch * 256; q < std::min(nb, (ch + 1) * 256); q++) {
                int k = order[q].first, b = order[q].second;
                const Tree &T = *trees[k];
                int o = F.lstart[t][q];
                for (int e = T.lstart[t][b]; e < T.lstart[t][b + 1]; e++) F.litems[t][o++] = nid[k][T.litems[t][e]];
            }
        });
    }
    int ns = 0, ng = 0;
    for (int k = 0; k < nt; k++) {
        ns = std::max(ns, soff[k] + (int)trees[k]->iz.size());
        ng = std::max(ng, toff[k] + (int)trees[k]->iztarg.size());
    }
    F.iz.resize(ns);
    F.iztarg.resize(ng);
    for (int k = 0; k < nt; k++) {
        const Tree &T = *trees[k];
        for (size_t i = 0; i < T.iz.size(); i++) F.iz[soff[k] + i] = soff[k] + T.iz[i];
        for (size_t i = 0; i < T.iztarg.size(); i++) F.iztarg[toff[k] + i] = toff[k] + T.iztarg[i];
    }
}

}  // namespace elfmm
