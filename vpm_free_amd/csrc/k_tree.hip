// Tree form of the infinite-domain boundary sums (pm.inp "tree = 1"):
//
//   links       : build_level_nbound_3d (pinfdomain.f90:875-1530) — per face, level lev
//                 groups 2^lev x 2^lev face cells; groups that do not fit are "dummy" cells
//                 that only link two finer cells.  The links follow the reference's rules
//                 exactly (including the finer cells those rules leave unreached when both
//                 face extents are not multiples of 2^lev), because the sums must be the
//                 reference's sums.
//   tree sums   : Bounds3d_lev -> calc_boundinf_3d_lev -> tree_calc_3d
//                 (pmbound.f90:980-1250), ibctyp=2; calc_boundinf_3d_lev_s -> tree_calc_3d_s
//                 (pmbound.f90:1255-1481), ibctyp=3 (panel sources, k_tree_eval_s).
//
// Device form.  The forest is flattened on the host into one preorder list per geometry:
// entry e is a (level, cell) node, its children follow it, and skip[e] is the first entry
// after its subtree.  The reference's recursion visits the children of a refined cell in
// link order, depth first — exactly this preorder — so walking the list with "refine:
// e+1, accept: skip[e]" takes the reference's terms.  A wave owns a patch of target nodes and
// walks trees with a wave-uniform cursor (every entry load is a broadcast): a lane that
// accepts a node waits until the cursor has passed that node's subtree while lanes that refine
// descend.  The trees are shared out over the launch (part p the trees p, p + parts, ...) and
// the parts' sums added in their order: one wave per patch over the whole list is some 6000
// entries one after another with two or three waves on a CU, all latency.
//
// The refinement test r < 10 sqrt(DS) decides which terms are taken, so r, the centroids
// and DS are formed with the reference's operation order and no contraction: for
// lattice-aligned centroids r can equal 10 sqrt(DS) to the last bit.  The accepted term
// is s * (DS / r) (the reference forms (s * DS) / r; the two differ in the last bit).
#include <hip/hip_ext.h>

#include <array>
#include <cmath>
#include <map>

#include "bnodes.h"
#include "panel.h"
#include "vpmx_ctx.h"
#include "vpmx_internal.h"

namespace vpmx {

namespace {

struct TreeLink {
    int32_t base;   // first level-0 cell of the group (0-based source index); -1 for a dummy
    int32_t pitch;  // level-0 cells per face row
    int32_t kind;   // +1 group, -1 dummy closing a row, -2 dummy in the closing row of a face
    int32_t ch[4];  // children (indices into the next finer level)
    int32_t nch;
};

// Target patches: work-group w of the evaluation covers tile w; the tiles of face q are
// [off[q], off[q+1]), nu[q] tiles along the face's inner target axis.
struct TreeTiles {
    int off[7];
    int nu[6];
};

struct TreePlan {
    int64_t nb = 0;
    int64_t nent = 0;
    TreeTiles tiles{};
    int4 *desc = nullptr;     // per entry: base, pitch, level, kind
    int *skip = nullptr;      // per entry
    double4 *line = nullptr;  // per entry: centroid, refinement parameter; sources (k_tree_entries)
    double2 *aux = nullptr;   // per entry: DS, refinement radius
    int nroot = 0;
    int *root = nullptr;      // first entry of each tree, and the end of the list
};

using PlanKey = std::array<int, 4>;
using PlanMap = std::map<PlanKey, TreePlan *>;

struct FaceDims {
    int64_t off;  // first level-0 cell of the face in the source order
    int A, B;     // cells per row, rows
};

// Level-0 face cells in the order of calc_normalderiv_3d: X faces rows of NNY cells (k outer),
// Y faces rows of NNX cells (k outer), Z faces rows of NNX cells (j outer).
void face_dims(const int n[3], FaceDims f[6]) {
    const int NNX = n[0] - 1, NNY = n[1] - 1, NNZ = n[2] - 1;
    const int A[6] = {NNY, NNY, NNX, NNX, NNX, NNX};
    const int B[6] = {NNZ, NNZ, NNZ, NNZ, NNY, NNY};
    int64_t off = 0;
    for (int q = 0; q < 6; q++) {
        f[q].off = off;
        f[q].A = A[q];
        f[q].B = B[q];
        off += (int64_t)A[q] * B[q];
    }
}

int ceil_div(int a, int b) { return a / b + (a % b != 0); }

// Links of every level, built face by face and, within a face, level by level (the order
// in which the reference numbers the cells of each level).
int build_links(Ctx *c, const int n[3], int levmax, std::vector<std::vector<TreeLink>> &lv) {
    FaceDims fd[6];
    face_dims(n, fd);
    lv.assign(levmax + 1, {});
    for (int q = 0; q < 6; q++) {
        const int A = fd[q].A, B = fd[q].B;
        std::vector<int32_t> start(levmax + 1, 0);  // first cell of this face per level
        for (int lev = 0; lev <= levmax; lev++) {
            const int s = 1 << lev;
            std::vector<TreeLink> &L = lv[lev];
            start[lev] = (int32_t)L.size();
            const int qa = A / s, qb = B / s;                  // whole groups per row, rows of groups
            const int nnl = lev > 0 ? ceil_div(A, s / 2) : 0;  // cells per row one level finer
            for (int b = 0; b < qb; b++) {
                for (int a = 0; a < qa; a++) {
                    TreeLink t{};
                    t.base = (int32_t)(fd[q].off + (int64_t)b * s * A + (int64_t)a * s);
                    t.pitch = A;
                    t.kind = 1;
                    if (lev > 0) {
                        int32_t nj;
                        if (a == 0 && (int32_t)L.size() == start[lev]) nj = start[lev - 1];  // face start
                        else if (a == 0) nj = L.back().kind < 0 ? L.back().ch[1] + 1 : L.back().ch[2] + 1;
                        else nj = L.back().ch[1] + 1;
                        t.ch[0] = nj;
                        t.ch[1] = nj + 1;
                        t.ch[2] = nj + nnl + 1;
                        t.ch[3] = nj + nnl;
                        t.nch = 4;
                    }
                    L.push_back(t);
                }
                if (A % s != 0 || A <= s) {
                    if (lev == 0 || L.empty()) return fail(c, VPMX_ERR_UNSUP, "tree: face narrower than 2^levmax cells");
                    TreeLink t{};
                    const int32_t nj = L.back().ch[1] + 1;
                    t.base = -1;
                    t.kind = -1;
                    t.ch[0] = nj;
                    t.ch[1] = nj + nnl;
                    t.nch = 2;
                    L.push_back(t);
                }
            }
            if (B % s != 0 || B <= s) {
                if (lev == 0 || L.empty()) return fail(c, VPMX_ERR_UNSUP, "tree: face narrower than 2^levmax cells");
                for (int a = 0; a < qa; a++) {
                    // the reference leaves out the corner when a*s == A-s with A % s != 0,
                    // which never holds; the test is kept so the cell count is its own
                    if (a * s == A - s && A % s != 0) continue;
                    const TreeLink &p = L.back();
                    const int32_t nj = (a == 0 && p.kind > 0) ? p.ch[2] + 1 : p.ch[1] + 1;
                    TreeLink t{};
                    t.base = -1;
                    t.kind = -2;
                    t.ch[0] = nj;
                    t.ch[1] = nj + 1;
                    t.nch = 2;
                    L.push_back(t);
                }
            }
        }
    }
    return VPMX_OK;
}

// Preorder of the forest rooted at every cell of level levmax.
int flatten(Ctx *c, const std::vector<std::vector<TreeLink>> &lv, int levmax, std::vector<int4> &desc,
            std::vector<int> &skip, std::vector<int> &root) {
    struct Frame {
        int lev, idx, next;
        size_t pos;
    };
    std::vector<Frame> st;
    for (int r = 0; r < (int)lv[levmax].size(); r++) {
        st.push_back({levmax, r, 0, desc.size()});
        root.push_back((int)desc.size());
        const TreeLink &t0 = lv[levmax][r];
        desc.push_back(make_int4(t0.base, t0.pitch, levmax, t0.kind));
        skip.push_back(0);
        while (!st.empty()) {
            Frame &f = st.back();
            const TreeLink &t = lv[f.lev][f.idx];
            if (f.lev > 0 && f.next < t.nch) {
                const int ch = t.ch[f.next++];
                const int fl = f.lev - 1;
                if (ch < 0 || ch >= (int)lv[fl].size())
                    return fail(c, VPMX_ERR_UNSUP, "tree: a cell links outside its level (faces too narrow for the levels)");
                const TreeLink &u = lv[fl][ch];
                st.push_back({fl, ch, 0, desc.size()});
                desc.push_back(make_int4(u.base, u.pitch, fl, u.kind));
                skip.push_back(0);
                if (desc.size() > (size_t)INT32_MAX / 2) return fail(c, VPMX_ERR_UNSUP, "tree: too many nodes");
                continue;
            }
            skip[f.pos] = (int)desc.size();
            st.pop_back();
        }
    }
    root.push_back((int)desc.size());
    return VPMX_OK;
}

// Entry aggregates from the level-0 cells (build_level_nbound_3d's sums, same order:
// rows of the group outer, cells of a row inner; area-weighted source).  pos.w encodes the
// refinement test of the traversal:
//   point sources (tree_calc_3d):   refine iff r < w, w = 10 sqrt(DS) above level 0, 0 at
//                                   level 0 (never), 1e150 at dummies (always); one 64-byte line
//                                   per entry: pos with w^2 (1 - 1e-14) for w, val the products
//                                   source * DS with the skip index in the bits of w; aux (DS, w);
//   panels (tree_calc_3d_s):        refine iff r / pos.w < 10 — sqrt(DS) above level 0, NaN at
//                                   level 0 (never), -1 at dummies of kind -1 (always), 0 at
//                                   dummies of kind -2 (never: the reference takes them as
//                                   cells of zero area, r / 0 = inf).
// Dummies sit at the origin with zero area and source, as the reference's zeroed level
// arrays leave them.
__global__ void k_tree_entries(int64_t nent, const int4 *__restrict__ desc, const int *__restrict__ skip, int64_t nb,
                               const double *__restrict__ cxyz, const double *__restrict__ sig,
                               const double *__restrict__ ds, double4 *__restrict__ line, double2 *__restrict__ aux,
                               int panels) {
#pragma clang fp contract(off)
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nent) return;
    const int4 d = desc[e];
    const double sk = __longlong_as_double(skip[e]);
    double4 *pos = line + 2 * e, *val = line + 2 * e + 1;
    if (d.w < 0) {
        const double w = panels ? (d.w == -1 ? -1.0 : 0.0) : 1e300;
        *pos = make_double4(0.0, 0.0, 0.0, w);
        *val = make_double4(0.0, 0.0, 0.0, panels ? 0.0 : sk);
        aux[e] = make_double2(0.0, 1e150);
        return;
    }
    const int s = 1 << d.z;
    double xc = 0, yc = 0, zc = 0, sc = 0, q0 = 0, q1 = 0, q2 = 0;
    for (int mm = 0; mm < s; mm++) {
        for (int nn = 0; nn < s; nn++) {
            const int64_t l = (int64_t)d.x + (int64_t)mm * d.y + nn;
            const double sv = ds[l];
            xc = cxyz[l] + xc;
            yc = cxyz[nb + l] + yc;
            zc = cxyz[2 * nb + l] + zc;
            sc = sv + sc;
            q0 = sig[l] * sv + q0;
            q1 = sig[nb + l] * sv + q1;
            q2 = sig[2 * nb + l] * sv + q2;
        }
    }
    const double fl = (double)(s * s);
    if (panels) {
        *pos = make_double4(xc / fl, yc / fl, zc / fl, d.z > 0 ? sqrt(sc) : __builtin_nan(""));
        *val = make_double4(sc, q0 / sc, q1 / sc, q2 / sc);
        return;
    }
    const double w = d.z > 0 ? 10.0 * sqrt(sc) : 0.0, w2 = w * w;
    *pos = make_double4(xc / fl, yc / fl, zc / fl, w2 * (1.0 - 1e-14));
    *val = make_double4(q0 / sc * sc, q1 / sc * sc, q2 / sc * sc, sk);
    aux[e] = make_double2(sc, w);
}

constexpr int TR_WAVES = 8, TR_PARTS = 16;

// The target node (1-based) t of lane `lane` of patch w (TR_T x 8 by 8 nodes, target t in its
// t-th 8 columns); face q, false past the face's edge.
constexpr int TR_T = 2;
__device__ __forceinline__ bool tree_target(const Grid &g, const TreeTiles &tt, int w, int lane, int t, int *q, int *i,
                                            int *j, int *k) {
    int f = 0;
    while (w >= tt.off[f + 1]) f++;
    *q = f;
    const int NX = g.n[0], NY = g.n[1], NZ = g.n[2];
    const int tl = w - tt.off[f];
    const int u = (tl % tt.nu[f]) * 8 * TR_T + 8 * t + (lane & 7);
    const int v = (tl / tt.nu[f]) * 8 + (lane >> 3);
    const int hi = f & 1;
    if (f < 2) {  // X faces: all (j, k)
        *i = hi ? NX : 1; *j = u + 1; *k = v + 1;
        return u < NY && v < NZ;
    }
    if (f < 4) {  // Y faces: i = 2..NX-1, all k
        *j = hi ? NY : 1; *i = u + 2; *k = v + 1;
        return u < NX - 2 && v < NZ;
    }
    // Z faces: i = 2..NX-1, j = 2..NY-1
    *k = hi ? NZ : 1; *i = u + 2; *j = v + 2;
    return u < NX - 2 && v < NY - 2;
}

// SOL(target) += SOURCE / (4 pi).  The test r < w needs r itself only where r^2 and w^2 agree to
// 1e-14; elsewhere the squares decide, and the accepted term's 1/r comes from the reciprocal
// square root and one third-order step.  What bounds the walk is the scalar loads of the entries:
// one 64-byte line per entry, the next one in list order fetched ahead (the list ends with one
// line of padding), TR_T targets per lane to each line, and the eight waves of a work-group on
// neighbouring patches of the same trees, so that they find each other's lines in the scalar
// cache (a 129 x 129 x 41 block: 0.87 ms with the waves of a work-group on different trees).
__global__ void __launch_bounds__(64 * TR_WAVES)
    k_tree_eval(Grid g, TreeTiles tt, int nroot, const int *__restrict__ root, const double4 *__restrict__ line,
                const double2 *__restrict__ aux, double *__restrict__ part) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = blockIdx.x * TR_WAVES + wave;
    if (tile >= tt.off[6]) return;
    double X[TR_T], Y[TR_T], Z[TR_T], S[TR_T][3];
    int until[TR_T];  // target t takes no term before entry until[t]
#pragma unroll
    for (int t = 0; t < TR_T; t++) {
        int q, i, j, k;
        until[t] = tree_target(g, tt, tile, lane, t, &q, &i, &j, &k) ? 0 : 0x7fffffff;
        X[t] = g.x0[0] + (double)(i - 1) * g.h[0];
        Y[t] = g.x0[1] + (double)(j - 1) * g.h[1];
        Z[t] = g.x0[2] + (double)(k - 1) * g.h[2];
        S[t][0] = S[t][1] = S[t][2] = 0.0;
    }
    for (int r0 = blockIdx.y; r0 < nroot; r0 += TR_PARTS) {
        int e = root[r0];
        const int end = root[r0 + 1];
        double4 p = line[2 * e], v = line[2 * e + 1];
        while (e < end) {
            const double4 p1 = line[2 * e + 2], v1 = line[2 * e + 3];
            const int sk = (int)__double_as_longlong(v.w);
            bool refine = false;
#pragma unroll
            for (int t = 0; t < TR_T; t++) {
                const double XR = p.x - X[t], YR = p.y - Y[t], ZR = p.z - Z[t];
                const double r2 = XR * XR + YR * YR + ZR * ZR;
                const bool live = e >= until[t];
                bool down = r2 < p.w;
                const bool close = live && ((!down && r2 <= p.w * (1.0 + 2.1e-14)) || r2 <= 1.1e-10);
                double y = __builtin_amdgcn_rsq(r2);
                const double er = fma(-r2 * y, y, 1.0);
                y = fma(y * er, fma(0.375, er, 0.5), y);
                if (__any(close)) {  // (whole wave: the square roots stay out of the common path)
                    const double r = sqrt(r2);
                    const double2 x = aux[e];
                    if (!down) down = r < x.y;
                    if (!down && !(r > 1e-05))  // self term of a cell whose centroid is the node
                        y = -sqrt(x.x) * (2.0 * log((sqrt(2.0) - 1) / (sqrt(2.0) + 1))) / x.x;
                }
                if (live && !down) {
                    S[t][0] = fma(-v.x, y, S[t][0]);
                    S[t][1] = fma(-v.y, y, S[t][1]);
                    S[t][2] = fma(-v.z, y, S[t][2]);
                    until[t] = sk;
                }
                refine = refine || (live && down);
            }
            const int next = __builtin_amdgcn_readfirstlane(__any(refine) ? e + 1 : sk);
            if (next == e + 1) {
                p = p1;
                v = v1;
            } else {
                p = line[2 * next];
                v = line[2 * next + 1];
            }
            e = next;
        }
    }
    const int64_t nt = (int64_t)tt.off[6] * 64 * TR_T;
#pragma unroll
    for (int t = 0; t < TR_T; t++)
        for (int c = 0; c < 3; c++)
            part[((int64_t)blockIdx.y * 3 + c) * nt + ((int64_t)tile * TR_T + t) * 64 + lane] = S[t][c];
}

// SOL(target) += (the parts' sums, in order) / div.
__global__ void __launch_bounds__(256) k_tree_sum(Grid g, TreeTiles tt, int parts, const double *__restrict__ part,
                                                  double div, GView sol) {
#pragma clang fp contract(off)
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x, nt = (int64_t)tt.off[6] * 64 * TR_T;
    if (e >= nt) return;
    const int lane = (int)(e & 63), t = (int)(e >> 6) % TR_T;
    int q, i, j, k;
    if (!tree_target(g, tt, (int)(e / (64 * TR_T)), lane, t, &q, &i, &j, &k)) return;
    const int64_t o = sol.at(i - 1, j - 1, k - 1);
    for (int c = 0; c < 3; c++) {
        double s = 0.0;
        for (int p = 0; p < parts; p++) s += part[((int64_t)p * 3 + c) * nt + e];
        sol.p[c * sol.cs + o] = sol.p[c * sol.cs + o] + s / div;
    }
}

// tree_calc_3d_s (pmbound.f90:1346-1481) under calc_boundinf_3d_lev_s (:1255-1345):
// refine iff r / sqrt(DS) < 10 above level 0 or at a dummy of kind -1; a cell taken below the
// top level adds -s DS / (4 pi r); a top-level cell adds FSOUR_A4 (the target plane's frame,
// the cell's area) times the source of the FIRST top-level cell, as the reference passes
// nv = 1 at the top.  SOL += SOURCE.
__global__ void __launch_bounds__(64 * TR_WAVES)
    k_tree_eval_s(Grid g, TreeTiles tt, int nroot, const int *__restrict__ root, int levmax,
                  const int4 *__restrict__ desc, const double4 *__restrict__ line, const int *__restrict__ skip,
                  double *__restrict__ part) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = blockIdx.x * TR_WAVES + wave;
    if (tile >= tt.off[6]) return;
    int q, i, j, k;
    const bool ok = tree_target(g, tt, tile, lane, blockIdx.z, &q, &i, &j, &k);
    const int iplane = (q & 1 ? -1 : 1) * (q < 2 ? 2 : (q < 4 ? 1 : 3));
    const PanelFrame fr = panel_frame(iplane, g.h);
    const double XO[3] = {g.x0[0] + (double)(i - 1) * g.h[0], g.x0[1] + (double)(j - 1) * g.h[1],
                          g.x0[2] + (double)(k - 1) * g.h[2]};
    const double PI4 = 4.0 * (4.0 * atan(1.0));
    const double4 first = line[1];  // the first top-level cell
    double S0 = 0.0, S1 = 0.0, S2 = 0.0;
    int until = ok ? 0 : 0x7fffffff;
    for (int t = blockIdx.y; t < nroot; t += TR_PARTS) {
        int e = root[t];
        const int end = root[t + 1];
        while (e < end) {
            const double4 p = line[2 * e];
            const double4 a = line[2 * e + 1];
            const int lev = desc[e].z;
            const int sk = skip[e];
            bool refine = false;
            if (e >= until) {
                const double d[3] = {XO[0] - p.x, XO[1] - p.y, XO[2] - p.z};
                const double r = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
                if (r / p.w < 10) {
                    refine = true;
                } else {
                    if (lev != levmax) {
                        const double PR = PI4 * r;
                        S0 = S0 - a.y * a.x / PR;
                        S1 = S1 - a.z * a.x / PR;
                        S2 = S2 - a.w * a.x / PR;
                    } else {
                        const double FIS = fsour_a4(fr, d, a.x, PI4);
                        S0 = S0 + first.y * FIS;
                        S1 = S1 + first.z * FIS;
                        S2 = S2 + first.w * FIS;
                    }
                    until = sk;
                }
            }
            e = __builtin_amdgcn_readfirstlane(__any(refine) ? e + 1 : sk);
        }
    }
    const int64_t nt = (int64_t)tt.off[6] * 64 * TR_T;
    double *o = part + (int64_t)blockIdx.y * 3 * nt + ((int64_t)tile * TR_T + blockIdx.z) * 64 + lane;
    o[0] = S0;
    o[nt] = S1;
    o[2 * nt] = S2;
}

void free_plan(TreePlan *p) {
    if (!p) return;
    (void)hipFree(p->desc);
    (void)hipFree(p->skip);
    (void)hipFree(p->line);
    (void)hipFree(p->root);
    (void)hipFree(p->aux);
    delete p;
}

int get_plan(Ctx *c, const Grid &g, int levmax, int64_t nb, TreePlan **out) {
    if (!c->tree) c->tree = new PlanMap();
    PlanMap &m = *(PlanMap *)c->tree;
    const PlanKey key{g.n[0], g.n[1], g.n[2], levmax};
    auto it = m.find(key);
    if (it != m.end()) {
        *out = it->second;
        return VPMX_OK;
    }
    if (levmax < 0 || levmax > 12) return fail(c, VPMX_ERR_UNSUP, "tree: levels must be 0..12");
    std::vector<std::vector<TreeLink>> lv;
    VPMX_TRY(build_links(c, g.n, levmax, lv));
    if ((int64_t)lv[0].size() != nb) return fail(c, VPMX_ERR_STATE, "tree: level-0 cells differ from the face sources");
    std::vector<int4> desc;
    std::vector<int> skip, root;
    desc.reserve((size_t)(nb * 4 / 3 + 64));
    skip.reserve(desc.capacity());
    VPMX_TRY(flatten(c, lv, levmax, desc, skip, root));
    TreePlan *p = new TreePlan();
    p->nb = nb;
    p->nent = (int64_t)desc.size();
    p->nroot = (int)root.size() - 1;
    const int NX = g.n[0], NY = g.n[1], NZ = g.n[2];
    const int U[6] = {NY, NY, NX - 2, NX - 2, NX - 2, NX - 2};
    const int V[6] = {NZ, NZ, NZ, NZ, NY - 2, NY - 2};
    p->tiles.off[0] = 0;
    for (int q = 0; q < 6; q++) {
        p->tiles.nu[q] = (U[q] + 8 * TR_T - 1) / (8 * TR_T);
        p->tiles.off[q + 1] = p->tiles.off[q] + p->tiles.nu[q] * ((V[q] + 7) / 8);
    }
    skip.push_back(p->nent);  // one entry of padding: the walks load ahead
    desc.push_back(make_int4(-1, 0, 0, -1));
    const size_t ne = (size_t)p->nent + 1;
    hipError_t e = hipMalloc((void **)&p->desc, sizeof(int4) * ne);
    if (e == hipSuccess) e = hipMalloc((void **)&p->skip, sizeof(int) * ne);
    if (e == hipSuccess) e = hipMalloc((void **)&p->line, sizeof(double4) * 2 * ne);
    if (e == hipSuccess) e = hipMalloc((void **)&p->aux, sizeof(double2) * ne);
    if (e == hipSuccess) e = hipMalloc((void **)&p->root, sizeof(int) * root.size());
    if (e == hipSuccess) e = hipMemcpy(p->root, root.data(), sizeof(int) * root.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->desc, desc.data(), sizeof(int4) * ne, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->skip, skip.data(), sizeof(int) * ne, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        free_plan(p);
        return fail(c, VPMX_ERR_HIP, std::string("tree plan: ") + hipGetErrorString(e));
    }
    m[key] = p;
    *out = p;
    return VPMX_OK;
}

}  // namespace

int boundary_sums_tree(Ctx *c, const Grid &g, int64_t nb, const double *sig, const double *cxyz, const double *ds,
                       GView sol, int levmax, bool fine, bool panels) {
    if (g.n[0] < 3 || g.n[1] < 3 || g.n[2] < 3) return fail(c, VPMX_ERR_ARG, "tree: grid too small");
    TreePlan *p = nullptr;
    VPMX_TRY(get_plan(c, g, levmax, nb, &p));
    hipLaunchKernelGGL(k_tree_entries, dim3((unsigned)((p->nent + 255) / 256)), dim3(256), 0, c->stream, p->nent,
                       p->desc, p->skip, nb, cxyz, sig, ds, p->line, p->aux, panels ? 1 : 0);
    VPMX_HIP(c, hipGetLastError());
    const int ntile = p->tiles.off[6];
    const int64_t nt = (int64_t)ntile * 64 * TR_T;
    int st = VPMX_OK;
    // (384 bytes a target, 200 MB for the faces of a 289^3 block; a plan has 24 trees or more)
    double *part = (double *)ensure(c, c->tree_part, sizeof(double) * 3 * TR_PARTS * (size_t)nt, &st);
    if (st) return st;
    const unsigned blocks = (unsigned)((ntile + TR_WAVES - 1) / TR_WAVES);
    hipEvent_t e0, e1;
    if (panels)
        hipLaunchKernelGGL(k_tree_eval_s, dim3(blocks, TR_PARTS, TR_T), dim3(64 * TR_WAVES), 0, c->stream, g, p->tiles,
                           p->nroot, p->root, levmax, p->desc, p->line, p->skip, part);
    else if (fine && kernel_events(c, K_BOUNDSUM, &e0, &e1))
        hipExtLaunchKernelGGL(k_tree_eval, dim3(blocks, TR_PARTS), dim3(64 * TR_WAVES), 0, c->stream, e0, e1, 0, g,
                              p->tiles, p->nroot, p->root, p->line, p->aux, part);
    else
        hipLaunchKernelGGL(k_tree_eval, dim3(blocks, TR_PARTS), dim3(64 * TR_WAVES), 0, c->stream, g, p->tiles, p->nroot,
                           p->root, p->line, p->aux, part);
    VPMX_HIP(c, hipGetLastError());
    const double PI4 = 4.0 * (4.0 * std::atan(1.0));
    hipLaunchKernelGGL(k_tree_sum, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, c->stream, g, p->tiles, TR_PARTS,
                       part, panels ? 1.0 : PI4, sol);
    VPMX_HIP(c, hipGetLastError());
    return VPMX_OK;
}

int64_t tree_entries(Ctx *c, const int n[3], int levmax) {
    if (!c->tree) return -1;
    PlanMap &m = *(PlanMap *)c->tree;
    auto it = m.find(PlanKey{n[0], n[1], n[2], levmax});
    return it == m.end() ? -1 : it->second->nent;
}

void free_tree(Ctx *c) {
    if (!c->tree) return;
    PlanMap *m = (PlanMap *)c->tree;
    for (auto &kv : *m) free_plan(kv.second);
    delete m;
    c->tree = nullptr;
}

}  // namespace vpmx
