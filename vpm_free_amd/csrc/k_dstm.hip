// DST-I passes of the Dirichlet solve (pmsolve.f90:284-432) as dense products with the sine
// matrix on the FP64 matrix cores (v_mfma_f64_16x16x4f64).
//
// S(j,k) = sin(pi j k / (m+1)) is symmetric about the middle of the line up to the sign (-1)^(k+1),
// so the outputs of odd k are a product with the sums x_j + x_{m+1-j} and those of even k one
// with the differences; with m odd the latter is a DST-I of (m-1)/2 points and folds once more.
// That leaves 3/8 m^2 multiply-adds per line: 6 transforms of 271 points over 3 x 271^3 values
// are 73 GFLOP against 1.2 ms of HBM time for the five passes, and on small grids the products
// are a few microseconds where a chain of FFT stages is one long dependent sequence.
//
// Operands: the A fragments (the sine matrix, in the lane order of the instruction, two k-steps
// of 4 per 16-byte load) come straight from L2, where one line length's 0.25 MB stay; the folded
// lines are staged once in LDS as B.  A wave owns 16-row blocks of the output (a list balanced
// by their lengths) against 16 or 32 lines.
//
//   k_dstm_plane  x and y transforms of a whole (x, y) plane held in LDS: a solve on a small grid
//                 is three launches (planes, z, planes) instead of five passes.
//   k_dstm_x/y/z  one axis, for planes that do not fit.
#include <hip/hip_ext.h>

#include <cmath>
#include <cstdio>
#include <map>
#include <vector>

#include "dstm.h"
#include "tune.h"
#include "vpmx_ctx.h"

namespace vpmx {

typedef double dm_acc __attribute__((ext_vector_type(4)));

// Longest lines of the matrix passes.  The products grow with the square of the length, the FFT
// passes hardly, but these depend on the factors of m + 1.  Whole solves of m^3 points, 3
// components, us, products against FFT.  FP64: 231 (8.29) 1233/4330, 239 1289/1489, 255 1548/1650,
// 263 (8.3.11) 1980/2991, 271 (16.17) 2065/2450, 279 2323/2489, and above 287 points, where an FFT line
// no longer fits one wave, 303 3155/13325, 319 4355/6821, 367 7405/23249.  The 288-point transform has a
// compile-time FFT plan and keeps it (by axis, products against FFT: x forward 600/425, y 440/370, z
// 800/806, x inverse 550/385); only z forward alone is the products' (465/618).  FP32 arrays (FP64
// sums: half the bytes, the same products): 191 481/563, 207 759/881, 215 847/793, 239 1189/1139, 255
// 1332/1117, 271 1907/1261, but with factors over 17 (no register transform) 231 1139/3079, 247
// 1296/3649.
// DM_MAX: three row blocks a wave (24 of them).
constexpr int DM_MAX = 367, DM_MAX32 = 208, DM_PLANE = 224;
constexpr int DM_PAD = 8;  // zero rows after a line: the products run over whole pairs of k-steps

// The folded transform of one length.  Segments: outputs k = k0 + ks i (i < nk, 1-based wave
// numbers) from the folded rows row0 .. of the line; kp pairs of k-steps (8 rows each).
struct DmPlan {
    int m, h, odd, nf, nrb;
    int row0[3], nk[3], kp[3], k0[3], ks[3], rb0[3], foff[3];
    const double2 *frag;
};

// Folding of one line: item i of nf combines the points it returns (0-based) into the folded
// rows of the same places.  m odd: four points (two pairs mirrored about the middle, and about
// the middle of the half line); m even: one pair.  The middle point of an odd line stays.
struct DmFold {
    int a, b, c, d;  // a + d, b + c: mirrored pairs; b < 0: one pair only
};
__device__ __forceinline__ DmFold dm_fold_at(const DmPlan &P, int i) {
    DmFold f;
    f.a = i;
    f.d = P.m - 1 - i;
    f.b = P.h - 1 - i;
    f.c = P.h + 1 + i;
    if (!P.odd || f.b == f.a) f.b = -1;
    return f;
}
// x: the points a, b, c, d -> the folded values of the same rows
__device__ __forceinline__ void dm_fold(bool two, double &xa, double &xb, double &xc, double &xd) {
    const double e = xa + xd, o = xa - xd;
    if (two) {
        const double e2 = xb + xc, o2 = xb - xc;
        xb = e2;
        xc = o - o2;
        xd = o + o2;
    } else {
        xd = o;
    }
    xa = e;
}

// Jobs (row block x column pair) of a wave: every other round runs backwards, so the longer row
// blocks, which come first, spread over the waves.
__device__ __forceinline__ int dm_job(int q, int wave, int nw) { return q * nw + ((q & 1) ? nw - 1 - wave : wave); }

// acc[q][j] = the wave's q-th job: 16 outputs x NB blocks of 16 columns.  Folded value (row, col)
// at L[row * rs + col * cs]; swz: the two halves of a row of 32 change places on odd rows, so
// the four rows that a wave reads at once fall on different banks.
// Row blocks [R.lo, R.lo + R.n) of the plan; its folded row r stands at LDS row r - R.shift.
struct DmRange {
    int lo, n, shift;
};
template <int Q, int NB, bool SWZ>
__device__ __forceinline__ void dm_product(const DmPlan &P, const DmRange &R, int ncp, int ncols, int wave, int nw,
                                           int lane, const double *__restrict__ L, int rs, int cs,
                                           dm_acc (&acc)[Q][NB]) {
    const int li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int q = 0; q < Q; q++) {
#pragma unroll
        for (int j = 0; j < NB; j++) acc[q][j] = dm_acc{0.0, 0.0, 0.0, 0.0};
        const int t = dm_job(q, wave, nw);
        if (t >= R.n * ncp) continue;
        const int tr = t / ncp, cp = t - tr * ncp, rb = R.lo + tr;
        const int s = rb >= P.rb0[2] ? 2 : (rb >= P.rb0[1] ? 1 : 0);
        const int kp = P.kp[s], row0 = P.row0[s] - R.shift;
        const double2 *__restrict__ f = P.frag + P.foff[s] + (rb - P.rb0[s]) * kp * 64 + lane;
        const double *b[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) {
            int col = (cp * NB + j) * 16 + li;
            if (SWZ) col ^= ((row0 + lk) & 1) << 4;
            else col = col < ncols ? col : ncols - 1;
            b[j] = L + (row0 + lk) * rs + col * cs;
        }
        double2 a = f[0], a1 = f[(kp > 1 ? 1 : 0) * 64];
        for (int p = 0; p < kp; p++) {
            const double2 a2 = f[(p + 2 < kp ? p + 2 : kp - 1) * 64];
            double x[NB], y[NB];
#pragma unroll
            for (int j = 0; j < NB; j++) {
                x[j] = b[j][8 * p * rs];
                y[j] = b[j][(8 * p + 4) * rs];
            }
#pragma unroll
            for (int j = 0; j < NB; j++) acc[q][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, x[j], acc[q][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < NB; j++) acc[q][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, y[j], acc[q][j], 0, 0, 0);
            a = a1;
            a1 = a2;
        }
    }
}

// f(k index (0-based), column, value, segment, column block, output of the segment) for the
// wave's outputs.
template <int Q, int NB, class F>
__device__ __forceinline__ void dm_outputs(const DmPlan &P, const DmRange &R, int ncp, int wave, int nw, int lane,
                                           const dm_acc (&acc)[Q][NB], F f) {
    const int li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int t = dm_job(q, wave, nw);
        if (t >= R.n * ncp) continue;
        const int tr = t / ncp, cp = t - tr * ncp, rb = R.lo + tr;
        const int s = rb >= P.rb0[2] ? 2 : (rb >= P.rb0[1] ? 1 : 0);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 16 * (rb - P.rb0[s]) + 4 * r + lk;
            if (i < P.nk[s]) {
                const int k = P.k0[s] + P.ks[s] * i - 1;
#pragma unroll
                for (int j = 0; j < NB; j++) f(k, (cp * NB + j) * 16 + li, acc[q][j][r], s, j, i);
            }
        }
    }
}

// The folds of lines already in LDS, in place.
template <bool SWZ>
__device__ __forceinline__ void dm_fold_lds(const DmPlan &P, double *L, int rs, int cs, int ncols, bool colfast,
                                            int tid, int nt) {
    const int tot = P.nf * ncols;
    for (int it = tid; it < tot; it += nt) {
        int i, col;
        if (colfast) { i = it / ncols; col = it - i * ncols; }
        else { col = it / P.nf; i = it - col * P.nf; }
        const DmFold f = dm_fold_at(P, i);
        auto at = [&](int row) -> double & { return L[row * rs + (SWZ ? col ^ ((row & 1) << 4) : col) * cs]; };
        const bool two = f.b >= 0;
        double xa = at(f.a), xd = at(f.d), xb = 0.0, xc = 0.0;
        if (two) { xb = at(f.b); xc = at(f.c); }
        dm_fold(two, xa, xb, xc, xd);
        at(f.a) = xa;
        at(f.d) = xd;
        if (two) { at(f.b) = xb; at(f.c) = xc; }
    }
}

// Lines of `ncols` columns from global memory (element (row, col) = ld(row, col)), folded on the
// way into LDS; zero rows after them.
template <bool SWZ, class LD>
__device__ __forceinline__ void dm_load(const DmPlan &P, double *L, int rs, int cs, int ncols, bool colfast, int tid,
                                        int nt, LD ld) {
    const int tot = P.nf * ncols;
    auto at = [&](int row, int col) -> double & { return L[row * rs + (SWZ ? col ^ ((row & 1) << 4) : col) * cs]; };
#pragma unroll 2
    for (int it = tid; it < tot; it += nt) {
        int i, col;
        if (colfast) { i = it / ncols; col = it - i * ncols; }
        else { col = it / P.nf; i = it - col * P.nf; }
        const DmFold f = dm_fold_at(P, i);
        const bool two = f.b >= 0;
        // (the loads of a single pair read its points twice: no load behind a branch)
        double xa = ld(f.a, col), xd = ld(f.d, col), xb = ld(two ? f.b : f.a, col), xc = ld(two ? f.c : f.d, col);
        dm_fold(two, xa, xb, xc, xd);
        at(f.a, col) = xa;
        at(f.d, col) = xd;
        if (two) { at(f.b, col) = xb; at(f.c, col) = xc; }
    }
    if (P.odd)
        for (int col = tid; col < ncols; col += nt) at(P.h, col) = ld(P.h, col);
    for (int it = tid; it < DM_PAD * ncols; it += nt) {
        const int r = it / ncols, col = it - r * ncols;
        at(P.m + r, col) = 0.0;
    }
}

// ---------------------------------------------------------------- z pass
struct DmZ {
    int px, mx, my;
    int64_t wcs;
    int pl;  // plane stride px * my
    int ncomp;
    const double *lx, *ly, *lz;
    double norm;
    double *zsum;
    const double *zw;
};
constexpr int DM_NT = 512, DM_NW = DM_NT / 64;

// A tile of 16 NB neighbouring lines of the flattened (x, y) plane: loaded once, transformed,
// scaled by the diagonal, transformed back and stored once.  The columns of the row padding run
// along (each column's values depend on that column alone).
template <int Q, int NB, class TI, class TO, bool INV>
__global__ void __launch_bounds__(DM_NT) k_dstm_z(DmPlan P, DmZ a, const TI *w, TO *wo) {
    extern __shared__ double L[];
    constexpr int BN = 16 * NB;
    const DmRange R{0, P.nrb, 0};
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * BN, comp = blockIdx.y, pl = a.pl;
    w += comp * a.wcs;
    wo += comp * a.wcs;
    dm_load<NB == 2>(P, L, BN, 1, BN, true, tid, DM_NT, [&](int row, int col) {
        const int n = n0 + col < pl ? n0 + col : pl - 1;
        return (double)w[row * pl + n];
    });
    const int li = lane & 15;
    double lxy[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int n = n0 + 16 * j + li < pl ? n0 + 16 * j + li : pl - 1;
        const int iy = n / a.px, ix = n - iy * a.px;
        lxy[j] = a.lx[ix < a.mx ? ix : a.mx - 1] + a.ly[iy];
    }
    __syncthreads();
    dm_acc acc[Q][NB];
    dm_product<Q, NB, NB == 2>(P, R, 1, BN, wave, DM_NW, lane, L, BN, 1, acc);
    if (INV) {
        __syncthreads();
        dm_outputs<Q, NB>(P, R, 1, wave, DM_NW, lane, acc, [&](int k, int col, double v, int, int j, int) {
            L[k * BN + (NB == 2 ? col ^ ((k & 1) << 4) : col)] = v * (a.norm / -(lxy[j] + a.lz[k]));
        });
        __syncthreads();
        dm_fold_lds<NB == 2>(P, L, BN, 1, BN, true, tid, DM_NT);
        __syncthreads();
        dm_product<Q, NB, NB == 2>(P, R, 1, BN, wave, DM_NW, lane, L, BN, 1, acc);
        dm_outputs<Q, NB>(P, R, 1, wave, DM_NW, lane, acc, [&](int k, int col, double v, int, int, int) {
            if (n0 + col < pl) wo[k * pl + n0 + col] = (TO)v;
        });
    } else {
        // the spectrum, and its weighted sums over odd and even k (one partial per wave)
        double so[NB], se[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) so[j] = se[j] = 0.0;
        dm_outputs<Q, NB>(P, R, 1, wave, DM_NW, lane, acc, [&](int k, int col, double v, int s, int j, int) {
            const double u = v * (a.norm / -(lxy[j] + a.lz[k]));
            const double t = a.zw[k] * u;
            if (s == 0) so[j] += t;
            else se[j] += t;
            if (n0 + col < pl) wo[k * pl + n0 + col] = (TO)u;
        });
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NB; j++) {
            so[j] += __shfl_xor(so[j], 16, 64);
            so[j] += __shfl_xor(so[j], 32, 64);
            se[j] += __shfl_xor(se[j], 16, 64);
            se[j] += __shfl_xor(se[j], 32, 64);
            if (lane < 16) {
                L[(2 * wave) * BN + 16 * j + lane] = so[j];
                L[(2 * wave + 1) * BN + 16 * j + lane] = se[j];
            }
        }
        __syncthreads();
        if (tid < BN && n0 + tid < pl) {
            double o = 0.0, e = 0.0;
            for (int v = 0; v < DM_NW; v++) {
                o += L[(2 * v) * BN + tid];
                e += L[(2 * v + 1) * BN + tid];
            }
            const int n = n0 + tid, iy = n / a.px, ix = n - iy * a.px;
            if (ix < a.mx) {
                const int64_t at = ((int64_t)comp * a.my + iy) * a.mx + ix;
                a.zsum[at] = o + e;
                a.zsum[(int64_t)a.ncomp * a.my * a.mx + at] = o - e;
            }
        }
    }
}

// ---------------------------------------------------------------- y pass (in place)
template <int Q, int NB, class T>
__global__ void __launch_bounds__(DM_NT) k_dstm_y(DmPlan P, T *w, int px, int64_t wcs) {
    extern __shared__ double L[];
    constexpr int BN = 16 * NB;
    const DmRange R{0, P.nrb, 0};
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int x0 = blockIdx.x * BN;
    w += blockIdx.z * wcs + (int64_t)blockIdx.y * px * P.m;
    dm_load<NB == 2>(P, L, BN, 1, BN, true, tid, DM_NT, [&](int row, int col) {
        return (double)w[row * px + (x0 + col < px ? x0 + col : px - 1)];
    });
    __syncthreads();
    dm_acc acc[Q][NB];
    dm_product<Q, NB, NB == 2>(P, R, 1, BN, wave, DM_NW, lane, L, BN, 1, acc);
    dm_outputs<Q, NB>(P, R, 1, wave, DM_NW, lane, acc, [&](int k, int col, double v, int, int, int) {
        if (x0 + col < px) w[k * px + x0 + col] = (T)v;
    });
}

// ---------------------------------------------------------------- x passes
struct DmX {
    GView v;   // RHS (forward) or output (inverse) view
    GView bc;  // Dirichlet values (forward, has_bc)
    int has_bc;
    double ih2[3];
    int px, my, mz;
    int64_t wcs;
    void *w;
    int pitch;  // LDS doubles per line
};

// The right-hand side at interior node (i, j, k) with the Dirichlet values next to it folded in.
__device__ __forceinline__ double dm_rhs(const DmX &a, int comp, int mx, int i, int j, int k) {
    double v = a.v.p[comp * a.v.cs + a.v.at(i + 1, j + 1, k + 1)];
    if (a.has_bc) {
        const double *b = a.bc.p + comp * a.bc.cs;
        if (i == 0) v -= b[a.bc.at(0, j + 1, k + 1)] * a.ih2[0];
        if (i == mx - 1) v -= b[a.bc.at(mx + 1, j + 1, k + 1)] * a.ih2[0];
        if (j == 0) v -= b[a.bc.at(i + 1, 0, k + 1)] * a.ih2[1];
        if (j == a.my - 1) v -= b[a.bc.at(i + 1, a.my + 1, k + 1)] * a.ih2[1];
        if (k == 0) v -= b[a.bc.at(i + 1, j + 1, 0)] * a.ih2[2];
        if (k == a.mz - 1) v -= b[a.bc.at(i + 1, j + 1, a.mz + 1)] * a.ih2[2];
    }
    return v;
}

// 32 rows (j, k) of one component; the transformed rows go back through LDS so that the stores
// are whole rows.
constexpr int DM_XR = 32;
template <int Q, bool FWD, class T>
__global__ void __launch_bounds__(DM_NT) k_dstm_x(DmPlan P, DmX a) {
    extern __shared__ double L[];
    __shared__ int rj[DM_XR], rk[DM_XR];
    const DmRange R{0, P.nrb, 0};
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r0 = blockIdx.x * DM_XR, comp = blockIdx.y, rows = a.my * a.mz, m = P.m;
    if (tid < DM_XR) {
        const int r = r0 + tid < rows ? r0 + tid : rows - 1;
        rk[tid] = r / a.my;
        rj[tid] = r - rk[tid] * a.my;
    }
    __syncthreads();
    T *w = (T *)a.w + comp * a.wcs;
    dm_load<false>(P, L, 1, a.pitch, DM_XR, false, tid, DM_NT, [&](int x, int row) {
        const int j = rj[row], k = rk[row];
        return FWD ? dm_rhs(a, comp, m, x, j, k) : (double)w[(int64_t)(k * a.my + j) * a.px + x];
    });
    __syncthreads();
    dm_acc acc[Q][2];
    dm_product<Q, 2, false>(P, R, 1, DM_XR, wave, DM_NW, lane, L, 1, a.pitch, acc);
    __syncthreads();
    dm_outputs<Q, 2>(P, R, 1, wave, DM_NW, lane, acc, [&](int k, int col, double v, int, int, int) { L[col * a.pitch + k] = v; });
    __syncthreads();
    for (int row = wave; row < DM_XR; row += DM_NW) {
        if (r0 + row >= rows) break;
        const int j = rj[row], k = rk[row];
        if (FWD) {
            T *o = w + (int64_t)(k * a.my + j) * a.px;
            for (int x = lane; x < m; x += 64) o[x] = (T)L[row * a.pitch + x];
        } else {
            double *o = a.v.p + comp * a.v.cs + a.v.at(1, j + 1, k + 1);
            for (int x = lane; x < m; x += 64) o[x] = L[row * a.pitch + x];
        }
    }
}

// ---------------------------------------------------------------- whole planes
// One (x, y) plane per pair of work-groups: forward x then y into the work array, inverse y then
// x into the output view.  The first fold along x already separates the outputs (forward: odd and
// even kx; inverse: odd and even x), so each work-group of the pair keeps one half of the folded
// plane in LDS and never meets the other: twice the work-groups with half the LDS each, which is
// what a small grid lacks.  The pair sits on one XCD (8 apart in launch order), whose L2 joins
// its interleaved stores.
template <int NT, int Q, bool FWD>
__global__ void __launch_bounds__(NT) k_dstm_plane(DmPlan X, DmPlan Y, DmX a) {
    extern __shared__ double L[];
    constexpr int NW = NT / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = (blockIdx.x >> 3) & 1, k = (blockIdx.x >> 4) * 8 + (blockIdx.x & 7), comp = blockIdx.y;
    if (k >= a.mz) return;
    const int mx = X.m, my = Y.m, pt = a.pitch;
    // this half of the folded line: its rows, its row blocks, the outputs of its first segment
    const int shift = half ? X.nk[0] : 0, W = half ? mx - X.nk[0] : X.nk[0];
    const DmRange RX{half ? X.rb0[1] : 0, half ? X.nrb - X.rb0[1] : X.rb0[1], shift}, RY{0, Y.nrb, 0};
    const int cx = (W + 31) / 32, cy = (my + 31) / 32;  // column pairs of the two products
    double *w = (double *)a.w + comp * a.wcs + (int64_t)k * a.px * my;
    dm_acc acc[Q][2];
    // lines along x, folded; this half's rows kept
    for (int it = tid; it < X.nf * my; it += NT) {
        const int row = it / X.nf;
        const DmFold f = dm_fold_at(X, it - row * X.nf);
        const bool two = f.b >= 0;
        auto ld = [&](int x) { return FWD ? dm_rhs(a, comp, mx, x, row, k) : w[row * a.px + x]; };
        double xa = ld(f.a), xd = ld(f.d), xb = ld(two ? f.b : f.a), xc = ld(two ? f.c : f.d);
        dm_fold(two, xa, xb, xc, xd);
        double *l = L + row * pt - shift;
        l[half ? f.d : f.a] = half ? xd : xa;
        if (two) l[half ? f.c : f.b] = half ? xc : xb;
    }
    if (X.odd && !half)
        for (int row = tid; row < my; row += NT)
            L[row * pt + X.h] = FWD ? dm_rhs(a, comp, mx, X.h, row, k) : w[row * a.px + X.h];
    auto zero_cols = [&]() {
        for (int it = tid; it < DM_PAD * my; it += NT) {
            const int r = it / DM_PAD, c = it - r * DM_PAD;
            L[r * pt + W + c] = 0.0;
        }
    };
    for (int it = tid; it < DM_PAD * W; it += NT) {  // zero rows after the lines along y
        const int r = it / W, c = it - r * W;
        L[(my + r) * pt + c] = 0.0;
    }
    if (FWD) {
        zero_cols();
        __syncthreads();
        dm_product<Q, 2, false>(X, RX, cy, my, wave, NW, lane, L, 1, pt, acc);
        __syncthreads();
        dm_outputs<Q, 2>(X, RX, cy, wave, NW, lane, acc, [&](int, int row, double v, int s, int, int i) {
            if (row < my) L[row * pt + (s == 2 ? X.nk[1] : 0) + i] = v;
        });
        __syncthreads();
        dm_fold_lds<false>(Y, L, pt, 1, W, true, tid, NT);
        __syncthreads();
        dm_product<Q, 2, false>(Y, RY, cx, W, wave, NW, lane, L, pt, 1, acc);
        dm_outputs<Q, 2>(Y, RY, cx, wave, NW, lane, acc, [&](int ky, int c, double v, int, int, int) {
            if (c >= W) return;
            // the wave number that column c holds
            const int s = half ? (c >= X.nk[1] ? 2 : 1) : 0;
            const int kx = X.k0[s] + X.ks[s] * (s == 2 ? c - X.nk[1] : c) - 1;
            w[ky * a.px + kx] = v;
        });
    } else {
        __syncthreads();
        dm_fold_lds<false>(Y, L, pt, 1, W, true, tid, NT);
        __syncthreads();
        dm_product<Q, 2, false>(Y, RY, cx, W, wave, NW, lane, L, pt, 1, acc);
        __syncthreads();
        dm_outputs<Q, 2>(Y, RY, cx, wave, NW, lane, acc, [&](int y, int c, double v, int, int, int) {
            if (c < W) L[y * pt + c] = v;
        });
        zero_cols();
        __syncthreads();
        dm_product<Q, 2, false>(X, RX, cy, my, wave, NW, lane, L, 1, pt, acc);
        __syncthreads();
        dm_outputs<Q, 2>(X, RX, cy, wave, NW, lane, acc, [&](int, int row, double v, int s, int, int i) {
            if (row < my) L[row * pt + (s == 2 ? X.nk[1] : 0) + i] = v;
        });
        __syncthreads();
        for (int row = wave; row < my; row += NW) {
            double *o = a.v.p + comp * a.v.cs + a.v.at(1, row + 1, k + 1);
            for (int c = lane; c < W; c += 64) {
                const int s = half ? (c >= X.nk[1] ? 2 : 1) : 0;
                o[X.k0[s] + X.ks[s] * (s == 2 ? c - X.nk[1] : c) - 1] = L[row * pt + c];
            }
        }
    }
}

// ---------------------------------------------------------------- host
// The plan of length m: segments and their A fragments, uploaded once per length.
static int dm_plan(Ctx *c, int m, DmPlan *out) {
    DmPlan P{};
    P.m = m;
    P.odd = m & 1;
    P.h = m / 2;
    P.nf = P.odd ? (P.h + 1) / 2 : P.h;
    auto seg = [&](int s, int row0, int nk, int nj, int k0, int ks) {
        P.row0[s] = row0;
        P.nk[s] = nk;
        P.kp[s] = (nj + 7) / 8;
        P.k0[s] = k0;
        P.ks[s] = ks;
    };
    int nj[3] = {0, 0, 0};
    if (P.odd) {
        const int fl = P.h / 2, ne = P.h - fl;
        nj[0] = P.h + 1;
        nj[1] = ne;
        nj[2] = fl;
        seg(0, 0, P.h + 1, nj[0], 1, 2);
        seg(1, P.h + 1 + fl, ne, ne, 2, 4);
        seg(2, P.h + 1, fl, fl, 4, 4);
    } else {
        nj[0] = nj[1] = P.h;
        seg(0, 0, P.h, P.h, 1, 2);
        seg(1, P.h, P.h, P.h, 2, 2);
    }
    int off = 0;
    P.nrb = 0;
    for (int s = 0; s < 3; s++) {
        P.rb0[s] = P.nrb;
        P.foff[s] = off;
        const int nr = (P.nk[s] + 15) / 16;
        P.nrb += nr;
        off += nr * P.kp[s] * 64;
    }
    auto it = c->sinf_cache.find(m);
    if (it != c->sinf_cache.end()) {
        P.frag = (const double2 *)it->second;
        *out = P;
        return VPMX_OK;
    }
    const long double PI = 3.141592653589793238462643383279502884L;
    std::vector<double> sn((size_t)2 * (m + 1));
    for (int t = 0; t < 2 * (m + 1); t++)
        sn[t] = t % (m + 1) == 0 ? 0.0 : (double)sinl(PI * (long double)t / (long double)(m + 1));
    std::vector<double> v((size_t)off * 2, 0.0);
    for (int s = 0; s < 3; s++)
        for (int i = 0; i < P.nk[s]; i++)
            for (int r = 0; r < nj[s]; r++) {
                // the point (1-based) that folded row row0 + r stands for
                int j;
                if (s == 0) j = r + 1;
                else if (!P.odd) j = P.h - r;
                else j = s == 1 ? nj[1] - r : r + 1;
                const long long k = P.k0[s] + (long long)P.ks[s] * i;
                const int rb = i / 16, li = i % 16, p = r / 8, half = (r % 8) / 4, lk = r % 4;
                v[2 * ((size_t)P.foff[s] + (size_t)(rb * P.kp[s] + p) * 64 + lk * 16 + li) + half] =
                    sn[(size_t)((k * j) % (2 * (m + 1)))];
            }
    void *d = nullptr;
    VPMX_HIP(c, hipMalloc(&d, sizeof(double) * v.size()));
    VPMX_HIP(c, hipMemcpy(d, v.data(), sizeof(double) * v.size(), hipMemcpyHostToDevice));
    c->sinf_cache[m] = d;
    P.frag = (const double2 *)d;
    *out = P;
    return VPMX_OK;
}

// n without its factors up to p
static int dm_without(int n, int p) {
    for (int q = 2; q <= p; q++)
        while (n % q == 0) n /= q;
    return n;
}
bool dstm_line_fits(int m, bool f32, bool forward) {
    if (m < 1 || m > DM_MAX) return false;
    if (f32) return m <= DM_MAX32 || dm_without(m + 1, 17) > 1;
    return forward || m + 1 != FFT64_LENGTH;
}

static int dm_pitch(int m) {  // 2 (mod 4): 16 lines of two neighbouring points fall on all banks
    int p = m + DM_PAD;
    while ((p & 3) != 2) p++;
    return p;
}
static size_t dm_plane_lds(const int m[3]) {
    return sizeof(double) * (size_t)((m[1] + DM_PAD) * dm_pitch(m[0] / 2 + 1) + 32);
}
// the most jobs (16 outputs x 32 columns) of one half plane's two products
static int dm_plane_jobs(const int m[3]) {
    auto blocks = [](int n) { return (n + 15) / 16; };
    const int hx = m[0] / 2, hy = m[1] / 2;
    const int px = std::max(blocks(hx + 1), blocks(hx - hx / 2) + blocks(hx / 2));
    const int ny = (m[1] & 1) ? blocks(hy + 1) + blocks(hy - hy / 2) + blocks(hy / 2) : 2 * blocks(hy);
    return std::max(px * ((m[1] + 31) / 32), ny * ((hx + 32) / 32));
}

bool dstm_plane_fits(const Ctx *c, const int m[3]) {
    for (int d = 0; d < 3; d++)
        if (m[d] < 1 || m[d] > DM_PLANE) return false;
    // above about 96 x 96 points a plane's work-group is one long chain (load, two products, two
    // folds): the separate passes are faster (y + x 79 points: 19.4 against 20.4 us, 95: 27 against
    // 30, 143: 83 against 116), below it one launch less counts more
    return m[0] * m[1] <= 96 * 96 && (int64_t)dm_plane_lds(m) + 256 <= c->max_lds && dm_plane_jobs(m) <= 16;
}

template <bool FWD>
static int launch_plane(Ctx *c, const DmSolve &s, DmX &a) {
    DmPlan X, Y;
    VPMX_TRY(dm_plan(c, s.m[0], &X));
    VPMX_TRY(dm_plan(c, s.m[1], &Y));
    a.px = s.px;
    a.my = s.m[1];
    a.mz = s.m[2];
    a.wcs = s.wcs;
    a.pitch = dm_pitch(s.m[0] / 2 + 1);
    const size_t lds = dm_plane_lds(s.m);
    const dim3 g((unsigned)((s.m[2] + 7) / 8 * 16), (unsigned)s.ncomp);
    const int jobs = dm_plane_jobs(s.m);
    if (jobs <= 8) hipLaunchKernelGGL((k_dstm_plane<512, 1, FWD>), g, dim3(512), lds, c->stream, X, Y, a);
    else hipLaunchKernelGGL((k_dstm_plane<512, 2, FWD>), g, dim3(512), lds, c->stream, X, Y, a);
    VPMX_HIP(c, hipGetLastError());
    return VPMX_OK;
}

int dstm_plane_fwd(Ctx *c, const DmSolve &s, const GView &rhs, const GView *bc, const double ih2[3], double *w) {
    DmX a{};
    a.v = rhs;
    a.has_bc = bc ? 1 : 0;
    if (bc) a.bc = *bc;
    for (int d = 0; d < 3; d++) a.ih2[d] = ih2[d];
    a.w = w;
    return launch_plane<true>(c, s, a);
}
int dstm_plane_inv(Ctx *c, const DmSolve &s, const double *w, const GView &out) {
    DmX a{};
    a.v = out;
    a.w = const_cast<double *>(w);
    return launch_plane<false>(c, s, a);
}

template <bool FWD, class T>
static int launch_x(Ctx *c, const DmSolve &s, DmX &a) {
    DmPlan P;
    VPMX_TRY(dm_plan(c, s.m[0], &P));
    a.px = s.px;
    a.my = s.m[1];
    a.mz = s.m[2];
    a.wcs = s.wcs;
    a.pitch = dm_pitch(s.m[0]);
    const dim3 g((unsigned)((s.m[1] * s.m[2] + DM_XR - 1) / DM_XR), (unsigned)s.ncomp);
    const size_t lds = sizeof(double) * (size_t)(DM_XR * a.pitch);
    if (P.nrb <= DM_NW) hipLaunchKernelGGL((k_dstm_x<1, FWD, T>), g, dim3(DM_NT), lds, c->stream, P, a);
    else if (P.nrb <= 2 * DM_NW) hipLaunchKernelGGL((k_dstm_x<2, FWD, T>), g, dim3(DM_NT), lds, c->stream, P, a);
    else hipLaunchKernelGGL((k_dstm_x<3, FWD, T>), g, dim3(DM_NT), lds, c->stream, P, a);
    VPMX_HIP(c, hipGetLastError());
    return VPMX_OK;
}

int dstm_x_fwd(Ctx *c, const DmSolve &s, const GView &rhs, const GView *bc, const double ih2[3], void *w) {
    DmX a{};
    a.v = rhs;
    a.has_bc = bc ? 1 : 0;
    if (bc) a.bc = *bc;
    for (int d = 0; d < 3; d++) a.ih2[d] = ih2[d];
    a.w = w;
    return s.f32 ? launch_x<true, float>(c, s, a) : launch_x<true, double>(c, s, a);
}
int dstm_x_inv(Ctx *c, const DmSolve &s, const void *w, const GView &out) {
    DmX a{};
    a.v = out;
    a.w = const_cast<void *>(w);
    return s.f32 ? launch_x<false, float>(c, s, a) : launch_x<false, double>(c, s, a);
}

// The kernels of the y and z passes for 16 and 32 lines per work-group (the tuner's variants:
// the same bits, a column's sums do not depend on its tile), q row blocks per wave.
template <class T>
static const void *y_kernel(int q, int nb) {
    if (nb == 1)
        return q == 1 ? (const void *)k_dstm_y<1, 1, T> : q == 2 ? (const void *)k_dstm_y<2, 1, T>
                                                                 : (const void *)k_dstm_y<3, 1, T>;
    return q == 1 ? (const void *)k_dstm_y<1, 2, T> : q == 2 ? (const void *)k_dstm_y<2, 2, T>
                                                             : (const void *)k_dstm_y<3, 2, T>;
}
template <class TI, class TO, bool INV>
static const void *z_kernel(int q, int nb) {
    if (nb == 1)
        return q == 1 ? (const void *)k_dstm_z<1, 1, TI, TO, INV> : q == 2 ? (const void *)k_dstm_z<2, 1, TI, TO, INV>
                                                                          : (const void *)k_dstm_z<3, 1, TI, TO, INV>;
    return q == 1 ? (const void *)k_dstm_z<1, 2, TI, TO, INV> : q == 2 ? (const void *)k_dstm_z<2, 2, TI, TO, INV>
                                                                      : (const void *)k_dstm_z<3, 2, TI, TO, INV>;
}
static size_t line_lds(int m, int nb) { return sizeof(double) * (size_t)((m + DM_PAD) * 16 * nb); }

// Scratch of at least `bytes` for the tuner's trials, zero-filled when it grows.
static int trial_scratch(Ctx *c, size_t bytes) {
    if (c->tune_scratch.p && c->tune_scratch.bytes >= bytes) return VPMX_OK;
    int st = VPMX_OK;
    if (!ensure(c, c->tune_scratch, bytes, &st)) return st;
    return fill(c, (double *)c->tune_scratch.p, (int64_t)(c->tune_scratch.bytes / sizeof(double)), 0.0);
}

static int launch_timed(Ctx *c, bool timed, int kc, double work, const void *fn, dim3 g, void **args, size_t lds) {
    hipEvent_t e0, e1;
    if (timed && kernel_events(c, kc, &e0, &e1)) {
        c->k_work[kc] = work;
        VPMX_HIP(c, hipExtLaunchKernel(fn, g, dim3(DM_NT), args, lds, c->stream, e0, e1, 0));
    } else {
        VPMX_HIP(c, hipLaunchKernel(fn, g, dim3(DM_NT), args, lds, c->stream));
    }
    VPMX_HIP(c, hipGetLastError());
    return VPMX_OK;
}

int dstm_y(Ctx *c, const DmSolve &s, void *w, bool timed) {
    DmPlan P;
    VPMX_TRY(dm_plan(c, s.m[1], &P));
    const int q = (P.nrb + DM_NW - 1) / DM_NW;
    const void *fns[2] = {s.f32 ? y_kernel<float>(q, 2) : y_kernel<double>(q, 2),
                          s.f32 ? y_kernel<float>(q, 1) : y_kernel<double>(q, 1)};
    const char *names[2] = {"32 lines per work-group", "16 lines per work-group"};
    const size_t lds[2] = {line_lds(s.m[1], 2), line_lds(s.m[1], 1)};
    const int thr[2] = {DM_NT, DM_NT};
    const size_t word = s.f32 ? sizeof(float) : sizeof(double);
    int px = s.px;
    int64_t wcs = s.wcs;
    auto grid = [&](int v) {
        const int bn = v ? 16 : 32;
        return dim3((unsigned)((px + bn - 1) / bn), (unsigned)s.m[2], (unsigned)s.ncomp);
    };
    auto trial = [&](int v, int) -> int {
        VPMX_TRY(trial_scratch(c, word * (size_t)wcs * s.ncomp));
        void *t = c->tune_scratch.p;
        void *args[] = {&P, &t, &px, &wcs};
        VPMX_HIP(c, hipLaunchKernel(fns[v], grid(v), dim3(DM_NT), args, lds[v], c->stream));
        return VPMX_OK;
    };
    char key[160];
    std::snprintf(key, sizeof key, "sine transforms y pass %s matrix products m=%d,%d,%d comps=%d", s.f32 ? "FP32" : "FP64",
                  s.m[0], s.m[1], s.m[2], s.ncomp);
    Ctx::Tuned ch;
    VPMX_TRY(tune_v(c, key, 2, fns, names, lds, thr, trial, &ch, false));
    void *args[] = {&P, &w, &px, &wcs};
    return launch_timed(c, timed, K_DST, 2.0 * word * s.m[0] * s.m[1] * (double)s.m[2] * s.ncomp, fns[ch.fi], grid(ch.fi),
                        args, lds[ch.fi]);
}

int dstm_z(Ctx *c, const DmSolve &s, const void *w, void *wo, bool out32, const double *const lam[3], double norm,
           double *zsum, const double *zw, bool timed) {
    DmPlan P;
    VPMX_TRY(dm_plan(c, s.m[2], &P));
    DmZ a{};
    a.px = s.px;
    a.mx = s.m[0];
    a.my = s.m[1];
    a.wcs = s.wcs;
    a.pl = s.px * s.m[1];
    a.ncomp = s.ncomp;
    a.lx = lam[0];
    a.ly = lam[1];
    a.lz = lam[2];
    a.norm = norm;
    a.zsum = zsum;
    a.zw = zw;
    if (out32 && !s.f32) return fail(c, VPMX_ERR_ARG, "sine transforms: FP32 results of FP32 arrays only");
    const int q = (P.nrb + DM_NW - 1) / DM_NW;
    const void *fns[2];
    for (int v = 0; v < 2; v++) {
        const int nb = v ? 1 : 2;
        if (!s.f32) fns[v] = zsum ? z_kernel<double, double, false>(q, nb) : z_kernel<double, double, true>(q, nb);
        else if (out32) fns[v] = zsum ? z_kernel<float, float, false>(q, nb) : z_kernel<float, float, true>(q, nb);
        else fns[v] = zsum ? z_kernel<float, double, false>(q, nb) : z_kernel<float, double, true>(q, nb);
    }
    const char *names[2] = {"32 lines per work-group", "16 lines per work-group"};
    const size_t red = sizeof(double) * 2 * DM_NW * 32;  // the partial face sums
    const size_t lds[2] = {std::max(line_lds(s.m[2], 2), red), std::max(line_lds(s.m[2], 1), red)};
    const int thr[2] = {DM_NT, DM_NT};
    auto grid = [&](int v) {
        const int bn = v ? 16 : 32;
        return dim3((unsigned)((a.pl + bn - 1) / bn), (unsigned)s.ncomp);
    };
    const size_t wi = s.f32 ? sizeof(float) : sizeof(double), wq = out32 ? sizeof(float) : sizeof(double);
    const size_t np = (size_t)s.wcs * s.ncomp;
    auto trial = [&](int v, int) -> int {
        const size_t zb = zsum ? sizeof(double) * 2 * (size_t)s.ncomp * s.m[0] * s.m[1] : 0;
        VPMX_TRY(trial_scratch(c, (wi + wq) * np + zb));
        DmZ t = a;
        char *to = (char *)c->tune_scratch.p;  // (np is a multiple of 16: every part stays aligned)
        const void *ti = to + wq * np;
        if (zsum) t.zsum = (double *)(to + (wi + wq) * np);
        void *args[] = {&P, &t, &ti, &to};
        VPMX_HIP(c, hipLaunchKernel(fns[v], grid(v), dim3(DM_NT), args, lds[v], c->stream));
        return VPMX_OK;
    };
    char key[160];
    std::snprintf(key, sizeof key, "sine transforms z pass %s matrix products m=%d,%d,%d comps=%d%s",
                  !s.f32 ? "FP64" : (out32 ? "FP32" : "FP32/FP64"), s.m[0], s.m[1], s.m[2], s.ncomp,
                  zsum ? " (forward and diagonal, z-face sums)" : "");
    Ctx::Tuned ch;
    VPMX_TRY(tune_v(c, key, 2, fns, names, lds, thr, trial, &ch, false));
    void *args[] = {&P, &a, &w, &wo};
    return launch_timed(c, timed && !zsum, K_DSTZ, (double)(wi + wq) * s.m[0] * s.m[1] * s.m[2] * s.ncomp, fns[ch.fi],
                        grid(ch.fi), args, lds[ch.fi]);
}

}  // namespace vpmx
