// DST-I passes as products with the sine matrix on the FP64 matrix cores (k_dstm.hip).
#pragma once
#include "vpmx_internal.h"

namespace vpmx {

// One Dirichlet solve's arrays: interior extents m, work array (mx, my, mz) per component with
// row pitch px (a multiple of 16) and component stride wcs, FP32 values when f32 (the sums are
// FP64 either way).
struct DmSolve {
    int m[3];
    int px;
    int64_t wcs;
    int ncomp;
    bool f32;
};

// Whether the x and y transforms of a plane fit one work-group (k_dstm_plane), and whether lines
// of m points take the matrix passes at all (forward: a pass of the forward transform alone).
bool dstm_plane_fits(const Ctx *c, const int m[3]);
bool dstm_line_fits(int m, bool f32, bool forward = false);

// RHS (interior of the view, Dirichlet values of bc folded in) -> x and y transforms in w; and
// back: x and y transforms of w into the interior of out.  One launch each (FP64 arrays).
int dstm_plane_fwd(Ctx *c, const DmSolve &s, const GView &rhs, const GView *bc, const double ih2[3], double *w);
int dstm_plane_inv(Ctx *c, const DmSolve &s, const double *w, const GView &out);
// Single passes: x forward from the RHS view, x inverse into the output view, y in place.
int dstm_x_fwd(Ctx *c, const DmSolve &s, const GView &rhs, const GView *bc, const double ih2[3], void *w);
int dstm_x_inv(Ctx *c, const DmSolve &s, const void *w, const GView &out);
int dstm_y(Ctx *c, const DmSolve &s, void *w, bool timed);
// z forward, diagonal, z inverse from w to wo (FP32 when out32; may be w when of one type).  With
// zsum: forward and diagonal only, wo receives the spectrum and zsum[side][comp][ky][kx] its
// sums with the weights zw (side 1: (-1)^(k+1) zw).
int dstm_z(Ctx *c, const DmSolve &s, const void *w, void *wo, bool out32, const double *const lam[3], double norm,
           double *zsum, const double *zw, bool timed);

}  // namespace vpmx
