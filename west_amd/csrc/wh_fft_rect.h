// Plane kernels for grids whose first two lengths differ or are not compiled
// sizes (declarations; wh_fft_rect.hip).
#pragma once

#include "wh_fft.h"

namespace wh {

// Fills p for the plan's first two axes; p.ok stays false where one of them is
// not a product of two radices of the kernels or a plane does not fit the LDS.
void rect_plan(const StickPlanDev& P, RectPlan& p);

// Same contracts as launch_plane_vloc / to_real / density, except that every
// real-space array (the potentials, the real grids) is laid out [a3][a1][a2],
// the second axis fastest.
void rect_plane_vloc(const StickPlanDev& P, const RectPlan& p, const FftItem* items, int n, const z64* sin, z64* sout,
                     const double* vpot, long ldpot, double scale, hipStream_t s);
void rect_plane_to_real(const StickPlanDev& P, const RectPlan& p, const FftItem* items, int n, const z64* sin,
                        double* out, long ldout, hipStream_t s);
void rect_plane_density(const StickPlanDev& P, const RectPlan& p, int npert, int nband, const z64* sin,
                        const double* occ, z64* sout, hipStream_t s);

// out[a3][a1][a2] = in[a3][a2][a1] (QE's grids, first axis fastest)
void rect_transpose_grid(int n1, int n2, int n3, const double* in, double* out, hipStream_t s);

}  // namespace wh
