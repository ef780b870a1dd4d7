// Device side of the two-radix plane transforms (wh_fft_rect.hip), shared with
// the kernels that keep a whole column's sticks in LDS (wh_kfft_lds.hip).
#pragma once

#include "wh_fft.h"
#include "wh_fft_pass2.h"

namespace wh {
namespace {

struct RectLds {
  z64* tw1;
  z64* tw2;
  z64* pl;   // [pz][nrows][rs2]
  z64* wa;   // a1 lines [nj][xs]
  double* acc;   // density: [n1][n2]
};

// at `base` in LDS; loads the twiddles (the caller's barrier after)
template <int NT>
__device__ __forceinline__ RectLds rect_lds(const StickPlanDev& P, const RectPlan& Q, int pz, z64* base) {
  RectLds S;
  S.tw1 = base;
  S.tw2 = S.tw1 + P.n1;
  S.pl = S.tw2 + P.n2;
  S.wa = S.pl + pz * P.nrows * Q.rs2;
  S.acc = reinterpret_cast<double*>(S.wa + Q.nj * Q.xs);
  const z64* t1 = reinterpret_cast<const z64*>(P.tw1);
  const z64* t2 = reinterpret_cast<const z64*>(P.tw2);
  for (int t = threadIdx.x; t < P.n1; t += NT) S.tw1[t] = t1[t];
  for (int t = threadIdx.x; t < P.n2; t += NT) S.tw2[t] = t2[t];
  return S;
}

// a2 transforms of the rows in place, Q.nrc rows at a time
template <int NT, int DIR>
__device__ __forceinline__ void rect_rows(const StickPlanDev& P, const RectPlan& Q, const RectLds& S, int nrow_all) {
  const int rs = Q.rs2;
  for (int q0 = 0; q0 < nrow_all; q0 += Q.nrc) {
    const int nl = min(Q.nrc, nrow_all - q0);
    z64* rows = S.pl + q0 * rs;
    auto ld = [=](int l, int x) { return rows[l * rs + x]; };
    auto st = [=](int l, int x, z64 v) { rows[l * rs + x] = v; };
    pass2<NT, DIR, PASS_FIRST, true>(nl, Q.r20, Q.r21, S.tw2, ld, no_mid, st);
    __syncthreads();
    pass2<NT, DIR, PASS_LAST, false>(nl, Q.r21, Q.r20, S.tw2, ld, no_mid, st);
  }
  __syncthreads();
}

// row of the sphere holding a1-frequency x, or -1
__device__ __forceinline__ int rect_row(int x, int n1, int imax) {
  if (x <= imax) return x + imax;
  if (x >= n1 - imax) return x - n1 + imax;
  return -1;
}

// the planes' rows: inverse along a2 and a1, times V scale, forward along a1
// and a2 (V at the first plane; the caller's barrier before, this one's after)
template <int NT>
__device__ __forceinline__ void rect_local(const StickPlanDev& P, const RectPlan& Q, const RectLds& S, int nz,
                                           const double* __restrict__ V, double scale) {
  rect_rows<NT, +1>(P, Q, S, nz * P.nrows);
  const int n1 = P.n1, n2 = P.n2, imax = P.imax, rs = Q.rs2, xs = Q.xs, pe = P.nrows * rs;
  const float inv_n2 = Q.inv_n2;
  z64 *wa = S.wa, *pl = S.pl;
  // a1 lines (plane p, second-axis position y): Q.nj at a time
  for (int l0 = 0; l0 < nz * n2; l0 += Q.nj) {
    const int nl = min(Q.nj, nz * n2 - l0);
    auto col = [=](int l) {
      const int p = fdiv(l0 + l, inv_n2);
      return pl + p * pe + (l0 + l - p * n2);
    };
    auto in_wa = [=](int l, int x) { return wa[l * xs + x]; };
    auto to_wa = [=](int l, int x, z64 v) { wa[l * xs + x] = v; };
    pass2<NT, +1, PASS_FIRST, false>(nl, Q.r10, Q.r11, S.tw1,
                                 [=](int l, int x) {
                                   const int r = rect_row(x, n1, imax);
                                   return r >= 0 ? col(l)[r * rs] : mk(0.0, 0.0);
                                 },
                                 no_mid, to_wa);
    __syncthreads();
    pass2<NT, +1, PASS_TURN, true>(nl, Q.r11, Q.r10, S.tw1, in_wa,
                               [=](int l, int x, z64 v) {
                                 const int p = fdiv(l0 + l, inv_n2);
                                 return cscale(v, V[(p * n1 + x) * n2 + (l0 + l - p * n2)] * scale);
                               },
                               to_wa);
    __syncthreads();
    pass2<NT, -1, PASS_LAST, false>(nl, Q.r10, Q.r11, S.tw1, in_wa, no_mid, [=](int l, int x, z64 v) {
      const int r = rect_row(x, n1, imax);
      if (r >= 0) col(l)[r * rs] = v;
    });
    __syncthreads();
  }
  rect_rows<NT, -1>(P, Q, S, nz * P.nrows);
}

}  // namespace
}  // namespace wh
