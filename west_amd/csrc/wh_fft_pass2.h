// Two-pass line transforms of run-time length n = r0 r1 with compiled
// butterflies (radices 3, 4, 5, 6, 8, 9, 10, 12), one butterfly per thread.
#pragma once

#include "wh_fft_dev.h"

namespace wh {
namespace {

// a / d for 0 <= a < 2^20 with inv = 1 / d: (a + 1/2) / d lies at least 1/(2d)
// from an integer, more than the rounding of the product
__device__ __forceinline__ int fdiv(int a, float inv) { return static_cast<int>((static_cast<float>(a) + 0.5f) * inv); }

template <class F>
__device__ __forceinline__ void with_radix(int r, F&& f) {
  switch (r) {
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    default: f(std::integral_constant<int, 12>{}); break;
  }
}

// v[j] *= exp(DIR 2 pi i j k / n), tw the forward roots of n
template <int R, int DIR>
__device__ __forceinline__ void twiddle(z64* v, const z64* tw, int k) {
  if (k == 0) return;
#pragma unroll
  for (int j = 1; j < R; ++j) {
    z64 w = tw[j * k];
    if (DIR > 0) w.y = -w.y;
    v[j] = cmul(v[j], w);
  }
}

// One pass over nl lines of a length n = r m (m butterflies of radix r a line,
// nl m <= NT, the workgroup).  FIRST: butterfly i takes the points i + j m and leaves the
// result at i r + j; otherwise (the second and last pass) it takes the points
// i + j m after the first pass's radix m, twiddles them and leaves them in
// place.  mid (the turn): the inverse's last pass, mid(line, point, value) and
// the first pass of the forward transform, whose radices are in reverse order.
// STAGE: the stores may hit what another thread loads, so a barrier separates
// the two.
enum PassKind : int { PASS_FIRST, PASS_LAST, PASS_TURN };
template <int NT, int DIR, PassKind KIND, bool STAGE, class Ld, class Mid, class St>
__device__ __forceinline__ void pass2(int nl, int r, int m, const z64* tw, Ld ld, Mid mid, St st) {
  const int bf = threadIdx.x;
  const int i = fdiv(bf, 1.0f / static_cast<float>(nl));
  const int line = bf - i * nl;
  const bool on = bf < nl * m;
  with_radix(r, [&](auto Rc) {
    constexpr int R = decltype(Rc)::value;
    z64 v[R];
    if (on) {
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = ld(line, i + j * m);
    }
    if (STAGE) __syncthreads();
    if (on) {
      if (KIND != PASS_FIRST) twiddle<R, DIR>(v, tw, i);
      dft<double, R, DIR>(v);
      if (KIND == PASS_TURN) {
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = mid(line, i + j * m, v[j]);
        dft<double, R, -DIR>(v);
      }
#pragma unroll
      for (int j = 0; j < R; ++j) st(line, KIND == PASS_LAST ? i + j * m : i * R + j, v[j]);
    }
  });
}
__device__ __forceinline__ z64 no_mid(int, int, z64 v) { return v; }

// the most even pair of radices, the larger one first; false where there is none
inline bool two_radices(int n, int& r0, int& r1) {
  r0 = r1 = 0;
  for (int r : {12, 10, 9, 8, 6, 5, 4, 3})
    if (n % r == 0) {
      const int q = n / r;
      if (q > r) break;
      for (int a : {12, 10, 9, 8, 6, 5, 4, 3})
        if (a == q) {
          r0 = r;
          r1 = q;
        }
    }
  return r0 != 0;
}

}  // namespace
}  // namespace wh
