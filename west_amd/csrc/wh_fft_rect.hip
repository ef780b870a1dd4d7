// Plane kernels for any n1 x n2 whose lengths are each a product of two of
// the radices 3, 4, 5, 6, 8, 9, 10, 12 (orthorhombic and slab cells: 40 x 54,
// 45 x 48 ...; every 2,3,5-smooth length from 15 to 108 but 75).
//
// Same step and stick layout as k_plane_vloc_t.  The lengths are run-time
// values, the radices select compiled butterflies, so a line is two LDS
// passes instead of the three or four of the radix-2/3/4/5 kernels, the zero
// padding, V(r) and the row selection are folded into the passes, and the
// inverse and forward a1 transforms meet in registers.
//
// What bounds it: instruction issue between barriers.  On 40 x 54 x 96 the
// vector ALUs are busy 58 % and the LDS 39 % of the cycles (27 % of those in bank
// conflicts), with 14 of 16 waves a CU resident and 0.8 TB/s of HBM traffic.
//  * Consecutive lanes take consecutive lines (not consecutive points): rows
//    and lines have odd strides of 16-byte elements, so neighbouring lanes of a
//    pass fall on other banks, and the twiddles of a butterfly are the
//    same for a whole line set (broadcast reads).  The potential must then be
//    contiguous along a2: real-space arrays of these plans are [a3][a1][a2].
//  * A pass is one butterfly per thread, staged in registers where it stores
//    over points that others load, so rows and lines need one LDS copy and
//    1,024 threads stay resident on a CU (passes between two LDS copies, with
//    a third of the lines: 25.5 ms against 19.5 ms for chi0 on 40 x 54 x 96;
//    the radix-2/3/4/5 kernels: 35.0 ms).
#include <mutex>

#include "wh_fft_pass2.h"
#include "wh_fft_rect.h"

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

__device__ __forceinline__ z64* rect_base() {
  extern __shared__ char smem_raw[];
  return reinterpret_cast<z64*>(smem_raw);
}

// nz planes of sticks into zeroed rows
template <int NT>
__device__ __forceinline__ void rect_fill(const StickPlanDev& P, const RectPlan& Q, const RectLds& S, const z64* src,
                                          int nz) {
  const int pe = P.nrows * Q.rs2;
  for (int t = threadIdx.x; t < nz * pe; t += NT) S.pl[t] = mk(0.0, 0.0);
  __syncthreads();
  for (int p = 0; p < nz; ++p)
    for (int c = threadIdx.x; c < P.nct; c += NT) {
      const int pos = P.col_pos[c];
      const int r = fdiv(pos, Q.inv_n2);
      S.pl[p * pe + r * Q.rs2 + (pos - r * P.n2)] = src[static_cast<long>(p) * P.nct + c];
    }
  __syncthreads();
}

// sticks -> (V(r) * .) -> sticks
template <int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_rect_vloc(
    StickPlanDev P, RectPlan Q, const FftItem* items, const z64* sin, z64* sout, const double* vpot, long ldpot,
    double scale) {
  const FftItem item = items[blockIdx.y];
  if (item.a < 0) return;   // inactive item (uniform per workgroup)
  const int z0 = blockIdx.x * Q.pz;
  const int nz = min(Q.pz, P.n3 - z0);
  const long sl = static_cast<long>(P.n3) * P.nct;
  const RectLds S = rect_lds<NT>(P, Q, Q.pz, rect_base());
  rect_fill<NT>(P, Q, S, sin + static_cast<long>(item.a) * sl + static_cast<long>(z0) * P.nct, nz);
  const double* V = vpot + (item.pot >= 0 ? static_cast<long>(item.pot) * ldpot : 0L) +
                    static_cast<long>(z0) * P.n1 * P.n2;
  rect_local<NT>(P, Q, S, nz, V, scale);
  const int n2 = P.n2, rs = Q.rs2, pe = P.nrows * rs;
  const float inv_n2 = Q.inv_n2;
  const z64* pl = S.pl;
  z64* dst = sout + static_cast<long>(blockIdx.y) * sl + static_cast<long>(z0) * P.nct;
  for (int p = 0; p < nz; ++p)
    for (int c = threadIdx.x; c < P.nct; c += NT) {
      const int pos = P.col_pos[c];
      const int r = fdiv(pos, inv_n2);
      dst[static_cast<long>(p) * P.nct + c] = pl[p * pe + r * rs + (pos - r * n2)];
    }
}

// inverse a1 transforms of one plane's rows; out(x, y, value) takes the grid
template <int NT, class Out>
__device__ __forceinline__ void rect_to_grid(const StickPlanDev& P, const RectPlan& Q, const RectLds& S, Out out) {
  const int n1 = P.n1, imax = P.imax, rs = Q.rs2, xs = Q.xs;
  z64 *wa = S.wa, *pl = S.pl;
  for (int y0 = 0; y0 < P.n2; y0 += Q.nj) {
    const int nl = min(Q.nj, P.n2 - y0);
    pass2<NT, +1, PASS_FIRST, false>(nl, Q.r10, Q.r11, S.tw1,
                                 [=](int l, int x) {
                                   const int r = rect_row(x, n1, imax);
                                   return r >= 0 ? pl[r * rs + y0 + l] : mk(0.0, 0.0);
                                 },
                                 no_mid, [=](int l, int x, z64 v) { wa[l * xs + x] = v; });
    __syncthreads();
    pass2<NT, +1, PASS_LAST, false>(nl, Q.r11, Q.r10, S.tw1, [=](int l, int x) { return wa[l * xs + x]; }, no_mid,
                                [=](int l, int x, z64 v) { out(x, y0 + l, v); });
    __syncthreads();
  }
}

// sticks -> real-space grid: Re -> row a, Im -> row b (if b >= 0)
template <int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_rect_to_real(
    StickPlanDev P, RectPlan Q, const FftItem* items, const z64* sin, double* out, long ldout) {
  const int z = blockIdx.x;
  const FftItem item = items[blockIdx.y];
  if (item.a < 0) return;   // inactive item (uniform per workgroup)
  const long sl = static_cast<long>(P.n3) * P.nct;
  const RectLds S = rect_lds<NT>(P, Q, 1, rect_base());
  rect_fill<NT>(P, Q, S, sin + static_cast<long>(blockIdx.y) * sl + static_cast<long>(z) * P.nct, 1);
  rect_rows<NT, +1>(P, Q, S, P.nrows);
  const long o = static_cast<long>(z) * P.n1 * P.n2;
  double* oa = out + static_cast<long>(item.a) * ldout + o;
  double* ob = item.b >= 0 ? out + static_cast<long>(item.b) * ldout + o : nullptr;
  const int n2 = P.n2;
  rect_to_grid<NT>(P, Q, S, [=](int x, int y, z64 v) {
    oa[x * n2 + y] = v.x;
    if (ob) ob[x * n2 + y] = v.y;
  });
}

// dn(r) = sum_v occ_v Re(psic_v) Im(psic_v), psic_v from the sticks of
// (psi_v + i dpsi_v); dn back to sticks.  sticks_in slot = p nband + v.
template <int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_rect_density(
    StickPlanDev P, RectPlan Q, int nband, const z64* sin, const double* occ, z64* sout) {
  const int z = blockIdx.x;
  const int pp = blockIdx.y;
  const long sl = static_cast<long>(P.n3) * P.nct;
  const RectLds S = rect_lds<NT>(P, Q, 1, rect_base());
  const int n1 = P.n1, n2 = P.n2, imax = P.imax, rs = Q.rs2, xs = Q.xs;
  double* acc = S.acc;
  for (int t = threadIdx.x; t < n1 * n2; t += NT) acc[t] = 0.0;
  for (int v = 0; v < nband; ++v) {
    rect_fill<NT>(P, Q, S, sin + (static_cast<long>(pp) * nband + v) * sl + static_cast<long>(z) * P.nct, 1);
    rect_rows<NT, +1>(P, Q, S, P.nrows);
    const double o = occ[v];
    // each (x, y) belongs to one thread within a band, and a barrier ends every pass
    rect_to_grid<NT>(P, Q, S, [=](int x, int y, z64 w) { acc[x * n2 + y] += o * w.x * w.y; });
  }
  z64 *wa = S.wa, *pl = S.pl;
  for (int y0 = 0; y0 < n2; y0 += Q.nj) {
    const int nl = min(Q.nj, n2 - y0);
    pass2<NT, -1, PASS_FIRST, false>(nl, Q.r11, Q.r10, S.tw1, [=](int l, int x) { return mk(acc[x * n2 + y0 + l], 0.0); },
                                 no_mid, [=](int l, int x, z64 v) { wa[l * xs + x] = v; });
    __syncthreads();
    pass2<NT, -1, PASS_LAST, false>(nl, Q.r10, Q.r11, S.tw1, [=](int l, int x) { return wa[l * xs + x]; }, no_mid,
                                [=](int l, int x, z64 v) {
                                  const int r = rect_row(x, n1, imax);
                                  if (r >= 0) pl[r * rs + y0 + l] = v;
                                });
    __syncthreads();
  }
  rect_rows<NT, -1>(P, Q, S, P.nrows);
  z64* dst = sout + static_cast<long>(pp) * sl + static_cast<long>(z) * P.nct;
  for (int c = threadIdx.x; c < P.nct; c += NT) {
    const int pos = P.col_pos[c];
    const int r = fdiv(pos, Q.inv_n2);
    dst[c] = pl[r * rs + (pos - r * n2)];
  }
}

// 32 x 33 tiles through LDS, both sides in runs along the fastest axis
__global__ __launch_bounds__(256) void k_transpose_planes(int n1, int n2, const double* in, double* out) {
  __shared__ double t[32][33];
  const long o = static_cast<long>(blockIdx.z) * n1 * n2;
  const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 32;
  const int lx = threadIdx.x & 31, ly = threadIdx.x >> 5;
  for (int y = ly; y < 32; y += 8)
    if (x0 + lx < n1 && y0 + y < n2) t[y][lx] = in[o + static_cast<long>(y0 + y) * n1 + x0 + lx];
  __syncthreads();
  for (int x = ly; x < 32; x += 8)
    if (x0 + x < n1 && y0 + lx < n2) out[o + static_cast<long>(x0 + x) * n2 + y0 + lx] = t[lx][x];
}

template <auto K>
void rect_smem_attr(size_t bytes) {
  static std::mutex mu;
  static size_t done = 0;
  std::lock_guard<std::mutex> lk(mu);
  if (done >= bytes) return;
  WH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(K), hipFuncAttributeMaxDynamicSharedMemorySize,
                             static_cast<int>(bytes)));
  done = bytes;
}

size_t rect_smem(const StickPlanDev& P, const RectPlan& Q, int pz, bool density) {
  return sizeof(z64) * (static_cast<size_t>(P.n1) + P.n2 + static_cast<size_t>(pz) * P.nrows * Q.rs2 +
                        static_cast<size_t>(Q.nj) * Q.xs) +
         (density ? sizeof(double) * static_cast<size_t>(P.n1) * P.n2 : 0);
}

constexpr size_t kLds = 160u * 1024u;

template <class F>
void rect_nt(const RectPlan& q, F&& launch) {
  if (q.nt == 256) launch(std::integral_constant<int, 256>{});
  else launch(std::integral_constant<int, 512>{});
  WH_HIP(hipGetLastError());
}

}  // namespace

void rect_plan(const StickPlanDev& P, RectPlan& q) {
  q = RectPlan{};
  // (the a1 turn, which holds two transforms, takes the smaller radix)
  if (!two_radices(P.n1, q.r10, q.r11) || !two_radices(P.n2, q.r20, q.r21)) return;
  q.rs2 = P.n2 | 1;
  q.xs = P.n1 | 1;
  q.inv_n2 = 1.0f / static_cast<float>(P.n2);
  // Workgroup size, planes a workgroup and a1 lines a pass: the fewest barrier
  // steps per plane over the workgroups that a CU holds (LDS, and registers
  // for four waves a SIMD), a step costing more the more threads it keeps
  // busy.  40 x 54 (chi0 of 8 perturbations, 40 bands, 96 planes): 256 threads,
  // one plane, 27 lines, four workgroups a CU 19.5 ms; 512 threads, two
  // planes, 54 lines 20.2; 512 and one plane 21.9; 1024 and four planes 21.8.
  double best = 0.0;
  RectPlan pick = q;
  for (int nt : {256, 512}) {
    const int lines1 = nt / std::max(q.r10, q.r11), lines2 = nt / std::max(q.r20, q.r21);
    for (int pz = 1; pz <= 4 && pz <= P.n3; ++pz)
      for (int most = std::min(lines1, pz * P.n2); most >= 4; most = most * 3 / 4) {
        RectPlan t = q;
        const int nch = ceil_div(pz * P.n2, most), rch = ceil_div(pz * P.nrows, std::min(lines2, pz * P.nrows));
        t.nt = nt;
        t.pz = pz;
        t.nj = ceil_div(pz * P.n2, nch);   // even chunks
        t.nrc = ceil_div(pz * P.nrows, rch);
        const size_t sm = rect_smem(P, t, pz, false);
        if (sm > kLds || rect_smem(P, t, 1, true) > kLds) continue;
        const int wgs = std::min<int>(static_cast<int>(kLds / sm), 1024 / nt);
        const double busy = std::min(1.0, wgs * t.nj * 0.5 * (q.r10 + q.r11) / 1024.0);
        const double cost = (3 * nch + 4 * rch + 2) * (0.4 + 0.6 * busy) / (pz * wgs);
        if (best == 0.0 || cost < best) {
          best = cost;
          pick = t;
        }
      }
  }
  q = pick;
  q.ok = best > 0.0;
}

void rect_plane_vloc(const StickPlanDev& P, const RectPlan& q, const FftItem* items, int n, const z64* sin, z64* sout,
                     const double* vpot, long ldpot, double scale, hipStream_t s) {
  const size_t sm = rect_smem(P, q, q.pz, false);
  rect_nt(q, [&](auto Nt) {
    constexpr int NT = decltype(Nt)::value;
    rect_smem_attr<k_rect_vloc<NT>>(sm);
    k_rect_vloc<NT><<<dim3(ceil_div(P.n3, q.pz), n), NT, sm, s>>>(P, q, items, sin, sout, vpot, ldpot, scale);
  });
}

void rect_plane_to_real(const StickPlanDev& P, const RectPlan& q, const FftItem* items, int n, const z64* sin,
                        double* out, long ldout, hipStream_t s) {
  const size_t sm = rect_smem(P, q, 1, false);
  rect_nt(q, [&](auto Nt) {
    constexpr int NT = decltype(Nt)::value;
    rect_smem_attr<k_rect_to_real<NT>>(sm);
    k_rect_to_real<NT><<<dim3(P.n3, n), NT, sm, s>>>(P, q, items, sin, out, ldout);
  });
}

void rect_plane_density(const StickPlanDev& P, const RectPlan& q, int npert, int nband, const z64* sin,
                        const double* occ, z64* sout, hipStream_t s) {
  const size_t sm = rect_smem(P, q, 1, true);
  rect_nt(q, [&](auto Nt) {
    constexpr int NT = decltype(Nt)::value;
    rect_smem_attr<k_rect_density<NT>>(sm);
    k_rect_density<NT><<<dim3(P.n3, npert), NT, sm, s>>>(P, q, nband, sin, occ, sout);
  });
}

void rect_transpose_grid(int n1, int n2, int n3, const double* in, double* out, hipStream_t s) {
  k_transpose_planes<<<dim3(ceil_div(n1, 32), ceil_div(n2, 32), n3), 256, 0, s>>>(n1, n2, in, out);
  WH_HIP(hipGetLastError());
}

}  // namespace wh
