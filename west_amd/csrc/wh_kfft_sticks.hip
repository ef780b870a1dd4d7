// z transforms of the k-point local term: sphere <-> sticks for complex
// functions on |k+G| spheres, several k points in one launch.
//
// The operator at k on grids beyond the LDS: sphere -> sticks (a3 lines of
// the columns that hold points) -> the plane kernels of the Gamma path, which
// see one complex function per item -> sticks -> sphere.  A 36^3 grid (8 atoms,
// 25 Ry) has 2,300 points in 300 columns, so a band moves 0.17 MB of sticks
// four times where full-grid transforms moved 0.75 MB fourteen times.
//
// Bound by memory (3.7 TB/s inverse, 4.4 forward, of the 4.4 that a large copy
// reaches).  A workgroup takes CW columns: lane -> column,
// so the sticks are read and written in runs of 16 CW bytes and the first
// (zfwd) and last (zinv) pass touch global memory directly; LDS holds the
// lines between the two passes and the sphere side.
#include "wh_fft_pass2.h"
#include "wh_fft.h"

namespace wh {

namespace {

constexpr int KZT = 256;

struct KzShape {
  int r0, r1;   // n3 = r0 r1
  int cw;       // columns per workgroup
  int ls;       // line stride (odd)
};

bool kz_shape(int n3, KzShape& q) {
  if (!two_radices(n3, q.r0, q.r1)) return false;
  q.cw = KZT / std::max(q.r0, q.r1);
  q.cw -= q.cw % 8;   // whole 128-byte lines of a stick row
  q.ls = n3 | 1;
  return q.cw >= 8 && sizeof(z64) * (static_cast<size_t>(n3) + static_cast<size_t>(q.cw) * q.ls) <= 64u * 1024u;
}

__device__ __forceinline__ const KStick& kz_stick(const KStick* tab, const int* l2i, int cols_per_k, int b) {
  return tab[cols_per_k > 0 ? (l2i ? l2i[b] : b) / cols_per_k : 0];
}

__global__ __launch_bounds__(KZT) void k_kzinv(StickPlanDev P, KzShape Q, const KStick* __restrict__ tab,
                                               const int* __restrict__ l2i, int cols_per_k, int b0,
                                               const int* __restrict__ d_nc, const z64* __restrict__ x, long ld,
                                               z64* __restrict__ sticks) {
  extern __shared__ char smem_raw[];
  const int b = b0 + blockIdx.y;
  if (d_nc && b >= *d_nc) return;   // uniform per workgroup
  const KStick K = kz_stick(tab, l2i, cols_per_k, b);
  z64* tw = reinterpret_cast<z64*>(smem_raw);
  z64* lines = tw + P.n3;
  const int n3 = P.n3, ls = Q.ls;
  const int c0 = blockIdx.x * Q.cw;
  const int nl = min(Q.cw, P.nct - c0);
  for (int t = threadIdx.x; t < n3; t += KZT) tw[t] = reinterpret_cast<const z64*>(P.tw3)[t];
  for (int t = threadIdx.x; t < nl * ls; t += KZT) lines[t] = mk(0.0, 0.0);
  __syncthreads();
  const z64* xb = x + b * ld;
  const int s1 = K.col_off[c0 + nl];
  for (int s = K.col_off[c0] + threadIdx.x; s < s1; s += KZT) {
    const int k = K.pt_k[s];
    lines[(K.pt_col[s] - c0) * ls + (k < 0 ? k + n3 : k)] = xb[s];
  }
  __syncthreads();
  auto ld_l = [=](int l, int z) { return lines[l * ls + z]; };
  pass2<KZT, +1, PASS_FIRST, true>(nl, Q.r0, Q.r1, tw, ld_l, no_mid,
                                   [=](int l, int z, z64 v) { lines[l * ls + z] = v; });
  __syncthreads();
  z64* out = sticks + static_cast<long>(blockIdx.y) * n3 * P.nct + c0;
  const int nct = P.nct;
  pass2<KZT, +1, PASS_LAST, false>(nl, Q.r1, Q.r0, tw, ld_l, no_mid,
                                   [=](int l, int z, z64 v) { out[z * nct + l] = v; });
}

__global__ __launch_bounds__(KZT) void k_kzfwd(StickPlanDev P, KzShape Q, const KStick* __restrict__ tab,
                                               const int* __restrict__ l2i, int cols_per_k, int b0,
                                               const int* __restrict__ d_nc, const z64* __restrict__ sticks,
                                               const z64* __restrict__ x, const double* __restrict__ e,
                                               z64* __restrict__ t, long ld) {
  extern __shared__ char smem_raw[];
  const int b = b0 + blockIdx.y;
  if (d_nc && b >= *d_nc) return;   // uniform per workgroup
  const KStick K = kz_stick(tab, l2i, cols_per_k, b);
  z64* tw = reinterpret_cast<z64*>(smem_raw);
  z64* lines = tw + P.n3;
  const int n3 = P.n3, ls = Q.ls, nct = P.nct;
  const int c0 = blockIdx.x * Q.cw;
  const int nl = min(Q.cw, nct - c0);
  for (int i = threadIdx.x; i < n3; i += KZT) tw[i] = reinterpret_cast<const z64*>(P.tw3)[i];
  const z64* src = sticks + static_cast<long>(blockIdx.y) * n3 * nct + c0;
  pass2<KZT, -1, PASS_FIRST, false>(nl, Q.r0, Q.r1, tw, [=](int l, int z) { return src[z * nct + l]; }, no_mid,
                                    [=](int l, int z, z64 v) { lines[l * ls + z] = v; });
  __syncthreads();
  pass2<KZT, -1, PASS_LAST, false>(nl, Q.r1, Q.r0, tw, [=](int l, int z) { return lines[l * ls + z]; }, no_mid,
                                   [=](int l, int z, z64 v) { lines[l * ls + z] = v; });
  __syncthreads();
  const double eb = e[b];
  const z64* xb = x + b * ld;
  z64* tb = t + b * ld;
  const int s1 = K.col_off[c0 + nl];
  for (int s = K.col_off[c0] + threadIdx.x; s < s1; s += KZT) {
    const int k = K.pt_k[s];
    tb[s] = lines[(K.pt_col[s] - c0) * ls + (k < 0 ? k + n3 : k)] + cscale(xb[s], K.g2[s] - eb);
  }
  if (blockIdx.x == 0)
    for (long s = K.npw + threadIdx.x; s < ld; s += KZT) tb[s] = mk(0.0, 0.0);
}

}  // namespace

bool kz_available(int n3) {
  KzShape q;
  return kz_shape(n3, q);
}

void launch_kzinv(const StickPlan& p, const KStick* tab, const int* l2i, int cols_per_k, int c0, int n,
                  const int* d_nc, const z64* x, long ld, z64* sticks, hipStream_t s) {
  if (n <= 0) return;
  KzShape q;
  WH_REQUIRE(kz_shape(p.dev.n3, q), "no k-point z kernel for this grid length");
  const size_t sm = sizeof(z64) * (p.dev.n3 + static_cast<size_t>(q.cw) * q.ls);
  k_kzinv<<<dim3(ceil_div(p.dev.nct, q.cw), n), KZT, sm, s>>>(p.dev, q, tab, l2i, cols_per_k, c0, d_nc, x, ld,
                                                              sticks);
  WH_HIP(hipGetLastError());
}

void launch_kzfwd(const StickPlan& p, const KStick* tab, const int* l2i, int cols_per_k, int c0, int n,
                  const int* d_nc, const z64* sticks, const z64* x, const double* e, z64* t, long ld, hipStream_t s) {
  if (n <= 0) return;
  KzShape q;
  WH_REQUIRE(kz_shape(p.dev.n3, q), "no k-point z kernel for this grid length");
  const size_t sm = sizeof(z64) * (p.dev.n3 + static_cast<size_t>(q.cw) * q.ls);
  k_kzfwd<<<dim3(ceil_div(p.dev.nct, q.cw), n), KZT, sm, s>>>(p.dev, q, tab, l2i, cols_per_k, c0, d_nc, sticks, x, e,
                                                              t, ld);
  WH_HIP(hipGetLastError());
}

}  // namespace wh
