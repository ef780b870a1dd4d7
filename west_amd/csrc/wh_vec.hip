// Vector kernels of the Sternheimer CG and the dfpt data movement (FP64).
//
// Vectors are rows of npw complex numbers in stick order (G = 0 first).
// Gamma inner products follow the reference: 2 Re sum a* b - Re a(G=0) Re b(G=0)
// (DFPT_kernel/linsolve_sternheimer_m_wfcts.f90:162-181, 253-276).
#include "wh_vec.h"

#include <type_traits>

namespace wh {

namespace {

constexpr int NT = 256;

// sum over the block (BT threads): wavefront reduction, then across the
// wavefronts in a fixed order
template <int BT = NT>
__device__ __forceinline__ double block_sum(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < BT / 64; ++i) s += red[i];
  return s;
}

__device__ __forceinline__ double gamma_dot_part(const z64* a, const z64* b, int npw) {
  double s = 0.0;
  for (int g = threadIdx.x; g < npw; g += NT) s += a[g].x * b[g].x + a[g].y * b[g].y;
  return s;
}

// rho[lb] = <M^-1 g|g> with M^-1 g = g[ib] / max(1, g2kin/eprec[ib])   (linsolve 150-181);
// M^-1 g itself is formed again by k_direction (one read of g here instead of
// a read of g and a write and re-read of M^-1 g).
// V is the vector precision; the inner products are summed in FP64.
template <typename V>
__global__ __launch_bounds__(NT) void k_prec_rho(int npw, int gstart, const int* l2i, const cplx<V>* g, long ld,
                                                 const double* g2kin, const double* eprec, double* rho,
                                                 bool by_band, const int* d_nc = nullptr) {
  __shared__ double red[NT / 64];
  const int lb = blockIdx.x;
  if (d_nc && lb >= *d_nc) return;   // uniform per workgroup
  const int ib = l2i[lb];
  const cplx<V>* gi = g + static_cast<long>(ib) * ld;
  const double ep = eprec[ib];
  double s = 0.0, r0 = 0.0;
  for (int q = threadIdx.x; q < npw; q += NT) {
    const V f = V(1.0 / fmax(1.0, g2kin[q] / ep));
    const cplx<V> gv = gi[q];
    const cplx<V> hv = mk<V>(gv.x * f, gv.y * f);
    s += static_cast<double>(hv.x) * gv.x + static_cast<double>(hv.y) * gv.y;
    if (q == 0) r0 = static_cast<double>(hv.x) * gv.x;
  }
  s = block_sum(s, red);
  r0 = block_sum(r0, red);
  if (threadIdx.x == 0) rho[by_band ? ib : lb] = 2.0 * s - (gstart == 2 ? r0 : 0.0);
}

// h[ib] = -M^-1 g[ib] + beta[lb] hold[ib];  bc[lb] = h[ib]   (linsolve 150-157, 226-240)
template <typename V>
__global__ __launch_bounds__(NT) void k_direction(int npw, const int* l2i, const double* beta, const cplx<V>* g,
                                                  const double* g2kin, const double* eprec, cplx<V>* h,
                                                  const cplx<V>* hold, cplx<V>* bc, long ld, long ldc,
                                                  const int* d_nc) {
  const int lb = blockIdx.y;
  if (d_nc && lb >= *d_nc) return;
  const int ib = l2i[lb];
  const int q = blockIdx.x * NT + threadIdx.x;
  if (q >= npw) return;
  const V bt = V(beta[lb]);
  const long o = static_cast<long>(ib) * ld + q;
  const V f = V(1.0 / fmax(1.0, g2kin[q] / eprec[ib]));
  const cplx<V> gv = g[o];
  cplx<V> v = mk<V>(-(gv.x * f), -(gv.y * f));
  if (bt != V(0)) {
    const cplx<V> w = hold[o];
    v = mk<V>(v.x + bt * w.x, v.y + bt * w.y);
  }
  h[o] = v;
  bc[static_cast<long>(lb) * ldc + q] = v;
}

// a = <h|g>, c = <h|t>; x -= (a/c) h; g -= (a/c) t   (linsolve 253-321)
template <typename V>
__global__ __launch_bounds__(NT) void k_cg_update(int npw, int gstart, const int* l2i, const cplx<V>* h, cplx<V>* g,
                                                  const cplx<V>* tc, cplx<V>* x, long ld, long ldc, double* ac_out,
                                                  const int* d_nc) {
  __shared__ double red[NT / 64];
  const int lb = blockIdx.x;
  if (d_nc && lb >= *d_nc) return;
  const int ib = l2i[lb];
  const cplx<V>* hi = h + static_cast<long>(ib) * ld;
  cplx<V>* gi = g + static_cast<long>(ib) * ld;
  const cplx<V>* ti = tc + static_cast<long>(lb) * ldc;
  cplx<V>* xi = x + static_cast<long>(ib) * ld;
  double sa = 0.0, sc = 0.0;
  for (int q = threadIdx.x; q < npw; q += NT) {
    const cplx<V> hv = hi[q];
    const cplx<V> gv = gi[q];
    const cplx<V> tv = ti[q];
    sa += static_cast<double>(hv.x) * gv.x + static_cast<double>(hv.y) * gv.y;
    sc += static_cast<double>(hv.x) * tv.x + static_cast<double>(hv.y) * tv.y;
  }
  sa = block_sum(sa, red);
  sc = block_sum(sc, red);
  double a = 2.0 * sa, c = 2.0 * sc;
  if (gstart == 2) {
    a -= static_cast<double>(hi[0].x) * gi[0].x;
    c -= static_cast<double>(hi[0].x) * ti[0].x;
  }
  __syncthreads();   // every thread has read gi[0] before it is updated
  const V step = V(a / c);
  if (threadIdx.x == 0 && ac_out) {
    ac_out[2 * lb] = a;
    ac_out[2 * lb + 1] = c;
  }
  for (int q = threadIdx.x; q < npw; q += NT) {
    const cplx<V> hv = hi[q];
    const cplx<V> tv = ti[q];
    cplx<V> xv = xi[q];
    cplx<V> gv = gi[q];
    xi[q] = mk<V>(xv.x - step * hv.x, xv.y - step * hv.y);
    gi[q] = mk<V>(gv.x - step * tv.x, gv.y - step * tv.y);
  }
}

// The same update with the band's h and t (and g when CG_ is set) held in
// registers between the inner products and the update (one read of each
// instead of two): 1024 threads, up to E elements each.
// With RHO the band's next rho = <M^-1 g|g> (as k_prec_rho forms it) is summed
// from the updated g while it is in registers and stored at rho[ib].
constexpr int NTU = 1024;
template <typename V, int E, bool CG_, bool RHO>
__global__ __launch_bounds__(NTU) void k_cg_update_reg(int npw, int gstart, const int* l2i, const cplx<V>* h,
                                                      cplx<V>* g, const cplx<V>* tc, cplx<V>* x, long ld, long ldc,
                                                      const double* g2kin, const double* eprec, double* rho,
                                                      const int* d_nc) {
  __shared__ double red[NTU / 64];
  const int lb = blockIdx.x;
  if (d_nc && lb >= *d_nc) return;
  const int ib = l2i[lb];
  const cplx<V>* hi = h + static_cast<long>(ib) * ld;
  cplx<V>* gi = g + static_cast<long>(ib) * ld;
  const cplx<V>* ti = tc + static_cast<long>(lb) * ldc;
  cplx<V>* xi = x + static_cast<long>(ib) * ld;
  cplx<V> hv[E], gv[CG_ ? E : 1], tv[E];
  double sa = 0.0, sc = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int q = threadIdx.x + e * NTU;
    if (q < npw) {
      hv[e] = hi[q];
      const cplx<V> gq = gi[q];
      if constexpr (CG_) gv[e] = gq;
      tv[e] = ti[q];
      sa += static_cast<double>(hv[e].x) * gq.x + static_cast<double>(hv[e].y) * gq.y;
      sc += static_cast<double>(hv[e].x) * tv[e].x + static_cast<double>(hv[e].y) * tv[e].y;
    }
  }
  sa = block_sum<NTU>(sa, red);
  sc = block_sum<NTU>(sc, red);
  double a = 2.0 * sa, c = 2.0 * sc;
  if (gstart == 2) {
    // element 0 belongs to thread 0; the block sums above end with a barrier
    a -= static_cast<double>(hi[0].x) * gi[0].x;
    c -= static_cast<double>(hi[0].x) * ti[0].x;
  }
  __syncthreads();   // every thread has read gi[0] before it is updated
  const V step = V(a / c);
  const double ep = RHO ? eprec[ib] : 1.0;
  double sr = 0.0, r0 = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int q = threadIdx.x + e * NTU;
    if (q < npw) {
      const cplx<V> xv = xi[q];
      cplx<V> gq;
      if constexpr (CG_) gq = gv[e];
      else gq = gi[q];
      xi[q] = mk<V>(xv.x - step * hv[e].x, xv.y - step * hv[e].y);
      const cplx<V> gn = mk<V>(gq.x - step * tv[e].x, gq.y - step * tv[e].y);
      gi[q] = gn;
      if constexpr (RHO) {
        const V f = V(1.0 / fmax(1.0, g2kin[q] / ep));
        const cplx<V> pv = mk<V>(gn.x * f, gn.y * f);
        const double t = static_cast<double>(pv.x) * gn.x + static_cast<double>(pv.y) * gn.y;
        sr += t;
        if (q == 0) r0 = static_cast<double>(pv.x) * gn.x;
      }
    }
  }
  if constexpr (RHO) {
    sr = block_sum<NTU>(sr, red);
    // element 0 is thread 0's
    if (threadIdx.x == 0) rho[ib] = 2.0 * sr - (gstart == 2 ? r0 : 0.0);
  }
}

// R values summed over the wavefront: lane l returns the sum of v[l % R].
// (log2 R exchange steps halve the values, the rest carry one: 10 exchanges
// for eight sums instead of 48.)
template <int R>
__device__ __forceinline__ double wave_sums(double (&v)[R]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int n = R / 2; n > 0; n >>= 1) {
    const bool up = lane & n;
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const double send = up ? v[i] : v[i + n];
      const double keep = up ? v[i + n] : v[i];
      v[i] = keep + __shfl_xor(send, n, 64);
    }
  }
  double t = v[0];
#pragma unroll
  for (int o = R; o < 64; o <<= 1) t += __shfl_xor(t, o, 64);
  return t;
}

// a value that is the same in every lane, in scalar registers
__device__ __forceinline__ double uniform(double v) {
  const long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<int>(b));
  const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<int>(b >> 32));
  return __longlong_as_double(static_cast<long>((static_cast<unsigned long>(hi) << 32) | lo));
}

// One band's share of a CG iteration after the local part of the operator, for
// few projector rows: t += Q s (Q^T h) (the projector part), a = <h|g>,
// c = <h|t>, x -= (a/c) h, g -= (a/c) t, rho = <M^-1 g|g> and the next
// direction h <- -M^-1 g + (rho / rho_old) h, one workgroup a band with h and
// M^-1 g in registers.  <h|Q s Q^T h> is the sum of s_i (Q_i^T h)^2, so t is complete
// only in the second pass and never stored.  (kCgProjRows rows: their two
// passes come from the L2 and cost 2 npw rows 16 bytes a band.)
// Bound: what one compute unit loads (the rows twice and nine passes of the
// vectors: 27 to 31 of its 64 bytes a cycle) around three block-wide sums; the
// vector ALUs are busy 3 to 8 % of the cycles.  Before, the same work was the
// products' three launches, the update and the direction: 35 bands, 7 rows,
// npw = 3,761: 12.2 + 4.3 + 4.5 + 8.9 + 4.1 -> 18 us; 192 bands, 6 rows, npw =
// 6,147: 10.3 + 4.9 + 7.5 + 16.7 + 8.5 -> 31 us; and four gaps less.
// Rows in groups of RG; beyond nq the last one is repeated and not used.
template <int E, int RG>
__global__ __launch_bounds__(NTU) void k_cg_project(unsigned npw, int gstart, int nq, const int* l2i, const z64* q,
                                                   const double* scale, z64* h, z64* g, const z64* t, z64* x,
                                                   const double* g2kin, const double* eprec, double* rho,
                                                   const int* d_nc) {
  constexpr int NW = NTU / 64;
  auto row = [&](int r) { return q + static_cast<long>(min(r, nq - 1)) * npw; };
  __shared__ double red[NW][kCgProjRows + 2];
  __shared__ double cs[kCgProjRows], cp[kCgProjRows];
  const int lb = blockIdx.x;
  if (lb >= *d_nc) return;   // uniform per workgroup
  const int ib = __builtin_amdgcn_readfirstlane(l2i[lb]);   // (scalar row addresses)
  const long o = static_cast<long>(ib) * npw;
  h += o;
  g += o;
  t += o;
  x += o;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  z64 hv[E], pv[E];
  double d[2] = {0.0, 0.0};
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const unsigned i = tid + e * NTU;
    hv[e] = mk(0.0, 0.0);
    if (i < npw) {
      hv[e] = h[i];
      const z64 gq = g[i], tq = t[i];
      d[0] += hv[e].x * gq.x + hv[e].y * gq.y;
      d[1] += hv[e].x * tq.x + hv[e].y * tq.y;
    }
    if (E > 4 && e % 3 == 2) __builtin_amdgcn_sched_barrier(0);   // no more loads ahead than registers for them
  }
  const double h0 = uniform(gstart == 2 ? h[0].x : 0.0);
  const double g0 = uniform(g[0].x), t0 = uniform(t[0].x), rho_old = uniform(rho[ib]), ep = uniform(eprec[ib]);
  const double dw = wave_sums<2>(d);
  if (lane < 2) red[w][kCgProjRows + lane] = dw;
#pragma unroll 1
  for (int r0 = 0; r0 < nq; r0 += RG) {
    constexpr int R2 = RG > 4 ? 8 : RG > 2 ? 4 : RG;
    double p[R2];
#pragma unroll
    for (int r = 0; r < R2; ++r) p[r] = 0.0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      // beyond npw h is zero: any element of the row may be read
      const unsigned i = min(static_cast<unsigned>(tid + e * NTU), npw - 1u);
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        const z64 v = row(r0 + r)[i];
        p[r] += v.x * hv[e].x + v.y * hv[e].y;
      }
      if (E > 4 || e % 2) __builtin_amdgcn_sched_barrier(0);
    }
    const double pw = wave_sums<R2>(p);
    if (lane < R2 && r0 + lane < kCgProjRows) red[w][r0 + lane] = pw;
  }
  __syncthreads();   // also: every thread has read h[0] and g[0]
  if (tid < nq) {
    double v = 0.0;
    for (int k = 0; k < NW; ++k) v += red[k][tid];
    v = 2.0 * v - h0 * q[static_cast<long>(tid) * npw].x;
    cs[tid] = scale[tid] * v;
    cp[tid] = v;
  }
  double a = 0.0, c = 0.0;
  for (int k = 0; k < NW; ++k) {
    a += red[k][kCgProjRows];
    c += red[k][kCgProjRows + 1];
  }
  __syncthreads();
  a = 2.0 * a - h0 * g0;
  c = 2.0 * c - h0 * t0;
  for (int r = 0; r < nq; ++r) c += cs[r] * cp[r];
  const double step = uniform(a / c);
  double s[2] = {0.0, 0.0};
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const unsigned i = tid + e * NTU;
    if (i < npw) {
      z64 tq = t[i];   // (again, from the L2: held through the first pass it would spill)
#pragma unroll 1
      for (int r0 = 0; r0 < nq; r0 += RG) {
#pragma unroll
        for (int r = 0; r < RG; ++r) {
          const z64 v = row(r0 + r)[i];
          const double f = r0 + r < nq ? uniform(cs[r0 + r]) : 0.0;
          tq.x += f * v.x;
          tq.y += f * v.y;
        }
      }
      const z64 xv = x[i], gv = g[i];
      x[i] = mk(xv.x - step * hv[e].x, xv.y - step * hv[e].y);
      const z64 gn = mk(gv.x - step * tq.x, gv.y - step * tq.y);
      g[i] = gn;
      const double f = 1.0 / fmax(1.0, g2kin[i] / ep);
      pv[e] = mk(gn.x * f, gn.y * f);   // M^-1 g
      s[0] += pv[e].x * gn.x + pv[e].y * gn.y;
      if (i == 0) s[1] = pv[e].x * gn.x;
    }
    if (E > 4) __builtin_amdgcn_sched_barrier(0);
  }
  const double sw = wave_sums<2>(s);
  // (the first sums' last readers are behind the barrier above)
  if (lane < 2) red[w][lane] = sw;
  __syncthreads();
  double r = 0.0;
  for (int k = 0; k < NW; ++k) r += red[k][0];
  r = 2.0 * r - (gstart == 2 ? red[0][1] : 0.0);   // element 0 is thread 0's
  if (tid == 0) rho[ib] = r;
  const double beta = r / rho_old;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const unsigned i = tid + e * NTU;
    if (i < npw) h[i] = mk(-pv[e].x + beta * hv[e].x, -pv[e].y + beta * hv[e].y);
  }
}

// The projector part alone, t += Q s (Q^T x), for the operator on few columns:
// as in k_cg_project, one workgroup a column with x in registers.  One launch
// where the products are three (one column, 6 rows, npw = 6,147: 17 us against
// 8.2 + 3.5 + 3.4 and two gaps; a whole call 96 -> 83 us with one item list and
// one wait for the caller's inputs).  project_pays: where it wins.
template <int E, int RG>
__global__ __launch_bounds__(NTU) void k_project(unsigned npw, int gstart, int nq, const z64* q, const double* scale,
                                                const z64* x, z64* t) {
  constexpr int NW = NTU / 64;
  auto row = [&](int r) { return q + static_cast<long>(min(r, nq - 1)) * npw; };
  __shared__ double red[NW][kCgProjRows];
  __shared__ double cs[kCgProjRows];
  x += static_cast<long>(blockIdx.x) * npw;
  t += static_cast<long>(blockIdx.x) * npw;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  z64 xv[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const unsigned i = tid + e * NTU;
    xv[e] = i < npw ? x[i] : mk(0.0, 0.0);
  }
#pragma unroll 1
  for (int r0 = 0; r0 < nq; r0 += RG) {
    constexpr int R2 = RG > 4 ? 8 : RG > 2 ? 4 : RG;
    double p[R2];
#pragma unroll
    for (int r = 0; r < R2; ++r) p[r] = 0.0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      // beyond npw x is zero: any element of the row may be read
      const unsigned i = min(static_cast<unsigned>(tid + e * NTU), npw - 1u);
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        const z64 v = row(r0 + r)[i];
        p[r] += v.x * xv[e].x + v.y * xv[e].y;
      }
    }
    const double pw = wave_sums<R2>(p);
    if (lane < R2 && r0 + lane < kCgProjRows) red[w][r0 + lane] = pw;
  }
  __syncthreads();
  if (tid < nq) {
    double v = 0.0;
    for (int k = 0; k < NW; ++k) v += red[k][tid];
    v = 2.0 * v - (gstart == 2 ? x[0].x * q[static_cast<long>(tid) * npw].x : 0.0);
    cs[tid] = scale[tid] * v;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const unsigned i = tid + e * NTU;
    if (i < npw) {
      z64 tq = t[i];
#pragma unroll 1
      for (int r0 = 0; r0 < nq; r0 += RG) {
#pragma unroll
        for (int r = 0; r < RG; ++r) {
          const z64 v = row(r0 + r)[i];
          const double f = r0 + r < nq ? cs[r0 + r] : 0.0;
          tq.x += f * v.x;
          tq.y += f * v.y;
        }
      }
      t[i] = tq;
    }
  }
}

// out[r][s] = in[r][perm[s]] * (w ? w[s] : 1)     caller order -> stick order
__global__ void k_gather(int m, int npw, const int* perm, const z64* in, long ldin, z64* out, long ldout,
                         const double* w) {
  const int r = blockIdx.y;
  const int s = blockIdx.x * NT + threadIdx.x;
  if (s >= npw || r >= m) return;
  z64 v = in[static_cast<long>(r) * ldin + perm[s]];
  if (w) v = cscale(v, w[s]);
  out[static_cast<long>(r) * ldout + s] = v;
}

// out[r][perm[s]] = in[r][s]; out[r][npw..ldout) = 0        stick order -> caller order
__global__ void k_scatter(int m, int npw, int npwx, const int* perm, const z64* in, long ldin, z64* out,
                          long ldout) {
  const int r = blockIdx.y;
  const int s = blockIdx.x * NT + threadIdx.x;
  if (r >= m) return;
  if (s < npw) out[static_cast<long>(r) * ldout + perm[s]] = in[static_cast<long>(r) * ldin + s];
  else if (s < npwx) out[static_cast<long>(r) * ldout + s] = mk(0.0, 0.0);
}

// pf[r] = f[r] / max(1, g2kin / eprec[r % period])
__global__ void k_precondition(int m, int npw, const z64* f, z64* pf, long ld, const double* g2kin,
                               const double* eprec, int period) {
  const int r = blockIdx.y;
  const int s = blockIdx.x * NT + threadIdx.x;
  if (s >= npw || r >= m) return;
  const double ep = eprec[r % period];
  const double fac = 1.0 / fmax(1.0, g2kin[s] / ep);
  pf[static_cast<long>(r) * ld + s] = cscale(f[static_cast<long>(r) * ld + s], fac);
}

// t[r] = (g2kin - e[r]) * x[r]      (k_psi - e psi)
template <typename V>
__global__ void k_kinetic(int m, int npw, const cplx<V>* x, cplx<V>* t, long ld, const double* g2kin,
                          const double* e) {
  const int r = blockIdx.y;
  const int s = blockIdx.x * NT + threadIdx.x;
  if (s >= npw || r >= m) return;
  t[static_cast<long>(r) * ld + s] = cscale(x[static_cast<long>(r) * ld + s], V(g2kin[s] - e[r]));
}

// x[ib] += dx[ib] (FP32 increment folded into the FP64 iterate); dx[ib] = 0; xc[u] = x[ib]
__global__ void k_fold(int npw, const int* u2i, z64* x, long ldx, z32* dx, long ld32, z64* xc) {
  const int u = blockIdx.y;
  const int ib = u2i[u];
  const int q = blockIdx.x * NT + threadIdx.x;
  if (q >= npw) return;
  const z32 d = dx[static_cast<long>(ib) * ld32 + q];
  const long o = static_cast<long>(ib) * ldx + q;
  const z64 v = mk(x[o].x + static_cast<double>(d.x), x[o].y + static_cast<double>(d.y));
  x[o] = v;
  dx[static_cast<long>(ib) * ld32 + q] = mk(0.f, 0.f);
  xc[static_cast<long>(u) * ldx + q] = v;
}

// FP64 residual of the refinement step: r = (A x)[u] - b[ib];
// rho[u] = <M^-1 r|r> (Gamma product); the FP32 iteration restarts from g[ib] = r.
__global__ __launch_bounds__(NT) void k_true_residual(int npw, int gstart, const int* u2i, const z64* tc,
                                                      const z64* b, long ldx, const double* g2kin,
                                                      const double* eprec, z32* g, long ld32, double* rho) {
  __shared__ double red[NT / 64];
  const int u = blockIdx.x;
  const int ib = u2i[u];
  const z64* ti = tc + static_cast<long>(u) * ldx;
  const z64* bi = b + static_cast<long>(ib) * ldx;
  z32* gi = g + static_cast<long>(ib) * ld32;
  const double ep = eprec[ib];
  double s = 0.0, r0 = 0.0;
  for (int q = threadIdx.x; q < npw; q += NT) {
    const z64 r = ti[q] - bi[q];
    const double f = 1.0 / fmax(1.0, g2kin[q] / ep);
    s += f * (r.x * r.x + r.y * r.y);
    if (q == 0) r0 = f * r.x * r.x;
    gi[q] = mk(static_cast<float>(r.x), static_cast<float>(r.y));
  }
  s = block_sum(s, red);
  r0 = block_sum(r0, red);
  if (threadIdx.x == 0) rho[u] = 2.0 * s - (gstart == 2 ? r0 : 0.0);
}

__global__ void k_residual32(int npw, const z32* t, long ld32, const z64* b, long ldb, z32* g) {
  const int r = blockIdx.y;
  const int q = blockIdx.x * NT + threadIdx.x;
  if (q >= npw) return;
  const z32 tv = t[static_cast<long>(r) * ld32 + q];
  const z64 bv = b[static_cast<long>(r) * ldb + q];
  g[static_cast<long>(r) * ld32 + q] = mk(static_cast<float>(static_cast<double>(tv.x) - bv.x),
                                          static_cast<float>(static_cast<double>(tv.y) - bv.y));
}

__global__ void k_to_f64(int cols, const float* in, long ld_in, double* out, long ld_out) {
  const int r = blockIdx.y;
  const long c = static_cast<long>(blockIdx.x) * NT + threadIdx.x;
  if (c >= cols) return;
  out[static_cast<long>(r) * ld_out + c] = static_cast<double>(in[static_cast<long>(r) * ld_in + c]);
}

__global__ void k_copy_rows(int npw, const int* list, const z64* in, long ld_in, z64* out, long ld_out, int scatter) {
  const int u = blockIdx.y;
  const int q = blockIdx.x * NT + threadIdx.x;
  if (q >= npw) return;
  const long src = static_cast<long>(scatter ? u : list[u]) * ld_in + q;
  const long dst = static_cast<long>(scatter ? list[u] : u) * ld_out + q;
  out[dst] = in[src];
}

__global__ void k_gather_real(int n, const int* list, const double* in, double* out) {
  const int u = blockIdx.x * NT + threadIdx.x;
  if (u < n) out[u] = in[list[u]];
}

__global__ void k_to_f32(int cols, const double* in, long ld_in, float* out, long ld_out) {
  const int r = blockIdx.y;
  const long c = static_cast<long>(blockIdx.x) * NT + threadIdx.x;
  if (c >= cols) return;
  out[static_cast<long>(r) * ld_out + c] = static_cast<float>(in[static_cast<long>(r) * ld_in + c]);
}

// y = a*x + b*y over n complex
__global__ void k_axpby(long n, double a, const z64* x, double b, z64* y) {
  const long i = static_cast<long>(blockIdx.x) * NT + threadIdx.x;
  if (i >= n) return;
  const z64 xv = x[i];
  const z64 yv = y[i];
  y[i] = mk(a * xv.x + b * yv.x, a * xv.y + b * yv.y);
}

__global__ void k_fill_pairs(FftItem* items, int n, int m, int row0, FftItem* ident, int chunk) {
  const int q = blockIdx.x * NT + threadIdx.x;
  if (q >= n) return;
  FftItem it;
  it.a = row0 + 2 * q;
  it.b = (2 * q + 1 < m) ? row0 + 2 * q + 1 : -1;
  it.pot = -1;
  it.pad = 0;
  items[q] = it;
  if (q < chunk) {
    it.a = q;
    it.b = -1;
    ident[q] = it;
  }
}

__global__ void k_iota(int* v, int n) {
  const int q = blockIdx.x * NT + threadIdx.x;
  if (q < n) v[q] = q;
}

// Convergence test, compaction and coefficients of one CG iteration on the
// device (linsolve_sternheimer_m_wfcts.f90:190-240): one workgroup walks the
// bands in order, so the active list keeps the ascending band order of
// map_lbnd2ibnd.  Along with it, the operator's work items of the launch's
// sel.npair pairs of columns (switched off beyond the active ones): the columns
// are the compacted ones, or (by_band) the bands themselves.  The count goes to
// sel.rec (host memory: the host reads it without a copy in between).
constexpr int NTS_SEL = 1024;
__global__ __launch_bounds__(NTS_SEL) void k_cg_select(int m, double tr2, int first, int group,
                                                       const double* __restrict__ rhob, double* __restrict__ rhoold,
                                                       int* __restrict__ conv, const double* __restrict__ e_col,
                                                       int* __restrict__ l2i, double* __restrict__ beta,
                                                       double* __restrict__ eu, int* __restrict__ nc_out,
                                                       CgSelect sel) {
  __shared__ int wcount[NTS_SEL / 64];
  __shared__ int base_s;
  __shared__ int calls_w[NTS_SEL / 64];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  if (tid == 0) base_s = 0;
  __syncthreads();
  for (int c0 = 0; c0 < m; c0 += NTS_SEL) {
    const int ib = c0 + tid;
    bool act = false;
    double r = 0.0;
    if (ib < m && !conv[ib]) {
      r = rhob[ib];
      if (r < tr2) conv[ib] = 1;
      else act = true;
    }
    const unsigned long long mask = __ballot(act);
    const int before = __popcll(mask & ((1ull << lane) - 1ull));
    if (lane == 0) wcount[w] = __popcll(mask);
    __syncthreads();
    int off = base_s;
    for (int k = 0; k < w; ++k) off += wcount[k];
    if (act) {
      const int pos = off + before;
      l2i[pos] = ib;
      beta[pos] = first ? 0.0 : r / rhoold[ib];
      rhoold[ib] = r;
      eu[pos] = e_col[ib];
    }
    __syncthreads();
    if (tid == 0) {
      int tot = 0;
      for (int k = 0; k < NTS_SEL / 64; ++k) tot += wcount[k];
      base_s += tot;
    }
    __syncthreads();
  }
  const int nc = base_s;
  const int npair = (nc + 1) / 2;
  for (int q = tid; q < sel.npair; q += NTS_SEL) {
    const int a = 2 * q, b = 2 * q + 1;
    FftItem it;
    it.pot = -1;
    it.pad = 0;
    it.a = a < nc ? (sel.by_band ? l2i[a] : a) : -1;
    it.b = b < nc ? (sel.by_band ? l2i[b] : b) : -1;
    sel.items[q] = it;
    it.a = q < npair ? q % sel.chunk : -1;
    it.b = -1;
    sel.ident[q] = it;
  }
  // perturbations among the active bands (the list is ascending)
  int calls = 0;
  for (int pos = tid; pos < nc; pos += NTS_SEL) {
    const int gp = group > 0 ? l2i[pos] / group : 0;
    const int gq = pos > 0 ? (group > 0 ? l2i[pos - 1] / group : 0) : -1;
    calls += gp != gq;
  }
  for (int o = 32; o > 0; o >>= 1) calls += __shfl_xor(calls, o, 64);
  if (lane == 0) calls_w[w] = calls;
  __syncthreads();
  if (tid == 0) {
    int tot = 0;
    for (int k = 0; k < NTS_SEL / 64; ++k) tot += calls_w[k];
    *nc_out = nc;
    __hip_atomic_store(sel.rec, nc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(sel.rec + 1, tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// eprec[v] = 1.35 sum_{g<npw} |evc_v(g)|^2 g2kin(g)   (Tools/set_eprec.f90:40-51)
__global__ __launch_bounds__(NT) void k_eprec(int npw, const z64* evc, long ld, const double* g2kin, double* eprec) {
  __shared__ double red[NT / 64];
  const int v = blockIdx.x;
  const z64* e = evc + static_cast<long>(v) * ld;
  double s = 0.0;
  for (int q = threadIdx.x; q < npw; q += NT) s += (e[q].x * e[q].x + e[q].y * e[q].y) * g2kin[q];
  s = block_sum(s, red);
  if (threadIdx.x == 0) eprec[v] = 1.35 * s;
}

}  // namespace

void prec_rho(int nc, int npw, int gstart, const int* l2i, const z64* g, long ld, const double* g2kin,
              const double* eprec, double* rho, hipStream_t s, bool by_band) {
  if (nc <= 0) return;
  k_prec_rho<double><<<nc, NT, 0, s>>>(npw, gstart, l2i, g, ld, g2kin, eprec, rho, by_band);
  WH_HIP(hipGetLastError());
}

void prec_rho(int nc, int npw, int gstart, const int* l2i, const z32* g, long ld, const double* g2kin,
              const double* eprec, double* rho, hipStream_t s, bool by_band) {
  if (nc <= 0) return;
  k_prec_rho<float><<<nc, NT, 0, s>>>(npw, gstart, l2i, g, ld, g2kin, eprec, rho, by_band);
  WH_HIP(hipGetLastError());
}

void direction(int nc, int npw, const int* l2i, const double* beta, const z64* g, const double* g2kin,
               const double* eprec, z64* h, const z64* hold, z64* bc, long ld, hipStream_t s, const int* d_nc) {
  if (nc <= 0) return;
  k_direction<double><<<dim3(ceil_div(npw, NT), nc), NT, 0, s>>>(npw, l2i, beta, g, g2kin, eprec, h, hold, bc, ld,
                                                                  ld, d_nc);
  WH_HIP(hipGetLastError());
}

void direction(int nc, int npw, const int* l2i, const double* beta, const z32* g, const double* g2kin,
               const double* eprec, z32* h, const z32* hold, z32* bc, long ld, hipStream_t s) {
  if (nc <= 0) return;
  k_direction<float><<<dim3(ceil_div(npw, NT), nc), NT, 0, s>>>(npw, l2i, beta, g, g2kin, eprec, h, hold, bc, ld,
                                                                 ld, nullptr);
  WH_HIP(hipGetLastError());
}

template <typename V, bool RHO>
static void cg_update_reg(int nc, int npw, int gstart, const int* l2i, const cplx<V>* h, cplx<V>* g,
                          const cplx<V>* tc, cplx<V>* x, long ld, const RhoOut& r, hipStream_t s, const int* d_nc) {
  // FP64 at 9 elements per thread keeps h and t only (g too would spill)
  if (npw <= 4 * NTU)
    k_cg_update_reg<V, 4, true, RHO><<<nc, NTU, 0, s>>>(npw, gstart, l2i, h, g, tc, x, ld, ld, r.g2kin, r.eprec,
                                                         r.rho, d_nc);
  else
    k_cg_update_reg<V, 9, (sizeof(V) == 4), RHO><<<nc, NTU, 0, s>>>(npw, gstart, l2i, h, g, tc, x, ld, ld, r.g2kin,
                                                                    r.eprec, r.rho, d_nc);
}

template <typename V>
static void cg_update_any(int nc, int npw, int gstart, const int* l2i, const cplx<V>* h, cplx<V>* g,
                          const cplx<V>* tc, cplx<V>* x, long ld, double* ac_out, const RhoOut* r, hipStream_t s,
                          const int* d_nc) {
  if (nc <= 0) return;
  if (!ac_out && npw <= 9 * NTU) {
    if (r) cg_update_reg<V, true>(nc, npw, gstart, l2i, h, g, tc, x, ld, *r, s, d_nc);
    else cg_update_reg<V, false>(nc, npw, gstart, l2i, h, g, tc, x, ld, RhoOut{}, s, d_nc);
  } else {
    k_cg_update<V><<<nc, NT, 0, s>>>(npw, gstart, l2i, h, g, tc, x, ld, ld, ac_out, d_nc);
    if (r) k_prec_rho<V><<<nc, NT, 0, s>>>(npw, gstart, l2i, g, ld, r->g2kin, r->eprec, r->rho, true, d_nc);
  }
  WH_HIP(hipGetLastError());
}

void cg_update(int nc, int npw, int gstart, const int* l2i, const z64* h, z64* g, const z64* tc, z64* x, long ld,
               double* ac_out, hipStream_t s, const RhoOut* rho, const int* d_nc) {
  cg_update_any<double>(nc, npw, gstart, l2i, h, g, tc, x, ld, ac_out, rho, s, d_nc);
}

void cg_update(int nc, int npw, int gstart, const int* l2i, const z32* h, z32* g, const z32* tc, z32* x, long ld,
               double* ac_out, hipStream_t s, const RhoOut* rho) {
  cg_update_any<float>(nc, npw, gstart, l2i, h, g, tc, x, ld, ac_out, rho, s, nullptr);
}

bool cg_project_fits(int nq, int m, int npw) { return nq <= kCgProjRows && m <= 256 && npw <= 9 * NTU; }

// The CG with k_cg_project against the general iteration (a solve of some 20
// iterations, ms).  Up to 4 elements a thread it wins throughout (npw = 3,761, 32
// rows, 1 / 16 / 128 columns: 1.19 / 1.44 / 2.44 against 1.37 / 1.86 / 3.25).  With 9 the
// one compute unit of a column goes through 2 x 9 x 16 kB of each row whatever npw
// is, which many rows and few columns leave in the open (ours, general):
//   npw, rows    1 column   8          16         32         64         128
//   4,193, 28   1.40 1.36  1.58 1.60  1.65 1.82  1.71 1.93  2.08 2.43
//   6,147, 16   1.18 1.15  1.37 1.38  1.50 1.57  1.74 1.86  2.04 2.31  2.73 3.21
//   6,147, 32   1.62 1.38  1.86 1.83  2.00 2.00  2.24 2.30  2.55 2.80  3.27 3.99
//   9,139, 10   1.21 1.21  1.50 1.48  1.61 1.64  1.95 2.04  2.39 2.59  3.62 4.25
//   9,139, 16   1.43 1.28  1.72 1.62  1.85 1.80  2.18 2.23  2.63 2.83  3.85 4.78
//   9,139, 32   2.15 1.54  2.47 2.12  2.65 2.38  2.96 2.84  3.35 3.54  4.57 5.89
// so beyond ten rows it takes the more columns the more elements there are.
bool cg_project_pays(int nq, int m, int npw) {
  if (!cg_project_fits(nq, m, npw)) return false;
  return npw <= 4 * NTU || nq <= 10 || m >= std::max(8, (ceil_div(npw, NTU) - 6) * (nq > 20 ? 16 : 10));
}

// k_project against the three products (a call, us; 1, 16, 256 columns): up to
// 4 elements a thread it wins throughout (npw = 1,820: 8 rows 69 / 70 / 140 against
// 92 / 92 / 175, 31 rows 86 / 88 / 161 against 102 / 104 / 213); with 9 the one
// compute unit of a column takes too long over many rows unless the columns
// fill the chip (npw = 6,147: 8 rows 86 / 101 / 309 against 84 / 97 / 327, 31 rows
// 142 / 170 / 402 against 103 / 128 / 475).
bool project_pays(int nq, int m, int npw) {
  return cg_project_fits(nq, m, npw) && (npw <= 4 * NTU || nq <= 6 || m > 128);
}

// Rows a group.  More of them share the reads of a column's elements and the
// sums' exchanges; fewer leave registers and repeat fewer rows that are not there.
// So: all of them where the registers allow (4 elements a thread: up to 7, except
// that six go faster in threes; 9: up to 4); fours, or threes, that leave none
// over; else fours unless more than an eighth (9 elements: a quarter) of their
// loads were for nothing, then twos.  With 9 elements threes stop at nine rows.
// A solve (cg_project), us, 128 columns, npw = 1,872 / 3,761: 7 rows at once 1,218 /
// 2,037, in twos 1,239 / 2,060, in fours 1,253 / 2,043; 6 in threes 1,207 / 2,025, at
// once 1,224 / 2,028; 10 in twos 1,293 / 2,084, in fours 1,317 / 2,095; 21 in threes
// 1,427 / 2,270, in fours 1,465 / 2,302.  npw = 6,147 / 9,139: 9 in threes 2,591 / 3,609,
// in fours 2,598 / 3,606 (one column 1,014 / 1,214 and 1,086 / 1,273); 24 in fours 3,009 /
// 4,205, in threes 3,186 / 4,415; 31 in fours 3,296 / 4,558, in twos 3,462 / 4,750; 5 and
// one column in twos 949 / 1,107, in fours 1,000 / 1,160.
static int project_group(int nq, bool small) {
  if (nq <= 4 || (small && (nq == 5 || nq == 7))) return std::max(nq, 1);
  if (nq % 4 == 0) return 4;
  if (nq % 3 == 0 && (small || nq <= 9)) return 3;
  const int over = ceil_div(nq, 4) * 4 - nq;
  return (small ? 8 : 4) * over > nq + over ? 2 : 4;
}

// run(elements a thread, rows a group)
template <typename F>
static void project_variant(int npw, int nq, F run) {
  using std::integral_constant;
  const bool small = npw <= 4 * NTU;
  const int rg = project_group(nq, small);
  auto with = [&](auto e) {
    if (rg == 1) run(e, integral_constant<int, 1>());
    else if (rg == 2) run(e, integral_constant<int, 2>());
    else if (rg == 3) run(e, integral_constant<int, 3>());
    else if (rg == 4) run(e, integral_constant<int, 4>());
    else if constexpr (decltype(e)::value == 4) {
      if (rg == 5) run(e, integral_constant<int, 5>());
      else run(e, integral_constant<int, 7>());
    }
  };
  if (small) with(integral_constant<int, 4>());
  else with(integral_constant<int, 9>());
}

void cg_project(int nc, int npw, int gstart, int nq, const int* l2i, const z64* q, const double* scale, z64* h, z64* g,
                const z64* t, z64* x, const double* g2kin, const double* eprec, double* rho, const int* d_nc,
                hipStream_t s) {
  if (nc <= 0) return;
  WH_REQUIRE(cg_project_fits(nq, nc, npw), "cg_project: outside the kernel's range");
  project_variant(npw, nq, [&](auto e, auto rg) {
    k_cg_project<decltype(e)::value, decltype(rg)::value><<<nc, NTU, 0, s>>>(npw, gstart, nq, l2i, q, scale, h, g, t, x,
                                                                             g2kin, eprec, rho, d_nc);
  });
  WH_HIP(hipGetLastError());
}

void project(int m, int npw, int gstart, int nq, const z64* q, const double* scale, const z64* x, z64* t,
             hipStream_t s) {
  if (m <= 0 || nq <= 0) return;
  WH_REQUIRE(cg_project_fits(nq, m, npw), "project: outside the kernel's range");
  project_variant(npw, nq, [&](auto e, auto rg) {
    k_project<decltype(e)::value, decltype(rg)::value><<<m, NTU, 0, s>>>(npw, gstart, nq, q, scale, x, t);
  });
  WH_HIP(hipGetLastError());
}

void gather_sticks(int m, int npw, const int* perm, const z64* in, long ldin, z64* out, long ldout, const double* w,
                   hipStream_t s) {
  if (m <= 0) return;
  k_gather<<<dim3(ceil_div(npw, NT), m), NT, 0, s>>>(m, npw, perm, in, ldin, out, ldout, w);
  WH_HIP(hipGetLastError());
}

void scatter_caller(int m, int npw, int npwx, const int* perm, const z64* in, long ldin, z64* out, long ldout,
                    hipStream_t s) {
  if (m <= 0) return;
  k_scatter<<<dim3(ceil_div(npwx, NT), m), NT, 0, s>>>(m, npw, npwx, perm, in, ldin, out, ldout);
  WH_HIP(hipGetLastError());
}

void precondition(int m, int npw, const z64* f, z64* pf, long ld, const double* g2kin, const double* eprec,
                  int period, hipStream_t s) {
  if (m <= 0) return;
  k_precondition<<<dim3(ceil_div(npw, NT), m), NT, 0, s>>>(m, npw, f, pf, ld, g2kin, eprec, period);
  WH_HIP(hipGetLastError());
}

void kinetic_minus_e(int m, int npw, const z64* x, z64* t, long ld, const double* g2kin, const double* e,
                     hipStream_t s) {
  if (m <= 0) return;
  k_kinetic<double><<<dim3(ceil_div(npw, NT), m), NT, 0, s>>>(m, npw, x, t, ld, g2kin, e);
  WH_HIP(hipGetLastError());
}

void kinetic_minus_e(int m, int npw, const z32* x, z32* t, long ld, const double* g2kin, const double* e,
                     hipStream_t s) {
  if (m <= 0) return;
  k_kinetic<float><<<dim3(ceil_div(npw, NT), m), NT, 0, s>>>(m, npw, x, t, ld, g2kin, e);
  WH_HIP(hipGetLastError());
}

void fold_increment(int nu, int npw, const int* u2i, z64* x, long ldx, z32* dx, long ld32, z64* xc, hipStream_t s) {
  if (nu <= 0) return;
  k_fold<<<dim3(ceil_div(npw, NT), nu), NT, 0, s>>>(npw, u2i, x, ldx, dx, ld32, xc);
  WH_HIP(hipGetLastError());
}

void true_residual(int nu, int npw, int gstart, const int* u2i, const z64* tc, const z64* b, long ldx,
                   const double* g2kin, const double* eprec, z32* g, long ld32, double* rho, hipStream_t s) {
  if (nu <= 0) return;
  k_true_residual<<<nu, NT, 0, s>>>(npw, gstart, u2i, tc, b, ldx, g2kin, eprec, g, ld32, rho);
  WH_HIP(hipGetLastError());
}

void residual32(int m, int npw, const z32* t, long ld32, const z64* b, long ldb, z32* g, hipStream_t s) {
  if (m <= 0) return;
  k_residual32<<<dim3(ceil_div(npw, NT), m), NT, 0, s>>>(npw, t, ld32, b, ldb, g);
  WH_HIP(hipGetLastError());
}

void to_f64(int rows, int cols, const float* in, long ld_in, double* out, long ld_out, hipStream_t s) {
  if (rows <= 0 || cols <= 0) return;
  k_to_f64<<<dim3(ceil_div(cols, NT), rows), NT, 0, s>>>(cols, in, ld_in, out, ld_out);
  WH_HIP(hipGetLastError());
}

void copy_rows(int n, int npw, const int* list, const z64* in, long ld_in, z64* out, long ld_out, bool scatter,
               hipStream_t s) {
  if (n <= 0) return;
  k_copy_rows<<<dim3(ceil_div(npw, NT), n), NT, 0, s>>>(npw, list, in, ld_in, out, ld_out, scatter ? 1 : 0);
  WH_HIP(hipGetLastError());
}

void gather_real(int n, const int* list, const double* in, double* out, hipStream_t s) {
  if (n <= 0) return;
  k_gather_real<<<ceil_div(n, NT), NT, 0, s>>>(n, list, in, out);
  WH_HIP(hipGetLastError());
}

void to_f32(int rows, int cols, const double* in, long ld_in, float* out, long ld_out, hipStream_t s) {
  if (rows <= 0 || cols <= 0) return;
  k_to_f32<<<dim3(ceil_div(cols, NT), rows), NT, 0, s>>>(cols, in, ld_in, out, ld_out);
  WH_HIP(hipGetLastError());
}

void axpby(long n, double a, const z64* x, double b, z64* y, hipStream_t s) {
  if (n <= 0) return;
  k_axpby<<<ceil_div(n, NT), NT, 0, s>>>(n, a, x, b, y);
  WH_HIP(hipGetLastError());
}

void fill_pairs(FftItem* items, int m, int row0, hipStream_t s, FftItem* ident, int chunk) {
  const int n = (m + 1) / 2;
  WH_REQUIRE(chunk <= n, "fill_pairs: more stick slots than pairs");
  if (n <= 0) return;
  k_fill_pairs<<<ceil_div(n, NT), NT, 0, s>>>(items, n, m, row0, ident, chunk);
  WH_HIP(hipGetLastError());
}

void iota(int* v, int n, hipStream_t s) {
  if (n <= 0) return;
  k_iota<<<ceil_div(n, NT), NT, 0, s>>>(v, n);
  WH_HIP(hipGetLastError());
}

void cg_select(int m, double tr2, int first, int group, const double* rhob, double* rhoold, int* conv,
               const double* e_col, int* l2i, double* beta, double* eu, int* nc, const CgSelect& sel, hipStream_t s) {
  k_cg_select<<<1, NTS_SEL, 0, s>>>(m, tr2, first, group, rhob, rhoold, conv, e_col, l2i, beta, eu, nc, sel);
  WH_HIP(hipGetLastError());
}

void eprec_of(int nb, int npw, const z64* evc, long ld, const double* g2kin, double* eprec, hipStream_t s) {
  if (nb <= 0) return;
  k_eprec<<<nb, NT, 0, s>>>(npw, evc, ld, g2kin, eprec);
  WH_HIP(hipGetLastError());
}

}  // namespace wh
