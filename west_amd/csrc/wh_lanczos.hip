// Wfreq's deflated Lanczos with full re-orthogonalisation at Gamma
// (Wfreq/solve_deflated_lanczos_w_full_ortho.f90:14-357, gamma_only branches)
// and the Gamma inner-product matrix of get_brak_hyper_parallel
// (Wfreq/get_brak_hyper_parallel.f90:14-143, Hamiltonian_kernel/glbrak.f90).
//
// All NRHS chains run together: each Lanczos step is one application of H to
// the NRHS current vectors (the Sternheimer operator's FFT and projector
// kernels with e = 0 and alpha = 0), one deflation P_c = 1 - sum_v |psi_v><psi_v|
// as a bra and a ket product, then one launch for the three-term recurrence,
// the modified Gram-Schmidt sweep over the earlier vectors, the norm and the
// next vector.  alpha, beta and the basis stay on the device until the end.
#include <algorithm>

#include "../../include/west_hip.h"
#include "wh_context.h"
#include "wh_gemm.h"
#include "wh_vec.h"

namespace wh {

namespace {

constexpr int NT = 256;

__device__ __forceinline__ double block_sum_l(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int k = 0; k < NT / 64; ++k) t += red[k];
  __syncthreads();
  return t;
}

// Gamma inner product of columns: 2 Re sum a* b - Re a(0) Re b(0) (gstart == 2)
__device__ __forceinline__ double gamma_dot(const z64* a, const z64* b, int npw, int gstart, double* red) {
  double s = 0.0;
  for (int g = threadIdx.x; g < npw; g += NT) s += a[g].x * b[g].x + a[g].y * b[g].y;
  s = block_sum_l(s, red);
  return 2.0 * s - (gstart == 2 ? a[0].x * b[0].x : 0.0);
}

// beta[ip] = sqrt(<r|r>); also into out[ip] when given (solve...ortho.f90:76-112, 290-339)
__global__ __launch_bounds__(NT) void k_lan_norm(int npw, int gstart, const z64* r, long ld, double* beta,
                                                 double* out) {
  __shared__ double red[NT / 64];
  const int ip = blockIdx.x;
  const z64* ri = r + static_cast<long>(ip) * ld;
  const double b = sqrt(gamma_dot(ri, ri, npw, gstart, red));
  if (threadIdx.x == 0) {
    beta[ip] = b;
    if (out) out[ip] = b;
  }
}

// q = r / beta  (solve...ortho.f90:118-124)
__global__ void k_lan_scale(int npw, const z64* r, const double* beta, z64* q, long ld) {
  const int ip = blockIdx.y;
  const int g = blockIdx.x * NT + threadIdx.x;
  if (g >= npw) return;
  const double inv = 1.0 / beta[ip];
  const z64 v = r[static_cast<long>(ip) * ld + g];
  q[static_cast<long>(ip) * ld + g] = mk<double>(v.x * inv, v.y * inv);
}

// The vector part of one Lanczos step, one workgroup per chain
// (solve...ortho.f90:145-339): r -= beta_prev q_prev (il > 0); alpha = <q|r>,
// r -= alpha q; the modified Gram-Schmidt sweep r -= <q_a|r> q_a over q_1 ..
// q_{il-2}, one vector at a time; beta = |r|; and the next q = r / beta.
//
// The sweep is a serial chain of dot products and reads every earlier vector
// of the chain once: 128 chains x 30 steps on 9,139 plane waves read 7.6 GB,
// 1.7 ms at this card's copy rate.  r therefore stays in registers (NE
// elements a thread) with the current vector beside it, and the next vector's
// first PF elements are loaded while the dot product is reduced.  The whole
// call on that case: one launch per vector with r in memory 27.2 ms (13.0 of
// it in those), <18, 4> 14.4, <18, 8> 15.1 and <18, 18> 17.6 (registers spill),
// each vector read twice instead of held 14.5, 1,024 threads 15.0 to 18.6.
// Bound by those reads: 310 MB a launch on average at 4.0 TB/s.
// Spheres beyond 18,432 points keep r in memory (k_lan_step_mem).
constexpr int LNT = 512;

struct LanArgs {
  int npw, gstart, il;
  z64* r;
  const z64* q;            // the basis: block j at q + j blk
  long blk, ld;
  z64* qnext;              // null at the last step
  const double* beta_prev;
  double *alpha, *beta, *beta_s;
};

// red: two sets of one slot per wave, used in turn (one barrier per sum)
__device__ __forceinline__ double lan_sum(double v, double (*red)[LNT / 64], int turn) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[turn & 1][threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int k = 0; k < LNT / 64; ++k) t += red[turn & 1][k];
  return t;
}

// PF elements of the next vector are loaded ahead (0: each vector is read
// twice, for the dot product and for the update, U elements at a time)
template <int NE, int PF>
__global__ __launch_bounds__(LNT) void k_lan_step(LanArgs A) {
  __shared__ double red[2][LNT / 64];
  constexpr int U = 6;
  static_assert(PF <= NE && (PF > 0 || NE % U == 0), "vector split");
  const int tid = threadIdx.x;
  const long o = static_cast<long>(blockIdx.x) * A.ld;
  const int npw = A.npw;
  // Gamma weight of the thread's first element: G = 0 counts once, the others twice
  const double w0 = (tid == 0 && A.gstart == 2) ? 0.5 : 1.0;
  const z64* q = A.q + o;
  const int nv = A.il;   // q_il (alpha), then q_0 .. q_{il-2}: max(1, il) vectors
  auto vec = [&](int k) { return q + (k == 0 ? A.il : k - 1) * A.blk; };
  // element tid + u LNT, 0 beyond npw: buffer loads bound by npw, one offset
  // register for all of a thread's elements
  auto at = [&](const z64* p, int u) {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<z64*>(p), 0, npw * static_cast<int>(sizeof(z64)), 0x00020000);
    typedef unsigned int v4u __attribute__((ext_vector_type(4)));
    const v4u w = __builtin_amdgcn_raw_buffer_load_b128(rs, tid * static_cast<int>(sizeof(z64)),
                                                        u * LNT * static_cast<int>(sizeof(z64)), 0);
    z64 v;
    __builtin_memcpy(&v, &w, sizeof v);
    return v;
  };
  z64 r[NE];
#pragma unroll
  for (int u = 0; u < NE; ++u) r[u] = at(A.r + o, u);
  if (A.il > 0) {
    const double bp = A.beta_prev[blockIdx.x];
    const z64* p = q + (A.il - 1) * A.blk;
#pragma unroll
    for (int u = 0; u < NE; ++u) r[u] = r[u] - cscale(at(p, u), bp);
  }
  auto term = [&](z64 a, int u) {
    const double x = a.x * r[u].x;
    return (u == 0 ? w0 * x : x) + a.y * r[u].y;
  };
  if constexpr (PF > 0) {
    z64 c[NE], n[PF];
#pragma unroll
    for (int u = 0; u < NE; ++u) c[u] = at(vec(0), u);
    for (int k = 0; k == 0 || k < nv; ++k) {
      const bool more = k + 1 < nv;
      const z64* pn = vec(k + 1);
      if (more) {
#pragma unroll
        for (int u = 0; u < PF; ++u) n[u] = at(pn, u);
      }
      double s = 0.0;
#pragma unroll
      for (int u = 0; u < NE; ++u) s += term(c[u], u);
      const double t = 2.0 * lan_sum(s, red, k);
      if (k == 0 && tid == 0) A.alpha[blockIdx.x] = t;
#pragma unroll
      for (int u = 0; u < NE; ++u) r[u] = r[u] - cscale(c[u], t);
      if (more) {
#pragma unroll
        for (int u = 0; u < NE; ++u) c[u] = u < PF ? n[u < PF ? u : 0] : at(pn, u);
      }
    }
  } else {
    for (int k = 0; k == 0 || k < nv; ++k) {
      const z64* p = vec(k);
      double s = 0.0;
#pragma unroll
      for (int u0 = 0; u0 < NE; u0 += U) {
        z64 c[U];
#pragma unroll
        for (int u = 0; u < U; ++u) c[u] = at(p, u0 + u);
#pragma unroll
        for (int u = 0; u < U; ++u) s += term(c[u], u0 + u);
        __builtin_amdgcn_sched_barrier(0);
      }
      const double t = 2.0 * lan_sum(s, red, k);
      if (k == 0 && tid == 0) A.alpha[blockIdx.x] = t;
#pragma unroll
      for (int u0 = 0; u0 < NE; u0 += U) {
        z64 c[U];
#pragma unroll
        for (int u = 0; u < U; ++u) c[u] = at(p, u0 + u);
#pragma unroll
        for (int u = 0; u < U; ++u) r[u0 + u] = r[u0 + u] - cscale(c[u], t);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  double s = 0.0;
#pragma unroll
  for (int u = 0; u < NE; ++u) s += term(r[u], u);
  const double b = sqrt(2.0 * lan_sum(s, red, nv > 0 ? nv : 1));
  if (tid == 0) {
    A.beta[blockIdx.x] = b;
    A.beta_s[blockIdx.x] = b;
  }
  if (A.qnext) {
    const double inv = 1.0 / b;
    z64* qn = A.qnext + o;
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      const int g = tid + u * LNT;
      if (g < npw) qn[g] = cscale(r[u], inv);
    }
  }
}

// the same with r in memory
__global__ __launch_bounds__(LNT) void k_lan_step_mem(LanArgs A) {
  __shared__ double red[2][LNT / 64];
  const int tid = threadIdx.x;
  const long o = static_cast<long>(blockIdx.x) * A.ld;
  const int npw = A.npw;
  z64* r = A.r + o;
  const z64* q = A.q + o;
  const double bp = A.il > 0 ? A.beta_prev[blockIdx.x] : 0.0;
  const int nv = A.il;
  for (int k = 0; k == 0 || k < nv; ++k) {
    const z64* c = q + (k == 0 ? A.il : k - 1) * A.blk;
    const z64* p = k == 0 && A.il > 0 ? q + (A.il - 1) * A.blk : nullptr;
    double s = 0.0;
    for (int g = tid; g < npw; g += LNT) {
      z64 v = r[g];
      if (p) {
        v = v - cscale(p[g], bp);
        r[g] = v;
      }
      const double x = c[g].x * v.x;
      s += (g == 0 && A.gstart == 2 ? 0.5 * x : x) + c[g].y * v.y;
    }
    const double t = 2.0 * lan_sum(s, red, k);
    if (k == 0 && tid == 0) A.alpha[blockIdx.x] = t;
    for (int g = tid; g < npw; g += LNT) r[g] = r[g] - cscale(c[g], t);
  }
  double s = 0.0;
  for (int g = tid; g < npw; g += LNT) {
    const double x = r[g].x * r[g].x;
    s += (g == 0 && A.gstart == 2 ? 0.5 * x : x) + r[g].y * r[g].y;
  }
  const double b = sqrt(2.0 * lan_sum(s, red, nv > 0 ? nv : 1));
  if (tid == 0) {
    A.beta[blockIdx.x] = b;
    A.beta_s[blockIdx.x] = b;
  }
  if (A.qnext)
    for (int g = tid; g < npw; g += LNT) A.qnext[o + g] = cscale(r[g], 1.0 / b);
}

void lan_step(int nrhs, const LanArgs& a, hipStream_t s) {
  const int ne = ceil_div(a.npw, LNT);
  if (ne <= 4) k_lan_step<4, 4><<<nrhs, LNT, 0, s>>>(a);
  else if (ne <= 9) k_lan_step<9, 9><<<nrhs, LNT, 0, s>>>(a);
  else if (ne <= 18) k_lan_step<18, 4><<<nrhs, LNT, 0, s>>>(a);
  else if (ne <= 36) k_lan_step<36, 0><<<nrhs, LNT, 0, s>>>(a);
  else k_lan_step_mem<<<nrhs, LNT, 0, s>>>(a);
  WH_HIP(hipGetLastError());
}

}  // namespace

}  // namespace wh

using namespace wh;

extern "C" int wh_solve_deflated_lanczos_w_full_ortho(int nbnd_to_deflate, int nrhs, int nlsteps, const double* b,
                                                       double* alpha_s, double* beta_s, double* q_s,
                                                       double* bnorm) {
  try {
    Context& c = ctx();
    require_ready(true);
    WH_REQUIRE(nrhs >= 0 && nlsteps >= 1, "nrhs must be >= 0 and nlsteps >= 1");
    WH_REQUIRE(nbnd_to_deflate >= 0 && nbnd_to_deflate <= c.nbndval,
               "nbnd_to_deflate must not exceed the registered states (nbndval)");
    WH_REQUIRE(!c.l_kinetic_only, "the Lanczos chains need the full Hamiltonian (l_kinetic_only is set)");
    WH_REQUIRE(c.precision == 0, "the Lanczos chains run in FP64 (precision mode 0)");
    if (nrhs == 0) return 0;
    hipStream_t s = c.stream;
    const int npw = c.npw;
    const long ld = npw;
    const long k2 = 2L * npw;
    const size_t blk = static_cast<size_t>(nrhs) * npw;
    // basis (nlsteps blocks of nrhs columns, stick order), residual, scalars
    z64* Q = c.lz_q.as<z64>(static_cast<size_t>(nlsteps) * blk);
    z64* R = c.lz_r.as<z64>(blk);
    double* sc = c.lz_sc.as<double>(static_cast<size_t>(2 * nlsteps + 3) * nrhs);
    double* d_alpha = sc;                                   // nlsteps x nrhs
    double* d_beta_s = sc + static_cast<size_t>(nlsteps) * nrhs;   // nlsteps x nrhs (last unused)
    double* d_beta = d_beta_s + static_cast<size_t>(nlsteps) * nrhs;
    double* d_bnorm = d_beta + nrhs;
    double* d_e0 = d_bnorm + nrhs;
    WH_HIP(hipMemsetAsync(d_e0, 0, sizeof(double) * nrhs, s));
    {
      const size_t cin = static_cast<size_t>(nrhs) * c.npwx;
      const z64* bin = nullptr;
      if (on_device_mem(b)) {
        wait_for_caller(c);
        bin = reinterpret_cast<const z64*>(b);
      } else {
        z64* t = c.w_in.as<z64>(cin);
        WH_HIP(hipMemcpyAsync(t, b, sizeof(z64) * cin, hipMemcpyHostToDevice, s));
        bin = t;
      }
      gather_sticks(nrhs, npw, c.d_perm, bin, c.npwx, R, ld, nullptr, s);
    }
    const double* q = reinterpret_cast<const double*>(c.d_q);
    double* cm = c.w_cmat.as<double>(static_cast<size_t>(std::max(nbnd_to_deflate, 1)) * nrhs);
    // r -> q & beta (76-112)
    k_lan_norm<<<nrhs, NT, 0, s>>>(npw, c.gstart, R, ld, d_beta, d_bnorm);
    WH_HIP(hipGetLastError());
    k_lan_scale<<<dim3(ceil_div(npw, NT), nrhs), NT, 0, s>>>(npw, R, d_beta, Q, ld);
    WH_HIP(hipGetLastError());
    for (int il = 0; il < nlsteps; ++il) {
      z64* qi = Q + static_cast<size_t>(il) * blk;
      // r = H q  (h_psi_: the operator with e = 0, alpha = 0), then r = P_c r (144-145)
      stern_apply(qi, R, d_e0, nrhs, 0.0);
      if (nbnd_to_deflate > 0) {
        glbrak_q(0, nbnd_to_deflate, R, nrhs, cm);
        WH_TIMED("gemm_ket", dgemm(false, static_cast<int>(k2), nrhs, nbnd_to_deflate, -1.0, q, k2, cm,
                                   nbnd_to_deflate, 1.0, reinterpret_cast<double*>(R), k2, s));
      }
      const size_t row = static_cast<size_t>(il) * nrhs;
      WH_TIMED("lanczos_step", lan_step(nrhs,
                                        LanArgs{npw, c.gstart, il, R, Q, static_cast<long>(blk), ld,
                                                il + 1 < nlsteps ? qi + blk : nullptr, d_beta, d_alpha + row, d_beta,
                                                d_beta_s + row},
                                        s));
    }
    // outputs in the reference's layouts: alpha_s(NLSTEPS, NRHS), beta_s(NLSTEPS-1, NRHS),
    // q_s(npwx, NRHS, NLSTEPS), bnorm(NRHS)
    // [alpha | beta_s | beta | bnorm], nrhs each row
    std::vector<double> h(static_cast<size_t>(2 * nlsteps + 2) * nrhs);
    WH_HIP(hipMemcpyAsync(h.data(), sc, sizeof(double) * h.size(), hipMemcpyDeviceToHost, s));
    if (q_s) {
      const size_t cin = static_cast<size_t>(nrhs) * c.npwx;
      const bool dout = on_device_mem(q_s);
      for (int il = 0; il < nlsteps; ++il) {
        z64* dst = reinterpret_cast<z64*>(q_s) + static_cast<size_t>(il) * cin;
        z64* o = dout ? dst : c.w_out.as<z64>(cin);
        scatter_caller(nrhs, npw, c.npwx, c.d_perm, Q + static_cast<size_t>(il) * blk, ld, o, c.npwx, s);
        if (!dout) {
          WH_HIP(hipMemcpyAsync(dst, o, sizeof(z64) * cin, hipMemcpyDeviceToHost, s));
          WH_HIP(hipStreamSynchronize(s));
        }
      }
    }
    WH_HIP(hipStreamSynchronize(s));
    for (int ip = 0; ip < nrhs; ++ip) {
      for (int il = 0; il < nlsteps; ++il)
        alpha_s[static_cast<size_t>(ip) * nlsteps + il] = h[static_cast<size_t>(il) * nrhs + ip];
      if (beta_s)
        for (int il = 0; il + 1 < nlsteps; ++il)
          beta_s[static_cast<size_t>(ip) * (nlsteps - 1) + il] =
              h[static_cast<size_t>(nlsteps + il) * nrhs + ip];
      if (bnorm) bnorm[ip] = h[static_cast<size_t>(2 * nlsteps + 1) * nrhs + ip];
    }
    if (c.prof.on) c.prof.flush();
    return 0;
  } catch (const Error& e) {
    set_error(e.msg);
    return e.code < 0 ? e.code : -1;
  } catch (const std::exception& e) {
    set_error(e.what());
    return -3;
  }
}

// c(na, nb) = 2 Re <a_i|b_j> - Re a_i(G=0) Re b_j(G=0) for a(npwx, na), b(npwx, nb)
extern "C" int wh_glbrak_gamma(int na, const double* a, int nb, const double* b, double* c_out) {
  try {
    Context& c = ctx();
    require_ready(false);
    WH_REQUIRE(na >= 0 && nb >= 0, "na and nb must be >= 0");
    if (na == 0 || nb == 0) return 0;
    hipStream_t s = c.stream;
    const int npw = c.npw;
    const long ld = npw;
    auto stage = [&](const double* p, int n, DevBuf& tmp, DevBuf& st) {
      const size_t cin = static_cast<size_t>(n) * c.npwx;
      const z64* in = nullptr;
      if (on_device_mem(p)) {
        wait_for_caller(c);
        in = reinterpret_cast<const z64*>(p);
      } else {
        z64* t = tmp.as<z64>(cin);
        WH_HIP(hipMemcpyAsync(t, p, sizeof(z64) * cin, hipMemcpyHostToDevice, s));
        in = t;
      }
      z64* o = st.as<z64>(static_cast<size_t>(n) * npw);
      gather_sticks(n, npw, c.d_perm, in, c.npwx, o, ld, nullptr, s);
      return o;
    };
    const z64* A = stage(a, na, c.w_in, c.lz_q);
    const z64* B = stage(b, nb, c.w_out, c.lz_r);
    double* d = c.w_cmat.as<double>(static_cast<size_t>(na) * nb);
    WH_TIMED("gemm_bra", dgemm_bra(na, nb, static_cast<int>(2 * npw), 2.0, reinterpret_cast<const double*>(A), 2L * npw,
                                   reinterpret_cast<const double*>(B), 2L * npw, c.gstart == 2 ? 1.0 : 0.0, nullptr,
                                   d, na, s));
    WH_HIP(hipMemcpyAsync(c_out, d, sizeof(double) * na * nb, hipMemcpyDefault, s));
    WH_HIP(hipStreamSynchronize(s));
    return 0;
  } catch (const Error& e) {
    set_error(e.msg);
    return e.code < 0 ? e.code : -1;
  } catch (const std::exception& e) {
    set_error(e.what());
    return -3;
  }
}
