// FP64 GEMMs on CDNA4 matrix cores (v_mfma_f64_16x16x4_f64).
//
//   C (M x N) = alpha * op(A) * B + beta * C,  all column major,
//   op(A) = A^T when TA (A stored K x M), A otherwise (A stored M x K).
//
// These carry the Gamma-point projections of the reference, which are DGEMMs
// on the real view of the complex arrays (Hamiltonian_kernel/glbrak.f90:38-39,
// apply_alpha_pc_to_m_wfcs.f90:59, apply_alpha_pv_to_m_wfcs.f90:71) and the
// Davidson subspace products (Wstat/wstat_tools.f90 build_hr/update/refresh).
//
// Tile 128 x (32 WN) x 16 per 256-thread workgroup (WN = 4, 2 or 1): four
// wavefronts in a 2 x 2 arrangement, each owning 64 x 16 WN = 4 x WN MFMA
// 16x16 blocks.  One tile is multiplied out of LDS while the next goes from
// registers to the other half of the double buffer and the ones after are on
// their way from memory; both are issued between the two halves of the K
// steps, so neither is waited for at the barrier.  Bound: the FP64 matrix pipe
// (64 cycles an instruction and SIMD); what is left is the address and LDS work
// between the matrix instructions, so tiles are loaded 16 bytes a lane and
// read from LDS two K steps at a time; with few columns, reading the long
// operand once.  TFLOP/s with 8-byte loads, [k][x] tiles for both operands,
// fixed splits and partial sums added a load at a time -> now: bra 384 x N over
// K = 18,278: N = 8,192 55 -> 64, 4,096 50 -> 60, 1,000 43 -> 46, 128 27.5 -> 38;
// ket of the same sizes 50 -> 56, 49 -> 55, 47 -> 49, 26.5 -> 27.5; bra / ket
// 1,296 x 432 over 61,446 38 -> 41 / 40 -> 45; 260 x 40 over 18,278 6.2 -> 7.7 /
// 9.2; 8,192^3 60 -> 66.
//
// The projection ("bra") products have a small M (occupied bands +
// projectors) and a long K (2 npw), so they split K (pick_split); the partial
// products are summed in a fixed order by the epilogue kernel, which also
// applies the G = 0 correction of glbrak_gamma (its DGER) and the per-row
// scale, so results do not depend on scheduling.
//
// Operand layout of the 16x16x4 f64 instruction (checked on the device):
// lane l holds A[l%16][l/16] and B[l/16][l%16]; result register r of lane l
// holds D[l/16 + 4r][l%16].  The kernel passes the B block as the
// instruction's A operand and the A block as its B operand, so it forms
// D = (A B)^T: the 16 lanes of a quarter wave then hold 16 consecutive rows
// of C, i.e. consecutive addresses of the column-major result, and the
// epilogue's loads and stores of C are whole 128-byte runs (the ket products
// read and write a C of 2 npw rows and up to thousands of columns).
#include "wh_gemm.h"

#include <algorithm>
#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>
#include <cstring>
#include <functional>

namespace wh {

namespace {

constexpr int BM = 128;
constexpr int BK = 16;
constexpr int NT = 256;

typedef double v4d __attribute__((ext_vector_type(4)));

// Tile loads, 16 bytes at a time (8-byte alignment is enough), mapped so that
// each load instruction of a wavefront reads contiguous memory:
//  * x-contiguous operand (element (k, x) at P[k*ld + x]: A of the plain
//    product, XT = 128): x = 2 (tid % 64), k = tid / 64 + 4q  (1 kB per
//    instruction); in LDS [k][x] with rows of 132;
//  * k-contiguous operand (element (k, x) at P[x*ld + k]: A of the bra
//    product, B of both): k = 2 (tid % 8), x = tid / 8 + 32q  (eight 128-byte
//    runs); in LDS [x][k] (kc_at), so that a lane reads two K steps of its
//    row at once.
// The rows' addresses are scalar sums and one 32-bit offset per thread.
// An MFMA's four k may be any four of the tile as long as both operands agree:
// lanes 16 g .. 16 g + 15 take k = 4 g + step, which are adjacent in the
// k-contiguous rows.  The LDS is busy 13 to 18 % of the cycles of the 1,296 x 432
// products over 61,446, a third of that in bank conflicts for the bra (both
// operands k-contiguous) and 11 % for the ket, beside 62 and 63 % of the matrix
// pipe: not what bounds them.
// CHK: zero-fill outside [0, X) x [k0, kend) (edge tiles only).
typedef double d2 __attribute__((ext_vector_type(2), aligned(8)));

template <bool KCONT, int XT>
constexpr int tile_elems() { return KCONT ? XT * BK : BK * 132; }
// k-contiguous rows: 16-byte chunk c of row x sits at chunk c ^ ((x / 2) % 8),
// so that 16 rows' same chunk spreads over all banks without padding (49 kB for
// the 128 x 64 tiles: three workgroups a CU)
__device__ __forceinline__ int kc_at(int x, int c) { return x * BK + 2 * (c ^ ((x >> 1) & 7)); }
template <int XT>
constexpr int tile_loads() { return BK * XT / NT / 2; }

template <bool KCONT, bool CHK, int XT>
__device__ __forceinline__ void load_tile(d2 (&r)[tile_loads<XT>()], const double* __restrict__ P, long ld, int X,
                                          int x0, int k0, int kend) {
  const int tid = threadIdx.x;
  static_assert(KCONT || XT == 128, "x-contiguous tiles are 128 wide");
  const unsigned ldu = static_cast<unsigned>(ld);
  if (KCONT) {
    const int tk = 2 * (tid & 7), tx = tid >> 3;
    const unsigned off = tx * ldu + tk;
#pragma unroll
    for (int q = 0; q < tile_loads<XT>(); ++q) {
      const double* row = P + static_cast<long>(x0 + 32 * q) * ld + k0;
      if (CHK) {
        const bool in = x0 + 32 * q + tx < X;
        r[q].x = in && k0 + tk < kend ? row[off] : 0.0;
        r[q].y = in && k0 + tk + 1 < kend ? row[off + 1] : 0.0;
      } else {
        r[q] = *reinterpret_cast<const d2*>(row + off);
      }
    }
  } else {
    const int tx = 2 * (tid & 63), tk = tid >> 6;
    const unsigned off = tk * ldu + tx;
#pragma unroll
    for (int q = 0; q < tile_loads<XT>(); ++q) {
      const double* row = P + static_cast<long>(k0 + 4 * q) * ld + x0;
      if (CHK) {
        const bool in = k0 + 4 * q + tk < kend;
        r[q].x = in && x0 + tx < X ? row[off] : 0.0;
        r[q].y = in && x0 + tx + 1 < X ? row[off + 1] : 0.0;
      } else {
        r[q] = *reinterpret_cast<const d2*>(row + off);
      }
    }
  }
}

template <bool KCONT, int XT>
__device__ __forceinline__ void store_tile(double* S, const d2 (&r)[tile_loads<XT>()]) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < tile_loads<XT>(); ++q) {
    const int o = KCONT ? kc_at((tid >> 3) + 32 * q, tid & 7) : ((tid >> 6) + 4 * q) * 132 + 2 * (tid & 63);
    *reinterpret_cast<double2*>(S + o) = make_double2(r[q].x, r[q].y);
  }
}

// operand rows x0 + 16 i + lane % 16 for the K steps 2 h, 2 h + 1
template <bool KCONT, int NB>
__device__ __forceinline__ void read_ops(double (&v)[NB][2], const double* S, int x0, int lane, int h) {
  const int g = lane >> 4, x = x0 + (lane & 15);
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if (KCONT) {
      const double2 w = *reinterpret_cast<const double2*>(S + kc_at(x + 16 * i, 2 * g + h));
      v[i][0] = w.x;
      v[i][1] = w.y;
    } else {
      v[i][0] = S[(4 * g + 2 * h) * 132 + x + 16 * i];
      v[i][1] = S[(4 * g + 2 * h + 1) * 132 + x + 16 * i];
    }
  }
}

// K chunks of a split product: the cost of s chunks is the rounds of slots_of
// workgroups, each with its share of the K steps and about kOvh more for its
// first loads and its stores, and the partial sums' write and read at about
// 1.7 kB a cycle; candidates fill one or two rounds (up to four measured the
// same).  Whole numbers throughout: the host, which sizes grids and buffers,
// and the device must come to the same answer.
// (Three fixed splits, aimed at 512, 1,024 or 2,048 workgroups and timed
// against each other, left a last round nearly empty, e.g. 576 workgroups for
// 384 x 8,192, and were sized for the launch's columns, not the active ones.)
__host__ __device__ constexpr int slots_of(int wn) { return wn == 4 ? 512 : 768; }   // workgroups the chip holds
constexpr int kMaxRounds = 2;
constexpr int kMaxSplit = 64;
constexpr int kOvh = 5;
__host__ __device__ inline int pick_split(int M, int N, int K, int wn) {
  const int tiles = ((M + BM - 1) / BM) * ((N + 32 * wn - 1) / (32 * wn));
  const int kt = max((K + BK - 1) / BK, 1);
  const int slots = slots_of(wn);
  int best = 1;
  long cost = 0;
  for (int r = 0; r <= kMaxRounds; ++r) {
    // each chunk at least 16 steps long
    const int s = r == 0 ? 1 : min(min(slots * r / max(tiles, 1), kMaxSplit), kt / 16);
    if (s < 1) continue;
    const int per = (kt + s - 1) / s;
    const int n = (kt + per - 1) / per;   // chunks that the steps fill
    const int rounds = (tiles * n + slots - 1) / slots;
    const long c = static_cast<long>(rounds) * (per + kOvh) * (wn == 4 ? 8192 : 3072 * wn) +
                   (n > 1 ? static_cast<long>(M) * N * n * 5 / 512 : 0L);
    if (r == 0 || c < cost) {
      cost = c;
      best = n;
    }
  }
  return best;
}
__host__ __device__ inline int split_chunk(int K, int split) {
  const int kt = (K + BK - 1) / BK;
  return (kt + split - 1) / split * BK;
}

// Tiles (bx, by, kz): gx x gy output tiles times split K chunks of
// split_chunk(K, split).  partial: raw partial sums go to C + kz ldc N (alpha,
// beta ignored; N the active columns).  d_split (with d_n): where fewer than
// the launch's columns are active, the split is pick_split of those, and the
// one taken is left in *d_split for the epilogue.  The grid is 1D and its blocks are
// dispatched round-robin over the 8 XCDs (block L on XCD L % 8); tile
// W = (L % 8) * ceil(tiles / 8) + L / 8 puts consecutive tiles, which share
// their B panel (same by, kz) or A panel (same bx, kz), on one XCD and its L2.
constexpr int kXcds = 8;
__host__ __device__ inline int xcd_blocks(int tiles) { return (tiles + kXcds - 1) / kXcds * kXcds; }

// WN: 16-column MFMA blocks per wavefront along N, i.e. tiles of
// BM x (32 WN) (WN = 4: 128 x 128; narrower tiles give more workgroups to
// products with few columns).
// GRP: the columns fall into groups with a left operand of their own (device
// tables G); a tile lies within one group.
template <bool TA, int WN, bool GRP = false>
__global__ __launch_bounds__(NT, WN == 4 ? 2 : 3) void k_dgemm(int M, int N, int K, int split, bool partial, double alpha,
                                              const double* __restrict__ A, long lda, const double* __restrict__ B,
                                              long ldb, double beta, double* __restrict__ C, long ldc,
                                              int gx, int gy, const int* __restrict__ d_n, int* d_split, DgemmGroups G) {
  constexpr int TN = 32 * WN;
  if (GRP) {
    gy = G.tstart[G.ng];
    if (gy == 0) return;   // no active column
  } else if (d_n) {
    // columns the device left active: the tiles of the active columns are
    // renumbered over the whole grid, so they still spread over all XCDs
    const int na = min(N, *d_n);
    gy = min(gy, (na + TN - 1) / TN);
    if (gy == 0) return;   // no active column
    if (d_split) {
      if (na < N) split = pick_split(M, na, K, WN);
      if (blockIdx.x == 0 && threadIdx.x == 0) *d_split = split;
    }
    N = na;
  }
  const long pstride = ldc * N;   // (grouped: of the launch's N)
  const int kchunk = split_chunk(K, split);
  __shared__ __align__(16) double As[2][tile_elems<TA, BM>()];
  __shared__ __align__(16) double Bs[2][tile_elems<true, TN>()];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave & 1;
  const int wn = wave >> 1;
  const int tiles = gx * gy * split;
  // (with fewer active tiles than the grid was sized for, only the first
  // xcd_blocks(tiles) workgroups take part, so each tile has exactly one)
  if (static_cast<int>(blockIdx.x) >= xcd_blocks(tiles)) return;
  const int W = static_cast<int>(blockIdx.x % kXcds) * (xcd_blocks(tiles) / kXcds) + static_cast<int>(blockIdx.x / kXcds);
  if (W >= tiles) return;   // uniform per workgroup
  const int m0 = (W % gx) * BM;
  int n0 = ((W / gx) % gy) * TN;
  if (GRP) {
    const int by = (W / gx) % gy;
    int lo = 0, hi = G.ng;   // the last group that starts at or before this tile
    while (hi - lo > 1) {
      const int mid = (lo + hi) / 2;
      if (G.tstart[mid] <= by) lo = mid;
      else hi = mid;
    }
    A = G.A[lo];
    n0 = G.starts[lo] + (by - G.tstart[lo]) * TN;
    N = G.starts[lo + 1];
  }
  if (n0 >= N) return;      // uniform per workgroup
  const int kz = W / (gx * gy);
  const int kbeg = kz * kchunk;
  const int kend = min(K, kbeg + kchunk);
  // interior tiles load without bounds checks (all but a short last K step)
  const bool interior = m0 + BM <= M && n0 + TN <= N;
  // C = alpha AB + beta C on an interior tile: the C loads of a row block are
  // issued while the previous block is combined and stored.  (Accumulators
  // that start from C, their loads under the first tiles', measured 2-4 %
  // faster, but every partial sum is then rounded at the size of C.)
  const bool rmw = !partial && beta != 0.0 && interior;
  double* Cz = C + (partial ? static_cast<long>(kz) * pstride : 0L);
  const int row0 = m0 + wm * 64 + (lane & 15);
  const int col0 = n0 + wn * (16 * WN) + (lane >> 4);
  double cv[4 * WN];
  auto load_c = [&](int i) {
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) cv[4 * j + r] = Cz[static_cast<long>(col0 + j * 16 + 4 * r) * ldc + row0 + i * 16];
  };
  v4d acc[4][WN];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  const int ntile = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;
  // PF tiles on their way from memory: narrow tiles have the registers for
  // two, and little else to cover the latency with
  constexpr int PF = WN == 4 ? 1 : 2;
  d2 ra[PF][tile_loads<BM>()], rb[PF][tile_loads<TN>()];
  auto load = [&](int t, d2 (&qa)[tile_loads<BM>()], d2 (&qb)[tile_loads<TN>()]) {
    if (t >= ntile) return;
    const int k0 = kbeg + t * BK;
    if (interior && k0 + BK <= kend) {
      load_tile<TA, false, BM>(qa, A, lda, M, m0, k0, kend);
      load_tile<true, false, TN>(qb, B, ldb, N, n0, k0, kend);
    } else {
      load_tile<TA, true, BM>(qa, A, lda, M, m0, k0, kend);
      load_tile<true, true, TN>(qb, B, ldb, N, n0, k0, kend);
    }
  };
  auto store = [&](int buf, const d2 (&qa)[tile_loads<BM>()], const d2 (&qb)[tile_loads<TN>()]) {
    store_tile<TA, BM>(As[buf], qa);
    store_tile<true, TN>(Bs[buf], qb);
  };
  load(0, ra[0], rb[0]);
  if (PF > 1) load(1, ra[PF - 1], rb[PF - 1]);
  if (ntile > 0) store(0, ra[0], rb[0]);
  load(PF, ra[0], rb[0]);
  __syncthreads();
  // Per tile: half of the K steps, then the next tile (in the registers q)
  // goes to the other LDS buffer (free since the last barrier) and the loads
  // of the one PF after are issued, so neither is waited for at the barrier,
  // then the other half.
  auto step = [&](int t, d2 (&qa)[tile_loads<BM>()], d2 (&qb)[tile_loads<TN>()]) {
    const int cur = t & 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      double a[4][2], b[WN][2];
      read_ops<TA, 4>(a, As[cur], wm * 64, lane, h);
      read_ops<true, WN>(b, Bs[cur], wn * (16 * WN), lane, h);
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < WN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j][st], a[i][st], acc[i][j], 0, 0, 0);
      if (h == 0) {
        if (t + 1 < ntile) store(cur ^ 1, qa, qb);
        load(t + 1 + PF, qa, qb);
      }
    }
    __syncthreads();
  };
  for (int t = 0; t < ntile; t += PF) {
    // tile t + 1 is in set (t + 1) % PF
    step(t, ra[PF - 1], rb[PF - 1]);
    if (PF > 1 && t + 1 < ntile) step(t + 1, ra[0], rb[0]);
  }
  // block (i, j) holds the transposed product: register r of lane l is
  // C(row i*16 + l%16, column j*16 + l/16 + 4r), so lanes 0..15 (and each
  // further quarter wave) touch 16 consecutive rows of one column of C
  if (rmw) {
    // row block i is combined in its accumulators, the next block's C loads
    // are issued, then block i is stored
    load_c(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = alpha * acc[i][j][r] + beta * cv[4 * j + r];
      if (i + 1 < 4) load_c(i + 1);
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) Cz[static_cast<long>(col0 + j * 16 + 4 * r) * ldc + row0 + i * 16] = acc[i][j][r];
    }
  } else if (partial || beta == 0.0) {
    const double f = partial ? 1.0 : alpha;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = row0 + i * 16, col = col0 + j * 16 + 4 * r;
          if (interior || (row < M && col < N)) Cz[static_cast<long>(col) * ldc + row] = f * acc[i][j][r];
        }
  } else {
    // edge tile of C = alpha AB + beta C
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = row0 + i * 16;
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int col = col0 + j * 16 + 4 * r;
          cv[4 * j + r] = (row < M && col < N) ? Cz[static_cast<long>(col) * ldc + row] : 0.0;
        }
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int col = col0 + j * 16 + 4 * r;
          if (row < M && col < N) Cz[static_cast<long>(col) * ldc + row] = alpha * acc[i][j][r] + beta * cv[4 * j + r];
        }
    }
  }
}

// Bra product with few rows (M <= MB, e.g. the bands of a small molecule with
// no projectors): one workgroup per (column j, K chunk z) streams B's column
// once and keeps the M running sums per thread (A's rows come through the
// caches); partial sums P_z(i, j) at P + z * pstride + j * ldc + i.  With
// FIN (one K chunk) the workgroup writes the result itself, as k_reduce_g0
// would: P(i, j) = s_i * (alpha * sum - g0 * A[i*lda] * B[j*ldb]).
constexpr int NTS = 256;
struct BraFin {
  double alpha, g0;
  const double* s;
};
template <int MB, bool FIN>
__global__ __launch_bounds__(NTS) void k_bra_skinny(int M, int K, int kchunk, const double* __restrict__ A, long lda,
                                                   const double* __restrict__ B, long ldb, double* __restrict__ P,
                                                   long ldc, long pstride, const int* __restrict__ d_n, BraFin fin) {
  __shared__ double red[MB][NTS / 64];
  const int j = blockIdx.x;
  if (d_n && j >= *d_n) return;
  const int z = blockIdx.y;
  const int kb = z * kchunk;
  const int ke = min(K, kb + kchunk);
  const double* Bj = B + static_cast<long>(j) * ldb;
  double acc[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) acc[i] = 0.0;
  for (int k = kb + threadIdx.x; k < ke; k += NTS) {
    const double b = Bj[k];
#pragma unroll
    for (int i = 0; i < MB; ++i)
      if (i < M) acc[i] += A[static_cast<long>(i) * lda + k] * b;
  }
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    if (i < M) {
      double v = acc[i];
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      if (lane == 0) red[i][w] = v;
    }
  }
  __syncthreads();
  if (threadIdx.x < M) {
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < NTS / 64; ++q) v += red[threadIdx.x][q];
    if (FIN) {
      const double acc = 0.0 + v;
      v = fin.alpha * acc - fin.g0 * A[static_cast<long>(threadIdx.x) * lda] * Bj[0];
      if (fin.s) v *= fin.s[threadIdx.x];
    }
    P[static_cast<long>(z) * pstride + static_cast<long>(j) * ldc + threadIdx.x] = v;
  }
}

// C = alpha A B + beta C (column major, A: M x K, B: K x N) for small K
// (the ket product of a molecule with a few bands and no projectors): one
// thread per element of C, B's column in LDS.
template <int KB>
__global__ __launch_bounds__(NTS) void k_ket_skinny(int M, int K, double alpha, const double* __restrict__ A, long lda,
                                                   const double* __restrict__ B, long ldb, double beta,
                                                   double* __restrict__ C, long ldc, const int* __restrict__ d_n) {
  __shared__ double bj[KB];
  const int j = blockIdx.y;
  if (d_n && j >= *d_n) return;
  if (threadIdx.x < K) bj[threadIdx.x] = B[static_cast<long>(j) * ldb + threadIdx.x];
  __syncthreads();
  const int r = blockIdx.x * NTS + threadIdx.x;
  if (r >= M) return;
  double acc = 0.0;
#pragma unroll
  for (int i = 0; i < KB; ++i)
    if (i < K) acc += A[static_cast<long>(i) * lda + r] * bj[i];
  double* c = C + static_cast<long>(j) * ldc + r;
  *c = (beta == 0.0) ? alpha * acc : alpha * acc + beta * (*c);
}

// C(i, j) = s_i * (alpha * sum_z P_z(i, j) - g0 * a(1, i) * b(1, j))
//   P_z: split partials (ldc, stride pstride); a(1, i) = A[i*lda], b(1, j) = B[j*ldb]
// pstride 0: ldc x the active columns; d_split: k_dgemm's split of those
__global__ void k_reduce_g0(int M, int N, int nsplit, const double* P, long pstride, double alpha, double g0,
                            const double* A, long lda, const double* B, long ldb, const double* s, double* C,
                            long ldc, const int* d_n, const int* d_split) {
  if (d_n) N = min(N, *d_n);
  if (pstride == 0) pstride = ldc * N;
  const long idx = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= static_cast<long>(M) * N) return;
  const int i = static_cast<int>(idx % M);
  const int j = static_cast<int>(idx / M);
  const long o = static_cast<long>(j) * ldc + i;
  if (d_split) nsplit = *d_split;
  // in order, four loads at a time
  double acc = 0.0;
  const double* p = P + o;
  int z = 0;
  for (; z + 4 <= nsplit; z += 4, p += 4 * pstride) {
    const double a0 = p[0], a1 = p[pstride], a2 = p[2 * pstride], a3 = p[3 * pstride];
    acc += a0;
    acc += a1;
    acc += a2;
    acc += a3;
  }
  for (; z < nsplit; ++z, p += pstride) acc += *p;
  double v = alpha * acc;
  if (g0 != 0.0) v -= g0 * A[static_cast<long>(i) * lda] * B[static_cast<long>(j) * ldb];
  if (s) v *= s[i];
  C[o] = v;
}

// C(i, j) = scale_i * (C(i, j) - g0 * A[i*lda] * B[j*ldb])   (scale may be null)
__global__ void k_g0_scale(int M, int N, double g0, const double* A, long lda, const double* B, long ldb,
                           const double* s, double* C, long ldc) {
  const long idx = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= static_cast<long>(M) * N) return;
  const int i = static_cast<int>(idx % M);
  const int j = static_cast<int>(idx / M);
  double v = C[static_cast<long>(j) * ldc + i] - g0 * A[static_cast<long>(i) * lda] * B[static_cast<long>(j) * ldb];
  if (s) v *= s[i];
  C[static_cast<long>(j) * ldc + i] = v;
}

// Grows on demand; before a larger buffer replaces the old one, the streams
// that used it (this host thread's calls only) are drained, so no other
// system's stream is waited for.
struct Scratch {
  double* p = nullptr;
  size_t n = 0;
  std::vector<hipStream_t> users;
  double* get(size_t count, hipStream_t s) {
    if (count > n) {
      if (p) {
        for (hipStream_t u : users) WH_HIP(hipStreamSynchronize(u));
        WH_HIP(hipFree(p));
      }
      users.clear();
      p = nullptr;
      WH_HIP(hipMalloc(&p, sizeof(double) * count));
      n = count;
    }
    if (std::find(users.begin(), users.end(), s) == users.end()) users.push_back(s);
    return p;
  }
};

// split-K partial sums, per host thread
Scratch& partials() {
  static thread_local Scratch s;
  return s;
}

}  // namespace

// split: K chunks; more than one, or partial: partial sums.  d_split: see k_dgemm
template <bool TA, int WN>
static void launch_tiles(int M, int N, int K, int split, bool partial, double alpha, const double* A, long lda,
                         const double* B, long ldb, double beta, double* C, long ldc, hipStream_t s, const int* d_n,
                         int* d_split) {
  const int gx = ceil_div(M, BM), gy = ceil_div(N, 32 * WN);
  // fewer active columns than N may be cut into more chunks: the most workgroups any split makes
  const int wgs = d_split ? std::max(gx * gy * split, slots_of(WN) * kMaxRounds) : gx * gy * split;
  k_dgemm<TA, WN><<<xcd_blocks(wgs), NT, 0, s>>>(M, N, K, split, partial, alpha, A, lda, B, ldb, beta, C, ldc, gx, gy,
                                                 d_n, d_split, DgemmGroups{});
  WH_HIP(hipGetLastError());
}

// tile width variants: WN = 4, 2, 1 (128-, 64- and 32-column tiles)
template <bool TA>
static void launch_wn(int v, int M, int N, int K, int split, bool partial, double alpha, const double* A, long lda,
                      const double* B, long ldb, double beta, double* C, long ldc, hipStream_t s,
                      const int* d_n = nullptr, int* d_split = nullptr) {
  if (v == 0) launch_tiles<TA, 4>(M, N, K, split, partial, alpha, A, lda, B, ldb, beta, C, ldc, s, d_n, d_split);
  else if (v == 1) launch_tiles<TA, 2>(M, N, K, split, partial, alpha, A, lda, B, ldb, beta, C, ldc, s, d_n, d_split);
  else launch_tiles<TA, 1>(M, N, K, split, partial, alpha, A, lda, B, ldb, beta, C, ldc, s, d_n, d_split);
}
constexpr int kWnVariants = 3;
inline int wn_of(int v) { return 4 >> v; }

// The variant of a product shape is chosen once, by timing every variant on
// the first call's own arguments (two rounds; the first warms the code up);
// results never depend on the choice beyond rounding of a fixed order.
using VariantKey = std::tuple<int, int, int, int, int>;
static std::map<VariantKey, int>& chosen_variants() {
  static std::map<VariantKey, int> m;
  return m;
}
static std::mutex g_variant_mutex;

static int time_variants(int nv, const std::function<void(int)>& run, hipStream_t s, float* t) {
  hipEvent_t a, b;
  WH_HIP(hipEventCreate(&a));
  WH_HIP(hipEventCreate(&b));
  for (int rep = 0; rep < 2; ++rep)
    for (int v = 0; v < nv; ++v) {
      WH_HIP(hipEventRecord(a, s));
      run(v);
      WH_HIP(hipEventRecord(b, s));
      WH_HIP(hipEventSynchronize(b));
      float ms = 0.f;
      WH_HIP(hipEventElapsedTime(&ms, a, b));
      if (rep == 1) t[v] = ms;
    }
  WH_HIP(hipEventDestroy(a));
  WH_HIP(hipEventDestroy(b));
  int best = 0;
  for (int v = 1; v < nv; ++v)
    if (t[v] < t[best]) best = v;
  return best;
}

static int log2_bucket(int n) {
  int lg = 0;
  while ((2 << lg) <= n) ++lg;
  return lg;
}

void dgemm(bool transa, int M, int N, int K, double alpha, const double* A, long lda, const double* B, long ldb,
           double beta, double* C, long ldc, hipStream_t s, const int* d_n) {
  if (M <= 0 || N <= 0) return;
  if (!transa && K > 0 && K <= 32 && N <= 256) {
    // inner dimension of a few bands: a streaming kernel (the matrix-core tiles would be nearly empty)
    dim3 grid(ceil_div(M, NTS), N);
    if (K <= 8) k_ket_skinny<8><<<grid, NTS, 0, s>>>(M, K, alpha, A, lda, B, ldb, beta, C, ldc, d_n);
    else if (K <= 16) k_ket_skinny<16><<<grid, NTS, 0, s>>>(M, K, alpha, A, lda, B, ldb, beta, C, ldc, d_n);
    else k_ket_skinny<32><<<grid, NTS, 0, s>>>(M, K, alpha, A, lda, B, ldb, beta, C, ldc, d_n);
    WH_HIP(hipGetLastError());
    return;
  }
  const int K0 = std::max(K, 0);
  auto run = [&](int v, double* Cv) {
    if (transa) launch_wn<true>(v, M, N, K0, 1, false, alpha, A, lda, B, ldb, beta, Cv, ldc, s, d_n);
    else launch_wn<false>(v, M, N, K0, 1, false, alpha, A, lda, B, ldb, beta, Cv, ldc, s, d_n);
  };
  // tile width, timed once per (op, M, log2 K, log2 N)
  const VariantKey key{0, transa ? 1 : 0, M, log2_bucket(std::max(K, 1)), log2_bucket(N)};
  std::unique_lock<std::mutex> lk(g_variant_mutex);
  auto it = chosen_variants().find(key);
  if (it == chosen_variants().end()) {
    // timed on a scratch copy of C's shape: C += AB must run once only
    double* tmp = nullptr;
    WH_HIP(hipMalloc(&tmp, sizeof(double) * static_cast<size_t>(ldc) * N));
    WH_HIP(hipMemsetAsync(tmp, 0, sizeof(double) * static_cast<size_t>(ldc) * N, s));
    float t[kWnVariants] = {};
    const int best = time_variants(kWnVariants, [&](int v) { run(v, tmp); }, s, t);
    WH_HIP(hipStreamSynchronize(s));
    WH_HIP(hipFree(tmp));
    if (tune_log())
      std::fprintf(stderr, "[west_hip] dgemm%s M=%d N=%d K=%d: tiles 128x128 %.3f 128x64 %.3f 128x32 %.3f ms -> %d\n",
                   transa ? "_t" : "", M, N, K, t[0], t[1], t[2], best);
    it = chosen_variants().emplace(key, best).first;
  }
  const int pick = it->second;
  lk.unlock();
  run(pick, C);
}

// doubles of partial sums for N columns, or (upto) for any count up to N:
// pick_split gives at most slots_of kMaxRounds workgroups beyond one chunk
static long partials_doubles(int M, int N, int K, long ldc, int wn, bool upto) {
  if (!upto) return static_cast<long>(pick_split(M, N, K, wn)) * ldc * N;
  const long cols = std::max<long>(N, static_cast<long>(slots_of(wn)) * kMaxRounds * 32 * wn / ceil_div(M, BM));
  return std::min<long>(cols, static_cast<long>(kMaxSplit) * N) * ldc;
}

// v: tile width variant.  P: room for the split-K partial sums (null: the per-thread scratch)
static void dgemm_bra_own(int M, int N, int K, double alpha, const double* A, long lda, const double* B, long ldb,
                          double g0, const double* scale, double* C, long ldc, hipStream_t s, int v = 0,
                          double* P = nullptr, const int* d_n = nullptr) {
  const int wn = wn_of(v);
  int* d_split = nullptr;   // behind the partial sums
  if (!P) {
    const long n = partials_doubles(M, N, K, ldc, wn, d_n != nullptr);
    P = partials().get(static_cast<size_t>(n) + 1, s);
    if (d_n) d_split = reinterpret_cast<int*>(P + n);
  }
  const int split = pick_split(M, N, K, wn);
  launch_wn<true>(v, M, N, std::max(K, 0), split, true, 1.0, A, lda, B, ldb, 0.0, P, ldc, s, d_n, d_split);
  const long n = static_cast<long>(M) * N;
  k_reduce_g0<<<ceil_div(n, 256), 256, 0, s>>>(M, N, split, P, 0, alpha, g0, A, lda, B, ldb, scale, C, ldc, d_n,
                                               d_split);
  WH_HIP(hipGetLastError());
}

static void skinny_split(int N, int K, int& split, int& kchunk) {
  // about 2048 workgroups, K chunks of at least 1024
  split = std::max(1, std::min(ceil_div(2048, N), K / 1024));
  kchunk = ceil_div(std::max(K, 1), split);
  split = ceil_div(std::max(K, 1), kchunk);
}

static void dgemm_bra_skinny(int M, int N, int K, double alpha, const double* A, long lda, const double* B, long ldb,
                             double g0, const double* scale, double* C, long ldc, hipStream_t s, double* P = nullptr,
                             const int* d_n = nullptr) {
  int split = 1, kchunk = 1;
  skinny_split(N, K, split, kchunk);
  const long pstride = static_cast<long>(ldc) * N;
  const BraFin fin{alpha, g0, scale};
  dim3 grid(N, split);
  if (split == 1) {   // one K chunk: the workgroups write C themselves
    if (M <= 8) k_bra_skinny<8, true><<<grid, NTS, 0, s>>>(M, K, kchunk, A, lda, B, ldb, C, ldc, pstride, d_n, fin);
    else if (M <= 16)
      k_bra_skinny<16, true><<<grid, NTS, 0, s>>>(M, K, kchunk, A, lda, B, ldb, C, ldc, pstride, d_n, fin);
    else k_bra_skinny<32, true><<<grid, NTS, 0, s>>>(M, K, kchunk, A, lda, B, ldb, C, ldc, pstride, d_n, fin);
    WH_HIP(hipGetLastError());
    return;
  }
  if (!P) P = partials().get(static_cast<size_t>(split) * pstride, s);
  if (M <= 8) k_bra_skinny<8, false><<<grid, NTS, 0, s>>>(M, K, kchunk, A, lda, B, ldb, P, ldc, pstride, d_n, fin);
  else if (M <= 16)
    k_bra_skinny<16, false><<<grid, NTS, 0, s>>>(M, K, kchunk, A, lda, B, ldb, P, ldc, pstride, d_n, fin);
  else k_bra_skinny<32, false><<<grid, NTS, 0, s>>>(M, K, kchunk, A, lda, B, ldb, P, ldc, pstride, d_n, fin);
  WH_HIP(hipGetLastError());
  const long n = static_cast<long>(M) * N;
  k_reduce_g0<<<ceil_div(n, 256), 256, 0, s>>>(M, N, split, P, pstride, alpha, g0, A, lda, B, ldb, scale, C, ldc,
                                               d_n, nullptr);
  WH_HIP(hipGetLastError());
}

void dgemm_bra(int M, int N, int K, double alpha, const double* A, long lda, const double* B, long ldb, double g0,
               const double* scale, double* C, long ldc, hipStream_t s, const int* d_n) {
  if (M <= 0 || N <= 0) return;
  // a few rows and columns: the matrix-core tiles (128 x 128) would be almost
  // empty (with many columns the tiles' reuse of A wins again)
  if (M <= 32 && N <= 256 && K > 0)
    return dgemm_bra_skinny(M, N, K, alpha, A, lda, B, ldb, g0, scale, C, ldc, s, nullptr, d_n);
  if (K <= 0 || N < 32) return dgemm_bra_own(M, N, K, alpha, A, lda, B, ldb, g0, scale, C, ldc, s, 2, nullptr, d_n);
  // tile widths, timed once per (M, K, log2 N); C is written (not accumulated),
  // so the timing runs on the call's own output
  constexpr int nv = kWnVariants;
  auto run = [&](int v) { dgemm_bra_own(M, N, K, alpha, A, lda, B, ldb, g0, scale, C, ldc, s, v, nullptr, d_n); };
  const VariantKey key{1, 1, M, K, log2_bucket(N)};
  std::unique_lock<std::mutex> lk(g_variant_mutex);
  auto it = chosen_variants().find(key);
  if (it == chosen_variants().end()) {
    float t[nv] = {};
    const int best = time_variants(nv, run, s, t);
    if (tune_log()) {
      std::fprintf(stderr, "[west_hip] dgemm_bra M=%d N=%d K=%d:", M, N, K);
      for (int v = 0; v < nv; ++v) std::fprintf(stderr, " 128x%d split %d %.3f", 32 * wn_of(v),
                                                pick_split(M, N, K, wn_of(v)), t[v]);
      std::fprintf(stderr, " ms -> %d\n", best);
    }
    it = chosen_variants().emplace(key, best).first;
  }
  const int pick = it->second;
  lk.unlock();
  // recomputed with the chosen variant, so the result does not depend on the timing order
  run(pick);
}

// ---- grouped products (one left operand per group of columns) -------------
// 64-column tiles: a group (one k point's active columns) has a few tens to
// a few hundred columns.
static_assert(kGroupTile == 64, "the grouped products run k_dgemm's WN = 2 tiles");

template <bool TA>
static void launch_groups(const DgemmGroups& G, int M, int N, int K, int split, bool partial, double alpha, long lda,
                          const double* B, long ldb, double beta, double* C, long ldc, hipStream_t s) {
  const int gx = ceil_div(M, BM), gy = ceil_div(N, kGroupTile) + G.ng;
  k_dgemm<TA, 2, true><<<xcd_blocks(gx * gy * split), NT, 0, s>>>(M, N, K, split, partial, alpha, nullptr, lda, B, ldb,
                                                                  beta, C, ldc, gx, gy, nullptr, nullptr, G);
  WH_HIP(hipGetLastError());
}

void dgemm_bra_groups(const DgemmGroups& G, int M, int N, int K, long lda, const double* B, long ldb,
                      const double* scale, double* C, long ldc, hipStream_t s, const int* d_n) {
  if (M <= 0 || N <= 0) return;
  // as pick_split, for the fewest tiles N columns can make
  const int split = pick_split(M, N, K, kGroupTile / 32);
  const long pstride = static_cast<long>(ldc) * N;
  double* P = partials().get(static_cast<size_t>(split) * pstride, s);
  launch_groups<true>(G, M, N, K, split, true, 1.0, lda, B, ldb, 0.0, P, ldc, s);
  const long n = static_cast<long>(M) * N;
  k_reduce_g0<<<ceil_div(n, 256), 256, 0, s>>>(M, N, split, P, pstride, 1.0, 0.0, nullptr, 0, nullptr, 0, scale, C,
                                               ldc, d_n, nullptr);
  WH_HIP(hipGetLastError());
}

void dgemm_ket_groups(const DgemmGroups& G, int M, int N, int K, long lda, const double* B, long ldb, double beta,
                      double* C, long ldc, hipStream_t s) {
  if (M <= 0 || N <= 0) return;
  launch_groups<false>(G, M, N, K, 1, false, 1.0, lda, B, ldb, beta, C, ldc, s);
}

// ---- products for callers that neither allocate nor time -------------------
// The variant an earlier timed call chose for the shape, else a fixed one.
static int chosen_or(const VariantKey& key, int dflt) {
  std::lock_guard<std::mutex> lk(g_variant_mutex);
  auto it = chosen_variants().find(key);
  return it != chosen_variants().end() ? it->second : dflt;
}

static int bra_untimed_variant(int M, int N, int K) {
  // default: 128 x 64 tiles (the most frequent winner of the timing)
  return (K <= 0 || N < 32) ? 2 : chosen_or(VariantKey{1, 1, M, K, log2_bucket(N)}, 1);
}

long bra_partials_doubles(int M, int N, int K, long ldc, int* variant) {
  *variant = 0;
  if (M <= 0 || N <= 0) return 0;
  int split = 1, kchunk = 1;
  if (M <= 32 && N <= 256 && K > 0) {
    skinny_split(N, K, split, kchunk);
  } else {
    *variant = bra_untimed_variant(M, N, K);
    return partials_doubles(M, N, K, ldc, wn_of(*variant), false);
  }
  return static_cast<long>(split) * ldc * N;
}

void dgemm_bra_into(int M, int N, int K, double alpha, const double* A, long lda, const double* B, long ldb,
                    double g0, const double* scale, double* C, long ldc, double* P, int variant, hipStream_t s) {
  if (M <= 0 || N <= 0) return;
  if (M <= 32 && N <= 256 && K > 0) return dgemm_bra_skinny(M, N, K, alpha, A, lda, B, ldb, g0, scale, C, ldc, s, P);
  dgemm_bra_own(M, N, K, alpha, A, lda, B, ldb, g0, scale, C, ldc, s, variant, P);
}

void dgemm_untimed(bool transa, int M, int N, int K, double alpha, const double* A, long lda, const double* B,
                   long ldb, double beta, double* C, long ldc, hipStream_t s) {
  if (M <= 0 || N <= 0) return;
  if (!transa && K > 0 && K <= 32 && N <= 256) return dgemm(transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, s);
  // default tile width: the widest that still gives two workgroups per compute unit
  int dflt = kWnVariants - 1;
  for (int v = 0; v < kWnVariants; ++v)
    if (static_cast<long>(ceil_div(M, BM)) * ceil_div(N, 32 * wn_of(v)) >= 512) {
      dflt = v;
      break;
    }
  const int v = chosen_or(VariantKey{0, transa ? 1 : 0, M, log2_bucket(std::max(K, 1)), log2_bucket(N)}, dflt);
  const int K0 = std::max(K, 0);
  if (transa) launch_wn<true>(v, M, N, K0, 1, false, alpha, A, lda, B, ldb, beta, C, ldc, s);
  else launch_wn<false>(v, M, N, K0, 1, false, alpha, A, lda, B, ldb, beta, C, ldc, s);
}

void g0_fix_scale(int M, int N, double g0, const double* A, long lda, const double* B, long ldb,
                  const double* scale, double* C, long ldc, hipStream_t s) {
  const long n = static_cast<long>(M) * N;
  if (n <= 0) return;
  k_g0_scale<<<ceil_div(n, 256), 256, 0, s>>>(M, N, g0, A, lda, B, ldb, scale, C, ldc);
  WH_HIP(hipGetLastError());
}

}  // namespace wh
