// J and K contraction kernels for gfx950 (see jk.hpp for the data layout).
//
// MFMA usage:
//   FP64   v_mfma_f64_16x16x4_f64   (A/B one element per lane, K = 4)
//   FP32   v_mfma_f32_16x16x4_f32   (same operand layout, FP32 accumulation)
//   BF16X3 v_mfma_f32_16x16x32_bf16 (8 bf16 per lane, K = 32); each FP32
//          operand x is split as hi = bf16(x), lo = bf16(x - hi) and the
//          product is accumulated as hi*hi + hi*lo + lo*hi in FP32.
// Accumulator layout (measured on gfx950): column lane % 16 in every case;
// row 4*(lane/16) + r in register r for the FP32 and BF16 instructions, but
// row lane/16 + 4*r for v_mfma_f64_16x16x4_f64 (AccRow below).
#include "jk.hpp"

#include <algorithm>
#include <cmath>

namespace vqc {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float fl2 __attribute__((ext_vector_type(2)));

template <class T>
struct AccOf;
template <>
struct AccOf<double> {
  using type = d4;
};
template <>
struct AccOf<float> {
  using type = f4;
};

// Row of accumulator register r held by `lane` in a 16x16 MFMA tile.
template <class T>
__device__ __forceinline__ int acc_row(int lane, int r) {
  return 4 * (lane >> 4) + r;
}
template <>
__device__ __forceinline__ int acc_row<double>(int lane, int r) {
  return (lane >> 4) + 4 * r;
}

__device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma(bf8 a, bf8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ std::size_t packed_index(int mu, int nu) {
  const std::size_t hi = mu > nu ? mu : nu, lo = mu > nu ? nu : mu;
  return hi * (hi + 1) / 2 + lo;
}

__device__ __forceinline__ void unpack_pair(std::size_t p, int& mu, int& nu) {
  int m = static_cast<int>((sqrt(8.0 * static_cast<double>(p) + 1.0) - 1.0) * 0.5);
  while (static_cast<std::size_t>(m) * (m + 1) / 2 > p) --m;
  while (static_cast<std::size_t>(m + 1) * (m + 2) / 2 <= p) ++m;
  mu = m;
  nu = static_cast<int>(p - static_cast<std::size_t>(m) * (m + 1) / 2);
}

__device__ __forceinline__ void split_bf16(float x, __bf16& hi, __bf16& lo) {
  hi = static_cast<__bf16>(x);
  lo = static_cast<__bf16>(x - static_cast<float>(hi));
}

// LDS tiles of 32 bf16 per row (64 bytes, four 16-byte chunks, no padding)
// that MFMA fragments read as 16 consecutive rows at one chunk: chunk c of
// row r is stored at position c ^ ((r >> 1) & 3), so the 16 reads of a
// fragment cover all 64 banks once (a padded 80-byte row leaves 2-way
// conflicts; measured 3.4e9 conflict cycles per (H2O)64 U launch, zero with
// this layout).
__device__ __forceinline__ int lds_chunk(int row, int chunk) { return chunk ^ ((row >> 1) & 3); }

// Split of eight floats into bf16 hi/lo fragments, two at a time (one packed
// conversion per pair for hi and one for lo).
__device__ __forceinline__ void split8_bf16(const float (&x)[8], bf8& hi, bf8& lo) {
  bf2 h[4], l[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const fl2 v = {x[2 * k], x[2 * k + 1]};
    h[k] = __builtin_convertvector(v, bf2);
    l[k] = __builtin_convertvector(v - __builtin_convertvector(h[k], fl2), bf2);
  }
  hi = __builtin_shufflevector(__builtin_shufflevector(h[0], h[1], 0, 1, 2, 3), __builtin_shufflevector(h[2], h[3], 0, 1, 2, 3),
                               0, 1, 2, 3, 4, 5, 6, 7);
  lo = __builtin_shufflevector(__builtin_shufflevector(l[0], l[1], 0, 1, 2, 3), __builtin_shufflevector(l[2], l[3], 0, 1, 2, 3),
                               0, 1, 2, 3, 4, 5, 6, 7);
}

// ---------------------------------------------------------------------------
// J
// ---------------------------------------------------------------------------

__global__ void pack_density_kernel(const double* __restrict__ D, int n, double* __restrict__ dp) {
  const std::size_t p = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= static_cast<std::size_t>(n) * (n + 1) / 2) return;
  int mu, nu;
  unpack_pair(p, mu, nu);
  const std::size_t a = static_cast<std::size_t>(mu) * n + nu, b = static_cast<std::size_t>(nu) * n + mu;
  dp[p] = mu == nu ? D[a] : D[a] + D[b];
}

constexpr int kRhoThreads = 256;

template <class T, int V>
__global__ __launch_bounds__(kRhoThreads) void coulomb_rho_kernel(const T* __restrict__ B,
                                                                  const double* __restrict__ dp,
                                                                  std::size_t npair, int ldq, std::size_t chunk,
                                                                  double* __restrict__ partial) {
  const int q = (blockIdx.x * kRhoThreads + threadIdx.x) * V;
  if (q >= ldq) return;
  const std::size_t p0 = static_cast<std::size_t>(blockIdx.y) * chunk;
  const std::size_t p1 = p0 + chunk < npair ? p0 + chunk : npair;
  double acc[V];
#pragma unroll
  for (int v = 0; v < V; ++v) acc[v] = 0.0;
  for (std::size_t p = p0; p < p1; ++p) {
    const double w = dp[p];
    const T* row = B + p * ldq + q;
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] += w * static_cast<double>(row[v]);
  }
  double* out = partial + static_cast<std::size_t>(blockIdx.y) * ldq + q;
#pragma unroll
  for (int v = 0; v < V; ++v) out[v] = acc[v];
}

// out[c] = sum_r partial[r][c]: 64 columns per block, 16 row groups per
// column reduced through LDS in a fixed order (deterministic).
constexpr int kSumCols = 64, kSumGroups = 16;
__global__ __launch_bounds__(kSumCols * kSumGroups) void sum_rows_kernel(const double* __restrict__ partial, int rows,
                                                                        int cols, double* __restrict__ out) {
  __shared__ double red[kSumGroups][kSumCols];
  const int lane = threadIdx.x % kSumCols, g = threadIdx.x / kSumCols;
  const int c = blockIdx.x * kSumCols + lane;
  double s = 0.0;
  if (c < cols) {
#pragma unroll 16
    for (int r = g; r < rows; r += kSumGroups) s += partial[static_cast<std::size_t>(r) * cols + c];
  }
  red[g][lane] = s;
  __syncthreads();
  if (g == 0 && c < cols) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < kSumGroups; ++k) t += red[k][lane];
    out[c] = t;
  }
}

template <class T>
struct Vec16;
template <>
struct Vec16<double> {
  using type = double __attribute__((ext_vector_type(2)));
};
template <>
struct Vec16<float> {
  using type = float __attribute__((ext_vector_type(4)));
};

constexpr int kJThreads = 1024, kJInFlight = 12;

// J_p = sum_Q B[p][Q] rho_Q, one wavefront per packed row.  Each lane keeps
// kJInFlight 16-byte loads of its row in flight before consuming them (12
// cover a 2432-wide FP32 row in one batch), and a 1024-thread block shares
// one LDS copy of rho, so with up to 128 VGPRs per lane one block (16 waves)
// per CU keeps enough bytes outstanding to stream B at HBM rate.
template <class T>
__global__ __launch_bounds__(kJThreads) __attribute__((amdgpu_waves_per_eu(4))) void coulomb_matrix_kernel(const T* __restrict__ B,
                                                                  const double* __restrict__ rho,
                                                                  std::size_t npair, int ldq, int n,
                                                                  double* __restrict__ J) {
  using V = typename Vec16<T>::type;
  constexpr int W = 16 / sizeof(T), STEP = 64 * W;
  extern __shared__ double srho[];
  for (int q = threadIdx.x; q < ldq; q += blockDim.x) srho[q] = rho[q];
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const std::size_t wave = static_cast<std::size_t>(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6);
  const std::size_t nwave = static_cast<std::size_t>(gridDim.x) * (blockDim.x / 64);
  for (std::size_t p = wave; p < npair; p += nwave) {
    const T* row = B + p * ldq;
    double s = 0.0;
    for (int q0 = lane * W; q0 < ldq; q0 += STEP * kJInFlight) {
      V v[kJInFlight];
#pragma unroll
      for (int u = 0; u < kJInFlight; ++u) {
        const int q = q0 + u * STEP;
        v[u] = q < ldq ? *reinterpret_cast<const V*>(row + q) : V{};
      }
#pragma unroll
      for (int u = 0; u < kJInFlight; ++u) {
        const int q = q0 + u * STEP;
        if (q < ldq) {
#pragma unroll
          for (int e = 0; e < W; ++e) s += static_cast<double>(v[u][e]) * srho[q + e];
        }
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) {
      int mu, nu;
      unpack_pair(p, mu, nu);
      J[static_cast<std::size_t>(mu) * n + nu] = s;
      J[static_cast<std::size_t>(nu) * n + mu] = s;
    }
  }
}

// ---------------------------------------------------------------------------
// K, step 1: U[mu][i][Q] = sum_nu B[(mu,nu)][Q] C[nu][i]
// Block: 2 x WQ waves (WQ along Q x 2 along i); tile 32*WQ (Q) x 32*NIW (i),
// i.e. all occupied columns up to 320 in one block, so each packed row of B
// is streamed once per mu.  Every wave owns 2 x NIW MFMA 16x16 tiles.  FP32 and
// BF16X3 use WQ = 8 (1024 threads, 256 rows of Q per C tile); FP64 uses
// WQ = 4 so its 2 x NIW x 4 double accumulators fit the register budget.
// ---------------------------------------------------------------------------

template <class T, int NIW, int WQ>
__global__ __launch_bounds__(128 * WQ) void occupied_u_kernel(const T* __restrict__ B, const T* __restrict__ C,
                                                             T* __restrict__ U, std::size_t us, int n, int ldq,
                                                             int ldc, int r, int nqb, const double* __restrict__ D,
                                                             double* __restrict__ rho_part) {
  using Acc = typename AccOf<T>::type;
  constexpr int BQ = 32 * WQ, BK = 16, BI = 32 * NIW, NT = 128 * WQ;
  constexpr int CP = (BK * BI + NT - 1) / NT;  // C elements staged per thread
  __shared__ T Bs[2][BK][BQ];
  __shared__ T Cs[2][BK][BI];
  // Q-tile-major order: the blocks in flight share one Q tile, so the
  // second gather of each packed row (as (mu, nu) and as (nu, mu)) finds it
  // in the last-level cache instead of HBM.
  const int mu = blockIdx.x % n;
  const int q0 = (blockIdx.x / n) * BQ;
  const int i0 = blockIdx.y * BI;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wq = wave % WQ, wi = wave / WQ;
  Acc acc[2][NIW];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < NIW; ++y) acc[x][y] = Acc{};
  const int bk = tid / (BQ / 4), bq = (tid % (BQ / 4)) * 4;
  // The first i-block also forms rho_Q partials, sum_nu D[mu][nu] B[(mu,nu)][Q],
  // from the B values it streams anyway (FP64 accumulation).
  const bool with_rho = rho_part != nullptr && blockIdx.y == 0;
  double racc[4] = {0.0, 0.0, 0.0, 0.0};
  extern __shared__ double drow[];  // D[mu][:], staged once when rho is formed
  if (with_rho)
    for (int k = tid; k < n; k += NT) drow[k] = D[static_cast<std::size_t>(mu) * n + k];
  __syncthreads();
  T rb[4], rc[CP];
  double rd = 0.0;
  // Stage the next k-step in registers so its global latency overlaps the
  // MFMAs of the current one; LDS is double-buffered (one barrier per step).
  // Staged values are only consumed in sstore, after the MFMAs.
  auto gload = [&](int nu0) {
    const int nu = nu0 + bk, q = q0 + bq;
    if (nu < n && q < ldq) {
      const T* src = B + packed_index(mu, nu) * ldq + q;
#pragma unroll
      for (int e = 0; e < 4; ++e) rb[e] = src[e];
      rd = nu;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) rb[e] = T(0);
      rd = -1.0;
    }
#pragma unroll
    for (int j = 0; j < CP; ++j) {
      const int e = tid + j * NT;
      const int k = e / BI, c = e % BI, nu2 = nu0 + k;
      rc[j] = (e < BK * BI && nu2 < n) ? C[static_cast<std::size_t>(nu2) * ldc + i0 + c] : T(0);
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int e = 0; e < 4; ++e) Bs[buf][bk][bq + e] = rb[e];
    if (with_rho) {
      const double d = rd >= 0.0 ? drow[static_cast<int>(rd)] : 0.0;
#pragma unroll
      for (int e = 0; e < 4; ++e) racc[e] += d * static_cast<double>(rb[e]);
    }
#pragma unroll
    for (int j = 0; j < CP; ++j) {
      const int e = tid + j * NT;
      if (e < BK * BI) Cs[buf][e / BI][e % BI] = rc[j];
    }
  };
  gload(0);
  sstore(0);
  __syncthreads();
  int cur = 0;
  for (int nu0 = 0; nu0 < n; nu0 += BK) {
    const bool more = nu0 + BK < n;
    if (more) gload(nu0 + BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      const int k = kk + (lane >> 4);
      const T a0 = Bs[cur][k][wq * 32 + (lane & 15)];
      const T a1 = Bs[cur][k][wq * 32 + 16 + (lane & 15)];
#pragma unroll
      for (int y = 0; y < NIW; ++y) {
        const T bv = Cs[cur][k][wi * 16 * NIW + y * 16 + (lane & 15)];
        acc[0][y] = mfma(a0, bv, acc[0][y]);
        acc[1][y] = mfma(a1, bv, acc[1][y]);
      }
    }
    if (more) sstore(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }
  if (with_rho) {
    // Reduce the BK row groups of each Q column through LDS (the B tiles are free).
    double* red = reinterpret_cast<double*>(&Bs[0][0][0]);
#pragma unroll
    for (int e = 0; e < 4; ++e) red[bk * BQ + bq + e] = racc[e];
    __syncthreads();
    if (tid < BQ && q0 + tid < ldq) {
      double t = 0.0;
#pragma unroll
      for (int k = 0; k < BK; ++k) t += red[k * BQ + tid];
      rho_part[static_cast<std::size_t>(mu) * ldq + q0 + tid] = t;
    }
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < NIW; ++y) {
      const int i = i0 + wi * 16 * NIW + y * 16 + (lane & 15);
      const int qb = q0 + wq * 32 + x * 16;
      if (i >= r || qb >= ldq) continue;
      T* dst = U + static_cast<std::size_t>(mu) * us + static_cast<std::size_t>(i) * ldq + qb;
#pragma unroll
      for (int v = 0; v < 4; ++v) dst[acc_row<T>(lane, v)] = acc[x][y][v];
    }
}

// BF16X3 U with the B operand taken straight from registers (i tiles of 32 to
// 320 columns).  Lane l of a wave gathers the adjacent Q rows q + 2 (l & 15)
// and q + 2 (l & 15) + 1 (one 8-byte load) at the eight consecutive nu of k
// group l >> 4: the even rows form one A fragment of
// v_mfma_f32_16x16x32_bf16 and the odd rows another, each in exactly the
// operand layout, split into hi/lo in registers; B never passes through LDS.
// Only the C^T tile (i x nu) is staged in LDS, double-buffered, one barrier
// per k-step.  8 waves x 32 Q rows per block (two blocks per CU).  The C^T
// global loads of the next step are issued before its B gathers, so the wait
// that precedes their LDS store never waits for the gathers.
template <int NIW, int TERMS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(NIW <= 3 ? 4 : 2))) void occupied_u_bf16x3_direct_kernel(
    const float* __restrict__ B, const __bf16* __restrict__ Cth, const __bf16* __restrict__ Ctl,
    __bf16* __restrict__ U, std::size_t us, int n, int ldq, int ldct, int r,
    const double* __restrict__ D, double* __restrict__ rho_part) {
  constexpr int NW = 8, NT = 64 * NW, BQ = 32 * NW, BK = 32, BI = 32 * NIW;
  constexpr int XF = 2, YF = BI / 16;
  constexpr int YP = (BI * 4 + NT - 1) / NT;  // 16-byte C^T chunks per thread and plane
  // C^T rows of 64 bytes, chunks swizzled (lds_chunk): the sixteen rows one
  // fragment read touches hit distinct banks.
  __shared__ __bf16 Yh[2][BI][BK], Yl[2][BI][BK];
  // Dynamic LDS: element offsets of the packed rows (mu, nu) for nu < n + BK
  // (rows past n repeat row n - 1, so gathers need no bounds test), then, for
  // the rho pass, D[mu][nu] as float.
  extern __shared__ double dyn[];
  std::size_t* rowoff = reinterpret_cast<std::size_t*>(dyn);
  float* drow = reinterpret_cast<float*>(rowoff + n + BK);
  const int mu = blockIdx.x % n;  // Q-tile-major block order
  const int q0 = (blockIdx.x / n) * BQ;
  const int i0 = blockIdx.y * BI;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kg = lane >> 4;  // k group: nu offset 8 kg within a step
  const int qw = q0 + wave * 32;
  const bool q_ok = qw < ldq;  // wave-uniform: ldq is a multiple of 32
  const int q_off = q_ok ? qw + 2 * (lane & 15) : 0;  // rows q_off (x = 0), q_off + 1 (x = 1)
  const bool with_rho = rho_part != nullptr && blockIdx.y == 0;
  for (int k = tid; k < n + BK; k += NT) rowoff[k] = packed_index(mu, k < n ? k : n - 1) * ldq;
  if (with_rho)
    for (int k = tid; k < n; k += NT) drow[k] = static_cast<float>(D[static_cast<std::size_t>(mu) * n + k]);
  f4 acc[XF][YF];
#pragma unroll
  for (int x = 0; x < XF; ++x)
#pragma unroll
    for (int y = 0; y < YF; ++y) acc[x][y] = f4{};
  double racc[XF] = {0.0, 0.0};
  fl2 rx[8] = {};
  bf8 rch[YP], rcl[YP];
  const float* Bq = B + q_off;
  auto gload = [&](int nu0) {
    const int nb = nu0 + 8 * kg;
#pragma unroll
    for (int j = 0; j < 8; ++j) rx[j] = *reinterpret_cast<const fl2*>(Bq + rowoff[nb + j]);
  };
  auto cload = [&](int nu0) {
#pragma unroll
    for (int jj = 0; jj < YP; ++jj) {
      const int e = tid + jj * NT;
      if (e < BI * 4) {
        const std::size_t off = static_cast<std::size_t>(i0 + (e >> 2)) * ldct + nu0 + (e & 3) * 8;
        rch[jj] = *reinterpret_cast<const bf8*>(Cth + off);
        rcl[jj] = *reinterpret_cast<const bf8*>(Ctl + off);
      }
    }
  };
  auto cstore = [&](int buf) {
#pragma unroll
    for (int jj = 0; jj < YP; ++jj) {
      const int e = tid + jj * NT;
      if (e < BI * 4) {
        const int yc = lds_chunk(e >> 2, e & 3) * 8;
        *reinterpret_cast<bf8*>(&Yh[buf][e >> 2][yc]) = rch[jj];
        *reinterpret_cast<bf8*>(&Yl[buf][e >> 2][yc]) = rcl[jj];
      }
    }
  };
  __syncthreads();  // rowoff and drow
  // Waves past ldq (only in the last Q tile) skip the gathers and MFMAs; they
  // still stage their share of C^T and meet every barrier.
  cload(0);
  if (q_ok) gload(0);
  cstore(0);
  __syncthreads();
  int cur = 0;
  for (int nu0 = 0; nu0 < n; nu0 += BK) {
    // This step's A fragments (waits for its gathers).  Lanes past ldq and
    // nu past n (only in the last step) contribute zeros.
    const int nb = nu0 + 8 * kg;
    float v0[8], v1[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v0[j] = rx[j].x;
      v1[j] = rx[j].y;
    }
    if (!q_ok || nu0 + BK > n) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (!q_ok || nb + j >= n) v0[j] = v1[j] = 0.0f;
    }
    if (with_rho) {
      // rho partials: FP32 over the step's eight nu, FP64 across steps.
      float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = nb + j < n ? drow[nb + j] : 0.0f;
        s0 = fmaf(d, v0[j], s0);
        s1 = fmaf(d, v1[j], s1);
      }
      racc[0] += static_cast<double>(s0);
      racc[1] += static_cast<double>(s1);
    }
    bf8 ah[XF], al[XF];
    split8_bf16(v0, ah[0], al[0]);
    split8_bf16(v1, ah[1], al[1]);
    const bool more = nu0 + BK < n;
    if (more) {
      cload(nu0 + BK);
      if (q_ok) gload(nu0 + BK);
    }
    const int kq = lds_chunk(lane & 15, kg) * 8;  // fragment rows start at multiples of 16
    if (q_ok) {
#pragma unroll
      for (int y = 0; y < YF; ++y) {
        const int row = y * 16 + (lane & 15);
        const bf8 bh = *reinterpret_cast<const bf8*>(&Yh[cur][row][kq]);
        const bf8 bl = *reinterpret_cast<const bf8*>(&Yl[cur][row][kq]);
#pragma unroll
        for (int x = 0; x < XF; ++x) acc[x][y] = mfma(ah[x], bh, acc[x][y]);
        if constexpr (TERMS == 3) {
#pragma unroll
          for (int x = 0; x < XF; ++x) acc[x][y] = mfma(ah[x], bl, acc[x][y]);
#pragma unroll
          for (int x = 0; x < XF; ++x) acc[x][y] = mfma(al[x], bh, acc[x][y]);
        }
      }
    }
    // The other buffer was last read before the previous barrier.
    if (more) cstore(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }
  if (with_rho) {
    // Sum the four k groups (lanes l, l ^ 16, l ^ 32, l ^ 48) of each row.
#pragma unroll
    for (int x = 0; x < XF; ++x) {
      double t = racc[x];
      t += __shfl_xor(t, 16);
      t += __shfl_xor(t, 32);
      if (kg == 0 && q_ok) rho_part[static_cast<std::size_t>(mu) * ldq + q_off + x] = t;
    }
  }
  // Fragment x row m holds Q = qw + 2 m + x; a lane's accumulator element v
  // is row m = 4 (l >> 4) + v of column i = l & 15.
  if (!q_ok) return;
#pragma unroll
  for (int y = 0; y < YF; ++y) {
    const int i = i0 + y * 16 + (lane & 15);
    if (i >= r) continue;
    // Eight consecutive k of this lane: 16 bytes of the hi half and of the lo
    // half of their 128-byte block of 32 k.  At (H2O)64 this costs U 1.5 ms
    // (32.65 -> 34.13; separate planes write 15.2 GB, blocks 16.4) and gains the
    // SYRK 4.5 (20.3 -> 15.8).
    const std::size_t off = 2 * (static_cast<std::size_t>(mu) * us + static_cast<std::size_t>(i) * ldq + qw) + 8 * (lane >> 4);
    bf8 h, l;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      __bf16 h0, l0, h1, l1;
      split_bf16(acc[0][y][v], h0, l0);
      split_bf16(acc[1][y][v], h1, l1);
      h[2 * v] = h0;
      l[2 * v] = l0;
      h[2 * v + 1] = h1;
      l[2 * v + 1] = l1;
    }
    *reinterpret_cast<bf8*>(U + off) = h;
    if constexpr (TERMS == 3) *reinterpret_cast<bf8*>(U + off + 32) = l;
  }
}

// ---------------------------------------------------------------------------
// K, step 2: lower-triangular split-K SYRK over W (n x kd, K-contiguous rows),
// partial results per split.  Bound by the matrix cores, so the tiles are small
// enough that little of their work falls above the diagonal or past n, and a
// wave whose whole part does skips its MFMAs (the other blocks of its CU use
// the cycles).  Block ids are remapped so the blocks resident on one XCD
// (hardware dispatch is round-robin over the 8 XCDs) work on the same k-range
// of W and share that XCD's L2.
// ---------------------------------------------------------------------------

constexpr int kSyrkBfT = 128;  // BF16X3 tile edge

// Lower-triangle tile t -> (row block, column block), RATIO columns of tiles to
// a row of them (the last row may hold fewer).
template <int RATIO>
__device__ __forceinline__ void syrk_tile_of(int t, int& rb, int& cb) {
  rb = 0;
  while (t >= RATIO * (rb + 1)) t -= RATIO * ++rb;
  cb = t;
}

// BF16X3 operands are rows of W as occupied_u writes them: blocks of 32 k, 64
// bytes of hi and 64 bytes of lo, so a k-step reads whole 128-byte lines of its
// rows.  In LDS a row's k-step keeps its PL parts (hi, or hi and lo) in 4 PL
// chunks of 16 bytes; chunk c is stored at position c ^ ((row >> 1) mod 4 PL),
// so the 16 rows of a fragment cover all 64 banks once.
template <int PL>
__device__ __forceinline__ int syrk_chunk(int row, int chunk) {
  return chunk ^ ((row >> 1) & (4 * PL - 1));
}

// 128 x 128 tiles, 4 waves as 2 x 2, each 64 x 64 = 4 x 4 MFMA 16x16x32 tiles:
// 48 MFMAs for 16 fragment reads per k-step of 32.  The next k-step is staged
// in registers while the current one runs (one 32 KB LDS buffer, two
// barriers); three blocks share a CU, so one block's barriers and stores hide
// behind the others' products.  With TERMS == 1 the lo parts are not read.
// CROSS: the column panels come from V instead of W and the tiles cover the
// whole n x n grid (ntiles = ncb^2): partial slices of W V^T, every element
// written.
template <bool CROSS, int TERMS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void exchange_syrk_bf16x3_kernel(
    const __bf16* __restrict__ W, std::size_t kd, int n, int ntiles, int ncb, int nwork, std::size_t kbegin,
    std::size_t kend, std::size_t kchunk, double sign, float* __restrict__ partial, const __bf16* __restrict__ V) {
  constexpr int T = kSyrkBfT, BK = 32, NT = 256, XF = 4, YF = 4, PL = TERMS == 3 ? 2 : 1, NC = 4 * PL;
  __shared__ __bf16 As[T][NC][8], Bs[T][NC][8];
  const int per = gridDim.x / 8;
  const int work = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (work >= nwork) return;
  const int split = work / ntiles, tile = work % ntiles;
  int rb, cb;
  if constexpr (CROSS) {
    rb = tile / ncb;
    cb = tile % ncb;
  } else {
    syrk_tile_of<1>(tile, rb, cb);
  }
  const int m0 = rb * T, l0 = cb * T;
  // A diagonal tile multiplies a panel by itself: one gather, one LDS copy.
  const bool diag = !CROSS && rb == cb;
  const __bf16* __restrict__ C = CROSS ? V : W;  // column-panel operand
  const std::size_t k0 = kbegin + static_cast<std::size_t>(split) * kchunk;
  const std::size_t k1 = k0 + kchunk < kend ? k0 + kchunk : kend;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const bool active = m0 + wr * 64 < n && l0 + wc * 64 < n && (!diag || wr >= wc);
  f4 acc[XF][YF];
#pragma unroll
  for (int i = 0; i < XF; ++i)
#pragma unroll
    for (int j = 0; j < YF; ++j) acc[i][j] = f4{};
  constexpr int CH = T * NC / NT;  // 16-byte chunks per thread and operand
  bf8 ra[CH], rbv[CH];
  auto gload = [&](std::size_t kb) {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int c = tid + j * NT, row = c / NC, kc = (c % NC) * 8;
      const int ga = m0 + row, gb = l0 + row;
      // Rows past n read row n - 1: their products land past n, unwritten.
      ra[j] = *reinterpret_cast<const bf8*>(W + 2 * (static_cast<std::size_t>(ga < n ? ga : n - 1) * kd + kb) + kc);
      if (!diag) rbv[j] = *reinterpret_cast<const bf8*>(C + 2 * (static_cast<std::size_t>(gb < n ? gb : n - 1) * kd + kb) + kc);
    }
  };
  auto sstore = [&]() {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int c = tid + j * NT, row = c / NC, pos = syrk_chunk<PL>(row, c % NC);
      *reinterpret_cast<bf8*>(As[row][pos]) = ra[j];
      if (!diag) *reinterpret_cast<bf8*>(Bs[row][pos]) = rbv[j];
    }
  };
  const __bf16(*Bt)[NC][8] = diag ? As : Bs;
  int at[PL];  // this lane's chunk of each part (fragment rows start at multiples of 16)
#pragma unroll
  for (int p = 0; p < PL; ++p) at[p] = syrk_chunk<PL>(lane & 15, 4 * p + (lane >> 4));
  gload(k0);
  sstore();
  __syncthreads();
  for (std::size_t kb = k0; kb < k1; kb += BK) {
    const bool more = kb + BK < k1;
    if (more) gload(kb + BK);
    if (active) {
      bf8 b[YF][PL];
#pragma unroll
      for (int j = 0; j < YF; ++j)
#pragma unroll
        for (int p = 0; p < PL; ++p) b[j][p] = *reinterpret_cast<const bf8*>(Bt[wc * 64 + j * 16 + (lane & 15)][at[p]]);
#pragma unroll
      for (int i = 0; i < XF; ++i) {
        bf8 a[PL];
#pragma unroll
        for (int p = 0; p < PL; ++p) a[p] = *reinterpret_cast<const bf8*>(As[wr * 64 + i * 16 + (lane & 15)][at[p]]);
        // Independent accumulators between dependent MFMAs keep the pipe full.
#pragma unroll
        for (int j = 0; j < YF; ++j) acc[i][j] = mfma(a[0], b[j][0], acc[i][j]);
        if constexpr (TERMS == 3) {
#pragma unroll
          for (int j = 0; j < YF; ++j) acc[i][j] = mfma(a[0], b[j][PL - 1], acc[i][j]);
#pragma unroll
          for (int j = 0; j < YF; ++j) acc[i][j] = mfma(a[PL - 1], b[j][0], acc[i][j]);
        }
      }
    }
    __syncthreads();
    if (more) {
      sstore();
      __syncthreads();
    }
  }
  // FP32 partials hold the FP32 accumulators exactly (sign is +-1).
  float* out = partial + static_cast<std::size_t>(split) * n * n;
  const float fsign = static_cast<float>(sign);
#pragma unroll
  for (int i = 0; i < XF; ++i)
#pragma unroll
    for (int j = 0; j < YF; ++j) {
      const int lam = l0 + wc * 64 + j * 16 + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int mu = m0 + wr * 64 + i * 16 + 4 * (lane >> 4) + v;
        if (mu < n && lam < n && (CROSS || lam <= mu)) out[static_cast<std::size_t>(mu) * n + lam] = fsign * acc[i][j][v];
      }
    }
}

// Eight fragments of 16 rows, complete on return: four from LDS byte address
// at0 and four from at1, STEP bytes apart.  Reading them in one asm block keeps
// the compiler from waiting for loads into the other LDS buffer (which it
// cannot tell apart) before them.
template <int OFFSET0, int OFFSET1, int STEP>
__device__ __forceinline__ void lds_read8(unsigned at0, unsigned at1, bf8 (&f)[4], bf8 (&g)[4]) {
  asm volatile(
      "ds_read_b128 %0, %8 offset:%10\n\t"
      "ds_read_b128 %1, %8 offset:%10+%12\n\t"
      "ds_read_b128 %2, %8 offset:%10+2*%12\n\t"
      "ds_read_b128 %3, %8 offset:%10+3*%12\n\t"
      "ds_read_b128 %4, %9 offset:%11\n\t"
      "ds_read_b128 %5, %9 offset:%11+%12\n\t"
      "ds_read_b128 %6, %9 offset:%11+2*%12\n\t"
      "ds_read_b128 %7, %9 offset:%11+3*%12\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(g[0]), "=&v"(g[1]), "=&v"(g[2]), "=&v"(g[3])
      : "v"(at0), "v"(at1), "n"(OFFSET0), "n"(OFFSET1), "n"(STEP)
      : "memory");
}

// For large n: 256 x 256 tiles, 8 waves as 2 x 4, each 128 x 64 = 8 x 4 MFMA
// tiles (96 MFMAs for 24 fragment reads per k-step of 32).  Panels go from
// global memory straight into LDS (16 bytes a lane, no staging registers or LDS
// stores), into the buffer the current k-step does not read; one barrier a
// step both ends the reads of one buffer and completes the loads of the other.
// The LDS side of such a load is linear in the lane, so the chunk swizzle is
// applied to the global address instead.  Bound by W's traffic: the tiles of a
// slice drift apart and 84% of their loads miss the XCD's L2, 25.7 GB at n =
// 1152, r ldq = 1.35e6, in 6.22 ms (4.1 TB/s); staged in registers, from
// separate hi and lo planes (64-byte pieces of rows), it took 7.62 ms, staged
// two steps ahead 8.45, and with look-ahead touches into the L2 6.47.
template <bool CROSS, int TERMS>
__global__ __launch_bounds__(512) void exchange_syrk_bf16x3_wide_kernel(
    const __bf16* __restrict__ W, std::size_t kd, int n, int ntiles, int ncb, int nwork, std::size_t kbegin,
    std::size_t kend, std::size_t kchunk, double sign, float* __restrict__ partial, const __bf16* __restrict__ V) {
  constexpr int T = 256, BK = 32, PL = TERMS == 3 ? 2 : 1, NC = 4 * PL, NW = 8, XF = 8, YF = 4;
  constexpr int ROW = 16 * NC, PANEL = T * ROW, FRAG = 16 * ROW;  // bytes: a row, an operand, a fragment's rows
  constexpr int LR = 64 / NC, LOADS = T / (LR * NW);              // rows of a wave's load, loads per wave and operand
  __shared__ __align__(128) unsigned char S[2][2 * PANEL];  // [buffer][operand, row, position]
  const int per = gridDim.x / 8;
  const int work = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (work >= nwork) return;
  const int split = work / ntiles, tile = work % ntiles;
  int rb, cb;
  if constexpr (CROSS) {
    rb = tile / ncb;
    cb = tile % ncb;
  } else {
    syrk_tile_of<1>(tile, rb, cb);
  }
  const int m0 = rb * T, l0 = cb * T;
  const bool diag = !CROSS && rb == cb;  // both operands are the A panel
  const std::size_t k0 = kbegin + static_cast<std::size_t>(split) * kchunk;
  const std::size_t k1 = k0 + kchunk < kend ? k0 + kchunk : kend;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 2, wc = wave & 3;
  const int r0 = m0 + wr * 16 * XF, c0 = l0 + wc * 16 * YF;
  const bool active = r0 < n && c0 < n && (CROSS || c0 < r0 + 16 * XF);
  f4 acc[XF][YF];
#pragma unroll
  for (int i = 0; i < XF; ++i)
#pragma unroll
    for (int j = 0; j < YF; ++j) acc[i][j] = f4{};
  // This lane's source of each load: row lane / NC of the load's rows and the
  // chunk stored at position lane % NC.  Rows past n repeat row n - 1: their
  // products land past n, unwritten.
  const __bf16* src[2][LOADS];
#pragma unroll
  for (int u = 0; u < LOADS; ++u) {
    const int row = (wave + u * NW) * LR + lane / NC, kc = syrk_chunk<PL>(row, lane % NC) * 8;
    src[0][u] = W + 2 * static_cast<std::size_t>(min(m0 + row, n - 1)) * kd + kc;
    src[1][u] = (CROSS ? V : W) + 2 * static_cast<std::size_t>(min(l0 + row, n - 1)) * kd + kc;
  }
  auto issue = [&](int buf, std::size_t kb) {
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      if (o && diag) break;
#pragma unroll
      for (int u = 0; u < LOADS; ++u)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[o][u] + 2 * kb),
                                         (__attribute__((address_space(3))) void*)&S[buf][o * PANEL + (wave + u * NW) * 1024],
                                         16, 0, 0);
    }
  };
  // Byte addresses of this lane's fragments (fragment rows start at multiples of 16).
  const unsigned lds0 = (unsigned)(std::size_t)(__attribute__((address_space(3))) void*)&S[0][0];
  const unsigned b_panel = (diag ? 0 : PANEL) + wc * YF * FRAG, a_panel = wr * XF * FRAG;
  unsigned frag[PL];
#pragma unroll
  for (int p = 0; p < PL; ++p)
    frag[p] = lds0 + static_cast<unsigned>((lane & 15) * ROW + syrk_chunk<PL>(lane & 15, 4 * p + (lane >> 4)) * 16);
  auto products = [&](int i0, const bf8(&a)[PL][4], const bf8(&b)[PL][4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < YF; ++j) acc[i0 + i][j] = mfma(a[0][i], b[0][j], acc[i0 + i][j]);
      if constexpr (TERMS == 3) {
#pragma unroll
        for (int j = 0; j < YF; ++j) acc[i0 + i][j] = mfma(a[0][i], b[PL - 1][j], acc[i0 + i][j]);
#pragma unroll
        for (int j = 0; j < YF; ++j) acc[i0 + i][j] = mfma(a[PL - 1][i], b[0][j], acc[i0 + i][j]);
      }
    }
  };
  auto compute = [&](int buf) {
    if (!active) return;
    const unsigned shift = buf * 2 * PANEL;
    bf8 a[PL][4], b[PL][4];
    lds_read8<0, 0, FRAG>(frag[0] + a_panel + shift, frag[0] + b_panel + shift, a[0], b[0]);
    if constexpr (PL == 2) lds_read8<0, 0, FRAG>(frag[PL - 1] + a_panel + shift, frag[PL - 1] + b_panel + shift, a[PL - 1], b[PL - 1]);
    products(0, a, b);
    if constexpr (PL == 2) {
      lds_read8<4 * FRAG, 4 * FRAG, FRAG>(frag[0] + a_panel + shift, frag[PL - 1] + a_panel + shift, a[0], a[PL - 1]);
    } else {
      lds_read8<4 * FRAG, 0, FRAG>(frag[0] + a_panel + shift, frag[0] + b_panel + shift, a[0], b[0]);
    }
    products(4, a, b);
  };
  constexpr int kVmcnt0 = 0x0f70;  // s_waitcnt vmcnt(0): this wave's loads into LDS are complete
  issue(0, k0);
  for (std::size_t kb = k0; kb < k1; kb += 2 * BK) {
    __builtin_amdgcn_s_waitcnt(kVmcnt0);
    __syncthreads();
    if (kb + BK < k1) issue(1, kb + BK);
    compute(0);
    if (kb + BK >= k1) break;
    __builtin_amdgcn_s_waitcnt(kVmcnt0);
    __syncthreads();
    if (kb + 2 * BK < k1) issue(0, kb + 2 * BK);
    compute(1);
  }
  float* out = partial + static_cast<std::size_t>(split) * n * n;
  const float fsign = static_cast<float>(sign);
#pragma unroll
  for (int i = 0; i < XF; ++i)
#pragma unroll
    for (int j = 0; j < YF; ++j) {
      const int lam = c0 + j * 16 + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int mu = r0 + i * 16 + 4 * (lane >> 4) + v;
        if (mu < n && lam < n && (CROSS || lam <= mu)) out[static_cast<std::size_t>(mu) * n + lam] = fsign * acc[i][j][v];
      }
    }
}

// FP64 / FP32 SYRK: WR x WC waves, each F x F MFMA 16x16x4 tiles.  LDS rows keep
// W's K-contiguous order with one element of padding, so the 16 rows a wave
// reads at one k fall on distinct banks; the next k-step is staged in registers
// and stored into the other LDS buffer (one barrier per step).
template <class T, int WR, int WC, int F>
__global__ __launch_bounds__(64 * WR * WC) void exchange_syrk_kernel(const T* __restrict__ W, std::size_t kd, int n,
                                                                     int ntiles, int nwork, std::size_t kbegin,
                                                                     std::size_t kend, std::size_t kchunk, double sign,
                                                                     T* __restrict__ partial) {
  using Acc = typename AccOf<T>::type;
  using V16 = typename Vec16<T>::type;
  constexpr int WE = 16 * F, TM = WR * WE, TN = WC * WE, BK = 16, PAD = 1, NT = 64 * WR * WC, V = 16 / sizeof(T);
  static_assert(TM % TN == 0, "whole tile columns to a tile row");
  __shared__ T As[2][TM][BK + PAD];
  __shared__ T Bs[2][TN][BK + PAD];
  const int per = gridDim.x / 8;
  const int work = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (work >= nwork) return;
  const int split = work / ntiles, tile = work % ntiles;
  int rb, cb;
  syrk_tile_of<TM / TN>(tile, rb, cb);
  const int m0 = rb * TM, l0 = cb * TN;
  const std::size_t k0 = kbegin + static_cast<std::size_t>(split) * kchunk;
  const std::size_t k1 = k0 + kchunk < kend ? k0 + kchunk : kend;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave / WC, wc = wave % WC;
  const int r0 = m0 + wr * WE, c0 = l0 + wc * WE;
  const bool active = r0 < n && c0 < n && c0 < r0 + WE;
  Acc acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = Acc{};
  constexpr int CH = BK / V;                          // 16-byte chunks per row
  constexpr int AC = TM * CH / NT, BC = TN * CH / NT;  // chunks per thread
  V16 ra[AC], rbv[BC];
  auto gload = [&](std::size_t kb) {
    // Rows past n read row n - 1: their products land past n, unwritten.
#pragma unroll
    for (int j = 0; j < AC; ++j) {
      const int c = tid + j * NT, row = min(m0 + c / CH, n - 1), kc = (c % CH) * V;
      ra[j] = *reinterpret_cast<const V16*>(W + static_cast<std::size_t>(row) * kd + kb + kc);
    }
#pragma unroll
    for (int j = 0; j < BC; ++j) {
      const int c = tid + j * NT, row = min(l0 + c / CH, n - 1), kc = (c % CH) * V;
      rbv[j] = *reinterpret_cast<const V16*>(W + static_cast<std::size_t>(row) * kd + kb + kc);
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int j = 0; j < AC; ++j) {
      const int c = tid + j * NT;
#pragma unroll
      for (int e = 0; e < V; ++e) As[buf][c / CH][(c % CH) * V + e] = ra[j][e];
    }
#pragma unroll
    for (int j = 0; j < BC; ++j) {
      const int c = tid + j * NT;
#pragma unroll
      for (int e = 0; e < V; ++e) Bs[buf][c / CH][(c % CH) * V + e] = rbv[j][e];
    }
  };
  gload(k0);
  sstore(0);
  __syncthreads();
  int cur = 0;
  for (std::size_t kb = k0; kb < k1; kb += BK) {
    const bool more = kb + BK < k1;
    if (more) gload(kb + BK);
    if (active) {
#pragma unroll
      for (int kk = 0; kk < BK; kk += 4) {
        const int k = kk + (lane >> 4);
        T b[F];
#pragma unroll
        for (int j = 0; j < F; ++j) b[j] = Bs[cur][wc * WE + j * 16 + (lane & 15)][k];
#pragma unroll
        for (int i = 0; i < F; ++i) {
          const T a = As[cur][wr * WE + i * 16 + (lane & 15)][k];
#pragma unroll
          for (int j = 0; j < F; ++j) acc[i][j] = mfma(a, b[j], acc[i][j]);
        }
      }
    }
    if (more) sstore(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }
  // Triangle elements in place (row-major, lambda <= mu) of the split's n x n slice.
  T* out = partial + static_cast<std::size_t>(split) * n * n;
  const T tsign = static_cast<T>(sign);
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const int lam = c0 + j * 16 + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int mu = r0 + i * 16 + acc_row<T>(lane, v);
        if (mu < n && lam < n && lam <= mu) out[static_cast<std::size_t>(mu) * n + lam] = tsign * acc[i][j][v];
      }
    }
}

// Sum of one element over the slices, in slice order; 32 loads in flight (107
// slices at n = 96: 4.6 us, 26.7 with one at a time).
template <class P>
__device__ __forceinline__ double slice_sum(const P* __restrict__ p, int slices, std::size_t stride) {
  constexpr int U = 32;
  double s = 0.0;
  int k = 0;
  for (; k + U <= slices; k += U) {
    P v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = p[static_cast<std::size_t>(k + u) * stride];
#pragma unroll
    for (int u = 0; u < U; ++u) s += static_cast<double>(v[u]);
  }
#pragma unroll 8
  for (; k < slices; ++k) s += static_cast<double>(p[static_cast<std::size_t>(k) * stride]);
  return s;
}
constexpr int kReduceThreads = 64;  // one wave a block: small n spreads over the CUs

// K = sum of the split partials (FP64 sum in slice order), mirrored.
template <class P>
__global__ void reduce_exchange_kernel(const P* __restrict__ partial, int slices, int n, double* __restrict__ K) {
  const std::size_t e = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= static_cast<std::size_t>(n) * n) return;
  const int mu = static_cast<int>(e / n), lam = static_cast<int>(e % n);
  if (lam > mu) return;
  const double s = slice_sum(partial + e, slices, static_cast<std::size_t>(n) * n);
  K[static_cast<std::size_t>(mu) * n + lam] = s;
  K[static_cast<std::size_t>(lam) * n + mu] = s;
}

// K = Kref + W + W^T with W the sum of the cross partial slices (FP64 sum in
// slice order); K is symmetric by construction.
__global__ void reduce_cross_kernel(const float* __restrict__ partial, int slices, int n,
                                    const double* __restrict__ Kref, double* __restrict__ K) {
  const std::size_t e = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= static_cast<std::size_t>(n) * n) return;
  const int mu = static_cast<int>(e / n), lam = static_cast<int>(e % n);
  if (lam > mu) return;
  const std::size_t et = static_cast<std::size_t>(lam) * n + mu;
  const std::size_t nn = static_cast<std::size_t>(n) * n;
  const double s = slice_sum(partial + e, slices, nn), t = slice_sum(partial + et, slices, nn);
  const double v = Kref[e] + (s + t);
  K[e] = v;
  K[et] = v;
}

__global__ void convert_kernel(const double* __restrict__ in, float* __restrict__ out, std::size_t count) {
  const std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const std::size_t stride = static_cast<std::size_t>(gridDim.x) * blockDim.x;
  for (std::size_t k = i; k < count; k += stride) out[k] = static_cast<float>(in[k]);
}

// C (n x ldc, FP64) -> C^T split: hi/lo bf16, ldc rows x ldct columns (zero beyond n).
__global__ void split_transpose_kernel(const double* __restrict__ C, int n, int ldc, int ldct,
                                       __bf16* __restrict__ hi, __bf16* __restrict__ lo) {
  const std::size_t e = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= static_cast<std::size_t>(ldc) * ldct) return;
  const int i = static_cast<int>(e / ldct), nu = static_cast<int>(e % ldct);
  const float x = nu < n ? static_cast<float>(C[static_cast<std::size_t>(nu) * ldc + i]) : 0.0f;
  __bf16 h, l;
  split_bf16(x, h, l);
  hi[e] = h;
  lo[e] = l;
}

template <int NIW>
void launch_u(Precision prec, const void* B, const OccupiedOperands& ops, int ldq, void* U, const double* D,
              double* rho_part, hipStream_t s) {
  const std::size_t dyn = rho_part ? static_cast<std::size_t>(ops.n) * sizeof(double) : 0;
  if (dyn > 32 * 1024) throw NotImplemented("fused rho supports nbf <= 4096");
  if (prec == Precision::FP64) {
    constexpr int WQ = 4;
    const int nqb = (ldq + 32 * WQ - 1) / (32 * WQ);
    dim3 grid(static_cast<unsigned>(ops.n) * nqb, ops.ldc / (32 * NIW));
    hipLaunchKernelGGL((occupied_u_kernel<double, NIW, WQ>), grid, dim3(128 * WQ), dyn, s,
                       static_cast<const double*>(B), ops.c64, static_cast<double*>(U), ops.ustride, ops.n, ldq,
                       ops.ldc, ops.r, nqb, D, rho_part);
  } else if (prec == Precision::FP32) {
    constexpr int WQ = 8;
    const int nqb = (ldq + 32 * WQ - 1) / (32 * WQ);
    dim3 grid(static_cast<unsigned>(ops.n) * nqb, ops.ldc / (32 * NIW));
    hipLaunchKernelGGL((occupied_u_kernel<float, NIW, WQ>), grid, dim3(128 * WQ), dyn, s, static_cast<const float*>(B),
                       ops.c32, static_cast<float*>(U), ops.ustride, ops.n, ldq, ops.ldc, ops.r, nqb, D, rho_part);
  } else {
    const int nqb = (ldq + 255) / 256;
    dim3 grid(static_cast<unsigned>(ops.n) * nqb, ops.ldc / (32 * NIW));
    // Row-offset table (n + 32 entries) and the rho row as float.
    const std::size_t ddyn = static_cast<std::size_t>(ops.n + 32) * sizeof(std::size_t) +
                             (rho_part ? static_cast<std::size_t>(ops.n) * sizeof(float) : 0);
    auto kernel = ops.terms == 1 ? occupied_u_bf16x3_direct_kernel<NIW, 1> : occupied_u_bf16x3_direct_kernel<NIW, 3>;
    hipLaunchKernelGGL(kernel, grid, dim3(512), ddyn, s, static_cast<const float*>(B),
                       static_cast<const __bf16*>(ops.ct_hi), static_cast<const __bf16*>(ops.ct_lo),
                       static_cast<__bf16*>(U), ops.ustride, ops.n, ldq, ops.ldct, ops.r, D, rho_part);
  }
  VQC_LAUNCH("occupied_u_kernel");
}


}  // namespace

int occupied_tile(int r) {
  // i-tiles of 16 per wave, two waves along i: one block covers 32 * NIW
  // columns, all of r up to 320.
  return std::max(1, std::min(10, (r + 31) / 32));
}

void pack_density(const double* D, int n, double* dpacked, hipStream_t s) {
  const std::size_t np = pair_count(n);
  hipLaunchKernelGGL(pack_density_kernel, dim3((np + 255) / 256), dim3(256), 0, s, D, n, dpacked);
  VQC_LAUNCH("pack_density_kernel");
}

namespace {
int rho_vector(Precision prec) { return prec == Precision::FP64 ? 2 : 4; }
int rho_chunks(std::size_t npair, int ldq, Precision prec) {
  const int cols = (ldq + kRhoThreads * rho_vector(prec) - 1) / (kRhoThreads * rho_vector(prec));
  const int want = std::max(1, 2048 / cols);
  return static_cast<int>(std::min<std::size_t>(want, std::max<std::size_t>(1, npair / 64)));
}
}  // namespace

std::size_t coulomb_partial_size(std::size_t npair, int ldq) {
  return static_cast<std::size_t>(std::max(rho_chunks(npair, ldq, Precision::FP64),
                                           rho_chunks(npair, ldq, Precision::FP32))) *
         ldq;
}

void coulomb_rho(Precision prec, const void* B, const double* dpacked, std::size_t npair, int ldq, double* rho,
                 double* partial, hipStream_t s) {
  const int v = rho_vector(prec);
  const int chunks = rho_chunks(npair, ldq, prec);
  const std::size_t chunk = (npair + chunks - 1) / chunks;
  dim3 grid((ldq + kRhoThreads * v - 1) / (kRhoThreads * v), chunks);
  if (prec == Precision::FP64)
    hipLaunchKernelGGL((coulomb_rho_kernel<double, 2>), grid, dim3(kRhoThreads), 0, s,
                       static_cast<const double*>(B), dpacked, npair, ldq, chunk, partial);
  else
    hipLaunchKernelGGL((coulomb_rho_kernel<float, 4>), grid, dim3(kRhoThreads), 0, s,
                       static_cast<const float*>(B), dpacked, npair, ldq, chunk, partial);
  VQC_LAUNCH("coulomb_rho_kernel");
  hipLaunchKernelGGL(sum_rows_kernel, dim3((ldq + kSumCols - 1) / kSumCols), dim3(kSumCols * kSumGroups), 0, s, partial,
                     chunks, ldq, rho);
  VQC_LAUNCH("sum_rows_kernel");
}

void rho_from_partials(const double* rho_part, int rows, int ldq, double* rho, hipStream_t s) {
  hipLaunchKernelGGL(sum_rows_kernel, dim3((ldq + kSumCols - 1) / kSumCols), dim3(kSumCols * kSumGroups), 0, s,
                     rho_part, rows, ldq, rho);
  VQC_LAUNCH("sum_rows_kernel");
}

void coulomb_matrix(Precision prec, const void* B, const double* rho, std::size_t npair, int ldq, int n, double* J,
                    hipStream_t s) {
  const std::size_t lds = static_cast<std::size_t>(ldq) * sizeof(double);
  if (lds > 160 * 1024) throw NotImplemented("auxiliary dimension exceeds the LDS-resident rho limit");
  // Up to two resident blocks per CU on 256 CUs (one when rho exceeds 80 KB);
  // waves stride over the packed rows.
  const std::size_t rows_per_block = kJThreads / 64;
  const unsigned blocks = static_cast<unsigned>(std::min<std::size_t>((npair + rows_per_block - 1) / rows_per_block, 512));
  if (prec == Precision::FP64)
    hipLaunchKernelGGL(coulomb_matrix_kernel<double>, dim3(blocks), dim3(kJThreads), lds, s,
                       static_cast<const double*>(B), rho, npair, ldq, n, J);
  else
    hipLaunchKernelGGL(coulomb_matrix_kernel<float>, dim3(blocks), dim3(kJThreads), lds, s,
                       static_cast<const float*>(B), rho, npair, ldq, n, J);
  VQC_LAUNCH("coulomb_matrix_kernel");
}

void prepare_occupied(Precision prec, OccupiedOperands& ops, hipStream_t s) {
  const std::size_t count = static_cast<std::size_t>(ops.n) * ops.ldc;
  if (prec == Precision::FP32) {
    hipLaunchKernelGGL(convert_kernel, dim3(std::min<std::size_t>((count + 255) / 256, 4096)), dim3(256), 0, s,
                       ops.c64, ops.c32, count);
    VQC_LAUNCH("convert_kernel");
  } else if (prec == Precision::BF16X3) {
    const std::size_t e = static_cast<std::size_t>(ops.ldc) * ops.ldct;
    hipLaunchKernelGGL(split_transpose_kernel, dim3((e + 255) / 256), dim3(256), 0, s, ops.c64, ops.n, ops.ldc,
                       ops.ldct, static_cast<__bf16*>(ops.ct_hi), static_cast<__bf16*>(ops.ct_lo));
    VQC_LAUNCH("split_transpose_kernel");
  }
}

void occupied_u(Precision prec, const void* B, const OccupiedOperands& ops, int ldq, void* U, const double* D,
                double* rho_part, hipStream_t s) {
  switch (ops.ni) {
    case 1: launch_u<1>(prec, B, ops, ldq, U, D, rho_part, s); break;
    case 2: launch_u<2>(prec, B, ops, ldq, U, D, rho_part, s); break;
    case 3: launch_u<3>(prec, B, ops, ldq, U, D, rho_part, s); break;
    case 4: launch_u<4>(prec, B, ops, ldq, U, D, rho_part, s); break;
    case 5: launch_u<5>(prec, B, ops, ldq, U, D, rho_part, s); break;
    case 6: launch_u<6>(prec, B, ops, ldq, U, D, rho_part, s); break;
    case 7: launch_u<7>(prec, B, ops, ldq, U, D, rho_part, s); break;
    case 8: launch_u<8>(prec, B, ops, ldq, U, D, rho_part, s); break;
    case 9: launch_u<9>(prec, B, ops, ldq, U, D, rho_part, s); break;
    case 10: launch_u<10>(prec, B, ops, ldq, U, D, rho_part, s); break;
    default: throw std::logic_error("occupied tile width out of range");
  }
}

namespace {
// Split-K slices per launch: at most 256 MB of FP64 partial slices (and 128).
int syrk_split_cap(int n) {
  const std::size_t slice = static_cast<std::size_t>(n) * n * sizeof(double);
  return static_cast<int>(std::max<std::size_t>(1, std::min<std::size_t>(128, (256ull << 20) / slice)));
}
// Lower-triangle tiles of tm x tn (tm a multiple of tn) over n rows.
int syrk_tiles(int n, int tm, int tn) {
  const int ncb = (n + tn - 1) / tn, nrb = (n + tm - 1) / tm;
  int t = 0;
  for (int rb = 0; rb < nrb; ++rb) t += std::min((tm / tn) * (rb + 1), ncb);
  return t;
}
// Equal-size work items fill the GPU in whole waves of `slots` resident
// blocks: take the fewest splits whose tiles x splits fill at least 95% of the
// last wave, else the best fill under the cap.
int syrk_splits(int tiles, int cap, int slots) {
  const int kSlots = slots;
  int best = 1;
  double best_fill = 0.0;
  for (int sp = 1; sp <= cap; ++sp) {
    const int w = tiles * sp;
    const double fill = static_cast<double>(w) / (static_cast<double>((w + kSlots - 1) / kSlots) * kSlots);
    if (w >= kSlots && fill >= 0.95) return sp;
    if (fill > best_fill + 1e-12) {
      best = sp;
      best_fill = fill;
    }
  }
  return best;
}
}  // namespace

std::size_t exchange_partial_size(int n) {
  return static_cast<std::size_t>(syrk_split_cap(n) + 1) * 2 * static_cast<std::size_t>(n) * n;
}

std::size_t u_row_stride(Precision prec, int r, int ldq) {
  const std::size_t dense = static_cast<std::size_t>(r) * ldq;
  if (prec == Precision::FP64) return dense;
  return dense + 32;
}

namespace {
// Slices per run: both runs (positive and negative columns) together must
// fit the partial buffer (n^2 doubles per FP64 slice; FP32 slices use half).
int syrk_cap(int n, std::size_t partial_capacity) {
  const std::size_t slice = static_cast<std::size_t>(n) * n;
  return partial_capacity == 0
             ? syrk_split_cap(n)
             : static_cast<int>(std::min<std::size_t>(syrk_split_cap(n), partial_capacity / (2 * slice)));
}
// BF16X3 tile edge.  Small n is padding-bound: at n = 384 the 128-wide tiles
// take 104 us where 256-wide ones took 187 (38% of a 256-wide triangle is K's).
// Large n is bound by W's traffic, of which wider tiles need less: n = 490
// 192 us at 128, 169 at 256; n = 1152 7.74 and 6.22 ms.
constexpr int kWideN = 400;
int bf16_edge(int n) { return n <= kWideN ? kSyrkBfT : 256; }
// FP64 / FP32 tiles: 64 x 64, or 256 x 128, which read W's panels a third as
// often but cover more than K's triangle.  A multiplied element costs the wide
// tiles 1 / 1.3 of what it costs the narrow ones (FP32 from n = 900: 1 / 1.5 to
// 1 / 1.7), so they are taken where their covered area is below that.  ms,
// narrow and wide, (H2O)n with all its occupied columns: FP64 n = 576 2.42 and
// 3.90, 768 8.11 and 7.66, 1152 41.7 and 41.9, 1344 76.2 and 80.3, 1536 130 and
// 105; FP32 576 1.32 and 1.71, 768 4.21 and 3.85, 1152 26.0 and 22.0, 1344 49.0
// and 41.3, 1536 84.6 and 54.3.
bool wide_syrk(Precision prec, int n) {
  const double gain = prec == Precision::FP32 && n >= 900 ? 1.5 : 1.3;
  return n > kWideN && 256.0 * 128.0 * syrk_tiles(n, 256, 128) <= gain * 64.0 * 64.0 * syrk_tiles(n, 64, 64);
}
int syrk_tile_count(Precision prec, int n) {
  if (prec == Precision::BF16X3) return syrk_tiles(n, bf16_edge(n), bf16_edge(n));
  return wide_syrk(prec, n) ? syrk_tiles(n, 256, 128) : syrk_tiles(n, 64, 64);
}
// Split-K slices per run.  Up to kWideN the slices stay those of 256-wide
// tiles on 256 single-block CUs: there are enough of them for any tile, and K
// (each slice's sums do not depend on the tile) keeps its rounding.  Beyond,
// they fill whole waves of the blocks that are resident: one per CU for the
// wide BF16X3 and FP64 tiles, two for the wide FP32 ones, four for the narrow
// FP64 ones (35 KB of LDS) and eight for FP32.
int syrk_rule(Precision prec, int n, int cap, bool cross) {
  if (n <= kWideN) {
    const int wide = prec == Precision::BF16X3 ? syrk_tiles(n, 256, 256) : syrk_tiles(n, 256, 128);
    const int edge = (n + 255) / 256;
    return syrk_splits(cross ? edge * edge : wide, cap, prec == Precision::FP32 ? 512 : 256);
  }
  const int resident = prec == Precision::FP32 ? 2 : 1;
  const int slots = prec == Precision::BF16X3 ? 256 : 256 * resident * (wide_syrk(prec, n) ? 1 : 4);
  const int blocks = (n + bf16_edge(n) - 1) / bf16_edge(n);
  return syrk_splits(cross ? blocks * blocks : syrk_tile_count(prec, n), cap, slots);
}
}  // namespace

int exchange_max_splits(int n, std::size_t partial_capacity) { return std::max(1, syrk_cap(n, partial_capacity)); }

int exchange_default_splits(Precision prec, int n, std::size_t partial_capacity) {
  const int cap = syrk_cap(n, partial_capacity);
  if (cap < 1) throw std::length_error("exchange partial buffer holds no slice");
  return syrk_rule(prec, n, cap, false);
}

namespace {
template <class T, class... Args>
void launch_syrk(unsigned grid, hipStream_t s, const T* w, std::size_t kd, int n, Args... args) {
  const bool wide = wide_syrk(sizeof(T) == 8 ? Precision::FP64 : Precision::FP32, n);
  auto kernel = wide ? exchange_syrk_kernel<T, 4, 2, 4> : exchange_syrk_kernel<T, 2, 2, 2>;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(wide ? 512 : 256), 0, s, w, kd, n, args...);
}
template <bool CROSS, class... Args>
void launch_syrk_bf16x3(int terms, unsigned grid, hipStream_t s, const __bf16* w, std::size_t kd, int n,
                        Args... args) {
  const int edge = bf16_edge(n);
  auto kernel = edge == kSyrkBfT ? (terms == 1 ? exchange_syrk_bf16x3_kernel<CROSS, 1> : exchange_syrk_bf16x3_kernel<CROSS, 3>)
                                 : (terms == 1 ? exchange_syrk_bf16x3_wide_kernel<CROSS, 1> : exchange_syrk_bf16x3_wide_kernel<CROSS, 3>);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(edge == kSyrkBfT ? 256 : 512), 0, s, w, kd, n, args...);
}
}  // namespace

void exchange_syrk(Precision prec, const void* U, std::size_t ustride, int n, int r, int r_pos, int ldq, double* K,
                   double* partial, hipStream_t s, std::size_t partial_capacity, int split_override, int terms) {
  const std::size_t kd = static_cast<std::size_t>(r) * ldq;
  if (ustride < kd) throw std::invalid_argument("U row stride shorter than r x ldq");
  const int cap = syrk_cap(n, partial_capacity);
  if (cap < 1) throw std::length_error("exchange partial buffer holds no slice");
  int slices = 0;
  auto run = [&](std::size_t kb, std::size_t ke, double sign) {
    if (ke <= kb) return;
    const std::size_t len = ke - kb;
    // FP64 partials for the FP64 build, FP32 (the accumulators' type) otherwise.
    const std::size_t at = static_cast<std::size_t>(slices) * n * n;
    double* out64 = partial + at;
    float* out32 = reinterpret_cast<float*>(partial) + at;
    const int tiles = syrk_tile_count(prec, n);
    const std::size_t bk = prec == Precision::BF16X3 ? 32 : 16;
    int splits = split_override > 0 ? std::min(split_override, cap) : syrk_rule(prec, n, cap, false);
    const std::size_t chunk = round_up((len + splits - 1) / splits, bk);
    splits = static_cast<int>((len + chunk - 1) / chunk);
    const int nwork = tiles * splits;
    const unsigned grid = static_cast<unsigned>(round_up(nwork, 8));
    if (prec == Precision::BF16X3) {
      const __bf16* w = static_cast<const __bf16*>(U);
      launch_syrk_bf16x3<false>(terms, grid, s, w, ustride, n, tiles, 0, nwork, kb, ke, chunk, sign, out32, w);
    } else if (prec == Precision::FP64) {
      launch_syrk(grid, s, static_cast<const double*>(U), ustride, n, tiles, nwork, kb, ke, chunk, sign, out64);
    } else {
      launch_syrk(grid, s, static_cast<const float*>(U), ustride, n, tiles, nwork, kb, ke, chunk, sign, out32);
    }
    VQC_LAUNCH("exchange_syrk_kernel");
    slices += splits;
  };
  run(0, static_cast<std::size_t>(r_pos) * ldq, 1.0);
  run(static_cast<std::size_t>(r_pos) * ldq, kd, -1.0);
  if (slices == 0) {
    VQC_HIP(hipMemsetAsync(K, 0, static_cast<std::size_t>(n) * n * sizeof(double), s));
    return;
  }
  const std::size_t e = static_cast<std::size_t>(n) * n;
  if (prec == Precision::FP64)
    hipLaunchKernelGGL(reduce_exchange_kernel<double>, dim3((e + kReduceThreads - 1) / kReduceThreads), dim3(kReduceThreads), 0, s, partial, slices, n, K);
  else
    hipLaunchKernelGGL(reduce_exchange_kernel<float>, dim3((e + kReduceThreads - 1) / kReduceThreads), dim3(kReduceThreads), 0, s,
                       reinterpret_cast<const float*>(partial), slices, n, K);
  VQC_LAUNCH("reduce_exchange_kernel");
}

void exchange_cross_bf16x3(const void* X, const void* Y, std::size_t ustride, int n, int r, int ldq,
                           const double* Kref, double* K, double* partial, hipStream_t s) {
  const std::size_t kd = static_cast<std::size_t>(r) * ldq;
  if (ustride < kd) throw std::invalid_argument("U row stride shorter than r x ldq");
  const int cap = syrk_cap(n, 0);
  const int edge = bf16_edge(n), ncb = (n + edge - 1) / edge;
  const int tiles = ncb * ncb;
  int splits = syrk_rule(Precision::BF16X3, n, cap, true);
  const std::size_t chunk = round_up((kd + splits - 1) / splits, 32);
  splits = static_cast<int>((kd + chunk - 1) / chunk);
  if (splits > 2 * cap) throw std::length_error("cross partial slices exceed the partial buffer");
  const int nwork = tiles * splits;
  const unsigned grid = static_cast<unsigned>(round_up(nwork, 8));
  float* out32 = reinterpret_cast<float*>(partial);
  launch_syrk_bf16x3<true>(3, grid, s, static_cast<const __bf16*>(X), ustride, n, tiles, ncb, nwork, std::size_t{0}, kd, chunk,
                           1.0, out32, static_cast<const __bf16*>(Y));
  VQC_LAUNCH("exchange_syrk_bf16x3_kernel (cross)");
  const std::size_t e = static_cast<std::size_t>(n) * n;
  hipLaunchKernelGGL(reduce_cross_kernel, dim3((e + kReduceThreads - 1) / kReduceThreads), dim3(kReduceThreads), 0, s, out32, splits, n, Kref, K);
  VQC_LAUNCH("reduce_cross_kernel");
}

namespace {
__global__ void occupied_factor_kernel(const double* __restrict__ C, int n, int nocc, int ldc,
                                       double* __restrict__ factor) {
  const std::size_t e = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= static_cast<std::size_t>(n) * ldc) return;
  const int nu = static_cast<int>(e / ldc), i = static_cast<int>(e % ldc);
  factor[e] = i < nocc ? 1.4142135623730951 * C[static_cast<std::size_t>(nu) * nocc + i] : 0.0;
}

// out = J then K, zeros for a null one.
__global__ void gather_results_kernel(const double* __restrict__ J, const double* __restrict__ K, std::size_t nn,
                                      double* __restrict__ out) {
  const std::size_t e = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= nn) return;
  out[e] = J ? J[e] : 0.0;
  out[nn + e] = K ? K[e] : 0.0;
}

// D[mu][nu] = sum_i F[mu][i] F[nu][i], one element per thread (fixed order).
__global__ void factor_product_kernel(const double* __restrict__ F, int n, int nocc, int ldc, double* __restrict__ D) {
  const std::size_t e = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= static_cast<std::size_t>(n) * n) return;
  const int mu = static_cast<int>(e / n), nu = static_cast<int>(e % n);
  const double* a = F + static_cast<std::size_t>(mu) * ldc;
  const double* b = F + static_cast<std::size_t>(nu) * ldc;
  double s = 0.0;
  for (int i = 0; i < nocc; ++i) s += a[i] * b[i];
  D[e] = s;
}
}  // namespace

void occupied_factor(const double* C, int n, int nocc, int ldc, double* factor, hipStream_t s) {
  const std::size_t ef = static_cast<std::size_t>(n) * ldc;
  hipLaunchKernelGGL(occupied_factor_kernel, dim3((ef + 255) / 256), dim3(256), 0, s, C, n, nocc, ldc, factor);
  VQC_LAUNCH("occupied_factor_kernel");
}

void gather_results(const double* J, const double* K, std::size_t nn, double* out, hipStream_t s) {
  hipLaunchKernelGGL(gather_results_kernel, dim3((nn + 255) / 256), dim3(256), 0, s, J, K, nn, out);
  VQC_LAUNCH("gather_results_kernel");
}

void occupied_factor_and_density(const double* C, int n, int nocc, int ldc, double* factor, double* D,
                                 hipStream_t s) {
  occupied_factor(C, n, nocc, ldc, factor, s);
  const std::size_t ed = static_cast<std::size_t>(n) * n;
  hipLaunchKernelGGL(factor_product_kernel, dim3((ed + 255) / 256), dim3(256), 0, s, factor, n, nocc, ldc, D);
  VQC_LAUNCH("factor_product_kernel");
}

void convert_f64_to_f32(const double* in, float* out, std::size_t count, hipStream_t s) {
  hipLaunchKernelGGL(convert_kernel, dim3(std::min<std::size_t>((count + 255) / 256, 65536)), dim3(256), 0, s, in,
                     out, count);
  VQC_LAUNCH("convert_kernel");
}

}  // namespace vqc
