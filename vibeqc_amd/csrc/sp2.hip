// One-launch SP2 purification (see scf.hpp): Gershgorin interval, first
// iterate, every step and the convergence test in one kernel, so a
// purification costs one launch instead of a DGEMM and an elementwise kernel
// per step with host polls between them.
//
// X stays symmetric, so a step is X X^T over the lower-triangle 16 x 16 tiles
// on v_mfma_f64_16x16x4 (one wave per tile), each written with its mirror.
// tr X^2 = |X|_F^2 is summed while X is written, so a step's choice (X^2 or
// 2 X - X^2) and its freeze test are known before its product starts and one
// barrier per step is enough.  MFMA sums over k in any order, so lane group g
// takes the four consecutive k = 16 b + 4 g + s of block b for step s: every
// operand load is 32 consecutive bytes of a row.  Bound by latency (operand
// loads and barriers), not by the matrix cores, at the sizes it serves.
// A purification of n = 96 takes 0.18 ms instead of 0.5 ms of kernels and as
// much again of gaps between the stepwise calls.
#include "scf.hpp"

#include <cstdlib>

namespace vqc {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ d4 mfma64(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ d4 load4(const double* p) {
  const d2 x = *reinterpret_cast<const d2*>(p), y = *reinterpret_cast<const d2*>(p + 2);
  return d4{x[0], x[1], y[0], y[1]};
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Lower-triangle tile t -> (row block, column block).
__device__ __forceinline__ void tile_of(int t, int& i, int& j) {
  i = static_cast<int>((sqrtf(8.0f * static_cast<float>(t) + 1.0f) - 1.0f) * 0.5f);
  while (i * (i + 1) / 2 > t) --i;
  while ((i + 1) * (i + 2) / 2 <= t) ++i;
  j = t - i * (i + 1) / 2;
}

// The choices of one step from tr X, tr X^2 and the error history (the rule
// of sp2_step_kernel).
struct StepRule {
  double trace, err1 = 0.0, err2 = 0.0;  // tr X; idempotency errors one and two steps back
  int k = 0;
  bool square = false, frozen = false, last = false;
  __device__ StepRule(double t) : trace(t) {}
  __device__ void choose(double trP, double nocc) {
    const double err = trace - trP;
    square = fabs(trP - nocc) < fabs(2.0 * trace - trP - nocc);
    const bool freeze = k >= 2 && (err <= 0.0 || (err < 1e-6 && err >= 0.5 * err2));
    err2 = err1;
    err1 = err;
    trace = square ? trP : 2.0 * trace - trP;
    frozen = freeze;
    last = freeze || k + 1 == kSp2MaxSteps;
    ++k;
  }
};

__device__ void write_state(double* state, const StepRule& rule, double lo, double hi, bool degenerate) {
  state[0] = state[1] = rule.trace;
  state[2] = state[3] = rule.frozen && !degenerate ? 1.0 : 0.0;
  state[4] = lo;
  state[5] = hi;
  state[6] = static_cast<double>(rule.k);
  state[7] = degenerate ? 1.0 : 0.0;
}

__device__ __forceinline__ bool degenerate_interval(double lo, double hi) {
  return !(hi - lo > 1e-12 * fmax(1.0, fmax(fabs(lo), fabs(hi))));
}

// ---- one workgroup, X in LDS -------------------------------------------------
constexpr int kLdsWaves = 16, kLdsThreads = 64 * kLdsWaves;  // at most one tile a wave

// LDS row length of np columns: 2 mod 32 doubles, so the 16-byte reads of the
// 16 rows of an operand cover all 64 banks once.
__host__ __device__ constexpr int lds_row(int np) { return (np + 29) / 32 * 32 + 2; }

__global__ __launch_bounds__(kLdsThreads) void sp2_lds_kernel(const double* __restrict__ F, int n, double nocc,
                                                              double* __restrict__ state, double* __restrict__ out) {
  extern __shared__ double X[];  // np rows of ld: F, then the iterates
  __shared__ double red[3][kLdsWaves];
  const int np = (n + 15) & ~15, ld = lds_row(np), nt = np / 16, ntile = nt * (nt + 1) / 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row16 = lane & 15, g = lane >> 4;
  for (int e = tid; e < np * np; e += kLdsThreads) {
    const int r = e / np, c = e % np;
    const int hi = max(r, c), lo = min(r, c);
    X[r * ld + c] = hi < n ? F[static_cast<std::size_t>(hi) * n + lo] : 0.0;
  }
  __syncthreads();
  // Gershgorin interval and trace: one row per wave and round.
  double lo = INFINITY, hi = -INFINITY, tr = 0.0;
  for (int r = wave; r < n; r += kLdsWaves) {
    double rad = 0.0;
    for (int c = lane; c < n; c += 64)
      if (c != r) rad += fabs(X[r * ld + c]);
    rad = wave_sum(rad);
    const double d = X[r * ld + r];
    lo = fmin(lo, d - rad);
    hi = fmax(hi, d + rad);
    tr += d;
  }
  if (lane == 0) {
    red[0][wave] = lo;
    red[1][wave] = hi;
    red[2][wave] = tr;
  }
  __syncthreads();
  lo = red[0][0];
  hi = red[1][0];
  tr = red[2][0];
  for (int w = 1; w < kLdsWaves; ++w) {
    lo = fmin(lo, red[0][w]);
    hi = fmax(hi, red[1][w]);
    tr += red[2][w];
  }
  const bool degenerate = degenerate_interval(lo, hi);
  const double width = degenerate ? 1.0 : hi - lo;
  StepRule rule(degenerate ? 0.0 : (n * hi - tr) / width);
  __syncthreads();
  double part = 0.0;
  for (int e = tid; e < np * np; e += kLdsThreads) {
    const int r = e / np, c = e % np;
    const double x = r < n && c < n ? ((r == c ? hi : 0.0) - X[r * ld + c]) / width : 0.0;
    X[r * ld + c] = x;
    part += x * x;
  }
  part = wave_sum(part);
  if (lane == 0) red[0][wave] = part;
  __syncthreads();
  if (degenerate) {
    if (tid == 0) write_state(state, rule, lo, hi, true);
    return;
  }
  int ti, tj;
  tile_of(min(wave, ntile - 1), ti, tj);
  const double* pa = X + (ti * 16 + row16) * ld + 4 * g;
  const double* pb = X + (tj * 16 + row16) * ld + 4 * g;
  for (;;) {
    d4 acc = d4{};
    if (wave < ntile) {
#pragma unroll 2
      for (int b = 0; b < nt; ++b) {
        const d4 va = load4(pa + 16 * b), vb = load4(pb + 16 * b);
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = mfma64(va[s], vb[s], acc);
      }
    }
    // The choice is needed from here on: its sum runs behind other waves' products.
    double trP = red[0][0];
    for (int w = 1; w < kLdsWaves; ++w) trP += red[0][w];
    rule.choose(trP, nocc);
    part = 0.0;
    if (wave < ntile) {
      const double weight = ti == tj ? 1.0 : 2.0;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const double p = acc[v];
        const double x = rule.square ? p : 2.0 * X[(ti * 16 + g + 4 * v) * ld + tj * 16 + row16] - p;
        acc[v] = x;
        part += weight * x * x;
      }
    }
    part = wave_sum(part);
    __syncthreads();  // every read of X and red is done
    if (lane == 0) red[0][wave] = part;
    if (wave < ntile) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = ti * 16 + g + 4 * v, c = tj * 16 + row16;
        X[r * ld + c] = acc[v];
        X[c * ld + r] = acc[v];
      }
    }
    __syncthreads();
    if (rule.last) break;
  }
  for (int e = tid; e < n * n; e += kLdsThreads) out[e] = X[(e / n) * ld + e % n];
  if (tid == 0) write_state(state, rule, lo, hi, false);
}

// ---- several workgroups, X in global memory ------------------------------------
// 160 blocks of two waves: an operand goes from L2 to each of the two waves of
// a CU that use it, and 80 blocks of four waves queue twice as long for it.
// Four launches at once (one per hardware queue) are resident together: 1280
// waves of the 2048 that 248 registers allow.  A purification of n = 192 / 384
// takes 287 / 503 us (80 blocks of four: 370 / 680; 325 of one: 292 / 612).
constexpr int kGridThreads = 128, kGridWaves = kGridThreads / 64, kGridBlocks = 160;
constexpr int kTile = 256;  // doubles of a 16 x 16 tile, row-major
// How long a block waits for the others before it gives up: the blocks of a
// launch are few enough to be resident together, so this only ends waits
// behind an oversubscribed device.  VIBEQC_SP2_WAIT_US sets another limit.
constexpr long long kGridWaitUs = 2000000, kTicksPerUs = 100;  // wall_clock64 counts 100 MHz
constexpr unsigned kGridEpochs = kSp2MaxSteps + 4;  // barriers of one launch, at most

// Values other blocks read are stored with device scope (written through the
// XCD's own L2), so once a thread's stores are acknowledged (vmcnt 0) they are
// visible device-wide and a barrier needs no write-back of the L2: only the
// readers drop their stale lines.
template <class T>
__device__ __forceinline__ void publish_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Every block stores its epoch into its own flag and its first wave polls
// all of them: no read-modify-write that the blocks would queue for.
// `epoch` grows from barrier to barrier and from launch to launch.
__device__ bool grid_barrier(unsigned* flags, unsigned epoch, long long wait, int* ok) {
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x < 64) {
    if (threadIdx.x == 0) publish_store(flags + blockIdx.x, epoch);
    const long long start = wall_clock64();
    bool good;
    for (;;) {
      bool here = true;
      for (unsigned k = threadIdx.x; k < gridDim.x; k += 64)
        here = here && static_cast<int>(__hip_atomic_load(flags + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - epoch) >= 0;
      good = __all(here);
      if (good || wall_clock64() - start > wait) break;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (threadIdx.x == 0) *ok = good ? 1 : 0;
  }
  __syncthreads();
  return *ok != 0;
}

struct GridArgs {
  const double* F;
  int n;
  double nocc;
  double* state;
  double* out;
  double* xa;       // lower-triangle tiles of the iterates
  double* xb;
  double* norms;    // [2][blocks] partial |X|_F^2 by step parity
  double* bounds;   // [3][blocks] partial lo, hi, trace
  unsigned* flags;  // [blocks] barrier epochs, then the count of blocks that finished
  unsigned epoch;   // first epoch of this launch
  long long wait;   // ticks
};

// Operand of row block i at k block b: element (16 i + row16, 16 b + 4 g + s)
// of X for s = 0..3, from the stored tile or, above the diagonal, its mirror.
__device__ __forceinline__ d4 tile_operand(const double* x, int i, int b, int row16, int g) {
  if (b <= i) return load4(x + (i * (i + 1) / 2 + b) * kTile + row16 * 16 + 4 * g);
  const double* t = x + (b * (b + 1) / 2 + i) * kTile + 4 * g * 16 + row16;
  return d4{t[0], t[16], t[32], t[48]};
}

__global__ __launch_bounds__(kGridThreads, 2) void sp2_grid_kernel(const GridArgs a) {
  __shared__ double red[3][kGridWaves];
  __shared__ int ok;
  const int n = a.n, np = (n + 15) & ~15, nt = np / 16, ntile = nt * (nt + 1) / 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row16 = lane & 15, g = lane >> 4;
  const int blocks = gridDim.x, nwave = blocks * kGridWaves, wid = blockIdx.x * kGridWaves + wave;
  unsigned epoch = a.epoch;
  // "Given up" until the last block to finish says otherwise: a block that gave
  // up a barrier (and returned) leaves it so.  The count starts at zero again
  // whatever the launch before left; no block adds to it before a barrier.
  if (blockIdx.x == 0 && tid == 0) {
    for (int k = 0; k < 8; ++k) publish_store(a.state + k, k == 6 ? -1.0 : 0.0);
    publish_store(a.flags + blocks, 0u);
  }
  double lo = INFINITY, hi = -INFINITY, tr = 0.0;
  for (int r = wid; r < n; r += nwave) {
    double rad = 0.0;
    for (int c = lane; c < n; c += 64)
      if (c != r) rad += fabs(a.F[static_cast<std::size_t>(max(r, c)) * n + min(r, c)]);
    rad = wave_sum(rad);
    const double d = a.F[static_cast<std::size_t>(r) * n + r];
    lo = fmin(lo, d - rad);
    hi = fmax(hi, d + rad);
    tr += d;
  }
  if (lane == 0) {
    red[0][wave] = lo;
    red[1][wave] = hi;
    red[2][wave] = tr;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kGridWaves; ++w) {
      lo = fmin(lo, red[0][w]);
      hi = fmax(hi, red[1][w]);
      tr += red[2][w];
    }
    publish_store(a.bounds + blockIdx.x, lo);
    publish_store(a.bounds + blocks + blockIdx.x, hi);
    publish_store(a.bounds + 2 * blocks + blockIdx.x, tr);
  }
  if (!grid_barrier(a.flags, epoch++, a.wait, &ok)) return;
  lo = INFINITY;
  hi = -INFINITY;
  tr = 0.0;
  for (int k = lane; k < blocks; k += 64) {
    lo = fmin(lo, a.bounds[k]);
    hi = fmax(hi, a.bounds[blocks + k]);
    tr += a.bounds[2 * blocks + k];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, off));
    hi = fmax(hi, __shfl_xor(hi, off));
  }
  tr = wave_sum(tr);
  const bool degenerate = degenerate_interval(lo, hi);
  const double width = degenerate ? 1.0 : hi - lo;
  StepRule rule(degenerate ? 0.0 : (n * hi - tr) / width);
  if (degenerate) {  // every block alike
    if (blockIdx.x == 0 && tid == 0) write_state(a.state, rule, lo, hi, true);
    return;
  }
  auto publish_norm = [&](double part, int slot) {
    part = wave_sum(part);
    __syncthreads();
    if (lane == 0) red[0][wave] = part;
    __syncthreads();
    if (tid == 0) {
      double s = red[0][0];
      for (int w = 1; w < kGridWaves; ++w) s += red[0][w];
      publish_store(a.norms + slot * blocks + blockIdx.x, s);
    }
  };
  double* cur = a.xa;
  double* next = a.xb;
  double part = 0.0;
  for (int t = wid; t < ntile; t += nwave) {
    int ti, tj;
    tile_of(t, ti, tj);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = ti * 16 + g + 4 * v, c = tj * 16 + row16;
      double x = 0.0;
      if (r < n && c < n) x = ((r == c ? hi : 0.0) - a.F[static_cast<std::size_t>(max(r, c)) * n + min(r, c)]) / width;
      publish_store(cur + t * kTile + (g + 4 * v) * 16 + row16, x);
      part += (ti == tj ? 1.0 : 2.0) * x * x;
    }
  }
  publish_norm(part, 0);
  for (;;) {
    if (!grid_barrier(a.flags, epoch++, a.wait, &ok)) return;
    // The norms are loaded here and consumed after the first product, so
    // their latency is not in front of the operand loads'.
    const int slot = rule.k & 1;
    double norm = 0.0;
    for (int k = lane; k < blocks; k += 64) norm += a.norms[slot * blocks + k];
    bool chosen = false;
    part = 0.0;
    for (int t = wid; t < ntile; t += nwave) {
      int ti, tj;
      tile_of(t, ti, tj);
      double old[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) old[v] = cur[t * kTile + (g + 4 * v) * 16 + row16];
      // U k blocks of both operands (20 16-byte loads a lane) are multiplied
      // while the next U are in flight.  U = 6 spills; 13, a row's half at once,
      // takes 292 / 529 us and one wave per SIMD.
      constexpr int U = 5;
      d4 va[U], vb[U], na[U], nb[U];
      auto fetch = [&](d4(&x)[U], d4(&y)[U], int b0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int b = min(b0 + u, nt - 1);
          x[u] = tile_operand(cur, ti, b, row16, g);
          y[u] = tile_operand(cur, tj, b, row16, g);
        }
      };
      d4 acc = d4{};
      auto multiply = [&](const d4(&x)[U], const d4(&y)[U], int b0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (b0 + u < nt)
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = mfma64(x[u][s], y[u][s], acc);
      };
      fetch(va, vb, 0);
      for (int b0 = 0; b0 < nt; b0 += 2 * U) {
        if (b0 + U < nt) fetch(na, nb, b0 + U);
        multiply(va, vb, b0);
        if (b0 + 2 * U < nt) fetch(va, vb, b0 + 2 * U);
        multiply(na, nb, b0 + U);
      }
      if (!chosen) rule.choose(wave_sum(norm), a.nocc);
      chosen = true;
      const double weight = ti == tj ? 1.0 : 2.0;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = ti * 16 + g + 4 * v, c = tj * 16 + row16;
        const double x = rule.square ? acc[v] : 2.0 * old[v] - acc[v];
        part += weight * x * x;
        if (rule.last) {
          if (r < n && c < n) {
            a.out[static_cast<std::size_t>(r) * n + c] = x;
            a.out[static_cast<std::size_t>(c) * n + r] = x;
          }
        } else {
          publish_store(next + t * kTile + (g + 4 * v) * 16 + row16, x);
        }
      }
    }
    if (!chosen) rule.choose(wave_sum(norm), a.nocc);  // a wave without tiles
    if (rule.last) break;
    publish_norm(part, slot ^ 1);
    double* t = cur;
    cur = next;
    next = t;
  }
  // The last block to finish publishes the outcome.
  __syncthreads();
  if (tid == 0) {
    unsigned* finished = a.flags + blocks;
    if (__hip_atomic_fetch_add(finished, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == static_cast<unsigned>(blocks) - 1)
      write_state(a.state, rule, lo, hi, false);
  }
}

// One workgroup while every wave has at most one tile (np <= 80: 15 tiles) and
// its step beats a grid step, which waits about 5 us for its barrier and
// operands whatever the size: a purification takes 134 us against 157 at n = 72,
// 210 (two tiles for some waves) against 184 at n = 96.
constexpr int kLdsMaxN = 80;
static_assert(kLdsMaxN / 16 * (kLdsMaxN / 16 + 1) / 2 <= kLdsWaves, "one tile a wave");
// Several workgroups up to here.  A step takes 8 us at n = 192 and 13 us at
// n = 384, where the DGEMM, the step kernel and the gap between them take 19
// to 25 and 22 to 26 us.  Further on they draw level: an iteration of a mixed
// SCF takes 2.56 ms in one launch and 2.66 stepwise at n = 408, 3.00 and 3.08 at
// 432, 3.69 and 3.84 at 480, 5.97 and 5.60 at 576.
constexpr int kGridMaxN = 400;

int padded(int n) { return (n + 15) & ~15; }

}  // namespace

bool sp2_fused_fits(int n) { return n >= 1 && n <= kGridMaxN; }

void Sp2Workspace::prepare(int n, hipStream_t s) {
  if (n <= kLdsMaxN || x.size()) return;
  const std::size_t nt = padded(n) / 16;
  x.resize(nt * (nt + 1) * kTile);
  partial.resize(5 * kGridBlocks);
  flags.resize(kGridBlocks + 1);
  const std::vector<unsigned> zero(flags.size(), 0u);
  flags.upload(zero.data(), zero.size(), s);
  epoch = 0;
  const char* limit = std::getenv("VIBEQC_SP2_WAIT_US");
  wait_us = limit ? std::max(0ll, std::min(std::atoll(limit), kGridWaitUs)) : kGridWaitUs;
}

void sp2_purify(const double* F, int n, double nocc, Sp2Workspace& work, double* state, double* X, hipStream_t s) {
  if (!sp2_fused_fits(n)) throw std::invalid_argument("one-launch SP2 size out of range");
  if (n <= kLdsMaxN) {
    const int np = padded(n);
    const std::size_t lds = static_cast<std::size_t>(np) * lds_row(np) * sizeof(double);
    hipLaunchKernelGGL(sp2_lds_kernel, dim3(1), dim3(kLdsThreads), lds, s, F, n, nocc, state, X);
    VQC_LAUNCH("sp2_lds_kernel");
    return;
  }
  const int nt = padded(n) / 16, ntile = nt * (nt + 1) / 2;
  const int blocks = std::min(kGridBlocks, (ntile + kGridWaves - 1) / kGridWaves);
  GridArgs a{};
  a.F = F;
  a.n = n;
  a.nocc = nocc;
  a.state = state;
  a.out = X;
  a.xa = work.x.data();
  a.xb = work.x.data() + static_cast<std::size_t>(ntile) * kTile;
  a.norms = work.partial.data();
  a.bounds = work.partial.data() + 2 * kGridBlocks;
  a.flags = work.flags.data();
  a.epoch = work.epoch + 1;
  a.wait = work.wait_us * kTicksPerUs;
  work.epoch += kGridEpochs;
  hipLaunchKernelGGL(sp2_grid_kernel, dim3(blocks), dim3(kGridThreads), 0, s, a);
  VQC_LAUNCH("sp2_grid_kernel");
}

}  // namespace vqc
