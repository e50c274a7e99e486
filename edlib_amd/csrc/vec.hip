// Vector kernels (FP64): dot products, fused axpy + norm, the Lanczos
// recurrence bookkeeping, and the Gram-Schmidt kernels of the eigensolver.
// Reductions are two-stage and deterministic: each block reduces with
// wavefront shuffles into one partial, one block then sums the partials in a
// fixed order.
#include "edh_internal.h"
#include "edh_kernels.h"
#include "hv_params.h"

namespace edh {

__device__ __forceinline__ double block_sum(double x, double* s_red) {
  for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s_red[wid] = x;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += s_red[q];
  return t;  // valid on thread 0
}

__global__ void dot_partial_kernel(const double* a, const double* b, int64_t n, double* partial) {
  __shared__ double s_red[16];
  double acc = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    acc = fma(a[i], b[i], acc);
  double t = block_sum(acc, s_red);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// Sums `n` partials in a fixed order into *out (optionally its square root).
__global__ void reduce_partials_kernel(const double* partial, int n, double* out, int take_sqrt) {
  __shared__ double s_red[16];
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) acc += partial[i];
  double t = block_sum(acc, s_red);
  if (threadIdx.x == 0) *out = take_sqrt ? sqrt(t) : t;
}

// Second half of Lanczos step k (Lanczos.h:56-60) of a single-sector run:
// alpha_k = the sum of the H*v's shares of <v, w>, formed by every block from
// the same shares in the same order, then w -= alpha_k v_k (stored as x with
// scale[k]) and the blocks' shares of |w|^2, from which the next step's H*v
// takes beta_k.  Two launches a step: the reductions that used to take a
// launch each read at most a few hundred numbers.
__global__ __launch_bounds__(kVecBlock) void lanczos_update_kernel(double* __restrict__ w, const double* __restrict__ x,
                                                                   int64_t n, const double* __restrict__ dot, int ndot,
                                                                   const double* __restrict__ scale, double* alpha,
                                                                   const int* __restrict__ st, int k,
                                                                   double* __restrict__ share) {
  __shared__ double s_red[16];
  if (st[1]) return;
  const double a = block_all_sum(dot, ndot, s_red);
  if (blockIdx.x == 0 && threadIdx.x == 0) alpha[k - 1] = a;
  const double c = -a * scale[k];
  const int64_t step = (int64_t)gridDim.x * blockDim.x, n2 = n >> 1;
  double2* w2 = reinterpret_cast<double2*>(w);
  const double2* x2 = reinterpret_cast<const double2*>(x);
  double s0 = 0.0, s1 = 0.0;
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  for (; i + step < n2; i += 2 * step) {
    const double2 p = x2[i], q = x2[i + step];
    double2 y = w2[i], z = w2[i + step];
    y.x = fma(c, p.x, y.x);
    y.y = fma(c, p.y, y.y);
    z.x = fma(c, q.x, z.x);
    z.y = fma(c, q.y, z.y);
    w2[i] = y;
    w2[i + step] = z;
    s0 = fma(y.x, y.x, s0);
    s1 = fma(y.y, y.y, s1);
    s0 = fma(z.x, z.x, s0);
    s1 = fma(z.y, z.y, s1);
  }
  if (i < n2) {
    const double2 p = x2[i];
    double2 y = w2[i];
    y.x = fma(c, p.x, y.x);
    y.y = fma(c, p.y, y.y);
    w2[i] = y;
    s0 = fma(y.x, y.x, s0);
    s1 = fma(y.y, y.y, s1);
  }
  if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
    const double y = fma(c, x[n - 1], w[n - 1]);
    w[n - 1] = y;
    s0 = fma(y, y, s0);
  }
  __syncthreads();  // s_red is read by block_all_sum's callers until here
  const double t = block_sum(s0 + s1, s_red);
  if (threadIdx.x == 0) share[blockIdx.x] = t;
}

// A step of a sector with many rows: what every work-group of its H*v and every
// block of its update would sum again is summed once, in two launches of their
// own.
//   scale: the sums of HvScales, left as {scale of v_k, of v_{k-1}} for the H*v
//   fold:  the H*v's shares of <v, w> into kLzFold
__global__ __launch_bounds__(kVecBlock) void lanczos_scale_kernel(LzStep lz, double* __restrict__ pair) {
  __shared__ double s_red[16];
  HvStepParams p;
  p.lz = lz;
  const HvScales sc(p, s_red);
  if (threadIdx.x != 0) return;
  pair[0] = sc.v;
  pair[1] = sc.w;
  HvScales::record(p, sc.v, sc.beta, sc.live);
}

__global__ __launch_bounds__(64) void lanczos_fold_kernel(const double* __restrict__ dot, int ndot,
                                                          const int* __restrict__ st, double* __restrict__ out) {
  if (st[1]) return;
  const int per = (ndot + gridDim.x - 1) / gridDim.x;
  const int e1 = min(ndot, ((int)blockIdx.x + 1) * per);
  double x = 0.0;
  for (int i = blockIdx.x * per + threadIdx.x; i < e1; i += 64) x += dot[i];
  for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
  if (threadIdx.x == 0) out[blockIdx.x] = x;
}

// ---- Gram-Schmidt of a new basis vector (eigensolver) ----------------------
// w (column cnt of V) against columns 0..cnt-1 by classical Gram-Schmidt, a
// second pass where ARPACK dsaitr's DGKS test asks for it (the first pass
// left less than 0.717 of the norm), and the normalisation, in three launches:
//   dots:    shares of h = V^T w and |w|^2
//   update:  w -= V h, and from the same registers the shares of s = V^T w
//            and |w|^2
//   finish:  w = (w - V s) / nrm where the test asks for it, else w / nrm,
//            with nrm^2 = |w|^2 - |s|^2 (exact up to rounding: |s| << |w|)
// Where the second pass takes a good part of what the first one left (the
// basis spans an invariant subspace and w is rounding noise) that difference
// is no norm: *nrm is then NaN, and the caller repeats the cycle in the exact
// form, which measures |w - V s| and scales in a fourth launch.
// A block's shares are sums over its tiles; every block of the next launch
// sums all of them itself, each the same numbers in the same order, so the
// reductions take no launch of their own.  Ten launches a step (two passes of
// dots, reduction, update, norm; scaling; H*v) became four; on 213,444 states
// with a basis of 11 the eight of them that are not H*v took 103 us, these
// three take 23.5 us.
constexpr int kGsBlock = 512;   // threads
constexpr int kGsElems = 2;     // elements per thread and tile
constexpr int kGsTile = kGsBlock * kGsElems;
constexpr int kGsGroup = 12;    // columns held in registers together (NCV = 11 in one group)
constexpr int kGsWaves = kGsBlock / 64;

// Sums of cnt values' shares (value i of block b at part[i * G + b]) into
// s_h, a value per wavefront at a time.
__device__ __forceinline__ void gs_sums(const double* __restrict__ part, int G, int cnt, double* s_h) {
  const int lane = threadIdx.x & 63;
  for (int i = threadIdx.x >> 6; i < cnt; i += kGsWaves) {
    double t = 0.0;
    for (int b = lane; b < G; b += 64) t += part[(size_t)i * G + b];
    for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
    if (lane == 0) s_h[i] = t;
  }
  __syncthreads();
}

// Block sums of acc[0..n) into part[(i0 + g) * G + block].
template <int K>
__device__ __forceinline__ void gs_store(const double (&acc)[K], int n, int i0, int G, double (*s_p)[K], double* part) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int g = 0; g < K; ++g) {
    if (g >= n) break;
    double x = acc[g];
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
    if (lane == 0) s_p[wave][g] = x;
  }
  __syncthreads();
  if ((int)threadIdx.x < n) {
    double t = 0.0;
    for (int q = 0; q < kGsWaves; ++q) t += s_p[q][threadIdx.x];
    part[(size_t)(i0 + threadIdx.x) * G + blockIdx.x] = t;
  }
  __syncthreads();
}

// Columns i0 + g < cnt of V, then w itself (slot cnt), at element e.
template <int K>
__device__ __forceinline__ void gs_load(const double* __restrict__ V, int64_t ldv, int i0, int cnt, int64_t e,
                                        double (&x)[K]) {
#pragma unroll
  for (int g = 0; g < K; ++g) x[g] = i0 + g < cnt ? V[(int64_t)(i0 + g) * ldv + e] : 0.0;
}

__global__ __launch_bounds__(kGsBlock) void gs_dots_kernel(const double* __restrict__ V, int64_t n, int cnt,
                                                           double* __restrict__ part) {
  __shared__ double s_p[kGsWaves][kGsGroup];
  const int G = gridDim.x;
  // the group's columns and, in the slot after the last one, w
  for (int i0 = 0; i0 <= cnt; i0 += kGsGroup) {
    double acc[kGsGroup];
#pragma unroll
    for (int g = 0; g < kGsGroup; ++g) acc[g] = 0.0;
    for (int64_t e0 = (int64_t)blockIdx.x * kGsTile; e0 < n; e0 += (int64_t)G * kGsTile) {
      double x[kGsElems][kGsGroup], we[kGsElems];
#pragma unroll
      for (int u = 0; u < kGsElems; ++u) {
        const int64_t e = e0 + u * kGsBlock + threadIdx.x;
        we[u] = e < n ? V[(int64_t)cnt * n + e] : 0.0;
        gs_load<kGsGroup>(V, n, i0, e < n ? cnt + 1 : 0, e, x[u]);
      }
#pragma unroll
      for (int u = 0; u < kGsElems; ++u)
#pragma unroll
        for (int g = 0; g < kGsGroup; ++g) acc[g] = fma(x[u][g], we[u], acc[g]);
    }
    gs_store<kGsGroup>(acc, min(kGsGroup, cnt + 1 - i0), i0, G, s_p, part);
  }
}

// ONE: the basis fits one group, so the columns stay in registers from the
// update to the projections; else they are read again.
template <bool ONE>
__global__ __launch_bounds__(kGsBlock) void gs_update_kernel(double* __restrict__ V, int64_t n, int cnt,
                                                             const double* __restrict__ part1,
                                                             double* __restrict__ part2, double* __restrict__ hcol) {
  __shared__ double s_h[kMaxBasis + kGsGroup];
  __shared__ double s_p[kGsWaves][kGsGroup + 1];
  const int G = gridDim.x;
  for (int i = threadIdx.x; i < kMaxBasis + kGsGroup; i += kGsBlock) s_h[i] = 0.0;
  __syncthreads();
  gs_sums(part1, G, cnt, s_h);
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < cnt; i += kGsBlock) hcol[i] = s_h[i];
  double* __restrict__ w = V + (int64_t)cnt * n;
  if (ONE) {
    double acc[kGsGroup + 1];
#pragma unroll
    for (int g = 0; g <= kGsGroup; ++g) acc[g] = 0.0;
    for (int64_t e0 = (int64_t)blockIdx.x * kGsTile; e0 < n; e0 += (int64_t)G * kGsTile) {
      double x[kGsElems][kGsGroup], y[kGsElems];
#pragma unroll
      for (int u = 0; u < kGsElems; ++u) {
        const int64_t e = e0 + u * kGsBlock + threadIdx.x;
        y[u] = e < n ? w[e] : 0.0;
        gs_load<kGsGroup>(V, n, 0, e < n ? cnt : 0, e, x[u]);
      }
#pragma unroll
      for (int u = 0; u < kGsElems; ++u) {
        const int64_t e = e0 + u * kGsBlock + threadIdx.x;
#pragma unroll
        for (int g = 0; g < kGsGroup; ++g) y[u] = fma(-s_h[g], x[u][g], y[u]);
        if (e < n) w[e] = y[u];
#pragma unroll
        for (int g = 0; g < kGsGroup; ++g) acc[g] = fma(x[u][g], y[u], acc[g]);
        acc[kGsGroup] = fma(y[u], y[u], acc[kGsGroup]);
      }
    }
    double v[kGsGroup + 1];
#pragma unroll
    for (int g = 0; g <= kGsGroup; ++g) v[g] = g < cnt ? acc[g < kGsGroup ? g : 0] : (g == cnt ? acc[kGsGroup] : 0.0);
    gs_store<kGsGroup + 1>(v, cnt + 1, 0, G, s_p, part2);
    return;
  }
  for (int64_t e0 = (int64_t)blockIdx.x * kGsTile; e0 < n; e0 += (int64_t)G * kGsTile)
#pragma unroll
    for (int u = 0; u < kGsElems; ++u) {
      const int64_t e = e0 + u * kGsBlock + threadIdx.x;
      if (e >= n) continue;
      double y = w[e];
      for (int i0 = 0; i0 < cnt; i0 += kGsGroup) {
        double x[kGsGroup];
        gs_load<kGsGroup>(V, n, i0, cnt, e, x);
#pragma unroll
        for (int g = 0; g < kGsGroup; ++g) y = fma(-s_h[i0 + g], x[g], y);
      }
      w[e] = y;
    }
  // a thread reads back only what it wrote
  for (int i0 = 0; i0 <= cnt; i0 += kGsGroup) {
    double acc[kGsGroup + 1];
#pragma unroll
    for (int g = 0; g <= kGsGroup; ++g) acc[g] = 0.0;
    for (int64_t e0 = (int64_t)blockIdx.x * kGsTile; e0 < n; e0 += (int64_t)G * kGsTile)
#pragma unroll
      for (int u = 0; u < kGsElems; ++u) {
        const int64_t e = e0 + u * kGsBlock + threadIdx.x;
        if (e >= n) continue;
        double x[kGsGroup];
        const double y = w[e];
        gs_load<kGsGroup>(V, n, i0, cnt, e, x);
#pragma unroll
        for (int g = 0; g < kGsGroup; ++g) acc[g] = fma(i0 + g == cnt ? y : x[g], y, acc[g]);
      }
    gs_store<kGsGroup + 1>(acc, min(kGsGroup, cnt + 1 - i0), i0, G, s_p, part2);
  }
}

// EXACT: w = w - V s, unscaled, and the shares of its norm in part1.
template <bool EXACT>
__global__ __launch_bounds__(kGsBlock) void gs_finish_kernel(double* __restrict__ V, int64_t n, int cnt,
                                                             double* part1,
                                                             const double* __restrict__ part2,
                                                             double* __restrict__ hcol, double* __restrict__ nrm_out) {
  __shared__ double s_h[kMaxBasis + kGsGroup];
  __shared__ double s_nb[1];
  __shared__ double s_p[kGsWaves][1];
  const int G = gridDim.x;
  for (int i = threadIdx.x; i < kMaxBasis + kGsGroup; i += kGsBlock) s_h[i] = 0.0;
  __syncthreads();
  gs_sums(part2, G, cnt + 1, s_h);
  gs_sums(part1 + (size_t)cnt * G, G, 1, s_nb);
  const double n2 = s_h[cnt], nrm1 = sqrt(n2);
  const bool again = nrm1 < 0.717 * sqrt(s_nb[0]);
  double nrm = nrm1;
  if (again) {
    double ss = 0.0;
    for (int i = 0; i < cnt; ++i) ss = fma(s_h[i], s_h[i], ss);
    nrm = ss <= 0.25 * n2 ? sqrt(n2 - ss) : __builtin_nan("");
  }
  if (blockIdx.x == 0) {
    if (again)
      for (int i = threadIdx.x; i < cnt; i += kGsBlock) hcol[i] += s_h[i];
    if (!EXACT && threadIdx.x == 0) *nrm_out = nrm;
  }
  __syncthreads();
  if (threadIdx.x == 0) s_h[cnt] = 0.0;  // the norm's slot is a column's coefficient below
  __syncthreads();
  const double f = EXACT ? 1.0 : 1.0 / nrm;
  double acc[1] = {0.0};
  double* __restrict__ w = V + (int64_t)cnt * n;
  for (int64_t e0 = (int64_t)blockIdx.x * kGsTile; e0 < n; e0 += (int64_t)G * kGsTile) {
    double y[kGsElems];
#pragma unroll
    for (int u = 0; u < kGsElems; ++u) {
      const int64_t e = e0 + u * kGsBlock + threadIdx.x;
      y[u] = e < n ? w[e] : 0.0;
    }
    if (again)
      for (int i0 = 0; i0 < cnt; i0 += kGsGroup) {
        double x[kGsElems][kGsGroup];
#pragma unroll
        for (int u = 0; u < kGsElems; ++u) {
          const int64_t e = e0 + u * kGsBlock + threadIdx.x;
          gs_load<kGsGroup>(V, n, i0, e < n ? cnt : 0, e, x[u]);
        }
#pragma unroll
        for (int u = 0; u < kGsElems; ++u)
#pragma unroll
          for (int g = 0; g < kGsGroup; ++g) y[u] = fma(-s_h[i0 + g], x[u][g], y[u]);
      }
#pragma unroll
    for (int u = 0; u < kGsElems; ++u) {
      const int64_t e = e0 + u * kGsBlock + threadIdx.x;
      if (e < n) w[e] = y[u] * f;
      acc[0] = fma(y[u], y[u], acc[0]);
    }
  }
  // (slot cnt of part1, which other blocks may still be reading, is not used)
  if (EXACT) gs_store<1>(acc, 1, 0, G, s_p, part1);
}

// *nrm = the norm from G shares, w /= it.
__global__ __launch_bounds__(kGsBlock) void gs_rescale_kernel(double* __restrict__ w, int64_t n,
                                                              const double* __restrict__ part,
                                                              double* __restrict__ nrm_out) {
  __shared__ double s_n[1];
  gs_sums(part, gridDim.x, 1, s_n);
  const double nrm = sqrt(s_n[0]), f = 1.0 / nrm;
  if (blockIdx.x == 0 && threadIdx.x == 0) *nrm_out = nrm;
  for (int64_t e = blockIdx.x * (int64_t)kGsBlock + threadIdx.x; e < n; e += (int64_t)gridDim.x * kGsBlock) w[e] *= f;
}

// out = x * (1 / *nrm)
__global__ void scale_inv_kernel(const double* x, const double* nrm, double* out, int64_t n) {
  const double s = 1.0 / *nrm;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x)
    out[e] = x[e] * s;
}

// Y (k columns) = V (m columns) * C (m x k, column-major), per element, and
// with `last` column k of Y = column m of V (the residual a thick restart
// continues from).  K >= m: the registers it takes set the occupancy.
template <int K>
__global__ __launch_bounds__(kVecBlock) void basis_combine_kernel(const double* __restrict__ V, int64_t n, int m,
                                                                  const double* __restrict__ C, int k,
                                                                  double* __restrict__ Y, int last) {
  __shared__ double s_c[K * K];
  for (int i = threadIdx.x; i < m * k; i += blockDim.x) s_c[i] = C[i];
  __syncthreads();
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    double v[K];
#pragma unroll
    for (int i = 0; i < K; ++i) v[i] = i < m ? V[i * n + e] : 0.0;
    if (last) Y[(int64_t)k * n + e] = V[(int64_t)m * n + e];
    for (int j = 0; j < k; ++j) {
      double y = 0.0;
#pragma unroll
      for (int i = 0; i < K; ++i)
        if (i < m) y = fma(s_c[j * m + i], v[i], y);
      Y[j * n + e] = y;
    }
  }
}

// ---------------------------------------------------------------------------
// Host launchers.
// ---------------------------------------------------------------------------
int reduce_grid(int64_t n) {
  int64_t g = (n + kVecBlock - 1) / kVecBlock;
  if (g > kMaxPartials) g = kMaxPartials;
  if (g < 1) g = 1;
  return (int)g;
}

void dev_dot(const double* a, const double* b, int64_t n, double* partial, double* out, hipStream_t s) {
  int g = reduce_grid(n);
  hipLaunchKernelGGL(dot_partial_kernel, dim3(g), dim3(kVecBlock), 0, s, a, b, n, partial);
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(1), dim3(kVecBlock), 0, s, partial, g, out, 0);
  EDH_HIP(hipGetLastError());
}

void dev_norm(const double* a, int64_t n, double* partial, double* out, hipStream_t s) {
  int g = reduce_grid(n);
  hipLaunchKernelGGL(dot_partial_kernel, dim3(g), dim3(kVecBlock), 0, s, a, a, n, partial);
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(1), dim3(kVecBlock), 0, s, partial, g, out, 1);
  EDH_HIP(hipGetLastError());
}

__global__ void fill_kernel(double* p, int64_t n, double x) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) p[e] = x;
}

// x[i] = uniform [-1, 1) value number i + 1 of the splitmix64 sequence
// started at st0 (state st0 + (i + 1) * 0x9E3779B97F4A7C15, then the
// splitmix64 output mix), top 53 bits scaled by 2^-52, minus 1: element i of
// the host generator's sequence, produced independently per element.
__global__ void splitmix_uniform_kernel(double* x, int64_t n, uint64_t st0) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    uint64_t z = st0 + (uint64_t)(i + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    x[i] = (double)(z >> 11) * (2.0 / 9007199254740992.0) - 1.0;
  }
}

void dev_random_uniform(double* x, int64_t n, uint64_t seed, hipStream_t s) {
  const uint64_t st0 = seed ? seed : 0x243F6A8885A308D3ull;
  const int g = (int)std::min<int64_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(splitmix_uniform_kernel, dim3(std::max(g, 1)), dim3(256), 0, s, x, n, st0);
  EDH_HIP(hipGetLastError());
}

void dev_fill(double* p, int64_t n, double x, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(fill_kernel, dim3(reduce_grid(n)), dim3(kVecBlock), 0, s, p, n, x);
  EDH_HIP(hipGetLastError());
}

void dev_scale_inv(const double* x, const double* nrm, double* out, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(scale_inv_kernel, dim3(reduce_grid(n)), dim3(kVecBlock), 0, s, x, nrm, out, n);
  EDH_HIP(hipGetLastError());
}

int gs_grid(int64_t n) {
  return (int)std::min<int64_t>(std::max<int64_t>((n + kGsTile - 1) / kGsTile, 1), kGsShares);
}

void dev_orthonormalize(double* V, int64_t n, int cnt, double* part, double* hcol, double* nrm, bool exact,
                        hipStream_t s) {
  EDH_CHECK(cnt >= 1 && cnt < kMaxBasis, EDH_ERR_LIMIT, "Krylov basis size outside the device limit");
  const int g = gs_grid(n);
  double* part2 = part + (size_t)(cnt + 1) * g;
  hipLaunchKernelGGL(gs_dots_kernel, dim3(g), dim3(kGsBlock), 0, s, V, n, cnt, part);
  auto update = cnt <= kGsGroup ? gs_update_kernel<true> : gs_update_kernel<false>;
  hipLaunchKernelGGL(update, dim3(g), dim3(kGsBlock), 0, s, V, n, cnt, part, part2, hcol);
  auto finish = exact ? gs_finish_kernel<true> : gs_finish_kernel<false>;
  hipLaunchKernelGGL(finish, dim3(g), dim3(kGsBlock), 0, s, V, n, cnt, part, part2, hcol, nrm);
  if (exact)
    hipLaunchKernelGGL(gs_rescale_kernel, dim3(g), dim3(kGsBlock), 0, s, V + (int64_t)cnt * n, n, part, nrm);
  EDH_HIP(hipGetLastError());
}

void dev_combine(const double* V, int64_t n, int m, const double* C, int k, double* Y, bool last, hipStream_t s) {
  EDH_CHECK(m <= kMaxBasis && k <= m, EDH_ERR_LIMIT, "Krylov basis larger than the device limit");
  auto kern = m <= 12 ? basis_combine_kernel<12> : m <= 24 ? basis_combine_kernel<24> : basis_combine_kernel<kMaxBasis>;
  hipLaunchKernelGGL(kern, dim3(reduce_grid(n)), dim3(kVecBlock), 0, s, V, n, m, C, k, Y, last ? 1 : 0);
  EDH_HIP(hipGetLastError());
}

int lanczos_update_grid(int64_t n) {
  // four elements a thread, at most 512 blocks (their shares are summed by
  // every work-group of the next H*v)
  return (int)std::min<int64_t>(std::max<int64_t>((n + 4 * kVecBlock - 1) / (4 * kVecBlock), 1), kLzShares);
}

void dev_lanczos_scale(const LzStep& step, double* pair, hipStream_t s) {
  hipLaunchKernelGGL(lanczos_scale_kernel, dim3(1), dim3(kVecBlock), 0, s, step, pair);
  EDH_HIP(hipGetLastError());
}

void dev_lanczos_fold(const double* dot, int ndot, const int* st, double* out, hipStream_t s) {
  hipLaunchKernelGGL(lanczos_fold_kernel, dim3(kLzFold), dim3(64), 0, s, dot, ndot, st, out);
  EDH_HIP(hipGetLastError());
}

void dev_lanczos_update(double* w, const double* x, int64_t n, const double* dot, int ndot, const double* scale,
                        double* alpha, const int* st, int k, double* share, hipStream_t s) {
  hipLaunchKernelGGL(lanczos_update_kernel, dim3(lanczos_update_grid(n)), dim3(kVecBlock), 0, s, w, x, n, dot, ndot,
                     scale, alpha, st, k, share);
  EDH_HIP(hipGetLastError());
}

}  // namespace edh
