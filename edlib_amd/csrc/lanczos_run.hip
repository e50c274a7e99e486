// A whole Lanczos run of a small sector in one launch of one work-group.
//
// A step of a few thousand states is two launches of about 6 us each in which
// the chip does next to nothing.  Here the current vector stays in LDS, the
// previous one and the diagonal in registers, and a step's two sums are
// barriers of a work-group instead of kernel boundaries.
//
// Thread t owns the down state d = t mod D_dn in rows u0, u0 + rows, ...: its
// entries of the down-spin table are the same for all of them and stay in
// registers.  The up-spin term takes the transposed assignment (one up state,
// several columns) and passes its sums through LDS.  The elements of a thread
// are gathered in pairs without a test: one past the last row reads the row
// after it, which lies in the same LDS block, and its sum is not used.
//
// What bounds it: about 3.5 us of barriers and dependent LDS reads a step, then
// the LDS reads themselves, one of 8 bytes per hop and element, by one CU.
// MI355X, us per step, two launches : this: 400 states 11.7 : 3.8, 8-site ring
// (3,920) 11.3 : 5.8, (4,900) 11.2 : 7.1, Anderson (4,900) 10.3 : 5.0,
// Kanamori (4,900, 16 hops) 12.7 : 10.9, all-to-all (4,900, 16 hops) 13.7 :
// 11.5, 12 x 495 states 11.3 : 5.7.  All that fit six elements a thread gain,
// so the limits are those of the registers and of LDS.
#include <algorithm>

#include "edh_kernels.h"
#include "hv_params.h"
#include "wave.h"

namespace edh {

namespace {

constexpr int kRunWG = 1024;
constexpr int kRunJ = 6;  // elements per thread

struct RunTables {
  const int32_t* dn_rowp;
  const uint32_t* dn_packed;
  int rows, cols;  // rows (columns) the work-group covers at a time, down (up) pass
  int ja, jb;      // elements per thread in the down (up) pass
  int ld;          // LDS row stride
  int nkp;         // entries of kan_ptr less one
};

// Sum over the work-group, the same value on every thread; slot alternates
// between two sets of 16 so that one barrier is enough.
__device__ __forceinline__ double run_sum(double x, double* s_red, int slot) {
  x = wave_sum(x);
  double* r = s_red + 16 * slot;
  if ((threadIdx.x & 63) == 0) r[threadIdx.x >> 6] = x;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int q = 0; q < kRunWG / 64; ++q) t += r[q];
  return t;
}

template <int H>
__global__ __launch_bounds__(kRunWG) void lanczos_run_kernel(HvParams p, RunTables t, int cross, int nl,
                                                             const double* __restrict__ v0, double* res) {
  extern __shared__ double s_run[];
  __shared__ double s_red[32];
  const int Dup = p.Dup, Ddn = p.Ddn, ld = t.ld;
  const int tid = threadIdx.x;
  double* const x = s_run;                    // the current vector
  double* const y = x + (size_t)Dup * ld;     // the up-spin term
  double* const vals = y + (size_t)Dup * ld;  // value table
  double* const kc = vals + p.nvals;          // impurity terms: coefficients,
  int* const ko = reinterpret_cast<int*>(kc + p.nkan);  // element offsets,
  int* const kp = ko + p.nkan;                          // and where a pair of patterns has them
  for (int i = tid; i < p.nvals; i += kRunWG) vals[i] = p.values[i];
  if (p.kan_ml > 0) {
    for (int i = tid; i < p.nkan; i += kRunWG) {
      kc[i] = p.kan_c[i];
      ko[i] = (int)p.kan_off[i];
    }
    for (int i = tid; i <= t.nkp; i += kRunWG) kp[i] = p.kan_ptr[i];
  }
  int* const st = reinterpret_cast<int*>(res);
  double* const alpha = res + 1;
  double* const beta = alpha + nl;

  // down pass
  const int d = tid % Ddn, u0 = tid / Ddn;
  const bool own = u0 < t.rows;
  const int na = 1 << (p.Ns - p.nb);
  uint32_t de[H], ue[H];
  int nd = 0, nu = 0;
  if (own) {
    const int b = t.dn_rowp[d];
    nd = t.dn_rowp[d + 1] - b;
#pragma unroll
    for (int k = 0; k < H; ++k) de[k] = k < nd ? t.dn_packed[b + k] : 0u;
  }
  // up pass
  const int u = tid % Dup, d0 = tid / Dup;
  const bool uown = d0 < t.cols;
  if (uown) {
    const int b = p.up_rowp[u];
    nu = p.up_rowp[u + 1] - b;
#pragma unroll
    for (int k = 0; k < H; ++k) ue[k] = k < nu ? p.up_packed[b + k] : 0u;
  }
  double diag[kRunJ], prev[kRunJ], w[kRunJ];
  int au[kRunJ];
  const int bd = own ? p.dn_bits[d] : 0;
#pragma unroll
  for (int j = 0; j < kRunJ; ++j) {
    diag[j] = prev[j] = w[j] = 0.0;
    au[j] = 0;
    const int r = u0 + j * t.rows;
    if (own && r < Dup) {
      const int bu = p.up_bits[r];
      au[j] = (bu >> p.nb) * na + (bd >> p.nb);
      double c = 0.0;
      if (cross == CROSS_POPC) c = cross_term<CROSS_POPC>(p, r, bu, bd, na);
      else if (cross == CROSS_IMP) c = cross_term<CROSS_IMP>(p, r, bu, bd, na);
      else if (cross == CROSS_GENERAL) c = cross_term<CROSS_GENERAL>(p, r, bu, bd, na);
      diag[j] = p.up_e[r] + p.dn_e[d] + c;
      x[r * ld + d] = v0[(size_t)r * Ddn + d];
    }
  }
  double b1 = 0.0, norm2 = 0.0;
  int taken = nl;
  for (int k = 1; k <= nl; ++k) {
    if (k > 1) {
      b1 = sqrt(norm2);
      if (tid == 0) beta[k - 1] = b1;
      if (fabs(b1) < 1e-10) {  // the same on every thread
        taken = k - 1;
        break;
      }
      const double s = 1.0 / b1;
#pragma unroll
      for (int j = 0; j < kRunJ; ++j) {
        const int r = u0 + j * t.rows;
        if (own && r < Dup) {
          prev[j] = x[r * ld + d];
          x[r * ld + d] = w[j] * s;
        }
      }
    }
    __syncthreads();
    // decoded anew in every step: kept over all of them, the addresses of
    // every entry and element would not fit the registers
#pragma unroll
    for (int q = 0; q < H; ++q) asm volatile("" : "+v"(ue[q]), "+v"(de[q]));
    int z = 0;
    asm volatile("" : "+v"(z));
    double* const xs = x + z;
    if (uown) {
      double acc[kRunJ];
#pragma unroll
      for (int j = 0; j < kRunJ; ++j) acc[j] = 0.0;
#pragma unroll
      for (int q = 0; q < H; ++q) {
        if (q < nu) {
          const double h = vals[ue[q] >> kColBits];
          const double* c = xs + (int)(ue[q] & kColMask) * ld;
#pragma unroll
          for (int j = 0; j < kRunJ; ++j)
            if ((j & ~1) < t.jb) acc[j] = fma(h, c[d0 + j * t.cols], acc[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < kRunJ; ++j) {
        const int col = d0 + j * t.cols;
        if (col < Ddn) y[u * ld + col] = acc[j];
      }
    }
    __syncthreads();
    double dot = 0.0;
    if (own) {
#pragma unroll
      for (int j = 0; j < kRunJ; ++j) {
        const int r = u0 + j * t.rows;
        if (r < Dup) w[j] = fma(diag[j], x[r * ld + d], fma(-b1, prev[j], y[r * ld + d]));
      }
#pragma unroll
      for (int q = 0; q < H; ++q) {
        if (q < nd) {
          const double h = vals[de[q] >> kColBits];
          const double* c = xs + u0 * ld + (int)(de[q] & kColMask);
#pragma unroll
          for (int j = 0; j < kRunJ; ++j)
            if ((j & ~1) < t.ja) w[j] = fma(h, c[j * t.rows * ld], w[j]);
        }
      }
      if (p.kan_ml > 0) {
#pragma unroll
        for (int j = 0; j < kRunJ; ++j) {
          const int r = u0 + j * t.rows;
          if (r < Dup)
            for (int q = kp[au[j]]; q < kp[au[j] + 1]; ++q) w[j] = fma(kc[q], x[r * ld + d + ko[q]], w[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < kRunJ; ++j) {
        const int r = u0 + j * t.rows;
        if (r < Dup) dot = fma(x[r * ld + d], w[j], dot);
      }
    }
    const double a = run_sum(dot, s_red, 0);
    if (tid == 0) alpha[k - 1] = a;
    double sq = 0.0;
    if (own) {
#pragma unroll
      for (int j = 0; j < kRunJ; ++j) {
        const int r = u0 + j * t.rows;
        if (r < Dup) {
          w[j] = fma(-a, x[r * ld + d], w[j]);
          sq = fma(w[j], w[j], sq);
        }
      }
    }
    norm2 = run_sum(sq, s_red, 1);
  }
  if (tid == 0) {
    st[0] = taken;
    st[1] = taken < nl ? 1 : 0;
  }
}

struct RunPlan {
  RunTables t;
  size_t smem = 0;
  int hops = 0;
  bool ok = false;
};

RunPlan run_plan(const DevSector& ds) {
  RunPlan r;
  const int64_t Du = ds.up.D, Dd = ds.dn.D;
  if (ds.N <= 0 || Du > kRunWG || Dd > kRunWG) return r;
  r.t.dn_rowp = ds.dn.rowp;
  r.t.dn_packed = ds.dn.packed;
  // (with more than half the rows at a time, twice as many are at most 2 D_up:
  // the gathers in pairs stay in the two vectors' LDS)
  r.t.rows = (int)std::min(kRunWG / Dd, Du);
  r.t.cols = (int)std::min(kRunWG / Du, Dd);
  r.t.ja = (int)((Du + r.t.rows - 1) / r.t.rows);
  r.t.jb = (int)((Dd + r.t.cols - 1) / r.t.cols);
  // an odd stride keeps a column off one LDS bank; the impurity terms' element
  // offsets hold for the plain stride
  r.t.ld = (int)(ds.kan_ml > 0 ? Dd : Dd | 1);
  r.t.nkp = ds.kan_ml > 0 ? 1 << (2 * ds.kan_ml) : 0;
  r.hops = std::max(ds.up.max_hops, ds.dn.max_hops);
  r.smem = ((size_t)2 * Du * r.t.ld + ds.nvalues + ds.nkan) * sizeof(double) +
           ((size_t)ds.nkan + r.t.nkp + 1) * sizeof(int);
  r.ok = r.t.ja <= kRunJ && r.t.jb <= kRunJ && r.hops <= 16 && r.smem <= lds_budget();
  return r;
}

}  // namespace

bool lanczos_run_fits(const DevSector& ds) { return run_plan(ds).ok; }

void dev_lanczos_run(const DevSector& ds, const double* v0, int nl, double* res, hipStream_t s) {
  const RunPlan r = run_plan(ds);
  EDH_CHECK(r.ok, EDH_ERR_INTERNAL, "Lanczos run: the sector does not fit one work-group");
  const HvParams p = make_params(ds, HvArgs{});
  auto k = r.hops <= 8 ? lanczos_run_kernel<8> : lanczos_run_kernel<16>;
  if (r.smem > 64 * 1024)
    EDH_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)r.smem));
  hipLaunchKernelGGL(k, dim3(1), dim3(kRunWG), r.smem, s, p, r.t, ds.cross_mode, nl, v0, res);
  EDH_HIP(hipGetLastError());
}

}  // namespace edh
