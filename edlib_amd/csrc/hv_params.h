// Operand and table descriptors shared by the H*v kernels.
#pragma once

#include "edh_internal.h"

namespace edh {

// What an H*v reads.  Every launch copies it and every work-group begins with
// loads from it, so size and order count in the smallest sectors: without the
// Lanczos step, in this order, kanamori (8 sites) takes 6.40 us a call and 16-bit
// and 32-bit entry sectors up to 13 sites 1 to 2.5 % less than with the single
// pass's fields together in front (6.50), where the loads are merged into wider
// ones; with the step inside 6.55.
struct HvParams {
  int Ns, nb;  // sites per spin, bath bits (Ns - ml) below the impurity bits
  int Dup, Ddn;
  const int32_t* row_order;
  // up spin
  const int32_t* up_bits;
  const double* up_e;
  const int32_t* up_rowp;
  const uint32_t* up_packed;
  const int32_t* up_slptr;
  const int32_t* up_sllen;
  const uint32_t* up_lell;
  // down spin
  const int32_t* dn_bits;
  const double* dn_e;
  const int32_t* dn_slptr;
  const int32_t* dn_sllen;
  const uint32_t* dn_ell;
  const uint32_t* dn_lell;
  const int32_t* dn_q4ptr;
  const uint64_t* dn_q4;
  double dn_vt[4];
  const uint32_t* dn_s4;
  double dn_s4_scale;
  const double* values;
  int nkan;   // impurity terms (staged in LDS by the multi-operand kernel)
  int nvals;  // entries of values (staged in LDS after the row with EF == 4)
  // cross term
  double cross_u;
  const double* cross_imp;
  const double* cross_rowtab;
  // impurity interaction
  int kan_ml;
  const int32_t* kan_ptr;
  const int64_t* kan_off;  // partner state's element offset per term
  const double* kan_c;
  int kan_t;  // the same by target pattern, and the row tiles they need (DevSector)
  const int32_t* row_tiles;
  const int32_t* kan_td;
  const double* kan_tc;
  // operands
  const double* v;
  double* w;
  const double* wprev;
  double vscale, wscale;
  int accumulate;
  double* dot_partial;
  const double* dscale;
  const int* done;
  // tile pass: per slice of two up rows (start, length) of its entries within
  // the tile and outside it
  const int32_t* up_slices;
  const uint32_t* up_in;
  const uint32_t* up_out;
  int xcd_rows;  // rows kernel: XCD-grouped row assignment (measured 2 % faster on the 16-site sector)
  // rows kernel in a batch: an eigensolver run's control block (v and w are
  // then columns col and col + 1 of the basis in v or v_alt; a run whose
  // state is not 0 is skipped)
  const double* ctl;
  const double* v_alt;
};

// With a step of a single-sector Lanczos run (lz.k = 0: without).
struct HvStepParams : HvParams {
  LzStep lz;
};

template <int CROSS>
__device__ __forceinline__ double cross_term(const HvParams& p, int u, int bu, int bd, int na) {
  if (CROSS == CROSS_POPC) return p.cross_u * (double)__builtin_popcount(bu & bd);
  if (CROSS == CROSS_IMP) return p.cross_imp[(bu >> p.nb) * na + (bd >> p.nb)];
  if (CROSS == CROSS_GENERAL) {
    double x = 0.0;
    const double* r = p.cross_rowtab + (size_t)u * p.Ns;
    unsigned m = (unsigned)bd;
    while (m) {
      int b = __builtin_ctz(m);
      x += r[b];
      m &= m - 1;
    }
    return x;
  }
  return 0.0;
}

__device__ __forceinline__ void block_reduce_store(double x, double* s_red, double* out) {
  for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s_red[wid] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += s_red[q];
    *out = t;
  }
}

// Sum of n shares, the same value on every thread: thread t takes shares t,
// t + T, ... in order, then a fixed tree per wavefront and the wavefronts in
// order.
__device__ __forceinline__ double block_all_sum(const double* share, int n, double* s_red) {
  double x = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) x += share[i];
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  __syncthreads();  // s_red may still be read from an earlier use
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = x;
  __syncthreads();
  double t = 0.0;
  for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += s_red[q];
  return t;
}

// A value that all lanes share, in scalar registers.
__device__ __forceinline__ double uniform_value(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readfirstlane((int)b);
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Scales of an operand; live false: the launch does nothing (uniform over the
// work-group, s_red: one double per wavefront).
struct HvScales {
  double v = 0.0, w = 0.0;
  double beta = 0.0;  // Lanczos step after the first: |W_k|
  bool live = false;
  __device__ __forceinline__ HvScales(const HvStepParams& p, double* s_red) {
    if (p.lz.k == 0) {
      if (p.done && *p.done) return;
      v = p.dscale ? p.dscale[0] : p.vscale;
      w = p.dscale ? p.dscale[1] : p.wscale;
      live = true;
      return;
    }
    if (p.lz.k == 1) {
      v = 1.0;
      live = true;
      return;
    }
    if (p.lz.st[1]) return;
    beta = uniform_value(sqrt(block_all_sum(p.lz.share, p.lz.nshare, s_red)));
    v = uniform_value(1.0 / beta);
    w = uniform_value(-beta * p.lz.scale[p.lz.k - 1]);
    live = __builtin_amdgcn_readfirstlane(!(fabs(beta) < 1e-10)) != 0;
  }
  // What one work-group of a Lanczos step's first pass records, at the very end
  // of its kernel, also for a stopped run: a store to memory that the compiler
  // may see ahead of the kernel's uniform table loads, in an early exit too,
  // turns them all from scalar into vector loads (the single pass then takes
  // 5.1 instead of 3.8 ms on the 16-site torus, 187 instead of 134 us on the
  // 14-site ring).
  static __device__ __forceinline__ void record(const HvStepParams& p, double v, double beta, bool live) {
    if (!p.lz.write || p.lz.k == 0 || threadIdx.x != 0) return;
    if (p.lz.k == 1) {
      p.lz.scale[1] = 1.0;
      p.lz.st[0] = p.lz.nl;
      p.lz.st[1] = 0;
      return;
    }
    if (p.lz.st[1]) return;
    p.lz.beta[p.lz.k - 1] = beta;
    p.lz.scale[p.lz.k] = v;
    if (!live) {
      p.lz.st[0] = p.lz.k - 1;
      p.lz.st[1] = 1;
    }
  }
};

// One signed byte-offset slot: a += (+-1) * row[e / 8], the sign in bit 0.
__device__ __forceinline__ double s4_fma(uint32_t e, const char* sv, double a) {
  const double sg = __hiloint2double((int)(0x3FF00000u | (e << 31)), 0);
  return fma(sg, *reinterpret_cast<const double*>(sv + (e & ~1u)), a);
}

struct HvBatchJob {
  HvParams p;
  int64_t row0;
  int cross, kan;
  const double* ctl;    // eigensolver control block or null
  const double* v_alt;  // second basis buffer (with ctl)
  double* tdot;         // per-task shares of <v, w>, or null
  const double* lzk;    // Lanczos run's step counter (buffers in rotation) or null
};

// The up-spin term in tiles (hv_tiles.hip): w += Hup v and the shares of
// <v, w>, hv_up_tiles_blocks of them.
int hv_up_tiles_blocks(const DevSector& ds);
void launch_hv_up_tiles(const DevSector& ds, const HvStepParams& p, hipStream_t s);

// The parameters of one operand (hv.hip).
HvParams make_params(const DevSector& ds, const HvArgs& a);
HvStepParams make_step_params(const DevSector& ds, const HvArgs& a);

// Largest dynamic LDS a block may use on the current device, less the
// static reduction scratch (hv.hip).
size_t lds_budget();

}  // namespace edh
