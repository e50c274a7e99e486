// Operand and table descriptors shared by the H*v kernels.
#pragma once

#include "edh_internal.h"

namespace edh {

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
  LzStep lz;
  // tile pass: per slice of two up rows (start, length) of its entries within
  // the tile and outside it
  const int32_t* up_slices;
  const uint32_t* up_in;
  const uint32_t* up_out;
  int row_t, col_t;  // line passes: threads that share a row, a column (hv_lines_threads)
  int xcd_rows;  // rows kernel: XCD-grouped row assignment (measured 2 % faster on the 16-site sector)
  // rows kernel in a batch: an eigensolver run's control block (v and w are
  // then columns col and col + 1 of the basis in v or v_alt; a run whose
  // state is not 0 is skipped)
  const double* ctl;
  const double* v_alt;
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

// Scales of an operand; false: the launch does nothing (uniform over the
// work-group, s_red: one double per wavefront).
__device__ __forceinline__ bool hv_scales(const HvParams& p, double* s_red, bool first, double& vs, double& ws) {
  if (p.lz.k == 0) {
    if (p.done && *p.done) return false;
    vs = p.dscale ? p.dscale[0] : p.vscale;
    ws = p.dscale ? p.dscale[1] : p.wscale;
    return true;
  }
  const bool write = first && p.lz.write && threadIdx.x == 0;
  if (p.lz.k == 1) {
    vs = 1.0;
    ws = 0.0;
    if (write) {
      p.lz.scale[1] = 1.0;
      p.lz.st[0] = p.lz.nl;
      p.lz.st[1] = 0;
    }
    return true;
  }
  if (p.lz.st[1]) return false;
  const double beta = sqrt(block_all_sum(p.lz.share, p.lz.nshare, s_red));
  const bool stop = fabs(beta) < 1e-10;
  vs = 1.0 / beta;
  ws = -beta * p.lz.scale[p.lz.k - 1];
  if (write) {
    p.lz.beta[p.lz.k - 1] = beta;
    p.lz.scale[p.lz.k] = vs;
    if (stop) {
      p.lz.st[0] = p.lz.k - 1;
      p.lz.st[1] = 1;
    }
  }
  return !stop;
}

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
void launch_hv_up_tiles(const DevSector& ds, const HvParams& p, hipStream_t s);

// Fills the descriptor of one operand (hv.hip).
HvBatchJob make_job(const DevSector& ds, const HvArgs& a);

// Largest dynamic LDS a block may use on the current device, less the
// static reduction scratch (hv.hip).
size_t lds_budget();

}  // namespace edh
