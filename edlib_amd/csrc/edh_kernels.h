// Launchers of the vector, Gram-Schmidt and Green's-function kernels.
#pragma once

#include "edh_internal.h"

namespace edh {

constexpr int kVecBlock = 256;      // threads per block of the vector kernels
constexpr int kMaxPartials = 2048;  // blocks of a grid-stride reduction
constexpr int kMaxBasis = 48;       // largest Krylov basis handled on the device

int reduce_grid(int64_t n);
void dev_dot(const double* a, const double* b, int64_t n, double* partial, double* out, hipStream_t s);
void dev_norm(const double* a, int64_t n, double* partial, double* out, hipStream_t s);
void dev_scale_inv(const double* x, const double* nrm, double* out, int64_t n, hipStream_t s);
void dev_fill(double* p, int64_t n, double x, hipStream_t s);  // a kernel, never a memset (graph-safe)
// Random start vector: uniform [-1, 1) from splitmix64 (seed 0 -> a fixed
// default), the same values as the sequential host generator.
void dev_random_uniform(double* x, int64_t n, uint64_t seed, hipStream_t s);
// Column cnt of V (n rows each) made orthogonal to columns 0..cnt-1 and
// normalised (see gs_dots_kernel): hcol[0..cnt) = its projections, *nrm = its
// norm before the normalisation (NaN: repeat with exact); part: 2 (cnt + 1)
// gs_grid(n) doubles.
constexpr int kGsShares = 512;
int gs_grid(int64_t n);
void dev_orthonormalize(double* V, int64_t n, int cnt, double* part, double* hcol, double* nrm, bool exact,
                        hipStream_t s);
// Y[:, j] = sum_i C[i + j*m] V[:, i]  (C on the device, column-major m x k);
// last: Y[:, k] = V[:, m] too
void dev_combine(const double* V, int64_t n, int m, const double* C, int k, double* Y, bool last, hipStream_t s);
// Second half of a single-sector Lanczos step (see LzStep): w -= alpha_k x
// scale[k] with alpha_k from the H*v's ndot shares, and lanczos_update_grid(n)
// shares of |w|^2.  w and x 16-byte aligned.
constexpr int kLzShares = 512;
int lanczos_update_grid(int64_t n);
// The same sums taken once, for sectors of many rows: the step's scales into
// pair (then the H*v takes them as dscale, and st[1] as done), the H*v's shares
// into kLzFold.
constexpr int kLzFold = 256;
void dev_lanczos_scale(const LzStep& step, double* pair, hipStream_t s);
void dev_lanczos_fold(const double* dot, int ndot, const int* st, double* out, hipStream_t s);
void dev_lanczos_update(double* w, const double* x, int64_t n, const double* dot, int ndot, const double* scale,
                        double* alpha, const int* st, int k, double* share, hipStream_t s);

// Green's-function helpers (gf.hip)
void dev_separable_gather(const double* in, int64_t ldin, const int32_t* mu, const int32_t* md, const int8_t* su,
                          const int8_t* sd, double* out, int64_t Dup, int64_t Ddn, hipStream_t s,
                          bool accumulate = false);
void dev_separable_scale(const double* in, const double* fu, const double* fd, double* out, int64_t Dup, int64_t Ddn,
                         hipStream_t s);
// One continued fraction of a batch (device pointers into a packed array).
struct CfJob {
  double ev, expb, excited;
  int isign, nlanc;
  const double* alpha;
  const double* beta;
};
// Run j at point q: z = (wr ? wr[q] : 0) + excited_j * isign_j + i wn[q].
void dev_cf_batch(int njobs, int nz, const double* wr, const double* wn, const CfJob* jobs, double* out_re,
                  double* out_im, hipStream_t s);
void dev_cf_eval(int nz, const double* zre, const double* zim, double ev, int nlanc, int isign, double expb,
                 const double* alpha, const double* beta, double* out_re, double* out_im, hipStream_t s);

// Symmetric eigen-decomposition on the host (eig.hip): A (n x n, row-major)
// is overwritten by the eigenvectors (columns), w by ascending eigenvalues.
void sym_eig(int n, std::vector<double>& A, std::vector<double>& w);

}  // namespace edh
