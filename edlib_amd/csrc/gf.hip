// Green's-function kernels (FP64):
//  * a_adag as a gather over the target sector (replaces the signed scatter of
//    SpinResolvedStorage::a_adag, SpinResolvedStorage.h:293-381): creating or
//    destroying one electron changes only one spin's pattern, so the source
//    index and sign factor into an up part and a down part;
//  * ChiLoc::operation (ChiLoc.h:474-530): the operator is diagonal and its
//    value is a sum of an up-pattern part and a down-pattern part;
//  * Lanczos::get_frac_point (Lanczos.h:201-224): one thread per energy point.
#include <cfloat>

#include "edh_internal.h"
#include "edh_kernels.h"

namespace edh {

// out = c(+)|in> (accumulate: out = c(+)|in> + out, the order in which the
// reference sums the vectors of several orbitals, GreensFunction.h:434-438)
__global__ void separable_gather_kernel(const double* in, int64_t ldin, const int32_t* mu, const int32_t* md,
                                        const int8_t* su, const int8_t* sd, double* out, int64_t Dup, int64_t Ddn,
                                        int accumulate) {
  const int64_t n = Dup * Ddn;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t u = e / Ddn, d = e - u * Ddn;
    const int32_t a = mu[u], b = md[d];
    double x = 0.0;
    if (a >= 0 && b >= 0) x = (double)(su[u] * sd[d]) * in[(int64_t)a * ldin + b];
    out[e] = accumulate ? x + out[e] : x;
  }
}

__global__ void separable_scale_kernel(const double* in, const double* fu, const double* fd, double* out, int64_t Dup,
                                       int64_t Ddn) {
  const int64_t n = Dup * Ddn;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t u = e / Ddn, d = e - u * Ddn;
    out[e] = (fu[u] + fd[d]) * in[e];
  }
}

struct cplx {
  double re, im;
};
__device__ __forceinline__ cplx cmul(cplx a, cplx b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ cplx csub(cplx a, cplx b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ cplx cscale(cplx a, double s) { return {a.re * s, a.im * s}; }
// Smith's algorithm for a / b.
__device__ __forceinline__ cplx cdiv(cplx a, cplx b) {
  if (fabs(b.re) >= fabs(b.im)) {
    const double r = b.im / b.re, den = b.re + b.im * r;
    return {(a.re + a.im * r) / den, (a.im - a.re * r) / den};
  }
  const double r = b.re / b.im, den = b.re * r + b.im;
  return {(a.re * r + a.im) / den, (a.im * r - a.re) / den};
}

// |d| > big without the overflow-safe hypot where the larger part decides
// (its cost was most of a recurrence step).
__device__ __forceinline__ bool exceeds(cplx d, double big) {
  const double m = fmax(fabs(d.re), fabs(d.im));
  if (m > big) return true;
  return m > 0.5 * big && hypot(d.re, d.im) > big;
}

// Coefficients staged in LDS, kCfLds steps at a time from the last one down,
// and a step's pair read while the one before is computed: the recurrence is a
// serial chain, and a global read per step was the longest part of it (256
// points, whole call: 500 steps 146 us with every read global, 107 staged, 100
// with the pair read ahead; 1500 steps 343, 364 with blocks of one wavefront and
// nothing staged beyond 1024, 250 now).
constexpr int kCfLds = 1024;

// Lanczos.h:201-224 at the point z; all threads of the block take part, those
// that are not live compute nothing.
__device__ __forceinline__ cplx fraction(bool live, cplx z, int n, int isign, double weight, const double* alpha,
                                         const double* beta, double2* s_ab) {
  const double big = (double)FLT_MAX / 2.0;
  const double shift = 1.0 / ((double)FLT_MAX / 1000.0);
  if (n == 1) return cdiv({weight, 0.0}, {z.re - alpha[0] * isign, z.im});
  cplx dA = z, dB = z;
  for (int hi = n; hi > 0; hi -= kCfLds) {
    const int lo = hi > kCfLds ? hi - kCfLds : 0;
    if (hi < n) __syncthreads();  // the steps above are done with
    // s_ab[i - lo] = {alpha_i, beta_{i+1}}
    for (int i = lo + threadIdx.x; i < hi; i += blockDim.x)
      s_ab[i - lo] = make_double2(alpha[i], i + 1 < n ? beta[i + 1] : 0.0);
    __syncthreads();
    if (!live) continue;
    int k = hi - lo - 1;
    if (hi == n) {
      const double b = s_ab[k - 1].y;
      const cplx dl1 = {z.re - s_ab[k].x * isign, z.im};
      const cplx dl2 = {z.re - s_ab[k - 1].x * isign, z.im};
      dA = dl1;                                 // det[i+2]
      dB = csub(cmul(dl2, dl1), {b * b, 0.0});  // det[i+1]
      k -= 2;
    }
    double2 c = s_ab[max(k, 0)];
    for (; k >= 0; --k) {
      const double2 ab = c;
      c = s_ab[max(k - 1, 0)];
      const cplx dli = {z.re - ab.x * isign, z.im};
      const double b2 = ab.y * ab.y;
      cplx d = csub(cmul(dli, dB), cscale(dA, b2));
      if (exceeds(d, big) && k + lo != 0) {
        d = cscale(d, shift);
        dB = cscale(dB, shift);
      }
      dA = dB;
      dB = d;
    }
  }
  return live ? cdiv(cscale(dA, weight), dB) : z;
}

__global__ __launch_bounds__(64) void cf_kernel(int nz, const double* zre, const double* zim, double ev, int nlanc,
                                                int isign, double expb, const double* alpha, const double* beta,
                                                double* out_re, double* out_im) {
  __shared__ double2 s_ab[kCfLds];
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  const int at = min(q, nz - 1);
  const cplx res = fraction(q < nz, {zre[at], zim[at]}, nlanc, isign, ev * expb, alpha, beta, s_ab);
  if (q >= nz) return;
  out_re[q] = res.re;
  out_im[q] = res.im;
}

// Many continued fractions at once: block row j evaluates job j at the
// points z = excited_j * isign_j + i wn[q].
__global__ __launch_bounds__(64) void cf_batch_kernel(int nz, const double* wr, const double* wn, const CfJob* jobs,
                                                      double* out_re, double* out_im) {
  __shared__ double2 s_ab[kCfLds];
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  const int at = min(q, nz - 1);
  const CfJob& J = jobs[blockIdx.y];
  // z = freq_point + isign * E (Lanczos.h:146-148): i w_n on the Matsubara
  // mesh (wr null), w + i pi/beta on the real axis
  const cplx z = {(wr ? wr[at] : 0.0) + J.excited * J.isign, wn[at]};
  const cplx res = fraction(q < nz, z, J.nlanc, J.isign, J.ev * J.expb, J.alpha, J.beta, s_ab);
  if (q >= nz) return;
  out_re[(size_t)blockIdx.y * nz + q] = res.re;
  out_im[(size_t)blockIdx.y * nz + q] = res.im;
}

void dev_cf_batch(int njobs, int nz, const double* wr, const double* wn, const CfJob* jobs, double* out_re,
                  double* out_im, hipStream_t s) {
  if (njobs <= 0 || nz <= 0) return;
  hipLaunchKernelGGL(cf_batch_kernel, dim3((nz + 63) / 64, njobs), dim3(64), 0, s, nz, wr, wn, jobs, out_re,
                     out_im);
  EDH_HIP(hipGetLastError());
}

void dev_separable_gather(const double* in, int64_t ldin, const int32_t* mu, const int32_t* md, const int8_t* su,
                          const int8_t* sd, double* out, int64_t Dup, int64_t Ddn, hipStream_t s, bool accumulate) {
  if (Dup * Ddn == 0) return;
  hipLaunchKernelGGL(separable_gather_kernel, dim3(reduce_grid(Dup * Ddn)), dim3(kVecBlock), 0, s, in, ldin, mu, md,
                     su, sd, out, Dup, Ddn, accumulate ? 1 : 0);
  EDH_HIP(hipGetLastError());
}

void dev_separable_scale(const double* in, const double* fu, const double* fd, double* out, int64_t Dup, int64_t Ddn,
                         hipStream_t s) {
  if (Dup * Ddn == 0) return;
  hipLaunchKernelGGL(separable_scale_kernel, dim3(reduce_grid(Dup * Ddn)), dim3(kVecBlock), 0, s, in, fu, fd, out,
                     Dup, Ddn);
  EDH_HIP(hipGetLastError());
}

void dev_cf_eval(int nz, const double* zre, const double* zim, double ev, int nlanc, int isign, double expb,
                 const double* alpha, const double* beta, double* out_re, double* out_im, hipStream_t s) {
  if (nz <= 0) return;
  hipLaunchKernelGGL(cf_kernel, dim3((nz + 63) / 64), dim3(64), 0, s, nz, zre, zim, ev, nlanc, isign, expb, alpha,
                     beta, out_re, out_im);
  EDH_HIP(hipGetLastError());
}

}  // namespace edh
