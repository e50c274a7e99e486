// H*v in two passes of LDS gathers, for sectors whose lines fit LDS several
// at a time.
//
// The state vector is the D_up x D_dn matrix V[u][d].  The down-spin hopping
// mixes the elements of a row, the up-spin hopping those of a column, both
// through a sparse table with one line of entries per basis state.  A
// work-group stages B whole lines (columns, then rows) in LDS with the B
// values of a basis state side by side, so that
//   * one table entry (index, value), loaded and decoded once, serves B
//     elements, and a gather is a 16-byte LDS read per two of them;
//   * neighbour rows of the up-spin term are never re-read from L2 or beyond:
//     each pass reads V once.
// Pass 1 (columns): w = up-spin hopping (+ w_in when that is w itself).
// Pass 2 (rows): w += diag v + w_in + down-spin hopping + impurity terms, and
// the shares of <v, w>.
//
// An element's sum runs in table order in one register whatever the other
// operands of the launch, and a row tile's share of <v, w> depends on the
// sector alone: an operand's result is bit-identical alone and in any mix.
//
// What bounds it (14-site sectors, 3432 x 3432, MI355X): a column pass moves
// 16 N bytes and a row pass 24 N (32 N with an accumulated input in another
// buffer), 37 and 60 us of their 55 and 70 us with 7 entries per state
// (Anderson); every further entry costs 2.6 us a pass, the LDS reads (two
// 16-byte and one 8-byte read per entry and four elements, half as long again
// with bank conflicts).  Kanamori sector (7,7): 83 + 107 us against 372 us in
// the single pass.  B = 2 (two work-groups per CU) took 98 + 137 us on the
// t, t' torus where B = 4 takes 92 + 108: the entries are decoded twice as
// often and every row's request is half as long.
#include <algorithm>
#include <cstring>

#include "hv_params.h"

namespace edh {

namespace {

// One operand of a launch.
struct LinesJob {
  HvStepParams p;
  int cross, kan;
};

// The operand with the scales of this launch.
struct View {
  const double* V;
  double* W;
  const double* Wp;
  double vs, ws;
  bool accum, live;
};

__device__ __forceinline__ View view_of(const HvParams& p, const HvScales& sc) {
  return View{p.v, p.w, p.wprev, sc.v, sc.w, p.accumulate != 0, sc.live};
}

// LDS image of B lines of D elements: planes of two lines, the pair of a
// basis state in 16 bytes, then a zero state (with all B values side by side a 16-byte read
// would use every other 16-byte slot of the banks only).
template <int B>
__device__ __forceinline__ void put_state(double* s, int ld, int i, const double (&x)[B]) {
#pragma unroll
  for (int q = 0; q < B / 2; ++q) reinterpret_cast<double2*>(s)[q * ld + i] = make_double2(x[2 * q], x[2 * q + 1]);
}

template <int B>
__device__ __forceinline__ void get_state(const double* s, int ld, int i, double (&x)[B]) {
#pragma unroll
  for (int q = 0; q < B / 2; ++q) {
    const double2 y = reinterpret_cast<const double2*>(s)[q * ld + i];
    x[2 * q] = y.x;
    x[2 * q + 1] = y.y;
  }
}

// acc[b] += sum over the entries of basis state i (slice i / 64) of
// value * line b[column].  An entry holds its column's byte offset in a plane
// and its value's byte offset in the value table (kLineOff), so decoding it
// takes two instructions.  The slice's slot count is wavefront-uniform.  Entries
// come in groups of U, the next group's loads issued before a group is worked on
// (B = 4, U = 8 against 4: 14-site Kanamori column pass 111 -> 94 us); but the
// tests of the count compile to a branch per entry and a wait for all loads per
// group, so neither these loads nor an entry's LDS reads overlap much else.
template <int B, int U>
__device__ __forceinline__ void gather_line(const double* s, int ld, const double* s_vals, const int32_t* slptr,
                                            const int32_t* sllen, const uint32_t* ell, int i, double (&acc)[B]) {
  const int sl = __builtin_amdgcn_readfirstlane(i >> 6);
  const int len = __builtin_amdgcn_readfirstlane(sllen[sl]);
  const uint32_t* el = ell + slptr[sl] + (i & 63);
  const char* const pl = reinterpret_cast<const char*>(s);
  const char* const vl = reinterpret_cast<const char*>(s_vals);
  uint32_t e[U];
#pragma unroll
  for (int r = 0; r < U; ++r) e[r] = r < len ? el[r * kSlice] : 0u;
  for (int k = 0; k < len; k += U) {
    uint32_t n[U];
#pragma unroll
    for (int r = 0; r < U; ++r) n[r] = k + U + r < len ? el[(k + U + r) * kSlice] : 0u;
#pragma unroll
    for (int r = 0; r < U; ++r) {
      if (k + r < len) {
        const uint32_t at = e[r] & ((1u << kLineOff) - 1u);
        double2 x[B / 2];
#pragma unroll
        for (int q = 0; q < B / 2; ++q) x[q] = *reinterpret_cast<const double2*>(pl + (size_t)q * ld * 16 + at);
        const double h = *reinterpret_cast<const double*>(vl + (e[r] >> kLineOff));
#pragma unroll
        for (int q = 0; q < B / 2; ++q) {
          acc[2 * q] = fma(h, x[q].x, acc[2 * q]);
          acc[2 * q + 1] = fma(h, x[q].y, acc[2 * q + 1]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < U; ++r) e[r] = n[r];
  }
}

// The rows of a row tile: listed where the impurity terms' tables need whole
// runs of rows together, else B consecutive ones.
template <int B>
struct Rows {
  int u[B], n;
  __device__ __forceinline__ Rows(const HvStepParams& p, int tile) {
    if (B == 4 && p.row_tiles) {
      n = 0;
#pragma unroll
      for (int r = 0; r < B; ++r) {
        u[r] = p.row_tiles[4 * tile + r];
        n += u[r] >= 0 ? 1 : 0;
      }
    } else {
      n = min(B, p.Dup - tile * B);
#pragma unroll
      for (int r = 0; r < B; ++r) u[r] = tile * B + r;
    }
#pragma unroll
    for (int r = 0; r < B; ++r)
      if (r >= n) u[r] = u[0];
  }
};

// (the slot's row for a lane-dependent slot)
template <int B>
__device__ __forceinline__ int row_of(const Rows<B>& R, int r) {
  int u = R.u[0];
#pragma unroll
  for (int q = 1; q < B; ++q) u = r == q ? R.u[q] : u;
  return u;
}

// Impurity terms of basis state d: acc[r] += sum over the terms of (a_r, b)
// of c * V[partner], from memory.
template <int B>
__device__ __forceinline__ void kan_terms(const HvParams& p, const View& o, const Rows<B>& R, const int (&a)[B], int b,
                                          int na, int d, double (&acc)[B]) {
#pragma unroll
  for (int r = 0; r < B; ++r) {
    if (r >= R.n) break;
    const int* kp = p.kan_ptr + a[r] * na + b;
    const int64_t at = (int64_t)R.u[r] * p.Ddn + d;
    for (int q = kp[0]; q < kp[1]; ++q) acc[r] = fma(p.kan_c[q], o.V[at + p.kan_off[q]] * o.vs, acc[r]);
  }
}

// The same in a tile of whole runs (DevSector::row_tiles): the states sharing
// their bath bits are neighbouring rows, so every partner is in LDS, and the
// rows a term leads to are the same for all states of a row.  The rows' reads
// are in flight together.
template <int B>
__device__ __forceinline__ void kan_targets(const HvStepParams& p, const double* tc, const int* td, const double* s,
                                            int ld, const int (&a)[B], int b, int na, int n, int d,
                                            double (&acc)[B]) {
  for (int j = 0; j < p.kan_t; ++j) {
    double c[B], x[B];
    int at[B];
#pragma unroll
    for (int r = 0; r < B; ++r) {
      const int q = (a[r] * p.kan_t + j) * na + b;
      c[r] = r < n ? tc[q] : 0.0;
      at[r] = row_tile_entry(r, n, td[q]);  // 8 * (state offset) + kOwnState + (row offset)
    }
#pragma unroll
    for (int r = 0; r < B; ++r) {
      const int rr = r + (at[r] & 7) - kOwnState;  // the partner's row in the tile
      x[r] = s[((size_t)(rr >> 1) * ld + d + (at[r] >> 3)) * 2 + (rr & 1)];
    }
    // (a state without this term must not pick up 0 * infinity)
#pragma unroll
    for (int r = 0; r < B; ++r) acc[r] = c[r] != 0.0 ? fma(c[r], x[r], acc[r]) : acc[r];
  }
}

// The work-groups of a launch stay and take tiles in turn; while a tile is
// worked on, the lines of the work-group's next tile are on their way into
// registers (NI basis states x B lines per thread), so that neither waits for
// the other: a tile of four 3432-element lines takes most of a CU's LDS, and
// one work-group per CU has no other one to fill the wait.
template <int B, int NI>
struct Ahead {
  double x[NI][B];
};

// The thread's index as a value of this tile: what depends on it is computed
// in every tile instead of being kept in registers over all of them.
__device__ __forceinline__ int fresh_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// Tables of a row tile in LDS after its lines: the value table, the impurity
// terms (coefficients, then state offsets), the rows' cross-term vectors (one
// value per row and site, CROSS_GENERAL).
template <int B>
struct RowTables {
  double *vals, *kc, *ct;
  int* kd;
  int nk;  // impurity-term table entries staged
  __device__ __forceinline__ RowTables(const LinesJob& J, double* s, int ld) {
    const HvStepParams& p = J.p;
    const int na = 1 << (p.Ns - p.nb);
    vals = s + (size_t)B * ld;
    nk = B == 4 && J.kan && p.row_tiles ? na * na * p.kan_t : 0;
    kc = vals + p.nvals;
    kd = reinterpret_cast<int*>(kc + nk);
    ct = kc + nk + (nk + 1) / 2;
  }
};

template <int B, int NI>
__device__ __forceinline__ void row_fetch(const LinesJob& J, const View& o, int tile, Ahead<B, NI>& f, int i0,
                                          int i1) {
  const HvStepParams& p = J.p;
  const int D = p.Ddn;
  const Rows<B> R(p, tile);
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (i < i0 || i >= i1) continue;
    const int d = threadIdx.x + i * blockDim.x;
#pragma unroll
    for (int r = 0; r < B; ++r) f.x[i][r] = d < D && r < R.n ? o.V[(size_t)R.u[r] * D + d] : 0.0;
  }
}

// One row tile whose lines are in f; the next tile's (tn, when there are more)
// are fetched into f on the way.
template <int B, int NI>
__device__ __forceinline__ void row_tile(const LinesJob& J, const View& o, int tile, bool tables, bool more, int tn,
                                         Ahead<B, NI>& f, double* s, double* s_red) {
  const HvStepParams& p = J.p;
  const int D = p.Ddn, T = blockDim.x;
  const int tid = fresh_tid();
  const int ld = D + 1;
  const Rows<B> R(p, tile);
  const int na = 1 << (p.Ns - p.nb);
  // the accumulated input is read here unless it is w itself (then the
  // column pass has read it)
  const bool accum = o.accum && o.Wp != o.W;
  const RowTables<B> t(J, s, ld);
  if (tables) {
    for (int i = tid; i < p.nvals; i += T) t.vals[i] = p.values[i];
    for (int i = tid; i < t.nk; i += T) {
      t.kc[i] = p.kan_tc[i];
      t.kd[i] = p.kan_td[i];
    }
  }
  if (tid < B) s[((size_t)(tid >> 1) * ld + D) * 2 + (tid & 1)] = 0.0;  // the padding entries' state
  if (J.cross == CROSS_GENERAL)
    for (int i = tid; i < p.Ns * B; i += T)
      t.ct[i] = p.cross_rowtab[(size_t)row_of(R, i % B) * p.Ns + i / B];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int d = tid + i * T;
    if (d < D) {
#pragma unroll
      for (int r = 0; r < B; ++r) f.x[i][r] *= o.vs;
      put_state<B>(s, ld, d, f.x[i]);
    }
  }
  __syncthreads();
  int bu[B], au[B];
  double eu[B];
#pragma unroll
  for (int r = 0; r < B; ++r) {
    bu[r] = p.up_bits[R.u[r]];
    au[r] = bu[r] >> p.nb;
    eu[r] = p.up_e[R.u[r]];
  }
  double dsum = 0.0;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int d = tid + i * T;
    if (d < D) {
      double acc[B], x[B], cr[B], wv[B];
      // the column pass's part and the accumulated input: issued here, added
      // last (the first group of entries waits for them with its own loads)
#pragma unroll
      for (int r = 0; r < B; ++r) wv[r] = r < R.n ? o.W[(int64_t)R.u[r] * D + d] : 0.0;
      if (accum) {
#pragma unroll
        for (int r = 0; r < B; ++r)
          if (r < R.n) wv[r] = fma(o.ws, __builtin_nontemporal_load(o.Wp + (int64_t)R.u[r] * D + d), wv[r]);
      }
      const int bd = p.dn_bits[d];
      const double ed = p.dn_e[d];
#pragma unroll
      for (int r = 0; r < B; ++r) cr[r] = 0.0;
      if (J.cross == CROSS_POPC) {
#pragma unroll
        for (int r = 0; r < B; ++r) cr[r] = p.cross_u * (double)__builtin_popcount(bu[r] & bd);
      } else if (J.cross == CROSS_IMP) {
#pragma unroll
        for (int r = 0; r < B; ++r) cr[r] = p.cross_imp[au[r] * na + (bd >> p.nb)];
      } else if (J.cross == CROSS_GENERAL) {
        // one walk over the state's electrons for all rows
        for (unsigned m = (unsigned)bd; m; m &= m - 1) {
          const double* c = t.ct + (size_t)__builtin_ctz(m) * B;
#pragma unroll
          for (int r = 0; r < B; ++r) cr[r] += c[r];
        }
      }
      get_state<B>(s, ld, d, x);
#pragma unroll
      for (int r = 0; r < B; ++r) acc[r] = (eu[r] + ed + cr[r]) * x[r];
      gather_line<B, B == 4 && NI == 1 ? 8 : 4>(s, ld, t.vals, p.dn_slptr, p.dn_sllen, p.dn_lell, d, acc);
      if (J.kan) {
        if (t.nk) kan_targets<B>(p, t.kc, t.kd, s, ld, au, bd >> p.nb, na, R.n, d, acc);
        else kan_terms<B>(p, o, R, au, bd >> p.nb, na, d, acc);
      }
#pragma unroll
      for (int r = 0; r < B; ++r)
        if (r < R.n) {
          acc[r] += wv[r];
          __builtin_nontemporal_store(acc[r], o.W + (int64_t)R.u[r] * D + d);
          dsum = fma(x[r], acc[r], dsum);
        }
    }
    // the next tile's lines behind the first half of this tile's states
    __builtin_amdgcn_sched_barrier(0);
    if (more) {
      if (NI == 1) row_fetch<B, NI>(J, o, tn, f, 0, 1);
      else if (i < NI / 2) row_fetch<B, NI>(J, o, tn, f, 2 * i, 2 * i + 2);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (p.dot_partial) block_reduce_store(dsum, s_red, p.dot_partial + tile);
  __syncthreads();  // the next tile's lines replace this one's
}

// B consecutive lanes read the B columns of a row: a load instruction touches
// 64 / B rows.  Load q of thread t is element q T + t of the D x B tile.
template <int B, int NI>
__device__ __forceinline__ void col_fetch(const LinesJob& J, const View& o, int c0, Ahead<B, NI>& f, int i0,
                                          int i1) {
  const HvStepParams& p = J.p;
  const int nc = min(B, p.Ddn - c0);
  const int c = threadIdx.x % B, row0 = threadIdx.x / B, rstep = blockDim.x / B;
  const double* __restrict__ src = o.V + c0;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (i < i0 || i >= i1) continue;
#pragma unroll
    for (int r = 0; r < B; ++r) {
      const int d = row0 + (i * B + r) * rstep;
      f.x[i][r] = d < p.Dup && c < nc ? src[(size_t)d * p.Ddn + c] : 0.0;
    }
  }
}

// LDS of a column tile after its lines: the value table, then 64 x B results
// per wavefront.
template <int B, int NI>
__device__ __forceinline__ void col_tile(const LinesJob& J, const View& o, int c0, bool tables, bool more, int cn,
                                         Ahead<B, NI>& f, double* s) {
  const HvStepParams& p = J.p;
  const int D = p.Dup, T = blockDim.x;
  const int tid = fresh_tid();
  const int ld = D + 1;
  const int nc = min(B, p.Ddn - c0);
  const bool accum = o.accum && o.Wp == o.W;
  double* s_vals = s + (size_t)B * ld;
  if (tables)
    for (int i = tid; i < p.nvals; i += T) s_vals[i] = p.values[i];
  const int c = tid % B;
  if (tid < B) s[((size_t)(tid >> 1) * ld + D) * 2 + (tid & 1)] = 0.0;  // the padding entries' state
  {
    const int row0 = tid / B, rstep = T / B;
    double* const sc = s + ((size_t)(c >> 1) * ld * 2 + (c & 1));
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int r = 0; r < B; ++r) {
        const int d = row0 + (i * B + r) * rstep;
        if (d < D) sc[(size_t)d * 2] = f.x[i][r] * o.vs;
      }
  }
  __syncthreads();
  const int lane = tid & 63;
  double* const t = s_vals + ((p.nvals + 1) & ~1) + (size_t)(tid >> 6) * (64 * B);
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    // whole wavefronts: lanes past the last row work on it again
    const int d1 = tid + i * T;
    if (d1 - lane < D) {
      const int d = min(d1, D - 1);
      double acc[B];
#pragma unroll
      for (int r = 0; r < B; ++r) acc[r] = accum && r < nc ? o.ws * o.W[(size_t)d * p.Ddn + c0 + r] : 0.0;
      gather_line<B, B == 4 ? 8 : 4>(s, ld, s_vals, p.up_slptr, p.up_sllen, p.up_lell, d, acc);
      // the wavefront's 64 x B results turn through its own piece of LDS, so
      // that B consecutive lanes store the B columns of a row (one request
      // per row instead of B / 2: the pass is 129 -> 111 us on the 14-site
      // Kanamori sector)
#pragma unroll
      for (int q = 0; q < B / 2; ++q)
        reinterpret_cast<double2*>(t)[lane * (B / 2) + q] = make_double2(acc[2 * q], acc[2 * q + 1]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int q = 0; q < B; ++q) {
        const int l = q * 64 + lane, row = d1 - lane + l / B;
        if (row < D && c < nc) o.W[(size_t)row * p.Ddn + c0 + c] = t[l];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) {
      if (NI == 1) col_fetch<B, NI>(J, o, cn, f, 0, 1);
      else if (i < NI / 2) col_fetch<B, NI>(J, o, cn, f, 2 * i, 2 * i + 2);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();  // the next tile's lines replace this one's
}

struct LinesArgs {
  LinesJob j[kLinesMax];
};

// Operand blockIdx.y: row tiles blockIdx.x, blockIdx.x + gridDim.x, ...
template <int B, int NI>
__global__ __launch_bounds__(1024) void hv_row_lines_kernel(LinesArgs a, int ntiles) {
  extern __shared__ double s_line[];
  __shared__ double s_red[16];
  const LinesJob& j = a.j[blockIdx.y];
  const View o = view_of(j.p, HvScales(j.p, s_red));
  if (!o.live) return;
  Ahead<B, NI> f;
  int t = blockIdx.x;
  if (t < ntiles) row_fetch<B, NI>(j, o, t, f, 0, NI);
  for (bool first = true; t < ntiles; first = false) {
    const int n = t + gridDim.x;
    row_tile<B, NI>(j, o, t, first, n < ntiles, n, f, s_line, s_red);
    t = n;
  }
}

// Consecutive column tiles share the 128-byte lines of every row: they go to
// one XCD (work-groups are dealt to the eight XCDs in turn; the grid is a
// multiple of eight).
template <int B, int NI>
__global__ __launch_bounds__(1024) void hv_col_lines_kernel(LinesArgs a, int ntiles, int per) {
  extern __shared__ double s_line[];
  __shared__ double s_red[16];
  const LinesJob& j = a.j[blockIdx.y];
  const HvScales sc(j.p, s_red);
  const View o = view_of(j.p, sc);
  const int x = blockIdx.x & 7, step = gridDim.x >> 3;
  const int t1 = o.live ? min(ntiles, (x + 1) * per) : 0;  // this XCD's tiles: [x per, t1)
  Ahead<B, NI> f;
  int t = x * per + (blockIdx.x >> 3);
  if (t < t1) col_fetch<B, NI>(j, o, t * B, f, 0, NI);
  for (bool first = true; t < t1; first = false) {
    const int n = t + step;
    col_tile<B, NI>(j, o, t * B, first, n < t1, n * B, f, s_line);
    t = n;
  }
  if (blockIdx.x == 0) HvScales::record(j.p, sc.v, sc.beta, sc.live);
}

// Work-groups that stay on the chip for a launch: as many as the CUs hold at
// this LDS and work-group size, a multiple of eight.
int stay_grid(int64_t ntiles, int block, size_t smem) {
  const int per_cu = (int)std::min<size_t>(std::max<size_t>(1, (lds_budget() + 1024) / (smem + 1024)),
                                           std::max(1, 2048 / block));
  return (int)std::min<int64_t>((ntiles + 7) / 8 * 8, (int64_t)256 * per_cu);
}

void allow_lds(const void* k, size_t smem) {
  if (smem > 64 * 1024)
    EDH_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
}

size_t pair_up(size_t n) { return (n + 1) & ~size_t(1); }

size_t row_smem(const DevSector& ds, int B) {
  size_t d = (size_t)B * (ds.dn.D + 1) + (size_t)ds.nvalues;
  if (ds.n_row_tiles > 0 && B == 4) {
    const size_t nk = ((size_t)1 << (2 * ds.kan_ml)) * ds.kan_t;
    d += nk + (nk + 1) / 2;
  }
  if (ds.cross_mode == CROSS_GENERAL) d += (size_t)B * ds.Ns;
  return pair_up(d) * sizeof(double);
}

size_t col_smem(const DevSector& ds, int B, int block) {
  return ((size_t)B * (ds.up.D + 1) + pair_up(ds.nvalues) + (size_t)block * B) * sizeof(double);
}

// Threads of a work-group for lines of D states: as few rounds as 1024 threads
// allow, split evenly.
int hv_lines_threads(int64_t D) {
  const int64_t it = (D + 1023) / 1024;
  return (int)std::max<int64_t>(64, ((D + it - 1) / std::max<int64_t>(it, 1) + 63) / 64 * 64);
}

int row_tiles(const DevSector& ds, const HvLinesPlan& L) {
  return L.row_b == 4 && ds.n_row_tiles > 0 ? ds.n_row_tiles : (int)((ds.up.D + L.row_b - 1) / L.row_b);
}
}  // namespace

HvLinesPlan hv_lines_plan(const DevSector& ds) {
  HvLinesPlan L;
  L.row_block = hv_lines_threads(ds.dn.D);
  L.col_block = hv_lines_threads(ds.up.D);
  const size_t room = lds_budget();
  for (L.row_b = 4; L.row_b >= 2; L.row_b /= 2)
    if (ds.dn.D * L.row_b <= 16 * 1024 && (L.row_smem = row_smem(ds, L.row_b)) <= room) break;
  for (L.col_b = 4; L.col_b >= 2; L.col_b /= 2)
    if (ds.up.D * L.col_b <= 16 * 1024 && (L.col_smem = col_smem(ds, L.col_b, L.col_block)) <= room) break;
  L.ok = ds.lines && ds.N > 0 && L.row_b >= 2 && L.col_b >= 2;
  return L;
}

int hv_lines_partials(const DevSector& ds) {
  const HvLinesPlan L = hv_lines_plan(ds);
  return L.ok ? row_tiles(ds, L) : 0;
}

// The two passes against the single pass for one operand: the hops of both
// spins per state from which on they are faster, by what the single pass's
// entry costs to decode (signed, compact, plain).  In place (w = H v + w) the
// column pass reads w in pieces of 32 bytes, so it takes more.  Measured
// (MI355X, single pass / two passes at hops, in place behind the comma; rings
// of one to four neighbours, tori, impurities of one to three orbitals,
// disordered):
//   four lines at a time, 0.6 to 2.5 M states: signed 924 x 924 1.02, 0.87 at 39
//     and 1.22, 1.05 at 66; compact 0.89, 0.76 at 26, 1.10, 0.94 at 39, 1.26,
//     1.08 at 52; plain 1.11, 0.92 at 26, 1.29, 1.07 at 39, Kanamori 1.23, 1.04
//     at 30, disordered 1.47, 1.24 at 29
//   below that two launches are most of the time: 495 x 924 and 924 x 495 0.74
//     to 1.03, in place 0.56 to 0.97 at any hops; 715 x 715 signed 0.96, compact
//     1.05, plain 1.16 at 48, disordered (general cross term) 1.31, 1.16 at 29
//   from 2.5 M on: signed 2002 x 2002 1.00, 0.84 at 21, 1.14, 0.96 at 28, 1.38,
//     1.17 at 42 (3432 x 3432 1.14, 0.95 at 23, 1.31, 1.10 at 30); compact 0.87,
//     0.72 at 14, 1.24, 1.04 at 28; plain 1.08, 0.89 at 14, 1.42, 1.17 at 28
//     (3003 x 3003 and 3432 x 3432 1.42 to 1.6, 1.11 to 1.24 at 14)
//     Calls of several contexts, on streams of their own, overlap, and the single
//     pass gains more by it where rows are many and short: signed 3432 x 2002
//     0.89 at 22 (1.04 one after the other), 1.14 at 29, 3003 x 2002 0.91 at 22,
//     1.16 at 29; compact 0.82 at 14, 1.28 at 29; plain 0.96 to 0.99 at 13 (1.12
//     to 1.16 one after the other); 2002 x 3003 and square ones 1.06 to 1.26
//   one spin two lines at a time (3003 x 6435, 6435 x 3003): signed 0.96 to
//     1.00, 0.84 to 0.89 at 30, 1.16, 1.03 at 45; compact 1.13, 0.97 at 30, 1.30,
//     1.13 at 45; plain 1.37, 1.18 at 30
//   both spins (5005 .. 8008): signed 0.83 to 0.94, 0.68 to 0.82 at 32, 1.04 to
//     1.12, 0.89 to 0.99 at 48, 1.02 to 1.12 in place at 63; compact 0.96, 0.78 at
//     32, 1.12, 0.95 at 47, 1.21, 1.08 at 63; plain 1.14, 0.94 at 31, 1.31, 1.11
//     at 47
bool hv_lines_faster(const DevSector& ds, bool in_place) {
  if (ds.N < kLinesMin) return false;
  const HvLinesPlan L = hv_lines_plan(ds);
  if (!L.ok) return false;
  static const double small[2][3] = {{39, 36, 28}, {56, 45, 34}};
  static const double large[2][3] = {{21, 20, 12}, {34, 28, 22}};
  static const double tall[3] = {27, 23, 18};
  static const double mixed[2][3] = {{36, 30, 30}, {45, 36, 30}};
  static const double pairs[2][3] = {{46, 40, 30}, {62, 54, 40}};
  const int q = in_place ? 1 : 0, f = ds.dn_form;
  const bool general = f == 2 && ds.cross_mode == CROSS_GENERAL;
  if (L.row_b < 4 && L.col_b < 4) return ds.hops >= pairs[q][f];
  if (L.row_b < 4 || L.col_b < 4) return ds.hops >= mixed[q][f];
  if (ds.N >= 2500000) {
    if (!in_place && 4 * ds.up.D > 5 * ds.dn.D) return ds.hops >= tall[f];
    return ds.hops >= (in_place && f == 2 && ds.N >= 9000000 ? 12 : large[q][f]);
  }
  if (ds.N < 600000) return general && ds.hops >= 28;
  // (the single pass's terms beyond the hopping make up for six hops)
  return ds.hops >= (in_place && f == 2 && (general || ds.kan_ml > 0) ? 28 : small[q][f]);
}

void launch_hv_lines(const DevSector& ds, const HvArgs* ops, int count, hipStream_t s) {
  const HvLinesPlan L = hv_lines_plan(ds);
  EDH_CHECK(L.ok && ds.two_pass, EDH_ERR_INTERNAL, "H*v lines: the sector has no tables for them");
  EDH_CHECK(count >= 1 && count <= kLinesMax, EDH_ERR_INTERNAL, "H*v lines: operand count");
  LinesArgs a;
  for (int q = 0; q < count; ++q) {
    a.j[q].p = make_step_params(ds, ops[q]);
    a.j[q].cross = ds.cross_mode;
    a.j[q].kan = ds.kan_ml > 0 ? 1 : 0;
  }
  for (int q = count; q < kLinesMax; ++q) a.j[q] = a.j[0];
  const bool r1 = ds.dn.D <= 1024, c1 = ds.up.D <= 1024;
  auto kr = L.row_b == 2 ? hv_row_lines_kernel<2, 8> : r1 ? hv_row_lines_kernel<4, 1> : hv_row_lines_kernel<4, 4>;
  auto kc = L.col_b == 2 ? hv_col_lines_kernel<2, 8> : c1 ? hv_col_lines_kernel<4, 1> : hv_col_lines_kernel<4, 4>;
  allow_lds((const void*)kr, L.row_smem);
  allow_lds((const void*)kc, L.col_smem);
  const int ct = (int)((ds.dn.D + L.col_b - 1) / L.col_b), per = (ct + 7) / 8;
  hipLaunchKernelGGL(kc, dim3(stay_grid(ct, L.col_block, L.col_smem), count), dim3(L.col_block), L.col_smem, s, a, ct,
                     per);
  const int rt = row_tiles(ds, L);
  hipLaunchKernelGGL(kr, dim3(stay_grid(rt, L.row_block, L.row_smem), count), dim3(L.row_block), L.row_smem, s, a, rt);
  EDH_HIP(hipGetLastError());
}

}  // namespace edh
