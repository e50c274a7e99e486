// The up-spin hopping of sectors whose lines do not fit LDS (hv_lines.hip):
// the second of two passes, after the rows kernel without that term.
//
// The vector V[u][d] is cut into slabs of 64 columns and those into tiles of
// 128 consecutive rows, one tile (64 KB) in LDS per work-group.  Basis states
// are in lexicographic order of their occupied positions, so consecutive ones
// share their low positions and two fifths of the hops stay in the tile (4x4
// torus, 12,870 rows of 17 hops).  Those are LDS reads; the others read the
// row's 512-byte segment from L2 or the memory-side cache.  Every slice of two
// rows has its own two lists of entries, padded to the longer row.
//
// A wavefront works on two rows, two columns per lane.  The grid is one
// work-group per CU (two of them, which LDS would hold, miss L2 for 137 M lines
// instead of 97 M); while a tile is worked on, the work-group's next one is on
// its way into registers, since nothing else would fill the wait.
//
// What bounds it: lines that miss the XCD's L2, 97 M of 183 M (128 bytes each,
// 6 TB/s) on the 4x4 torus, 2.0 ms; a pass that gathered every hop from a slab
// of 16 columns in L2 took 3.5 ms.  Narrower slabs fit L2 but touch more lines
// (a row of 12,870 elements is no multiple of a line) and take more address
// work: 16 columns x 1024 rows 2.44 ms, 32 x 512 2.17 ms, 64 x 256 2.04 ms, 64 x
// 128 2.02 ms (the one here: half the LDS), 128 x 128 2.44 ms.  The whole H*v of
// that sector, one after the other for seconds: 4.8 -> 3.3 ms (from rest 3.8 ->
// 3.3: the single pass's 25 GB of gathers cost clock).
#include <algorithm>

#include "hv_params.h"

namespace edh {

namespace {

constexpr int kTileW = 64;                // columns
constexpr int kTileRows = 128;
constexpr int kPairs = kTileW / 2;        // lanes per row
constexpr int kSliceRows = 64 / kPairs;   // rows per wavefront
constexpr int kTileWG = 1024;
constexpr int kRound = kTileWG / kPairs;  // rows a round covers
constexpr int kTileNI = kTileRows / kRound;
constexpr uint32_t kNoEntry = ~0u;

// Two neighbouring elements; VEC: both exist and their address is a multiple
// of 16 bytes.
typedef double pair_t __attribute__((ext_vector_type(2)));

template <bool VEC>
__device__ __forceinline__ double2 get_pair(const double* q, bool two) {
  if (VEC) return *reinterpret_cast<const double2*>(q);
  return make_double2(q[0], two ? q[1] : 0.0);
}

template <bool VEC>
__global__ __launch_bounds__(kTileWG) void hv_up_tiles_kernel(HvStepParams p, int ntiles, int nslabs, int per) {
  extern __shared__ double s_tile[];  // the tile, a zero row, the value table
  __shared__ double s_red[16];
  const HvScales sc(p, s_red);
  if (!sc.live) return;
  const double vs = sc.v;
  const int Dup = p.Dup, Ddn = p.Ddn;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = tid / kPairs;       // the thread's row of a round
  const int sub = row0 % kSliceRows;        // and in its slice
  double2* const s2 = reinterpret_cast<double2*>(s_tile);
  double* const s_vals = s_tile + (size_t)(kTileRows + 1) * kTileW;
  for (int i = tid; i < p.nvals; i += kTileWG) s_vals[i] = p.values[i];
  if (tid < kTileW) s_tile[(size_t)kTileRows * kTileW + tid] = 0.0;

  // Work-groups are dealt to the eight XCDs in turn; XCD x takes slabs
  // [x per, x per + per) one after the other, neighbouring slabs (which share
  // 128-byte lines) at about the same time.
  const int x = blockIdx.x & 7, step = gridDim.x >> 3;
  const int nt = max(0, min(per, nslabs - x * per)) * ntiles;
  double2 f[kTileNI];
  auto fetch = [&](int t, int i0, int i1) {
    const int c = (x * per + t / ntiles) * kTileW + 2 * (tid % kPairs);
    const int r = (t % ntiles) * kTileRows + row0;
#pragma unroll
    for (int i = 0; i < kTileNI; ++i) {
      if (i < i0 || i >= i1) continue;
      const int row = r + i * kRound;
      f[i] = row < Dup && c < Ddn ? get_pair<VEC>(p.v + (size_t)row * Ddn + c, c + 1 < Ddn) : make_double2(0.0, 0.0);
    }
  };
  double dsum = 0.0;
  int t = blockIdx.x >> 3;
  if (t < nt) fetch(t, 0, kTileNI);
  while (t < nt) {
    const int g0 = (t % ntiles) * kTileRows;
    const int c = (x * per + t / ntiles) * kTileW + 2 * (tid % kPairs);
    const bool one = c < Ddn, two = c + 1 < Ddn;
    const int next = t + step;
#pragma unroll
    for (int i = 0; i < kTileNI; ++i) s2[i * kTileWG + tid] = make_double2(f[i].x * vs, f[i].y * vs);
    __syncthreads();
    const char* const lane_s = reinterpret_cast<const char*>(s2 + (tid % kPairs));
    const char* const vl = reinterpret_cast<const char*>(s_vals);
    const double* const Vc = p.v + c;
#pragma unroll
    for (int i = 0; i < kTileNI; ++i) {
      const int first = g0 + i * kRound + wave * kSliceRows;  // the wavefront's slice
      if (first < Dup) {
        const int4 h = reinterpret_cast<const int4*>(p.up_slices)[first / kSliceRows];
        const int in_len = __builtin_amdgcn_readfirstlane(h.y), out_len = __builtin_amdgcn_readfirstlane(h.w);
        const uint32_t* ei = p.up_in + __builtin_amdgcn_readfirstlane(h.x) + sub;
        const uint32_t* eo = p.up_out + __builtin_amdgcn_readfirstlane(h.z) + sub;
        const int row = g0 + i * kRound + row0;
        const bool live = row < Dup && one;
        double2 wv = make_double2(0.0, 0.0);
        double* const W = p.w + (size_t)row * Ddn + c;
        if (live) {
          if (VEC) {
            const pair_t w2 = __builtin_nontemporal_load(reinterpret_cast<const pair_t*>(W));
            wv = make_double2(w2.x, w2.y);
          } else {
            wv = get_pair<VEC>(W, two);
          }
        }
        double2 a = make_double2(0.0, 0.0), b = make_double2(0.0, 0.0);
        for (int k = 0; k < max(out_len, 1); k += 8) {
          uint32_t e[8];
          double2 y[8];
#pragma unroll
          for (int r = 0; r < 8; ++r) e[r] = k + r < out_len ? eo[(k + r) * kSliceRows] : kNoEntry;
#pragma unroll
          for (int r = 0; r < 8; ++r) {
            y[r] = make_double2(0.0, 0.0);
            if (e[r] != kNoEntry && one) y[r] = get_pair<VEC>(Vc + (size_t)(e[r] & kColMask) * Ddn, two);
          }
          if (k == 0)
            for (int q = 0; q < in_len; q += 4) {
              uint32_t d[4];
#pragma unroll
              for (int r = 0; r < 4; ++r) d[r] = ei[(q + r) * kSliceRows];  // (lists are multiples of four long)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const double2 z = *reinterpret_cast<const double2*>(lane_s + (d[r] & ((1u << kLineOff) - 1u)));
                const double hv = *reinterpret_cast<const double*>(vl + (d[r] >> kLineOff));
                a.x = fma(hv, z.x, a.x);
                a.y = fma(hv, z.y, a.y);
              }
            }
#pragma unroll
          for (int r = 0; r < 8; ++r) {
            const double hv = e[r] != kNoEntry ? s_vals[e[r] >> kColBits] : 0.0;
            b.x = fma(hv, y[r].x, b.x);
            b.y = fma(hv, y[r].y, b.y);
          }
        }
        if (live) {
          const double2 own = s2[i * kTileWG + tid];
          wv.x += fma(b.x, vs, a.x);
          wv.y += fma(b.y, vs, a.y);
          if (VEC) {
            const pair_t w2 = {wv.x, wv.y};
            __builtin_nontemporal_store(w2, reinterpret_cast<pair_t*>(W));
          } else {
            W[0] = wv.x;
            if (two) W[1] = wv.y;
          }
          dsum = fma(own.x, wv.x, dsum);
          if (two) dsum = fma(own.y, wv.y, dsum);
        }
      }
      // the next tile behind the first half of this one's rounds
      if (next < nt && i < kTileNI / 2) fetch(next, 2 * i, 2 * i + 2);
    }
    __syncthreads();  // the next tile replaces this one
    t = next;
  }
  if (p.dot_partial) block_reduce_store(dsum, s_red, p.dot_partial + blockIdx.x);
}

struct TileGrid {
  int ntiles, nslabs, per, grid;
};

TileGrid tile_grid(const DevSector& ds) {
  TileGrid g;
  g.ntiles = (int)((ds.up.D + kTileRows - 1) / kTileRows);
  g.nslabs = (int)((ds.dn.D + kTileW - 1) / kTileW);
  g.per = (g.nslabs + 7) / 8;
  g.grid = 8 * (int)std::min<int64_t>(32, (int64_t)g.per * g.ntiles);
  return g;
}

}  // namespace

// The up spin's entries by slices of two rows, within the row's tile (LDS byte
// offset of the row, value's byte offset above it; padding at the zero row,
// lists a multiple of four long) and outside it (packed as in the CSR form;
// padding kNoEntry).
void up_tile_tables(const SpinTables& sp, std::vector<int32_t>& slices, std::vector<uint32_t>& in,
                    std::vector<uint32_t>& out) {
  const int64_t D = sp.D;
  slices.clear();
  in.clear();
  out.clear();
  std::vector<uint32_t> li[kSliceRows], lo[kSliceRows];
  for (int64_t s = 0; s < D; s += kSliceRows) {
    size_t ni = 0, no = 0;
    for (int q = 0; q < kSliceRows; ++q) {
      li[q].clear();
      lo[q].clear();
      const int64_t u = s + q, t = u / kTileRows;
      if (u >= D) continue;
      for (int k = sp.rowp[u]; k < sp.rowp[u + 1]; ++k) {
        const uint32_t e = sp.packed[k], col = e & kColMask;
        if (col / kTileRows == t)
          li[q].push_back((col % kTileRows) * (kTileW * 8) | (e >> kColBits) << (kLineOff + 3));
        else
          lo[q].push_back(e);
      }
      ni = std::max(ni, li[q].size());
      no = std::max(no, lo[q].size());
    }
    ni = (ni + 3) / 4 * 4;
    const int32_t h[4] = {(int32_t)in.size(), (int32_t)ni, (int32_t)out.size(), (int32_t)no};
    slices.insert(slices.end(), h, h + 4);
    for (size_t k = 0; k < ni; ++k)
      for (int q = 0; q < kSliceRows; ++q) in.push_back(k < li[q].size() ? li[q][k] : (uint32_t)(kTileRows * kTileW * 8));
    for (size_t k = 0; k < no; ++k)
      for (int q = 0; q < kSliceRows; ++q) out.push_back(k < lo[q].size() ? lo[q][k] : kNoEntry);
  }
}

int hv_up_tiles_blocks(const DevSector& ds) { return tile_grid(ds).grid; }

void launch_hv_up_tiles(const DevSector& ds, const HvStepParams& p, hipStream_t s) {
  EDH_CHECK(ds.two_pass && ds.up_slices, EDH_ERR_INTERNAL, "H*v tiles: the sector has no tables for them");
  const TileGrid g = tile_grid(ds);
  const size_t smem = ((size_t)(kTileRows + 1) * kTileW + ds.nvalues) * sizeof(double);
  const bool vec = ds.dn.D % 2 == 0 && ((uintptr_t)p.v | (uintptr_t)p.w) % 16 == 0;
  auto k = vec ? hv_up_tiles_kernel<true> : hv_up_tiles_kernel<false>;
  EDH_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
  hipLaunchKernelGGL(k, dim3(g.grid), dim3(kTileWG), smem, s, p, g.ntiles, g.nslabs, g.per);
  EDH_HIP(hipGetLastError());
}

}  // namespace edh
