// Upload of one sector's tables to the device.
#include <algorithm>
#include <cstdint>
#include <cstring>
#include <functional>
#include <mutex>

#include "hv_params.h"

namespace edh {

namespace {

// All tables of a sector go to the device as one allocation and one copy:
// the host arrays are first packed (256-byte aligned) into one blob, and
// the device pointers are set once the blob has its device address.
class Packer {
 public:
  template <class T>
  void add(T*& field, const std::vector<T>& h) {
    field = nullptr;
    if (h.empty()) return;
    const size_t off = (blob_.size() + 255) & ~size_t(255);
    blob_.resize(off + h.size() * sizeof(T));
    std::memcpy(blob_.data() + off, h.data(), h.size() * sizeof(T));
    set_.push_back([&field, off](char* base) { field = reinterpret_cast<T*>(base + off); });
  }
  // Without a stage the blob must stay alive until the copy has completed
  // (the caller synchronises the stream); with one the copy reads pinned
  // staging memory that the stage keeps until the copy is done.
  void commit(DevSector& ds, hipStream_t s, UploadStage* stage) {
    if (blob_.empty()) return;
    void* p = nullptr;
    check_alloc(hipMallocAsync(&p, blob_.size(), s), "hipMallocAsync");
    ds.allocs.push_back(p);
    if (stage) {
      int c = -1;
      char* h = stage->take(blob_.size(), c);
      std::memcpy(h, blob_.data(), blob_.size());
      EDH_HIP(hipMemcpyAsync(p, h, blob_.size(), hipMemcpyHostToDevice, s));
      stage->mark(c, s);
    } else {
      EDH_HIP(hipMemcpyAsync(p, blob_.data(), blob_.size(), hipMemcpyHostToDevice, s));
    }
    for (auto& f : set_) f(static_cast<char*>(p));
  }

 private:
  std::vector<char> blob_;
  std::vector<std::function<void(char*)>> set_;
};

// The sliced ELL's slots as line-pass entries (kLineOff), padding slots at the
// zero state after the line.
std::vector<uint32_t> line_entries(const SpinTables& sp) {
  std::vector<uint32_t> out(sp.ell.size());
  for (size_t q = 0; q < out.size(); ++q)
    out[q] = ((sp.ell_pad[q] ? (uint32_t)sp.D : sp.ell[q] & kColMask) << 4) |
             ((sp.ell[q] >> kColBits) << (kLineOff + 3));
  return out;
}

void upload_spin(Packer& pk, const SpinTables& sp, DevSpin& d) {
  d.D = sp.D;
  pk.add(d.bits, sp.bits);
  pk.add(d.ediag, sp.ediag);
  pk.add(d.rowp, sp.rowp);
  pk.add(d.packed, sp.packed);
  pk.add(d.sl_ptr, sp.sl_ptr);
  pk.add(d.sl_len, sp.sl_len);
  pk.add(d.ell, sp.ell);
  for (int q = 0; q < 4; ++q) d.vt16[q] = sp.vt16[q];
  d.nvt16 = sp.nvt16;
  pk.add(d.q4_ptr, sp.q4_ptr);
  pk.add(d.ell_q4, sp.ell_q4);
  pk.add(d.ell_s4, sp.ell_s4);
  d.s4_scale = sp.s4_scale;
  d.max_hops = 0;
  for (size_t r = 0; r + 1 < sp.rowp.size(); ++r) d.max_hops = std::max(d.max_hops, sp.rowp[r + 1] - sp.rowp[r]);
}

// Reverse Cuthill-McKee order of the graph whose adjacency is the CSR
// structure (rows and columns are basis states of one spin): breadth-first
// from a minimum-degree vertex of each component, neighbours by increasing
// degree, then reversed.
std::vector<int32_t> rcm_order(const std::vector<int32_t>& rowp, const std::vector<int32_t>& col, int64_t n) {
  std::vector<int32_t> deg(n), order;
  order.reserve(n);
  for (int64_t i = 0; i < n; ++i) deg[i] = rowp[i + 1] - rowp[i];
  std::vector<char> seen(n, 0);
  std::vector<int32_t> byDeg(n);
  for (int64_t i = 0; i < n; ++i) byDeg[i] = (int32_t)i;
  std::stable_sort(byDeg.begin(), byDeg.end(), [&](int32_t a, int32_t b) { return deg[a] < deg[b]; });
  std::vector<int32_t> nb;
  for (int32_t start : byDeg) {
    if (seen[start]) continue;
    size_t head = order.size();
    order.push_back(start);
    seen[start] = 1;
    while (head < order.size()) {
      const int32_t x = order[head++];
      nb.clear();
      for (int q = rowp[x]; q < rowp[x + 1]; ++q)
        if (!seen[col[q]]) {
          seen[col[q]] = 1;
          nb.push_back(col[q]);
        }
      std::stable_sort(nb.begin(), nb.end(), [&](int32_t a, int32_t b) { return deg[a] < deg[b]; });
      order.insert(order.end(), nb.begin(), nb.end());
    }
  }
  std::reverse(order.begin(), order.end());
  return order;
}

}  // namespace

// A run of rows sharing their bath bits has C(ml, k) <= 3 rows for up to
// three orbitals; a tile takes a run of several rows and fills up with single
// ones.
RowTileTables row_tile_tables(const SectorTables& st, int Ns) {
  RowTileTables out;
  const int ml = st.kan_ml, na = 1 << ml, nb = Ns - ml;
  if (ml < 1 || ml > 3) return out;
  std::vector<std::vector<int>> tgt(na);
  int nt = 0;
  for (int a = 0; a < na; ++a) {
    for (int q = st.kan_ptr[a * na]; q < st.kan_ptr[(a + 1) * na]; ++q)
      if (std::find(tgt[a].begin(), tgt[a].end(), st.kan[q].new_a) == tgt[a].end()) tgt[a].push_back(st.kan[q].new_a);
    nt = std::max(nt, (int)tgt[a].size());
  }
  if (nt == 0) return out;
  std::vector<int32_t> td((size_t)na * nt * na, kOwnState);
  std::vector<double> tc(td.size(), 0.0);
  for (int a = 0; a < na; ++a)
    for (int b = 0; b < na; ++b)
      for (int q = st.kan_ptr[a * na + b]; q < st.kan_ptr[a * na + b + 1]; ++q) {
        const size_t j = std::find(tgt[a].begin(), tgt[a].end(), st.kan[q].new_a) - tgt[a].begin();
        const size_t at = ((size_t)a * nt + j) * na + b;
        if (tc[at] != 0.0) return out;  // two terms of (a, b) lead to this up pattern
        const int32_t lu = (int32_t)((1ll << (st.nup - __builtin_popcount(a))) - 1);
        const int32_t ld = (int32_t)((1ll << (st.ndn - __builtin_popcount(b))) - 1);
        const int du = st.up.rank[lu | (st.kan[q].new_a << nb)] - st.up.rank[lu | (a << nb)];
        const int dd = st.dn.rank[ld | (st.kan[q].new_b << nb)] - st.dn.rank[ld | (b << nb)];
        if (du < -2 || du > 2) return out;
        td[at] = 8 * dd + kOwnState + du;
        tc[at] = st.kan[q].coef;
      }
  // runs of rows with the same bath bits
  const int32_t bath = (int32_t)((1ll << nb) - 1);
  std::vector<int32_t> single, tiles;
  for (int64_t u = 0; u < st.up.D;) {
    int64_t e = u + 1;
    while (e < st.up.D && (st.up.bits[e] & bath) == (st.up.bits[u] & bath)) ++e;
    if (e - u > 4) return out;
    if (e - u == 1) {
      single.push_back((int32_t)u);
    } else {
      for (int k = 0; k < 4; ++k) tiles.push_back(u + k < e ? (int32_t)(u + k) : -1);
    }
    u = e;
  }
  size_t next = 0;
  for (int32_t& t : tiles)
    if (t < 0 && next < single.size()) t = single[next++];
  while (next < single.size())
    for (int k = 0; k < 4; ++k) tiles.push_back(next < single.size() ? single[next++] : -1);
  out.t = nt;
  out.tiles = std::move(tiles);
  out.td = std::move(td);
  out.tc = std::move(tc);
  return out;
}

void DevSector::release() {
  for (void* p : allocs) (void)hipFreeAsync(p, astream);
  allocs.clear();
  *this = DevSector();
}

void configure_mem_pool(int device) {
  static bool done[64] = {false};
  if (device < 0 || device >= 64 || done[device]) return;
  hipMemPool_t pool;
  EDH_HIP(hipDeviceGetDefaultMemPool(&pool, device));
  uint64_t keep = UINT64_MAX;
  EDH_HIP(hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep));
  done[device] = true;
}

namespace {
std::mutex g_pinned_mu;
std::vector<std::pair<double*, size_t>> g_pinned_free;  // (buffer, capacity in doubles)
constexpr size_t kPinnedKept = 64, kPinnedLargest = size_t(1) << 22;  // buffers, doubles
}  // namespace

double* pinned_take(size_t need, size_t& cap) {
  {
    std::lock_guard<std::mutex> lk(g_pinned_mu);
    size_t best = g_pinned_free.size();
    for (size_t q = 0; q < g_pinned_free.size(); ++q)
      if (g_pinned_free[q].second >= need &&
          (best == g_pinned_free.size() || g_pinned_free[q].second < g_pinned_free[best].second))
        best = q;
    if (best < g_pinned_free.size()) {
      const auto r = g_pinned_free[best];
      g_pinned_free.erase(g_pinned_free.begin() + (std::ptrdiff_t)best);
      cap = r.second;
      return r.first;
    }
  }
  double* h = nullptr;
  EDH_HIP(hipHostMalloc((void**)&h, need * sizeof(double)));
  cap = need;
  return h;
}

void pinned_give(double* h, size_t cap) {
  if (cap <= kPinnedLargest) {
    std::lock_guard<std::mutex> lk(g_pinned_mu);
    if (g_pinned_free.size() < kPinnedKept) {
      g_pinned_free.push_back({h, cap});
      return;
    }
  }
  (void)hipHostFree(h);
}

char* UploadStage::take(size_t bytes, int& c) {
  // a chunk with room, else one whose copies have all completed, else a new one
  for (size_t q = 0; q < chunks.size(); ++q)
    if (chunks[q].cap - chunks[q].used >= bytes) {
      c = (int)q;
      char* h = chunks[q].host + chunks[q].used;
      chunks[q].used = (chunks[q].used + bytes + 255) & ~size_t(255);
      return h;
    }
  for (size_t q = 0; q < chunks.size(); ++q)
    if (chunks[q].cap >= bytes && hipEventQuery(chunks[q].ev) == hipSuccess) {
      c = (int)q;
      chunks[q].used = (bytes + 255) & ~size_t(255);
      return chunks[q].host;
    }
  Chunk k;
  k.cap = std::max<size_t>(size_t(16) << 20, bytes);
  EDH_HIP(hipHostMalloc((void**)&k.host, k.cap, hipHostMallocDefault));
  EDH_HIP(hipEventCreateWithFlags(&k.ev, hipEventDisableTiming));
  k.used = (bytes + 255) & ~size_t(255);
  chunks.push_back(k);
  c = (int)chunks.size() - 1;
  return k.host;
}

void UploadStage::mark(int c, hipStream_t s) { EDH_HIP(hipEventRecord(chunks[c].ev, s)); }

void UploadStage::release() {
  for (Chunk& k : chunks) {
    if (k.host) (void)hipHostFree(k.host);
    if (k.ev) (void)hipEventDestroy(k.ev);
  }
  chunks.clear();
}

namespace {

// Geometry of the impurity terms' row tiles (their tables are returned).
RowTileTables set_row_tiles(const SectorTables& st, DevSector& ds) {
  RowTileTables r;
  if (ds.lines && st.kan_ml > 0) r = row_tile_tables(st, ds.Ns);
  ds.kan_t = r.t;
  ds.n_row_tiles = (int)(r.tiles.size() / 4);
  return r;
}

// Tables of the line passes, or of the tile pass where lines do not fit.
void add_two_pass(Packer& pk, const SectorTables& st, DevSector& ds) {
  const RowTileTables r = set_row_tiles(st, ds);
  if (hv_lines_plan(ds).ok) {
    pk.add(ds.up.lell, line_entries(st.up));
    pk.add(ds.dn.lell, line_entries(st.dn));
    pk.add(ds.row_tiles, r.tiles);
    pk.add(ds.kan_td, r.td);
    pk.add(ds.kan_tc, r.tc);
    return;
  }
  std::vector<int32_t> slices;
  std::vector<uint32_t> in, out;
  up_tile_tables(st.up, slices, in, out);
  pk.add(ds.up_slices, slices);
  pk.add(ds.up_in, in);
  pk.add(ds.up_out, out);
}

}  // namespace

void upload_sector(const SectorTables& st, int Ns, DevSector& ds, hipStream_t s, UploadStage* stage) {
  ds.release();
  ds.astream = s;
  ds.lds_room = lds_budget();
  ds.Ns = Ns;
  ds.nup = st.nup;
  ds.ndn = st.ndn;
  ds.N = st.N;
  ds.imp_ml = st.imp_ml;
  ds.table_bytes = st.table_bytes;
  Packer pk;
  ds.nvalues = (int)st.values.size();
  ds.hops = (double)st.up.col.size() / (double)std::max<int64_t>(st.up.D, 1) +
            (double)st.dn.col.size() / (double)std::max<int64_t>(st.dn.D, 1);
  ds.up.D = st.up.D;
  ds.dn.D = st.dn.D;
  ds.dn_form = !st.dn.ell_s4.empty() ? 0 : !st.dn.ell_q4.empty() ? 1 : 2;
  ds.lines = std::max(st.up.D, st.dn.D) < (1 << (kLineOff - 4)) - 1;
  upload_spin(pk, st.up, ds.up);
  upload_spin(pk, st.dn, ds.dn);
  pk.add(ds.values, st.values);
  ds.cross_mode = st.cross_mode;
  ds.cross_u = st.cross_u;
  pk.add(ds.cross_imp, st.cross_imp);
  pk.add(ds.cross_rowtab, st.cross_rowtab);
  ds.kan_ml = st.kan_ml;
  if (st.kan_ml > 0) {
    // Each impurity term moves the impurity bits (a, b) -> (a', b') with the
    // same occupation counts.  In the basis order (positions in ascending
    // lexicographic order, impurity orbitals on the highest positions) the
    // states sharing their bath bits form one contiguous run ordered by the
    // impurity pattern alone, so the partner of (u, d) is (u + du, d + dd)
    // with du, dd fixed by (a, a') and (b, b'): one element offset per term,
    // du * D_dn + dd, read from the representative state of its group.
    const int ml = st.kan_ml, na = 1 << ml, nb = ds.Ns - ml;
    std::vector<int64_t> koff(st.kan.size());
    std::vector<double> kc(st.kan.size());
    for (int a = 0; a < na; ++a)
      for (int b = 0; b < na; ++b) {
        const int idx = a * na + b;
        if (st.kan_ptr[idx + 1] == st.kan_ptr[idx]) continue;
        const int bath_up = st.nup - __builtin_popcount(a), bath_dn = st.ndn - __builtin_popcount(b);
        const int32_t lu = (int32_t)((1ll << bath_up) - 1), ld = (int32_t)((1ll << bath_dn) - 1);
        const int32_t ru = st.up.rank[lu | (a << nb)], rd = st.dn.rank[ld | (b << nb)];
        for (int q = st.kan_ptr[idx]; q < st.kan_ptr[idx + 1]; ++q) {
          const KanEntry& e = st.kan[q];
          EDH_CHECK(__builtin_popcount(e.new_a) == __builtin_popcount(a) &&
                        __builtin_popcount(e.new_b) == __builtin_popcount(b),
                    EDH_ERR_INTERNAL, "impurity term changes an occupation count");
          const int64_t du = st.up.rank[lu | (e.new_a << nb)] - ru, dd = st.dn.rank[ld | (e.new_b << nb)] - rd;
          koff[q] = du * st.dn.D + dd;
          kc[q] = e.coef;
        }
      }
    pk.add(ds.kan_ptr, st.kan_ptr);
    pk.add(ds.kan_off, koff);
    pk.add(ds.kan_c, kc);
    ds.nkan = (int)kc.size();
    if (st.N >= kLinesMin) (void)set_row_tiles(st, ds);  // the choice below depends on their LDS
  }
  pk.add(ds.row_order, rcm_order(st.up.rowp, st.up.col, st.up.D));
  // the two passes' tables where they are taken by themselves: in a batch by
  // its Lanczos operands, else by the sector's own choice
  const int variant = stage ? HV_SINGLE : hv_choose(ds, false), in_place = stage ? HV_SINGLE : hv_choose(ds, true);
  const bool two_pass =
      ds.N > 0 && (stage ? hv_batch_lines(ds) : variant == HV_TWO_PASS || in_place == HV_TWO_PASS);
  if (two_pass) add_two_pass(pk, st, ds);
  pk.commit(ds, s, stage);
  ds.two_pass = two_pass;
  if (stage) return;
  EDH_HIP(hipStreamSynchronize(s));
  ds.variant = variant;
  ds.variant_in_place = in_place;
}

void hv_two_pass_tables(const SectorTables& st, DevSector& ds, hipStream_t s) {
  if (ds.two_pass || ds.N == 0) return;
  Packer pk;
  add_two_pass(pk, st, ds);
  pk.commit(ds, s, nullptr);
  EDH_HIP(hipStreamSynchronize(s));
  ds.two_pass = true;
}

}  // namespace edh
