// Walks every row tile of a three-orbital impurity sector as the row pass of
// H*v does and prints how many slots hold no row, how many of the partners
// that the slots read lie outside the tile's four rows (or, for a slot with a
// row, outside its rows or the line), and how many tiles there are.
//   row_tiles <sites> <orbitals> <nup> <ndn>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "edh_internal.h"

int main(int argc, char** argv) {
  if (argc != 5) return 2;
  const int Ns = atoi(argv[1]), ml = atoi(argv[2]), nup = atoi(argv[3]), ndn = atoi(argv[4]), nb = Ns - ml;
  std::vector<double> eps(2 * nb, 0.1), vk(2 * ml * nb, 0.3), h0(2 * ml * ml, 0.0), ut(4 * ml * ml * ml * ml, 0.0);
  auto u = [&](int s, int i, int j, int k, int l) -> double& { return ut[(((s * ml + i) * ml + j) * ml + k) * ml + l]; };
  for (int s = 0; s < 4; ++s)
    for (int i = 0; i < ml; ++i) {
      u(s, i, i, i, i) = 4.0;
      for (int j = 0; j < ml; ++j)
        if (i != j) u(s, i, j, i, j) = 2.6, u(s, i, j, j, i) = 0.7, u(s, i, i, j, j) = 0.7;
    }
  edh::Model* m = edh::build_siam(Ns, ml, eps.data(), vk.data(), h0.data(), ut.data(), 1.0);
  edh::SectorTables st;
  edh::build_sector(*m, nup, ndn, st, false);
  const edh::RowTileTables t = edh::row_tile_tables(st, Ns);
  const int na = 1 << ml;
  long empty = 0, outside = 0;
  for (size_t q = 0; q < t.tiles.size(); q += 4) {
    int n = 0;
    for (int r = 0; r < 4; ++r) n += t.tiles[q + r] >= 0;
    empty += 4 - n;
    for (int r = 0; r < 4; ++r) {
      const int a = st.up.bits[t.tiles[q + (r < n ? r : 0)]] >> nb;
      for (int64_t d = 0; d < st.dn.D; ++d)
        for (int j = 0; j < t.t; ++j) {
          const int at = edh::row_tile_entry(r, n, t.td[(a * t.t + j) * na + (st.dn.bits[d] >> nb)]);
          const int row = r + (at & 7) - edh::kOwnState;
          const int64_t state = d + (at >> 3);
          if (row < 0 || row >= 4 || (r < n && row >= n) || state < 0 || state >= st.dn.D) ++outside;
        }
    }
  }
  printf("%ld %ld %zu\n", empty, outside, t.tiles.size() / 4);
  delete m;
  return 0;
}
