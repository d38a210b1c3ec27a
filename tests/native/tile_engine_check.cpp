// Host check of the small-tile engine's work items (pan2_amd/csrc/pm_tiles.hpp):
// xcd_runs is a permutation that keeps an XCD's items in runs, and the tile
// decoders at its row-group sizes cover every tile of an extent once.
#include <cstdio>
#include <vector>

#include "../../pan2_amd/csrc/pm_tiles.hpp"

int main() {
  int bad = 0;
  for (int n = 1; n <= 1500; n += (n < 300 ? 1 : 7)) {
    std::vector<int> seen(n, 0);
    for (int b = 0; b < n; ++b) {
      const int t = pm::xcd_runs<16>(b, n);
      if (t < 0 || t >= n || seen[t]++) {
        if (bad++ < 5) std::printf("xcd_runs n=%d b=%d -> %d\n", n, b, t);
        continue;
      }
      // block b + 8 (the same XCD) takes the next item of the run
      if (b + 8 < n && b % 128 < 120 && (b < n / 128 * 128) == (b + 8 < n / 128 * 128) &&
          pm::xcd_runs<16>(b + 8, n) != t + 1) {
        if (bad++ < 5) std::printf("xcd_runs n=%d b=%d: run broken\n", n, b);
      }
    }
  }
  for (int edge : {64, 128}) {
    for (int m = 129; m <= 1100; m += 31) {
      const int np = pm::mt_edge_tiles(m, edge);
      if ((np - 1) * edge >= m || np * edge < m) ++bad;
      std::vector<int> sym(np * np, 0);
      for (int lt = 0; lt < pm::mt_sym_tiles(m, edge); ++lt) {
        int ti, tj;
        pm::sym_tile(lt, np, ti, tj, 512 / edge);
        if (ti < 0 || tj >= np || ti > tj || sym[ti * np + tj]++) {
          if (bad++ < 5) std::printf("sym edge=%d m=%d lt=%d -> (%d,%d)\n", edge, m, lt, ti, tj);
        }
      }
      for (int n : {m, m + 1, m + 700, 4 * m}) {
        const int nq = pm::mt_edge_tiles(n, edge);
        std::vector<int> seen(np * nq, 0);
        for (int lt = 0; lt < pm::mt_full_tiles(m, n, edge); ++lt) {
          int ti, tj;
          pm::full_tile_cols(lt, np, nq, ti, tj, 512 / edge);
          if (ti < 0 || ti >= np || tj < 0 || tj >= nq || seen[ti * nq + tj]++) {
            if (bad++ < 5) std::printf("full edge=%d m=%d n=%d lt=%d -> (%d,%d)\n", edge, m, n, lt, ti, tj);
          }
        }
      }
      // the tiles' K-split partials fit the 256-tile engine's
      const int nt = (m + 255) / 256;
      if ((long)pm::mt_sym_tiles(m, edge) * edge * edge > (long)nt * (nt + 1) / 2 * 65536) {
        if (bad++ < 5) std::printf("partials edge=%d m=%d\n", edge, m);
      }
    }
  }
  std::printf(bad ? "FAIL %d\n" : "OK\n", bad);
  return bad != 0;
}
