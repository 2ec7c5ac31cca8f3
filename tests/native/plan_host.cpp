// Plans of the tile kernel as the library makes them, for the tests: "rows N K" of a problem or two ("rows0 rows1 N K") on each line of stdin -> tile
// height, parts of a tile and whole tiles; "pad rows tile ld K" -> the row that a tile's rows of padding are fetched as; "shares rows N K workers" -> TileShares.
#include <cstdio>
#include <cstring>
#include <iostream>
#include <sstream>

#include "gemm_bf16.h"

int main() {
  using namespace odit;
  for (std::string line; std::getline(std::cin, line);) {
    std::istringstream in(line);
    std::string word;
    if (line.rfind("pad ", 0) == 0) {
      long long rows, tile, ld, k;
      in >> word >> rows >> tile >> ld >> k;
      printf("%d\n", tile_padding_row(static_cast<int>(rows), static_cast<int>(tile), ld, static_cast<int>(k)));
      continue;
    }
    if (line.rfind("shares ", 0) == 0) {
      int rows, N, K, workers;
      in >> word >> rows >> N >> K >> workers;
      const TileShares t = tile_shares(rows, N, K, workers);
      printf("%d %d %d %d %d\n", t.known ? 1 : 0, t.tiles, t.from, t.share, t.more);
      continue;
    }
    int v[4], n = 0;
    while (n < 4 && in >> v[n]) ++n;
    const int count = n - 2;
    GemmCall c[2] = {};
    for (int i = 0; i < count; ++i) { c[i].M = v[i]; c[i].N = v[count]; c[i].K = v[count + 1]; }
    const TilePlan p = plan_gemm_tile(c, count, 256, true);
    printf("%d %d %d\n", p.bm, p.parts, p.whole);
  }
}
