// Tile records made in pieces against all of them at once.
#include <stddef.h>

#include <vector>

#include "../../pentago_amd/csrc/mid_tiles.h"

extern "C" int rc_pieces(int64_t piece) {
  using namespace pe;
  const MidTabs M = mid_tabs().view();
  const std::vector<uint32_t> all = mid_records(M);
  const int64_t tiles = int64_t(all.size()) / kRecWords;
  std::vector<uint32_t> out(size_t(kRecWords * piece) + 1, 7u);   // pieces leave dirt behind, the word past them stays
  for (int64_t t = 0; t < tiles; t += piece) {
    const int64_t n = piece < tiles - t ? piece : tiles - t;
    mid_records(M, t, n, out.data());
    for (int64_t i = 0; i < kRecWords * n; i++)
      if (out[size_t(i)] != all[size_t(kRecWords * t + i)]) return 1;
    if (out.back() != 7u) return 2;
  }
  return tiles > 0 ? 0 : 3;
}
