// Midsolve: retrograde sweep over the positions below one board with >= 18 stones.
//
// Entries are 32-byte (win, notlose) halfsuper pairs, so both of the reference's aggressive
// passes (pentago/mid/midengine.cc:155-160) run as one: the reference's pass a at level n is
// the win component when a ^ (n & 1) == 1 and the notlose component otherwise, and the two
// passes exchange roles through ~ exactly as ~(win, notlose) = (~notlose, ~win) does.  Where
// the entries of a level are kept is this library's own layout (mid_tiles.h).
#pragma once
#include <cstdint>

#include "../../include/pentago_amd.h"

namespace pe {

// A board to solve: its empty cells in increasing order.
struct MidInfo {
  uint64_t side[2];
  uint32_t ply;
  int32_t spots;
  uint8_t empty[20];
};

int choose_host(int n, int k);
int bottleneck(int spots);
bool make_mid_info(const pe_high_board& b, MidInfo* I);

// high_board_t helpers (pentago/high/board.{h,cc})
int high_count(const pe_high_board& b);
bool high_done_and_value(const pe_high_board& b, int* value);
pe_high_board high_place(const pe_high_board& b, int bit);
pe_high_board high_rotate(const pe_high_board& b, int q, int d);
uint64_t high_raw(const pe_high_board& b);
int mid_traverse(const pe_high_board& b, const pe_halfsupers* supers, pe_mid_value* out);

}  // namespace pe
