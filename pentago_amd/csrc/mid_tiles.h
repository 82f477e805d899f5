// Midsolve tiles: how the positions below a board are cut into units that a workgroup sweeps
// from its LDS.
//
// The board's empty cells are split into L low cells (cells 0..L-1) and H = spots - L high
// cells.  A tile is every position with the same stones on the high cells: its configuration
// (p, q), the high cells holding stones of the player to move at the root (M0) and of the
// other player (M1), and within it every way to place stones on the low cells that keeps the
// players in turn.  With a = |p|, b = |q| and l stones on the low cells a position is at level
// n = a + b + l, where M0 holds ceil(n/2) stones, so it has la = ceil((l - (a - b)) / 2) low
// stones of M0 and lb = l - la of M1: the classes (la, lb) of a tile depend on a - b only, and
// the members of a class (pairs of disjoint masks) and the ranks of their children inside the
// tile are the same for every board.  A move to a low cell stays in the tile, at class l + 1; a
// move to a high cell c leads to the same low stones, the same rank of the same class, of the
// tile with c added.
//
// So a tile is swept for l = L..0 with its last class in LDS, reading only the tiles one high
// stone up from memory, as contiguous runs, and a board is swept tile layer by tile layer
// (a + b = H..0).  Of a tile's entries those of odd levels (M0 moved last) are read by the
// tiles (a - 1, b) only and those of even levels by the tiles (a, b - 1) only; each half is
// stored apart, and its memory is free again once that one group of tiles is done.  The half that
// a tile's classes of one parity read of a tile one stone up holds the same classes in the same
// order, so its layout is that of the half they are in.
#pragma once
#include <cstdint>
#include <vector>

namespace pe {

constexpr int kMidSpots = 18;        // most empty cells
constexpr int kTileCells = 7;        // most low cells
constexpr int kTileClass = 210;      // largest class: 8! / (3! 3! 2!)
constexpr int kTileEntries = 750;    // largest tile (a = b): sum over l of 7! / ((7-l)! ceil(l/2)! floor(l/2)!)
constexpr uint32_t kNotStored = 0xffffffffu;

inline int mid_low_cells(int spots) { return spots < kTileCells ? spots : kTileCells; }

// One spots value: its tiles in the order they are computed, in steps (one launch each).
struct MidSched {
  int32_t low, high, steps;
  int32_t tiles;                     // first of its tiles in MidTabs::tiles
  int32_t bases;                     // start of its rows in MidTabs::bases
  int32_t work_entries;              // entries below this are in the workspace, the rest in the spill area
  int32_t first[kMidSpots + 2];      // step k: tiles [first[k], first[k + 1]) from `tiles` on
};

// A tile: its configuration and the base-3 code of it (digit c: 0 empty, 1 M0, 2 M1).
struct MidTile { uint32_t p, q, code, pad; };

// Class l of the tiles with a - b = d, for `low` low cells: row ((low * 23) + d + 11) * 9 + l.
// Packed: a lane holds one.
struct MidClass {
  uint32_t w[2];
  constexpr int count() const { return int(w[0] & 0xff); }     // 0: no such class
  constexpr int members() const { return int(w[0] >> 8); }     // members of the classes before it (kids: twice that)
  constexpr int at() const { return int(w[1]); }               // its first entry within the tile's half (levels of its parity)
};

// One member (A, B) of a class, the low cells of M0 and of M1: 16 times the ranks of its children
// inside the tile, by ascending cell, and A | B << 8.
struct Kids { uint16_t rank16[kTileCells], mem; };

// Lookup tables on the host.
struct MidTabs {
  const MidSched* sched;             // [kMidSpots + 1]
  const MidTile* tiles;
  const uint32_t* bases;             // [2 * (bases + code) + parity]: first entry of the tile's half
  const MidClass* classes;
  const Kids* kids;                  // [2 * members + mover * count + rank]
};
struct MidTabsHost {
  std::vector<MidSched> sched;
  std::vector<MidTile> tiles;
  std::vector<uint32_t> bases;
  std::vector<MidClass> classes;
  std::vector<Kids> kids;
  MidTabs view() const;
};
constexpr int mid_class_row(int low, int d, int l) { return (low * 23 + d + 11) * 9 + l; }

// The device's form of the tables, which a workgroup has in two dependent loads (the tile's
// record, then everything that the record leads to).
//
// A tile's record is 32 words, one to a lane: p | q << 16; the first entries of its own halves
// (even levels, odd levels); entries of its classes of even l | of odd l << 16; the classes'
// counts, a byte each; and by empty high cell in ascending order the first entries of the halves
// it may read there: the odd levels of the tile with the cell filled by M0, the even ones of the
// tile with it filled by M1.
constexpr int kRecWords = 32, kRecOwn = 1, kRecSizes = 3, kRecCounts = 4, kRecUp = 6, kRecUp1 = kMidSpots - kTileCells;
// Ranks of a member's children by ascending cell, a byte each, and in the last two bytes its masks
// A and B; the one member of class 0 (no stones) may have a seventh child, in the place of A.
struct KidRanks { uint32_t w[2]; };
// The mover of class l is (d + l) & 1 (d and a + b have one parity): a row of kTileClass members.
constexpr int mid_kid_row(int low, int d, int l) { return ((low * 23 + d + 11) * (kTileCells + 1) + l) * kTileClass; }
struct MidTabsDev {
  const MidSched* sched;
  const uint32_t* records;           // kRecWords a tile, in the order of MidTabs::tiles
  const KidRanks* kids;              // [mid_kid_row + rank]
};
// Records of n tiles from `first` on (kRecWords each); of all tiles.
void mid_records(const MidTabs& M, int64_t first, int64_t n, uint32_t* out);
std::vector<uint32_t> mid_records(const MidTabs& M);
std::vector<KidRanks> mid_kid_ranks(const MidTabs& M);

// Entries (32 bytes) of a board's two areas: its workspace, and its table area, which holds
// the wins tables (2 << spots entries) and then the spill area.
int64_t mid_work_entries(int spots);
int64_t mid_table_area_bytes(int spots);
int64_t mid_spill_entries(int spots);

// Built once (thread-safe); throws std::runtime_error if a board's tiles did not fit its areas.
const MidTabsHost& mid_tabs();

}  // namespace pe
