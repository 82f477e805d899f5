// Midsolve device code shared by the level-synchronous and the work-queue kernels: the
// per-board descriptor, the wins tables and the tile sweep (pentago/mid/internal.h:122-131 and
// 358-408, both aggressive passes at once; tiles: mid_tiles.h).
#pragma once
#include <hip/hip_runtime.h>

#include "device.h"
#include "mid.h"
#include "mid_tiles.h"
#include "super.h"

namespace pe {

struct MidBoardDev {
  MidInfo I;
  uint64_t* wins;           // [mover of the root, other][mask of empty cells]: halves of parity 0, 1
  uint64_t* spill;          // tile entries that the workspace has no room for
  uint64_t* work;           // tile entries, 4 u64 each
  pe_halfsupers* results;   // 19 entries
};

// One entry of a board's wins tables: idx = player << spots | mask of empty cells, player 0 the
// one to move at the root.  Masks with more stones than the player ever places are not read.
__device__ inline void mid_wins_entry(const MidBoardDev& B, int64_t idx, const DevTables& T) {
  const int spots = B.I.spots;
  const int player = int(idx >> spots);
  const uint32_t mask = uint32_t(idx) & ((1u << spots) - 1);
  if (__popc(mask) > (spots + 1 - player) / 2) return;
  uint64_t side = B.I.side[(spots + player) & 1];
  for (uint32_t r = mask; r; r &= r - 1) side |= uint64_t(1) << B.I.empty[__builtin_ctz(r)];
  const S4 w = super_wins<true>(side, T.superwin);
  const H2 even = split_half(w, 0), odd = split_half(w, 1);
  ulonglong2* o = reinterpret_cast<ulonglong2*>(B.wins + 4 * idx);
  o[0] = make_ulonglong2(even.w[0], even.w[1]);
  o[1] = make_ulonglong2(odd.w[0], odd.w[1]);
}

constexpr int kTileThreads = 256;   // threads that sweep one tile: the largest class at once
static_assert(kTileClass <= kTileThreads, "a class is one round");
// Loads of the tiles above in flight for a thread: slots of this tile times tiles.  2 x 4 and
// 1 x 4 (44 registers) take 6 % and 14 % longer, 6 x 1 9 %, 6 x 2 spills.
constexpr int kSlots = 3, kAbove = 2;

// LDS of a tile: its entries as they are stored (classes of even l, then of odd l; a class's win
// halves, then its notlose halves), and the wins of both players' stones on the low cells beside
// the tile's high ones, halves of parity 0 and 1.
struct TileLds {
  uint4 half[2 * kTileEntries];
  uint4 wins[2][2][1 << kTileCells];
};

// Barrier between the classes of a tile: orders the LDS, and leaves global loads and stores
// in flight (a tile reads only tiles of earlier launches or earlier full barriers).
__device__ __forceinline__ void tile_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

struct Two { uint4 win, nl; };   // an entry
__device__ __forceinline__ void or4(uint4& a, const uint4& b) {
  a.x |= b.x; a.y |= b.y; a.z |= b.z; a.w |= b.w;
}
__device__ __forceinline__ void or4(uint4& a, const uint4& b, const uint4& c) {
  a.x = lop3_32<kOr3>(a.x, b.x, c.x); a.y = lop3_32<kOr3>(a.y, b.y, c.y);
  a.z = lop3_32<kOr3>(a.z, b.z, c.z); a.w = lop3_32<kOr3>(a.w, b.w, c.w);
}
__device__ __forceinline__ void or_two(Two& a, const Two& b) { or4(a.win, b.win); or4(a.nl, b.nl); }
__device__ __forceinline__ void or_two(Two& a, const Two& b, const Two& c) {
  or4(a.win, b.win, c.win); or4(a.nl, b.nl, c.nl);
}
// hrmax of four words (super.h), then OR with `extra`
__device__ __forceinline__ uint4 hrmax4(const uint4& v, const uint4& extra) {
  uint4 r;
  r.x = hrmax_word(v.x, v.w, v.y, extra.x);
  r.y = hrmax_word(v.y, v.x, v.z, extra.y);
  r.z = hrmax_word(v.z, v.y, v.w, extra.z);
  r.w = hrmax_word(v.w, v.z, v.x, extra.w);
  return r;
}

// A store that does not stay in the L2.
__device__ __forceinline__ void store_stream(uint4* p, const uint4& v) {
  typedef uint32_t v4 __attribute__((ext_vector_type(4)));
  const v4 x = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(x, reinterpret_cast<v4*>(p));
}

// What a tile needs of its board and schedule, the same for every tile of a launch.
struct TileJob {
  const uint4* wins;        // MidBoardDev::wins
  uint64_t* work;
  uint64_t* spill;
  pe_halfsupers* results;
  const MidTile* tiles;     // the board's tiles in order
  const uint2* bases;       // first entries of a tile's halves (even levels, odd levels), by code
  int32_t ply, low, high, in_work;
  bool stream;              // entries are read again only once they have left the L2 (store_stream)
};
__device__ __forceinline__ TileJob tile_job(const MidBoardDev& B, uint64_t* work, const MidSched& S, const MidTabs& M,
                                                bool stream) {
  TileJob J;
  J.wins = reinterpret_cast<const uint4*>(B.wins);
  J.work = work;
  J.spill = B.spill;
  J.results = B.results;
  J.tiles = M.tiles + S.tiles;
  J.bases = reinterpret_cast<const uint2*>(M.bases) + S.bases;
  J.ply = int(B.I.ply);
  J.low = S.low;
  J.high = S.high;
  J.in_work = S.work_entries;
  J.stream = stream;
  return J;
}

// Sweep one tile (`tile` counts from the board's first; negative: only take part in the
// barriers) with the kTileThreads threads tid = 0.. of a workgroup.  Every tile of a board runs
// the same number of barriers (low + 2).
//
// What bounds it: the reads of the tiles one high stone up, 32 bytes a position and empty high
// cell.  The half that a class reads of such a tile has the same layout as the half of this tile
// that the class is in, so all of them are ORed into the LDS first, entry by entry, with every
// load of the tile independent of every other; the sweep that follows, a barrier a class, touches
// the LDS only, but for the child ranks, which are loaded a class ahead.
__device__ __forceinline__ void mid_tile(const TileJob& J, const MidTabs& M, int tile, TileLds& lds, int tid) {
  const int wave0 = __builtin_amdgcn_readfirstlane(tid & ~63);
  const int lane = tid & 63;
  const int low = J.low, high = J.high, spots = low + high;
  const MidTile cfg = J.tiles[max(tile, 0)];
  const uint32_t p = cfg.p, q = cfg.q;
  const int a = __popc(p), h = a + __popc(q), d = 2 * a - h;
  const int nhigh = tile < 0 ? 0 : high - h;
  auto entry = [&](uint32_t e) {
    return e < uint32_t(J.in_work) ? J.work + 4 * uint64_t(e) : J.spill + 4 * uint64_t(e - uint32_t(J.in_work));
  };
  // lane l: class l; lane j: the tiles above with the j-th empty high cell filled by M0 (of which
  // the odd levels are read) and by M1 (the even ones)
  MidClass mine = {{0, 0}};
  if (tile >= 0 && lane <= low) mine = M.classes[mid_class_row(low, d, lane)];
  uint64_t up0 = 0, up1 = 0;
  if (lane < nhigh) {
    uint32_t rest = ((1u << high) - 1) & ~(p | q);
    for (int j = 0; j < lane; j++) rest &= rest - 1;
    uint32_t c3 = 1;
    for (int i = __builtin_ctz(rest); i > 0; i--) c3 *= 3;
    up0 = reinterpret_cast<uint64_t>(entry(J.bases[cfg.code + c3].y));
    up1 = reinterpret_cast<uint64_t>(entry(J.bases[cfg.code + 2 * c3].x));
  }
  const uint2 own = J.bases[cfg.code];
  if (tile >= 0)
    for (int i = tid; i < 4 << low; i += kTileThreads) {   // player, mask, parity
      const int player = i >> (low + 1), k = i & ((2 << low) - 1);
      const uint64_t row = player ? (uint64_t(1) << spots) + (uint64_t(q) << low) : uint64_t(p) << low;
      lds.wins[player][k & 1][k >> 1] = J.wins[2 * row + k];
    }
  auto get_class = [&](int l) {
    MidClass c = {{0, 0}};
    if (l >= 0)
      for (int i = 0; i < 2; i++) c.w[i] = uint32_t(__builtin_amdgcn_readlane(int(mine.w[i]), l));
    return c;
  };
  // entries of the classes of even l, which come first, and of odd l
  int size[2];
  for (int e = 0; e < 2; e++) {
    const MidClass top = get_class(low - ((low + e) & 1));
    size[e] = top.at() + top.count();
  }
  if (nhigh)
    for (int e = 0; e < 2; e++) {
      const uint64_t up = (h + e) & 1 ? up1 : up0;
      auto above = [&](int j) {
        return reinterpret_cast<const uint4*>(uint64_t(uint32_t(__builtin_amdgcn_readlane(int(up), j))) |
                                              uint64_t(uint32_t(__builtin_amdgcn_readlane(int(up >> 32), j))) << 32);
      };
      // whole waves (a lane of `up` is read only with every lane active): lanes past the end
      // take the last slot once more
      for (int i = wave0; i < 2 * size[e]; i += kSlots * kTileThreads) {
        uint4 acc[kSlots];
        int at[kSlots];
#pragma unroll
        for (int u = 0; u < kSlots; u++) at[u] = min(i + lane + u * kTileThreads, 2 * size[e] - 1);
        const uint4* in = above(0);
#pragma unroll
        for (int u = 0; u < kSlots; u++) acc[u] = in[at[u]];
        int j = 1;
        for (; j + kAbove <= nhigh; j += kAbove) {
          uint4 x[kAbove][kSlots];
#pragma unroll
          for (int k = 0; k < kAbove; k++) {
            const uint4* in = above(j + k);
#pragma unroll
            for (int u = 0; u < kSlots; u++) x[k][u] = in[at[u]];
          }
#pragma unroll
          for (int k = 0; k < kAbove; k++)
#pragma unroll
            for (int u = 0; u < kSlots; u++) or4(acc[u], x[k][u]);
        }
        for (; j < nhigh; j++) {
          const uint4* in = above(j);
#pragma unroll
          for (int u = 0; u < kSlots; u++) or4(acc[u], in[at[u]]);
        }
#pragma unroll
        for (int u = 0; u < kSlots; u++) lds.half[(e ? 2 * size[0] : 0) + at[u]] = acc[u];
      }
    }
  const uint4 none = make_uint4(0, 0, 0, 0);
  MidClass c = get_class(low);
  Kids kids, ahead;
  if (wave0 < c.count()) kids = M.kids[2 * c.members() + ((h + low) & 1) * c.count() + min(tid, c.count() - 1)];
  const uint4* kid_half = nullptr;   // class l + 1
  int kid_count = 0;
  for (int l = low; l >= 0; l--) {
    const int n = h + l, mover = n & 1, par = (n + J.ply) & 1;
    const MidClass cn = get_class(l - 1);
    if (wave0 < cn.count())
      ahead = M.kids[2 * cn.members() + ((h + l - 1) & 1) * cn.count() + min(tid, cn.count() - 1)];
    uint4* half = lds.half + 2 * ((l & 1 ? size[0] : 0) + c.at());
    tile_barrier();   // the tiles above (first round) or class l + 1 are in the LDS
    if (wave0 < c.count()) {
      const int r = min(tid, c.count() - 1);
      Two acc = {none, none};
      if (nhigh) acc = Two{half[r], half[c.count() + r]};
      if (n == spots) acc.nl = make_uint4(~0u, ~0u, ~0u, ~0u);   // the board is full: not lost
      auto kid = [&](uint32_t rank16) {
        const char* in = reinterpret_cast<const char*>(kid_half) + rank16;
        return Two{*reinterpret_cast<const uint4*>(in), *reinterpret_cast<const uint4*>(in + 16 * kid_count)};
      };
#pragma unroll
      for (int j = 0; j < kTileCells; j += 2) {
        if (j + 1 < kTileCells && j + 1 < low - l)
          or_two(acc, kid(kids.rank16[j]), kid(kids.rank16[j + 1]));
        else if (j < low - l)
          or_two(acc, kid(kids.rank16[j]));
      }
      const uint32_t A = kids.mem & 0xff, Bm = kids.mem >> 8;
      const uint4 imm0 = lds.wins[mover][par][mover ? Bm : A];
      const uint4 after = lds.wins[mover ^ 1][par][mover ? A : Bm];
      const uint4 before = lds.wins[mover ^ 1][par ^ 1][mover ? A : Bm];
      // The side to move wins at once (imm0) unless the other side has five too (after), else
      // by a child; not lost likewise.  Of (children, imm0, after): win (c & ~(i | a)) | (i & ~a)
      // = 0x54, not lost (c & ~(i | a)) | i = 0xDC; here their complements, whose hrmax,
      // exchanged, is the other side's view, which the parents read.
      uint4 lw, ln;
      lw.x = lop3_32<0xAB>(acc.win.x, imm0.x, after.x); ln.x = lop3_32<0x23>(acc.nl.x, imm0.x, after.x);
      lw.y = lop3_32<0xAB>(acc.win.y, imm0.y, after.y); ln.y = lop3_32<0x23>(acc.nl.y, imm0.y, after.y);
      lw.z = lop3_32<0xAB>(acc.win.z, imm0.z, after.z); ln.z = lop3_32<0x23>(acc.nl.z, imm0.z, after.z);
      lw.w = lop3_32<0xAB>(acc.win.w, imm0.w, after.w); ln.w = lop3_32<0x23>(acc.nl.w, imm0.w, after.w);
      if (n <= 1 && tid < c.count()) {
        const uint32_t root = p << low | A;
        uint4* res = reinterpret_cast<uint4*>(&J.results[n ? 1 + __builtin_ctz(root) : 0]);
        res[0] = make_uint4(~lw.x, ~lw.y, ~lw.z, ~lw.w);
        res[1] = make_uint4(~ln.x, ~ln.y, ~ln.z, ~ln.w);
      }
      const uint4 sw = hrmax4(ln, before), sn = hrmax4(lw, before);
      if (tid < c.count()) {
        half[tid] = sw;
        half[c.count() + tid] = sn;
        const uint32_t to = n & 1 ? own.y : own.x;
        if (to != kNotStored) {
          uint4* out = reinterpret_cast<uint4*>(entry(to + uint32_t(c.at())));
          if (J.stream) {
            store_stream(&out[tid], sw);
            store_stream(&out[c.count() + tid], sn);
          } else {
            out[tid] = sw;
            out[c.count() + tid] = sn;
          }
        }
      }
    }
    kid_half = half;
    kid_count = c.count();
    c = cn;
    kids = ahead;
  }
}

}  // namespace pe
