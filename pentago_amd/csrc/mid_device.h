// Midsolve device code shared by the step and the work-queue kernels: the wins tables and the tile sweep (pentago/mid/internal.h:122-131 and
// 358-408, both aggressive passes at once; tiles: mid_tiles.h).
#pragma once
#include <hip/hip_runtime.h>

#include "device.h"
#include "mid.h"
#include "mid_queue.h"
#include "mid_tiles.h"
#include "super.h"

namespace pe {

// One entry of a board's wins tables: idx = player << spots | mask of empty cells, player 0 the
// one to move at the root.  Masks with more stones than the player ever places are not written:
// a tile copies them to its LDS with the rest and never uses them.
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

constexpr int kTileThreads = 256;   // threads of a sweep, or of each of its two chains: the largest class at once
static_assert(kTileClass <= kTileThreads, "a class is one round");

// A level's win halves come from the notlose halves of the level below it and the other way
// round, so a tile's entries are two chains that never meet: chain 0 is the win halves of even
// levels and the notlose halves of odd ones (as stored, which is the other side's view, the
// halves that those are made from), chain 1 the rest.  They are kept apart, each thread reads and
// writes the slots of its own chain only.
//
// LDS of a tile (kAlone: of one chain of a tile): its entries as they are stored (classes of even l,
// then of odd l, of each chain 0, then chain 1), and the wins of both players' stones on the low
// cells beside the tile's high ones, halves of parity 0 and 1.
template <bool kAlone>
struct TileLds {
  uint4 half[(kAlone ? 1 : 2) * kTileEntries];
  uint4 wins[2][2][1 << kTileCells];
};

// Barrier between the classes of a tile: orders the LDS, and leaves global loads and stores
// in flight (a tile reads only tiles of earlier launches or earlier full barriers).
__device__ __forceinline__ void tile_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ void or4(uint4& a, const uint4& b) {
  a.x |= b.x; a.y |= b.y; a.z |= b.z; a.w |= b.w;
}
__device__ __forceinline__ void or4(uint4& a, const uint4& b, const uint4& c) {
  a.x = lop3_32<kOr3>(a.x, b.x, c.x); a.y = lop3_32<kOr3>(a.y, b.y, c.y);
  a.z = lop3_32<kOr3>(a.z, b.z, c.z); a.w = lop3_32<kOr3>(a.w, b.w, c.w);
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
  const uint32_t* records;  // of the board's tiles in order
  const KidRanks* kids;     // rows of its number of low cells, from d = 0, l = 0 on
  int32_t ply, low, high, in_work;
  bool stream;              // entries are read again only once they have left the L2 (store_stream)
};
__host__ __device__ __forceinline__ TileJob tile_job(const MidBoardDev& B, uint64_t* work, const MidSched& S,
                                                     const MidTabsDev& M, bool stream) {
  TileJob J;
  J.wins = reinterpret_cast<const uint4*>(B.wins);
  J.work = work;
  J.spill = B.spill;
  J.results = B.results;
  J.records = M.records + int64_t(kRecWords) * S.tiles;
  J.kids = M.kids + mid_kid_row(S.low, 0, 0);
  J.ply = int(B.I.ply);
  J.low = S.low;
  J.high = S.high;
  J.in_work = S.work_entries;
  J.stream = stream;
  return J;
}

// Sweep one tile (`tile` counts from the board's first; negative: only take part in the
// barriers) with the threads tid = 0.. of a workgroup: kTileThreads that each take both chains
// (kChains = 1), kTileThreads for each chain (2), or kTileThreads for the chain `alone` only (2 and
// kAlone).  Every tile of a board runs the same number of barriers (low + 1).
//
// What bounds it: for a launch that fills the chip, the reads of the tiles one high stone up, 32
// bytes a position and empty high cell; else the latency of one tile.  The half that a class
// reads of such a tile has the same layout as the half of this tile that the class is in, so all
// of them are ORed into the LDS first, entry by entry, with every load of the tile independent of
// every other; the sweep that follows, a barrier a class, touches the LDS only.  The loads of a
// tile are two deep: its record, then the children's ranks of all its classes (two registers
// each), the wins and the tiles above at once.  Ranks loaded a class ahead and first entries
// looked up cell by cell took 9.5 against 7.5 us for a step of 26 stones.  One MI355X: 26 stones 68
// -> 58 us, 18 stones 2.57 -> 2.29 ms, of which 0.19 by 8 waves a SIMD with a thread a chain, where
// both chains a thread allow 5.
template <int kChains, bool kAlone = false>
__device__ __forceinline__ void mid_tile(const TileJob& J, int tile, TileLds<kAlone>& lds, int tid, int alone = 0) {
  // Loads of the tiles above in flight for a thread: slots of this tile times tiles (a chain's
  // slots are two rounds of its threads, both chains' three).  One chain a thread, in the 64
  // registers of 8 waves a SIMD: 2 x 3 and 2 x 2 alike, 2 x 4 20 % longer (spills), 2 x 5 with 6 waves 17 %.
  // Both: 2 x 4 and 1 x 4 take 6 % and 14 % longer, 6 x 1 9 %.
  constexpr int kSlots = kChains == 2 ? 2 : 3, kAbove = kChains == 2 ? 3 : 2;
  const int chain0 = kAlone ? alone : kChains == 2 ? __builtin_amdgcn_readfirstlane(tid / kTileThreads) : 0;
  const int t = kChains == 2 && !kAlone ? tid % kTileThreads : tid;   // member of a class
  const int wave0 = __builtin_amdgcn_readfirstlane(t & ~63);
  const int lane = tid & 63;
  const int low = J.low, high = J.high, spots = low + high;
  uint32_t rec = 0;
  if (tile >= 0 && lane < kRecWords) rec = J.records[int64_t(kRecWords) * tile + lane];
  auto word = [&](int i) { return uint32_t(__builtin_amdgcn_readlane(int(rec), i)); };
  const uint32_t p = word(0) & 0xffff, q = word(0) >> 16;
  const int a = __popc(p), h = a + __popc(q), d = 2 * a - h;
  const int nhigh = tile < 0 ? 0 : high - h;
  const uint64_t counts = uint64_t(word(kRecCounts)) | uint64_t(word(kRecCounts + 1)) << 32;
  auto count = [&](int l) { return int(counts >> (8 * l) & 0xff); };
  auto entry = [&](uint32_t e) {
    return reinterpret_cast<uint4*>(e < uint32_t(J.in_work) ? J.work + 4 * uint64_t(e)
                                                            : J.spill + 4 * uint64_t(e - uint32_t(J.in_work)));
  };
  KidRanks kids[kTileCells + 1];
  const KidRanks* row = J.kids + mid_kid_row(0, d, 0) - mid_kid_row(0, 0, 0) + min(t, kTileClass - 1);
#pragma unroll
  for (int l = kTileCells; l >= 0; l--)
    if (wave0 < count(l)) kids[l] = row[l * kTileClass];
  if (tile >= 0)
    for (int i = tid; i < 4 << low; i += kAlone ? kTileThreads : kTileThreads * kChains) {   // player, mask, parity
      const int player = i >> (low + 1), k = i & ((2 << low) - 1);
      const uint64_t first = player ? (uint64_t(1) << spots) + (uint64_t(q) << low) : uint64_t(p) << low;
      lds.wins[player][k & 1][k >> 1] = J.wins[2 * first + k];
    }
  // entries of the classes of even l, which come first, and of odd l
  const int size[2] = {int(word(kRecSizes) & 0xffff), int(word(kRecSizes) >> 16)};
  if (nhigh)
    for (int e = 0; e < 2; e++) {
      const int up = kRecUp + ((h + e) & 1 ? kRecUp1 : 0);
      const int first = chain0 * size[e], end = kChains == 2 ? first + size[e] : 2 * size[e];
      // whole waves (a word of the record is taken with every lane active): lanes past the end
      // take the last slot once more
      for (int i = first + wave0; i < end; i += kSlots * kTileThreads) {
        uint4 acc[kSlots];
        int at[kSlots];
#pragma unroll
        for (int u = 0; u < kSlots; u++) at[u] = min(i + lane + u * kTileThreads, end - 1);
        const uint4* in = entry(word(up));
#pragma unroll
        for (int u = 0; u < kSlots; u++) acc[u] = in[at[u]];
        int j = 1;
        for (; j + kAbove <= nhigh; j += kAbove) {
          uint4 x[kAbove][kSlots];
#pragma unroll
          for (int k = 0; k < kAbove; k++) {
            const uint4* in = entry(word(up + j + k));
#pragma unroll
            for (int u = 0; u < kSlots; u++) x[k][u] = in[at[u]];
          }
#pragma unroll
          for (int k = 0; k < kAbove; k++)
#pragma unroll
            for (int u = 0; u < kSlots; u++) or4(acc[u], x[k][u]);
        }
        for (; j < nhigh; j++) {
          const uint4* in = entry(word(up + j));
#pragma unroll
          for (int u = 0; u < kSlots; u++) or4(acc[u], in[at[u]]);
        }
#pragma unroll
        for (int u = 0; u < kSlots; u++) lds.half[kAlone ? (e ? size[0] : 0) + at[u] - first : (e ? 2 * size[0] : 0) + at[u]] = acc[u];
      }
    }
  // first slots of the classes from the highest on, below the class's own chain 0
  int at[2] = {size[0], size[1]};
  const uint4* kid_half = nullptr;   // class l + 1, chain 0
#pragma unroll
  for (int l = kTileCells; l >= 0; l--) {
    if (l > low) continue;
    const int n = h + l, mover = n & 1, par = (n + J.ply) & 1, e = l & 1, c = count(l);
    at[e] -= c;
    uint4* half = lds.half + (e ? (kAlone ? 1 : 2) * size[0] : 0) + at[e];
    tile_barrier();   // the tiles above (first round) or class l + 1 are in the LDS
    if (wave0 < c) {
      const int r = min(t, c - 1);
      const uint32_t mem = l ? kids[l].w[1] >> 16 : 0, A = mem & 0xff, Bm = mem >> 8;
      const uint4 imm0 = lds.wins[mover][par][mover ? Bm : A];
      const uint4 after = lds.wins[mover ^ 1][par][mover ? A : Bm];
      const uint4 before = lds.wins[mover ^ 1][par ^ 1][mover ? A : Bm];
      const uint32_t own = word(kRecOwn + mover);
#pragma unroll
      for (int k = 0; k < 3 - kChains; k++) {
        const int chain = chain0 + k;
        const bool notlose = (mover ^ chain) != 0;   // wave-uniform
        uint4 acc = make_uint4(0, 0, 0, 0);
        const int lc = kAlone ? 0 : chain;   // in the LDS
        if (nhigh) acc = half[lc * size[e] + r];
        if (n == spots && notlose) acc = make_uint4(~0u, ~0u, ~0u, ~0u);   // the board is full: not lost
        auto kid = [&](int j) {
          return kid_half[lc * size[e ^ 1] + int(kids[l].w[j >> 2] >> (8 * (j & 3)) & 0xff)];
        };
#pragma unroll
        for (int j = 0; j < kTileCells - l; j += 2) {
          if (j + 1 < low - l) or4(acc, kid(j), kid(j + 1));
          else if (j < low - l) or4(acc, kid(j));
        }
        // The side to move wins at once (imm0) unless the other side has five too (after), else
        // by a child; not lost likewise.  Of (children, imm0, after): win (c & ~(i | a)) | (i & ~a)
        // = 0x54, not lost (c & ~(i | a)) | i = 0xDC; here their complements, whose hrmax is the
        // other side's view, which the parents read.
        uint4 x;
        if (notlose) {
          x.x = lop3_32<0x23>(acc.x, imm0.x, after.x); x.y = lop3_32<0x23>(acc.y, imm0.y, after.y);
          x.z = lop3_32<0x23>(acc.z, imm0.z, after.z); x.w = lop3_32<0x23>(acc.w, imm0.w, after.w);
        } else {
          x.x = lop3_32<0xAB>(acc.x, imm0.x, after.x); x.y = lop3_32<0xAB>(acc.y, imm0.y, after.y);
          x.z = lop3_32<0xAB>(acc.z, imm0.z, after.z); x.w = lop3_32<0xAB>(acc.w, imm0.w, after.w);
        }
        if (n <= 1 && t < c) {
          const uint32_t root = p << low | A;
          uint4* res = reinterpret_cast<uint4*>(&J.results[n ? 1 + __builtin_ctz(root) : 0]);
          res[notlose] = make_uint4(~x.x, ~x.y, ~x.z, ~x.w);
        }
        x = hrmax4(x, before);
        if (t < c) {
          half[lc * size[e] + t] = x;
          if (own != kNotStored) {
            uint4* out = entry(own) + (chain * size[e] + at[e]);
            if (J.stream) store_stream(&out[t], x);
            else out[t] = x;
          }
        }
      }
    }
    kid_half = half;
  }
}

}  // namespace pe
