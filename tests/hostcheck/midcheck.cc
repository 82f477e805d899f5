// CPU build of the midsolve tiles (pentago_amd/csrc/mid_tiles.{h,cc}): the tables walked as the
// device kernels walk them.
#include <cstring>
#include <map>
#include <vector>

#include "../../pentago_amd/csrc/mid.h"
#include "../../pentago_amd/csrc/mid_tiles.h"
#include "../../pentago_amd/csrc/super.h"
#include "../../pentago_amd/csrc/tables.h"

using namespace pe;

static uint32_t pow3(int n) { return n ? 3 * pow3(n - 1) : 1; }

extern "C" {

// Where every half of a tile lies and who reads it, step by step: the number of faults (a half
// outside its area or over another that is still to be read, a read of a half that does not
// hold the tile expected, a tile computed before its children or twice, positions missed).
int mc_layout(int spots) {
  const MidTabs M = mid_tabs().view();
  const MidSched& S = M.sched[spots];
  const int64_t work = mid_work_entries(spots), all = work + mid_spill_entries(spots);
  int faults = 0;
  int64_t positions = 0, expect = 0;
  for (int n = 0; n <= spots; n++) expect += int64_t(choose_host(spots, n)) * choose_host(n, n / 2);
  struct Half { int64_t size; uint32_t id; };
  std::map<int64_t, Half> held;   // by first entry: tiles in memory
  std::vector<int> done(size_t(1) << 20, -1);
  auto size = [&](int a, int b, int par) {
    int64_t t = 0;
    for (int l = 0; l <= S.low; l++)
      if (((a + b + l) & 1) == par) t += M.classes[mid_class_row(S.low, a - b, l)].count();
    return t;
  };
  for (int k = 0; k < S.steps; k++) {
    std::vector<int64_t> read;
    std::vector<std::pair<int64_t, Half>> wrote;
    for (int t = S.first[k]; t < S.first[k + 1]; t++) {
      const uint32_t p = M.tiles[S.tiles + t].p, q = M.tiles[S.tiles + t].q, code = M.tiles[S.tiles + t].code;
      const int a = __builtin_popcount(p), b = __builtin_popcount(q);
      uint32_t digits = 0;
      for (int c = 0; c < S.high; c++) digits += ((p >> c & 1) + 2 * (q >> c & 1)) * pow3(c);
      faults += digits != code;
      faults += (p & q) || (p | q) >> S.high || done[code] >= 0;
      done[code] = k;
      for (int l = 0; l <= S.low; l++) positions += M.classes[mid_class_row(S.low, a - b, l)].count();
      for (int c = 0; c < S.high; c++) {
        if ((p | q) >> c & 1) continue;
        for (int m = 0; m < 2; m++) {   // as many levels as the tile has with mover m
          bool needs = false;
          for (int l = 0; l <= S.low; l++)
            needs |= ((a + b + l) & 1) == m && M.classes[mid_class_row(S.low, a - b, l)].count();
          if (!needs) continue;
          const uint32_t child = code + (m + 1u) * pow3(c);
          const int64_t at = M.bases[2 * (S.bases + child) + 1 - m];
          const auto it = held.find(at);
          if (it == held.end() || it->second.id != 2 * child + 1 - m) faults++;
          else read.push_back(at);
        }
      }
      for (int par = 0; par < 2; par++) {
        const int64_t at = M.bases[2 * (S.bases + code) + par], n = size(a, b, par);
        if (at == kNotStored) { faults += (par ? a : b) > 0 && n > 0; continue; }
        faults += at + n > all || (at < work && at + n > work);
        wrote.push_back({at, Half{n, 2 * code + par}});
      }
    }
    // written while the step's reads go on: over nothing that is held
    for (const auto& w : wrote) {
      const auto it = held.lower_bound(w.first);
      if (it != held.end() && it->first < w.first + w.second.size) faults++;
      if (it != held.begin()) {
        const auto pr = std::prev(it);
        if (pr->first + pr->second.size > w.first) faults++;
      }
      held[w.first] = w.second;
    }
    for (int64_t at : read) held.erase(at);   // each half is read in one step only
  }
  return faults + (positions != expect) + int(held.size());
}

// The records and child ranks that the device reads, against the tables: the number of words
// that differ, of tiles and members whose low cells number mid_low_cells(spots).
int mc_device_tables(int spots) {
  const MidTabs M = mid_tabs().view();
  const MidSched& S = M.sched[spots];
  const std::vector<uint32_t> recs = mid_records(M);
  const std::vector<KidRanks> ranks = mid_kid_ranks(M);
  int faults = 0;
  for (int t = S.tiles; t < S.tiles + S.first[S.steps]; t++) {
    const uint32_t* r = recs.data() + size_t(kRecWords) * size_t(t);
    const MidTile& X = M.tiles[t];
    const int d = __builtin_popcount(X.p) - __builtin_popcount(X.q);
    faults += (r[0] & 0xffff) != X.p || r[0] >> 16 != X.q;
    for (int par = 0; par < 2; par++) faults += r[kRecOwn + par] != M.bases[2 * (S.bases + X.code) + par];
    uint32_t size[2] = {0, 0};
    for (int l = 0; l <= kTileCells; l++) {
      const uint32_t n = l <= S.low ? uint32_t(M.classes[mid_class_row(S.low, d, l)].count()) : 0;
      size[l & 1] += n;
      faults += (r[kRecCounts + l / 4] >> (8 * (l % 4)) & 0xff) != n;
    }
    faults += r[kRecSizes] != (size[0] | size[1] << 16);
    for (int c = 0, j = 0; c < S.high; c++)
      if (!((X.p | X.q) >> c & 1)) {
        faults += r[kRecUp + j] != M.bases[2 * (S.bases + X.code + pow3(c)) + 1];
        faults += r[kRecUp + kRecUp1 + j] != M.bases[2 * (S.bases + X.code + 2 * pow3(c))];
        j++;
      }
  }
  for (int d = -11; d <= 11; d++)
    for (int l = 0; l <= S.low; l++) {
      const MidClass& c = M.classes[mid_class_row(S.low, d, l)];
      for (int i = 0; i < c.count(); i++) {
        const KidRanks& k = ranks[size_t(mid_kid_row(S.low, d, l) + i)];
        const Kids& x = M.kids[2 * c.members() + ((d + l) & 1) * c.count() + i];
        for (int j = 0; j < S.low - l; j++) faults += 16 * (k.w[j >> 2] >> (8 * (j & 3)) & 0xff) != x.rank16[j];
        faults += l && k.w[1] >> 16 != x.mem;
      }
    }
  return faults;
}

// One board solved on the CPU, as mid_tile does; 0 on success.
int mc_solve(uint64_t side0, uint64_t side1, uint32_t ply, uint64_t* results) {
  pe_high_board hb{{side0, side1}, ply};
  MidInfo I;
  if (!make_mid_info(hb, &I)) return 1;
  const int spots = I.spots;
  const MidTabs M = mid_tabs().view();
  const MidSched& S = M.sched[spots];
  const int low = S.low, high = S.high;
  std::vector<H2> wins(size_t(4) << spots);
  for (int player = 0; player < 2; player++)
    for (uint32_t mask = 0; mask < 1u << spots; mask++) {
      uint64_t side = I.side[(spots + player) & 1];
      for (int i = 0; i < spots; i++)
        if (mask >> i & 1) side |= uint64_t(1) << I.empty[i];
      const S4 w = super_wins(side, tables().superwin);
      for (int par = 0; par < 2; par++) wins[2 * ((size_t(player) << spots) + mask) + par] = split_half(w, par);
    }
  struct Entry { H2 win, nl; };
  std::vector<Entry> mem(size_t(mid_work_entries(spots) + mid_spill_entries(spots)));
  for (int k = 0; k < S.steps; k++)
    for (int t = S.first[k]; t < S.first[k + 1]; t++) {
      const uint32_t p = M.tiles[S.tiles + t].p, q = M.tiles[S.tiles + t].q, code = M.tiles[S.tiles + t].code;
      const int a = __builtin_popcount(p), h = a + __builtin_popcount(q), d = 2 * a - h;
      std::vector<Entry> tile[2];
      for (int l = low; l >= 0; l--) {
        const MidClass& c = M.classes[mid_class_row(low, d, l)];
        if (!c.count()) continue;
        const int n = h + l, mover = n & 1, par = (n + int(ply)) & 1;
        tile[l & 1].resize(size_t(c.count()));
        for (int r = 0; r < c.count(); r++) {
          Entry e{};
          if (n == spots) e.nl.w[0] = e.nl.w[1] = ~uint64_t(0);
          auto add = [&](const Entry& x) { e.win = h2_or(e.win, x.win); e.nl = h2_or(e.nl, x.nl); };
          for (int cell = 0; cell < high; cell++)
            if (!((p | q) >> cell & 1)) {
              const uint32_t up = code + (mover + 1u) * pow3(cell);
              add(mem.at(size_t(M.bases[2 * (S.bases + up) + 1 - mover]) + size_t(c.at() + r)));
            }
          const Kids& kids = M.kids[2 * c.members() + mover * c.count() + r];
          for (int j = 0; j < low - l; j++) add(tile[(l + 1) & 1].at(kids.rank16[j] / 16));
          const uint32_t A = kids.mem & 0xff, B = kids.mem >> 8;
          const size_t w0 = 2 * size_t(p << low | A), w1 = 2 * ((size_t(1) << spots) + (q << low | B));
          const H2 imm = wins[(mover ? w1 : w0) + par];
          const H2 after = wins[(mover ? w0 : w1) + par], before = wins[(mover ? w0 : w1) + (par ^ 1)];
          H2 win, nl, nw, nn;
          for (int i = 0; i < 2; i++) {
            win.w[i] = lop3<0x54>(e.win.w[i], imm.w[i], after.w[i]);
            nl.w[i] = lop3<0xDC>(e.nl.w[i], imm.w[i], after.w[i]);
            nw.w[i] = ~nl.w[i];
            nn.w[i] = ~win.w[i];
          }
          if (n <= 1) {
            uint64_t* res = results + 4 * (n ? 1 + __builtin_ctz(p << low | A) : 0);
            res[0] = win.w[0]; res[1] = win.w[1]; res[2] = nl.w[0]; res[3] = nl.w[1];
          }
          e.win = h2_or(hrmax(nw), before);
          e.nl = h2_or(hrmax(nn), before);
          tile[l & 1][size_t(r)] = e;
          const uint32_t own = M.bases[2 * (S.bases + code) + (n & 1)];
          if (own != kNotStored) mem.at(size_t(own) + size_t(c.at() + r)) = e;
        }
      }
    }
  return 0;
}

}  // extern "C"
