// Tables of the midsolve tiles (see mid_tiles.h): class members and children, and per number
// of empty cells the order of the tiles and where each stores its entries.
#include "mid_tiles.h"

#include <algorithm>
#include <stdexcept>
#include <string>

#include "mid.h"

namespace pe {

namespace {

// M0's share of l low stones in a tile with a - b = d
int low0(int l, int d) { return (l - d + 1) >> 1; }   // ceil((l - d) / 2), floor shift

int class_count(int low, int d, int l) {
  const int la = low0(l, d), lb = l - la;
  return la < 0 || lb < 0 || l < 0 || l > low ? 0 : choose_host(low, l) * choose_host(l, la);
}

// Entries of the half with levels n = parity (mod 2) of a tile (a, b), 0 if nothing reads it.
int half_entries(int low, int a, int b, int parity) {
  if ((parity ? a : b) == 0) return 0;
  int t = 0;
  for (int l = 0; l <= low; l++)
    if (((a + b + l) & 1) == parity) t += class_count(low, a - b, l);
  return t;
}
bool tile_empty(int low, int d) {
  for (int l = 0; l <= low; l++)
    if (class_count(low, d, l)) return false;
  return true;
}

// Free extents of the entry space, lowest first; whole tiles are taken from as many extents as
// it needs.
struct Extents {
  std::vector<std::pair<int64_t, int64_t>> free;   // (first, entries)
  // n tiles of `tile` entries each: their first entries, or false with nothing taken
  bool take(int64_t tile, int64_t n, std::vector<uint32_t>* out) {
    const auto before = free;
    out->clear();
    for (auto& f : free)
      while (int64_t(out->size()) < n && f.second >= tile) {
        out->push_back(uint32_t(f.first));
        f.first += tile;
        f.second -= tile;
      }
    if (int64_t(out->size()) < n) {
      free = before;
      return false;
    }
    return true;
  }
  void give(int64_t tile, const std::vector<uint32_t>& at, int64_t border) {
    int64_t end = -1;   // of the run before: tiles taken from one extent follow each other
    for (uint32_t x : at) {
      if (int64_t(x) == end && end != border) free.back().second += tile;
      else free.emplace_back(int64_t(x), tile);
      end = int64_t(x) + tile;
    }
    std::sort(free.begin(), free.end());
    std::vector<std::pair<int64_t, int64_t>> m;
    for (const auto& f : free) {
      if (!f.second) continue;
      // the workspace and the spill area are two memory ranges
      if (!m.empty() && m.back().first + m.back().second == f.first && f.first != border) m.back().second += f.second;
      else m.push_back(f);
    }
    free.swap(m);
  }
};

struct Placed { int a = 0, b = 0; std::vector<uint32_t> half[2]; };

// The steps of one spots value: groups (a, b) of one layer a + b, in order of a, as many to a
// step as the memory holds; a step frees the halves that only its groups read.
bool plan_steps(int spots, bool down, std::vector<std::vector<Placed>>* steps) {
  const int low = mid_low_cells(spots), high = spots - low;
  const int64_t work = mid_work_entries(spots);
  Extents X;
  X.free.emplace_back(0, work);
  if (mid_spill_entries(spots) > 0) X.free.emplace_back(work, mid_spill_entries(spots));
  std::vector<Placed> live;
  steps->clear();
  for (int h = high; h >= 0; h--) {
    std::vector<std::pair<int, int>> todo;
    for (int i = 0; i <= h; i++) {
      const int a = down ? h - i : i;
      if (!tile_empty(low, 2 * a - h)) todo.emplace_back(a, h - a);
    }
    for (size_t at = 0; at < todo.size();) {
      std::vector<Placed> step;
      for (; at < todo.size(); at++) {
        Placed g;
        g.a = todo[at].first;
        g.b = todo[at].second;
        const int64_t n = int64_t(choose_host(high, h)) * choose_host(h, g.a);
        int64_t size[2];
        bool ok = true;
        for (int par = 0; par < 2 && ok; par++) {
          size[par] = half_entries(low, g.a, g.b, par);
          if (size[par] && !X.take(size[par], n, &g.half[par])) {
            if (par) X.give(size[0], g.half[0], work);
            ok = false;
          }
        }
        if (!ok) break;
        step.push_back(std::move(g));
      }
      if (step.empty()) return false;
      for (const Placed& g : step)
        for (Placed& c : live)
          for (int par = 0; par < 2; par++)
            if (c.a == g.a + par && c.b == g.b + 1 - par && !c.half[par].empty()) {
              X.give(half_entries(low, c.a, c.b, par), c.half[par], work);
              c.half[par].clear();
            }
      for (const Placed& g : step) live.push_back(g);
      steps->push_back(std::move(step));
    }
  }
  return true;
}

MidTabsHost build() {
  MidTabsHost T;
  std::vector<uint32_t> code3(size_t(1) << (kMidSpots - kTileCells));   // base-3 value of a mask
  for (uint32_t m = 0; m < code3.size(); m++) {
    uint32_t c = 0;
    for (int i = kMidSpots - kTileCells - 1; i >= 0; i--) c = 3 * c + (m >> i & 1);
    code3[m] = c;
  }
  // classes: members in order of (A, B), children by rank
  std::vector<uint32_t> members;   // A | B << 16
  T.classes.assign(size_t(mid_class_row(kTileCells, 11, 8)) + 1, MidClass{{0, 0}});
  for (int low = 0; low <= kTileCells; low++) {
    int at[kTileCells + 2][kTileCells + 2];
    std::vector<int> rank(size_t(1) << (2 * low));   // of (A, B) in its class
    for (auto& r : at)
      for (int& x : r) x = -1;
    for (int la = 0; la <= low; la++)
      for (int lb = 0; la + lb <= low; lb++) {
        at[la][lb] = int(members.size());
        int k = 0;
        for (uint32_t A = 0; A < 1u << low; A++)
          for (uint32_t B = 0; B < 1u << low; B++)
            if (!(A & B) && __builtin_popcount(A) == la && __builtin_popcount(B) == lb) {
              rank[A << low | B] = k++;
              members.push_back(A | B << 16);
            }
      }
    T.kids.resize(2 * members.size());
    for (int la = 0; la <= low; la++)
      for (int lb = 0; la + lb <= low; lb++) {
        const int n = choose_host(low, la + lb) * choose_host(la + lb, la);
        for (int m = 0; m < 2; m++)
          for (int r = 0; r < n; r++) {
            const uint32_t A = members[size_t(at[la][lb] + r)] & 0xffff, B = members[size_t(at[la][lb] + r)] >> 16;
            Kids k{};
            int j = 0;
            for (int c = 0; c < low; c++)
              if (!((A | B) >> c & 1))
                k.rank16[j++] = uint16_t(16 * (m ? rank[A << low | (B | 1u << c)] : rank[(A | 1u << c) << low | B]));
            k.mem = uint16_t(A | B << 8);
            T.kids[size_t(2 * at[la][lb] + m * n + r)] = k;
          }
      }
    auto start = [&](int d, int l) {
      int n = 0;
      for (int k = l - 2; k >= 0; k -= 2) n += class_count(low, d, k);
      return n;
    };
    for (int d = -11; d <= 11; d++) {
      int entries = 0;
      for (int l = 0; l <= low; l++) {
        const int n = class_count(low, d, l);
        if (!n) continue;
        if (n > kTileClass || (entries += n) > kTileEntries) throw std::runtime_error("midsolve tile sizes");
        T.classes[size_t(mid_class_row(low, d, l))] =
            MidClass{{uint32_t(n) | uint32_t(at[low0(l, d)][l - low0(l, d)]) << 8, uint32_t(start(d, l))}};
      }
    }
  }
  // tiles
  T.sched.resize(kMidSpots + 1);
  for (int spots = 0; spots <= kMidSpots; spots++) {
    MidSched& S = T.sched[size_t(spots)];
    S = MidSched{};
    S.low = mid_low_cells(spots);
    S.high = spots - S.low;
    S.work_entries = int32_t(mid_work_entries(spots));
    std::vector<std::vector<Placed>> steps, other;
    const bool up = plan_steps(spots, false, &steps), dn = plan_steps(spots, true, &other);
    if (dn && (!up || other.size() < steps.size())) steps.swap(other);
    // prep and the steps are at most as many launches as prep and one per level
    if ((!up && !dn) || int(steps.size()) > spots + 1)
      throw std::runtime_error("midsolve tiles of " + std::to_string(spots) + " cells do not fit");
    S.steps = int32_t(steps.size());
    S.tiles = int32_t(T.tiles.size());
    S.bases = int32_t(T.bases.size() / 2);
    int codes = 1;
    for (int i = 0; i < S.high; i++) codes *= 3;
    T.bases.resize(T.bases.size() + 2 * size_t(codes), kNotStored);
    for (size_t k = 0; k < steps.size(); k++) {
      S.first[k] = int32_t(T.tiles.size()) - S.tiles;
      for (const Placed& g : steps[k]) {
        size_t i = 0;
        for (uint32_t p = 0; p < 1u << S.high; p++) {
          if (__builtin_popcount(p) != g.a) continue;
          const uint32_t rest = ((1u << S.high) - 1) & ~p;
          uint32_t q = rest;   // the subsets of rest in ascending order, 0 first
          do {
            q = (q - rest) & rest;
            if (__builtin_popcount(q) != g.b) continue;
            const uint32_t code = code3[p] + 2 * code3[q];
            for (int par = 0; par < 2; par++)
              if (!g.half[par].empty()) T.bases[2 * (size_t(S.bases) + code) + size_t(par)] = g.half[par][i];
            T.tiles.push_back(MidTile{p, q, code, 0});
            i++;
          } while (q != rest);
        }
      }
    }
    S.first[steps.size()] = int32_t(T.tiles.size()) - S.tiles;
  }
  return T;
}

}  // namespace

MidTabs MidTabsHost::view() const {
  return MidTabs{sched.data(), tiles.data(), bases.data(), classes.data(), kids.data()};
}

std::vector<uint32_t> mid_records(const MidTabs& M) {
  int64_t tiles = 0;
  for (int spots = 0; spots <= kMidSpots; spots++) tiles += M.sched[spots].first[M.sched[spots].steps];
  std::vector<uint32_t> out(size_t(kRecWords * tiles));
  mid_records(M, 0, tiles, out.data());
  return out;
}

void mid_records(const MidTabs& M, int64_t first, int64_t n, uint32_t* r) {
  std::fill(r, r + kRecWords * n, 0u);
  for (int spots = 0; spots <= kMidSpots; spots++) {
    const MidSched& S = M.sched[spots];
    const int begin = int(std::max<int64_t>(S.tiles, first));
    const int end = int(std::min<int64_t>(S.tiles + S.first[S.steps], first + n));
    if (begin >= end) continue;
    const uint32_t* bases = M.bases + 2 * size_t(S.bases);
    uint32_t sizes[23] = {}, counts[23][2] = {};   // by d + 11
    for (int d = -11; d <= 11; d++)
      for (int l = 0; l <= S.low; l++) {
        const uint32_t n = uint32_t(M.classes[mid_class_row(S.low, d, l)].count());
        sizes[d + 11] += n << (l & 1 ? 16 : 0);
        counts[d + 11][l / 4] |= n << (8 * (l % 4));
      }
    for (int t = begin; t < end; t++, r += kRecWords) {
      const MidTile& X = M.tiles[t];
      const int d = __builtin_popcount(X.p) - __builtin_popcount(X.q) + 11;
      r[0] = X.p | X.q << 16;
      for (int par = 0; par < 2; par++) r[kRecOwn + par] = bases[2 * X.code + uint32_t(par)];
      r[kRecSizes] = sizes[d];
      r[kRecCounts] = counts[d][0];
      r[kRecCounts + 1] = counts[d][1];
      uint32_t c3 = 1;
      for (int c = 0, j = 0; c < S.high; c++, c3 *= 3) {
        if ((X.p | X.q) >> c & 1) continue;
        r[kRecUp + j] = bases[2 * (X.code + c3) + 1];
        r[kRecUp + kRecUp1 + j] = bases[2 * (X.code + 2 * c3)];
        j++;
      }
    }
  }
}

std::vector<KidRanks> mid_kid_ranks(const MidTabs& M) {
  std::vector<KidRanks> out(size_t(mid_kid_row(kTileCells + 1, -11, 0)), KidRanks{{0, 0}});
  for (int low = 0; low <= kTileCells; low++)
    for (int d = -11; d <= 11; d++)
      for (int l = 0; l <= low; l++) {
        const MidClass& c = M.classes[mid_class_row(low, d, l)];
        for (int r = 0; r < c.count(); r++) {
          const Kids& k = M.kids[2 * c.members() + ((d + l) & 1) * c.count() + r];
          KidRanks& o = out[size_t(mid_kid_row(low, d, l) + r)];
          o.w[1] = uint32_t(k.mem) << 16;
          for (int j = 0; j < low - l; j++) o.w[j / 4] |= uint32_t(k.rank16[j] / 16) << (8 * (j % 4));
        }
      }
  return out;
}

int64_t mid_work_entries(int spots) { return bottleneck(spots); }

// Part of the plans' memory contract (pe_mid_schedule_info reports it, budgets are checked
// against it): what per-level tables over the subsets of each side would take, 256 bytes a
// subset of the mover and 32 a subset of the other side, with masks and 16-bit remaps.
int64_t mid_table_area_bytes(int spots) {
  auto up = [](int64_t x) { return (x + 255) & ~int64_t(255); };
  int64_t set0 = 0, wins1 = 0, remap = 0, masks = 0;
  for (int n = 0; n <= spots; n++) {
    const int k0 = n >> 1, k1 = n - k0;
    set0 += choose_host(spots, k0);
    wins1 += choose_host(spots, k1);
    masks += choose_host(spots - k0, k1);
    remap += int64_t(choose_host(spots - k0, k1)) * (spots - k0);
  }
  return up(256 * set0) + up(32 * wins1) + up(2 * remap) + up(4 * masks);
}
int64_t mid_spill_entries(int spots) { return mid_table_area_bytes(spots) / 32 - (int64_t(2) << spots); }

const MidTabsHost& mid_tabs() {
  static const MidTabsHost T = build();
  return T;
}

}  // namespace pe
