// Tile order and launch rules of the MXFP8 GEMM: which tile a product takes, how many workgroups walk its
// tiles, which tile a workgroup walks when, what a run of tiles reads. Plain C++ without HIP (the constexpr
// functions serve the kernels too), so that the rules are checked over their whole range on the CPU.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace wanmi {

constexpr int TN = 256;      // weight rows (output features) per tile
constexpr int TM = 256;      // tokens per tile
constexpr int TS = 128;      // features and tokens of the small tile
constexpr int kGroupM = 4;   // 256-token m tiles per group (4: the XCD's 32 concurrent tiles are 4 m x 8 n)
constexpr int kTsGroupM = 8;  // m tiles per group of the 128 x 128 tiles' order

// ------------------------------------------------------------------------------------------------
// Tile order
// ------------------------------------------------------------------------------------------------
// Position of tile number v in the order: XCD v & 7 takes a contiguous run of it.
constexpr int run_position(int v, int total) {
  const int x = v & 7, r = total & 7;
  return x * (total >> 3) + (x < r ? x : r) + (v >> 3);
}

struct TileAt {
  int tm, tn;
};
// Tile number v of tiles_m x tiles_n: the order walks groups of `group` m tiles along n.
constexpr TileAt tile_at(int v, int tiles_m, int tiles_n, int group) {
  const int pid = run_position(v, tiles_m * tiles_n);
  const int in_group = group * tiles_n;
  const int first_m = pid / in_group * group;
  const int left = tiles_m - first_m, gsz = left < group ? left : group;
  return TileAt{first_m + (pid % in_group) % gsz, (pid % in_group) / gsz};
}

// What the run of tiles of XCD `x` reads: its token rows [m_lo, m_hi) and n tiles, [n0, n0 + n_hi) and, over
// several groups, [0, n_lo) (kGroup m tiles of kTm tokens per group).
struct RunPanels {
  int64_t m_lo, m_hi;
  int n0, n_hi, n_lo;
};
template <int kTm, int kGroup>
constexpr RunPanels run_panels(int64_t M, int tiles_m, int tiles_n, int x) {
  const int total = tiles_m * tiles_n, r = total & 7;
  const int first = x * (total >> 3) + (x < r ? x : r), tiles = (total >> 3) + (x < r ? 1 : 0);
  if (tiles == 0) return RunPanels{0, 0, 0, 0, 0};
  const int in_group = kGroup * tiles_n, last = first + tiles - 1;
  const int g0 = first / in_group, g1 = last / in_group;
  const int s0 = tiles_m - g0 * kGroup, s1 = tiles_m - g1 * kGroup;  // m tiles of the groups
  const int tn0 = first % in_group / (s0 < kGroup ? s0 : kGroup), tn1 = last % in_group / (s1 < kGroup ? s1 : kGroup);
  const int64_t m_end = (int64_t)(g1 + 1) * kGroup * kTm;
  // the first group's n tiles from tn0 on, the last group's up to tn1; a group between walks all of them
  const int n_lo = g1 - g0 > 1 || tn1 + 1 > tn0 ? tn0 : tn1 + 1;
  return RunPanels{(int64_t)g0 * kGroup * kTm, m_end < M ? m_end : M, tn0, g0 == g1 ? tn1 - tn0 + 1 : tiles_n - tn0,
                   g0 == g1 ? 0 : n_lo};
}

// ------------------------------------------------------------------------------------------------
// Launch rules
// ------------------------------------------------------------------------------------------------
// Which tile a product of M tokens takes on `cus` CUs (one workgroup each), and at what cost.
struct TilePlan {
  int nj;      // token fragments per wave of the 256-feature kernel (tiles of 64 nj tokens); 0: 128 x 128 tiles
  int64_t cost;
  int qk_wgs;  // Q|K and V in one launch on 256-feature tiles: workgroups of the Q|K part
};

// Every CU takes one tile at a time, so a product costs its rounds of `cus` tiles times one tile's
// time, which is the same for all full tiles of a kind but not proportional to the tile: the loads
// bound it, and a smaller tile needs more of them per flop. Measured per k stage in rounds of 5120 x
// 5120 (one to twenty rounds): 256 x 256 tiles 1.30-1.60 us, 192 tokens x 256 1.05-1.25, 128 x 256
// 0.87-0.97, 128 x 128 0.55-0.58; K = 13824 and the GELU epilogue give the same ratios within 3%. A
// smaller tile pays where it saves a round or fills the only one: 5120 x 5120 at 512 tokens 54 -> 23 us
// (128 x 128), 1024 55 -> 37 (128 x 256), 1560 57 -> 47 (192), 3120 119 -> 83 (128 x 256), 4100 122 ->
// 101 (192); at 5500 tokens 130 against 146 (192) and at 16380 338 against 364, the 256 x 256 tile.
constexpr int kTileCost[5] = {40, 0, 67, 82, 100};  // by nj (0: 128 x 128 tiles)

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Best tile for n output columns (a multiple of 256); a larger tile wins a tie. V^T columns are
// written for whole tiles only, so tiles that end before vt_ld are not taken.
inline TilePlan select_tile(int64_t M, int64_t n, int64_t cus, int64_t vt_ld) {
  TilePlan best{4, kTileCost[4] * ceil_div(ceil_div(M, 256) * (n / TN), cus), 0};
  for (int nj : {3, 2, 0}) {
    const int64_t tm = nj ? 64 * nj : TS, tn = nj ? TN : TS;
    const int64_t mt = ceil_div(M, tm);
    if (mt * tm < vt_ld) continue;
    const int64_t cost = kTileCost[nj] * ceil_div(mt * (n / tn), cus);
    if (cost < best.cost) best = TilePlan{nj, cost, 0};
  }
  return best;
}

// The same for Q|K (qk columns) and V (v columns) in one launch: on 256-feature tiles the CUs are split
// between the two parts so that the longer one is shortest, neither part with more of them than it has tiles;
// 128 x 128 tiles mix freely. The first such split is taken. Where a part's count is no multiple of 8 its later tiles
// leave its XCDs' runs; whole eights at the same cost helped or hurt by what else the split changed (10240 + 5120
// columns: 1560 tokens 124.5 -> 121.5 us, 1200 104.8 -> 102.9, 3600 258 -> 263, nine other counts within 1%).
inline TilePlan select_qkv_tile(int64_t M, int64_t qk, int64_t v, int64_t cus, int64_t vt_ld) {
  TilePlan best{4, INT64_MAX, 0};
  for (int nj : {4, 3, 2, 0}) {
    const int64_t tm = nj ? 64 * nj : TS;
    const int64_t mt = ceil_div(M, tm);
    if (mt * tm < vt_ld) continue;
    if (nj == 0) {
      const int64_t cost = kTileCost[0] * ceil_div(mt * ((qk + v) / TS), cus);
      if (cost < best.cost) best = TilePlan{0, cost, 0};
      continue;
    }
    const int64_t tq = mt * (qk / TN), tv = mt * (v / TN);
    if (tq + tv <= cus) {  // one tile per workgroup
      if (kTileCost[nj] < best.cost) best = TilePlan{nj, kTileCost[nj], (int)tq};
      continue;
    }
    if (cus < 2) continue;  // no CU for one of the parts
    // The fewest rounds in which both parts fit: from the rounds of all tiles on, one or two steps.
    int64_t rounds = ceil_div(tq + tv, cus);
    while (ceil_div(tq, rounds) + ceil_div(tv, rounds) > cus) ++rounds;
    const int64_t cost = kTileCost[nj] * rounds;
    if (cost < best.cost) best = TilePlan{nj, cost, (int)std::max(ceil_div(tq, rounds), cus - tv)};
  }
  return best;
}

// Workgroups that compute tiles: 128 x 128 tiles one each, 256-feature tiles one per CU at most, a round at
// a time (workgroup w of a part of n walks tiles w, w + n, ...).
inline int64_t tile_workgroups(const TilePlan& plan, int64_t tiles, int64_t cus) {
  return plan.nj == 0 ? tiles : std::min(tiles, cus);
}

// Workgroups per XCD that fetch ahead of a product of one round: as many as walk the longest run's panels at
// twice the tiles' pace, one CU touching about 900 lines per us and a k stage (one line per row) taking the
// tiles of nj `kStageNs`; none if the idle CUs cannot at least keep pace. 1000 tokens, 13824 deep, 0 / 2 / 3 /
// 4 / 5 / 6 / 8 of them: 120 / 117 / 108 / 92 / 87 / 89 / 91 us; 512 tokens 72 / 74 / 70 / 61 / 54 / 50 / 51;
// four where the rule asks for thirteen (2000 tokens) 127 -> 212. Not with 256 x 256 tiles, whose MFMAs take
// as long as the loads (216 tiles: 56.5 -> 58.2 us).
// (Those figures with the weights in memory. n workgroups of an XCD share its path: 2, 4, 6, 9 of them touch 1750,
// 3190, 4200, 5110 lines per us where tiles overtake them. Nine at 900 each seem to keep pace with the deep run
// that 1025 to 1152 tokens of 5120 columns have, and do not: with the weights in the caches 1100 tokens take 45 us
// with them and 37 without, 13824 deep 130 and 91. From memory, as a model's layers come, it is 44.5 and 48.9,
// and 125 and 118; 1152 tokens 43.9 and 51.9, 124 and 125: there they stay.)
constexpr int kStageNs[5] = {560, 0, 920, 1100, 0};

template <int kTm, int kTn, int kGroup>
inline int64_t fetch_wgs(int64_t M, int tiles_m, int tiles_n, int64_t idle, int nj) {
  int64_t lines = 0;
  for (int x = 0; x < 8; ++x) {
    const RunPanels p = run_panels<kTm, kGroup>(M, tiles_m, tiles_n, x);
    lines = std::max(lines, p.m_hi - p.m_lo + (int64_t)(p.n_hi + p.n_lo) * kTn);
  }
  const int64_t pace = 900 * kStageNs[nj] / 1000;  // lines per stage and workgroup
  const int64_t n = std::min(idle, (2 * lines + pace / 2) / pace);
  return n * pace >= lines ? n : 0;
}

}  // namespace wanmi
