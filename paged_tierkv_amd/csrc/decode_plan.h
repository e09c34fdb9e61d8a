// Wave and split counts of a decode launch and the layout of its workspace
// (host code without HIP, also compiled by a CPU test).
#pragma once

#include <algorithm>
#include <cstdint>

namespace tierkv {

constexpr int FBS = 16;            // tokens per block on the fast path
constexpr int MAX_LIST = 512;      // resident blocks per workgroup (LDS list)
constexpr int MAX_WAVES = 8;
constexpr int PRE_CHUNKS = 4;      // table-row chunks loaded together by the list build
constexpr int MERGE_UNROLL = 8;    // split partials loaded together by the merge
constexpr int MAX_LDS_STAGE = 48 * 1024;   // bytes of per-block score statistics kept in LDS
constexpr int MAX_SPLIT_UNITS = 1 << 16;   // units per launch when a unit is split

struct Plan {
  int nw;
  int splits;
};

inline bool fast_path_ok(int block_size, int head_dim, int groups) {
  return block_size == FBS && (head_dim == 64 || head_dim == 128) && groups >= 1 && groups <= 16;
}

// The fewest splits whose lists hold any row of num_blocks: a split's list
// holds ceil(hot / splits) + ceil(warm / splits) entries, at most
// ceil(num_blocks / splits) + 1; MAX_LIST - 1 blocks per split keep the HOT
// (front) and WARM (back) halves of the list apart.
inline int min_splits(int num_blocks) { return std::max(1, (num_blocks + MAX_LIST - 2) / (MAX_LIST - 1)); }

// Splits of a launch in the smallest workspace that is accepted: the hint, or
// enough to put about 2048 waves on the chip with at least four tiles per
// wave.  (A launch takes the plan below when its workspace has room.)
inline int required_splits(int64_t units, int num_blocks, int groups, int splits_hint) {
  const int nw = groups <= 8 ? 8 : 4;
  int64_t splits = splits_hint;
  if (splits_hint <= 0) {
    splits = std::max<int64_t>(1, (2048 + units * nw - 1) / (units * nw));
    splits = std::min<int64_t>(splits, std::max(1, num_blocks / (4 * nw)));
    if (num_blocks < 12 * nw) splits = 1;
  }
  splits = std::max<int64_t>(splits, min_splits(num_blocks));
  return int(std::max<int64_t>(1, std::min<int64_t>(splits, num_blocks)));
}

// Expected time (us, less the launch itself) of a launch with nw waves per
// workgroup and s splits per unit.  A CU moves about 26 B/ns whether one or
// two workgroups and four or eight waves stream on it, so what counts is how
// many workgroups the busiest CU gets, how many of them run together (by
// registers: one of eight waves at head_dim 128, two at 64; twice as many of
// four), and each pass's fixed part (list build, first loads, wave merge).
// A split adds its publication, arrival and merge, and with score sums the
// finalisation launch.  The constants are a fit to 6,192 timings (16
// unit counts from 4 to 1024, ten row lengths from 9 to 2048 blocks, up to 12
// split counts, both wave counts and head dims, with and without score sums;
// 10 % HOT, 60 % WARM): over these shapes the plan chosen by it is on average
// 1 % slower than the fastest measured one, where aiming at 2048 waves with
// eight per workgroup was 15 % slower (head_dim 64: 9 %, with score sums 17 %;
// up to 2.1x: 248 units made 496 workgroups of 256 that fit at a time).
inline double plan_cost(int64_t units, int num_blocks, int head_dim, bool scores, int nw, int s) {
  const double per_block = head_dim == 64 ? 0.038 : 0.091;   // a block's tiles at a CU's rate
  const double per_wave = 0.231;                             // a block's round trips in one wave
  const double fixed = nw == 4 ? 6.0 : 6.4;
  const int64_t room = (head_dim == 64 ? 2 : 1) * (nw == 4 ? 2 : 1);
  const int64_t on_cu = (units * s + 255) / 256;
  const int64_t passes = (on_cu + room - 1) / room;
  const double refill = room == 1 ? 1.0 : nw == 4 ? 1.8 : 0.3;   // a further pass against the first
  const double blocks = double(num_blocks) / s;
  // One pass with so many workgroups together on the CU.  Four waves alone
  // stream 3 % slower than eight (256 units of 1024 blocks: 145 against 141
  // us), three workgroups of four where four fit (head_dim 64) 8 % (632
  // units of 496 blocks: 88.8 against 81.8).
  auto pass = [&](int64_t together) {
    const double slower = nw == 4 && together == 1 && s == 1 ? 1.03 : nw == 4 && room == 4 && together == 3 ? 1.08 : 1.0;
    return std::max(slower * per_block * blocks * together, per_wave * blocks / nw);
  };
  double t = fixed + (passes - 1) * (fixed * refill + pass(std::min(on_cu, room))) +
             pass(on_cu - (passes - 1) * room);
  if (s > 1)
    t += 1.7 + (scores ? (nw == 4 ? 4.9 : 4.1) : 0.0) + 1.5 * ((s + MERGE_UNROLL - 1) / MERGE_UNROLL) +
         0.3 * (std::min(on_cu, room) - 1);
  // Rows longer than one pass of the list build (with score sums, the blanks
  // of the later passes are written one by one).
  t += ((num_blocks - 1) / (PRE_CHUNKS * nw * 64)) * (scores ? 3.5 : 1.0);
  return t;
}

// Split counts a plan may take: at most MAX_PLAN_GRID workgroups, four blocks
// per split.
constexpr int PLAN_SPLITS[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 24, 32};
constexpr int64_t MAX_PLAN_GRID = 1024;
inline bool plan_split_ok(int64_t units, int num_blocks, int s) {
  return s == 1 || (units * s <= MAX_PLAN_GRID && s <= num_blocks / 4);
}

struct WsLayout {
  int64_t err, cnt, acc, ml, stage, total;
};

inline WsLayout ws_layout(int batch, int num_heads, int kv_heads, int num_blocks, int block_size,
                          int head_dim, bool scores, int splits) {
  WsLayout l{};
  const int groups = num_heads / std::max(kv_heads, 1);
  auto up = [](int64_t x) { return (x + 255) & ~int64_t(255); };
  l.err = 0;
  int64_t off = 256;
  if (fast_path_ok(block_size, head_dim, groups)) {
    const int64_t units = int64_t(batch) * kv_heads;
    // The arrival counters come first and have the same place and size in
    // every layout, so a launch of any shape finds them zero.
    l.cnt = off;
    off = up(off + int64_t(MAX_SPLIT_UNITS) * 4);
    l.acc = off;
    if (splits > 1) off = up(off + units * splits * groups * head_dim * 4);
    l.ml = off;
    if (splits > 1) off = up(off + units * splits * groups * 2 * 4);
    l.stage = off;
    if (scores) off = up(off + int64_t(batch) * num_heads * num_blocks * 2 * 4);
  } else {
    l.cnt = l.acc = l.ml = l.stage = off;
  }
  l.total = off;
  return l;
}

// Bytes of the smallest workspace that a launch is accepted with.
inline int64_t least_workspace(int batch, int num_heads, int kv_heads, int num_blocks, int block_size, int head_dim,
                               bool scores, int splits_hint) {
  const int splits = required_splits(int64_t(batch) * kv_heads, num_blocks, num_heads / kv_heads, splits_hint);
  return ws_layout(batch, num_heads, kv_heads, num_blocks, block_size, head_dim, scores, splits).total;
}

// Wave and split counts of a fast-path launch: the cheapest by plan_cost whose
// workspace fits workspace_bytes (that of required_splits always does); a
// split hint fixes the splits.  GQA groups above 8 take four waves, to bound
// the LDS accumulators.
// The plan decides in which groups a deterministic launch adds its partial
// sums, so its output's bits are the plan's: such a launch takes the free plan
// in every workspace with room for it, and in every smaller one the plan of
// the smallest (not the best that fits, which would change with each size).
inline Plan plan_launch(int batch, int num_heads, int kv_heads, int num_blocks, int block_size, int head_dim,
                        bool scores, int splits_hint, bool deterministic, int64_t workspace_bytes) {
  const int groups = num_heads / kv_heads;
  const int64_t units = int64_t(batch) * kv_heads;
  auto bytes = [&](int s) {
    return ws_layout(batch, num_heads, kv_heads, num_blocks, block_size, head_dim, scores, s).total;
  };
  auto cheapest = [&](int64_t room) -> Plan {
    Plan best{4, required_splits(units, num_blocks, groups, splits_hint)};
    double best_cost = 1e300;
    auto consider = [&](int s) {
      for (int nw = 8; nw >= 4; nw -= 4) {
        if (nw == 8 && groups > 8) continue;
        const double c = plan_cost(units, num_blocks, head_dim, scores, nw, s);
        if (c < best_cost) {
          best_cost = c;
          best = Plan{nw, s};
        }
      }
    };
    consider(best.splits);
    if (splits_hint > 0) return best;
    const int lo = min_splits(num_blocks);
    for (int s : PLAN_SPLITS) {
      if (s < lo || !plan_split_ok(units, num_blocks, s)) continue;
      if (bytes(s) > room) break;
      consider(s);
    }
    return best;
  };
  if (!deterministic) return cheapest(workspace_bytes);
  const Plan best = cheapest(INT64_MAX);
  if (bytes(best.splits) <= workspace_bytes) return best;
  return cheapest(
      least_workspace(batch, num_heads, kv_heads, num_blocks, block_size, head_dim, scores, splits_hint));
}

// Splits that the reported workspace has room for: whatever plan_launch may
// take for this many blocks or fewer.
inline int reported_splits(int64_t units, int num_blocks, int groups, int splits_hint) {
  int splits = required_splits(units, num_blocks, groups, splits_hint);
  if (splits_hint <= 0)
    for (int s : PLAN_SPLITS)
      if (plan_split_ok(units, num_blocks, s)) splits = std::max(splits, s);
  return splits;
}

}  // namespace tierkv
