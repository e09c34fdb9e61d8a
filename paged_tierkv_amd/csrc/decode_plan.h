// Wave and split counts of a decode launch and the layout of its workspace
// (host code without HIP, also compiled by a CPU test).
#pragma once

#include <algorithm>
#include <cstdint>

#include "tierkv_hip.h"

namespace tierkv {

constexpr int FBS = 16;            // tokens per block on the fast path
constexpr int MAX_LIST = 512;      // resident blocks per workgroup (LDS list)
constexpr int MAX_WAVES = 8;
constexpr int PRE_CHUNKS = 4;      // table-row chunks loaded together by the list build
constexpr int MERGE_UNROLL = 8;    // split partials loaded together by the merge
constexpr int MAX_LDS_STAGE = 48 * 1024;   // bytes of per-block score statistics kept in LDS
// Where a score launch stages each block's (max, sum) per head:
//   STAGE_LDS_BLOCK LDS [G][num_blocks] by logical block (unsplit launches),
//                   finalised by the workgroup itself;
//   STAGE_LDS_LIST  LDS [G][MAX_LIST] by list position, copied to the
//                   workspace [B][H][num_blocks] at the end of the workgroup
//                   (split launches);
//   STAGE_GLOBAL    the workspace, written per tile (rows too long for LDS).
// The workspace stages are finalised by finalize_scores_kernel, launched
// after the decode kernel: one workgroup per (sequence, q head) row spreads
// that work over the chip, where a unit's last workgroup would read every
// staged pair of the unit and write its whole score rows from one CU.
constexpr int STAGE_GLOBAL = 0;
constexpr int STAGE_LDS_BLOCK = 1;
constexpr int STAGE_LDS_LIST = 2;
constexpr int MAX_SPLIT_UNITS = 1 << 16;   // units per launch when a unit is split
constexpr int CUS = 256;           // compute units of the GPU, 32 in each of 8 XCDs
constexpr int CU_LDS = 160 * 1024; // bytes of LDS per compute unit

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

// The stage of a launch: unsplit score launches keep the statistics in LDS
// (up to MAX_LDS_STAGE bytes per workgroup) and finalise them in the workgroup;
// split ones stage them in LDS by list position.
inline int score_stage(bool scores, int groups, int num_blocks, int splits) {
  const int64_t pair = 2 * int64_t(sizeof(float));
  if (!scores) return STAGE_GLOBAL;
  if (splits == 1) return int64_t(groups) * num_blocks * pair <= MAX_LDS_STAGE ? STAGE_LDS_BLOCK : STAGE_GLOBAL;
  return groups * MAX_LIST * pair <= MAX_LDS_STAGE ? STAGE_LDS_LIST : STAGE_GLOBAL;
}

// LDS of a workgroup: the wave accumulators and the stage, beside the kernel's
// own arrays (the list and the waves' counts and sums).
constexpr int STATIC_LDS = 9728;
inline int64_t dynamic_lds(int nw, int groups, int head_dim, int num_blocks, int stage) {
  int64_t bytes = int64_t(nw) * groups * head_dim * int64_t(sizeof(float));
  if (stage == STAGE_LDS_BLOCK) bytes += int64_t(groups) * num_blocks * 2 * int64_t(sizeof(float));
  if (stage == STAGE_LDS_LIST) bytes += int64_t(groups) * MAX_LIST * 2 * int64_t(sizeof(float));
  return bytes;
}

// Waves of the decode kernel that a SIMD's 512 vector registers hold: 206 to
// 230 registers at head_dim 128, at head_dim 64 127 in the absmax format and
// 132 to 151 in the reference format or with score sums.
inline int waves_per_simd(int head_dim, int warm_format, bool scores) {
  if (head_dim == 128) return 2;
  return warm_format == TIERKV_WARM_ABSMAX_I8 && !scores ? 4 : 3;
}

// Workgroups of nw waves that run together on a CU (four SIMDs).  A score launch of a large group at head_dim 64 is held to fewer by
// its statistics than by registers.
inline int64_t workgroups_per_cu(int num_blocks, int groups, int head_dim, int warm_format, bool scores, int nw,
                                 int s) {
  const int64_t by_registers = 4 * waves_per_simd(head_dim, warm_format, scores) / nw;
  const int64_t lds = STATIC_LDS + dynamic_lds(nw, groups, head_dim, num_blocks,
                                               score_stage(scores, groups, num_blocks, s));
  return std::max<int64_t>(1, std::min(by_registers, CU_LDS / lds));
}

// Expected time (us, less the launch itself) of a launch with nw waves per
// workgroup and s splits per unit: what counts is how many workgroups the
// busiest CU gets, how many of them run together (workgroups_per_cu), their
// blocks' time, and what is fixed in each pass (list build, first loads, wave
// merge) and in each split (publication, arrival, merge, and with score sums
// the finalisation launch).
// The constants are one least-squares fit (of the logarithm) to 17,589
// timings: 1,336 shapes of 1 to 1024 units, 8 to 2048 blocks, GQA groups 1 to
// 16, both head dims and formats, with and without score sums, 5 to 30 % HOT
// and 40 to 65 % WARM, each with both wave counts and up to 13 split counts,
// in graphs over four layers' buffers.  The plan chosen by it is on average
// 0.6 % slower than the fastest measured one, also over 1,200 further shapes
// that the fit has not seen; the plain rule of required_splits with the most
// waves is 15 % slower, up to 3.5 times (units * s just above what runs at
// once).  1 shape in 60 is more than 3 % slower than with it (worst
// 1.12 times).
inline double plan_cost(int64_t units, int num_blocks, int groups, int head_dim, int warm_format, bool scores, int nw,
                        int s) {
  // A block's tiles in a workgroup, alone or sharing its CU: 256 units, D =
  // 128, 10 % HOT, 60 % WARM (3.3 KB per block) take 25.6 us at 144 blocks and
  // 58.3 at 400, 0.128 per block (26 B/ns; smaller launches are served by the
  // caches in part).  Four waves alone at D = 64 have too few loads in flight
  // (64 units of 256 blocks: 25.1 us, 18.6 with eight).
  const double per_block = head_dim == 64 ? 0.063 : 0.117;
  const double alone = head_dim == 64 && nw == 4 ? 1.38 : 1.0;
  const double fixed = head_dim == 64 ? (nw == 4 ? 4.19 : 4.97) : (nw == 4 ? 5.07 : 5.94);
  const int64_t room = workgroups_per_cu(num_blocks, groups, head_dim, warm_format, scores, nw, s);
  const int64_t on_cu = (units * s + CUS - 1) / CUS;
  const int64_t passes = (on_cu + room - 1) / room;
  const double refill = nw == 4 && room > 1 ? 1.48 : 1.3;   // a further pass's fixed part against the first's
  auto pass = [&](int64_t together) { return per_block * num_blocks / s * std::max(double(together), alone); };
  double t = fixed + (passes - 1) * (fixed * refill + pass(std::min(on_cu, room))) +
             pass(on_cu - (passes - 1) * room);
  if (s > 1) {
    // Publication and merge, by the unit's elements and MERGE_UNROLL splits
    // per round trip (in four splits instead of one, four waves, under 48
    // blocks, D = 128: 0.1 us more with four heads, 0.7 with eight, 4.3 with
    // sixteen); workgroups on one CU publish in turn (64 units of 256 blocks,
    // D = 64, G = 4: 14.5 us in two splits of eight waves, 12.0 in four, 14.7
    // in five, where two share a CU).
    const int rounds = (s + MERGE_UNROLL - 1) / MERGE_UNROLL;
    t += 0.95 * rounds + (0.57 + 0.89 * rounds) * (groups * head_dim / 512.0) + 1.59 * (std::min(on_cu, room) - 1);
  }
  // Score sums: the workgroup's own waves, a head or a part of one each (8
  // units of 64 blocks unsplit, G = 4: 10.9 -> 13.8 us with eight waves, 11.5
  // -> 15.4 with four), or a finalisation launch of a workgroup per (sequence,
  // head) row (the same in eight splits 8.8 -> 13.4 us; 1024 rows, 128 units
  // of 256 blocks at D = 64 in two splits: 29.7 us, 23.2 unsplit).
  if (scores && score_stage(scores, groups, num_blocks, s) == STAGE_LDS_BLOCK)
    t += 1.7 * (((groups <= 8 ? 8 / groups * groups : groups) + nw - 1) / nw);
  else if (scores)
    t += 4.22 + 5.05 * double(units * groups) / 512;
  // The list build of rows beyond one chunk (256 units, D = 128, four waves
  // against eight: 0.5 us less at 256 blocks, 0.6 more at 320), and beyond one
  // pass (32 units of 2048 blocks in eight splits: 30.7 us with eight waves,
  // one pass; 32.1 with four, two), where the blanks of the score sums are
  // written one by one.
  const int threads = 64 * nw;
  if (num_blocks > threads) t += 1.17;
  t += ((num_blocks - 1) / (PRE_CHUNKS * threads)) * (scores ? 5.28 : 1.5);
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
// the LDS accumulators.  Another plan has to promise 2 % over the plain rule's
// (its splits with the most waves): of 2,536 shapes those then measured more
// than 3 % slower than it fall from 54 to 43, the mean stays.
// The plan decides in which groups a deterministic launch adds its partial
// sums, so its output's bits are the plan's: such a launch takes the free plan
// in every workspace with room for it, and in every smaller one the plan of
// the smallest (not the best that fits, which would change with each size).
inline Plan plan_launch(int batch, int num_heads, int kv_heads, int num_blocks, int block_size, int head_dim,
                        int warm_format, bool scores, int splits_hint, bool deterministic, int64_t workspace_bytes) {
  const int groups = num_heads / kv_heads;
  const int64_t units = int64_t(batch) * kv_heads;
  auto bytes = [&](int s) {
    return ws_layout(batch, num_heads, kv_heads, num_blocks, block_size, head_dim, scores, s).total;
  };
  auto cheapest = [&](int64_t room) -> Plan {
    Plan best{groups <= 8 ? 8 : 4, required_splits(units, num_blocks, groups, splits_hint)};
    auto cost = [&](int nw, int s) {
      return plan_cost(units, num_blocks, groups, head_dim, warm_format, scores, nw, s);
    };
    double best_cost = cost(best.nw, best.splits) / 1.02;
    auto consider = [&](int s) {
      for (int nw = 8; nw >= 4; nw -= 4) {
        if (nw == 8 && groups > 8) continue;
        const double c = cost(nw, s);
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
