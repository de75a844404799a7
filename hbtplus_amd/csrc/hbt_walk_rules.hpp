// hbt_walk_rules.hpp -- which form of the tree walk a call takes, by its sizes.
// Host code only, without HIP, so that the rules are checked by themselves.
#pragma once
#include <stdint.h>

#include "../../include/hbt_unbind.h"

namespace hbt {

// Trees whose items the walks of 8, 16 and 32 lanes can reach: their positions
// are 32-bit byte offsets of 32-byte items from the segment's first.  n sources
// have at most 2 n - 1 items, the sentinel follows and the item after it is
// fetched.  Larger trees take walks that stand at item indices: 64 lanes
// together, or each lane by itself.
constexpr int64_t BYTE_WALK_SOURCES = (int64_t)1 << 26;
constexpr bool byte_walk(int64_t n_src) { return n_src < BYTE_WALK_SOURCES; }

// Lanes per walk group of a list of up to len particles.
inline int walk_group_for(const hbt_tuning &t, int64_t len) {
  if (!byte_walk(len)) return 64;
  return len < t.bin_edge[0] ? t.walk_group[0] : (len < t.bin_edge[1] ? t.walk_group[1] : t.walk_group[2]);
}

// Lanes per walk group of a launch whose longest list has up to len particles; 0:
// each segment's own.
inline int launch_group(const hbt_tuning &t, int64_t len) {
  const int32_t *g = t.walk_group;
  return byte_walk(len) && g[0] == g[1] && g[1] == g[2] ? g[0] : 0;
}

// Waves that share a chunk's walk (1, 2, 4, 8 or 16): about eight waves per
// SIMD.  From six without sharing on a second wave no longer pays: a list of
// 420,000 (6,563 chunks) walks 1.71 ms alone and 1.78 shared by two, 50 lists of
// together 5,900 chunks 0.81 and 0.62, one list of 24,000 (375) 0.53 and, by 16,
// 0.147.
inline int walk_parts(int64_t chunks, int cus) {
  const int64_t simds = 4 * (int64_t)cus;
  if (chunks >= 6 * simds) return 1;
  int parts = 2;
  while (parts < 16 && chunks * parts < 8 * simds) parts *= 2;
  return parts;
}

// How hbt_tree_potential walks its targets: each lane by itself, over the targets
// as they came or in tree order, or lanes together (16 of them, or 64 beyond
// byte_walk; FAST shares a chunk among several waves).  The bits are the same (in
// FAST while its FP64 sums of FP32 terms are exact).
// Lanes that walk together wait for the union of their paths, which is long where
// few targets lie far apart in a large tree, and ordering the targets costs five
// launches and the digits' sort.  ms a call, periodic box, alone / ordered /
// together:
//   REPLAY sums in the reference's order, so no chunk is shared: alone, in order
//   from where two waves a SIMD hide each other's loads (20,000 to 1 million sources
//   at 262,144 targets 1.20-4.57 / 1.10-3.52 / 1.42-3.63; 100,000 at 32,768 1.16 /
//   1.19 / 1.60; 300 at any number fastest unordered).
//   FP32 adds in one order too; together where targets are dense (10,000 sources,
//   4,096 targets 0.69 / 0.69 / 0.57; 100,000 and 32,768 1.02 / 1.00 / 0.85), alone
//   below a target in 16 sources (30,000 and 512 0.90 / 0.88 / 1.11; 1 million and
//   64 1.64 / 1.45 / 4.77), up to two targets being paths of their own (0.70 together
//   for one among a million, 1.08 alone).
//   FAST, its chunks shared, only below one in 1,500 of a large tree (1 million
//   and 64 1.64 / 1.45 / 3.14; 300,000 and 64 1.36 / 1.19 / 2.05, and 512 1.37 / 1.45
//   / 1.30).
//   Trees of a wave's sources are walked in less time than the ordering's launches
//   take (16 sources, 4,096 targets 0.043 / 0.095 / 0.095).
enum class TargetWalk { alone, alone_ordered, together };
inline TargetWalk target_walk(int64_t n_src, int64_t n_tgt, int precision) {
  if (precision == HBT_PREC_REPLAY)
    return n_tgt >= 131072 && n_src >= 1000 ? TargetWalk::alone_ordered : TargetWalk::alone;
  if (n_src <= 64) return TargetWalk::alone;
  const bool sparse = precision == HBT_PREC_FP32 ? n_tgt > 2 && n_src > 16 * n_tgt
                                                 : n_tgt > 8 && n_src > 1500 * n_tgt && n_src >= 131072;
  return sparse ? TargetWalk::alone : TargetWalk::together;
}

// The most sources per target for ordered targets to walk together (chunk_alone).
// FP32: with 3.8 (a million sources, 262,144 targets) 1.8 ms together and 4.1
// alone, with 6 (100,000 and 16,384 among as many others) 1.39 and 1.14.  FAST: 12
// and 24 are alike, with 48 targets spread over the box of a million sources
// take 2.5 ms for 2.3, with 96 2.9.
inline int target_reach(int precision) { return precision == HBT_PREC_FAST ? 24 : 5; }

}  // namespace hbt
