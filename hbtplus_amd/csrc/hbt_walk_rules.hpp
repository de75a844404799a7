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

}  // namespace hbt
