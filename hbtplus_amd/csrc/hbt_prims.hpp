// hbt_prims.hpp -- segmented device primitives for gfx950 (wave64).
//
// Every batch is a set of segments (one per subhalo).  Segment k owns the
// slot range [base[k], base[k] + cap[k]) of every per-particle work array;
// the number of live elements of the current operation is a per-segment
// device value (n[k]), so launches have static shapes (graph friendly) and
// work inside them is data dependent.  Segments are cut into TILE-element
// tiles (Tile table, built once per batch) for block-level work.
//
// Primitives:
//   segmented sort of (u64 key, u32 value) pairs by (key, value):
//     sort_tile, sort_tile_spare, sort_tile_words : a workgroup's run, as pairs or
//                           as words that carry their place
//     tile_sort_kernel    : each tile's pairs
//     merge_pass_kernel   : one bottom-up merge level (co-rank by binary search)
//     rank_merge_kernel   : a level of 16 runs, for launches of few tiles
//   segmented exclusive scan (load/store functors):
//     scan_tiles_kernel / scan_add_kernel
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hbt {

typedef unsigned long long u64;
typedef unsigned int u32;

constexpr int WAVE = 64;
constexpr int BLOCK = 256;
constexpr int TILE = 1024;           // elements per tile (4 per thread)
constexpr int ITEMS = TILE / BLOCK;

struct Tile {
  int seg;     // segment index
  int start;   // local offset of the tile inside the segment
};

__device__ __forceinline__ bool pair_less(u64 ka, u32 va, u64 kb, u32 vb) {
  return ka < kb || (ka == kb && va < vb);
}

// ---- wave / block scans ----------------------------------------------------

template <class T>
__device__ __forceinline__ T wave_inclusive_scan(T x) {
  const int lane = threadIdx.x & (WAVE - 1);
#pragma unroll
  for (int d = 1; d < WAVE; d <<= 1) {
    T y = __shfl_up(x, d, WAVE);
    if (lane >= d) x += y;
  }
  return x;
}

// A double moved across lanes by a DPP control (both halves).
template <int CTRL>
__device__ __forceinline__ double dpp_double(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double readlane_double(double x, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}

// Sum of x over the wave (every lane active), returned in every lane: DPP
// butterflies within each row of 16 lanes (quad permutes, half-row and row
// mirrors), then the four row sums read from lanes 0, 16, 32 and 48.  The
// order of the additions is fixed, so the result is deterministic.
__device__ __forceinline__ double wave_total(double x) {
#pragma clang fp contract(off)
  x += dpp_double<0xb1>(x);   // quad_perm [1,0,3,2]
  x += dpp_double<0x4e>(x);   // quad_perm [2,3,0,1]
  x += dpp_double<0x141>(x);  // row_half_mirror
  x += dpp_double<0x140>(x);  // row_mirror
  return (readlane_double(x, 0) + readlane_double(x, 16)) + (readlane_double(x, 32) + readlane_double(x, 48));
}

template <class T>
__device__ __forceinline__ T wave_reduce_sum(T x) {
#pragma unroll
  for (int d = WAVE / 2; d > 0; d >>= 1) x += __shfl_down(x, d, WAVE);
  return x;  // valid in lane 0
}

// Exclusive scan over the block (BLOCK threads, one value each); returns the
// exclusive prefix and writes the block total to *total.
template <class T>
__device__ __forceinline__ T block_exclusive_scan(T x, T *total) {
  __shared__ T wsum[BLOCK / WAVE];
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  T inc = wave_inclusive_scan(x);
  if (lane == WAVE - 1) wsum[w] = inc;
  __syncthreads();
  T off = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < BLOCK / WAVE; i++) {
    if (i < w) off += wsum[i];
    tot += wsum[i];
  }
  __syncthreads();
  *total = tot;
  return off + inc - x;
}

// ---- one-wave tiles ------------------------------------------------------------
// The tile table lists a level's segments largest first, so the tiles of the
// segments of at most SMALL_CAP slots -- one tile each, most segments of a
// level -- are a suffix of it.  Their kernels give each tile one wave instead
// of one workgroup: no workgroup barriers, four tiles per workgroup, and less
// LDS per tile in flight.
constexpr int SMALL_CAP = 4 * WAVE;  // one-wave tiles: 4 elements per lane ...
constexpr int TINY_CAP = WAVE;       // ... or 1 for the segments of at most one wave

// LDS writes of the wave visible to its other lanes.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Tiles t0 <= t < ntiles, one per wave (t is uniform across the wave).
#define WAVE_TILE_LOOP(t, t0, ntiles)                                                            \
  for (int t = (t0) + (int)(blockIdx.x * (BLOCK / WAVE) + threadIdx.x / WAVE); t < (ntiles); \
       t += (int)gridDim.x * (BLOCK / WAVE))

// ---- XCD-aware block order -----------------------------------------------------
// MI355X has 8 accelerator dies (XCDs), each with its own L2; the workgroups of
// a launch are dispatched to them round-robin (block b runs on XCD b % 8).
// xcd_block returns a virtual block index under which each XCD receives runs
// of `run` consecutive virtual blocks, so neighbouring slots (spatially close
// targets of one subhalo) share an L2.  Identity when run <= 1 or the grid is
// not a multiple of 8*run.
constexpr int NXCD = 8;

__device__ __forceinline__ int xcd_block(int run) {
  const int G = (int)gridDim.x, b = (int)blockIdx.x;
  if (run <= 1 || G % (NXCD * run) != 0) return b;
  const int x = b % NXCD, i = b / NXCD;
  return ((i / run) * NXCD + x) * run + (i % run);
}

// ---- segmented sort ----------------------------------------------------------

// Number of merge levels a segment of n elements needs after the sort of its
// runs of `run` elements, joining pairs of runs or, ranked, RANK_RUNS of them.
constexpr int RANK_RUNS = 16;
__device__ __forceinline__ int merge_levels(int n, int run, bool ranked = false) {
  int m = 0;
  for (int64_t w = run; w < n; w *= ranked ? RANK_RUNS : 2) m++;
  return m;
}

// ---- sorting networks of one wave ---------------------------------------------
// Lane l holds elements R l .. R l + R - 1 (padding sorts last), a bitonic
// network up to the power of two that covers them, partners less than R apart
// swapped in the lane and the others read across lanes.

// Lane x ^ M of the wave (within 32 lanes through the crossbar's bit mode,
// whose pattern is part of the instruction).
template <int M>
__device__ __forceinline__ u32 lane_xor(u32 v) {
  if constexpr (M < 32) return (u32)__builtin_amdgcn_ds_swizzle((int)v, 0x1f | (M << 10));
  else return (u32)__shfl_xor((int)v, M, WAVE);
}
template <int M>
__device__ __forceinline__ u64 lane_xor(u64 v) {
  return ((u64)lane_xor<M>((u32)(v >> 32)) << 32) | lane_xor<M>((u32)v);
}

__device__ __forceinline__ void sort_keep(bool keep_small, u64 ko, u32 vo, u64 &k, u32 &v) {
  const bool other_less = pair_less(ko, vo, k, v);
  if (keep_small ? other_less : !other_less) {
    k = ko;
    v = vo;
  }
}

// Elements a < b of one lane: the lower keeps the smaller in an ascending run.
__device__ __forceinline__ void sort_pair(bool up, u64 &ka, u32 &va, u64 &kb, u32 &vb) {
  if (pair_less(kb, vb, ka, va) == up) {
    const u64 tk = ka; ka = kb; kb = tk;
    const u32 tv = va; va = vb; vb = tv;
  }
}

// The network's stage (SIZE, J): partners J apart in runs of SIZE.
template <int R, int SIZE, int J>
__device__ __forceinline__ void sort_stage(u64 (&k)[R], u32 (&v)[R], int lane) {
  const int e0 = R * lane;
  if constexpr (J >= R) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int e = e0 + r;
      // the lower element of a pair keeps the smaller one in an ascending run
      sort_keep(((e & J) == 0) == ((e & SIZE) == 0), lane_xor<J / R>(k[r]), lane_xor<J / R>(v[r]), k[r], v[r]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < R; r++)
      if ((r & J) == 0) sort_pair(((e0 + r) & SIZE) == 0, k[r], v[r], k[r | J], v[r | J]);
  }
  if constexpr (J > 1) sort_stage<R, SIZE, J / 2>(k, v, lane);
}

// Sorts the wave's R * WAVE elements, of which the first `cnt` matter (the
// rest are padding): runs of SIZE, then of twice that, up to cnt.
template <int R, int SIZE = 2>
__device__ __forceinline__ void sort_wave(u64 (&k)[R], u32 (&v)[R], int lane, int cnt) {
  if (SIZE / 2 >= cnt) return;  // uniform across the wave
  sort_stage<R, SIZE, SIZE / 2>(k, v, lane);
  if constexpr (SIZE < R * WAVE) sort_wave<R, SIZE * 2>(k, v, lane, cnt);
}

// ---- the same for single words ---------------------------------------------------
// Where what orders the elements and each one's place fit one 64-bit word, the
// words alone are sorted: two registers to exchange instead of three and one
// comparison, which no tie follows.  All runs ascend, the first partners of a
// run being mirrored, so that neighbours in a lane need no direction; and lanes
// are exchanged in the vector unit: the crossbar behind ds_swizzle is shared by
// the four SIMDs.  Energies of 200,000 subhalos' passes as words 0.60 ms, keys
// included; as keys with values 0.94 and 0.57 for the keys.

// Lane x ^ M of the wave; M is a power of two or one less.
template <int M>
__device__ __forceinline__ u32 lane_flip(u32 v) {
  constexpr int ROW = M & 15;
  if constexpr (ROW == 1) v = (u32)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, false);        // quad_perm [1,0,3,2]
  else if constexpr (ROW == 2) v = (u32)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, false);   // quad_perm [2,3,0,1]
  else if constexpr (ROW == 3 || ROW == 4) v = (u32)__builtin_amdgcn_mov_dpp((int)v, 0x1b, 0xf, 0xf, false);  // [3,2,1,0]
  else if constexpr (ROW == 8) v = (u32)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, false);  // row_ror:8
  else if constexpr (ROW == 15) v = (u32)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xf, 0xf, false); // row_mirror
  if constexpr (ROW == 4 || ROW == 7) v = (u32)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xf, 0xf, false);  // half_mirror
  if constexpr ((M & 16) != 0) {  // rows 0, 1 and 2, 3 change places
    const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = (threadIdx.x & 16) ? p[0] : p[1];
  }
  if constexpr ((M & 32) != 0) {  // the halves change places
    const auto p = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = (threadIdx.x & 32) ? p[0] : p[1];
  }
  return v;
}
template <int M>
__device__ __forceinline__ u64 lane_flip(u64 v) {
  return ((u64)lane_flip<M>((u32)(v >> 32)) << 32) | lane_flip<M>((u32)v);
}

__device__ __forceinline__ void order_words(u64 &a, u64 &b) {
  const u64 x = a, y = b;
  const bool swap = y < x;
  a = swap ? y : x;
  b = swap ? x : y;
}

// Partners J apart, then J / 2 and so on.
template <int R, int J>
__device__ __forceinline__ void word_stages(u64 (&x)[R], int lane) {
  if constexpr (J >= R) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const u64 o = lane_flip<J / R>(x[r]);
      x[r] = (o < x[r]) == ((lane & (J / R)) == 0) ? o : x[r];
    }
  } else if constexpr (J > 0) {
#pragma unroll
    for (int r = 0; r < R; r++)
      if ((r & J) == 0) order_words(x[r], x[r | J]);
  }
  if constexpr (J > 1) word_stages<R, J / 2>(x, lane);
}

// Sorts the wave's R * WAVE words, of which the first cnt matter (the rest are ~0).
template <int R, int SIZE = 2>
__device__ __forceinline__ void sort_words(u64 (&x)[R], int lane, int cnt) {
  if (SIZE / 2 >= cnt) return;  // uniform across the wave
  if constexpr (SIZE <= R) {
#pragma unroll
    for (int r = 0; r < R; r++)
      if ((r & (SIZE / 2)) == 0) order_words(x[r], x[r ^ (SIZE - 1)]);
  } else {
    u64 o[R];
#pragma unroll
    for (int r = 0; r < R; r++) o[r] = lane_flip<SIZE / R - 1>(x[R - 1 - r]);
#pragma unroll
    for (int r = 0; r < R; r++) x[r] = (o[r] < x[r]) == ((lane & (SIZE / R / 2)) == 0) ? o[r] : x[r];
  }
  word_stages<R, SIZE / 4>(x, lane);
  if constexpr (SIZE < R * WAVE) sort_words<R, SIZE * 2>(x, lane, cnt);
}

// Outputs among the first d of the merge of A (la) and B (lb) that come from A.
// less(i, j): element i of A before element j of B.
template <class Less>
__device__ __forceinline__ int merge_split(Less less, int la, int lb, int d) {
  int lo = d > lb ? d - lb : 0, hi = d < la ? d : la;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (less(mid, d - 1 - mid)) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// The same by a whole wave, 64 places at a time: three rounds of loads where
// halving takes seventeen.
template <class Less>
__device__ __forceinline__ int merge_split_wave(Less less, int la, int lb, int d) {
  int lo = d > lb ? d - lb : 0, hi = d < la ? d : la;
  while (lo < hi) {
    const int step = (hi - lo + WAVE - 1) / WAVE;
    const int at = lo + step * ((int)(threadIdx.x & (WAVE - 1)) + 1) - 1;
    const int c = __popcll(__ballot(at < hi && less(at, d - 1 - at)));
    hi = min(hi, lo + step * (c + 1) - 1);
    lo += step * c;
  }
  return lo;
}

// Element i of the pairs (ka, va) before element j of (kb, vb); the values are
// read for equal keys only.
struct PairsLess {
  const u64 *ka;
  const u32 *va;
  const u64 *kb;
  const u32 *vb;
  __device__ __forceinline__ bool operator()(int i, int j) const {
    const u64 x = ka[i], y = kb[j];
    return x != y ? x < y : va[i] < vb[j];
  }
};

// Sorts the cnt <= 4 T elements of a workgroup of T threads, four per thread
// (element 4 i + r in thread i, padding ~0 / ~0 past cnt), into sk / sv: each wave
// sorts its 256 in registers, then merges in LDS join 2, 4, ... of those runs,
// each thread finding its split of its pair of runs and its four outputs.  One LDS network
// over the whole tile is a chain of 55 barriers: 25 us for a tile alone, 10 so.
template <int T>
__device__ __forceinline__ void sort_tile(u64 (&k)[ITEMS], u32 (&v)[ITEMS], int cnt, u64 *sk, u32 *sv) {
  constexpr int RUN = ITEMS * WAVE;
  const int i0 = ITEMS * (int)threadIdx.x;
  const int w0 = i0 & ~(RUN - 1);
  if (w0 < cnt) sort_wave<ITEMS>(k, v, threadIdx.x & (WAVE - 1), min(RUN, cnt - w0));
#pragma unroll
  for (int r = 0; r < ITEMS; r++) { sk[i0 + r] = k[r]; sv[i0 + r] = v[r]; }
  __syncthreads();
  for (int width = RUN; width < cnt; width *= 2) {  // uniform across the block
    const int a0 = i0 & ~(2 * width - 1), d = i0 - a0;
    const u64 *ka = sk + a0, *kb = ka + width;
    const u32 *va = sv + a0, *vb = va + width;
    const int lb = min(width, max(0, cnt - a0 - width));  // past cnt there is padding only
    const bool merge = lb > 0;
    if (merge) {
      int i = merge_split(PairsLess{ka, va, kb, vb}, width, width, d);
      int j = d - i;
      u64 x = i < width ? ka[i] : ~0ull, y = j < width ? kb[j] : ~0ull;
      u32 xv = i < width ? va[i] : ~0u, yv = j < width ? vb[j] : ~0u;
#pragma unroll
      for (int r = 0; r < ITEMS; r++) {
        const bool take_a = j >= width || (i < width && !pair_less(y, yv, x, xv));
        k[r] = take_a ? x : y;
        v[r] = take_a ? xv : yv;
        if (take_a) {
          i++;
          x = i < width ? ka[i] : ~0ull;
          xv = i < width ? va[i] : ~0u;
        } else {
          j++;
          y = j < width ? kb[j] : ~0ull;
          yv = j < width ? vb[j] : ~0u;
        }
      }
    }
    __syncthreads();
    if (merge) {
#pragma unroll
      for (int r = 0; r < ITEMS; r++) { sk[i0 + r] = k[r]; sv[i0 + r] = v[r]; }
    }
    __syncthreads();
  }
}

// The same for words, into sk.
template <int T>
__device__ __forceinline__ void sort_tile_words(u64 (&x)[ITEMS], int cnt, u64 *sk) {
  constexpr int RUN = ITEMS * WAVE;
  const int i0 = ITEMS * (int)threadIdx.x;
  const int w0 = i0 & ~(RUN - 1);
  if (w0 < cnt) sort_words<ITEMS>(x, threadIdx.x & (WAVE - 1), min(RUN, cnt - w0));
#pragma unroll
  for (int r = 0; r < ITEMS; r++) sk[i0 + r] = x[r];
  __syncthreads();
  for (int width = RUN; width < cnt; width *= 2) {  // uniform across the block
    const int a0 = i0 & ~(2 * width - 1), d = i0 - a0;
    const u64 *ka = sk + a0, *kb = ka + width;
    const bool merge = min(width, cnt - a0 - width) > 0;  // past cnt there is padding only
    if (merge) {
      int i = merge_split([&](int p, int q) { return ka[p] < kb[q]; }, width, width, d);
      int j = d - i;
      u64 a = i < width ? ka[i] : ~0ull, b = j < width ? kb[j] : ~0ull;
#pragma unroll
      for (int r = 0; r < ITEMS; r++) {
        const bool take_a = j >= width || (i < width && a <= b);
        x[r] = take_a ? a : b;
        if (take_a) a = ++i < width ? ka[i] : ~0ull;
        else b = ++j < width ? kb[j] : ~0ull;
      }
    }
    __syncthreads();
    if (merge) {
#pragma unroll
      for (int r = 0; r < ITEMS; r++) sk[i0 + r] = x[r];
    }
    __syncthreads();
  }
}

constexpr int log2_of(int n) { return n <= 1 ? 0 : 1 + log2_of(n / 2); }

// Orders by value the elements of equal keys that start at e, in place; false
// if there are more than SHORT of them.
__device__ __forceinline__ bool order_equal(const u64 *sk, u32 *sv, int e, int cnt) {
  constexpr int SHORT = 8;
  const u64 k = sk[e];
  if (e + 1 >= cnt || sk[e + 1] != k || (e > 0 && sk[e - 1] == k)) return true;
  int n = 2;
  while (e + n < cnt && sk[e + n] == k)
    if (++n > SHORT) return false;
  for (int i = 1; i < n; i++) {
    const u32 v = sv[e + i];
    int at = i;
    for (; at > 0 && sv[e + at - 1] > v; at--) sv[e + at] = sv[e + at - 1];
    sv[e + at] = v;
  }
  return true;
}

// Keys k whose low `spare` bits are zero, with values v, as sort_tile: as words
// that carry the element's place in those bits where they are enough, the few
// equal keys (sources in one cell of the smallest size) then ordered by their
// values; with long runs of equal keys as pairs after all.
template <int T>
__device__ __forceinline__ void sort_tile_spare(u64 (&k)[ITEMS], u32 (&v)[ITEMS], int cnt, int spare, u64 *sk,
                                                u32 *sv) {
  constexpr int BITS = log2_of(ITEMS * T);
  constexpr u64 PLACE = (1ull << BITS) - 1;
  if (spare >= BITS) {  // uniform across the block
    u64 x[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int e = ITEMS * (int)threadIdx.x + r;
      x[r] = e < cnt ? k[r] | (u64)e : ~0ull;
      sv[e] = v[r];
    }
    sort_tile_words<T>(x, cnt, sk);
    u32 w[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int e = (int)threadIdx.x + T * r;
      x[r] = sk[e];
      w[r] = e < cnt ? sv[x[r] & PLACE] : ~0u;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int e = (int)threadIdx.x + T * r;
      sk[e] = e < cnt ? x[r] & ~PLACE : ~0ull;
      sv[e] = w[r];
    }
    __syncthreads();
    bool ordered = true;
#pragma unroll 1
    for (int e = threadIdx.x; e < cnt; e += T) ordered &= order_equal(sk, sv, e, cnt);
    if (!__syncthreads_or(!ordered)) return;
#pragma unroll
    for (int r = 0; r < ITEMS; r++) { k[r] = sk[ITEMS * threadIdx.x + r]; v[r] = sv[ITEMS * threadIdx.x + r]; }
    __syncthreads();
  }
  sort_tile<T>(k, v, cnt, sk, sv);
}

// The same for a wave, R elements per lane, through sk / sv of its own.
template <int R>
__device__ __forceinline__ void sort_wave_spare(u64 (&k)[R], u32 (&v)[R], int lane, int cnt, int spare, u64 *sk,
                                                u32 *sv) {
  constexpr int BITS = log2_of(R * WAVE);
  constexpr u64 PLACE = (1ull << BITS) - 1;
  if (spare >= BITS) {  // uniform across the wave
    u64 x[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int e = R * lane + r;
      x[r] = e < cnt ? k[r] | (u64)e : ~0ull;
      sv[e] = v[r];
    }
    sort_words<R>(x, lane, cnt);
    wave_sync();
#pragma unroll
    for (int r = 0; r < R; r++) {
      const bool live = R * lane + r < cnt;
      k[r] = live ? x[r] & ~PLACE : ~0ull;
      v[r] = live ? sv[x[r] & PLACE] : ~0u;
    }
    wave_sync();
#pragma unroll
    for (int r = 0; r < R; r++) { sk[R * lane + r] = k[r]; sv[R * lane + r] = v[r]; }
    wave_sync();
    bool ordered = true;
#pragma unroll 1
    for (int e = lane; e < cnt; e += WAVE) ordered &= order_equal(sk, sv, e, cnt);
    wave_sync();
    if (__ballot(!ordered) == 0) return;
#pragma unroll
    for (int r = 0; r < R; r++) v[r] = sv[R * lane + r];
  }
  sort_wave<R>(k, v, lane, cnt);
#pragma unroll
  for (int r = 0; r < R; r++) { sk[R * lane + r] = k[r]; sv[R * lane + r] = v[r]; }
}

// Sorts each tile's live elements [start, min(start+TILE, n[seg])) from
// (k0, v0) into the buffer from which the segment's merge levels end in
// (k0, v0): (k1, v1) when it needs an odd number of levels, else in place.
__global__ void __launch_bounds__(BLOCK)
tile_sort_kernel(const Tile *__restrict__ tiles, int ntiles, const int64_t *__restrict__ base,
                 const int *__restrict__ n, u64 *k0, u32 *v0, u64 *k1, u32 *v1) {
  __shared__ u64 sk[TILE];
  __shared__ u32 sv[TILE];
  __shared__ int slive[BLOCK];
  // The block's tiles (blockIdx.x + k gridDim.x) are checked BLOCK at a time,
  // one per thread, and only the non-empty ones are sorted: a sort of a few
  // entries per segment (the energy sort of a removed block) skips its empty
  // tiles without a chain of header loads.
  for (int tb = blockIdx.x; tb < ntiles; tb += gridDim.x * BLOCK) {
    const int tc = tb + (int)threadIdx.x * (int)gridDim.x;
    int live = 0;
    if (tc < ntiles) live = n[tiles[tc].seg] - tiles[tc].start > 0 ? 1 : 0;
    int nlive;
    const int at = block_exclusive_scan(live, &nlive);
    if (live) slive[at] = tc;
    __syncthreads();
    for (int li = 0; li < nlive; li++) {
      const int t = slive[li];
      const Tile tl = tiles[t];
      const int nseg = n[tl.seg];
      const int cnt = min(TILE, nseg - tl.start);
      const int64_t off = base[tl.seg] + tl.start;
      u64 *kout = (merge_levels(nseg, TILE) & 1) ? k1 : k0;
      u32 *vout = (merge_levels(nseg, TILE) & 1) ? v1 : v0;
      if (cnt == 1) {
        if (threadIdx.x == 0) { kout[off] = k0[off]; vout[off] = v0[off]; }
        continue;
      }
      u64 k[ITEMS];
      u32 v[ITEMS];
#pragma unroll
      for (int r = 0; r < ITEMS; r++) {
        const int e = ITEMS * (int)threadIdx.x + r;
        k[r] = e < cnt ? k0[off + e] : ~0ull;
        v[r] = e < cnt ? v0[off + e] : ~0u;
      }
      sort_tile<BLOCK>(k, v, cnt, sk, sv);
      for (int i = threadIdx.x; i < cnt; i += BLOCK) { kout[off + i] = sk[i]; vout[off + i] = sv[i]; }
      __syncthreads();
    }
    __syncthreads();  // slive is rewritten for the next batch of tiles
  }
}

// Merge level `level` (runs of width run << level merged pairwise).  A
// segment that needs m levels takes part in levels 0..m-1 and ping-pongs
// between the two buffers so that level m-1 writes (k0, v0); segments with
// m <= level are done and are not touched.  Merge path: one block per tile of
// output; two waves search how many of the tile's outputs come from the left run
// at its two ends, the block stages those parts of the two runs in LDS, and each
// thread finds its own split in LDS and merges MERGE_PER outputs.  Keys with
// their values are distinct, so the merged order is unique.  Two threads halving
// their ranges kept the block waiting on seventeen dependent loads: a level over
// one list of 24,000 took 7.2 us, 5.4 now, the levels of 200,000 subhalos' passes
// 4.8 ms, 3.6 now (24 bytes an element and level are 2.2 at 4.7 TB/s).
constexpr int MERGE_PER = TILE / BLOCK;

__global__ void __launch_bounds__(BLOCK)
merge_pass_kernel(const Tile *__restrict__ tiles, int ntiles, const int64_t *__restrict__ base,
                  const int *__restrict__ n, int run, int level, u64 *k0, u32 *v0, u64 *k1, u32 *v1) {
  __shared__ u64 sk[TILE];
  __shared__ u32 sv[TILE];
  __shared__ int ssplit[2];
  const int width = run << level;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const int cnt = n[tl.seg];
    if (cnt <= width || tl.start >= cnt) continue;  // uniform across the block
    const int m = merge_levels(cnt, run);
    // buffer holding the input of this level: the tile sort wrote parity m&1
    const bool in1 = ((m + level) & 1) != 0;
    const u64 *kin = in1 ? k1 : k0;
    const u32 *vin = in1 ? v1 : v0;
    u64 *kout = in1 ? k0 : k1;
    u32 *vout = in1 ? v0 : v1;
    const int64_t bs = base[tl.seg];
    const int a0 = tl.start / (2 * width) * (2 * width);  // start of the merged pair
    const int la = min(width, cnt - a0);
    const int lb = max(0, min(width, cnt - a0 - width));
    const u64 *ka = kin + bs + a0, *kb = ka + width;
    const u32 *va = vin + bs + a0, *vb = va + width;
    const int o0 = tl.start - a0, o1 = min(tl.start + TILE, cnt) - a0;  // outputs of this tile
    const int w = threadIdx.x / WAVE;
    if (w < 2) {
      const int at = merge_split_wave(PairsLess{ka, va, kb, vb}, la, lb, w == 0 ? o0 : o1);
      if ((threadIdx.x & (WAVE - 1)) == 0) ssplit[w] = at;
    }
    __syncthreads();
    const int i0 = ssplit[0], i1 = ssplit[1];
    const int j0 = o0 - i0, j1 = o1 - i1;
    const int na = i1 - i0, nb = j1 - j0;  // na + nb = o1 - o0 <= TILE
    for (int i = threadIdx.x; i < na; i += BLOCK) { sk[i] = ka[i0 + i]; sv[i] = va[i0 + i]; }
    for (int i = threadIdx.x; i < nb; i += BLOCK) { sk[na + i] = kb[j0 + i]; sv[na + i] = vb[j0 + i]; }
    __syncthreads();
    const int d = (int)threadIdx.x * MERGE_PER;
    if (d < na + nb) {
      const PairsLess less{sk, sv, sk + na, sv + na};
      int i = merge_split(less, na, nb, d), j = d - i;
      u64 k[MERGE_PER];
      u32 v[MERGE_PER];
      const int e = min(MERGE_PER, na + nb - d);
#pragma unroll
      for (int o = 0; o < MERGE_PER; o++) {
        if (o >= e) break;
        const int at = j >= nb || (i < na && less(i, j)) ? i++ : na + j++;
        k[o] = sk[at];
        v[o] = sv[at];
      }
      u64 *ko = kout + bs + a0 + o0 + d;
      u32 *vo = vout + bs + a0 + o0 + d;
      if (e == MERGE_PER && (((uintptr_t)ko | (uintptr_t)vo) & 15) == 0) {  // bases are multiples of four mostly
        static_assert(MERGE_PER == 4, "outputs are stored four at a time");
        reinterpret_cast<ulonglong2 *>(ko)[0] = make_ulonglong2(k[0], k[1]);
        reinterpret_cast<ulonglong2 *>(ko)[1] = make_ulonglong2(k[2], k[3]);
        *reinterpret_cast<uint4 *>(vo) = make_uint4(v[0], v[1], v[2], v[3]);
      } else {
        for (int o = 0; o < e; o++) { ko[o] = k[o]; vo[o] = v[o]; }
      }
    }
    __syncthreads();
  }
}

// The merge level `level` of RANK_RUNS runs (run * RANK_RUNS^level long) each, with
// the buffers of merge_pass_kernel's levels: an element's place is its place in
// its own run and the number of elements before it in each of the others, which a
// wave per run counts for 64 elements by halving.  For launches of few tiles,
// which wait on each level's chain of loads: the four levels of pairs of one list
// of 24,000 took 22 us and three gaps between launches, this takes 5.6.  It
// searches the runs anew for every element, so larger launches merge.
__global__ void __launch_bounds__(RANK_RUNS *WAVE)
rank_merge_kernel(const Tile *__restrict__ tiles, const int64_t *__restrict__ base, const int *__restrict__ n, int run,
                  int level, u64 *k0, u32 *v0, u64 *k1, u32 *v1) {
  __shared__ int place[WAVE];
  constexpr int CHUNKS = TILE / WAVE;  // workgroups per tile
  const Tile tl = tiles[blockIdx.x / CHUNKS];
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const int cnt = n[tl.seg], e0 = tl.start + (int)(blockIdx.x % CHUNKS) * WAVE, e = e0 + lane;
  int width = run;
  for (int i = 0; i < level; i++) width *= RANK_RUNS;
  if (cnt <= width || e0 >= cnt) return;  // uniform across the block
  const bool in1 = ((merge_levels(cnt, run, true) + level) & 1) != 0;
  const int64_t b = base[tl.seg];
  const int g0 = e0 / (width * RANK_RUNS) * (width * RANK_RUNS);  // first element of the joined runs
  const int own = (e0 - g0) / width;
  const u64 *k = (in1 ? k1 : k0) + b;
  const u32 *v = (in1 ? v1 : v0) + b;
  const u64 key = e < cnt ? k[e] : ~0ull;
  const u32 val = e < cnt ? v[e] : ~0u;
  if (w == 0) place[lane] = e - own * width;
  __syncthreads();
  const int r0 = g0 + w * width;
  if (w != own && r0 < cnt) {
    int lo = 0, hi = min(width, cnt - r0);  // first element of the run that is not before this one
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      const u64 x = k[r0 + mid];
      if (x < key || (x == key && v[r0 + mid] < val)) lo = mid + 1; else hi = mid;
    }
    if (lo) atomicAdd(&place[lane], lo);
  }
  __syncthreads();
  if (w == 0 && e < cnt) {
    (in1 ? k0 : k1)[b + place[lane]] = key;
    (in1 ? v0 : v1)[b + place[lane]] = val;
  }
}

// ---- segmented exclusive scan ----------------------------------------------
// Load(seg, local) -> T for local < n[seg]; Store(seg, local, exclusive prefix).
// Pass 1 scans each tile and stores tile-local prefixes and the tile total;
// pass 2 adds to every tile the totals of the tiles before it in its segment.

template <class T, class Load, class Store>
__global__ void __launch_bounds__(BLOCK)
scan_tiles_kernel(const Tile *__restrict__ tiles, int ntiles, const int *__restrict__ n,
                  T *__restrict__ tile_sum, Load load, Store store) {
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const int cnt = min(TILE, n[tl.seg] - tl.start);
    if (cnt <= 0) {
      if (threadIdx.x == 0) tile_sum[t] = T(0);
      continue;
    }
    T v[ITEMS];
    T s = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
      const int l = threadIdx.x * ITEMS + i;
      v[i] = l < cnt ? load(tl.seg, tl.start + l) : T(0);
      s += v[i];
    }
    T total;
    T off = block_exclusive_scan(s, &total);
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
      const int l = threadIdx.x * ITEMS + i;
      if (l < cnt) store(tl.seg, tl.start + l, off);
      off += v[i];
    }
    if (threadIdx.x == 0) tile_sum[t] = total;
  }
}

// Pass 2: adds to each tile the sum of the earlier tiles of its segment (the
// tiles of a segment are consecutive in the table; tile t is the
// start/TILE-th of its segment).
template <class T, class Update>
__global__ void __launch_bounds__(BLOCK)
scan_add_kernel(const Tile *__restrict__ tiles, int ntiles, const int *__restrict__ n,
                const T *__restrict__ tile_sum, Update update) {
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    if (tl.start == 0) continue;  // first tile of a segment has offset 0
    const int cnt = min(TILE, n[tl.seg] - tl.start);
    if (cnt <= 0) continue;
    const int t0 = t - tl.start / TILE;
    T part = 0;
    for (int u = t0 + (int)threadIdx.x; u < t; u += BLOCK) part += tile_sum[u];
    T o;
    (void)block_exclusive_scan(part, &o);
    for (int l = threadIdx.x; l < cnt; l += BLOCK) update(tl.seg, tl.start + l, o);
  }
}

}  // namespace hbt
