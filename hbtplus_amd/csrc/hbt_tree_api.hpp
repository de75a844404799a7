// hbt_tree_api.hpp -- hbt_tree_potential: GravityTree_t::Build over a source
// set in the given order followed by EvaluatePotential at arbitrary targets
// (src/oct_tree.tpp:17-144, src/gravity_tree.cpp:79-164), on the same tree
// kernels as the unbinding passes.  Included by hbt_unbind.hip.
#pragma once

namespace {

__global__ void tree_only_setup_kernel(Work W, int n) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    Seg &S = W.seg[0];
    W.ncount[NC_SRC * W.nseg] = n;
    S.flags = F_ACTIVE;
    S.n_src = n; S.src_lo = 0; S.n_tgt = 0; S.nsort = n; S.nlast = n; S.nbound = n;
    for (int j = 0; j < 3; j++) { S.bmin[j] = 0xffffffffu; S.bmax[j] = 0u; }
  }
}

__global__ void tree_sources_kernel(Work W, int n, const float *x, const float *y, const float *z,
                                    const float *m) {
  for (int i = blockIdx.x * BLOCK + threadIdx.x; i < n; i += gridDim.x * BLOCK) {
    W.pos[i] = make_float4(x[i], y[i], z[i], m[i]);
    W.el[i] = i;
  }
}

// The targets in an order that follows the tree, so that neighbouring lanes
// walk together: a target's bucket is the place of its octant digits among the
// sources' sorted digits, BUCKET sources to a bucket, and a counting sort puts
// the buckets in order (the order inside one is arbitrary; no result depends
// on it).  Walked lane by lane in the caller's order, 120,000 targets spent
// 1.44 of their call's 1.68 ms in the walk; in tree order, 16 lanes together
// and without the wrap's FP64 separations where nothing wraps, 0.60 of 0.91
// (and 0.32 of 0.65 where several waves share a chunk).
constexpr int BUCKET_BITS = 4;
constexpr int64_t TGT_SLICE = 1 << 24;  // targets per round (their scratch is 12 bytes each)

struct TgtArgs {
  const float *x, *y, *z, *m;
  double *out;
  int n;
  int *bucket, *rank, *order;  // [n]
  int *count;                  // [buckets] targets per bucket
  u64 *first;                  // [buckets] exclusive prefix of count
  u32 *box;                    // [6] targets' bounding box, ordered-integer encoding
  int *apart;                  // chunks whose lanes walk alone
};

struct TgtLoad {
  const int *count;
  __device__ u64 operator()(int, int l) const { return (u64)count[l]; }
};
struct TgtStore {
  u64 *first;
  __device__ void operator()(int, int l, u64 x) const { first[l] = x; }
};
struct TgtAdd {
  u64 *first;
  __device__ void operator()(int, int l, u64 x) const { first[l] += x; }
};

__global__ void __launch_bounds__(BLOCK) tgt_clear_kernel(Work W, TgtArgs A, int nb) {
  const int i = blockIdx.x * BLOCK + threadIdx.x;
  if (i < 6) A.box[i] = i < 3 ? 0xffffffffu : 0u;
  if (i == 0) {
    W.ncount[NC_SORT * W.nseg] = nb;  // the scan's element count
    *A.apart = 0;
  }
  for (int j = i; j < nb; j += gridDim.x * BLOCK) A.count[j] = 0;
}

// The target's bucket: the place of the first source whose digits are not below
// its own; the last one outside the sources' cube, whose outermost sources' digits
// would bring targets from everywhere together.
__device__ __forceinline__ int tgt_bucket(const Work &W, const Seg &S, int outside, float x, float y, float z) {
  const double half = 0.5 * S.Len;
  if (fabs(x - S.center[0]) > half || fabs(y - S.center[1]) > half || fabs(z - S.center[2]) > half) return outside;
  const u64 key = octant_key(S.center, S.Len, S.D, x, y, z);
  int lo = 0, hi = S.n_src;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (W.k0[mid] < key) lo = mid + 1; else hi = mid;
  }
  return lo >> BUCKET_BITS;
}

// Folds a position into a thread's box (ordered-integer encoding).
__device__ __forceinline__ void box_take(u32 mn[3], u32 mx[3], float x, float y, float z) {
  const u32 o[3] = {f2ord(x), f2ord(y), f2ord(z)};
  for (int j = 0; j < 3; j++) { mn[j] = min(mn[j], o[j]); mx[j] = max(mx[j], o[j]); }
}

// Bucket of each target, its place among the bucket's targets, the box of all.
// Atomics on one address are served one after another, 28 ns each, and few buckets
// hold many targets each: up to LDS_BUCKETS a block counts its run of the targets
// in LDS and takes a range of each bucket with one atomic (2 million targets among
// 100 sources 8.8 -> 0.33 ms a call, among 1,000 4.3 -> 0.91).  With more buckets a
// wave takes its places in memory, one atomic for each bucket its targets are in
// (2 million close to a few of a million sources: target by target 12.4 ms a call,
// so 3.5).
constexpr int LDS_BUCKETS = 4096;

__global__ void __launch_bounds__(BLOCK) tgt_bucket_lds_kernel(Work W, TgtArgs A, int nb, int per_block) {
  __shared__ int cnt[LDS_BUCKETS];
  const Seg &S = W.seg[0];
  u32 mn[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, mx[3] = {0u, 0u, 0u};
  const int i0 = blockIdx.x * per_block, i1 = min(A.n, i0 + per_block);
  for (int j = threadIdx.x; j < nb; j += BLOCK) cnt[j] = 0;
  __syncthreads();
  for (int i = i0 + (int)threadIdx.x; i < i1; i += BLOCK) {
    const float x = A.x[i], y = A.y[i], z = A.z[i];
    box_take(mn, mx, x, y, z);
    const int b = tgt_bucket(W, S, nb - 1, x, y, z);
    A.bucket[i] = b;
    A.rank[i] = atomicAdd(&cnt[b], 1);
  }
  __syncthreads();
  for (int j = threadIdx.x; j < nb; j += BLOCK)
    if (cnt[j]) cnt[j] = atomicAdd(&A.count[j], cnt[j]);
  __syncthreads();
  for (int i = i0 + (int)threadIdx.x; i < i1; i += BLOCK) A.rank[i] += cnt[A.bucket[i]];
  fold_box(mn, mx, A.box, A.box + 3);
}

__global__ void __launch_bounds__(BLOCK) tgt_bucket_kernel(Work W, TgtArgs A, int nb) {
  const Seg &S = W.seg[0];
  u32 mn[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, mx[3] = {0u, 0u, 0u};
  for (int i0 = blockIdx.x * BLOCK; i0 < A.n; i0 += gridDim.x * BLOCK) {  // uniform across the block
    const int i = i0 + (int)threadIdx.x;
    int b = -1;
    if (i < A.n) {
      const float x = A.x[i], y = A.y[i], z = A.z[i];
      box_take(mn, mx, x, y, z);
      b = tgt_bucket(W, S, nb - 1, x, y, z);
      A.bucket[i] = b;
    }
    // the lanes of each bucket among the wave's: their first, how many, how many before;
    // four buckets with one lane each, and the rest are taken to be so too
    const int lane = threadIdx.x & (WAVE - 1);
    int head = lane, size = b >= 0 ? 1 : 0, before = 0, lone = 0;
    for (u64 todo = __ballot(b >= 0); todo != 0ull && lone < 4;) {  // uniform across the wave
      const int first = __ffsll((long long)todo) - 1;
      const u64 same = __ballot(b == __builtin_amdgcn_readlane(b, first));
      if ((same >> lane) & 1ull) {
        head = first;
        size = __popcll(same);
        before = __popcll(same & ((1ull << lane) - 1ull));
      }
      lone += __popcll(same) == 1 ? 1 : 0;
      todo &= ~same;
    }
    int r = 0;
    if (size > 0 && lane == head) r = atomicAdd(&A.count[b], size);
    r = __shfl(r, head, WAVE) + before;
    if (b >= 0) A.rank[i] = r;
  }
  fold_box(mn, mx, A.box, A.box + 3);
}

__global__ void __launch_bounds__(BLOCK) tgt_order_kernel(TgtArgs A) {
  for (int i = blockIdx.x * BLOCK + threadIdx.x; i < A.n; i += gridDim.x * BLOCK)
    A.order[A.first[A.bucket[i]] + A.rank[i]] = i;
}

// The FP32 walk wraps separations only where some target and source can be
// more than half a box apart (sources' and targets' boxes; a node's centre may
// lie a rounding outside its sources').
__device__ __forceinline__ bool targets_wrap(const Seg &S, const DevParams &P, const TgtArgs &A) {
  bool wrap = false;
  if (P.periodic)
    for (int j = 0; j < 3; j++) {
      const double s0 = ord2f(S.bmin[j]), s1 = ord2f(S.bmax[j]), t0 = ord2f(A.box[j]), t1 = ord2f(A.box[3 + j]);
      const double far = t1 - s0 > s1 - t0 ? t1 - s0 : s1 - t0;
      if (!(far <= (double)P.box_half * (1.0 - 1e-6)) || !(t0 <= t1)) wrap = true;  // also where one is not a number
    }
  return wrap;
}

// Whether the lanes of a chunk of 64 ordered targets walk alone, as target_walk
// decides for a call's sizes: most of its targets lie outside the sources' cube, or
// the buckets between neighbours add up to more than `reach` (a step counts for a
// quarter of it at most: one from an octant to the next passes over any number),
// and their paths have little in common.  Targets spread over the box of one halo,
// together / so / each lane alone as they came (ms a call, FAST): a million sources
// and as many targets 4.4 / 2.3 / 2.5, 262,144 targets 3.2 / 1.7 / 1.9, 100,000
// sources and a million targets 2.6 / 1.9 / 1.6.  A chunk that four waves or more share
// is walked together: they are the chunks of calls with few targets, whose longest
// path alone would be the call.  Called by whole waves; t: the lane's target.
__device__ __forceinline__ bool chunk_alone(const TgtArgs &A, bool live, int t, int nb, int reach) {
  const int b = live ? A.bucket[t] : nb - 1;
  const int next = __shfl_down(b, 1, WAVE);
  const bool last = (threadIdx.x & (WAVE - 1)) == WAVE - 1;
  int apart = last || next == nb - 1 ? 0 : min(next - b, reach / 4);
  for (int d = WAVE / 2; d > 0; d >>= 1) apart += __shfl_xor(apart, d, WAVE);
  return 2 * __popcll(__ballot(live && b == nb - 1)) > __popcll(__ballot(live)) || apart > reach;
}

// The chunks that walk alone, counted.
__global__ void __launch_bounds__(BLOCK) tgt_apart_kernel(TgtArgs A, int nb, int reach) {
  int n = 0;
  for (int i0 = blockIdx.x * BLOCK + (threadIdx.x & ~(WAVE - 1)); i0 < A.n; i0 += gridDim.x * BLOCK) {
    const int i = i0 + (int)(threadIdx.x & (WAVE - 1));
    n += chunk_alone(A, i < A.n, i < A.n ? A.order[i] : 0, nb, reach) ? 1 : 0;
  }
  if (n > 0 && (threadIdx.x & (WAVE - 1)) == 0) atomicAdd(A.apart, n);
}

// Each lane walks a path of its own, over the targets in tree order or as they
// came (then a periodic box always takes the wrapped separations, which give the
// same bits where nothing wraps).
template <bool ORDERED>
__global__ void __launch_bounds__(BLOCK) walk_points_lane_kernel(Work W, DevParams P, TgtArgs A) {
  Seg S = W.seg[0];
  S.straddle = ORDERED ? (targets_wrap(S, P, A) ? 1 : 0) : P.periodic;
  unsigned ni = 0, no = 0;
  for (int i = blockIdx.x * BLOCK + threadIdx.x; i < A.n; i += gridDim.x * BLOCK) {
    const int t = ORDERED ? A.order[i] : i;
    A.out[t] = walk_dispatch<false>(W, P, S, A.x[t], A.y[t], A.z[t], A.m ? A.m[t] : 0.f, ni, no);
  }
}

// One target per lane, in tree order, GROUP lanes together: 16, or 64 in trees
// beyond byte_walk.  MIXED: some chunks' lanes alone.  Both forms are launched and
// one runs, the mixed one where more than one chunk in 20 is to walk alone: with
// both walks in one kernel the walk together takes 8% longer.
template <int GROUP, bool MIXED>
__global__ void __launch_bounds__(BLOCK) walk_points_kernel(Work W, DevParams P, TgtArgs A,
                                                            const Item *__restrict__ it, int nb, int reach) {
  if ((*A.apart > A.n / (20 * WAVE)) != MIXED) return;
  Seg S = W.seg[0];
  S.straddle = targets_wrap(S, P, A) ? 1 : 0;
  WalkCount wc;
  for (int i0 = blockIdx.x * BLOCK + (threadIdx.x & ~(WAVE - 1)); i0 < A.n; i0 += gridDim.x * BLOCK) {
    const int i = i0 + (int)(threadIdx.x & (WAVE - 1));
    const bool live = i < A.n;
    const int t = live ? A.order[i] : 0;
    const float x = A.x[t], y = A.y[t], z = A.z[t], tm = A.m ? A.m[t] : 0.f;
    if (MIXED && chunk_alone(A, live, t, nb, reach)) {  // uniform across the wave
      unsigned ni = 0, no = 0;
      if (live) A.out[t] = walk_dispatch<false>(W, P, S, x, y, z, tm, ni, no);
      continue;
    }
    const double pot = walk_group_dispatch<GROUP, false, false>(it, P, S, 0, S.n_items, live, x, y, z, tm, wc);
    if (live) A.out[t] = pot * (double)P.G / (double)P.a;
  }
}

// The same with PARTS waves to 64 targets, one chunk per workgroup.
template <int PARTS>
__global__ void __launch_bounds__(PARTS *WAVE) walk_points_split_kernel(Work W, DevParams P, TgtArgs A,
                                                                        const Item *__restrict__ it, int nb,
                                                                        int reach) {
  __shared__ double part[PARTS - 1][WAVE];
  const Seg &S = W.seg[0];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int i = blockIdx.x * WAVE + (int)(threadIdx.x & (WAVE - 1));
  const bool live = i < A.n;
  const int t = live ? A.order[i] : 0;
  const float x = A.x[t], y = A.y[t], z = A.z[t], tm = A.m ? A.m[t] : 0.f;
  if (PARTS == 2 && chunk_alone(A, live, t, nb, reach)) {  // uniform across the workgroup; each wave takes a part of the targets
    Seg T = S;
    T.straddle = targets_wrap(S, P, A) ? 1 : 0;
    unsigned ni = 0, no = 0;
    if (live && (int)(threadIdx.x & (WAVE - 1)) / (WAVE / PARTS) == w) A.out[t] = walk_dispatch<false>(W, P, T, x, y, z, tm, ni, no);
    return;
  }
  const int M = S.n_items;
  const int mid = A.bucket[A.order[min((int)blockIdx.x * WAVE + WAVE / 2, A.n - 1)]] << BUCKET_BITS;
  const int own = __builtin_amdgcn_readfirstlane((int)((int64_t)M * min(mid, S.n_src) / S.n_src));
  double pot;
  if (targets_wrap(S, P, A)) pot = walk_part<PARTS, FastTerm<true, true>>(it, P, w, own, M, live, x, y, z, tm);
  else pot = walk_part<PARTS, FastTerm<false, true>>(it, P, w, own, M, live, x, y, z, tm);
  pot = add_parts<PARTS>(pot, part);
  if (w == 0 && live) A.out[t] = pot * (double)P.G / (double)P.a;
}

}  // namespace

extern "C" int hbt_tree_potential(hbt_ctx *ctx, int64_t n_src, const float *sx, const float *sy,
                                  const float *sz, const float *smass, int64_t n_tgt, const float *tx,
                                  const float *ty, const float *tz, const float *target_mass,
                                  double *out_phi) {
  if (!ctx || n_src < 1 || n_tgt < 0 || !sx || !sy || !sz || !smass || (n_tgt > 0 && (!tx || !ty || !tz || !out_phi)))
    return fail(HBT_ERR_INVALID_ARG, "bad argument");
  if (n_src >= INT32_MAX / 2) return fail(HBT_ERR_UNSUPPORTED, "too many sources");
  HIPCHK(hipSetDevice(ctx->device));
  hbt_subhalo h{};
  h.count = n_src;
  h.parent = -1;
  Nest N;
  RETCHK(plan_nests(&h, 1, N));
  Level L;
  build_level(N, std::vector<int>{0}, ctx->tune, nullptr, 1, L);
  RETCHK(ensure_slots(ctx, L.nslots, 1, (int64_t)L.tiles.size()));
  const TargetWalk form = target_walk(n_src, n_tgt, ctx->params.precision);
  if (n_tgt > 0 && form != TargetWalk::alone)
    RETCHK(ctx->tgt.ensure(((size_t)(n_src >> BUCKET_BITS) + 2) * 12 + 28 + (size_t)std::min(n_tgt, TGT_SLICE) * 12));
  RETCHK(stage_level(ctx, L));
  Runner R;
  R.c = ctx;
  R.L = &L;
  R.P = make_dev_params(ctx->params);
  R.W = make_work(ctx, L, nullptr, nullptr, nullptr, nullptr);
  R.max_n = L.maxcap;
  R.list_all();
  R.gseg = 1;
  hipStream_t st = ctx->stream;
  seg_expand_kernel<<<1, BLOCK, 0, st>>>(R.W, R.P, ctx->segin.as<SegIn>(), 0);
  seg_of_slot_kernel<<<grid_for(L.nslots, ctx->cus), BLOCK, 0, st>>>(1, R.W.ibase, L.nslots,
                                                                      ctx->seg_of_slot.as<int>());
  tree_only_setup_kernel<<<1, 1, 0, st>>>(R.W, (int)n_src);
  tree_sources_kernel<<<grid_for(n_src, ctx->cus), BLOCK, 0, st>>>(R.W, (int)n_src, sx, sy, sz, smass);
  RETCHK(R.build_tree(false, form != TargetWalk::alone));  // the targets' order reads the sorted digits
  const int nb = (int)(n_src >> BUCKET_BITS) + 2;  // a target's place among the sources is 0 .. n_src, or far from them
  for (int64_t t0 = 0; t0 < n_tgt; t0 += TGT_SLICE) {
    TgtArgs A{};
    A.n = (int)std::min<int64_t>(TGT_SLICE, n_tgt - t0);
    A.x = tx + t0; A.y = ty + t0; A.z = tz + t0;
    A.m = target_mass ? target_mass + t0 : nullptr;
    A.out = out_phi + t0;
    if (form == TargetWalk::alone) {
      walk_points_lane_kernel<false><<<grid_for(A.n, ctx->cus), BLOCK, 0, st>>>(R.W, R.P, A);
      continue;
    }
    A.first = ctx->tgt.as<u64>();
    A.count = (int *)(A.first + nb);
    A.box = (u32 *)(A.count + nb);
    A.apart = (int *)(A.box + 6);
    A.bucket = A.apart + 1;
    A.rank = A.bucket + A.n;
    A.order = A.rank + A.n;
    const int *n = R.count_row(NC_SORT);
    tgt_clear_kernel<<<grid_for(nb, ctx->cus), BLOCK, 0, st>>>(R.W, A, nb);
    if (nb <= LDS_BUCKETS) {
      const int per = std::max((A.n + ctx->cus - 1) / ctx->cus, BLOCK);
      tgt_bucket_lds_kernel<<<(A.n + per - 1) / per, BLOCK, 0, st>>>(R.W, A, nb, per);
    } else {
      tgt_bucket_kernel<<<grid_for(A.n, ctx->cus), BLOCK, 0, st>>>(R.W, A, nb);
    }
    // the level's tile table starts at the buckets' tiles (fewer buckets than sources)
    const int nt = (nb + TILE - 1) / TILE, g = std::min(nt, ctx->cus * 8);
    scan_tiles_kernel<u64><<<g, BLOCK, 0, st>>>(R.tl_cur, nt, n, ctx->tsum.as<u64>(), TgtLoad{A.count}, TgtStore{A.first});
    if (nt > 1) scan_add_kernel<u64><<<g, BLOCK, 0, st>>>(R.tl_cur, nt, n, ctx->tsum.as<u64>(), TgtAdd{A.first});
    tgt_order_kernel<<<grid_for(A.n, ctx->cus), BLOCK, 0, st>>>(A);
    if (form == TargetWalk::alone_ordered) {
      walk_points_lane_kernel<true><<<grid_for(A.n, ctx->cus), BLOCK, 0, st>>>(R.W, R.P, A);
      continue;
    }
    const int chunks = (A.n + WAVE - 1) / WAVE;
    const int parts = byte_walk(n_src) && R.P.wide_sum ? walk_parts(chunks, ctx->cus) : 1;
    const int reach = WAVE * target_reach(ctx->params.precision) >> BUCKET_BITS;
    const int blocks = (A.n + BLOCK - 1) / BLOCK;
    switch (parts) {
      case 16: walk_points_split_kernel<16><<<chunks, 16 * WAVE, 0, st>>>(R.W, R.P, A, R.W.items, nb, reach); break;
      case 8: walk_points_split_kernel<8><<<chunks, 8 * WAVE, 0, st>>>(R.W, R.P, A, R.W.items, nb, reach); break;
      case 4: walk_points_split_kernel<4><<<chunks, 4 * WAVE, 0, st>>>(R.W, R.P, A, R.W.items, nb, reach); break;
      case 2: walk_points_split_kernel<2><<<chunks, 2 * WAVE, 0, st>>>(R.W, R.P, A, R.W.items, nb, reach); break;
      default:
        tgt_apart_kernel<<<grid_for(A.n, ctx->cus), BLOCK, 0, st>>>(A, nb, reach);
        if (byte_walk(n_src)) {
          walk_points_kernel<16, false><<<blocks, BLOCK, 0, st>>>(R.W, R.P, A, R.W.items, nb, reach);
          walk_points_kernel<16, true><<<blocks, BLOCK, 0, st>>>(R.W, R.P, A, R.W.items, nb, reach);
        } else {
          walk_points_kernel<64, false><<<blocks, BLOCK, 0, st>>>(R.W, R.P, A, R.W.items, nb, reach);
          walk_points_kernel<64, true><<<blocks, BLOCK, 0, st>>>(R.W, R.P, A, R.W.items, nb, reach);
        }
    }
  }
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(st));
  return HBT_OK;
}
