// hbt_mask.hpp -- hbt_mask_subhalos: exclusive particle ownership inside each
// host halo (SubhaloMasker_t / SubhaloSnapshot_t::MaskSubhalos,
// src/subhalo_tracking.cpp:793-841).  Included by hbt_unbind.hip.
//
// The host orders each group's subhalos in the reference's visit order
// (post-order from the central, the other heads nested in it after its own
// nested subhalos) and lays the entries of the subhalos that claim (Nbound >
// 1) out group by group in that order, so an entry's position in its group is
// its claim order.  On the device:
//   mask_gather   key = particle ID (sign bit flipped: unsigned order =
//                 signed order), value = claim order
//   groups of up to CLAIM_CAP entries, mask_claim: a table in LDS holds the
//   first claim of each ID; the keep flags and their scan
//   larger ones: segmented sort by (ID, claim order), mask_owner (the first
//   entry of every run of equal IDs keeps its particle), segmented scan
//   mask_write    each subhalo's kept entries in list order at the front of its
//                 range
// Subhalos that do not claim (orphans, field) keep their lists (mask_copy).
#pragma once

namespace {

struct MaskSub {
  int64_t offset;  // list range in the particle columns
  int64_t count;
  int grp;         // group segment, -1: list kept as it is
  int gstart;      // first claim position in the group segment
};

// Groups whose first claims a workgroup finds in LDS: of up to CLAIM_SMALL
// entries by one of 256 threads, of up to CLAIM_CAP by one of 1,024.
constexpr int CLAIM_SMALL = 1024, CLAIM_CAP = 8192;

struct MaskArgs {
  const MaskSub *sub;
  int nsub;
  const int64_t *gbase;  // first slot of each group segment
  const int *gn;         // entries per group segment
  const int64_t *id;
  u64 *k0;
  u32 *v0;
  unsigned char *keep;
  u64 *scan;
  int64_t *out_list;
  int64_t *new_count;
};

__global__ void __launch_bounds__(BLOCK) mask_copy_kernel(MaskArgs A) {
  for (int s = blockIdx.x; s < A.nsub; s += gridDim.x) {
    const MaskSub m = A.sub[s];
    if (m.grp >= 0) continue;
    for (int64_t l = threadIdx.x; l < m.count; l += BLOCK) A.out_list[m.offset + l] = m.offset + l;
    if (threadIdx.x == 0) A.new_count[s] = m.count;
  }
}

__global__ void __launch_bounds__(BLOCK) mask_gather_kernel(MaskArgs A) {
  for (int s = blockIdx.x; s < A.nsub; s += gridDim.x) {
    const MaskSub m = A.sub[s];
    if (m.grp < 0) continue;
    const int64_t b = A.gbase[m.grp] + m.gstart;
    const bool sorted = A.gn[m.grp] > CLAIM_CAP;
    for (int64_t l = threadIdx.x; l < m.count; l += BLOCK) {
      A.k0[b + l] = (u64)A.id[m.offset + l] ^ (1ull << 63);
      if (sorted) A.v0[b + l] = (u32)(m.gstart + l);
    }
  }
}

// The first claims of a group of n <= T PER entries, a workgroup's: a table of
// twice as many places holds a claim for each ID, the smallest once all are in.  A
// place keeps the ID it was taken for, so a claim is compared with whichever
// claim of that ID stands there, and half of the places stay empty, so every
// probe ends.  The IDs themselves stay in memory: a probe of a taken place reads
// one through the L2, which bounds the kernel, and the table of a group of 8,192
// leaves room for a second workgroup on the CU.  1,000 groups (4.0 M entries)
// take 54 us in both sizes where their sort, owners and scan took 190; the call
// 0.67 -> 0.44 ms, with 20 groups 0.20 -> 0.08.
// Both sides of the line, us a call with 400 groups (20 groups) of one size: 2,000
// entries 123 by table, 185 sorted (58, 107); 4,096 128, 231 (61, 113); 8,192 153,
// 330 (67, 128).  A table for 16,384, 128 KiB and one workgroup on a CU, in this
// one's place costs groups of 8,192 180 (77) and gives those of 12,000 200 for 444
// sorted (84, 146), of 16,384 221 for 554 (90, 147): it would pay as a third size
// beside these two, which is not built.
template <int T, int PER>
__global__ void __launch_bounds__(T) mask_claim_kernel(MaskArgs A, const int *groups, int ngroups) {
  constexpr u32 SLOTS = 2u * T * PER, EMPTY = ~0u;
  __shared__ u32 claim[SLOTS];
  __shared__ u32 wsum[T / WAVE];
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  for (int i = blockIdx.x; i < ngroups; i += gridDim.x) {
    const int n = A.gn[groups[i]];
    const int64_t b = A.gbase[groups[i]];
    const u64 *id = A.k0 + b;
    u32 slots = 2 * WAVE;  // no more than needed: they are cleared
    while (slots < 2 * (u32)n) slots *= 2;
    for (u32 h = threadIdx.x; h < slots; h += T) claim[h] = EMPTY;
    u64 key[PER];
    const int c0 = PER * (int)threadIdx.x;
#pragma unroll
    for (int r = 0; r < PER; r++) key[r] = id[min(c0 + r, n - 1)];
    __syncthreads();
    u32 at[PER];
#pragma unroll
    for (int r = 0; r < PER; r++) {
      const u32 c = (u32)(c0 + r);
      at[r] = 0;
      if (c >= (u32)n) continue;
      u32 h = (u32)id_hash((long long)key[r]) & (slots - 1);
      for (;;) {
        const u32 p = atomicCAS(&claim[h], EMPTY, c);
        if (p == EMPTY) break;
        if (id[p] == key[r]) {
          if (c < p) atomicMin(&claim[h], c);
          break;
        }
        h = (h + 1) & (slots - 1);
      }
      at[r] = h;
    }
    __syncthreads();
    u32 kept = 0, mine = 0;
#pragma unroll
    for (int r = 0; r < PER; r++) {
      const bool first = c0 + r < n && claim[at[r]] == (u32)(c0 + r);
      mine |= (u32)first << r;
      kept += first;
    }
    u32 ex = wave_inclusive_scan(kept);
    if (lane == WAVE - 1) wsum[w] = ex;
    __syncthreads();
    ex -= kept;
    for (int u = 0; u < w; u++) ex += wsum[u];
#pragma unroll
    for (int r = 0; r < PER; r++) {
      if (c0 + r >= n) continue;
      A.keep[b + c0 + r] = mine >> r & 1;
      A.scan[b + c0 + r] = ex;
      ex += mine >> r & 1;
    }
    __syncthreads();  // the table and wsum are written again
  }
}

// sorted position i of a larger group: owner iff its ID differs from position i-1
__global__ void __launch_bounds__(BLOCK) mask_owner_kernel(MaskArgs A, const Tile *tiles, int ntiles) {
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const int64_t b = A.gbase[tl.seg];
    const int end = min(tl.start + TILE, A.gn[tl.seg]);
    for (int i = tl.start + (int)threadIdx.x; i < end; i += BLOCK) {
      const bool owner = i == 0 || A.k0[b + i - 1] != A.k0[b + i];
      A.keep[b + A.v0[b + i]] = owner ? 1 : 0;
    }
  }
}

struct KeepLoad {
  const int64_t *gbase; const unsigned char *keep;
  __device__ u64 operator()(int g, int l) const { return (u64)keep[gbase[g] + l]; }
};
struct KeepStore {
  const int64_t *gbase; u64 *scan;
  __device__ void operator()(int g, int l, u64 x) const { scan[gbase[g] + l] = x; }
};
struct KeepAdd {
  const int64_t *gbase; u64 *scan;
  __device__ void operator()(int g, int l, u64 x) const { scan[gbase[g] + l] += x; }
};

__global__ void __launch_bounds__(BLOCK) mask_write_kernel(MaskArgs A) {
  for (int s = blockIdx.x; s < A.nsub; s += gridDim.x) {
    const MaskSub m = A.sub[s];
    if (m.grp < 0) continue;
    const int64_t b = A.gbase[m.grp] + m.gstart;
    const u64 first = A.scan[b];
    u64 kept = 0;
    for (int64_t l = threadIdx.x; l < m.count; l += BLOCK) {
      if (!A.keep[b + l]) continue;
      A.out_list[m.offset + (int64_t)(A.scan[b + l] - first)] = m.offset + l;
      kept++;
    }
    u64 tot;
    (void)block_exclusive_scan(kept, &tot);
    if (threadIdx.x == 0) A.new_count[s] = (int64_t)tot;
  }
}

}  // namespace

extern "C" int hbt_mask_subhalos(hbt_ctx *ctx, const hbt_particles *particles, const hbt_subhalo *subs_host,
                                 const int64_t *host_group, const int64_t *visit_rank, int64_t nsub, int64_t *out_list,
                                 int64_t *new_count) {
  if (!ctx || !particles || nsub < 0 || (nsub > 0 && (!subs_host || !host_group || !out_list || !new_count)))
    return fail(HBT_ERR_INVALID_ARG, "bad argument");
  if (nsub == 0) return HBT_OK;
  if (nsub >= (int64_t)INT32_MAX) return fail(HBT_ERR_UNSUPPORTED, "too many subhalos");
  if (!particles->id) return fail(HBT_ERR_INVALID_ARG, "particle IDs are required");
  HIPCHK(hipSetDevice(ctx->device));
  // nesting and heads per group
  std::vector<std::vector<int>> nested(nsub);
  std::vector<int> head_of_group;  // central per group segment
  std::unordered_map<int64_t, int> gidx;
  std::vector<std::vector<int>> heads;
  for (int64_t s = 0; s < nsub; s++) {
    const hbt_subhalo &r = subs_host[s];
    if (r.count < 0 || r.offset < 0 || r.offset + r.count > particles->n)
      return fail(HBT_ERR_INVALID_ARG, "subhalo list outside the particle columns");
    const int64_t p = r.parent;
    if (p >= 0) {
      if (p >= nsub || p == s || host_group[p] != host_group[s])
        return fail(HBT_ERR_INVALID_ARG, "a nested subhalo must share its parent's host group");
      nested[p].push_back((int)s);
    } else if (host_group[s] >= 0) {
      auto it = gidx.find(host_group[s]);
      if (it == gidx.end()) {
        gidx.emplace(host_group[s], (int)heads.size());
        heads.push_back({(int)s});
      } else {
        heads[it->second].push_back((int)s);
      }
    }
  }
  // siblings in the caller's visit order (the reference's SubGroups order for
  // a group's heads, its central first; NestedSubhalos order for nested ones)
  if (visit_rank) {
    auto by_rank = [&](int a, int b) { return visit_rank[a] != visit_rank[b] ? visit_rank[a] < visit_rank[b] : a < b; };
    for (auto &v : nested) std::sort(v.begin(), v.end(), by_rank);
    for (auto &v : heads) std::sort(v.begin(), v.end(), by_rank);
  }
  // visit order (post-order from the central; the other heads nested in the
  // central after its own nested subhalos), claim positions per group
  std::vector<MaskSub> ms(nsub);
  for (int64_t s = 0; s < nsub; s++) ms[s] = MaskSub{subs_host[s].offset, subs_host[s].count, -1, 0};
  std::vector<int64_t> gbase;
  std::vector<int> gn, claims[2];
  std::vector<Tile> tiles;  // of the groups that are sorted
  std::vector<char> seen(nsub, 0);
  int64_t off = 0;
  int maxn = 0;
  for (size_t g = 0; g < heads.size(); g++) {
    const int central = heads[g][0];
    int64_t pos = 0;
    // iterative post-order: (node, next child index)
    std::vector<std::pair<int, size_t>> stack{{central, 0}};
    while (!stack.empty()) {
      auto &top = stack.back();
      const int s = top.first;
      const std::vector<int> &kids = nested[s];
      const size_t nk = kids.size() + (s == central ? heads[g].size() - 1 : 0);
      if (top.second < nk) {
        const size_t i = top.second++;
        const int c = i < kids.size() ? kids[i] : heads[g][1 + (i - kids.size())];
        if (seen[c]) return fail(HBT_ERR_INVALID_ARG, "nesting has a cycle");
        seen[c] = 1;
        stack.push_back({c, 0});
        continue;
      }
      stack.pop_back();
      if (subs_host[s].nbound_prev > 1 && subs_host[s].count > 0) {
        ms[s].grp = (int)gbase.size();
        ms[s].gstart = (int)pos;
        pos += subs_host[s].count;
      }
    }
    if (pos >= (int64_t)INT32_MAX / 2) return fail(HBT_ERR_UNSUPPORTED, "host group too large");
    if (pos == 0) continue;
    const int k = (int)gbase.size();
    gbase.push_back(off);
    gn.push_back((int)pos);
    off += (pos + WAVE - 1) / WAVE * WAVE;
    if (pos <= CLAIM_CAP) {
      claims[pos <= CLAIM_SMALL ? 0 : 1].push_back(k);
      continue;
    }
    const int nt = (int)((pos + TILE - 1) / TILE);
    for (int t = 0; t < nt; t++) tiles.push_back(Tile{k, t * TILE});
    maxn = std::max(maxn, (int)pos);
  }
  // groups whose central never got a segment keep -1; map group ids for subhalos
  // that claim: ms[s].grp was set to the segment about to be created
  const int ngrp = (int)gbase.size();
  hipStream_t st = ctx->stream;
  RETCHK(ensure_slots(ctx, std::max<int64_t>(off, 1), std::max(ngrp, 1), std::max<int64_t>((int64_t)tiles.size(), 1)));
  DBuf dcnt;
  RETCHK(dcnt.ensure(nsub * 8));
  void *d[6];
  int rc = stage_blobs(ctx, {{ms.data(), ms.size() * sizeof(MaskSub)},
                             {gbase.data(), gbase.size() * 8},
                             {gn.data(), gn.size() * 4},
                             {claims[0].data(), claims[0].size() * 4},
                             {claims[1].data(), claims[1].size() * 4},
                             {tiles.data(), tiles.size() * sizeof(Tile)}},
                       d);
  if (rc != HBT_OK) { dcnt.release(); return rc; }
  MaskArgs A{};
  A.sub = (const MaskSub *)d[0];
  A.nsub = (int)nsub;
  A.gbase = (const int64_t *)d[1];
  A.gn = (const int *)d[2];
  A.id = particles->id;
  A.k0 = ctx->k0.as<u64>();
  A.v0 = ctx->v0.as<u32>();
  A.keep = ctx->isb.as<unsigned char>();
  A.scan = ctx->scan64.as<u64>();
  A.out_list = out_list;
  A.new_count = dcnt.as<int64_t>();
  const int gsub = (int)std::min<int64_t>(nsub, (int64_t)ctx->cus * 8);
  mask_copy_kernel<<<gsub, BLOCK, 0, st>>>(A);
  if (ngrp > 0) {
    mask_gather_kernel<<<gsub, BLOCK, 0, st>>>(A);
    const int nc0 = (int)claims[0].size(), nc1 = (int)claims[1].size(), nt = (int)tiles.size();
    if (nc0 > 0)
      mask_claim_kernel<BLOCK, CLAIM_SMALL / BLOCK><<<std::min(nc0, ctx->cus * 8), BLOCK, 0, st>>>(A, (const int *)d[3], nc0);
    if (nc1 > 0)
      mask_claim_kernel<1024, CLAIM_CAP / 1024><<<std::min(nc1, ctx->cus * 2), 1024, 0, st>>>(A, (const int *)d[4], nc1);
    if (nt > 0) {
      const Tile *dt = (const Tile *)d[5];
      const int gt = std::min(nt, ctx->cus * 8);
      const int gm = (int)std::min<int64_t>((int64_t)nt * (TILE / BLOCK), (int64_t)ctx->cus * 16);
      tile_sort_kernel<<<gt, BLOCK, 0, st>>>(dt, nt, A.gbase, A.gn, A.k0, A.v0, ctx->k1.as<u64>(), ctx->v1.as<u32>());
      int level = 0;
      for (int64_t w = TILE; w < maxn; w *= 2, level++)
        merge_pass_kernel<<<gm, BLOCK, 0, st>>>(dt, nt, A.gbase, A.gn, TILE, level, A.k0, A.v0, ctx->k1.as<u64>(),
                                                ctx->v1.as<u32>());
      mask_owner_kernel<<<gt, BLOCK, 0, st>>>(A, dt, nt);
      u64 *ts = ctx->tsum.as<u64>();
      scan_tiles_kernel<u64><<<gt, BLOCK, 0, st>>>(dt, nt, A.gn, ts, KeepLoad{A.gbase, A.keep}, KeepStore{A.gbase, A.scan});
      scan_add_kernel<u64><<<gt, BLOCK, 0, st>>>(dt, nt, A.gn, ts, KeepAdd{A.gbase, A.scan});
    }
    mask_write_kernel<<<gsub, BLOCK, 0, st>>>(A);
  }
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(new_count, dcnt.p, nsub * 8, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  dcnt.release();
  if (e != hipSuccess) return fail(HBT_ERR_DEVICE, std::string("mask_subhalos: ") + hipGetErrorString(e));
  return HBT_OK;
}
