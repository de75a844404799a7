// hbt_kernels.hpp -- the unbinding pass kernels (gfx950).
//
// One pass of the reference's Unbind loop (src/subhalo_unbind.cpp:310-422)
// runs for every active segment (subhalo) of a level at once:
//   begin_pass        full pass over Elist[0,Nlast) or correction pass over the
//                     freshly removed block Elist[Nbound,Nlast) (:312-356), set
//                     up at the end of the pass before
//   tree_one          a segment of one tile: its whole tree in one launch
//   bbox / keys_sort / (merge levels) / emit / items_tile / moments_super, _cross
//                     the others: root cube and per-particle octant digits
//                     computed with the reference's double-precision centre
//                     iteration (src/oct_tree.tpp:118-224), their segmented sort,
//                     and from the sorted digits the compressed octree in pre-order
//                     with skip pointers; node moments accumulated in double over
//                     float children in son order (src/gravity_tree.cpp:18-77)
//   walk              stackless walk per target (src/gravity_tree.cpp:79-175)
//   post_one          a segment of one tile: the rest of the pass in one launch
//   partition_*       the others: parallel replica of PartitionBindingEnergy (:21-58)
//   frames            FP64 AverageVelocity/AveragePosition, convergence (:357-421)
//   output            permuted list, kinematics, particle-type counts (:405-431)
#pragma once
#include "hbt_device.hpp"
#include "../../include/hbt_unbind.h"

namespace hbt {

// One tree item (leaf or node) in DFS pre-order, one 32-byte record: the
// walk reads both halves of an item at once.
// Rows of Work::ncount, each written by the kernel that decides the count:
// sources of the tree (begin_pass), the energy sort (frames), the tree's nodes
// that span super-tiles (bbox, items).
enum { NC_SRC = 0, NC_SORT = 1, NC_CROSS = 2, NC_ROWS = 3 };

struct __align__(32) Item {
  float4 pm;   // x, y, z, mass (a node: centre of mass and total mass)
  int2 ax;     // float bits of len^2 (0 for a leaf), skip (first item after the subtree)
  int2 sb;     // skip as a byte offset from the segment's first item (32 * skip); float bits of the
               // squared distance below which the FP32 walk opens the node (0 for a leaf)
};

static_assert(sizeof(Item) == 32, "the walks step by 32 bytes");

struct Work {
  // per level
  Seg *seg;
  int nseg;
  int nmulti;                // segments of more than one tile
  int64_t nslots;
  // the slots a pass visits: all (act_chunk null, nact = nslots) or the
  // wave-sized chunks of the segments still active (nact = 64 * chunks)
  const int *act_chunk;
  int64_t nact;
  int *segact;               // [nseg] nonzero: the segment stays active after the pass
  const int *seg_of_slot;
  const int64_t *ibase;
  int *ncount;               // [NC_ROWS][nseg] element counts of the pass's scans and sorts
  // particle columns of the caller (device)
  const int64_t *g_id;
  const float *g_x, *g_y, *g_z, *g_vx, *g_vy, *g_vz, *g_m;
  const int32_t *g_type;
  const int64_t *g_index;    // optional: list entry -> particle column position
  const float4 *g_packed;    // optional: the columns interleaved, 2 float4 per particle
  // working arrays [nslots]
  int *gidx;
  float4 *pos;               // x, y, z, mass: one record, so a gather reads one line
  float4 *vel;               // vx, vy, vz, type (int bits)
  float *E;
  float *Er;                 // energies of the refinement pass (RefineBindingEnergyOrder)
  int *el, *el2, *sp;
  u64 *k0, *k1;
  u32 *v0, *v1;
  signed char *dl;
  u32 *bits;
  int *pre, *nlo, *nhi, *npos;
  int *cross;                // per super-tile: pairs of the nodes whose leaves span tiles in it
  int *cross2;               // per segment: pairs of the nodes whose leaves span super-tiles
  int *tcount;               // per tile of the pass's table: list length of the super-tile it starts
  Item *items;               // [2*nslots] tree items in pre-order
  unsigned char *isb;
  int *active;               // [4]: segments active after the pass, the largest Nlast among them, blocks that
                             // have counted, refinements pending in the level
  int *host_active;          // the same for the host (pinned)
  unsigned long long *counters;  // interactions, opened nodes, targets (instrumented passes); [4] evaluations
  // caller outputs
  hbt_subhalo *subs;
  int64_t *out_index;
  float *out_energy;
};

// counts list entries that are not positions in [0, n)
__global__ void check_index_kernel(const int64_t *idx, int64_t n_list, int64_t n, int *bad) {
  int cnt = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_list; i += (int64_t)gridDim.x * blockDim.x)
    cnt += (idx[i] < 0 || idx[i] >= n) ? 1 : 0;
  if (cnt) atomicAdd(bad, cnt);
}

// The slots a wave visits form one wave-aligned chunk, and segments start at
// multiples of WAVE, so a wave's slots share one segment: the lookups read
// one entry for the wave (scalar loads of a wave-uniform address).
__device__ __forceinline__ int seg_lane_local(const Work &W, int64_t s, int &k) {
  const int64_t s0 = (int64_t)__builtin_amdgcn_readfirstlane((int)(s >> 6)) << 6;
  k = W.seg_of_slot[s0];
  if (k < 0) return -1;
  return (int)(s - W.ibase[k]);
}

// i-th visited slot (the active lists hold wave-sized chunks, nact a multiple of WAVE)
__device__ __forceinline__ int64_t slot_at(const Work &W, int64_t i) {
  if (W.act_chunk && i < W.nact) {
    const int c = __builtin_amdgcn_readfirstlane((int)(i >> 6));
    return (int64_t)W.act_chunk[c] * WAVE + (i & (WAVE - 1));
  }
  return i;
}

#define SLOT_LOOP(s, W)                                                                        \
  for (int64_t s##_i = (int64_t)blockIdx.x * BLOCK + threadIdx.x, s = slot_at((W), s##_i);    \
       s##_i < (W).nact; s##_i += (int64_t)gridDim.x * BLOCK, s = slot_at((W), s##_i))

// The segments of more than one tile come first in a level.
#define MULTI_SEG_LOOP(k, W) \
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < (W).nmulti; k += gridDim.x * blockDim.x)

#define SEG_LOOP(k, W) \
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < (W).nseg; k += gridDim.x * blockDim.x)

// One wave per segment of the first n (k is wave-uniform).
#define WAVE_SEG_LOOP(k, n)                                                     \
  for (int k = (int)((blockIdx.x * blockDim.x + threadIdx.x) / WAVE); k < (n); \
       k += (int)(gridDim.x * blockDim.x / WAVE))

// Sums of C values over the tiles t0 .. t0+nt-1 of part: the wave's lanes take
// strided tiles, then wave_total; the sums are valid in every lane.
template <int C>
__device__ __forceinline__ void wave_sum_tiles(const double *__restrict__ part, int t0, int nt, double v[C]) {
#pragma clang fp contract(off)
  for (int c = 0; c < C; c++) v[c] = 0;
  for (int t = t0 + (int)(threadIdx.x & (WAVE - 1)); t < t0 + nt; t += WAVE)
    for (int c = 0; c < C; c++) v[c] += part[(int64_t)t * C + c];
  for (int c = 0; c < C; c++) v[c] = wave_total(v[c]);
}

// ---------------------------------------------------------------------------
// Level initialisation

// Fills seg_of_slot for the level.
__global__ void fill_seg_of_slot_kernel(int nseg, const int64_t *ibase, const int *cap_aligned,
                                        int *seg_of_slot) {
  for (int k = blockIdx.x; k < nseg; k += gridDim.x) {
    const int64_t b = ibase[k];
    const int c = cap_aligned[k];
    for (int i = threadIdx.x; i < c; i += blockDim.x) seg_of_slot[b + i] = k;
  }
}

// The same, slot-parallel, for a level whose segments tile the slots in order
// (ibase ascending, each segment's slots followed by the next one's): a slot's
// segment is the last one starting at or before it.  A giant segment is then
// not left to one workgroup.
__global__ void __launch_bounds__(BLOCK) seg_of_slot_kernel(int nseg, const int64_t *__restrict__ ibase,
                                                            int64_t nslots, int *seg_of_slot) {
  for (int64_t s = (int64_t)blockIdx.x * BLOCK + threadIdx.x; s < nslots; s += (int64_t)gridDim.x * BLOCK) {
    int lo = 0, hi = nseg - 1;  // ibase[lo] <= s
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (ibase[mid] <= s) lo = mid; else hi = mid - 1;
    }
    seg_of_slot[s] = lo;
  }
}

// The same for a level whose segments start at multiples of WAVE slots: one
// search per WAVE slots.  Each wave takes WAVE such chunks, lane i searching
// chunk i, then writes the chunks' slots one chunk per store across the lanes.
__global__ void __launch_bounds__(BLOCK) seg_of_chunk_kernel(int nseg, const int64_t *__restrict__ ibase,
                                                             int64_t nslots, int *seg_of_slot) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int64_t nchunk = (nslots + WAVE - 1) / WAVE;
  const int64_t waves = (int64_t)gridDim.x * (BLOCK / WAVE);
  for (int64_t g = (int64_t)blockIdx.x * (BLOCK / WAVE) + threadIdx.x / WAVE; g * WAVE < nchunk; g += waves) {
    const int64_t c = g * WAVE + lane;
    int lo = 0;
    if (c < nchunk) {
      const int64_t s = c * WAVE;
      int hi = nseg - 1;  // ibase[lo] <= s
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (ibase[mid] <= s) lo = mid; else hi = mid - 1;
      }
    }
    for (int j = 0; j < WAVE; j++) {
      const int k = __shfl(lo, j, WAVE);
      const int64_t s = (g * WAVE + j) * WAVE + lane;
      if (s < nslots) seg_of_slot[s] = k;
    }
  }
}

// Unbind entry (src/subhalo_unbind.cpp:263-309): early exits, initial Elist;
// the shuffle's sort count (steps 1..ulen-1) of a shuffled list.
__device__ __forceinline__ void init_segment(const Work &W, const DevParams &P, Seg &S, int k) {
  hbt_subhalo &r = W.subs[S.sub];
  const bool orphan = S.nbprev <= 1;
  S.ulen = orphan ? S.count : S.len;
  S.flags = orphan ? F_ORPHAN : 0;
  S.iter = 0;
  S.evals = 0;
  for (int j = 0; j < 3; j++) { S.ref_pos[j] = r.ref_pos[j]; S.ref_vel[j] = r.ref_vel[j]; }
  if (S.ulen < P.min_part && r.snapshot_index_of_death == -1) r.snapshot_index_of_death = P.snap;
  if (S.ulen <= 1) {
    S.flags |= F_EARLY;
    S.nbound = S.ulen;
    S.nlast = S.ulen;
  } else {
    S.flags |= F_ACTIVE;
    S.nbound = S.ulen;
    S.nlast = S.ulen;
  }
  // the host shuffles exactly the lists longer than the sample (:302), with
  // draws counted for the same length (a list of another length would read
  // other segments' draws: it is not shuffled, and parity tests show it)
  if (S.draw_off >= 0 && S.ulen > P.max_sample && P.max_sample > 0 && S.ulen == S.shuf_len) S.flags |= F_SHUF;
  else S.draw_off = -1;
  W.ncount[NC_SRC * W.nseg + k] = S.draw_off >= 0 ? S.ulen - 1 : 0;
}

// Setup of a segment's next pass: full over Elist[0, Nbound), or a correction
// over the block just removed.
__device__ __forceinline__ void begin_pass(const Work &W, const DevParams &P, Seg &S, int k) {
  S.flags &= ~(F_FINAL | F_SAMP);
  S.mf = 1.f;
  S.n_src = 0; S.n_tgt = 0; S.src_lo = 0; S.nsort = 0; S.sort_lo = 0; S.n_items = 0;
  S.K = 0; S.nP = 0; S.nG = 0;
  if (S.flags & F_ACTIVE) {
    S.iter++;
    if (S.flags & F_CORR) {
      // RelativeVelocity(OldRefPos, OldRefVel, RefPos, RefVel), dK (:314-316)
      rel_vel(P, S.old_pos[0], S.old_pos[1], S.old_pos[2], S.old_vel[0], S.old_vel[1],
              S.old_vel[2], S.ref_pos, S.ref_vel, S.rvd);
      S.dK = (float)(0.5 * (double)vnorm_f(S.rvd));
      S.src_lo = S.nbound;
      S.n_src = S.nlast - S.nbound;
      S.n_tgt = S.nbound;
      S.nlast = S.nbound;  // Nlast=Nbound after the correction loop (:329)
    } else {
      S.nlast = S.nbound;
      S.src_lo = 0;
      S.n_src = S.nlast;
      S.n_tgt = S.nlast;
      if (P.max_sample > 0 && S.nlast > P.max_sample) {
        // sampled tree: the first MaxSampleSize entries with their masses
        // scaled by Nlast / MaxSampleSize (float / long -> float, :334-339)
        S.n_src = P.max_sample;
        S.mf = (float)S.nlast / (float)P.max_sample;
        S.flags |= F_SAMP;
      }
    }
    S.evals += S.n_tgt;
    S.nsort = S.n_src;
    for (int j = 0; j < 3; j++) { S.bmin[j] = 0xffffffffu; S.bmax[j] = 0u; }
  }
  W.ncount[NC_SRC * W.nseg + k] = S.n_src;
  W.ncount[NC_SORT * W.nseg + k] = 0;
}

__device__ __forceinline__ void clear_level_counts(const Work &W) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int i = 0; i < 4; i++) W.active[i] = 0;
    W.counters[4] = 0;  // evaluations, summed after the last level
  }
}

// After build_lists_kernel (a level with nested subhalos' tails).
__global__ void seg_init_kernel(Work W, DevParams P) {
  clear_level_counts(W);
  SEG_LOOP(k, W) init_segment(W, P, W.seg[k], k);
}

// The level's segment records: zero, then the host's fixed fields.  begin: 1, the
// lists are the segments' own, and their unbinding starts here too; 2, and
// none is shuffled: their first pass also.
__global__ void __launch_bounds__(BLOCK) seg_expand_kernel(Work W, DevParams P, const SegIn *in, int begin) {
  if (begin) clear_level_counts(W);
  SEG_LOOP(k, W) {
    const SegIn a = in[k];
    Seg S{};
    S.ibase = a.ibase;
    S.out_off = a.out_off;
    S.sub = a.sub;
    S.cap = a.cap;
    S.count = a.count;
    S.list_off = a.list_off;
    S.nbprev = a.nbprev;
    S.wgroup = a.wgroup;
    S.draw_off = a.draw_off;
    S.shuf_len = a.shuf_len;
    S.mf = 1.f;
    S.swapq = INT_MAX;
    if (begin) {
      S.len = S.count;
      init_segment(W, P, S, k);
      if (begin == 2) begin_pass(W, P, S, k);
    }
    W.segact[k] = 1;
    W.seg[k] = S;
  }
}

// Builds the working list of every segment: own particles in source order
// (their positions are written by gather_kernel), then the unbound tails of
// nested subhalos (read from their output lists, src/subhalo_unbind.cpp:437-443).
// child_ptr/child_list: CSR list of the subhalos nested in each segment.
__global__ void build_lists_kernel(Work W, const int *child_ptr, const int *child_list) {
  for (int k = blockIdx.x; k < W.nseg; k += gridDim.x) {
    Seg &S = W.seg[k];
    const int64_t b = S.ibase;
    int pos = S.count;
    for (int c = child_ptr[k]; c < child_ptr[k + 1]; c++) {
      const hbt_subhalo &q = W.subs[child_list[c]];
      const int tail = (int)(q.list_len - q.nbound);
      for (int i = threadIdx.x; i < tail; i += blockDim.x)
        W.gidx[b + pos + i] = (int)W.out_index[q.out_offset + q.nbound + i];
      pos += tail;
    }
    if (threadIdx.x == 0) S.len = pos;
    __syncthreads();
  }
}

// The snapshot's columns interleaved per particle (x, y, z, mass | vx, vy, vz,
// type): a gather in list order, which is random in the snapshot, then reads
// one 32-byte record per particle instead of eight scattered words.
__global__ void __launch_bounds__(BLOCK) pack_particles_kernel(hbt_particles P, float4 *out) {
  for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < P.n; i += (int64_t)gridDim.x * BLOCK) {
    out[2 * i] = make_float4(P.x[i], P.y[i], P.z[i], P.mass[i]);
    out[2 * i + 1] = make_float4(P.vx[i], P.vy[i], P.vz[i], __int_as_float(P.type ? P.type[i] : 1));
  }
}

// Column position of list entry l of a segment's own list.
__device__ __forceinline__ int own_entry(const Work &W, const Seg &S, int l) {
  const int64_t o = S.list_off + l;
  return W.g_index ? (int)W.g_index[o] : (int)o;
}

// Column positions of the segments' own particles (phase bit 1), local copies
// of the listed particles' columns and the initial Elist (phase bit 2),
// slot-parallel.  A shuffled list is permuted between the two phases.
__global__ void __launch_bounds__(BLOCK) gather_kernel(Work W, int phase) {
  SLOT_LOOP(s, W) {
    int k;
    int l = seg_lane_local(W, s, k);
    if (l < 0 || l >= W.seg[k].len) continue;
    int g;
    if ((phase & 1) && l < W.seg[k].count) {
      g = own_entry(W, W.seg[k], l);
      W.gidx[s] = g;
    } else {
      g = W.gidx[s];
    }
    if (!(phase & 2)) continue;
    if (l < W.seg[k].ulen) W.el[s] = l;
    if (W.g_packed) {
      W.pos[s] = W.g_packed[2 * (int64_t)g];
      W.vel[s] = W.g_packed[2 * (int64_t)g + 1];
    } else {
      W.pos[s] = make_float4(W.g_x[g], W.g_y[g], W.g_z[g], W.g_m[g]);
      W.vel[s] = make_float4(W.g_vx[g], W.g_vy[g], W.g_vz[g], __int_as_float(W.g_type ? W.g_type[g] : 1));
    }
  }
}

// ---------------------------------------------------------------------------
// Shuffle (std::random_shuffle at src/subhalo_unbind.cpp:302; libstdc++'s
// form: step i = 1..n-1 swaps positions i and j_i = rand() % (i+1)), replayed
// in parallel.  Before step i position i still holds element i, so the last
// step that moves an element into position p from above (the largest i > p
// with j_i = p) leaves element i there for good.  A position that no later
// step reaches keeps what step p left: element p if j_p = p, else what
// position q = j_p held just before step p -- the element of the latest step
// i in (q, p) with j_i = q, or, if none, what step q left there, and so on
// down the chain p -> j_p -> ...  Sorting the pairs (j_i, i) groups each
// position's movers in step order; pre = j_i, nlo = the previous mover into
// j_i (-1: none), nhi = the last mover into a position (-1: none), npos =
// the list before the shuffle.

// Keys (j_i << 32 | i) of steps i = 1..ulen-1 at sort positions i-1.
__global__ void __launch_bounds__(BLOCK) shuffle_keys_kernel(Work W, const int *__restrict__ draws) {
  SLOT_LOOP(s, W) {
    int k;
    int l = seg_lane_local(W, s, k);
    if (l < 0) continue;
    Seg &S = W.seg[k];
    if (S.draw_off < 0 || l >= S.ulen) continue;
    const int64_t b = S.ibase;
    W.npos[s] = W.gidx[s];
    W.nlo[s] = -1;
    W.nhi[s] = -1;
    if (l == 0) {
      W.pre[s] = 0;
      S.old_mb_id = W.g_id[W.gidx[s]];  // OldMostboundParticle is taken before the shuffle (:297)
      continue;
    }
    const int j = (int)((unsigned)draws[S.draw_off + l - 1] % (unsigned)(l + 1));
    W.pre[s] = j;
    W.k0[b + l - 1] = ((u64)(unsigned)j << 32) | (u64)(unsigned)l;
    W.v0[b + l - 1] = 0u;
  }
}

// Previous mover into the same position, and the last mover into each position.
__global__ void __launch_bounds__(BLOCK) shuffle_links_kernel(Work W) {
  SLOT_LOOP(s, W) {
    int k;
    int t = seg_lane_local(W, s, k);
    if (t < 0) continue;
    const Seg &S = W.seg[k];
    const int n = S.ulen - 1;  // sorted steps
    if (S.draw_off < 0 || t >= n) continue;
    const int64_t b = S.ibase;
    const u64 e = W.k0[s];
    const int q = (int)(e >> 32), i = (int)(e & 0xffffffffu);
    if (i == q) continue;  // a step that swaps a position with itself moves nothing
    int prev = -1;
    if (t > 0) {
      const u64 f = W.k0[s - 1];
      if ((int)(f >> 32) == q && (int)(f & 0xffffffffu) > q) prev = (int)(f & 0xffffffffu);
    }
    W.nlo[b + i] = prev;
    if (t + 1 == n || (int)(W.k0[s + 1] >> 32) != q) W.nhi[b + q] = i;
  }
}

// The shuffled list: position p takes the element the chain above names.
__global__ void __launch_bounds__(BLOCK) shuffle_apply_kernel(Work W) {
  SLOT_LOOP(s, W) {
    int k;
    int p = seg_lane_local(W, s, k);
    if (p < 0) continue;
    const Seg &S = W.seg[k];
    if (S.draw_off < 0 || p >= S.ulen) continue;
    const int64_t b = S.ibase;
    int src = W.nhi[s];
    if (src < 0) {
      int cur = p;  // strictly decreases along the chain
      while (true) {
        if (cur == 0) { src = 0; break; }
        const int q = W.pre[b + cur];
        if (q == cur) { src = cur; break; }
        const int w = W.nlo[b + cur];
        if (w >= 0) { src = w; break; }
        cur = q;
      }
    }
    W.gidx[s] = W.npos[b + src];
  }
}

// Spatial target order of a shuffled list (its sampled trees hold only the
// first MaxSampleSize entries): a sort of every particle's octant digits in
// the cube of the whole list.  Setup: the whole unbound list as the sources.
__global__ void prelude_setup_kernel(Work W) {
  SEG_LOOP(k, W) {
    Seg &S = W.seg[k];
    const bool on = S.draw_off >= 0 && (S.flags & F_ACTIVE);
    S.n_src = on ? S.ulen : 0;
    S.src_lo = 0;
    S.n_tgt = 0;
    for (int j = 0; j < 3; j++) { S.bmin[j] = 0xffffffffu; S.bmax[j] = 0u; }
    W.ncount[NC_SRC * W.nseg + k] = S.n_src;
  }
}

// After the digit sort: the order becomes the target list, and the whole
// list's periodic straddle bounds every later pass of the segment.
__global__ void __launch_bounds__(BLOCK) prelude_sp_kernel(Work W) {
  SLOT_LOOP(s, W) {
    int k;
    int l = seg_lane_local(W, s, k);
    if (l < 0) continue;
    Seg &S = W.seg[k];
    if (S.draw_off < 0 || !(S.flags & F_ACTIVE) || l >= S.ulen) continue;
    W.sp[s] = (int)W.v0[s];
    if (l == 0) S.sall = S.straddle;
  }
}

// First pass of a level whose lists were shuffled or hold nested tails (else
// seg_expand_kernel sets it up; pass_end_kernel sets up the later ones).
__global__ void pass_begin_kernel(Work W, DevParams P) {
  SEG_LOOP(k, W) begin_pass(W, P, W.seg[k], k);
}

// ---------------------------------------------------------------------------
// Tree.  Segments of one tile (cap <= TILE) build theirs in one launch, a wave
// or a workgroup each, everything between the sources and the finished items in
// LDS (tree_one_kernel).  Larger ones go through their tiles: box, digits and
// tile sort, merge levels, nodes, pre-order positions, items and moments.  The
// trees of 200,000 subhalos' passes take 8.7 ms this way, without the merge levels
// (5.8 of it the larger segments'), 50,000 small ones' 5.8; with every stage a launch over all
// segments, through memory, 12.4 and 8.4.

// Folds every thread's box (ordered-integer encoding of the floats) over the
// block and into lo[3], hi[3].  Atomics on one address are served one after
// another at the memory side (4,000 tiles of one segment: 0.27 ms of them), so a
// block only sends those that its read of the box so far calls for; a read that
// is behind costs an atomic, never a bound.
__device__ __forceinline__ void fold_box(u32 mn[3], u32 mx[3], u32 *lo, u32 *hi) {
  __shared__ u32 sh[6][BLOCK / WAVE];
  for (int d = WAVE / 2; d > 0; d >>= 1)
    for (int j = 0; j < 3; j++) {
      mn[j] = min(mn[j], (u32)__shfl_xor((int)mn[j], d, WAVE));
      mx[j] = max(mx[j], (u32)__shfl_xor((int)mx[j], d, WAVE));
    }
  if ((threadIdx.x & (WAVE - 1)) == 0)
    for (int j = 0; j < 3; j++) { sh[j][threadIdx.x / WAVE] = mn[j]; sh[3 + j][threadIdx.x / WAVE] = mx[j]; }
  __syncthreads();
  if (threadIdx.x < 3) {
    u32 a = sh[threadIdx.x][0];
    for (int w = 1; w < BLOCK / WAVE; w++) a = min(a, sh[threadIdx.x][w]);
    if (a < __hip_atomic_load(&lo[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&lo[threadIdx.x], a);
  } else if (threadIdx.x < 6) {
    u32 a = sh[threadIdx.x][0];
    for (int w = 1; w < BLOCK / WAVE; w++) a = max(a, sh[threadIdx.x][w]);
    if (a > __hip_atomic_load(&hi[threadIdx.x - 3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(&hi[threadIdx.x - 3], a);
  }
  __syncthreads();
}

// Bounding box of each segment's sources, a block per tile.
__global__ void __launch_bounds__(BLOCK) bbox_kernel(Work W, const Tile *tiles, int ntiles) {
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    Seg &S = W.seg[tl.seg];
    if (threadIdx.x == 0) {
      W.tcount[t] = 0;  // node lists of the pass's moments
      if (tl.start == 0) W.ncount[NC_CROSS * W.nseg + tl.seg] = 0;
    }
    const int cnt = min(TILE, S.n_src - tl.start);
    if (cnt <= 0) continue;  // uniform
    const int64_t b = S.ibase;
    u32 mn[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, mx[3] = {0u, 0u, 0u};
    for (int i = threadIdx.x; i < cnt; i += BLOCK) {
      const int li = W.el[b + S.src_lo + tl.start + i];
      const float4 q = W.pos[b + li];
      const u32 e[3] = {f2ord(q.x), f2ord(q.y), f2ord(q.z)};
      for (int j = 0; j < 3; j++) { mn[j] = min(mn[j], e[j]); mx[j] = max(mx[j], e[j]); }
    }
    fold_box(mn, mx, S.bmin, S.bmax);
  }
}

// Root cube exactly as OctTree_t::Build (src/oct_tree.tpp:118-139) and the
// depth schedule: node length halves while >= TreeNodeResolution
// (src/gravity_tree.cpp:37-40); a node created at depth >= max(1, dlen) is
// below the resolution floor (src/oct_tree.tpp:200).
struct RootCube {
  double center[3], Len;
  int dlen, D;
  bool deep;  // D truncated at MAX_DEPTH
};

__device__ __forceinline__ RootCube root_cube(const DevParams &P, const u32 bmin[3], const u32 bmax[3]) {
#pragma clang fp contract(off)
  RootCube R;
  double xmin[3], xmax[3];
  for (int j = 0; j < 3; j++) { xmin[j] = ord2f(bmin[j]); xmax[j] = ord2f(bmax[j]); }
  double Len = xmax[0] - xmin[0];
  for (int j = 1; j < 3; j++)
    if ((xmax[j] - xmin[j]) > Len) Len = xmax[j] - xmin[j];
  for (int j = 0; j < 3; j++) R.center[j] = 0.5 * (xmax[j] + xmin[j]);
  R.Len = Len;
  int dlen = 0;
  while (dlen < 1100 && ldexp(Len, -dlen) >= (double)P.res) dlen++;
  R.dlen = dlen;
  int D = dlen < 1 ? 1 : dlen;
  R.deep = D > MAX_DEPTH;
  R.D = R.deep ? MAX_DEPTH : D;
  return R;
}

// The root cube into the segment's state, by one thread.
__device__ __forceinline__ void store_root_cube(const DevParams &P, const RootCube &R, Seg &S) {
  for (int j = 0; j < 3; j++) S.center[j] = R.center[j];
  S.Len = R.Len;
  S.dlen = R.dlen;
  if (R.deep) S.flags |= F_DEEP;
  S.D = R.D;
  // a correction pass builds its tree over the block just removed, which
  // lies inside the latest full pass's sources but not inside the previous
  // correction pass's: the latest full pass bounds the depth of later passes
  if (!(S.flags & F_CORR)) S.Dfull = R.D;
  // the FP32 walk drops the periodic wrap unless some target-source pair can
  // be more than half a box apart: a correction pass's sources (the block
  // just removed) may lie on one side of the box edge while its targets lie
  // on both, so its flag also takes the latest full pass's, whose sources
  // hold both sets
  const int st = (P.periodic && R.Len > 0.5 * (double)P.box_half) ? 1 : 0;
  if (!(S.flags & F_CORR)) S.sfull = st;
  // a shuffled list's sampled sources may span less than its targets: the
  // straddle of the whole list (prelude) bounds every pass
  S.straddle = st | S.sfull | S.sall;
}

// Octant digits of a source for depths 1..D: the reference's insertion
// descends with lenhalf *= 0.5 and centre +/- lenhalf in double and compares
// the float coordinate with strict '>' (src/oct_tree.tpp:151-184).  Digits
// are packed most significant first in bits 62..0.
__device__ __forceinline__ u64 octant_key(const double center[3], double Len, int D, float x, float y, float z) {
#pragma clang fp contract(off)
  double c0 = center[0], c1 = center[1], c2 = center[2], lh = 0.5 * Len;
  u64 key = 0;
  for (int d = 0; d < D; d++) {
    lh *= 0.5;
    int sub = 0;
    if (x > c0) { c0 += lh; sub |= 1; } else c0 -= lh;
    if (y > c1) { c1 += lh; sub |= 2; } else c1 -= lh;
    if (z > c2) { c2 += lh; sub |= 4; } else c2 -= lh;
    key = (key << 3) | (u64)sub;
  }
  return key << (3 * (MAX_DEPTH - D));
}

// Sorted runs of RUN elements (a workgroup of RUN_THREADS), a segment's merge
// levels starting there: longer than a tile, since a level reads and writes
// every element once more, but a workgroup's phases overlap only with another's.
// Digits, energies and merge levels of 200,000 subhalos' passes take 5.5 ms with
// runs of 1,024, 5.3 with 2,048 and 5.7 with 4,096 (7.2 with 1,024 sorted as keys
// with values, the energy keys by a launch of their own).
constexpr int RUN_THREADS = 512, RUN = ITEMS * RUN_THREADS;

// The runs with elements (count n(segment)) among the block's tiles
// (blockIdx.x + k gridDim.x, a multiple of RUN into their segments), checked
// RUN_THREADS at a time: an operation on a few entries per segment skips the
// others without a chain of header loads.  f(tile) for each.
template <class Count, class F>
__device__ __forceinline__ void for_runs(const Tile *__restrict__ tiles, int ntiles, Count n, F f) {
  __shared__ int live[RUN_THREADS], nlive;
  for (int tb = blockIdx.x; tb < ntiles; tb += gridDim.x * RUN_THREADS) {
    if (threadIdx.x == 0) nlive = 0;
    __syncthreads();
    const int tc = tb + (int)threadIdx.x * (int)gridDim.x;
    if (tc < ntiles && tiles[tc].start % RUN == 0 && n(tiles[tc].seg) > tiles[tc].start) live[atomicAdd(&nlive, 1)] = tc;
    __syncthreads();
    const int m = nlive;
    for (int i = 0; i < m; i++) f(tiles[live[i]]);
    __syncthreads();
  }
}

// A run's digits, sorted, into the buffer from which the merge levels end in
// (k0, v0); the root cube from the box, into the segment's state by its first
// run.  In one kernel the keys reach memory sorted: digits and sort in kernels
// of their own wrote and read 12 bytes per source in between.
__global__ void __launch_bounds__(RUN_THREADS, 8) keys_sort_kernel(Work W, DevParams P, const Tile *__restrict__ tiles,
                                                                   int ntiles, bool ranked) {
  __shared__ u64 sk[RUN];
  __shared__ u32 sv[RUN];
  __shared__ RootCube cube;
  for_runs(tiles, ntiles, [&](int k) { return W.ncount[NC_SRC * W.nseg + k]; }, [&](const Tile &tl) {
    Seg &S = W.seg[tl.seg];
    const int n = S.n_src;
    const int cnt = min(RUN, n - tl.start);
    if (threadIdx.x == 0) {
      cube = root_cube(P, S.bmin, S.bmax);
      if (tl.start == 0) store_root_cube(P, cube, S);
    }
    const int64_t off = S.ibase + tl.start;
    u32 v[ITEMS];
    float4 q[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int e = ITEMS * (int)threadIdx.x + r;
      v[r] = e < cnt ? (u32)W.el[off + S.src_lo + e] : ~0u;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; r++)
      if (v[r] != ~0u) q[r] = W.pos[S.ibase + v[r]];
    __syncthreads();
    u64 k[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++)
      k[r] = v[r] != ~0u ? octant_key(cube.center, cube.Len, cube.D, q[r].x, q[r].y, q[r].z) : ~0ull;
    sort_tile_spare<RUN_THREADS>(k, v, cnt, 3 * (MAX_DEPTH - cube.D), sk, sv);
    const bool odd = (merge_levels(n, RUN, ranked) & 1) != 0;
    u64 *kout = odd ? W.k1 : W.k0;
    u32 *vout = odd ? W.v1 : W.v0;
    for (int i = threadIdx.x; i < cnt; i += RUN_THREADS) {
      kout[off + i] = sk[i];
      vout[off + i] = sv[i];
      W.bits[off + i] = 0u;  // node-start masks, set by emit_kernel
    }
    __syncthreads();
  });
}

// ---------------------------------------------------------------------------
// Structure from sorted keys.  Pair l joins sorted sources l and l+1;
// delta = number of leading digits they share (D when the keys are equal: the
// two are in one cell at the depth of the resolution floor).  A node of the
// compressed octree is a maximal run of sources whose pairs all have
// delta >= v, split by pairs with delta == v; it sits at depth v.

__device__ __forceinline__ int key_delta(u64 a, u64 b, int D) {
  if (a == b) return D;
  int d = (__clzll((long long)(a ^ b)) - 1) / 3;
  return d < D ? d : D;
}

// First v octant digits of a key (digit 0 in bits 62..60).
__device__ __forceinline__ u64 key_prefix(u64 k, int v) { return v == 0 ? 0ull : k >> (63 - 3 * v); }

// First index in [lo, hi+1] whose v-digit prefix is >= p (keys ascending).
__device__ __forceinline__ int prefix_lower(const u64 *key, int lo, int hi, int v, u64 p) {
  while (lo <= hi) {
    const int m = (lo + hi) >> 1;
    if (key_prefix(key[m], v) < p) lo = m + 1;
    else hi = m - 1;
  }
  return lo;
}

// Keys 0 .. n-1 at sk: sk(i), and the first index in [a, h + 1] whose v-digit
// prefix is >= p.
struct KeyAll {
  const u64 *sk;
  __device__ __forceinline__ u64 at(int i) const { return sk[i]; }
  __device__ __forceinline__ int lower(int a, int h, int v, u64 p) const { return prefix_lower(sk, a, h, v, p); }
};

// The node whose leftmost split is pair l of n sources: sources lo..hi at
// depth v; false if l is no node's leftmost split.  v: the pair's delta (-1:
// l is the last source).
template <class Keys>
__device__ __forceinline__ bool node_of_pair(const Keys &K, int l, int n, int D, int &lo, int &hi, int &v) {
  v = (l + 1 < n) ? key_delta(K.at(l), K.at(l + 1), D) : -1;
  if (v < 0) return false;
  const int vl = l > 0 ? key_delta(K.at(l - 1), K.at(l), D) : -1;
  if (vl == v) return false;  // source l-1 is in the node, in another child
  const int vr = l + 2 < n ? key_delta(K.at(l + 1), K.at(l + 2), D) : -1;
  const u64 p = key_prefix(K.at(l), v);
  lo = l;
  hi = l + 1;
  if (vl > v) {
    lo = K.lower(0, l - 1, v, p);
    // leftmost split iff sources lo and l are in the same child
    if (key_delta(K.at(lo), K.at(l), D) <= v) return false;
  }
  if (vr >= v) hi = K.lower(l + 2, n - 1, v, p + 1) - 1;
  return true;
}

// A tile's keys and those around them, w_lo .. w_hi of the segment's n, in LDS;
// every pair of the tile has its neighbours' keys there.  `inside` is cleared by
// a search whose answer lies beyond the window.
struct KeyWin {
  const u64 *sk;
  int w_lo, w_hi, n;
  mutable bool inside = true;
  __device__ __forceinline__ u64 at(int i) const { return sk[max(i, w_lo) - w_lo]; }
  __device__ __forceinline__ int lower(int a, int h, int v, u64 p) const {
    const int wa = max(a, w_lo), wh = min(h, w_hi);
    const int i = prefix_lower(sk, wa - w_lo, wh - w_lo, v, p) + w_lo;
    if ((i == wa && wa > a) || (i > wh && wh < h)) inside = false;
    return i;
  }
};

// A pair's node that reaches beyond the window: both of its ends searched
// together in device memory, where one step waits on the other.
__device__ __forceinline__ bool node_of_pair_far(const u64 *sk, int w_lo, int w_hi, const u64 *key, int l, int n,
                                                 int D, int &lo, int &hi) {
  auto win = [&](int i) { return sk[i - w_lo]; };
  const u64 kl = win(l);
  const int v = key_delta(kl, win(l + 1), D);
  const int vl = l > 0 ? key_delta(win(l - 1), kl, D) : -1;
  const int vr = l + 2 < n ? key_delta(win(l + 1), win(l + 2), D) : -1;
  const u64 p = key_prefix(kl, v);
  // first source of [a0, a1 + 1] with prefix p, first of [b0, b1 + 1] beyond it
  int a0 = l, a1 = l - 1, b0 = l + 2, b1 = l + 1;
  if (vl > v) {
    if (w_lo == 0 || key_prefix(win(w_lo), v) < p) { a0 = prefix_lower(sk, 0, l - 1 - w_lo, v, p) + w_lo; a1 = a0 - 1; }
    else { a0 = 0; a1 = w_lo - 1; }
  }
  if (vr >= v) {
    if (w_hi == n - 1 || key_prefix(win(w_hi), v) > p) { b0 = prefix_lower(sk, l + 2 - w_lo, w_hi - w_lo, v, p + 1) + w_lo; b1 = b0 - 1; }
    else { b0 = w_hi + 1; b1 = n - 1; }
  }
  while (a0 <= a1 || b0 <= b1) {
    const int ma = (a0 + a1) >> 1, mb = (b0 + b1) >> 1;
    const u64 xa = a0 <= a1 ? key[ma] : 0ull, xb = b0 <= b1 ? key[mb] : 0ull;
    if (a0 <= a1) { if (key_prefix(xa, v) < p) a0 = ma + 1; else a1 = ma - 1; }
    if (b0 <= b1) { if (key_prefix(xb, v) < p + 1) b0 = mb + 1; else b1 = mb - 1; }
  }
  lo = a0;
  hi = vr >= v ? b0 - 1 : l + 1;
  return !(vl > v) || key_delta(lo >= w_lo ? win(lo) : key[lo], kl, D) > v;
}

// Per pair l of sorted sources: its delta, and the node of which it is the
// leftmost split.  In a full pass the sorted order also becomes the spatial
// target order.  A tile's keys are in LDS (window t0 - 1 .. t0 + TILE + 1), so
// the searches for a node's ends run there; the pairs whose nodes reach beyond
// it, a few per depth, are listed and searched together at the end: among the
// others, each of a thread's four pairs could wait on two chains of loads: one
// list of 24,000 took 25 us (19 now), 200,000 subhalos' passes 1.27 ms (0.94).
__global__ void __launch_bounds__(BLOCK) emit_kernel(Work W, const Tile *__restrict__ tiles, int ntiles,
                                                     int full_copy_sp) {
  __shared__ u64 sk[TILE + 3];
  __shared__ unsigned short far[TILE];
  __shared__ int nfar;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    const int n = S.n_src;
    const int cnt = min(TILE, n - tl.start);
    if (cnt <= 0) continue;  // uniform across the block
    const int64_t b = S.ibase;
    const bool copy_sp = full_copy_sp && !(S.flags & (F_CORR | F_SAMP | F_REFINE));
    const int D = S.D, w_lo = tl.start > 0 ? tl.start - 1 : 0, w_hi = min(n - 1, tl.start + TILE + 1);
    const u64 *key = W.k0 + b;
    for (int i = w_lo + (int)threadIdx.x; i <= w_hi; i += BLOCK) sk[i - w_lo] = key[i];
    if (threadIdx.x == 0) nfar = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < cnt; i += BLOCK) {
      const int l = tl.start + i;
      const int64_t s = b + l;
      if (copy_sp) W.sp[s] = (int)W.v0[s];
      KeyWin K{sk, w_lo, w_hi, n};
      int lo, hi, v;
      const bool node = node_of_pair(K, l, n, D, lo, hi, v);
      W.dl[s] = (signed char)v;
      if (!K.inside) {
        far[atomicAdd(&nfar, 1)] = (unsigned short)i;
        continue;
      }
      W.nlo[s] = node ? lo : -1;
      if (node) {
        W.nhi[s] = hi;
        atomicOr(&W.bits[b + lo], 1u << v);
      }
    }
    __syncthreads();
    for (int f = threadIdx.x; f < nfar; f += BLOCK) {
      const int l = tl.start + far[f];
      int lo, hi;
      const bool node = node_of_pair_far(sk, w_lo, w_hi, key, l, n, D, lo, hi);
      W.nlo[b + l] = node ? lo : -1;
      if (node) {
        W.nhi[b + l] = hi;
        atomicOr(&W.bits[b + lo], 1u << key_delta(sk[l - w_lo], sk[l + 1 - w_lo], D));
      }
    }
    __syncthreads();  // the next tile restages sk
  }
}

// Node length at depth v: Len halved while >= resolution, stored as float.
__device__ __forceinline__ float node_len(double Len, int dlen, int v) {
  const int e = v < dlen ? v : dlen;
  return (float)ldexp(Len, -e);
}

// The squared distance below which the FP32 walk opens a node: the smallest
// float r2 for which lsq > r2 * theta2 (rounded to float) fails, so that
// r2 < open_below(lsq, theta2) is that test for every r2 >= 0 (the product is
// monotonic in r2).  The quotient is off by a step or two; where the product
// is subnormal a plateau can be longer, and the bits are bisected.
__device__ __forceinline__ float open_below(float lsq, float theta2) {
#pragma clang fp contract(off)
  if (!(lsq > 0.f)) return 0.f;
  auto opens = [&](u32 bits) { return lsq > __uint_as_float(bits) * theta2; };
  const float t0 = lsq / theta2;
  if (!(t0 >= 0.f)) return 0.f;  // theta2 is NaN: nothing opens
  u32 t = __float_as_uint(t0);
  for (int i = 0; i < 3 && t < 0x7f800000u && opens(t); i++) t++;
  for (int i = 0; i < 3 && t > 0u && !opens(t - 1u); i++) t--;
  const bool low = t < 0x7f800000u && opens(t), high = t > 0u && !opens(t - 1u);
  if (low || high) {
    u32 a = 0u, b = 0x7f800000u;  // the answer lies in [a, b]
    while (a < b) {
      const u32 m = (a + b) >> 1;
      if (opens(m)) a = m + 1u; else b = m;
    }
    t = a;
  }
  return __uint_as_float(t);
}

// The opening lengths of a tree's depths, filled by the first NLEVEL threads.
struct DepthTable {
  float lsq[NLEVEL], below[NLEVEL];
  __device__ __forceinline__ void fill(int v, double Len, int dlen, float theta2) {
    if (v < NLEVEL) {
      const float len = node_len(Len, dlen, v);
      lsq[v] = len * len;
      below[v] = open_below(lsq[v], theta2);
    }
  }
};

// (not read in trees that are too large for it)
__device__ __forceinline__ int byte_offset(int item) { return (int)((u32)sizeof(Item) * (u32)item); }
__device__ __forceinline__ Item leaf_item(const float4 &pm, int pos) {
  return Item{pm, make_int2(0, pos + 1), make_int2(byte_offset(pos + 1), 0)};
}
__device__ __forceinline__ Item node_item(const float4 &pm, int skip, float lsq, float below) {
  return Item{pm, make_int2(__float_as_int(lsq), skip), make_int2(byte_offset(skip), __float_as_int(below))};
}
// Sentinel after the last item: massless, far from every target, never
// opened, its skip is itself, so a group walk that has finished reads it, adds
// nothing and stays put.
__device__ __forceinline__ Item sentinel_item(int pos) {
  return Item{make_float4(1e18f, 1e18f, 1e18f, 0.f), make_int2(0, pos), make_int2(byte_offset(pos), 0)};
}

// A leaf: a sampled tree's leaves carry mass * MassFactor (EnergySnapshot_t::GetMass, :79).
__device__ __forceinline__ float4 leaf_pm(const Work &W, const Seg &S, int li) {
  float4 q = W.pos[S.ibase + li];
  if (S.flags & F_SAMP) q.w = q.w * S.mf;
  return q;
}

// Node moments: mass and centre of mass accumulated in double over the float
// values of the children in son order, stored as float
// (UpdateInternalNodes/ProcessNode/FillNodeCenter, src/gravity_tree.cpp:18-77).
// pm(i) and skip(i) read item i; g is the node, end its skip.
template <class Pm, class Skip>
__device__ __forceinline__ float4 sum_children(Pm pm, Skip skip, int g, int end) {
#pragma clang fp contract(off)
  double mass = 0., cx = 0., cy = 0., cz = 0.;
  int c = g + 1;
  while (c < end) {
    const float4 q = pm(c);
    const double m = q.w;
    mass += m;
    cx += (double)q.x * m;
    cy += (double)q.y * m;
    cz += (double)q.z * m;
    const int nx = skip(c);
    c = nx > c ? nx : end;  // skips always advance
  }
  return make_float4((float)(cx / mass), (float)(cy / mass), (float)(cz / mass), (float)mass);
}

// The same over a segment's items in device memory (positions and skips are
// segment-local: a level's items may number more than 2^31).
__device__ __forceinline__ void node_moments(Item *it, int g) {
  it[g].pm = sum_children([&](int c) { return it[c].pm; }, [&](int c) { return it[c].ax.y; }, g, it[g].ax.y);
}

// A team: the threads that build one tile's tree (one wave, or the workgroup),
// R elements each.
template <int T_, int R_>
struct Team {
  static constexpr int T = T_, R = R_, CAP = T_ * R_;
  static_assert(T_ == WAVE || T_ == BLOCK, "a wave or a workgroup");
  static __device__ __forceinline__ int id() { return T == WAVE ? threadIdx.x & (WAVE - 1) : threadIdx.x; }
  static __device__ __forceinline__ void sync() {
    if (T == WAVE) wave_sync();
    else __syncthreads();
  }
  template <class X>
  static __device__ __forceinline__ X exclusive_scan(X x, X *total) {
    if (T == BLOCK) return block_exclusive_scan(x, total);
    const X inc = wave_inclusive_scan(x);
    *total = __shfl(inc, WAVE - 1, WAVE);
    return inc - x;
  }
};

// The nodes whose leaves all lie in the tile, computed deepest first: depth
// counts and places, and the LDS items they work on.
template <int NI, int NN>
struct TileNodes {
  float4 pm[NI];
  unsigned short skip[NI];
  unsigned short node[NN];       // nodes (item index) grouped by depth, deepest first
  int count[NLEVEL], first[NLEVEL + 1];
};

// Fills in the moments of a tile's nodes.  at[r] < 0: no node in thread's slot
// r; otherwise its LDS item and its depth v[r] (headers' skips and every leaf
// are in place).  Called by the whole team; leaves the team synchronised.
template <class TM, int R, int NI, int NN>
__device__ __forceinline__ void tile_moments(TileNodes<NI, NN> &N, const int (&at)[R], const int (&v)[R]) {
  for (int d = TM::id(); d < NLEVEL; d += TM::T) N.count[d] = 0;
  TM::sync();
  int rank[R];
#pragma unroll
  for (int r = 0; r < R; r++)
    if (at[r] >= 0) rank[r] = atomicAdd(&N.count[v[r]], 1);
  TM::sync();
  if (TM::id() == 0) {
    int o = 0;
    for (int d = MAX_DEPTH; d >= 0; d--) { N.first[d] = o; o += N.count[d]; }
    N.first[NLEVEL] = o;
  }
  TM::sync();
#pragma unroll
  for (int r = 0; r < R; r++)
    if (at[r] >= 0) N.node[N.first[v[r]] + rank[r]] = (unsigned short)at[r];
  TM::sync();
  for (int d = MAX_DEPTH; d >= 0; d--) {
    const int p0 = N.first[d], p1 = d > 0 ? N.first[d - 1] : N.first[NLEVEL];
    if (p0 == p1) continue;  // uniform
    for (int p = p0 + TM::id(); p < p1; p += TM::T) {
      const int g = N.node[p];
      N.pm[g] = sum_children([&](int c) { return N.pm[c]; }, [&](int c) { return (int)N.skip[c]; }, g, N.skip[g]);
    }
    TM::sync();
  }
}

// LDS of a one-tile tree: the sorted keys with what places the items, then, in
// the same memory, the items.
template <int CAP>
struct OneTile {
  union {
    struct {
      u64 key[CAP];
      u32 val[CAP];
      u32 bits[CAP];
      unsigned short pre[CAP];
    } s;
    TileNodes<2 * CAP, CAP> n;
  };
  DepthTable depth;
  u32 box[6][BLOCK / WAVE];
};

// The whole tree of a segment of at most CAP sources: box, root cube, digits,
// sort, nodes, pre-order positions, items and moments, between one read of the
// sources and one write of the items.  A chain of LDS steps bounds it: a tree of
// 300 alone takes 19 us, in launches of their own, each waiting on its chain of
// loads per source, the stages took 36 and their gaps.  LDS (40 KB) and registers
// (held to 128) each let four waves run per SIMD.
template <class TM>
__device__ __forceinline__ void tree_one(const Work &W, const DevParams &P, const Tile &tl, int full_copy_sp,
                                         OneTile<TM::CAP> &L) {
  constexpr int R = TM::R, CAP = TM::CAP;
  Seg &S = W.seg[tl.seg];
  const int n = min(CAP, S.n_src);
  if (n <= 0) return;  // uniform across the team
  const int64_t b = S.ibase;
  const int id = TM::id();
  u32 v[R];
  float4 q[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int e = R * id + r;
    v[r] = e < n ? (u32)W.el[b + S.src_lo + e] : ~0u;
  }
  u32 mn[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, mx[3] = {0u, 0u, 0u};
#pragma unroll
  for (int r = 0; r < R; r++)
    if (v[r] != ~0u) {
      q[r] = W.pos[b + v[r]];
      const u32 o[3] = {f2ord(q[r].x), f2ord(q[r].y), f2ord(q[r].z)};
      for (int j = 0; j < 3; j++) { mn[j] = min(mn[j], o[j]); mx[j] = max(mx[j], o[j]); }
    }
  for (int d = WAVE / 2; d > 0; d >>= 1)
    for (int j = 0; j < 3; j++) {
      mn[j] = min(mn[j], (u32)__shfl_xor((int)mn[j], d, WAVE));
      mx[j] = max(mx[j], (u32)__shfl_xor((int)mx[j], d, WAVE));
    }
  if (TM::T > WAVE) {
    if ((threadIdx.x & (WAVE - 1)) == 0)
      for (int j = 0; j < 3; j++) { L.box[j][threadIdx.x / WAVE] = mn[j]; L.box[3 + j][threadIdx.x / WAVE] = mx[j]; }
    TM::sync();
    for (int w = 0; w < TM::T / WAVE; w++)
      for (int j = 0; j < 3; j++) { mn[j] = min(mn[j], L.box[j][w]); mx[j] = max(mx[j], L.box[3 + j][w]); }
  }
  const RootCube cube = root_cube(P, mn, mx);
  L.depth.fill(id, cube.Len, cube.dlen, P.theta2);
  const bool copy_sp = full_copy_sp && !(S.flags & (F_CORR | F_SAMP | F_REFINE));
  u64 k[R];
#pragma unroll
  for (int r = 0; r < R; r++)
    k[r] = v[r] != ~0u ? octant_key(cube.center, cube.Len, cube.D, q[r].x, q[r].y, q[r].z) : ~0ull;
  const int spare = 3 * (MAX_DEPTH - cube.D);
  if constexpr (TM::T == WAVE) sort_wave_spare<R>(k, v, id, n, spare, L.s.key, L.s.val);
  else sort_tile_spare<TM::T>(k, v, n, spare, L.s.key, L.s.val);
#pragma unroll
  for (int r = 0; r < R; r++) L.s.bits[id + r * TM::T] = 0u;
  TM::sync();
  // nodes, by their leftmost split
  int lo[R], hi[R], dv[R], at[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int l = id + r * TM::T;
    at[r] = -1;
    if (l < n && node_of_pair(KeyAll{L.s.key}, l, n, cube.D, lo[r], hi[r], dv[r])) {
      at[r] = 0;
      atomicOr(&L.s.bits[lo[r]], 1u << dv[r]);
    }
  }
  TM::sync();
  // pre-order: the nodes that start before each source
  int own = 0, nodes;
#pragma unroll
  for (int r = 0; r < R; r++) own += __popc(L.s.bits[R * id + r]);
  int run = TM::exclusive_scan(own, &nodes);
#pragma unroll
  for (int r = 0; r < R; r++) {
    L.s.pre[R * id + r] = (unsigned short)run;
    run += __popc(L.s.bits[R * id + r]);
  }
  TM::sync();
  int leaf[R], nskip[R];
  float4 pm[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int l = id + r * TM::T;
    leaf[r] = -1;
    if (l < n) {
      const int li = (int)L.s.val[l];
      if (copy_sp) W.sp[b + l] = li;
      leaf[r] = l + L.s.pre[l] + __popc(L.s.bits[l]);
      pm[r] = leaf_pm(W, S, li);
    }
    if (at[r] >= 0) {
      at[r] = lo[r] + L.s.pre[lo[r]] + __popc(L.s.bits[lo[r]] & ((1u << dv[r]) - 1u));
      nskip[r] = hi[r] + L.s.pre[hi[r]] + __popc(L.s.bits[hi[r]]) + 1;
    }
  }
  TM::sync();  // the items take the keys' place
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (leaf[r] >= 0) {
      L.n.pm[leaf[r]] = pm[r];
      L.n.skip[leaf[r]] = (unsigned short)(leaf[r] + 1);
    }
    if (at[r] >= 0) L.n.skip[at[r]] = (unsigned short)nskip[r];
  }
  tile_moments<TM>(L.n, at, dv);
  Item *out = W.items + 2 * b;
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (leaf[r] >= 0) out[leaf[r]] = leaf_item(pm[r], leaf[r]);
    if (at[r] >= 0) out[at[r]] = node_item(L.n.pm[at[r]], nskip[r], L.depth.lsq[dv[r]], L.depth.below[dv[r]]);
  }
  if (id == 0) {
    const int ni = n + nodes;
    out[ni] = sentinel_item(ni);
    store_root_cube(P, cube, S);
    S.n_items = ni;
  }
  TM::sync();  // the next tile reuses the LDS
}

// Tiles t0 <= t < ntiles, one team each.
template <int R>
__global__ void __launch_bounds__(BLOCK, 4) tree_one_wave_kernel(Work W, DevParams P, const Tile *__restrict__ tiles,
                                                              int t0, int ntiles, int full_copy_sp) {
  using TM = Team<WAVE, R>;
  __shared__ OneTile<TM::CAP> L[BLOCK / WAVE];
  WAVE_TILE_LOOP(t, t0, ntiles) tree_one<TM>(W, P, tiles[t], full_copy_sp, L[threadIdx.x / WAVE]);
}
__global__ void __launch_bounds__(BLOCK, 4) tree_one_kernel(Work W, DevParams P, const Tile *__restrict__ tiles, int t0,
                                                         int ntiles, int full_copy_sp) {
  using TM = Team<BLOCK, ITEMS>;
  __shared__ OneTile<TM::CAP> L;
  for (int t = t0 + (int)blockIdx.x; t < ntiles; t += gridDim.x) tree_one<TM>(W, P, tiles[t], full_copy_sp, L);
}

// items_tile_kernel: one workgroup per tile places
// the tile's leaves and the nodes whose leaves all lie in it in LDS (leaves plus
// the headers of the nodes whose leftmost leaf it holds: fewer than 2 TILE +
// MAX_DEPTH), computes those nodes deepest first (their children are there too)
// and writes both out; of the nodes whose leaves cross a tile edge (at most one
// per depth per edge) it writes the header and lists the pair: in W.cross, by
// super-tile (SUPER_TILES tiles), when the node lies in one, else in W.cross2 by
// segment.  moments_super_kernel: one workgroup per super-tile computes its
// listed nodes, deepest first; moments_cross_kernel (only for segments of more
// than one super-tile): one workgroup per segment computes the rest, deepest
// first.  A node's children are inside a tile (done by the first launch) or
// listed at the same or a lower level and deeper.  Each node sums its children
// in son order (sum_children), so the results do not depend on which launch
// computes a node.  With the items placed in LDS they reach memory once and
// finished, 32 bytes each; placed by a launch of its own and staged again for
// the moments they were written, read and half written again (200,000 subhalos:
// 5.2 ms with the smaller segments', 2.0 now).
constexpr int TILE_ITEMS = 2 * TILE + MAX_DEPTH + 2;
constexpr int SUPER_TILES = 64;
constexpr int SUPER = SUPER_TILES * TILE;

// Lists the pair l (in tile t) of a node with leaves lo..hi that crosses a tile edge.
__device__ __forceinline__ void list_crossing(const Work &W, int t, const Tile &tl, int64_t b, int l, int lo,
                                              int hi, int *ncross) {
  if (lo / SUPER == hi / SUPER) {
    const int st = tl.start / SUPER * SUPER;  // first leaf of the super-tile
    const int ts = t - (tl.start - st) / TILE;  // its first tile in the table
    W.cross[b + st + atomicAdd(&W.tcount[ts], 1)] = l;
  } else {
    W.cross2[b + atomicAdd(ncross, 1)] = l;
  }
}

// pre = exclusive prefix of popcount(bits) over the segment's sorted sources.
__global__ void __launch_bounds__(BLOCK, 4) items_tile_kernel(Work W, DevParams P, const Tile *__restrict__ tiles,
                                                           int ntiles) {
  using TM = Team<BLOCK, ITEMS>;
  struct Place { u32 bits[TILE]; int pre[TILE]; };
  __shared__ union { Place p; TileNodes<TILE_ITEMS, TILE> n; } L;
  __shared__ DepthTable depth;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    const int n = S.n_src;
    const int nl = min(TILE, n - tl.start);
    if (nl <= 0) continue;  // uniform across the block
    const int64_t b = S.ibase, ib = 2 * b, s0 = b + tl.start;
    const int t_lo = tl.start, t_hi = tl.start + TILE - 1;
    depth.fill(threadIdx.x, S.Len, S.dlen, P.theta2);
    // one batch of loads per thread: four neighbouring sources and pairs
    // (4-aligned slots inside the segment's wave-aligned slots)
    static_assert(ITEMS == 4, "sources are loaded four at a time");
    const int p0 = ITEMS * (int)threadIdx.x;
    int plo[ITEMS], phi[ITEMS], pdl[ITEMS], li[ITEMS], pre[ITEMS];
    u32 bits[ITEMS];
    if (p0 < nl) {
      const int4 a = *reinterpret_cast<const int4 *>(W.nlo + s0 + p0);
      const int4 h = *reinterpret_cast<const int4 *>(W.nhi + s0 + p0);
      const int4 x = *reinterpret_cast<const int4 *>(W.v0 + s0 + p0);
      const int4 e = *reinterpret_cast<const int4 *>(W.pre + s0 + p0);
      const int4 m = *reinterpret_cast<const int4 *>(W.bits + s0 + p0);
      const char4 d = *reinterpret_cast<const char4 *>(W.dl + s0 + p0);
      plo[0] = a.x; plo[1] = a.y; plo[2] = a.z; plo[3] = a.w;
      phi[0] = h.x; phi[1] = h.y; phi[2] = h.z; phi[3] = h.w;
      li[0] = x.x; li[1] = x.y; li[2] = x.z; li[3] = x.w;
      pre[0] = e.x; pre[1] = e.y; pre[2] = e.z; pre[3] = e.w;
      bits[0] = (u32)m.x; bits[1] = (u32)m.y; bits[2] = (u32)m.z; bits[3] = (u32)m.w;
      pdl[0] = d.x; pdl[1] = d.y; pdl[2] = d.z; pdl[3] = d.w;
    }
    float4 pm[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
      if (p0 + j < nl) {
        pm[j] = leaf_pm(W, S, li[j]);
        L.p.bits[p0 + j] = bits[j];
        L.p.pre[p0 + j] = pre[j];
      } else {
        plo[j] = -1;
      }
    }
    __syncthreads();
    const int first = t_lo + L.p.pre[0];  // the tile's first item
    int *ncross = W.ncount + NC_CROSS * W.nseg + tl.seg;
    int leaf[ITEMS], at[ITEMS], nskip[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
      const int l = t_lo + p0 + j;
      leaf[j] = p0 + j < nl ? l + pre[j] + __popc(bits[j]) : -1;
      at[j] = -1;
      if (plo[j] < 0) continue;
      const bool lo_in = plo[j] >= t_lo, hi_in = phi[j] <= t_hi;
      const u32 blo = lo_in ? L.p.bits[plo[j] - t_lo] : W.bits[b + plo[j]];
      const int elo = lo_in ? L.p.pre[plo[j] - t_lo] : W.pre[b + plo[j]];
      const u32 bhi = hi_in ? L.p.bits[phi[j] - t_lo] : W.bits[b + phi[j]];
      const int ehi = hi_in ? L.p.pre[phi[j] - t_lo] : W.pre[b + phi[j]];
      const int pos = plo[j] + elo + __popc(blo & ((1u << pdl[j]) - 1u));
      nskip[j] = phi[j] + ehi + __popc(bhi) + 1;
      if (lo_in && hi_in) {
        at[j] = pos - first;
      } else {
        W.items[ib + pos] = node_item(make_float4(0.f, 0.f, 0.f, 0.f), nskip[j], depth.lsq[pdl[j]], depth.below[pdl[j]]);
        W.npos[b + l] = pos;
        list_crossing(W, t, tl, b, l, plo[j], phi[j], ncross);
      }
    }
    __syncthreads();  // the items take the places' memory
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
      if (leaf[j] >= 0) {
        L.n.pm[leaf[j] - first] = pm[j];
        L.n.skip[leaf[j] - first] = (unsigned short)(leaf[j] + 1 - first);
      }
      if (at[j] >= 0) L.n.skip[at[j]] = (unsigned short)(nskip[j] - first);
    }
    tile_moments<TM>(L.n, at, pdl);
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
      if (leaf[j] >= 0) {
        W.items[ib + leaf[j]] = leaf_item(pm[j], leaf[j]);
        if (t_lo + p0 + j + 1 == n) {
          W.seg[tl.seg].n_items = leaf[j] + 1;
          W.items[ib + leaf[j] + 1] = sentinel_item(leaf[j] + 1);
        }
      }
      if (at[j] >= 0)
        W.items[ib + first + at[j]] = node_item(L.n.pm[at[j]], nskip[j], depth.lsq[pdl[j]], depth.below[pdl[j]]);
    }
    __syncthreads();
  }
}

// The nodes of a list (pairs at list[0..ng)) of segment S, deepest first.  Where
// the list fits in LDS its nodes are grouped by depth and their children's places
// found for all of them at once: one after another down the skips, child after
// child and depth after depth, the loads of a list's nodes were a chain that took
// 24 us for one list of 24,000 (14 now).
constexpr int LISTED = 1024, SONS = 8;  // nodes, children of a node (more only where digits are equal)
struct ListNodes {
  int son[SONS][LISTED];
  unsigned short node[LISTED];  // grouped by depth, deepest first
  unsigned char sons[LISTED];
  int count[NLEVEL], first[NLEVEL + 1];
};

__device__ __forceinline__ void moments_of_list(const Work &W, const Seg &S, const int *list, int ng, ListNodes &L) {
#pragma clang fp contract(off)
  const int64_t b = S.ibase;
  Item *it = W.items + 2 * b;
  if (ng > LISTED) {
    for (int v = min(max(S.D, S.Dfull), MAX_DEPTH); v >= 0; v--) {
      for (int i = threadIdx.x; i < ng; i += BLOCK) {
        const int64_t s = b + list[i];
        if (W.dl[s] == v) node_moments(it, W.npos[s]);
      }
      __syncthreads();
    }
    return;
  }
  constexpr int PER = LISTED / BLOCK;
  for (int d = threadIdx.x; d < NLEVEL; d += BLOCK) L.count[d] = 0;
  __syncthreads();
  int pos[PER], depth[PER], rank[PER];
#pragma unroll
  for (int r = 0; r < PER; r++) {
    const int i = (int)threadIdx.x + BLOCK * r;
    if (i >= ng) continue;
    const int64_t s = b + list[i];
    pos[r] = W.npos[s];
    depth[r] = W.dl[s];
    rank[r] = atomicAdd(&L.count[depth[r]], 1);
    const int end = it[pos[r]].ax.y;
    int c = pos[r] + 1, k = 0;
    for (; c < end && k < SONS; k++) {
      L.son[k][i] = c;
      const int nx = it[c].ax.y;
      c = nx > c ? nx : end;  // skips always advance
    }
    L.sons[i] = (unsigned char)(c < end ? SONS + 1 : k);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int o = 0;
    for (int d = MAX_DEPTH; d >= 0; d--) { L.first[d] = o; o += L.count[d]; }
    L.first[NLEVEL] = o;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < PER; r++) {
    const int i = (int)threadIdx.x + BLOCK * r;
    if (i < ng) L.node[L.first[depth[r]] + rank[r]] = (unsigned short)i;
  }
  __syncthreads();
  for (int d = MAX_DEPTH; d >= 0; d--) {
    const int p0 = L.first[d], p1 = d > 0 ? L.first[d - 1] : L.first[NLEVEL];
    if (p0 == p1) continue;  // uniform
    for (int p = p0 + (int)threadIdx.x; p < p1; p += BLOCK) {
      const int i = L.node[p], n = L.sons[i], g = L.son[0][i] - 1;
      if (n > SONS) {
        node_moments(it, g);
        continue;
      }
      float4 q[SONS];
#pragma unroll
      for (int k = 0; k < SONS; k++) q[k] = it[L.son[k < n ? k : 0][i]].pm;
      double mass = 0., cx = 0., cy = 0., cz = 0.;  // as sum_children
#pragma unroll
      for (int k = 0; k < SONS; k++)
        if (k < n) {
          const double m = q[k].w;
          mass += m;
          cx += (double)q[k].x * m;
          cy += (double)q[k].y * m;
          cz += (double)q[k].z * m;
        }
      it[g].pm = make_float4((float)(cx / mass), (float)(cy / mass), (float)(cz / mass), (float)mass);
    }
    __syncthreads();
  }
}

__global__ void __launch_bounds__(BLOCK) moments_super_kernel(Work W, const Tile *__restrict__ tiles, int ntiles) {
  __shared__ ListNodes L;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    if (tl.start % SUPER != 0) continue;  // a super-tile's first tile stands for it
    const int ng = W.tcount[t];
    if (ng == 0) continue;  // uniform
    const Seg &S = W.seg[tl.seg];
    moments_of_list(W, S, W.cross + S.ibase + tl.start, ng, L);
  }
}

__global__ void __launch_bounds__(BLOCK) moments_cross_kernel(Work W, const Tile *__restrict__ tiles, int ntiles) {
  __shared__ ListNodes L;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    if (tl.start != 0) continue;  // the segment's first tile stands for it
    const int ng = W.ncount[NC_CROSS * W.nseg + tl.seg];
    if (ng == 0) continue;  // uniform
    const Seg &S = W.seg[tl.seg];
    moments_of_list(W, S, W.cross2 + S.ibase, ng, L);
  }
}

// ---------------------------------------------------------------------------
// Walk.  Pre-order items: an internal node is opened when
// len^2 > r^2 * theta^2 (then the next item is its first child), otherwise its
// monopole is used and the walk continues at its skip pointer; a leaf has
// len^2 = 0 and skip = next item.

// Reference arithmetic (src/gravity_tree.cpp:79-164): FP64 walk over float data.
template <bool COUNT>
__device__ double walk_replay(const Item *it, const DevParams &P, int end, float tx, float ty, float tz, float tmass,
                              unsigned &ni, unsigned &no) {
#pragma clang fp contract(off)
  const double h = 2.8 * (double)P.eps, hinv = 1.0 / h;
  double pot = (double)(float)(tmass / P.eps);
  const double x = tx, y = ty, z = tz;
  int j = 0;
  while (j < end) {
    const float4 q = it[j].pm;
    const int2 a = it[j].ax;
    double dx = (double)q.x - x, dy = (double)q.y - y, dz = (double)q.z - z;
    if (P.periodic) { dx = nearest_d(dx, P); dy = nearest_d(dy, P); dz = nearest_d(dz, P); }
    const double r2 = dx * dx + dy * dy + dz * dz;
    const float lsq = __int_as_float(a.x);
    if ((double)lsq > r2 * (double)P.theta2) { j++; if (COUNT) no++; continue; }
    j = a.y > j ? a.y : end;  // skips always advance
    if (COUNT) ni++;
    pot += kernel_term_d((double)q.w, sqrt(r2), h, hinv);
  }
  return pot * (double)P.G / (double)P.a;
}

// FP32 walk, the terms summed in FP64 (or in FP32 when !P.wide_sum), as the
// group walk's FastTerm sums them.  Straddling segments (a periodic subhalo
// wider than a quarter box) form the separation in double.
template <bool STRADDLE, bool COUNT>
__device__ double walk_fast(const Item *it, const DevParams &P, int end, float tx, float ty, float tz, float tmass,
                            unsigned &ni, unsigned &no) {
#pragma clang fp contract(off)
  const float h = 2.8f * P.eps, h2 = h * h, hinv = 1.0f / h;
  const float self = tmass / P.eps;
  double accd = self;
  float accf = self;
  int j = 0;
  while (j < end) {
    const float4 q = it[j].pm;
    const int2 a = it[j].ax;
    float dx, dy, dz;
    if (STRADDLE) {
      dx = (float)nearest_d((double)q.x - (double)tx, P);
      dy = (float)nearest_d((double)q.y - (double)ty, P);
      dz = (float)nearest_d((double)q.z - (double)tz, P);
    } else {
      dx = q.x - tx; dy = q.y - ty; dz = q.z - tz;
    }
    const float r2 = pair_r2(dx, dy, dz);
    if (__int_as_float(a.x) > r2 * P.theta2) { j++; if (COUNT) no++; continue; }
    j = a.y > j ? a.y : end;  // skips always advance
    if (COUNT) ni++;
    const float t = kernel_term_f(q.w, r2, h2, hinv);
    if (P.wide_sum) accd += t;
    else accf += t;
  }
  return (P.wide_sum ? accd : (double)accf) * (double)P.G / (double)P.a;
}

template <bool COUNT>
__device__ __forceinline__ double walk_dispatch(const Work &W, const DevParams &P, const Seg &S,
                                                float tx, float ty, float tz, float tmass,
                                                unsigned &ni, unsigned &no) {
  const Item *it = W.items + 2 * S.ibase;  // positions and skips are segment-local
  if (P.replay) return walk_replay<COUNT>(it, P, S.n_items, tx, ty, tz, tmass, ni, no);
  if (S.straddle) return walk_fast<true, COUNT>(it, P, S.n_items, tx, ty, tz, tmass, ni, no);
  return walk_fast<false, COUNT>(it, P, S.n_items, tx, ty, tz, tmass, ni, no);
}

__device__ __forceinline__ void flush_counts(const Work &W, unsigned ni, unsigned no, unsigned nt,
                                             unsigned ns = 0, unsigned nw = 0) {
  unsigned long long a = ni, b = no, c = nt, d = ns, e = nw;
  a = wave_reduce_sum(a); b = wave_reduce_sum(b); c = wave_reduce_sum(c); d = wave_reduce_sum(d);
  e = wave_reduce_sum(e);
  if ((threadIdx.x & (WAVE - 1)) == 0) {
    atomicAdd(&W.counters[0], a); atomicAdd(&W.counters[1], b); atomicAdd(&W.counters[2], c);
    atomicAdd(&W.counters[3], d); atomicAdd(&W.counters[6], e);
  }
}

// Counts of an instrumented group walk, per lane: summed sources, opened
// nodes, targets, lane slots spent by the groups (leader lanes), wave steps
// (lane 0 of each wave).
struct WalkCount {
  unsigned ni = 0, no = 0, nt = 0, ns = 0, nw = 0;
  __device__ void flush(const Work &W) const { flush_counts(W, ni, no, nt, ns, nw); }
};

// Group-shared traversal.  The wave's 64 targets (consecutive in spatial
// order, one segment) are split into groups of GROUP lanes; each group walks
// the pre-order items together: the group stands on item j, every lane whose
// own path reaches j decides for itself (open, or use the monopole and skip
// the subtree), and the group moves to j+1 if any of its lanes opened j, else
// to skip(j) -- lanes still skipping an accepted ancestor A have
// skip(A) >= skip(j), so no lane's next item is passed over.  Each lane sees
// exactly the items, decisions and summation order of its own walk, whatever
// GROUP is.  GROUP = 64: the item index is wave-uniform and items are read
// with scalar loads; smaller groups visit fewer items that none of their lanes
// needs, at the price of vector loads and of the wave running until its
// slowest group is done.
template <int GROUP>
__device__ __forceinline__ u64 group_lanes() {
  if (GROUP == WAVE) return ~0ull;
  const int base = (int)(threadIdx.x & (WAVE - 1)) & ~(GROUP - 1);
  return (GROUP >= WAVE ? ~0ull : ((1ull << (GROUP & 63)) - 1ull)) << base;
}

template <int GROUP>
__device__ __forceinline__ bool group_any(bool p, u64 lanes) {
  if (GROUP == WAVE) return __any(p);
  return (__ballot(p) & lanes) != 0ull;
}

// Lane K of the caller's aligned group of GROUP (8, 16 or 32) lanes, read by
// every lane of the group (ds_swizzle, bit mode: source lane = (lane & AND) |
// K within each half-wave).  Every lane of the wave must be active.
template <int GROUP, int K>
__device__ __forceinline__ int group_field(int v) {
  static_assert(GROUP >= 8 && GROUP <= 32 && K < 8, "group_field: 8 to 32 lanes");
  constexpr int AND = 0x1f & ~(GROUP - 1);
  return __builtin_amdgcn_ds_swizzle(v, AND | (K << 5));
}

// Lane K of the caller's row of 16 lanes, read by every lane of the row (DPP
// row_newbcast: a source modifier of the consuming vector instruction, no LDS
// crossbar).  Every lane of the wave must be active.
template <int K>
__device__ __forceinline__ int row_field(int v) {
  return __builtin_amdgcn_mov_dpp(v, 0x150 + K, 0xf, 0xf, true);
}
// the same value in an instruction of its own
template <int K>
__device__ __forceinline__ int row_field_again(int v) {
  return __builtin_amdgcn_update_dpp(v, v, 0x150 + K, 0xf, 0xf, false);
}

// Lane mask m with every GROUP-lane field that holds a set bit filled (GROUP =
// 16 or 32), on the scalar unit.
template <int GROUP>
__device__ __forceinline__ u64 fill_fields(u64 m) {
  static_assert(GROUP == 16 || GROUP == 32, "16- or 32-lane fields");
  if (GROUP == 32) return ((u32)m ? 0xffffffffull : 0ull) | ((m >> 32) ? ~0xffffffffull : 0ull);
  // one bit per quad of lanes, filled per four quads, each bit widened to four again
  u64 q, r;
  u32 w;
  asm("s_quadmask_b64 %0, %1" : "=s"(q) : "s"(m) : "scc");
  asm("s_wqm_b32 %0, %1" : "=s"(w) : "s"((u32)q) : "scc");
  asm("s_bitreplicate_b64_b32 %0, %1" : "=s"(r) : "s"(w));
  asm("s_bitreplicate_b64_b32 %0, %1" : "=s"(q) : "s"((u32)r));
  return q;
}

// Per-target arithmetic of one item in FP32: sep2 = squared separation,
// opens = the opening test, add = the softened monopole term, the terms summed
// in FP64 (WIDE: the FAST precision; one conversion and one FP64 add per term,
// exact for a few thousand terms of one sign) or in FP32.  Straddling segments
// (a periodic subhalo wider than a quarter box) form the separation in double.
template <bool STRADDLE, bool WIDE>
struct FastTerm {
  using real = float;
  static constexpr bool WIDE_F32 = WIDE;
  float h2, hinv;
  typename std::conditional<WIDE, double, float>::type acc;
  __device__ __forceinline__ void init(const DevParams &P, bool live, float tmass) {
#pragma clang fp contract(off)
    const float h = 2.8f * P.eps;
    h2 = h * h;
    hinv = 1.0f / h;
    acc = live ? tmass / P.eps : 0.f;
  }
  __device__ __forceinline__ float sep2(const DevParams &P, const float4 &q, float tx, float ty,
                                        float tz) const {
#pragma clang fp contract(off)
    float dx, dy, dz;
    if (STRADDLE) {
      dx = (float)nearest_d((double)q.x - (double)tx, P);
      dy = (float)nearest_d((double)q.y - (double)ty, P);
      dz = (float)nearest_d((double)q.z - (double)tz, P);
    } else {
      dx = q.x - tx; dy = q.y - ty; dz = q.z - tz;
    }
    return pair_r2(dx, dy, dz);
  }
  __device__ __forceinline__ bool opens(const DevParams &P, float lsq, float r2) const {
#pragma clang fp contract(off)
    return lsq > r2 * P.theta2;
  }
  // the same test as a wave lane mask (every lane active)
  __device__ __forceinline__ u64 opens_mask(const DevParams &P, float lsq, float r2) const {
#pragma clang fp contract(off)
    return __builtin_amdgcn_fcmpf(lsq, r2 * P.theta2, 2 /* ordered > */);
  }
  // the same against the row's item v (its bound on r2)
  __device__ __forceinline__ u64 opens_row(const DevParams &, int v, float r2) const {
    return __builtin_amdgcn_fcmpf(r2, __int_as_float(row_field<7>(v)), 4 /* ordered < */);
  }
  __device__ __forceinline__ void add(float m, float r2) {
#pragma clang fp contract(off)
    acc += kernel_term_f(m, r2, h2, hinv);
  }
  // add() for the lanes in `accept` without branching on it: kernel_term_f's
  // Newtonian form is computed for every lane, the spline only for accepting
  // lanes within the softening length (rare), and the others add zero
  __device__ __forceinline__ void add_masked(bool accept, u64, float m, float r2) {
#pragma clang fp contract(off)
    float term = -m * __builtin_amdgcn_rsqf(r2);
    if (accept && !(r2 >= h2)) term = kernel_term_f(m, r2, h2, hinv);
    const float added = accept ? term : 0.f;
    acc += added;
  }
  // the lanes' terms of the row's item v, negated: the Newtonian form for every
  // lane, the spline only in steps where a lane of amask lies within the
  // softening length (the mass is read again there, so that the common product
  // takes it as a DPP operand)
  __device__ __forceinline__ float row_term(u64 amask, int v, float r2) const {
#pragma clang fp contract(off)
    float term = __int_as_float(row_field<3>(v)) * __builtin_amdgcn_rsqf(r2);
    const u64 near = amask & __builtin_amdgcn_fcmpf(r2, h2, 12 /* unordered or < */);
    if (near != 0ull) {
      const float m = __int_as_float(row_field_again<3>(v));
      if (__builtin_amdgcn_inverse_ballot_w64(near)) term = -kernel_term_f(m, r2, h2, hinv);
    }
    return term;
  }
  __device__ __forceinline__ double result() const { return (double)acc; }
};

// Reference arithmetic (src/gravity_tree.cpp:79-164): FP64 over float data.
struct ReplayTerm {
  using real = double;
  static constexpr bool WIDE_F32 = false;
  double h, hinv, pot;
  __device__ __forceinline__ void init(const DevParams &P, bool live, float tmass) {
#pragma clang fp contract(off)
    h = 2.8 * (double)P.eps;
    hinv = 1.0 / h;
    pot = live ? (double)(float)(tmass / P.eps) : 0.0;
  }
  __device__ __forceinline__ double sep2(const DevParams &P, const float4 &q, float tx, float ty,
                                         float tz) const {
#pragma clang fp contract(off)
    double dx = (double)q.x - (double)tx, dy = (double)q.y - (double)ty, dz = (double)q.z - (double)tz;
    if (P.periodic) { dx = nearest_d(dx, P); dy = nearest_d(dy, P); dz = nearest_d(dz, P); }
    return dx * dx + dy * dy + dz * dz;
  }
  __device__ __forceinline__ bool opens(const DevParams &P, float lsq, double r2) const {
#pragma clang fp contract(off)
    return (double)lsq > r2 * (double)P.theta2;
  }
  __device__ __forceinline__ u64 opens_mask(const DevParams &P, float lsq, double r2) const {
#pragma clang fp contract(off)
    return __builtin_amdgcn_fcmp((double)lsq, r2 * (double)P.theta2, 2 /* ordered > */);
  }
  __device__ __forceinline__ u64 opens_row(const DevParams &P, int v, double r2) const {
    return opens_mask(P, __int_as_float(row_field<4>(v)), r2);
  }
  __device__ __forceinline__ void add(float m, double r2) {
#pragma clang fp contract(off)
    pot += kernel_term_d((double)m, sqrt(r2), h, hinv);
  }
  __device__ __forceinline__ void add_masked(bool accept, u64, float m, double r2) {
    if (accept) add(m, r2);
  }
  __device__ __forceinline__ double result() const { return pot; }
};

// The items come in as a restrict-qualified kernel argument pointing at the
// segment's first item (wave-uniform; item positions and skips are
// segment-local): nothing in the walk kernel writes them, so reads at a
// group-uniform index compile to scalar loads when GROUP = 64, and both
// possible successors of item j (j+1 and skip(j)) are fetched while j is
// evaluated.  Smaller groups read with vector loads at a 32-bit byte offset
// from the scalar base, one dword of the item per lane, and spread the fields
// over the group -- 16 and 32 lanes with DPP row broadcasts, 8 lanes with
// crossbar swizzles; every lane of the wave takes
// part in every step (lanes off their path discard the result), the dwords of
// both possible successors are fetched as soon as skip(j) is known, the
// group's vote takes the group's field of the opened-lane mask, and the
// accepting lanes add their terms without a branch; a finished group sits on
// the sentinel item at `end`, whose skip is itself.  The 64-lane form
// clamps its reads to the segment's last item, a leaf whose skip is `end`, and
// its skips always advance (max with j+1).
//
// RANGE (16 lanes and up): only the items ib <= j < end of a longer array, a
// lane joining its path at item `join`; a group past `end` takes part in no
// further step.
template <int GROUP, bool COUNT, class Term, bool RANGE = false>
__device__ double walk_group(const Item *__restrict__ it, const DevParams &P, int ib, int end,
                             bool live, float tx, float ty, float tz, float tmass, WalkCount &wc, int join = 0) {
  Term t;
  t.init(P, live, tmass);
  const u64 lanes = group_lanes<GROUP>();
  const bool leader = (threadIdx.x & (GROUP - 1)) == 0;
  int until = live ? ib : INT_MAX;  // lane is on its path at j iff until <= j
  int j = group_any<GROUP>(live, lanes) ? ib : end;
  const int last = end - 1 > ib ? end - 1 : ib;
  if constexpr (GROUP == WAVE) {
    j = __builtin_amdgcn_readfirstlane(j);
    float4 q = it[(unsigned)min(j, last)].pm;
    int2 a = it[(unsigned)min(j, last)].ax;
    while (j < end) {
      const int j1 = j + 1;
      const int js = max(a.y, j1);
      const unsigned c1 = (unsigned)min(j1, last), cs = (unsigned)min(js, last);
      const float4 q1 = it[c1].pm, qs = it[cs].pm;
      const int2 a1 = it[c1].ax, as = it[cs].ax;
      bool opened = false;
      if (COUNT && leader) wc.ns += GROUP;
      if (COUNT && (threadIdx.x & (WAVE - 1)) == 0) wc.nw++;
      if (until <= j) {
        const typename Term::real r2 = t.sep2(P, q, tx, ty, tz);
        opened = t.opens(P, __int_as_float(a.x), r2);
        if (opened) {
          if (COUNT) wc.no++;
        } else {
          t.add(q.w, r2);
          until = a.y;
          if (COUNT) wc.ni++;
        }
      }
      const bool go = __any(opened);
      j = go ? j1 : js;
      q = go ? q1 : qs;
      a = go ? a1 : as;
    }
  } else if constexpr (GROUP >= 16) {
    // Vector issue bounds this loop: a step is about 20 vector instructions,
    // and products, sums and moves of vector registers issue in half the time
    // of compares, selects, conversions, FMAs and DPP forms (measured: 2.4
    // against 4.4 cycles per wave; the reciprocal root 8.3), so item fields
    // are DPP operands where an instruction can take them, the vote runs on
    // the scalar unit and selects are moves under an exec mask.  With the
    // items read through ds_swizzle and 8 lanes the 200,000-subhalo share's
    // walks took 91.8 ms; so, with 16 lanes, 78.2 ms (86 cycles of a SIMD per
    // wave step), the 4M-particle host's 14.9 -> 11.8 ms.
    // lane r of every 8 fetches dword r of its group's item; a row of 16 lanes shares the group's item, so its fields are
    // DPP row broadcasts inside the instructions that use them.  Positions are
    // byte offsets from the segment's first item plus the lane's dword offset
    // (< 32): J = 32 j + dw, and a skip becomes JS = 32 skip + dw.  A finished
    // group sits on the sentinel item (skip = itself, massless, far away, never
    // opened), where steps change nothing, so the exit is tested every UNROLL
    // steps; a lane without a target is never on its path.
    // (the address is the wave's: kept in scalar registers)
    using Global = const __attribute__((address_space(1))) char;
    Global *base = (Global *)(((u64)(u32)__builtin_amdgcn_readfirstlane((int)((u64)it >> 32)) << 32) |
                              (u32)__builtin_amdgcn_readfirstlane((int)(u64)it));
    auto dword = [base](unsigned off) { return *(const __attribute__((address_space(1))) int *)(base + off); };
    auto dword_next = [base](unsigned off) { return *(const __attribute__((address_space(1))) int *)(base + off + 32); };
    const unsigned dw = 4u * (threadIdx.x & 7u);
    const unsigned endb = 32u * (unsigned)end;
    unsigned J = 32u * (unsigned)j + dw;
    unsigned untilb = live ? 32u * (unsigned)(RANGE ? join : ib) + dw : UINT_MAX;
    int v = dword(J);
    const u64 full = __builtin_amdgcn_read_exec();
    constexpr int UNROLL = COUNT ? 1 : 4;
    while (__any(J < endb)) {
#pragma unroll
      for (int u = 0; u < UNROLL; u++) {
        const unsigned JS = (unsigned)row_field<6>(v) + dw;
        // both possible successors are fetched under the work on item j
        // (j + 1 = end + 1 reads the next region or the buffer's two spare items)
        const int v1 = dword_next(J), vs = dword(JS);
        const float4 q = make_float4(__int_as_float(row_field<0>(v)), __int_as_float(row_field<1>(v)),
                                     __int_as_float(row_field<2>(v)), __int_as_float(row_field<3>(v)));
        u64 pmask = __builtin_amdgcn_uicmp(untilb, J, 37 /* unsigned <= */);
        if (RANGE) pmask &= __builtin_amdgcn_uicmp(J, endb, 36 /* unsigned < */);
        const typename Term::real r2 = t.sep2(P, q, tx, ty, tz);
        const u64 omask = pmask & t.opens_row(P, v, r2);
        const u64 amask = pmask & ~omask;
        if (COUNT) {
          if (J < endb && leader) wc.ns += GROUP;
          if ((threadIdx.x & (WAVE - 1)) == 0) wc.nw++;
          const bool on = J < endb;
          wc.no += on && __builtin_amdgcn_inverse_ballot_w64(omask) ? 1u : 0u;
          wc.ni += on && __builtin_amdgcn_inverse_ballot_w64(amask) ? 1u : 0u;
        }
        const u64 gmask = fill_fields<GROUP>(omask);
        if constexpr (Term::WIDE_F32) {
          // under the accepting lanes' exec mask, and under that of the groups
          // that step into item j, plain moves and adds (half the issue time of
          // selects)
          const float term = t.row_term(amask, v, r2);
          double wide;
          asm volatile("s_mov_b64 exec, %3\n\t"
                       "v_mov_b32 %0, %4\n\t"
                       "v_cvt_f64_f32 %2, %5\n\t"
                       "v_add_f64 %1, %1, -%2\n\t"
                       "s_mov_b64 exec, %6"
                       : "+v"(untilb), "+v"(t.acc), "=&v"(wide)
                       : "s"(amask), "v"(JS), "v"(term), "s"(full));
          // v is written two instructions before its next use, a DPP read
          unsigned Jn = JS;
          int vn = vs;
          asm volatile("s_mov_b64 exec, %2\n\t"
                       "v_mov_b32 %0, %3\n\t"
                       "v_add_u32 %1, 32, %4\n\t"
                       "s_mov_b64 exec, %5"
                       : "+v"(vn), "+v"(Jn)
                       : "s"(gmask), "v"(v1), "v"(J), "s"(full));
          J = Jn;
          v = vn;
        } else {
          const bool go = __builtin_amdgcn_inverse_ballot_w64(gmask);
          J = go ? J + 32u : JS;
          v = go ? v1 : vs;
          const bool accept = __builtin_amdgcn_inverse_ballot_w64(amask);
          if (accept) t.add(q.w, r2);
          untilb = accept ? JS : untilb;
        }
      }
    }
  } else {
    // lane r of every 8 fetches dword r of its group's item (r = 5, 7 are
    // not used) and the group takes the six fields it needs from those lanes
    // through the LDS crossbar: 4 bytes per lane through the vector memory
    // pipe.  Positions are byte offsets from the segment's first item: J =
    // 32 j + the lane's dword offset (< 32), so J < 32 end iff j < end, and a
    // skip kept as 32 skip (the item's sb field) is <= J iff skip <= j.
    const char *base = (const char *)it;
    const unsigned dw = 4u * (threadIdx.x & 7u);
    // the group's lanes in a wave mask: the vote takes the group's field of a
    // lane mask with one 64-bit shift per lane (vector unit) instead of
    // folding the mask on the scalar unit
    const unsigned gbase = threadIdx.x & (WAVE - GROUP);
    constexpr u64 GFIELD = GROUP >= 64 ? ~0ull : ((1ull << (GROUP & 63)) - 1ull);
    const unsigned endb = 32u * (unsigned)end;
    unsigned J = 32u * (unsigned)j + dw;
    unsigned untilb = live ? 32u * (unsigned)ib : UINT_MAX;
    int v = *(const int *)(base + J);
    while (__any(J < endb)) {
      const bool on = J < endb;
      const float4 q = make_float4(__int_as_float(group_field<GROUP, 0>(v)), __int_as_float(group_field<GROUP, 1>(v)),
                                   __int_as_float(group_field<GROUP, 2>(v)), __int_as_float(group_field<GROUP, 3>(v)));
      const float lsq = __int_as_float(group_field<GROUP, 4>(v));
      const unsigned sb = (unsigned)group_field<GROUP, 6>(v);
      // J <= 32 end + dw throughout: every item's skip lies in (j, end], the sentinel's is end
      const unsigned J1 = J + 32u, JS = sb + dw;
      // both possible successors are fetched now, under the work on item j
      // (j + 1 = end + 1 reads the next region or the buffer's two spare items)
      const int v1 = *(const int *)(base + J1), vs = *(const int *)(base + JS);
      // lane masks straight from the compares (every lane is active here):
      // the group's vote runs on them without a round trip through VGPRs
      const u64 pmask = __builtin_amdgcn_uicmp(J, endb, 36 /* unsigned < */) &
                        __builtin_amdgcn_uicmp(untilb, J, 37 /* unsigned <= */);
      const typename Term::real r2 = t.sep2(P, q, tx, ty, tz);
      const u64 omask = pmask & t.opens_mask(P, lsq, r2);
      const u64 amask = pmask & ~omask;
      const bool accept = __builtin_amdgcn_inverse_ballot_w64(amask);
      if (COUNT) {
        if (on && leader) wc.ns += GROUP;
        if ((threadIdx.x & (WAVE - 1)) == 0) wc.nw++;
        wc.no += __builtin_amdgcn_inverse_ballot_w64(omask) ? 1u : 0u;
        wc.ni += accept ? 1u : 0u;
      }
      const bool go = ((omask >> gbase) & GFIELD) != 0ull;
      J = go ? J1 : JS;
      v = go ? v1 : vs;
      t.add_masked(accept, amask, q.w, r2);
      untilb = accept ? sb : untilb;
    }
  }
  return t.result();
}

template <int GROUP, bool COUNT, bool REPLAY>
__device__ __forceinline__ double walk_group_dispatch(const Item *__restrict__ it,
                                                      const DevParams &P, const Seg &S, int ib,
                                                      int end, bool live, float x, float y, float z,
                                                      float tm, WalkCount &wc) {
  if (REPLAY)
    return walk_group<GROUP, COUNT, ReplayTerm>(it, P, ib, end, live, x, y, z, tm, wc);
  if (!P.wide_sum) {
    if (S.straddle)
      return walk_group<GROUP, COUNT, FastTerm<true, false>>(it, P, ib, end, live, x, y, z, tm, wc);
    return walk_group<GROUP, COUNT, FastTerm<false, false>>(it, P, ib, end, live, x, y, z, tm, wc);
  }
  if (S.straddle)
    return walk_group<GROUP, COUNT, FastTerm<true, true>>(it, P, ib, end, live, x, y, z, tm, wc);
  return walk_group<GROUP, COUNT, FastTerm<false, true>>(it, P, ib, end, live, x, y, z, tm, wc);
}

// Lanes per group chosen per segment (S.wgroup, set from its size: 64 where
// 32-bit byte offsets do not reach).  The straddling and uncompensated forms (rare; precision study) keep 64.
template <bool COUNT, bool REPLAY>
__device__ __forceinline__ double walk_binned(const Item *__restrict__ it, const DevParams &P,
                                              const Seg &S, int ib, int end, bool live, float x,
                                              float y, float z, float tm, WalkCount &wc) {
  if (REPLAY) {
    switch (S.wgroup) {
      case 8: return walk_group<8, COUNT, ReplayTerm>(it, P, ib, end, live, x, y, z, tm, wc);
      case 16: return walk_group<16, COUNT, ReplayTerm>(it, P, ib, end, live, x, y, z, tm, wc);
      case 32: return walk_group<32, COUNT, ReplayTerm>(it, P, ib, end, live, x, y, z, tm, wc);
      default: return walk_group<64, COUNT, ReplayTerm>(it, P, ib, end, live, x, y, z, tm, wc);
    }
  }
  if (!P.wide_sum || S.straddle)
    return walk_group_dispatch<64, COUNT, false>(it, P, S, ib, end, live, x, y, z, tm, wc);
  using T = FastTerm<false, true>;
  switch (S.wgroup) {
    case 8: return walk_group<8, COUNT, T>(it, P, ib, end, live, x, y, z, tm, wc);
    case 16: return walk_group<16, COUNT, T>(it, P, ib, end, live, x, y, z, tm, wc);
    case 32: return walk_group<32, COUNT, T>(it, P, ib, end, live, x, y, z, tm, wc);
    default: return walk_group<64, COUNT, T>(it, P, ib, end, live, x, y, z, tm, wc);
  }
}

// The target mass that removes a target's own softened self term: none in a
// correction pass (its tree holds the removed block only); in a sampled pass
// the scaled mass of the sampled entries and none for the rest (:344-349);
// otherwise the particle's mass m.  isb flags the sampled entries.
__device__ __forceinline__ float target_mass(const Work &W, const Seg &S, int64_t b, int li, float m) {
  if (S.flags & F_CORR) return 0.f;
  if (S.flags & F_SAMP) return W.isb[b + li] ? m * S.mf : 0.f;
  return m;
}

// A target's binding energy from its potential.
// Full pass: E = 0.5|dv|^2 + phi (BindingEnergy, src/subhalo_unbind.cpp:341-354).
// Correction pass: E += OldVel.RefVelDiff + dK - phi_removed (:319-328).
template <bool REPLAY>
__device__ __forceinline__ void finish_target(const Work &W, const DevParams &P, const Seg &S, int64_t b,
                                              int li, float x, float y, float z, double pot) {
#pragma clang fp contract(off)
  pot = pot * (double)P.G / (double)P.a;
  const float4 v = W.vel[b + li];
  const float vx = v.x, vy = v.y, vz = v.z;
  if (!(S.flags & F_CORR)) {
    float dv[3];
    rel_vel(P, x, y, z, vx, vy, vz, S.ref_pos, S.ref_vel, dv);
    // the refinement pass keeps the unbinding energies (:252-259)
    float *E = (S.flags & F_REFINE) ? W.Er : W.E;
    if (REPLAY) {
      E[b + li] = (float)((double)vnorm_f(dv) * 0.5 + pot);
    } else {
      const double kin = 0.5 * ((double)dv[0] * dv[0] + (double)dv[1] * dv[1] + (double)dv[2] * dv[2]);
      E[b + li] = (float)(kin + pot);
    }
  } else {
    float ov[3];
    rel_vel(P, x, y, z, vx, vy, vz, S.old_pos, S.old_vel, ov);
    const float kin = vdot_f(ov, S.rvd) + S.dK;
    W.E[b + li] = (float)((double)W.E[b + li] + ((double)kin - pot));
  }
}

// The targets of one wave-aligned chunk of slots, one per lane.
template <int GROUP, bool COUNT, bool REPLAY>
__device__ __forceinline__ void walk_chunk(const Work &W, const DevParams &P, const Item *__restrict__ it,
                                           int64_t s, WalkCount &wc) {
  // segments are wave-aligned: the whole wave belongs to one segment
  const int k = __builtin_amdgcn_readfirstlane(W.seg_of_slot[s]);
  const Seg &S = W.seg[k];
  const int64_t b = S.ibase;
  const int l = (int)(s - b);
  const bool live = l < S.n_tgt;
  if (!__any(live)) return;
  if (COUNT && live) wc.nt++;
  const int li = live ? W.sp[s] : 0;
  const float4 q = W.pos[b + li];
  const float x = q.x, y = q.y, z = q.z;
  const float tm = target_mass(W, S, b, li, q.w);
  const Item *seg_it = it + 2 * b;  // item positions and skips are segment-local
  const int end = S.n_items;
  double pot;
  if (GROUP == 0)
    pot = walk_binned<COUNT, REPLAY>(seg_it, P, S, 0, end, live, x, y, z, tm, wc);
  else
    pot = walk_group_dispatch<GROUP == 0 ? 64 : GROUP, COUNT, REPLAY>(seg_it, P, S, 0, end, live, x, y, z,
                                                                     tm, wc);
  if (live) finish_target<REPLAY>(W, P, S, b, li, x, y, z, pot);
}

// Binding energies with the group-shared walk (same results as walk_kernel
// for every group size).  GROUP = 0: lanes per group from each segment's bin.
template <int GROUP, bool COUNT, bool REPLAY>
__global__ void __launch_bounds__(BLOCK) walk_shared_kernel(Work W, DevParams P,
                                                            const Item *__restrict__ it, int xcd_run) {
  WalkCount wc;
  const int vb = xcd_block(xcd_run);
  for (int64_t i = (int64_t)vb * BLOCK + threadIdx.x; i < W.nact; i += (int64_t)gridDim.x * BLOCK)
    walk_chunk<GROUP, COUNT, REPLAY>(W, P, it, slot_at(W, i), wc);
  if (COUNT) wc.flush(W);
}

// ---- one chunk's walk shared by several waves ---------------------------------
// A launch of few chunks leaves the chip waiting on each wave's chain of
// steps, one load after another (450 cycles a step at one wave per SIMD, 86
// with the chip full).  PARTS waves then walk a part of the item array each for
// the same 64 targets, and their sums are added.  The FP64 sum of FP32 terms
// is exact while it is below 2^29 times its smallest term (a list of millions of
// equal masses: 2^25), so the parts change no bit of it there; beyond it they may.
// One list of 24,000 particles (375 chunks, 16 parts): walks 0.53 -> 0.147 ms.

// First item of part w of PARTS for targets at item `own` of M: equal shares of
// a step density that falls off as a power of the distance from the targets,
// F(d) ~ d^s, with s measured on NFW lists (s = 1, even, up to 900 items; 0.76
// at 3,500; 0.35 at 174,000).  Equal item counts would give 8 parts of a
// 24,000-particle list a speedup of 2.4 in steps, this 4.0.
template <int PARTS>
__device__ __forceinline__ int part_start(int w, int own, int M) {
  if (w <= 0) return 0;
  if (w >= PARTS) return M;
  const float s = fminf(1.f, fmaxf(0.25f, 0.76f - 0.07f * __log2f((float)M / 3500.f)));
  const float a = exp2f(s * __log2f((float)max(own, 1))), b = exp2f(s * __log2f((float)max(M - own, 1)));
  const float v = (a + b) * (float)w / (float)PARTS - a;  // signed share from the targets' place
  const float d = exp2f(__log2f(fmaxf(fabsf(v), 1e-20f)) / s);
  return min(M, max(0, v < 0.f ? own - (int)d : own + (int)d));
}

// The part's share of the potential of 64 targets (lane's target at tx, ty, tz;
// own: their place among the items).  The wave first goes down to its first
// item e past every subtree that ends before it; a lane that accepts a node
// around e leaves the part at that node's skip.
template <int PARTS, class Term>
__device__ __forceinline__ double walk_part(const Item *__restrict__ it, const DevParams &P, int w, int own, int M,
                                            bool live, float tx, float ty, float tz, float tmass) {
  const int e = __builtin_amdgcn_readfirstlane(part_start<PARTS>(w, own, M));
  const int end = __builtin_amdgcn_readfirstlane(part_start<PARTS>(w + 1, own, M));
  const float self = w == 0 ? tmass : 0.f;
  WalkCount wc;
  int join = e;
  if (e < end) {
    Term t;
    t.init(P, false, 0.f);
    bool on = true;
    for (int j = 0; j < e;) {  // uniform across the wave
      const int skip = it[j].ax.y;
      if (skip <= e) {
        j = skip > j ? skip : j + 1;
        continue;
      }
      const typename Term::real r2 = t.sep2(P, it[j].pm, tx, ty, tz);
      if (on && !t.opens(P, __int_as_float(it[j].ax.x), r2)) {
        on = false;
        join = skip;
      }
      j++;
    }
  }
  return walk_group<16, false, Term, true>(it, P, e, max(e, end), live, tx, ty, tz, self, wc, join);
}

// The waves' shares added in order, in wave 0; part: PARTS - 1 rows in LDS.
// Called by the whole workgroup of PARTS waves.
template <int PARTS>
__device__ __forceinline__ double add_parts(double pot, double (*part)[WAVE]) {
#pragma clang fp contract(off)
  const int w = threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
  if (w > 0) part[w - 1][lane] = pot;
  __syncthreads();
  if (w == 0)
    for (int i = 0; i < PARTS - 1; i++) pot += part[i][lane];
  return pot;
}

template <int PARTS>
__global__ void __launch_bounds__(PARTS *WAVE) walk_split_kernel(Work W, DevParams P, const Item *__restrict__ it) {
  __shared__ double part[PARTS - 1][WAVE];
  const int lane = threadIdx.x & (WAVE - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int64_t i = (int64_t)blockIdx.x * WAVE + lane;
  if (i >= W.nact) return;  // nact is a multiple of WAVE: the whole workgroup
  const int64_t s = slot_at(W, i);
  const int k = __builtin_amdgcn_readfirstlane(W.seg_of_slot[s]);
  const Seg &S = W.seg[k];
  const int64_t b = S.ibase;
  const int l = (int)(s - b), n = S.n_tgt;
  const bool live = l < n;
  if (!__any(live)) return;  // the same in every wave of the workgroup
  const int li = live ? W.sp[s] : 0;
  const float4 q = W.pos[b + li];
  const float tm = target_mass(W, S, b, li, q.w);
  const Item *seg_it = it + 2 * b;
  const int M = S.n_items;
  const int mid = __builtin_amdgcn_readfirstlane(min(l - lane + WAVE / 2, n - 1));
  const int own = (int)((int64_t)M * mid / n);
  double pot;
  if (S.straddle) pot = walk_part<PARTS, FastTerm<true, true>>(seg_it, P, w, own, M, live, q.x, q.y, q.z, tm);
  else pot = walk_part<PARTS, FastTerm<false, true>>(seg_it, P, w, own, M, live, q.x, q.y, q.z, tm);
  pot = add_parts<PARTS>(pot, part);
  if (w == 0 && live) finish_target<false>(W, P, S, b, li, q.x, q.y, q.z, pot);
}

// What a sort's runs read and write per element: of lists that are one run, and
// of those whose merge levels (24 bytes each: key and value in and out) follow.
struct SortBytes {
  int one_run, merged;
};
constexpr SortBytes SORT_DIGITS{20 + 16, 20 + 16};  // Elist entry, position; key, value, node mask
constexpr SortBytes SORT_ENERGIES{8 + 4, 8 + 12};   // Elist entry, energy; the entry, or key and value
constexpr SortBytes SORT_PAIRS{24, 24};

// Instrumented passes: the elements a segmented sort ordered (counters[8]),
// the elements times the merge levels each needed (counters[9]) and the bytes of
// both (counters[10]).
__global__ void sort_count_kernel(Work W, const int *n, int above, int run, bool ranked, SortBytes B) {
  unsigned long long e = 0, el = 0, by = 0;
  SEG_LOOP(k, W) {
    const int c = W.seg[k].cap > above && n[k] > 0 ? n[k] : 0;
    e += (unsigned long long)c;
    const int levels = merge_levels(c, run, ranked);
    el += (unsigned long long)c * (unsigned long long)levels;
    by += (unsigned long long)c * (unsigned long long)(levels > 0 ? B.merged + 24 * levels : B.one_run);
  }
  e = wave_reduce_sum(e);
  el = wave_reduce_sum(el);
  by = wave_reduce_sum(by);
  if ((threadIdx.x & (WAVE - 1)) == 0 && (e | el)) {
    atomicAdd(&W.counters[8], e);
    atomicAdd(&W.counters[9], el);
    atomicAdd(&W.counters[10], by);
  }
}

// Instrumented passes: the items of the trees the walk read (counters[5]).
__global__ void tree_items_kernel(Work W) {
  SEG_LOOP(k, W) {
    const Seg &S = W.seg[k];
    if (S.n_tgt > 0 && S.n_items > 0) atomicAdd(&W.counters[5], (unsigned long long)S.n_items);
  }
}

// Binding energies of the pass's targets, in spatial order.
// Full pass: E = 0.5|dv|^2 + phi (BindingEnergy, :341-354).
// Correction pass: E += OldVel.RefVelDiff + dK - phi_removed (:319-328).
template <bool COUNT>
__global__ void __launch_bounds__(BLOCK) walk_kernel(Work W, DevParams P) {
  unsigned ni = 0, no = 0, nt = 0;
  SLOT_LOOP(s, W) {
#pragma clang fp contract(off)
    int k;
    int l = seg_lane_local(W, s, k);
    if (l < 0) continue;
    const Seg &S = W.seg[k];
    if (l >= S.n_tgt) continue;
    if (COUNT) nt++;
    const int64_t b = S.ibase;
    const int li = W.sp[s];
    const float4 q = W.pos[b + li], w = W.vel[b + li];
    const float x = q.x, y = q.y, z = q.z;
    const float vx = w.x, vy = w.y, vz = w.z;
    if (!(S.flags & F_CORR)) {
      const double pot = walk_dispatch<COUNT>(W, P, S, x, y, z, target_mass(W, S, b, li, q.w), ni, no);
      float dv[3];
      rel_vel(P, x, y, z, vx, vy, vz, S.ref_pos, S.ref_vel, dv);
      float *E = (S.flags & F_REFINE) ? W.Er : W.E;
      if (P.replay) {
        E[b + li] = (float)((double)vnorm_f(dv) * 0.5 + pot);
      } else {
        const double kin = 0.5 * ((double)dv[0] * dv[0] + (double)dv[1] * dv[1] + (double)dv[2] * dv[2]);
        E[b + li] = (float)(kin + pot);
      }
    } else {
      const double pot = walk_dispatch<COUNT>(W, P, S, x, y, z, 0.f, ni, no);
      float ov[3];
      rel_vel(P, x, y, z, vx, vy, vz, S.old_pos, S.old_vel, ov);
      const float kin = vdot_f(ov, S.rvd) + S.dK;
      W.E[b + li] = (float)((double)W.E[b + li] + ((double)kin - pot));
    }
  }
  if (COUNT) flush_counts(W, ni, no, nt);
}

// ---------------------------------------------------------------------------
// Partition (PartitionBindingEnergy, src/subhalo_unbind.cpp:21-58), in
// parallel.  Over positions 1..len-1, p_k is the k-th position from the front
// holding E>0 and g_k the k-th from the back holding E<0.  The two-pointer
// loop moves g_k to p_{k-1} (p_0 = 0) and p_k to g_k for k = 1..K, where K is
// the largest k with p_k < g_k; then g_{K+1} moves to p_K if g_{K+1} > p_K.
// Element 0 fills the last hole h, and Nbound = h + (E_0 < 0).
//
// Segments of several tiles, a workgroup per tile: signs and their counts by
// tile, the positions listed, K and the hole by segment, the moves with the
// bound flags, the flags' masks by tile, then the compacted spatial list with
// the new Elist's copy and its frame sums.  A sign is a byte and 64 flags one
// word between these launches, and ranks are found again from them: stored as
// 64-bit prefixes that every later launch read again, in fourteen launches, the
// larger segments' part of 200,000 subhalos' passes took 7.2 ms here and, with
// the frame sums it includes, takes 3.1 (37 million entries in the first pass).
//
// The tree's scratch is free after the walk: nlo holds the positions p_k (at
// k), nhi those of E<0 from the front (the j-th at j), npos the new Elist, dl
// the signs, k0 the masks (one per 64 slots).

// Sum of the tile totals t0 .. t-1, in every thread.
__device__ __forceinline__ u64 tiles_before(const u64 *__restrict__ tile_sum, int t0, int t) {
  u64 part = 0, all;
  for (int u = t0 + (int)threadIdx.x; u < t; u += BLOCK) part += tile_sum[u];
  (void)block_exclusive_scan(part, &all);
  return all;
}

// Elements of the tile that the pass partitions.
__device__ __forceinline__ int part_count(const Seg &S, const Tile &tl) {
  return (S.flags & F_ACTIVE) ? min(TILE, S.nlast - tl.start) : 0;
}

// Counts of both signs among a thread's four, E>0 in the low half.
__device__ __forceinline__ u32 sign_counts(const char4 &c) {
  auto one = [](signed char x) { return x > 0 ? 1u : x < 0 ? 0x10000u : 0u; };
  return one(c.x) + one(c.y) + one(c.z) + one(c.w);
}

__global__ void __launch_bounds__(BLOCK) part_signs_kernel(Work W, const Tile *__restrict__ tiles, int ntiles,
                                                           u64 *tile_sum) {
  static_assert(ITEMS == 4, "elements are loaded four at a time");
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    const int cnt = part_count(S, tl);
    if (cnt <= 0) continue;  // uniform
    const int64_t b = S.ibase, s0 = b + tl.start;
    const int p0 = ITEMS * (int)threadIdx.x;
    u32 own = 0, all;
    if (p0 < cnt) {
      const int4 a = *reinterpret_cast<const int4 *>(W.el + s0 + p0);
      auto sign = [&](int i, int li) -> signed char {
        if (p0 + i >= cnt || tl.start + p0 + i < 1) return 0;
        const float e = W.E[b + li];
        return e > 0.f ? 1 : e < 0.f ? -1 : 0;
      };
      const char4 c = make_char4(sign(0, a.x), sign(1, a.y), sign(2, a.z), sign(3, a.w));
      *reinterpret_cast<char4 *>(W.dl + s0 + p0) = c;
      own = sign_counts(c);
    }
    (void)block_exclusive_scan(own, &all);
    if (threadIdx.x == 0) tile_sum[t] = (u64)(all & 0xffffu) | ((u64)(all >> 16) << 32);
  }
}

// The tile's signs, four to a thread, and the number of each sign before them
// in the segment.
struct SignRank {
  signed char c[ITEMS];
  int p, g;
};
__device__ __forceinline__ SignRank sign_ranks(const Work &W, const Tile &tl, int t, int64_t s0, int cnt,
                                               const u64 *__restrict__ tile_sum) {
  SignRank K;
  const u64 pre = tiles_before(tile_sum, t - tl.start / TILE, t);
  char4 c = make_char4(0, 0, 0, 0);
  if (ITEMS * (int)threadIdx.x < cnt) c = *reinterpret_cast<const char4 *>(W.dl + s0 + ITEMS * threadIdx.x);
  u32 all;
  const u32 ex = block_exclusive_scan(sign_counts(c), &all);
  K.c[0] = c.x; K.c[1] = c.y; K.c[2] = c.z; K.c[3] = c.w;
  K.p = (int)(pre & 0xffffffffu) + (int)(ex & 0xffffu);
  K.g = (int)(pre >> 32) + (int)(ex >> 16);
  return K;
}

__global__ void __launch_bounds__(BLOCK) part_list_kernel(Work W, const Tile *__restrict__ tiles, int ntiles,
                                                          const u64 *tile_sum) {
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    const int cnt = part_count(S, tl);
    if (cnt <= 0) continue;  // uniform
    const int64_t b = S.ibase;
    SignRank K = sign_ranks(W, tl, t, b + tl.start, cnt, tile_sum);
    const int l0 = tl.start + ITEMS * (int)threadIdx.x;
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      if (K.c[r] > 0) W.nlo[b + ++K.p] = l0 + r;
      if (K.c[r] < 0) W.nhi[b + K.g++] = l0 + r;
    }
  }
}

// K, the hole, Nbound and the disruption test (:357-379), a workgroup per
// segment; K by a search 64 positions at a time (p_k < g_k holds up to K).
__global__ void __launch_bounds__(BLOCK) part_hole_kernel(Work W, DevParams P, const int *__restrict__ first_tile,
                                                          const u64 *tile_sum) {
  for (int k = blockIdx.x; k < W.nmulti; k += gridDim.x) {
    Seg &S = W.seg[k];
    if (!(S.flags & F_ACTIVE)) continue;  // uniform
    const int64_t b = S.ibase;
    const int n = S.nlast, t0 = first_tile[k];
    const u64 tot = tiles_before(tile_sum, t0, t0 + (n + TILE - 1) / TILE);
    const int nP = (int)(tot & 0xffffffffu), nG = (int)(tot >> 32);
    if (threadIdx.x < WAVE) {
      const int lane = threadIdx.x;
      const int *p = W.nlo + b, *g = W.nhi + b;
      int lo = 0, hi = min(nP, nG) + 1;  // p_k < g_k at lo (or lo is 0), not at hi
      while (hi - lo > 1) {
        const int step = (hi - lo - 1 + WAVE - 1) / WAVE;
        const int at = lo + step * (lane + 1);
        const int c = __popcll(__ballot(at < hi && p[at] < g[nG - at]));
        hi = min(hi, lo + step * (c + 1));
        lo += step * c;
      }
      if (lane == 0) {
        const int K = lo, pK = K ? p[K] : 0;
        const bool extra = K + 1 <= nG && g[nG - K - 1] > pK;
        S.K = K;
        S.nG = nG;
        S.nP = extra ? K + 1 : K;  // number of g moves
        S.hole = extra ? g[nG - K - 1] : pK;
        // the original element 0 ends in the last hole (Etmp, :37-38 and :50-51)
        const int nb = n == 0 ? 0 : S.hole + (W.E[b + W.el[b]] < 0.f ? 1 : 0);
        S.nbound = nb;
        if (nb < P.min_part) {
          S.flags = (S.flags & ~F_ACTIVE) | F_DISR | F_FINAL;
          S.nbound = 1;
          S.nlast = 1;
        }
        S.nsort = 0;  // the energy sort follows the frames
      }
    }
  }
}

// The new Elist (in npos) and the flags of the bound entries (isb).
__global__ void __launch_bounds__(BLOCK) part_move_kernel(Work W, const Tile *__restrict__ tiles, int ntiles,
                                                          const u64 *tile_sum) {
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    const int cnt = part_count(S, tl);
    if (cnt <= 0) continue;  // uniform
    const int64_t b = S.ibase;
    const int p0 = ITEMS * (int)threadIdx.x;
    int4 a = make_int4(0, 0, 0, 0);
    if (p0 < cnt) a = *reinterpret_cast<const int4 *>(W.el + b + tl.start + p0);
    SignRank K = sign_ranks(W, tl, t, b + tl.start, cnt, tile_sum);
    const int li[ITEMS] = {a.x, a.y, a.z, a.w};
    const int nb = S.nbound, moves = S.nP, nK = S.K, nG = S.nG;
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int l = tl.start + p0 + r;
      if (p0 + r >= cnt) continue;
      int dest = l;
      if (l == 0) dest = S.hole;
      if (K.c[r] > 0 && ++K.p <= nK) dest = W.nhi[b + nG - K.p];
      if (K.c[r] < 0) {
        const int k = nG - K.g++;
        if (k <= moves) dest = k == 1 ? 0 : W.nlo[b + k - 1];
      }
      W.npos[b + dest] = li[r];
      W.isb[b + li[r]] = dest < nb ? 1 : 0;
    }
  }
}

// The spatial list's bound flags, 64 to a mask, and their count by tile.
__global__ void __launch_bounds__(BLOCK) bound_masks_kernel(Work W, const Tile *__restrict__ tiles, int ntiles,
                                                            u64 *tile_sum) {
  __shared__ int wcount[BLOCK / WAVE];
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    const int cnt = part_count(S, tl);
    if (cnt <= 0) continue;  // uniform
    const int64_t b = S.ibase, s0 = b + tl.start;
    int q[ITEMS], have = 0;
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int i = (int)threadIdx.x + BLOCK * r;
      q[r] = i < cnt ? W.sp[s0 + i] : -1;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const u64 m = __ballot(q[r] >= 0 && W.isb[b + q[r]] != 0);
      have += __popcll(m);
      if ((threadIdx.x & (WAVE - 1)) == 0 && BLOCK * r + (int)threadIdx.x < cnt)
        W.k0[(s0 + BLOCK * r + threadIdx.x) / WAVE] = m;
    }
    if ((threadIdx.x & (WAVE - 1)) == 0) wcount[threadIdx.x / WAVE] = have;
    __syncthreads();
    if (threadIdx.x == 0) {
      int all = 0;
      for (int w = 0; w < BLOCK / WAVE; w++) all += wcount[w];
      tile_sum[t] = (u64)all;
    }
    __syncthreads();
  }
}

// A shuffled list that is disrupted puts its old most-bound particle (the
// first list entry before the shuffle) back in front: the first particle
// with its ID swaps with position 0 (:363-370).  Find, then swap.
__global__ void __launch_bounds__(BLOCK) disrupt_find_kernel(Work W) {
  SLOT_LOOP(s, W) {
    int k;
    int l = seg_lane_local(W, s, k);
    if (l < 0) continue;
    Seg &S = W.seg[k];
    if (!(S.flags & F_SHUF) || (S.flags & (F_DISR | F_FINAL)) != (F_DISR | F_FINAL) || l >= S.ulen) continue;
    if (W.g_id[W.gidx[s]] == S.old_mb_id) atomicMin(&S.swapq, l);
  }
}

__device__ __forceinline__ void swap_entries(const Work &W, int64_t a, int64_t c) {
  auto sw = [](auto *v, int64_t i, int64_t j) { const auto t = v[i]; v[i] = v[j]; v[j] = t; };
  sw(W.gidx, a, c); sw(W.pos, a, c); sw(W.vel, a, c);
}

__global__ void disrupt_swap_kernel(Work W) {
  MULTI_SEG_LOOP(k, W) {
    Seg &S = W.seg[k];
    if (!(S.flags & F_SHUF) || (S.flags & (F_DISR | F_FINAL)) != (F_DISR | F_FINAL)) continue;
    const int q = S.swapq;
    S.swapq = INT_MAX;
    if (q == INT_MAX || q == 0) continue;
    swap_entries(W, S.ibase, S.ibase + q);
  }
}

// Sampled pass: isb flags the sampled entries Elist[0, MaxSampleSize) (read
// by the walk for the self term; the partition then reuses isb).
__global__ void __launch_bounds__(BLOCK) sample_flags_kernel(Work W) {
  SLOT_LOOP(s, W) {
    int k;
    int l = seg_lane_local(W, s, k);
    if (l < 0) continue;
    const Seg &S = W.seg[k];
    if (!(S.flags & F_SAMP) || l >= S.nlast) continue;
    W.isb[S.ibase + W.el[s]] = l < S.n_src ? 1 : 0;
  }
}

// A captured pass sequence's spatial list back from el2.
__global__ void __launch_bounds__(BLOCK) spatial_copy_kernel(Work W) {
  SLOT_LOOP(s, W) {
    int k;
    int l = seg_lane_local(W, s, k);
    if (l < 0) continue;
    const Seg &S = W.seg[k];
    if (!(S.flags & F_ACTIVE) || l >= S.nbound) continue;
    W.sp[s] = W.el2[s];
  }
}

// What orders Elist by energy: (block, E), position breaking ties (a stable
// order).  The block bit keeps the bound block Elist[0, nbound) and the removed
// block Elist[nbound, nlast) apart, so one segmented sort orders each in place.
// Position `at` of a run or tile of 2^BITS from position `first`, as one word ...
template <int BITS>
__device__ __forceinline__ u64 energy_word(int at, int first, int nbound, float E) {
  return ((u64)(at >= nbound ? 1u : 0u) << (32 + BITS)) | ((u64)f2ord(E) << BITS) | (u64)(unsigned)(at - first);
}
// ... and as the key of the merge levels over the whole segment.
template <int BITS>
__device__ __forceinline__ u64 energy_key(u64 w, int first) {
  return ((w >> (32 + BITS)) << 63) | (((w >> BITS) & 0xffffffffull) << 31) |
         (u64)(unsigned)(first + (int)(w & ((1ull << BITS) - 1)));
}

// Energies of Elist[sort_lo, sort_lo + nsort), sorted by runs: into Elist where
// that is all, else into the buffer from which the merge levels end in (k0, v0).
__global__ void __launch_bounds__(RUN_THREADS, 8) energy_sort_kernel(Work W, const Tile *__restrict__ tiles,
                                                                     int ntiles, bool ranked) {
  constexpr int BITS = log2_of(RUN);
  __shared__ u64 sk[RUN];
  __shared__ int sv[RUN];
  for_runs(tiles, ntiles, [&](int k) { return W.ncount[NC_SORT * W.nseg + k]; }, [&](const Tile &tl) {
    const Seg &S = W.seg[tl.seg];
    const int64_t b = S.ibase;
    const int n = S.nsort, first = S.sort_lo + tl.start, nb = S.nbound;
    const int cnt = min(RUN, n - tl.start);
    u64 x[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int e = ITEMS * (int)threadIdx.x + r;
      const int li = e < cnt ? W.el[b + first + e] : -1;
      sv[e] = li;
      x[r] = e < cnt ? energy_word<BITS>(first + e, first, nb, W.E[b + li]) : ~0ull;
    }
    sort_tile_words<RUN_THREADS>(x, cnt, sk);
    const int m = merge_levels(n, RUN, ranked);
    u64 *kout = (m & 1) != 0 ? W.k1 : W.k0;
    u32 *vout = (m & 1) != 0 ? W.v1 : W.v0;
    for (int i = threadIdx.x; i < cnt; i += RUN_THREADS) {
      const u64 w = sk[i];
      const int li = sv[w & (RUN - 1)];
      if (m == 0) {
        W.el[b + first + i] = li;
      } else {
        kout[b + tl.start + i] = energy_key<BITS>(w, first);
        vout[b + tl.start + i] = (u32)li;
      }
    }
    __syncthreads();
  });
}

// ---------------------------------------------------------------------------
// FAST frame sums, tile-parallel: every tile of an active segment sums its part
// of the bound block in FP64 (mass, m*v, m*x relative to the periodic origin,
// part_finish_kernel); frames_combine_kernel adds the tiles of each segment in tile order, so the
// result does not depend on scheduling.
constexpr int FRAME_SUMS = 7;

// The frame sums of a bound entry at q, w: mass, momentum, mass-weighted position
// (relative to the most-bound entry o when periodic).
__device__ __forceinline__ void frame_accum(const DevParams &P, const float4 &q, const float4 &w, const double o[3],
                                            double v[FRAME_SUMS]) {
#pragma clang fp contract(off)
  const float m = q.w;
  v[0] += m;
  v[1] += w.x * m; v[2] += w.y * m; v[3] += w.z * m;
  if (P.periodic) {
    v[4] += nearest_d((double)q.x - o[0], P) * (double)m;
    v[5] += nearest_d((double)q.y - o[1], P) * (double)m;
    v[6] += nearest_d((double)q.z - o[2], P) * (double)m;
  } else {
    v[4] += q.x * m; v[5] += q.y * m; v[6] += q.z * m;
  }
}

// The bound entries of the spatial list in order into sp_out, the new Elist
// copied back, and (FAST) the frame sums of the tile's part of the bound block.
template <bool SUMS>
__global__ void __launch_bounds__(BLOCK) part_finish_kernel(Work W, DevParams P, const Tile *__restrict__ tiles,
                                                            int ntiles, const u64 *tile_sum, int *sp_out,
                                                            double *part) {
#pragma clang fp contract(off)
  __shared__ u64 mask[TILE / WAVE];
  __shared__ int first[TILE / WAVE];
  __shared__ double sh[FRAME_SUMS][BLOCK / WAVE];
  const int lane = threadIdx.x & (WAVE - 1);
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    const int cnt = part_count(S, tl);
    if (cnt <= 0) continue;  // uniform
    const int64_t b = S.ibase, s0 = b + tl.start;
    int q[ITEMS], li[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int i = (int)threadIdx.x + BLOCK * r;
      q[r] = i < cnt ? W.sp[s0 + i] : 0;
      li[r] = i < cnt ? W.npos[s0 + i] : 0;
    }
    const int before = (int)tiles_before(tile_sum, t - tl.start / TILE, t);
    if (threadIdx.x < TILE / WAVE) {
      const u64 m = WAVE * (int)threadIdx.x < cnt ? W.k0[s0 / WAVE + threadIdx.x] : 0ull;
      mask[threadIdx.x] = m;
      int run = __popcll(m);
#pragma unroll
      for (int d = 1; d < TILE / WAVE; d <<= 1) {
        const int y = __shfl_up(run, d, WAVE);
        if (lane >= d) run += y;
      }
      first[threadIdx.x] = before + run - __popcll(m);
    }
    __syncthreads();
    const float4 p0 = W.pos[b + W.npos[b]];
    const double o[3] = {p0.x, p0.y, p0.z};
    const int bound = min(TILE, S.nbound - tl.start);
    double v[FRAME_SUMS] = {0, 0, 0, 0, 0, 0, 0};
    float4 pos[ITEMS], vel[ITEMS];  // before the stores, so that they load together
    if (SUMS) {
#pragma unroll
      for (int r = 0; r < ITEMS; r++)
        if ((int)threadIdx.x + BLOCK * r < bound) { pos[r] = W.pos[b + li[r]]; vel[r] = W.vel[b + li[r]]; }
    }
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int i = (int)threadIdx.x + BLOCK * r;
      if (i >= cnt) continue;
      const int w = i / WAVE;
      if ((mask[w] >> lane) & 1ull) sp_out[b + first[w] + __popcll(mask[w] & ((1ull << lane) - 1ull))] = q[r];
      W.el[s0 + i] = li[r];
      if (SUMS && i < bound) frame_accum(P, pos[r], vel[r], o, v);
    }
    if (SUMS) {
      for (int c = 0; c < FRAME_SUMS; c++) {
        const double r = wave_total(v[c]);
        if (lane == 0) sh[c][threadIdx.x / WAVE] = r;
      }
      __syncthreads();
      if (threadIdx.x < FRAME_SUMS) {
        double r = 0;
        for (int w = 0; w < BLOCK / WAVE; w++) r += sh[threadIdx.x][w];
        part[(int64_t)t * FRAME_SUMS + threadIdx.x] = r;
      }
    }
    __syncthreads();
  }
}

// Correction switch, new frame, convergence (:380-421) for one segment, given
// its most-bound entry and the FP64 sums over its bound block.
__device__ void frame_update(Work &W, const DevParams &P, Seg &S, int l0, double msum, double s1, double s2,
                             double s3, double q1, double q2, double q3) {
#pragma clang fp contract(off)
  const int64_t b = S.ibase;
  const int nb = S.nbound;
  const float4 p0 = W.pos[b + l0], v0 = W.vel[b + l0];
  const double o[3] = {p0.x, p0.y, p0.z};
  // correction switch (uses the frame of the pass just done); with sampling
  // only when fewer than MaxSampleSize were removed (:383-389)
  if (S.nlast - nb < nb && (P.max_sample <= 0 || S.nlast - nb < P.max_sample)) {
    S.flags |= F_CORR;
    for (int j = 0; j < 3; j++) { S.old_pos[j] = S.ref_pos[j]; S.old_vel[j] = S.ref_vel[j]; }
  }
  if (nb == 0) {
    msum = 0.;
  } else if (nb == 1) {
    S.ref_vel[0] = v0.x; S.ref_vel[1] = v0.y; S.ref_vel[2] = v0.z;
    msum = p0.w;
    S.ref_pos[0] = p0.x; S.ref_pos[1] = p0.y; S.ref_pos[2] = p0.z;
  } else {
    S.ref_vel[0] = (float)(s1 / msum); S.ref_vel[1] = (float)(s2 / msum); S.ref_vel[2] = (float)(s3 / msum);
    double q[3] = {q1 / msum, q2 / msum, q3 / msum};
    for (int j = 0; j < 3; j++) {
      if (P.periodic) q[j] += o[j];
      S.ref_pos[j] = (float)q[j];
    }
  }
  S.mbound = (float)msum;
  // energy sort of the removed block Elist[nb, nlast) (:359-360) and, on
  // convergence, of the bound block Elist[0, nb) too (:401)
  if ((float)nb >= (float)S.nlast * P.bmp) {
    // RefineBindingEnergyOrder (:406-407) runs after the level's passes; the
    // outputs wait for it
    if (P.refine && nb > P.max_sample) {
      S.flags = (S.flags & ~F_ACTIVE) | F_CONV | F_REFPEND;
      atomicAdd(&W.active[3], 1);
    } else {
      S.flags = (S.flags & ~F_ACTIVE) | F_CONV | F_FINAL;
    }
    S.sort_lo = 0;
    S.nsort = S.nlast;
  } else {
    S.sort_lo = nb;
    S.nsort = S.nlast - nb;
  }
  W.ncount[NC_SORT * W.nseg + (int)(&S - W.seg)] = S.nsort;
}

// v[c] += part[(t0 + i * step) * C + c] for i = 0 .. cnt-1, in that order, with
// the values of the next few tiles loaded ahead of their use.
template <int C>
__device__ __forceinline__ void sum_tiles_in_order(const double *__restrict__ part, int t0, int cnt, int step,
                                                   double v[C]) {
#pragma clang fp contract(off)
  constexpr int PREF = 4;
  int i = 0;
  for (; i + PREF <= cnt; i += PREF) {
    double x[PREF][C];
#pragma unroll
    for (int u = 0; u < PREF; u++)
#pragma unroll
      for (int c = 0; c < C; c++) x[u][c] = part[(int64_t)(t0 + (i + u) * step) * C + c];
#pragma unroll
    for (int u = 0; u < PREF; u++)
#pragma unroll
      for (int c = 0; c < C; c++) v[c] += x[u][c];
  }
  for (; i < cnt; i++)
#pragma unroll
    for (int c = 0; c < C; c++) v[c] += part[(int64_t)(t0 + i * step) * C + c];
}

// Segments whose bound block spans more than SUPER_TILES tiles: one thread per
// run of SUPER_TILES tiles sums the run's partials in tile order into gpart
// (at the run's first tile), so that frames_combine_kernel adds runs.
__global__ void __launch_bounds__(BLOCK) frames_runs_kernel(Work W, const Tile *__restrict__ tiles, int ntiles,
                                                            const double *part, double *gpart) {
#pragma clang fp contract(off)
  for (int t = blockIdx.x * BLOCK + threadIdx.x; t < ntiles; t += gridDim.x * BLOCK) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    const int nt = (S.flags & F_ACTIVE) ? (S.nbound + TILE - 1) / TILE : 0;
    const int r = tl.start / TILE;  // tile number within the segment
    if (nt <= SUPER_TILES || r >= nt || r % SUPER_TILES != 0) continue;
    double v[FRAME_SUMS] = {0, 0, 0, 0, 0, 0, 0};
    sum_tiles_in_order<FRAME_SUMS>(part, t, min(SUPER_TILES, nt - r), 1, v);
    for (int c = 0; c < FRAME_SUMS; c++) gpart[(int64_t)t * FRAME_SUMS + c] = v[c];
  }
}

// One thread per segment.  A bound block of more than SUPER_TILES tiles is
// summed over the runs of frames_runs_kernel.
__global__ void frames_combine_kernel(Work W, DevParams P, const int *first_tile, const double *part,
                                      const double *gpart) {
#pragma clang fp contract(off)
  MULTI_SEG_LOOP(k, W) {
    Seg &S = W.seg[k];
    if (!(S.flags & F_ACTIVE)) continue;
    double v[FRAME_SUMS] = {0, 0, 0, 0, 0, 0, 0};
    const int nt = (S.nbound + TILE - 1) / TILE;
    if (nt <= SUPER_TILES)
      sum_tiles_in_order<FRAME_SUMS>(part, first_tile[k], nt, 1, v);
    else
      sum_tiles_in_order<FRAME_SUMS>(gpart, first_tile[k], (nt + SUPER_TILES - 1) / SUPER_TILES, SUPER_TILES, v);
    frame_update(W, P, S, W.el[S.ibase], v[0], v[1], v[2], v[3], v[4], v[5], v[6]);
  }
}

// ---------------------------------------------------------------------------
// Frame update (:380-421) with the reference's summation order (REPLAY): one
// thread per segment sums the bound block serially in Elist order.
__global__ void frames_serial_kernel(Work W, DevParams P) {
#pragma clang fp contract(off)
  SEG_LOOP(k, W) {
    Seg &S = W.seg[k];
    if (!(S.flags & F_ACTIVE)) continue;
    const int64_t b = S.ibase;
    const int nb = S.nbound;
    const float4 p0 = W.pos[b + W.el[b]];
    const double o[3] = {p0.x, p0.y, p0.z};
    double msum = 0, s1 = 0, s2 = 0, s3 = 0, q1 = 0, q2 = 0, q3 = 0;
    if (nb > 1) {
      for (int i = 0; i < nb; i++) {
        const int li = W.el[b + i];
        const float4 q = W.pos[b + li], w = W.vel[b + li];
        const float m = q.w;
        msum += m;
        s1 += w.x * m; s2 += w.y * m; s3 += w.z * m;
        if (P.periodic) {
          q1 += nearest_d((double)q.x - o[0], P) * (double)m;
          q2 += nearest_d((double)q.y - o[1], P) * (double)m;
          q3 += nearest_d((double)q.z - o[2], P) * (double)m;
        } else {
          q1 += q.x * m; q2 += q.y * m; q3 += q.z * m;
        }
      }
    }
    frame_update(W, P, S, W.el[b], msum, s1, s2, s3, q1, q2, q3);
  }
}

// ---------------------------------------------------------------------------
// Outputs for segments that finished in this pass, early exits and orphans.

// Output list and energies of entry l.  li: Elist's entry at l, for l < ulen.
// Split in what is read and what is written, so that a thread's entries load
// together.
struct OutEntry {
  int64_t index;
  float energy;
};
template <class Energy>
__device__ __forceinline__ OutEntry output_entry(const Work &W, const Seg &S, int l, int li, Energy energy) {
  const bool sorted = (S.flags & F_CONV) && !(S.flags & F_ORPHAN) && l < S.ulen;
  OutEntry e;
  e.index = W.gidx[S.ibase + (sorted ? li : l)];
  e.energy = sorted ? energy() : __builtin_nanf("");
  // disrupted, early, orphan: the list keeps its order -- an orphan's own list
  // as it came in, even when a shuffled copy of it was unbound (:434-446)
  if ((S.flags & F_ORPHAN) && (S.flags & F_SHUF) && l < S.count) e.index = own_entry(W, S, l);
  return e;
}
__device__ __forceinline__ OutEntry output_entry(const Work &W, const Seg &S, int l, int li) {
  return output_entry(W, S, l, li, [&]() { return W.E[S.ibase + li]; });
}
__device__ __forceinline__ void write_entry(const Work &W, const Seg &S, int l, const OutEntry &e) {
  W.out_index[S.out_off + l] = e.index;
  W.out_energy[S.out_off + l] = e.energy;
}

// Writes the record of a segment that finished, from its sums over the bound
// block: kinematics (AverageKinematics, :189-232), particle types
// (CountParticleTypes / CountParticles, src/subhalo.cpp:400-499) and the
// state markers of Unbind (:269-421).
__device__ void write_record(Work &W, const DevParams &P, Seg &S, double E, double K, double A0,
                             double A1, double A2, double M, const int nt[HBT_TYPE_MAX],
                             const float mts[HBT_TYPE_MAX]) {
#pragma clang fp contract(off)
  hbt_subhalo &r = W.subs[S.sub];
  const int64_t b = S.ibase;
  const bool conv = (S.flags & F_CONV) != 0;
  const int nb = S.nbound;
  if (S.flags & F_EARLY) {
    float mb = 0.f;  // CountParticles: Mbound = float sum of MboundType
    for (int t = 0; t < HBT_TYPE_MAX; t++) mb += mts[t];
    r.mbound = mb;
    r.status = HBT_STATUS_EARLY;
  } else {
    if (nb <= 1) {
      r.specific_self_potential_energy = 0.f;
      r.specific_self_kinetic_energy = 0.f;
      r.specific_angular_momentum[0] = r.specific_angular_momentum[1] = r.specific_angular_momentum[2] = 0.f;
    } else {
      E /= M;
      K *= 0.5 / M;
      r.specific_self_potential_energy = (float)(E - K);
      r.specific_self_kinetic_energy = (float)K;
      r.specific_angular_momentum[0] = (float)(A0 / M);
      r.specific_angular_momentum[1] = (float)(A1 / M);
      r.specific_angular_momentum[2] = (float)(A2 / M);
    }
    if (conv) {
      r.status = HBT_STATUS_CONVERGED;
      if (r.snapshot_index_of_death != -1) r.snapshot_index_of_death = -1;
      if (r.sink_track_id != -1) { r.snapshot_index_of_sink = -1; r.sink_track_id = -1; }
      for (int j = 0; j < 3; j++) { r.ref_pos[j] = S.ref_pos[j]; r.ref_vel[j] = S.ref_vel[j]; }
      const int l0 = W.el[b];
      const float4 q = W.pos[b + l0], w = W.vel[b + l0];
      r.mostbound_pos[0] = q.x; r.mostbound_pos[1] = q.y; r.mostbound_pos[2] = q.z;
      r.mostbound_vel[0] = w.x; r.mostbound_vel[1] = w.y; r.mostbound_vel[2] = w.z;
      r.mbound = S.mbound;
    } else {
      // disruption (:361-379): frame <- previous most-bound coordinates
      r.status = HBT_STATUS_DISRUPTED;
      if (r.snapshot_index_of_death == -1) r.snapshot_index_of_death = P.snap;
      for (int j = 0; j < 3; j++) { r.ref_pos[j] = r.mostbound_pos[j]; r.ref_vel[j] = r.mostbound_vel[j]; }
      r.mbound = W.pos[b].w;
    }
  }
  for (int t = 0; t < HBT_TYPE_MAX; t++) { r.nbound_type[t] = nt[t]; r.mbound_type[t] = mts[t]; }
  r.nbound = nb;
  r.list_len = S.len;
  long long ns = nb <= 1 ? nb : (long long)((float)nb * P.relax);
  if (ns > S.len) ns = S.len;
  r.nsource = ns;
  r.n_iter = S.iter;
  r.n_evals = S.evals;
  S.flags &= ~F_FINAL;
}

// Kinematics of one bound particle (AverageKinematics, :205-224).
__device__ __forceinline__ void kin_accum(const Work &W, const DevParams &P, const Seg &S, int li,
                                          double v[6]) {
#pragma clang fp contract(off)
  const int64_t b = S.ibase;
  const float4 q = W.pos[b + li], w = W.vel[b + li];
  const float m = q.w;
  v[0] += W.E[b + li] * m;
  const float x[3] = {q.x, q.y, q.z};
  const float vel[3] = {w.x, w.y, w.z};
  double dx[3], dv[3];
  for (int j = 0; j < 3; j++) {
    dx[j] = x[j] - S.ref_pos[j];
    if (P.periodic) dx[j] = nearest_d(dx[j], P);
    dx[j] *= P.a;
    dv[j] = (double)(vel[j] - S.ref_vel[j]) + P.hz * dx[j];
    v[1] += dv[j] * dv[j] * m;
  }
  v[2] += (dx[1] * dv[2] - dx[2] * dv[1]) * m;
  v[3] += (dx[2] * dv[0] - dx[0] * dv[2]) * m;
  v[4] += (dx[0] * dv[1] - dx[1] * dv[0]) * m;
  v[5] += m;
}

// Serial form (REPLAY and early exits): sums in list order as the reference
// does with one thread.
__device__ __forceinline__ void record_serial(Work &W, const DevParams &P, Seg &S) {
#pragma clang fp contract(off)
  const int64_t b = S.ibase;
  const bool conv = (S.flags & F_CONV) != 0;
  const int nb = S.nbound;
  const bool skip_null = !(S.flags & F_EARLY) && nb <= 100;
  double v[6] = {0, 0, 0, 0, 0, 0};
  int nt[HBT_TYPE_MAX] = {0, 0, 0, 0, 0, 0};
  float mts[HBT_TYPE_MAX] = {0, 0, 0, 0, 0, 0};
  for (int i = 0; i < nb; i++) {
    const int li = conv ? W.el[b + i] : i;
    if (nb > 1) kin_accum(W, P, S, li, v);
  }
  for (int i = 0; i < nb; i++) {
    const int li = conv ? W.el[b + i] : i;
    if (skip_null && W.g_id[W.gidx[b + li]] == -1) continue;
    const int t = __float_as_int(W.vel[b + li].w);
    nt[t]++;
    mts[t] += W.pos[b + li].w;
  }
  write_record(W, P, S, v[0], v[1], v[2], v[3], v[4], v[5], nt, mts);
}

__global__ void output_record_kernel(Work W, DevParams P) {
  SEG_LOOP(k, W) {
    Seg &S = W.seg[k];
    if (S.flags & F_FINAL) record_serial(W, P, S);
  }
}

// Lists and records of the early exits (0 or 1 particles to unbind), a wave per
// segment: over every slot they took 0.26 ms of a level of 54 million.  An orphan
// host's list holds its subhalos' tails too, whatever their number: of more than a
// tile, it goes by tiles (early_tiles_kernel; ten tails of 300,000 by one wave took
// 26 ms of a call, 10 without them).
__global__ void __launch_bounds__(BLOCK) output_early_kernel(Work W, DevParams P) {
  WAVE_SEG_LOOP(k, W.nseg) {
    Seg &S = W.seg[k];
    if (!(S.flags & F_EARLY)) continue;  // uniform across the wave
    const int lane = threadIdx.x & (WAVE - 1);
    if (S.len <= TILE)
      for (int l = lane; l < S.len; l += WAVE) write_entry(W, S, l, output_entry(W, S, l, 0));  // (none of them converged)
    if (lane == 0) record_serial(W, P, S);
  }
}

__global__ void __launch_bounds__(BLOCK) early_tiles_kernel(Work W, const Tile *__restrict__ tiles, int ntiles) {
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    if (!(S.flags & F_EARLY) || S.len <= TILE) continue;  // uniform
    const int end = min(tl.start + TILE, S.len);
    for (int l = tl.start + (int)threadIdx.x; l < end; l += BLOCK) write_entry(W, S, l, output_entry(W, S, l, 0));
  }
}

// FAST form, tile-parallel: partial sums per tile (6 kinematic sums, 6 type
// counts, 6 type masses in FP64), combined per segment in tile order.  A
// converged segment's bound set is read in slot order -- the slots of the
// list it unbound, [0, ulen), flagged in isb (every pass's partition flags the
// slots it keeps, so the flags hold the final bound set) -- so the reads
// stream through the columns instead of following the energy order; other
// finished segments sum their first nbound slots.
constexpr int REC_SUMS = 18;

__device__ __forceinline__ int record_span(const Seg &S) { return (S.flags & F_CONV) ? S.ulen : S.nbound; }

// The record sums of slot li: kinematics of a bound entry, and its type
// count and mass unless it is a null particle of a small subhalo.
__device__ __forceinline__ void record_accum(const Work &W, const DevParams &P, const Seg &S, int64_t b, int li,
                                             int nb, bool skip_null, double (&v)[REC_SUMS]) {
#pragma clang fp contract(off)
  if (nb > 1) kin_accum(W, P, S, li, v);
  if (skip_null && W.g_id[W.gidx[b + li]] == -1) return;
  const int ty = __float_as_int(W.vel[b + li].w);
  const float m = W.pos[b + li].w;
  for (int q = 0; q < HBT_TYPE_MAX; q++) {
    const bool hit = q == ty;
    v[6 + q] += hit ? 1.0 : 0.0;
    v[12 + q] += hit ? (double)m : 0.0;
  }
}

// After the energy sort, a workgroup per tile: the merged order into Elist where
// more than `run` elements were sorted (shorter ones are there), and the lists of
// the segments that finished.  keyed: the merged keys hold the entries' energies,
// which are then not gathered.  As two launches over the slots, a thread's entries
// one after another, 1.24 ms of 200,000 subhalos' passes, 0.76 now; with the
// record sums in the same launch, whose registers leave five waves per SIMD, both
// took 1.6 together (1.4 apart).
__global__ void __launch_bounds__(BLOCK)
output_tile_kernel(Work W, const Tile *__restrict__ tiles, int ntiles, int run, bool keyed) {
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    const bool fin = (S.flags & F_FINAL) != 0;
    const int lo = S.sort_lo, nsort = S.nsort;
    const bool merged = nsort > run;
    const int end = fin ? S.len : merged ? lo + nsort : 0;
    const int cnt = min(TILE, end - tl.start);
    if (cnt <= 0) continue;  // uniform
    const int64_t b = S.ibase;
    int li[ITEMS];
    OutEntry e[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int i = (int)threadIdx.x + BLOCK * r, l = tl.start + i;
      const bool in = merged && l >= lo && l < lo + nsort;
      li[r] = i >= cnt ? 0 : in ? (int)W.v0[b + l - lo] : W.el[b + l];
    }
    if (fin) {
#pragma unroll
      for (int r = 0; r < ITEMS; r++) {
        const int i = (int)threadIdx.x + BLOCK * r, l = tl.start + i;
        const bool key = keyed && merged && l >= lo && l < lo + nsort;
        if (i < cnt)
          e[r] = output_entry(W, S, l, li[r], [&]() {
            return key ? ord2f((u32)(W.k0[b + l - lo] >> 31)) : W.E[b + li[r]];
          });
      }
    }
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
      const int i = (int)threadIdx.x + BLOCK * r, l = tl.start + i;
      if (i >= cnt) continue;
      if (merged && l >= lo && l < lo + nsort) W.el[b + l] = li[r];
      if (fin) write_entry(W, S, l, e[r]);
    }
  }
}

__global__ void __launch_bounds__(BLOCK)
output_partial_kernel(Work W, DevParams P, const Tile *tiles, int ntiles, double *part) {
#pragma clang fp contract(off)
  __shared__ double sh[REC_SUMS][BLOCK / WAVE];
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const Seg &S = W.seg[tl.seg];
    const bool fin = (S.flags & F_FINAL) != 0;
    const int cnt = fin ? min(TILE, record_span(S) - tl.start) : 0;
    if (cnt <= 0) continue;  // uniform
    const int64_t b = S.ibase;
    const bool conv = (S.flags & F_CONV) != 0;
    const int nb = S.nbound;
    const bool skip_null = nb <= 100;
    double v[REC_SUMS];
    for (int c = 0; c < REC_SUMS; c++) v[c] = 0;
    for (int i = threadIdx.x; i < cnt; i += BLOCK)
      if (!conv || W.isb[b + tl.start + i]) record_accum(W, P, S, b, tl.start + i, nb, skip_null, v);
    for (int c = 0; c < REC_SUMS; c++) {
      const double r = wave_total(v[c]);
      if ((threadIdx.x & (WAVE - 1)) == 0) sh[c][threadIdx.x / WAVE] = r;
    }
    __syncthreads();
    if (threadIdx.x < REC_SUMS) {
      double r = 0;
      for (int w = 0; w < BLOCK / WAVE; w++) r += sh[threadIdx.x][w];
      part[(int64_t)t * REC_SUMS + threadIdx.x] = r;
    }
    __syncthreads();
  }
}

// The record of a segment that finished, from its sums.
__device__ __forceinline__ void write_record_sums(Work &W, const DevParams &P, Seg &S, const double (&v)[REC_SUMS]) {
  int nt[HBT_TYPE_MAX];
  float mts[HBT_TYPE_MAX];
  for (int q = 0; q < HBT_TYPE_MAX; q++) { nt[q] = (int)v[6 + q]; mts[q] = (float)v[12 + q]; }
  write_record(W, P, S, v[0], v[1], v[2], v[3], v[4], v[5], nt, mts);
}

// The first nseg segments, a wave each.
__global__ void __launch_bounds__(BLOCK) output_combine_kernel(Work W, DevParams P, int nseg, const int *first_tile,
                                                               const double *part) {
  WAVE_SEG_LOOP(k, nseg) {
    Seg &S = W.seg[k];
    if (!(S.flags & F_FINAL)) continue;  // uniform across the wave
    double v[REC_SUMS];
    wave_sum_tiles<REC_SUMS>(part, first_tile[k], (record_span(S) + TILE - 1) / TILE, v);
    if ((threadIdx.x & (WAVE - 1)) == 0) write_record_sums(W, P, S, v);
  }
}

// ---------------------------------------------------------------------------
// Everything after the walk for a segment of one tile, in one launch: the
// partition, the spatial list, the frame, the energy sort and, where the
// segment finished, its outputs, a wave or a workgroup each (the teams of
// tree_one), Elist and energies in LDS in between.  REPLAY sums in the
// reference's order between two stages of it.  As fifteen launches over every
// slot, each behind its own loads of segment, list and record, this took 7.0 ms
// of a batch of 200,000 subhalos' passes (3.4 now) and 35 us of a pass of a
// 300-particle list (12 now); the record's 18 FP64 sums bound it, so their
// registers are kept to four waves per SIMD.
enum { POST_PART = 1, POST_FRAME = 2, POST_SORT = 4, POST_RECORD = 8 };
constexpr int POST_ALL = POST_PART | POST_FRAME | POST_SORT | POST_RECORD;

template <int CAP>
struct OnePost {
  union {
    struct { unsigned short p[CAP + 1], g[CAP + 1]; } part;  // p_k, g_k of the partition
    u64 key[CAP];                                            // energy sort of a workgroup
  };
  float E[CAP];             // by Elist position, until the energy sort
  unsigned short el[CAP];   // Elist
  unsigned char bound[CAP]; // by list entry
  double sums[REC_SUMS][BLOCK / WAVE];
  int K;
};

// Sums of C values over the elements 0 .. cnt-1 of a tile, add(e, v) adding
// element e's; in the team's first thread.  Up to BLOCK elements, which any team
// may hold, both forms add the totals of 64 neighbouring ones to zero in order:
// the same bits.
template <class TM, int C, class Add>
__device__ __forceinline__ void tile_sums(int cnt, double (&out)[C], double (*sh)[BLOCK / WAVE], Add add) {
#pragma clang fp contract(off)
  if constexpr (TM::T == WAVE) {
    double sum = 0;
    for (int e0 = 0; e0 < cnt; e0 += WAVE) {
      double v[C];
      for (int c = 0; c < C; c++) v[c] = 0;
      if (e0 + TM::id() < cnt) add(e0 + TM::id(), v);
      for (int c = 0; c < C; c++) {
        const double t = wave_total(v[c]);
        if (TM::id() == c) sum += t;  // lane c keeps sum c
      }
    }
    for (int c = 0; c < C; c++) out[c] = readlane_double(sum, c);
  } else {
    double v[C];
    for (int c = 0; c < C; c++) v[c] = 0;
    for (int e = TM::id(); e < cnt; e += TM::T) add(e, v);
    for (int c = 0; c < C; c++) {
      const double r = wave_total(v[c]);
      if ((threadIdx.x & (WAVE - 1)) == 0) sh[c][threadIdx.x / WAVE] = r;
    }
    TM::sync();
    if (TM::id() < C) {
      double r = 0;
      for (int w = 0; w < BLOCK / WAVE; w++) r += sh[TM::id()][w];
      sh[TM::id()][0] = r;
    }
    TM::sync();
    if (TM::id() == 0)
      for (int c = 0; c < C; c++) out[c] = sh[c][0];
  }
}

template <class TM, int STAGE>
__device__ __forceinline__ void post_one(Work &W, const DevParams &P, const Tile &tl, int *sp_out,
                                         OnePost<TM::CAP> &L) {
  constexpr int R = TM::R, CAP = TM::CAP, T = TM::T;
  Seg &S = W.seg[tl.seg];
  const int64_t b = S.ibase;
  const int id = TM::id();
  int n = min(CAP, S.nlast);
  if constexpr ((STAGE & POST_PART) != 0) {
    if (!(S.flags & F_ACTIVE)) return;  // uniform across the team
    int li[R], cls[R], rank[R];
    float e[R];
    u32 own = 0, all;  // low half: E > 0, high half: E < 0
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int l = R * id + r;
      li[r] = l < n ? W.el[b + l] : 0;
      e[r] = l < n ? W.E[b + li[r]] : 0.f;
      cls[r] = (l < 1 || l >= n) ? 0 : e[r] > 0.f ? 1 : e[r] < 0.f ? 2 : 0;
      own += cls[r] == 1 ? 1u : cls[r] == 2 ? 0x10000u : 0u;
    }
    const u32 before = TM::exclusive_scan(own, &all);
    const int nP = (int)(all & 0xffffu), nG = (int)(all >> 16);
    int p = (int)(before & 0xffffu), g = (int)(before >> 16);
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int l = R * id + r;
      if (cls[r] == 1) L.part.p[rank[r] = ++p] = (unsigned short)l;
      if (cls[r] == 2) L.part.g[rank[r] = nG - g++] = (unsigned short)l;
    }
    if (id == 0) L.K = 0;
    TM::sync();
    const int m = min(nP, nG);
    for (int k = 1 + id; k <= m; k += T)
      if (L.part.p[k] < L.part.g[k] && (k == m || L.part.p[k + 1] >= L.part.g[k + 1])) L.K = k;
    TM::sync();
    const int K = L.K, pK = K ? L.part.p[K] : 0;
    const bool extra = K + 1 <= nG && L.part.g[K + 1] > pK;
    const int hole = extra ? L.part.g[K + 1] : pK, moves = extra ? K + 1 : K;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int l = R * id + r;
      if (l >= n) continue;
      int dest = l;
      if (l == 0) dest = hole;
      else if (cls[r] == 1 && rank[r] <= K) dest = L.part.g[rank[r]];
      else if (cls[r] == 2 && rank[r] <= moves) dest = rank[r] == 1 ? 0 : L.part.p[rank[r] - 1];
      L.el[dest] = (unsigned short)li[r];
      L.E[dest] = e[r];
    }
    for (int i = id; i < CAP; i += T) L.bound[i] = 0;
    TM::sync();
    // Nbound after the partition; disruption test (:357-379): the original
    // element 0 ends in the last hole (Etmp, :37-38 and :50-51)
    const int nb = n == 0 ? 0 : hole + (L.E[hole] < 0.f ? 1 : 0);
    const bool disrupted = nb < P.min_part;
    if (id == 0) {
      S.nbound = nb;
      S.nsort = 0;
      if (disrupted) {
        S.flags = (S.flags & ~F_ACTIVE) | F_DISR | F_FINAL;
        S.nbound = 1;
        S.nlast = 1;
      }
    }
    if (disrupted) {
      if (S.flags & F_SHUF) {
        // the old most-bound particle back in front (see disrupt_find_kernel)
        int q = INT_MAX;
        for (int l = id; l < S.ulen; l += T)
          if (W.g_id[W.gidx[b + l]] == S.old_mb_id) q = min(q, l);
        if (id == 0) L.K = INT_MAX;
        TM::sync();
        if (q != INT_MAX) atomicMin(&L.K, q);
        TM::sync();
        if (id == 0 && L.K != INT_MAX) swap_entries(W, b, b + L.K);
      }
      n = 0;  // its Elist is not read again
    } else {
      for (int l = id; l < nb; l += T) L.bound[L.el[l]] = 1;
      TM::sync();
      int q[R], keep[R], kept = 0, total;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int l = R * id + r;
        q[r] = l < n ? W.sp[b + l] : 0;
        keep[r] = l < n ? L.bound[q[r]] : 0;
        kept += keep[r];
      }
      int at = TM::exclusive_scan(kept, &total);
      TM::sync();  // the list may be compacted in place
#pragma unroll
      for (int r = 0; r < R; r++)
        if (keep[r]) sp_out[b + at++] = q[r];
      if (P.refine)  // the outputs after a refinement read the flags
        for (int l = id; l < n; l += T) W.isb[b + L.el[l]] = l < nb ? 1 : 0;
    }
    if constexpr ((STAGE & POST_FRAME) != 0) {
      if (!disrupted) {
        const int l0 = L.el[0];
        const float4 p0 = W.pos[b + l0];
        const double o[3] = {p0.x, p0.y, p0.z};
        double v[FRAME_SUMS];
        tile_sums<TM, FRAME_SUMS>(nb, v, L.sums,
                                  [&](int i, double (&x)[FRAME_SUMS]) {
                                    frame_accum(P, W.pos[b + L.el[i]], W.vel[b + L.el[i]], o, x);
                                  });
        if (id == 0) frame_update(W, P, S, l0, v[0], v[1], v[2], v[3], v[4], v[5], v[6]);
      }
    }
    TM::sync();
  }
  if constexpr ((STAGE & POST_SORT) != 0) {
    const int flags = S.flags, nsort = S.nsort, lo = S.sort_lo;
    if constexpr ((STAGE & POST_PART) == 0) {
      if (nsort <= 0 && !(flags & F_FINAL)) return;  // uniform across the team
      if (flags & F_DISR) n = 0;
      for (int l = id; l < n; l += T) {
        const int li = W.el[b + l];
        L.el[l] = (unsigned short)li;
        L.E[l] = W.E[b + li];
      }
      TM::sync();
    }
    // energy sort of Elist[lo, lo + nsort)
    if (nsort > 0) {
      constexpr int BITS = log2_of(CAP);
      u64 x[R];
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int i = R * id + r;
        x[r] = i < nsort ? energy_word<BITS>(lo + i, lo, S.nbound, L.E[lo + i]) : ~0ull;
      }
      if constexpr (T == WAVE) {
        sort_words<R>(x, id, nsort);
      } else {
        sort_tile_words<T>(x, nsort, L.key);
#pragma unroll
        for (int r = 0; r < R; r++) x[r] = L.key[R * id + r];
      }
      unsigned short li[R];
#pragma unroll
      for (int r = 0; r < R; r++)
        if (R * id + r < nsort) li[r] = L.el[lo + (int)(x[r] & (CAP - 1))];
      TM::sync();
#pragma unroll
      for (int r = 0; r < R; r++)
        if (R * id + r < nsort) L.el[lo + R * id + r] = li[r];
      TM::sync();
    }
  }
  for (int l = id; l < n; l += T) W.el[b + l] = L.el[l];
  if constexpr ((STAGE & POST_SORT) != 0) {
    if (S.flags & F_FINAL) {  // uniform across the team
      for (int l = id; l < S.len; l += T) write_entry(W, S, l, output_entry(W, S, l, l < n ? L.el[l] : l < S.ulen ? W.el[b + l] : 0));
      if constexpr ((STAGE & POST_RECORD) != 0) {
        const bool conv = (S.flags & F_CONV) != 0;
        const int nb = S.nbound;
        double v[REC_SUMS];
        tile_sums<TM, REC_SUMS>(record_span(S), v, L.sums, [&](int i, double (&x)[REC_SUMS]) {
          if (!conv || L.bound[i]) record_accum(W, P, S, b, i, nb, nb <= 100, x);
        });
        if (id == 0) write_record_sums(W, P, S, v);
      }
    }
  }
  TM::sync();  // the next tile reuses the LDS
}

// Tiles t0 <= t < ntiles, one team each.
template <int R, int STAGE>
__global__ void __launch_bounds__(BLOCK, 4) post_one_wave_kernel(Work W, DevParams P, const Tile *__restrict__ tiles,
                                                              int t0, int ntiles, int *sp_out) {
  using TM = Team<WAVE, R>;
  __shared__ OnePost<TM::CAP> L[BLOCK / WAVE];
  WAVE_TILE_LOOP(t, t0, ntiles) post_one<TM, STAGE>(W, P, tiles[t], sp_out, L[threadIdx.x / WAVE]);
}
template <int STAGE>
__global__ void __launch_bounds__(BLOCK, 4) post_one_kernel(Work W, DevParams P, const Tile *__restrict__ tiles, int t0,
                                                         int ntiles, int *sp_out) {
  using TM = Team<BLOCK, ITEMS>;
  __shared__ OnePost<TM::CAP> L;
  for (int t = t0 + (int)blockIdx.x; t < ntiles; t += gridDim.x) post_one<TM, STAGE>(W, P, tiles[t], sp_out, L);
}

// The end of a pass: the segments still active and the largest Nlast among them,
// and the setup of their next pass.  A segment that was not active before is not
// read.  Counted by blocks, since atomics on one address are served one after
// another; the last block writes the counts where the host reads them and clears
// them.  Setup, count and copy as three launches took 14 us of a 300-particle
// list's pass of 60.
__global__ void __launch_bounds__(BLOCK) pass_end_kernel(Work W, DevParams P) {
  __shared__ int sh[2][BLOCK / WAVE];
  int cnt = 0, most = 0;
  SEG_LOOP(k, W) {
    if (W.segact[k] == 0) continue;
    Seg &S = W.seg[k];
    const bool active = (S.flags & F_ACTIVE) != 0;
    if (active) {
      cnt++;
      most = max(most, S.nlast);
    }
    W.segact[k] = active ? 1 : 0;
    begin_pass(W, P, S, k);
  }
  for (int d = WAVE / 2; d > 0; d >>= 1) {
    cnt += __shfl_xor(cnt, d, WAVE);
    most = max(most, __shfl_xor(most, d, WAVE));
  }
  if ((threadIdx.x & (WAVE - 1)) == 0) { sh[0][threadIdx.x / WAVE] = cnt; sh[1][threadIdx.x / WAVE] = most; }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < BLOCK / WAVE; w++) {
    cnt += sh[0][w];
    most = max(most, sh[1][w]);
  }
  if (cnt) {
    atomicAdd(&W.active[0], cnt);
    atomicMax(&W.active[1], most);  // bounds every count of the next pass
  }
  __threadfence();
  if (atomicAdd(&W.active[2], 1) != (int)gridDim.x - 1) return;
  __threadfence();
  for (int i = 0; i < 4; i++) {
    if (i == 2) continue;
    W.host_active[i] = __hip_atomic_load(&W.active[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  for (int i = 0; i < 3; i++) __hip_atomic_store(&W.active[i], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __threadfence_system();
}

// ---------------------------------------------------------------------------
// RefineBindingEnergyOrder (src/subhalo_unbind.cpp:234-262), for the segments
// that converged with more bound particles than MaxSampleSize: a tree over the
// first MaxSampleSize entries of the energy-sorted list (full masses), each of
// them a target with its own mass (self term removed) in the final frame,
// then those entries re-ordered by that energy; they keep their unbinding
// energies.  Runs once per level after its passes.

__global__ void refine_setup_kernel(Work W, DevParams P) {
  SEG_LOOP(k, W) {
    Seg &S = W.seg[k];
    const bool on = (S.flags & F_REFPEND) != 0;
    S.flags &= ~(F_CORR | F_SAMP | F_FINAL);
    if (on) S.flags |= F_REFINE;
    S.mf = 1.f;
    S.src_lo = 0;
    S.n_src = on ? P.max_sample : 0;
    S.n_tgt = S.n_src;
    S.nsort = S.n_src;
    S.sort_lo = 0;
    S.n_items = 0;
    for (int j = 0; j < 3; j++) { S.bmin[j] = 0xffffffffu; S.bmax[j] = 0u; }
    W.ncount[NC_SRC * W.nseg + k] = S.n_src;
    W.ncount[NC_SORT * W.nseg + k] = S.n_src;
  }
}

// targets: the entries themselves (their order does not change any result)
__global__ void __launch_bounds__(BLOCK) refine_targets_kernel(Work W) {
  SLOT_LOOP(s, W) {
    int k;
    int l = seg_lane_local(W, s, k);
    if (l < 0) continue;
    const Seg &S = W.seg[k];
    if (!(S.flags & F_REFINE) || l >= S.n_tgt) continue;
    W.sp[s] = W.el[s];
  }
}

// sort keys (refinement energy, position): ties keep the energy order
__global__ void __launch_bounds__(BLOCK) refine_keys_kernel(Work W) {
  SLOT_LOOP(s, W) {
    int k;
    int l = seg_lane_local(W, s, k);
    if (l < 0) continue;
    const Seg &S = W.seg[k];
    if (!(S.flags & F_REFINE) || l >= S.nsort) continue;
    const int li = W.el[s];
    W.k0[s] = ((u64)f2ord(W.Er[S.ibase + li]) << 31) | (u64)(unsigned)l;
    W.v0[s] = (u32)li;
  }
}

__global__ void refine_done_kernel(Work W) {
  SEG_LOOP(k, W) {
    Seg &S = W.seg[k];
    if (!(S.flags & F_REFINE)) continue;
    S.flags = (S.flags & ~(F_REFINE | F_REFPEND)) | F_FINAL;
    S.n_src = S.n_tgt = 0;
  }
}

}  // namespace hbt
