// hbt_props.hpp -- hbt_subhalo_properties: Subhalo_t::CalculateProfileProperties
// and Subhalo_t::CalculateShape (src/subhalo.cpp:242-398) for a batch of
// subhalos after unbinding, on the bound lists resident on the device.
// Included by hbt_unbind.hip.
//
// One segment per subhalo with Nbound > 1.  Of at most a tile:
//   props_one      everything in one pass: distance to the most-bound particle
//                  (PeriodicDistance, src/config_parser.h:143-156), sort by it,
//                  running mass (m_cum, :296-297), first maximum of
//                  m(<r)/max(r, eps) (:299-306), the outermost radius enclosing
//                  200 times the critical density
//                  (Snapshot_t::SphericalOverdensitySize,
//                  src/snapshot.cpp:259-280), RHalf and R2Sigma; the 12 FP64
//                  inertia sums over bound particles 1..Nbound-1 (:355-384)
// Longer ones, per tile:
//   props_tile     distances and masses, the tile sorted, the inertia sums
//   merge levels of the unbinding, segmented FP64 scan of the masses
//   props_elem     the profile of a tile in distance order
// props_combine    per subhalo: tiles in order, outputs
#pragma once

namespace {

struct PropSeg {
  int64_t ibase;    // first slot
  int64_t out_off;  // the caller's out_offset
  int sub;          // record index
  int nb;           // Nbound (> 1)
};

struct PropsArgs {
  const PropSeg *seg;
  int nseg;
  const int64_t *ibase;
  const int *n;  // Nbound per segment
  const hbt_subhalo *subs;
  const int64_t *out_index;
  hbt_properties *props;
  const float *gx, *gy, *gz, *gm;
  u64 *k0, *k1;
  u32 *v0, *v1;
  float *m;      // per slot, list order
  double *cum;   // per slot, distance order: exclusive prefix of the masses
};

constexpr int PROF_PART = 5;   // per tile: v, its position, its radius, SO position, SO mass
constexpr int SHAPE_SUMS = 12;

__device__ __forceinline__ float periodic_distance_f(const DevParams &P, const float c[3], float x,
                                                     float y, float z) {
#pragma clang fp contract(off)
  float d0 = c[0] - x, d1 = c[1] - y, d2 = c[2] - z;
  if (P.periodic) { d0 = nearest_f(d0, P); d1 = nearest_f(d1, P); d2 = nearest_f(d2, P); }
  return sqrtf(d0 * d0 + d1 * d1 + d2 * d2);
}

// 200 times the critical density in comoving units, with the reference's
// float/double promotions (src/snapshot.cpp:268, VirialFactor = 200 at c200).
__device__ __forceinline__ float rho_c200(const DevParams &P) {
#pragma clang fp contract(off)
  const float f = 200.f * P.hz * P.hz;
  return (float)((double)f / 2.0 / (double)P.G * (double)P.a * (double)P.a * (double)P.a);
}

// Nbound <= 1: zero profile and shape (src/subhalo.cpp:262-279, 339-351).
__global__ void props_small_kernel(const hbt_subhalo *subs, int64_t nsub, hbt_properties *props) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nsub; i += (int64_t)gridDim.x * blockDim.x) {
    if (subs[i].nbound > 1) continue;
    hbt_properties &o = props[i];
    o.rmax_comoving = 0.f; o.vmax_physical = 0.f; o.r2sigma_comoving = 0.f; o.rhalf_comoving = 0.f;
    o.bound_r200crit_comoving = 0.f; o.bound_m200crit = 0.f;
    for (int j = 0; j < 6; j++) { o.inertial_tensor[j] = 0.f; o.inertial_tensor_weighted[j] = 0.f; }
  }
}

// scan functors: masses in distance order
struct CumLoad {
  const int64_t *ibase; const u32 *v0; const float *m;
  __device__ double operator()(int k, int l) const {
    const int64_t b = ibase[k];
    return (double)m[b + v0[b + l]];
  }
};
struct CumStore {
  const int64_t *ibase; double *cum;
  __device__ void operator()(int k, int l, double x) const { cum[ibase[k] + l] = x; }
};
struct CumAdd {
  const int64_t *ibase; double *cum;
  __device__ void operator()(int k, int l, double x) const { cum[ibase[k] + l] += x; }
};

// Entry i of a list in distance order: its radius and place are word i.  A word
// orders by distance, then by place, so the place is the sort's value too.
__device__ __forceinline__ u64 radius_word(float rr, int l) { return ((u64)f2ord(rr) << 32) | (u64)(unsigned)l; }
__device__ __forceinline__ float word_radius(u64 w) { return ord2f((unsigned)(w >> 32)); }

// Per tile of a segment in distance order.  v = m(<r)/max(r, eps) with
// m(<r) the float of the FP64 running sum; the first maximum wins (max_element).
// The tile's maxima are folded across lanes (one thread scanning the block's
// 256 candidates took 0.40 of the kernel's 0.49 ms for 5.4 M particles).
__global__ void __launch_bounds__(BLOCK)
props_elem_kernel(PropsArgs A, DevParams P, const Tile *tiles, int ntiles, double *part) {
#pragma clang fp contract(off)
  __shared__ float sv[BLOCK / WAVE], sr[BLOCK / WAVE], sm[BLOCK / WAVE];
  __shared__ int sl[BLOCK / WAVE], so[BLOCK / WAVE];
  const float rho = rho_c200(P);
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const PropSeg &S = A.seg[tl.seg];
    const int cnt = min(TILE, S.nb - tl.start);
    if (cnt <= 0) continue;  // uniform
    const int64_t b = S.ibase;
    float bv = -1.f, br = 0.f, bm = 0.f;
    int bl = INT_MAX, bso = -1;
    for (int i = threadIdx.x; i < cnt; i += BLOCK) {
      const int ls = tl.start + i;
      const int li = (int)A.v0[b + ls];
      float rr = word_radius(A.k0[b + ls]);
      const float mc = (float)(A.cum[b + ls] + (double)A.m[b + li]);
      if (rr < P.eps) rr = P.eps;  // SofteningHalo
      const float v = mc / rr;
      if (v > bv || (v == bv && ls < bl)) { bv = v; bl = ls; br = rr; }
      if (mc > rho * rr * rr * rr && ls > bso) { bso = ls; bm = mc; }
      if (ls == S.nb / 2) A.props[S.sub].rhalf_comoving = rr;
      if (ls == (int)((int64_t)S.nb * 0.955)) A.props[S.sub].r2sigma_comoving = rr;
    }
    auto take = [&](float v, int l, float r, int o, float m) {
      if (v > bv || (v == bv && l < bl)) { bv = v; bl = l; br = r; }
      if (o > bso) { bso = o; bm = m; }
    };
    for (int d = WAVE / 2; d > 0; d >>= 1)
      take(__shfl_xor(bv, d, WAVE), __shfl_xor(bl, d, WAVE), __shfl_xor(br, d, WAVE), __shfl_xor(bso, d, WAVE),
           __shfl_xor(bm, d, WAVE));
    if ((threadIdx.x & (WAVE - 1)) == 0) {
      const int w = threadIdx.x / WAVE;
      sv[w] = bv; sl[w] = bl; sr[w] = br; so[w] = bso; sm[w] = bm;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < BLOCK / WAVE; w++) take(sv[w], sl[w], sr[w], so[w], sm[w]);
      double *p = part + (int64_t)t * PROF_PART;
      p[0] = bv; p[1] = bl; p[2] = br; p[3] = bso; p[4] = bm;
    }
    __syncthreads();
  }
}

// Adds the products of an entry at (dx, dy, dz) with mass m (dr2 its squared
// distance) to the inertia sums.
__device__ __forceinline__ void add_shape(double (&v)[SHAPE_SUMS], float dx, float dy, float dz, float dr2, float m) {
#pragma clang fp contract(off)
  const float dx2 = dx * dx, dy2 = dy * dy, dz2 = dz * dz;
  v[0] += dx2 * m; v[1] += dx * dy * m; v[2] += dx * dz * m;
  v[3] += dy2 * m; v[4] += dy * dz * m; v[5] += dz2 * m;
  dr2 /= m;
  v[6] += dx2 / dr2; v[7] += dx * dy / dr2; v[8] += dx * dz / dr2;
  v[9] += dy2 / dr2; v[10] += dy * dz / dr2; v[11] += dz2 / dr2;
}

// One tile of a longer bound list: distance to the most-bound particle and mass
// of each entry, the tile's entries sorted by distance (into the buffer from
// which the list's merge levels end in (k0, v0)), and the inertia sums of
// particles 1..Nbound-1 in list order.  The four scattered column reads bound
// it; the distances and the sums share them, and the sort takes the distances
// out of LDS (3.7 M entries 0.28 ms; with the sort of pairs in a launch of its
// own 5.4 M took 0.43 + 0.17).
__global__ void __launch_bounds__(BLOCK)
props_tile_kernel(PropsArgs A, DevParams P, const Tile *tiles, int ntiles, double *part) {
#pragma clang fp contract(off)
  __shared__ double sh[SHAPE_SUMS][BLOCK / WAVE];
  __shared__ u64 sk[TILE];
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const PropSeg &S = A.seg[tl.seg];
    const int cnt = min(TILE, S.nb - tl.start);
    if (cnt <= 0) continue;  // uniform
    const float *c = A.subs[S.sub].mostbound_pos;
    const float c0 = c[0], c1 = c[1], c2 = c[2];
    double v[SHAPE_SUMS];
    for (int q = 0; q < SHAPE_SUMS; q++) v[q] = 0.;
    constexpr int PER = TILE / BLOCK;
    int64_t g[PER];
    float gx[PER], gy[PER], gz[PER], gm[PER];
    // the tile's reads in two batches (past its end the last entry again)
#pragma unroll
    for (int k = 0; k < PER; k++) g[k] = A.out_index[S.out_off + tl.start + min((int)threadIdx.x + k * BLOCK, cnt - 1)];
#pragma unroll
    for (int k = 0; k < PER; k++) { gx[k] = A.gx[g[k]]; gy[k] = A.gy[g[k]]; gz[k] = A.gz[g[k]]; gm[k] = A.gm[g[k]]; }
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int i = (int)threadIdx.x + k * BLOCK;
      sk[i] = ~0ull;
      if (i >= cnt) continue;
      const int l = tl.start + i;
      const float m = gm[k];
      float dx = gx[k] - c0, dy = gy[k] - c1, dz = gz[k] - c2;
      if (P.periodic) { dx = nearest_f(dx, P); dy = nearest_f(dy, P); dz = nearest_f(dz, P); }
      const float dr2 = dx * dx + dy * dy + dz * dz;
      const float rr = sqrtf(dr2);  // PeriodicDistance (src/config_parser.h:143-156)
      A.m[S.ibase + l] = m;
      sk[i] = radius_word(rr, l);
      if (l > 0) add_shape(v, dx, dy, dz, dr2, m);
    }
    for (int q = 0; q < SHAPE_SUMS; q++) {
      const double r = wave_reduce_sum(v[q]);
      if ((threadIdx.x & (WAVE - 1)) == 0) sh[q][threadIdx.x / WAVE] = r;
    }
    __syncthreads();
    if (threadIdx.x < SHAPE_SUMS) {
      double r = 0;
      for (int w = 0; w < BLOCK / WAVE; w++) r += sh[threadIdx.x][w];
      part[(int64_t)t * SHAPE_SUMS + threadIdx.x] = r;
    }
    u64 x[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) x[r] = sk[ITEMS * threadIdx.x + r];
    __syncthreads();
    sort_tile_words<BLOCK>(x, cnt, sk);
    const bool odd = (merge_levels(S.nb, TILE) & 1) != 0;
    u64 *kout = odd ? A.k1 : A.k0;
    u32 *vout = odd ? A.v1 : A.v0;
    const int64_t s = S.ibase + tl.start;
    for (int i = threadIdx.x; i < cnt; i += BLOCK) { kout[s + i] = sk[i]; vout[s + i] = (u32)sk[i]; }
    __syncthreads();
  }
}

// Lists of at most R T entries: distances, sort, running mass, profile and
// shape without a store in between, by one wave (R T of 64 or 256) or one
// workgroup (1,024).  Thread i holds the entries R i .. R i + R - 1, before the
// sort of the list's order and after it of the distances'.  The scattered reads
// bound it, and for the shortest lists the reductions.  19,400 lists of up to a
// tile among 20,000 (1.7 M entries): 41 us for those of one lane an entry, 55 and
// 65 for the longer classes; through the tiles' launches a list of 43 entries
// kept a workgroup in each of five.  The call with its host part 2.59 -> 2.10 ms.
template <int R, int T>
__global__ void __launch_bounds__(BLOCK)
props_one_kernel(PropsArgs A, DevParams P, const Tile *tiles, int ntiles, double *prof_part, double *shape_part) {
#pragma clang fp contract(off)
  constexpr int GROUPS = BLOCK / T, NW = T / WAVE;
  __shared__ float smass[R > 1 ? GROUPS : 1][R > 1 ? R * T : 1];
  __shared__ u64 sk[T > WAVE ? R * T : 1];
  __shared__ double sh[T > WAVE ? SHAPE_SUMS : 1][NW];
  __shared__ float sv[NW], sr[NW], som[NW];
  __shared__ int so[NW];
  const float rho = rho_c200(P);
  const int id = threadIdx.x % T, grp = threadIdx.x / T, lane = threadIdx.x & (WAVE - 1);
  for (int t = blockIdx.x * GROUPS + grp; t < ntiles; t += gridDim.x * GROUPS) {  // uniform across T threads
    const PropSeg &S = A.seg[tiles[t].seg];
    const int cnt = S.nb;
    const float *c = A.subs[S.sub].mostbound_pos;
    const float c0 = c[0], c1 = c[1], c2 = c[2];
    double v[SHAPE_SUMS];
    for (int q = 0; q < SHAPE_SUMS; q++) v[q] = 0.;
    int64_t g[R];
    float gx[R], gy[R], gz[R], gm[R];
#pragma unroll
    for (int r = 0; r < R; r++) g[r] = A.out_index[S.out_off + min(R * id + r, cnt - 1)];
#pragma unroll
    for (int r = 0; r < R; r++) { gx[r] = A.gx[g[r]]; gy[r] = A.gy[g[r]]; gz[r] = A.gz[g[r]]; gm[r] = A.gm[g[r]]; }
    u64 x[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int l = R * id + r;
      x[r] = ~0ull;
      if (R > 1) smass[R > 1 ? grp : 0][R > 1 ? l : 0] = gm[r];
      if (l >= cnt) continue;
      float dx = gx[r] - c0, dy = gy[r] - c1, dz = gz[r] - c2;
      if (P.periodic) { dx = nearest_f(dx, P); dy = nearest_f(dy, P); dz = nearest_f(dz, P); }
      const float dr2 = dx * dx + dy * dy + dz * dz;
      x[r] = radius_word(sqrtf(dr2), l);
      if (l > 0) add_shape(v, dx, dy, dz, dr2, gm[r]);
    }
    double mine = 0;  // lane q: sum q
    for (int q = 0; q < SHAPE_SUMS; q++) {
      const double s = wave_total(v[q]);
      if (lane == q) mine = s;
    }
    if constexpr (T > WAVE) {
      if (lane < SHAPE_SUMS) sh[lane][threadIdx.x / WAVE] = mine;
      sort_tile_words<T>(x, cnt, sk);  // its barriers also cover sh and smass
#pragma unroll
      for (int r = 0; r < R; r++) x[r] = sk[R * id + r];
      if (id < SHAPE_SUMS) {
        mine = 0;
        for (int w = 0; w < NW; w++) mine += sh[id][w];
      }
    } else {
      sort_words<R>(x, lane, cnt);
      wave_sync();
    }
    if (id < SHAPE_SUMS) shape_part[(int64_t)t * SHAPE_SUMS + id] = mine;
    // masses in distance order and their running sum
    float m[R];
    double sum = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
      if constexpr (R > 1) m[r] = R * id + r < cnt ? smass[grp][(u32)x[r]] : 0.f;
      else {
        m[r] = __shfl(gm[0], (int)(u32)x[0] & (WAVE - 1), WAVE);
        if (id >= cnt) m[r] = 0.f;
      }
      sum += (double)m[r];
    }
    double off, all;
    if constexpr (T > WAVE) off = block_exclusive_scan(sum, &all);
    else off = wave_inclusive_scan(sum) - sum;
    float bv = -1.f, br = 0.f, bm = 0.f;
    int bso = -1;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int ls = R * id + r;
      const float mc = (float)(off + (double)m[r]);
      off += (double)m[r];
      if (ls >= cnt) continue;
      float rr = word_radius(x[r]);
      if (rr < P.eps) rr = P.eps;  // SofteningHalo
      const float vv = mc / rr;
      if (vv > bv) { bv = vv; br = rr; }
      if (mc > rho * rr * rr * rr) { bso = ls; bm = mc; }
      if (ls == cnt / 2) A.props[S.sub].rhalf_comoving = rr;
      if (ls == (int)((int64_t)cnt * 0.955)) A.props[S.sub].r2sigma_comoving = rr;
    }
    // the first of the largest: the lowest lane that holds the maximum
    float top = bv;
    for (int d = WAVE / 2; d > 0; d >>= 1) top = fmaxf(top, __shfl_xor(top, d, WAVE));
    const int first = __ffsll((unsigned long long)__ballot(bv == top)) - 1;
    br = __shfl(br, first, WAVE);
    const unsigned long long in = __ballot(bso >= 0);
    const int last = in ? 63 - __clzll((long long)in) : 0;
    bso = __shfl(bso, last, WAVE);
    bm = __shfl(bm, last, WAVE);
    if constexpr (T > WAVE) {
      const int w = threadIdx.x / WAVE;
      if (lane == 0) { sv[w] = top; sr[w] = br; so[w] = bso; som[w] = bm; }
      __syncthreads();
      for (int u = 0; u < NW; u++) {
        if (u == 0 || sv[u] > top) { top = sv[u]; br = sr[u]; }
        if (u == 0 || so[u] >= 0) { bso = so[u]; bm = som[u]; }
      }
      __syncthreads();
    } else {
      wave_sync();
    }
    if (id == 0) {
      double *p = prof_part + (int64_t)t * PROF_PART;
      p[0] = top; p[1] = 0; p[2] = br; p[3] = bso; p[4] = bm;
    }
  }
}

__global__ void __launch_bounds__(BLOCK) props_combine_kernel(PropsArgs A, DevParams P, const int *first_tile,
                                     const double *prof_part, const double *shape_part) {
#pragma clang fp contract(off)
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < A.nseg; k += gridDim.x * blockDim.x) {
    const PropSeg &S = A.seg[k];
    const hbt_subhalo &h = A.subs[S.sub];
    hbt_properties &o = A.props[S.sub];
    const int t0 = first_tile[k], nt = (S.nb + TILE - 1) / TILE;
    double v = -1., rr = 0., mso = 0.;
    int lso = -1;
    double sums[SHAPE_SUMS];
    for (int q = 0; q < SHAPE_SUMS; q++) sums[q] = 0.;
    // tiles in order (the first maximum stays; the sums keep their order);
    // PREF tiles are loaded ahead of their use, so a subhalo of thousands of
    // tiles does not wait for each load in turn
    constexpr int PREF = 4;
    int t = t0;
    for (; t + PREF <= t0 + nt; t += PREF) {
      double pv[PREF], pr[PREF], pl[PREF], pm[PREF], sp[PREF][SHAPE_SUMS];
#pragma unroll
      for (int u = 0; u < PREF; u++) {
        const double *p = prof_part + (int64_t)(t + u) * PROF_PART;
        pv[u] = p[0]; pr[u] = p[2]; pl[u] = p[3]; pm[u] = p[4];
#pragma unroll
        for (int q = 0; q < SHAPE_SUMS; q++) sp[u][q] = shape_part[(int64_t)(t + u) * SHAPE_SUMS + q];
      }
#pragma unroll
      for (int u = 0; u < PREF; u++) {
        if (pv[u] > v) { v = pv[u]; rr = pr[u]; }
        if ((int)pl[u] > lso) { lso = (int)pl[u]; mso = pm[u]; }
#pragma unroll
        for (int q = 0; q < SHAPE_SUMS; q++) sums[q] += sp[u][q];
      }
    }
    for (; t < t0 + nt; t++) {
      const double *p = prof_part + (int64_t)t * PROF_PART;
      if (p[0] > v) { v = p[0]; rr = p[2]; }
      if ((int)p[3] > lso) { lso = (int)p[3]; mso = p[4]; }
      for (int q = 0; q < SHAPE_SUMS; q++) sums[q] += shape_part[(int64_t)t * SHAPE_SUMS + q];
    }
    const float vel_unit = P.G / P.a;
    o.rmax_comoving = (float)rr;
    o.vmax_physical = sqrtf((float)v * vel_unit);
    if (lso >= 0) {
      const float rho = rho_c200(P);
      o.bound_m200crit = (float)mso;
      o.bound_r200crit_comoving = (float)pow((double)((float)mso / rho), 1.0 / 3);
    }
    if (o.vmax_physical >= o.last_max_vmax_physical) {
      o.snapshot_index_of_last_max_vmax = P.snap;
      o.last_max_vmax_physical = o.vmax_physical;
    }
    for (int j = 0; j < 6; j++) {  // {xx, xy, xz, yy, yz, zz}, then divided by Mbound
      float a = (float)sums[j];
      a /= h.mbound;
      o.inertial_tensor[j] = a;
      float w = (float)sums[6 + j];
      w /= h.mbound;
      o.inertial_tensor_weighted[j] = w;
    }
  }
}

}  // namespace

extern "C" int hbt_subhalo_properties(hbt_ctx *ctx, const hbt_particles *particles,
                                      const hbt_subhalo *subs, int64_t nsub, const int64_t *out_index,
                                      hbt_properties *props) {
  if (!ctx || !particles || nsub < 0 || (nsub > 0 && (!subs || !out_index || !props)))
    return fail(HBT_ERR_INVALID_ARG, "bad argument");
  if (nsub == 0) return HBT_OK;
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  std::vector<hbt_subhalo> rec(nsub);
  HIPCHK(hipMemcpyAsync(rec.data(), subs, nsub * sizeof(hbt_subhalo), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  // segments: subhalos with Nbound > 1
  std::vector<PropSeg> seg;
  std::vector<int64_t> ibase;
  std::vector<int> first_tile, nb;
  std::vector<Tile> tiles, one[3];  // of longer lists; lists of at most a wave, four, a tile
  int64_t off = 0;
  int maxn = 0;
  for (int64_t i = 0; i < nsub; i++) {
    const int64_t n = rec[i].nbound;
    if (n <= 1) continue;
    if (n >= (int64_t)INT32_MAX / 2 || rec[i].out_offset < 0)
      return fail(HBT_ERR_INVALID_ARG, "bad nbound or out_offset");
    const int k = (int)seg.size();
    seg.push_back(PropSeg{off, rec[i].out_offset, (int)i, (int)n});
    ibase.push_back(off);
    nb.push_back((int)n);
    first_tile.push_back((int)tiles.size());
    if (n <= TILE) {
      one[n <= TINY_CAP ? 0 : n <= SMALL_CAP ? 1 : 2].push_back(Tile{k, 0});
      continue;
    }
    const int nt = (int)((n + TILE - 1) / TILE);
    for (int t = 0; t < nt; t++) tiles.push_back(Tile{k, t * TILE});
    off += (n + WAVE - 1) / WAVE * WAVE;
    maxn = std::max(maxn, (int)n);
  }
  const int nmulti = (int)tiles.size();
  for (const auto &list : one)
    for (const Tile &tl : list) {
      first_tile[tl.seg] = (int)tiles.size();
      tiles.push_back(tl);
    }
  const DevParams P = make_dev_params(ctx->params);
  props_small_kernel<<<grid_for(nsub, ctx->cus), BLOCK, 0, st>>>(subs, nsub, props);
  if (seg.empty()) {
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(st));
    return HBT_OK;
  }
  const int nseg = (int)seg.size(), ntiles = (int)tiles.size();
  RETCHK(ensure_slots(ctx, off, nseg, ntiles));
  void *d[5];
  RETCHK(stage_blobs(ctx, {{seg.data(), seg.size() * sizeof(PropSeg)},
                           {ibase.data(), ibase.size() * 8},
                           {first_tile.data(), first_tile.size() * 4},
                           {nb.data(), nb.size() * 4},
                           {tiles.data(), tiles.size() * sizeof(Tile)}},
                     d));
  PropsArgs A{};
  A.seg = (const PropSeg *)d[0];
  A.nseg = nseg;
  A.ibase = (const int64_t *)d[1];
  A.n = (const int *)d[3];
  A.subs = subs;
  A.out_index = out_index;
  A.props = props;
  A.gx = particles->x; A.gy = particles->y; A.gz = particles->z; A.gm = particles->mass;
  A.k0 = ctx->k0.as<u64>(); A.k1 = ctx->k1.as<u64>();
  A.v0 = ctx->v0.as<u32>(); A.v1 = ctx->v1.as<u32>();
  A.m = ctx->Er.as<float>();
  A.cum = (double *)ctx->scan64.as<u64>();
  const Tile *dt = (const Tile *)d[4];
  const auto grid = [&](int64_t blocks, int per_cu) {
    return (int)std::max<int64_t>(1, std::min<int64_t>(blocks, (int64_t)ctx->cus * per_cu));
  };
  double *prof_part = ctx->tpart.as<double>();
  double *shape_part = prof_part + (size_t)(ntiles + 1) * PROF_PART;
  if (nmulti > 0) {
    const int gt = grid(nmulti, 8), gm = grid((int64_t)nmulti * (TILE / BLOCK), 16);
    props_tile_kernel<<<gt, BLOCK, 0, st>>>(A, P, dt, nmulti, shape_part);
    int level = 0;
    for (int64_t w = TILE; w < maxn; w *= 2, level++)
      merge_pass_kernel<<<gm, BLOCK, 0, st>>>(dt, nmulti, A.ibase, A.n, TILE, level, A.k0, A.v0, A.k1, A.v1);
    // running mass in distance order
    double *ts = (double *)ctx->tsum.as<u64>();
    scan_tiles_kernel<double><<<gt, BLOCK, 0, st>>>(dt, nmulti, A.n, ts, CumLoad{A.ibase, A.v0, A.m},
                                                    CumStore{A.ibase, A.cum});
    scan_add_kernel<double><<<gt, BLOCK, 0, st>>>(dt, nmulti, A.n, ts, CumAdd{A.ibase, A.cum});
    props_elem_kernel<<<gt, BLOCK, 0, st>>>(A, P, dt, nmulti, prof_part);
  }
  const auto lists = [&](auto kernel, int t0, const std::vector<Tile> &list, int per_block) {
    const int n = (int)list.size();
    if (n > 0)
      kernel<<<grid((n + per_block - 1) / per_block, 8), BLOCK, 0, st>>>(
          A, P, dt + t0, n, prof_part + (size_t)t0 * PROF_PART, shape_part + (size_t)t0 * SHAPE_SUMS);
    return t0 + n;
  };
  int t0 = lists(props_one_kernel<1, WAVE>, nmulti, one[0], BLOCK / WAVE);
  t0 = lists(props_one_kernel<SMALL_CAP / WAVE, WAVE>, t0, one[1], BLOCK / WAVE);
  lists(props_one_kernel<ITEMS, BLOCK>, t0, one[2], 1);
  props_combine_kernel<<<grid_for(nseg, ctx->cus), BLOCK, 0, st>>>(A, P, (const int *)d[2], prof_part, shape_part);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(st));
  return HBT_OK;
}
