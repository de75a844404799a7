// hbt_direct.hpp -- hbt_direct_potential: exact pair sums with the walk's
// softened kernel (src/gravity_tree.cpp:144-160), self term excluded, for
// groups of particles (one group per subhalo).  Sources are staged through
// LDS in tiles of BLOCK particles; each thread owns one target.
// Modes: FP32, FP32 with Kahan-compensated sums, FP64.  Included by
// hbt_unbind.hip.
#pragma once

namespace {

struct DTile { int64_t seg_lo, seg_hi, tgt0; };

// 1 / sqrt(x) in double: the hardware's estimate and one third-order step,
// within an ulp or two of the rounded value (x: finite, not 0).  A division
// and a square root by the compiler take about four times the instructions.
__device__ __forceinline__ double rsqrt_d(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-(x * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}

// One staged source: float4, or its values in double.
struct Src64 { double x, y, z, m; };
template <int MODE> struct SrcOf { using type = float4; };
template <> struct SrcOf<HBT_DIRECT_FP64> { using type = Src64; };

// The sum over one target's pairs.  FP32: one sum (compensated or plain), term
// by term in source order.  FP64: four sums taken in turn.
template <int MODE>
struct PairSum {
  using real = float;
  Kahan<MODE == HBT_DIRECT_FP32_KAHAN> acc;
  float h2, hinv;
  __device__ __forceinline__ void init(const DevParams &P) {
    const float h = 2.8f * P.eps;
    h2 = h * h;
    hinv = 1.0f / h;
    acc.init(0.f);
  }
  template <bool WRAP>
  __device__ __forceinline__ float sep2(const DevParams &P, const float4 &s, float tx, float ty, float tz) const {
    float dx = s.x - tx, dy = s.y - ty, dz = s.z - tz;
    if (WRAP) { dx = nearest_f(dx, P); dy = nearest_f(dy, P); dz = nearest_f(dz, P); }
    return pair_r2(dx, dy, dz);
  }
  __device__ __forceinline__ bool near(float r2) const { return !(r2 >= h2); }
  __device__ __forceinline__ float far_term(const float4 &s, float r2) const {
#pragma clang fp contract(off)
    return -s.w * __builtin_amdgcn_rsqf(r2);
  }
  __device__ __forceinline__ float near_term(const float4 &s, float r2) const { return kernel_term_f(s.w, r2, h2, hinv); }
  __device__ __forceinline__ void add(int, float t) { acc.add(t); }
  __device__ __forceinline__ double result() const { return (double)acc.s; }
};

template <>
struct PairSum<HBT_DIRECT_FP64> {
  using real = double;
  double acc[4], h, hinv, h2;
  __device__ __forceinline__ void init(const DevParams &P) {
    h = 2.8 * (double)P.eps;
    hinv = 1.0 / h;
    h2 = h * h;
    for (int k = 0; k < 4; k++) acc[k] = 0.0;
  }
  template <bool WRAP>
  __device__ __forceinline__ double sep2(const DevParams &P, const Src64 &s, double tx, double ty, double tz) const {
    double dx = s.x - tx, dy = s.y - ty, dz = s.z - tz;
    if (WRAP) { dx = nearest_d(dx, P); dy = nearest_d(dy, P); dz = nearest_d(dz, P); }
    return __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
  }
  __device__ __forceinline__ bool near(double r2) const { return !(r2 >= h2); }
  // (an infinite r2 has no term: the largest finite ones stand in for it)
  __device__ __forceinline__ double far_term(const Src64 &s, double r2) const {
    return -s.m * rsqrt_d(__builtin_fmin(r2, 1e300));
  }
  __device__ __forceinline__ double near_term(const Src64 &s, double r2) const {
    return kernel_term_d(s.m, sqrt(r2), h, hinv);
  }
  __device__ __forceinline__ void add(int k, double t) { acc[k] += t; }
  __device__ __forceinline__ double result() const { return (acc[0] + acc[1]) + (acc[2] + acc[3]); }
};

// Smallest and largest of x over the wave, in every lane.
__device__ __forceinline__ void wave_min_max(float &mn, float &mx) {
  for (int d = WAVE / 2; d > 0; d >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, d, WAVE));
    mx = fmaxf(mx, __shfl_xor(mx, d, WAVE));
  }
}

// The pairs of the sources src(0) .. src(nj - 1) with this lane's target; `self` is
// the target's own place among them (left out), or outside [0, nj).  K pairs at
// a time; the spline only where a lane of the wave is inside the softening
// length, behind one scalar branch for the K.
template <int K, int MODE, bool WRAP, bool SELF, class Real, class Source>
__device__ __forceinline__ void direct_pairs(PairSum<MODE> &sum, const DevParams &P, Source src, int q, int self,
                                             Real tx, Real ty, Real tz) {
  typename SrcOf<MODE>::type s[K];
  Real r2[K], t[K];
  bool close[K];
  u64 near = 0;
#pragma unroll
  for (int k = 0; k < K; k++) {
    s[k] = src(q + k);
    r2[k] = sum.template sep2<WRAP>(P, s[k], tx, ty, tz);
    t[k] = sum.far_term(s[k], r2[k]);
    close[k] = sum.near(r2[k]) && !(SELF && q + k == self);  // (the target is its own nearest)
    near |= __ballot(close[k]);
  }
  if (near != 0ull) {
#pragma unroll
    for (int k = 0; k < K; k++)
      if (close[k]) t[k] = sum.near_term(s[k], r2[k]);
  }
#pragma unroll
  for (int k = 0; k < K; k++)
    if (!SELF || q + k != self) sum.add((q + k) & 3, t[k]);
}

template <int MODE, bool WRAP, bool SELF, class Real, class Source>
__device__ __forceinline__ void direct_chunk(PairSum<MODE> &sum, const DevParams &P, Source src, int nj, int self,
                                             Real tx, Real ty, Real tz) {
  int q = 0;
  for (; q + 4 <= nj; q += 4) direct_pairs<4, MODE, WRAP, SELF, Real>(sum, P, src, q, self, tx, ty, tz);
  for (; q < nj; q++) direct_pairs<1, MODE, WRAP, SELF, Real>(sum, P, src, q, self, tx, ty, tz);
}

// The groups of at most a wave's particles, one to a wave: a particle to a lane,
// the sources read from the lanes.  The wrap is left out where every particle lies
// within a quarter box of the first (then no pair is half a box apart, and the
// selects change nothing).  20,000 groups of 5 take 45 us a call in FP32 and 68 in
// FP64, 20,000 of 20 69 and 110; as tiles, three of four waves idle and the boxes of
// targets and sources to find for each, 98 to 127 and 159 to 189, 122 to 144 and 220
// to 255.
template <int MODE>
__device__ __forceinline__ void direct_small(const int64_t *__restrict__ seg_offset, int64_t nseg, const float *x,
                                             const float *y, const float *z, const float *m, const DevParams &P,
                                             double *out) {
  using Real = typename PairSum<MODE>::real;
  using Src = typename SrcOf<MODE>::type;
  const int lane = threadIdx.x & (WAVE - 1);
  const int64_t waves = (int64_t)gridDim.x * (BLOCK / WAVE);
  for (int64_t s = (int64_t)blockIdx.x * (BLOCK / WAVE) + threadIdx.x / WAVE; s < nseg; s += waves) {  // uniform across the wave
    const int64_t lo = seg_offset[s], len = seg_offset[s + 1] - lo;
    if (len <= 0 || len > WAVE) continue;
    const int n = __builtin_amdgcn_readfirstlane((int)len);
    const int64_t i = lo + min(lane, n - 1);
    const float px = x[i], py = y[i], pz = z[i], pm = m[i];
    const auto lane_of = [](float v, int q) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), q)); };
    const auto src = [&](int q) { return Src{lane_of(px, q), lane_of(py, q), lane_of(pz, q), lane_of(pm, q)}; };
    const float near = 0.5f * P.box_half * (1.f - 1e-6f);
    const bool inside = fabsf(px - lane_of(px, 0)) <= near && fabsf(py - lane_of(py, 0)) <= near &&
                        fabsf(pz - lane_of(pz, 0)) <= near;
    PairSum<MODE> sum;
    sum.init(P);
    if (P.periodic && __any(!inside)) direct_chunk<MODE, true, true, Real>(sum, P, src, n, lane, px, py, pz);
    else direct_chunk<MODE, false, true, Real>(sum, P, src, n, lane, px, py, pz);
    if (lane < n) out[i] = sum.result() * (double)P.G / (double)P.a;
  }
}

template <int MODE>
__global__ void __launch_bounds__(BLOCK)
direct_small_kernel(const int64_t *__restrict__ seg_offset, int64_t nseg, const float *x, const float *y, const float *z,
                    const float *m, DevParams P, double *out) {
  direct_small<MODE>(seg_offset, nseg, x, y, z, m, P, out);
}

// One tile of targets (BLOCK consecutive particles of a group) against every
// particle of its group; the workgroup stages the sources through sh.  The
// wrap's selects and the test for the target itself would cost as much as a
// pair's arithmetic: a wave wraps only against chunks that reach more than
// half a box from one of its targets (boxes of its targets and of the chunk:
// differences are monotonic, so the decision is exact), and looks for itself
// only in chunks that hold it.  Vector issue bounds it: 1.25e9 pairs of 600
// groups (20 to 4,700 particles, periodic) take 0.47 ms in FP32, 0.54 compensated
// and 1.03 in FP64, where tests and wrap in every pair, a branch for its spline
// and FP64 by division and root took 1.64, 1.62 and 3.23.
template <int MODE>
__device__ __forceinline__ void direct_tile(const DTile T, const float *x, const float *y, const float *z,
                                            const float *m, const DevParams &P, double *out,
                                            typename SrcOf<MODE>::type *sh) {
  using Real = typename PairSum<MODE>::real;
  const int64_t i = T.tgt0 + threadIdx.x;
  const bool live = i < T.seg_hi;
  const int64_t w0 = T.tgt0 + (int64_t)(threadIdx.x & ~(WAVE - 1));  // the wave's first target
  const bool busy = w0 < T.seg_hi;
  const int64_t it = live ? i : T.seg_lo;
  const Real tx = x[it], ty = y[it], tz = z[it];
  float b0[3], b1[3];  // box of the wave's targets
  if (P.periodic) {
    // (lanes without a target stand at the group's first particle: a larger box only)
    const float t[3] = {(float)tx, (float)ty, (float)tz};
    for (int j = 0; j < 3; j++) { b0[j] = b1[j] = t[j]; wave_min_max(b0[j], b1[j]); }
  }
  PairSum<MODE> sum;
  sum.init(P);
  for (int64_t j0 = T.seg_lo; j0 < T.seg_hi; j0 += BLOCK) {
    const int nj = (int)min<int64_t>(BLOCK, T.seg_hi - j0);
    if ((int)threadIdx.x < nj) {
      const int64_t j = j0 + threadIdx.x;
      sh[threadIdx.x] = {x[j], y[j], z[j], m[j]};
    }
    __syncthreads();
    if (busy) {  // uniform across the wave
      bool wrap = false;
      if (P.periodic) {
        float c0[3], c1[3];
        bool nan = false;
        for (int k = 0; k < BLOCK / WAVE; k++) {
          const auto s = sh[min((int)(threadIdx.x & (WAVE - 1)) + k * WAVE, nj - 1)];
          const float v[3] = {(float)s.x, (float)s.y, (float)s.z};
          for (int j = 0; j < 3; j++) {
            nan = nan || v[j] != v[j];
            c0[j] = k ? fminf(c0[j], v[j]) : v[j];
            c1[j] = k ? fmaxf(c1[j], v[j]) : v[j];
          }
        }
        for (int j = 0; j < 3; j++) {
          wave_min_max(c0[j], c1[j]);
          wrap = wrap || !((Real)c1[j] - (Real)b0[j] <= (Real)P.box_half && (Real)b1[j] - (Real)c0[j] <= (Real)P.box_half);
        }
        nan = nan || tx != tx || ty != ty || tz != tz;  // (a minimum passes over one)
        wrap = __any(nan || wrap);
      }
      const auto src = [sh](int q) { return sh[q]; };
      const bool self = j0 < w0 + WAVE && w0 < j0 + nj;
      const int own = live ? (int)min<int64_t>(i - j0, BLOCK) : BLOCK;
      if (wrap) {
        if (self) direct_chunk<MODE, true, true, Real>(sum, P, src, nj, own, tx, ty, tz);
        else direct_chunk<MODE, true, false, Real>(sum, P, src, nj, own, tx, ty, tz);
      } else {
        if (self) direct_chunk<MODE, false, true, Real>(sum, P, src, nj, own, tx, ty, tz);
        else direct_chunk<MODE, false, false, Real>(sum, P, src, nj, own, tx, ty, tz);
      }
    }
    __syncthreads();
  }
  if (live) out[i] = sum.result() * (double)P.G / (double)P.a;
}

template <int MODE>
__global__ void __launch_bounds__(BLOCK)
direct_kernel(const DTile *tiles, int ntiles, const int64_t *__restrict__ seg_offset, int64_t nseg, const float *x,
              const float *y, const float *z, const float *m, DevParams P, double *out) {
  __shared__ typename SrcOf<MODE>::type sh[BLOCK];
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) direct_tile<MODE>(tiles[t], x, y, z, m, P, out, sh);
  direct_small<MODE>(seg_offset, nseg, x, y, z, m, P, out);
}

// ---- the entry point that allocates nothing ---------------------------------
// Its scratch -- the first tile of every group and the tile total, then a flag
// for offsets that are not ascending -- lives in this file-scope device array.
// Each GPU holds its own copy until the process ends; host code reaches it only
// through the address hipGetSymbolAddress gives for the device (the array's
// name in host code is not a device address).
constexpr int64_t NOALLOC_MAX_GROUPS = 65536;
static __device__ __align__(256) int64_t scratch[NOALLOC_MAX_GROUPS + 2];

constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};

// Once per device, with that device current (hbt_ctx_create).
int noalloc_scratch_setup(int device) {
  if (device < 0 || device >= NOALLOC_MAX_DEVICES) return fail(HBT_ERR_UNSUPPORTED, "device index above 63");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return HBT_OK;
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr)
    return fail(HBT_ERR_DEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  g_scratch_ptr[device] = ptr;
  return HBT_OK;
}

// First tile of every group of more than a wave's particles (ceil(len / BLOCK)
// tiles each, an exclusive scan in one workgroup), the total at tstart[nseg], and *bad = 1 when a group's
// offsets descend (such a group gets no tiles).
__global__ void __launch_bounds__(BLOCK) direct_tile_starts_kernel(const int64_t *__restrict__ seg_offset,
                                                                   int64_t nseg, int64_t *tstart, int *bad) {
  __shared__ int sbad;
  if (threadIdx.x == 0) sbad = 0;
  __syncthreads();
  int64_t run = 0;
  for (int64_t s0 = 0; s0 < nseg; s0 += BLOCK) {  // uniform across the block
    const int64_t s = s0 + threadIdx.x;
    int64_t nt = 0;
    if (s < nseg) {
      const int64_t len = seg_offset[s + 1] - seg_offset[s];
      if (len < 0) atomicOr(&sbad, 1);
      nt = len > WAVE ? (len + BLOCK - 1) / BLOCK : 0;  // (direct_small takes the others)
    }
    unsigned long long tot;
    const unsigned long long ex = block_exclusive_scan((unsigned long long)nt, &tot);
    if (s < nseg) tstart[s] = run + (int64_t)ex;
    run += (int64_t)tot;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    tstart[nseg] = run;
    *bad = sbad;
  }
}

// Tile t belongs to the last group whose first tile is at or before it.
template <int MODE>
__global__ void __launch_bounds__(BLOCK)
direct_noalloc_kernel(const int64_t *__restrict__ seg_offset, int64_t nseg, const int64_t *__restrict__ tstart,
                      const float *x, const float *y, const float *z, const float *m, DevParams P, double *out) {
  __shared__ typename SrcOf<MODE>::type sh[BLOCK];
  const int64_t ntiles = tstart[nseg];
  for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    int64_t lo = 0, hi = nseg - 1;
    while (lo < hi) {
      const int64_t mid = (lo + hi + 1) >> 1;
      if (tstart[mid] <= t) lo = mid; else hi = mid - 1;
    }
    const DTile T{seg_offset[lo], seg_offset[lo + 1], seg_offset[lo] + (t - tstart[lo]) * BLOCK};
    direct_tile<MODE>(T, x, y, z, m, P, out, sh);
  }
  direct_small<MODE>(seg_offset, nseg, x, y, z, m, P, out);
}

}  // namespace

extern "C" int hbt_direct_potential(hbt_ctx *ctx, int64_t nseg, const int64_t *seg_offset,
                                    const float *x, const float *y, const float *z,
                                    const float *mass, int mode, double *out_phi) {
  if (!ctx || nseg < 0 || !seg_offset) return fail(HBT_ERR_INVALID_ARG, "bad argument");
  if (mode != HBT_DIRECT_FP32 && mode != HBT_DIRECT_FP32_KAHAN && mode != HBT_DIRECT_FP64)
    return fail(HBT_ERR_INVALID_ARG, "bad mode");
  if (nseg == 0) return HBT_OK;
  HIPCHK(hipSetDevice(ctx->device));
  std::vector<int64_t> off(nseg + 1);
  // ordered after whatever the caller enqueued on the context's stream
  HIPCHK(hipMemcpyAsync(off.data(), seg_offset, (nseg + 1) * 8, hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  std::vector<DTile> tiles;
  bool small = false;
  for (int64_t s = 0; s < nseg; s++) {
    if (off[s + 1] < off[s]) return fail(HBT_ERR_INVALID_ARG, "seg_offset not ascending");
    if (off[s + 1] - off[s] <= WAVE) {
      small = small || off[s + 1] > off[s];
      continue;
    }
    for (int64_t t = off[s]; t < off[s + 1]; t += BLOCK) tiles.push_back(DTile{off[s], off[s + 1], t});
  }
  if (tiles.empty() && !small) return HBT_OK;
  DBuf tb;
  hipStream_t st = ctx->stream;
  hipError_t e = hipSuccess;
  if (!tiles.empty()) {
    RETCHK(tb.ensure(tiles.size() * sizeof(DTile)));
    e = hipMemcpyAsync(tb.p, tiles.data(), tiles.size() * sizeof(DTile), hipMemcpyHostToDevice, st);
  }
  if (e == hipSuccess) {
    const DevParams P = make_dev_params(ctx->params);
    const int nt = (int)tiles.size();
    // small groups alone: a kernel that leaves more waves to a SIMD; else after the tiles
    const auto launch = [&](auto tile_kernel, auto small_kernel) {
      const int64_t sb = small ? (nseg + BLOCK / WAVE - 1) / (BLOCK / WAVE) : 0;
      const int g = (int)std::min<int64_t>(std::max<int64_t>(sb, nt), (int64_t)ctx->cus * 16);
      if (nt == 0) small_kernel<<<g, BLOCK, 0, st>>>(seg_offset, nseg, x, y, z, mass, P, out_phi);
      else
        tile_kernel<<<g, BLOCK, 0, st>>>(tb.as<DTile>(), nt, seg_offset, small ? nseg : 0, x, y, z, mass, P, out_phi);
    };
    if (mode == HBT_DIRECT_FP64) launch(direct_kernel<HBT_DIRECT_FP64>, direct_small_kernel<HBT_DIRECT_FP64>);
    else if (mode == HBT_DIRECT_FP32_KAHAN)
      launch(direct_kernel<HBT_DIRECT_FP32_KAHAN>, direct_small_kernel<HBT_DIRECT_FP32_KAHAN>);
    else launch(direct_kernel<HBT_DIRECT_FP32>, direct_small_kernel<HBT_DIRECT_FP32>);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(st);
  }
  tb.release();
  if (e != hipSuccess) return fail(HBT_ERR_DEVICE, std::string("direct potential: ") + hipGetErrorString(e));
  return HBT_OK;
}

// hbt_direct_potential without allocating: no hipMalloc, hipFree or other
// allocating call; the tile table goes to the device's scratch array.  Calls
// that overlap on one GPU race for it.
extern "C" int hbt_direct_potential_noalloc(hbt_ctx *ctx, int64_t nseg, const int64_t *seg_offset,
                                            const float *x, const float *y, const float *z,
                                            const float *mass, int mode, double *out_phi) {
  if (!ctx || nseg < 0 || !seg_offset) return fail(HBT_ERR_INVALID_ARG, "bad argument");
  if (mode != HBT_DIRECT_FP32 && mode != HBT_DIRECT_FP32_KAHAN && mode != HBT_DIRECT_FP64)
    return fail(HBT_ERR_INVALID_ARG, "bad mode");
  if (nseg > NOALLOC_MAX_GROUPS)
    return fail(HBT_ERR_CAPACITY, "hbt_direct_potential_noalloc takes at most 65536 groups");
  if (nseg == 0) return HBT_OK;
  HIPCHK(hipSetDevice(ctx->device));
  void *ptr = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (ctx->device >= 0 && ctx->device < NOALLOC_MAX_DEVICES) ptr = g_scratch_ptr[ctx->device];
  }
  if (!ptr) return fail(HBT_ERR_DEVICE, "no scratch address for the context's device");
  int64_t *tstart = (int64_t *)ptr;
  int *bad = (int *)(tstart + NOALLOC_MAX_GROUPS + 1);
  hipStream_t st = ctx->stream;
  const DevParams P = make_dev_params(ctx->params);
  direct_tile_starts_kernel<<<1, BLOCK, 0, st>>>(seg_offset, nseg, tstart, bad);
  const int g = ctx->cus * 8;  // (twice what a CU holds of the FP64 form)
  if (mode == HBT_DIRECT_FP64)
    direct_noalloc_kernel<HBT_DIRECT_FP64><<<g, BLOCK, 0, st>>>(seg_offset, nseg, tstart, x, y, z, mass, P, out_phi);
  else if (mode == HBT_DIRECT_FP32_KAHAN)
    direct_noalloc_kernel<HBT_DIRECT_FP32_KAHAN><<<g, BLOCK, 0, st>>>(seg_offset, nseg, tstart, x, y, z, mass, P,
                                                                     out_phi);
  else
    direct_noalloc_kernel<HBT_DIRECT_FP32><<<g, BLOCK, 0, st>>>(seg_offset, nseg, tstart, x, y, z, mass, P, out_phi);
  HIPCHK(hipGetLastError());
  int h_bad = 0;
  HIPCHK(hipMemcpyAsync(&h_bad, bad, sizeof(int), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  if (h_bad) return fail(HBT_ERR_INVALID_ARG, "seg_offset not ascending");
  return HBT_OK;
}
