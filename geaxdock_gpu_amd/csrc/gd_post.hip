// gd_post.hip -- post-MC clustering on the device: k-means over the nine
// energy terms of accepted-step records and one medoid per cluster.
//
// The reference clusters the records of each replica into 50 groups, then
// the collected medoids into 500 (src/post_mc.C:40-101), each time with
// clusterByKmeans (src/util.C:1801-1880) over seq_kmeans
// (src/seq_kmeans.c): centers start at the first k objects of a shuffled
// list, Lloyd passes repeat while more than `threshold` of the objects change
// cluster (at most 501 passes), and each cluster reports one member. This
// file keeps that algorithm with three changes, each for reproducibility:
//   - the shuffle is seeded: the first k objects of a uniformly random
//     permutation are drawn by k steps of Fisher-Yates from Philox
//     (the reference seeds it from the clock);
//   - the medoid is the member nearest the final center, ties to the lower
//     index (the reference never updates its running distance and so keeps
//     the last member);
//   - cluster sums are exact: each term is added as a 48.16 fixed-point
//     integer (clamped to +-2^27), so the centers do not depend on the order
//     in which device threads add, and the means are rounded once from double.
//
// Layout in HBM: features SoA [9][n] (coalesced per term), membership [n],
// per group: centers [k][9] float, sums [k][9] int64, counts [k], pass count,
// change count and the pass that ended it. A pass is two launches over all
// groups at once: assign (workgroups of a few waves over tiles of a group's
// objects) and update (the centers). The sums live on between passes: an object
// that changes cluster takes its terms from one sum to the other, which is
// exact in integers, so a pass adds only what moved. The host checks the
// number of live groups every 8 passes; finished groups cost one early return
// per tile.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <memory>
#include <new>
#include <thread>
#include <vector>

namespace gd {

constexpr int KM_DIM = GD_MAXWEI - 1;  // vdw .. dst
constexpr int KM_MAX_K = 512;
constexpr int KM_GATHER_K = 128;  // all passes gather in LDS up to this many centers
constexpr int KM_ROUNDS_K = 15;   // fewer than are ever split over waves
constexpr int KM_MAX_GROUP = 1 << 19;  // objects per group (fixed-point sum range)
constexpr float KM_CLAMP = 134217728.0f;  // 2^27

struct KmArgs {
  const float *feat;  // [KM_DIM][n_total]
  int64_t n_total;
  const int64_t *off;  // [n_groups + 1]
  const int *tile_g;   // tile -> group
  const int *tile_s;   // tile -> first object (group-local)
  int *memb;           // [n_total], group-local cluster id or -1
  float *cent;         // [n_groups][k][KM_DIM]
  long long *sum;      // [n_groups][k][KM_DIM]
  int *cnt;            // [n_groups][k]
  int *delta, *pass;         // [n_groups]
  int *done;                 // [n_groups]: the pass that ended the group (-1: never run)
  int *active;
  int rounds;  // tiles of a gathering workgroup
  unsigned long long *best;  // [n_groups][k]: (distance bits << 32) | member
  int *size;                 // [n_groups][k]
  int k;
  float threshold;
  int max_pass;
};

__host__ __device__ inline long long km_fixed(float v) {
  if (!(v == v)) return 0;
  v = v > KM_CLAMP ? KM_CLAMP : (v < -KM_CLAMP ? -KM_CLAMP : v);
  return (long long)rint((double)v * 65536.0);
}

// Squared Euclidean distance: terms in order, each square added with one
// fused multiply-add (the CPU restatement calls fmaf the same way).
__host__ __device__ inline float km_dist2(const float *a, const float *b) {
#pragma clang fp contract(off)
  float s = 0.0f;
#pragma unroll
  for (int d = 0; d < KM_DIM; ++d) {
    const float t = a[d] - b[d];
    s = fmaf(t, t, s);
  }
  return s;
}

// One assignment pass. A workgroup of 4 waves takes 64 O (4 / S) objects of a
// group, O per lane; S waves share the same objects and take k / S centers
// each, then the lowest distance in center order wins (ties to the lower
// index, as in one loop over all centers). The rule (km_run) gives every CU
// several waves: S = 4 for a group of few objects and many centers (22,000
// objects and 500 centers ran on 22 CUs before: 190 us a pass, 29 us now),
// O = 2 only when the objects alone fill the chip many times, where two
// objects share each center's scalar loads.
//
// The centers are read-only here and wave-uniform: passed as their own
// restrict pointer they are fetched with scalar loads and feed the distance
// arithmetic as scalar operands. Bound: VALU, 22 instructions per object and
// center.
//
// GATHER (S = 1): a workgroup's changes to the sums are gathered in LDS and
// flushed once. It serves the first pass, where every object is new, and all
// passes of up to KM_GATHER_K centers, whose few sums the objects' atomics
// would all meet on: 400,000 objects, 3 centers, 159 us a pass with global
// atomics, 35 so; 24 centers 51 and 32 us, 100 centers 42 and 41. With more
// centers later passes move the objects that changed with global atomics (500
// centers 110 us, 126 by LDS: few objects of a workgroup share a center).
template <int O, int S, bool GATHER>
__global__ void __launch_bounds__(256) gd_km_assign_kernel(KmArgs A, const float *__restrict__ cent,
                                                           int pass) {
  const int g = A.tile_g[blockIdx.x];
  if (A.done[g] < pass) return;
  const int k = A.k;
  extern __shared__ __align__(16) unsigned char km_lds[];
  long long *lsum = (long long *)km_lds;              // GATHER: [k][KM_DIM]
  int *lcnt = (int *)(lsum + (size_t)k * KM_DIM);     // GATHER: [k]
  __shared__ float pd[S > 1 ? 4 : 1][O][64];
  __shared__ int pb[S > 1 ? 4 : 1][O][64];
  if constexpr (GATHER) {
    for (int j = threadIdx.x; j < k * KM_DIM; j += 256) lsum[j] = 0;
    for (int c = threadIdx.x; c < k; c += 256) lcnt[c] = 0;
    __syncthreads();
  }
  const float *cen = cent + (size_t)g * k * KM_DIM;
  const int64_t base = A.off[g];
  const int n = (int)(A.off[g + 1] - base);
  const int l = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int part = wv % S, og = wv / S;
  long long *gs = A.sum + (size_t)g * k * KM_DIM;
  int *gn = A.cnt + (size_t)g * k;
  int changed = 0;
  // a gathering workgroup takes `rounds` tiles
  const int t1 = GATHER ? min(n, A.tile_s[blockIdx.x] + A.rounds * 256 * O) : n;
  for (int t0 = A.tile_s[blockIdx.x];;) {
    const int i0 = t0 + og * 64 * O + l;
    float f[O][KM_DIM], dist[O];
    int best[O];
    bool has[O];
#pragma unroll
    for (int o = 0; o < O; ++o) {
      has[o] = i0 + 64 * o < n;
      const int64_t i = base + (has[o] ? i0 + 64 * o : 0);
#pragma unroll
      for (int d = 0; d < KM_DIM; ++d) f[o][d] = A.feat[(size_t)d * A.n_total + i];
      // the first center is taken whatever its distance; later parts start from
      // nothing
      best[o] = part == 0 ? 0 : -1;
      dist[o] = part == 0 ? km_dist2(f[o], cen) : __builtin_inff();
    }
    const int c1 = (k * (part + 1)) / S;
#pragma unroll 4
    for (int c = part == 0 ? 1 : (k * part) / S; c < c1; ++c) {
      const float *cc = cen + (size_t)c * KM_DIM;
#pragma unroll
      for (int o = 0; o < O; ++o) {
        const float e = km_dist2(f[o], cc);
        if (e < dist[o]) {
          dist[o] = e;
          best[o] = c;
        }
      }
    }
    if constexpr (S > 1) {
#pragma unroll
      for (int o = 0; o < O; ++o) {
        pd[wv][o][l] = dist[o];
        pb[wv][o][l] = best[o];
      }
      __syncthreads();
      if (part != 0) return;
#pragma unroll
      for (int o = 0; o < O; ++o)
        for (int q = 1; q < S; ++q)
          if (pd[wv + q][o][l] < dist[o]) {
            dist[o] = pd[wv + q][o][l];
            best[o] = pb[wv + q][o][l];
          }
    }
#pragma unroll
    for (int o = 0; o < O; ++o) {
      int *m = A.memb + base + i0 + 64 * o;
      const int old = has[o] ? *m : 0, now = best[o];
      const bool move = has[o] && old != now;
      changed += __popcll(__ballot(move));
      if (!move) continue;
      *m = now;
      if constexpr (GATHER) {
#pragma unroll
        for (int d = 0; d < KM_DIM; ++d) {
          const unsigned long long v = (unsigned long long)km_fixed(f[o][d]);
          atomicAdd((unsigned long long *)&lsum[now * KM_DIM + d], v);
          if (old >= 0) atomicAdd((unsigned long long *)&lsum[old * KM_DIM + d], 0ull - v);
        }
        atomicAdd(&lcnt[now], 1);
        if (old >= 0) atomicAdd(&lcnt[old], -1);
      } else {
#pragma unroll
        for (int d = 0; d < KM_DIM; ++d) {
          const unsigned long long v = (unsigned long long)km_fixed(f[o][d]);
          atomicAdd((unsigned long long *)&gs[now * KM_DIM + d], v);
          if (old >= 0) atomicAdd((unsigned long long *)&gs[old * KM_DIM + d], 0ull - v);
        }
        atomicAdd(&gn[now], 1);
        if (old >= 0) atomicAdd(&gn[old], -1);
      }
    }
    t0 += 256 * O;
    if (!GATHER || t0 >= t1) break;
  }
  if (l == 0 && changed) atomicAdd(A.delta + g, changed);
  if constexpr (GATHER) {
    __syncthreads();
    for (int c = threadIdx.x; c < k; c += 256)
      if (lcnt[c]) atomicAdd(gn + c, lcnt[c]);
    for (int j = threadIdx.x; j < k * KM_DIM; j += 256)
      if (lsum[j]) atomicAdd((unsigned long long *)&gs[j], (unsigned long long)lsum[j]);
  }
}

__host__ __device__ inline float km_mean(long long s, int n) {
  return (float)((double)s / (double)n / 65536.0);
}

// Centers of pass `pass` (256 terms per workgroup, grid.y of them per group)
// and each group's end: the group that ends now still gets its centers, so
// workgroups look for earlier ends only.
__global__ void __launch_bounds__(256) gd_km_update_kernel(KmArgs A, int pass) {
  const int g = blockIdx.x;
  if (A.done[g] < pass) return;
  const int k = A.k;
  const int j = blockIdx.y * 256 + threadIdx.x;
  if (j < k * KM_DIM) {
    const int n = A.cnt[(size_t)g * k + j / KM_DIM];
    const size_t q = (size_t)g * k * KM_DIM + j;
    if (n > 0) A.cent[q] = km_mean(A.sum[q], n);
  }
  if (j == 0) {
    const int n = (int)(A.off[g + 1] - A.off[g]);
    const float frac = (float)A.delta[g] / (float)n;
    A.delta[g] = 0;
    A.pass[g] = pass + 1;
    if (!(frac > A.threshold) || pass + 1 >= A.max_pass) A.done[g] = pass;
    else atomicAdd(A.active, 1);
  }
}

// Per cluster, the member with the smallest (distance bits, index). One thread
// per object of a tile of `tile` objects.
__global__ void __launch_bounds__(256) gd_km_medoid_kernel(KmArgs A, int tile) {
  const int g = A.tile_g[blockIdx.x];
  const int k = A.k;
  const float *cen = A.cent + (size_t)g * k * KM_DIM;
  const int64_t base = A.off[g];
  const int n = (int)(A.off[g + 1] - base);
  const int s0 = A.tile_s[blockIdx.x];
  const int s1 = min(n, s0 + tile);
  for (int i = s0 + (int)threadIdx.x; i < s1; i += 256) {
    const int c = A.memb[base + i];
    if (c < 0 || c >= k) continue;
    float f[KM_DIM];
#pragma unroll
    for (int d = 0; d < KM_DIM; ++d) f[d] = A.feat[(size_t)d * A.n_total + base + i];
    const float dd = km_dist2(f, cen + (size_t)c * KM_DIM);
    const unsigned long long key = ((unsigned long long)__float_as_uint(dd) << 32) | (unsigned)i;
    atomicMin(A.best + (size_t)g * k + c, key);
    atomicAdd(A.size + (size_t)g * k + c, 1);
  }
}

// First k positions of a uniformly random permutation of [0, n): k steps of
// Fisher-Yates, position i swapped with i + floor(u * (n - i)), u from
// Philox (i, group, level, 0x6B6D) under the seed.
inline void km_init_indices(int n, int k, int group, int level, uint64_t seed, std::vector<int> &perm,
                            int *out) {
  if ((int)perm.size() < n) {
    const int old = (int)perm.size();
    perm.resize(n);
    for (int i = old; i < n; ++i) perm[i] = i;
  }
  std::vector<int> touched;
  for (int i = 0; i < k; ++i) {
    const u32x4 r = philox4x32_10({(uint32_t)i, (uint32_t)group, (uint32_t)level, 0x6B6Du},
                                  (uint32_t)seed, (uint32_t)(seed >> 32));
    const int j = i + (int)(((uint64_t)r.x * (uint64_t)(n - i)) >> 32);
    std::swap(perm[i], perm[j]);
    out[i] = perm[i];
    touched.push_back(i);
    touched.push_back(j);
  }
  for (int t : touched) perm[t] = t;  // back to the identity for the next group
}

}  // namespace gd

namespace {

// Host loops over millions of records run on up to 16 threads.
template <class F>
void par_for(int64_t n, F f) {
  const int64_t hw = std::max(1u, std::thread::hardware_concurrency());
  const int nt = (int)std::min<int64_t>(std::min<int64_t>(hw, 16), std::max<int64_t>(1, n / 32768));
  if (nt <= 1) {
    f(0, (int64_t)0, n);
    return;
  }
  std::vector<std::thread> th;
  for (int t = 0; t < nt; ++t)
    th.emplace_back([&, t] { f(t, n * t / nt, n * (t + 1) / nt); });
  for (auto &x : th) x.join();
}
// Host arrays that every element of is written before use: no zero fill.
template <class T>
std::unique_ptr<T[]> uninit(size_t n) {
  return std::unique_ptr<T[]>(new T[std::max<size_t>(n, 1)]);
}

inline int par_threads(int64_t n) {
  const int64_t hw = std::max(1u, std::thread::hardware_concurrency());
  return (int)std::min<int64_t>(std::min<int64_t>(hw, 16), std::max<int64_t>(1, n / 32768));
}

// Device k-means of n_groups groups of objects whose features are given as
// SoA [9][n_total] on the host. medoid/size: [n_groups][k], group-local
// member index or -1.
gd_status km_run(gd_ctx *ctx, int n_groups, const int64_t *off, const float *soa_in, int k,
                 float threshold, int max_pass, uint64_t seed, int level, int *medoid, int *size,
                 int *passes, double *device_ms) {
  using namespace gd;
  if (n_groups < 0 || !off || (!soa_in && off[n_groups] > 0) || !medoid || !size)
    return fail(ctx, GD_ERR_INVALID, "kmeans: bad arguments");
  if (k < 1 || k > KM_MAX_K) return fail(ctx, GD_ERR_CAPACITY, "kmeans: k %d outside [1, %d]", k, KM_MAX_K);
  if (max_pass < 1) return fail(ctx, GD_ERR_INVALID, "kmeans: max_pass %d < 1", max_pass);
  if (off[0] != 0) return fail(ctx, GD_ERR_INVALID, "kmeans: group offsets must start at 0");
  for (int g = 0; g < n_groups; ++g) {
    const int64_t n = off[g + 1] - off[g];
    if (n < 0) return fail(ctx, GD_ERR_INVALID, "kmeans: group %d has negative size", g);
    if (n > KM_MAX_GROUP)
      return fail(ctx, GD_ERR_CAPACITY, "kmeans: group %d has %lld objects (max %d)", g,
                  (long long)n, KM_MAX_GROUP);
  }
  const int64_t n_total = n_groups ? off[n_groups] : 0;
  if (n_total > INT32_MAX) return fail(ctx, GD_ERR_CAPACITY, "kmeans: %lld objects", (long long)n_total);
  for (int i = 0; i < n_groups * k; ++i) {
    medoid[i] = -1;
    size[i] = 0;
  }
  // groups with fewer than k objects: every object is its own medoid
  std::vector<int> tile_g, tile_s;
  std::vector<float> cent((size_t)n_groups * k * KM_DIM, 0.0f);
  std::vector<int> done(n_groups, -1), init(k);
  std::vector<int> perm;
  int64_t waves = 0, n_live = 0;
  for (int g = 0; g < n_groups; ++g) {
    const int n = (int)(off[g + 1] - off[g]);
    if (passes) passes[g] = 0;
    if (n < k) {
      for (int i = 0; i < n; ++i) {
        medoid[(size_t)g * k + i] = i;
        size[(size_t)g * k + i] = 1;
      }
      continue;
    }
    done[g] = INT32_MAX;
    n_live += 1;
    waves += (n + 63) / 64;
    km_init_indices(n, k, g, level, seed, perm, init.data());
    for (int c = 0; c < k; ++c)
      for (int d = 0; d < KM_DIM; ++d)
        cent[((size_t)g * k + c) * KM_DIM + d] = soa_in[(size_t)d * n_total + off[g] + init[c]];
  }
  // objects per lane and waves per object set (see the kernel): two objects per
  // lane from 32 waves of objects per CU on, centers split four ways below two
  // waves per CU (and not for a handful of centers)
  const int o_lane = waves >= (int64_t)32 * ctx->n_cu ? 2 : 1;
  const int c_split = waves < (int64_t)2 * ctx->n_cu && k >= 16 ? 4 : 1;
  // a workgroup of few centers takes four tiles of groups of thousands of objects,
  // where that leaves one for every other CU: four times as many flushes would
  // meet on the same sums (10 groups of 20,000 objects, 3 centers, 43 us a pass,
  // 33 so; 300 groups of 2,000, whose sums few meet on, would go from 20 to 23)
  const int rounds = k <= KM_ROUNDS_K && waves >= (int64_t)8 * o_lane * ctx->n_cu &&
                             waves >= (int64_t)64 * n_live
                         ? 4
                         : 1;
  const int tile = 64 * o_lane * (4 / c_split) * rounds;
  for (int g = 0; g < n_groups; ++g) {
    if (done[g] < 0) continue;
    const int n = (int)(off[g + 1] - off[g]);
    for (int s = 0; s < n; s += tile) {
      tile_g.push_back(g);
      tile_s.push_back(s);
    }
  }
  const int n_tiles = (int)tile_g.size();
  if (n_tiles == 0) return GD_OK;
  HIPCHK(hipSetDevice(ctx->device));
  const size_t gk = (size_t)n_groups * k;
  const ScratchTrim trim{ctx};
  Regions R;
  const size_t o_feat = R.add((size_t)KM_DIM * n_total * 4);
  const size_t o_off = R.add((size_t)(n_groups + 1) * 8);
  const size_t o_tg = R.add((size_t)n_tiles * 4), o_ts = R.add((size_t)n_tiles * 4);
  const size_t o_cent = R.add(gk * KM_DIM * 4), o_done = R.add((size_t)n_groups * 4);
  const size_t o_zero = R.end;  // cleared: sums, counts, changes, passes, sizes
  const size_t o_sum = R.add(gk * KM_DIM * 8), o_cnt = R.add(gk * 4);
  const size_t o_delta = R.add((size_t)n_groups * 4), o_pass = R.add((size_t)n_groups * 4);
  const size_t o_size = R.add(gk * 4), o_active = R.add(4);
  const size_t o_ones = R.end;  // set to all ones: memberships, medoid keys
  const size_t o_memb = R.add((size_t)n_total * 4), o_best = R.add(gk * 8);
  TRY(scratch_need(ctx, ctx->dev, R.end, false));
  unsigned char *base = ctx->dev.p;
  KmArgs A{};
  float *d_feat = (float *)(base + o_feat);
  int64_t *d_off = (int64_t *)(base + o_off);
  int *d_tg = (int *)(base + o_tg), *d_ts = (int *)(base + o_ts);
  A.cent = (float *)(base + o_cent);
  A.done = (int *)(base + o_done);
  A.sum = (long long *)(base + o_sum);
  A.cnt = (int *)(base + o_cnt);
  A.delta = (int *)(base + o_delta);
  A.pass = (int *)(base + o_pass);
  A.size = (int *)(base + o_size);
  A.active = (int *)(base + o_active);
  A.memb = (int *)(base + o_memb);
  A.best = (unsigned long long *)(base + o_best);
  hipStream_t st = ctx->stream;
  HIPCHK(hipMemcpyAsync(d_feat, soa_in, (size_t)KM_DIM * n_total * 4, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(d_off, off, (size_t)(n_groups + 1) * 8, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(d_tg, tile_g.data(), (size_t)n_tiles * 4, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(d_ts, tile_s.data(), (size_t)n_tiles * 4, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(A.cent, cent.data(), gk * KM_DIM * 4, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(A.done, done.data(), (size_t)n_groups * 4, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemsetAsync(base + o_zero, 0, o_ones - o_zero, st));
  HIPCHK(hipMemsetAsync(base + o_ones, 0xFF, R.end - o_ones, st));
  A.feat = d_feat;
  A.n_total = n_total;
  A.off = d_off;
  A.tile_g = d_tg;
  A.tile_s = d_ts;
  A.k = k;
  A.threshold = threshold;
  A.max_pass = max_pass;
  A.rounds = rounds;
  // LDS sums of the gathering passes (unsplit centers)
  const size_t lds_gather = (size_t)k * KM_DIM * 8 + (size_t)k * 4 + 16;
  void (*assign)(KmArgs, const float *, int) = nullptr, (*first)(KmArgs, const float *, int) = nullptr;
  if (c_split == 4) {
    assign = first = gd_km_assign_kernel<1, 4, false>;
  } else if (o_lane == 2) {
    assign = gd_km_assign_kernel<2, 1, false>;
    first = gd_km_assign_kernel<2, 1, true>;
  } else {
    assign = gd_km_assign_kernel<1, 1, false>;
    first = gd_km_assign_kernel<1, 1, true>;
  }
  if (c_split == 1) {
    HIPCHK(hipFuncSetAttribute((const void *)first, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds_gather));
    if (k <= KM_GATHER_K) assign = first;
  }
  const dim3 upd((unsigned)n_groups, (unsigned)((k * KM_DIM + 255) / 256));
  HIPCHK(hipEventRecord(ctx->ev0, st));
  for (int p = 0; p < max_pass;) {
    const int batch = std::min(8, max_pass - p);
    for (int b = 0; b < batch; ++b, ++p) {
      if (b == batch - 1) HIPCHK(hipMemsetAsync(A.active, 0, 4, st));
      const bool gather = c_split == 1 && (p == 0 || k <= KM_GATHER_K);
      hipLaunchKernelGGL(p == 0 ? first : assign, dim3(n_tiles), dim3(256), gather ? lds_gather : 0,
                         st, A, (const float *)A.cent, p);
      HIPCHK(hipGetLastError());
      hipLaunchKernelGGL(gd_km_update_kernel, upd, dim3(256), 0, st, A, p);
      HIPCHK(hipGetLastError());
    }
    int live = 0;
    HIPCHK(hipMemcpyAsync(&live, A.active, 4, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (live == 0) break;
  }
  hipLaunchKernelGGL(gd_km_medoid_kernel, dim3(n_tiles), dim3(256), 0, st, A, tile);
  HIPCHK(hipGetLastError());
  HIPCHK(hipEventRecord(ctx->ev1, st));
  std::vector<unsigned long long> best(gk);
  std::vector<int> sz(gk), pass(n_groups);
  HIPCHK(hipMemcpyAsync(best.data(), A.best, gk * 8, hipMemcpyDeviceToHost, st));
  HIPCHK(hipMemcpyAsync(sz.data(), A.size, gk * 4, hipMemcpyDeviceToHost, st));
  HIPCHK(hipMemcpyAsync(pass.data(), A.pass, (size_t)n_groups * 4, hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  if (device_ms) {
    float ms = 0.0f;
    HIPCHK(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    *device_ms += ms;
  }
  for (int g = 0; g < n_groups; ++g) {
    if (off[g + 1] - off[g] < k) continue;
    if (passes) passes[g] = pass[g];
    for (int c = 0; c < k; ++c) {
      const size_t j = (size_t)g * k + c;
      if (sz[j] > 0) {
        medoid[j] = (int)(best[j] & 0xFFFFFFFFull);
        size[j] = sz[j];
      }
    }
  }
  return GD_OK;
}

}  // namespace

extern "C" {

gd_status gd_kmeans_medoids(gd_ctx *ctx, int n_groups, const int64_t *group_off,
                            const float *features, int k, float threshold, int max_pass,
                            uint64_t seed, int *medoid, int *size, int *passes,
                            double *device_ms) {
  if (!ctx) return GD_ERR_INVALID;
  if (device_ms) *device_ms = 0.0;
  try {
    using namespace gd;
    if (n_groups < 0 || !group_off || (n_groups > 0 && group_off[n_groups] > INT32_MAX))
      return fail(ctx, GD_ERR_INVALID, "kmeans: bad group offsets");
    const int64_t n_total = n_groups > 0 ? std::max<int64_t>(group_off[n_groups], 0) : 0;
    if (n_total > 0 && !features) return fail(ctx, GD_ERR_INVALID, "kmeans: null features");
    // row-major objects to SoA terms
    auto soa_v = uninit<float>((size_t)KM_DIM * n_total);
    float *soa = soa_v.get();
    par_for(n_total, [&](int, int64_t a, int64_t b) {
      for (int d = 0; d < KM_DIM; ++d)
        for (int64_t i = a; i < b; ++i) soa[(size_t)d * n_total + i] = features[i * KM_DIM + d];
    });
    return km_run(ctx, n_groups, group_off, soa, k, threshold, max_pass, seed, 0, medoid, size,
                  passes, device_ms);
  } catch (const std::bad_alloc &) {
    return fail(ctx, GD_ERR_NOMEM, "kmeans: out of host memory");
  }
}

}  // extern "C"

namespace {
gd_status post_mc_impl(gd_ctx *ctx, const gd_record *recs, int64_t n, int k_replica, int k_final,
                       uint64_t seed, int64_t *medoid_rec, int *medoid_size, int *n_medoids,
                       double *device_ms);
}  // namespace

extern "C" {

gd_status gd_post_mc(gd_ctx *ctx, const gd_record *recs, int64_t n, int k_replica, int k_final,
                     uint64_t seed, int64_t *medoid_rec, int *medoid_size, int *n_medoids,
                     double *device_ms) {
  if (!ctx) return GD_ERR_INVALID;
  try {
    return post_mc_impl(ctx, recs, n, k_replica, k_final, seed, medoid_rec, medoid_size,
                        n_medoids, device_ms);
  } catch (const std::bad_alloc &) {
    return fail(ctx, GD_ERR_NOMEM, "post_mc: out of host memory");
  }
}

}  // extern "C"

namespace {
gd_status post_mc_impl(gd_ctx *ctx, const gd_record *recs, int64_t n, int k_replica, int k_final,
                       uint64_t seed, int64_t *medoid_rec, int *medoid_size, int *n_medoids,
                       double *device_ms) {
  using namespace gd;
  if (device_ms) *device_ms = 0.0;
  if (n < 0 || (n > 0 && !recs) || !medoid_rec || !medoid_size || !n_medoids)
    return fail(ctx, GD_ERR_INVALID, "post_mc: bad arguments");
  if (k_replica < 1 || k_replica > KM_MAX_K || k_final < 1 || k_final > KM_MAX_K)
    return fail(ctx, GD_ERR_CAPACITY, "post_mc: k %d / %d outside [1, %d]", k_replica, k_final,
                KM_MAX_K);
  *n_medoids = 0;
  if (n == 0) return GD_OK;
  // records grouped by replica (ascending replica, each in the given order):
  // a stable counting sort, chunk-parallel, over the replica indices (read from
  // the records once)
  const int nt = par_threads(n);
  auto rep_v = uninit<int>((size_t)n);
  int *rep = rep_v.get();
  std::vector<int> tmax(nt, -1), tbad(nt, -1);
  par_for(n, [&](int t, int64_t a, int64_t b) {
    int mx = -1;
    for (int64_t i = a; i < b; ++i) {
      const int r = recs[i].replica.idx_rep;
      if (r < 0 && tbad[t] < 0) tbad[t] = (int)std::min<int64_t>(i, INT32_MAX);
      mx = std::max(mx, r);
      rep[i] = r;
    }
    tmax[t] = mx;
  });
  for (int t = 0; t < nt; ++t)
    if (tbad[t] >= 0)
      return fail(ctx, GD_ERR_INVALID, "post_mc: record %d has a negative replica", tbad[t]);
  const int max_rep = *std::max_element(tmax.begin(), tmax.end());
  const size_t nr = (size_t)max_rep + 1;
  // per-thread counts, then each thread's first slot per replica
  std::vector<int64_t> tcnt((size_t)nt * nr, 0);
  par_for(n, [&](int t, int64_t a, int64_t b) {
    int64_t *c = tcnt.data() + (size_t)t * nr;
    for (int64_t i = a; i < b; ++i) c[rep[i]] += 1;
  });
  std::vector<int64_t> cnt(nr + 1, 0);
  for (size_t r = 0; r < nr; ++r) {
    int64_t s0 = cnt[r];
    for (int t = 0; t < nt; ++t) {
      const int64_t c = tcnt[(size_t)t * nr + r];
      tcnt[(size_t)t * nr + r] = s0;
      s0 += c;
    }
    cnt[r + 1] = s0;
  }
  // groups: replicas that have records
  std::vector<int64_t> off{0};
  for (size_t r = 0; r < nr; ++r)
    if (cnt[r + 1] > cnt[r]) off.push_back(cnt[r + 1]);
  const int n_groups = (int)off.size() - 1;
  // order and features (SoA terms) of the grouped records, the features in
  // the context's pinned staging unless they are more than it keeps
  HIPCHK(hipSetDevice(ctx->device));
  const ScratchTrim trim{ctx};
  auto order = uninit<int64_t>((size_t)n);
  std::unique_ptr<float[]> feat_v;
  float *feat = nullptr;
  const size_t feat_bytes = (size_t)KM_DIM * n * sizeof(float);
  if (feat_bytes <= SCRATCH_KEEP / 2) {
    TRY(scratch_need(ctx, ctx->pin, feat_bytes, true));
    feat = reinterpret_cast<float *>(ctx->pin.p);
  } else {
    feat_v = uninit<float>((size_t)KM_DIM * n);
    feat = feat_v.get();
  }
  par_for(n, [&](int t, int64_t a, int64_t b) {
    int64_t *pos = tcnt.data() + (size_t)t * nr;
    for (int64_t i = a; i < b; ++i) {
      const int64_t at = pos[rep[i]]++;
      order[(size_t)at] = i;
      const float *e = recs[i].energy.e;
      for (int d = 0; d < KM_DIM; ++d) feat[(size_t)d * n + at] = e[d];
    }
  });
  std::vector<int> med((size_t)n_groups * k_replica), sz((size_t)n_groups * k_replica);
  TRY(km_run(ctx, n_groups, off.data(), feat, k_replica, 0.001f, 501, seed, 1, med.data(),
             sz.data(), nullptr, device_ms));
  // level 2 over the level-1 medoids, in replica and cluster order
  std::vector<int64_t> l1;
  for (int g = 0; g < n_groups; ++g)
    for (int c = 0; c < k_replica; ++c) {
      const int m = med[(size_t)g * k_replica + c];
      if (m >= 0) l1.push_back(order[off[g] + m]);
    }
  const size_t n1 = l1.size();
  std::vector<float> f2((size_t)KM_DIM * std::max<size_t>(n1, 1));
  for (size_t i = 0; i < n1; ++i)
    for (int d = 0; d < KM_DIM; ++d) f2[(size_t)d * n1 + i] = recs[l1[i]].energy.e[d];
  const int64_t off2[2] = {0, (int64_t)l1.size()};
  std::vector<int> med2(k_final), sz2(k_final);
  TRY(km_run(ctx, 1, off2, f2.data(), k_final, 0.001f, 501, seed, 2, med2.data(), sz2.data(),
             nullptr, device_ms));
  int m = 0;
  for (int c = 0; c < k_final; ++c)
    if (med2[c] >= 0) {
      medoid_rec[m] = l1[med2[c]];
      medoid_size[m] = sz2[c];
      m += 1;
    }
  *n_medoids = m;
  return GD_OK;
}
}  // namespace
