// gd_sur.hip -- learned energy surrogate kernels: receptor feature grids,
// feature rows, BF16 MFMA MLP forward/backward (FP32 accumulate), fixed-order
// gradient sums, FP32 Adam. Building blocks and layouts: gd_sur.h.
#include <type_traits>

#include "gd_sur.h"

namespace gd {

// Feature grids of all protein conformers (grid.y) of a complex: n^3 nodes at
// origin + h*(i,j,k), 32 floats per node, node index (i*n + j)*n + k.
//
// A wave owns a brick of 4 x 4 x 4 nodes, so its lanes share most of the
// receptor points within the cut-off. It tests 64 points at a time against
// the brick (grown by the cut-off), one per lane, and takes the points that
// pass, class by class, from the owning lane's registers as scalars: each class
// then adds to its own eight registers without selects, in the point order of
// a plain loop over the receptor (same bits). Bound: VALU, the eight expf of a
// node-point pair. One wave per 64 nodes along z and a 32-way select per pair
// took 744 us for 65^3 nodes and 2,400 points; this takes 182 us.
extern "C" __global__ void __launch_bounds__(256) gd_sur_grid_kernel(
    const float4 *xyze_all, const int *type, int pnp, float ox, float oy, float oz, float h, int n,
    float *grid_all) {
  const int l = threadIdx.x & 63;
  const int nb = (n + 3) / 4;
  const int brick = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (brick >= nb * nb * nb) return;  // whole wave leaves; no block barrier
  const float4 *xyze = xyze_all + (size_t)blockIdx.y * pnp;
  const int bi = 4 * (brick / (nb * nb)), bj = 4 * ((brick / nb) % nb), bk = 4 * (brick % nb);
  const int i = bi + (l >> 4), j = bj + ((l >> 2) & 3), k = bk + (l & 3);
  const float x = ox + h * i, y = oy + h * j, z = oz + h * k;
  // squared distance of a point to the brick; a margin covers its rounding
  const float lx = ox + h * bi, ly = oy + h * bj, lz = oz + h * bk, w = 3.0f * h;
  const float reach = SUR_CUT * SUR_CUT * 1.001f;
  float f[32];
#pragma unroll
  for (int q = 0; q < 32; ++q) f[q] = 0.0f;
  float4 P = make_float4(0.f, 0.f, 0.f, 0.f);
  int c = -1;
  if (l < pnp) {
    P = xyze[l];
    c = type[l] % SUR_NCLS;
  }
  for (int p0 = 0; p0 < pnp; p0 += 64) {
    const int pn = p0 + 64 + l;
    float4 Pn = make_float4(0.f, 0.f, 0.f, 0.f);
    int cn = -1;
    if (pn < pnp) {
      Pn = xyze[pn];
      cn = type[pn] % SUR_NCLS;
    }
    const float dx = fmaxf(fmaxf(lx - P.x, P.x - (lx + w)), 0.0f);
    const float dy = fmaxf(fmaxf(ly - P.y, P.y - (ly + w)), 0.0f);
    const float dz = fmaxf(fmaxf(lz - P.z, P.z - (lz + w)), 0.0f);
    const bool in = dx * dx + dy * dy + dz * dz <= reach;
    auto add = [&](auto cls_c) {
      constexpr int C = decltype(cls_c)::value;
      for (unsigned long long m = __ballot(in && c == C); m != 0; m &= m - 1) {
        const int s = __builtin_ctzll(m);
        radial_add<C>(x, y, z,
                      __int_as_float(__builtin_amdgcn_readlane(__float_as_int(P.x), s)),
                      __int_as_float(__builtin_amdgcn_readlane(__float_as_int(P.y), s)),
                      __int_as_float(__builtin_amdgcn_readlane(__float_as_int(P.z), s)), f);
      }
    };
    add(std::integral_constant<int, 0>{});
    add(std::integral_constant<int, 1>{});
    add(std::integral_constant<int, 2>{});
    add(std::integral_constant<int, 3>{});
    P = Pn;
    c = cn;
  }
  if (i < n && j < n && k < n) {
    float4 *o = reinterpret_cast<float4 *>(
        grid_all + (((size_t)blockIdx.y * n + i) * n + j) * n * 32 + (size_t)k * 32);
#pragma unroll
    for (int q = 0; q < 8; ++q) o[q] = make_float4(f[4 * q], f[4 * q + 1], f[4 * q + 2], f[4 * q + 3]);
  }
}

// Feature rows of poses of one complex: one thread per ligand atom of each
// pose, rows from row0 on.
extern "C" __global__ void gd_sur_feat_kernel(const DevComplex *cxs, int cxi, SurGrid G, int n,
                                              const int *idx_lig, const int *idx_prt,
                                              const float *mm, int64_t row0,
                                              unsigned short *X, float *xf) {
  const DevComplex &C = cxs[cxi];
  const int lna = C.lna;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)n * lna) return;
  const int pose = (int)(t / lna), l = (int)(t % lna);
  feat_row(C, G, mm + (size_t)pose * 6, idx_lig[pose], idx_prt[pose], l, row0 + t, X,
           xf ? xf + (size_t)t * SUR_NF : nullptr);
}

// Feature rows of poses of many complexes: one workgroup per pose, its rows
// from row_of[pose] on; the grid geometry comes from the complex record.
extern "C" __global__ void gd_sur_feat_multi_kernel(const DevComplex *cxs, int n, const int *cid,
                                                    const int *idx_lig, const int *idx_prt,
                                                    const float *mm, const int64_t *row_of,
                                                    unsigned short *X) {
  const int pose = blockIdx.x;
  if (pose >= n) return;
  const DevComplex &C = cxs[cid[pose]];
  SurGrid G;
  G.grid = C.sgrid;
  G.ox = C.sox;
  G.oy = C.soy;
  G.oz = C.soz;
  G.h = C.sh;
  G.n = C.sn;
  for (int l = threadIdx.x; l < C.lna; l += blockDim.x)
    feat_row(C, G, mm + (size_t)pose * 6, idx_lig[pose], idx_prt[pose], l, row_of[pose] + l, X,
             nullptr);
}

// Row strides (bf16) of the LDS tiles of the batch kernels: 64 + 8 and
// 128 + 8 (multiples of 8, so 16-byte reads stay aligned; the padding
// spreads a fragment's rows over the LDS banks).
constexpr int SUR_XS = SUR_F + 8;
constexpr int SUR_AS = SUR_H + 8;
constexpr int SUR_TR = 72;    // transposed tiles: 64 rows + 8
constexpr int SUR_STEP = 64;  // rows per step: 4 row tiles of 16

// Column-split MLP of the batch kernels. A workgroup takes 64 rows at a time;
// each of its waves owns 16 NC columns of both 128-wide layers for all 64
// rows, so its slices of W1, W2 and W2^T stay in registers for the whole
// kernel (B fragments: col tile c, K block kb), and the rows' X and A1 tiles
// are shared through LDS.
template <int NC>
struct ColW {
  bf16x8_t w1[NC][2];    // W1[:, 16 (NC w + c) ..]: K = 64
  bf16x8_t w2[NC][4];    // W2[:, 16 (NC w + c) ..]: K = 128
  float b2[NC], w3[NC];  // per lane: column 16 (NC w + c) + l % 16
};

template <int NC>
__device__ inline void load_colw(const SurW &W, int wv, ColW<NC> &cw) {
  const int l = threadIdx.x & 63, lr = l & 15, lq = l >> 4;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int n = 16 * (NC * wv + c) + lr;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) cw.w1[c][kb] = ld8(W.W1T + n * SUR_F + 32 * kb + 8 * lq);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) cw.w2[c][kb] = ld8(W.W2T + n * SUR_H + 32 * kb + 8 * lq);
    cw.b2[c] = W.b2[n];
    cw.w3[c] = W.w3[n];
  }
}

// X rows [r0, r0 + 64) as 512 pieces of 8 bf16, NV per thread (512 / NV
// threads): read into registers, then written to xs (row-major) and, when xt
// is given, xt (transposed, [64 features][SUR_TR]).
template <int NV>
__device__ inline void load_x(const unsigned short *X, int64_t r0, uint4 (&v)[NV]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int h = 0; h < NV; ++h) {
    const int e = t + (512 / NV) * h;
    const int r = e >> 3, c8 = (e & 7) * 8;
    v[h] = *reinterpret_cast<const uint4 *>(X + (r0 + r) * SUR_F + c8);
  }
}

template <int NV>
__device__ inline void put_x(const uint4 (&v)[NV], unsigned short *xs, unsigned short *xt) {
  const int t = threadIdx.x;
#pragma unroll
  for (int h = 0; h < NV; ++h) {
    const int e = t + (512 / NV) * h;
    const int r = e >> 3, c8 = (e & 7) * 8;
    *reinterpret_cast<uint4 *>(xs + r * SUR_XS + c8) = v[h];
    if (xt) {
      const unsigned int w[4] = {v[h].x, v[h].y, v[h].z, v[h].w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        xt[(c8 + 2 * q) * SUR_TR + r] = (unsigned short)(w[q] & 0xFFFFu);
        xt[(c8 + 2 * q + 1) * SUR_TR + r] = (unsigned short)(w[q] >> 16);
      }
    }
  }
}

// Layer 1 of the wave's column slice: h1[rt][c] = C tile (rows 16 rt.., the
// wave's column tile c), from the staged X tile.
template <int NC>
__device__ inline void col_layer1(const unsigned short *xs, const ColW<NC> &cw,
                                  f32x4_t (&h1)[4][NC]) {
  const int l = threadIdx.x & 63, lr = l & 15, lq = l >> 4;
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int c = 0; c < NC; ++c) h1[rt][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const bf16x8_t a = ld8(xs + (16 * rt + lr) * SUR_XS + 32 * kb + 8 * lq);
#pragma unroll
      for (int c = 0; c < NC; ++c) h1[rt][c] = mfma32(a, cw.w1[c][kb], h1[rt][c]);
    }
}

// Layer 2 of the wave's column slice from the shared A1 tile (+ b2).
template <int NC>
__device__ inline void col_layer2(const unsigned short *a1s, const ColW<NC> &cw,
                                  f32x4_t (&h2)[4][NC]) {
  const int l = threadIdx.x & 63, lr = l & 15, lq = l >> 4;
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int c = 0; c < NC; ++c) h2[rt][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const bf16x8_t a = ld8(a1s + (16 * rt + lr) * SUR_AS + 32 * kb + 8 * lq);
#pragma unroll
      for (int c = 0; c < NC; ++c) h2[rt][c] = mfma32(a, cw.w2[c][kb], h2[rt][c]);
    }
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) h2[rt][c][i] += cw.b2[c];
}

// Store the C tiles v (rows 16 rt + 4 lq + i, column 16 (NC w + c) + lr) as
// bf16: row-major into rm (row stride SUR_AS) and, when tr is given,
// transposed into tr ([128][SUR_TR]).
template <int NC>
__device__ inline void put_tiles(const float (&v)[4][NC][4], int wv, unsigned short *rm,
                                 unsigned short *tr) {
  const int l = threadIdx.x & 63, lr = l & 15, lq = l >> 4;
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int col = 16 * (NC * wv + c) + lr;
      const unsigned int p01 = pk_bf16(v[rt][c][0], v[rt][c][1]);
      const unsigned int p23 = pk_bf16(v[rt][c][2], v[rt][c][3]);
      if (rm) {
        unsigned short *r = rm + (16 * rt + 4 * lq) * SUR_AS + col;
        r[0] = (unsigned short)p01;
        r[SUR_AS] = (unsigned short)(p01 >> 16);
        r[2 * SUR_AS] = (unsigned short)p23;
        r[3 * SUR_AS] = (unsigned short)(p23 >> 16);
      }
      if (tr) *reinterpret_cast<uint2 *>(tr + col * SUR_TR + 16 * rt + 4 * lq) = make_uint2(p01, p23);
    }
}

// Per-row outputs of a batch: y[r] = w3 . silu(H2[r]) + b3. Workgroup b
// takes 64-row steps b, b + G, ... (G = gridDim.x); the next step's X rows
// are read into registers while a step is evaluated.
extern "C" __global__ void __launch_bounds__(256) gd_mlp_fwd_kernel(const unsigned short *X,
                                                                    int64_t n_rows, SurW W,
                                                                    float *y) {
  __shared__ __attribute__((aligned(16))) unsigned short xs[SUR_STEP * SUR_XS];
  __shared__ __attribute__((aligned(16))) unsigned short a1s[SUR_STEP * SUR_AS];
  __shared__ float red[4][SUR_STEP];
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, lr = l & 15, lq = l >> 4;
  ColW<2> cw;
  load_colw(W, wv, cw);
  const float b3 = W.b3[0];
  const int64_t n_steps = n_rows / SUR_STEP;
  uint4 xv[2];
  if (blockIdx.x < n_steps) load_x(X, (int64_t)blockIdx.x * SUR_STEP, xv);
  for (int64_t st = blockIdx.x; st < n_steps; st += gridDim.x) {
    const int64_t r0 = st * SUR_STEP;
    put_x(xv, xs, nullptr);
    if (st + gridDim.x < n_steps) load_x(X, (st + gridDim.x) * SUR_STEP, xv);
    __syncthreads();
    f32x4_t h1[4][2], h2[4][2];
    col_layer1(xs, cw, h1);
    float a1[4][2][4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) a1[rt][c][i] = silu(h1[rt][c][i]);
    put_tiles(a1, wv, a1s, nullptr);
    __syncthreads();
    col_layer2(a1s, cw, h2);
    // this wave's 32 columns of w3 . silu(H2) per row, then across the waves
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = row16_sum(fmaf(silu(h2[rt][0][i]), cw.w3[0], silu(h2[rt][1][i]) * cw.w3[1]));
        if (lr == 0) red[wv][16 * rt + 4 * lq + i] = v;
      }
    __syncthreads();
    if (threadIdx.x < SUR_STEP) {
      const int r = threadIdx.x;
      y[r0 + r] = ((red[0][r] + red[1][r]) + (red[2][r] + red[3][r])) + b3;
    }
    __syncthreads();  // xs, a1s and red are rewritten by the next step
  }
}

// Network output at every grid point for each listed ligand atom type:
// Y[conformer][type][point] = MLP(onehot(type), features(point)), the features
// being the grid's own values (no interpolation).
//
// A wave keeps W1 and W2 in registers (192) and takes tiles of 16 points, each
// through all the types: the points' features are read and rounded once per
// tile, and only the one-hot half of the first K block changes. Both layers
// are computed transposed (weights as the A operand, points as columns), so a
// lane holds four consecutive hidden units of one point: A1 goes to LDS as
// 8-byte rows instead of 32 two-byte stores, and the output's sum over units
// needs two cross-lane steps instead of sixteen. Products, K order and the sum
// tree are those of mlp_fwd16 and mlp_out16, so values have the same bits.
// Bound: VALU (SiLU: 64 exp2 and 64 rcp per lane and tile), then MFMA. Reading
// the weights from L2 for every tile took 2,217 us for 65^3 points and 20
// types (122 TFLOP/s); this takes 520 us (520 TFLOP/s).
constexpr int SUR_TAB_LD = SUR_H + 8;  // A1 row stride in LDS
extern "C" __global__ void __launch_bounds__(256, 2) gd_sur_tab_kernel(
    const float *fgrid, int n_pts, int n_prt, const int *types, int n_types, SurW W, float *Y) {
  __shared__ __attribute__((aligned(16))) unsigned short a1s[4][16 * SUR_TAB_LD];
  __shared__ __attribute__((aligned(16))) float b2s[SUR_H], w3s[SUR_H];
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, lr = l & 15, lq = l >> 4;
  for (int i = threadIdx.x; i < SUR_H; i += blockDim.x) {
    b2s[i] = W.b2[i];
    w3s[i] = W.w3[i];
  }
  __syncthreads();
  bf16x8_t w1[8][2], w2[8][4];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) w1[t][ks] = ld8(W.W1T + (16 * t + lr) * SUR_F + 32 * ks + 8 * lq);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) w2[t][ks] = ld8(W.W2T + (16 * t + lr) * SUR_H + 32 * ks + 8 * lq);
  }
  const float b3 = W.b3[0];
  unsigned short *a1 = a1s[wv] + lr * SUR_TAB_LD;  // this lane's point
  const int tiles = (n_pts + 15) / 16;
  const int64_t n_tiles = (int64_t)tiles * n_prt;
  for (int64_t job = (int64_t)blockIdx.x * 4 + wv; job < n_tiles; job += (int64_t)gridDim.x * 4) {
    const int prt = (int)(job / tiles);
    const int p0 = (int)(job % tiles) * 16;
    // feature columns: K block 0 holds the one-hot (lq 0..2) and radial 0..7
    // (lq 3), block 1 radial 8..31 (lq 0..2) and the bias column (lq 3)
    const int pt = min(p0 + lr, n_pts - 1);
    const float4 *f = reinterpret_cast<const float4 *>(
        fgrid + ((size_t)prt * n_pts + pt) * 32 + (lq == 3 ? 0 : 8 + 8 * lq));
    const float4 fa = f[0], fb = f[1];
    const uint4 fx = make_uint4(pk_bf16(fa.x, fa.y), pk_bf16(fa.z, fa.w), pk_bf16(fb.x, fb.y),
                                pk_bf16(fb.z, fb.w));
    const uint4 x1 = lq == 3 ? make_uint4(0x3F80u, 0u, 0u, 0u) : fx;
    for (int ti = 0; ti < n_types; ++ti) {
      const int type = types[ti];
      const int rel = type - 8 * lq;  // one-hot column within the lane's eight
      auto hot = [&](int w) {
        return rel == 2 * w ? 0x3F80u : (rel == 2 * w + 1 ? 0x3F800000u : 0u);
      };
      const uint4 x0 = lq == 3 ? fx : make_uint4(hot(0), hot(1), hot(2), hot(3));
      const bf16x8_t xb0 = __builtin_bit_cast(bf16x8_t, x0);
      const bf16x8_t xb1 = __builtin_bit_cast(bf16x8_t, x1);
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        f32x4_t c = {0.f, 0.f, 0.f, 0.f};
        c = mfma32(w1[t][0], xb0, c);
        c = mfma32(w1[t][1], xb1, c);
        *reinterpret_cast<uint2 *>(a1 + 16 * t + 4 * lq) =
            make_uint2(pk_bf16(silu(c[0]), silu(c[1])), pk_bf16(silu(c[2]), silu(c[3])));
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): A1 is in LDS
      __builtin_amdgcn_wave_barrier();
      bf16x8_t ab[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) ab[ks] = ld8(a1 + 32 * ks + 8 * lq);
      float y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) c = mfma32(w2[u][ks], ab[ks], c);
        const float4 bb = *reinterpret_cast<const float4 *>(b2s + 16 * u + 4 * lq);
        const float4 ww = *reinterpret_cast<const float4 *>(w3s + 16 * u + 4 * lq);
        y[0] = fmaf(silu(c[0] + bb.x), ww.x, y[0]);
        y[1] = fmaf(silu(c[1] + bb.y), ww.y, y[1]);
        y[2] = fmaf(silu(c[2] + bb.z), ww.z, y[2]);
        y[3] = fmaf(silu(c[3] + bb.w), ww.w, y[3]);
      }
      __builtin_amdgcn_wave_barrier();  // the next type's A1 goes to the same rows
      float v = (y[0] + y[1]) + (y[2] + y[3]);
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      if (lq == 0 && p0 + lr < n_pts) Y[((size_t)prt * NLT + type) * n_pts + p0 + lr] = v + b3;
    }
  }
}

// Pose sums over poses [p0, p1): S = sum of row outputs, residual against the
// target, dS = 2 (S - target) / (p1 - p0), squared residuals for the loss, and
// (with dyr) the output gradient of every row of the batch's n_rows: its
// pose's dS, 0 for the rows that pad the batch to whole steps. Row offsets and
// y are absolute, dyr is relative to the batch's first row.
//
// One workgroup per 64 poses. Their rows are adjacent, so they are read in
// whole lines into LDS, SUR_POSE_ROWS at a time; one lane per pose then adds
// its rows in row order. Latency bound (64 workgroups for a batch of 4,096):
// 7.7 us and a separate kernel for the rows' gradients before, 6.9 us now.
constexpr int SUR_POSE_ROWS = 4096;
extern "C" __global__ void __launch_bounds__(256) gd_mlp_pose_kernel(
    const float *y, const int64_t *off, int p0, int p1, const float *target, float *dS, float *sq,
    float *S_out, float *dyr, int64_t n_rows) {
  __shared__ float ys[SUR_POSE_ROWS];
  const int pb = p0 + blockIdx.x * 64, pe = min(pb + 64, p1);
  const int t = threadIdx.x;
  const bool mine = t < pe - pb;  // this thread's pose
  const int p = mine ? pb + t : pb;
  const int64_t base = off[p0], rb = off[pb], re = off[pe];
  const int64_t mb = off[p], me = mine ? off[p + 1] : mb;
  float s = 0.0f;
  for (int64_t r = rb; r < re; r += SUR_POSE_ROWS) {
    const int n = (int)min(re - r, (int64_t)SUR_POSE_ROWS);
    for (int i = t; i < n; i += 256) ys[i] = y[r + i];
    __syncthreads();
    const int b = (int)max(mb - r, (int64_t)0), e = (int)min(me - r, (int64_t)n);
#pragma unroll 8
    for (int i = b; i < e; ++i) s += ys[i];
    __syncthreads();
  }
  const float res = s - target[p];
  const float g = 2.0f * res / (float)(p1 - p0);
  if (mine) {
    dS[p] = g;
    sq[p] = res * res;
    if (S_out) S_out[p] = s;
  }
  if (!dyr) return;
  for (int64_t r = rb; r < re; r += SUR_POSE_ROWS) {
    const int n = (int)min(re - r, (int64_t)SUR_POSE_ROWS);
    const int b = (int)max(mb - r, (int64_t)0), e = (int)min(me - r, (int64_t)n);
    for (int i = b; i < e; ++i) ys[i] = g;
    __syncthreads();
    for (int i = t; i < n; i += 256) dyr[r + i - base] = ys[i];
    __syncthreads();
  }
  if (pe == p1)
    for (int64_t i = re - base + t; i < n_rows; i += 256) dyr[i] = 0.0f;
}

// Backward of one batch fused with its weight gradients, column-split like
// gd_mlp_fwd_kernel, in 8 waves of 16 columns. Workgroup b takes the contiguous 64-row steps
// [b S / G, (b + 1) S / G) (S steps, G = gridDim.x). Per step, wave w
// recomputes H1 and H2 of its columns, forms
//   dy = dyr of the row (gd_mlp_pose_kernel),  dH2 = dy w3 * silu'(H2),
//   dA1 = dH2 W2^T (all of dH2 from LDS, W2^T slice in registers),
//   dH1 = dA1 * silu'(H1)
// and accumulates its columns of
//   dW2 += A1^T dH2   (A1^T of all waves from LDS),
//   dW1 += X^T dH1    (row 56 of dW1 is the b1 gradient)
// in MFMA accumulators, with b2, w3 and b3. Only fixed-order partials go to
// HBM: p1g[b][64][128], p2g[b][128][128], pb2[b][128], pw3[b][129]
// (summed in a fixed order by gd_mlp_update_kernel or gd_mlp_gradsum_kernel,
// so training is deterministic). The next step's X rows are read into
// registers while a step is evaluated, and a step's dy rows are read at its
// start, so neither load stalls the step.
//
// Bound: VALU (SiLU and its derivative, bf16 conversions) and the LDS round
// trips between layers. Four waves of 32 columns filled the register file
// with one wave per SIMD, which waited out each of them; 16 columns per wave
// leave room for two. 156,000 rows (4,096 poses): 69.6 -> 50 us.
extern "C" __global__ void __launch_bounds__(512) gd_mlp_train_kernel(
    const unsigned short *X, int64_t n_rows, const float *dyr, SurW W, float *p1g, float *p2g,
    float *pb2, float *pw3) {
  extern __shared__ __attribute__((aligned(16))) unsigned char sm_train[];
  // X [64][SUR_XS] and X^T [64][SUR_TR], two of each (even and odd steps)
  unsigned short *xb = reinterpret_cast<unsigned short *>(sm_train);
  unsigned short *a1s = xb + 2 * (SUR_STEP * SUR_XS + SUR_F * SUR_TR);  // A1 [64][SUR_AS]
  unsigned short *a1t = a1s + SUR_STEP * SUR_AS;                        // A1^T [128][SUR_TR]
  unsigned short *d2s = a1t + SUR_H * SUR_TR;                           // dH2 [64][SUR_AS]
  unsigned short *d2t = d2s + SUR_STEP * SUR_AS;                        // dH2^T [128][SUR_TR]
  unsigned short *d1t = d2t + SUR_H * SUR_TR;                           // dH1^T [128][SUR_TR]
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, lr = l & 15, lq = l >> 4;
  constexpr int NC = 1;
  ColW<NC> cw;
  load_colw(W, wv, cw);
  bf16x8_t w2r[NC][4];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      w2r[c][kb] = ld8(W.W2R + (16 * (NC * wv + c) + lr) * SUR_H + 32 * kb + 8 * lq);
  f32x4_t g2[8][NC], g1[4][NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
#pragma unroll
    for (int t = 0; t < 8; ++t) g2[t][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; ++t) g1[t][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  float gw3[NC] = {}, gb2[NC] = {}, gb3 = 0.0f;
  const int64_t n_steps = n_rows / SUR_STEP;
  const int64_t s_beg = n_steps * blockIdx.x / gridDim.x;
  const int64_t s_end = n_steps * (blockIdx.x + 1) / gridDim.x;
  uint4 xv[1];
  if (s_beg < s_end) load_x(X, s_beg * SUR_STEP, xv);
  for (int64_t st = s_beg; st < s_end; ++st) {
    const int64_t r0 = st * SUR_STEP;
    unsigned short *xs = xb + (st & 1) * (SUR_STEP * SUR_XS + SUR_F * SUR_TR);
    unsigned short *xt = xs + SUR_STEP * SUR_XS;
    // dy of the rows 16 rt + 4 lq + i
    float4 dyv[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
      dyv[rt] = *reinterpret_cast<const float4 *>(dyr + r0 + 16 * rt + 4 * lq);
    put_x(xv, xs, xt);
    if (st + 1 < s_end) load_x(X, r0 + SUR_STEP, xv);
    __syncthreads();
    f32x4_t h1[4][NC], h2[4][NC];
    col_layer1(xs, cw, h1);
    {
      float a1[4][NC][4];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) a1[rt][c][i] = silu(h1[rt][c][i]);
      put_tiles(a1, wv, a1s, a1t);
    }
    __syncthreads();
    col_layer2(a1s, cw, h2);
    // dy of the rows 16 rt + 4 lq + i; w3, b2, b3 gradients
    float dy[4][4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      dy[rt][0] = dyv[rt].x;
      dy[rt][1] = dyv[rt].y;
      dy[rt][2] = dyv[rt].z;
      dy[rt][3] = dyv[rt].w;
    }
    if (wv == 0 && lr == 0)
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) gb3 += (dy[rt][0] + dy[rt][1]) + (dy[rt][2] + dy[rt][3]);
    {
      float d2[4][NC][4];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            gw3[c] = fmaf(silu(h2[rt][c][i]), dy[rt][i], gw3[c]);
            const float dyw = dy[rt][i] * cw.w3[c], ds = dsilu(h2[rt][c][i]);
            gb2[c] = fmaf(dyw, ds, gb2[c]);
            d2[rt][c][i] = dyw * ds;
          }
      put_tiles(d2, wv, d2s, d2t);
    }
    __syncthreads();
    // dA1 = dH2 W2^T for this wave's columns, dH1 transposed
    {
      f32x4_t da[4][NC];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int c = 0; c < NC; ++c) da[rt][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
          const bf16x8_t a = ld8(d2s + (16 * rt + lr) * SUR_AS + 32 * kb + 8 * lq);
#pragma unroll
          for (int c = 0; c < NC; ++c) da[rt][c] = mfma32(a, w2r[c][kb], da[rt][c]);
        }
      float d1[4][NC][4];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) d1[rt][c][i] = da[rt][c][i] * dsilu(h1[rt][c][i]);
      put_tiles(d1, wv, nullptr, d1t);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // this wave's dH1^T stores are in LDS
    __builtin_amdgcn_wave_barrier();
    // weight gradients over the step's 64 rows (two K blocks of 32)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const int ko = 32 * kb + 8 * lq;
      bf16x8_t b2v[NC], b1v[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        b2v[c] = ld8(d2t + (16 * (NC * wv + c) + lr) * SUR_TR + ko);
        b1v[c] = ld8(d1t + (16 * (NC * wv + c) + lr) * SUR_TR + ko);
      }
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const bf16x8_t a = ld8(a1t + (16 * t + lr) * SUR_TR + ko);
#pragma unroll
        for (int c = 0; c < NC; ++c) g2[t][c] = mfma32(a, b2v[c], g2[t][c]);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bf16x8_t a = ld8(xt + (16 * t + lr) * SUR_TR + ko);
#pragma unroll
        for (int c = 0; c < NC; ++c) g1[t][c] = mfma32(a, b1v[c], g1[t][c]);
      }
    }
    // no barrier here: the next step writes the other X buffer, and its
    // first barrier precedes every write to the shared A1 and dH2 tiles
  }

  // partials of this workgroup: its waves own disjoint columns
  float *o2 = p2g + (int64_t)blockIdx.x * SUR_H * SUR_H;
  float *o1 = p1g + (int64_t)blockIdx.x * SUR_F * SUR_H;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int col = 16 * (NC * wv + c) + lr;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int t = 0; t < 8; ++t) o2[(16 * t + 4 * lq + i) * SUR_H + col] = g2[t][c][i];
#pragma unroll
      for (int t = 0; t < 4; ++t) o1[(16 * t + 4 * lq + i) * SUR_H + col] = g1[t][c][i];
    }
  }
  float *w3o = pw3 + (int64_t)blockIdx.x * (SUR_H + 1);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    float v = gw3[c];
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    float b = gb2[c];
    b += __shfl_xor(b, 16);
    b += __shfl_xor(b, 32);
    if (lq == 0) {
      w3o[16 * (NC * wv + c) + lr] = v;
      pb2[(int64_t)blockIdx.x * SUR_H + 16 * (NC * wv + c) + lr] = b;
    }
  }
  gb3 += __shfl_xor(gb3, 16);
  gb3 += __shfl_xor(gb3, 32);
  if (wv == 0 && l == 0) w3o[SUR_H] = gb3;
}

// Dynamic LDS bytes of gd_mlp_train_kernel.
constexpr int SUR_TRAIN_LDS =
    (2 * (SUR_STEP * SUR_XS + SUR_F * SUR_TR) + 2 * SUR_STEP * SUR_AS + 3 * SUR_H * SUR_TR) * 2;

// Gradient of a parameter as the fixed-order sum of n partials: eight
// interleaved sums (partials c, c + 8, ...), then a fixed tree. A workgroup
// takes 32 parameters; thread (j, i) adds interleave j of parameter i, so 128
// adjacent bytes are read at a time and eight times as many loads are in
// flight as with one thread per parameter. The sum is left in threads 0..31.
__device__ inline float grad_sum(const float *p1, const float *p2, const float *pb2,
                                 const float *pw3, int n, int q, float (&red)[8][33]) {
  const int i = threadIdx.x & 31, j = threadIdx.x >> 5;
  const float *part = nullptr;
  int64_t stride = 0;
  if (q < SP_W2) {
    part = p1 + q;
    stride = (int64_t)SUR_F * SUR_H;
  } else if (q < SP_B2) {
    part = p2 + (q - SP_W2);
    stride = (int64_t)SUR_H * SUR_H;
  } else if (q < SP_W3) {
    part = pb2 + (q - SP_B2);
    stride = SUR_H;
  } else if (q < SUR_NPARAM) {
    part = pw3 + (q - SP_W3);
    stride = SUR_H + 1;
  }
  float a = 0.0f;
  if (part) {
#pragma unroll 8
    for (int c = j; c < n; c += 8) a += part[c * stride];
  }
  red[j][i] = a;
  __syncthreads();
  return ((red[0][i] + red[1][i]) + (red[2][i] + red[3][i])) +
         ((red[4][i] + red[5][i]) + (red[6][i] + red[7][i]));
}

// Sums gradient partials into g[SUR_NPARAM] (fixed order: deterministic).
extern "C" __global__ void __launch_bounds__(256) gd_mlp_gradsum_kernel(
    const float *p1, const float *p2, const float *pb2, const float *pw3, int n, float *g) {
  __shared__ float red[8][33];
  const int q = blockIdx.x * 32 + (threadIdx.x & 31);
  const float s = grad_sum(p1, p2, pb2, pw3, n, q, red);
  if (threadIdx.x < 32 && q < SUR_NPARAM) g[q] = s;
}

// One training update: each parameter's gradient from the fixed-order sum of
// the backward's per-workgroup partials (ng of each), then Adam on it and the
// refresh of its bf16 copies. The gradient is also left in g. The last
// workgroup adds the batch's n_sq squared residuals into *loss instead
// (strided partial sums, then a fixed tree). Bound: 25 MB of partials from L2,
// 13.6 us with one thread per parameter, 7.6 us now.
extern "C" __global__ void __launch_bounds__(256) gd_mlp_update_kernel(
    const float *p1, const float *p2, const float *pb2, const float *pw3, int ng, float *p,
    float *m, float *v, float *g, float lr, float b1, float b2, float eps, float c1, float c2,
    unsigned short *W1T, unsigned short *W2T, unsigned short *W2R, const float *sq, int n_sq,
    float *loss) {
  __shared__ float red[8][33];
  if (blockIdx.x == gridDim.x - 1) {
    float *r = &red[0][0];
    float s = 0.0f;
    for (int i = threadIdx.x; i < n_sq; i += 256) s += sq[i];
    r[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
      if (threadIdx.x < h) r[threadIdx.x] += r[threadIdx.x + h];
      __syncthreads();
    }
    if (threadIdx.x == 0) *loss = r[0];
    return;
  }
  const int q = blockIdx.x * 32 + (threadIdx.x & 31);
  const float gq = grad_sum(p1, p2, pb2, pw3, ng, q, red);
  if (threadIdx.x >= 32 || q >= SUR_NPARAM) return;
  g[q] = gq;
  const float mq = fmaf(1.0f - b1, gq, mul_rn(b1, m[q]));
  const float vq = fmaf(gq, mul_rn(1.0f - b2, gq), mul_rn(b2, v[q]));
  m[q] = mq;
  v[q] = vq;
  const float x = p[q] - lr * (mq / c1) / (sqrtf(vq / c2) + eps);
  p[q] = x;
  if (q < SP_W2) {
    const int f = q / SUR_H, i = q % SUR_H;
    W1T[i * SUR_F + f] = f2bf(x);
  } else if (q < SP_B2) {
    const int i = (q - SP_W2) / SUR_H, j = (q - SP_W2) % SUR_H;
    W2T[j * SUR_H + i] = f2bf(x);
    W2R[i * SUR_H + j] = f2bf(x);
  }
}

// Adam on the FP32 master parameters; refreshes the bf16 layouts.
extern "C" __global__ void gd_mlp_adam_kernel(float *p, float *m, float *v, const float *g,
                                              float lr, float b1, float b2, float eps, float c1,
                                              float c2, unsigned short *W1T, unsigned short *W2T,
                                              unsigned short *W2R) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= SUR_NPARAM) return;
  float x = p[q];
  if (lr > 0.0f) {
    const float gq = g[q];
    const float mq = b1 * m[q] + (1.0f - b1) * gq;
    const float vq = b2 * v[q] + (1.0f - b2) * gq * gq;
    m[q] = mq;
    v[q] = vq;
    x -= lr * (mq / c1) / (sqrtf(vq / c2) + eps);
    p[q] = x;
  }
  if (q < SP_W2) {
    const int f = q / SUR_H, i = q % SUR_H;
    W1T[i * SUR_F + f] = f2bf(x);
  } else if (q < SP_B2) {
    const int i = (q - SP_W2) / SUR_H, j = (q - SP_W2) % SUR_H;
    W2T[j * SUR_H + i] = f2bf(x);
    W2R[i * SUR_H + j] = f2bf(x);
  }
}

}  // namespace gd
