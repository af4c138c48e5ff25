// gd_mc.h -- the MC step kernel for CDNA4 (gfx950): device code and the
// gd_mc_kernel template, instantiated per atoms-per-lane in gd_mc_inst.hip.
//
// One workgroup owns a pack: whole temperature ladders of one complex that
// share one protein conformer. The receptor conformer, the type-pair
// parameter records and the KDE points are staged into LDS once per launch;
// each replica is `lpr` lanes of one wave (8..64), each lane owns `APL`
// ligand atoms, and every replica-level sum is a butterfly over its lanes, so
// the MC step needs no workgroup barrier. Barriers occur only at replica-
// exchange points, where one thread per ladder performs the swap sweep.
//
// Reference step order (src/kernel_cuda_l1_montecarlo.cu:95-119): Move_d,
// CalcRmsd_d, CalcMcc_d, CalcEnergy_d (+CombineEnergy_d), Accept_d,
// RecordLigand_d; ExchangeReplicas_d between segments
// (src/kernel_cuda_lancher_siglegpu.cu:25-31).
#pragma once

#include <type_traits>

#include "gd_device.h"
#include "gd_kernels.h"
#include "gd_sur.h"

namespace gd {

struct Lds {
  const float4 *xyze;
  const float *hpp;
  const int *psp;
  const float *par;
  const float4 *kde;  // LDS, or HBM for tiled receptors
  const int2 *kr;
  const int4 *ch;
  const float4 *fl;  // units of the flat pair loop
  float *xe;
  int *xi;
  int *xa;
  int *xo;
  float *xp;
  // tiled receptors: the pack's conformer in HBM (sorted order) and the two
  // LDS tile buffers of `tile` points each
  const float4 *gx;
  const float *ghpp;
  const int *gpsp;
  float4 *tx;
  float *th;
  int *tp;
  int tile;
};

// Pointers read from device structures are generic; their loads would count
// as LDS accesses too and stall the LDS pipeline. Data in HBM is read through
// global pointers.
typedef const __attribute__((address_space(1))) float *gfloat_p;
typedef const __attribute__((address_space(1))) f32x4_t *gfloat4_p;
__device__ __forceinline__ gfloat_p glob(const float *p) { return (gfloat_p)p; }
typedef int i32x2_t __attribute__((ext_vector_type(2)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) int *gint_p;
typedef const __attribute__((address_space(1))) i32x2_t *gint2_p;
typedef const __attribute__((address_space(1))) i32x4_t *gint4_p;

// n items from HBM to LDS by the workgroup's nt threads, four reads of up to 16
// bytes in flight per thread: one of 4 bytes at a time waited out the latency
// for each (14 rounds for the parameter records alone). A launch that finds
// them outside L2 47.6 -> 43.3 us, a call on 8 poses 65.2 -> 63.8 us.
template <class T, class G, class F>
__device__ __forceinline__ void stage_lds(T *dst, G src, int n, int nt, F &&f) {
  for (int i0 = threadIdx.x; i0 < n; i0 += 4 * nt) {
    T v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = src[min(i0 + j * nt, n - 1)];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (i0 + j * nt < n) dst[i0 + j * nt] = f(v[j]);
  }
}
template <class T, class G>
__device__ __forceinline__ void stage_lds(T *dst, G src, int n, int nt) {
  stage_lds(dst, src, n, nt, [](T v) { return v; });
}

// Receptor split of one workgroup: lanes [h*half, (h+1)*half) form group h
// of ns (1, 2, 4 or 8, per pack); every group holds the same replicas and
// covers its share of each receptor chunk. `par` selects the LDS parity
// buffer of the next exchange (each exchange flips it, so one barrier per
// exchange suffices).
struct Split {
  int h, ns, half, ltid, slot, slots;
  int xp_floats;
  int par;
};

// Sums over the `lpr` lanes (8, 16, 32 or 64) of each replica, left in every
// lane; several sums share the level tests and overlap.
template <class... T>
__device__ __forceinline__ void seg_sums(int lpr, T &...v) {
  (dpp_add<DPP_XOR1>(v), ...);
  (dpp_add<DPP_XOR2>(v), ...);
  (dpp_add<DPP_HALF_MIRROR>(v), ...);
  if (lpr > 8) (dpp_add<DPP_MIRROR>(v), ...);
  if (lpr > 16) (swap16_add(v), ...);
  if (lpr > 32) (swap32_add(v), ...);
}
__device__ __forceinline__ float seg_sum(float v, int lpr) {
  seg_sums(lpr, v);
  return v;
}

// Poses evaluated with fewer lanes than the complex's lane shape has (J > 1,
// see eval_poses in gd_engine.hip): slot k of a lane belongs to block k % J of
// the wider shape's lanes. Each block's sum over its lanes is a subtree of the
// wider shape's butterfly; its last levels add the blocks in pairs (blocks
// without an atom would add zeros).
template <int J>
__device__ __forceinline__ float block_total(const float (&t)[J]) {
  if constexpr (J == 1) return t[0];
  else if constexpr (J == 2) return t[0] + t[1];
  else if constexpr (J == 3) return (t[0] + t[1]) + t[2];
  else return (t[0] + t[1]) + (t[2] + t[3]);
}

// KDE sum of one atom over points [b, e) of its type's range:
// sum_j exp2(kde2l |x - q_j|^2) (src/kernel_cuda_l2_calcenergy.cu:232-246).
// Four points are read and exponentiated ahead of their additions, which stay
// in point order, so the sum has the bits of the one-point-at-a-time loop
// while the LDS read latency of the next points overlaps the arithmetic.
__device__ __forceinline__ float kde_sum(const float4 *kde, float kde2l, float x, float y,
                                         float z, int b, int e) {
  float ks = 0.0f;
  int j = b;
  for (; j + 4 <= e; j += 4) {
    const float4 Q0 = kde[j], Q1 = kde[j + 1], Q2 = kde[j + 2], Q3 = kde[j + 3];
    const float e0 = fast_exp2(kde2l * pair_d2(x, y, z, Q0.x, Q0.y, Q0.z));
    const float e1 = fast_exp2(kde2l * pair_d2(x, y, z, Q1.x, Q1.y, Q1.z));
    const float e2 = fast_exp2(kde2l * pair_d2(x, y, z, Q2.x, Q2.y, Q2.z));
    const float e3 = fast_exp2(kde2l * pair_d2(x, y, z, Q3.x, Q3.y, Q3.z));
    ks += e0;
    ks += e1;
    ks += e2;
    ks += e3;
  }
  for (; j < e; ++j) {
    const float4 Q = kde[j];
    ks += fast_exp2(kde2l * pair_d2(x, y, z, Q.x, Q.y, Q.z));
  }
  return ks;
}

// HPC switching polynomial (src/kernel_cuda_l2_calcenergy.cu:116-121):
// 1 - (3.5 x - 4.5 x^2 + 2.5 x^3 - 0.5 x^4), x = d^2 / 81, which factors as
// (1 - x)^3 (1 - x/2) = u^3 (1 + u) / 2 with u = 1 - x. Clamping u at 0 makes
// it exactly 0 beyond d = 9 (the reference's d^2 <= 81 test; u never exceeds
// 1, so the clamp to [0, 1] of the fma's output modifier does it), and the factored
// form has no cancellation near the cut-off. The 1/2 is folded into the
// receptor's hpp values when they are staged into LDS (an exact scaling).
constexpr float INV81 = 1.0f / 81.0f;
constexpr float LOG2E = 1.44269504088896340736f;

struct PairConst {
  float el0, el1, a1, b1;
};

// Per-lane parameters of one chunk (one receptor type) for one ligand atom.
struct ChunkPar {
  float p1a, p2a, pmf0, pmf1, pb, pc, ha, hb, hc;
  float a0, a1;  // p1a lj0, p1a lj0 lj1: den = a0 + a1 d^2 + d^9
  float nr2;  // contacts and the near electrostatic form lie within sqrt(nr2)
};

// Squared distances that let a group of pairs skip terms without a change of
// bits, per lane for one receptor type.
struct Range {
  float nr2;   // contacts, the near electrostatic form and PSP lie within
  float far2;  // beyond: the PMF's exponential does not change 1 + e, HPC is 0
  float hb2;   // beyond: every H-bond term is exactly 0
};

// Largest squared distance at which an H-bond term of these records is not 0:
// exp2(-h^2) is 0 below 2^-126 (the hardware's exp2 has no denormals), h = 11.3
// lies beyond it. `all` (a pose or a complex outside the range that the skips
// are proven for): every distance.
template <int APL>
__device__ __forceinline__ float hb_range2(const ChunkPar (&cp)[APL], bool all) {
  float r = 0.0f;
#pragma unroll
  for (int k = 0; k < APL; ++k)
    if (cp[k].hc != 0.0f) r = fmaxf(r, (11.3f - cp[k].hb) * fast_rcp(cp[k].ha));
  return all ? __builtin_huge_valf() : r * r * 1.001f;
}

// Receptor points [p, p + NP) of one chunk against the lane's APL atoms.
// All terms of src/kernel_cuda_l2_calcenergy.cu:105-184 plus the contact
// count of CalcMcc_d:
//   vdW  (p1 - p2) / (p1 lj0 (1 + lj1 d^2) + 1), p1 = p1a/d^9, p2 = p2a/d^6,
//        evaluated multiplied through by d^9:
//        num/den = (p1a - p2a d^3) / (a0 + a1 d^2 + d^6 d^3);
//   ele  ele_p * g(el1 d) (the ligand charge is applied per atom later);
//        g = 1/(el1 d) is accumulated for every pair (the point stores
//        ele_p/el1); where el1 d < 1 the near form replaces it;
//   pmf  pmf1 / (1 + exp((6 - d/2)(d - pmf0))), exponent in base 2 as
//        A d^2 + B d + C; vdW and PMF share one reciprocal 1/(den (1 + e));
//        `pmf` here sums 1/(1 + e) over the chunk (pmf1 is applied per chunk);
//   hdb  -hdb1/sqrt(2 pi) exp(-((d - hdb0) hdb1)^2 / 2) (zero record if hdb0 <= 0.1);
//   hpc  hpp * switch(d^2) for d^2 <= 81 (KIND >= 1; S.hpp holds hpp / 2);
//   psp  psp[lig_t][seq3r] when class 2 and d <= pmf0 (KIND == 2);
//   contacts  d <= pmf0.
// Every pair takes the full form of every term, so a pair's contribution is
// a function of that pair alone. Wave-uniform branches skip only what leaves
// every lane's sums as they are, bit for bit (Range): where all lanes are
// beyond far2 (about 15.5 A) the PMF's exponential is below 2^-26, so den + den e
// and num + num e round to den and num, and HPC and contacts are exact zeros;
// beyond a lane's hb2 its H-bond terms are exact zeros; contacts, the near
// electrostatic form and PSP run only when some lane is within contact range
// (the terms inside test each pair exactly). Two chunk-uniform choices are
// template parameters: CLAMP keeps the PMF exponent finite where the chunk's
// pmf0 lets it grow past 60, HB evaluates the H-bond term where some lane's
// atom has an H-bond record with the chunk's receptor type.
// Bound: VALU issue (95 % on the CUs that hold a pack). The two distance tests
// cost a compare each per group of points; in the ensemble of 3,520 replicas
// (3,000 points) they take 12 % of the transcendentals and 6 % of the VALU
// instructions away, 21.6 -> 20.5 ms a kernel of 40 steps; 2,000 poses on 8,000
// points 1,624 -> 1,535 us a call. With kind, clamp and H-bond as run-time
// branches instead (one variant of the loop) the ensemble took 5 % longer. Without
// SKIP every pair takes all terms: where few points are far, or a SIMD holds one
// wave, the tests cost more than they save (rule and figures: NEAR_SHARE in
// gd_engine.hip). The flat loop below goes without them too: its units hold
// points of smaller receptors, and they cost 3 % there.
template <int APL, int KIND, int NP, bool CLAMP, bool HB, bool SKIP>
__device__ __forceinline__ void pair_group(const Lds &S, int p, const float4 (&P)[NP],
                                           const PairConst &K, const Range &G,
                                           const float (&x)[APL], const float (&y)[APL],
                                           const float (&z)[APL], const ChunkPar (&cp)[APL],
                                           const float *const (&psprow)[APL],
                                           float (&vdw)[APL], float (&ele)[APL],
                                           float (&pmf)[APL], float (&psp)[APL],
                                           float (&hdb)[APL], float (&hpc)[APL],
                                           int (&cnt)[APL]) {
  const float pa = -0.5f * LOG2E;
  float hp[NP];
  int ps[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    hp[j] = (KIND >= KIND_HPC) ? S.hpp[p + j] : 0.0f;
    ps[j] = (KIND == KIND_PSP) ? S.psp[p + j] : 0;
  }
  float d2[NP][APL], rd[NP][APL], dd[NP][APL], num[NP][APL], den[NP][APL], dn[NP][APL];
  // the distance tests go by blocks of points, of one where a lane has several
  // atoms (independent work enough), else of two: four at once are seldom far
  // from every atom of a wave (four -> two -> this, in tiles: 2,000 poses of 61
  // atoms on 8,000 points 1.30 -> 1.22 -> 1.21 ms, of 45 atoms on 6,000 points 0.76
  // -> 0.70 -> 0.66)
  constexpr int NB = !SKIP ? NP : NP < 2 || APL >= 2 ? 1 : 2;
  float qm[NP];  // the lane's nearest atom to each point
#pragma unroll
  for (int j = 0; j < NP; ++j) {
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      const float q2 = pair_d2(x[k], y[k], z[k], P[j].x, P[j].y, P[j].z);
      const float r = fast_rsq(q2);
      const float d = q2 * r;
      d2[j][k] = q2;
      rd[j][k] = r;
      dd[j][k] = d;
      qm[j] = k == 0 ? q2 : fminf(qm[j], q2);
      const float d3 = q2 * d;
      const float d6 = d3 * d3;
      num[j][k] = fmaf(-cp[k].p2a, d3, cp[k].p1a);
      den[j][k] = dn[j][k] = fmaf(d6, d3, fmaf(cp[k].a1, q2, cp[k].a0));
      ele[k] = fmaf(P[j].w, r, ele[k]);
    }
  }
#pragma unroll
  for (int j0 = 0; j0 < NP; j0 += NB) {
    float qmin = qm[j0];
#pragma unroll
    for (int j = j0 + 1; j < j0 + NB; ++j) qmin = fminf(qmin, qm[j]);
    if (!SKIP || __ballot(!(qmin > G.far2)) != 0) {
#pragma unroll
      for (int j = j0; j < j0 + NB; ++j)
#pragma unroll
        for (int k = 0; k < APL; ++k) {
          const float q2 = d2[j][k];
          // the exponent is clamped at 64 (exp2 must stay finite) only in chunks
          // whose parameters let it reach 60; elsewhere the clamp is a no-op
          const float wv0 = fmaf(pa, q2, fmaf(cp[k].pb, dd[j][k], cp[k].pc));
          const float wv = CLAMP ? fminf(wv0, 64.0f) : wv0;
          // den (1 + e) and num (1 + e) as den + den e and num + num e: one
          // fma each, one rounding each
          const float e = fast_exp2(wv);
          dn[j][k] = fmaf(den[j][k], e, den[j][k]);
          num[j][k] = fmaf(num[j][k], e, num[j][k]);
          if (KIND >= KIND_HPC) {
            // u <= 1, so clamping to [0, 1] is max(u, 0): the fma's own clamp
            const float u = __builtin_amdgcn_fmed3f(fmaf(q2, -INV81, 1.0f), 0.0f, 1.0f);
            const float u3 = u * u * u;
            hpc[k] = fmaf(hp[j], fmaf(u3, u, u3), hpc[k]);
          }
        }
      // contact range: the lane's nearest atom against the largest of its
      // atoms' near radii (a superset of the pairs the branch needs; the terms
      // inside test each pair exactly)
      if (__ballot(qmin <= G.nr2) != 0) {
#pragma unroll
        for (int j = j0; j < j0 + NB; ++j)
#pragma unroll
          for (int k = 0; k < APL; ++k) {
            const float d = dd[j][k];
            const bool c = d <= cp[k].pmf0;
            cnt[k] += c ? 1 : 0;
            const float s = K.el1 * d;
            if (s < 1.0f) {
              const float gn = fmaf(s * s, fmaf(K.b1, s, K.a1), K.el0);
              ele[k] = fmaf(P[j].w, fmaf(K.el1, gn, -rd[j][k]), ele[k]);
            }
            if (KIND == KIND_PSP) {
              if (c) psp[k] += psprow[k][ps[j]];
            }
          }
      }
    }
    // H-bond: only in chunks where some lane's atom has an H-bond record with
    // this receptor type (elsewhere every term would be 0 * exp2), and there
    // only where such a lane is within its records' range
    if (HB && (!SKIP || __ballot(!(qmin > G.hb2)) != 0)) {
#pragma unroll
      for (int j = j0; j < j0 + NB; ++j)
#pragma unroll
        for (int k = 0; k < APL; ++k) {
          const float h = fmaf(dd[j][k], cp[k].ha, cp[k].hb);
          hdb[k] = fmaf(cp[k].hc, fast_exp2(-(h * h)), hdb[k]);
        }
    }
  }
#pragma unroll
  for (int j = 0; j < NP; ++j)
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      const float r = fast_rcp(dn[j][k]);
      vdw[k] = fmaf(num[j][k], r, vdw[k]);
      pmf[k] = fmaf(den[j][k], r, pmf[k]);
    }
}

// Points per group of a lane shape: enough independent pairs per lane to cover
// latency.
__host__ __device__ constexpr int group_points(int apl) { return apl >= 3 ? 1 : (apl == 2 ? 2 : 4); }

template <int APL, int NP, int KIND, bool CLAMP, bool HB, bool SKIP>
__device__ __forceinline__ void chunk_pairs(const Lds &S, int beg, int end, const PairConst &K,
                                            const Range &G,
                                            const float (&x)[APL], const float (&y)[APL],
                                            const float (&z)[APL], const ChunkPar (&cp)[APL],
                                            const float *const (&psprow)[APL],
                                            float (&vdw)[APL], float (&ele)[APL],
                                            float (&pmf)[APL], float (&psp)[APL],
                                            float (&hdb)[APL], float (&hpc)[APL],
                                            int (&cnt)[APL]) {
  int p = beg;
  // the chunk's PMF sum is taken without pmf1, which multiplies it once at
  // the end
  float pmfc[APL];
#pragma unroll
  for (int k = 0; k < APL; ++k) pmfc[k] = 0.0f;
  // the next group's points are read from LDS one group ahead, so the read
  // latency overlaps the current group's arithmetic (indices clamped into
  // the chunk: the last prefetch re-reads its final point)
  // two register sets in turn (no copies): while one group is evaluated the
  // other is being read
  if (p + NP <= end) {
    float4 Pa[NP], Pb[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) Pa[j] = S.xyze[p + j];
    for (; p + 2 * NP <= end; p += 2 * NP) {
#pragma unroll
      for (int j = 0; j < NP; ++j) Pb[j] = S.xyze[p + NP + j];
      pair_group<APL, KIND, NP, CLAMP, HB, SKIP>(S, p, Pa, K, G, x, y, z, cp, psprow, vdw, ele,
                                           pmfc, psp, hdb, hpc, cnt);
#pragma unroll
      for (int j = 0; j < NP; ++j) Pa[j] = S.xyze[min(p + 2 * NP + j, end - 1)];
      pair_group<APL, KIND, NP, CLAMP, HB, SKIP>(S, p + NP, Pb, K, G, x, y, z, cp, psprow, vdw,
                                           ele, pmfc, psp, hdb, hpc, cnt);
    }
    if (p + NP <= end) {
      pair_group<APL, KIND, NP, CLAMP, HB, SKIP>(S, p, Pa, K, G, x, y, z, cp, psprow, vdw, ele,
                                           pmfc, psp, hdb, hpc, cnt);
      p += NP;
    }
  }
  for (; p < end; ++p) {
    const float4 P1[1] = {S.xyze[p]};
    pair_group<APL, KIND, 1, CLAMP, HB, SKIP>(S, p, P1, K, G, x, y, z, cp, psprow, vdw, ele, pmfc,
                                        psp, hdb, hpc, cnt);
  }
#pragma unroll
  for (int k = 0; k < APL; ++k) pmf[k] = fmaf(cp[k].pmf1, pmfc[k], pmf[k]);
}

// ---- flat pair loop ---------------------------------------------------------
// Under a receptor split of 8 a group's share of a chunk is a few points (2 of
// a 1,200-point receptor, 1 of a 670-point one), and the chunk loop above
// spends its time between them: chunk header, parameter records, loop set-up
// and one of twelve code variants, each waiting out its LDS reads. Here a
// group's points are listed as units of at most two (build_flat_units), by
// receptor type, each unit's points and attributes together in LDS in the
// order they are used. A type's records are read once for all its chunks and the
// units one ahead. One variant serves all kinds: terms a unit
// cannot have are skipped by its flags, and what runs without need adds exact
// zeros (hpp is 0 at plain points, the H-bond factor of pairs without a record
// is 0).
//
// Sums keep the bits of the chunk loop. Every accumulator adds the points in
// the same order, and the near electrostatic corrections, which chunk_pairs
// adds after the main terms of each group of NP points, follow the unit's mode:
// FLAT_SINGLES (each point's correction after its own term), FLAT_BLOCK (a
// group of two: both terms, then both corrections), FLAT_FIRST and FLAT_SECOND
// (the halves of a group of four: the first half's corrections wait for the
// second's terms).
//
// Bound: VALU issue of the CUs that hold a pack (71 % of it on one complex of
// 8 replicas, 77 % on a coarse receptor; the rest is the two waves' latencies).
// Measured per MC step, chunk loop -> units, together with the paired groups
// of run_pack and the prefetched MCS templates: one complex of 8 replicas
// (1,200 points) 48.9 -> 35 us, a coarse receptor of 672 points with 4,408 KDE
// points and 196 MCS templates (408 replicas) 72 -> 50 us; scoring 16,384
// poses on 2,400 points 5.1 -> 3.9 ms.
template <int APL>
struct FlatAcc {
  float vdw[APL], ele[APL], pmf[APL], psp[APL], hdb[APL], hpc[APL];
  float pmfc[APL];          // the current chunk's PMF sum, without pmf1
  // the last PSP value read and its lanes' contact masks: added when the next
  // one is read (or at the end), so no read is waited for
  float pps[APL];
  int ppm[APL];
  float pv[2][APL], pw[2];  // corrections of a FLAT_FIRST unit, with its ele parameters
  bool pend;
  int cnt[APL];
};

struct FlatUnit {
  float4 P[2];  // x, y, z, ele
  int4 a;       // flags, hpp / 2 of both points, PSP columns (16 bits each, -1: none)
};

template <int APL>
__device__ __forceinline__ void flat_psp_add(FlatAcc<APL> &A) {
#pragma unroll
  for (int k = 0; k < APL; ++k)
    A.psp[k] += __int_as_float(__float_as_int(A.pps[k]) & A.ppm[k]);
}

// Keeps a rare wave-uniform branch a branch: if-converted, its instructions
// and selects would run for every unit.
__device__ __forceinline__ void keep_branch() { asm volatile("" ::: "memory"); }

template <int APL, int N, bool PEND>
__device__ __forceinline__ void flat_unit(int ux, bool hb, bool wide, const FlatUnit &U, const PairConst &K,
                                          float nr2max, const float (&x)[APL],
                                          const float (&y)[APL], const float (&z)[APL],
                                          const ChunkPar (&cp)[APL],
                                          gfloat_p const (&psprow)[APL], FlatAcc<APL> &A) {
  const float pa = -0.5f * LOG2E;
  float d2[N][APL], rd[N][APL], dd[N][APL], num[N][APL], den[N][APL];
  bool near = false;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    float qmin = 0.0f;
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      const float q2 = pair_d2(x[k], y[k], z[k], U.P[j].x, U.P[j].y, U.P[j].z);
      const float r = fast_rsq(q2);
      const float d = q2 * r;
      d2[j][k] = q2;
      rd[j][k] = r;
      dd[j][k] = d;
      qmin = k == 0 ? q2 : fminf(qmin, q2);
      const float d3 = q2 * d;
      const float d6 = d3 * d3;
      num[j][k] = fmaf(-cp[k].p2a, d3, cp[k].p1a);
      den[j][k] = fmaf(d6, d3, fmaf(cp[k].a1, q2, cp[k].a0));
    }
    near |= qmin <= nr2max;
  }
  const bool any_near = __ballot(near) != 0;
  float wv[N][APL], pt[N][APL];
#pragma unroll
  for (int j = 0; j < N; ++j)
#pragma unroll
    for (int k = 0; k < APL; ++k)
      wv[j][k] = fmaf(pa, d2[j][k], fmaf(cp[k].pb, dd[j][k], cp[k].pc));
  if (wide) {
    keep_branch();
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
      for (int k = 0; k < APL; ++k) wv[j][k] = fminf(wv[j][k], 64.0f);
  }
#pragma unroll
  for (int j = 0; j < N; ++j)
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      const float e = fast_exp2(wv[j][k]);
      const float r = fast_rcp(fmaf(den[j][k], e, den[j][k]));
      A.vdw[k] = fmaf(fmaf(num[j][k], e, num[j][k]), r, A.vdw[k]);
      pt[j][k] = r;
    }
  auto end_chunk = [&] {
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      A.pmf[k] = fmaf(cp[k].pmf1, A.pmfc[k], A.pmf[k]);
      A.pmfc[k] = 0.0f;
    }
  };
#pragma unroll
  for (int k = 0; k < APL; ++k) A.pmfc[k] = fmaf(den[0][k], pt[0][k], A.pmfc[k]);
  if (ux & FLAT_END0) {  // the first point is its chunk's last
    keep_branch();
    end_chunk();
  }
  if constexpr (N == 2) {
#pragma unroll
    for (int k = 0; k < APL; ++k) A.pmfc[k] = fmaf(den[1][k], pt[1][k], A.pmfc[k]);
    if (ux & FLAT_END1) {
      keep_branch();
      end_chunk();
    }
  }
  if (hb) {
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
      for (int k = 0; k < APL; ++k) {
        const float h = fmaf(dd[j][k], cp[k].ha, cp[k].hb);
        A.hdb[k] = fmaf(cp[k].hc, fast_exp2(-(h * h)), A.hdb[k]);
      }
  }
  if (ux & FLAT_HPC) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const float hp = __int_as_float(j == 0 ? U.a.y : U.a.z);
#pragma unroll
      for (int k = 0; k < APL; ++k) {
        const float u = __builtin_amdgcn_fmed3f(fmaf(d2[j][k], -INV81, 1.0f), 0.0f, 1.0f);
        const float u3 = u * u * u;
        A.hpc[k] = fmaf(hp, fmaf(u3, u, u3), A.hpc[k]);
      }
    }
  }
  const int mode = ux & FLAT_MODE;
  if (!any_near) {
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
      for (int k = 0; k < APL; ++k) A.ele[k] = fmaf(U.P[j].w, rd[j][k], A.ele[k]);
    if constexpr (PEND && N == 2) {
      if (mode == FLAT_SECOND && A.pend) {
        keep_branch();
        A.pend = false;
#pragma unroll
        for (int k = 0; k < APL; ++k)
          A.ele[k] = fmaf(A.pw[1], A.pv[1][k], fmaf(A.pw[0], A.pv[0][k], A.ele[k]));
      }
    }
    return;
  }
  // contacts, the pocket-specific potential and the near electrostatic form
  // (the correction is 0 where that form does not hold)
  const int pscol = __builtin_amdgcn_readfirstlane(U.a.w);
  float v[N][APL];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int ps = j == 0 ? (pscol << 16) >> 16 : pscol >> 16;
    const bool has_psp = ps >= 0;
    if (has_psp) flat_psp_add(A);
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      const float d = dd[j][k];
      const bool c = d <= cp[k].pmf0;
      A.cnt[k] += c ? 1 : 0;
      const float s = K.el1 * d;
      const float gn = fmaf(s * s, fmaf(K.b1, s, K.a1), K.el0);
      v[j][k] = s < 1.0f ? fmaf(K.el1, gn, -rd[j][k]) : 0.0f;
      if (has_psp) {
        A.pps[k] = psprow[k][ps];
        A.ppm[k] = c ? -1 : 0;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < APL; ++k) A.ele[k] = fmaf(U.P[0].w, rd[0][k], A.ele[k]);
  if (N == 1 || mode == FLAT_SINGLES) {
#pragma unroll
    for (int k = 0; k < APL; ++k) A.ele[k] = fmaf(U.P[0].w, v[0][k], A.ele[k]);
  }
  if constexpr (N == 2) {
#pragma unroll
    for (int k = 0; k < APL; ++k) A.ele[k] = fmaf(U.P[1].w, rd[1][k], A.ele[k]);
    if constexpr (PEND) {
      if (mode == FLAT_FIRST) {
        A.pend = true;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
          for (int k = 0; k < APL; ++k) A.pv[j][k] = v[j][k];
          A.pw[j] = U.P[j].w;
        }
        return;
      }
      if (mode == FLAT_SECOND && A.pend) {
        keep_branch();
        A.pend = false;
#pragma unroll
        for (int k = 0; k < APL; ++k)
          A.ele[k] = fmaf(A.pw[1], A.pv[1][k], fmaf(A.pw[0], A.pv[0][k], A.ele[k]));
      }
    }
    if (mode != FLAT_SINGLES) {
#pragma unroll
      for (int k = 0; k < APL; ++k) A.ele[k] = fmaf(U.P[0].w, v[0][k], A.ele[k]);
    }
#pragma unroll
    for (int k = 0; k < APL; ++k) A.ele[k] = fmaf(U.P[1].w, v[1][k], A.ele[k]);
  }
}

// Unit list of a receptor split (1, 2, 4 or 8).
__device__ __forceinline__ int flat_index(int ns) { return 31 - __builtin_clz(ns); }

// All units of lane group h (list bounds `off`). A receptor type's units come in
// an even number (the last may be empty), two register sets in turn.
template <int APL, bool PEND>
__device__ __forceinline__ void flat_pairs(const int *off, const Lds &S, int h,
                                           const PairConst &K, const float (&x)[APL],
                                           const float (&y)[APL], const float (&z)[APL],
                                           const int (&lt)[APL], gfloat_p const (&psprow)[APL],
                                           FlatAcc<APL> &A) {
  const int u0 = __builtin_amdgcn_readfirstlane(off[h]);
  int left = __builtin_amdgcn_readfirstlane(off[h + 1]) - u0;
  if (left <= 0) return;
  const float *rec[APL];
#pragma unroll
  for (int k = 0; k < APL; ++k) rec[k] = S.par + lt[k] * NPAR;
  const float4 *U = S.fl + (size_t)u0 * FLAT_F4;
  auto read_unit = [&](FlatUnit &V) {
    V.P[0] = U[0];
    V.P[1] = U[1];
    const float4 a = U[2];
    V.a = make_int4(__float_as_int(a.x), __float_as_int(a.y), __float_as_int(a.z),
                    __float_as_int(a.w));
    U += FLAT_F4;
  };
  FlatUnit Va, Vb;
  read_unit(Va);
  int ua = __builtin_amdgcn_readfirstlane(Va.a.x);
  while (left > 0) {
    ChunkPar cp[APL];
    float nr2max = 0.0f;
    bool hbond = false, wide_l = false;
    const int type = ua & FLAT_TYPE;
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      const float4 *r = reinterpret_cast<const float4 *>(rec[k] + type * (NLT * NPAR));
      const float4 a = r[0], b = r[1], c = r[2];
      cp[k].p1a = a.x;
      cp[k].p2a = a.y;
      cp[k].pmf0 = a.z;
      cp[k].pmf1 = a.w;
      cp[k].ha = b.x;
      cp[k].hb = b.y;
      cp[k].hc = b.z;
      cp[k].nr2 = b.w;
      cp[k].a0 = c.x;
      cp[k].a1 = c.y;
      cp[k].pb = c.z;
      cp[k].pc = c.w;
      const float t = cp[k].pmf0 - 12.0f;
      wide_l |= !(0.125f * LOG2E * t * t <= 60.0f);  // as in pose_energy's chunks
      hbond |= cp[k].hc != 0.0f;
      nr2max = k == 0 ? cp[k].nr2 : fmaxf(nr2max, cp[k].nr2);
    }
    const bool hb = __ballot(hbond) != 0, wide = __ballot(wide_l) != 0;
    int pairs = (ua >> FLAT_PAIRS) & FLAT_PAIR_MASK;
    left -= 2 * pairs;
    for (; pairs > 0; --pairs) {
      read_unit(Vb);
      if (ua & FLAT_ONE) flat_unit<APL, 1, PEND>(ua, hb, wide, Va, K, nr2max, x, y, z, cp, psprow, A);
      else flat_unit<APL, 2, PEND>(ua, hb, wide, Va, K, nr2max, x, y, z, cp, psprow, A);
      const int ub = __builtin_amdgcn_readfirstlane(Vb.a.x);
      read_unit(Va);  // past the group's end: the next group's first unit, or the pad
      if (!(ub & FLAT_EMPTY)) {
        if (ub & FLAT_ONE) flat_unit<APL, 1, PEND>(ub, hb, wide, Vb, K, nr2max, x, y, z, cp, psprow, A);
        else flat_unit<APL, 2, PEND>(ub, hb, wide, Vb, K, nr2max, x, y, z, cp, psprow, A);
      }
      ua = __builtin_amdgcn_readfirstlane(Va.a.x);
    }
  }
  flat_psp_add(A);
}

// Sum over MCS templates [m_begin, m_end) of tcc_m * sqrt(mean squared
// distance of the template's atoms), src/kernel_cuda_l2_calcenergy.cu:274-313. Templates go
// Q at a time: their loads are issued together, one round ahead of their
// use (a round waited out three dependent reads from L2 before: 196 templates
// of a coarse receptor took 37,000 cycles of a step's 124,000 per wave), and
// their lane sums share each butterfly step. Per template the additions are
// the same as one template at a time. Lanes of three and four atoms take two
// templates a round: four ahead hold 48 registers and more, which the step loop
// then spilled (42 around the plain chunk loop of three atoms, 5 with two).
template <int APL, int J>
__device__ __forceinline__ float mcs_sum(const DevComplex &C, int lpr, const float (&x)[APL],
                                         const float (&y)[APL], const float (&z)[APL],
                                         const int (&li)[APL], const bool (&val)[APL],
                                         int m_begin, int m_end) {
  float elhm = 0.0f;
  if (m_begin >= m_end) return elhm;
  const gfloat4_p mcs = (gfloat4_p)C.mcs;
  const gfloat_p cnt = glob(C.mcs_cnt), tcc = glob(C.mcs_tcc);
  const int lna = C.lna;
  constexpr int Q = APL >= 3 ? 2 : 4;
  f32x4_t M[Q][APL];
  float n[Q], t[Q];
  auto read = [&](int m0) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int m = min(m0 + q, m_end - 1);
#pragma unroll
      for (int k = 0; k < APL; ++k) M[q][k] = mcs[(size_t)m * lna + li[k]];
      n[q] = cnt[m];
      t[q] = tcc[m];
    }
  };
  read(m_begin);
  for (int m0 = m_begin; m0 < m_end; m0 += Q) {
    float s[Q][J], nc[Q], tc[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
#pragma unroll
      for (int j = 0; j < J; ++j) s[q][j] = 0.0f;
      nc[q] = n[q];
      tc[q] = t[q];
#pragma unroll
      for (int k = 0; k < APL; ++k) {
        if (!val[k]) continue;
        if (M[q][k][3] != 0.0f) s[q][k % J] += pair_d2(x[k], y[k], z[k], M[q][k][0], M[q][k][1], M[q][k][2]);
      }
    }
    if (m0 + Q < m_end) read(m0 + Q);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      if constexpr (Q == 4) seg_sums(lpr, s[0][j], s[1][j], s[2][j], s[3][j]);
      else seg_sums(lpr, s[0][j], s[1][j]);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (m0 + q < m_end && nc[q] > 0.0f) elhm += tc[q] * sqrtf(block_total(s[q]) / nc[q]);
  }
  return elhm;
}

// Energy, RMSD and MCC of one pose held by `lpr` lanes (CalcEnergy_d +
// CombineEnergy_d + CalcRmsd_d + CalcMcc_d). Every lane of the replica ends
// with the same bit pattern in E.
//
// With a receptor split (sp.ns > 1) every thread of the workgroup must call
// this together: `live` (wave-uniform) says whether the wave has a pose to
// evaluate; the groups exchange their partial sums through LDS behind one
// workgroup barrier and add them in group order, so every group ends with
// identical bits (with two groups this is the order-free g0 + g1).
//
// TILE: the receptor does not stay resident in LDS; its sorted points stream
// through two LDS tile buffers of S.tile points. While a tile is evaluated
// the next one is read from HBM into registers (one point per thread; points
// beyond the workgroup size after the evaluation) and written to the other
// buffer; one workgroup barrier per tile.
// Every thread runs the tile loop (waves without a pose only stage). Chunks
// that cross a tile boundary are evaluated as one fragment per tile.
//
// FLAT: every pack of the launch has the unit list of its split in LDS; the
// pair loop is flat_pairs.
template <int APL, bool TILE, bool FLAT, int J = 1, int NP = group_points(APL), bool SKIP = true>
__device__ __forceinline__ void pose_energy(const DevComplex &C, const Lds &S, int lpr, Split &sp,
                            bool live, const float (&x)[APL],
                            const float (&y)[APL], const float (&z)[APL],
                            const float (&ox)[APL], const float (&oy)[APL],
                            const float (&oz)[APL], const int (&lt)[APL],
                            const float (&q)[APL], const int (&li)[APL],
                            const bool (&val)[APL], const float mm[6], gd_energy &E) {
  const int n_chunks = __builtin_amdgcn_readfirstlane(C.n_chunks);
  PairConst K;
  K.el0 = C.el0;
  K.el1 = C.el1;
  K.a1 = C.a1;
  K.b1 = C.b1;

  float vdw[APL], ele[APL], pmf[APL], psp[APL], hdb[APL], hpc[APL];
  int cnt[APL];
  const float *psprow[APL];
#pragma unroll
  for (int k = 0; k < APL; ++k) {
    vdw[k] = ele[k] = pmf[k] = psp[k] = hdb[k] = hpc[k] = 0.0f;
    cnt[k] = 0;
    psprow[k] = C.psp + (size_t)lt[k] * C.n_res;
  }

  // A pose of ordinary coordinates (so that no power of a distance overflows)
  // on a complex of ordinary parameters may skip terms by distance.
  float far2 = C.far2;
  bool odd;
  {
    bool o = false;
#pragma unroll
    for (int k = 0; k < APL; ++k)
      o |= !(fabsf(x[k]) < FAR_COORD && fabsf(y[k]) < FAR_COORD && fabsf(z[k]) < FAR_COORD);
    odd = live && __ballot(o) != 0;
  }
  odd |= !(far2 < __builtin_huge_valf());
  if (odd) far2 = __builtin_huge_valf();

  // fragment [fb, fe) of chunk ci, indices into T's point arrays; each lane
  // group of a receptor split takes its share
  auto fragment = [&](const Lds &T, int ci, int fb, int fe) {
    const int4 ch = S.ch[ci];
    const int fl = fe - fb;
    const int beg = fb + (fl * sp.h) / sp.ns;
    const int end = fb + (fl * (sp.h + 1)) / sp.ns;
    const int type = __builtin_amdgcn_readfirstlane(ch.z);
    const int kind = __builtin_amdgcn_readfirstlane(ch.w);
    ChunkPar cp[APL];
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      const float *r = S.par + (type * NLT + lt[k]) * NPAR;
      // the record holds the chunk constants precomputed on the host:
      // a0 = p1a lj0, a1 = p1a lj0 lj1; (6 - d/2)(d - pmf0) log2(e) =
      // A d^2 + B d + C with B = log2(e)(6 + pmf0/2), C = -6 log2(e) pmf0;
      // contacts (d <= pmf0) and the near electrostatic form (d < 1/el1) lie
      // within sqrt(nr2), nr2 = (1.0001 max(pmf0, 1/el1))^2 (the margin covers
      // the rounding of d)
      const float4 a = *reinterpret_cast<const float4 *>(r);
      const float4 b = *reinterpret_cast<const float4 *>(r + 4);
      const float4 c = *reinterpret_cast<const float4 *>(r + 8);
      cp[k].p1a = a.x;
      cp[k].p2a = a.y;
      cp[k].pmf0 = a.z;
      cp[k].pmf1 = a.w;
      cp[k].ha = b.x;
      cp[k].hb = b.y;
      cp[k].hc = b.z;
      cp[k].nr2 = b.w;
      cp[k].a0 = c.x;
      cp[k].a1 = c.y;
      cp[k].pb = c.z;
      cp[k].pc = c.w;
    }
    // the PMF exponent (6 - d/2)(d - pmf0) log2(e) peaks at (pmf0 - 12)^2 / 8
    // log2(e); only a chunk where some lane's peak passes 60 needs the clamp
    bool wide = false, hbond = false;
    Range G;
    G.nr2 = cp[0].nr2;
    G.far2 = far2;
    G.hb2 = hb_range2<APL>(cp, odd);
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      const float t = cp[k].pmf0 - 12.0f;
      wide |= !(0.125f * LOG2E * t * t <= 60.0f);
      hbond |= cp[k].hc != 0.0f;
      G.nr2 = fmaxf(G.nr2, cp[k].nr2);
    }
    const bool clamp = __ballot(wide) != 0;
    const bool hb = __ballot(hbond) != 0;
    auto pairs = [&](auto kind_c, auto clamp_c, auto hb_c) {
      chunk_pairs<APL, NP, decltype(kind_c)::value, decltype(clamp_c)::value,
                  decltype(hb_c)::value, SKIP>(T, beg, end, K, G, x, y, z, cp, psprow, vdw, ele,
                                         pmf, psp, hdb, hpc, cnt);
    };
    auto by_hb = [&](auto kind_c, auto clamp_c) {
      if (hb) pairs(kind_c, clamp_c, std::true_type{});
      else pairs(kind_c, clamp_c, std::false_type{});
    };
    auto by_clamp = [&](auto kind_c) {
      if (clamp) by_hb(kind_c, std::true_type{});
      else by_hb(kind_c, std::false_type{});
    };
    if (kind == KIND_PLAIN) by_clamp(std::integral_constant<int, KIND_PLAIN>{});
    else if (kind == KIND_HPC) by_clamp(std::integral_constant<int, KIND_HPC>{});
    else by_clamp(std::integral_constant<int, KIND_PSP>{});
  };

  if constexpr (FLAT) {
    if (live) {
      FlatAcc<APL> A;
      gfloat_p prow[APL];
#pragma unroll
      for (int k = 0; k < APL; ++k) {
        A.vdw[k] = A.ele[k] = A.pmf[k] = A.psp[k] = A.hdb[k] = A.hpc[k] = A.pmfc[k] = 0.0f;
        A.pps[k] = 0.0f;
        A.ppm[k] = 0;
        A.cnt[k] = 0;
        prow[k] = glob(psprow[k]);
      }
      A.pend = false;
      flat_pairs<APL, (APL == 1 || J > 1)>(C.flat_off[flat_index(sp.ns)], S, sp.h, K, x, y, z, lt, prow, A);
#pragma unroll
      for (int k = 0; k < APL; ++k) {
        vdw[k] = A.vdw[k];
        ele[k] = A.ele[k];
        pmf[k] = A.pmf[k];
        psp[k] = A.psp[k];
        hdb[k] = A.hdb[k];
        hpc[k] = A.hpc[k];
        cnt[k] = A.cnt[k];
      }
    }
  } else if constexpr (!TILE) {
    for (int ci = 0; live && ci < n_chunks; ++ci) {
      const int4 ch = S.ch[ci];
      const int cb = __builtin_amdgcn_readfirstlane(ch.x);
      const int cl = __builtin_amdgcn_readfirstlane(ch.y);
      fragment(S, ci, cb, cb + cl);
    }
  } else {
    const int T = S.tile, pnp = C.pnp;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int n_tiles = (pnp + T - 1) / T;
    for (int i = tid; i < min(T, pnp); i += nt) {
      S.tx[i] = S.gx[i];
      S.th[i] = 0.5f * S.ghpp[i];
      S.tp[i] = S.gpsp[i];
    }
    __syncthreads();
    int ci = 0;
    for (int t = 0; t < n_tiles; ++t) {
      const int tb = t * T, te = min(tb + T, pnp);
      // this thread's point of the next tile, read while this tile is evaluated
      const int ni = te + tid;
      const bool stage = tid < T && ni < min(te + T, pnp);
      float4 nx = make_float4(0.f, 0.f, 0.f, 0.f);
      float nh = 0.0f;
      int np = 0;
      if (stage) {
        nx = S.gx[ni];
        nh = S.ghpp[ni];
        np = S.gpsp[ni];
      }
      if (live) {
        Lds Tl = S;
        const int cur = (t & 1) * T;
        Tl.xyze = S.tx + cur;
        Tl.hpp = S.th + cur;
        Tl.psp = S.tp + cur;
        while (ci < n_chunks) {
          const int4 ch = S.ch[ci];
          const int cb = __builtin_amdgcn_readfirstlane(ch.x);
          const int ce = cb + __builtin_amdgcn_readfirstlane(ch.y);
          const int fb = max(cb, tb), fe = min(ce, te);
          if (fb < fe) fragment(Tl, ci, fb - tb, fe - tb);
          if (ce > te) break;  // the chunk continues in the next tile
          ++ci;
        }
      }
      if (stage) {
        const int o = ((t + 1) & 1) * T + tid;
        S.tx[o] = nx;
        S.th[o] = 0.5f * nh;
        S.tp[o] = np;
      }
      // a tile longer than the workgroup: the rest of it, read now
      for (int i = ni + nt; i < min(te + T, pnp); i += nt) {
        const int o = ((t + 1) & 1) * T + (i - te);
        S.tx[o] = S.gx[i];
        S.th[o] = 0.5f * S.ghpp[i];
        S.tp[o] = S.gpsp[i];
      }
      __syncthreads();
    }
  }

  // Per-atom lists that the groups of a receptor split share out the way they
  // share the receptor's chunks: each group takes its part of the KDE points
  // of every atom's type, of every atom's reference contacts and of the MCS
  // templates, and the partial sums join the exchange below. With one group
  // the parts are the whole lists.
  const float kde2l = C.kde2l;
  float b_kde[J] = {}, elhm = 0.f;
  int t_tp = 0;
  if (live) {
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      if (!val[k]) continue;
      // KDE: mean over same-type points, src/kernel_cuda_l2_calcenergy.cu:224-253
      const int2 kr = S.kr[lt[k]];
      const int kl = kr.y - kr.x;
      const int kb = kr.x + (kl * sp.h) / sp.ns, ke = kr.x + (kl * (sp.h + 1)) / sp.ns;
      const float ks = kde_sum(S.kde, kde2l, x[k], y[k], z[k], kb, ke);
      if (kl > 0) b_kde[k % J] += ks / (float)kl;
      // true positives against the reference contact list
      const int nr = C.ref_cnt[li[k]];
      const int2 *rl = C.ref + (size_t)li[k] * KMAX;
      const int rb0 = (nr * sp.h) / sp.ns, re0 = (nr * (sp.h + 1)) / sp.ns;
      int j = rb0;
      // four contacts at a time: their list entries, then their points, are
      // read together (the count is order-free)
      for (; j + 4 <= re0; j += 4) {
        int2 r[4];
        float4 P[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) r[u] = rl[j + u];
#pragma unroll
        for (int u = 0; u < 4; ++u) P[u] = TILE || FLAT ? S.gx[r[u].x] : S.xyze[r[u].x];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float d2 = pair_d2(x[k], y[k], z[k], P[u].x, P[u].y, P[u].z);
          const float d = d2 * fast_rsq(d2);
          t_tp += (d <= __int_as_float(r[u].y)) ? 1 : 0;
        }
      }
      for (; j < re0; ++j) {
        const int2 r = rl[j];
        const float4 P = TILE || FLAT ? S.gx[r.x] : S.xyze[r.x];
        const float d2 = pair_d2(x[k], y[k], z[k], P.x, P.y, P.z);
        const float d = d2 * fast_rsq(d2);
        t_tp += (d <= __int_as_float(r.y)) ? 1 : 0;
      }
    }
    // MCS restraints, src/kernel_cuda_l2_calcenergy.cu:274-313
    elhm = mcs_sum<APL, J>(C, lpr, x, y, z, li, val, (C.pos * sp.h) / sp.ns,
                        (C.pos * (sp.h + 1)) / sp.ns);
  }

  // pair sums that are linear in the receptor points
  float b_vdw[J] = {}, b_ele[J] = {}, b_pmf[J] = {}, b_psp[J] = {}, b_hdb[J] = {};
  int t_cnt = 0;
#pragma unroll
  for (int k = 0; k < APL; ++k) {
    if (!val[k]) continue;
    b_vdw[k % J] += vdw[k];
    b_ele[k % J] += q[k] * ele[k];
    b_pmf[k % J] += pmf[k];
    b_psp[k % J] += psp[k];
    b_hdb[k % J] += hdb[k];
    t_cnt += cnt[k];
  }
  seg_sums(lpr, b_vdw[0], b_ele[0], b_pmf[0], b_psp[0], b_hdb[0], t_cnt, b_kde[0], t_tp);
#pragma unroll
  for (int j = 1; j < J; ++j)
    seg_sums(lpr, b_vdw[j], b_ele[j], b_pmf[j], b_psp[j], b_hdb[j], b_kde[j]);
  float t_vdw = block_total(b_vdw), t_ele = block_total(b_ele), t_pmf = block_total(b_pmf);
  float t_psp = block_total(b_psp), t_hdb = block_total(b_hdb), t_kde = block_total(b_kde);
  if (sp.ns > 1) {
    // exchange: per-atom HPC sums (the restraint is nonlinear in them) and
    // the replica's linear sums. Every group adds the ns partials in group
    // order, so all groups end with the same bits.
    float *buf = S.xp + sp.par * sp.xp_floats;
    float *hb = buf;                                // [ns*half][4]
    float *rb = buf + (size_t)sp.ns * sp.half * 4;  // [ns][slots][12]
    if (live) {
      float hg[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < APL; ++k) hg[k] = hpc[k];
      *reinterpret_cast<float4 *>(hb + ((size_t)sp.h * sp.half + sp.ltid) * 4) = make_float4(hg[0], hg[1], hg[2], hg[3]);
      if ((sp.ltid - sp.slot * lpr) == 0) {
        float4 *r = reinterpret_cast<float4 *>(rb + ((size_t)sp.h * sp.slots + sp.slot) * 12);
        r[0] = make_float4(t_vdw, t_ele, t_pmf, t_psp);
        r[1] = make_float4(t_hdb, __int_as_float(t_cnt), t_kde, __int_as_float(t_tp));
        r[2] = make_float4(elhm, 0.f, 0.f, 0.f);
      }
    }
    __syncthreads();
    if (live) {
      for (int g = 0; g < sp.ns; ++g) {
        const float4 hv = *reinterpret_cast<const float4 *>(hb + ((size_t)g * sp.half + sp.ltid) * 4);
        const float4 *r = reinterpret_cast<const float4 *>(rb + ((size_t)g * sp.slots + sp.slot) * 12);
        const float4 r0 = r[0], r1 = r[1], r2 = r[2];
        const float hg[4] = {hv.x, hv.y, hv.z, hv.w};
        if (g == 0) {
#pragma unroll
          for (int k = 0; k < APL; ++k) hpc[k] = hg[k];
          t_vdw = r0.x;
          t_ele = r0.y;
          t_pmf = r0.z;
          t_psp = r0.w;
          t_hdb = r1.x;
          t_cnt = __float_as_int(r1.y);
          t_kde = r1.z;
          t_tp = __float_as_int(r1.w);
          elhm = r2.x;
        } else {
#pragma unroll
          for (int k = 0; k < APL; ++k) hpc[k] += hg[k];
          t_vdw += r0.x;
          t_ele += r0.y;
          t_pmf += r0.z;
          t_psp += r0.w;
          t_hdb += r1.x;
          t_cnt += __float_as_int(r1.y);
          t_kde += r1.z;
          t_tp += __float_as_int(r1.w);
          elhm += r2.x;
        }
      }
    }
    sp.par ^= 1;
  }
  if (!live) return;

  // per-atom terms
  float b_hpc[J] = {}, b_rms[J] = {};
#pragma unroll
  for (int k = 0; k < APL; ++k) {
    if (!val[k]) continue;
    // hydrophobic restraint, src/kernel_cuda_l2_calcenergy.cu:200-205
    const float h2 = (hpc[k] - C.hpl0[lt[k]]) / C.hpl1[lt[k]];
    b_hpc[k % J] += 0.5f * h2 * h2 - C.hpl2[lt[k]];
    // RMSD against the start pose
    const float dx = x[k] - (ox[k] + C.pocket[0]);
    const float dy = y[k] - (oy[k] + C.pocket[1]);
    const float dz = z[k] - (oz[k] + C.pocket[2]);
    b_rms[k % J] += dx * dx + dy * dy + dz * dz;
  }
  const int pos = C.pos;

#pragma unroll
  for (int j = 0; j < J; ++j) seg_sums(lpr, b_hpc[j], b_rms[j]);
  const float t_hpc = block_total(b_hpc), t_rms = block_total(b_rms);

  // src/kernel_cuda_l2_calcenergy.cu:334-359, src/kernel_cuda_l3_combineenergy.cu:28-37
  const float lna = (float)C.lna;
  float e[GD_MAXWEI];
  e[0] = t_vdw / lna;
  e[1] = t_ele / lna;
  e[2] = t_pmf / lna;
  e[3] = t_psp / lna;
  e[4] = t_hdb / lna;
  e[5] = t_hpc / lna;
  e[6] = (t_kde / C.kde3) / lna;
  e[7] = pos > 0 ? logf(elhm / (float)pos) : 0.0f;
  {
    const float cx = C.pocket[0] + mm[0], cy = C.pocket[1] + mm[1], cz = C.pocket[2] + mm[2];
    const float dx = cx - C.pocket[0], dy = cy - C.pocket[1], dz = cz - C.pocket[2];
    e[8] = sqrtf(dx * dx + dy * dy + dz * dz);
  }
  float total = 0.0f;
#pragma unroll
  for (int i = 0; i < GD_MAXWEI - 1; ++i) {
    e[i] = C.a_para[i] * e[i] + C.b_para[i];
    E.e[i] = e[i];
    total += e[i] * C.w[i];
  }
  E.e[GD_MAXWEI - 1] = total;
  E.rmsd = sqrtf(t_rms / lna);
  // Matthews correlation of the contact maps, src/kernel_cuda_l2_calcmcc.cu:194-206
  const int tp = t_tp, fp = t_cnt - t_tp, fn = C.ref_total - t_tp;
  const int tn = C.lna * C.pnp - C.ref_total - fp;
  const float tp0 = (float)tp, fn0 = (float)fn, fp0 = (float)fp, tn0 = (float)tn;
  const float dv = sqrtf((tp0 + fp0) * (tp0 + fn0) * (tn0 + fp0) * (tn0 + fn0));
  E.cms = dv != 0.0f ? (tp0 * tn0 - fp0 * fn0) / dv : 0.0f;
}

// Weighted KDE, MCS and pocket-distance terms (e[6..8] after normalization)
// of one pose: the cheap part of the energy, evaluated exactly inside the
// surrogate (src/kernel_cuda_l2_calcenergy.cu:224-326).
//
// SHARE (a split pack of a complex with large KDE or MCS sets): the groups of
// the receptor split take their parts of each atom's KDE points and of the
// MCS templates and exchange the partial sums through the split's LDS
// buffers behind one barrier, adding them in group order. Every thread of the
// workgroup must then call this together; `live` (wave-uniform) says whether
// the wave has a pose. Without SHARE the lists are evaluated whole by every
// group, and only waves with a pose call it.
template <int APL, bool SHARE>
__device__ __forceinline__ float cheap_terms(const DevComplex &C, const Lds &S, int lpr,
                                             Split &sp, bool live,
                                             const float (&x)[APL], const float (&y)[APL],
                                             const float (&z)[APL], const int (&lt)[APL],
                                             const bool (&val)[APL], const float mm[6],
                                             const Rot &R, int a, int ilig) {
  const int gh = SHARE ? sp.h : 0, gn = SHARE ? sp.ns : 1;
  const int pos = C.pos;
  float t_kde = 0.0f, elhm = 0.0f;
  if (live) {
    const float kde2l = C.kde2l;
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      if (!val[k]) continue;
      const int2 kr = S.kr[lt[k]];
      const int kl = kr.y - kr.x;
      const float ks = kde_sum(S.kde, kde2l, x[k], y[k], z[k], kr.x + (kl * gh) / gn,
                               kr.x + (kl * (gh + 1)) / gn);
      if (kl > 0) t_kde += ks / (float)kl;
    }
    // MCS restraints in closed form from the conformer's template moments:
    // sum |R o + t - m|^2 = A + n |R obar + t - mbar|^2 - 2 <R, M>; the
    // replica's lanes take the group's templates in turn
    const float4 *qm = C.mcsq + (size_t)ilig * pos * 4;
    const float tx = mm[0] + C.pocket[0], ty = mm[1] + C.pocket[1], tz = mm[2] + C.pocket[2];
    const int mb = (pos * gh) / gn, me = (pos * (gh + 1)) / gn;
    for (int m = mb + a; m < me; m += lpr) {
      const float n = C.mcs_cnt[m];
      if (!(n > 0.0f)) continue;
      const float4 q0 = qm[4 * m], q1 = qm[4 * m + 1], q2 = qm[4 * m + 2], q3 = qm[4 * m + 3];
      const float ux = R.r00 * q0.y + R.r01 * q0.z + R.r02 * q0.w + tx - q1.x;
      const float uy = R.r10 * q0.y + R.r11 * q0.z + R.r12 * q0.w + ty - q1.y;
      const float uz = R.r20 * q0.y + R.r21 * q0.z + R.r22 * q0.w + tz - q1.z;
      const float rm = R.r00 * q1.w + R.r01 * q2.x + R.r02 * q2.y + R.r10 * q2.z +
                       R.r11 * q2.w + R.r12 * q3.x + R.r20 * q3.y + R.r21 * q3.z + R.r22 * q3.w;
      const float sq = fmaxf(q0.x + n * (ux * ux + uy * uy + uz * uz) - 2.0f * rm, 0.0f);
      elhm += C.mcs_tcc[m] * sqrtf(sq / n);
    }
    seg_sums(lpr, elhm, t_kde);
  }
  if constexpr (SHARE) {
    float *rb = S.xp + sp.par * sp.xp_floats + (size_t)sp.ns * sp.half * 4;  // [ns][slots][12]
    if (live && (sp.ltid - sp.slot * lpr) == 0)
      *reinterpret_cast<float4 *>(rb + ((size_t)sp.h * sp.slots + sp.slot) * 12) =
          make_float4(t_kde, elhm, 0.f, 0.f);
    __syncthreads();
    if (live) {
      for (int g = 0; g < sp.ns; ++g) {
        const float4 r = *reinterpret_cast<const float4 *>(rb + ((size_t)g * sp.slots + sp.slot) * 12);
        t_kde = g == 0 ? r.x : t_kde + r.x;
        elhm = g == 0 ? r.y : elhm + r.y;
      }
    }
    sp.par ^= 1;
  }
  if (!live) return 0.0f;
  const float lna = (float)C.lna;
  const float e6 = (t_kde / C.kde3) / lna;
  const float e7 = pos > 0 ? logf(elhm / (float)pos) : 0.0f;
  const float cx = C.pocket[0] + mm[0], cy = C.pocket[1] + mm[1], cz = C.pocket[2] + mm[2];
  const float dx = cx - C.pocket[0], dy = cy - C.pocket[1], dz = cz - C.pocket[2];
  const float e8 = sqrtf(dx * dx + dy * dy + dz * dz);
  return (C.a_para[6] * e6 + C.b_para[6]) * C.w[6] + (C.a_para[7] * e7 + C.b_para[7]) * C.w[7] +
         (C.a_para[8] * e8 + C.b_para[8]) * C.w[8];
}

// Surrogate total of the pose held by each replica of the wave: the MLP's
// receptor-pair estimate, scale * sum_atoms y / lna, plus the exact cheap
// terms. Rows are the
// wave's atoms, 16 per MFMA tile: tile (k, sub) holds atom k of lanes
// 16 sub .. 16 sub + 15. `da` is the wave's scratch: X tile [16][64] bf16,
// A1 tile [16][128] bf16, y[16].
template <int APL, int DAM, bool SHARE>
__device__ __forceinline__ float sur_total(const KParams &P, const DevComplex &C, const Lds &S,
                                           Split &sp, bool live,
                                           unsigned char *da, int lpr, int prt,
                                           const float (&x)[APL], const float (&y)[APL],
                                           const float (&z)[APL], const int (&lt)[APL],
                                           const bool (&val)[APL], const float mm[6],
                                           const Rot &R, int a, int ilig) {
  if (!live) {  // the cheap terms' exchange only (a workgroup barrier)
    if constexpr (SHARE)
      (void)cheap_terms<APL, true>(C, S, lpr, sp, false, x, y, z, lt, val, mm, R, a, ilig);
    return 0.0f;
  }
  if constexpr (DAM == 2) {
    // tabulated network: trilinear interpolation of the atom type's output
    // grid (same grid geometry and clamping as the feature grid)
    const int n = C.sn;
    const size_t n3 = (size_t)n * n * n;
    const float lim = (float)(n - 1) - 1e-4f;
    const float ih = 1.0f / C.sh;
    float ys = 0.0f;
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      const float ux = fminf(fmaxf((x[k] - C.sox) * ih, 0.0f), lim);
      const float uy = fminf(fmaxf((y[k] - C.soy) * ih, 0.0f), lim);
      const float uz = fminf(fmaxf((z[k] - C.soz) * ih, 0.0f), lim);
      const int ix = (int)ux, iy = (int)uy, iz = (int)uz;
      const float tx = ux - ix, ty = uy - iy, tz = uz - iz;
      const float *g = C.stab + ((size_t)prt * NLT + lt[k]) * n3 + ((size_t)ix * n + iy) * n + iz;
      const size_t sx = (size_t)n * n, sy = n;
      const float c00 = fmaf(tz, g[1] - g[0], g[0]);
      const float c01 = fmaf(tz, g[sy + 1] - g[sy], g[sy]);
      const float c10 = fmaf(tz, g[sx + 1] - g[sx], g[sx]);
      const float c11 = fmaf(tz, g[sx + sy + 1] - g[sx + sy], g[sx + sy]);
      const float c0 = fmaf(ty, c01 - c00, c00);
      const float c1 = fmaf(ty, c11 - c10, c10);
      const float v = fmaf(tx, c1 - c0, c0);
      ys += val[k] ? v : 0.0f;
    }
    ys = seg_sum(ys, lpr);
    return P.sur_scale * (ys / (float)C.lna) +
           cheap_terms<APL, SHARE>(C, S, lpr, sp, true, x, y, z, lt, val, mm, R, a, ilig);
  }
  const int l = threadIdx.x & 63;
  unsigned short *Xs = reinterpret_cast<unsigned short *>(da);
  unsigned short *A1s = Xs + 16 * SUR_F;
  float *ys = reinterpret_cast<float *>(A1s + 16 * SUR_H);
  SurW W;
  W.W1T = P.sW1T;
  W.W2T = P.sW2T;
  W.W2R = nullptr;
  W.b2 = P.sb2;
  W.w3 = P.sw3;
  W.b3 = P.sb3;
  SurGrid G;
  G.grid = C.sgrid;
  G.ox = C.sox;
  G.oy = C.soy;
  G.oz = C.soz;
  G.h = C.sh;
  G.n = C.sn;
  float ysum = 0.0f;
#pragma unroll
  for (int k = 0; k < APL; ++k) {
    float f[32];
    grid_radial(G, prt, x[k], y[k], z[k], f);
    for (int sub = 0; sub < 4; ++sub) {
      if ((l >> 4) == sub) {
        unsigned short *row = Xs + (l & 15) * SUR_F;
#pragma unroll
        for (int q = 0; q < NLT; ++q) row[q] = (q == lt[k]) ? (unsigned short)0x3F80 : (unsigned short)0;
#pragma unroll
        for (int q = 0; q < 32; ++q) row[NLT + q] = f2bf(f[q]);
        row[SUR_BIAS_COL] = 0x3F80;  // 1.0
#pragma unroll
        for (int q = SUR_BIAS_COL + 1; q < SUR_F; ++q) row[q] = 0;
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();
      f32x4_t h1[8], h2[8];
      mlp_fwd16(Xs, 0, W, A1s, h1, h2);
      float yy[4];
      mlp_out16(h2, W, yy);
      if ((l & 15) == 0)
#pragma unroll
        for (int i = 0; i < 4; ++i) ys[4 * (l >> 4) + i] = yy[i];
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();
      if ((l >> 4) == sub && val[k]) ysum += ys[l & 15];
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();
    }
  }
  ysum = seg_sum(ysum, lpr);
  // the network sums per-atom pair energies; the terms are per-atom means
  return P.sur_scale * (ysum / (float)C.lna) +
         cheap_terms<APL, SHARE>(C, S, lpr, sp, true, x, y, z, lt, val, mm, R, a, ilig);
}

// ExchangeReplicas_d for one ladder (src/kernel_cuda_l1_exchangereplicas.cu:33-78):
// temperature i1 = 2 pair + mode_t and i1 + 1 trade slots when
// exp((mb1 - mb2)(E2 - E1)) > U.
template <class U>
__device__ __forceinline__ void exchange_ladder(int n_tmp, int mode_t, const float *et, const float *mb,
                                int *temps, int *acs, int *order, U &&uni) {
  for (int t = 0; t < n_tmp; ++t) order[temps[t]] = t;
  const int maxpair = n_tmp / 2 - ((n_tmp % 2 == 0) && (mode_t == 1));
  for (int pair = 0; pair < maxpair; ++pair) {
    const int i1 = (pair << 1) + mode_t;
    const int i2 = i1 + 1;
    const int o1 = order[i1];
    const int o2 = order[i2];
    const int tt = temps[o1];
    const float e1 = et[o1], e2 = et[o2];
    const float mb1 = mb[temps[o1]], mb2 = mb[temps[o2]];
    const float d1 = mb1 - mb2;
    const float d2 = e2 - e1;
    const float delta = d1 * d2;
    const float prob = decision_expf(delta);
    if (prob > uni(pair)) {
      temps[o1] = temps[o2];
      temps[o2] = tt;
      acs[o1] += 1;
      acs[o2] += 1;
    }
  }
}

// ---- MC steps by a tree of energies -----------------------------------------
// A context with few packs leaves most CUs idle, and one MC step waits for the
// one before it. But a step's proposal needs only the random numbers of its
// step and the state it starts from, and that state is known up to the outcomes
// of the steps between: from one known state, the 2^D - 1 poses that the next D
// steps can propose are the nodes of a binary tree (node v's children: 2v after
// a rejection, 2v + 1 after an acceptance). MODE_TREE evaluates them all at once,
// one workgroup per pack and node; the last workgroup of a pack to finish then
// takes the D decisions in order along the tree and leaves the state, records
// and counts as D single steps do. Every energy and decision is the same
// expression of the same numbers, so results keep their bits.
//
// Bound: one evaluation and its launch, 50 us for 5 steps of 1,200 points
// against 35 us for each step in turn. One complex of 8 replicas (4 packs), 200
// steps: 7.3 -> 2.3 ms; 96 replicas of 40 atoms and 1,311 points (20 packs),
// 159 steps 6.5 -> 4.7 ms; 8 replicas of 120 atoms and 6,000 points, 100 steps
// 21.4 -> 4.9 ms. The count needs no wait: whichever workgroup is last decides.
//
// The pose `from` moved by the offsets that wave lane `src` holds.
__device__ __forceinline__ void tree_move(const float from[6], const float dm[6], int src,
                                          float to[6]) {
  float d[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) d[i] = __shfl(dm[i], src);
  apply_move(from, d, to);
}

// The pose of tree node v (1-based) of a replica: `a` its lane, `base` the
// wave lane of its lane 0. Called by whole waves with a uniform v.
__device__ __forceinline__ void tree_pose(const KParams &P, const DevComplex &C, int flat, int a,
                                          int base, int step0, int v, float mo[6]) {
  const int depth = 31 - __builtin_clz(v);
  float u[8], dm[6], scale[6], mn[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) scale[i] = C.move_scale[i];
  mc_uniforms(P.k0, P.k1, C.cid, flat, step0 + min(a, depth), u);
  move_offsets(u, scale, C.move_kind, dm);
  for (int i = 0; i < depth; ++i)
    if (v >> (depth - 1 - i) & 1) {
      tree_move(mo, dm, base + i, mn);
#pragma unroll
      for (int q = 0; q < 6; ++q) mo[q] = mn[q];
    }
  tree_move(mo, dm, base + depth, mn);
#pragma unroll
  for (int q = 0; q < 6; ++q) mo[q] = mn[q];
}

// Decisions of replica sv's steps [step0, step0 + n_steps) by one wave, whose
// lane l holds the energy of node l + 1 and the random numbers of step l.
__device__ __forceinline__ void tree_decide(const KParams &P, const DevComplex &C, int prt,
                                            int sv, int step0) {
  const int l = threadIdx.x & 63;
  const int flat = P.rep_flat[sv];
  const int ilig = flat % C.n_lig, itmp = P.idx_tmp[sv];
  const float mb = C.minus_beta[itmp];
  gd_energy E = P.ev_out[(size_t)sv * P.tree_nodes + min(l, P.tree_nodes - 1)];
  float mo[6], scale[6], u[8], dm[6], mn[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    mo[i] = P.mm[(size_t)sv * 6 + i];
    scale[i] = C.move_scale[i];
  }
  mc_uniforms(P.k0, P.k1, C.cid, flat, step0 + min(l, P.n_steps - 1), u);
  move_offsets(u, scale, C.move_kind, dm);
  float e = P.e_old[sv].e[GD_MAXWEI - 1];
  float best = P.best_e[sv];
  int rc = P.rec ? P.rec_cnt[sv] : 0;
  int acs = 0, kept = 0, v = 1;
  for (int i = 0; i < P.n_steps; ++i) {
    const float en = __shfl(E.e[GD_MAXWEI - 1], v - 1);
    const bool yes = metropolis(en, e, mb, __shfl(u[6], i));
    if (yes) {
      tree_move(mo, dm, i, mn);
#pragma unroll
      for (int q = 0; q < 6; ++q) mo[q] = mn[q];
      e = en;
      acs += 1;
      kept = v;
      if (P.rec) {
        if (l == v - 1 && rc < P.rec_cap) {
          gd_record &r = P.rec[(size_t)sv * P.rec_cap + rc];
          r.replica.idx_rep = flat;
          r.replica.idx_prt = prt;
          r.replica.idx_tmp = itmp;
          r.replica.idx_lig = ilig;
          r.energy = E;
#pragma unroll
          for (int q = 0; q < 6; ++q) r.movematrix[q] = mo[q];
          r.step = step0 + i;
        }
        rc += 1;
      }
      if (e < best) {
        best = e;
        if (l == 0)
#pragma unroll
          for (int q = 0; q < 6; ++q) P.best_mm[(size_t)sv * 6 + q] = mo[q];
      }
    }
    v = 2 * v + (yes ? 1 : 0);
  }
  if (kept > 0 && l == kept - 1) P.e_old[sv] = E;
  if (l == 0) {
#pragma unroll
    for (int q = 0; q < 6; ++q) P.mm[(size_t)sv * 6 + q] = mo[q];
    P.best_e[sv] = best;
    P.acs_mc[sv] += acs;
    if (P.rec) P.rec_cnt[sv] = rc < P.rec_cap ? rc : P.rec_cap;
  }
}

// DA: 0 plain Metropolis (DA_TREE: by a tree of energies, in instances of its
// own, so that the step loop's registers stay as they are; DA_POSES and
// DA_POSES2: poses with fewer lanes than the complex's shape has, slot k in
// block k or k % 2 of block_total); delayed acceptance with the surrogate from
// the network evaluated per atom (1) or from its tabulated outputs (2); 3 and 4
// are 1 and 2 with the split groups' shared surrogate sums compiled in. MODE is
// DA, with DA_NEAR added where the pair loop goes without distance tests.
template <int APL, int MODE, bool TILE, bool FLAT>
__device__ __forceinline__ void run_pack(const KParams &P, const Pack &pk, const DevComplex &C, const Lds &S,
                         int lpr, int step0, int idx, int node, int &par) {
  constexpr int DA = MODE & ~DA_NEAR;
  constexpr bool SKIP = (MODE & DA_NEAR) == 0;
  constexpr bool TREE = DA == DA_TREE, POSES = DA == DA_POSES || DA == DA_POSES2;
  constexpr int DAM = TREE || POSES ? 0 : DA > 2 ? DA - 2 : DA;
  constexpr int J = !POSES ? 1 : DA == DA_POSES2 ? 2 : APL;
  // the wide shape has one atom per lane (DA_POSES) or two
  constexpr int NP = group_points(DA == DA_POSES ? 1 : DA == DA_POSES2 ? 2 : APL);
  constexpr bool SHARED = DAM != 0 && DA > 2;
  const int tid = threadIdx.x;
  Split sp;
  sp.ns = P.unsplit ? 1 : pk.ns;
  sp.half = P.unsplit ? (int)blockDim.x : pk.half;
  // half is a multiple of 64, so the group index is wave-uniform. Shares of a
  // chunk are rounded so that later groups hold more points; waves i and i + 4
  // share a SIMD, so the second half of the waves takes the groups in reverse
  // order and every SIMD gets a long and a short one.
  const int hw = __builtin_amdgcn_readfirstlane(tid / sp.half);
  sp.h = 2 * hw < sp.ns || hw >= sp.ns ? hw : sp.ns + sp.ns / 2 - 1 - hw;
  sp.ltid = tid - hw * sp.half;
  sp.slots = sp.half / 8;
  sp.xp_floats = P.xp_floats;
  sp.par = par;
  const int slot = sp.ltid / lpr;
  sp.slot = slot;
  const int a = sp.ltid - slot * lpr;
  const bool lead = a == 0 && sp.h == 0;  // writes the replica's results
  const int n_slots = pk.n_slots;
  const bool active = slot < n_slots && sp.h < sp.ns;
  const int sl = active ? slot : 0;
  const int sv = P.slots[pk.slot_off + sl];  // replica id or pose index
  const int lna = C.lna;
  const int n_lig = C.n_lig;

  int flat = 0, ilig;
  float mo[6];
  gd_energy eo;
  if (POSES || P.mode == MODE_EVAL || P.mode == MODE_SUREVAL) {
    ilig = P.ev_lig[sv];
#pragma unroll
    for (int i = 0; i < 6; ++i) mo[i] = P.ev_mm[(size_t)sv * 6 + i];
  } else {
    flat = P.rep_flat[sv];
    ilig = flat % n_lig;
#pragma unroll
    for (int i = 0; i < 6; ++i) mo[i] = P.mm[(size_t)sv * 6 + i];
    eo = P.e_old[sv];
  }

  // the lane's atoms: l = a + k*lpr
  float ox[APL], oy[APL], oz[APL], q[APL];
  int lt[APL], li[APL];
  bool val[APL];
  const float *orig = C.lig_orig + (size_t)ilig * 3 * lna;
#pragma unroll
  for (int k = 0; k < APL; ++k) {
    const int l = a + k * lpr;
    val[k] = l < lna;
    const int lc = val[k] ? l : 0;
    li[k] = lc;
    ox[k] = orig[lc];
    oy[k] = orig[lna + lc];
    oz[k] = orig[2 * lna + lc];
    lt[k] = C.lig_t[lc];
    q[k] = C.lig_c[lc];
  }

  float x[APL], y[APL], z[APL];
  Rot Rp{};  // rotation of the last placed pose (the surrogate's MCS moments use it)
  auto place = [&](const float m[6]) {
    const Rot R = euler(m[3], m[4], m[5]);
    Rp = R;
#pragma unroll
    for (int k = 0; k < APL; ++k) {
      x[k] = R.r00 * ox[k] + R.r01 * oy[k] + R.r02 * oz[k] + m[0] + C.pocket[0];
      y[k] = R.r10 * ox[k] + R.r11 * oy[k] + R.r12 * oz[k] + m[1] + C.pocket[1];
      z[k] = R.r20 * ox[k] + R.r21 * oy[k] + R.r22 * oz[k] + m[2] + C.pocket[2];
    }
  };

  if constexpr (DAM) {
    if (P.mode == MODE_SUREVAL) {
      extern __shared__ __attribute__((aligned(16))) unsigned char lds_se[];
      unsigned char *dse = lds_se + P.off_da + (threadIdx.x >> 6) * 6208;
      place(mo);
      const bool live = __ballot(active) != 0;
      float sv_s;
      if constexpr (SHARED) {
        sv_s = (sp.ns > 1 && C.da_share != 0)
                   ? sur_total<APL, DAM, true>(P, C, S, sp, live, dse, lpr, pk.prt, x, y, z, lt,
                                               val, mo, Rp, a, ilig)
                   : sur_total<APL, DAM, false>(P, C, S, sp, live, dse, lpr, pk.prt, x, y, z, lt,
                                                val, mo, Rp, a, ilig);
      } else {
        sv_s = sur_total<APL, DAM, false>(P, C, S, sp, live, dse, lpr, pk.prt, x, y, z, lt, val,
                                          mo, Rp, a, ilig);
      }
      if (active && lead) P.ev_sur[sv] = sv_s;
      par = sp.par;
      return;
    }
  }
  if (TREE || POSES || P.mode != MODE_MC) {
    if constexpr (TREE) tree_pose(P, C, flat, a, (threadIdx.x & 63) - a, step0, node + 1, mo);
    place(mo);
    gd_energy E;
    pose_energy<APL, TILE, FLAT, J, NP, SKIP>(C, S, lpr, sp, true, x, y, z, ox, oy, oz, lt, q, li, val, mo, E);
    par = sp.par;
    if constexpr (TREE) {
      // the wave of group 0 writes: its energies are visible on the device
      // before the node is counted, and are read after the last count
      if (active && lead) P.ev_out[(size_t)sv * P.tree_nodes + node] = E;
      if (sp.h == 0) __threadfence();
      __syncthreads();
      if (tid == 0) S.xo[0] = atomicAdd(P.tree_cnt + P.pack_base + idx, 1);
      __syncthreads();
      if (S.xo[0] != P.tree_nodes - 1) return;
      __threadfence();
      if (tid == 0) P.tree_cnt[P.pack_base + idx] = 0;
      for (int i = __builtin_amdgcn_readfirstlane(tid >> 6); i < n_slots;
           i += (int)(blockDim.x >> 6))
        tree_decide(P, C, pk.prt, P.slots[pk.slot_off + i], step0);
      return;
    }
    if (active && lead) {
      if (POSES || P.mode == MODE_EVAL) {
        P.ev_out[sv] = E;
      } else {
        P.e_old[sv] = E;
        P.best_e[sv] = E.e[GD_MAXWEI - 1];
#pragma unroll
        for (int i = 0; i < 6; ++i) P.best_mm[(size_t)sv * 6 + i] = mo[i];
        if (P.rec) {
          const int rc = P.rec_cnt[sv];
          if (rc < P.rec_cap) {
            gd_record &r = P.rec[(size_t)sv * P.rec_cap + rc];
            r.replica.idx_rep = flat;
            r.replica.idx_prt = pk.prt;
            r.replica.idx_tmp = P.idx_tmp[sv];
            r.replica.idx_lig = ilig;
            r.energy = E;
            for (int i = 0; i < 6; ++i) r.movematrix[i] = mo[i];
            r.step = step0;
            P.rec_cnt[sv] = rc + 1;
          }
        }
      }
    }
    return;
  }

  // ---- MC steps ------------------------------------------------------------
  const int cid = C.cid;
  const int nc = P.nc;
  float mb = C.minus_beta[S.xi[sl]];
  int acs = 0;
  int rc = P.rec ? P.rec_cnt[sv] : 0;
  float best = P.best_e[sv];
  auto track_best = [&]() {
    if (eo.e[GD_MAXWEI - 1] < best) {
      best = eo.e[GD_MAXWEI - 1];
      if (active && lead)
#pragma unroll
        for (int i = 0; i < 6; ++i) P.best_mm[(size_t)sv * 6 + i] = mo[i];
    }
  };
  const bool wave_active = __ballot(active) != 0;
  float scale[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) scale[i] = C.move_scale[i];

  auto record = [&](const gd_energy &E, int step) {
    if (P.rec && active) {
      if (lead && rc < P.rec_cap) {
        gd_record &r = P.rec[(size_t)sv * P.rec_cap + rc];
        r.replica.idx_rep = flat;
        r.replica.idx_prt = pk.prt;
        r.replica.idx_tmp = S.xi[sl];
        r.replica.idx_lig = ilig;
        r.energy = E;
        for (int i = 0; i < 6; ++i) r.movematrix[i] = mo[i];
        r.step = step;
      }
      rc += 1;
    }
  };
  // delayed acceptance (surrogate transition): K surrogate Metropolis
  // sub-steps, then one exact test of the composite move with
  // min(1, exp(-beta [(E(y) - E(x)) - (S(y) - S(x))]))
  const int K = DAM ? P.da_k : 1;
  unsigned char *da = nullptr;
  float s_old = 0.0f;
  // the split's groups share the surrogate's KDE and MCS sums for complexes
  // with large KDE or MCS sets (one exchange per surrogate evaluation, so
  // every thread evaluates it together)
  const bool share = SHARED && sp.ns > 1 && C.da_share != 0;
  if constexpr (DAM) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_da[];
    da = lds_da + P.off_da + (threadIdx.x >> 6) * 6208;
    if (wave_active) place(mo);
    if constexpr (SHARED) {
      if (share)
        s_old = sur_total<APL, DAM, true>(P, C, S, sp, wave_active, da, lpr, pk.prt, x, y, z, lt,
                                          val, mo, Rp, a, ilig);
    }
    if (!share && wave_active)
      s_old = sur_total<APL, DAM, false>(P, C, S, sp, true, da, lpr, pk.prt, x, y, z, lt, val, mo,
                                         Rp, a, ilig);
  }

  for (int s = step0; s < step0 + P.n_steps; s += K) {
    if constexpr (!DAM) {
      float u[8], mn[6];
      if (wave_active) {
        float dm[6];
        mc_uniforms(P.k0, P.k1, cid, flat, s, u);
        move_offsets(u, scale, C.move_kind, dm);
        apply_move(mo, dm, mn);
        place(mn);
      }
      gd_energy E;
      pose_energy<APL, TILE, FLAT, J, NP, SKIP>(C, S, lpr, sp, wave_active, x, y, z, ox, oy, oz, lt, q, li, val, mn, E);
      if (wave_active && metropolis(E.e[GD_MAXWEI - 1], eo.e[GD_MAXWEI - 1], mb, u[6])) {
#pragma unroll
        for (int i = 0; i < 6; ++i) mo[i] = mn[i];
        eo = E;
        acs += 1;
        record(E, s);
        track_best();
      }
    } else {
      float yv[6];
#pragma unroll
      for (int i = 0; i < 6; ++i) yv[i] = mo[i];
      float s_y = s_old, u7 = 1.0f;
      bool moved = false;
      if (!share) {
        for (int j = 0; wave_active && j < K; ++j) {
          float u[8], dm[6], mn[6];
          mc_uniforms(P.k0, P.k1, cid, flat, s + j, u);
          move_offsets(u, scale, C.move_kind, dm);
          apply_move(yv, dm, mn);
          place(mn);
          const float s_n = sur_total<APL, DAM, false>(P, C, S, sp, true, da, lpr, pk.prt, x, y,
                                                       z, lt, val, mn, Rp, a, ilig);
          if (metropolis(s_n, s_y, mb, u[6])) {
#pragma unroll
            for (int i = 0; i < 6; ++i) yv[i] = mn[i];
            s_y = s_n;
            moved = true;
          }
          u7 = u[7];
        }
      } else if constexpr (SHARED) {
        // every wave runs the K evaluations: their exchanges are workgroup
        // barriers
        for (int j = 0; j < K; ++j) {
          float u[8], dm[6], mn[6];
          if (wave_active) {
            mc_uniforms(P.k0, P.k1, cid, flat, s + j, u);
            move_offsets(u, scale, C.move_kind, dm);
            apply_move(yv, dm, mn);
            place(mn);
          }
          const float s_n = sur_total<APL, DAM, true>(P, C, S, sp, wave_active, da, lpr, pk.prt,
                                                      x, y, z, lt, val, mn, Rp, a, ilig);
          if (wave_active) {
            if (metropolis(s_n, s_y, mb, u[6])) {
#pragma unroll
              for (int i = 0; i < 6; ++i) yv[i] = mn[i];
              s_y = s_n;
              moved = true;
            }
            u7 = u[7];
          }
        }
      }
      const bool eval = wave_active && __ballot(moved) != 0;
      if (eval) place(yv);
      gd_energy E;
      pose_energy<APL, TILE, FLAT, J, NP, SKIP>(C, S, lpr, sp, eval, x, y, z, ox, oy, oz, lt, q, li, val, yv, E);
      if (eval) {
        const float d1 = E.e[GD_MAXWEI - 1] - eo.e[GD_MAXWEI - 1];
        const float d2 = s_y - s_old;
        const float delta = d1 - d2;
        const float prod = delta * mb;
        if (moved && u7 < decision_expf(prod)) {
#pragma unroll
          for (int i = 0; i < 6; ++i) mo[i] = yv[i];
          eo = E;
          s_old = s_y;
          acs += 1;
          record(E, s + K - 1);
          track_best();
        }
      }
    }
    if (nc > 0 && ((s + K) % nc) == 0) {
      if (active && lead) S.xe[slot] = eo.e[GD_MAXWEI - 1];
      __syncthreads();
      if (tid < pk.n_groups) {
        const int n_tmp = C.n_tmp;
        const int seg = (s + K) / nc - 1;
        const int mode_t = (seg % 2 == 0) ? 1 : 0;
        const int f0 = P.rep_flat[P.slots[pk.slot_off + tid * n_tmp]];
        const int group = (f0 / (n_tmp * n_lig)) * n_lig + (f0 % n_lig);
        const int b = tid * n_tmp;
        exchange_ladder(n_tmp, mode_t, S.xe + b, C.minus_beta, S.xi + b, S.xa + b, S.xo + b,
                        [&](int pair) {
                          return exchange_uniform(P.k0, P.k1, cid, group, seg, pair);
                        });
      }
      __syncthreads();
      mb = C.minus_beta[S.xi[sl]];
    }
  }

  if (active && lead) {
#pragma unroll
    for (int i = 0; i < 6; ++i) P.mm[(size_t)sv * 6 + i] = mo[i];
    P.e_old[sv] = eo;
    P.best_e[sv] = best;
    P.idx_tmp[sv] = S.xi[slot];
    P.acs_mc[sv] += acs;
    P.acs_x[sv] = S.xa[slot];
    if (P.rec) P.rec_cnt[sv] = rc < P.rec_cap ? rc : P.rec_cap;
  }
}

template <int APL, int DA, bool TILE, bool FLAT>
__device__ __forceinline__ void mc_kernel_body(const KParams &P, int idx, int step0) {
  int node = 0;
  if constexpr (DA == DA_TREE) {
    node = idx / P.tree_packs;
    idx -= node * P.tree_packs;
  }
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const Pack pk = P.packs[P.pack_base + idx];
  const DevComplex &C = P.cxs[pk.cx];
  Lds S;
  S.xyze = reinterpret_cast<const float4 *>(lds);
  S.hpp = reinterpret_cast<const float *>(lds + P.off_hpp);
  S.psp = reinterpret_cast<const int *>(lds + P.off_psp);
  S.par = reinterpret_cast<const float *>(lds + P.off_par);
  S.kde = reinterpret_cast<const float4 *>(lds + P.off_kde);
  S.kr = reinterpret_cast<const int2 *>(lds + P.off_kr);
  S.ch = reinterpret_cast<const int4 *>(lds + P.off_ch);
  S.fl = reinterpret_cast<const float4 *>(lds);
  S.xe = reinterpret_cast<float *>(lds + P.off_xe);
  S.xi = reinterpret_cast<int *>(lds + P.off_xi);
  S.xa = reinterpret_cast<int *>(lds + P.off_xa);
  S.xo = reinterpret_cast<int *>(lds + P.off_xo);
  S.xp = reinterpret_cast<float *>(lds + P.off_xp);
  const int pnp = C.pnp;
  const float4 *src = C.prt_xyze + (size_t)pk.prt * pnp;
  S.gx = src;
  S.ghpp = C.prt_hpp;
  S.gpsp = C.prt_psp;
  S.tx = reinterpret_cast<float4 *>(lds);
  S.th = reinterpret_cast<float *>(lds + P.off_hpp);
  S.tp = reinterpret_cast<int *>(lds + P.off_psp);
  S.tile = P.tile;
  if constexpr (TILE) S.kde = C.kde;  // KDE points are read from HBM

  // stage the pack's receptor conformer (unless it streams in tiles) and tables
  const int nt = blockDim.x;
  {
    float4 *xyze = reinterpret_cast<float4 *>(lds);
    float *hpp = reinterpret_cast<float *>(lds + P.off_hpp);
    int *psp = reinterpret_cast<int *>(lds + P.off_psp);
    const gfloat4_p gsrc = (gfloat4_p)src;
    const gfloat_p ghpp = glob(C.prt_hpp);
    const gint_p gpsp = (gint_p)C.prt_psp;
    if constexpr (FLAT) {
      // each unit: its two points of this conformer and its attributes
      const int fi = flat_index(pk.ns);
      const int n_units = C.flat_off[fi][pk.ns];
      const gint4_p units = (gint4_p)C.flat[fi];
      for (int i0 = threadIdx.x; i0 < n_units; i0 += 2 * nt) {
        i32x4_t f[2];
        f32x4_t A[2], B[2];
        float h0[2], h1[2];
        int s0[2], s1[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) f[j] = units[min(i0 + j * nt, n_units - 1)];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int p0 = f[j][1] & 0xffff, p1 = (unsigned)f[j][1] >> 16;
          A[j] = gsrc[p0];
          B[j] = gsrc[p1];
          h0[j] = ghpp[p0];
          h1[j] = ghpp[p1];
          s0[j] = gpsp[p0];
          s1[j] = gpsp[p1];
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int i = i0 + j * nt;
          if (i >= n_units) break;
          f32x4_t *u = reinterpret_cast<f32x4_t *>(xyze + FLAT_F4 * i);
          u[0] = A[j];
          u[1] = B[j];
          *reinterpret_cast<int4 *>(xyze + FLAT_F4 * i + 2) =
              make_int4(f[j][0], __float_as_int(0.5f * h0[j]), __float_as_int(0.5f * h1[j]),
                        (s0[j] & 0xffff) | (s1[j] << 16));
        }
      }
    } else if constexpr (!TILE) {
      stage_lds(reinterpret_cast<f32x4_t *>(xyze), gsrc, pnp, nt);
      stage_lds(hpp, ghpp, pnp, nt, [](float v) { return 0.5f * v; });
      stage_lds(psp, gpsp, pnp, nt);
    }
    if constexpr (!TILE)
      stage_lds(reinterpret_cast<f32x4_t *>(lds + P.off_kde), (gfloat4_p)C.kde, C.pnk, nt);
    static_assert(PAR_FLOATS % 4 == 0, "parameter records are staged 16 bytes at a time");
    stage_lds(reinterpret_cast<f32x4_t *>(lds + P.off_par), (gfloat4_p)C.params, PAR_FLOATS / 4, nt);
    stage_lds(reinterpret_cast<i32x2_t *>(lds + P.off_kr), (gint2_p)C.kde_range, NLT, nt);
    stage_lds(reinterpret_cast<i32x4_t *>(lds + P.off_ch), (gint4_p)C.chunks, C.n_chunks, nt);
    if (P.mode == MODE_MC) {
      for (int i = threadIdx.x; i < pk.n_slots; i += nt) {
        const int g = P.slots[pk.slot_off + i];
        S.xi[i] = P.idx_tmp[g];
        S.xa[i] = P.acs_x[g];
      }
    }
  }
  __syncthreads();

  int par = 0;
  const int lpr = DA == DA_POSES || DA == DA_POSES2 ? P.ev_lpr : C.lpr;
  if constexpr (FLAT) {
    // rounds of poses on the staged receptor (MC packs have one round); the
    // exchange buffers' parity runs on, so a round's first exchange does not
    // touch what the round before it may still be reading
    Pack q = pk;
    for (int b = 0; b < pk.n_slots; b += pk.round) {
      q.slot_off = pk.slot_off + b;
      q.n_slots = min(pk.round, pk.n_slots - b);
      run_pack<APL, DA, TILE, FLAT>(P, q, C, S, lpr, step0, idx, node, par);
    }
  } else {
    run_pack<APL, DA, TILE, FLAT>(P, pk, C, S, lpr, step0, idx, node, par);
  }
}

// MC kernel for packs whose complexes place APL ligand atoms on each lane:
// plain MC, start-pose evaluation and pose evaluation (DA = 0), plain MC by a
// tree of energies (DA_TREE), or delayed acceptance with surrogate sub-steps. One instance per
// APL keeps each variant's register allocation to what it needs.
template <int APL, int DA, bool TILE, bool FLAT>
__global__ void __launch_bounds__(512) gd_mc_kernel(KParams P) {
  const int step0 = P.step_dev ? *P.step_dev : P.step0;
  // persistent launches: each workgroup takes packs in LPT order from a
  // counter until none is left; otherwise one pack per workgroup
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_q[];
  int *next = reinterpret_cast<int *>(lds_q + P.off_q);
  const bool persistent = P.queue != nullptr;
  int idx = blockIdx.x;
  for (;;) {
    if (persistent) {
      if (threadIdx.x == 0) *next = atomicAdd(P.queue, 1);
      __syncthreads();
      idx = *next;
      __syncthreads();  // every thread has read the index; the previous pack's LDS is free
      if (idx >= P.n_queue) break;
    }
    mc_kernel_body<APL, DA, TILE, FLAT>(P, idx, step0);
    if (!persistent) break;
  }
}

}  // namespace gd
