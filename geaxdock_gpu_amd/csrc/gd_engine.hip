// gd_engine.hip -- host side of the C ABI in include/geauxdock.h.
//
// Replaces Run() and its single-GPU launcher (src/run.cu:33-289,
// src/kernel_cuda_lancher_siglegpu.cu:5-69): uploads complexes once, keeps
// all replica state resident in HBM, and advances every replica of every
// complex with one fused kernel launch per record window.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <limits>
#include <string>
#include <vector>

#include "gd_sur.hip"
#include "gd_util.hip"

using namespace gd;

// Device scratch of gd_calc_energy_noalloc: the pose tables and the energies
// of one call (packs, slots, conformer indices, movematrices, outputs), so
// that entry point allocates nothing. One copy per GPU, held until the
// process ends; host code reaches it only through the address
// hipGetSymbolAddress returns for the current device (gd_ctx::scratch).
static __device__ __align__(256) unsigned char scratch[GD_NOALLOC_SCRATCH_BYTES];

namespace {

// One kernel launch of a pack set: packs [begin, end) share the atoms-per-lane
// kernel instance, the LDS layout and the block shape.
struct LaunchClass {
  int apl = 1, begin = 0, end = 0;
  int tile = 0;      // receptor tile length (0: receptor resident in LDS)
  int block = 64;    // lanes: each pack's ns groups of its `half` lanes
  int half_max = 64;  // largest pack half (the block of an unsplit launch)
  size_t lds = 0;    // dynamic LDS bytes
  KParams lay{};     // LDS offsets and exchange-buffer fields
  size_t lds_flat = 0;  // the same with the receptor as units of the flat
  KParams lay_flat{};   // pair loop (0: none)
  bool near = false;  // chunk loop without distance tests (DA_NEAR)
};

struct HostComplex {
  gd_complex_desc d;  // sizes, scalars (pointers are not kept)
  int n_rep = 0, rep_base = 0;
  int lpr = 0, apl = 0, n_chunks = 0;
  int lpr0 = 0, apl0 = 0;  // the shape of fewest lane slots (lpr and apl may be widened)
  bool tiled = false;  // receptor streamed through LDS tiles
  bool ref_built = false;
  float far_share = 0.0f;  // share of receptor points far from the start pose
  int flat_n[4] = {0, 0, 0, 0};  // units of the flat pair loop by split (0: no list)
  bool shape_final = false;  // lane shape fixed (the complex's energies have bits)
  std::vector<int4> chunks;  // receptor chunks (host copy)
  std::vector<int> lig_t;  // ligand atom types (host copy)
  std::vector<int> lig_ns;  // receptor split of each ligand conformer's MC packs
  DevComplex dev{};
  std::vector<void *> bufs;  // device allocations owned by this complex
  size_t lds_bytes = 0;
};

// A buffer that a context keeps between calls, grown to the largest need so
// far and given back after a call that needed more than SCRATCH_KEEP bytes.
struct Scratch {
  unsigned char *p = nullptr;
  size_t cap = 0;
};
constexpr size_t SCRATCH_KEEP = (size_t)256 << 20;

constexpr int GRID_ROWS = 32768;  // rows (grid.y, 16 bits) of a launch
constexpr int SIDE_STREAMS = 3;  // streams beside the main one for launch classes

}  // namespace

struct gd_ctx {
  gd_opts opts{};
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  // side streams for concurrent launches of the per-APL kernel classes
  hipStream_t aux[SIDE_STREAMS] = {};
  hipEvent_t ev_fork = nullptr, ev_join[SIDE_STREAMS] = {};
  std::string err;
  int n_cu = 0;
  size_t max_lds = 65536;
  unsigned char *scratch = nullptr;  // this device's copy of the file-scope scratch array
  // staging of the calls that take or return host arrays: pinned host memory
  // (also read and written by kernels directly for small calls) and device
  // memory; `drain` is the record drains' own pinned staging (a drain runs
  // beside a window)
  Scratch pin, dev, drain_pin, tree;
  int64_t *h_counts = nullptr;  // pinned: accepted moves and exchanges before and after a run
  std::vector<HostComplex> cx;
  std::vector<void *> flat_bufs;  // unit lists of the flat pair loop
  bool flat = false;              // packs with unit lists use them
  DevComplex *d_cx = nullptr;
  bool cx_dirty = true;
  // replica state
  bool state_alloc = false, initialized = false;
  int n_rep = 0;
  int64_t step = 0;
  float *d_mm = nullptr;
  gd_energy *d_eold = nullptr;
  float *d_best_e = nullptr, *d_best_mm = nullptr;
  int *d_idx_tmp = nullptr, *d_acs_mc = nullptr, *d_acs_x = nullptr, *d_rep_flat = nullptr;
  // record rings: the MC kernels append accepted states to ring `ring`; with
  // a sink, windows alternate between two rings so one window's records are
  // drained while the next window runs (ring 1 is allocated on first use)
  gd_record *d_ring[2] = {nullptr, nullptr};
  int *d_ring_cnt[2] = {nullptr, nullptr};
  int ring = 0;
  int rec_cap = 0;
  hipStream_t drain_stream = nullptr;
  hipEvent_t ev_compact = nullptr;  // the pending window is compacted
  // record drains: device offsets and compacted window, and the pinned host
  // staging buffer the sink reads, grown as needed and reused across windows
  int64_t *d_drain_off = nullptr;
  gd_record *d_drain = nullptr, *h_drain = nullptr;
  int64_t d_drain_cap = 0, h_drain_cap = 0;
  int64_t drain_total = 0;  // records of the compacted window (their offsets: drain_pin)
  // packs of the MC launch
  Pack *d_packs = nullptr;
  int *d_slots = nullptr;
  int n_packs = 0, ladders_per_pack = 0;
  // spread packing: ladders exchanged between launches, (complex, ladder,
  // replica of slot 0, replica stride)
  int4 *d_ladders = nullptr;
  int n_ladders = 0;
  std::vector<LaunchClass> mc_classes;  // kernel launches of the MC pack set
  // device control words: [0] first step of a graph replay, [1 + i] pack
  // counter of class i in persistent launches
  int *d_ctrl = nullptr;
  int h_step = 0;  // host source of the step upload (outlives the async copy)
  // captured MC launch per record ring (one graph per window shape)
  struct GraphSlot {
    hipGraphExec_t exec = nullptr;
    bool valid = false;
    int mode = -1, win = 0, nc = 0, da = 0, tab = 0, persistent = 0;
    float scale = 0.0f;
  } gslot[2];
  // learned surrogate
  struct Sur {
    std::vector<float *> grid;  // per complex [n_prt][n^3][32]
    std::vector<SurGrid> g;
    std::vector<float *> tab;   // per complex [n_prt][NLT][n^3] network outputs
    std::vector<size_t> grid_n, tab_n;  // floats held by each of them
    bool tab_valid = false;     // tab holds the current parameters' outputs
    float *p = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr;  // FP32 master + Adam
    unsigned short *W1T = nullptr, *W2T = nullptr, *W2R = nullptr;    // bf16 layouts
    int64_t adam_t = 0;
    bool have_params = false;
    // dataset (rows padded, last 64 rows zero)
    unsigned short *X = nullptr;  // feature rows [cap + 64][64] bf16
    int64_t rows = 0, cap = 0;
    std::vector<int64_t> off{0};  // pose row offsets
    std::vector<float> target;
    std::vector<int> pose_cx;
    int64_t *d_off = nullptr;
    float *d_target = nullptr;
    bool dirty = true;
    // work buffers
    float *y = nullptr, *dS = nullptr, *sq = nullptr, *S = nullptr;
    float *p1 = nullptr, *p2 = nullptr, *pb2 = nullptr, *pw3 = nullptr;
    float *dyr = nullptr;  // per-row output gradient of the current batch
    float *bl = nullptr;   // per-batch sums of squared residuals of an epoch
    int64_t work_rows = 0, work_poses = 0, work_batches = 0;
    int last_groups = 0;  // backward workgroups (partials) of the last batch
  } sur;
};

namespace {

gd_status fail(gd_ctx *c, gd_status s, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  if (c) c->err = buf;
  // the runtime keeps a failed call's error until it is asked for: it is
  // reported here and must not be found by the next call's launch check
  if (s == GD_ERR_HIP || s == GD_ERR_NOMEM) (void)hipGetLastError();
  return s;
}

#define HIPCHK(expr)                                                                  \
  do {                                                                                \
    hipError_t e_ = (expr);                                                           \
    if (e_ != hipSuccess)                                                             \
      return fail(ctx, GD_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(e_));    \
  } while (0)

#define TRY(expr)                      \
  do {                                 \
    gd_status s_ = (expr);             \
    if (s_ != GD_OK) return s_;        \
  } while (0)

void scratch_free(Scratch &s, bool pinned) {
  if (s.p) (void)(pinned ? hipHostFree(s.p) : hipFree(s.p));
  s = Scratch{};
}

// At least `bytes` in the scratch buffer (its contents are lost when it grows).
gd_status scratch_need(gd_ctx *ctx, Scratch &s, size_t bytes, bool pinned) {
  if (s.cap >= bytes) return GD_OK;
  scratch_free(s, pinned);
  const size_t cap = (bytes + bytes / 4 + 65535) & ~(size_t)65535;
  void *p = nullptr;
  if (pinned) HIPCHK(hipHostMalloc(&p, cap, hipHostMallocDefault));
  else HIPCHK(hipMalloc(&p, cap));
  s.p = static_cast<unsigned char *>(p);
  s.cap = cap;
  return GD_OK;
}

// Gives the context's scratch back at the end of a call if it is large.
struct ScratchTrim {
  gd_ctx *ctx;
  ~ScratchTrim() {
    if (ctx->pin.cap > SCRATCH_KEEP) scratch_free(ctx->pin, true);
    if (ctx->dev.cap > SCRATCH_KEEP) scratch_free(ctx->dev, false);
  }
};

// Regions of one scratch buffer, each 256-byte aligned.
struct Regions {
  size_t end = 0;
  size_t add(size_t bytes) {
    const size_t o = end;
    end = (end + bytes + 255) & ~(size_t)255;
    return o;
  }
};

// Calls whose arrays stay below this go without copies: kernels read their
// inputs from the pinned staging and write their results there. A copy costs
// 5 to 10 us each way whatever its size; these reads cross the bus once.
constexpr size_t ZERO_COPY_BYTES = 65536;

// Squared distance beyond which every pair of the complex can go without the
// PMF's exponential, HPC and the contact terms, with the same bits: there
// e <= 2^-26, so den + den e and num + num e round to den and num; u is 0; no
// contact or near electrostatic form holds. The PMF exponent's upper root of
// (d - 12)(d - pmf0) = 2 * 26 / log2(e). Infinite (nothing is skipped) for
// values with which a skipped term could be other than an exact zero: those
// not finite, or so large that a distance's ninth power overflows.
float skip_range2(const gd_complex_desc &d, const std::vector<float> &par) {
  const float none = std::numeric_limits<float>::infinity();
  for (size_t i = 0; i < (size_t)d.n_prt * d.pnp; ++i)
    if (!(std::fabs(d.prt_x[i]) < FAR_COORD && std::fabs(d.prt_y[i]) < FAR_COORD &&
          std::fabs(d.prt_z[i]) < FAR_COORD))
      return none;
  bool lt[NLT] = {}, pt[NPT] = {};
  for (int l = 0; l < d.lna; ++l) lt[d.lig_t[l]] = true;
  for (int p = 0; p < d.pnp; ++p) {
    pt[d.prt_t[p]] = true;
    if (!std::isfinite(d.prt_hpp[p])) return none;
  }
  double r2 = 82.0;
  for (int j = 0; j < NPT; ++j)
    for (int i = 0; i < NLT; ++i) {
      if (!pt[j] || !lt[i]) continue;
      const float *r = &par[(j * NLT + i) * NPAR];
      for (int q : {P_P1A, P_P2A, P_A0, P_A1, P_HA, P_HB, P_HC})
        if (!(std::fabs(r[q]) < 1e20f)) return none;
      if (!(std::fabs(r[P_PMF0]) < 1e4f) || !(r[P_HA] >= 0.0f)) return none;
      const double p = r[P_PMF0], D = (12.0 - p) * (12.0 - p) + 8.0 * 26.0 / 1.4426950408889634;
      const double F = 0.5 * (12.0 + p + std::sqrt(D));
      r2 = std::max({r2, F * F, (double)r[P_NR2]});
    }
  return (float)(r2 * 1.002);
}

// Share of the receptor's points (first conformer) whose pairs the distance
// tests can skip around the start pose: points beyond far2 of a sphere of half
// the ligand's radius (which counts within 0.08 of the points that are that
// far from every atom).
float far_share(const gd_complex_desc &d, float far2) {
  if (!std::isfinite(far2)) return 0.0f;
  float r2 = 0.0f;
  for (int l = 0; l < d.lna; ++l)
    r2 = std::max(r2, d.lig_x[l] * d.lig_x[l] + d.lig_y[l] * d.lig_y[l] + d.lig_z[l] * d.lig_z[l]);
  const float reach = std::sqrt(far2) + 0.5f * std::sqrt(r2);
  int n = 0;
  for (int p = 0; p < d.pnp; ++p) {
    const float x = d.prt_x[p] - d.pocket_center[0], y = d.prt_y[p] - d.pocket_center[1],
                z = d.prt_z[p] - d.pocket_center[2];
    n += x * x + y * y + z * z > reach * reach ? 1 : 0;
  }
  return (float)n / (float)d.pnp;
}

// Launches by chunks or tiles go without the loop's distance tests (DA_NEAR, same bits)
// where these cost more than they skip. At a wave per SIMD (blocks of at most
// 256 lanes) nothing hides the tests' branches: 64 ladders of 4 replicas of 30
// atoms, split 1, 2,000 points, 14.2 ms with tests and 12.1 without, 3,500 points
// 22.8 and 20.4; one pose on 1,200 points 116 us and 106; in tiles of 6,000 points
// (share 0.84) 14 atoms 22.9 and 26.2. At two waves per SIMD
// the tests pay from a share of far points on that falls with the atoms per
// lane (batches and ladders, tests first): 1 atom, 2,000 points (share 0.6) 5.8 ms
// and 5.5, 3,500 (0.77) 8.4 and 8.7; 2 atoms, 1,000 points (0.13) 65.8 and 63.1,
// 2,000 (0.44) 10.6 and 10.4, 2,500 (0.52) 139.9 and 142.9; 3 atoms, 800 points
// (0.07) 6.98 and 6.81, 1,000 (0.14) 76.6 and 77.3, 2,000 (0.46) 78.0 and 81.4.
constexpr int NEAR_BLOCK = 256;
constexpr float NEAR_SHARE_1WAVE = 0.8f;
constexpr float NEAR_SHARE[4] = {0.65f, 0.45f, 0.1f, 0.1f};

// Lanes per replica and atoms per lane: the fewest lane slots lpr*apl that
// hold lna atoms with apl <= 4, preferring 2..3 atoms per lane on ties (more
// independent work per lane), with a whole ladder within 512 lanes.
void choose_shape(int lna, int n_tmp, int force_lpr, int force_apl, int *lpr, int *apl) {
  int best_l = 64, best_a = (lna + 63) / 64, best_cost = 1 << 30;
  const int cands[4] = {8, 16, 32, 64};
  for (int ci = 0; ci < 4; ++ci) {
    const int l = cands[ci];
    if (force_lpr && l != force_lpr) continue;
    const int a = (lna + l - 1) / l;
    if (a > 4 || (force_apl && a > force_apl)) continue;
    const int aa = force_apl ? force_apl : a;
    if (l * n_tmp > 512 && !force_lpr) continue;
    const int cost = l * aa * 8 + std::abs(aa - 2);
    if (cost < best_cost) {
      best_cost = cost;
      best_l = l;
      best_a = aa;
    }
  }
  *lpr = best_l;
  *apl = best_a;
}

// Without spread packing, packs of the automatic split take the flat pair loop
// where a lane group's share of a receptor chunk is at most this many points on
// average (a split that the caller fixed keeps the chunk loop, with the block
// sizes it brings): short shares spend their time on a chunk's ends, which units do not have. Batches
// of 40 to 100 complexes of 600 to 3,300 points, whose packs are split 2, 4 and
// 8 ways (9 to 10 points a share): 38.7 ms by chunks, 36.1 by units at 64
// complexes, 26.8 and 25.8 at 40, 55.1 and 52.1 at 100. Unsplit packs (20 to
// 22 points): 77.3 ms by chunks, 104 by units at 150 complexes, 145.8 and
// 149.6 at 300, 21.7 and 22.0 for one complex of 220 ladders.
constexpr int FLAT_SHARE = 14;

// Default tile length of receptors that do not fit in LDS.
constexpr int DEFAULT_TILE = 256;

// LDS bytes of a complex's pack with `slots` replicas: the resident layout
// (tile = 0) holds the receptor conformer and KDE points, the tiled layout two
// receptor tiles.
size_t lds_need(const HostComplex &h, int slots, int tile) {
  const gd_complex_desc &d = h.d;
  const size_t pts = tile > 0 ? (size_t)2 * tile : (size_t)d.pnp;
  const size_t kde = tile > 0 ? 0 : (size_t)d.pnk * 16;
  // the receptor split's two exchange buffers of a 512-lane workgroup (any
  // pack of the complex may be split)
  const size_t xp = (size_t)2 * (11 * 512 / 2) * 4;
  return pts * 24 + PAR_FLOATS * 4 + kde + NLT * 8 + (size_t)h.n_chunks * 16 +
         (size_t)slots * 16 + xp + 256;
}

// Tile length of a complex's packs, 0 when its receptor stays resident.
int complex_tile(const gd_ctx *ctx, const HostComplex &h);

}  // namespace

extern "C" {

const char *gd_last_error(const gd_ctx *c) { return c ? c->err.c_str() : "null context"; }

gd_status gd_create(gd_ctx **out, const gd_opts *opts) {
  if (!out) return GD_ERR_INVALID;
  *out = nullptr;
  gd_ctx *ctx = new (std::nothrow) gd_ctx();
  if (!ctx) return GD_ERR_NOMEM;
  if (opts) ctx->opts = *opts;
  if (ctx->opts.steps_per_dump <= 0) ctx->opts.steps_per_dump = 2000;
  ctx->device = ctx->opts.device;
  int ndev = 0;
  hipError_t e = hipGetDeviceCount(&ndev);
  if (e != hipSuccess || ndev <= 0) {
    *out = ctx;
    return fail(ctx, GD_ERR_HIP, "no HIP device available (%s)", hipGetErrorString(e));
  }
  *out = ctx;
  HIPCHK(hipSetDevice(ctx->device));
  hipDeviceProp_t prop;
  HIPCHK(hipGetDeviceProperties(&prop, ctx->device));
  ctx->n_cu = prop.multiProcessorCount;
  ctx->max_lds = prop.sharedMemPerBlock;
  if (prop.maxSharedMemoryPerMultiProcessor > 0)
    ctx->max_lds = std::max<size_t>(ctx->max_lds, std::min<size_t>(prop.maxSharedMemoryPerMultiProcessor, 160 * 1024));
  if (ctx->opts.verbose)
    fprintf(stderr, "[geauxdock] %s: %d CUs, LDS/block %zu, LDS/CU %zu, regs/block %d\n",
            prop.gcnArchName, prop.multiProcessorCount, (size_t)prop.sharedMemPerBlock,
            (size_t)prop.maxSharedMemoryPerMultiProcessor, prop.regsPerBlock);
  HIPCHK(hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking));
  HIPCHK(hipEventCreate(&ctx->ev0));
  HIPCHK(hipEventCreate(&ctx->ev1));
  HIPCHK(hipGetSymbolAddress((void **)&ctx->scratch, HIP_SYMBOL(scratch)));
  return GD_OK;
}

void gd_destroy(gd_ctx *ctx) {
  if (!ctx) return;
  if (ctx->stream) {
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
  }
  for (auto &h : ctx->cx)
    for (void *p : h.bufs) (void)hipFree(p);
  for (void *p : ctx->flat_bufs) (void)hipFree(p);
  void *ps[] = {ctx->d_cx, ctx->d_mm, ctx->d_eold, ctx->d_idx_tmp,
                ctx->d_acs_mc, ctx->d_acs_x, ctx->d_rep_flat, ctx->d_ring[0], ctx->d_ring_cnt[0],
                ctx->d_packs, ctx->d_slots, ctx->d_best_e, ctx->d_best_mm, ctx->d_ctrl,
                ctx->d_drain_off, ctx->d_drain, ctx->d_ring[1], ctx->d_ring_cnt[1],
                ctx->d_ladders};
  if (ctx->h_drain) (void)hipHostFree(ctx->h_drain);
  if (ctx->h_counts) (void)hipHostFree(ctx->h_counts);
  scratch_free(ctx->pin, true);
  scratch_free(ctx->drain_pin, true);
  scratch_free(ctx->dev, false);
  scratch_free(ctx->tree, false);
  for (auto &g : ctx->gslot)
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
  for (void *p : ps)
    if (p) (void)hipFree(p);
  {
    auto &S = ctx->sur;
    for (float *g : S.grid)
      if (g) (void)hipFree(g);
    for (float *g : S.tab)
      if (g) (void)hipFree(g);
    void *qs[] = {S.p, S.m, S.v, S.grad, S.W1T, S.W2T, S.W2R, S.X, S.bl,
                  S.d_off, S.d_target, S.y, S.dS, S.sq, S.S, S.p1, S.p2, S.pb2, S.pw3,
                  S.dyr};
    for (void *p : qs)
      if (p) (void)hipFree(p);
  }
  if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
  if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
  if (ctx->ev_fork) (void)hipEventDestroy(ctx->ev_fork);
  for (int i = 0; i < SIDE_STREAMS; ++i) {
    if (ctx->ev_join[i]) (void)hipEventDestroy(ctx->ev_join[i]);
    if (ctx->aux[i]) (void)hipStreamDestroy(ctx->aux[i]);
  }
  if (ctx->ev_compact) (void)hipEventDestroy(ctx->ev_compact);
  if (ctx->drain_stream) (void)hipStreamDestroy(ctx->drain_stream);
  if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
  delete ctx;
}

gd_status gd_complex_shape(const gd_ctx *ctx, int cid, int *lpr, int *apl) {
  if (!ctx || cid < 0 || cid >= (int)ctx->cx.size() || !lpr || !apl) return GD_ERR_INVALID;
  *lpr = ctx->cx[cid].lpr;
  *apl = ctx->cx[cid].apl;
  return GD_OK;
}

int gd_num_replicas(const gd_ctx *ctx, int cid) {
  if (!ctx || cid < 0 || cid >= (int)ctx->cx.size()) return -1;
  return ctx->cx[cid].n_rep;
}

static gd_status add_complex(gd_ctx *ctx, const gd_complex_desc *d, int *complex_id);

gd_status gd_add_complex(gd_ctx *ctx, const gd_complex_desc *d, int *complex_id) {
  if (!ctx || !d) return GD_ERR_INVALID;
  const size_t n = ctx->cx.size();
  const gd_status st = add_complex(ctx, d, complex_id);
  // a complex that failed half-way has arrays missing: it leaves the context
  if (st != GD_OK && ctx->cx.size() > n) {
    for (void *p : ctx->cx.back().bufs) (void)hipFree(p);
    ctx->cx.pop_back();
  }
  return st;
}

static gd_status add_complex(gd_ctx *ctx, const gd_complex_desc *d, int *complex_id) {
  if (ctx->state_alloc) return fail(ctx, GD_ERR_STATE, "complexes must be added before gd_run");
  if (d->n_lig <= 0 || d->n_prt <= 0 || d->n_tmp <= 0 || d->lna <= 0 || d->pnp <= 0 ||
      d->pnk < 0 || d->pos < 0)
    return fail(ctx, GD_ERR_INVALID, "non-positive size in complex description");
  if (d->lna > GD_MAX_LNA) return fail(ctx, GD_ERR_CAPACITY, "lna %d > %d", d->lna, GD_MAX_LNA);
  if (d->n_tmp > GD_MAX_NTMP)
    return fail(ctx, GD_ERR_CAPACITY, "n_tmp %d > %d", d->n_tmp, GD_MAX_NTMP);
  if (!d->lig_x || !d->lig_y || !d->lig_z || !d->lig_t || !d->lig_c || !d->lig_n || !d->prt_x ||
      !d->prt_y || !d->prt_z || !d->prt_t || !d->prt_c || !d->prt_ele || !d->prt_seq3r ||
      !d->prt_c0_and_d12_or_c2 || !d->prt_hpp || !d->enepara || !d->temp)
    return fail(ctx, GD_ERR_INVALID, "null array in complex description");
  if (d->pnk > 0 && (!d->kde_x || !d->kde_y || !d->kde_z || !d->kde_t))
    return fail(ctx, GD_ERR_INVALID, "null KDE array");
  if (d->pos > 0 && (!d->mcs_x || !d->mcs_y || !d->mcs_z || !d->mcs_tcc || d->n_mcs <= 0))
    return fail(ctx, GD_ERR_INVALID, "null MCS array");
  const int lna = d->lna, pnp = d->pnp, pnk = d->pnk, pos = d->pos;
  for (int l = 0; l < lna; ++l) {
    if (d->lig_t[l] < 0 || d->lig_t[l] >= NLT)
      return fail(ctx, GD_ERR_INVALID, "ligand atom %d type %d out of range", l, d->lig_t[l]);
    if (pos > 0 && (d->lig_n[l] + 1 < 0 || d->lig_n[l] + 1 >= d->n_mcs))
      return fail(ctx, GD_ERR_INVALID, "ligand atom %d number %d outside MCS fields", l, d->lig_n[l]);
  }
  bool any_psp = false;
  for (int p = 0; p < pnp; ++p) {
    if (d->prt_t[p] < 0 || d->prt_t[p] >= NPT)
      return fail(ctx, GD_ERR_INVALID, "receptor point %d type %d out of range", p, d->prt_t[p]);
    if (d->prt_c[p] == 2) {
      any_psp = true;
      if (d->prt_seq3r[p] < 0 || d->prt_seq3r[p] >= d->n_res)
        return fail(ctx, GD_ERR_INVALID, "receptor point %d seq3r %d outside [0,%d)", p,
                    d->prt_seq3r[p], d->n_res);
    }
  }
  if (any_psp && !d->psp) return fail(ctx, GD_ERR_INVALID, "null PSP table");
  for (int k = 0; k < pnk; ++k)
    if (d->kde_t[k] < 0 || d->kde_t[k] >= NLT)
      return fail(ctx, GD_ERR_INVALID, "KDE point %d type out of range", k);

  if (!(d->enepara->el1 > 0.0f) || !(d->enepara->lj0 > 0.0f))
    return fail(ctx, GD_ERR_INVALID, "el1 and lj0 must be positive");
  HIPCHK(hipSetDevice(ctx->device));
  ctx->cx.emplace_back();
  HostComplex &h = ctx->cx.back();
  const int cid = (int)ctx->cx.size() - 1;
  h.d = *d;
  h.n_rep = d->n_lig * d->n_prt * d->n_tmp;
  h.lig_t.assign(d->lig_t, d->lig_t + d->lna);
  choose_shape(lna, d->n_tmp, ctx->opts.lanes_per_replica, ctx->opts.atoms_per_lane, &h.lpr,
               &h.apl);
  if (h.lpr * h.apl < lna || h.apl < 1 || h.apl > 4)
    return fail(ctx, GD_ERR_INVALID, "no lane shape for lna %d (lpr %d apl %d)", lna, h.lpr, h.apl);
  h.lpr0 = h.lpr;
  h.apl0 = h.apl;

  // receptor sorted by (type, kind); kind: 2 = class 2, 1 = hydrophobic flag
  std::vector<int> kind(pnp), perm(pnp);
  for (int p = 0; p < pnp; ++p) {
    kind[p] = d->prt_c[p] == 2 ? KIND_PSP : (d->prt_c0_and_d12_or_c2[p] == 1 ? KIND_HPC : KIND_PLAIN);
    perm[p] = p;
  }
  std::stable_sort(perm.begin(), perm.end(), [&](int a, int b) {
    if (d->prt_t[a] != d->prt_t[b]) return d->prt_t[a] < d->prt_t[b];
    return kind[a] < kind[b];
  });
  std::vector<float4> xyze((size_t)d->n_prt * pnp);
  for (int c = 0; c < d->n_prt; ++c)
    for (int i = 0; i < pnp; ++i) {
      const int p = perm[i];
      const size_t o = (size_t)c * pnp;
      // the electrostatic parameter is stored divided by el1 (far-field form)
      xyze[o + i] = make_float4(d->prt_x[o + p], d->prt_y[o + p], d->prt_z[o + p],
                                d->prt_ele[p] / d->enepara->el1);
    }
  std::vector<float> hpp(pnp);
  std::vector<int> pspi(pnp);
  for (int i = 0; i < pnp; ++i) {
    const int p = perm[i];
    hpp[i] = d->prt_c0_and_d12_or_c2[p] == 1 ? d->prt_hpp[p] : 0.0f;
    pspi[i] = d->prt_c[p] == 2 ? d->prt_seq3r[p] : -1;
  }
  std::vector<int4> chunks;
  for (int i = 0; i < pnp;) {
    int j = i;
    const int t = d->prt_t[perm[i]], k = kind[perm[i]];
    while (j < pnp && d->prt_t[perm[j]] == t && kind[perm[j]] == k) ++j;
    chunks.push_back(make_int4(i, j - i, t, k));
    i = j;
  }
  h.n_chunks = (int)chunks.size();
  h.chunks = chunks;

  // type-pair parameter records [receptor type][ligand type]
  const gd_enepara &ep = *d->enepara;
  std::vector<float> par(PAR_FLOATS, 0.0f);
  const float hsc = sqrtf(0.5f * 1.44269504088896340736f);
  const float sqrt_2_pi_m1 = -1.0f / sqrtf(2.0f * 3.1415926535f);
  for (int pt = 0; pt < NPT; ++pt)
    for (int lt = 0; lt < NLT; ++lt) {
      float *r = &par[(pt * NLT + lt) * NPAR];
      r[P_P1A] = ep.p1a[lt][pt];
      r[P_P2A] = ep.p2a[lt][pt];
      r[P_PMF0] = ep.pmf0[lt][pt];
      r[P_PMF1] = ep.pmf1[lt][pt];
      const float h0 = ep.hdb0[lt][pt], h1 = ep.hdb1[lt][pt];
      const bool on = h0 > 0.1f;
      r[P_HA] = on ? h1 * hsc : 0.0f;
      r[P_HB] = on ? -h0 * h1 * hsc : 0.0f;
      r[P_HC] = on ? sqrt_2_pi_m1 * h1 : 0.0f;
      // the per-chunk constants of the pair loop, with its FP32 expressions
      const float p1a = r[P_P1A], pmf0 = r[P_PMF0];
      const float rn = fmaxf(pmf0, 1.0f / ep.el1) * 1.0001f;
      r[P_NR2] = rn * rn;
      r[P_A0] = p1a * ep.lj0;
      r[P_A1] = p1a * (ep.lj0 * ep.lj1);
      r[P_PB] = LOG2E * fmaf(0.5f, pmf0, 6.0f);
      r[P_PC] = -6.0f * LOG2E * pmf0;
    }

  // ligand conformers [n_lig][3][lna]
  std::vector<float> orig((size_t)d->n_lig * 3 * lna);
  for (int c = 0; c < d->n_lig; ++c)
    for (int l = 0; l < lna; ++l) {
      const size_t o = (size_t)c * lna + l;
      orig[(size_t)c * 3 * lna + l] = d->lig_x[o];
      orig[(size_t)c * 3 * lna + lna + l] = d->lig_y[o];
      orig[(size_t)c * 3 * lna + 2 * lna + l] = d->lig_z[o];
    }
  // MCS fields by atom: [pos][lna]
  std::vector<float4> mcs((size_t)std::max(pos, 1) * lna);
  std::vector<float> mcnt(std::max(pos, 1), 0.0f), tcc(std::max(pos, 1), 0.0f);
  for (int m = 0; m < pos; ++m) {
    tcc[m] = d->mcs_tcc[m];
    for (int l = 0; l < lna; ++l) {
      const size_t o = (size_t)m * d->n_mcs + d->lig_n[l] + 1;
      const bool ok = d->mcs_x[o] != GD_MCS_INVALID_COORD;
      mcs[(size_t)m * lna + l] = make_float4(d->mcs_x[o], d->mcs_y[o], d->mcs_z[o], ok ? 1.0f : 0.0f);
      mcnt[m] += ok ? 1.0f : 0.0f;
    }
  }
  // MCS moments per (ligand conformer, template) for the closed-form
  // restraint of the surrogate path (double sums, stored as float)
  std::vector<float4> mcsq((size_t)std::max(d->n_lig * pos, 1) * 4, make_float4(0, 0, 0, 0));
  for (int c = 0; c < d->n_lig; ++c)
    for (int m = 0; m < pos; ++m) {
      double so[3] = {0, 0, 0}, sm[3] = {0, 0, 0};
      int n = 0;
      for (int l = 0; l < lna; ++l) {
        const float4 f = mcs[(size_t)m * lna + l];
        if (f.w == 0.0f) continue;
        const size_t o = (size_t)c * 3 * lna + l;
        so[0] += orig[o];
        so[1] += orig[o + lna];
        so[2] += orig[o + 2 * lna];
        sm[0] += f.x;
        sm[1] += f.y;
        sm[2] += f.z;
        n += 1;
      }
      if (n == 0) continue;
      double ob[3], mb[3], A = 0.0, M[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
      for (int i = 0; i < 3; ++i) {
        ob[i] = so[i] / n;
        mb[i] = sm[i] / n;
      }
      for (int l = 0; l < lna; ++l) {
        const float4 f = mcs[(size_t)m * lna + l];
        if (f.w == 0.0f) continue;
        const size_t o = (size_t)c * 3 * lna + l;
        const double op[3] = {orig[o] - ob[0], orig[o + lna] - ob[1], orig[o + 2 * lna] - ob[2]};
        const double mp[3] = {f.x - mb[0], f.y - mb[1], f.z - mb[2]};
        for (int i = 0; i < 3; ++i) {
          A += op[i] * op[i] + mp[i] * mp[i];
          for (int j = 0; j < 3; ++j) M[i][j] += mp[i] * op[j];
        }
      }
      float4 *q = &mcsq[((size_t)c * pos + m) * 4];
      q[0] = make_float4((float)A, (float)ob[0], (float)ob[1], (float)ob[2]);
      q[1] = make_float4((float)mb[0], (float)mb[1], (float)mb[2], (float)M[0][0]);
      q[2] = make_float4((float)M[0][1], (float)M[0][2], (float)M[1][0], (float)M[1][1]);
      q[3] = make_float4((float)M[1][2], (float)M[2][0], (float)M[2][1], (float)M[2][2]);
    }
  // KDE sorted by type with per-type ranges
  std::vector<int> kperm(pnk);
  for (int k = 0; k < pnk; ++k) kperm[k] = k;
  std::stable_sort(kperm.begin(), kperm.end(), [&](int a, int b) { return d->kde_t[a] < d->kde_t[b]; });
  std::vector<float4> kde(std::max(pnk, 1));
  std::vector<int2> krange(NLT, make_int2(0, 0));
  for (int i = 0; i < pnk; ++i) {
    const int k = kperm[i];
    kde[i] = make_float4(d->kde_x[k], d->kde_y[k], d->kde_z[k], 0.0f);
  }
  for (int t = 0; t < NLT; ++t) {
    int b = 0;
    while (b < pnk && d->kde_t[kperm[b]] < t) ++b;
    int e = b;
    while (e < pnk && d->kde_t[kperm[e]] == t) ++e;
    krange[t] = make_int2(b, e);
  }

  DevComplex &D = h.dev;
  D.lna = lna;
  D.pnp = pnp;
  D.pnk = pnk;
  D.pos = pos;
  D.n_res = d->n_res;
  D.n_lig = d->n_lig;
  D.n_prt = d->n_prt;
  D.n_tmp = d->n_tmp;
  D.n_chunks = h.n_chunks;
  D.lpr = h.lpr;
  D.apl = h.apl;
  D.move_kind = d->move_kind;
  D.ref_total = 0;
  D.cid = cid;
  // a surrogate step evaluates the KDE and MCS terms exactly; for large sets
  // the receptor split's groups share them (one exchange per step)
  D.da_share = (d->pnk >= 256 || d->pos >= 32) ? 1 : 0;
  for (int i = 0; i < 3; ++i) D.pocket[i] = d->pocket_center[i];
  for (int i = 0; i < 6; ++i) D.move_scale[i] = d->move_scale[i];
  D.el0 = ep.el0;
  D.el1 = ep.el1;
  D.a1 = ep.a1;
  D.b1 = ep.b1;
  D.kde2l = ep.kde2 * 1.44269504088896340736f;
  D.kde3 = ep.kde3;
  D.far2 = skip_range2(*d, par);
  h.far_share = far_share(*d, D.far2);
  for (int i = 0; i < GD_MAXWEI; ++i) {
    D.w[i] = ep.w[i];
    D.a_para[i] = ep.a_para[i];
    D.b_para[i] = ep.b_para[i];
  }
  for (int i = 0; i < NLT; ++i) {
    D.hpl0[i] = ep.hpl0[i];
    D.hpl1[i] = ep.hpl1[i];
    D.hpl2[i] = ep.hpl2[i];
  }
  for (int t = 0; t < GD_MAX_NTMP; ++t) D.minus_beta[t] = t < d->n_tmp ? d->temp[t].minus_beta : 0.0f;

  const float *psp_src = d->psp;
  std::vector<float> psp_zero;
  size_t psp_n = (size_t)NLT * std::max(d->n_res, 1);
  if (!psp_src) {
    psp_zero.assign(psp_n, 0.0f);
    psp_src = psp_zero.data();
  }
  // one device block and one copy for all arrays of the complex
  std::vector<int> type(pnp);
  for (int i = 0; i < pnp; ++i) type[i] = d->prt_t[perm[i]];
  Regions R;
  struct Part {
    const void *src;
    size_t bytes, at;
    void **dst;
  };
  std::vector<Part> parts;
  auto part = [&](auto **dst, const void *src, size_t n_items) {
    const size_t bytes = n_items * sizeof(**dst);
    parts.push_back({src, bytes, R.add(std::max<size_t>(bytes, 16)), (void **)dst});
  };
  part(&D.prt_xyze, xyze.data(), xyze.size());
  part(&D.prt_hpp, hpp.data(), hpp.size());
  part(&D.prt_psp, pspi.data(), pspi.size());
  part(&D.prt_type, type.data(), type.size());
  part(&D.chunks, chunks.data(), chunks.size());
  part(&D.params, par.data(), par.size());
  part(&D.lig_orig, orig.data(), orig.size());
  part(&D.lig_t, d->lig_t, (size_t)lna);
  part(&D.lig_c, d->lig_c, (size_t)lna);
  part(&D.mcs, mcs.data(), mcs.size());
  part(&D.mcs_tcc, tcc.data(), tcc.size());
  part(&D.mcs_cnt, mcnt.data(), mcnt.size());
  part(&D.mcsq, mcsq.data(), mcsq.size());
  part(&D.kde, kde.data(), kde.size());
  part(&D.kde_range, krange.data(), krange.size());
  part(&D.psp, psp_src, psp_n);
  const size_t up_bytes = R.end;
  part(&D.ref, nullptr, (size_t)lna * KMAX);
  part(&D.ref_cnt, nullptr, (size_t)lna);
  void *block = nullptr;
  HIPCHK(hipMalloc(&block, R.end));
  h.bufs.push_back(block);
  {
    const ScratchTrim trim{ctx};
    TRY(scratch_need(ctx, ctx->pin, up_bytes, true));
    for (const Part &q : parts) {
      *q.dst = static_cast<unsigned char *>(block) + q.at;
      if (q.src) memcpy(ctx->pin.p + q.at, q.src, q.bytes);
    }
    HIPCHK(hipMemcpyAsync(block, ctx->pin.p, up_bytes, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
  }
  h.lds_bytes = lds_need(h, 512 / h.lpr, 0);
  h.tiled = ctx->opts.receptor_tile > 0 || h.lds_bytes > ctx->max_lds;
  if (h.tiled) {
    h.lds_bytes = lds_need(h, 512 / h.lpr, complex_tile(ctx, h));
    if (h.lds_bytes > ctx->max_lds)
      return fail(ctx, GD_ERR_CAPACITY, "complex needs %zu bytes of LDS with receptor tiles, "
                  "device has %zu", h.lds_bytes, ctx->max_lds);
  }
  ctx->cx_dirty = true;
  if (complex_id) *complex_id = cid;
  return GD_OK;
}

}  // extern "C"

namespace {

// Side streams and their events for a launch of n classes (made when a context
// first may need them: a stream costs about 50 us and as much again to destroy).
hipError_t side_streams(gd_ctx *ctx, int n) {
  hipError_t e = hipSuccess;
  if (n > 1 && !ctx->ev_fork) e = hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming);
  for (int i = 0; i < std::min(n - 1, SIDE_STREAMS) && e == hipSuccess; ++i) {
    if (!ctx->aux[i]) e = hipStreamCreateWithFlags(&ctx->aux[i], hipStreamNonBlocking);
    if (e == hipSuccess && !ctx->ev_join[i])
      e = hipEventCreateWithFlags(&ctx->ev_join[i], hipEventDisableTiming);
  }
  return e;
}

bool spread_packing(const gd_ctx *ctx);
int auto_gmax(const gd_ctx *ctx);
std::vector<int> lig_splits(const gd_ctx *ctx, const HostComplex &h, int gmax);

// Packs of one wave of replicas (spread packing) for a complex at lpr lanes
// per replica.
int64_t spread_pack_count(const HostComplex &h, int lpr) {
  const int r = std::max(1, 64 / lpr);
  return (int64_t)h.d.n_prt * h.d.n_lig * ((h.d.n_tmp + r - 1) / r);
}

// Lane shapes under spread packing, fixed when a complex is first put on the
// device. Spread packs hold one wave of replicas, so more lanes per replica
// make more packs: a complex takes the shape with the fewest rounds of packs
// over the CUs times atoms per lane (the fewest packs on a tie), among the
// shapes whose ladder fits a workgroup. Forced shapes are kept.
gd_status widen_shapes(gd_ctx *ctx) {
  const bool widen = spread_packing(ctx) && ctx->opts.lanes_per_replica == 0 &&
                     ctx->opts.atoms_per_lane == 0;
  int64_t packs = 0;
  for (const HostComplex &h : ctx->cx)
    if (h.shape_final) packs += spread_pack_count(h, h.lpr);
  for (HostComplex &h : ctx->cx) {
    if (h.shape_final) continue;
    h.shape_final = true;
    if (!widen) continue;
    const int lna = h.d.lna;
    auto cost = [&](int l, int a) {
      return (double)((packs + spread_pack_count(h, l) + ctx->n_cu - 1) / ctx->n_cu) * a;
    };
    int best_l = h.lpr, best_a = h.apl;
    double best = cost(best_l, best_a);
    for (int l = 8; l <= 64; l *= 2) {
      const int a = (lna + l - 1) / l;
      if (a > 4 || l * h.d.n_tmp > 512) continue;
      const double c = cost(l, a);
      if (c < best || (c == best && l < best_l)) {
        best = c;
        best_l = l;
        best_a = a;
      }
    }
    if (best_l != h.lpr) {
      const int ol = h.lpr, oa = h.apl;
      h.lpr = best_l;
      h.apl = best_a;
      const size_t need = lds_need(h, 512 / h.lpr, h.tiled ? complex_tile(ctx, h) : 0);
      if (need > ctx->max_lds) {  // keep the shape add_complex chose
        h.lpr = ol;
        h.apl = oa;
      } else {
        h.lds_bytes = need;
        h.dev.lpr = h.lpr;
        h.dev.apl = h.apl;
      }
    }
    packs += spread_pack_count(h, h.lpr);
  }
  return GD_OK;
}

int flat_index(int ns) { return ns >= 8 ? 3 : ns >= 4 ? 2 : ns >= 2 ? 1 : 0; }

// Unit list of the flat pair loop (gd_mc.h) for lane groups of a split of ns:
// group g's share of every chunk, in chunk order, cut into units of one
// receptor type, an even number for each type. `apl` sets the groups of NP
// points that chunk_pairs forms (4, 2 and 1 for 1, 2 and more atoms per lane),
// which the units' modes keep.
std::vector<int4> build_flat_units(const std::vector<int4> &chunks, int apl, int ns,
                                   int (&off)[9]) {
  std::vector<int4> U;
  const int np = apl >= 3 ? 1 : (apl == 2 ? 2 : 4);
  for (int g = 0; g < ns; ++g) {
    off[g] = (int)U.size();
    std::vector<int> first, types;  // each type's first unit
    int lone = -1;                  // a unit of one point that may take a second
    auto even = [&] {
      if (!first.empty() && ((int)U.size() - first.back()) % 2 != 0)
        U.push_back(make_int4(FLAT_EMPTY, U.back().y, 0, 0));
    };
    for (const int4 &ch : chunks) {
      const int fb = ch.x + (ch.y * g) / ns, fe = ch.x + (ch.y * (g + 1)) / ns;
      if (fb >= fe) continue;
      if (types.empty() || types.back() != ch.z) {
        even();
        first.push_back((int)U.size());
        types.push_back(ch.z);
        lone = -1;
      }
      const int hpc = ch.w >= KIND_HPC ? FLAT_HPC : 0;
      auto emit = [&](int p0, int p1, int flags) {
        U.push_back(make_int4(flags | hpc, p0 | (p1 << 16), 0, 0));
      };
      int p = fb;
      for (; np == 4 && p + 4 <= fe; p += 4) {
        emit(p, p + 1, FLAT_FIRST);
        emit(p + 2, p + 3, FLAT_SECOND | (p + 4 == fe ? FLAT_END1 : 0));
        lone = -1;
      }
      for (; np == 2 && p + 2 <= fe; p += 2) {
        emit(p, p + 1, FLAT_BLOCK | (p + 2 == fe ? FLAT_END1 : 0));
        lone = -1;
      }
      for (; p < fe; ++p) {
        const bool last = p + 1 == fe;
        if (lone >= 0) {
          int4 &u = U[lone];
          u.x = (u.x & ~FLAT_ONE) | (last ? FLAT_END1 : 0) | hpc;
          u.y = (u.y & 0xffff) | (p << 16);
          lone = -1;
        } else {
          emit(p, p, FLAT_SINGLES | FLAT_ONE | (last ? FLAT_END0 : 0));
          lone = (int)U.size() - 1;
        }
      }
    }
    even();
    for (size_t i = 0; i < first.size(); ++i) {
      const int end = i + 1 < first.size() ? first[i + 1] : (int)U.size();
      U[first[i]].x |= types[i] | (((end - first[i]) / 2) << FLAT_PAIRS);
    }
  }
  off[ns] = (int)U.size();
  return U;
}

// Unit lists of the complexes that lack one for a split their packs have, in
// one device block (points and PSP columns are 16-bit in a unit and a type has
// at most FLAT_PAIR_MASK unit pairs in a group).
gd_status build_flat(gd_ctx *ctx) {
  const bool spread = spread_packing(ctx);
  const int gmax = spread ? 0 : auto_gmax(ctx);
  std::vector<int> want(ctx->cx.size(), 0);  // bit f: packs of split 1 << f
  int64_t points = 0, shares = 0;
  for (size_t c = 0; c < ctx->cx.size(); ++c) {
    const HostComplex &h = ctx->cx[c];
    if (h.tiled) continue;
    for (int ns : lig_splits(ctx, h, gmax)) {
      points += (int64_t)h.d.n_prt * h.d.pnp;
      shares += (int64_t)h.d.n_prt * h.n_chunks * ns;
      want[c] |= 1 << flat_index(ns);
    }
  }
  ctx->flat = spread || (ctx->opts.receptor_split == 0 && points <= FLAT_SHARE * shares);
  if (!ctx->flat) return GD_OK;
  struct Todo {
    HostComplex *h;
    int f;
    size_t at;
    int n;
  };
  std::vector<Todo> todo;
  std::vector<int4> all;
  for (size_t c = 0; c < ctx->cx.size(); ++c) {
    HostComplex &h = ctx->cx[c];
    if (h.d.pnp > 4 * FLAT_PAIR_MASK || h.d.n_res > 0x7fff) continue;
    for (int f = 0; f < 4; ++f) {
      if (!(want[c] >> f & 1) || h.flat_n[f] > 0) continue;
      const std::vector<int4> U = build_flat_units(h.chunks, h.apl, 1 << f, h.dev.flat_off[f]);
      todo.push_back({&h, f, all.size(), (int)U.size()});
      all.insert(all.end(), U.begin(), U.end());
    }
  }
  if (todo.empty()) return GD_OK;
  void *p = nullptr;
  HIPCHK(hipMalloc(&p, all.size() * sizeof(int4)));
  ctx->flat_bufs.push_back(p);
  HIPCHK(hipMemcpyAsync(p, all.data(), all.size() * sizeof(int4), hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  // a list counts (flat_n) from here on, when the device holds it
  for (const Todo &t : todo) {
    t.h->dev.flat[t.f] = static_cast<int4 *>(p) + t.at;
    t.h->flat_n[t.f] = t.n;
  }
  return GD_OK;
}

gd_status sync_complexes(gd_ctx *ctx) {
  if (!ctx->cx_dirty) return GD_OK;
  TRY(widen_shapes(ctx));
  TRY(build_flat(ctx));
  // runs and feature kernels do not come through here: the table they use stays
  // until the new one is on the device
  std::vector<DevComplex> v;
  for (auto &h : ctx->cx) v.push_back(h.dev);
  DevComplex *table = nullptr;
  HIPCHK(hipMalloc(&table, std::max<size_t>(v.size(), 1) * sizeof(DevComplex)));
  hipError_t e = hipMemcpyAsync(table, v.data(), v.size() * sizeof(DevComplex),
                                hipMemcpyHostToDevice, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  if (e != hipSuccess) {
    (void)hipFree(table);
    return fail(ctx, GD_ERR_HIP, "complex table: %s", hipGetErrorString(e));
  }
  if (ctx->d_cx) (void)hipFree(ctx->d_cx);
  ctx->d_cx = table;
  for (auto &g : ctx->gslot) g.valid = false;  // captured launches hold the old pointer
  ctx->cx_dirty = false;
  return GD_OK;
}

// Contact maps of replica 0's start pose for the complexes that lack one, in
// one launch.
gd_status ensure_ref(gd_ctx *ctx) {
  TRY(sync_complexes(ctx));
  std::vector<int> todo;
  int lna_max = 0;
  for (int c = 0; c < (int)ctx->cx.size(); ++c)
    if (!ctx->cx[c].ref_built) {
      todo.push_back(c);
      lna_max = std::max(lna_max, ctx->cx[c].d.lna);
    }
  if (todo.empty()) return GD_OK;
  // pose calls without allocations come after this call and may need a launch
  // for each block size (packs of a split below 8)
  if (!spread_packing(ctx)) HIPCHK(side_streams(ctx, SIDE_STREAMS + 1));
  const size_t n = todo.size();
  int2 *d_out = nullptr;  // per complex: contacts, atoms beyond the limit; then the list
  HIPCHK(hipMalloc(&d_out, n * (sizeof(int2) + sizeof(int))));
  int *d_todo = reinterpret_cast<int *>(d_out + n);
  std::vector<int2> out(n);
  hipError_t e = hipMemcpyAsync(d_todo, todo.data(), n * sizeof(int), hipMemcpyHostToDevice, ctx->stream);
  if (e == hipSuccess) e = hipMemsetAsync(d_out, 0, n * sizeof(int2), ctx->stream);
  for (size_t b = 0; b < n && e == hipSuccess; b += GRID_ROWS) {
    hipLaunchKernelGGL(gd_ref_kernel,
                       dim3((unsigned)lna_max, (unsigned)std::min<size_t>(GRID_ROWS, n - b)), dim3(64),
                       0, ctx->stream, ctx->d_cx, d_todo + b, d_out + b);
    e = hipGetLastError();
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(out.data(), d_out, n * sizeof(int2), hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  (void)hipFree(d_out);
  if (e != hipSuccess) return fail(ctx, GD_ERR_HIP, "contact maps: %s", hipGetErrorString(e));
  for (size_t i = 0; i < n; ++i) {
    if (out[i].y > 0)
      return fail(ctx, GD_ERR_CAPACITY,
                  "complex %d: more than %d reference contacts for one ligand atom", todo[i], KMAX);
    ctx->cx[todo[i]].dev.ref_total = out[i].x;
  }
  for (int c : todo) ctx->cx[c].ref_built = true;
  ctx->cx_dirty = true;
  return sync_complexes(ctx);
}

int complex_tile(const gd_ctx *ctx, const HostComplex &h) {
  if (!h.tiled) return 0;
  return ctx->opts.receptor_tile > 0 ? ctx->opts.receptor_tile : DEFAULT_TILE;
}

// LDS layout for a launch covering packs with these maxima, in blocks of
// `block` lanes; `split` adds the partial-sum exchange buffers of packs with
// more than one lane group ([ns*half][4] HPC sums and [ns][half/8][12] replica
// sums, ns*half = block). With tile > 0 the receptor arrays are two tiles of
// `tile` points and KDE stays in HBM; with flat_max > 0 the receptor is that many
// units of the flat pair loop (and a pad, which its reads run into).
void layout(KParams &P, size_t *bytes, int pnp_max, int pnk_max, int nch_max, int slots_max,
            int block, bool split, int tile = 0, int flat_max = 0) {
  auto al = [](size_t v) { return (v + 15) & ~(size_t)15; };
  P.tile = tile;
  if (tile > 0) {
    pnp_max = 2 * tile;
    pnk_max = 0;
  }
  size_t o = al((size_t)pnp_max * 16);
  P.off_hpp = (int)o;
  o = al(o + (size_t)pnp_max * 4);
  P.off_psp = (int)o;
  o = al(o + (size_t)pnp_max * 4);
  if (flat_max > 0) o = (size_t)(flat_max + 1) * FLAT_F4 * 16;
  P.off_par = (int)o;
  o = al(o + (size_t)PAR_FLOATS * 4);
  P.off_kde = (int)o;
  o = al(o + (size_t)std::max(pnk_max, 1) * 16);
  P.off_kr = (int)o;
  o = al(o + NLT * 8);
  P.off_ch = (int)o;
  o = al(o + (size_t)std::max(nch_max, 1) * 16);
  P.off_xe = (int)o;
  o = al(o + (size_t)slots_max * 4);
  P.off_xi = (int)o;
  o = al(o + (size_t)slots_max * 4);
  P.off_xa = (int)o;
  o = al(o + (size_t)slots_max * 4);
  P.off_xo = (int)o;
  o = al(o + (size_t)slots_max * 4);
  // split exchange: 4 floats of per-atom HPC sums per lane, 12 floats of
  // partial sums per replica (at most block/8 replicas): 5.5 floats per lane
  P.xp_floats = split ? (11 * block) / 2 : 0;
  P.off_xp = (int)o;
  o = al(o + (size_t)2 * P.xp_floats * 4);
  P.off_q = (int)o;
  o = al(o + 16);
  *bytes = o;
}

struct PackSet {
  std::vector<Pack> packs;
  std::vector<int> slots;
  std::vector<LaunchClass> classes;
};

// Copy the LDS layout and split fields of a launch class into P.
void apply_layout(KParams &P, const KParams &L) {
  P.off_hpp = L.off_hpp;
  P.off_psp = L.off_psp;
  P.off_par = L.off_par;
  P.off_kde = L.off_kde;
  P.off_kr = L.off_kr;
  P.off_ch = L.off_ch;
  P.off_xe = L.off_xe;
  P.off_xi = L.off_xi;
  P.off_xa = L.off_xa;
  P.off_xo = L.off_xo;
  P.off_xp = L.off_xp;
  P.xp_floats = L.xp_floats;
  P.off_q = L.off_q;
  P.tile = L.tile;
}

// Group packs into launch classes by (atoms per lane, tile, block shape,
// workgroups per CU that the LDS allows), each class longest packs first so
// the hardware dispatcher (or the persistent queue) fills the CUs in LPT
// order. Every pack of a class has the class's block (its ns groups of `half`
// lanes), so no wave of a workgroup is idle. A class's LDS is the largest need
// among its packs: a class closes when the next pack would lower the
// workgroups per CU it allows. Workgroups of 512 lanes take a CU's register
// file alone (two waves per SIMD), so LDS does not split their classes.
void pack_finish(const gd_ctx *ctx, PackSet &ps, int lpr = 0, int apl_of_lpr = 0) {
  const size_t n_pk = ps.packs.size();
  std::vector<int> res(n_pk), block(n_pk), apl(n_pk), tile(n_pk), units(n_pk);
  std::vector<double> cost(n_pk);
  for (size_t i = 0; i < n_pk; ++i) {
    Pack &p = ps.packs[i];
    const HostComplex &h = ctx->cx[p.cx];
    p.half = ((p.round * (lpr > 0 ? lpr : h.lpr) + 63) / 64) * 64;
    block[i] = p.half * p.ns;
    apl[i] = lpr > 0 ? apl_of_lpr : h.apl;
    // the tile length depends on the options only (not on the pack's block),
    // so every launch of a complex sums its chunks in the same order
    tile[i] = complex_tile(ctx, h);
    cost[i] = (double)h.d.pnp * (double)p.half * apl[i];
    KParams L{};
    size_t need = 0;
    // units of the flat pair loop, where they fit
    units[i] = ctx->flat && tile[i] == 0 && block[i] == 512 ? h.flat_n[flat_index(p.ns)] : 0;
    if (units[i] > 0) {
      layout(L, &need, 0, h.d.pnk, h.n_chunks, p.round, block[i], p.ns > 1, 0, units[i]);
      if (need > ctx->max_lds) units[i] = 0;
    }
    layout(L, &need, (h.d.pnp + 3) & ~3, h.d.pnk, h.n_chunks, p.round, block[i], p.ns > 1,
           tile[i]);
    res[i] = block[i] >= 512
                 ? 1
                 : (int)std::max<size_t>(1, std::min<size_t>(512 / block[i],
                                                             ctx->max_lds / std::max<size_t>(need, 1)));
  }
  // all per-pack keys are indexed by the pack's position before sorting
  std::vector<int> order(n_pk);
  for (size_t i = 0; i < n_pk; ++i) order[i] = (int)i;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    if (apl[a] != apl[b]) return apl[a] < apl[b];
    if (tile[a] != tile[b]) return tile[a] < tile[b];
    if ((units[a] > 0) != (units[b] > 0)) return units[a] > 0;
    if (block[a] != block[b]) return block[a] > block[b];
    if (res[a] != res[b]) return res[a] < res[b];
    return cost[a] > cost[b];
  });
  std::vector<Pack> sorted;
  for (int i : order) sorted.push_back(ps.packs[i]);
  ps.packs.swap(sorted);
  ps.classes.clear();
  for (size_t b = 0; b < n_pk;) {
    const int o0 = order[b];
    LaunchClass lc;
    lc.apl = apl[o0];
    lc.begin = (int)b;
    lc.block = block[o0];
    lc.tile = tile[o0];
    int pnp_max = 0, pnk_max = 0, nch_max = 0, slots_max = 1, half_max = 64, flat_max = 0;
    bool split = false;
    double far = 0.0, all = 0.0;
    const bool flat = units[o0] > 0;
    size_t e = b;
    for (; e < n_pk; ++e) {
      const int oe = order[e];
      if (apl[oe] != lc.apl || tile[oe] != lc.tile || block[oe] != lc.block ||
          res[oe] != res[o0] || (units[oe] > 0) != flat)
        break;
      const Pack &p = ps.packs[e];
      const HostComplex &h = ctx->cx[p.cx];
      const int np = std::max(pnp_max, h.d.pnp), nk = std::max(pnk_max, h.d.pnk);
      const int nc = std::max(nch_max, h.n_chunks), ns = std::max(slots_max, p.round);
      const bool sp = split || p.ns > 1;
      KParams L{};
      size_t need = 0;
      layout(L, &need, (np + 3) & ~3, nk, nc, ns, lc.block, sp, lc.tile);
      const size_t fit = ctx->max_lds / std::max<size_t>(need, 1);
      if (e > b && (fit < 1 || (res[o0] > 1 && fit < (size_t)res[o0]))) break;
      const int nu = std::max(flat_max, units[oe]);
      if (flat) {
        layout(L, &need, 0, nk, nc, ns, lc.block, sp, 0, nu);
        if (e > b && need > ctx->max_lds) break;
      }
      flat_max = nu;
      pnp_max = np;
      pnk_max = nk;
      nch_max = nc;
      slots_max = ns;
      split = sp;
      half_max = std::max(half_max, p.half);
      far += cost[oe] * h.far_share;
      all += cost[oe];
    }
    lc.end = (int)e;
    lc.near = far < (lc.block <= NEAR_BLOCK ? NEAR_SHARE_1WAVE : NEAR_SHARE[lc.apl - 1]) * all;
    lc.half_max = half_max;
    layout(lc.lay, &lc.lds, (pnp_max + 3) & ~3, pnk_max, nch_max, slots_max, lc.block, split,
           lc.tile);
    if (flat) {
      layout(lc.lay_flat, &lc.lds_flat, 0, pnk_max, nch_max, slots_max, lc.block, split, 0,
             flat_max);
    }
    ps.classes.push_back(lc);
    b = e;
  }
}

// Ladders of one (complex, protein conformer) grouped into packs, in
// ligand-conformer order: {first ligand conformer, ladders, receptor split}.
// The same grouping serves every protein conformer of the complex.
//
// A fixed split (receptor_split 1, 2, 4 or 8) takes `ladders_per_pack`
// ladders per pack (default: about 256 lanes), within 512 lanes per workgroup.
// The automatic split (0) fills every workgroup to 8 waves, the two waves per
// SIMD that the kernels' registers allow: ladders of w waves are grouped by
// powers of two, at most `gmax` ladders (and 8 waves) per pack, and each pack
// takes the smallest split that fills 8 waves with its groups, so a ladder
// left over from an odd count runs with more groups instead of leaving waves
// idle. A ladder of 5 or more waves runs unsplit.
struct LadderGroup {
  int l0, ng, ns;
};

std::vector<LadderGroup> ladder_groups(const gd_ctx *ctx, const HostComplex &h, int gmax) {
  std::vector<LadderGroup> out;
  const int n_lig = h.d.n_lig, glanes = h.d.n_tmp * h.lpr;
  const int fixed = ctx->opts.receptor_split, ladders = ctx->opts.ladders_per_pack;
  if (fixed > 0) {
    int G = ladders > 0 ? ladders : std::max(1, 256 / glanes);
    while (G > 1 && G * glanes > 512 / fixed) --G;
    for (int l0 = 0; l0 < n_lig; l0 += G) out.push_back({l0, std::min(G, n_lig - l0), fixed});
    return out;
  }
  const int w = (glanes + 63) / 64;
  if (w >= 5) {
    for (int l0 = 0; l0 < n_lig; ++l0) out.push_back({l0, 1, 1});
    return out;
  }
  const int gcap = std::max(1, std::min(gmax, 8 / w));
  for (int l0 = 0; l0 < n_lig;) {
    int G = 1;
    while (2 * G <= std::min(gcap, n_lig - l0)) G *= 2;
    int ns = 1;
    while (2 * ns * G * w <= 8) ns *= 2;
    out.push_back({l0, G, ns});
    l0 += G;
  }
  return out;
}

// Ladders per pack of the automatic split for the context's complexes:
// `ladders_per_pack` when set, else the most (up to 8) that still leaves at
// least four packs per CU for the longest-first balancing, down to one ladder
// per pack (each then filled by its split) when the batch is small.
int auto_gmax(const gd_ctx *ctx) {
  if (ctx->opts.ladders_per_pack > 0) return ctx->opts.ladders_per_pack;
  int g = 8;
  for (; g > 1; g /= 2) {
    int64_t packs = 0;
    for (const HostComplex &h : ctx->cx) packs += (int64_t)h.d.n_prt * ladder_groups(ctx, h, g).size();
    if (packs >= (int64_t)4 * ctx->n_cu) break;
  }
  return g;
}

// Spread packing: on request, or by default when the workload has at most
// one temperature ladder per two CUs (ladder-per-workgroup packing would
// leave most CUs idle) and no fixed split or ladders per pack is set.
bool spread_packing(const gd_ctx *ctx) {
  const int L = ctx->opts.launch;
  if (L & GD_LAUNCH_SPREAD) return true;
  if ((L & GD_LAUNCH_NO_SPREAD) || ctx->opts.receptor_split > 0 || ctx->opts.ladders_per_pack > 0)
    return false;
  int64_t ladders = 0;
  for (const HostComplex &h : ctx->cx) ladders += (int64_t)h.d.n_prt * h.d.n_lig;
  return ladders > 0 && 2 * ladders <= ctx->n_cu;
}

// Receptor split of each ligand conformer's MC packs. The split sets the
// summation order, so a pose's energy bits follow it; gd_calc_energy uses it.
// `gmax`: auto_gmax(ctx) (unused under spread packing).
std::vector<int> lig_splits(const gd_ctx *ctx, const HostComplex &h, int gmax) {
  std::vector<int> ns(h.d.n_lig, spread_packing(ctx) ? 8 : 1);
  if (spread_packing(ctx)) return ns;
  for (const LadderGroup &lg : ladder_groups(ctx, h, gmax))
    for (int g = 0; g < lg.ng; ++g) ns[lg.l0 + g] = lg.ns;
  return ns;
}

// Spread packing: each pack holds one wave of replicas of one ladder
// (64 / lanes-per-replica temperature slots, in slot order) at a receptor
// split of 8, so each workgroup is 8 waves; a ladder of more slots spans
// several packs, and its exchanges run between launches.
PackSet build_spread_packs(gd_ctx *ctx) {
  PackSet ps;
  for (int c = 0; c < (int)ctx->cx.size(); ++c) {
    HostComplex &h = ctx->cx[c];
    const int n_tmp = h.d.n_tmp, n_lig = h.d.n_lig;
    const int r = std::max(1, 64 / h.lpr);
    h.lig_ns.assign(n_lig, 8);
    for (int p = 0; p < h.d.n_prt; ++p)
      for (int l = 0; l < n_lig; ++l)
        for (int t0 = 0; t0 < n_tmp; t0 += r) {
          Pack pk{};
          pk.cx = c;
          pk.prt = p;
          pk.n_groups = 0;
          pk.n_slots = pk.round = std::min(r, n_tmp - t0);
          pk.ns = 8;
          pk.slot_off = (int)ps.slots.size();
          for (int t = t0; t < t0 + pk.n_slots; ++t)
            ps.slots.push_back(h.rep_base + n_tmp * n_lig * p + n_lig * t + l);
          ps.packs.push_back(pk);
        }
  }
  pack_finish(ctx, ps);
  return ps;
}

// MC packs: the ladder groups of every (complex, protein conformer).
PackSet build_mc_packs(gd_ctx *ctx) {
  if (spread_packing(ctx)) return build_spread_packs(ctx);
  PackSet ps;
  const int gmax = auto_gmax(ctx);
  for (int c = 0; c < (int)ctx->cx.size(); ++c) {
    HostComplex &h = ctx->cx[c];
    const int n_tmp = h.d.n_tmp, n_lig = h.d.n_lig;
    const std::vector<LadderGroup> groups = ladder_groups(ctx, h, gmax);
    h.lig_ns.assign(n_lig, 1);
    for (const LadderGroup &lg : groups)
      for (int g = 0; g < lg.ng; ++g) h.lig_ns[lg.l0 + g] = lg.ns;
    for (int p = 0; p < h.d.n_prt; ++p)
      for (const LadderGroup &lg : groups) {
        Pack pk{};
        pk.cx = c;
        pk.prt = p;
        pk.n_groups = lg.ng;
        pk.n_slots = pk.round = lg.ng * n_tmp;
        pk.ns = lg.ns;
        pk.slot_off = (int)ps.slots.size();
        for (int g = 0; g < lg.ng; ++g)
          for (int t = 0; t < n_tmp; ++t)
            ps.slots.push_back(h.rep_base + n_tmp * n_lig * p + n_lig * t + (lg.l0 + g));
        ps.packs.push_back(pk);
      }
  }
  pack_finish(ctx, ps);
  return ps;
}

gd_status alloc_state(gd_ctx *ctx) {
  if (ctx->state_alloc) return GD_OK;
  TRY(ensure_ref(ctx));
  int n = 0;
  for (auto &h : ctx->cx) {
    h.rep_base = n;
    n += h.n_rep;
  }
  if (n == 0) return fail(ctx, GD_ERR_STATE, "no complexes added");
  ctx->n_rep = n;
  HIPCHK(hipMalloc(&ctx->d_mm, (size_t)n * 6 * sizeof(float)));
  HIPCHK(hipMalloc(&ctx->d_eold, (size_t)n * sizeof(gd_energy)));
  HIPCHK(hipMalloc(&ctx->d_best_e, (size_t)n * sizeof(float)));
  HIPCHK(hipMalloc(&ctx->d_best_mm, (size_t)n * 6 * sizeof(float)));
  HIPCHK(hipMalloc(&ctx->d_idx_tmp, (size_t)n * sizeof(int)));
  HIPCHK(hipMalloc(&ctx->d_acs_mc, (size_t)n * sizeof(int)));
  HIPCHK(hipMalloc(&ctx->d_acs_x, (size_t)n * sizeof(int)));
  HIPCHK(hipMalloc(&ctx->d_rep_flat, (size_t)n * sizeof(int)));
  HIPCHK(hipMalloc(&ctx->d_ring_cnt[0], (size_t)n * sizeof(int)));
  std::vector<int> flat(n), itmp(n);
  for (auto &h : ctx->cx)
    for (int f = 0; f < h.n_rep; ++f) {
      flat[h.rep_base + f] = f;
      itmp[h.rep_base + f] = (f / h.d.n_lig) % h.d.n_tmp;  // SetReplica, src/util.C:846-852
    }
  HIPCHK(hipMemcpyAsync(ctx->d_rep_flat, flat.data(), n * sizeof(int), hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipMemcpyAsync(ctx->d_idx_tmp, itmp.data(), n * sizeof(int), hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipMemsetAsync(ctx->d_mm, 0, (size_t)n * 6 * sizeof(float), ctx->stream));
  HIPCHK(hipMemsetAsync(ctx->d_eold, 0, (size_t)n * sizeof(gd_energy), ctx->stream));
  HIPCHK(hipMemsetAsync(ctx->d_acs_mc, 0, (size_t)n * sizeof(int), ctx->stream));
  HIPCHK(hipMemsetAsync(ctx->d_acs_x, 0, (size_t)n * sizeof(int), ctx->stream));
  HIPCHK(hipMemsetAsync(ctx->d_ring_cnt[0], 0, (size_t)n * sizeof(int), ctx->stream));
  // receptor split: automatic (0, per pack) or fixed
  const int ns = ctx->opts.receptor_split;
  if (ns != 0 && ns != 1 && ns != 2 && ns != 4 && ns != 8)
    return fail(ctx, GD_ERR_INVALID, "receptor_split must be 0, 1, 2, 4 or 8");
  for (auto &h : ctx->cx)
    if (ns > 1 && h.d.n_tmp * h.lpr > 512 / ns)
      return fail(ctx, GD_ERR_CAPACITY,
                  "receptor split %d needs ladders of at most %d lanes (a ladder has %d)", ns,
                  512 / ns, h.d.n_tmp * h.lpr);
  if ((ctx->opts.launch & GD_LAUNCH_SPREAD) && (ns > 0 || ctx->opts.ladders_per_pack > 0))
    return fail(ctx, GD_ERR_INVALID,
                "GD_LAUNCH_SPREAD sets its own packs: leave receptor_split and ladders_per_pack 0");
  PackSet ps = build_mc_packs(ctx);
  if (spread_packing(ctx)) {
    std::vector<int4> lad;
    for (int c = 0; c < (int)ctx->cx.size(); ++c) {
      const HostComplex &h = ctx->cx[c];
      const int n_tmp = h.d.n_tmp, n_lig = h.d.n_lig;
      for (int p = 0; p < h.d.n_prt; ++p)
        for (int l = 0; l < n_lig; ++l)
          lad.push_back(make_int4(c, p * n_lig + l, h.rep_base + n_tmp * n_lig * p + l, n_lig));
    }
    ctx->n_ladders = (int)lad.size();
    HIPCHK(hipMalloc(&ctx->d_ladders, lad.size() * sizeof(int4)));
    HIPCHK(hipMemcpyAsync(ctx->d_ladders, lad.data(), lad.size() * sizeof(int4),
                          hipMemcpyHostToDevice, ctx->stream));
  }
  HIPCHK(hipMalloc(&ctx->d_packs, ps.packs.size() * sizeof(Pack)));
  HIPCHK(hipMalloc(&ctx->d_slots, ps.slots.size() * sizeof(int)));
  HIPCHK(hipMemcpyAsync(ctx->d_packs, ps.packs.data(), ps.packs.size() * sizeof(Pack),
                        hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipMemcpyAsync(ctx->d_slots, ps.slots.data(), ps.slots.size() * sizeof(int),
                        hipMemcpyHostToDevice, ctx->stream));
  ctx->n_packs = (int)ps.packs.size();
  ctx->mc_classes = ps.classes;
  HIPCHK(hipMalloc(&ctx->d_ctrl, (1 + ps.classes.size()) * sizeof(int)));
  HIPCHK(hipMemsetAsync(ctx->d_ctrl, 0, (1 + ps.classes.size()) * sizeof(int), ctx->stream));
  for (const LaunchClass &lc : ps.classes) {
    if (lc.lds > ctx->max_lds)
      return fail(ctx, GD_ERR_CAPACITY, "launch needs %zu bytes of LDS, device has %zu", lc.lds,
                  ctx->max_lds);
    if (lc.block > 512)
      return fail(ctx, GD_ERR_CAPACITY, "a temperature ladder needs %d lanes (> 512)", lc.block);
  }
  HIPCHK(hipStreamSynchronize(ctx->stream));
  ctx->state_alloc = true;
  if (ctx->opts.verbose) {
    fprintf(stderr, "[geauxdock] %d replicas, %d packs, split %s, %zu launch classes\n", n,
            ctx->n_packs, ns ? "fixed" : "auto", ctx->mc_classes.size());
    for (const LaunchClass &lc : ctx->mc_classes) {
      int nsp[4] = {0, 0, 0, 0};
      for (int i = lc.begin; i < lc.end; ++i) {
        const int v = ps.packs[i].ns;
        ++nsp[v >= 8 ? 3 : v >= 4 ? 2 : v >= 2 ? 1 : 0];
      }
      fprintf(stderr,
              "[geauxdock]   apl %d packs %d block %d LDS %zu B tile %d (split 1/2/4/8: %d/%d/%d/%d)\n",
              lc.apl, lc.end - lc.begin, lc.block, lc.lds, lc.tile, nsp[0], nsp[1], nsp[2],
              nsp[3]);
    }
  }
  return GD_OK;
}

KParams base_params(gd_ctx *ctx) {
  KParams P{};
  P.cxs = ctx->d_cx;
  P.packs = ctx->d_packs;
  P.slots = ctx->d_slots;
  P.mm = ctx->d_mm;
  P.e_old = ctx->d_eold;
  P.best_e = ctx->d_best_e;
  P.best_mm = ctx->d_best_mm;
  P.idx_tmp = ctx->d_idx_tmp;
  P.acs_mc = ctx->d_acs_mc;
  P.acs_x = ctx->d_acs_x;
  P.rep_flat = ctx->d_rep_flat;
  P.rec = ctx->d_ring[ctx->ring];
  P.rec_cnt = ctx->d_ring_cnt[ctx->ring];
  P.rec_cap = ctx->rec_cap;
  P.k0 = (uint32_t)ctx->opts.seed;
  P.k1 = (uint32_t)(ctx->opts.seed >> 32);
  return P;
}

// Kernel instance for atoms per lane `apl` and mode `da`: 0 plain,
// 1 delayed acceptance with the network per atom, 2 with its tables, 3 and 4
// the same with the split groups' shared surrogate sums compiled in; and the
// other modes of gd_kernels.h.
const void *mc_kernel_fn(int apl, int da, int rec) {
  switch (apl) {
    case 1: return mc_kernel_handle<1>(da, rec);
    case 2: return mc_kernel_handle<2>(da, rec);
    case 3: return mc_kernel_handle<3>(da, rec);
    default: return mc_kernel_handle<4>(da, rec);
  }
}

// Instance mode of a delayed-acceptance or surrogate launch (see
// mc_kernel_fn): the shared-sum variants only when some complex's KDE or MCS
// sets are large enough to share, so other workloads run code without them.
int da_instance(const gd_ctx *ctx, bool tab) {
  bool any = false;
  for (const HostComplex &h : ctx->cx) any = any || h.dev.da_share != 0;
  return (tab ? 2 : 1) + (any ? 2 : 0);
}

// Launch every class of a pack set, the classes concurrently on side streams
// forked from and joined to `stream`. With `da`, the delayed-acceptance
// instances run; `da_scratch` adds the per-wave LDS scratch of the direct
// network evaluation (a class whose LDS would overflow then runs each pack as
// one lane group: the same packs and decisions' inputs, with the pair sums in
// one group's order).
// Per-class kernel arguments of a launch (persistent grids when `queue`).
struct ClassLaunch {
  const void *f;
  KParams P;
  int grid, block, packs;
  size_t lds;
};

hipError_t plan_classes(gd_ctx *ctx, const std::vector<LaunchClass> &classes, const KParams &P0,
                        int da, bool da_scratch, int *queue, std::vector<ClassLaunch> &out) {
  out.clear();
  for (size_t i = 0; i < classes.size(); ++i) {
    const LaunchClass &lc = classes[i];
    ClassLaunch cl;
    cl.P = P0;
    KParams &P = cl.P;
    // the flat pair loop where the packs have unit lists; the direct network
    // evaluation keeps the layout its scratch fits in
    const bool flat = lc.lds_flat > 0 && !da_scratch;
    apply_layout(P, flat ? lc.lay_flat : lc.lay);
    P.pack_base = lc.begin;
    cl.block = lc.block;
    cl.lds = flat ? lc.lds_flat : lc.lds;
    if (da && da_scratch) {
      P.off_da = (int)((cl.lds + 15) & ~(size_t)15);
      cl.lds = P.off_da + (size_t)(cl.block / 64) * 6208;
      if (cl.lds > ctx->max_lds && lc.half_max < cl.block) {
        P.unsplit = 1;
        cl.block = lc.half_max;
        cl.lds = P.off_da + (size_t)(cl.block / 64) * 6208;
      }
      if (cl.lds > ctx->max_lds) return hipErrorInvalidValue;
    } else if (da) {
      P.off_da = (int)((cl.lds + 15) & ~(size_t)15);
    }
    const int n_pk = lc.end - lc.begin;
    cl.grid = cl.packs = n_pk;
    if (queue) {
      // resident workgroups: LDS-limited, and at most 8 waves per CU (the
      // kernels' register use allows two waves per SIMD)
      const int by_lds = (int)std::max<size_t>(1, ctx->max_lds / std::max<size_t>(cl.lds, 1));
      const int by_waves = std::max(1, 8 / std::max(1, cl.block / 64));
      cl.grid = std::min(n_pk, ctx->n_cu * std::min(by_lds, by_waves));
      P.queue = queue + i;
      P.n_queue = n_pk;
    }
    const int rec = lc.tile > 0 ? REC_TILED : flat ? REC_FLAT : REC_CHUNKS;
    cl.f = mc_kernel_fn(lc.apl, lc.near && da <= 4 ? da | DA_NEAR : da, rec);
    out.push_back(cl);
  }
  // the dynamic LDS limit of every instance used is the device's: classes
  // (and pose-evaluation launches) of different sizes share instances
  for (const ClassLaunch &cl : out) {
    const hipError_t e =
        hipFuncSetAttribute(cl.f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ctx->max_lds);
    if (e != hipSuccess) return e;
  }
  return side_streams(ctx, (int)out.size());
}

// Enqueue planned class launches, the classes concurrently on side streams
// forked from and joined to `stream` (capturable).
hipError_t enqueue_classes(gd_ctx *ctx, std::vector<ClassLaunch> &cls, int *queue,
                           hipStream_t stream) {
  const int n = (int)cls.size();
  hipError_t e = hipSuccess;
  if (queue && n > 0) {
    hipLaunchKernelGGL(gd_queue_reset_kernel, dim3((n + 63) / 64), dim3(64), 0, stream, queue, n);
    e = hipGetLastError();
  }
  const int n_side = std::min(n - 1, SIDE_STREAMS);
  if (e == hipSuccess && n_side > 0) {
    e = hipEventRecord(ctx->ev_fork, stream);
    for (int i = 0; i < n_side && e == hipSuccess; ++i) e = hipStreamWaitEvent(ctx->aux[i], ctx->ev_fork, 0);
  }
  for (int i = 0; i < n && e == hipSuccess; ++i) {
    void *args[] = {&cls[i].P};
    const int side = i % (SIDE_STREAMS + 1);  // 0: the main stream
    hipStream_t s = side == 0 ? stream : ctx->aux[side - 1];
    e = hipLaunchKernel(cls[i].f, dim3(cls[i].grid), dim3(cls[i].block), args, cls[i].lds, s);
  }
  for (int i = 0; i < n_side && e == hipSuccess; ++i) {
    e = hipEventRecord(ctx->ev_join[i], ctx->aux[i]);
    if (e == hipSuccess) e = hipStreamWaitEvent(stream, ctx->ev_join[i], 0);
  }
  return e;
}

hipError_t launch_classes(gd_ctx *ctx, const std::vector<LaunchClass> &classes, const KParams &P0,
                          int da, bool da_scratch, hipStream_t stream) {
  std::vector<ClassLaunch> cls;
  hipError_t e = plan_classes(ctx, classes, P0, da, da_scratch, nullptr, cls);
  if (e == hipSuccess) e = enqueue_classes(ctx, cls, nullptr, stream);
  return e;
}

// A drain of record ring r hands its accepted-state records to the sink in two
// halves. compact_ring gathers them on the device into one window and restarts
// the ring's counts, before the next window begins: MC workgroups may leave no
// registers to its kernels, which then waited for that window's end (1,024
// complexes with records 7.9M replica-steps/s, 9.7M now). deliver_records
// copies the window to the pinned staging buffer and hands it out per complex:
// copy engines work beside the next window.
gd_status compact_ring(gd_ctx *ctx, int r, hipStream_t stream) {
  ctx->drain_total = 0;
  if (!ctx->d_ring[r]) return GD_OK;
  const int n = ctx->n_rep;
  int *cnt_d = ctx->d_ring_cnt[r];
  Regions R;
  const size_t o_off = R.add((n + 1) * sizeof(int64_t)), o_cnt = R.add(n * sizeof(int));
  TRY(scratch_need(ctx, ctx->drain_pin, R.end, true));
  int64_t *off = reinterpret_cast<int64_t *>(ctx->drain_pin.p + o_off);
  int *cnt = reinterpret_cast<int *>(ctx->drain_pin.p + o_cnt);
  HIPCHK(hipMemcpyAsync(cnt, cnt_d, n * sizeof(int), hipMemcpyDeviceToHost, stream));
  HIPCHK(hipStreamSynchronize(stream));
  off[0] = 0;
  for (int i = 0; i < n; ++i) off[i + 1] = off[i] + cnt[i];
  const int64_t tot = off[n];
  if (tot > 0) {
    if (tot > ctx->d_drain_cap) {
      if (ctx->d_drain) (void)hipFree(ctx->d_drain);
      ctx->d_drain = nullptr;
      ctx->d_drain_cap = 0;
      const int64_t cap = tot + tot / 8;
      HIPCHK(hipMalloc(&ctx->d_drain, cap * sizeof(gd_record)));
      ctx->d_drain_cap = cap;
    }
    if (!ctx->d_drain_off) HIPCHK(hipMalloc(&ctx->d_drain_off, (n + 1) * sizeof(int64_t)));
    HIPCHK(hipMemcpyAsync(ctx->d_drain_off, off, (n + 1) * sizeof(int64_t),
                          hipMemcpyHostToDevice, stream));
    hipLaunchKernelGGL(gd_compact_kernel, dim3(n), dim3(256), 0, stream, n, ctx->d_ring[r],
                       cnt_d, ctx->d_drain_off, ctx->rec_cap, ctx->d_drain);
    HIPCHK(hipGetLastError());
  }
  HIPCHK(hipMemsetAsync(cnt_d, 0, n * sizeof(int), stream));
  ctx->drain_total = tot;
  return GD_OK;
}

// The compacted window to the sink; `stream` (compact_ring's) is synchronized
// before.
gd_status deliver_records(gd_ctx *ctx, gd_record_sink sink, void *user, hipStream_t stream) {
  const int64_t tot = ctx->drain_total;
  ctx->drain_total = 0;
  if (tot == 0) return GD_OK;
  if (tot > ctx->h_drain_cap) {
    if (ctx->h_drain) (void)hipHostFree(ctx->h_drain);
    ctx->h_drain = nullptr;
    ctx->h_drain_cap = 0;
    HIPCHK(hipHostMalloc(&ctx->h_drain, ctx->d_drain_cap * sizeof(gd_record),
                         hipHostMallocDefault));
    ctx->h_drain_cap = ctx->d_drain_cap;
  }
  HIPCHK(hipMemcpyAsync(ctx->h_drain, ctx->d_drain, tot * sizeof(gd_record),
                        hipMemcpyDeviceToHost, stream));
  HIPCHK(hipStreamSynchronize(stream));
  const int64_t *off = reinterpret_cast<const int64_t *>(ctx->drain_pin.p);
  for (int c = 0; c < (int)ctx->cx.size(); ++c) {
    const HostComplex &h = ctx->cx[c];
    const int64_t b = off[h.rep_base], e = off[h.rep_base + h.n_rep];
    if (e > b) sink(user, c, ctx->h_drain + b, e - b);
  }
  return GD_OK;
}

// Drains the current ring on the main stream; without a sink its records go.
gd_status drain_records(gd_ctx *ctx, gd_record_sink sink, void *user) {
  if (!ctx->d_ring[ctx->ring]) return GD_OK;
  if (!sink) {
    HIPCHK(hipMemsetAsync(ctx->d_ring_cnt[ctx->ring], 0, ctx->n_rep * sizeof(int), ctx->stream));
    return GD_OK;
  }
  TRY(compact_ring(ctx, ctx->ring, ctx->stream));
  return deliver_records(ctx, sink, user, ctx->stream);
}

// Record rings for windows of up to `win` steps (and the start poses): ring 0,
// and ring 1 when windows alternate. Called between runs, when they are empty.
// They grow with the longest window asked for, not to steps_per_dump at once
// (93 MB and 1 ms for a first run of 200 steps of 504 replicas). Rings that do
// not fit are all given back, so a run of shorter windows sizes its own.
gd_status ensure_rings(gd_ctx *ctx, int win, bool both) {
  if (!ctx->opts.record) return GD_OK;
  const size_t n = ctx->n_rep;
  auto drop = [&] {
    for (int r = 0; r < 2; ++r) {
      if (ctx->d_ring[r]) (void)hipFree(ctx->d_ring[r]);
      ctx->d_ring[r] = nullptr;
    }
    for (auto &g : ctx->gslot) g.valid = false;  // captured launches hold the old rings
    ctx->rec_cap = 0;
  };
  if (win + 1 > ctx->rec_cap) {
    drop();
    for (int r = 0; r < 2; ++r)
      if (ctx->d_ring_cnt[r]) HIPCHK(hipMemsetAsync(ctx->d_ring_cnt[r], 0, n * sizeof(int), ctx->stream));
    ctx->rec_cap = win + 1;
  }
  for (int r = 0; r < 2; ++r) {
    // the ring in use may be the second, left current by windows that alternated
    const bool used = r == 0 || both || r == ctx->ring;
    if (used && !ctx->d_ring[r]) {
      const hipError_t e = hipMalloc(&ctx->d_ring[r], n * ctx->rec_cap * sizeof(gd_record));
      if (e != hipSuccess) {
        ctx->d_ring[r] = nullptr;
        const int cap = ctx->rec_cap;
        drop();
        return fail(ctx, GD_ERR_HIP, "record rings of %d steps: %s", cap, hipGetErrorString(e));
      }
    }
    if (used && !ctx->d_ring_cnt[r]) {
      HIPCHK(hipMalloc(&ctx->d_ring_cnt[r], n * sizeof(int)));
      HIPCHK(hipMemsetAsync(ctx->d_ring_cnt[r], 0, n * sizeof(int), ctx->stream));
    }
  }
  if (both && !ctx->drain_stream)
    HIPCHK(hipStreamCreateWithFlags(&ctx->drain_stream, hipStreamNonBlocking));
  if (both && !ctx->ev_compact)
    HIPCHK(hipEventCreateWithFlags(&ctx->ev_compact, hipEventDisableTiming));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return GD_OK;
}

// Kernel arguments of an MC launch; with da_k > 0 of the delayed-acceptance
// kernels.
KParams mc_params(gd_ctx *ctx, int da_k, float sur_scale) {
  KParams P = base_params(ctx);
  P.mode = MODE_MC;
  if (da_k > 0) {
    auto &S = ctx->sur;
    P.da_k = da_k;
    P.sur_scale = sur_scale;
    P.sW1T = S.W1T;
    P.sW2T = S.W2T;
    P.sb2 = S.p + SP_B2;
    P.sw3 = S.p + SP_W3;
    P.sb3 = S.p + SP_B3;
    P.sur_tab = S.tab_valid ? 1 : 0;
  }
  return P;
}

// Enqueue one MC launch (mode, window of n_steps from step0) on ctx->stream
// between the timing events ev0 and ev1; launch_mc_wait waits for it.
gd_status launch_mc_enqueue(gd_ctx *ctx, int mode, int step0, int n_steps, int nc, int da_k = 0,
                            float sur_scale = 1.0f) {
  KParams P = mc_params(ctx, mode == MODE_MC ? da_k : 0, sur_scale);
  P.mode = mode;
  P.step0 = step0;
  P.n_steps = n_steps;
  P.nc = nc;
  // the direct network evaluation needs per-wave LDS scratch
  const bool scratch = P.da_k > 0 && !P.sur_tab;
  const int da = P.da_k > 0 ? da_instance(ctx, P.sur_tab != 0) : 0;
  const bool persistent = (ctx->opts.launch & GD_LAUNCH_PERSISTENT) && mode == MODE_MC;
  const bool use_graph = !(ctx->opts.launch & GD_LAUNCH_NO_GRAPH) && mode == MODE_MC;
  int *queue = persistent ? ctx->d_ctrl + 1 : nullptr;
  if (use_graph) {
    // the first step comes from device memory so one graph serves every window
    P.step_dev = ctx->d_ctrl;
    // one graph slot per record ring (the ring's pointers are kernel arguments)
    auto &G = ctx->gslot[ctx->ring];
    const bool same = G.valid && G.mode == mode && G.win == n_steps && G.nc == nc &&
                      G.da == P.da_k && G.tab == P.sur_tab && G.scale == P.sur_scale &&
                      G.persistent == (int)persistent;
    if (!same) {
      if (G.exec) (void)hipGraphExecDestroy(G.exec);
      G.exec = nullptr;
      G.valid = false;
      std::vector<ClassLaunch> cls;
      hipError_t e = plan_classes(ctx, ctx->mc_classes, P, da, scratch, queue, cls);
      if (e == hipErrorInvalidValue)
        return fail(ctx, GD_ERR_CAPACITY, "delayed acceptance scratch does not fit in LDS");
      HIPCHK(e);
      hipGraph_t g = nullptr;
      HIPCHK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
      e = enqueue_classes(ctx, cls, queue, ctx->stream);
      const hipError_t e2 = hipStreamEndCapture(ctx->stream, &g);
      HIPCHK(e);
      HIPCHK(e2);
      e = hipGraphInstantiate(&G.exec, g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      HIPCHK(e);
      G.valid = true;
      G.mode = mode;
      G.win = n_steps;
      G.nc = nc;
      G.da = P.da_k;
      G.tab = P.sur_tab;
      G.scale = P.sur_scale;
      G.persistent = (int)persistent;
    }
    ctx->h_step = step0;
    HIPCHK(hipMemcpyAsync(ctx->d_ctrl, &ctx->h_step, sizeof(int), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipEventRecord(ctx->ev0, ctx->stream));
    HIPCHK(hipGraphLaunch(G.exec, ctx->stream));
  } else {
    std::vector<ClassLaunch> cls;
    hipError_t e = plan_classes(ctx, ctx->mc_classes, P, da, scratch, queue, cls);
    if (e == hipErrorInvalidValue)
      return fail(ctx, GD_ERR_CAPACITY, "delayed acceptance scratch does not fit in LDS");
    HIPCHK(e);
    HIPCHK(hipEventRecord(ctx->ev0, ctx->stream));
    HIPCHK(enqueue_classes(ctx, cls, queue, ctx->stream));
  }
  HIPCHK(hipGetLastError());
  HIPCHK(hipEventRecord(ctx->ev1, ctx->stream));
  return GD_OK;
}

gd_status launch_mc_wait(gd_ctx *ctx, float *ms) {
  HIPCHK(hipEventSynchronize(ctx->ev1));
  if (ms) HIPCHK(hipEventElapsedTime(ms, ctx->ev0, ctx->ev1));
  return GD_OK;
}

gd_status launch_mc(gd_ctx *ctx, int mode, int step0, int n_steps, int nc, float *ms,
                    int da_k = 0, float sur_scale = 1.0f) {
  TRY(launch_mc_enqueue(ctx, mode, step0, n_steps, nc, da_k, sur_scale));
  return launch_mc_wait(ctx, ms);
}

// Steps that one launch of a small context takes through a tree of energies
// (MODE_TREE in gd_mc.h): the deepest tree whose nodes, one workgroup each per
// pack, still run side by side, one workgroup per CU. 1: plain MC launches.
// A launch of two steps already pays at the line (85 packs, small receptors
// of 300 points: 2.4 -> 2.25 ms for 100 steps; 2,000 points: 5.5 -> 2.9 ms at
// 32 packs); beyond it the nodes would queue.
int tree_depth(const gd_ctx *ctx) {
  int64_t packs = 0;
  for (const LaunchClass &lc : ctx->mc_classes) packs += lc.end - lc.begin;
  int d = 1;
  while (d < TREE_DEPTH && packs * ((2 << d) - 1) <= ctx->n_cu) ++d;
  return d;
}

// The packs' counts of finished nodes (zero between launches), then the
// energies of the tree's nodes for every replica.
gd_status tree_buffers(gd_ctx *ctx, int depth, int **cnt, gd_energy **e) {
  size_t packs = 0;
  for (const LaunchClass &lc : ctx->mc_classes) packs = std::max(packs, (size_t)lc.end);
  Regions R;
  const size_t o_cnt = R.add(packs * sizeof(int));
  const size_t o_e = R.add((size_t)ctx->n_rep * ((1 << depth) - 1) * sizeof(gd_energy));
  TRY(scratch_need(ctx, ctx->tree, R.end, false));
  *cnt = reinterpret_cast<int *>(ctx->tree.p + o_cnt);
  *e = reinterpret_cast<gd_energy *>(ctx->tree.p + o_e);
  HIPCHK(hipMemsetAsync(*cnt, 0, packs * sizeof(int), ctx->stream));
  return GD_OK;
}

// One window of spread packing: MC launches that end on exchange steps, each
// followed by the ladder exchange kernel, all enqueued at once and timed
// together (waiting for each launch left the GPU idle for 60 to 90 us every
// exchange interval). ctx->step follows each launch as it is enqueued, so a window
// that ends in an error does not take the same random numbers again.
gd_status spread_window(gd_ctx *ctx, int win, int nc, int da_k, float sur_scale, double *ms_sum,
                        int *launches) {
  KParams P = mc_params(ctx, da_k, sur_scale);
  const bool persistent = (ctx->opts.launch & GD_LAUNCH_PERSISTENT) != 0;
  const int depth = da_k > 0 || persistent ? 1 : tree_depth(ctx);
  const int da = P.da_k > 0 ? da_instance(ctx, P.sur_tab != 0) : depth > 1 ? DA_TREE : 0;
  int *queue = persistent ? ctx->d_ctrl + 1 : nullptr;
  std::vector<ClassLaunch> cls;
  const hipError_t pe =
      plan_classes(ctx, ctx->mc_classes, P, da, P.da_k > 0 && !P.sur_tab, queue, cls);
  if (pe == hipErrorInvalidValue)
    return fail(ctx, GD_ERR_CAPACITY, "delayed acceptance scratch does not fit in LDS");
  HIPCHK(pe);
  int *tree_cnt = nullptr;
  gd_energy *tree_e = nullptr;
  if (depth > 1) TRY(tree_buffers(ctx, depth, &tree_cnt, &tree_e));
  HIPCHK(hipEventRecord(ctx->ev0, ctx->stream));
  for (int done = 0; done < win;) {
    const int s = (int)ctx->step;
    int sub = win - done;
    if (nc > 0) sub = std::min(sub, nc - s % nc);
    if (depth > 1) {
      // even shares of the interval, none deeper than `depth`
      const int rounds = (sub + depth - 1) / depth;
      for (int r = 0, at = s; r < rounds; ++r) {
        const int d = (s + sub - at) / (rounds - r);
        for (ClassLaunch &cl : cls) {
          cl.P.mode = MODE_TREE;
          cl.P.tree_cnt = tree_cnt;
          cl.P.ev_out = tree_e;
          cl.P.step0 = at;
          cl.P.n_steps = d;
          cl.P.tree_nodes = (1 << d) - 1;
          cl.P.tree_packs = cl.packs;
          cl.grid = cl.packs * cl.P.tree_nodes;
        }
        HIPCHK(enqueue_classes(ctx, cls, nullptr, ctx->stream));
        ctx->step += d;
        at += d;
      }
      *launches += rounds - 1;
    } else {
      for (ClassLaunch &cl : cls) {
        cl.P.step0 = s;
        cl.P.n_steps = sub;
      }
      HIPCHK(enqueue_classes(ctx, cls, queue, ctx->stream));
      ctx->step += sub;
    }
    if (nc > 0 && (s + sub) % nc == 0) {
      hipLaunchKernelGGL(gd_ladder_exchange_kernel, dim3((ctx->n_ladders + 63) / 64), dim3(64),
                         0, ctx->stream, ctx->d_cx, ctx->d_ladders, ctx->n_ladders, s + sub, nc,
                         P.k0, P.k1, ctx->d_eold, ctx->d_idx_tmp, ctx->d_acs_x);
      HIPCHK(hipGetLastError());
    }
    *launches += 1;
    done += sub;
  }
  HIPCHK(hipEventRecord(ctx->ev1, ctx->stream));
  float ms = 0.f;
  TRY(launch_mc_wait(ctx, &ms));
  *ms_sum += ms;
  return GD_OK;
}

}  // namespace

extern "C" {

static gd_status run_impl(gd_ctx *ctx, int64_t n_steps, int steps_per_exchange,
                          gd_record_sink sink, void *user, gd_run_stats *stats, int da_k,
                          float sur_scale);

gd_status gd_run(gd_ctx *ctx, int64_t n_steps, int steps_per_exchange, gd_record_sink sink,
                 void *user, gd_run_stats *stats) {
  return run_impl(ctx, n_steps, steps_per_exchange, sink, user, stats, 0, 1.0f);
}

gd_status gd_run_da(gd_ctx *ctx, int64_t n_steps, int steps_per_exchange, int k_sub,
                    float sur_scale, gd_record_sink sink, void *user, gd_run_stats *stats) {
  if (!ctx) return GD_ERR_INVALID;
  if (k_sub < 1) return fail(ctx, GD_ERR_INVALID, "k_sub must be >= 1");
  if (ctx->sur.g.size() != ctx->cx.size()) return fail(ctx, GD_ERR_STATE, "call gd_sur_build_grids first");
  if (!ctx->sur.have_params) return fail(ctx, GD_ERR_STATE, "no surrogate parameters");
  if (n_steps % k_sub != 0 || (steps_per_exchange > 0 && steps_per_exchange % k_sub != 0) ||
      ctx->step % k_sub != 0)
    return fail(ctx, GD_ERR_INVALID, "step counts must be multiples of k_sub");
  return run_impl(ctx, n_steps, steps_per_exchange, sink, user, stats, k_sub, sur_scale);
}

static gd_status run_impl(gd_ctx *ctx, int64_t n_steps, int steps_per_exchange,
                          gd_record_sink sink, void *user, gd_run_stats *stats, int da_k,
                          float sur_scale) {
  if (!ctx) return GD_ERR_INVALID;
  if (n_steps < 0 || steps_per_exchange < 0) return fail(ctx, GD_ERR_INVALID, "negative step count");
  if (ctx->step + n_steps > 2000000000LL) return fail(ctx, GD_ERR_CAPACITY, "step counter overflow");
  HIPCHK(hipSetDevice(ctx->device));
  const auto t_start = std::chrono::steady_clock::now();
  TRY(alloc_state(ctx));
  gd_run_stats st{};
  const bool spread = spread_packing(ctx);
  const bool overlap = sink && ctx->opts.record && n_steps > 0 && !spread;
  const int win0 = (int)std::min<int64_t>(n_steps, ctx->opts.steps_per_dump);
  TRY(ensure_rings(ctx, da_k > 0 ? std::max(da_k, win0) : win0, overlap));
  // accepted moves and exchanges before and after, summed on the device
  // (the sinks may call back: these words are not part of the scratch)
  if (!ctx->h_counts)
    HIPCHK(hipHostMalloc((void **)&ctx->h_counts, 4 * sizeof(int64_t), hipHostMallocDefault));
  int64_t *counts = ctx->h_counts;
  hipLaunchKernelGGL(gd_counts_kernel, dim3(1), dim3(1024), 0, ctx->stream, ctx->n_rep,
                     ctx->d_acs_mc, ctx->d_acs_x, counts);
  HIPCHK(hipGetLastError());
  if (!ctx->initialized) {
    float ms = 0.f;
    TRY(launch_mc(ctx, MODE_INIT, (int)ctx->step, 0, 0, &ms));
    ctx->initialized = true;
  }
  int64_t left = n_steps;
  double t_ms = 0.0;
  // with records and a sink, windows alternate between the two rings: the
  // previous window's records, compacted between the windows, are delivered (on
  // the drain stream, sinks called here) while the next window runs
  bool pending = false;
  while (left > 0) {
    int win = (int)std::min<int64_t>(left, ctx->opts.steps_per_dump);
    if (da_k > 0) win = std::max(da_k, win / da_k * da_k);
    if (spread) {
      TRY(spread_window(ctx, win, steps_per_exchange, da_k, sur_scale, &t_ms, &st.kernel_launches));
      left -= win;
      TRY(drain_records(ctx, sink, user));
      continue;
    }
    float ms = 0.f;
    TRY(launch_mc_enqueue(ctx, MODE_MC, (int)ctx->step, win, steps_per_exchange, da_k, sur_scale));
    // a failed drain is reported after the window in flight has finished
    const gd_status ds =
        pending ? deliver_records(ctx, sink, user, ctx->drain_stream) : GD_OK;
    TRY(launch_mc_wait(ctx, &ms));
    t_ms += ms;
    st.kernel_launches += 1;
    ctx->step += win;
    left -= win;
    if (ds != GD_OK) return ds;
    if (overlap) {
      TRY(compact_ring(ctx, ctx->ring, left > 0 ? ctx->drain_stream : ctx->stream));
      if (left > 0) {
        HIPCHK(hipEventRecord(ctx->ev_compact, ctx->drain_stream));
        HIPCHK(hipStreamWaitEvent(ctx->stream, ctx->ev_compact, 0));
      }
      pending = true;
      ctx->ring ^= 1;
    } else {
      TRY(drain_records(ctx, sink, user));
    }
  }
  if (pending) TRY(deliver_records(ctx, sink, user, ctx->stream));
  if (n_steps == 0) TRY(drain_records(ctx, sink, user));
  hipLaunchKernelGGL(gd_counts_kernel, dim3(1), dim3(1024), 0, ctx->stream, ctx->n_rep,
                     ctx->d_acs_mc, ctx->d_acs_x, counts + 2);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(ctx->stream));
  st.accepted = counts[2] - counts[0];
  st.exchanges_accepted = counts[3] - counts[1];
  st.t_compute = t_ms * 1e-3;
  st.steps = n_steps;
  st.replica_steps = n_steps * (int64_t)ctx->n_rep;
  st.kernel_ms_avg = st.kernel_launches ? t_ms / st.kernel_launches : 0.0;
  st.t_wall = std::chrono::duration<double>(std::chrono::steady_clock::now() - t_start).count();
  if (stats) *stats = st;
  return GD_OK;
}

// Copies device arrays to host ones: one kernel gathers them into the pinned
// staging (five copies of a few KB each took 100 us and more).
struct HostCopy {
  const void *src;
  void *dst;  // null: left out
  size_t bytes;
};

static gd_status copy_out(gd_ctx *ctx, std::initializer_list<HostCopy> parts) {
  GatherArgs A{};
  size_t words = 0;
  for (const HostCopy &c : parts) {
    if (!c.dst || c.bytes == 0) continue;
    A.src[A.n] = static_cast<const int *>(c.src);
    words += c.bytes / sizeof(int);
    A.end[A.n++] = (long long)words;
  }
  if (A.n == 0) return GD_OK;
  const ScratchTrim trim{ctx};
  TRY(scratch_need(ctx, ctx->pin, words * sizeof(int), true));
  hipLaunchKernelGGL(gd_gather_kernel, dim3((unsigned)std::min<size_t>((words + 255) / 256, 1024)),
                     dim3(256), 0, ctx->stream, A, reinterpret_cast<int *>(ctx->pin.p));
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(ctx->stream));
  const unsigned char *p = ctx->pin.p;
  for (const HostCopy &c : parts) {
    if (!c.dst || c.bytes == 0) continue;
    memcpy(c.dst, p, c.bytes);
    p += c.bytes;
  }
  return GD_OK;
}

gd_status gd_get_state(gd_ctx *ctx, int cid, float *movematrix, gd_energy *energy_old,
                       gd_replica *replica, int32_t *acs_mc, int32_t *acs_x) {
  if (!ctx || cid < 0 || cid >= (int)ctx->cx.size()) return GD_ERR_INVALID;
  if (!ctx->state_alloc) return fail(ctx, GD_ERR_STATE, "no state before gd_run");
  HIPCHK(hipSetDevice(ctx->device));
  const HostComplex &h = ctx->cx[cid];
  const size_t b = h.rep_base, n = h.n_rep;
  std::vector<int> it(replica ? n : 0);
  TRY(copy_out(ctx, {{ctx->d_mm + b * 6, movematrix, n * 6 * sizeof(float)},
                     {ctx->d_eold + b, energy_old, n * sizeof(gd_energy)},
                     {ctx->d_acs_mc + b, acs_mc, n * sizeof(int)},
                     {ctx->d_acs_x + b, acs_x, n * sizeof(int)},
                     {ctx->d_idx_tmp + b, replica ? it.data() : nullptr, n * sizeof(int)}}));
  if (replica) {
    for (size_t f = 0; f < n; ++f) {
      replica[f].idx_rep = (int)f;
      replica[f].idx_prt = (int)(f / (h.d.n_tmp * h.d.n_lig));
      replica[f].idx_tmp = it[f];
      replica[f].idx_lig = (int)(f % h.d.n_lig);
    }
  }
  return GD_OK;
}

gd_status gd_get_best(gd_ctx *ctx, int cid, float *best_e, float *best_mm) {
  if (!ctx || cid < 0 || cid >= (int)ctx->cx.size()) return GD_ERR_INVALID;
  if (!ctx->initialized) return fail(ctx, GD_ERR_STATE, "no state before gd_run");
  HIPCHK(hipSetDevice(ctx->device));
  const HostComplex &h = ctx->cx[cid];
  const size_t b = h.rep_base, n = h.n_rep;
  return copy_out(ctx, {{ctx->d_best_e + b, best_e, n * sizeof(float)},
                        {ctx->d_best_mm + b * 6, best_mm, n * 6 * sizeof(float)}});
}

gd_status gd_reset_best(gd_ctx *ctx) {
  if (!ctx) return GD_ERR_INVALID;
  if (!ctx->initialized) return fail(ctx, GD_ERR_STATE, "no state before gd_run");
  HIPCHK(hipSetDevice(ctx->device));
  const int n = ctx->n_rep;
  hipLaunchKernelGGL(gd_reset_best_kernel, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n,
                     ctx->d_eold, ctx->d_mm, ctx->d_best_e, ctx->d_best_mm);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return GD_OK;
}

static const uint32_t kCkptMagic = 0x47444b32u;  // "GDK2"

gd_status gd_checkpoint(gd_ctx *ctx, void *buf, size_t *size) {
  if (!ctx || !size) return GD_ERR_INVALID;
  if (!ctx->state_alloc) return fail(ctx, GD_ERR_STATE, "no state before gd_run");
  const size_t n = ctx->n_rep;
  const size_t need = 32 + n * (13 * sizeof(float) + sizeof(gd_energy) + 3 * sizeof(int));
  if (!buf || *size < need) {
    *size = need;
    return buf ? fail(ctx, GD_ERR_INVALID, "checkpoint buffer too small") : GD_OK;
  }
  HIPCHK(hipSetDevice(ctx->device));
  char *o = (char *)buf;
  uint32_t hdr[8] = {kCkptMagic, (uint32_t)n, (uint32_t)ctx->initialized, 0,
                     (uint32_t)(ctx->step & 0xffffffffu), (uint32_t)(ctx->step >> 32),
                     (uint32_t)ctx->cx.size(), 0};
  memcpy(o, hdr, 32);
  o += 32;
  HIPCHK(hipMemcpyAsync(o, ctx->d_mm, n * 6 * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
  o += n * 6 * sizeof(float);
  HIPCHK(hipMemcpyAsync(o, ctx->d_eold, n * sizeof(gd_energy), hipMemcpyDeviceToHost, ctx->stream));
  o += n * sizeof(gd_energy);
  HIPCHK(hipMemcpyAsync(o, ctx->d_idx_tmp, n * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  o += n * sizeof(int);
  HIPCHK(hipMemcpyAsync(o, ctx->d_acs_mc, n * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  o += n * sizeof(int);
  HIPCHK(hipMemcpyAsync(o, ctx->d_acs_x, n * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  o += n * sizeof(int);
  HIPCHK(hipMemcpyAsync(o, ctx->d_best_e, n * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
  o += n * sizeof(float);
  HIPCHK(hipMemcpyAsync(o, ctx->d_best_mm, n * 6 * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  *size = need;
  return GD_OK;
}

gd_status gd_restore(gd_ctx *ctx, const void *buf, size_t size) {
  if (!ctx || !buf) return GD_ERR_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  TRY(alloc_state(ctx));
  const size_t n = ctx->n_rep;
  const size_t need = 32 + n * (13 * sizeof(float) + sizeof(gd_energy) + 3 * sizeof(int));
  uint32_t hdr[8];
  if (size < need) return fail(ctx, GD_ERR_INVALID, "checkpoint too small");
  memcpy(hdr, buf, 32);
  if (hdr[0] != kCkptMagic || hdr[1] != n || hdr[6] != ctx->cx.size())
    return fail(ctx, GD_ERR_INVALID, "checkpoint does not match this context");
  const char *o = (const char *)buf + 32;
  HIPCHK(hipMemcpyAsync(ctx->d_mm, o, n * 6 * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
  o += n * 6 * sizeof(float);
  HIPCHK(hipMemcpyAsync(ctx->d_eold, o, n * sizeof(gd_energy), hipMemcpyHostToDevice, ctx->stream));
  o += n * sizeof(gd_energy);
  HIPCHK(hipMemcpyAsync(ctx->d_idx_tmp, o, n * sizeof(int), hipMemcpyHostToDevice, ctx->stream));
  o += n * sizeof(int);
  HIPCHK(hipMemcpyAsync(ctx->d_acs_mc, o, n * sizeof(int), hipMemcpyHostToDevice, ctx->stream));
  o += n * sizeof(int);
  HIPCHK(hipMemcpyAsync(ctx->d_acs_x, o, n * sizeof(int), hipMemcpyHostToDevice, ctx->stream));
  o += n * sizeof(int);
  HIPCHK(hipMemcpyAsync(ctx->d_best_e, o, n * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
  o += n * sizeof(float);
  HIPCHK(hipMemcpyAsync(ctx->d_best_mm, o, n * 6 * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
  for (int r = 0; r < 2; ++r)
    if (ctx->d_ring_cnt[r]) HIPCHK(hipMemsetAsync(ctx->d_ring_cnt[r], 0, n * sizeof(int), ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  ctx->initialized = hdr[2] != 0;
  ctx->step = (int64_t)hdr[4] | ((int64_t)hdr[5] << 32);
  return GD_OK;
}

static gd_status eval_poses(gd_ctx *ctx, int cid, int n, const int *idx_lig, const int *idx_prt,
                            const float *movematrix, gd_energy *out, float *out_sur,
                            float sur_scale, bool no_alloc = false);

gd_status gd_calc_energy_noalloc(gd_ctx *ctx, int cid, int n, const int *idx_lig,
                                 const int *idx_prt, const float *movematrix, gd_energy *out) {
  if (!ctx || cid < 0 || cid >= (int)ctx->cx.size() || n < 0) return GD_ERR_INVALID;
  if (n == 0) return GD_OK;
  if (!idx_lig || !idx_prt || !movematrix || !out) return GD_ERR_INVALID;
  if (n > GD_NOALLOC_MAX_POSES)
    return fail(ctx, GD_ERR_CAPACITY, "gd_calc_energy_noalloc: %d poses > %d per call", n,
                GD_NOALLOC_MAX_POSES);
  if (!ctx->scratch) return fail(ctx, GD_ERR_STATE, "no device scratch address");
  if (ctx->cx_dirty || !ctx->cx[cid].ref_built)
    return fail(ctx, GD_ERR_STATE,
                "gd_calc_energy_noalloc: the complex table and contact map are not on the device "
                "yet; call gd_calc_energy or gd_run once after the last gd_add_complex");
  return eval_poses(ctx, cid, n, idx_lig, idx_prt, movematrix, out, nullptr, 0.0f, true);
}

gd_status gd_calc_energy(gd_ctx *ctx, int cid, int n, const int *idx_lig, const int *idx_prt,
                         const float *movematrix, gd_energy *out) {
  if (!ctx || cid < 0 || cid >= (int)ctx->cx.size() || n < 0) return GD_ERR_INVALID;
  if (n == 0) return GD_OK;
  if (!idx_lig || !idx_prt || !movematrix || !out) return GD_ERR_INVALID;
  return eval_poses(ctx, cid, n, idx_lig, idx_prt, movematrix, out, nullptr, 0.0f);
}

gd_status gd_sur_surrogate(gd_ctx *ctx, int cid, int n, const int *idx_lig, const int *idx_prt,
                           const float *movematrix, float sur_scale, float *out) {
  if (!ctx || cid < 0 || cid >= (int)ctx->cx.size() || n < 0) return GD_ERR_INVALID;
  if (n == 0) return GD_OK;
  if (!idx_lig || !idx_prt || !movematrix || !out) return GD_ERR_INVALID;
  if (ctx->sur.g.size() != ctx->cx.size()) return fail(ctx, GD_ERR_STATE, "call gd_sur_build_grids first");
  if (!ctx->sur.have_params) return fail(ctx, GD_ERR_STATE, "no surrogate parameters");
  return eval_poses(ctx, cid, n, idx_lig, idx_prt, movematrix, nullptr, out, sur_scale);
}

// Energies (or surrogate totals) of n poses of one complex. With no_alloc the
// pose tables and outputs live in the device scratch array (the caller has
// checked n and that the complex table and contact map are on the device);
// otherwise in the context's staging: pinned memory that the kernel reads and
// writes itself for small calls, else device memory with a copy each way.
static gd_status eval_poses(gd_ctx *ctx, int cid, int n, const int *idx_lig, const int *idx_prt,
                            const float *movematrix, gd_energy *out, float *out_sur,
                            float sur_scale, bool no_alloc) {
  HostComplex &h = ctx->cx[cid];
  for (int i = 0; i < n; ++i)
    if (idx_lig[i] < 0 || idx_lig[i] >= h.d.n_lig || idx_prt[i] < 0 || idx_prt[i] >= h.d.n_prt)
      return fail(ctx, GD_ERR_INVALID, "pose %d: conformer index out of range", i);
  HIPCHK(hipSetDevice(ctx->device));
  if (!no_alloc) TRY(ensure_ref(ctx));
  // each pose is evaluated with the receptor split of its ligand conformer's
  // MC packs, so a pose's energy has the bits an MC step gives it
  std::vector<int> lig_ns = h.lig_ns;
  if (lig_ns.size() != (size_t)h.d.n_lig) lig_ns = lig_splits(ctx, h, auto_gmax(ctx));
  // poses by protein conformer and split
  std::vector<int> key(n), start(h.d.n_prt * 4 + 1, 0), order(n);
  for (int i = 0; i < n; ++i) {
    const int ns = lig_ns[idx_lig[i]];
    key[i] = idx_prt[i] * 4 + (ns >= 8 ? 3 : ns >= 4 ? 2 : ns >= 2 ? 1 : 0);
    start[key[i] + 1] += 1;
  }
  for (size_t k = 1; k < start.size(); ++k) start[k] += start[k - 1];
  {
    std::vector<int> at(start.begin(), start.end() - 1);
    for (int i = 0; i < n; ++i) order[at[key[i]]++] = i;
  }
  // the launch takes the flat pair loop (plan_classes): a list that fits, and
  // no scratch of the direct network evaluation
  auto flat_fits = [&](int lpr) {
    KParams L{};
    size_t need = 0;
    layout(L, &need, 0, h.d.pnk, h.n_chunks, std::max(1, 64 / lpr), 512, true, 0, h.flat_n[3]);
    return need <= ctx->max_lds;
  };
  const bool flat = ctx->flat && h.flat_n[3] > 0 && !(out_sur && !ctx->sur.tab_valid) &&
                    flat_fits(h.lpr);
  // Spread packing widens the lane shape of complexes with few packs, at the
  // cost of lanes without an atom and of independent work per lane. Larger
  // pose sets take the shape of fewest lane slots, in the wide shape's order of
  // additions (J in gd_mc.h), where its rounds of packs over the CUs cost
  // less: per atom of a lane 0.65 of the wide shape's time with unit lists,
  // 0.75 with tiles. 16,384 poses of 38 atoms (64 lanes of one atom, 16 of
  // three) on 2,400 points 3.77 -> 2.38 ms; 2,000 of 61 atoms on 8,000 points
  // (tiles) 1.54 -> 1.30; 1,100 of 45 atoms on 6,000 points, near the line, 0.79
  // -> 0.74.
  int lpr = h.lpr, apl = h.apl, da_poses = 0;
  if ((h.tiled || (flat && flat_fits(h.lpr0))) && !out_sur && spread_packing(ctx) &&
      h.lpr0 < h.lpr && h.apl0 > 1 && h.apl0 < 4) {
    auto cost = [&](int l, int a) {
      const int64_t packs = ((int64_t)n * l + 63) / 64;
      return (double)((packs + ctx->n_cu - 1) / ctx->n_cu) * a;
    };
    if (cost(h.lpr0, h.apl0) * (h.tiled ? 0.75 : 0.65) < 0.95 * cost(h.lpr, h.apl)) {
      lpr = h.lpr0;
      apl = h.apl0;
      da_poses = h.apl == 2 ? DA_POSES2 : DA_POSES;
    }
  }
  PackSet ps;
  ps.slots = order;
  for (int k = 0; k < h.d.n_prt * 4; ++k) {
    const int cnt = start[k + 1] - start[k], ns = 1 << (k & 3);
    const int per = std::max(1, (512 / ns) / lpr);
    // With the flat pair loop (a split of 8: a few poses at a time) a workgroup
    // stages the receptor once for several rounds of poses, as long as that
    // leaves four workgroups per CU: 16,384 poses on 2,400 points staged about
    // 100 KB for every pose otherwise (4.6 ms, 3.8 ms with rounds)
    const int rounds = (cnt + per - 1) / per;
    const int many = ns == 8 && flat ? std::max(1, rounds / (4 * std::max(1, ctx->n_cu))) : 1;
    for (int b = 0; b < cnt; b += per * many) {
      Pack pk{};
      pk.cx = cid;
      pk.prt = k / 4;
      pk.n_slots = std::min(per * many, cnt - b);
      pk.round = std::min(per, pk.n_slots);
      pk.n_groups = 0;
      pk.ns = ns;
      pk.slot_off = start[k] + b;
      ps.packs.push_back(pk);
    }
  }
  if (da_poses) pack_finish(ctx, ps, lpr, apl);
  else pack_finish(ctx, ps);
  for (const LaunchClass &lc : ps.classes)
    for (int i = lc.begin; i < lc.end; ++i)
      if (lc.lds_flat == 0 && ((da_poses && lc.tile == 0) || ps.packs[i].round < ps.packs[i].n_slots))
        return fail(ctx, GD_ERR_STATE, "pose packs without the flat pair loop");
  for (const LaunchClass &lc : ps.classes)
    if (lc.lds > ctx->max_lds && lc.lds_flat == 0) return fail(ctx, GD_ERR_CAPACITY, "LDS %zu > %zu", lc.lds, ctx->max_lds);
  KParams P{};
  const bool sur = out_sur != nullptr;
  if (sur) {
    auto &S = ctx->sur;
    P.sur_scale = sur_scale;
    P.sur_tab = S.tab_valid ? 1 : 0;
    P.sW1T = S.W1T;
    P.sW2T = S.W2T;
    P.sb2 = S.p + SP_B2;
    P.sw3 = S.p + SP_W3;
    P.sb3 = S.p + SP_B3;
  }
  // inputs (packs, slots, conformers, poses), then results
  Regions R;
  const size_t o_packs = R.add(ps.packs.size() * sizeof(Pack));
  const size_t o_slots = R.add(ps.slots.size() * sizeof(int));
  const size_t o_lig = R.add((size_t)n * sizeof(int));
  const size_t o_mm = R.add((size_t)n * 6 * sizeof(float));
  const size_t o_out = R.end;
  const size_t res_bytes = (size_t)n * (sur ? sizeof(float) : sizeof(gd_energy));
  R.add(res_bytes);
  const ScratchTrim trim{ctx};
  unsigned char *base = nullptr;  // where the kernel reads and writes
  const bool direct = !no_alloc && R.end <= ZERO_COPY_BYTES;
  if (no_alloc) {
    if (R.end > GD_NOALLOC_SCRATCH_BYTES)
      return fail(ctx, GD_ERR_CAPACITY, "gd_calc_energy_noalloc: %zu scratch bytes needed, %d held",
                  R.end, GD_NOALLOC_SCRATCH_BYTES);
    base = ctx->scratch;
    HIPCHK(hipMemcpyAsync(base + o_packs, ps.packs.data(), ps.packs.size() * sizeof(Pack), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(base + o_slots, ps.slots.data(), ps.slots.size() * sizeof(int), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(base + o_lig, idx_lig, n * sizeof(int), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(base + o_mm, movematrix, (size_t)n * 6 * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
  } else {
    TRY(scratch_need(ctx, ctx->pin, R.end, true));
    memcpy(ctx->pin.p + o_packs, ps.packs.data(), ps.packs.size() * sizeof(Pack));
    memcpy(ctx->pin.p + o_slots, ps.slots.data(), ps.slots.size() * sizeof(int));
    memcpy(ctx->pin.p + o_lig, idx_lig, (size_t)n * sizeof(int));
    memcpy(ctx->pin.p + o_mm, movematrix, (size_t)n * 6 * sizeof(float));
    base = ctx->pin.p;
    if (!direct) {
      TRY(scratch_need(ctx, ctx->dev, R.end, false));
      base = ctx->dev.p;
      HIPCHK(hipMemcpyAsync(base, ctx->pin.p, o_out, hipMemcpyHostToDevice, ctx->stream));
    }
  }
  Pack *d_packs = reinterpret_cast<Pack *>(base + o_packs);
  int *d_slots = reinterpret_cast<int *>(base + o_slots);
  int *d_lig = reinterpret_cast<int *>(base + o_lig);
  float *d_mm = reinterpret_cast<float *>(base + o_mm);
  gd_energy *d_out = reinterpret_cast<gd_energy *>(base + o_out);
  float *d_sur = reinterpret_cast<float *>(base + o_out);
  P.cxs = ctx->d_cx;
  P.packs = d_packs;
  P.slots = d_slots;
  P.ev_mm = d_mm;
  P.ev_lig = d_lig;
  P.ev_out = d_out;
  P.ev_sur = d_sur;
  P.mode = sur ? MODE_SUREVAL : MODE_EVAL;
  P.ev_lpr = lpr;
  hipError_t le = launch_classes(ctx, ps.classes, P, sur ? da_instance(ctx, P.sur_tab != 0) : da_poses,
                                 sur && !P.sur_tab, ctx->stream);
  void *res = sur ? static_cast<void *>(out_sur) : static_cast<void *>(out);
  if (le == hipSuccess && no_alloc)
    le = hipMemcpyAsync(res, base + o_out, res_bytes, hipMemcpyDeviceToHost, ctx->stream);
  else if (le == hipSuccess && !direct)
    le = hipMemcpyAsync(ctx->pin.p + o_out, base + o_out, res_bytes, hipMemcpyDeviceToHost, ctx->stream);
  if (le == hipSuccess) le = hipStreamSynchronize(ctx->stream);
  if (le == hipSuccess && !no_alloc) memcpy(res, ctx->pin.p + o_out, res_bytes);
  if (le != hipSuccess) return fail(ctx, GD_ERR_HIP, "energy evaluation: %s", hipGetErrorString(le));
  return GD_OK;
}

}  // extern "C"

namespace {
template <class T>
gd_status tmp_dev(gd_ctx *ctx, std::vector<void *> &keep, T **p, const T *src, size_t n) {
  HIPCHK(hipMalloc((void **)p, std::max<size_t>(n, 1) * sizeof(T)));
  keep.push_back(*p);
  if (src && n) HIPCHK(hipMemcpyAsync(*p, src, n * sizeof(T), hipMemcpyHostToDevice, ctx->stream));
  return GD_OK;
}

void free_all(std::vector<void *> &keep) {
  for (void *p : keep) (void)hipFree(p);
  keep.clear();
}
}  // namespace

extern "C" {

gd_status gd_accept(gd_ctx *ctx, int n, const float *e_new, const float *e_old,
                    const float *minus_beta, const float *u, int32_t *accept) {
  if (!ctx || n < 0) return GD_ERR_INVALID;
  if (n == 0) return GD_OK;
  if (!e_new || !e_old || !minus_beta || !u || !accept) return GD_ERR_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  std::vector<void *> keep;
  float *a, *b, *c, *d;
  int *r;
  gd_status s = GD_OK;
  if ((s = tmp_dev(ctx, keep, &a, e_new, n)) || (s = tmp_dev(ctx, keep, &b, e_old, n)) ||
      (s = tmp_dev(ctx, keep, &c, minus_beta, n)) || (s = tmp_dev(ctx, keep, &d, u, n)) ||
      (s = tmp_dev<int>(ctx, keep, &r, nullptr, n))) {
    free_all(keep);
    return s;
  }
  hipLaunchKernelGGL(gd_accept_kernel, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n, a, b, c, d, r);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(accept, r, n * sizeof(int), hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  free_all(keep);
  if (e != hipSuccess) return fail(ctx, GD_ERR_HIP, "gd_accept: %s", hipGetErrorString(e));
  return GD_OK;
}

gd_status gd_exchange(gd_ctx *ctx, int n_groups, int n_tmp, int mode_t, const float *etot,
                      const float *minus_beta, const float *u, int32_t *idx_tmp, int32_t *acs) {
  if (!ctx || n_groups < 0 || n_tmp <= 0) return GD_ERR_INVALID;
  if (n_tmp > GD_MAX_NTMP) return fail(ctx, GD_ERR_CAPACITY, "n_tmp %d > %d", n_tmp, GD_MAX_NTMP);
  if (mode_t != 0 && mode_t != 1) return fail(ctx, GD_ERR_INVALID, "mode_t must be 0 or 1");
  if (n_groups == 0) return GD_OK;
  if (!etot || !minus_beta || !u || !idx_tmp || !acs) return GD_ERR_INVALID;
  const size_t ns = (size_t)n_groups * n_tmp;
  for (size_t i = 0; i < ns; ++i)
    if (idx_tmp[i] < 0 || idx_tmp[i] >= n_tmp)
      return fail(ctx, GD_ERR_INVALID, "idx_tmp[%zu] = %d outside [0,%d)", i, idx_tmp[i], n_tmp);
  HIPCHK(hipSetDevice(ctx->device));
  std::vector<void *> keep;
  float *de, *dm, *du;
  int *di, *da;
  gd_status s = GD_OK;
  const size_t nu = (size_t)n_groups * (n_tmp / 2);
  if ((s = tmp_dev(ctx, keep, &de, etot, ns)) || (s = tmp_dev(ctx, keep, &dm, minus_beta, (size_t)n_tmp)) ||
      (s = tmp_dev(ctx, keep, &du, u, nu)) || (s = tmp_dev<int>(ctx, keep, &di, idx_tmp, ns)) ||
      (s = tmp_dev<int>(ctx, keep, &da, acs, ns))) {
    free_all(keep);
    return s;
  }
  hipLaunchKernelGGL(gd_exchange_kernel, dim3((n_groups + 63) / 64), dim3(64), 0, ctx->stream,
                     n_groups, n_tmp, mode_t, de, dm, du, di, da);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(idx_tmp, di, ns * sizeof(int), hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(acs, da, ns * sizeof(int), hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  free_all(keep);
  if (e != hipSuccess) return fail(ctx, GD_ERR_HIP, "gd_exchange: %s", hipGetErrorString(e));
  return GD_OK;
}

gd_status gd_philox(gd_ctx *ctx, int n, const uint32_t *ctr, const uint32_t *key, uint32_t *out) {
  if (!ctx || n < 0) return GD_ERR_INVALID;
  if (n == 0) return GD_OK;
  if (!ctr || !key || !out) return GD_ERR_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  std::vector<void *> keep;
  uint32_t *dc, *dk, *dout;
  gd_status s = GD_OK;
  if ((s = tmp_dev(ctx, keep, &dc, ctr, (size_t)4 * n)) || (s = tmp_dev(ctx, keep, &dk, key, (size_t)2 * n)) ||
      (s = tmp_dev<uint32_t>(ctx, keep, &dout, nullptr, (size_t)4 * n))) {
    free_all(keep);
    return s;
  }
  hipLaunchKernelGGL(gd_philox_kernel, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n, dc, dk, dout);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(out, dout, (size_t)4 * n * sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  free_all(keep);
  if (e != hipSuccess) return fail(ctx, GD_ERR_HIP, "gd_philox: %s", hipGetErrorString(e));
  return GD_OK;
}

}  // extern "C"

// ===========================================================================
// Learned surrogate: feature grids, dataset, BF16 MFMA training, prediction.
// ===========================================================================
namespace {

gd_status sur_alloc_params(gd_ctx *ctx) {
  auto &S = ctx->sur;
  // each that is missing: an earlier call may have failed half-way
  auto need = [](auto **p, size_t n) {
    return *p ? hipSuccess : hipMalloc(p, n * sizeof(**p));
  };
  for (float **p : {&S.p, &S.m, &S.v, &S.grad}) HIPCHK(need(p, SUR_NPARAM));
  HIPCHK(need(&S.W1T, SUR_F * SUR_H));
  HIPCHK(need(&S.W2T, SUR_H * SUR_H));
  HIPCHK(need(&S.W2R, SUR_H * SUR_H));
  return GD_OK;
}

SurW sur_weights(gd_ctx *ctx) {
  auto &S = ctx->sur;
  SurW W;
  W.W1T = S.W1T;
  W.W2T = S.W2T;
  W.W2R = S.W2R;
  W.b2 = S.p + SP_B2;
  W.w3 = S.p + SP_W3;
  W.b3 = S.p + SP_B3;
  return W;
}

// refresh the bf16 layouts from the FP32 master (Adam with lr = 0)
gd_status sur_refresh(gd_ctx *ctx) {
  auto &S = ctx->sur;
  hipLaunchKernelGGL(gd_mlp_adam_kernel, dim3((SUR_NPARAM + 255) / 256), dim3(256), 0, ctx->stream,
                     S.p, S.m, S.v, S.grad, 0.0f, 0.f, 0.f, 0.f, 1.f, 1.f, S.W1T, S.W2T, S.W2R);
  HIPCHK(hipGetLastError());
  return GD_OK;
}

gd_status sur_upload_index(gd_ctx *ctx) {
  auto &S = ctx->sur;
  if (!S.dirty) return GD_OK;
  const int64_t np = (int64_t)S.target.size();
  if (S.d_off) (void)hipFree(S.d_off);
  if (S.d_target) (void)hipFree(S.d_target);
  S.d_off = nullptr;
  S.d_target = nullptr;
  HIPCHK(hipMalloc(&S.d_off, (np + 1) * sizeof(int64_t)));
  HIPCHK(hipMalloc(&S.d_target, std::max<int64_t>(np, 1) * sizeof(float)));
  // per-row outputs are indexed by absolute dataset row
  if (S.y) (void)hipFree(S.y);
  S.y = nullptr;
  HIPCHK(hipMalloc(&S.y, (S.cap + 64) * sizeof(float)));
  HIPCHK(hipMemcpyAsync(S.d_off, S.off.data(), (np + 1) * sizeof(int64_t), hipMemcpyHostToDevice, ctx->stream));
  if (np) HIPCHK(hipMemcpyAsync(S.d_target, S.target.data(), np * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  S.dirty = false;
  return GD_OK;
}

// Workgroups of the batch kernels: the fused backward runs one per CU (its
// LDS tiles take 124 KB), the forward three (its registers allow three waves
// per SIMD); each walks 64-row steps.
int sur_train_groups(const gd_ctx *ctx, int64_t rows) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(rows / 64, ctx->n_cu));
}
int sur_fwd_groups(const gd_ctx *ctx, int64_t rows) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(rows / 64, 3 * (int64_t)ctx->n_cu));
}

// work buffers for batches of up to `rows` rows (rounded up to 64): the
// gradient partials of the fused backward's workgroups and per-pose outputs
gd_status sur_work(gd_ctx *ctx, int64_t rows, int64_t n_pose_total) {
  auto &S = ctx->sur;
  rows = (rows + 63) / 64 * 64 + 64;
  if (rows > S.work_rows) {
    float **qs[] = {&S.p1, &S.p2, &S.pb2, &S.pw3, &S.dyr};
    S.work_rows = 0;
    for (float **q : qs) {
      if (*q) (void)hipFree(*q);
      *q = nullptr;
    }
    const int64_t ng = std::max(1, ctx->n_cu);
    HIPCHK(hipMalloc(&S.dyr, (size_t)rows * sizeof(float)));
    HIPCHK(hipMalloc(&S.p1, (size_t)ng * SUR_F * SUR_H * sizeof(float)));
    HIPCHK(hipMalloc(&S.p2, (size_t)ng * SUR_H * SUR_H * sizeof(float)));
    HIPCHK(hipMalloc(&S.pb2, (size_t)ng * SUR_H * sizeof(float)));
    HIPCHK(hipMalloc(&S.pw3, (size_t)ng * (SUR_H + 1) * sizeof(float)));
    HIPCHK(hipFuncSetAttribute((const void *)gd_mlp_train_kernel,
                               hipFuncAttributeMaxDynamicSharedMemorySize, SUR_TRAIN_LDS));
    S.work_rows = rows;
  }
  const int64_t np = std::max<int64_t>(n_pose_total, 1);
  if (np > S.work_poses) {
    float **qs[] = {&S.dS, &S.sq, &S.S};
    S.work_poses = 0;
    for (float **q : qs) {
      if (*q) (void)hipFree(*q);
      *q = nullptr;
      HIPCHK(hipMalloc(q, np * sizeof(float)));
    }
    S.work_poses = np;
  }
  return GD_OK;
}

// forward (+ backward and gradient when grad) over poses [p0, p1) of the dataset
// With `update`, the gradient partials are left for gd_mlp_update_kernel
// (the training step sums them and applies Adam in one launch).
gd_status sur_batch(gd_ctx *ctx, int64_t p0, int64_t p1, bool grad, double *loss,
                    bool update = false) {
  auto &S = ctx->sur;
  const int64_t r0 = S.off[p0], r1 = S.off[p1];
  const int64_t nr = (r1 - r0 + 63) / 64 * 64;  // padded rows read from the dataset
  const int np = (int)(p1 - p0);
  const SurW W = sur_weights(ctx);
  const unsigned short *X = S.X + r0 * SUR_F;
  hipLaunchKernelGGL(gd_mlp_fwd_kernel, dim3(sur_fwd_groups(ctx, nr)), dim3(256), 0, ctx->stream, X,
                     nr, W, S.y + r0);
  hipLaunchKernelGGL(gd_mlp_pose_kernel, dim3((np + 63) / 64), dim3(256), 0, ctx->stream, S.y,
                     S.d_off, (int)p0, (int)p1, S.d_target, S.dS, S.sq, S.S,
                     grad ? S.dyr : (float *)nullptr, nr);
  if (grad) {
    const int ng = sur_train_groups(ctx, nr);
    hipLaunchKernelGGL(gd_mlp_train_kernel, dim3(ng), dim3(512), SUR_TRAIN_LDS, ctx->stream, X,
                       nr, S.dyr, W, S.p1, S.p2, S.pb2, S.pw3);
    S.last_groups = ng;
    if (!update)
      hipLaunchKernelGGL(gd_mlp_gradsum_kernel, dim3((SUR_NPARAM + 31) / 32), dim3(256), 0,
                         ctx->stream, S.p1, S.p2, S.pb2, S.pw3, ng, S.grad);
  }
  HIPCHK(hipGetLastError());
  if (loss) {
    std::vector<float> sq(np);
    HIPCHK(hipMemcpyAsync(sq.data(), S.sq + p0, np * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    double s = 0.0;
    for (float v : sq) s += v;
    *loss = s / np;
  }
  return GD_OK;
}

}  // namespace

extern "C" {

int gd_sur_num_params(void) { return SUR_NPARAM; }

gd_status gd_sur_build_grids(gd_ctx *ctx, float spacing, float half_width) {
  if (!ctx || !(spacing > 0.0f) || !(half_width > spacing)) return GD_ERR_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  TRY(sync_complexes(ctx));
  auto &S = ctx->sur;
  const int n = (int)std::ceil(2.0f * half_width / spacing) + 1;
  const size_t nodes = (size_t)n * n * n;
  // no grids (S.g is what calls ask) until all of them are there and in the
  // complex table: a failure below leaves some replaced, some freed
  S.tab_valid = false;
  S.g.clear();
  for (HostComplex &h : ctx->cx) {
    h.dev.sgrid = nullptr;
    h.dev.stab = nullptr;
  }
  ctx->cx_dirty = true;
  // grids and tables of the sizes they had are kept, others replaced (the
  // number of complexes only grows)
  const size_t n_cx = ctx->cx.size();
  S.grid.resize(n_cx, nullptr);
  S.tab.resize(n_cx, nullptr);
  S.grid_n.resize(n_cx, 0);
  S.tab_n.resize(n_cx, 0);
  std::vector<SurGrid> grids(n_cx);
  for (size_t c = 0; c < n_cx; ++c) {
    const HostComplex &h = ctx->cx[c];
    const size_t need = (size_t)h.d.n_prt * nodes * 32;
    if (S.tab_n[c] != (size_t)h.d.n_prt * NLT * nodes) {
      if (S.tab[c]) (void)hipFree(S.tab[c]);
      S.tab[c] = nullptr;
      S.tab_n[c] = 0;
    }
    if (S.grid_n[c] != need) {
      if (S.grid[c]) (void)hipFree(S.grid[c]);
      S.grid[c] = nullptr;
      S.grid_n[c] = 0;
      HIPCHK(hipMalloc(&S.grid[c], need * sizeof(float)));
      S.grid_n[c] = need;
    }
    SurGrid G;
    G.grid = S.grid[c];
    G.ox = h.d.pocket_center[0] - half_width;
    G.oy = h.d.pocket_center[1] - half_width;
    G.oz = h.d.pocket_center[2] - half_width;
    G.h = spacing;
    G.n = n;
    grids[c] = G;
    ctx->cx[c].dev.sgrid = G.grid;
    ctx->cx[c].dev.sox = G.ox;
    ctx->cx[c].dev.soy = G.oy;
    ctx->cx[c].dev.soz = G.oz;
    ctx->cx[c].dev.sh = G.h;
    ctx->cx[c].dev.sn = G.n;
    const int64_t nb = (n + 3) / 4, bricks = nb * nb * nb;
    for (int p = 0; p < h.d.n_prt; p += GRID_ROWS) {
      hipLaunchKernelGGL(gd_sur_grid_kernel,
                         dim3((unsigned)((bricks + 3) / 4),
                              (unsigned)std::min(GRID_ROWS, h.d.n_prt - p)),
                         dim3(256), 0, ctx->stream, h.dev.prt_xyze + (size_t)p * h.d.pnp,
                         h.dev.prt_type, h.d.pnp, G.ox, G.oy, G.oz, G.h, n,
                         S.grid[c] + (size_t)p * nodes * 32);
      HIPCHK(hipGetLastError());
    }
  }
  HIPCHK(hipStreamSynchronize(ctx->stream));
  TRY(sync_complexes(ctx));
  S.g = std::move(grids);
  return GD_OK;
}

// Pose arrays of a call on the device: one staged copy. `cid` and `row` may be
// null; `extra_bytes` of device scratch follow them.
struct PoseInputs {
  int *cid = nullptr, *lig = nullptr, *prt = nullptr;
  float *mm = nullptr;
  int64_t *row = nullptr;
  unsigned char *extra = nullptr;
};

static gd_status stage_poses(gd_ctx *ctx, int n, const int *cid, const int *idx_lig,
                             const int *idx_prt, const float *movematrix, const int64_t *row,
                             size_t extra_bytes, PoseInputs &in) {
  Regions R;
  const size_t o_row = R.add(row ? (size_t)n * sizeof(int64_t) : 0);
  const size_t o_cid = R.add(cid ? (size_t)n * sizeof(int) : 0);
  const size_t o_lig = R.add((size_t)n * sizeof(int));
  const size_t o_prt = R.add((size_t)n * sizeof(int));
  const size_t o_mm = R.add((size_t)n * 6 * sizeof(float));
  const size_t o_extra = R.end;
  TRY(scratch_need(ctx, ctx->pin, o_extra, true));
  TRY(scratch_need(ctx, ctx->dev, o_extra + extra_bytes, false));
  unsigned char *p = ctx->pin.p, *d = ctx->dev.p;
  if (row) memcpy(p + o_row, row, (size_t)n * sizeof(int64_t));
  if (cid) memcpy(p + o_cid, cid, (size_t)n * sizeof(int));
  memcpy(p + o_lig, idx_lig, (size_t)n * sizeof(int));
  memcpy(p + o_prt, idx_prt, (size_t)n * sizeof(int));
  memcpy(p + o_mm, movematrix, (size_t)n * 6 * sizeof(float));
  HIPCHK(hipMemcpyAsync(d, p, o_extra, hipMemcpyHostToDevice, ctx->stream));
  in.row = reinterpret_cast<int64_t *>(d + o_row);
  in.cid = reinterpret_cast<int *>(d + o_cid);
  in.lig = reinterpret_cast<int *>(d + o_lig);
  in.prt = reinterpret_cast<int *>(d + o_prt);
  in.mm = reinterpret_cast<float *>(d + o_mm);
  in.extra = d + o_extra;
  return GD_OK;
}

gd_status gd_sur_features(gd_ctx *ctx, int cid, int n, const int *idx_lig, const int *idx_prt,
                          const float *movematrix, float *out) {
  if (!ctx || cid < 0 || cid >= (int)ctx->cx.size() || n < 0) return GD_ERR_INVALID;
  if ((int)ctx->sur.g.size() <= cid) return fail(ctx, GD_ERR_STATE, "call gd_sur_build_grids first");
  if (n == 0) return GD_OK;
  const HostComplex &h = ctx->cx[cid];
  for (int i = 0; i < n; ++i)
    if (idx_lig[i] < 0 || idx_lig[i] >= h.d.n_lig || idx_prt[i] < 0 || idx_prt[i] >= h.d.n_prt)
      return fail(ctx, GD_ERR_INVALID, "pose %d: conformer index out of range", i);
  HIPCHK(hipSetDevice(ctx->device));
  const size_t rows = (size_t)n * h.d.lna;
  const ScratchTrim trim{ctx};
  PoseInputs in;
  TRY(stage_poses(ctx, n, nullptr, idx_lig, idx_prt, movematrix, nullptr,
                  rows * SUR_NF * sizeof(float), in));
  float *dout = reinterpret_cast<float *>(in.extra);
  hipLaunchKernelGGL(gd_sur_feat_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0,
                     ctx->stream, ctx->d_cx, cid, ctx->sur.g[cid], n, in.lig, in.prt, in.mm,
                     (int64_t)0, (unsigned short *)nullptr, dout);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(out, dout, rows * SUR_NF * sizeof(float), hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  if (e != hipSuccess) return fail(ctx, GD_ERR_HIP, "gd_sur_features: %s", hipGetErrorString(e));
  return GD_OK;
}

gd_status gd_sur_set_params(gd_ctx *ctx, const float *params) {
  if (!ctx || !params) return GD_ERR_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  TRY(sur_alloc_params(ctx));
  auto &S = ctx->sur;
  HIPCHK(hipMemcpyAsync(S.p, params, SUR_NPARAM * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
  HIPCHK(hipMemsetAsync(S.m, 0, SUR_NPARAM * sizeof(float), ctx->stream));
  HIPCHK(hipMemsetAsync(S.v, 0, SUR_NPARAM * sizeof(float), ctx->stream));
  S.adam_t = 0;
  S.tab_valid = false;
  TRY(sur_refresh(ctx));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  S.have_params = true;
  return GD_OK;
}

gd_status gd_sur_tabulate(gd_ctx *ctx) {
  if (!ctx) return GD_ERR_INVALID;
  auto &S = ctx->sur;
  if (S.g.size() != ctx->cx.size()) return fail(ctx, GD_ERR_STATE, "call gd_sur_build_grids first");
  if (!S.have_params) return fail(ctx, GD_ERR_STATE, "no surrogate parameters");
  HIPCHK(hipSetDevice(ctx->device));
  SurW W{S.W1T, S.W2T, S.W2R, S.p + SP_B2, S.p + SP_W3, S.p + SP_B3};
  const size_t n_cx = ctx->cx.size();
  // only the ligands' atom types are evaluated: NLT slots per complex
  std::vector<int> types(n_cx * NLT, 0), n_types(n_cx, 0);
  for (size_t c = 0; c < n_cx; ++c) {
    const HostComplex &h = ctx->cx[c];
    for (int t = 0; t < NLT; ++t)
      if (std::find(h.lig_t.begin(), h.lig_t.end(), t) != h.lig_t.end())
        types[c * NLT + n_types[c]++] = t;
    if (S.tab[c]) continue;
    const size_t need = (size_t)h.d.n_prt * NLT * S.g[c].n * S.g[c].n * S.g[c].n;
    if (hipMalloc(&S.tab[c], need * sizeof(float)) != hipSuccess) {
      S.tab[c] = nullptr;
      return fail(ctx, GD_ERR_NOMEM, "surrogate table of complex %zu", c);
    }
    S.tab_n[c] = need;
  }
  int *d_types = nullptr;
  HIPCHK(hipMalloc(&d_types, std::max<size_t>(types.size(), 1) * sizeof(int)));
  hipError_t e = hipMemcpyAsync(d_types, types.data(), types.size() * sizeof(int),
                                hipMemcpyHostToDevice, ctx->stream);
  for (size_t c = 0; c < n_cx && e == hipSuccess; ++c) {
    HostComplex &h = ctx->cx[c];
    const int n = S.g[c].n;
    const size_t n3 = (size_t)n * n * n;
    // two workgroups of four waves per CU, which walk the tiles of 16 points
    const int64_t tiles = (int64_t)((n3 + 15) / 16) * h.d.n_prt;
    const int64_t grid = std::min<int64_t>((tiles + 3) / 4, 2 * (int64_t)ctx->n_cu);
    hipLaunchKernelGGL(gd_sur_tab_kernel, dim3((unsigned)grid), dim3(256), 0, ctx->stream,
                       S.grid[c], (int)n3, h.d.n_prt, d_types + c * NLT, n_types[c], W, S.tab[c]);
    e = hipGetLastError();
    h.dev.stab = S.tab[c];
    ctx->cx_dirty = true;
  }
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  (void)hipFree(d_types);
  if (e != hipSuccess) return fail(ctx, GD_ERR_HIP, "tabulation: %s", hipGetErrorString(e));
  TRY(sync_complexes(ctx));
  S.tab_valid = true;
  return GD_OK;
}

gd_status gd_sur_get_params(gd_ctx *ctx, float *params) {
  if (!ctx || !params) return GD_ERR_INVALID;
  if (!ctx->sur.have_params) return fail(ctx, GD_ERR_STATE, "no surrogate parameters");
  HIPCHK(hipSetDevice(ctx->device));
  HIPCHK(hipMemcpyAsync(params, ctx->sur.p, SUR_NPARAM * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return GD_OK;
}

gd_status gd_sur_dataset_clear(gd_ctx *ctx) {
  if (!ctx) return GD_ERR_INVALID;
  auto &S = ctx->sur;
  S.rows = 0;
  S.off.assign(1, 0);
  S.target.clear();
  S.pose_cx.clear();
  S.dirty = true;
  return GD_OK;
}

gd_status gd_sur_dataset_reserve(gd_ctx *ctx, int64_t rows) {
  if (!ctx || rows < 0) return GD_ERR_INVALID;
  auto &S = ctx->sur;
  if (rows <= S.cap) return GD_OK;
  HIPCHK(hipSetDevice(ctx->device));
  unsigned short *X = nullptr;
  const int64_t cap = (rows + 63) / 64 * 64;
  HIPCHK(hipMalloc(&X, (size_t)(cap + 64) * SUR_F * 2));
  HIPCHK(hipMemsetAsync(X, 0, (size_t)(cap + 64) * SUR_F * 2, ctx->stream));
  if (S.rows > 0)
    HIPCHK(hipMemcpyAsync(X, S.X, (size_t)S.rows * SUR_F * 2, hipMemcpyDeviceToDevice, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  if (S.X) (void)hipFree(S.X);
  S.X = X;
  S.cap = cap;
  S.dirty = true;
  return GD_OK;
}

gd_status gd_sur_dataset_add(gd_ctx *ctx, int cid, int n, const int *idx_lig, const int *idx_prt,
                             const float *movematrix, const float *target) {
  if (!ctx || cid < 0 || cid >= (int)ctx->cx.size() || n < 0) return GD_ERR_INVALID;
  if ((int)ctx->sur.g.size() <= cid) return fail(ctx, GD_ERR_STATE, "call gd_sur_build_grids first");
  if (n == 0) return GD_OK;
  if (!idx_lig || !idx_prt || !movematrix || !target) return GD_ERR_INVALID;
  const HostComplex &h = ctx->cx[cid];
  for (int i = 0; i < n; ++i)
    if (idx_lig[i] < 0 || idx_lig[i] >= h.d.n_lig || idx_prt[i] < 0 || idx_prt[i] >= h.d.n_prt)
      return fail(ctx, GD_ERR_INVALID, "pose %d: conformer index out of range", i);
  auto &S = ctx->sur;
  const int64_t add = (int64_t)n * h.d.lna;
  if (S.rows + add > S.cap) TRY(gd_sur_dataset_reserve(ctx, std::max<int64_t>(S.rows + add, 2 * S.cap)));
  HIPCHK(hipSetDevice(ctx->device));
  const ScratchTrim trim{ctx};
  PoseInputs in;
  TRY(stage_poses(ctx, n, nullptr, idx_lig, idx_prt, movematrix, nullptr, 0, in));
  hipLaunchKernelGGL(gd_sur_feat_kernel, dim3((unsigned)((add + 255) / 256)), dim3(256), 0,
                     ctx->stream, ctx->d_cx, cid, S.g[cid], n, in.lig, in.prt, in.mm, S.rows, S.X,
                     (float *)nullptr);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  if (e != hipSuccess) return fail(ctx, GD_ERR_HIP, "gd_sur_dataset_add: %s", hipGetErrorString(e));
  for (int i = 0; i < n; ++i) {
    S.off.push_back(S.off.back() + h.d.lna);
    S.target.push_back(target[i]);
    S.pose_cx.push_back(cid);
  }
  S.rows += add;
  S.dirty = true;
  return GD_OK;
}

gd_status gd_sur_dataset_add_multi(gd_ctx *ctx, int n, const int *cid, const int *idx_lig,
                                   const int *idx_prt, const float *movematrix,
                                   const float *target) {
  if (!ctx || n < 0) return GD_ERR_INVALID;
  if (n == 0) return GD_OK;
  if (!cid || !idx_lig || !idx_prt || !movematrix || !target) return GD_ERR_INVALID;
  auto &S = ctx->sur;
  if (S.g.size() != ctx->cx.size()) return fail(ctx, GD_ERR_STATE, "call gd_sur_build_grids first");
  std::vector<int64_t> row_of(n);
  int64_t add = 0;
  for (int i = 0; i < n; ++i) {
    if (cid[i] < 0 || cid[i] >= (int)ctx->cx.size())
      return fail(ctx, GD_ERR_INVALID, "pose %d: complex id out of range", i);
    const HostComplex &h = ctx->cx[cid[i]];
    if (idx_lig[i] < 0 || idx_lig[i] >= h.d.n_lig || idx_prt[i] < 0 || idx_prt[i] >= h.d.n_prt)
      return fail(ctx, GD_ERR_INVALID, "pose %d: conformer index out of range", i);
    row_of[i] = S.rows + add;
    add += h.d.lna;
  }
  if (S.rows + add > S.cap) TRY(gd_sur_dataset_reserve(ctx, std::max<int64_t>(S.rows + add, 2 * S.cap)));
  HIPCHK(hipSetDevice(ctx->device));
  TRY(sync_complexes(ctx));
  const ScratchTrim trim{ctx};
  PoseInputs in;
  TRY(stage_poses(ctx, n, cid, idx_lig, idx_prt, movematrix, row_of.data(), 0, in));
  hipLaunchKernelGGL(gd_sur_feat_multi_kernel, dim3((unsigned)n), dim3(64), 0, ctx->stream,
                     ctx->d_cx, n, in.cid, in.lig, in.prt, in.mm, in.row, S.X);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  if (e != hipSuccess) return fail(ctx, GD_ERR_HIP, "gd_sur_dataset_add_multi: %s", hipGetErrorString(e));
  for (int i = 0; i < n; ++i) {
    S.off.push_back(S.off.back() + ctx->cx[cid[i]].d.lna);
    S.target.push_back(target[i]);
    S.pose_cx.push_back(cid[i]);
  }
  S.rows += add;
  S.dirty = true;
  return GD_OK;
}

int64_t gd_sur_dataset_size(const gd_ctx *ctx) { return ctx ? (int64_t)ctx->sur.target.size() : -1; }

gd_status gd_sur_loss_grad(gd_ctx *ctx, int pose_begin, int pose_end, double *loss, float *grad) {
  if (!ctx) return GD_ERR_INVALID;
  auto &S = ctx->sur;
  if (!S.have_params) return fail(ctx, GD_ERR_STATE, "no surrogate parameters");
  if (pose_begin < 0 || pose_end > (int)S.target.size() || pose_begin >= pose_end)
    return fail(ctx, GD_ERR_INVALID, "pose range [%d,%d) outside the dataset", pose_begin, pose_end);
  HIPCHK(hipSetDevice(ctx->device));
  TRY(sur_upload_index(ctx));
  TRY(sur_work(ctx, S.off[pose_end] - S.off[pose_begin], (int64_t)S.target.size()));
  TRY(sur_batch(ctx, pose_begin, pose_end, grad != nullptr, loss));
  if (grad) {
    HIPCHK(hipMemcpyAsync(grad, S.grad, SUR_NPARAM * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
  }
  return GD_OK;
}

gd_status gd_sur_predict(gd_ctx *ctx, int pose_begin, int pose_end, float *out) {
  if (!ctx || !out) return GD_ERR_INVALID;
  auto &S = ctx->sur;
  if (!S.have_params) return fail(ctx, GD_ERR_STATE, "no surrogate parameters");
  if (pose_begin < 0 || pose_end > (int)S.target.size() || pose_begin >= pose_end)
    return fail(ctx, GD_ERR_INVALID, "pose range outside the dataset");
  HIPCHK(hipSetDevice(ctx->device));
  TRY(sur_upload_index(ctx));
  TRY(sur_work(ctx, S.off[pose_end] - S.off[pose_begin], (int64_t)S.target.size()));
  // in chunks that bound the work buffers
  const int step = 65536;
  for (int p = pose_begin; p < pose_end; p += step)
    TRY(sur_batch(ctx, p, std::min(pose_end, p + step), false, nullptr));
  HIPCHK(hipMemcpyAsync(out, S.S + pose_begin, (size_t)(pose_end - pose_begin) * sizeof(float),
                        hipMemcpyDeviceToHost, ctx->stream));
  HIPCHK(hipStreamSynchronize(ctx->stream));
  return GD_OK;
}

gd_status gd_sur_train(gd_ctx *ctx, int pose_begin, int pose_end, int epochs, int batch_poses,
                       float lr, double *epoch_loss, double *seconds) {
  if (!ctx || epochs < 0 || batch_poses <= 0 || !(lr > 0.0f)) return GD_ERR_INVALID;
  auto &S = ctx->sur;
  if (!S.have_params) return fail(ctx, GD_ERR_STATE, "no surrogate parameters");
  if (pose_begin < 0 || pose_end > (int)S.target.size() || pose_begin >= pose_end)
    return fail(ctx, GD_ERR_INVALID, "pose range outside the dataset");
  HIPCHK(hipSetDevice(ctx->device));
  TRY(sur_upload_index(ctx));
  int64_t maxrows = 0;
  for (int p = pose_begin; p < pose_end; p += batch_poses) {
    const int q = std::min(pose_end, p + batch_poses);
    maxrows = std::max<int64_t>(maxrows, S.off[q] - S.off[p]);
  }
  TRY(sur_work(ctx, maxrows, (int64_t)S.target.size()));
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const int n_batch = (pose_end - pose_begin + batch_poses - 1) / batch_poses;
  // per-batch sums of squared residuals (before each batch's update)
  if (n_batch > S.work_batches) {
    if (S.bl) (void)hipFree(S.bl);
    S.bl = nullptr;
    S.work_batches = 0;
    HIPCHK(hipMalloc(&S.bl, (size_t)n_batch * sizeof(float)));
    S.work_batches = n_batch;
  }
  float *d_bl = S.bl;
  std::vector<float> bl(n_batch);
  const auto t0 = std::chrono::steady_clock::now();
  S.tab_valid = false;  // the parameters change
  gd_status st = GD_OK;
  for (int ep = 0; ep < epochs && st == GD_OK; ++ep) {
    int b = 0;
    for (int p = pose_begin; p < pose_end && st == GD_OK; p += batch_poses, ++b) {
      const int q = std::min(pose_end, p + batch_poses);
      st = sur_batch(ctx, p, q, true, nullptr, true);
      if (st != GD_OK) break;
      S.adam_t += 1;
      const float c1 = 1.0f - std::pow(b1, (float)S.adam_t);
      const float c2 = 1.0f - std::pow(b2, (float)S.adam_t);
      hipLaunchKernelGGL(gd_mlp_update_kernel, dim3((SUR_NPARAM + 31) / 32 + 1), dim3(256), 0,
                         ctx->stream, S.p1, S.p2, S.pb2, S.pw3, S.last_groups, S.p, S.m, S.v,
                         S.grad, lr, b1, b2, eps, c1, c2, S.W1T, S.W2T, S.W2R, S.sq + p, q - p,
                         d_bl + b);
      if (hipGetLastError() != hipSuccess) st = fail(ctx, GD_ERR_HIP, "training launch failed");
    }
    if (st != GD_OK || !epoch_loss) continue;
    if (ep + 1 < epochs) {
      // the epoch's batch losses, each taken before its batch's update
      if (hipMemcpyAsync(bl.data(), d_bl, (size_t)n_batch * sizeof(float),
                         hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
          hipStreamSynchronize(ctx->stream) != hipSuccess) {
        st = fail(ctx, GD_ERR_HIP, "batch loss copy failed");
        break;
      }
      double tot = 0.0;
      for (float v : bl) tot += v;
      epoch_loss[ep] = tot / (double)(pose_end - pose_begin);
    } else {
      // last epoch: the loss over the whole range with the final parameters
      // (every batch's residuals in one copy)
      double tot = 0.0;
      for (int p = pose_begin; p < pose_end && st == GD_OK; p += batch_poses)
        st = sur_batch(ctx, p, std::min(pose_end, p + batch_poses), false, nullptr);
      if (st != GD_OK) break;
      std::vector<float> sq(pose_end - pose_begin);
      if (hipMemcpyAsync(sq.data(), S.sq + pose_begin, sq.size() * sizeof(float),
                         hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
          hipStreamSynchronize(ctx->stream) != hipSuccess) {
        st = fail(ctx, GD_ERR_HIP, "residual copy failed");
        break;
      }
      for (int p = pose_begin; p < pose_end; p += batch_poses) {
        const int q = std::min(pose_end, p + batch_poses);
        double l = 0.0;
        for (int i = p; i < q; ++i) l += sq[i - pose_begin];
        tot += l / (q - p) * (q - p);
      }
      epoch_loss[ep] = tot / (double)(pose_end - pose_begin);
    }
  }
  (void)hipStreamSynchronize(ctx->stream);
  TRY(st);
  HIPCHK(hipStreamSynchronize(ctx->stream));
  if (seconds) *seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return GD_OK;
}

}  // extern "C"

#include "gd_post.hip"
