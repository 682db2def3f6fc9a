// Batched parallel-beam CGLS: many independent problems of uneven sizes
// advanced together.
//
// No counterpart in the reference (it reconstructs one problem per call;
// the iteration body is cgls_3d, Core/src/Algorithms/cgls.cpp:26-157).
// Every step of an iteration is ONE launch over a flat work list that spans
// all problems:
//   FP    items (problem, 64 rays of an angle, 4*lr-row block) -> Ad, partial ||Ad||^2
//   alpha one workgroup per problem: fixed-order sum of its partials
//   x/r   items (problem, element chunk)               -> x += a d, r -= a Ad
//   BP    items (problem, 16x16-column tile or 256-column block, slice
//         block)                                    -> s, partial ||s||^2
//   beta  one workgroup per problem
//   d     items (problem, element chunk)               -> d = s + b d
// The six launches are captured once in a hipGraph and replayed per
// iteration; scalars (gamma, alpha, beta, iteration index) live in the
// problem descriptors in device memory, so a replay needs no host work.
// The norms of the projector outputs are produced by the projector
// epilogues (per work item, deterministic), so no separate reduction pass
// re-reads Ad or s.  The BP's rows per lane and grid (one workgroup per
// item, or a persistent grid of 2 / 4 / 8 workgroups per CU dealing the items
// out by a fixed stride) are picked by timing candidates on the batch itself
// (tune_batch, cached per batch shape), and so is the grid of the FP items that
// the shared walk does not take.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <memory>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "batch_tune.hpp"
#include "par_body.hpp"
#include "plan.hpp"
#include "solvers.hpp"

namespace ccpi {

struct BatchProb {
  ParArgs g;
  float *r, *x, *d, *s, *Ad;
  double *norms;       // [iters]
  long long nvox, npix;
  int fp_nbx, fp_nby, bp_nbx, bp_nby;
  double gamma;
  float alpha, beta;
  int it;
  int fp_lr;           // FP lanes per ray
  int fp_part, fp_parts;   // its norm partials: first and count
  int bp_tiled;        // BP items are 16 x 16 column tiles staged in LDS
  int bp_hmax, bp_ab;  // their staged detector columns per angle, angles per block
  int bp_groups;       // angle groups of the problem's one-problem tiled BP
};

struct BatchLists {
  int count;
  const int *fs_off;   // [count + 1] item prefix per kernel type: shared-walk FP
  const int *fp_off;   // other FP
  const int *bp_off;
  const int *vx_off;   // volume chunks
  const int *px_off;   // sinogram chunks
  double *part_fp;     // one per live shared-walk item, 4 per other FP item
  double *part_bp;     // [4 * bp items]
};

constexpr int kChunk = 2048;  // elements per vector work item

__device__ inline int find_prob(const int *off, int count, int item) {
  int lo = 0, hi = count;  // last p with off[p] <= item
  while (hi - lo > 1) {
    const int m = (lo + hi) >> 1;
    if (off[m] <= item) lo = m; else hi = m;
  }
  return lo;
}

__device__ inline double wave_sum_d(double v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// FP of d into Ad for every problem whose rows and slices go one to one: one
// workgroup per item, 64 rays of an angle walked by its first wavefront for
// the other four (par_fp_shared), up to 8 lanes of 4 rows per ray.  Item
// counts are multiples of 8 per problem, so an item's XCD is its place in its
// problem's tiles (par_share_item).  With every lane walking on its own (the
// form that batch_proj_kernel keeps for the other problems) an iteration of
// the 64-problem mix took 27.8 ms, now 20.2 (7 waves per SIMD; 20.7 at 6).
constexpr int kBatchShareThreads = 64 * 5, kBatchShareLanes = 8;

__global__ __launch_bounds__(kBatchShareThreads)
__attribute__((amdgpu_waves_per_eu(kParShareWavesPerSimd, 8))) void batch_fp_shared_kernel(
    const BatchProb *__restrict__ P, BatchLists L) {
  __shared__ ParShare sh;
  const int id = wg_index();
  if (id >= L.fs_off[L.count]) return;
  const int p = find_prob(L.fs_off, L.count, id);
  const BatchProb &B = P[p];
  const ParArgs g = B.g;
  const int lr = B.fp_lr;
  const ParShareItem it = par_share_item(g, lr, id - L.fs_off[p]);
  if (!it.live) return;
  const float *d = B.d;
  float *Ad = B.Ad;
  const int ns = lr == kBatchShareLanes ? 2 : 1;
  double ss;
  if (g.nz >= 4)
    ss = ns == 2 ? par_fp_shared<2, true, float>(g, it.a, it.h0, it.v0, lr, d, Ad, false, sh)
                 : par_fp_shared<1, true, float>(g, it.a, it.h0, it.v0, lr, d, Ad, false, sh);
  else
    ss = ns == 2 ? par_fp_shared<2, false, float>(g, it.a, it.h0, it.v0, lr, d, Ad, false, sh)
                 : par_fp_shared<1, false, float>(g, it.a, it.h0, it.v0, lr, d, Ad, false, sh);
  block_part(ss, L.part_fp, B.fp_part + it.index);
}

// FP of d into Ad for the problems that the shared walk does not take (mode
// 0), or, for every problem, BP of r into s (mode 1) or into d (mode 2,
// initial direction).  FP work is taken per
// wavefront: a wave takes a block item (256 rays' lanes) and runs its four
// 64-lane quarters in turn, so no wave waits at a barrier for the longest
// walk of its workgroup.  BP work is taken per workgroup: a 16 x 16 column
// tile whose detector rows the workgroup stages in LDS (par_bp_tile, the
// one-problem path's tiled body, with its angle groups folded in registers
// so the sums are those of the one-problem launch) or, for problems the
// tiled form does not take, 256 columns of the column-per-lane body.  Every
// quarter (FP) or wave (BP) of an item leaves one FP64 partial norm.
// BPK: the BP bodies a batch needs (1 tiled, 2 column-per-lane, 3 both);
// a kernel holding both bodies is sized for the larger of their register
// sets, so a batch of one kind gets the kernel of that body alone.
// Waves per SIMD the registers must allow.  The FP items wait on their
// gathers: 6 waves took the 64-problem mix from 23.7 to 24.2 CGLS iterations
// a second.  The tiled BP items: an iteration of the mix takes 17.4 / 17.7 /
// 18.2 ms with them at 6 / 5 / 4 waves, one of 8 problems up to 300 columns
// 0.60 / 0.62 / 0.61.
template <int MODE, int BPK>
constexpr int batch_min_waves() { return MODE == 0 || BPK == 1 ? 6 : 1; }

template <int RC, int MODE, int BPK>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(batch_min_waves<MODE, BPK>(), 8))) void batch_proj_kernel(
    BatchProb *__restrict__ P, BatchLists L) {
  const int *off = MODE == 0 ? L.fp_off : L.bp_off;
  double *part = MODE == 0 ? L.part_fp : L.part_bp;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (MODE == 0) {
    // a wavefront takes the four 64-thread quarters of a block item one
    // after another: one problem lookup (a binary search and the
    // descriptor's scalar loads) per 256 threads' worth of rays
    const int total = off[L.count];
    const int wid = blockIdx.x * 4 + wave;
    for (int item = wid; item < total; item += 4 * gridDim.x) {
      const int p = find_prob(off, L.count, item);
      const BatchProb &B = P[p];
      // the problem's geometry as a local value (scalar registers), as the
      // one-problem kernels get it through their arguments
      const ParArgs g = B.g;
      const int local = item - off[p];
      for (int qtr = 0; qtr < 4; ++qtr) {
        double ss = par_fp_lanes(g, local % B.fp_nbx, local / B.fp_nbx, qtr * 64 + lane,
                                 B.fp_lr, B.d, B.Ad, false);
        ss = wave_sum_d(ss);
        if (lane == 0) part[B.fp_part + 4 * local + qtr] = ss;
      }
    }
    return;
  }
  extern __shared__ __align__(16) float smem[];
  const int total = off[L.count];
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const int p = find_prob(off, L.count, item);
    const BatchProb &B = P[p];
    const ParArgs g = B.g;
    const int local = item - off[p];
    const float *r = B.r;
    float *dst = MODE == 1 ? B.s : B.d;
    double ss;
    if (BPK == 1 || (BPK == 3 && B.bp_tiled)) {
      ss = par_bp_tile<RC, float, true>(g, local % B.bp_nbx, local / B.bp_nbx, 0, g.na,
                                        B.bp_hmax, B.bp_ab, false, r, dst, smem, true,
                                        B.bp_groups);
    } else {
      ss = par_bp_thread<RC>(g, local % B.bp_nbx, local / B.bp_nbx, threadIdx.x, r, dst,
                             false);
    }
    ss = wave_sum_d(ss);
    if (lane == 0) part[4 * item + wave] = ss;
    __syncthreads();   // the next item's first block overwrites this one's LDS
  }
}

// Per-problem scalars.  STEP 0: gamma = ||d||^2 (start), 1: alpha,
// 2: beta / gamma update / norm record.
template <int STEP>
__global__ __launch_bounds__(256) void batch_scalar_kernel(BatchProb *__restrict__ P,
                                                           BatchLists L) {
  const int p = blockIdx.x;
  const double *part = STEP == 1 ? L.part_fp : L.part_bp;
  const int q0 = STEP == 1 ? P[p].fp_part : 4 * L.bp_off[p];
  const int q1 = STEP == 1 ? q0 + P[p].fp_parts : 4 * L.bp_off[p + 1];
  __shared__ double sh[256];
  double s = 0.0;
  for (int q = q0 + threadIdx.x; q < q1; q += 256) s += part[q];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    BatchProb &B = P[p];
    const double t = sh[0];
    if (STEP == 0) {
      B.gamma = t;
      B.it = 0;
    } else if (STEP == 1) {
      B.alpha = t > 0.0 ? (float)(B.gamma / t) : 0.f;  // zero direction: stop
    } else {
      B.beta = B.gamma > 0.0 ? (float)(t / B.gamma) : 0.f;
      B.gamma = t;
      B.norms[B.it] = sqrt(t);
      B.it = B.it + 1;
    }
  }
}

// x += alpha d, r -= alpha Ad (MODE 0); d = s + beta d (MODE 1)
template <int MODE>
__global__ __launch_bounds__(256) void batch_vec_kernel(BatchProb *__restrict__ P,
                                                        BatchLists L) {
  const int tv = L.vx_off[L.count];
  const int total = MODE == 0 ? tv + L.px_off[L.count] : tv;
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const bool vox = item < tv;
    const int it2 = vox ? item : item - tv;
    const int *off = vox ? L.vx_off : L.px_off;
    const int p = find_prob(off, L.count, it2);
    const BatchProb &B = P[p];
    const long long n = vox ? B.nvox : B.npix;
    const long long q0 = (long long)(it2 - off[p]) * kChunk;
    const long long q1 = q0 + kChunk < n ? q0 + kChunk : n;
    if (MODE == 0) {
      const float a = B.alpha;
      if (vox)
        for (long long q = q0 + threadIdx.x; q < q1; q += 256) B.x[q] = B.x[q] + a * B.d[q];
      else
        for (long long q = q0 + threadIdx.x; q < q1; q += 256) B.r[q] = B.r[q] + (-a) * B.Ad[q];
    } else {
      const float b = B.beta;
      for (long long q = q0 + threadIdx.x; q < q1; q += 256) B.d[q] = b * B.d[q] + B.s[q];
    }
  }
}

// ---------------------------------------------------------------------------

namespace {

std::mutex g_tune_mu;
std::map<std::string, Tuned> g_tuned;

int cu_count();

// A persistent grid is capped at the workgroups that are resident at once:
// the work items are dealt out by a fixed stride, so a workgroup that only
// starts when another one ends would run its share at the tail.
template <class K>
int blocks_per_cu(K kernel, size_t lds) {
  int per_cu = 0;
  CCPI_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 256, lds));
  return std::max(per_cu, 1);
}

// grid: Tuned's fp_grid / bp_grid; items: the launch's work items (FP
// block items, four wavefront items each, or BP items); lds: dynamic LDS of
// the BP launches (the tiled items' staged rows)
template <int RC, int MODE, int BPK>
void launch_one(int grid, int items, size_t lds, BatchProb *P, const BatchLists &L,
                hipStream_t st) {
  const size_t l = MODE == 0 ? 0 : lds;
  int g;
  if (grid > 0) {
    const int per_cu = blocks_per_cu(batch_proj_kernel<RC, MODE, BPK>, l);
    g = std::min(grid, per_cu * cu_count());
  } else {
    g = MODE == 0 ? (items + 3) / 4 : items;
  }
  g = std::max(1, g);
  hipLaunchKernelGGL((batch_proj_kernel<RC, MODE, BPK>), dim3(g), dim3(256), l, st, P, L);
}

template <int RC, int MODE>
void launch_bp(int bpk, int grid, int items, size_t lds, BatchProb *P, const BatchLists &L,
               hipStream_t st) {
  if (bpk == 1)
    launch_one<RC, MODE, 1>(grid, items, lds, P, L, st);
  else if (bpk == 2)
    launch_one<RC, MODE, 2>(grid, items, lds, P, L, st);
  else
    launch_one<RC, MODE, 3>(grid, items, lds, P, L, st);
}

template <int RC>
void launch_bp_mode(int mode, int bpk, int grid, int items, size_t lds, BatchProb *P,
                    const BatchLists &L, hipStream_t st) {
  if (mode == 1)
    launch_bp<RC, 1>(bpk, grid, items, lds, P, L, st);
  else
    launch_bp<RC, 2>(bpk, grid, items, lds, P, L, st);
}

struct BatchRun;
// One projector step of every problem (mode 0 FP, 1 BP, 2 initial BP)
// with the launch shape T.
void proj(const BatchRun &R, const Tuned &T, int mode, hipStream_t st);

struct BatchRun {
  Workspace &W;
  ParBatchPlan plan;
  std::vector<BatchProb> host;
  BatchLists L{};
  int count = 0;
  int fs_total = 0, fp_total = 0, bp_total = 0;
  size_t bp_lds = 0;   // dynamic LDS of the BP launches
  int bp_kinds = 0;    // BP bodies of the problems: 1 tiled, 2 column-per-lane
};

// FP items outside the shared walk (they have neither BP body nor slices per
// item: one instance).
void proj_fp_items(const BatchRun &R, int grid, hipStream_t st) {
  launch_one<8, 0, 3>(grid, R.fp_total, R.bp_lds, R.W.probs.as<BatchProb>(), R.L, st);
  CCPI_HIP(hipGetLastError());
}

void proj(const BatchRun &R, const Tuned &T, int mode, hipStream_t st) {
  BatchProb *P = R.W.probs.as<BatchProb>();
  if (mode == 0) {
    if (R.fs_total > 0) {
      hipLaunchKernelGGL(batch_fp_shared_kernel,
                         wg_dim3(R.fs_total, kBatchShareThreads, "batched CGLS: too many rays"),
                         dim3(kBatchShareThreads), 0, st, P, R.L);
      CCPI_HIP(hipGetLastError());
    }
    if (R.fp_total > 0) proj_fp_items(R, T.fp_grid, st);
    return;
  }
  if (T.rc == 8)
    launch_bp_mode<8>(mode, R.bp_kinds, T.bp_grid, R.bp_total, R.bp_lds, P, R.L, st);
  else
    launch_bp_mode<16>(mode, R.bp_kinds, T.bp_grid, R.bp_total, R.bp_lds, P, R.L, st);
  CCPI_HIP(hipGetLastError());
}

// Item lists for row/slice blocks of `rc`.  A problem whose plan takes the
// tiled BP gets tile items of rc slices, its staged span and angle groups
// from the plan and its angles per staged block for rc slices.
void layout(BatchRun &R, int rc, hipStream_t st) {
  std::vector<int> off(5 * (R.count + 1), 0);
  long long parts = 0;
  R.bp_lds = 0;
  R.bp_kinds = 0;
  for (int p = 0; p < R.count; p++) {
    BatchProb &B = R.host[p];
    const ParArgs &g = B.g;
    const ParBpShape &S = R.plan.bp[p];
    B.fp_lr = par_fp_lanes_per_ray(g.nv);
    const bool share = par_share_fits(g);
    if (share) B.fp_lr = std::min(B.fp_lr, kBatchShareLanes);
    B.fp_nbx = (g.na * g.nh + 256 / B.fp_lr - 1) / (256 / B.fp_lr);
    B.fp_nby = (g.nv + 4 * B.fp_lr - 1) / (4 * B.fp_lr);
    B.bp_tiled = S.tiled;
    R.bp_kinds |= S.tiled ? 1 : 2;
    if (S.tiled) {
      B.bp_hmax = S.hmax;
      B.bp_groups = S.groups;
      B.bp_ab = par_bp_block_angles(S.hmax, rc);
      R.bp_lds = std::max(R.bp_lds, par_bp_tile_bytes(S.hmax, rc, B.bp_ab));
      B.bp_nbx = ((g.nx + 15) / 16) * ((g.ny + 15) / 16);
    } else {
      B.bp_nbx = (g.nx * g.ny + 255) / 256;
    }
    B.bp_nby = (g.nz + rc - 1) / rc;
    const long long fs = share ? par_share_items(g, B.fp_lr) : 0;
    const long long fp = share ? 0 : (long long)B.fp_nbx * B.fp_nby;
    B.fp_part = (int)parts;
    B.fp_parts = share ? (int)par_share_parts(g, B.fp_lr) : (int)(4 * fp);
    parts += B.fp_parts;
    CCPI_REQUIRE(off[4 * (R.count + 1) + p] + fs < (1LL << 31) && off[p] + fp < (1LL << 31) &&
                     parts < (1LL << 31),
                 CCPI_E_LIMIT, "batched CGLS: too many rays");
    off[p + 1] = off[p] + (int)fp;
    off[4 * (R.count + 1) + p + 1] = off[4 * (R.count + 1) + p] + (int)fs;
    off[(R.count + 1) + p + 1] = off[(R.count + 1) + p] + B.bp_nbx * B.bp_nby;
    off[2 * (R.count + 1) + p + 1] =
        off[2 * (R.count + 1) + p] + (int)((B.nvox + kChunk - 1) / kChunk);
    off[3 * (R.count + 1) + p + 1] =
        off[3 * (R.count + 1) + p] + (int)((B.npix + kChunk - 1) / kChunk);
  }
  R.fp_total = off[R.count];
  R.bp_total = off[2 * R.count + 1];
  R.fs_total = off[5 * R.count + 4];
  R.W.offs.upload(off, st);
  R.W.part.alloc((size_t)std::max(parts, 1LL) * sizeof(double));
  R.W.part2.alloc((size_t)std::max(4 * R.bp_total, 1) * sizeof(double));
  int *o = R.W.offs.as<int>();
  R.L.count = R.count;
  R.L.fp_off = o;
  R.L.bp_off = o + (R.count + 1);
  R.L.vx_off = o + 2 * (R.count + 1);
  R.L.px_off = o + 3 * (R.count + 1);
  R.L.fs_off = o + 4 * (R.count + 1);
  R.L.part_fp = R.W.part.as<double>();
  R.L.part_bp = R.W.part2.as<double>();
  R.W.probs.upload(R.host, st);
}

int cu_count() {
  int dev = 0, n = 0;
  CCPI_HIP(hipGetDevice(&dev));
  CCPI_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
  return std::max(n, 1);
}

}  // namespace

void run_pb_cgls_batched(const std::vector<Geometry> &geoms, float *const *b,
                         float *const *x, int iters, double *norms_out, hipStream_t caller) {
  if (geoms.empty()) return;
  WorkspaceLease lease;
  std::vector<char> tables;
  BatchRun R{*lease};
  R.count = (int)geoms.size();
  CCPI_HIP(hipStreamSynchronize(caller));
  hipStream_t st;
  CCPI_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  struct StreamGuard {
    hipStream_t s;
    ~StreamGuard() { (void)hipStreamDestroy(s); }
  } guard{st};

  // per-problem work vectors carved from one allocation
  size_t total = 0;
  for (const Geometry &G : geoms) total += 2 * G.n_vox() + G.n_pix();
  R.W.v1.alloc(total * sizeof(float));
  R.W.norms.alloc((size_t)R.count * std::max(iters, 1) * sizeof(double));
  float *w = R.W.v1.as<float>();
  for (const Geometry &G : geoms)
    CCPI_REQUIRE(G.kind == CCPI_PARALLEL, CCPI_E_ARG, "batched CGLS takes parallel-beam problems");
  // no plans: 64 problems would go through a cache of 8, each with uploads of
  // its own and, for the small ones, a walk table that a batch does not use
  R.plan = par_batch_plan(geoms, tables, R.W.tabs, st);
  std::string sig;
  for (int p = 0; p < R.count; p++) {
    const Geometry &G = geoms[p];
    BatchProb B{};
    B.g = R.plan.args[p];
    B.r = b[p];
    B.x = x[p];
    B.d = w;
    w += G.n_vox();
    B.s = w;
    w += G.n_vox();
    B.Ad = w;
    w += G.n_pix();
    B.norms = R.W.norms.as<double>() + (size_t)p * std::max(iters, 1);
    B.nvox = (long long)G.n_vox();
    B.npix = (long long)G.n_pix();
    R.host.push_back(B);
    sig += std::to_string(G.na) + "," + std::to_string(G.nh) + "," + std::to_string(G.nv) +
           "," + std::to_string(G.nx) + "," + std::to_string(G.ny) + "," + std::to_string(G.nz) + ";";
  }

  // slices per BP item and the grids, tuned once per batch shape
  Tuned T{16, 0, 0};
  bool have = false;
  if (const char *env = std::getenv("CCPI_BATCH_TUNE")) {
    // "rc,fp_blocks_per_cu,bp_blocks_per_cu" pins the launch shape (skips
    // the timing sweep); 0 blocks per CU is one workgroup / wavefront per item
    int rc = 16, fm = 0, bm = 0;
    if (std::sscanf(env, "%d,%d,%d", &rc, &fm, &bm) == 3 && (rc == 8 || rc == 16) &&
        fm >= 0 && bm >= 0) {
      T = Tuned{rc, fm * cu_count(), bm * cu_count()};
      have = true;
    }
  }
  if (!have) {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    auto it = g_tuned.find(sig);
    if (it != g_tuned.end()) {
      T = it->second;
      have = true;
    }
  }
  if (!have) {
    struct Events {
      hipEvent_t a = nullptr, b = nullptr;
      Events() {
        CCPI_HIP(hipEventCreate(&a));
        CCPI_HIP(hipEventCreate(&b));
      }
      ~Events() {
        if (a) (void)hipEventDestroy(a);
        if (b) (void)hipEventDestroy(b);
      }
    } ev;
    auto time = [&](auto launch) {
      CCPI_HIP(hipEventRecord(ev.a, st));
      launch();
      CCPI_HIP(hipEventRecord(ev.b, st));
      CCPI_HIP(hipEventSynchronize(ev.b));
      float ms = 0.f;
      CCPI_HIP(hipEventElapsedTime(&ms, ev.a, ev.b));
      return ms;
    };
    // FP of d (scratch, contents irrelevant) and BP of r into s, outputs
    // discarded; the first launch of each loads its kernel
    int rc = 16;
    layout(R, rc, st);
    if (R.fp_total > 0) proj_fp_items(R, 0, st);
    T = tune_batch(
        R.fp_total > 0, cu_count(),
        [&](int slices) {
          rc = slices;
          layout(R, rc, st);
          proj(R, Tuned{rc, 0, 0}, 1, st);
        },
        [&](int grid) { return time([&] { proj_fp_items(R, grid, st); }); },
        [&](int grid) { return time([&] { proj(R, Tuned{rc, 0, grid}, 1, st); }); });
    std::lock_guard<std::mutex> lock(g_tune_mu);
    g_tuned[sig] = T;
  }
  layout(R, T.rc, st);
  BatchProb *P = R.W.probs.as<BatchProb>();
  const int vgrid = 4 * cu_count();

  // start: d = A^T b, gamma = ||d||^2 (cgls.cpp:45-49)
  proj(R, T, 2, st);
  hipLaunchKernelGGL(batch_scalar_kernel<0>, dim3(R.count), dim3(256), 0, st, P, R.L);
  CCPI_HIP(hipGetLastError());

  // one iteration, captured once and replayed
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  CCPI_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  proj(R, T, 0, st);
  hipLaunchKernelGGL(batch_scalar_kernel<1>, dim3(R.count), dim3(256), 0, st, P, R.L);
  hipLaunchKernelGGL(batch_vec_kernel<0>, dim3(vgrid), dim3(256), 0, st, P, R.L);
  proj(R, T, 1, st);
  hipLaunchKernelGGL(batch_scalar_kernel<2>, dim3(R.count), dim3(256), 0, st, P, R.L);
  hipLaunchKernelGGL(batch_vec_kernel<1>, dim3(vgrid), dim3(256), 0, st, P, R.L);
  CCPI_HIP(hipStreamEndCapture(st, &graph));
  struct GraphGuard {
    hipGraph_t g;
    hipGraphExec_t e;
    ~GraphGuard() {
      if (e) (void)hipGraphExecDestroy(e);
      if (g) (void)hipGraphDestroy(g);
    }
  } gg{graph, nullptr};
  CCPI_HIP(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
  gg.e = exec;
  for (int it = 0; it < iters; it++) CCPI_HIP(hipGraphLaunch(exec, st));
  if (norms_out && iters > 0)
    CCPI_HIP(hipMemcpyAsync(norms_out, R.W.norms.p, (size_t)R.count * iters * sizeof(double),
                            hipMemcpyDeviceToHost, st));
  CCPI_HIP(hipStreamSynchronize(st));
  lease.keep();
}

}  // namespace ccpi
