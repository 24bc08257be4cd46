// The implicit TSQR Q (or Qᵀ) applied to a block of columns, panel by panel
// (alg/QR/tsqr/apply_tsqr_QT.cxx:31-165): a wave holds 16 columns of a leaf's
// rows of B (or of a tree pair's top rows) in registers as 16×16 tiles and
// applies the factorization's 16-column panels to them one after another,
//   W = V_kᵀ·B,  U = op(T_kk)·W,  B −= V_k·U,
// as the factorization itself does (ptree_kernel.hip): Q_l is the product of
// the panels' I − V_k·T_kk·V_kᵀ, T_kk the diagonal tiles of its compact-WY T.
// Qᵀ takes the panels in order with T_kkᵀ, Q backwards with T_kk.  The waves
// of a workgroup share the panel in LDS (two buffers, the next one fetched
// into registers under the products).
//
// Every value of B is read and written once by the leaves and, for the top b
// rows of a leaf, once per tree level it takes part in.  Qᵀ of a 32768×128
// panel's tree (128 leaves, seven levels) on 2000 columns: 5.25 ms as three
// batched products per leaf and five per pair, each a pass over B; 1.30 ms
// here.  The leaves' 0.65 ms stand against 0.35 ms of MFMA issue and 0.21 ms
// of moving B once at the copy rate, which two workgroups a CU overlap in
// part; the levels' first two (0.20 and 0.11 ms) move B's rows at 2.5 TB/s,
// the last four (0.035 ms each) wait on eight panels in a row.
// Four waves a workgroup, so that a CU holds two or three and one's loads and
// stores of B run under another's products: eight waves measured 0.72 ms in
// the leaves and 0.23 ms in the first level.
#include "cqr_device.h"
#include "cqr_internal.h"
#include "panel16.h"

namespace cqr {

namespace {

constexpr int W = 4;   // waves, and strips of 16 columns, of a workgroup

// acc + Σ V_tᵀ·a_t, and a_t += V_t·u, over the groups of four tiles that meet
// [lo, hi); tiles of such a group outside it are zero in V.
template <int N>
__device__ __forceinline__ dbl4 range_vta(const double* Vk, const dbl4 (&a)[N], int lo, int hi, dbl4 acc, int lane) {
  const double* vp = Vk + (lane >> 4) * P16_LD + (lane & 15);
  dbl4 acc2 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int q = 0; q < (N + 3) / 4; ++q)
    if (4 * q + 3 >= lo && 4 * q < hi) {
#pragma unroll
      for (int t = 4 * q; t < 4 * q + 4; ++t)
        if (t < N) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const double x = vp[t * P16_TILE + 4 * v * P16_LD];
            if (v & 1) acc2 = __builtin_amdgcn_mfma_f64_16x16x4f64(x, a[t][v], acc2, 0, 0, 0);
            else acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x, a[t][v], acc, 0, 0, 0);
          }
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  return acc + acc2;
}
template <int N>
__device__ __forceinline__ void range_vu(const double* Vk, dbl4 (&a)[N], int lo, int hi, const dbl4& u, int lane) {
  const double* vp = Vk + (lane & 15) * P16_LD + (lane >> 4);
#pragma unroll
  for (int q = 0; q < (N + 3) / 4; ++q)
    if (4 * q + 3 >= lo && 4 * q < hi) {
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int t = 4 * q; t < 4 * q + 4; ++t)
          if (t < N) a[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vp[t * P16_TILE + 4 * v], u[v], a[t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
}

// The diagonal tile (k, k) of T (b×b) in LDS as the left operand of U:
// T_kkᵀ (trans) or T_kk, row-major; one value per thread and step.
template <int NT>
struct TTile {
  static constexpr int PER = (256 + NT - 1) / NT;
  double v[PER];
  __device__ __forceinline__ void fetch(const double* T, int b, int k, int tid) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + i * NT, r = 16 * k + (e & 15), q = 16 * k + (e >> 4);
      v[i] = (e < 256 && r <= q && q < b) ? T[r + (int64_t)q * b] : 0.0;
    }
  }
  __device__ __forceinline__ void put(double* X, bool trans, int tid) const {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + i * NT, r = e & 15, q = e >> 4;
      if (e < 256) X[trans ? q * P16_LD + r : r * P16_LD + q] = v[i];
    }
  }
};

}  // namespace

// Leaves: workgroup (leaf, 16·W columns) of W waves, leaf rows ≤ 16·RT.
template <int RT>
__global__ void __launch_bounds__(64 * W)
apply_leaf16_kernel(const double* __restrict__ Y, int64_t ldy, const double* __restrict__ leafT, double* __restrict__ B,
                    int64_t ldb, int64_t m, int L, int b, int64_t k, int trans) {
  constexpr int NT = 64 * W, TPW = RT / W;        // tiles of a panel fetched by each wave
  extern __shared__ double smem[];
  double* Vs = smem;                              // two panels of RT tiles, then two T tiles
  double* Ts = smem + 2 * RT * P16_TILE;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int c = lane & 15, g = lane >> 4;
  const int leaf = blockIdx.x;
  const int64_t r0 = leaf_off(leaf, m, L);
  const int r = (int)(leaf_off(leaf + 1, m, L) - r0);
  const int nblk = (b + 15) / 16, rt = (r + 15) / 16;
  const double* Yl = Y + r0;
  const double* Tl = leafT + (int64_t)leaf * b * b;
  const int64_t col = (int64_t)blockIdx.y * (16 * W) + 16 * w + c;
  const bool ok = col < k;
  double* Bc = B + r0 + (ok ? col : 0) * ldb + 4 * g;

  dbl4 pv[TPW];
  TTile<NT> pt;
  auto fetch = [&](int kk) {
    const int cc = 16 * kk + c;
    const double* p = Yl + (int64_t)min(cc, b - 1) * ldy;
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const int t = w + W * i, row = 16 * t + 4 * g;
      pv[i] = p16_rows_load(p + row, r - row, t >= kk && cc < b);
      if (t == kk)
#pragma unroll
        for (int v = 0; v < 4; ++v) pv[i][v] = 4 * g + v > c ? pv[i][v] : (4 * g + v == c && cc < b ? 1.0 : 0.0);
    }
    pt.fetch(Tl, b, kk, tid);
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TPW; ++i) p16_store(Vs + (buf * RT + w + W * i) * P16_TILE, pv[i], lane);
    pt.put(Ts + buf * P16_TILE, trans, tid);
  };
  auto panel = [&](int s) { return trans ? s : nblk - 1 - s; };

  fetch(panel(0));
  dbl4 a[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) a[t] = p16_rows_load(Bc + 16 * t, r - 16 * t - 4 * g, ok);
  put(0);
  for (int s = 0; s < nblk; ++s) {
    const int kk = panel(s), buf = s & 1;
    __syncthreads();
    if (s + 1 < nblk) fetch(panel(s + 1));
    const double* Vk = Vs + buf * RT * P16_TILE;
    const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
    const dbl4 wt = range_vta<RT>(Vk, a, kk, rt, zero, lane);
    const dbl4 u = -p16_xy(Ts + buf * P16_TILE, wt, zero, lane);
    range_vu<RT>(Vk, a, kk, rt, u, lane);
    if (s + 1 < nblk) put(buf ^ 1);
  }
#pragma unroll
  for (int t = 0; t < RT; ++t)
    if (16 * t < r) p16_rows_store(Bc + 16 * t, a[t], r - 16 * t - 4 * g, ok);
}

// One tree level: workgroup (pair, 16·W columns); the pair's receiver is leaf
// z, its sender leaf z + half, nodes node0 + z.  N tiles of b ≤ 16·N rows.
template <int N>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(3)))  // 164 VGPRs; 182 without
apply_node16_kernel(const double* __restrict__ nodeV2, const double* __restrict__ nodeT, double* __restrict__ B,
                    int64_t ldb, int64_t m, int L, int b, int64_t k, int half, int trans) {
  constexpr int NT = 64 * W, TPW = (N + W - 1) / W;
  extern __shared__ double smem[];
  double* Vs = smem;
  double* Ts = smem + 2 * N * P16_TILE;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int c = lane & 15, g = lane >> 4;
  const int z = blockIdx.x, nblk = (b + 15) / 16;
  const int64_t bb = (int64_t)b * b;
  const double* V2 = nodeV2 + z * bb;
  const double* Tn = nodeT + z * bb;
  const int64_t col = (int64_t)blockIdx.y * (16 * W) + 16 * w + c;
  const bool ok = col < k;
  double* Bz = B + leaf_off(z, m, L) + (ok ? col : 0) * ldb;
  double* Bs = B + leaf_off(z + half, m, L) + (ok ? col : 0) * ldb + 4 * g;

  dbl4 pv[TPW], pz;
  TTile<NT> pt;
  auto fetch = [&](int kk) {
    const int cc = 16 * kk + c;
    const double* p = V2 + (int64_t)min(cc, b - 1) * b;
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const int t = w + W * i, row = 16 * t + 4 * g;
      pv[i] = p16_rows_load(p + row, b - row, t <= kk && cc < b);
      if (t == kk)
#pragma unroll
        for (int v = 0; v < 4; ++v) pv[i][v] = 4 * g + v <= c ? pv[i][v] : 0.0;
    }
    pt.fetch(Tn, b, kk, tid);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 16 * kk + g + 4 * v;
      pz[v] = ok && row < b ? Bz[row] : 0.0;
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TPW; ++i)
      if (w + W * i < N) p16_store(Vs + (buf * N + w + W * i) * P16_TILE, pv[i], lane);
    pt.put(Ts + buf * P16_TILE, trans, tid);
  };
  auto panel = [&](int s) { return trans ? s : nblk - 1 - s; };

  fetch(panel(0));
  dbl4 a[N];
#pragma unroll
  for (int t = 0; t < N; ++t) a[t] = p16_rows_load(Bs + 16 * t, b - 16 * t - 4 * g, ok);
  put(0);
  for (int s = 0; s < nblk; ++s) {
    const int kk = panel(s), buf = s & 1;
    dbl4 top = pz;
    __syncthreads();
    if (s + 1 < nblk) fetch(panel(s + 1));
    const double* Vk = Vs + buf * N * P16_TILE;
    const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
    const dbl4 wt = range_vta<N>(Vk, a, 0, kk + 1, top, lane);
    const dbl4 u = -p16_xy(Ts + buf * P16_TILE, wt, zero, lane);
    top += u;
    range_vu<N>(Vk, a, 0, kk + 1, u, lane);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 16 * kk + g + 4 * v;
      if (ok && row < b) Bz[row] = top[v];
    }
    if (s + 1 < nblk) put(buf ^ 1);
  }
#pragma unroll
  for (int t = 0; t < N; ++t)
    if (16 * t < b) p16_rows_store(Bs + 16 * t, a[t], b - 16 * t - 4 * g, ok);
}

template <int RT>
static int leaf_launch16(cqr_ctx* c, const double* Y, int64_t ldy, const double* leafT, double* B, int64_t ldb, int64_t m,
                         int L, int b, int64_t k, int trans) {
  const size_t lds = sizeof(double) * (2 * RT + 2) * P16_TILE;
  auto kern = apply_leaf16_kernel<RT>;
  CQR_TRY(set_max_lds(c, (const void*)kern, (int)lds));
  hipLaunchKernelGGL(kern, dim3((unsigned)L, (unsigned)((k + 16 * W - 1) / (16 * W))), dim3(64 * W), lds, c->stream, Y,
                     ldy, leafT, B, ldb, m, L, b, k, trans);
  return check_launch(c, "apply_leaf16");
}
template <int N>
static int node_launch16(cqr_ctx* c, const double* V2, const double* T, double* B, int64_t ldb, int64_t m, int L, int b,
                         int64_t k, int npairs, int half, int trans) {
  const size_t lds = sizeof(double) * (2 * N + 2) * P16_TILE;
  auto kern = apply_node16_kernel<N>;
  CQR_TRY(set_max_lds(c, (const void*)kern, (int)lds));
  hipLaunchKernelGGL(kern, dim3((unsigned)npairs, (unsigned)((k + 63) / 64)), dim3(256), lds, c->stream, V2, T, B, ldb, m,
                     L, b, k, half, trans);
  return check_launch(c, "apply_node16");
}

// Leaves of at most 512 rows (rows: the largest) fit the strips' registers.
bool apply16_takes(const TsqrPlan& p, int64_t k) {
  return p.max_leaf_rows <= 512 && p.b <= 128 && (k + 63) / 64 <= 65535;
}

int apply16_leaves(cqr_ctx* c, int trans, const TsqrPlan& p, const double* Y, int64_t ldy, const double* leafT, double* B,
                   int64_t ldb, int64_t k) {
  const int L = (int)p.nleaves, b = (int)p.b;
  const int64_t r = p.max_leaf_rows;
  hipEvent_t ev = prof_begin(c);
  if (r <= 128) CQR_TRY(leaf_launch16<8>(c, Y, ldy, leafT, B, ldb, p.m, L, b, k, trans));
  else if (r <= 256) CQR_TRY(leaf_launch16<16>(c, Y, ldy, leafT, B, ldb, p.m, L, b, k, trans));
  else CQR_TRY(leaf_launch16<32>(c, Y, ldy, leafT, B, ldb, p.m, L, b, k, trans));
  prof_end(c, ev, PK_BGEMM, 4.0 * p.m * b * (double)k, 8.0 * ((double)p.m * b + 2.0 * p.m * k));
  return CQR_OK;
}

int apply16_level(cqr_ctx* c, int trans, const TsqrPlan& p, int lv, const double* nodeV2, const double* nodeT, double* B,
                  int64_t ldb, int64_t k) {
  const int npairs = (int)p.levels[lv].size(), b = (int)p.b, L = (int)p.nleaves;
  if (npairs == 0) return CQR_OK;
  const int half = p.levels[lv][0].second;   // sender of pair 0 = ⌈n/2⌉
  const int64_t bb = p.b * p.b;
  const double* V2 = nodeV2 + p.level_node0[lv] * bb;
  const double* T = nodeT + p.level_node0[lv] * bb;
  hipEvent_t ev = prof_begin(c);
  if (b <= 16) CQR_TRY(node_launch16<1>(c, V2, T, B, ldb, p.m, L, b, k, npairs, half, trans));
  else if (b <= 32) CQR_TRY(node_launch16<2>(c, V2, T, B, ldb, p.m, L, b, k, npairs, half, trans));
  else if (b <= 64) CQR_TRY(node_launch16<4>(c, V2, T, B, ldb, p.m, L, b, k, npairs, half, trans));
  else CQR_TRY(node_launch16<8>(c, V2, T, B, ldb, p.m, L, b, k, npairs, half, trans));
  prof_end(c, ev, PK_BGEMM, 4.0 * npairs * b * (double)b * k, 8.0 * npairs * ((double)b * b + 4.0 * b * k));
  return CQR_OK;
}

}  // namespace cqr
