// TSQR leaves and reduction tree on sixteen-column panels (panel16.h).
//
// The tree is the reference's binary schedule (alg/QR/tsqr/bitree_tsqr.cxx:
// 172-232): on a level with n live ranks, receiver z stacks its R on the R
// of sender z + ceil(n/2) and refactors the 2b×b triangle pair (dtpqrt with
// l = b, :20-34).
//
// Leaves and nodes advance right-looking by panels of 16 columns; wave w of
// the workgroup owns the columns [16w, 16w + 16) for the whole
// factorization, in registers.  In step k wave k factors its strip and puts
// the vectors and T_kk in LDS; after one barrier every later wave applies
// them to its own strip (W = Vᵀ·A, U = T_kkᵀ·W, A −= V·U, all on FP64 MFMA
// with A as accumulator and B operand), wave k + 1 going straight on to its
// panel, while the finished waves turn V into their tiles of T.  So a step
// costs one panel and one application of it, with one barrier.
//
// Row block k of R is final after step k, and step k of a tree node needs
// only row block k of its two inputs.  Each wave publishes its 16×16 tile
// R(k, w) as soon as it is final and waits only for the tiles of its own
// column block, so all levels of the tree advance together, a step or so
// apart: the tree costs about (b/16 + depth) steps.  Node ids follow forward
// level order, so every producer has a smaller block id than its consumer
// and is dispatched first; waits are bounded (a timeout raises a device flag
// and the node finishes with whatever it has).
//
// Bound: the serial chain of columns, not bytes or flops.  A 256×128 leaf
// takes 0.17 ms (25 k cycles a panel, 1.0–1.2 k a column, and 8.5–10.5 k for
// the next strip's products); a tree level adds about 13 µs.  Before, with
// one reflector at a time broadcast through LDS (leaf) and 8-column blocks
// with four products and six barriers each (node), a leaf took 0.25–0.30 ms
// and a level 21 µs: with this and the other kernels' gains hh_recon_qr of
// 32768×128 went 0.88 → 0.49 ms, of 4099×100 (a width that took a
// column-at-a-time node) 0.95 → 0.34 ms, 512 batched problems of up to
// 16384×128 17.4 → 10.4 ms, QR 32768×4096 43.9 → 33.0 ms.
#include "cqr_device.h"
#include "cqr_internal.h"
#include "panel16.h"

namespace cqr {

// Producer of rank r's current R when entering level `lv` (level sizes
// n_0 = L, n_{k+1} = ceil(n_k / 2)): the node of the last earlier level at
// which r was a receiver, or leaf r.  Returns a node id, or −1 for a leaf.
__device__ inline int producer_of(int r, int lv, int L) {
  int n = L, node0 = 0, best = -1;
  for (int k = 0; k < lv; ++k) {
    const int pairs = n / 2;
    if (r < pairs) best = node0 + r;
    node0 += pairs;
    n = n / 2 + (n & 1);
  }
  return best;
}

// Zeros below the diagonal tiles of columns [16w, 16w + 16) of a b×b matrix.
__device__ __forceinline__ void zero_below(double* __restrict__ M, int b, int w, int lane) {
  for (int cc = 0; cc < P16 && 16 * w + cc < b; ++cc)
    for (int rr = 16 * (w + 1) + lane; rr < b; rr += 64) M[rr + (int64_t)(16 * w + cc) * b] = 0.0;
}

// Tile (i, k) of T, given transposed (as p16_tcol and the T slots hold it).
__device__ __forceinline__ void put_t_tile(double* __restrict__ T, int b, int i, int k, const dbl4& x, int lane) {
  const int row = 16 * i + (lane & 15);
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int col = 16 * k + (lane >> 4) + 4 * v;
    if (row < b && col < b) T[row + (int64_t)col * b] = x[v];
  }
}

// LDS (doubles): the vectors of two panels (RT row tiles each), the tiles of
// T for W column blocks, and one tile where a panel keeps its pivot tile.
template <int W, int RT>
constexpr int p16_smem_doubles() { return (2 * RT + W * (W + 1) / 2 + 1) * P16_TILE; }

// ---------------------------------------------------------------------------
// One leaf per workgroup of W waves: dgeqrf of r ≤ 16·RT rows × b ≤ 16·W
// columns (b > 16·(W − 1) is not needed: waves without columns only attend
// the barriers).  Writes [V\R] over A, R (b×b), T (b×b) and tau.  With lcnt
// set, tile R(k, w) is announced in lcnt[8·leaf + w] = epoch·256 + k + 1.
// ---------------------------------------------------------------------------
template <int W, int RT>
__device__ __forceinline__ void leaf16_body(double* __restrict__ A, int64_t lda, int64_t m, int L, int b,
                                            double* __restrict__ Rout, double* __restrict__ Tout,
                                            double* __restrict__ tauout, const BatchProb* __restrict__ bp, int nprob,
                                            int gleaf, double* smem, uint64_t* __restrict__ lcnt, uint64_t epoch) {
  constexpr int NB = RT - 1;   // tiles below the pivot tile
  int leaf = gleaf;
  if (bp) {                    // batched: A is the group's base, the problem's block at aoff
    const BatchProb P = bp[bp_find(bp, nprob, gleaf, BP_LEAF)];
    A += P.aoff;
    lda = P.m;
    m = P.m;
    L = P.L;
    leaf = gleaf - P.leaf0;
  }
  const int64_t r0 = leaf_off(leaf, m, L);
  const int r = (int)(leaf_off(leaf + 1, m, L) - r0);
  const int64_t bb = (int64_t)b * b;
  double* Al = A + r0;
  double* Rl = Rout + (int64_t)gleaf * bb;
  double* Tl = Tout + (int64_t)gleaf * bb;
  double* taul = tauout + (int64_t)gleaf * b;
  double* Vs = smem;                              // two panels
  double* S = smem + 2 * RT * P16_TILE;           // tiles of T

  const int lane = threadIdx.x & 63, w = wave_id();
  const int c = lane & 15, g = lane >> 4;
  const int nblk = (b + P16 - 1) / P16, rt = (r + 15) / 16;
  const int col = 16 * w + c;
  const bool colok = col < b;
  // a lane's four rows of a tile are contiguous: two 16-byte accesses where
  // every column starts on a 16-byte boundary
  const bool vec = ((lda & 1) == 0) && ((reinterpret_cast<uintptr_t>(Al) & 15) == 0);
  typedef double dbl2 __attribute__((ext_vector_type(2)));
  double* Ac = Al + (int64_t)(colok ? col : 0) * lda + 4 * g;
  const int rg = r - 4 * g;                      // rows left from this lane group's first
  dbl4 D, a[NB];
  if (vec && r == 16 * RT && b == 16 * W) {      // the usual full leaf
    auto full = [&](int t) {
      const dbl2 lo = *reinterpret_cast<const dbl2*>(Ac + 16 * t), hi = *reinterpret_cast<const dbl2*>(Ac + 16 * t + 2);
      return dbl4{lo[0], lo[1], hi[0], hi[1]};
    };
    D = full(0);
#pragma unroll
    for (int t = 0; t < NB; ++t) a[t] = full(t + 1);
  } else {
    // loads from clamped rows, then masked: no branch, no mask kept
    auto part = [&](int t) {
      dbl4 x;
#pragma unroll
      for (int v = 0; v < 4; ++v) x[v] = Ac[max(min(16 * t + v, rg - 1), -4 * g)];
#pragma unroll
      for (int v = 0; v < 4; ++v) x[v] = (colok && 16 * t + v < rg) ? x[v] : 0.0;
      return x;
    };
    D = part(0);
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      a[t] = part(t + 1);
      if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
  auto store_tile = [&](int t, const dbl4& x) {
    double* p = Ac + 16 * t;
    if (!colok) return;
    if (vec && 16 * t + 16 <= r) {
      *reinterpret_cast<dbl2*>(p) = dbl2{x[0], x[1]};
      *reinterpret_cast<dbl2*>(p + 2) = dbl2{x[2], x[3]};
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (16 * t + v < rg) p[v] = x[v];
    }
  };
  if (w < nblk) {
    zero_below(Rl, b, w, lane);
    zero_below(Tl, b, w, lane);
  }
  dbl4 tnew = {0.0, 0.0, 0.0, 0.0};   // tile (w, k−1) of T, waiting for its slot
  for (int k = 0; k <= nblk; ++k) {
    double* Vk = Vs + (k & 1) * (RT * P16_TILE);
    const int nact = rt - 1 - k;
    if (w == k && k < nblk) {
      __builtin_amdgcn_s_setprio(3);
      Panel16<NB, false> P;
      P.factor(D, a, nact, min(P16, b - 16 * k), lane, S + p16_slot(k, k), Vk + P16_TILE, S + p16_slot(0, W));
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 4 * g + v;
        Vk[(g + 4 * v) * P16_LD + c] = row > c ? D[v] : (row == c ? 1.0 : 0.0);
      }
      if (g == 0 && colok) taul[col] = P.tau;
      __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
    const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
    auto apply = [&]() {
      dbl4 top[1] = {D};
      dbl4 wt = p16_vta<1>(Vk, top, 1, zero, lane);
      wt = p16_vta<NB>(Vk + P16_TILE, a, nact, wt, lane);
      const dbl4 u = -p16_xy(S + p16_slot(k, k), wt, zero, lane);
      p16_vu<1>(Vk, top, 1, u, lane);
      D = top[0];
      p16_vu<NB>(Vk + P16_TILE, a, nact, u, lane);
    };
    // The next panel's strip goes first, alone: another strip's MFMAs on its
    // SIMD would halve its rate, and they fit beside that panel's VALU work.
    if (k + 1 < nblk) {
      if (w == k + 1) apply();
      __syncthreads();
    }
    if (w >= nblk) continue;
    if (w < k - 2) p16_store(S + p16_slot(w, k - 2), tnew, lane);
    if (k < nblk) {
      if (w > k + 1) {
        apply();
      } else if (w < k) {
        dbl4 top[1] = {D};
        dbl4 gt = p16_vta<1>(Vk, top, 1, zero, lane);
        gt = p16_vta<NB>(Vk + P16_TILE, a, nact, gt, lane);
        p16_store(S + p16_slot(w, k), gt, lane);
      }
      if (w == k) {                              // the scaled vectors back from LDS (every tile that factor() touched)
        put_t_tile(Tl, b, k, k, p16_load(S + p16_slot(k, k), lane), lane);
#pragma unroll
        for (int t = 0; t < NB; ++t)
          if (t < Panel16<NB, false>::H || nact > Panel16<NB, false>::H) a[t] = p16_load(Vk + (t + 1) * P16_TILE, lane);
      }
      // row block k of this strip is final: R(k, w), and vectors for w ≤ k
      if (w >= k) {
        const int row = 16 * k + 4 * g;
        if (colok) {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (row + v < b) store_coherent(Rl + row + v + (int64_t)col * b, row + v <= col ? D[v] : 0.0);
        }
        // the wave whose panel is next announces this tile together with its
        // own panel's, so that it does not wait for the stores now
        if (lcnt && w != k + 1) {
          wait_memory();
          if (lane == 0) flag_store(lcnt + 8 * (int64_t)gleaf + w, epoch * 256 + (uint64_t)(k + 1));
        }
      }
      store_tile(k, D);
      D = a[0];
#pragma unroll
      for (int t = 0; t + 1 < NB; ++t) a[t] = a[t + 1];
      a[NB - 1] = zero;
    }
    if (w < k - 1) {
      tnew = p16_tcol(S, w, k - 1, lane);
      put_t_tile(Tl, b, w, k - 1, tnew, lane);
    }
  }
  // the rows below the last panel's block
  if (w < nblk) {
    store_tile(nblk, D);
#pragma unroll
    for (int t = 0; t < NB; ++t)
      if (16 * (nblk + 1 + t) < r) {
        store_tile(nblk + 1 + t, a[t]);
        __builtin_amdgcn_sched_barrier(0);
      }
  }
}

// ---------------------------------------------------------------------------
// A leaf taller than a wave's registers (r ≤ 256·P rows, b ≤ 16·S columns):
// P waves share a strip, 256 rows each, the first of them with the pivot
// tile.  They factor a panel together (a barrier a column) and add their
// shares of each product in LDS (X), so the steps run one after another, with
// one panel of V in LDS.  Three loops rather than one with roles: the factor()
// of the strip's own panel then stands in no loop, where its registers
// spilled.  512×64 leaves take 0.11 ms (0.125 with a reflector at a time over
// 64-row lanes); hh_recon_qr of 65536×16 225 → 147 µs, ×32 321 → 234,
// 8192×64 416 → 275 (with the other kernels' gains).  A single strip (b ≤ 16)
// keeps its vectors in registers, so that two or four leaves share a CU: 4500
// leaves of 1024×16 take 0.43 ms, 0.70 with V in 143 KB of LDS, a leaf a CU.
// ---------------------------------------------------------------------------
template <int S, int P>
constexpr int tall_smem_doubles() {
  return ((S > 1 ? 16 * P : P - 1) + S * (S + 1) / 2 + 1 + (S - 1) * P) * P16_TILE + p16_ex_doubles(P);
}

template <int S, int P>
__device__ __forceinline__ void leaf16_tall_body(double* __restrict__ A, int64_t lda, int64_t m, int L, int b,
                                                 double* __restrict__ Rout, double* __restrict__ Tout,
                                                 double* __restrict__ tauout, const BatchProb* __restrict__ bp,
                                                 int nprob, int gleaf, double* smem) {
  constexpr int NB = P16 - 1;
  int leaf = gleaf;
  if (bp) {                    // batched: A is the group's base, the problem's block at aoff
    const BatchProb B = bp[bp_find(bp, nprob, gleaf, BP_LEAF)];
    A += B.aoff;
    lda = B.m;
    m = B.m;
    L = B.L;
    leaf = gleaf - B.leaf0;
  }
  const int64_t r0 = leaf_off(leaf, m, L);
  const int r = (int)(leaf_off(leaf + 1, m, L) - r0);
  const int64_t bb = (int64_t)b * b;
  double* Rl = Rout + (int64_t)gleaf * bb;
  double* Tl = Tout + (int64_t)gleaf * bb;
  double* taul = tauout + (int64_t)gleaf * b;
  // the panel, tile by tile; of a single strip only a tile for each low part's D
  double* Vk = smem;
  double* Ts = Vk + (S > 1 ? 16 * P : P - 1) * P16_TILE;   // tiles of T, and one for the pivot tile
  double* X = Ts + (S * (S + 1) / 2 + 1) * P16_TILE;
  double* ex = X + (S - 1) * P * P16_TILE;

  const int lane = threadIdx.x & 63, w = wave_id(), strip = w / P, part = w % P;
  const int c = lane & 15, g = lane >> 4;
  const int nblk = (b + P16 - 1) / P16;
  const int col = 16 * strip + c;
  const bool colok = col < b;
  const int rg = r - 256 * part - 4 * g;          // rows left from this lane group's first
  double* Ac = A + r0 + 256 * part + 4 * g + (int64_t)(colok ? col : 0) * lda;
  const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
  // loads from clamped rows, then masked: no branch, no mask kept
  const double* A0 = Ac - 4 * g - 256 * part;     // the leaf's first row
  auto load = [&](int t) {
    dbl4 x;
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] = A0[min(256 * part + 4 * g + 16 * t + v, r - 1)];
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] = (colok && 16 * t + v < rg) ? x[v] : 0.0;
    return x;
  };
  dbl4 D = load(0), a[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    a[t] = load(t + 1);
    if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  }
  if (part == 0 && strip < nblk) {
    zero_below(Rl, b, strip, lane);
    zero_below(Tl, b, strip, lane);
  }
  double* Vp = Vk + (S > 1 ? 16 * part : part - 1) * P16_TILE;   // this part's tiles of the panel
  auto panel = [&](int k) {                       // another strip's panel: its columns, then V and T_kk are there
    for (int j = 16 * k; j < min(b, 16 * k + 16); ++j) __syncthreads();
    int bar = 0;
    do __syncthreads();
    while (ex[p16_more(P) + (bar++ & 1)] != 0.0);
  };
  // this part's share of V_kᵀ·(D; a) into X, for all parts after a barrier
  auto share = [&](int k) {
    dbl4 top[1] = {D};
    dbl4 wt = p16_vta<1>(Vp, top, 1, zero, lane);
    wt = p16_vta<NB>(Vp + P16_TILE, a, NB, wt, lane);
    p16_store(X + ((strip < k ? strip : strip - 1) * P + part) * P16_TILE, wt, lane);
  };
  auto sum = [&](int k) {
    const double* Xs = X + (strip < k ? strip : strip - 1) * P * P16_TILE;
    dbl4 wt = p16_load(Xs, lane);
#pragma unroll
    for (int q = 1; q < P; ++q) wt += p16_load(Xs + q * P16_TILE, lane);
    return wt;
  };
  // row block k of this strip is final: R(k, strip), and vectors for strip ≤ k
  auto finish = [&](int k) {
    if (part != 0) return;
    if (strip >= k && colok) {
      const int row = 16 * k + 4 * g;
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (row + v < b) Rl[row + v + (int64_t)col * b] = row + v <= col ? D[v] : 0.0;
    }
    p16_rows_store(Ac + 16 * k, D, rg - 16 * k, colok);
    D = a[0];
#pragma unroll
    for (int t = 0; t + 1 < NB; ++t) a[t] = a[t + 1];
    a[NB - 1] = zero;
  };
  // before its own panel the strip takes the earlier ones in
  for (int k = 0; k < min(strip, nblk); ++k) {
    panel(k);
    if (strip < nblk) share(k);
    __syncthreads();
    if (strip < nblk) {
      const dbl4 u = -p16_xy(Ts + p16_slot(k, k), sum(k), zero, lane);
      dbl4 top[1] = {D};
      p16_vu<1>(Vp, top, 1, u, lane);
      D = top[0];
      p16_vu<NB>(Vp + P16_TILE, a, NB, u, lane);
      finish(k);
    }
    __syncthreads();
  }
  if (strip >= nblk) return;                      // (no barrier is left)
  {
    const int k = strip;
    __builtin_amdgcn_s_setprio(3);
    Panel16<NB, false, P, S == 1> F;
    F.col = Ac - 4 * g;
    F.rows = colok ? r - 256 * part : 0;
    F.ex = ex;
    F.part = part;
    F.factor(D, a, NB, min(P16, b - 16 * k), lane, Ts + p16_slot(k, k), Vp + P16_TILE,
             part == 0 ? Ts + p16_slot(0, S) : Vp);
    if (part == 0) {
      if (S > 1)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 4 * g + v;
          Vk[(g + 4 * v) * P16_LD + c] = row > c ? D[v] : (row == c ? 1.0 : 0.0);
        }
      if (g == 0 && colok) taul[col] = F.tau;
    }
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();
    __syncthreads();
    // the scaled vectors back from LDS
    if (part == 0) put_t_tile(Tl, b, k, k, p16_load(Ts + p16_slot(k, k), lane), lane);
    if constexpr (S > 1) {
      if (part != 0) D = p16_load(Vp, lane);
#pragma unroll
      for (int t = 0; t < NB; ++t) a[t] = p16_load(Vp + (t + 1) * P16_TILE, lane);
    } else {
      if (part != 0) D = p16_load(Vp, lane);
    }
    finish(k);
    __syncthreads();
  }
  // after it, the strip's tiles of T
  dbl4 tnew = zero;
  for (int k = strip + 1; k < nblk; ++k) {
    panel(k);
    share(k);
    if (part == 0 && strip < k - 2) p16_store(Ts + p16_slot(strip, k - 2), tnew, lane);
    __syncthreads();
    if (part == 0) {
      p16_store(Ts + p16_slot(strip, k), sum(k), lane);
      if (strip < k - 1) {
        tnew = p16_tcol(Ts, strip, k - 1, lane);
        put_t_tile(Tl, b, strip, k - 1, tnew, lane);
      }
    }
    finish(k);
    __syncthreads();
  }
  if (part == 0 && strip < nblk - 1) {
    if (strip < nblk - 2) p16_store(Ts + p16_slot(strip, nblk - 2), tnew, lane);
    put_t_tile(Tl, b, strip, nblk - 1, p16_tcol(Ts, strip, nblk - 1, lane), lane);
  }
  // the rows below the last panel's block
  const int t0 = part == 0 ? nblk : 0;
  p16_rows_store(Ac + 16 * t0, D, rg - 16 * t0, colok);
#pragma unroll
  for (int t = 0; t < NB; ++t)
    if (t0 + t + 1 < 16) p16_rows_store(Ac + 16 * (t0 + t + 1), a[t], rg - 16 * (t0 + t + 1), colok);
}

// ---------------------------------------------------------------------------
// One tree node per workgroup of W waves (b ≤ 16·W).  The reflectors are
// [e; v2] with v2 in the bottom triangle: wave w holds the bottom tiles
// (0..w, w) of its columns and one tile of the top triangle at a time, which
// takes part in step k with row block k only:
//   W = Top(k, w) + V2_kᵀ·Bot,  Top(k, w) −= T_kkᵀ·W,  Bot −= V2_k·T_kkᵀ·W.
// A producer that is a node is waited for through cnt (8 words a node, one
// per column block); a leaf is complete at launch unless lcnt is set (fused
// launch), in which case its words there are waited for.
// ---------------------------------------------------------------------------
template <int W>
__device__ __forceinline__ void node16_body(const double* __restrict__ leafR, double* __restrict__ nodeR,
                                            double* __restrict__ V2out, double* __restrict__ Tout,
                                            double* __restrict__ tauout, uint64_t* __restrict__ cnt, uint64_t epoch,
                                            int L, int b, int* __restrict__ err, const BatchProb* __restrict__ bp,
                                            const BatchSeg* __restrict__ seg, int nseg, int nid, double* smem,
                                            const uint64_t* __restrict__ lcnt) {
  const int lane = threadIdx.x & 63, w = wave_id();
  const int c = lane & 15, g = lane >> 4;
  const int64_t bb = (int64_t)b * b;
  if (bp) {  // batched: this problem's leaves and nodes are contiguous slices
    const BatchSeg sg = seg[seg_find(seg, nseg, nid)];
    const BatchProb P = bp[sg.prob];
    nid = sg.local0 + (nid - sg.g0);
    L = P.L;
    leafR += (int64_t)P.leaf0 * bb;
    nodeR += (int64_t)P.node0 * bb;
    V2out += (int64_t)P.node0 * bb;
    Tout += (int64_t)P.node0 * bb;
    tauout += (int64_t)P.node0 * b;
    cnt += (int64_t)P.node0 * CQR_TREE_FLAGS;
  }
  // locate this node: level lv, pair z, live ranks n
  int lv = 0, n = L, node0 = 0;
  while (nid >= node0 + n / 2) {
    node0 += n / 2;
    n = n / 2 + (n & 1);
    ++lv;
  }
  const int z = nid - node0, snd = z + (n + 1) / 2;
  const int ptop = producer_of(z, lv, L), pbot = producer_of(snd, lv, L);
  const double* Rt = ptop >= 0 ? nodeR + ptop * bb : leafR + z * bb;
  const double* Rb = pbot >= 0 ? nodeR + pbot * bb : leafR + snd * bb;
  double* Ro = nodeR + nid * bb;
  double* Tn = Tout + nid * bb;
  double* V2 = V2out + nid * bb;

  double* Vs = smem;                          // vectors of two panels, W row tiles each
  double* S = smem + 2 * W * P16_TILE;        // tiles of T
  const int nblk = (b + P16 - 1) / P16;
  const int col = 16 * w + c;
  const bool colok = col < b;
  // this wave's column block of either input; null when complete at launch
  const uint64_t* ftop = ptop >= 0 ? cnt + CQR_TREE_FLAGS * ptop + w : lcnt ? lcnt + CQR_TREE_FLAGS * z + w : nullptr;
  const uint64_t* fbot = pbot >= 0 ? cnt + CQR_TREE_FLAGS * pbot + w : lcnt ? lcnt + CQR_TREE_FLAGS * snd + w : nullptr;
  uint64_t* fout = cnt + CQR_TREE_FLAGS * (int64_t)nid + w;
  const long limit = wait_limit(err);
  bool live = true;                           // no wait of this wave has given up

  dbl4 a[W], top = {0.0, 0.0, 0.0, 0.0}, tnew = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int t = 0; t < W; ++t) a[t] = dbl4{0.0, 0.0, 0.0, 0.0};
  if (w < nblk) {
    zero_below(Ro, b, w, lane);
    zero_below(V2, b, w, lane);
    zero_below(Tn, b, w, lane);
  }
  for (int k = 0; k <= nblk; ++k) {
    double* Vk = Vs + (k & 1) * (W * P16_TILE);
    if (k < nblk && w >= k && w < nblk) {
      // tiles (k, w) of both inputs (upper triangles)
      const uint64_t want = epoch * 256 + (uint64_t)(k + 1);
      if (live && ftop) live = flag_wait(ftop, want, limit);
      if (live && fbot) live = flag_wait(fbot, want, limit);
      if (!live && lane == 0) *err = 1;
      asm volatile("" ::: "memory");          // the loads below stay behind the waits
      dbl4 bot = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int rt = 16 * k + g + 4 * v, rb = 16 * k + 4 * g + v;
        top[v] = colok && rt <= col ? load_coherent(Rt + rt + (int64_t)col * b) : 0.0;
        bot[v] = colok && rb <= col ? load_coherent(Rb + rb + (int64_t)col * b) : 0.0;
      }
#pragma unroll
      for (int t = 0; t < W; ++t)
        if (t == k) a[t] = bot;
      if (w == k) {
        __builtin_amdgcn_s_setprio(3);
        Panel16<W, true> P;
        P.factor(top, a, k + 1, min(P16, b - 16 * k), lane, S + p16_slot(k, k), Vk, S + p16_slot(0, W));
        if (g == 0 && colok) tauout[(int64_t)nid * b + col] = P.tau;
        __builtin_amdgcn_s_setprio(0);
      }
    }
    __syncthreads();
    if (w >= nblk) continue;
    if (w < k - 2) p16_store(S + p16_slot(w, k - 2), tnew, lane);
    if (k < nblk) {
      const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
      if (w > k) {
        if (w == k + 1) __builtin_amdgcn_s_setprio(3);
        const dbl4 wt = p16_vta<W>(Vk, a, k + 1, top, lane);
        const dbl4 u = -p16_xy(S + p16_slot(k, k), wt, zero, lane);
        top += u;
        p16_vu<W>(Vk, a, k + 1, u, lane);
      } else if (w < k) {
        p16_store(S + p16_slot(w, k), p16_vta<W>(Vk, a, w + 1, zero, lane), lane);
      }
      if (w >= k) {
        if (colok) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int row = 16 * k + g + 4 * v;
            if (row < b) store_coherent(Ro + row + (int64_t)col * b, row <= col ? top[v] : 0.0);
          }
        }
        // (see leaf16_body: the next panel's wave announces this tile with its own)
        if (w != k + 1) {
          wait_memory();
          if (lane == 0) flag_store(fout, epoch * 256 + (uint64_t)(k + 1));
        }
      }
      if (w == k) {                           // the scaled vectors back from LDS (every tile that factor() touched)
        put_t_tile(Tn, b, k, k, p16_load(S + p16_slot(k, k), lane), lane);
#pragma unroll
        for (int t = 0; t < W; ++t)
          if (t < Panel16<W, true>::H || k + 1 > Panel16<W, true>::H) a[t] = p16_load(Vk + t * P16_TILE, lane);
      }
      if (w == k && colok) {                  // this strip of V2 is final
#pragma unroll
        for (int t = 0; t < W; ++t)
          if (t <= k) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const int row = 16 * t + 4 * g + v;
              if (row < b) V2[row + (int64_t)col * b] = row <= col ? a[t][v] : 0.0;
            }
          }
      }
    }
    if (w < k - 1) {
      tnew = p16_tcol(S, w, k - 1, lane);
      put_t_tile(Tn, b, w, k - 1, tnew, lane);
    }
  }
}

template <int W>
__global__ void __launch_bounds__(64 * W)
node16_kernel(const double* __restrict__ leafR, double* __restrict__ nodeR, double* __restrict__ V2out,
              double* __restrict__ Tout, double* __restrict__ tauout, uint64_t* __restrict__ cnt, uint64_t epoch,
              int L, int b, int* __restrict__ err, const BatchProb* __restrict__ bp, const BatchSeg* __restrict__ seg,
              int nseg) {
  extern __shared__ double smem[];
  node16_body<W>(leafR, nodeR, V2out, Tout, tauout, cnt, epoch, L, b, err, bp, seg, nseg, blockIdx.x, smem, nullptr);
}

template <int W, int RT>
__global__ void __launch_bounds__(64 * W)
leaf16_kernel(double* __restrict__ A, int64_t lda, int64_t m, int L, int b, double* __restrict__ Rout,
              double* __restrict__ Tout, double* __restrict__ tauout, const BatchProb* __restrict__ bp, int nprob) {
  extern __shared__ double smem[];
  leaf16_body<W, RT>(A, lda, m, L, b, Rout, Tout, tauout, bp, nprob, blockIdx.x, smem, nullptr, 0);
}

template <int S, int P>
__global__ void __launch_bounds__(64 * S * P) __attribute__((amdgpu_waves_per_eu(2)))
leaf16_tall_kernel(double* __restrict__ A, int64_t lda, int64_t m, int L, int b, double* __restrict__ Rout,
                   double* __restrict__ Tout, double* __restrict__ tauout, const BatchProb* __restrict__ bp, int nprob) {
  extern __shared__ double smem[];
  leaf16_tall_body<S, P>(A, lda, m, L, b, Rout, Tout, tauout, bp, nprob, blockIdx.x, smem);
}

// Leaves and tree in one launch (b in (64, 128], leaves of at most 256
// rows): workgroups [0, L) factor the leaves and announce their R tile by
// tile, workgroups [L, L + nnodes) are the tree nodes, which start on a
// leaf's first row block while the leaf is still running.  Block ids order
// every producer before its consumers, so dispatch order alone guarantees
// progress.
template <int RT>
__global__ void __launch_bounds__(512)
leaf_tree_kernel(double* __restrict__ A, int64_t lda, int64_t m, int L, int b, double* __restrict__ leafR,
                 double* __restrict__ leafT, double* __restrict__ leafTau, double* __restrict__ nodeR,
                 double* __restrict__ V2out, double* __restrict__ Tout, double* __restrict__ tauout,
                 uint64_t* __restrict__ cnt, uint64_t* __restrict__ lcnt, uint64_t epoch, int* __restrict__ err) {
  extern __shared__ double smem[];
  if ((int)blockIdx.x < L)
    leaf16_body<8, RT>(A, lda, m, L, b, leafR, leafT, leafTau, nullptr, 0, blockIdx.x, smem, lcnt, epoch);
  else
    node16_body<8>(leafR, nodeR, V2out, Tout, tauout, cnt, epoch, L, b, err, nullptr, nullptr, 0, blockIdx.x - L, smem,
                   lcnt);
}

template <int W>
static int node16_launch(cqr_ctx* c, const double* leafR, double* nodeR, double* V2, double* T, double* tau,
                         uint64_t* cnt, int L, int nnodes, int b, uint64_t epoch, const BatchProb* bp,
                         const BatchSeg* seg, int nseg) {
  const size_t lds = sizeof(double) * p16_smem_doubles<W, W>();
  auto k = node16_kernel<W>;
  CQR_TRY(set_max_lds(c, (const void*)k, (int)lds));
  hipEvent_t ev = prof_begin(c);
  {
    SpinScope gate(c, (const void*)k, nnodes, 64 * W, lds);
    CQR_TRY(gate.status());
    hipLaunchKernelGGL(k, dim3(nnodes), dim3(64 * W), lds, c->stream, leafR, nodeR, V2, T, tau, cnt, epoch, L, b,
                       c->d_terr, bp, seg, nseg);
  }
  prof_end(c, ev, PK_TREE, nnodes * (2.0 / 3.0) * b * (double)b * b, nnodes * 40.0 * b * b);
  return check_launch(c, "node16");
}

static int tree_dispatch(cqr_ctx* c, const double* leafR, double* nodeR, double* V2, double* T, double* tau,
                         uint64_t* cnt, int L, int nnodes, int b, uint64_t epoch, const BatchProb* bp,
                         const BatchSeg* seg, int nseg) {
  // one wave per 16 columns
  if (b <= 16) return node16_launch<1>(c, leafR, nodeR, V2, T, tau, cnt, L, nnodes, b, epoch, bp, seg, nseg);
  if (b <= 32) return node16_launch<2>(c, leafR, nodeR, V2, T, tau, cnt, L, nnodes, b, epoch, bp, seg, nseg);
  if (b <= 64) return node16_launch<4>(c, leafR, nodeR, V2, T, tau, cnt, L, nnodes, b, epoch, bp, seg, nseg);
  return node16_launch<8>(c, leafR, nodeR, V2, T, tau, cnt, L, nnodes, b, epoch, bp, seg, nseg);
}

// Leaf QR of every row block, rows the largest leaf; with bp the leaves of a
// batched group.  A wave holds 16 columns of up to 256 rows; taller leaves
// (b ≤ 64) take two or four waves a strip.
int leaf16(cqr_ctx* c, double* A, int64_t lda, int64_t m, int L, int64_t rows, int b, double* R, double* T, double* tau,
           const BatchProb* bp, int nprob) {
  if (b < 1 || b > 128 || rows > (b <= 32 ? 1024 : b <= 64 ? 512 : 256))
    return set_err(c, CQR_ERR_UNSUPPORTED, "leaf: b = %d, rows = %lld", b, (long long)rows);
  auto run = [&](auto k, int waves, int lds_doubles) {
    const size_t lds = sizeof(double) * lds_doubles;
    CQR_TRY(set_max_lds(c, (const void*)k, (int)lds));
    hipEvent_t ev = prof_begin(c);
    hipLaunchKernelGGL(k, dim3(L), dim3(64 * waves), lds, c->stream, A, lda, m, L, b, R, T, tau, bp, nprob);
    prof_end(c, ev, PK_LEAF, 2.0 * m * b * b - (2.0 / 3.0) * L * (double)b * b * b, 16.0 * m * b);
    return check_launch(c, "leaf16");
  };
#define CQR_LEAF(W, RT) run(leaf16_kernel<W, RT>, W, p16_smem_doubles<W, RT>())
#define CQR_TALL(S, P) run(leaf16_tall_kernel<S, P>, S * P, tall_smem_doubles<S, P>())
  if (rows <= 256) {
    const bool low = rows <= 128;
    if (b <= 16) return low ? CQR_LEAF(1, 8) : CQR_LEAF(1, 16);
    if (b <= 32) return low ? CQR_LEAF(2, 8) : CQR_LEAF(2, 16);
    if (b <= 64) return low ? CQR_LEAF(4, 8) : CQR_LEAF(4, 16);
    return low ? CQR_LEAF(8, 8) : CQR_LEAF(8, 16);
  }
  if (rows <= 512) return b <= 16 ? CQR_TALL(1, 2) : b <= 32 ? CQR_TALL(2, 2) : CQR_TALL(4, 2);
  return b <= 16 ? CQR_TALL(1, 4) : CQR_TALL(2, 4);
#undef CQR_LEAF
#undef CQR_TALL
}

template <int RT>
static int leaf_tree_launch(cqr_ctx* c, double* A, int64_t lda, int64_t m, int L, int b, double* leafR,
                            double* leafT, double* leafTau, double* nodeR, double* V2, double* T, double* tau,
                            int nnodes) {
  const size_t lds = sizeof(double) * std::max(p16_smem_doubles<8, RT>(), p16_smem_doubles<8, 8>());
  auto k = leaf_tree_kernel<RT>;
  CQR_TRY(set_max_lds(c, (const void*)k, (int)lds));
  const uint64_t epoch = ++c->tree_epoch;
  hipEvent_t ev = prof_begin(c);
  {
    SpinScope gate(c, (const void*)k, L + nnodes, 512, lds);
    CQR_TRY(gate.status());
    hipLaunchKernelGGL(k, dim3(L + nnodes), dim3(512), lds, c->stream, A, lda, m, L, b, leafR, leafT, leafTau, nodeR,
                       V2, T, tau, c->d_cnt, c->d_cnt + CQR_TREE_FLAGS * CQR_MAX_TREE_NODES, epoch, c->d_terr);
  }
  prof_end(c, ev, PK_TREE,
           2.0 * m * b * b - (2.0 / 3.0) * L * (double)b * b * b + nnodes * (2.0 / 3.0) * b * (double)b * b,
           16.0 * m * b + nnodes * 40.0 * b * b);
  return check_launch(c, "leaf_tree");
}

// Leaf QR of every row block, then the reduction tree; one launch when the
// shapes allow the fused kernel, else the two kernels in stream order.
int leaf_tree(cqr_ctx* c, double* A, int64_t lda, int64_t m, int L, int b, double* leafR, double* leafT,
              double* leafTau, double* nodeR, double* V2, double* T, double* tau, int nnodes) {
  const int64_t rows = (m + L - 1) / L;
  // fused only while every leaf and node workgroup is resident at once (one
  // per CU, for the LDS): beyond that the nodes start only as leaves retire
  // and the two launches in order are faster (65536×2048: 32.6 → 30.4 ms)
  const bool fuse = nnodes > 0 && b > 64 && b <= 128 && rows <= 256 && L <= CQR_MAX_TREE_NODES &&
                    nnodes <= CQR_MAX_TREE_NODES && L + nnodes <= c->num_cu;
  if (!fuse) {
    CQR_TRY(leaf_qr(c, A, lda, m, L, b, leafR, leafT, leafTau));
    return launch_ptree(c, leafR, nodeR, V2, T, tau, L, nnodes, b);
  }
  if (rows <= 128) return leaf_tree_launch<8>(c, A, lda, m, L, b, leafR, leafT, leafTau, nodeR, V2, T, tau, nnodes);
  return leaf_tree_launch<16>(c, A, lda, m, L, b, leafR, leafT, leafTau, nodeR, V2, T, tau, nnodes);
}

int launch_ptree(cqr_ctx* c, const double* leafR, double* nodeR, double* V2, double* T, double* tau,
                 int L, int nnodes, int b) {
  if (nnodes <= 0) return CQR_OK;
  if (nnodes > CQR_MAX_TREE_NODES) return set_err(c, CQR_ERR_UNSUPPORTED, "tree of %d nodes", nnodes);
  return tree_dispatch(c, leafR, nodeR, V2, T, tau, c->d_cnt, L, nnodes, b, ++c->tree_epoch, nullptr, nullptr, 0);
}

// Batched: all trees of a group in one launch; cnt (CQR_TREE_FLAGS words per node) must
// hold values below 256 (the batch driver zeroes it with a kernel before
// every run, so the launch is graph-replayable with epoch 1).
int launch_ptree_batched(cqr_ctx* c, const double* leafR, double* nodeR, double* V2, double* T, double* tau,
                         uint64_t* cnt, int total_nodes, int b, const BatchProb* bp, const BatchSeg* seg, int nseg) {
  if (total_nodes <= 0) return CQR_OK;
  return tree_dispatch(c, leafR, nodeR, V2, T, tau, cnt, 0, total_nodes, b, 1, bp, seg, nseg);
}

}  // namespace cqr
