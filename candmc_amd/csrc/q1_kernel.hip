// construct_Q1 in one launch: the explicit first b columns of the TSQR Q
// (alg/QR/tsqr/construct_tsqr_Q.cxx:34-242).
//
// The reference walks the tree from the root down: the root starts from
// C = [I; 0]; every node (receiver z, sender s) turns the b×b block of its
// receiver into [C_z; C_s] = Q_node·[C_z; 0] with Q_node = I − [I;V2]·T·[I;V2]ᵀ
// (the dtprfb of :195-208):
//     X = T·C_z,   C_s = −V2·X,   C_z = C_z − X;
// and every leaf l finally expands its block with its own reflectors (the
// dormqr of :229-232):
//     Q1_l = [C_l; 0] − V_l·(T_l·(V_topᵀ·C_l)).
// Columns never mix, so the work splits into (node, strips) and (leaf, strips)
// items, a strip being 16 columns.  All blocks C are upper triangular (the
// root's identity is, and T, V2 keep it so): strip j has rows below 16(j+1)
// only, and an item takes the strips p and nb−1−p together, which evens out
// their sizes and reads each operand once for two strips.  Items are numbered
// root first, then down the tree, then the leaves: an item only waits for the
// item of its parent node and strips, which has a smaller block id and is
// therefore dispatched earlier.  Blocks C pass between items through
// device-coherent atomics and a flag per (node, strip pair) (see
// cqr_device.h).  Waits are bounded; a timeout raises a flag that the host
// reads at the next synchronisation.
//
// Bound: the chain of levels, then the leaves' MFMAs.  A wave owns the tile
// rows w and 7−w of every product: nine tiles of a triangular operand, the
// same for each of the four SIMDs.  It fetches them into registers (72 VGPRs
// each for T and V2, or for V_top and T of a leaf) before it waits for its
// parent, so that a level costs the hand-over and two products of 36 MFMAs.
// Two items fit a CU (205 VGPRs; 52 KB of LDS).  A 32768×128 panel with 128
// leaves: 90 µs, seven levels of 9 and the leaves' 25; with an item per strip
// that fetched its operands after its parent's flag 172 µs (18 a level).  A
// batch of 512 problems, group by group: 4.7 → 2.4 ms.
#include "cqr_device.h"
#include "cqr_internal.h"

namespace cqr {

namespace {

constexpr int CW = 16;     // columns of a strip
constexpr int LD = CW + 1;
constexpr int NWV = 4;

// The node consuming rank r's block above level `lv` (lv = −1 for a leaf):
// the first level k > lv at which r is a receiver (node z = r) or a sender
// (node z = r − ⌈n_k/2⌉); −1 when none exists (the root, or a one-leaf tree).
__device__ inline int parent_node(int r, int lv, int L) {
  int n = L, node0 = 0;
  for (int k = 0; n > 1; ++k) {
    const int pairs = n / 2, half = (n + 1) / 2;
    if (k > lv) {
      if (r < pairs) return node0 + r;
      if (r >= half && r < n) return node0 + (r - half);
    }
    node0 += pairs;
    n = half;
  }
  return -1;
}

// Slot s of wave w's nine tiles: tile (t, kt) of an upper triangular operand,
// row w first, then row 7 − w.
__device__ __forceinline__ int slot_row(int s, int w) { return s < 8 - w ? w : 7 - w; }
__device__ __forceinline__ int slot_col(int s, int w) { return s < 8 - w ? w + s : s - 1; }

}  // namespace

__global__ void __launch_bounds__(64 * NWV) __attribute__((amdgpu_waves_per_eu(2)))
q1_kernel(const double* __restrict__ nodeV2, const double* __restrict__ nodeT, const double* __restrict__ leafT,
          const double* __restrict__ V, int64_t ldv, int64_t m, double* __restrict__ C,
          double* __restrict__ Q, int64_t ldq, uint64_t* __restrict__ flags, uint64_t epoch, int L,
          int nnodes, int b, int* __restrict__ err, const BatchProb* __restrict__ bp,
          const BatchSeg* __restrict__ seg, int nseg) {
  // [row][column of the strip]: the wide strip (128 rows) and the narrow one
  __shared__ double S0[192 * LD];
  __shared__ double S1[192 * LD];
  __shared__ int s_ok;

  const int nb = (b + CW - 1) / CW, nsp = (nb + 1) / 2;
  int item = blockIdx.x;
  if (bp) {  // batched: V is the group's base; the problem's slices of every buffer
    const int64_t bb0 = (int64_t)b * b;
    // the table counts nb strips a node or leaf, a block takes two of them
    const int s0 = item / nsp * nb;
    const BatchSeg S = seg[seg_find(seg, nseg, s0)];
    const BatchProb P = bp[S.prob];
    item = (S.local0 + (s0 - S.g0)) / nb * nsp + item % nsp;
    L = P.L;
    nnodes = P.L - 1;
    nodeV2 += (int64_t)P.node0 * bb0;
    nodeT += (int64_t)P.node0 * bb0;
    leafT += (int64_t)P.leaf0 * bb0;
    V += P.aoff;
    ldv = P.m;
    m = P.m;
    C += (int64_t)P.leaf0 * bb0;
    Q += P.yoff;
    ldq = P.m;
    flags += (int64_t)P.node0 * nsp;
  }
  {
    // The leaf items of eight consecutive leaves are dealt so that all items
    // of a leaf run on one XCD (blocks go to XCD blockIdx mod 8) and share its
    // L2's copy of V and T; in a single problem that is the XCD of the leaf's
    // factorization (leaf z is block z there).  A partial last group keeps the
    // linear order.  A batch of 512 problems of 128 columns takes 30.6 ms so, 31.6
    // with a leaf's items on four XCDs.
    const int s0 = nnodes * nsp, rel = item - s0;
    if (rel >= 0) {
      const int grp = rel / (8 * nsp);
      if (8 * (grp + 1) <= L) item = s0 + (8 * grp + ((int)blockIdx.x & 7)) * nsp + (rel - grp * 8 * nsp) / 8;
    }
  }
  const int lo = item % nsp, hi = nb - 1 - lo;   // the item's strips; one strip if they are the same
  const bool two = lo != hi;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int tr = lane & 15, tc = lane >> 4;
  const int64_t bb = (int64_t)b * b;

  const bool is_node = item < nnodes * nsp;
  int z, parent, nid = -1, snd = -1;
  if (is_node) {
    nid = nnodes - 1 - item / nsp;
    int lv = 0, n = L, node0 = 0;  // level, live ranks and first node of nid's level
    while (nid >= node0 + n / 2) {
      node0 += n / 2;
      n = n / 2 + (n & 1);
      ++lv;
    }
    z = nid - node0;
    snd = z + (n + 1) / 2;
    parent = parent_node(z, lv, L);
  } else {
    z = item / nsp - nnodes;
    parent = parent_node(z, -1, L);
  }
  // ---- leaf z: rows [r0, r1) of V = [V\R] (unit lower in its top b×b)
  const int64_t r0 = ((int64_t)z * m) / L, r1 = ((int64_t)(z + 1) * m) / L;
  const int ml = (int)(r1 - r0);
  const double* Vl = V + r0;

  // Products X·y on FP64 MFMA tiles with the operands exchanged, yᵀ·Xᵀ: lane
  // l supplies X(l & 15, (l >> 4) + 4v) and receives the result's row (l & 15),
  // columns (l >> 4) + 4v of the strip.
  // Rows and columns past the ends are fetched from the last one in range: a
  // product's row past the end is dropped by put(), and a column past it meets
  // zeros.  Nothing looks at a fetched value before the parent's blocks are
  // there.  The address walks along k (a table of offsets would not fit the
  // registers).
  struct Walk {
    const double* q;
    int k;
  };
  auto walk_from = [&](const double* row, int k, int64_t cs) {
    k = min(k, b - 1);
    return Walk{row + k * cs, k};
  };
  auto walk4 = [&](Walk& p, int64_t cs, dbl4& x) {   // four steps of four columns
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      x[v] = *p.q;
      const bool in = p.k + 4 < b;
      p.q += in ? 4 * cs : 0;
      p.k += in ? 4 : 0;
    }
  };
  auto fetch9 = [&](const double* p, int64_t rs, int64_t cs, dbl4 (&x)[9]) {   // element (r, k) at r·rs + k·cs
    Walk q = walk_from(p + min(16 * w + tr, b - 1) * rs, 16 * w + tc, cs);
#pragma unroll
    for (int s = 0; s < 9; ++s) {
      if (s >= 5 && s == 8 - w) q = walk_from(p + min(16 * (7 - w) + tr, b - 1) * rs, 16 * (7 - w) + tc, cs);
      if (slot_col(s, w) <= hi) walk4(q, cs, x[s]);
    }
  };
  // out[0], out[1]: rows w and 7 − w of X·S, each for the wide and the narrow strip
  auto product9 = [&](const dbl4 (&x)[9], const double* S, dbl4 (&out)[2][2]) {
    const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
    const double* sp = S + tc * LD + tr;
    dbl4 h0 = zero, h1 = zero, l0 = zero;
#pragma unroll
    for (int s = 0; s < 9; ++s) {
      const int kt = slot_col(s, w);
      if (s >= 5 && s == 8 - w) {
        out[0][0] = h0 + h1;
        out[0][1] = l0;
        h0 = h1 = l0 = zero;
      }
      if (kt <= hi) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const double y = sp[(16 * kt + 4 * v) * LD];
          if (v & 1) h1 = __builtin_amdgcn_mfma_f64_16x16x4f64(y, x[s][v], h1, 0, 0, 0);
          else h0 = __builtin_amdgcn_mfma_f64_16x16x4f64(y, x[s][v], h0, 0, 0, 0);
        }
        if (two && kt <= lo)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const double y = sp[(128 + 16 * kt + 4 * v) * LD];
            l0 = __builtin_amdgcn_mfma_f64_16x16x4f64(y, x[s][v], l0, 0, 0, 0);
          }
      }
    }
    out[1][0] = h0 + h1;
    out[1][1] = l0;
  };
  // for the item's tiles (q: row w or 7 − w, j: wide or narrow strip)
  auto each_tile = [&](auto f) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int t = q ? 7 - w : w, strip = j ? lo : hi;
        if (t <= strip && (j == 0 || two)) f(q, j, t, strip);
      }
  };
  auto put = [&](double* S, int j, int t, const dbl4& x) {
#pragma unroll
    for (int v = 0; v < 4; ++v) S[(128 * j + 16 * t + tr) * LD + tc + 4 * v] = 16 * t + tr < b ? x[v] : 0.0;
  };

  auto get = [&](const double* S, int j, int t) {
    dbl4 x;
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] = S[(128 * j + 16 * t + tr) * LD + tc + 4 * v];
    return x;
  };
  // The strips of C_z (identity at the root) into S0 once the parent has
  // written them.
  double* Cz = C + (int64_t)z * bb;
  auto input = [&] {
    if (tid == 0) s_ok = parent < 0 || flag_wait(flags + (int64_t)parent * nsp + lo, epoch, wait_limit(err));
    __syncthreads();
    if (!s_ok) {
      if (tid == 0) *err = 1;
      return false;
    }
    dbl4 x[2][2];
    each_tile([&](int q, int j, int t, int strip) {
      const int row = 16 * t + tr;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int col = 16 * strip + tc + 4 * v;
        x[q][j][v] = row < b && col < b ? (parent >= 0 ? load_coherent(Cz + row + (int64_t)col * b) : (row == col ? 1.0 : 0.0))
                                        : 0.0;
      }
    });
    each_tile([&](int q, int j, int t, int) { put(S0, j, t, x[q][j]); });
    __syncthreads();
    return true;
  };
  dbl4 y[2][2];

  if (is_node) {
    dbl4 x0[9], x1[9];
    fetch9(nodeT + (int64_t)nid * bb, 1, b, x0);
    fetch9(nodeV2 + (int64_t)nid * bb, 1, b, x1);
    if (!input()) return;
    double* Cs = C + (int64_t)snd * bb;
    product9(x0, S0, y);   // X = T·C_z
    each_tile([&](int q, int j, int t, int) { put(S1, j, t, y[q][j]); });
    __syncthreads();
    each_tile([&](int q, int j, int t, int strip) {
      const dbl4 cz = get(S0, j, t) - y[q][j];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * t + tr, col = 16 * strip + tc + 4 * v;
        if (row < b && col < b) store_coherent(Cz + row + (int64_t)col * b, cz[v]);
      }
    });
    product9(x1, S1, y);
    each_tile([&](int q, int j, int t, int strip) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * t + tr, col = 16 * strip + tc + 4 * v;
        if (row < b && col < b) store_coherent(Cs + row + (int64_t)col * b, -y[q][j][v]);
      }
    });
    wait_memory();
    __syncthreads();
    if (tid == 0) flag_store(flags + (int64_t)nid * nsp + lo, epoch);
    return;
  }

  // V_l's tiles (t, 0..min(t, hi)) of 16 rows
  auto vrow = [&](int t, dbl4 (&x)[8]) {
    Walk q = walk_from(Vl + min(16 * t + tr, ml - 1), tc, ldv);
#pragma unroll
    for (int kt = 0; kt < 8; ++kt)
      if (kt <= hi && kt <= t) walk4(q, ldv, x[kt]);
  };
  // tile rows of wave w: w, 7 − w, then w + 8, w + 12, ...
  auto row_of = [&](int i) { return i == 0 ? w : i == 1 ? 7 - w : w + 4 * i; };
  dbl4 x0[9], x1[9], vt[8];
  fetch9(Vl, ldv, 1, x0);   // V_topᵀ
  fetch9(leafT + (int64_t)z * bb, 1, b, x1);
  if (!input()) return;
#pragma unroll
  for (int s = 0; s < 9; ++s)   // its diagonal tiles: unit upper
    if (s == 0 || (s >= 5 && s == 8 - w))
#pragma unroll
      for (int v = 0; v < 4; ++v) x0[s][v] = tc + 4 * v > tr ? x0[s][v] : (tc + 4 * v == tr ? 1.0 : 0.0);
  product9(x0, S0, y);   // Z = V_topᵀ·C_l
  each_tile([&](int q, int j, int t, int) { put(S1, j, t, y[q][j]); });
  __syncthreads();
  vrow(w, vt);
  product9(x1, S1, y);   // M = T_l·Z, in place of Z
  __syncthreads();
  each_tile([&](int q, int j, int t, int) { put(S1, j, t, y[q][j]); });
  __syncthreads();
  // Q1_l = [C_l; 0] − V_l·M over the leaf rows
  const double* sp = S1 + tc * LD + tr;
  const int nrow = (ml + 15) / 16;
  auto row_product = [&](int t, dbl4 (&x)[8]) {
    const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
    dbl4 h0 = zero, h1 = zero, l0 = zero;
#pragma unroll
    for (int kt = 0; kt < 8; ++kt)
      if (kt <= hi && kt <= t) {
        if (kt == t)   // unit lower
#pragma unroll
          for (int v = 0; v < 4; ++v) x[kt][v] = tc + 4 * v < tr ? x[kt][v] : (tc + 4 * v == tr ? 1.0 : 0.0);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const double a = -sp[(16 * kt + 4 * v) * LD];
          if (v & 1) h1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x[kt][v], h1, 0, 0, 0);
          else h0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x[kt][v], h0, 0, 0, 0);
        }
        if (two && kt <= lo)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const double a = -sp[(128 + 16 * kt + 4 * v) * LD];
            l0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x[kt][v], l0, 0, 0, 0);
          }
      }
    // C_l last: summed onto it (a value near 1 on the diagonal) the product
    // would round at its size in every step
    h0 += h1;
    if (t <= hi) h0 += get(S0, 0, t);
    if (two && t <= lo) l0 += get(S0, 1, t);
    const int row = 16 * t + tr;
    if (row < ml)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int ch = 16 * hi + tc + 4 * v, cl = 16 * lo + tc + 4 * v;
        if (ch < b) Q[r0 + row + (int64_t)ch * ldq] = h0[v];
        if (two) Q[r0 + row + (int64_t)cl * ldq] = l0[v];
      }
  };
  dbl4 vn[8];
#pragma unroll 1
  for (int i = 0; row_of(i) < nrow || i == 0; i += 2) {
    const int ta = row_of(i), tb = row_of(i + 1), tn = row_of(i + 2);
    if (tb < nrow) vrow(tb, vn);
    if (ta < nrow) row_product(ta, vt);
    if (tn < nrow) vrow(tn, vt);
    if (tb < nrow) row_product(tb, vn);
  }
}

int launch_q1(cqr_ctx* c, const double* nodeV2, const double* nodeT, const double* leafT, const double* V,
              int64_t ldv, int64_t m, double* C, double* Q, int64_t ldq, int L, int nnodes, int b) {
  if (b > 128 || b < 1) return set_err(c, CQR_ERR_UNSUPPORTED, "construct_Q1: b = %d", b);
  const int nb = (b + CW - 1) / CW;
  if ((int64_t)nnodes * nb > CQR_MAX_TREE_NODES * 8)
    return set_err(c, CQR_ERR_UNSUPPORTED, "construct_Q1: tree of %d nodes", nnodes);
  const uint64_t epoch = ++c->q1_epoch;
  hipEvent_t ev = prof_begin(c);
  const int64_t items = (int64_t)(nnodes + L) * ((nb + 1) / 2);
  {
    SpinScope gate(c, (const void*)q1_kernel, items, 64 * NWV, 0);
    CQR_TRY(gate.status());
    hipLaunchKernelGGL(q1_kernel, dim3((unsigned)items), dim3(64 * NWV), 0, c->stream, nodeV2, nodeT, leafT, V, ldv, m, C,
                       Q, ldq, c->d_qflags, epoch, L, nnodes, b, c->d_terr, nullptr, nullptr, 0);
  }
  prof_end(c, ev, PK_BGEMM, 4.0 * nnodes * (double)b * b * b + 4.0 * (double)m * b * b,
           8.0 * (3.0 * nnodes * b * b + 2.0 * m * b + 2.0 * L * b * b));
  return check_launch(c, "q1_kernel");
}

// Batched: every problem of a group, strips (total_items) in the order of the
// segment table (node levels from the top across all problems, then the leaves);
// flags must be zero before the launch (epoch 1, graph-replayable).
int launch_q1_batched(cqr_ctx* c, const double* nodeV2, const double* nodeT, const double* leafT, const double* Vbase,
                      double* C, double* Y, uint64_t* flags, int total_items, int b, const BatchProb* bp,
                      const BatchSeg* seg, int nseg) {
  if (total_items <= 0) return CQR_OK;
  const int nb = (b + CW - 1) / CW, blocks = total_items / nb * ((nb + 1) / 2);
  hipEvent_t ev = prof_begin(c);
  {
    SpinScope gate(c, (const void*)q1_kernel, blocks, 64 * NWV, 0);
    CQR_TRY(gate.status());
    hipLaunchKernelGGL(q1_kernel, dim3((unsigned)blocks), dim3(64 * NWV), 0, c->stream, nodeV2, nodeT, leafT, Vbase,
                       (int64_t)0, (int64_t)0, C, Y, (int64_t)0, flags, (uint64_t)1, 0, 0, b, c->d_terr, bp, seg, nseg);
  }
  prof_end(c, ev, PK_BGEMM, 0.0, 0.0);
  return check_launch(c, "q1_kernel_batched");
}

int q1_items_per_problem(int L, int b) { return (2 * L - 1) * ((b + CW - 1) / CW); }

}  // namespace cqr
