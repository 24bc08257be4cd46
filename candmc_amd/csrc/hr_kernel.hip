// Householder reconstruction core (alg/QR/hh_recon/hh_recon.cxx:43-111,
// 282-308) on sixteen-column strips: signed LU of the b×b block Q1_top − S,
// the inverses of its factors and every b×b product the panel needs, in one
// workgroup.
//
// Wave by wave the matrix is cut into 16-column strips held in registers as
// 16×16 tiles (lane l = 16g + c, value v of a tile: row 4g + v of column c),
// the layout a v_mfma_f64_16x16x4f64 result has when lane m of the left
// operand carries row 4(m & 3) + (m >> 2); such a tile is directly a right
// operand, its value v the k-slices 4g + v.  Left operands are read from
// 16×16 tiles in LDS.
//
// The LU goes like the leaf QR (ptree_kernel.hip): the strip's own wave
// factors its panel with the DPP row broadcast, one barrier later the next
// strip is updated first, then the others beside that panel.  The inverses
// need no more synchronisation: strip w of L⁻¹ (and of U⁻¹) depends on tiles
// of L (U) and the inverted diagonal tiles only,
//   X(t, w) = −L_tt⁻¹·Σ_{w≤j<t} L(t, j)·X(j, w),
// and so does strip w of Tᵀ = −L⁻¹·Wᵀ, whose tiles then are the right
// operands of U⁻¹·Tᵀ.
//
// Bound: the serial chain of b columns (one recip and one broadcast FMA per
// tile row each), then MFMA issue on one CU.  At b = 128 with Tᵀ and U⁻¹·Tᵀ
// 88–100 µs, b = 64 37 µs, b = 32 15 µs; the form before (8-column steps
// through LDS, in-place inverses one after the other) took 160–210, 75 and
// 47 µs and left T, T⁻ᵀ, and below b = 128 Tᵀ, U⁻¹·Tᵀ and the top rows of
// Y and Y·Tᵀ, to small products of 6–20 µs each.
#include "cqr_device.h"
#include "cqr_internal.h"
#include "panel16.h"

namespace cqr {

namespace {

constexpr int HT = P16_TILE;

// Row 4(m & 3) + (m >> 2) that lane m of a left operand carries.
__device__ __forceinline__ int perm16(int m) { return 4 * (m & 3) + (m >> 2); }

__device__ __forceinline__ dbl4 ht_load(const double* X, int lane) {
  const double* p = X + 4 * (lane >> 4) * P16_LD + (lane & 15);
  return dbl4{p[0], p[P16_LD], p[2 * P16_LD], p[3 * P16_LD]};
}
// the same of Xᵀ
__device__ __forceinline__ dbl4 ht_load_t(const double* X, int lane) {
  const double* p = X + (lane & 15) * P16_LD + 4 * (lane >> 4);
  return dbl4{p[0], p[1], p[2], p[3]};
}
__device__ __forceinline__ void ht_store(double* X, const dbl4& y, int lane) {
  double* p = X + 4 * (lane >> 4) * P16_LD + (lane & 15);
#pragma unroll
  for (int v = 0; v < 4; ++v) p[v * P16_LD] = y[v];
}
// acc + X·y
__device__ __forceinline__ dbl4 ht_mm(const double* X, const dbl4& y, dbl4 acc, int lane) {
  const double* p = X + perm16(lane & 15) * P16_LD + 4 * (lane >> 4);
#pragma unroll
  for (int v = 0; v < 4; ++v) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(p[v], y[v], acc, 0, 0, 0);
  return acc;
}
// acc + Xᵀ·y
__device__ __forceinline__ dbl4 ht_mmt(const double* X, const dbl4& y, dbl4 acc, int lane) {
  const double* p = X + 4 * (lane >> 4) * P16_LD + perm16(lane & 15);
#pragma unroll
  for (int v = 0; v < 4; ++v) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(p[v * P16_LD], y[v], acc, 0, 0, 0);
  return acc;
}
// X·y for the unit lower triangle of X (what lies on and above its diagonal is
// other data): y added to the strict triangle's product
__device__ __forceinline__ dbl4 ht_mm_unit(const double* X, const dbl4& y, int lane) {
  const int r = perm16(lane & 15), k0 = 4 * (lane >> 4);
  const double* p = X + r * P16_LD + k0;
  dbl4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const double x = p[v];
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(r > k0 + v ? x : 0.0, y[v], acc, 0, 0, 0);
  }
  return acc + y;
}

// One panel of the signed LU: RT tiles below the diagonal tile, whose rows
// are replicated in every lane group.
template <int RT>
struct LuPanel {
  static constexpr int RT1 = RT > 0 ? RT : 1;
  static constexpr int H = RT > 4 ? 4 : RT;
  double pr[P16];
  double rpl, sgl;     // lane c: reciprocal pivot and sign of column c

  template <int J, int T0, int T1>
  __device__ static __forceinline__ void axpys(dbl4 (&a)[RT1], double f) {
#pragma unroll
    for (int t = T0; t < T1; t += 2) {
      if (t + 1 < T1) p16_axpy2<J>(a[t], a[t + 1 < T1 ? t + 1 : t], f);
      else p16_axpy1<J>(a[t], f);
    }
  }
  template <int J>
  __device__ __forceinline__ void column(dbl4 (&a)[RT1], int nact) {
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n v_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lane), "+s"(nact));
    const int c = lane & 15;
    constexpr int N = P16 - 1 - J;
    const double p = pr[J], pv = readlane_d(p, J);
    const double sg = pv > 0.0 ? -1.0 : 1.0;
    const double piv = pv - sg, rp = recip_nr(piv);     // |piv| ≥ 1
    const double f = c > J ? -(p * rp) : 0.0;
#pragma unroll
    for (int q = 0; q + 4 <= N; q += 4) p16_axpyrows<J, 4>(pr + J + 1 + q, f);
    if constexpr (N % 4 != 0) p16_axpyrows<J, N % 4>(pr + P16 - N % 4, f);
    axpys<J, 0, H>(a, f);
    if constexpr (RT > H)
      if (__builtin_expect(nact > H, 1)) axpys<J, H, RT>(a, f);
    pr[J] = c == J ? piv : p;
    rpl = c == J ? rp : rpl;
    sgl = c == J ? sg : sgl;
  }

  // The panel with a masked update and true quotients, in LDS: the diagonal
  // tile in Ds, nt tiles from Bs, stride bst.
  __device__ static __forceinline__ void slow(double* Ds, double* Bs, int bst, int nt, int nb, double& rpl, double& sgl) {
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    auto sync = []() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup"); };
#pragma unroll 1
    for (int j = 0; j < nb; ++j) {
      const double u = Ds[j * P16_LD + c], pv = readlane_d(u, j);
      const double sg = pv > 0.0 ? -1.0 : 1.0, piv = pv - sg, rp = 1.0 / piv;
#pragma unroll 1
      for (int t = -1; t < nt; ++t)
#pragma unroll 1
        for (int v = 0; v < 4; ++v) {
          double* x = (t < 0 ? Ds : Bs + t * bst) + (4 * g + v) * P16_LD;
          if (t < 0 && 4 * g + v <= j) continue;
          const double l = x[j] * rp, old = x[c];
          sync();
          if (c == j) x[c] = l;
          else if (c > j) x[c] = old - l * u;
        }
      sync();
      if (g == 0 && c == j) Ds[j * P16_LD + j] = piv;
      if (c == j) {
        rpl = rp;
        sgl = sg;
      }
      sync();
    }
  }

  // Factors the first nb columns of (D; a), nact tiles of a nonzero: leaves
  // L\U of the diagonal tile in Ds and the scaled tiles of L in Bs (bst
  // doubles apart).
  __device__ __forceinline__ void factor(const dbl4& D, dbl4 (&a)[RT1], int nact, int nb, int lane, double* Ds, double* Bs,
                                         int bst) {
    const int c = lane & 15;
    rpl = sgl = 1.0;
    __builtin_amdgcn_sched_barrier(0);     // (see Panel16::factor)
    asm volatile("s_nop 15\n s_nop 15\n s_nop 15");
    __builtin_amdgcn_sched_barrier(0);
    ht_store(Ds, D, lane);
#pragma unroll
    for (int t = 0; t < RT; ++t)
      if (t < nact) ht_store(Bs + t * bst, a[t], lane);
#pragma unroll
    for (int q = 0; q < P16; ++q) pr[q] = Ds[q * P16_LD + c];
#define HR_STEP(J)              \
  asm volatile("" : "+s"(nb));  \
  if (J == 0 || __builtin_expect(J < nb, 1)) column<J>(a, nact);
    HR_STEP(0) HR_STEP(1) HR_STEP(2) HR_STEP(3) HR_STEP(4) HR_STEP(5) HR_STEP(6) HR_STEP(7)
    HR_STEP(8) HR_STEP(9) HR_STEP(10) HR_STEP(11) HR_STEP(12) HR_STEP(13) HR_STEP(14) HR_STEP(15)
#undef HR_STEP
    // a NaN or infinity anywhere in the panel, or a pivot too large for its
    // refined reciprocal: redo it without letting it reach the columns before
    // its own
    double chk = 0.0;
#pragma unroll
    for (int q = 0; q < P16; ++q) chk = fma(pr[q], 0.0, chk);
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) chk = fma(a[t][v], 0.0, chk);
    if (__builtin_amdgcn_ballot_w64(!(chk == 0.0 && fabs(rpl) > 0x1p-1000)) != 0) {
      slow(Ds, Bs, bst, max(nact, 0), nb, rpl, sgl);
#pragma unroll
      for (int q = 0; q < P16; ++q) pr[q] = Ds[q * P16_LD + c];
    } else {
#pragma unroll
      for (int t = 0; t < RT; ++t)
        if (t < nact) ht_store(Bs + t * bst, a[t] * rpl, lane);
#pragma unroll
      for (int q = 0; q < P16; ++q) {
        pr[q] = q > c ? pr[q] * rpl : pr[q];
        Ds[q * P16_LD + c] = pr[q];
      }
    }
  }

  // Column c of the inverse of the unit lower triangle of pr, and of its
  // upper triangle, by substitution; the matrix entry (R, Q) is broadcast
  // from lane Q of row R.
  template <int R, int Q = 0>
  __device__ __forceinline__ void lsum(double& acc, const double (&nx)[P16]) const {
    if constexpr (Q < R) {
      p16_fma_bc<Q>(acc, pr[R], nx[Q]);
      lsum<R, Q + 1>(acc, nx);
    }
  }
  template <int R = 0>
  __device__ __forceinline__ void linv(double (&nx)[P16], double* Li, int c) const {
    if constexpr (R < P16) {
      double acc = R == c ? 1.0 : 0.0;
      asm("s_nop 1" : "+v"(acc) : "v"(pr[R]));
      lsum<R>(acc, nx);
      nx[R] = -acc;
      Li[R * P16_LD] = R > c ? acc : pr[R];          // [L⁻¹ \ U] in one tile
      linv<R + 1>(nx, Li, c);
    }
  }
  template <int R, int Q = R + 1>
  __device__ __forceinline__ void usum(double& acc, const double (&nx)[P16]) const {
    if constexpr (Q < P16) {
      p16_fma_bc<Q>(acc, pr[R], nx[Q]);
      usum<R, Q + 1>(acc, nx);
    }
  }
  template <int R = P16 - 1>
  __device__ __forceinline__ void uinv(double (&nx)[P16], double* Ui, int c) const {
    if constexpr (R >= 0) {
      double acc = R == c ? 1.0 : 0.0;
      asm("s_nop 1" : "+v"(acc) : "v"(pr[R]));
      usum<R>(acc, nx);
      const double x = acc * readlane_d(rpl, R);
      nx[R] = -x;
      Ui[R * P16_LD] = R <= c ? x : 0.0;
      uinv<R - 1>(nx, Ui, c);
    }
  }
};

// LDS of a body of W strips: the W×W tiles of the matrix (diagonal tiles:
// U_kk⁻¹), W tiles [L_kk⁻¹ \ U_kk], the signs.
template <int W>
constexpr int hr_smem_doubles() { return (W * W + W) * HT + 16 * W; }

// The strip of wave w: on eight waves, strips s and 7 − s share a SIMD, so
// that the triangular products load the four SIMDs alike.
template <int W>
__device__ __forceinline__ int strip_of(int w) { return W == 8 && w >= 4 ? 11 - w : w; }

template <int W>
__device__ __forceinline__ double* hr_tile(double* smem, int i, int j) { return smem + (i * W + j) * HT; }

// Signed LU (b ≤ 16·W) of the block at src: L and U in the off-diagonal
// tiles, [L_kk⁻¹ \ U_kk] and U_kk⁻¹ per diagonal tile, signs in sgn.  Wave
// w returns its strip's diagonal tile L\U in D.
template <int W>
__device__ __forceinline__ void lu16(const double* src, int64_t ld, double* smem, double* sgn, int b, dbl4& D) {
  constexpr int RT = W - 1, RT1 = RT > 0 ? RT : 1;
  const int lane = threadIdx.x & 63, s = strip_of<W>(wave_id());
  const int c = lane & 15, g = lane >> 4;
  const int n = (b + P16 - 1) / P16, col = 16 * s + c;
  double* LI = smem + W * W * HT;
  dbl4 a[RT1], own = {0.0, 0.0, 0.0, 0.0};
  {
    const double* p = src + (int64_t)min(col, b - 1) * ld;
    dbl4 x[W];
#pragma unroll
    for (int t = 0; t < W; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) x[t][v] = p[min(16 * t + 4 * g + v, b - 1)];
#pragma unroll
    for (int t = 0; t < W; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) x[t][v] = col < b && 16 * t + 4 * g + v < b ? x[t][v] : 0.0;
    D = x[0];
#pragma unroll
    for (int t = 0; t < RT; ++t) a[t] = x[t + 1];
  }
  for (int k = 0; k < n; ++k) {
    const int nact = n - 1 - k;
    LuPanel<RT> P;
    if (s == k) {
      __builtin_amdgcn_s_setprio(3);
      P.factor(D, a, nact, min(P16, b - 16 * k), lane, hr_tile<W>(smem, k, k), hr_tile<W>(smem, k + 1, k), W * HT);
      double nx[P16];
      P.linv(nx, LI + k * HT + c, c);
      __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
    auto apply = [&]() {
      const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
      const dbl4 u = ht_mm_unit(LI + k * HT, D, lane);
      ht_store(hr_tile<W>(smem, k, s), u, lane);
#pragma unroll
      for (int t = 0; t < RT; ++t)
        if (t < nact) a[t] -= ht_mm(hr_tile<W>(smem, k + 1 + t, k), u, zero, lane);
    };
    if (k + 1 < n) {   // the next strip first, alone (see leaf16_body)
      if (s == k + 1) apply();
      __syncthreads();
      if (s > k + 1 && s < n) apply();
    }
    if (s == k) {
      own = ht_load(hr_tile<W>(smem, k, k), lane);
      if (g == 0) sgn[col] = P.sgl;
      double nx[P16];
      P.uinv(nx, hr_tile<W>(smem, k, k) + c, c);
    } else {
      D = a[0];
#pragma unroll
      for (int t = 0; t + 1 < RT; ++t) a[t] = a[t + 1];
    }
  }
  D = own;
  __syncthreads();
}

// A column strip of a b×b result in memory, tile by tile; op is applied to
// each value with its row and column.
struct Strip {
  double* p;      // column start (row 0) of this lane
  int g4, b;
  bool ok;
  __device__ Strip(double* M, int64_t ld, int s, int b_, int lane)
      : p(M ? M + (int64_t)min(16 * s + (lane & 15), b_ - 1) * ld : nullptr), g4(4 * (lane >> 4)), b(b_),
        ok(16 * s + (lane & 15) < b_) {}
  __device__ void put(int t, const dbl4& x) const {
    if (!ok) return;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (16 * t + g4 + v < b) p[16 * t + g4 + v] = x[v];
  }
};
// Tile (i, j) of a result given transposed (rows from lanes, columns 4g + v).
__device__ __forceinline__ void put_transposed(double* M, int64_t ld, int b, int i, int j, const dbl4& x, int lane) {
  const int row = 16 * i + (lane & 15), col = 16 * j + 4 * (lane >> 4);
#pragma unroll
  for (int v = 0; v < 4; ++v)
    if (row < b && col + v < b) M[row + (col + v) * ld] = x[v];
}

struct HrArgs {
  const double* Q1top;
  int64_t ldq;
  const double* Rroot;
  double* Atop;        // L below the diagonal, S·R on and above it
  int64_t lda;
  double* W;           // W = U·S
  double* Uinv;        // U⁻¹, zeros below the diagonal
  int64_t* signs;
  double* Tt;          // Tᵀ = −L⁻¹·Wᵀ
  double* T;
  double* invTT;       // T⁻ᵀ = −W⁻ᵀ·L (needs Uinv)
  double* M2;          // U⁻¹·Tᵀ (needs Tt)
  double* Ye;          // top rows of the explicit Y and of Y·Tᵀ = −Wᵀ there
  double* YT;
  int64_t ldy;
  int b;
};

}  // namespace

// Everything but Q1top, Rroot, Atop and W may be null; M2 needs Tt and Uinv,
// invTT needs Uinv (U⁻¹'s tiles are formed for it only).
template <int W>
__device__ __forceinline__ void hr16_body(const HrArgs& h, double* smem) {
  const int lane = threadIdx.x & 63, s = strip_of<W>(wave_id());
  const int c = lane & 15, g = lane >> 4, b = h.b;
  const int n = (b + P16 - 1) / P16;
  const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
  double* LI = smem + W * W * HT;
  double* sgn = LI + W * HT;
  dbl4 D;
  lu16<W>(h.Q1top, h.ldq, smem, sgn, b, D);
  const bool act = s < n;
  const bool tri = h.Tt || h.T || h.M2;
  const Strip oA(h.Atop, h.lda, s, b, lane), oW(h.W, b, s, b, lane), oU(h.Uinv, b, s, b, lane),
      oE(h.Ye, h.ldy, s, b, lane), oY(h.YT, h.ldy, s, b, lane);
  const double sc = act ? sgn[16 * s + c] : 1.0;

  // x[d] = L⁻¹(s + d, s), y[d] = U⁻¹(s − d, s)
  dbl4 x[W], y[W];
#pragma unroll
  for (int d = 0; d < W; ++d) x[d] = y[d] = zero;
  if (act) {
    if (h.signs && g == 0 && 16 * s + c < b) h.signs[16 * s + c] = (int64_t)sc;
    // R's strip, in flight under the products below
    dbl4 r[W];
    {
      const double* p = h.Rroot + (int64_t)min(16 * s + c, b - 1) * b;
#pragma unroll
      for (int t = 0; t < W; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) r[t][v] = t <= s ? p[min(16 * t + 4 * g + v, b - 1)] : 0.0;
    }
    if (tri) {
      const dbl4 l = ht_load(LI + s * HT, lane);
#pragma unroll
      for (int v = 0; v < 4; ++v) x[0][v] = 4 * g + v > c ? l[v] : (4 * g + v == c ? 1.0 : 0.0);
#pragma unroll
      for (int d = 1; d < W; ++d)
        if (s + d < n) {
          dbl4 acc = zero;
#pragma unroll
          for (int e = 0; e < d; ++e) acc = ht_mm(hr_tile<W>(smem, s + d, s + e), x[e], acc, lane);
          x[d] = -ht_mm_unit(LI + (s + d) * HT, acc, lane);
        }
    }
    if (h.Uinv) {
      y[0] = ht_load(hr_tile<W>(smem, s, s), lane);
#pragma unroll
      for (int d = 1; d < W; ++d)
        if (d <= s) {
          dbl4 acc = zero;
#pragma unroll
          for (int e = 0; e < d; ++e) acc = ht_mm(hr_tile<W>(smem, s - d, s - e), y[e], acc, lane);
          y[d] = -ht_mm(hr_tile<W>(smem, s - d, s - d), acc, zero, lane);
        }
#pragma unroll
      for (int d = 0; d < W; ++d)
        if (d <= s) oU.put(s - d, y[d]);
      for (int t = s + 1; t < n; ++t) oU.put(t, zero);
    }
    // [L \ S·R], W, the explicit Y's top
#pragma unroll
    for (int t = 0; t < W; ++t)
      if (t < n) {
        dbl4 l = zero, u = zero, av, ev;
        if (t < s) u = ht_load(hr_tile<W>(smem, t, s), lane);
        if (t > s) l = ht_load(hr_tile<W>(smem, t, s), lane);
        if (t == s) l = u = D;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const bool low = t > s || (t == s && 4 * g + v > c);
          const double sr = 4 * g + v + 16 * t < b ? sgn[16 * t + 4 * g + v] : 1.0;
          av[v] = low ? l[v] : sr * r[t][v];
          ev[v] = low ? l[v] : (t == s && 4 * g + v == c ? 1.0 : 0.0);
          u[v] = low ? 0.0 : u[v] * sc;
        }
        oA.put(t, av);
        oW.put(t, u);
        if (h.Ye) oE.put(t, ev);
      }
  }
  if (!tri && !h.invTT) return;
  // wt[d] = Wᵀ(s + d, s), the strip's right operands
  dbl4 wt[W];
#pragma unroll
  for (int d = 0; d < W; ++d) {
    wt[d] = zero;
    if (act && s + d < n) {
      wt[d] = ht_load_t(d == 0 ? LI + s * HT : hr_tile<W>(smem, s, s + d), lane);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * (s + d) + 4 * g + v;
        wt[d][v] = (d > 0 || 4 * g + v >= c) && row < b ? wt[d][v] * sgn[row] : 0.0;
      }
      if (h.YT) oY.put(s + d, -wt[d]);
    }
  }
  if (h.YT && act)
    for (int t = 0; t < s; ++t) oY.put(t, zero);
  __syncthreads();                       // every wave is done with L and U
  dbl4 tt[W];
#pragma unroll
  for (int d = 0; d < W; ++d) tt[d] = zero;
  if (tri) {
    if (act)
#pragma unroll
      for (int d = 1; d < W; ++d)
        if (s + d < n) ht_store(hr_tile<W>(smem, s + d, s), x[d], lane);
    __syncthreads();
    if (act) {
#pragma unroll
      for (int d = 0; d < W; ++d)
        if (s + d < n) {
          dbl4 acc = ht_mm_unit(LI + (s + d) * HT, wt[d], lane);
#pragma unroll
          for (int e = 0; e < d; ++e) acc = ht_mm(hr_tile<W>(smem, s + d, s + e), wt[e], acc, lane);
          tt[d] = -acc;
        }
      const Strip oT(h.Tt, b, s, b, lane);
#pragma unroll
      for (int d = 0; d < W; ++d)
        if (s + d < n) {
          if (h.Tt) oT.put(s + d, tt[d]);
          if (h.T) put_transposed(h.T, b, b, s, s + d, tt[d], lane);
        }
      for (int t = 0; t < s; ++t) {
        if (h.Tt) oT.put(t, zero);
        if (h.T) put_transposed(h.T, b, b, s, t, zero, lane);
      }
    }
  }
  if (!h.M2 && !h.invTT) return;
  if (act)
#pragma unroll
    for (int d = 1; d < W; ++d)
      if (d <= s) ht_store(hr_tile<W>(smem, s - d, s), y[d], lane);
  __syncthreads();
  if (!act) return;
  if (h.M2) {
    const Strip oM(h.M2, b, s, b, lane);
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
      dbl4 acc = zero;
#pragma unroll
      for (int e = 0; e < W; ++e)
        if (s + e < n && s + e >= i) acc = ht_mm(hr_tile<W>(smem, i, s + e), tt[e], acc, lane);
      oM.put(i, acc);
    }
  }
  if (h.invTT) {
    // T⁻ᵀ(i, s) = −Σ_{s≤k≤i} U⁻¹(k, i)ᵀ·S_k·L(k, s); L's strip as this wave
    // wrote it to Atop (and D)
    dbl4 l[W];
#pragma unroll
    for (int d = 0; d < W; ++d) {
      l[d] = zero;
      if (s + d < n)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * (s + d) + 4 * g + v;
          double val = d == 0 ? (4 * g + v > c ? D[v] : (4 * g + v == c ? 1.0 : 0.0)) : 0.0;
          if (d > 0 && row < b && oA.ok) val = oA.p[row];
          l[d][v] = row < b ? val * sgn[row] : 0.0;
        }
    }
    const Strip oI(h.invTT, b, s, b, lane);
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
      dbl4 acc = zero;
#pragma unroll
      for (int e = 0; e < W; ++e)
        if (s + e <= i && s + e < n) acc = ht_mmt(hr_tile<W>(smem, s + e, i), l[e], acc, lane);
      oI.put(i, -acc);
    }
  }
}

template <int W>
__global__ void __launch_bounds__(64 * W) hr_core_kernel(HrArgs h) {
  extern __shared__ double smem[];
  hr16_body<W>(h, smem);
}

// Batched: workgroup p handles problem p (its Q1 top in Y, its root R).
template <int W>
__global__ void __launch_bounds__(64 * W)
hr_core_batched_kernel(const BatchProb* __restrict__ bp, const double* __restrict__ Y, const double* __restrict__ leafR,
                       const double* __restrict__ nodeR, double* __restrict__ Abase, double* __restrict__ Wm,
                       double* __restrict__ Uinv, double* __restrict__ Tt, int b) {
  extern __shared__ double smem[];
  const BatchProb P = bp[blockIdx.x];
  const int64_t bb = (int64_t)b * b, p = blockIdx.x;
  HrArgs h{};
  h.Q1top = Y + P.yoff;
  h.ldq = P.m;
  h.Rroot = P.L > 1 ? nodeR + (int64_t)(P.node0 + P.L - 2) * bb : leafR + (int64_t)P.leaf0 * bb;
  h.Atop = Abase + P.aoff;
  h.lda = P.m;
  h.W = Wm + p * bb;
  h.Uinv = Uinv + p * bb;
  h.Tt = Tt + P.toff;
  h.b = b;
  hr16_body<W>(h, smem);
}

// a5 standalone: signed LU of a b×b block with R scaling.
template <int W>
__global__ void __launch_bounds__(64 * W)
signed_nlu_kernel(double* A, int64_t lda, double* __restrict__ R, int64_t ldr, int64_t* __restrict__ signs, int b) {
  extern __shared__ double smem[];
  double* sgn = smem + (W * W + W) * HT;
  dbl4 D;
  lu16<W>(A, lda, smem, sgn, b, D);
  const int lane = threadIdx.x & 63, s = strip_of<W>(wave_id()), n = (b + P16 - 1) / P16;
  const int c = lane & 15, g = lane >> 4, col = 16 * s + c;
  if (s >= n) return;
  const Strip oA(A, lda, s, b, lane);
  for (int t = 0; t < n; ++t) oA.put(t, t == s ? D : ht_load(hr_tile<W>(smem, t, s), lane));
  if (signs && g == 0 && col < b) signs[col] = (int64_t)sgn[col];
  if (R && col < b)
    for (int row = g; row <= col; row += 4)
      if (sgn[row] < 0) R[row + col * ldr] = -R[row + col * ldr];
}

template <int W>
static int hr_core_launch(cqr_ctx* c, const HrArgs& h) {
  const size_t lds = sizeof(double) * hr_smem_doubles<W>();
  CQR_TRY(set_max_lds(c, (const void*)hr_core_kernel<W>, (int)lds));
  hipLaunchKernelGGL(hr_core_kernel<W>, dim3(1), dim3(64 * W), lds, c->stream, h);
  return CQR_OK;
}

int hr_core(cqr_ctx* c, const HrCore& a) {
  const int b = a.b;
  if (b < 1 || b > 128) return set_err(c, CQR_ERR_UNSUPPORTED, "hr_core: b = %d", b);
  if (a.M2 && !(a.Tt && a.Uinv)) return set_err(c, CQR_ERR_INVALID, "hr_core: M2 needs Tt and Uinv");
  if (a.invTT && !a.Uinv) return set_err(c, CQR_ERR_INVALID, "hr_core: invTT needs Uinv");
  HrArgs h{};
  h.Q1top = a.Q1top; h.ldq = a.ldq; h.Rroot = a.Rroot; h.Atop = a.Atop; h.lda = a.lda; h.W = a.W; h.Uinv = a.Uinv;
  h.signs = a.signs; h.Tt = a.Tt; h.T = a.T; h.invTT = a.invTT; h.M2 = a.M2; h.Ye = a.Ye; h.YT = a.YT; h.ldy = a.ldy;
  h.b = b;
  hipEvent_t ev = prof_begin(c);
  if (b <= 16) CQR_TRY(hr_core_launch<1>(c, h));
  else if (b <= 32) CQR_TRY(hr_core_launch<2>(c, h));
  else if (b <= 64) CQR_TRY(hr_core_launch<4>(c, h));
  else CQR_TRY(hr_core_launch<8>(c, h));
  const double bbb = (double)b * b * b;
  prof_end(c, ev, PK_HR, (2.0 / 3.0) * bbb + (a.Tt ? bbb / 3.0 : 0.0) + (a.M2 ? bbb : 0.0), 64.0 * b * b);
  return check_launch(c, "hr_core");
}

template <int W>
static int hr_batched_launch(cqr_ctx* c, const BatchProb* bp, int nprob, const double* Y, const double* leafR,
                             const double* nodeR, double* Abase, double* Wm, double* Uinv, double* Tt, int b) {
  const size_t lds = sizeof(double) * hr_smem_doubles<W>();
  CQR_TRY(set_max_lds(c, (const void*)hr_core_batched_kernel<W>, (int)lds));
  hipLaunchKernelGGL(hr_core_batched_kernel<W>, dim3(nprob), dim3(64 * W), lds, c->stream, bp, Y, leafR, nodeR, Abase,
                     Wm, Uinv, Tt, b);
  return CQR_OK;
}

int hr_core_batched(cqr_ctx* c, const BatchProb* bp, int nprob, const double* Y, const double* leafR,
                    const double* nodeR, double* Abase, double* Wm, double* Uinv, double* Tt, int b) {
  if (b < 1 || b > 128) return set_err(c, CQR_ERR_UNSUPPORTED, "hr_core_batched: b = %d", b);
  hipEvent_t ev = prof_begin(c);
  if (b <= 16) CQR_TRY(hr_batched_launch<1>(c, bp, nprob, Y, leafR, nodeR, Abase, Wm, Uinv, Tt, b));
  else if (b <= 32) CQR_TRY(hr_batched_launch<2>(c, bp, nprob, Y, leafR, nodeR, Abase, Wm, Uinv, Tt, b));
  else if (b <= 64) CQR_TRY(hr_batched_launch<4>(c, bp, nprob, Y, leafR, nodeR, Abase, Wm, Uinv, Tt, b));
  else CQR_TRY(hr_batched_launch<8>(c, bp, nprob, Y, leafR, nodeR, Abase, Wm, Uinv, Tt, b));
  prof_end(c, ev, PK_HR, nprob * (2.0 / 3.0) * b * (double)b * b, nprob * 64.0 * b * b);
  return check_launch(c, "hr_core_batched");
}

template <int W>
static int nlu_launch(cqr_ctx* c, double* A, int64_t lda, double* R, int64_t lda_R, int64_t* signs, int b) {
  const size_t lds = sizeof(double) * hr_smem_doubles<W>();
  CQR_TRY(set_max_lds(c, (const void*)signed_nlu_kernel<W>, (int)lds));
  hipLaunchKernelGGL(signed_nlu_kernel<W>, dim3(1), dim3(64 * W), lds, c->stream, A, lda, R, lda_R, signs, b);
  return check_launch(c, "signed_nlu");
}

int launch_signed_nlu(cqr_ctx* c, double* A, int64_t lda, double* R, int64_t lda_R, int64_t* signs, int b) {
  if (b <= 16) return nlu_launch<1>(c, A, lda, R, lda_R, signs, b);
  if (b <= 32) return nlu_launch<2>(c, A, lda, R, lda_R, signs, b);
  if (b <= 64) return nlu_launch<4>(c, A, lda, R, lda_R, signs, b);
  return nlu_launch<8>(c, A, lda, R, lda_R, signs, b);
}

}  // namespace cqr
