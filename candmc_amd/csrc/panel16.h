// Sixteen-column panel steps shared by the leaf QR and the tree nodes.
//
// One wave holds a 16-column strip of the matrix as 16×16 tiles in the
// layout of a v_mfma_f64_16x16x4f64 result: lane l, value v of a tile holds
// tile row "i = (l >> 4) + 4v" of column l & 15.  A tile in this layout is
// directly the B operand of the next product (value v is its k-slice v), so
// the strip never leaves its registers.  Which matrix row tile row i stands
// for is free as long as every tile of a launch agrees: `PERM` strips map
// (g = l >> 4, v) to row 4g + v, so that a lane's four values are 32
// contiguous bytes of a column; the pivot tiles of tree nodes use i itself.
//
// The panel is factored by the wave that owns its strip, without LDS and
// without barriers: in a column step every lane needs column jj's value of
// its own row, which the DPP row broadcast of v_fmac_f64_dpp supplies for
// free, so the sixteen dot products x·a_c (‖x‖² among them) and the rank-1
// update are one FMA per value.  (Measured on gfx950: the broadcast FMA
// issues in 4 cycles, as the plain one does.)
#pragma once

#include "cqr_device.h"

namespace cqr {

constexpr int P16 = 16;               // panel width
constexpr int P16_LD = 17;            // pitch of a 16×16 tile in LDS (row-major)
constexpr int P16_TILE = 16 * P16_LD;

// The tile stored row-major in LDS, in tile layout, and back.
__device__ __forceinline__ dbl4 p16_load(const double* __restrict__ X, int lane) {
  const double* xp = X + (lane >> 4) * P16_LD + (lane & 15);
  return dbl4{xp[0], xp[4 * P16_LD], xp[8 * P16_LD], xp[12 * P16_LD]};
}
__device__ __forceinline__ void p16_store(double* __restrict__ X, const dbl4& y, int lane) {
  double* xp = X + (lane >> 4) * P16_LD + (lane & 15);
#pragma unroll
  for (int v = 0; v < 4; ++v) xp[4 * v * P16_LD] = y[v];
}

typedef double dbl2a __attribute__((ext_vector_type(2), aligned(8)));

// Four rows p[0..3] of a column, of which `left` exist.
__device__ __forceinline__ dbl4 p16_rows_load(const double* p, int left, bool ok) {
  if (ok && left >= 4) {
    const dbl2a lo = *reinterpret_cast<const dbl2a*>(p), hi = *reinterpret_cast<const dbl2a*>(p + 2);
    return dbl4{lo[0], lo[1], hi[0], hi[1]};
  }
  dbl4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int v = 0; v < 4; ++v)
    if (ok && v < left) x[v] = p[v];
  return x;
}
__device__ __forceinline__ void p16_rows_store(double* p, const dbl4& x, int left, bool ok) {
  if (!ok) return;
  if (left >= 4) {
    *reinterpret_cast<dbl2a*>(p) = dbl2a{x[0], x[1]};
    *reinterpret_cast<dbl2a*>(p + 2) = dbl2a{x[2], x[3]};
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (v < left) p[v] = x[v];
  }
}

// s[v] += x_t[v](column J)·x_t[v] over four tiles.  The leading s_nop covers
// the two wait states a DPP source needs after a VALU write.
template <int J>
__device__ __forceinline__ void p16_dot4(double (&s)[4], const dbl4& a, const dbl4& b, const dbl4& c, const dbl4& d) {
  asm("s_nop 1\n"
      "v_fmac_f64_dpp %0, %4, %4 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %5, %5 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %6, %6 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %7, %7 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %8, %8 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %9, %9 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %10, %10 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %11, %11 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %12, %12 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %13, %13 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %14, %14 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %15, %15 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %16, %16 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %17, %17 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %18, %18 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %19, %19 row_newbcast:%20 row_mask:0xf bank_mask:0xf"
      : "+&v"(s[0]), "+&v"(s[1]), "+&v"(s[2]), "+&v"(s[3])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]), "v"(c[0]), "v"(c[1]),
        "v"(c[2]), "v"(c[3]), "v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]), "n"(J));
}

// N rows of the pivot tile (N ≤ 4): s[v & 1] += x_v(column J)·x_v, and
// x_v += x_v(column J)·f.
#define P16_BC " row_newbcast:%c[j] row_mask:0xf bank_mask:0xf\n"
template <int J, int N>
__device__ __forceinline__ void p16_dotrows(double (&s)[2], const double* x) {
  if constexpr (N == 1)
    asm("s_nop 1\n v_fmac_f64_dpp %0, %2, %2" P16_BC : "+&v"(s[0]), "+&v"(s[1]) : "v"(x[0]), [j] "n"(J));
  else if constexpr (N == 2)
    asm("s_nop 1\n v_fmac_f64_dpp %0, %2, %2" P16_BC "v_fmac_f64_dpp %1, %3, %3" P16_BC
        : "+&v"(s[0]), "+&v"(s[1]) : "v"(x[0]), "v"(x[1]), [j] "n"(J));
  else if constexpr (N == 3)
    asm("s_nop 1\n v_fmac_f64_dpp %0, %2, %2" P16_BC "v_fmac_f64_dpp %1, %3, %3" P16_BC "v_fmac_f64_dpp %0, %4, %4" P16_BC
        : "+&v"(s[0]), "+&v"(s[1]) : "v"(x[0]), "v"(x[1]), "v"(x[2]), [j] "n"(J));
  else
    asm("s_nop 1\n v_fmac_f64_dpp %0, %2, %2" P16_BC "v_fmac_f64_dpp %1, %3, %3" P16_BC "v_fmac_f64_dpp %0, %4, %4" P16_BC
        "v_fmac_f64_dpp %1, %5, %5" P16_BC
        : "+&v"(s[0]), "+&v"(s[1]) : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), [j] "n"(J));
}
template <int J, int N>
__device__ __forceinline__ void p16_axpyrows(double* x, double f) {
  if constexpr (N == 1)
    asm("s_nop 1\n v_fmac_f64_dpp %0, %0, %[f]" P16_BC : "+&v"(x[0]) : [f] "v"(f), [j] "n"(J));
  else if constexpr (N == 2)
    asm("s_nop 1\n v_fmac_f64_dpp %0, %0, %[f]" P16_BC "v_fmac_f64_dpp %1, %1, %[f]" P16_BC
        : "+&v"(x[0]), "+&v"(x[1]) : [f] "v"(f), [j] "n"(J));
  else if constexpr (N == 3)
    asm("s_nop 1\n v_fmac_f64_dpp %0, %0, %[f]" P16_BC "v_fmac_f64_dpp %1, %1, %[f]" P16_BC "v_fmac_f64_dpp %2, %2, %[f]" P16_BC
        : "+&v"(x[0]), "+&v"(x[1]), "+&v"(x[2]) : [f] "v"(f), [j] "n"(J));
  else
    asm("s_nop 1\n v_fmac_f64_dpp %0, %0, %[f]" P16_BC "v_fmac_f64_dpp %1, %1, %[f]" P16_BC "v_fmac_f64_dpp %2, %2, %[f]" P16_BC
        "v_fmac_f64_dpp %3, %3, %[f]" P16_BC
        : "+&v"(x[0]), "+&v"(x[1]), "+&v"(x[2]), "+&v"(x[3]) : [f] "v"(f), [j] "n"(J));
}

// a[v] += a[v](column J)·f (one tile in place)
template <int J>
__device__ __forceinline__ void p16_axpy1(dbl4& a, double f) {
  double a0 = a[0], a1 = a[1], a2 = a[2], a3 = a[3];
  asm("s_nop 1\n"
      "v_fmac_f64_dpp %0, %0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
      : "+&v"(a0), "+&v"(a1), "+&v"(a2), "+&v"(a3)
      : "v"(f), "n"(J));
  a = dbl4{a0, a1, a2, a3};
}

// a[v] += a[v](column J)·f, b likewise (two tiles in place).
template <int J>
__device__ __forceinline__ void p16_axpy2(dbl4& a, dbl4& b, double f) {
  double a0 = a[0], a1 = a[1], a2 = a[2], a3 = a[3], b0 = b[0], b1 = b[1], b2 = b[2], b3 = b[3];
  asm("s_nop 1\n"
      "v_fmac_f64_dpp %0, %0, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %1, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %2, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %3, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %4, %4, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %5, %5, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %6, %6, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %7, %7, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
      : "+&v"(a0), "+&v"(a1), "+&v"(a2), "+&v"(a3), "+&v"(b0), "+&v"(b1), "+&v"(b2), "+&v"(b3)
      : "v"(f), "n"(J));
  a = dbl4{a0, a1, a2, a3};
  b = dbl4{b0, b1, b2, b3};
}

// acc += z(lane C of the row)·t
template <int C>
__device__ __forceinline__ void p16_fma_bc(double& acc, double z, double t) {
  asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+&v"(acc) : "v"(z), "v"(t), "n"(C));
}

// sqrt and the two reciprocals of dlarfg for ss = ‖x‖² above 2^-960 and
// alpha² + ss below overflow (tau is NaN beyond it): beta =
// −sign(alpha)·sqrt(alpha² + ss) by the Goldschmidt iteration from the
// hardware's reciprocal square root with two residual corrections; no operand
// scaling is needed in this range (the residual g² − x is a multiple of
// 2^-1064, and 1/beta at most 2^480).
__device__ __forceinline__ void p16_larfg(double alpha, double ss, double& beta, double& tau, double& scal, double& rb) {
  const double x = fma(alpha, alpha, ss);
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  h = fma(h, r, h);
  g = fma(g, r, g);
  g = fma(fma(-g, g, x), h, g);
  g = fma(fma(-g, g, x), h, g);
  beta = -copysign(g, alpha);
  // 1/beta from the refined reciprocal root h ≈ 1/(2g)
  double q = h + h;
  q = fma(q, fma(-g, q, 1.0), q);
  rb = copysign(q, beta);
  scal = recip_nr(alpha - beta);
  tau = (beta - alpha) * rb;
}

// One panel: RT tiles below the pivot tile, the pivot tile's sixteen rows
// (row q of every column, the same in all four lane groups), and per lane
// (column c = lane & 15) its reflector's tau and the scale still to be
// applied to its vector.
//   NODE = false: the pivot tile's rows below the diagonal belong to the
//     reflectors (a leaf; tile rows map as 4g + v).
//   NODE = true:  the pivot tile is the top triangle of a stacked pair: a
//     reflector is [e_jj; x] and only row jj takes part (rows map as g + 4v).
// LDS: Zs, a 16×16 tile whose row J receives −tau_J·v_qᵀv_J (q < J) and in
// the end the panel's compact-WY T, transposed; Vs (RT tiles), where the
// strip is kept for slow() and the scaled vectors are left; Ds (one
// tile), the pivot tile before and after.
// With PARTS > 1 a leaf's panel is spread over as many waves, `part` of them
// this one, all with RT tiles and one more, the pivot tile in part 0 and an
// ordinary one in the others (its values then live in pr[0..3]; Ds is its
// place in Vs).  Each part publishes its share of a column's dot products in
// `ex` (p16_ex_doubles: two buffers of PARTS + 1 rows of sixteen, the last one
// the pivot row, then slow()'s), and after a workgroup barrier all of them form
// the same reflector.  Other strips' waves meet these barriers by count; where
// more of them follow (zero columns, slow()), the word p16_more of `ex` says so,
// and ends at 0 for the barrier that publishes the panel.
//
// With GLOB (a leaf of one strip) nobody else reads the vectors: the tiles stay
// in registers, scaled in place, and slow() works on the leaf in memory, which
// still holds the strip; col is this part's first row of this lane's column, of
// which it has `rows` rows (none past the matrix's last column).
constexpr int p16_more(int parts) { return 2 * P16 * (parts + 1) + 2 * P16 * (2 * parts + 1); }   // (two words, taken in turn)
constexpr int p16_ex_doubles(int parts) { return p16_more(parts) + 2; }

template <int RT, bool NODE, int PARTS = 1, bool GLOB = false>
struct Panel16 {
  double* ex = nullptr;
  int part = 0;
  double* col = nullptr;
  int rows = 0;
  // the tiles [H, RT) are skipped as a whole once they are zero (never in a
  // tall leaf, whose parts stay full)
  static constexpr int H = PARTS > 1 ? RT : RT > 8 ? 8 : RT > 4 ? 4 : RT;
  double pr[P16];          // pivot rows
  double tau, scale;
  uint32_t ssmin;          // the smallest high word of a column's ‖x‖² (see factor()), less one

  // part ≠ 0, opaque as nact in column()
  __device__ __forceinline__ bool low() const {
    int p = part;
    asm volatile("" : "+s"(p));
    return p != 0;
  }
  // tile row that holds matrix row q of the pivot tile
  __device__ static constexpr int trow_of(int q) { return NODE ? q : (q >> 2) + 4 * (q & 3); }

  template <int J, int T0, int T1>
  __device__ static __forceinline__ void dots(double (&s4)[4], const dbl4 (&a)[RT]) {
    const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = T0; t < T1; t += 4)
      p16_dot4<J>(s4, a[t], t + 1 < T1 ? a[t + 1 < T1 ? t + 1 : 0] : zero, t + 2 < T1 ? a[t + 2 < T1 ? t + 2 : 0] : zero,
                  t + 3 < T1 ? a[t + 3 < T1 ? t + 3 : 0] : zero);
  }
  template <int J, int T0, int T1>
  __device__ static __forceinline__ void axpys(dbl4 (&a)[RT], double f) {
#pragma unroll
    for (int t = T0; t < T1; t += 2) {
      if (t + 1 < T1) p16_axpy2<J>(a[t], a[t + 1 < T1 ? t + 1 : t], f);
      else p16_axpy1<J>(a[t], f);
    }
  }

  // Column J.  Exact in the fast range (checked for all columns at the end:
  // outside it the panel is redone by slow()).
  template <int J>
  __device__ __forceinline__ void column(dbl4 (&a)[RT], int nact, double* __restrict__ Zc) {
    // an opaque copy: the code is not duplicated per number of active tiles,
    // and no lane mask lives across columns
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n v_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lane), "+s"(nact));
    const int c = lane & 15;
    constexpr int N = P16 - 1 - J;              // pivot rows below row J
    double s4[4] = {0.0, 0.0, 0.0, 0.0}, d2[2] = {0.0, 0.0};
    dots<J, 0, H>(s4, a);
    if constexpr (RT > H)
      if (__builtin_expect(nact > H, 1)) dots<J, H, RT>(s4, a);
    double s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
    if (PARTS > 1 && low()) {
      p16_dotrows<J, 4>(d2, pr);
      s += d2[0] + d2[1];
    } else if constexpr (!NODE) {
#pragma unroll
      for (int q = 0; q + 4 <= N; q += 4) p16_dotrows<J, 4>(d2, pr + J + 1 + q);
      if constexpr (N % 4 != 0) p16_dotrows<J, N % 4>(d2, pr + P16 - N % 4);
    }
    s = xr_cross_rows(s);
    if constexpr (!NODE) s += PARTS > 1 && low() ? 0.0 : d2[0] + d2[1];
    double p = pr[J];
    if constexpr (PARTS > 1) {
      double* E = ex + (J & 1) * (P16 * (PARTS + 1)) + c;
      E[P16 * part] = s;                        // four lanes, one value
      if (!low()) E[P16 * PARTS] = p;
      __syncthreads();
      s = E[0];
#pragma unroll
      for (int q = 1; q < PARTS; ++q) s += E[P16 * q];
      p = E[P16 * PARTS];
    }
    const double ss = readlane_d(s, J), alpha = readlane_d(p, J);
    // a column without anything below its diagonal: H = I (by masks alone, as
    // the values of p16_larfg then need not be numbers)
    int sh = __double2hiint(ss);
    asm("" : "+s"(sh));                         // (tested in scalar registers)
    const int cj = sh != 0 ? J : P16;
    ssmin = min(ssmin, (uint32_t)sh - 1u);
    double beta, tj, scal, rb;
    p16_larfg(alpha, ss, beta, tj, scal, rb);
    const double wv = fma(scal, s, p);          // v_Jᵀ·(column c), v_J = [1; scal·x]
    const double f = c > cj ? wv * rb : 0.0;    // −tau·scal = 1/beta
    axpys<J, 0, H>(a, f);
    asm volatile("" : "+s"(nact));
    if constexpr (RT > H)
      if (__builtin_expect(nact > H, 1)) axpys<J, H, RT>(a, f);
    if (PARTS > 1 && low()) {
      p16_axpyrows<J, 4>(pr, f);
    } else {
      if constexpr (!NODE) {
#pragma unroll
        for (int q = 0; q + 4 <= N; q += 4) p16_axpyrows<J, 4>(pr + J + 1 + q, f);
        if constexpr (N % 4 != 0) p16_axpyrows<J, N % 4>(pr + P16 - N % 4, f);
      }
      pr[J] = c > cj ? fma(-tj, wv, p) : (c == cj ? beta : p);
      Zc[J * P16_LD] = wv * scale * -tj;        // four lanes, one value
    }
    tau = c == cj ? tj : tau;
    scale = c == cj ? scal : scale;
  }

  // The whole panel again with dlarfg's general semantics (norms that have to
  // be rescaled, non-finite columns), on this part's copy: nt tiles in Vs (GLOB:
  // the leaf in memory), the pivot tile in Ds; one column at a time with the
  // updates masked to the columns behind it.  A column of very large or small
  // entries is first scaled by a power of two, which leaves its reflector as it
  // is and brings data of any common size into the range of p16_larfg; what is
  // left (entries too far apart, NaN, infinities) takes up to three more passes
  // and dlarfg_scalar.  Two passes a column, two or four tiles in flight; keeping
  // the strip in the registers that are free here spilled in the straight-line
  // steps.  hh_recon_qr with every entry around 1e-200: 256×16 100 µs (49 in
  // range), 32768×128 1030 (460), 65536×16 420 (147); with one value in flight,
  // a division an element and one wave for a whole tall leaf 347, 3540 and 4400.
  __device__ __forceinline__ double slow(double* Vs, double* Ds, double* Zs, int nt, int nb, int& bar) const {
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const bool first = PARTS == 1 || part == 0;   // holds the pivot tile
    asm volatile("" : "+s"(nt));                  // (a count the loops do not unroll by)
    auto sync = []() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup"); };
    auto load = [&](int t) {                      // this lane's column in tile t
      if constexpr (GLOB) return p16_rows_load(col + 16 * (t + 1) + 4 * g, rows - 16 * (t + 1) - 4 * g, rows > 0);
      else return p16_load(Vs + t * P16_TILE, lane);
    };
    auto load_j = [&](int t, int j) {             // column j there
      if constexpr (GLOB) {
        const double* q = reinterpret_cast<const double*>(__double_as_longlong(
            readlane_d(__longlong_as_double(reinterpret_cast<uintptr_t>(col)), j)));
        const int left = __builtin_amdgcn_readlane(rows, j) - 16 * (t + 1) - 4 * g;
        return p16_rows_load(q + 16 * (t + 1) + 4 * g, left, true);
      } else {
        return p16_load(Vs + t * P16_TILE, (lane & 48) | j);
      }
    };
    auto store = [&](int t, const dbl4& x) {
      if constexpr (GLOB) p16_rows_store(col + 16 * (t + 1) + 4 * g, x, rows - 16 * (t + 1) - 4 * g, rows > 0);
      else p16_store(Vs + t * P16_TILE, x, lane);
    };
    // f(t, x_t) for all tiles, CH of them loaded at a time
    constexpr int CH = PARTS > 1 ? 4 : 2;
    auto each = [&](auto get, auto f) {
#pragma unroll 1
      for (int t = 0; t < nt; t += CH) {
        decltype(get(0)) x[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) x[i] = get(min(t + i, nt - 1));
#pragma unroll
        for (int i = 0; i < CH; ++i)
          if (t + i < nt) f(t + i, x[i]);
      }
    };
    struct Two {
      dbl4 j, c;
    };
    auto both = [&](int j) { return [&, j](int t) { return Two{load_j(t, j), load(t)}; }; };
    auto top = [](const dbl4& x) { return fmax(fmax(fabs(x[0]), fabs(x[1])), fmax(fabs(x[2]), fabs(x[3]))); };
    auto rows_max = [](double m) {
      m = fmax(m, __shfl_xor(m, 16));
      return fmax(m, __shfl_xor(m, 32));
    };
    auto ldexp4 = [](const dbl4& x, int e) { return dbl4{ldexp(x[0], e), ldexp(x[1], e), ldexp(x[2], e), ldexp(x[3], e)}; };
    // the values of the pivot tile (or of a low part's first one) below the
    // diagonal of column j, which belong to a leaf's vectors
    auto low_row = [&](int v, int j) { return !NODE && (!first || 4 * g + v > j); };
    auto below = [&](const dbl4& x, int j) {
      dbl4 y;
#pragma unroll
      for (int v = 0; v < 4; ++v) y[v] = low_row(v, j) ? x[v] : 0.0;
      return y;
    };
    // sums and largest values over all parts, and the pivot part's q
    auto exchange = [&](double& sum, double& m, double& q) {
      if constexpr (PARTS > 1) {
        double* E = ex + 2 * P16 * (PARTS + 1) + (bar & 1) * (P16 * (2 * PARTS + 1)) + c;
        E[P16 * part] = sum;
        E[P16 * (PARTS + part)] = m;
        if (first) {
          E[P16 * 2 * PARTS] = q;
          if (lane == 0) ex[p16_more(PARTS) + (bar & 1)] = 1.0;
        }
        __syncthreads();
        sum = E[0];
        m = E[P16 * PARTS];
#pragma unroll
        for (int i = 1; i < PARTS; ++i) {
          sum += E[P16 * i];
          m = fmax(m, E[P16 * (PARTS + i)]);
        }
        q = E[P16 * 2 * PARTS];
        ++bar;
      }
    };
    double none = 0.0, zero = 0.0;

    double mx = top(p16_load(Ds, lane));
    each(load, [&](int, const dbl4& x) { mx = fmax(mx, top(x)); });
    mx = rows_max(mx);
    exchange(zero, mx, none);
    int e = mx > 0.0 && mx < INFINITY ? __builtin_amdgcn_frexp_exp(mx) : 0;
    if (abs(e) < 400) e = 0;
    if (__builtin_amdgcn_ballot_w64(e != 0) != 0) {
      p16_store(Ds, ldexp4(p16_load(Ds, lane), -e), lane);
      each(load, [&](int t, const dbl4& x) { store(t, ldexp4(x, -e)); });
    }
    double tl = 0.0, scale = 1.0;
    sync();
#pragma unroll 1
    for (int j = 0; j < nb; ++j) {
      const int jr = trow_of(j);
      double p = Ds[jr * P16_LD + c];             // (a low part's is not used)
      auto dots = [&](double& m) {
        const dbl4 xd = below(p16_load(Ds, (lane & 48) | j), j), d = below(p16_load(Ds, lane), j);
        dbl4 s = xd * d;
        m = top(d);
        each(both(j), [&](int, const Two& x) {
          s += x.j * x.c;
          m = fmax(m, top(x.c));
        });
        m = rows_max(m);
        return xr_cross_rows((s[0] + s[1]) + (s[2] + s[3]));
      };
      double m, s = dots(m);
      exchange(s, m, p);
      const double ss = readlane_d(s, j), alpha = readlane_d(p, j);
      m = readlane_d(m, j);
      double beta, tj, fs, sc, wv;                // sc: the vector's scale, fs: the update's factor
      if (ss > 0x1p-960 && ss < 0x1p960 && fabs(alpha) < 0x1p480) {
        p16_larfg(alpha, ss, beta, tj, sc, fs);
        wv = fma(sc, s, p);
      } else {
        double xnorm = m == 0.0 ? 0.0 : NAN;      // (a NaN beside entries that are none)
        if (m > 0.0 && m < INFINITY && ss == ss) {
          const int em = __builtin_amdgcn_frexp_exp(m);
          dbl4 q = ldexp4(below(p16_load(Ds, lane), j), -em);
          q *= q;
          each(load, [&](int, const dbl4& x) {
            const dbl4 y = ldexp4(x, -em);
            q += y * y;
          });
          double n2 = xr_cross_rows((q[0] + q[1]) + (q[2] + q[3]));
          exchange(n2, zero, none);
          xnorm = ldexp(sqrt(readlane_d(n2, j)), em);
        }
        const Reflector h = dlarfg_scalar(alpha, xnorm);
        if (h.tau != 0.0) {
          if (c == j) {
            auto vec = [&](dbl4 x) {
              for (int k = 0; k < h.knt; ++k) x *= 0x1p969;
              return x * h.scal;
            };
            const dbl4 d = p16_load(Ds, lane), y = vec(d);
            dbl4 z;
#pragma unroll
            for (int v = 0; v < 4; ++v) z[v] = low_row(v, j) ? y[v] : d[v];
            p16_store(Ds, z, lane);
#pragma unroll 1
            for (int t = 0; t < nt; ++t) store(t, vec(load(t)));
          }
          sync();
          s = dots(m);
          exchange(s, m, p);
        }
        wv = p + s;
        beta = h.beta;
        tj = h.tau;
        fs = -h.tau;
        sc = 1.0;
      }
      if (c > j) {
        const double f = wv * fs;
        const dbl4 xd = p16_load(Ds, (lane & 48) | j), d = p16_load(Ds, lane);
        dbl4 z;
#pragma unroll
        for (int v = 0; v < 4; ++v) z[v] = low_row(v, j) ? fma(xd[v], f, d[v]) : d[v];
        p16_store(Ds, z, lane);
        each(both(j), [&](int t, const Two& x) { store(t, x.j * f + x.c); });
      }
      sync();
      if (first && g == 0) {
        Ds[jr * P16_LD + c] = c > j ? fma(-tj, wv, p) : (c == j ? beta : p);
        Zs[j * P16_LD + c] = c < j ? wv * scale * -tj : 0.0;
      }
      if (c == j) {
        tl = tj;
        scale = sc;
      }
      sync();
    }
    const dbl4 d = p16_load(Ds, lane);
    dbl4 z;
#pragma unroll
    for (int v = 0; v < 4; ++v) z[v] = low_row(v, c) ? d[v] * scale : ldexp(d[v], e);
    p16_store(Ds, z, lane);
    each(load, [&](int t, const dbl4& x) { store(t, x * scale); });
    sync();
    return tl;
  }

  template <int J, int Q = 0>
  __device__ static __forceinline__ void tsum(double& acc, const double& z, const double (&trow)[P16]) {
    if constexpr (Q < J) {
      p16_fma_bc<Q>(acc, z, trow[Q]);
      tsum<J, Q + 1>(acc, z, trow);
    }
  }
  // T(0:J, J) = −tau_J·T(0:J, 0:J)·(v_qᵀv_J)_q, T(J, J) = tau_J, from column J on
  template <int J>
  __device__ __forceinline__ void tcols(double (&trow)[P16], const double (&z)[P16], int c) const {
    if constexpr (J < P16) {
      double acc = c == J ? tau : 0.0;
      asm("s_nop 1" : "+v"(acc) : "v"(z[J]));
      tsum<J>(acc, z[J], trow);
      trow[J] = acc;
      tcols<J + 1>(trow, z, c);
    }
  }

  // Factors the first nb columns of the strip (D; a); nact tiles of `a` may
  // be nonzero.  On return Vs holds the vectors scaled as dlarfg's (every
  // tile that can be nonzero, and zeros up to tile H), Ds and D the pivot
  // tile (R rows and, for a leaf, the vectors below its diagonal) and Zs the
  // panel's T, transposed; `a` is left unscaled.
  __device__ __forceinline__ void factor(dbl4& D, dbl4 (&a)[RT], int nact, int nb, int lane, double* Zs, double* Vs,
                                         double* Ds) {
    const int c = lane & 15;
    tau = 0.0;
    scale = 1.0;
    ssmin = ~0u;
    // the strip may come straight from MFMAs, whose results the inline VALU
    // code below must not read before they land
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n s_nop 15\n s_nop 15");
    __builtin_amdgcn_sched_barrier(0);
    // kept for slow(): straight-line columns with one test at the end
    // cost less than a way out of every column
    p16_store(Ds, D, lane);
    if constexpr (!GLOB)
#pragma unroll
      for (int t = 0; t < RT; ++t)
        if (t < H || nact > H) p16_store(Vs + t * P16_TILE, a[t], lane);
    double* Zc = Zs + c;
#pragma unroll
    for (int q = 0; q < P16; ++q) pr[q] = Ds[trow_of(q) * P16_LD + c];
    if (PARTS > 1 && part != 0) {
#pragma unroll
      for (int v = 0; v < 4; ++v) pr[v] = D[v];
    } else if (nb < P16)
      for (int q = nb; q < P16; ++q) Zc[q * P16_LD] = 0.0;
#define P16_STEP(J)                 \
  asm volatile("" : "+s"(nb));      \
  if (J == 0 || __builtin_expect(J < nb, 1)) column<J>(a, nact, Zc);
    P16_STEP(0) P16_STEP(1) P16_STEP(2) P16_STEP(3) P16_STEP(4) P16_STEP(5) P16_STEP(6) P16_STEP(7)
    P16_STEP(8) P16_STEP(9) P16_STEP(10) P16_STEP(11) P16_STEP(12) P16_STEP(13) P16_STEP(14) P16_STEP(15)
#undef P16_STEP
    int bar = 0;
    // Exact as they stand are columns with ‖x‖² above 2^-960 (dots of two of
    // them lose nothing to underflow that counts, 2^-1074 against 2^-960) and
    // no overflow, which makes its column infinite and that column's tau NaN,
    // as a NaN or an infinity in the data does, and columns with x = 0.
    bool redo = __builtin_amdgcn_ballot_w64(tau != tau) != 0 || ssmin < 0x03f00000u;
    const uint64_t zero = __builtin_amdgcn_ballot_w64(tau == 0.0 && c < nb);
    if (__builtin_expect(zero != 0, 0)) {
      // really nothing there, or entries too small to square?  (they are as
      // their column's own step found them)
      double nz = 0.0;
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) nz = fmax(nz, fabs(a[t][v]));
      if (!NODE)
#pragma unroll
        for (int q = 0; q < P16; ++q) nz = fmax(nz, (PARTS > 1 && part != 0 ? q < 4 : q > c) ? fabs(pr[q]) : 0.0);
      bool some = __builtin_amdgcn_ballot_w64(tau == 0.0 && nz > 0.0) != 0;
      if constexpr (PARTS > 1) {                  // one decision for all parts
        double* E = ex + 2 * P16 * (PARTS + 1);
        if (lane == 0) {
          E[part] = some ? 1.0 : 0.0;
          if (part == 0) ex[p16_more(PARTS)] = 1.0;
        }
        __syncthreads();
        some = false;
#pragma unroll
        for (int q = 0; q < PARTS; ++q) some |= E[q] != 0.0;
        some = __builtin_amdgcn_readfirstlane(some) != 0;
        bar = 1;
      }
      redo |= some;
      if (PARTS == 1 || part == 0)
        for (int q = 0; q < P16; ++q)
          if (zero >> q & 1) Zc[q * P16_LD] = 0.0;
    }
    if constexpr (GLOB)   // (without meaning if the panel is redone)
#pragma unroll
      for (int t = 0; t < RT; ++t) a[t] *= scale;
    if (__builtin_expect(redo, 0)) {
      tau = slow(Vs, Ds, Zs, nact > H ? RT : H, nb, bar);
      if constexpr (GLOB)
#pragma unroll
        for (int t = 0; t < RT; ++t)
          a[t] = p16_rows_load(col + 16 * (t + 1) + 4 * (lane >> 4), rows - 16 * (t + 1) - 4 * (lane >> 4), rows > 0);
      if (PARTS > 1 && part != 0) return;
    } else {
      if constexpr (!GLOB)
#pragma unroll
        for (int t = 0; t < RT; ++t)
          if (t < H || nact > H) p16_store(Vs + t * P16_TILE, a[t] * scale, lane);
      if (PARTS > 1 && part != 0) {
        p16_store(Ds, dbl4{pr[0], pr[1], pr[2], pr[3]} * scale, lane);
        return;
      }
#pragma unroll
      for (int q = 0; q < P16; ++q) Ds[trow_of(q) * P16_LD + c] = !NODE && q > c ? pr[q] * scale : pr[q];
    }
    if (PARTS > 1 && lane == 0) ex[p16_more(PARTS) + (bar & 1)] = 0.0;
    D = p16_load(Ds, lane);
    double z[P16], trow[P16];
#pragma unroll
    for (int q = 0; q < P16; ++q) z[q] = Zc[q * P16_LD];
    tcols<0>(trow, z, c);
#pragma unroll
    for (int q = 0; q < P16; ++q) Zc[q * P16_LD] = trow[q];
  }
};

// Products with a published panel: Vk holds its vectors as 16×16 tiles in
// LDS (row-major, tile row i, pitch P16_LD), a[0..N) the caller's strip.
// acc (16×16) + Σ_t V_tᵀ·a_t over tiles t < nact (tiles past nact are zero).
// Four tiles at a time are summed from zero and then added: one chain over all
// rows would round 4·N times at the size of its sum.
template <int N>
__device__ __forceinline__ dbl4 p16_vta(const double* __restrict__ Vk, const dbl4 (&a)[N], int nact, dbl4 acc, int lane) {
  const double* vp = Vk + (lane >> 4) * P16_LD + (lane & 15);
  dbl4 s0 = {0.0, 0.0, 0.0, 0.0}, s1 = s0;
#pragma unroll
  for (int q = 0; q < (N + 3) / 4; ++q)
    if (q == 0 || 4 * q < nact) {
      const dbl4 r0 = s0, r1 = s1;
      s0 = s1 = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int t = 4 * q; t < 4 * q + 4; ++t)
        if (t < N) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const double x = vp[t * P16_TILE + 4 * v * P16_LD];
            if (v & 1) s1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x, a[t][v], s1, 0, 0, 0);
            else s0 = __builtin_amdgcn_mfma_f64_16x16x4f64(x, a[t][v], s0, 0, 0, 0);
          }
        }
      if (q > 0) acc += r0 + r1;
      __builtin_amdgcn_sched_barrier(0);   // sixteen operand loads ahead, no more registers than that
    }
  return acc + (s0 + s1);
}

// a_t += V_t·u over tiles t < nact (u: 16×16, tile layout).
template <int N>
__device__ __forceinline__ void p16_vu(const double* __restrict__ Vk, dbl4 (&a)[N], int nact, const dbl4& u, int lane) {
  const double* vp = Vk + (lane & 15) * P16_LD + (lane >> 4);
#pragma unroll
  for (int q = 0; q < (N + 3) / 4; ++q)
    if (q == 0 || 4 * q < nact) {
      // four tiles' chains interleaved: consecutive MFMAs are independent
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int t = 4 * q; t < 4 * q + 4; ++t)
          if (t < N) a[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vp[t * P16_TILE + 4 * v], u[v], a[t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
}

// X·y for a 16×16 X in LDS, row-major (y: tile layout).
__device__ __forceinline__ dbl4 p16_xy(const double* __restrict__ X, const dbl4& y, dbl4 acc, int lane) {
  const double* xp = X + (lane & 15) * P16_LD + (lane >> 4);
#pragma unroll
  for (int v = 0; v < 4; ++v) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(xp[4 * v], y[v], acc, 0, 0, 0);
  return acc;
}
// The compact-WY T of a factorization advancing by 16-column panels, kept in
// LDS as 16×16 tiles (transposed, one slot per pair i ≤ k).  Wave i owns tile
// row i.  In step k (after its barrier) wave j < k leaves the Gram tile
// V_kᵀV_j in slot (j, k); in step k + 1 wave i < k forms
//   T(i,k)ᵀ = −T_kkᵀ·Σ_{i≤j<k} (V_kᵀV_j)·T(i,j)ᵀ
// from those tiles, and in step k + 2, when every wave has read them, puts it
// into slot (i, k), where only wave i needs it again.
__device__ __forceinline__ int p16_slot(int i, int k) { return (k * (k + 1) / 2 + i) * P16_TILE; }

__device__ __forceinline__ dbl4 p16_tcol(const double* __restrict__ S, int i, int k, int lane) {
  dbl4 x = {0.0, 0.0, 0.0, 0.0};
  for (int j = i; j < k; ++j) x = p16_xy(S + p16_slot(j, k), p16_load(S + p16_slot(i, j), lane), x, lane);
  const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
  return -p16_xy(S + p16_slot(k, k), x, zero, lane);
}

}  // namespace cqr
