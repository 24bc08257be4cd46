// Solve and refinement of many one-panel least-squares requests at once
// (n ≤ 128, at most 16 right-hand sides each), from the batched factors
// A = Q·R, Q = I − Y·T·Yᵀ.  Per request and column this is the computation of
// lstsq_refine (lsq.cpp) while its corrected semi-normal-equation steps
// converge:
//   x  = R⁻¹·(Qᵀb)(0:n),   then   x += R⁻¹R⁻ᵀAᵀ(b − A·x).
// Each of the two lines is two launches over all requests:
//   slab:   partial sums of Yᵀb, or of Aᵀ(b − A·x), over row slabs; A is read
//           once, a wave forming r = b − A·x for sixteen rows and multiplying
//           it into Aᵀ from the registers the rows already are in;
//   solve:  a workgroup per request sums its slabs and solves with R, whose
//           tiles it holds in registers; it also takes the step (or not) and
//           records the request's state.
// A request that is done, or whose steps stopped contracting, drops out of
// later launches by its state; the caller takes the latter through
// lstsq_refine.
//
// Bound: the chains inside a workgroup (a slab's rows one after another, the
// solve's sixteen tile steps), then HBM.  32 requests of 64 columns, rows
// around 4096 and 1 to 16 right-hand sides: 7.3 ms with a chain of a hundred
// small launches and a synchronisation per step and request, 0.92 ms so, of
// it the factorization 0.57 ms, a slab launch 55 (Yᵀb) or 83 µs (Aᵀ(b − A·x)),
// a solve 30 µs.
#include "cqr_device.h"
#include "cqr_internal.h"
#include "panel16.h"

namespace cqr {

namespace {

constexpr int MT = CQR_MAX_B / 16;   // tile rows of the widest request

// Between one lane's LDS writes and other lanes' reads of them in one wave.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace

// Y := A, slab by slab (grid: slabs of the longest request × requests).
__global__ void __launch_bounds__(256) lsq_copy_kernel(const LsqProb* __restrict__ probs) {
  const LsqProb& P = probs[blockIdx.y];
  const int64_t r0 = (int64_t)blockIdx.x * P.slab;
  if (r0 >= P.m) return;
  const int rows = (int)min(P.slab, P.m - r0);
  const double* a = P.A + r0;
  double* y = P.Y + r0;
  for (int r = threadIdx.x & 127; r < rows; r += 128)
#pragma unroll 8
    for (int j = threadIdx.x >> 7; j < P.n; j += 2) y[r + j * P.m] = a[r + j * P.lda];
}

// Partial sums over one slab, sixteen rows of A (or Y) a wave at a time as
// tiles whose lane l holds row (l & 15), columns (l >> 4) + 4v: the left
// operand of A·x; through a tile in LDS they become that of Aᵀ·r.
// n ≤ 16·NT: with four tiles a row four workgroups fit a CU, with eight two.
template <bool REFINE, int NT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(16 / NT)))
lsq_slab_kernel(const LsqProb* __restrict__ probs, const LsqState* __restrict__ states) {
  __shared__ double xs[NT * P16_TILE];     // x, then the sum over the waves
  __shared__ double tr[4][2][P16_TILE];
  const LsqProb& P = probs[blockIdx.y];
  const int64_t r0 = (int64_t)blockIdx.x * P.slab, m = P.m;
  if (r0 >= m || (REFINE && states[blockIdx.y].state != LSQ_ACTIVE)) return;
  const int n = P.n, nr = P.nr, nbn = (n + 15) / 16;
  const int nt = (int)((min(P.slab, m - r0) + 15) / 16);
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int c = lane & 15, g = lane >> 4;
  const double* A = REFINE ? P.A : P.Y;
  const int64_t lda = REFINE ? P.lda : m;
  const double* Bc = P.B + (int64_t)min(c, nr - 1) * P.ldb;
  const dbl4 zero = {0.0, 0.0, 0.0, 0.0};

  dbl4 a[NT], b;
  // columns past n come from the last one in range and meet zeros; the
  // address walks along the row
  auto fetch = [&](int t) {
    const int64_t row = r0 + 16 * t;
    int k = min(g, n - 1);
    const double* p = A + min(row + c, m - 1) + k * lda;
#pragma unroll
    for (int kt = 0; kt < NT; ++kt)
      if (kt < nbn)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          a[kt][v] = *p;
          const bool in = k + 4 < n;
          p += in ? 4 * lda : 0;
          k += in ? 4 : 0;
        }
#pragma unroll
    for (int v = 0; v < 4; ++v) b[v] = Bc[min(row + g + 4 * v, m - 1)];
  };
  if (w < nt) fetch(w);
  if (REFINE) {
    for (int e = tid; e < 16 * nbn * 16; e += 256) {
      const int i = e % (16 * nbn), j = e / (16 * nbn);
      xs[(i >> 4) * P16_TILE + (i & 15) * P16_LD + j] = i < n && j < nr ? P.X[i + j * P.ldx] : 0.0;
    }
    __syncthreads();
  }
  dbl4 acc[NT];
#pragma unroll
  for (int kt = 0; kt < NT; ++kt) acc[kt] = zero;
#pragma unroll 1
  for (int t = w; t < nt; t += 4) {
    const int64_t row = r0 + 16 * t;
    dbl4 r = b;
    if (REFINE) {
      dbl4 s0 = zero, s1 = zero;
#pragma unroll
      for (int kt = 0; kt < NT; ++kt)
        if (kt < nbn) {
          const dbl4 xk = p16_load(xs + kt * P16_TILE, lane);
          s0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kt][0], xk[0], s0, 0, 0, 0);
          s1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kt][1], xk[1], s1, 0, 0, 0);
          s0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kt][2], xk[2], s0, 0, 0, 0);
          s1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kt][3], xk[3], s1, 0, 0, 0);
        }
      r -= s0 + s1;
    } else if (row < n) {   // Y's top is unit lower
#pragma unroll
      for (int kt = 0; kt < NT; ++kt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int d = (int)row + c - (16 * kt + g + 4 * v);
          a[kt][v] = d > 0 ? a[kt][v] : d == 0 ? 1.0 : 0.0;
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) r[v] = c < nr && row + g + 4 * v < m ? r[v] : 0.0;
#pragma unroll
    for (int kt = 0; kt < NT; ++kt)
      if (kt < nbn) {
        double* T = tr[w][kt & 1];
#pragma unroll
        for (int v = 0; v < 4; ++v) T[c * P16_LD + g + 4 * v] = a[kt][v];
        wave_lds_sync();
        const dbl4 xt = p16_load(T, lane);
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[kt] = __builtin_amdgcn_mfma_f64_16x16x4f64(xt[v], r[v], acc[kt], 0, 0, 0);
      }
    if (t + 4 < nt) fetch(t + 4);
  }
  __syncthreads();
  for (int q = 0; q < 4; ++q) {   // the waves' sums in order
    if (w == q)
#pragma unroll
      for (int kt = 0; kt < NT; ++kt)
        if (kt < nbn) p16_store(xs + kt * P16_TILE, q ? p16_load(xs + kt * P16_TILE, lane) + acc[kt] : acc[kt], lane);
    __syncthreads();
  }
  double* out = P.part + (int64_t)blockIdx.x * n * nr;
  for (int e = tid; e < n * nr; e += 256) {
    const int i = e % n, j = e / n;
    out[e] = xs[(i >> 4) * P16_TILE + (i & 15) * P16_LD + j];
  }
}

// A workgroup per request.  Wave w owns the tile rows w and 7 − w of every
// product and solve.  Without REFINE: x = R⁻¹·(b − Y·Tᵀ·Σ)(0:n).  With it: the
// correction R⁻¹R⁻ᵀ·Σ, and the step.
template <bool REFINE>
__global__ void __launch_bounds__(256)
lsq_solve_kernel(const LsqProb* __restrict__ probs, LsqState* __restrict__ states, int it, double tol) {
  __shared__ double S0[MT * P16_TILE], S1[MT * P16_TILE];
  __shared__ double inv[MT * P16_TILE];   // inverses of R's diagonal tiles
  __shared__ double dinv[CQR_MAX_B];
  __shared__ double red[2][4][16];
  __shared__ int flag;
  const LsqProb& P = probs[blockIdx.x];
  LsqState& st = states[blockIdx.x];
  if (REFINE && st.state != LSQ_ACTIVE) return;
  const int n = P.n, nr = P.nr, nbn = (n + 15) / 16;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int c = lane & 15, g = lane >> 4;
  const int64_t ldy = P.m;
  const double* Y = P.Y;
  const dbl4 zero = {0.0, 0.0, 0.0, 0.0};

  // Tile (t, kt) of an n×n operand with element (r, k) at r·rs + k·cs, as a
  // left operand; entries past the ends come from the last row or column, and
  // meet zeros or are dropped.
  auto fetch = [&](const double* p, int64_t rs, int64_t cs, int t, int kt) {
    dbl4 x;
    const double* q = p + min(16 * t + c, n - 1) * rs;
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] = q[min(16 * kt + g + 4 * v, n - 1) * cs];
    return x;
  };
  auto mul = [&](const dbl4& x, const dbl4& y, dbl4 acc) {
#pragma unroll
    for (int v = 0; v < 4; ++v) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[v], y[v], acc, 0, 0, 0);
    return acc;
  };
  auto row_of = [&](int q) { return q ? 7 - w : w; };

  // R's tiles right of the diagonal, by row (R⁻¹) and by column (R⁻ᵀ)
  dbl4 ru[2][MT], rl[2][MT];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int kt = 0; kt < MT; ++kt) {
      const int t = row_of(q);
      if (t < nbn && kt > t && kt < nbn) ru[q][kt] = fetch(Y, 1, ldy, t, kt);
      if (REFINE && t < nbn && kt < t) rl[q][kt] = fetch(Y, ldy, 1, t, kt);
    }
  // its diagonal tiles, unit past the end, into LDS
  for (int e = tid; e < 256 * nbn; e += 256) {
    const int t = e >> 8, r = e & 15, k = (e >> 4) & 15, i = 16 * t + r, j = 16 * t + k;
    inv[t * P16_TILE + r * P16_LD + k] = i < n && j < n ? (r <= k ? Y[i + j * ldy] : 0.0) : (r == k ? 1.0 : 0.0);
  }
  // Σ: the slab sums in slab order
  const int nn = n * nr;
  for (int e = tid; e < 256 * nbn; e += 256) {
    const int i = e % (16 * nbn), j = e / (16 * nbn);
    double s = 0.0;
    if (i < n && j < nr) {
      const double* p = P.part + j * n + i;
      for (int z0 = 0; z0 < P.nslab; z0 += 8) {
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = p[(int64_t)min(z0 + u, P.nslab - 1) * nn];
#pragma unroll
        for (int u = 0; u < 8; ++u) s += z0 + u < P.nslab ? x[u] : 0.0;
      }
    }
    S0[(i >> 4) * P16_TILE + (i & 15) * P16_LD + j] = s;
  }
  if (tid == 0) flag = 0;
  __syncthreads();
  if (tid < 16 * nbn) {
    const double d = inv[(tid >> 4) * P16_TILE + (tid & 15) * P16_LD + (tid & 15)];
    dinv[tid] = 1.0 / d;
    if (!REFINE && !(fabs(d) < INFINITY)) flag = 1;
  }
  __syncthreads();
  // column c of the tile's inverse by back substitution, four tiles a wave
  double xi[16];
  const int ti = 4 * w + g;
  if (ti < nbn) {
    const double* D = inv + ti * P16_TILE;
#pragma unroll
    for (int i = 0; i < 16; ++i) xi[i] = i == c ? 1.0 : 0.0;
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      xi[i] = i <= c ? xi[i] * dinv[16 * ti + i] : 0.0;
#pragma unroll
      for (int p = 0; p < i; ++p) xi[p] -= D[p * P16_LD + i] * xi[i];
    }
  }
  __syncthreads();
  if (ti < nbn)
#pragma unroll
    for (int i = 0; i < 16; ++i) inv[ti * P16_TILE + i * P16_LD + c] = xi[i];

  dbl4 y[2] = {zero, zero};
  if (!REFINE) {
    // Z' = Tᵀ·Σ (T holds Tᵀ, lower), then y = (b − Y·Z')(0:n)
    auto lower = [&](const double* p, int64_t ld, bool unit, const double* S, dbl4 (&out)[2]) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int t = row_of(q);
        out[q] = zero;
        if (t >= nbn) continue;
        dbl4 x[MT];
#pragma unroll
        for (int kt = 0; kt < MT; ++kt)
          if (kt <= t) x[kt] = fetch(p, 1, ld, t, kt);
#pragma unroll
        for (int kt = 0; kt < MT; ++kt)
          if (kt <= t) {
            if (kt == t)
#pragma unroll
              for (int v = 0; v < 4; ++v)
                x[kt][v] = g + 4 * v < c ? x[kt][v] : g + 4 * v > c ? 0.0 : unit ? 1.0 : x[kt][v];
            out[q] = mul(x[kt], p16_load(S + kt * P16_TILE, lane), out[q]);
          }
      }
    };
    dbl4 z[2];
    lower(P.T, n, false, S0, z);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int t = row_of(q);
      if (t >= nbn) continue;
#pragma unroll
      for (int v = 0; v < 4; ++v) z[q][v] = 16 * t + g + 4 * v < n ? z[q][v] : 0.0;
      p16_store(S1 + t * P16_TILE, z[q], lane);
    }
    __syncthreads();
    lower(Y, ldy, true, S1, z);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int t = row_of(q);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * t + g + 4 * v;
        y[q][v] = row < n && c < nr ? P.B[row + c * P.ldb] - z[q][v] : 0.0;
      }
    }
    __syncthreads();
  } else {
#pragma unroll
    for (int q = 0; q < 2; ++q)
      if (row_of(q) < nbn) y[q] = p16_load(S0 + row_of(q) * P16_TILE, lane);
    __syncthreads();
    // u = R⁻ᵀ·Σ, forwards; the inverses are read transposed
#pragma unroll
    for (int kt = 0; kt < MT; ++kt) {
      if (kt >= nbn) continue;
      const int q = kt < 4 ? 0 : 1;
      if (row_of(q) == kt) {
        y[q] = mul(p16_load(inv + kt * P16_TILE, lane), y[q], zero);
        if (kt == nbn - 1)   // nothing in the rows past the end
#pragma unroll
          for (int v = 0; v < 4; ++v) y[q][v] = 16 * kt + g + 4 * v < n ? y[q][v] : 0.0;
        p16_store(S1 + kt * P16_TILE, y[q], lane);
      }
      __syncthreads();
      const dbl4 u = -p16_load(S1 + kt * P16_TILE, lane);
#pragma unroll
      for (int q2 = 0; q2 < 2; ++q2)
        if (row_of(q2) > kt && row_of(q2) < nbn) y[q2] = mul(rl[q2][kt], u, y[q2]);
    }
  }
  // x = R⁻¹·y, backwards
#pragma unroll
  for (int kt = MT - 1; kt >= 0; --kt) {
    if (kt >= nbn) continue;
    const int q = kt < 4 ? 0 : 1;
    if (row_of(q) == kt) {
      y[q] = p16_xy(inv + kt * P16_TILE, y[q], zero, lane);
      p16_store(S0 + kt * P16_TILE, y[q], lane);
    }
    __syncthreads();
    const dbl4 x = -p16_load(S0 + kt * P16_TILE, lane);
#pragma unroll
    for (int q2 = 0; q2 < 2; ++q2)
      if (row_of(q2) < kt) y[q2] = mul(ru[q2][kt], x, y[q2]);
  }
  auto each = [&](auto f) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * row_of(q) + g + 4 * v;
        if (row < n && c < nr) f(q, v, P.X + row + c * P.ldx);
      }
  };
  if (!REFINE) {
    if (flag) {   // R is not finite
      if (tid == 0) st = LsqState{LSQ_LEFT, 0, 0.0};
      return;
    }
    each([&](int q, int v, double* x) { *x = y[q][v]; });
    if (tid == 0) st = LsqState{LSQ_ACTIVE, 0, 0.0};
    return;
  }
  // ‖dx‖ / ‖x‖ column by column, both scaled by their largest entries; a NaN
  // anywhere makes the ratio NaN
  double xo[2][4];
  double md = 0.0, mx = 0.0;
  bool nan = false;
  each([&](int q, int v, double* x) {
    xo[q][v] = *x;
    nan |= xo[q][v] != xo[q][v] || y[q][v] != y[q][v];
    md = fmax(md, fabs(y[q][v]));
    mx = fmax(mx, fabs(xo[q][v]));
  });
  auto columns = [&](double& p, double& q, bool sum) {   // over the rows of each column
#pragma unroll
    for (int o = 16; o <= 32; o <<= 1) {
      const double a = __shfl_xor(p, o), b = __shfl_xor(q, o);
      p = sum ? p + a : fmax(p, a);
      q = sum ? q + b : fmax(q, b);
    }
    __syncthreads();
    if (g == 0) {
      red[0][w][c] = p;
      red[1][w][c] = q;
    }
    __syncthreads();
    p = red[0][0][c];
    q = red[1][0][c];
#pragma unroll
    for (int i = 1; i < 4; ++i) {
      p = sum ? p + red[0][i][c] : fmax(p, red[0][i][c]);
      q = sum ? q + red[1][i][c] : fmax(q, red[1][i][c]);
    }
  };
  if (nan) flag = 1;
  columns(md, mx, false);
  double sd = 0.0, sx = 0.0;
  each([&](int q, int v, double*) {
    const double d = md > 0.0 ? y[q][v] / md : 0.0, x = mx > 0.0 ? xo[q][v] / mx : 0.0;
    sd += d * d;
    sx += x * x;
  });
  columns(sd, sx, true);
  const double nd = md * sqrt(sd), nx = mx * sqrt(sx);
  double rel = flag || nd != nd || nx != nx ? NAN : nd / fmax(nx, 1e-300);
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    const double a = __shfl_xor(rel, o);
    rel = rel != rel || a != a ? NAN : fmax(rel, a);
  }
  const bool take = rel <= 0.5 && (it == 1 || rel <= st.rel / 8);
  if (take) each([&](int q, int v, double* x) { *x = xo[q][v] + y[q][v]; });
  __syncthreads();   // every thread has read st
  if (tid == 0) {
    if (take) st = LsqState{rel <= tol ? LSQ_DONE : LSQ_ACTIVE, it, rel};
    else st.state = LSQ_LEFT;
  }
}

// The workgroups' row count: 128, or more where a request would have more
// than 64 slabs (its solve sums them all).
int64_t lsq_slab_rows(int64_t m) { return std::max<int64_t>(128, (m + 64 * 64 - 1) / (64 * 64) * 64); }

int launch_lsq_copy(cqr_ctx* c, const LsqProb* probs, int np, int nslab) {
  hipLaunchKernelGGL(lsq_copy_kernel, dim3(nslab, np), dim3(256), 0, c->stream, probs);
  return check_launch(c, "lsq_copy");
}

int launch_lsq_solve(cqr_ctx* c, const LsqProb* probs, LsqState* states, int np, int nslab, int nmax, int it, double tol) {
  auto slab = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(nslab, np), dim3(256), 0, c->stream, probs, states);
    return check_launch(c, "lsq_slab");
  };
  if (it == 0) {
    CQR_TRY(nmax <= 64 ? slab(lsq_slab_kernel<false, 4>) : slab(lsq_slab_kernel<false, 8>));
    hipLaunchKernelGGL(lsq_solve_kernel<false>, dim3(np), dim3(256), 0, c->stream, probs, states, it, tol);
  } else {
    CQR_TRY(nmax <= 64 ? slab(lsq_slab_kernel<true, 4>) : slab(lsq_slab_kernel<true, 8>));
    hipLaunchKernelGGL(lsq_solve_kernel<true>, dim3(np), dim3(256), 0, c->stream, probs, states, it, tol);
  }
  return check_launch(c, "lsq_solve");
}

}  // namespace cqr
