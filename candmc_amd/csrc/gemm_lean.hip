// FP64 MFMA kernel for Z = Yᵀ·A of the compact-WY trailing update
// (alg/QR/qr_2d/qr_2d.cxx:259-265, the first dgemm of upd_A): raw split-K
// partials of Aᵀ·B, both operands k-contiguous (column-major K×M and K×N).
// No structural masks: the unit-lower top block of an implicit Y goes
// through the general kernel.
//
// 128×128 tile, 256 threads (4 waves of 64×64, 16 MFMA tiles each), 16-deep
// k slabs double-buffered in LDS, k-contiguous there too, so the global loads
// and the LDS writes are 16 bytes wide, and eight lanes read one 128-byte
// line of a column.  Slab s + 1 goes from registers to LDS before the MFMAs
// of slab s, and slab s + 2 is fetched under them: the loads have a whole
// slab's time, and nothing but the barrier stands between two slabs' MFMAs.
// Register use is bounded for two workgroups per CU, so one workgroup's
// prologue and epilogue overlap the other's MFMAs.  Items are ordered XCD by
// XCD, columns fastest, so the workgroups of one XCD share a k chunk of Y in
// its L2.
//
// Bound: MFMA issue (a v_mfma_f64_16x16x4f64 holds its SIMD 64 cycles).
// Z = Yᵀ·A at 32768×3968×128: 669 → 550 µs (50 → 60.5 TFLOP/s; a large
// square product reaches 73 on this card).  The loop before had two threads
// per column and wrote slab s + 1 to LDS after the MFMAs of slab s; it took
// 562 µs even without its global loads.
#include "cqr_device.h"
#include "cqr_internal.h"

namespace cqr {

namespace {

typedef double d4l __attribute__((ext_vector_type(4)));
typedef double d2l __attribute__((ext_vector_type(2)));
// a 16-byte global access at any 8-byte boundary (odd leading dimensions)
typedef double d2u8 __attribute__((ext_vector_type(2), aligned(8)));

constexpr int BM = 128, BN = 128, BK = 16;
constexpr int PK = BK + 2;   // pitch of a slab row [idx][k]: 16 rows × 2 k cover all banks

struct LeanArgs {
  int64_t M, N, K;
  const double* A;
  int64_t lda;
  const double* B;
  int64_t ldb;
  double* C;                 // partial of split z at C + z·M·N (ld M)
  int64_t kchunk;            // k per split (multiple of 16)
  int ntm, ntn, nsplit;      // tile grid and number of k splits
  int per_xcd;               // work items (split, tile) per XCD
};

}  // namespace

// FULL: the tile and its k chunk need no bounds checks, so every access is
// unconditional (a branch around a slab's loads would make each wait for the
// ones before it).
template <bool FULL>
__device__ __forceinline__ void lean_tile(const LeanArgs& g, int z, int64_t m0, int64_t n0, int64_t kbeg, int64_t kend,
                                          double (*As)[BM * PK], double (*Bs)[BN * PK]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm0 = (wave & 1) * 64, wn0 = (wave >> 1) * 64;
  // a thread's slab elements: rows ri + 32s, k = kh, kh + 1
  const int ri = tid >> 3, kh = (tid & 7) * 2;
  d2l ra[4], rb[4];
  auto load = [&](int64_t k0) {
    const int64_t k = k0 + kh;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int64_t m = m0 + ri + 32 * s, n = n0 + ri + 32 * s;
      if (FULL) {
        ra[s] = *reinterpret_cast<const d2u8*>(g.A + k + m * g.lda);
        rb[s] = *reinterpret_cast<const d2u8*>(g.B + k + n * g.ldb);
      } else {
        ra[s].x = (k < kend && m < g.M) ? g.A[k + m * g.lda] : 0.0;
        ra[s].y = (k + 1 < kend && m < g.M) ? g.A[k + 1 + m * g.lda] : 0.0;
        rb[s].x = (k < kend && n < g.N) ? g.B[k + n * g.ldb] : 0.0;
        rb[s].y = (k + 1 < kend && n < g.N) ? g.B[k + 1 + n * g.ldb] : 0.0;
      }
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      *reinterpret_cast<d2l*>(&As[buf][(ri + 32 * s) * PK + kh]) = ra[s];
      *reinterpret_cast<d2l*>(&Bs[buf][(ri + 32 * s) * PK + kh]) = rb[s];
    }
  };

  d4l acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = d4l{0.0, 0.0, 0.0, 0.0};

  const int fr = lane >> 4, fc = lane & 15;
  auto compute = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      double af[4], bf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) af[i] = As[buf][(wm0 + 16 * i + fc) * PK + kk + fr];
#pragma unroll
      for (int j = 0; j < 4; ++j) bf[j] = Bs[buf][(wn0 + 16 * j + fc) * PK + kk + fr];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf[j], af[i], acc[i][j], 0, 0, 0);
    }
  };

  const int64_t nslab = (kend - kbeg + BK - 1) / BK;
  load(kbeg);
  store(0);
  if (nslab > 1) load(kbeg + BK);
  __syncthreads();
  for (int64_t sl = 0; sl < nslab; ++sl) {
    const int buf = (int)(sl & 1);
    if (sl + 1 < nslab) store(buf ^ 1);
    if (sl + 2 < nslab) load(kbeg + (sl + 2) * BK);
    __builtin_amdgcn_sched_barrier(0);
    compute(buf);
    __syncthreads();
  }

  // lane l, register v of acc[i][j] holds C[m0+wm0+16i+(l&15)][n0+wn0+16j+(l>>4)+4v]
  double* C = g.C + (int64_t)z * g.M * g.N;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t gm = m0 + wm0 + 16 * i + fc;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t gn = n0 + wn0 + 16 * j + fr + 4 * v;
        if (FULL || (gm < g.M && gn < g.N)) C[gm + gn * g.M] = acc[i][j][v];
      }
  }
}

__global__ void __launch_bounds__(256, 2) lean_gemm_f64(LeanArgs g) {
  __shared__ __align__(16) double As[2][BM * PK];
  __shared__ __align__(16) double Bs[2][BN * PK];
  // workgroups are dealt to the 8 XCDs round-robin; XCD x takes the
  // contiguous item range [x·per_xcd, (x+1)·per_xcd), items ordered split
  // by split with column tiles fastest
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int tiles = g.ntm * g.ntn;
  const int u = xcd * g.per_xcd + slot;
  if (slot >= g.per_xcd || u >= tiles * g.nsplit) return;
  const int z = u / tiles, t = u - z * tiles;
  const int tm = t / g.ntn, tn = t - tm * g.ntn;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int64_t kbeg = (int64_t)z * g.kchunk, kend = min(g.K, kbeg + g.kchunk);
  if ((m0 + BM <= g.M) && (n0 + BN <= g.N) && ((kend - kbeg) % BK == 0))
    lean_tile<true>(g, z, m0, n0, kbeg, kend, As, Bs);
  else
    lean_tile<false>(g, z, m0, n0, kbeg, kend, As, Bs);
}

// k splits (at most cap) for `tiles` output tiles of `out` values and K rows.
// Two workgroups share a CU and its matrix cores, so a round of up to 512
// items lasts as long as two chunks, however few of its slots are taken: 31
// tiles × 17 splits = 527 items ran as two rounds, the second for 15 of them
// (Yᵀ·A at 32768×3968×128: 934 µs against 669 with 16 splits).  The
// rounds' time at the card's product rate (0.115 µs a row of a 128×128 tile
// alone on a CU, a quarter more where one workgroup hides its own latency)
// is weighed against writing and reading one more partial (5 TB/s).
static int lean_splits(int64_t tiles, int64_t K, int64_t out, int cap) {
  double best = 0.0;
  int pick = 1;
  for (int s = 1; s <= cap; ++s) {
    const int64_t kc = ((K + s - 1) / s + BK - 1) / BK * BK, used = (K + kc - 1) / kc, items = tiles * used;
    const int64_t rem = items % 512;
    const double rounds = 2.0 * (double)(items / 512) + (rem > 256 ? 2.0 : rem > 0 ? 1.25 : 0.0);
    const double t = rounds * (double)kc * 0.115 + 16.0 * (double)used * (double)out / 5e6;
    if (s == 1 || t < best) {
      best = t;
      pick = s;
    }
  }
  return pick;
}

// Partial sums of Aᵀ·B (A K×M, B K×N, K ≥ 1) over at most `cap` k chunks, in
// scratch + z·M·N (ld M); *used receives their number.
int lean_gemm(cqr_ctx* c, int64_t M, int64_t N, int64_t K, const double* A, int64_t lda, const double* B, int64_t ldb,
              double* scratch, int cap, int kind, int* used) {
  *used = 0;
  if (M <= 0 || N <= 0 || K <= 0) return CQR_OK;
  LeanArgs g{};
  g.M = M; g.N = N; g.K = K; g.A = A; g.lda = lda; g.B = B; g.ldb = ldb; g.C = scratch;
  g.ntm = (int)((M + BM - 1) / BM);
  g.ntn = (int)((N + BN - 1) / BN);
  const int64_t tiles = (int64_t)g.ntm * g.ntn;
  const int s = lean_splits(tiles, K, M * N, std::max(cap, 1));
  g.kchunk = ((K + s - 1) / s + BK - 1) / BK * BK;
  g.nsplit = (int)((K + g.kchunk - 1) / g.kchunk);
  *used = g.nsplit;
  if (tiles * g.nsplit >= (int64_t)1 << 30) return CQR_ERR_INVALID;
  g.per_xcd = (int)((tiles * g.nsplit + 7) / 8);
  hipEvent_t ev = prof_begin(c);
  hipLaunchKernelGGL(lean_gemm_f64, dim3((unsigned)(8 * g.per_xcd)), dim3(256), 0, c->stream, g);
  prof_end(c, ev, kind, 2.0 * M * N * K, 8.0 * ((double)M * K + (double)K * N + g.nsplit * (double)M * N));
  return check_launch(c, "lean_gemm_f64");
}

}  // namespace cqr
