// Host-only check of how cqr_lstsq_batched (candmc_amd/csrc/batch.cpp) ends
// when a step of it fails: the call returns the error and every request it had
// not settled reports it too, with no iterations.  The steps that would touch
// the GPU before the failure are replaced by the stand-ins below and the arena
// is host memory, so nothing is ever launched.  Built by
// tests/test_lsq_batch_status.py.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <vector>

static int memcpys, fail_memcpy = 1 << 30;
static hipError_t test_memcpy(void*, const void*, size_t, hipMemcpyKind, hipStream_t) {
  return memcpys++ < fail_memcpy ? hipSuccess : hipErrorUnknown;
}
static hipError_t test_sync(hipStream_t) { return hipSuccess; }
static hipError_t test_set_device(int) { return hipSuccess; }
#define hipMemcpyAsync test_memcpy
#define hipStreamSynchronize test_sync
#define hipSetDevice test_set_device
#define launch_lsq_copy test_lsq_copy
#include "../../candmc_amd/csrc/batch.cpp"

namespace cqr {
int test_lsq_copy(cqr_ctx* c, const LsqProb*, int, int) { return set_err(c, CQR_ERR_DEVICE, "no copy"); }
}  // namespace cqr

static int fails = 0;

// The call on three requests of two widths, which fails at its `at`-th upload
// or, if that is later, at the copy of A.
static void check(int at) {
  std::vector<cqr_request> rq(3);
  for (int p = 0; p < 3; ++p) {
    cqr_request& r = rq[p];
    r = cqr_request{};
    r.m = r.lda = r.ldb = 300 + p;
    r.n = r.ldx = p < 2 ? 20 : 33;
    r.nrhs = 1;
    // distinct addresses, never dereferenced
    r.A = reinterpret_cast<double*>(uintptr_t(1) << 32 | uintptr_t(p) << 24);
    r.B = reinterpret_cast<double*>(uintptr_t(2) << 32 | uintptr_t(p) << 24);
    r.X = reinterpret_cast<double*>(uintptr_t(3) << 32 | uintptr_t(p) << 24);
  }
  cqr_ctx c;
  std::vector<char> arena(cqr_lstsq_batched_workspace_bytes(3, rq.data()));
  c.ws = arena.data();
  c.ws_bytes = arena.size();
  memcpys = 0;
  fail_memcpy = at;
  int status[3] = {77, 77, 77}, iters[3] = {77, 77, 77};
  double upd[3] = {77.0, 77.0, 77.0};
  const int rc = cqr_lstsq_batched(&c, 3, rq.data(), 4, 1e-12, status, iters, upd);
  for (int p = 0; p < 3; ++p)
    if (rc != CQR_ERR_DEVICE || status[p] != rc || iters[p] != 0 || upd[p] != 0.0) {
      std::printf("FAIL: upload %d fails: rc %d, request %d: status %d, iters %d, update %g\n", at, rc, p, status[p],
                  iters[p], upd[p]);
      ++fails;
    }
}

int main() {
  check(0);        // the first group's table
  check(1);        // the second group's
  check(2);        // the requests' table
  check(1 << 30);  // the copy of A
  if (fails) return 1;
  std::printf("status ok\n");
  return 0;
}
