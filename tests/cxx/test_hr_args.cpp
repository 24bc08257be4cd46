// Host-only check of the reconstruction core's arguments
// (candmc_amd/csrc/hr_kernel.hip): outputs that are formed from U⁻¹ (M2 and
// T⁻ᵀ) are refused without it, before anything is launched.  Built by
// tests/test_hr_args.py.
#include "../../candmc_amd/csrc/cqr_internal.h"

#include <cstdint>
#include <cstdio>

int main() {
  int fails = 0;
  auto check = [&](bool tt, bool m2, bool invtt) {
    cqr_ctx c;
    double* some = reinterpret_cast<double*>(uintptr_t(1) << 32);   // never dereferenced
    cqr::HrCore h{};
    h.Q1top = h.Rroot = h.Atop = h.W = some;
    h.ldq = h.lda = 32;
    h.b = 32;
    if (tt) h.Tt = some;
    if (m2) h.M2 = some;
    if (invtt) h.invTT = some;
    const int rc = cqr::hr_core(&c, h);
    if (rc != CQR_ERR_INVALID) {
      std::printf("FAIL: Tt %d, M2 %d, T^-T %d without U^-1: %d\n", tt, m2, invtt, rc);
      ++fails;
    }
  };
  check(true, true, false);
  check(false, false, true);
  check(true, false, true);
  if (fails) return 1;
  std::printf("hr args ok\n");
  return 0;
}
