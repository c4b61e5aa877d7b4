// The kernel test harness touches no more of a caller's arrays than there is.
#include "fake_hip.hpp"
extern "C" hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
#include "ktest.cpp"

namespace spq {
int rrqr_form(int, int) { return 1; }
int rrqr_init_tiles(int) { return 1; }
int rrqr_update_cols() { return 16; }
template <> void launch_rrqr_init<double>(hipStream_t, const RrqrDesc<double>*, const int*, int, int) {}
std::vector<double> C(30, 7.0);  // other owners' memory behind the empty matrix
template <> void launch_rrqr_panel<double>(hipStream_t, const RrqrDesc<double>* d, int, int) {
  d->st->done = 1;
  C.assign(30, 8.0);  // it changes meanwhile
}
template <> void launch_rrqr_update<double>(hipStream_t, const RrqrDesc<double>*, const int*, int, int, int) {}
}  // namespace spq

int main() {
  const int k = 30;
  std::vector<double> V((size_t)k * k), tau(k);
  std::vector<int> perm(4, 7);
  int rounds = 0;
  CHECK(ktest_rrqr(k, 0, spq::C.data(), V.data(), tau.data(), 1e-2, 1, perm.data(), &rounds) == 0);
  for (double v : spq::C) CHECK(v == 8.0);
  for (int v : perm) CHECK(v == 7);
  return 0;
}
