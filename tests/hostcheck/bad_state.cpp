// The host path's answer to a device state it must not take for a result, on the
// host-only build (stub_runtime.cpp): a panel that gave up (flags bit 3) in a call
// whose columns are all fixed.  Prints the call's return code.
#define launch_panel_exact model_panel_exact
#include "stub_runtime.cpp"
#undef launch_panel_exact

namespace qrdm {
void launch_panel_exact(double* A, int lda, int j, int m, int fjb, double tau_dm, int truncate,
                        double* tau, DevState* st, hipStream_t s, int mode) {
  model_panel_exact(A, lda, j, m, fjb, tau_dm, truncate, tau, st, s, mode);
  submit(s, [=] { st->flags |= 8; });
}
}  // namespace qrdm

int main() {
  const int m = 700, n = 300;
  std::vector<double> a((size_t)m * n), tau(n);
  std::vector<int> jp(n, 1), nc(n, 0);
  const double th[3] = {0.9, 0.15, 0.0};
  printf("%d\n", qrdm_dgeqrdm_dev(102, m, n, a.data(), m, jp.data(), tau.data(), nc.data(), th,
                                  64, nullptr));
  return 0;
}
