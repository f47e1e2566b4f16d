// The host path's answers to two device states it must not take for results, on
// the host-only build (stub_runtime.cpp): a panel that gave up (flags bit 3) in a
// call whose columns are all fixed, and a wide step's candidate index past the
// columns.  usage: bad_state panel|index; prints the call's return code.
#define launch_panel_exact model_panel_exact
#define launch_topk_wide model_topk_wide
#include "stub_runtime.cpp"
#undef launch_panel_exact
#undef launch_topk_wide

namespace {
bool g_panel = false;
}

namespace qrdm {
void launch_panel_exact(double* A, int lda, int j, int m, int fjb, double tau_dm, int truncate,
                        double* tau, DevState* st, hipStream_t s, int mode) {
  model_panel_exact(A, lda, j, m, fjb, tau_dm, truncate, tau, st, s, mode);
  if (g_panel) submit(s, [=] { st->flags |= 8; });
}
void launch_topk_wide(const double* work, int nsub, int kmax, double* val[2], int* idx[2],
                      const double** out_val, hipStream_t s) {
  model_topk_wide(work, nsub, kmax, val, idx, out_val, s);
  if (!g_panel) submit(s, [=] { idx[0][0] = 0x7fffffff; });
}
}  // namespace qrdm

int main(int argc, char** argv) {
  g_panel = argc > 1 && strcmp(argv[1], "panel") == 0;
  const int m = 700, n = 300;
  std::vector<double> a((size_t)m * n), tau(n);
  std::vector<int> jp(n, g_panel ? 1 : 0), nc(n, 0);
  const double th[3] = {0.9, 0.15, 0.0};
  printf("%d\n", qrdm_dgeqrdm_dev(102, m, n, a.data(), m, jp.data(), tau.data(), nc.data(), th,
                                  g_panel ? 64 : 128, nullptr));
  return 0;
}
