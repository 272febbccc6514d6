// Test harness: C entry point over the acceptance of the diagonalised solves
// (channel_flow_amd/csrc/helmholtz.h), loaded by tests/test_helmholtz_accept_host.py.
#include "../../channel_flow_amd/csrc/helmholtz.h"

// 1 when the half system's decomposition, its solutions off by the factor 1 + off, is
// accepted at k^2 = 0, k2lo and k2hi; -1 when there is no decomposition
extern "C" int accept_c(int N, int par, double c, double k2lo, double k2hi, double off) {
  chf::la::HelmholtzHalf h;
  if (!chf::la::helmholtz_half(N, par, h)) return -1;
  for (double& v : h.V) v *= 1.0 + off;
  return chf::la::helmholtz_accept(N, par, h, c, {0.0, k2lo, k2hi});
}
