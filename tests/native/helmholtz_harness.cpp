// Test harness: C entry points over the host set-up of the diagonalised solves
// (channel_flow_amd/csrc/helmholtz.h), loaded by tests/test_helmholtz_host.py.
#include "../../channel_flow_amd/csrc/helmholtz.h"

// x[n] of one half system's v (is_v = 1, rows f of p = 2 ..) or omega_y solve
extern "C" int helmholtz_c(int N, int par, int is_v, double c, double k2, const double* f, double* x) {
  chf::la::HelmholtzHalf h;
  if (!chf::la::helmholtz_half(N, par, h)) return 1;
  if (!chf::la::helmholtz_verify(par, h, c, k2)) return 2;
  chf::la::helmholtz_solve(h, is_v != 0, c, k2, f, x);
  return 0;
}
