// Host-side run of rustb_amd/csrc/refine_core.hpp (the cluster Rayleigh-Ritz
// executed per k-point by the GPU refinement kernel).  Test-only.
#include "../../rustb_amd/csrc/refine_core.hpp"

extern "C" void emul_cluster_rr(int n, double* Z, const double* HZ, double* E, double gap_rel) {
  static rtb::C2 buf[7][rtb::kMaxCluster][rtb::kMaxCluster];
  rtb::cluster_rr_one(n, reinterpret_cast<rtb::Cd*>(Z), reinterpret_cast<const rtb::Cd*>(HZ), E, gap_rel, buf);
}

// The c x c problem alone: G, M in; ev and X out.  Returns the Jacobi sweeps (-1:
// G not positive definite).
extern "C" int emul_cluster_small(int c, const double* G, const double* M, double* ev, double* X) {
  static rtb::C2 buf[7][rtb::kMaxCluster][rtb::kMaxCluster];
  for (int a = 0; a < c; ++a)
    for (int b = 0; b < c; ++b) {
      buf[0][a][b] = {G[2 * (a * c + b)], G[2 * (a * c + b) + 1]};
      buf[1][a][b] = {M[2 * (a * c + b)], M[2 * (a * c + b) + 1]};
    }
  int sweeps = 0;
  if (!rtb::cluster_rr_small(c, buf, ev, &sweeps)) return -1;
  for (int a = 0; a < c; ++a)
    for (int b = 0; b < c; ++b) {
      X[2 * (a * c + b)] = buf[6][a][b].re;
      X[2 * (a * c + b) + 1] = buf[6][a][b].im;
    }
  return sweeps;
}
