// Test-only host build of the leg-elimination forward dynamics (spi_fwd.h), in double
// (SPI_HOST_DOUBLE) or float.
#ifdef SPI_HOST_DOUBLE
#define SPI_REAL_T double
#endif
#include "spi_fwd.h"

extern "C" void spi_host_forward_elim(const SpiSimArgs* a, const double* par, const double* s37, const double* tau12,
                                      double* acc18, double* force12) {
  using namespace spi;
  Real p[25], s[37], tau[12], qdd[12], ff[12];
  for (int i = 0; i < 25; ++i) p[i] = Real(par[i]);
  for (int i = 0; i < 37; ++i) s[i] = Real(s37[i]);
  for (int i = 0; i < 12; ++i) tau[i] = Real(tau12[i]);
  LaneParams lp;
  lp.base = base_with_legs(make_base_inertia(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9]));
  for (int l = 0; l < 4; ++l) { lp.kp_s[l] = p[10 + l]; lp.kd_s[l] = p[14 + l]; lp.fric[l] = p[18 + l]; }
  for (int g = 0; g < 3; ++g) lp.motor[g] = p[22 + g];
  State st;
  state_from_root(st, s, s + 13, s + 25, 1);
  M6 a0;
  forward_dynamics_elim(*a, LaneRegs{lp, tau}, st, a0, qdd, ff);
  acc18[0] = a0.w.x; acc18[1] = a0.w.y; acc18[2] = a0.w.z;
  acc18[3] = a0.v.x; acc18[4] = a0.v.y; acc18[5] = a0.v.z;
  for (int j = 0; j < 12; ++j) { acc18[6 + j] = qdd[j]; force12[j] = ff[j]; }
}
