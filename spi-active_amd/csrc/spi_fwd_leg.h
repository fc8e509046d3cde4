// Leg elimination (spi_fwd.h) with four lanes per rollout: lane % 4 is a leg, eliminated in the
// same instruction stream with the leg's constants in registers; the four legs' contributions
// to the base are summed by DPP quad steps and the base is solved identically in the four lanes.
// For batches that leave most SIMDs idle, where one wavefront's instruction count is the time:
// 1,010 -> 770 vector instructions per sub-interval against the articulated-body form; 256 candidates
// x 64 segments x H 5 (one wave on every SIMD) 163 -> 126 us.
#pragma once
#include "spi_dyn_leg.h"
#include "spi_fwd.h"

namespace SPI_DYN_NS {

// Parameters of lane i from their rows [25][ld], the base with the legs' axial mass.
__device__ __forceinline__ LaneParams load_params(const float* __restrict__ par, int ld, int i) {
  LaneParams lp;
  lp.base = base_with_legs(make_base_inertia(par[0 * ld + i], par[1 * ld + i], par[2 * ld + i], par[3 * ld + i],
                                             par[4 * ld + i], par[5 * ld + i], par[6 * ld + i], par[7 * ld + i],
                                             par[8 * ld + i], par[9 * ld + i]));
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    lp.kp_s[l] = par[(10 + l) * ld + i];
    lp.kd_s[l] = par[(14 + l) * ld + i];
    lp.fric[l] = par[(18 + l) * ld + i];
  }
#pragma unroll
  for (int g = 0; g < 3; ++g) lp.motor[g] = par[(22 + g) * ld + i];
  return lp;
}

struct ElimTable { LegC<float> k[4]; };
constexpr ElimTable elim_table() { return ElimTable{{leg_c<float>(0), leg_c<float>(1), leg_c<float>(2), leg_c<float>(3)}}; }
static __constant__ ElimTable kElimTab = elim_table();

// forward_dynamics_elim, leg-parallel: k this lane's leg; lp.base is base_with_legs(); foot_force
// (optional) this leg's.  All four lanes of a rollout must be active.
__device__ __forceinline__ void forward_dynamics_elim_leg(const SpiSimArgs& a, const LegParams& lp,
                                                          const LegC<float>& k, const LegState& st,
                                                          const Real* tau_motor, M6& acc0, Real* qdd,
                                                          Real* foot_force = nullptr) {
  const G3 R = quat_to_rot(st.qx, st.qy, st.qz, st.qw);
  const BaseMotion b = base_motion(st.w, st.v, V3{R.m20, R.m21, R.m22}, st.p.z, lp.base);
  Real tau[3];
#pragma unroll
  for (int j = 0; j < 3; ++j)
    tau[j] = joint_friction(tau_motor[j], lp.fric, st.qd[j], a.fric_vel_inv * kTwoLog2e);
  ABI I, t;
  F6 p, pt;
  LegElim e;
  leg_eliminate<false, false>(a, k, b, st.q, st.qd, tau, t, pt, e, &R, foot_force);
  sum4(t);
  sum4(pt.n);
  sum4(pt.f);
  base_terms(lp.base, b, I, p);
  abi_add(I, t);
  const M6 a0 = solve_base(I, F6{-1.0f * (p.n + pt.n), -1.0f * (p.f + pt.f)});
  leg_resolve(k, e, a0, qdd);
  acc0 = base_rate(a0, st.w, st.v, b.up, a.gravity);
}

__device__ __forceinline__ void physics_step_elim_leg(const SpiSimArgs& a, const LegParams& lp, const LegC<float>& k,
                                                      LegState& st, const Real* tau_motor,
                                                      Real* foot_force = nullptr) {
  const Real h = a.dt / Real(a.substeps);
  for (int i = 0; i < a.substeps; ++i) {
    M6 acc0;
    Real qdd[3];
    forward_dynamics_elim_leg(a, lp, k, st, tau_motor, acc0, qdd, foot_force);
    integrate_leg(st, acc0, qdd, h);
  }
}

}  // namespace SPI_DYN_NS
