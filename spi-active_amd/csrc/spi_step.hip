// Single physics steps, forward dynamics and record mode (the states of a rollout after every
// control step), one env per lane.  In a source of its own, so that a simulator's trajectories and
// recorded data sets do not change in the last bit when a scoring kernel does.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "spi_fwd_leg.h"
#include "spi_launch.h"

using namespace spi;

namespace {

int rfail(int code, const char* msg) {
  spi_set_error(msg);
  return code;
}

__global__ __launch_bounds__(256) void physics_step_kernel(SpiSimArgs a, const float* __restrict__ par, int ld,
                                                           int n, float* __restrict__ root, float* __restrict__ dof,
                                                           const float* __restrict__ torques,
                                                           float* __restrict__ foot_force) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const LaneParams lp = load_params(par, ld, i);
  State st;
  float* r = root + static_cast<size_t>(i) * 13;
  float* d = dof + static_cast<size_t>(i) * 24;
  state_from_root(st, r, d, d + 1, 2);
  float tau[12];
#pragma unroll
  for (int j = 0; j < 12; ++j) tau[j] = torques[static_cast<size_t>(i) * 12 + j];
  float ff[12];
  physics_step_elim(a, LaneRegs{lp, tau}, st, foot_force ? ff : nullptr);
  state_to_root(st, r, d, d + 1, 2);
  if (foot_force) {
#pragma unroll
    for (int k = 0; k < 12; ++k) foot_force[static_cast<size_t>(i) * 12 + k] = ff[k];
  }
}

// physics_step_kernel with four lanes per env, one per leg.  Up to kLegStepMaxEnvs: an env loop of a
// few thousand envs is one wave's latency, and a leg's share of the step is a third of it (4096
// envs 19 -> 9 us; one wave per SIMD carries 16,384 envs here and 65,536 above).
constexpr int kLegStepMaxEnvs = 32768;
__global__ __launch_bounds__(256) void physics_step_leg_kernel(SpiSimArgs a, const float* __restrict__ par, int ld,
                                                               int n, float* __restrict__ root,
                                                               float* __restrict__ dof,
                                                               const float* __restrict__ torques,
                                                               float* __restrict__ foot_force) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = t >> 2, l = t & 3;
  if (i >= n) return;  // the four lanes of an env leave together
  LegParams lp;
  lp.base = base_with_legs(make_base_inertia(par[0 * ld + i], par[1 * ld + i], par[2 * ld + i], par[3 * ld + i],
                                             par[4 * ld + i], par[5 * ld + i], par[6 * ld + i], par[7 * ld + i],
                                             par[8 * ld + i], par[9 * ld + i]));
  lp.fric = par[(18 + l) * ld + i];
  LegState st;
  float* r = root + static_cast<size_t>(i) * 13;
  float* d = dof + static_cast<size_t>(i) * 24 + 6 * l;
  st.p = V3{r[0], r[1], r[2]};
  st.qx = r[3]; st.qy = r[4]; st.qz = r[5]; st.qw = r[6];
  const G3 R = quat_to_rot(st.qx, st.qy, st.qz, st.qw);
  st.v = mulT(R, V3{r[7], r[8], r[9]});
  st.w = mulT(R, V3{r[10], r[11], r[12]});
  float tau[3], ff[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    st.q[k] = d[2 * k];
    st.qd[k] = d[2 * k + 1];
    tau[k] = torques[static_cast<size_t>(i) * 12 + 3 * l + k];
  }
  physics_step_elim_leg(a, lp, kElimTab.k[l], st, tau, ff);
  if (l == 0) leg_root(st, r);   // after every lane of the quad has read the root (one wavefront)
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    d[2 * k] = st.q[k];
    d[2 * k + 1] = st.qd[k];
    if (foot_force) foot_force[static_cast<size_t>(i) * 12 + 3 * l + k] = ff[k];
  }
}

__global__ __launch_bounds__(256) void forward_dynamics_kernel(SpiSimArgs a, const float* __restrict__ par, int ld,
                                                               int n, const float* __restrict__ root,
                                                               const float* __restrict__ dof,
                                                               const float* __restrict__ torques,
                                                               float* __restrict__ acc, float* __restrict__ foot_force) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const LaneParams lp = load_params(par, ld, i);
  State st;
  state_from_root(st, root + static_cast<size_t>(i) * 13, dof + static_cast<size_t>(i) * 24,
                  dof + static_cast<size_t>(i) * 24 + 1, 2);
  float tau[12], qdd[12], ff[12];
#pragma unroll
  for (int j = 0; j < 12; ++j) tau[j] = torques[static_cast<size_t>(i) * 12 + j];
  M6 a0;
  // one evaluation, bound by its memory and launch: accurate angles cost it nothing
  forward_dynamics_elim(a, LaneRegsT<true>{lp, tau}, st, a0, qdd, foot_force ? ff : nullptr);
  float* o = acc + static_cast<size_t>(i) * 18;
  o[0] = a0.w.x; o[1] = a0.w.y; o[2] = a0.w.z; o[3] = a0.v.x; o[4] = a0.v.y; o[5] = a0.v.z;
#pragma unroll
  for (int j = 0; j < 12; ++j) o[6 + j] = qdd[j];
  if (foot_force) {
#pragma unroll
    for (int k = 0; k < 12; ++k) foot_force[static_cast<size_t>(i) * 12 + k] = ff[k];
  }
}

// Record mode: per-lane params, initial state and action sequence; state after every control step.
__global__ __launch_bounds__(256) void simulate_kernel(SpiSimArgs a, const float* __restrict__ par, int ld, int n,
                                                       const float* __restrict__ init,
                                                       const float* __restrict__ actions, int T,
                                                       float* __restrict__ states) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const LaneParams lp = load_params(par, ld, i);
  State st;
  const float* s0 = init + static_cast<size_t>(i) * SPI_STATE_DIM;
  state_from_root(st, s0, s0 + 13, s0 + 25, 1);
  for (int t = 0; t < T; ++t) {
    float act[12];
#pragma unroll
    for (int j = 0; j < 12; ++j) act[j] = actions[(static_cast<size_t>(i) * T + t) * 12 + j];
    for (int d = 0; d < a.decimation; ++d) {
      float tau[12];
      control_torques(a, lp, act, st, tau);
      physics_step_elim(a, LaneRegs{lp, tau}, st, nullptr);
    }
    float* o = states + (static_cast<size_t>(i) * T + t) * SPI_STATE_DIM;
    state_to_root(st, o, o + 13, o + 25, 1);
  }
}

int launched() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SPI_OK : rfail(SPI_ERR_HIP, hipGetErrorString(e));
}

}  // namespace

extern "C" {

int spi_physics_step(const SpiSimArgs* sim, const float* params_dev, int ld, int n, float* root_dev,
                     float* dof_state_dev, const float* torques_dev, float* foot_force_dev, hipStream_t stream) {
  if (!spi_launch::sim_args_ok(sim)) return rfail(SPI_ERR_INVALID_ARG, "spi_physics_step: invalid SpiSimArgs");
  if (n < 0 || ld < n || !params_dev || !root_dev || !dof_state_dev || !torques_dev)
    return rfail(SPI_ERR_INVALID_ARG, "spi_physics_step: bad sizes or null pointer");
  if (n == 0) return SPI_OK;
  if (n <= kLegStepMaxEnvs)
    physics_step_leg_kernel<<<(n + 63) / 64, 256, 0, stream>>>(*sim, params_dev, ld, n, root_dev, dof_state_dev,
                                                               torques_dev, foot_force_dev);
  else
    physics_step_kernel<<<(n + 255) / 256, 256, 0, stream>>>(*sim, params_dev, ld, n, root_dev, dof_state_dev,
                                                            torques_dev, foot_force_dev);
  return launched();
}

int spi_forward_dynamics(const SpiSimArgs* sim, const float* params_dev, int ld, int n, const float* root_dev,
                         const float* dof_state_dev, const float* torques_dev, float* acc_dev, float* foot_force_dev,
                         hipStream_t stream) {
  if (!spi_launch::sim_args_ok(sim)) return rfail(SPI_ERR_INVALID_ARG, "spi_forward_dynamics: invalid SpiSimArgs");
  if (n < 0 || ld < n || !params_dev || !root_dev || !dof_state_dev || !torques_dev || !acc_dev)
    return rfail(SPI_ERR_INVALID_ARG, "spi_forward_dynamics: bad sizes or null pointer");
  if (n == 0) return SPI_OK;
  forward_dynamics_kernel<<<(n + 255) / 256, 256, 0, stream>>>(*sim, params_dev, ld, n, root_dev, dof_state_dev,
                                                              torques_dev, acc_dev, foot_force_dev);
  return launched();
}

int spi_simulate(const SpiSimArgs* sim, const float* params_dev, int ld, int n, const float* init_dev,
                 const float* actions_dev, int n_steps, float* states_dev, hipStream_t stream) {
  if (!spi_launch::sim_args_ok(sim)) return rfail(SPI_ERR_INVALID_ARG, "spi_simulate: invalid SpiSimArgs");
  if (n < 0 || ld < n || n_steps < 0 || !params_dev || !init_dev || !actions_dev || !states_dev)
    return rfail(SPI_ERR_INVALID_ARG, "spi_simulate: bad sizes or null pointer");
  if (n == 0 || n_steps == 0) return SPI_OK;
  simulate_kernel<<<(n + 255) / 256, 256, 0, stream>>>(*sim, params_dev, ld, n, init_dev, actions_dev, n_steps,
                                                       states_dev);
  return launched();
}

}  // extern "C"
