// Command sequences of the active-exploration optimizer: one thread per (trial, step), all
// command dimensions of the step.  Strict IEEE float32 arithmetic in the order of the
// reference's numpy code, so the sequences match it to float rounding.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>

#include "spi_types.h"

namespace {

int cfail(int code, const char* msg) {
  spi_set_error(msg);
  return code;
}

int n_params_of(const SpiCommandSpec& c) {
  switch (c.mode) {
    case SPI_COMMAND_CONSTANT: return c.n_sampled * c.n_updates;
    case SPI_COMMAND_POLYNOMIAL: return c.n_updates * c.n_sampled * (c.poly_degree + 1);
    case SPI_COMMAND_BEZIER: return c.n_updates * c.n_sampled * c.n_bezier;
    default: return -1;
  }
}

__device__ float binom_f(int n, int k) {   // C(n, k) as the reference forms it: product, then int
  if (k > n - k) k = n - k;
  double r = 1.0;
  for (int i = 0; i < k; ++i) r *= static_cast<double>(n - i) / (i + 1);
  return static_cast<float>(static_cast<long long>(r));
}

constexpr int kMaxBasis = 8;    // polynomial degree + 1 or Bezier points held in registers

// A step's place in its update window (u, position t) and its power or Bernstein basis, formed once
// per step (unrolled over kMaxBasis with guards, so that it stays in registers).
struct StepBasis { int u, nb; float t, b[kMaxBasis]; };
__device__ __forceinline__ StepBasis step_basis(const SpiCommandSpec& c, int step) {
  StepBasis r;
  const int S = c.steps_per_update;
  r.u = step / S;
  const int i = step - r.u * S;
  // np.linspace(0, 1, S, dtype=float32): computed in float64, then rounded
  const float t = S > 1 ? static_cast<float>(static_cast<double>(i) / (S - 1)) : 0.0f;
  r.t = t;
  r.nb = c.mode == SPI_COMMAND_POLYNOMIAL ? c.poly_degree + 1 : c.mode == SPI_COMMAND_BEZIER ? c.n_bezier : 0;
  if (c.mode == SPI_COMMAND_POLYNOMIAL) {
#pragma unroll
    for (int q = 0; q < kMaxBasis; ++q)
      if (q < r.nb) r.b[q] = q == 0 ? 1.0f : powf(t, static_cast<float>(q));
  } else if (c.mode == SPI_COMMAND_BEZIER) {
    const int n = r.nb - 1;
    const float omt = 1.0f - t;
#pragma unroll
    for (int j = 0; j < kMaxBasis; ++j)
      if (j <= n)
        r.b[j] = binom_f(n, j) * (j == 0 ? 1.0f : powf(t, static_cast<float>(j))) *
                 (n - j == 0 ? 1.0f : powf(omt, static_cast<float>(n - j)));
  }
  return r;
}

// Command of sampled dimension d (dimension k of the command) of the trial with parameters p.
__device__ __forceinline__ float sampled_command(const SpiCommandSpec& c, const StepBasis& s,
                                                 const float* __restrict__ p, int d, int k) {
  const float lo = c.lo[k], hi = c.hi[k], t = s.t;
  const int nb = s.nb;
  if (c.mode == SPI_COMMAND_CONSTANT) return p[d * c.n_updates + s.u];
  const float* cf = p + (static_cast<size_t>(s.u) * c.n_sampled + d) * nb;
  if (c.mode == SPI_COMMAND_POLYNOMIAL) {
    float poly = 0.0f;
#pragma unroll
    for (int q = 0; q < kMaxBasis; ++q)
      if (q < nb) poly = poly + cf[q] * s.b[q];
    for (int q = kMaxBasis; q < nb; ++q) poly = poly + cf[q] * powf(t, static_cast<float>(q));
    poly = tanhf(poly);
    return lo + (poly + 1.0f) * 0.5f * (hi - lo);
  }
  const int n = nb - 1;
  const float omt = 1.0f - t;
  float acc = 0.0f;
#pragma unroll
  for (int j = 0; j < kMaxBasis; ++j)
    if (j <= n) acc = acc + s.b[j] * cf[j];
  for (int j = kMaxBasis; j <= n; ++j)
    acc = acc + binom_f(n, j) * powf(t, static_cast<float>(j)) *
                    (n - j == 0 ? 1.0f : powf(omt, static_cast<float>(n - j))) * cf[j];
  return fminf(fmaxf(acc, lo), hi);
}

// The sampled dimension that fills command dimension k, -1 for the default.
__device__ __forceinline__ int sampled_slot(const SpiCommandSpec& c, int k) {
  int d = -1;
  for (int m = 0; m < c.n_sampled; ++m)
    if (c.sampled_idx[m] == k) d = m;               // the last listed wins, as the reference's fill loop
  return d;
}

// A workgroup takes 256 consecutive steps of up to `per` consecutive trials: a thread forms its
// step's basis once for all of them, each trial's sampled commands go through LDS, and its run of
// 256 n_dims output words is written in float4 (VEC: n_dims and the steps of a trial make every
// run a multiple of 16 bytes; word by word otherwise).  Bound by the output: 1024 Bezier trials x 1250
// steps x 14 (71.7 MB) in 26 us; 45 us with a basis per (trial, step) and all 14 commands through LDS.
// The streaming stores hold for small outputs too: with a kernel that reads all of it behind, 16, 128
// and 1024 trials of 1250 steps 11.4 -> 9.6, 19.8 -> 17.7 and 68 -> 50 us.
typedef float FloatX4 __attribute__((ext_vector_type(4)));
constexpr int kStepThreads = 256, kTrialsPerBlock = 8;
template <bool VEC>
__global__ __launch_bounds__(kStepThreads) void command_trials_kernel(SpiCommandSpec c, const float* __restrict__ params,
                                                                      int n_trials, int n_params, int T, int per,
                                                                      float* __restrict__ out) {
  __shared__ float val[SPI_MAX_COMMAND_DIMS * (kStepThreads + 1)];   // sampled slots, then the defaults
  __shared__ int2 at[SPI_MAX_COMMAND_DIMS];            // dimension k of step s is val[at[k].x + at[k].y s]
  const int tid = threadIdx.x, step = blockIdx.x * kStepThreads + tid, nd = c.n_dims;
  const int n_steps = min(kStepThreads, T - static_cast<int>(blockIdx.x) * kStepThreads);
  float* def = val + SPI_MAX_COMMAND_DIMS * kStepThreads;
  if (tid < nd) {
    const int d = sampled_slot(c, tid);
    at[tid] = d >= 0 ? make_int2(d * kStepThreads, 1) : make_int2(SPI_MAX_COMMAND_DIMS * kStepThreads + tid, 0);
    def[tid] = c.default_cmd[tid];
  }
  const StepBasis sb = step_basis(c, min(step, T - 1));
  const int b0 = blockIdx.y * per, b1 = min(b0 + per, n_trials);
  // step and dimension of this thread's first W words, and what 256 of these further adds
  constexpr int W = VEC ? 4 : 1;
  const int sv = W * tid / nd, kv = W * tid - sv * nd, ds = W * kStepThreads / nd, dk = W * kStepThreads - ds * nd;
  for (int b = b0; b < b1; ++b) {
    const float* p = params + static_cast<size_t>(b) * n_params;
    for (int d = 0; d < c.n_sampled; ++d) val[d * kStepThreads + tid] = sampled_command(c, sb, p, d, c.sampled_idx[d]);
    __syncthreads();
    float* o = out + (static_cast<size_t>(b) * T + static_cast<size_t>(blockIdx.x) * kStepThreads) * nd;
    const int n_out = n_steps * nd;
    int s0 = sv, k0 = kv;
    for (int e = tid; W * e < n_out; e += kStepThreads) {
      float v[W];
      int s = s0, k = k0;
#pragma unroll
      for (int q = 0; q < W; ++q) {
        const int2 a = at[k];
        v[q] = val[a.x + a.y * s];
        if (++k == nd) { k = 0; ++s; }
      }
      if constexpr (VEC)    // written once, not read here
        __builtin_nontemporal_store(FloatX4{v[0], v[1], v[2], v[3]}, reinterpret_cast<FloatX4*>(o) + e);
      else
        o[e] = v[0];
      s0 += ds;
      k0 += dk;
      if (k0 >= nd) { k0 -= nd; ++s0; }
    }
    __syncthreads();
  }
}

// Short trials, constants: one thread per (trial, step) over the flat run of all trials, its
// commands staged in LDS; the workgroup's 256 steps are one
// contiguous run of the output, written back with consecutive threads on consecutive words.
// Idx: int while the launch has fewer than 2^31 (trial, step) pairs, long long above.
template <typename Idx>
__global__ __launch_bounds__(256) void command_kernel(SpiCommandSpec c, const float* __restrict__ params,
                                                     int n_trials, int n_params, float* __restrict__ out) {
  __shared__ float stage[256 * SPI_MAX_COMMAND_DIMS];
  const Idx T = static_cast<Idx>(c.n_updates) * c.steps_per_update;
  const Idx pairs = static_cast<Idx>(n_trials) * T;
  const Idx base = static_cast<Idx>(blockIdx.x) * blockDim.x;
  const Idx idx = base + threadIdx.x;
  if (idx < pairs) {
    const int b = static_cast<int>(idx / T);
    const StepBasis sb = step_basis(c, static_cast<int>(idx - static_cast<Idx>(b) * T));
    const float* p = params + static_cast<size_t>(b) * n_params;
    float* o = stage + threadIdx.x * c.n_dims;
    for (int k = 0; k < c.n_dims; ++k) o[k] = c.default_cmd[k];
    for (int d = 0; d < c.n_sampled; ++d)      // the last listed wins, as in sampled_slot
      o[c.sampled_idx[d]] = sampled_command(c, sb, p, d, c.sampled_idx[d]);
  }
  __syncthreads();
  const Idx left = pairs - base;
  const int n_out = static_cast<int>((left < static_cast<Idx>(blockDim.x) ? left : static_cast<Idx>(blockDim.x)) *
                                     c.n_dims);
  float* o = out + static_cast<size_t>(base) * c.n_dims;
  for (int e = threadIdx.x; e < n_out; e += blockDim.x) o[e] = stage[e];
}

}  // namespace

extern "C" {

int spi_command_sequences(const SpiCommandSpec* spec, const float* params_dev, int n_trials, int n_params,
                          float* out_dev, hipStream_t stream) {
  if (!spec || spec->n_dims < 1 || spec->n_dims > SPI_MAX_COMMAND_DIMS || spec->n_sampled < 0 ||
      spec->n_sampled > SPI_MAX_COMMAND_DIMS || spec->n_updates < 1 || spec->steps_per_update < 1 ||
      spec->poly_degree < 0 || spec->n_bezier < 1)
    return cfail(SPI_ERR_INVALID_ARG, "spi_command_sequences: bad spec");
  for (int m = 0; m < spec->n_sampled; ++m)
    if (spec->sampled_idx[m] < 0 || spec->sampled_idx[m] >= spec->n_dims)
      return cfail(SPI_ERR_INVALID_ARG, "spi_command_sequences: sampled index out of range");
  const int need = n_params_of(*spec);
  if (need < 0) return cfail(SPI_ERR_INVALID_ARG, "spi_command_sequences: unknown mode");
  if (n_trials < 0 || n_params != need || (n_trials > 0 && (!params_dev || !out_dev)))
    return cfail(SPI_ERR_INVALID_ARG, "spi_command_sequences: n_params does not match the spec");
  const long long pairs = static_cast<long long>(n_trials) * spec->n_updates * spec->steps_per_update;
  if (pairs == 0) return SPI_OK;
  const long long T = static_cast<long long>(spec->n_updates) * spec->steps_per_update;
  // A workgroup per 256 steps of some trials where the basis that these share costs more than the part of
  // the last workgroup that stands idle (4096 trials x 14, us against the flat run): Bezier from 192
  // steps on (195 steps 24.7 / 29.4, 260 32.3 / 35.1, 1250 81 / 142), polynomials with at least two
  // thirds of the threads at work (200 19.2 / 21.4, 520 36.6 / 45.6, 625 47.8 / 55.7; but 265 39.4 / 26.4,
  // 300 32.0 / 29.4), constants, which have no basis, for the wide stores of one workgroup per trial (200
  // 11.4 / 12.6; but 255 15.4 / 14.1, 1250 72 / 50).
  const bool vec = (T * spec->n_dims) % 4 == 0 && reinterpret_cast<uintptr_t>(out_dev) % 16 == 0;
  const long long gx256 = (T + kStepThreads - 1) / kStepThreads * kStepThreads;
  const bool by_trial = T >= 192 && (spec->mode == SPI_COMMAND_BEZIER ? true
                                     : spec->mode == SPI_COMMAND_POLYNOMIAL ? 3 * T >= 2 * gx256
                                                                            : vec && T <= kStepThreads);
  if (by_trial && T <= 0x7fffffffLL - kStepThreads) {
    const unsigned gx = static_cast<unsigned>((T + kStepThreads - 1) / kStepThreads);
    // enough trials per workgroup to share a basis, few enough to leave four workgroups per CU
    const long long groups = static_cast<long long>(gx) * n_trials;
    int per = static_cast<int>(groups / 1024 < kTrialsPerBlock ? groups / 1024 : kTrialsPerBlock);
    if (per < 1) per = 1;
    while ((n_trials + per - 1) / per > 65535) per *= 2;
    const dim3 grid(gx, static_cast<unsigned>((n_trials + per - 1) / per));
    const int Ti = static_cast<int>(T);
    if (vec) command_trials_kernel<true><<<grid, kStepThreads, 0, stream>>>(*spec, params_dev, n_trials, n_params, Ti, per, out_dev);
    else command_trials_kernel<false><<<grid, kStepThreads, 0, stream>>>(*spec, params_dev, n_trials, n_params, Ti, per, out_dev);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return cfail(SPI_ERR_HIP, hipGetErrorString(e));
    return SPI_OK;
  }
  const long long blocks = (pairs + 255) / 256;
  if (blocks > 0x7fffffffLL) return cfail(SPI_ERR_TOO_LARGE, "spi_command_sequences: too large");
  if (blocks * 256 < 0x7fffffffLL)
    command_kernel<int><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(*spec, params_dev, n_trials, n_params,
                                                                           out_dev);
  else
    command_kernel<long long><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(*spec, params_dev, n_trials,
                                                                                 n_params, out_dev);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return cfail(SPI_ERR_HIP, hipGetErrorString(e));
  return SPI_OK;
}

}  // extern "C"
