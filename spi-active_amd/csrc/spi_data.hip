// Device-resident dataset windows: packs sliding windows of a recorded trajectory straight
// into the rollout kernels' segment records (init state, then per step actions + target).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>

#include "spi_types.h"

namespace {

constexpr int kRow = SPI_STATE_DIM + 12;   // one staged row: state, then action
constexpr int kWinPerBlock = 64;            // windows per workgroup
constexpr int kMaxStagedRows = 320;         // 62,720 bytes of LDS

// Where window w starts.
struct RowTable {      // rows[w]
  const int* rows;
  __device__ __forceinline__ int operator()(int w, int) const { return rows[w]; }
};
struct RowRun {        // first + w
  int first;
  __device__ __forceinline__ int operator()(int w, int) const { return first + w; }
};
// Trajectories back to back, each longer than H: trajectory i starts at row first[i] and its
// windows at window first[i] - i H, so window w starts at row w + i H.
struct RowStore {
  const int* first;
  int n_traj;
  __device__ __forceinline__ int operator()(int w, int H) const {
    int lo = 0, hi = n_traj - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (first[mid] - mid * H <= w) lo = mid; else hi = mid - 1;
    }
    return w + lo * H;
  }
};

// Element e of the record of a window starting at row t, read from the buffers: a record is
// state t, action t, state t + 1, ..., state t + H.
__device__ __forceinline__ float record_elem(const float* states, const float* actions, int t, int e) {
  const int k = e / kRow, c = e - k * kRow;
  return c < SPI_STATE_DIM ? states[static_cast<size_t>(t + k) * SPI_STATE_DIM + c]
                           : actions[static_cast<size_t>(t + k) * 12 + (c - SPI_STATE_DIM)];
}

// Workgroup g packs windows g * 64 .. + 63.  With its rows staged in LDS as (state, action), a
// window's record is the run of `stride` staged floats from its first row on, and the group's
// records are one run of the output, written in float4.  A group is staged when its windows'
// rows lie within `cap` rows of its first one (consecutive windows share all rows but one; a
// group across the end of a trajectory has a gap of H); otherwise each element is read from the
// buffers: short records in one run over the group (5000 random rows, H 1 23 us by window, which
// leaves two thirds of the threads idle, 9 us so), long ones by window (H 400 1,118 us in one run,
// 1,066 by window, its row in a scalar register).  A single short window is not worth staging (H 1 2.8 ->
// 2.4 us).  A window whose rows r .. r + H do not all lie below n_rows is written as NaN and
// nothing outside the buffers is read.  Bound by the output: 64 x 2500 steps, H 20 (646 MB) in
// 151 us; 232 us with a division per element, word stores and groups across trajectories
// read element by element.
constexpr int kShortRecord = 1024;
template <class Rows>
__global__ __launch_bounds__(256) void pack_windows_kernel(const float* __restrict__ states,
                                                           const float* __restrict__ actions, Rows rows, int n_rows,
                                                           int H, int n_windows, int stride, int cap,
                                                           float* __restrict__ out) {
  extern __shared__ float stage[];
  __shared__ int at[kWinPerBlock];      // stage offset of each window's record
  __shared__ int last;
  const int tid = threadIdx.x, w0 = blockIdx.x * kWinPerBlock, nw = min(kWinPerBlock, n_windows - w0);
  const int r0 = rows(w0, H);
  const int rj = tid < nw ? rows(w0 + tid, H) : r0;
  if (tid == 0) last = 0;
  const bool near = (nw > 1 || stride > kShortRecord) && rj >= 0 && r0 >= 0 && rj >= r0 && static_cast<long long>(rj) - r0 + H < cap &&
                    static_cast<long long>(rj) + H < n_rows;
  const bool staged = __syncthreads_and(near);
  float* o = out + static_cast<size_t>(w0) * stride;
  if (staged) {
    if (tid < nw) {
      at[tid] = (rj - r0) * kRow;
      atomicMax(&last, rj - r0);
    }
    __syncthreads();
    const int n_stage = last + H + 1;
    const float* sp = states + static_cast<size_t>(r0) * SPI_STATE_DIM;
    for (int i = tid; i < n_stage * SPI_STATE_DIM; i += 256) {
      const int row = i / SPI_STATE_DIM;
      stage[row * kRow + (i - row * SPI_STATE_DIM)] = sp[i];
    }
    const float* ap = actions + static_cast<size_t>(r0) * 12;
    for (int i = tid; i < n_stage * 12; i += 256) {
      const int row = i / 12;
      stage[row * kRow + SPI_STATE_DIM + (i - row * 12)] = ap[i];
    }
    __syncthreads();
    const int n_out = nw * stride;
    int done = 0;
    if ((reinterpret_cast<uintptr_t>(o) & 15) == 0) {
      float4* o4 = reinterpret_cast<float4*>(o);
      const int n4 = n_out >> 2, qw = 1024 / stride, qe = 1024 - qw * stride;
      int w = 4 * tid / stride, e = 4 * tid - w * stride;
      for (int f = tid; f < n4; f += 256) {
        float v[4];
        if (e + 4 <= stride) {
          const float* x = stage + at[w] + e;
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = x[q];
        } else {
          int ww = w, ee = e;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            v[q] = stage[at[ww] + ee];
            if (++ee == stride) { ee = 0; ++ww; }
          }
        }
        o4[f] = make_float4(v[0], v[1], v[2], v[3]);
        w += qw;
        e += qe;
        if (e >= stride) { e -= stride; ++w; }
      }
      done = n4 << 2;
    }
    for (int f = done + tid; f < n_out; f += 256) {
      const int w = f / stride;
      o[f] = stage[at[w] + (f - w * stride)];
    }
    return;
  }
  if (stride > kShortRecord) {
    for (int w = 0; w < nw; ++w) {
      const int t = rows(w0 + w, H);
      const bool ok = t >= 0 && static_cast<long long>(t) + H < n_rows;
      for (int e = tid; e < stride; e += 256)
        o[static_cast<size_t>(w) * stride + e] = ok ? record_elem(states, actions, t, e) : __int_as_float(0x7fc00000);
    }
    return;
  }
  if (tid < nw) at[tid] = rj >= 0 && static_cast<long long>(rj) + H < n_rows ? rj : -1;
  __syncthreads();
  const int n_out = nw * stride, qw = 256 / stride, qe = 256 - qw * stride;
  int w = tid / stride, e = tid - w * stride;
  for (int f = tid; f < n_out; f += 256) {
    const int t = at[w];
    o[f] = t >= 0 ? record_elem(states, actions, t, e) : __int_as_float(0x7fc00000);
    w += qw;
    e += qe;
    if (e >= stride) { e -= stride; ++w; }
  }
}

template <class Rows>
int pack_launch(const float* states_dev, const float* actions_dev, Rows rows, int n_rows, int horizon, int n_windows,
                float* segments_dev, hipStream_t stream) {
  const int stride = SPI_STATE_DIM + horizon * kRow;
  const int blocks = (n_windows + kWinPerBlock - 1) / kWinPerBlock;
  // room for 64 consecutive windows and one gap of H; 0: longer horizons read the rows directly
  const long long want = kWinPerBlock + 2LL * horizon;
  const int cap = want <= kMaxStagedRows ? static_cast<int>(want) : horizon < kMaxStagedRows ? kMaxStagedRows : 0;
  pack_windows_kernel<<<blocks, 256, static_cast<size_t>(cap) * kRow * sizeof(float), stream>>>(
      states_dev, actions_dev, rows, n_rows, horizon, n_windows, stride, cap, segments_dev);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    spi_set_error(hipGetErrorString(e));
    return SPI_ERR_HIP;
  }
  return SPI_OK;
}

}  // namespace

extern "C" {

int spi_pack_windows(const float* states_dev, const float* actions_dev, int n_steps, int horizon, int first,
                     int n_windows, float* segments_dev, hipStream_t stream) {
  if (n_steps < 0 || horizon < 1 || first < 0 || n_windows < 0 ||
      static_cast<long long>(first) + n_windows + horizon > n_steps ||
      (n_windows > 0 && (!states_dev || !actions_dev || !segments_dev))) {
    spi_set_error("spi_pack_windows: windows must lie inside the trajectory (first + n + horizon <= n_steps)");
    return SPI_ERR_INVALID_ARG;
  }
  if (n_windows == 0) return SPI_OK;
  return pack_launch(states_dev, actions_dev, RowRun{first}, n_steps, horizon, n_windows, segments_dev, stream);
}

int spi_pack_windows_rows(const float* states_dev, const float* actions_dev, int n_rows, const int* rows_dev,
                          int n_windows, int horizon, float* segments_dev, hipStream_t stream) {
  if (n_rows < 0 || horizon < 1 || n_windows < 0 ||
      (n_windows > 0 && (!states_dev || !actions_dev || !rows_dev || !segments_dev))) {
    spi_set_error("spi_pack_windows_rows: bad sizes or null pointer");
    return SPI_ERR_INVALID_ARG;
  }
  if (n_windows == 0) return SPI_OK;
  return pack_launch(states_dev, actions_dev, RowTable{rows_dev}, n_rows, horizon, n_windows, segments_dev, stream);
}

int spi_window_index(int n, const int* traj, const int* counts, const int* first, const float* kp, const float* kd,
                     unsigned char* ends_out, int* traj_out, int* start_out, float* kp_out, float* kd_out,
                     int* rows_out) {
  size_t o = 0;
  for (int k = 0; k < n; ++k) {
    const int c = counts[k];
    for (int i = 0; i < c; ++i) traj_out[o + i] = traj[k];
    for (int i = 0; i < c; ++i) start_out[o + i] = i;
    for (int i = 0; i < c; ++i) kp_out[o + i] = kp[k];
    for (int i = 0; i < c; ++i) kd_out[o + i] = kd[k];
    for (int i = 0; i < c; ++i) ends_out[o + i] = 0;
    if (rows_out)
      for (int i = 0; i < c; ++i) rows_out[o + i] = first[k] + i;
    if (c > 0) ends_out[o + c - 1] = 1;
    o += c > 0 ? c : 0;
  }
  return SPI_OK;
}

int spi_pack_windows_store(const float* states_dev, const float* actions_dev, int n_rows, const int* first_dev,
                           int n_traj, int n_windows, int horizon, float* segments_dev, hipStream_t stream) {
  if (n_rows < 0 || horizon < 1 || n_windows < 0 || n_traj < 1 ||
      static_cast<long long>(n_windows) + static_cast<long long>(n_traj) * horizon != n_rows ||
      (n_windows > 0 && (!states_dev || !actions_dev || !first_dev || !segments_dev))) {
    spi_set_error("spi_pack_windows_store: every trajectory must be longer than the horizon, or a null pointer");
    return SPI_ERR_INVALID_ARG;
  }
  if (n_windows == 0) return SPI_OK;
  return pack_launch(states_dev, actions_dev, RowStore{first_dev, n_traj}, n_rows, horizon, n_windows, segments_dev,
                     stream);
}

}  // extern "C"
