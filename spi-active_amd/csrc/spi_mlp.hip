// Policy network inference (gfx950): the actor MLP of the locomotion policy (Linear layers with
// ELU between them, spigym/agents/modules/modules.py:47-63; hidden sizes 512-256-128 from
// config/algo/ppo.yaml), one launch per layer with bias and ELU in the epilogue.
// linear_split_kernel: layers of at least 64 inputs and outputs, float32 products formed exactly
// enough on the bf16 matrix pipe.  linear_kernel: the others and the fused last two layers, FP32
// MFMA (v_mfma_f32_32x32x2f32); a workgroup of 4 wavefronts owns a 32-row x 128-column output
// tile, rows of X and the weight rows staged through LDS in K chunks of 64 (even columns, then odd
// ones, 65 words per row, so the operand reads of a wavefront hit 64 distinct banks).  Strict IEEE
// float32 (no fast-math).
// The actor (900 -> 512 -> 256 -> 128 -> 12): 2048 rows 63 -> 54 us, 16384 rows 222 -> 200 us.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <mutex>

#include "spi_types.h"

// Workspace of spi_mlp_forward_noalloc: the ping-pong hidden activations live in this
// file-scope device array (one copy per GPU, held until the process ends) instead of a buffer
// the caller allocates.  In host code the name stands for the symbol, not for a device
// address: the address of the current device's copy comes from hipGetSymbolAddress.
static __device__ __align__(256) float scratch[SPI_MLP_SCRATCH_FLOATS];

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kCols = 128;   // output columns per workgroup (4 wavefronts x MFMA N)
constexpr int kKc = 64;      // K chunk staged per pass
constexpr int kPad = kKc + 1;
constexpr int kMaxLayers = 8;
constexpr int kMaxRingK = 1024;  // widest ring-gathered input

// LDS slot of tile element (row, k): the even columns of a row first, then the odd ones, so
// the MFMA operand reads of a wavefront (lane -> row l % 32, column kk + l / 32) cover 64
// distinct banks: row * 65 + 32 (l / 32) + kk / 2.
__device__ __forceinline__ int lds_at(int row, int k) { return row * kPad + ((k & 1) << 5) + (k >> 1); }

// Layer input gathered from a ring of per-step observation terms, stored term-major
// ring[slot][term][m] (m = row, fastest): X[m][k] = clip(ring[slot_k][term_k][m]) with
// slot_k = (head - kmap[k].x) mod n_slots and term_k = kmap[k].y.
struct RingSrc {
  const float* ring;
  int ld;          // row stride of a (slot, term) line: >= M
  int n_slots, n_terms, head;
  const int2* kmap;
  float clip;
};

// LDS slot of element (row, k) of a tile staged in K chunks of kC: the even columns of a row
// first, then the odd ones, rows padded to kC + 1 words (lds_at is the kC = 64 case).
template <int kC> __device__ __forceinline__ int lds_at_c(int row, int k) {
  return row * (kC + 1) + (k & 1) * (kC / 2) + (k >> 1);
}

// Y[m][n] = act(sum_k X[m][k] W[n][k] + b[n]); W row-major [N][K] (torch Linear layout).
// MFMA operands: lane l supplies A[l % 32][k + l / 32] = X-tile element and
// B[k + l / 32][l % 32] = W[n0 + l % 32][k + l / 32]; accumulator r of lane l holds
// D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].  The next K chunk is fetched from global memory
// into registers while the MFMAs consume the current one from LDS.
// kSrc 0: X row-major, scalar loads; 1: X and W rows 16-byte aligned with K % 4 == 0, float4
// loads; 2: X gathered from a RingSrc (32 consecutive rows of one column per load), W as in 1;
// 3: as 2 with float4 loads along the rows.
// Split K (kS groups of 4 wavefronts, 256 kS threads): group g multiplies chunks g, g + kS,
// g + 2 kS, ... of K (chunks of 64, of 32 for kS = 4) into its own accumulators from its own
// LDS tiles; at the end groups 1 .. kS-1 hand theirs to group 0 through LDS, which adds them in
// group order (a fixed order: the result does not depend on timing) and runs the epilogue.
// For small batches, whose 32 x 128 tiles leave SIMDs idle or alone: kS wavefronts per SIMD
// hide each other's load latency and each K loop is kS times shorter.  kS = 1 is the plain
// tile loop.
// kFuse: the layer's outputs (N <= 128: one column tile) never leave the workgroup; after the
// epilogue (bias, ELU) they go to LDS and the workgroup computes the next, last layer from them
// (W2 [N2][N], b2, N2 <= 32, no activation: for each row and output, multiply-add chains over
// the two halves of the N inputs in index order, then the two halves and the bias in that
// order), writing Y2 [M][N2].
template <bool kElu, int kSrc, int kS, bool kFuse = false>
__global__ __launch_bounds__(256 * kS) void linear_kernel(const float* __restrict__ X, int ldx, RingSrc rs, int M, int K,
                                                          const float* __restrict__ W, const float* __restrict__ b, int N,
                                                          float* __restrict__ Y, int ldy,
                                                          const float* __restrict__ W2 = nullptr,
                                                          const float* __restrict__ b2 = nullptr, int N2 = 0,
                                                          float* __restrict__ Y2 = nullptr) {
  constexpr int kRows = 32;
  constexpr int kKs = kS == 4 ? 32 : kKc;              // K chunk of one group
  constexpr int kPs = kKs + 1;
  constexpr int kGroupFloats = (kRows + kCols) * kPs;
  static_assert(kS == 1 || (kS - 1) * 16 * 256 <= kS * kGroupFloats, "reduction buffer fits the tiles");
  static_assert(kRows * (kCols + 1) + 2 * kRows * 32 + 32 * (kCols + 1) <= (kFuse ? kS * kGroupFloats : 1 << 20), "a fused tail's tile fits the tiles");
  __shared__ float smem[kS * kGroupFloats];
  __shared__ int Kr[kSrc >= 2 ? kMaxRingK : 1];       // ring line of each input column
  const int m0 = blockIdx.x * kRows, n0 = blockIdx.y * kCols;
  const int grp = threadIdx.x >> 8, tid = threadIdx.x & 255, wave = tid >> 6, lane = tid & 63;
  float* As = smem + grp * kGroupFloats;
  float* Ws = As + kRows * kPs;
  const int col = lane & 31, half = lane >> 5;
  const bool live = n0 + wave * 32 < N;  // uniform per wavefront
  if (kSrc >= 2) {
    // any table entry is folded into the ring: slots back in [0, n_slots), term in [0, n_terms)
    for (int k = threadIdx.x; k < K; k += 256 * kS) {
      const int2 km = rs.kmap[k];
      const int back = min(max(km.x, 0), rs.n_slots - 1);
      const int slot = rs.head >= back ? rs.head - back : rs.head - back + rs.n_slots;
      Kr[k] = slot * rs.n_terms + min(max(km.y, 0), rs.n_terms - 1);
    }
    __syncthreads();
  }
  floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  constexpr int kV = kSrc == 0 ? 1 : 4;                // floats per W (and row-major X) load
  constexpr int kTPR = kKs / kV;                       // threads per tile row
  constexpr int kRowStep = 256 / kTPR;                 // rows covered by one pass of the group
  constexpr int kAV = kSrc == 2 ? 1 : kV;
  // ring gather: thread -> row (tid % 32), columns kk_r + i * 8; float4 ring gather (kSrc 3):
  // thread -> rows 4 (tid % 8) .. + 3, columns kk4 + i * 32
  constexpr int kGStep = 256 / kRows;
  constexpr int kG4 = kRows / 4, kG4Step = 256 / kG4;
  constexpr int kAPer = kSrc == 2 ? kRows * kKs / 256 : (kSrc == 3 ? kRows * kKs / 1024 : kRows / kRowStep);
  constexpr int kWPer = kCols / kRowStep;
  static_assert(kAPer >= 1 && kWPer >= 1, "tile staging covers the chunk");
  const int r0 = tid / kTPR, c0 = (tid % kTPR) * kV;
  const int gm_r = m0 + tid % kRows, kk_r = tid / kRows;
  const int m4 = (tid % kG4) * 4, kk4 = tid / kG4;
  float ra[kAPer][kAV], rw[kWPer][kV];
  auto fetch = [&](int k0) {
    const int gk = k0 + c0;
#pragma unroll
    for (int i = 0; i < kAPer; ++i) {
      if (kSrc == 2) {
        const int k = k0 + kk_r + kGStep * i;
        float v = 0.0f;
        if (gm_r < M && k < K) {
          v = rs.ring[static_cast<size_t>(Kr[k]) * rs.ld + gm_r];
          v = fminf(fmaxf(v, -rs.clip), rs.clip);
        }
        ra[i][0] = v;
      } else if (kSrc == 3) {
        const int k = k0 + kk4 + kG4Step * i;
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (m0 + m4 < M && k < K)
          v = *reinterpret_cast<const float4*>(rs.ring + static_cast<size_t>(Kr[k]) * rs.ld + m0 + m4);
        ra[i][0] = fminf(fmaxf(v.x, -rs.clip), rs.clip);
        ra[i][kAV > 1 ? 1 : 0] = fminf(fmaxf(v.y, -rs.clip), rs.clip);
        ra[i][kAV > 2 ? 2 : 0] = fminf(fmaxf(v.z, -rs.clip), rs.clip);
        ra[i][kAV > 3 ? 3 : 0] = fminf(fmaxf(v.w, -rs.clip), rs.clip);
      } else {
        const int gm = m0 + r0 + i * kRowStep;
        if (kSrc == 1) {
          float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          if (gm < M && gk < K) v = *reinterpret_cast<const float4*>(X + static_cast<size_t>(gm) * ldx + gk);
          ra[i][0] = v.x; ra[i][kAV > 1 ? 1 : 0] = v.y; ra[i][kAV > 2 ? 2 : 0] = v.z; ra[i][kAV > 3 ? 3 : 0] = v.w;
        } else {
          ra[i][0] = (gm < M && gk < K) ? X[static_cast<size_t>(gm) * ldx + gk] : 0.0f;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kWPer; ++i) {
      const int gn = n0 + r0 + i * kRowStep;
      if (kV == 4) {
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (gn < N && gk < K) v = *reinterpret_cast<const float4*>(W + static_cast<size_t>(gn) * K + gk);
        rw[i][0] = v.x; rw[i][kV > 1 ? 1 : 0] = v.y; rw[i][kV > 2 ? 2 : 0] = v.z; rw[i][kV > 3 ? 3 : 0] = v.w;
      } else {
        rw[i][0] = (gn < N && gk < K) ? W[static_cast<size_t>(gn) * K + gk] : 0.0f;
      }
    }
  };
  // every group runs the same number of passes (chunks past K load zeros), so the barriers match
  const int n_pass = (K + kKs * kS - 1) / (kKs * kS);
  fetch(grp * kKs);
  for (int it = 0; it < n_pass; ++it) {
#pragma unroll
    for (int i = 0; i < kAPer; ++i) {
      if (kSrc == 2) {
        As[lds_at_c<kKs>(tid % kRows, kk_r + kGStep * i)] = ra[i][0];
      } else if (kSrc == 3) {
#pragma unroll
        for (int v = 0; v < 4; ++v) As[lds_at_c<kKs>(m4 + v, kk4 + kG4Step * i)] = ra[i][v];
      } else {
#pragma unroll
        for (int v = 0; v < kAV; ++v) As[lds_at_c<kKs>(r0 + i * kRowStep, c0 + v)] = ra[i][v];
      }
    }
#pragma unroll
    for (int i = 0; i < kWPer; ++i)
#pragma unroll
      for (int v = 0; v < kV; ++v) Ws[lds_at_c<kKs>(r0 + i * kRowStep, c0 + v)] = rw[i][v];
    __syncthreads();
    if (it + 1 < n_pass) fetch(((it + 1) * kS + grp) * kKs);
    if (live) {
      const float* ap = As + col * kPs + (kKs / 2) * half;
      const float* bp = Ws + (wave * 32 + col) * kPs + (kKs / 2) * half;
#pragma unroll
      for (int kk = 0; kk < kKs; kk += 2)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ap[kk / 2], bp[kk / 2], acc, 0, 0, 0);
    }
    __syncthreads();
  }
  if (kS > 1) {
    // the loop ended on a barrier: the tiles are free; groups 1 .. kS-1 -> [kS-1][16][256]
    float* red = smem;
    if (grp > 0 && live) {
#pragma unroll
      for (int r = 0; r < 16; ++r) red[((grp - 1) * 16 + r) * 256 + tid] = acc[r];
    }
    __syncthreads();
    if (grp > 0 && !kFuse) return;
    if (grp == 0 && live) {
      for (int g = 1; g < kS; ++g)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] += red[((g - 1) * 16 + r) * 256 + tid];
    }
  }
  if (kFuse) {
    // every thread of every group reaches both barriers; group 0 holds the finished tile
    constexpr int kHs = kCols + 1;
    float* h = smem;                                   // [32][kHs] after the reduction reads
    float* part = h + kRows * kHs;                     // [2][32][32] partial sums of the last layer
    // the last layer's weights, each read 32 times: from global memory the 64-deep chains waited
    // on a load every 8 steps
    float* w2s = part + 2 * kRows * 32;                // [N2][kHs]
    __syncthreads();
    for (int u = threadIdx.x; u < N2 * N; u += blockDim.x) {
      const int j = u / N;
      w2s[j * kHs + (u - j * N)] = W2[u];
    }
    if (grp == 0) {
      const int gn = wave * 32 + col;
      const float bias = gn < N ? b[gn] : 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 8 * (r >> 2) + 4 * half + (r & 3);
        float v = 0.0f;
        if (live && gn < N) {
          v = acc[r] + bias;
          if (kElu) v = v > 0.0f ? v : expm1f(v);
        }
        h[row * kHs + gn] = v;
      }
    }
    __syncthreads();
    // every thread: partial sums over the two halves of the N inputs, (half, row, output) per
    // thread, then half 0 + half 1 + bias in that order
    const int nh = (N + 1) / 2;
    for (int u = threadIdx.x; u < 2 * kRows * N2; u += blockDim.x) {
      const int q = u / (kRows * N2), rem = u - q * (kRows * N2), row = rem / N2, j = rem - row * N2;
      const int k0 = q * nh, k1 = min(N, k0 + nh);
      const float* hr = h + row * kHs;
      const float* w2 = w2s + j * kHs;
      float sum = 0.0f;
#pragma unroll 8
      for (int k = k0; k < k1; ++k) sum = fmaf(hr[k], w2[k], sum);
      part[(q * kRows + row) * 32 + j] = sum;
    }
    __syncthreads();
    for (int u = threadIdx.x; u < kRows * N2; u += blockDim.x) {
      const int row = u / N2, j = u - row * N2, gm = m0 + row;
      if (gm < M) Y2[static_cast<size_t>(gm) * N2 + j] = (part[row * 32 + j] + part[(kRows + row) * 32 + j]) + b2[j];
    }
    return;
  }
  if (!live) return;
  const int gn = n0 + wave * 32 + col;
  if (gn >= N) return;
  const float bias = b[gn];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int gm = m0 + 8 * (r >> 2) + 4 * half + (r & 3);
    if (gm < M) {
      float v = acc[r] + bias;
      if (kElu) v = v > 0.0f ? v : expm1f(v);
      Y[static_cast<size_t>(gm) * ldy + gn] = v;
    }
  }
}

// Groups of 4 wavefronts per 32 x 128 tile: split K while the tiles alone would leave SIMDs
// idle or with one wavefront (kS needs K >= 128: a chunk per group).
int split_for(int M, int K, int N) {
  const long long tiles = static_cast<long long>((M + 31) / 32) * ((N + kCols - 1) / kCols);
  if (K < 128 || tiles >= 512) return 1;
  return tiles <= 128 ? 4 : 2;
}

// float32 products on the bf16 matrix pipe.  A float is exactly the sum of three bf16 values (each
// part rounded to nearest, the next one takes what it left), so a product is nine bf16 products.
// Eight are formed; the ninth, of the two last parts, is below 2^-34 of the product and no larger in
// sum than the rounding of the accumulators.  (With the six largest of truncated parts an output of
// one non-zero input was off by up to 4.1e-7 of itself, always towards zero; now as by one float32
// rounding, 6.0e-8.)  Operands are scaled by 2^16, so that the last part of any float is a bf16,
// subnormal floats' too: unscaled, inputs or weights of 1e-36 lost 5e-5 of the result.  Eight
// v_mfma_f32_32x32x16_bf16 of 32 cycles replace eight v_mfma_f32_32x32x2_f32 of 64.
// The leading products and the seven small ones have an accumulator each, so the leading one adds
// 57 times where the float32 pipe added 450 times for 900 inputs: relative error of such a layer
// against 64 bits 3.8e-7 on the float32 pipe, 1.2e-7 here; with 1, 4 and 16 non-zero inputs 2.53e-8,
// 4.2e-8 and 6.1e-8 there, 2.53e-8, 3.6e-8 and 4.0e-8 here.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
constexpr float kOperandScale = 65536.0f, kResultScale = 1.0f / (kOperandScale * kOperandScale);
struct Split4 { uint2 p[3]; };      // the three parts of four consecutive inputs
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {   // v_cvt_pk_bf16_f32, a in the low half
  return __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a, b}, bf16x2));
}
__device__ __forceinline__ Split4 split4(const float* x) {
  float r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = kOperandScale * x[i];
  Split4 s;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    s.p[q] = make_uint2(bf16_pair(r[0], r[1]), bf16_pair(r[2], r[3]));
    if (q == 2) break;
    r[0] -= __uint_as_float(s.p[q].x << 16);
    r[1] -= __uint_as_float(s.p[q].x & 0xffff0000u);
    r[2] -= __uint_as_float(s.p[q].y << 16);
    r[3] -= __uint_as_float(s.p[q].y & 0xffff0000u);
  }
  return s;
}

// Tile of a workgroup: ids go round-robin over the 8 XCDs, and all column tiles of a row tile go to
// one XCD one after the other, so that X is read from memory once and then from that XCD's L2.
__device__ __forceinline__ void tile_of(int id, int n_tiles, int n_col, int* row, int* col) {
  const int full = (n_tiles / n_col) / 8 * 8 * n_col;   // tiles of whole groups of 8 row tiles
  if (id < full) {
    const int j = id >> 3;
    *row = j / n_col * 8 + (id & 7);
    *col = j % n_col;
  } else {
    *row = id / n_col;
    *col = id % n_col;
  }
}

// linear_kernel's layer on the split products: 4 wavefronts own a 64 x 64 kN output tile, each a
// quarter of 32 x 32 kN.  K goes in chunks of 32 through two LDS buffers: while chunk c is
// multiplied, chunk c + 1 is split into the other buffer and chunks c + 2 and c + 3 are in flight.
// LDS rows are four 16-byte units of 8 columns, unit u of row r at u ^ (r / 2) % 4: the 16-byte
// operand reads of 8 rows and the 8-byte stores of a row's columns each cover the banks once.
// Lane l supplies row l % 32 and columns 8 (l / 32) .. + 7 of both operands.
// A wavefront issues 16 kN MFMAs (32 cycles each) and splits 8 (1 + kN) values (6.5 vector
// instructions of 4 cycles each) per chunk, and the two do not overlap on a SIMD: kN = 2 halves
// the splitting per product where the tiles still fill the chip.  kG groups of 4 wavefronts take
// alternate chunks and add up in group order at the end: for batches of one tile per CU, whose
// wavefronts would sit alone on their SIMDs.
// kSrc 0: X row-major; 1: X gathered from a RingSrc in blocks of 2 rows x 4 columns, float2 along
// the rows (lines 8-byte aligned, ld even); 2: the same blocks in scalar loads.  The accumulation
// order does not depend on the source: dense and ring input give the same bits.
// A result that is not finite (an infinite or NaN operand, or one of 2^112 and more, has no finite
// parts) is formed again on the float32 pipe, by its wavefront together: 16 bad rows of 2048 1220 us
// with a loop per element, 90 us so
// (66 where every batch took the float32 pipe).
constexpr int kSpTile = 64, kSpK = 32;
constexpr int kSpGroupTiles = 256, kSpWideTiles = 1024;   // tiles of 64 x 64
template <bool kElu, int kSrc, int kN, int kG>
__global__ __launch_bounds__(256 * kG, 2) void linear_split_kernel(const float* __restrict__ X, int ldx, RingSrc rs,
                                                                   int M, int K, const float* __restrict__ W,
                                                                   const float* __restrict__ b, int N,
                                                                   float* __restrict__ Y, int ldy) {
  constexpr int kTc = kSpTile * kN, kRowsLds = kSpTile + kTc, kWPer = 2 * kN;
  __shared__ uint4 lds[kG][2][3][kRowsLds * 4];        // [group][buffer][part][X rows, W rows][unit]
  constexpr bool kRing = kSrc != 0;
  __shared__ int Kr[kRing ? kMaxRingK : 1];
  int rb, cb;
  tile_of(blockIdx.x, gridDim.x, (N + kTc - 1) / kTc, &rb, &cb);
  const int m0 = rb * kSpTile, n0 = cb * kTc;
  const int grp = threadIdx.x >> 8, tid = threadIdx.x & 255, wave = tid >> 6, lane = tid & 63;
  const int col = lane & 31, half = lane >> 5;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32 * kN;
  if (kRing) {
    for (int k = threadIdx.x; k < K; k += 256 * kG) {
      const int2 km = rs.kmap[k];
      const int back = min(max(km.x, 0), rs.n_slots - 1);
      const int slot = rs.head >= back ? rs.head - back : rs.head - back + rs.n_slots;
      Kr[k] = slot * rs.n_terms + min(max(km.y, 0), rs.n_terms - 1);
    }
    __syncthreads();
  }
  const int sr = tid >> 3, sc = (tid & 7) * 4;         // row-major: rows sr + 32 i, columns sc .. + 3
  const int gr = (tid & 31) * 2, gc = (tid >> 5) * 4;  // ring: rows gr, gr + 1, columns gc .. + 3
  // rows past the matrix read its last ones (their results are not stored)
  const float* xsrc[2];
  const float* wsrc[kWPer];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    xsrc[i] = kRing ? nullptr : X + static_cast<size_t>(min(m0 + sr + 32 * i, M - 1)) * ldx + sc;
#pragma unroll
  for (int i = 0; i < kWPer; ++i) wsrc[i] = W + static_cast<size_t>(min(n0 + sr + 32 * i, N - 1)) * K + sc;
  const int gq = min(m0 + gr, (M - 1) & ~1);           // rows up to M rounded to 2 exist in every line
  struct Chunk { float x[2][4], w[kWPer][4]; };
  auto load4 = [](float* o, const float* p, bool in) {
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (in) v = *reinterpret_cast<const float4*>(p);
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
  };
  auto fetch_at = [&](Chunk& o, int k0, bool whole) {   // whole: no column at or past K
    const bool in = whole || k0 + sc < K;
#pragma unroll
    for (int i = 0; i < kWPer; ++i) load4(o.w[i], wsrc[i] + k0, in);
    if (!kRing) {
#pragma unroll
      for (int i = 0; i < 2; ++i) load4(o.x[i], xsrc[i] + k0, in);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = k0 + gc + e;
        float2 q = make_float2(0.0f, 0.0f);
        if (whole || k < K) {
          const float* line = rs.ring + static_cast<size_t>(Kr[k]) * rs.ld;
          if (kSrc == 1) q = *reinterpret_cast<const float2*>(line + gq);
          else q = make_float2(line[min(m0 + gr, M - 1)], line[min(m0 + gr + 1, M - 1)]);
        }
        o.x[0][e] = q.x;
        o.x[1][e] = q.y;
      }
    }
  };
  auto fetch = [&](Chunk& o, int c) {                   // chunk c of this group
    const int k0 = (c * kG + grp) * kSpK;
    if (k0 + kSpK <= K) fetch_at(o, k0, true);
    else fetch_at(o, k0, false);
  };
  auto put = [&](const float* v, int buf, int row, int c) {
    const Split4 s = split4(v);
    const int unit = row * 4 + ((c >> 3) ^ ((row >> 1) & 3));
#pragma unroll
    for (int q = 0; q < 3; ++q) reinterpret_cast<uint2*>(&lds[grp][buf][q][unit])[(c >> 2) & 1] = s.p[q];
  };
  auto stage = [&](Chunk& o, int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (kRing) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o.x[i][e] = fminf(fmaxf(o.x[i][e], -rs.clip), rs.clip);
        put(o.x[i], buf, gr + i, gc);
      } else {
        put(o.x[i], buf, sr + 32 * i, sc);
      }
    }
#pragma unroll
    for (int i = 0; i < kWPer; ++i) put(o.w[i], buf, kSpTile + sr + 32 * i, sc);
  };
  floatx16 hi[kN], lo[kN];
#pragma unroll
  for (int n = 0; n < kN; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) hi[n][r] = lo[n][r] = 0.0f;
  auto operand = [&](int buf, int q, int row, int ks) {
    return *reinterpret_cast<const bf16x8*>(&lds[grp][buf][q][row * 4 + ((2 * ks + half) ^ ((row >> 1) & 3))]);
  };
  auto compute = [&](int buf) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 x[3], w[kN][3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        x[q] = operand(buf, q, wr + col, ks);
#pragma unroll
        for (int n = 0; n < kN; ++n) w[n][q] = operand(buf, q, kSpTile + wc + 32 * n + col, ks);
      }
#define SPI_MM(A, P, Q)                                                                                  \
  _Pragma("unroll") for (int n = 0; n < kN; ++n)                                                         \
      A[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[P], w[n][Q], A[n], 0, 0, 0);
      SPI_MM(lo, 2, 1)
      SPI_MM(hi, 0, 0)
      SPI_MM(lo, 1, 2)
      SPI_MM(lo, 2, 0)
      SPI_MM(lo, 0, 2)
      SPI_MM(lo, 1, 1)
      SPI_MM(lo, 1, 0)
      SPI_MM(lo, 0, 1)
#undef SPI_MM
    }
  };
  const int nch = (K + kSpK * kG - 1) / (kSpK * kG);    // per group; chunks past K are zeros
  Chunk even, odd;
  fetch(even, 0);
  fetch(odd, 1);
  stage(even, 0);
  fetch(even, 2);
  __syncthreads();
  for (int c = 0; c < nch; c += 2) {
    compute(0);
    stage(odd, 1);
    fetch(odd, c + 3);
    __syncthreads();
    if (c + 1 < nch) compute(1);
    stage(even, 0);
    fetch(even, c + 4);
    __syncthreads();
  }
  if (kG > 1) {                                        // the loop ended on a barrier: the tiles are free
    static_assert((kG - 1) * kN * 16 * 256 * 4 <= sizeof(lds), "the partial sums fit the tiles");
    float* red = reinterpret_cast<float*>(lds);
    if (grp > 0) {
#pragma unroll
      for (int n = 0; n < kN; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) red[(((grp - 1) * kN + n) * 16 + r) * 256 + tid] = hi[n][r] + lo[n][r];
    }
    __syncthreads();
    if (grp > 0) return;
  }
  // results of the wavefront's tile n that are not finite over again from float32 products, K in
  // steps of 8 (4 columns per half), four steps multiplied while four are in flight; a row's results
  // never depend on the rows beside it
  auto in_float32 = [&](int n, float* y) {
    const int gm = min(m0 + wr + col, M - 1), gn = min(n0 + wc + 32 * n + col, N - 1);
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    struct Step { float x[4][4], w[4][4]; };
    auto load = [&](Step& s, int k0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = k0 + 8 * j + 4 * half;
        const bool in = k < K;
        load4(s.w[j], W + static_cast<size_t>(gn) * K + k, in);
        if (!kRing) {
          load4(s.x[j], X + static_cast<size_t>(gm) * ldx + k, in);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) s.x[j][e] = in ? rs.ring[static_cast<size_t>(Kr[k + e]) * rs.ld + gm] : 0.0f;
        }
      }
    };
    Step s;
    load(s, 0);
    for (int k0 = 0; k0 < K; k0 += 32) {
      Step t;
      load(t, k0 + 32);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kRing ? fminf(fmaxf(s.x[j][e], -rs.clip), rs.clip) : s.x[j][e],
                                                     s.w[j][e], acc, 0, 0, 0);
      s = t;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) y[r] = isfinite(y[r]) ? y[r] : acc[r];
  };
#pragma unroll
  for (int n = 0; n < kN; ++n) {
    const int gn = n0 + wc + 32 * n + col, gm0 = m0 + wr + 4 * half;   // row of register r: gm0 + 8 (r / 4) + r % 4
    float y[16];
    bool finite = true;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      y[r] = hi[n][r] + lo[n][r];
      for (int g = 1; g < kG; ++g) y[r] += reinterpret_cast<const float*>(lds)[(((g - 1) * kN + n) * 16 + r) * 256 + tid];
      y[r] *= kResultScale;
      finite = finite && isfinite(y[r]);
    }
    if (__any(!finite)) in_float32(n, y);
    if (gn < N) {
      const float bias = b[gn];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gm = gm0 + 8 * (r >> 2) + (r & 3);
        if (gm < M) {
          const float v = y[r] + bias;
          Y[static_cast<size_t>(gm) * ldy + gn] = kElu ? (v > 0.0f ? v : expm1f(v)) : v;
        }
      }
    }
  }
}

int mfail(int code, const char* msg) {
  spi_set_error(msg);
  return code;
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// rs.ring != nullptr: X comes from the ring (K % 4 == 0 and W 16-byte aligned required).
int launch_linear(const float* X, int ldx, const RingSrc& rs, int M, int K, const float* W, const float* b, int N,
                  float* Y, int ldy, bool elu, hipStream_t stream) {
  const bool wvec = K % 4 == 0 && aligned16(W);
  const bool xvec = rs.ring ? true : (wvec && ldx % 4 == 0 && aligned16(X));
  if (rs.ring && !wvec)
    return mfail(SPI_ERR_INVALID_ARG, "ring-gathered layer needs K % 4 == 0 and 16-byte aligned weights");
  // rows of the ring read as float4: needs ld % 4 == 0 (then rows up to round4(M) <= ld exist)
  const bool ring4 = rs.ring && rs.ld % 4 == 0 && aligned16(rs.ring);
  if (N >= kSpTile && K >= 2 * kSpK && wvec && xvec) {
    const long long rows = (M + kSpTile - 1) / kSpTile, tiles = rows * ((N + kSpTile - 1) / kSpTile);
    // us of a layer 900 -> 512, two groups / one group per 64 x 64 tile / 64 x 128 tiles / the float32
    // pipe.  A tile per CU or less, two groups share its chunks: 16 rows 20.5 / 23.7 / 37 / 25.5, 256 rows
    // 21.4 / 24.6 / 39 / 26.8, 2048 rows (256 tiles) 24.5 / 26.3 / 40 / 28.4.  Above, one: 4096 rows 44.7 /
    // 40.0 / 43.0 / 44.1.  From two 64 x 128 tiles per CU on, those: 8192 rows 85 / 72 / 68 / 78, 16384
    // rows 168 / 134 / 127 / 131.
    const int shape = tiles <= kSpGroupTiles ? 0 : tiles < kSpWideTiles ? 1 : 2;
#define SPI_SP_G(E, S, NN, G) \
  linear_split_kernel<E, S, NN, G><<<static_cast<int>(rows * ((N + kSpTile * NN - 1) / (kSpTile * NN))), 256 * G, 0, stream>>>( \
      X, ldx, rs, M, K, W, b, N, Y, ldy)
#define SPI_SP(E, S)                            \
  do {                                          \
    if (shape == 0) SPI_SP_G(E, S, 1, 2);       \
    else if (shape == 1) SPI_SP_G(E, S, 1, 1);  \
    else SPI_SP_G(E, S, 2, 1);                  \
  } while (0)
    // float2 along the ring's rows: rows up to M rounded to 2 exist (ld even and >= M)
    const bool ring2 = rs.ring && rs.ld % 2 == 0 && reinterpret_cast<uintptr_t>(rs.ring) % 8 == 0;
    if (ring2) {
      if (elu) SPI_SP(true, 1); else SPI_SP(false, 1);
    } else if (rs.ring) {
      if (elu) SPI_SP(true, 2); else SPI_SP(false, 2);
    } else {
      if (elu) SPI_SP(true, 0); else SPI_SP(false, 0);
    }
#undef SPI_SP_G
#undef SPI_SP
  } else {
    const dim3 grid((M + 31) / 32, (N + kCols - 1) / kCols);
    const int split = split_for(M, K, N);
#define SPI_LINEAR_S(E, S, P) linear_kernel<E, S, P><<<grid, 256 * P, 0, stream>>>(X, ldx, rs, M, K, W, b, N, Y, ldy)
#define SPI_LINEAR(E, S)            \
  do {                              \
    if (split == 4)                 \
      SPI_LINEAR_S(E, S, 4);        \
    else if (split == 2)            \
      SPI_LINEAR_S(E, S, 2);        \
    else                            \
      SPI_LINEAR_S(E, S, 1);        \
  } while (0)
    if (ring4) {
      if (elu) SPI_LINEAR(true, 3); else SPI_LINEAR(false, 3);
    } else if (rs.ring) {
      if (elu) SPI_LINEAR(true, 2); else SPI_LINEAR(false, 2);
    } else if (xvec) {
      if (elu) SPI_LINEAR(true, 1); else SPI_LINEAR(false, 1);
    } else {
      if (elu) SPI_LINEAR(true, 0); else SPI_LINEAR(false, 0);
    }
#undef SPI_LINEAR
#undef SPI_LINEAR_S
  }
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return SPI_OK;
  char buf[256];
  std::snprintf(buf, sizeof(buf), "linear_kernel: %s", hipGetErrorString(e));
  spi_set_error(buf);
  return SPI_ERR_HIP;
}

// The last two layers in one launch (linear_kernel with kFuse) when the second-to-last has at
// most 128 outputs (one column tile) and the last at most 32, and the input is a dense buffer
// with 16-byte rows; returns false (nothing launched) when that does not hold.
bool fused_tail(const float* X, int ldx, int M, int K, const float* W, const float* b, int N, const float* W2,
                const float* b2, int N2, float* Y2, hipStream_t stream, int* rc) {
  if (N > kCols || N2 > 32 || K % 4 != 0 || ldx % 4 != 0 || !aligned16(W) || !aligned16(X)) return false;
  const RingSrc none{nullptr, 0, 0, 0, 0, nullptr, 0.0f};
  const dim3 grid((M + 31) / 32, 1);
  const int split = split_for(M, K, N);
  if (split == 4)
    linear_kernel<true, 1, 4, true><<<grid, 1024, 0, stream>>>(X, ldx, none, M, K, W, b, N, nullptr, 0, W2, b2, N2, Y2);
  else if (split == 2)
    linear_kernel<true, 1, 2, true><<<grid, 512, 0, stream>>>(X, ldx, none, M, K, W, b, N, nullptr, 0, W2, b2, N2, Y2);
  else
    linear_kernel<true, 1, 1, true><<<grid, 256, 0, stream>>>(X, ldx, none, M, K, W, b, N, nullptr, 0, W2, b2, N2, Y2);
  const hipError_t e = hipGetLastError();
  *rc = e == hipSuccess ? SPI_OK : mfail(SPI_ERR_HIP, hipGetErrorString(e));
  return true;
}

long long param_floats(int n_layers, const int* dims) {
  if (n_layers < 1 || n_layers > kMaxLayers || !dims) return -1;
  long long n = 0;
  for (int l = 0; l < n_layers; ++l) {
    if (dims[l] < 1 || dims[l + 1] < 1) return -1;
    n += static_cast<long long>(dims[l + 1]) * dims[l] + dims[l + 1];
  }
  return n;
}

int widest_hidden(int n_layers, const int* dims) {
  int w = 0;
  for (int l = 1; l < n_layers; ++l) w = dims[l] > w ? dims[l] : w;
  return w;
}

int mlp_layers(const float* x_dev, const RingSrc& rs, int M, int n_layers, const int* dims, const float* params_dev,
               float* work_dev, long long work_floats, float* y_dev, hipStream_t stream) {
  if (M < 0 || param_floats(n_layers, dims) < 0 || !params_dev || !y_dev || (n_layers > 1 && !work_dev))
    return mfail(SPI_ERR_INVALID_ARG, "spi_mlp_forward: bad arguments");
  const int widest = widest_hidden(n_layers, dims);
  if (work_floats < 2LL * M * widest) return mfail(SPI_ERR_INVALID_ARG, "spi_mlp_forward: work buffer too small");
  for (int l = 0; l <= n_layers; ++l)
    if (static_cast<long long>(M) * dims[l] > 0x7fffffffLL)
      return mfail(SPI_ERR_TOO_LARGE, "spi_mlp_forward: activations exceed 2^31 elements");
  if (M == 0) return SPI_OK;
  const float* in = x_dev;
  const float* p = params_dev;
  for (int l = 0; l < n_layers; ++l) {
    const int K = dims[l], N = dims[l + 1];
    const bool last = l == n_layers - 1;
    if (l > 0 && l == n_layers - 2) {                 // hidden layer + output layer in one launch
      const float* p2 = p + static_cast<size_t>(N) * K + N;
      const int N2 = dims[l + 2];
      int rc = SPI_OK;
      if (fused_tail(in, K, M, K, p, p + static_cast<size_t>(N) * K, N, p2, p2 + static_cast<size_t>(N2) * N, N2,
                     y_dev, stream, &rc))
        return rc;
    }
    float* out = last ? y_dev : work_dev + static_cast<size_t>(l & 1) * M * widest;
    const RingSrc none{nullptr, 0, 0, 0, 0, nullptr, 0.0f};
    const int rc = launch_linear(in, K, l == 0 ? rs : none, M, K, p, p + static_cast<size_t>(N) * K, N, out, N,
                                 !last, stream);
    if (rc != SPI_OK) return rc;
    p += static_cast<size_t>(N) * K + N;
    in = out;
  }
  return SPI_OK;
}

}  // namespace

extern "C" {

long long spi_mlp_param_floats(int n_layers, const int* dims) { return param_floats(n_layers, dims); }

long long spi_mlp_work_floats(int M, int n_layers, const int* dims) {
  if (M < 0 || param_floats(n_layers, dims) < 0) return -1;
  return 2LL * M * widest_hidden(n_layers, dims);
}

int spi_mlp_forward(const float* x_dev, int M, int n_layers, const int* dims, const float* params_dev, float* work_dev,
                    long long work_floats, float* y_dev, hipStream_t stream) {
  if (!x_dev) return mfail(SPI_ERR_INVALID_ARG, "spi_mlp_forward: null input");
  const RingSrc none{nullptr, 0, 0, 0, 0, nullptr, 0.0f};
  return mlp_layers(x_dev, none, M, n_layers, dims, params_dev, work_dev, work_floats, y_dev, stream);
}

int spi_mlp_forward_noalloc(const float* x_dev, int M, int n_layers, const int* dims, const float* params_dev,
                            float* y_dev, hipStream_t stream) {
  // device address of this GPU's scratch array, looked up once per device with it current
  static std::mutex mu;
  static float* addr[64] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= 64)
    return mfail(SPI_ERR_HIP, "spi_mlp_forward_noalloc: no current device");
  float* work = nullptr;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
      void* ptr = nullptr;
      e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !ptr) {
        char buf[256];
        std::snprintf(buf, sizeof(buf), "spi_mlp_forward_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
        return mfail(SPI_ERR_HIP, buf);
      }
      addr[dev] = static_cast<float*>(ptr);
    }
    work = addr[dev];
  }
  if (!x_dev) return mfail(SPI_ERR_INVALID_ARG, "spi_mlp_forward_noalloc: null input");
  if (M < 0 || param_floats(n_layers, dims) < 0)
    return mfail(SPI_ERR_INVALID_ARG, "spi_mlp_forward_noalloc: bad arguments");
  if (2LL * M * widest_hidden(n_layers, dims) > SPI_MLP_SCRATCH_FLOATS)
    return mfail(SPI_ERR_TOO_LARGE, "spi_mlp_forward_noalloc: 2 * M * (widest hidden layer) exceeds "
                                    "SPI_MLP_SCRATCH_FLOATS; use spi_mlp_forward with a caller workspace");
  const RingSrc none{nullptr, 0, 0, 0, 0, nullptr, 0.0f};
  return mlp_layers(x_dev, none, M, n_layers, dims, params_dev, work, SPI_MLP_SCRATCH_FLOATS, y_dev, stream);
}

int spi_mlp_forward_ring(const float* ring_dev, int ld, int n_slots, int n_terms, int head, const int* kmap_dev,
                         float clip, int M, int n_layers, const int* dims, const float* params_dev, float* work_dev,
                         long long work_floats, float* y_dev, hipStream_t stream) {
  if (!ring_dev || !kmap_dev || ld < M || n_slots < 1 || n_terms < 1 || head < 0 || head >= n_slots ||
      !(clip > 0.0f) || reinterpret_cast<uintptr_t>(kmap_dev) % 8 != 0 || !dims || dims[0] > kMaxRingK)
    return mfail(SPI_ERR_INVALID_ARG, "spi_mlp_forward_ring: bad ring arguments (input width <= 1024)");
  const RingSrc rs{ring_dev, ld, n_slots, n_terms, head, reinterpret_cast<const int2*>(kmap_dev), clip};
  return mlp_layers(nullptr, rs, M, n_layers, dims, params_dev, work_dev, work_floats, y_dev, stream);
}

}  // extern "C"
