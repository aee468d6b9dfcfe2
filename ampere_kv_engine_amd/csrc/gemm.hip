// Matrix products y = x W^T for x [rows, k], W [out, k] (row-major, as checkpoints store them).
//
// `linear_tiled` is the plain path: float32 multiply-add on 64x64 output tiles staged through LDS, for any
// mix of float32 / bfloat16 operands and any sizes.  Every output element is one sum over k in ascending order
// inside fixed k-tiles, so a row's result does not depend on how many other rows the call carries.  It is the
// fallback for operand mixes and widths that no matrix-core kernel takes.
//
// `linear_f32_pairs`, `linear_f32_few` and `linear_f32_wide` are the float32 path on the matrix cores (see below).

#include "common.h"
#include "api.h"

using namespace akv;

namespace {

constexpr int kTile = 64;   // output tile edge
constexpr int kDepth = 16;  // k-tile

template <typename TX, typename TW, typename TY>
__global__ __launch_bounds__(256) void linear_tiled_kernel(const TX* __restrict__ x, const TW* __restrict__ w,
                                                           TY* __restrict__ y, int rows, int outs, int k,
                                                           const float* __restrict__ bias) {
  __shared__ float xs[kDepth][kTile + 1];
  __shared__ float ws[kDepth][kTile + 1];
  const int row0 = blockIdx.y * kTile, out0 = blockIdx.x * kTile;
  const int tr = threadIdx.x / 16, tc = threadIdx.x % 16;  // 16 x 16 threads, each a 4 x 4 patch
  float acc[4][4] = {};
  for (int k0 = 0; k0 < k; k0 += kDepth) {
    // 64 x 16 elements of each operand, 4 per thread; out-of-range elements are zeros
    for (int e = threadIdx.x; e < kTile * kDepth; e += 256) {
      const int r = e / kDepth, c = e % kDepth;
      const bool in_k = k0 + c < k;
      xs[c][r] = (in_k && row0 + r < rows) ? to_float(x[static_cast<size_t>(row0 + r) * k + k0 + c]) : 0.f;
      ws[c][r] = (in_k && out0 + r < outs) ? to_float(w[static_cast<size_t>(out0 + r) * k + k0 + c]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kDepth; ++c) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = xs[c][tr * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = ws[c][tc * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = row0 + tr * 4 + i;
    if (r >= rows) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int o = out0 + tc * 4 + j;
      if (o < outs) y[static_cast<size_t>(r) * outs + o] = from_float<TY>(bias != nullptr ? acc[i][j] + bias[o] : acc[i][j]);
    }
  }
}

template <typename TX, typename TW, typename TY>
int launch_tiled(const void* x, const void* w, void* y, int rows, int outs, int k, const float* bias, hipStream_t stream) {
  dim3 grid((outs + kTile - 1) / kTile, (rows + kTile - 1) / kTile);
  linear_tiled_kernel<TX, TW, TY><<<grid, 256, 0, stream>>>(static_cast<const TX*>(x), static_cast<const TW*>(w),
                                                            static_cast<TY*>(y), rows, outs, k, bias);
  return AKV_LAUNCH_STATUS();
}

// ---- float32 on the matrix cores -----------------------------------------------------------------------------------------
// v_mfma_f32_16x16x4_f32 multiplies and adds in float32 at twice the vector units' rate (157 TFLOP/s), with no rounding
// of an operand.  A lane's operands of four such instructions are 16 consecutive bytes of a matrix row: lane (r, g) holds
// elements 16 b + 4 g .. + 3 of row r, and instruction j takes element j of every group g.  All three kernels sum every output
// the same way, so that a row's result depends neither on how many rows a call carries nor on which kernel takes it:
// k is cut into segments of 128, a segment is one chain of instructions in the order (b, j), and the segments' sums are
// added in their order.  (Rows and outputs beyond the matrices repeat the last one and are not stored; elements beyond k are
// zeros and change no sum.)
typedef float floats4 __attribute__((ext_vector_type(4)));
constexpr int kSegment = 128;        // k of one chain
constexpr int kSegmentBlocks = kSegment / 16;

__device__ __forceinline__ floats4 mfma4(const floats4 a, const floats4 b, floats4 sums) {
#pragma unroll
  for (int j = 0; j < 4; ++j) sums = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], sums, 0, 0, 0);
  return sums;
}

// The sums of 16 outputs (4 g .. 4 g + 3 of them in this lane) for row `row`, with their bias, to y.
__device__ __forceinline__ void store_f32(float* __restrict__ y, long row, int out, int outs, floats4 sums,
                                          const float* __restrict__ bias, bool wide_stores) {
  if (bias != nullptr) {
#pragma unroll
    for (int j = 0; j < 4; ++j) sums[j] += bias[min(out + j, outs - 1)];
  }
  float* at = y + row * outs + out;
  if (wide_stores && out + 4 <= outs) {
    *reinterpret_cast<floats4*>(at) = sums;
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (out + j < outs) at[j] = sums[j];
}

// GATED: y = silu(x Wgate^T) * (x Wup^T) of a matrix whose first half is the gate's, in steps of up to 16 rows, where a launch costs as
// much as it does: a block owns as many outputs of either half and forms what the activation's kernel forms from the stored
// product, the same bits (us, the product and the activation's kernel / gated: 3 rows of 6144 x 2048 15.1 / 13.3, 16 rows 23.5 / 20.9, of
// 8192 x 4096 42.9 / 41.6).
__device__ __forceinline__ float silu(float v) { return v / (1.f + expf(-v)); }

// Up to 32 rows: the matrix is read once and its reads are what the product waits for.  A block owns 16 outputs and all of
// k; its waves take a segment each (a second round where k has more than 16), with the whole segment's loads in flight - 8 KB
// a wave, 128 KB a block -, and leave their sums in LDS, where the first waves add them in order.  Rows lie in cache and
// are read by every wave in operand order, without LDS: NT tiles of 16 rows.
template <int NT, bool GATED>
__global__ __launch_bounds__(1024) void linear_f32_few_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             float* __restrict__ y, int rows, int outs, int k, int segments,
                                                             const float* __restrict__ bias, bool wide_stores) {
  static_assert(NT == 1 || !GATED, "");
  extern __shared__ floats4 pieces[];                      // [waves][NT][64]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int out0 = blockIdx.x * (GATED ? 8 : 16);          // (of the result; of the gate's half of the matrix and of the up's eight each)
  const float* wp = w + static_cast<long>(GATED && r >= 8 ? outs + min(out0 + r - 8, outs - 1) : min(out0 + (GATED ? r & 7 : r), outs - 1)) * k + 4 * g;
  const float* xp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) xp[t] = x + static_cast<long>(min(16 * t + r, rows - 1)) * k + 4 * g;
  const floats4 zero = {0.f, 0.f, 0.f, 0.f};
  floats4 total = zero;
  for (int first = 0; first < segments; first += waves) {
    const int segment = first + wave;
    if (segment < segments) {
      const int k0 = segment * kSegment;
      floats4 sums[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) sums[t] = zero;
      if (k0 + kSegment <= k) {
        floats4 a[kSegmentBlocks];
#pragma unroll
        for (int b = 0; b < kSegmentBlocks; ++b) a[b] = *reinterpret_cast<const floats4*>(wp + k0 + 16 * b);
        __builtin_amdgcn_sched_barrier(0);                 // (else the loads are moved down to where they are used)
        floats4 v[kSegmentBlocks][NT];
#pragma unroll
        for (int b = 0; b < kSegmentBlocks; ++b)
#pragma unroll
          for (int t = 0; t < NT; ++t) v[b][t] = *reinterpret_cast<const floats4*>(xp[t] + k0 + 16 * b);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < kSegmentBlocks; ++b)
#pragma unroll
          for (int t = 0; t < NT; ++t) sums[t] = mfma4(a[b], v[b][t], sums[t]);
      } else {
        for (int b = 0; k0 + 16 * b < k; ++b) {
          const int at = k0 + 16 * b;
          const bool inside = at + 4 * g < k;              // (k is a multiple of 4: a group of four is whole or absent)
          const floats4 a = inside ? *reinterpret_cast<const floats4*>(wp + at) : zero;
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const floats4 v = inside ? *reinterpret_cast<const floats4*>(xp[t] + at) : zero;
            sums[t] = mfma4(a, v, sums[t]);
          }
        }
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) pieces[(wave * NT + t) * 64 + lane] = sums[t];
    }
    __syncthreads();
    if (wave < NT) {
      const int there = min(waves, segments - first);
      for (int s = 0; s < there; ++s) total += pieces[(s * NT + wave) * 64 + lane];
    }
    __syncthreads();
  }
  if (wave >= NT) return;                                  // (a block has at least NT waves: the launch sees to it)
  if constexpr (GATED) {
#pragma unroll
    for (int n = 0; n < 4; ++n) total[n] = silu(total[n]) * __shfl_xor(total[n], 32, 64);   // lane (row, g + 2): the up's four
    if (g >= 2) return;
  }
  if (16 * wave + r < rows) store_f32(y, 16 * wave + r, out0 + 4 * g, outs, total, bias, wide_stores);
}

// Up to 8 rows: bound by what the units have on their way from memory; a block a tile of 16 outputs leaves half of them without
// one at 2,048 outputs, and its sixteen waves share a unit with no other block at more.  Here a block owns 8 outputs,
// and an instruction carries two segments of k - its rows 0 .. 7 the outputs' first and its rows 8 .. 15 their second, its
// columns likewise the rows of x, so that two quarters of its sums are the two segments' and the others mean nothing (the matrix
// cores have nothing else to do).  Each sum is the chain that the other kernels form, and the segments are added in their order.
template <bool GATED>
__global__ __launch_bounds__(1024) void linear_f32_pairs_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                               float* __restrict__ y, int rows, int outs, int k, int segments,
                                                               const float* __restrict__ bias, bool wide_stores) {
  extern __shared__ floats4 pieces[];                      // [2 waves][16]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int r = lane & 7, second = lane >> 3 & 1, g = lane >> 4;
  const int out0 = blockIdx.x * (GATED ? 4 : 8);           // (of the result; of the gate's half of the matrix and of the up's four each)
  const float* wp = w + static_cast<long>(GATED && r >= 4 ? outs + min(out0 + r - 4, outs - 1) : min(out0 + (GATED ? r & 3 : r), outs - 1)) * k;
  const float* xp = x + static_cast<long>(min(r, rows - 1)) * k;
  const floats4 zero = {0.f, 0.f, 0.f, 0.f};
  floats4 total = zero;
  for (int first = 0; first < segments; first += 2 * waves) {
    const int segment = first + 2 * wave + second, at = segment * kSegment + 4 * g;
    floats4 a[kSegmentBlocks], v[kSegmentBlocks];
    // (beyond k - a multiple of 4: a group of four is whole or absent - the last elements once more, which count as zeros)
#pragma unroll
    for (int b = 0; b < kSegmentBlocks; ++b) a[b] = *reinterpret_cast<const floats4*>(wp + min(at + 16 * b, k - 4));
#pragma unroll
    for (int b = 0; b < kSegmentBlocks; ++b) v[b] = *reinterpret_cast<const floats4*>(xp + min(at + 16 * b, k - 4));
    __builtin_amdgcn_sched_barrier(0);                     // (else the loads are moved down to where they are used)
    floats4 sums = zero;
    if ((first + 2 * wave + 2) * kSegment <= k) {          // (the same for the wave)
#pragma unroll
      for (int b = 0; b < kSegmentBlocks; ++b) sums = mfma4(a[b], v[b], sums);
    } else {
#pragma unroll
      for (int b = 0; b < kSegmentBlocks; ++b) {
        const bool inside = at + 16 * b < k;
        sums = mfma4(inside ? a[b] : zero, inside ? v[b] : zero, sums);
      }
    }
    // lane (column, g) holds the sums of instruction rows 4 g .. 4 g + 3: of outputs 4 (g & 1) .. + 3 and segment g / 2
    if (second == g >> 1) pieces[(2 * wave + second) * 16 + (g & 1) * 8 + r] = sums;
    __syncthreads();
    if (threadIdx.x < 16) {
      const int there = min(2 * waves, segments - first);
      for (int s = 0; s < there; ++s) total += pieces[s * 16 + threadIdx.x];
    }
    __syncthreads();
  }
  if constexpr (GATED) {
    if (wave > 0) return;
#pragma unroll
    for (int n = 0; n < 4; ++n) total[n] = silu(total[n]) * __shfl_xor(total[n], 8, 64);    // lane (row, second): the up's four
    if (lane < 8 && r < rows) store_f32(y, r, out0, outs, total, bias, wide_stores);
    return;
  }
  if (threadIdx.x < 16 && r < rows) store_f32(y, r, out0 + 4 * static_cast<int>(threadIdx.x >> 3), outs, total, bias, wide_stores && out0 + 8 <= outs);
}

// More rows: tiles of 32 TM outputs by 32 TN rows, four waves of TM x TN tiles of 16 each, operands through two LDS buffers
// of 32 k (row stride 36 floats: 16-byte reads of eight rows meet no bank twice), the next AHEAD steps of 32 k on their way in
// registers.  Bound by the matrix cores where tiles fill the chip (8 TM TN instructions of 32 cycles a step and wave for
// 2 (TM + TN) reads of 1 KB), so a step is written in the order in which they never wait: either half of a step's 32 k is
// read from LDS while the half before it is multiplied, the next step is filed between a half's instructions, and the one
// barrier of a step stands between its halves - the reads behind it have the second half's time, those before it are long
// there.  (Read where they are used and filed at the end, with the barrier after it, 999 rows of 2048 x 2048 / 6144 x 2048 /
// 2048 x 3072 took 85 / 237 / 125 us instead of 75 / 214 / 110 with tiles of 64 x 64, 333 rows of 2048 x 2048 / 6144 x 2048 38 /
// 101 instead of 33 / 95 with tiles of 32 x 32, 2048 rows of 6144 x 2048 462 instead of 419, 123 TFLOP/s; weights that no cache
// holds, as in the table at `launch_f32`.)  Where a unit holds one or two blocks a read from memory takes longer than a step:
// 2048 outputs, k 2048 with 333 rows (64 x 64) take 69 / 43 / 42 us with 1 / 2 / 4 steps on their way, with 999 rows 79 / 75 / 74.  Steps are a multiple of AHEAD, so that no register is copied
// at a loop's end: steps beyond k add zeros.  ZEROS: k is no multiple of AHEAD steps, so some of what is filed counts as zeros.
template <int TM, int TN, int AHEAD, bool ZEROS>
__global__ __launch_bounds__(256) void linear_f32_wide_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                              float* __restrict__ y, int rows, int outs, int k,
                                                              const float* __restrict__ bias, bool wide_stores) {
  constexpr int kStride = 36, kDeep = 32, kOuts = 32 * TM, kRows = 32 * TN;
  __shared__ float ws[2][kOuts * kStride];
  __shared__ float xs[2][kRows * kStride];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int out0 = blockIdx.x * kOuts, row0 = blockIdx.y * kRows;
  const int file_row = threadIdx.x >> 3, file_k = (threadIdx.x & 7) * 4;   // thread t fetches 16 bytes of rows t / 8 + 32 i
  const float* wp[TM];
  const float* xp[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) wp[i] = w + static_cast<long>(min(out0 + file_row + 32 * i, outs - 1)) * k;
#pragma unroll
  for (int i = 0; i < TN; ++i) xp[i] = x + static_cast<long>(min(row0 + file_row + 32 * i, rows - 1)) * k;
  const floats4 zero = {0.f, 0.f, 0.f, 0.f};
  floats4 sums[TM][TN], total[TM][TN], next_w[AHEAD][TM], next_x[AHEAD][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) sums[i][j] = total[i][j] = zero;
  auto fetch = [&](int slot, int k0) {
    const int at = min(k0 + file_k, k - 4);
#pragma unroll
    for (int i = 0; i < TM; ++i) next_w[slot][i] = *reinterpret_cast<const floats4*>(wp[i] + at);
#pragma unroll
    for (int i = 0; i < TN; ++i) next_x[slot][i] = *reinterpret_cast<const floats4*>(xp[i] + at);
  };
  auto file = [&](int slot, int buffer, int k0) {
    const bool inside = !ZEROS || k0 + file_k < k;
#pragma unroll
    for (int i = 0; i < TM; ++i)
      *reinterpret_cast<floats4*>(&ws[buffer][(file_row + 32 * i) * kStride + file_k]) = inside ? next_w[slot][i] : zero;
#pragma unroll
    for (int i = 0; i < TN; ++i)
      *reinterpret_cast<floats4*>(&xs[buffer][(file_row + 32 * i) * kStride + file_k]) = inside ? next_x[slot][i] : zero;
  };
  const int w_at = ((wave >> 1) * 16 * TM + r) * kStride + 4 * g, x_at = ((wave & 1) * 16 * TN + r) * kStride + 4 * g;
  floats4 a[2][TM], v[2][TN];                              // the operands of either half of a step
  auto read = [&](int half, int buffer) {
#pragma unroll
    for (int i = 0; i < TM; ++i) a[half][i] = *reinterpret_cast<const floats4*>(&ws[buffer][w_at + 16 * i * kStride + 16 * half]);
#pragma unroll
    for (int j = 0; j < TN; ++j) v[half][j] = *reinterpret_cast<const floats4*>(&xs[buffer][x_at + 16 * j * kStride + 16 * half]);
  };
  auto multiply = [&](int half, int first, int last) {
#pragma unroll
    for (int e = first; e < last; ++e)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          sums[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[half][i][e], v[half][j][e], sums[i][j], 0, 0, 0);
  };
  const int steps = (k + AHEAD * kDeep - 1) / (AHEAD * kDeep) * AHEAD;
  fetch(0, 0);
#pragma unroll
  for (int i = 1; i < AHEAD; ++i) fetch(i, i * kDeep);
  file(0, 0, 0);
  __syncthreads();
  read(0, 0);
  for (int first = 0; first < steps; first += AHEAD) {
#pragma unroll
    for (int turn = 0; turn < AHEAD; ++turn) {
      const int step = first + turn;
      const int buffer = step & 1;
      fetch(turn, (step + AHEAD) * kDeep);                 // (beyond k the last elements once more; they are filed as zeros or not multiplied)
      __builtin_amdgcn_sched_barrier(0);                   // (left alone the compiler moves all of these to where they are used)
      read(1, buffer);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, 0, 2);
      __builtin_amdgcn_sched_barrier(0);
      file((turn + 1) % AHEAD, buffer ^ 1, (step + 1) * kDeep);   // (read last before the barrier of the step before)
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, 2, 4);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
      read(0, buffer ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      multiply(1, 0, 4);
      __builtin_amdgcn_sched_barrier(0);
      if ((step & 3) == 3 || step + 1 == steps) {          // the end of a segment of 128
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            total[i][j] += sums[i][j];
            sums[i][j] = zero;
          }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int row = row0 + (wave & 1) * 16 * TN + 16 * j + r;
    if (row >= rows) continue;
#pragma unroll
    for (int i = 0; i < TM; ++i)
      store_f32(y, row, out0 + (wave >> 1) * 16 * TM + 16 * i + 4 * g, outs, total[i][j], bias, wide_stores);
  }
}

template <int NT, bool GATED = false>
int launch_f32_few(const float* x, const float* w, float* y, int rows, int outs, int k, const float* bias, bool wide_stores,
                   hipStream_t stream) {
  constexpr int kOuts = GATED ? 8 : 16;
  const int segments = (k + kSegment - 1) / kSegment, rounds = (segments + 15) / 16;
  const int waves = max((segments + rounds - 1) / rounds, NT);
  const size_t lds = static_cast<size_t>(waves) * NT * 64 * sizeof(floats4);     // 32 KB at most
  linear_f32_few_kernel<NT, GATED><<<(outs + kOuts - 1) / kOuts, waves * 64, lds, stream>>>(x, w, y, rows, outs, k, segments, bias, wide_stores);
  return AKV_LAUNCH_STATUS();
}

template <bool GATED>
int launch_f32_pairs(const float* x, const float* w, float* y, int rows, int outs, int k, const float* bias, bool wide_stores,
                     hipStream_t stream) {
  constexpr int kOuts = GATED ? 4 : 8;
  const int segments = (k + kSegment - 1) / kSegment, pairs = (segments + 1) / 2, rounds = (pairs + 15) / 16;
  const int waves = (pairs + rounds - 1) / rounds;
  linear_f32_pairs_kernel<GATED><<<(outs + kOuts - 1) / kOuts, waves * 64, 2 * waves * 16 * sizeof(floats4), stream>>>(
      x, w, y, rows, outs, k, segments, bias, wide_stores);
  return AKV_LAUNCH_STATUS();
}

template <int TM, int TN>
int launch_f32_wide(const float* x, const float* w, float* y, int rows, int outs, int k, const float* bias, bool wide_stores,
                    hipStream_t stream) {
  dim3 grid((outs + 32 * TM - 1) / (32 * TM), (rows + 32 * TN - 1) / (32 * TN));
  constexpr int kAhead = TM * TN == 4 ? 2 : 4;
  if (k <= 32)       // (one step: those that are asked for ahead would add zeros)
    linear_f32_wide_kernel<TM, TN, 1, true><<<grid, 256, 0, stream>>>(x, w, y, rows, outs, k, bias, wide_stores);
  else if (k % (32 * kAhead) != 0)
    linear_f32_wide_kernel<TM, TN, kAhead, true><<<grid, 256, 0, stream>>>(x, w, y, rows, outs, k, bias, wide_stores);
  else
    linear_f32_wide_kernel<TM, TN, kAhead, false><<<grid, 256, 0, stream>>>(x, w, y, rows, outs, k, bias, wide_stores);
  return AKV_LAUNCH_STATUS();
}

// Up to 16 rows (see `launch_f32`); gated: `outs` of the result, half of what is read.
template <bool GATED>
int launch_f32_few_rows(const float* x, const float* w, float* y, int rows, int outs, int k, const float* bias, hipStream_t stream) {
  const bool wide_stores = outs % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
  const long units = device_facts().compute_units, read = GATED ? 2l * outs : outs, tiles = (read + 15) / 16;
  if (k > kSegment && (rows <= 4 || (rows <= 8 && ((read + 7) / 8 <= units || (tiles > units && tiles <= 4 * units)))))
    return launch_f32_pairs<GATED>(x, w, y, rows, outs, k, bias, wide_stores, stream);
  return launch_f32_few<1, GATED>(x, w, y, rows, outs, k, bias, wide_stores, stream);
}

// float32 operands whose rows are 16-byte aligned.  Which kernel takes a product is a matter of time alone (the bits are the
// same).  Measured, us, on weights that no cache holds (outs x k = 2048 x 2048 / 6144 x 2048 / 4096 x 12288 / 32768 x 2048;
// tiles of outputs x rows):
//     16 rows: few 9.8 / 20 / 59 / 74     32 x 32 as with 17 rows
//     17 rows: few 13.3 / 26 / 74 / 86    32 x 32 16 / 18 / 87 / 58       32 x 64 23 / 25 / 125 / 90     64 x 64 41 / 42 / 233 / 84
//     64 rows: few 22 / 45 / 129 / -      32 x 32 17 / 25 / 92 / 106      32 x 64 24 / 25 / 134 / 90     64 x 64 42 / 43 / 238 / 85
//    300 rows:                            32 x 32 33 / 86 / 336 / 483     32 x 64 40 / 79 / 350 / 414    64 x 64 42 / 75 / 427 / 367
//    700 rows:                            32 x 32 62 / 184 / 718 / 1036   32 x 64 58 / 173 / 669 / 899   64 x 64 74 / 177 / 618 / 801
//    999 rows:                            32 x 32 82 / 265 / 1026 / 1477  32 x 64 77 / 233 / 894 / 1288  64 x 64 75 / 214 / 834 / 1160
// (123 TFLOP/s at best; the vector kernel above: 511 us on average over 999 rows of 2048 x 2048 and 2048 x 3072).  So: few
// rows stay with the kernels that read the matrix once, from 17 on only where blocks of 16 outputs are one a unit; tiles
// are the kind whose busiest unit has the least to do - the blocks it gets times their area, a block of 32 x 64 taking 5 % and
// one of 32 x 32 15 % longer for its area than one of 64 x 64.  (Tiles of 128 are slower everywhere: the matrix cores wait for
// nothing that larger tiles would spare.)
// Up to 8 rows, blocks of 8 outputs (pairs) against blocks of 16 (few), outs x k = 2048 x 2048 / 2048 x 6144 / 3072 x 2048 /
// 4096 x 2048 / 6144 x 2048 / 12288 x 2048 / 32768 x 2048:
//      1 row:  pairs 5.5 / 12.7 / 7.7 / 7.9 / 11.7 / 20.1 / 48     few 7.5 / 20.3 / 8.0 / 9.2 / 15.5 / 23.7 / 55
//      8 rows: pairs 6.5 / 16.0 / 9.9 / 10.1 / 14.6 / 26.0 / 64    few 8.6 / 22.6 / 8.9 / 9.8 / 16.9 / 26.2 / 62
// So: pairs up to 4 rows (also with 3: 2048 x 6144 13.4 against 20.6); from 5 on where they are one block a unit, or where
// blocks of 16 are several a unit, but not many (100,000 x 1024 with 8 rows: 96 against 87).
// Never where k is one segment: an instruction's second would be empty (32768 x 16 with 1 row 6.7 against 4.0, 32768 x 128 8.2
// against 5.6).
int launch_f32(const float* x, const float* w, float* y, int rows, int outs, int k, const float* bias, hipStream_t stream) {
  const bool wide_stores = outs % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
  const long units = device_facts().compute_units;
  const auto rounds = [&](int out_tile, int row_tile) {
    const long blocks = static_cast<long>((outs + out_tile - 1) / out_tile) * ((rows + row_tile - 1) / row_tile);
    return (blocks + units - 1) / units;
  };
  if (rows <= 16) return launch_f32_few_rows<false>(x, w, y, rows, outs, k, bias, stream);
  if (rows <= 32 && (outs + 15) / 16 <= units) return launch_f32_few<2>(x, w, y, rows, outs, k, bias, wide_stores, stream);
  // (The caller counts the grid's limit in tiles of 64 rows.  Where tiles of 32 would pass it they are not taken: by then tiles of 64
  // are more than a hundred rounds, and from eleven on twice the tiles at 115 cost more than 210.)
  const long large = 400 * rounds(64, 64), middle = 210 * rounds(32, 64), small = 115 * rounds(32, 32);
  if (large <= middle && large <= small) return launch_f32_wide<2, 2>(x, w, y, rows, outs, k, bias, wide_stores, stream);
  if (middle <= small) return launch_f32_wide<1, 2>(x, w, y, rows, outs, k, bias, wide_stores, stream);
  return launch_f32_wide<1, 1>(x, w, y, rows, outs, k, bias, wide_stores, stream);
}

}  // namespace

// `bias` [outs] float32 or null: added to a sum after its last product, before it is rounded to y's type.
extern "C" int akv_linear_tiled(const void* x, int x_dtype, const void* w, int w_dtype, void* y, int y_dtype, int rows,
                                int outs, int k, const float* bias, hipStream_t stream) {
  if (rows <= 0 || outs <= 0) return 0;
  if (((rows + kTile - 1) / kTile) > 65535) return -2;
  const int code = x_dtype * 4 + w_dtype * 2 + y_dtype;
  switch (code) {
    case 0:
      if (k > 0 && k % 4 == 0 && (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0)
        return launch_f32(static_cast<const float*>(x), static_cast<const float*>(w), static_cast<float*>(y), rows, outs, k,
                          bias, stream);
      return launch_tiled<float, float, float>(x, w, y, rows, outs, k, bias, stream);
    case 2: return launch_tiled<float, bf16_t, float>(x, w, y, rows, outs, k, bias, stream);
    case 4: return launch_tiled<bf16_t, float, float>(x, w, y, rows, outs, k, bias, stream);
    case 5: return launch_tiled<bf16_t, float, bf16_t>(x, w, y, rows, outs, k, bias, stream);
    case 6: return launch_tiled<bf16_t, bf16_t, float>(x, w, y, rows, outs, k, bias, stream);
    case 7: return launch_tiled<bf16_t, bf16_t, bf16_t>(x, w, y, rows, outs, k, bias, stream);
    default: return -1;
  }
}

// y [rows, inter] = silu(x W[:inter]^T) * (x W[inter:]^T), w [2 inter, k]: float32 throughout, up to 16 rows, k a multiple of 4, x and w
// on 16-byte boundaries (else -2).
extern "C" int akv_linear_f32_gated(const float* x, const float* w, float* y, int rows, int inter, int k, hipStream_t stream) {
  if (rows <= 0 || inter <= 0) return 0;
  if (rows > 16 || k <= 0 || k % 4 != 0 || inter >= (1 << 30) ||
      (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 != 0)
    return -2;
  return launch_f32_few_rows<true>(x, w, y, rows, inter, k, nullptr, stream);
}
