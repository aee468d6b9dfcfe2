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
// v_mfma_f32_16x16x4_f32 multiplies float32 operands at a sixteenth of the rate of v_mfma_f32_16x16x32_bf16, whose products of
// bfloat16 numbers are exact and whose sums are float32.  So an operand becomes three bfloat16 numbers, each what the ones before
// it leave, rounded: 24 bits of mantissa in all, its value exactly.  (The instruction takes numbers below 2^-126 as zeros: operands
// are multiplied by 2^24 before they are split, which keeps the last bit of every float32 number above that, and sums by 2^-48.)
// Of the nine products of two such operands six are formed, from the smallest to the largest - the three left out are at most
// 2^-23 of the product, 2^-26 of it on average and of either sign.  Against 64 bits the sums are closer than the float32
// instruction's, which rounds after every four products where this one rounds after 32: normal operands, k 2,048, relative error
// 1.6e-7 / 2.2e-7; positive ones, whose sums grow, k 12,288, 5.7e-8 / 1.5e-7, largest error in units of 2^-24 sum |x w| 3.9 / 12.3;
// the logits of a model of 8 layers 1.1e-6 / 1.35e-6.
// A result that is no finite number is formed anew from the operands as they are, by the float32 instruction (`redo_f32`): an
// infinite operand, or one that bfloat16 rounds to infinity, has no parts, and sums beyond 2^80 have left float32's range.
// A lane's operand of an instruction is 32 bytes of a matrix row: lane (r, g) holds elements 4 g .. + 3 and 16 + 4 g .. + 3 of 32
// of row r.  All kernels sum every output the same way, so that a row's result depends neither on how many rows a call carries nor
// on which kernel takes it: k is cut into segments of 128, a segment is one chain of instructions (32 elements after 32, the six
// products of each in their order), every fourth segment's sums are added in their order, from the first, second, third and fourth
// on, and then those four, the even ones and the odd ones first.  The instruction cuts a sum's low bits off towards minus infinity:
// every result would be 0.02 x 2^-24 sum |x w| too low, which a model's residual sum collects layer by layer; so the rows' elements
// of odd segments are negated, and what their sums make is subtracted.  (Rows and outputs beyond the matrices repeat the last one
// and are not stored; elements beyond k are zeros and change no sum.)
typedef float floats4 __attribute__((ext_vector_type(4)));
typedef uint32_t uints4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
constexpr int kSegment = 128;        // k of one chain
constexpr int kSegmentBlocks = kSegment / 16;

struct Parts4 { uint2 p[3]; };       // four values as three bfloat16 numbers each
struct Parts8 { uints4 p[3]; };      // eight: operands of an instruction

constexpr float kRaised = 16777216.f, kLowered = 1.f / (kRaised * kRaised);
// What the rows' elements of a segment are multiplied by.
__device__ __forceinline__ float raised_in(int segment) { return segment & 1 ? -kRaised : kRaised; }

__device__ __forceinline__ Parts4 split4(floats4 v, float raised) {
  Parts4 s;
  v *= raised;
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    s.p[p] = uint2{bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3])};
    if (p == 2) break;
    v[0] -= __uint_as_float(s.p[p].x << 16);
    v[1] -= __uint_as_float(s.p[p].x & 0xffff0000u);
    v[2] -= __uint_as_float(s.p[p].y << 16);
    v[3] -= __uint_as_float(s.p[p].y & 0xffff0000u);
  }
  return s;
}

__device__ __forceinline__ Parts8 split8(const floats4 low, const floats4 high, float raised = kRaised) {
  const Parts4 a = split4(low, raised), b = split4(high, raised);
  Parts8 s;
#pragma unroll
  for (int p = 0; p < 3; ++p) s.p[p] = uints4{a.p[p].x, a.p[p].y, b.p[p].x, b.p[p].y};
  return s;
}

__device__ __forceinline__ floats4 mfma32(const uints4 a, const uints4 b, const floats4 sums) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), sums, 0, 0, 0);
}

// The parts of the six products, the smallest products first.
constexpr int kProducts = 6, kPartOfW[kProducts] = {2, 0, 1, 1, 0, 0}, kPartOfX[kProducts] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ floats4 products(const Parts8& w, const Parts8& x, floats4 sums) {
#pragma unroll
  for (int n = 0; n < kProducts; ++n) sums = mfma32(w.p[kPartOfW[n]], x.p[kPartOfX[n]], sums);
  return sums;
}

// The sums of 16 outputs (4 g .. 4 g + 3 of them in this lane) by 16 rows, `w` and `x` the lane's row of either: float32
// operands as they are, 128 of k in one chain.
__device__ __forceinline__ floats4 redo_f32(const float* __restrict__ w, const float* __restrict__ x, int k, int g) {
  const floats4 zero = {0.f, 0.f, 0.f, 0.f};
  floats4 total = zero;
#pragma unroll 1
  for (int k0 = 0; k0 < k; k0 += kSegment) {
    floats4 sums = zero;
#pragma unroll 1
    for (int at = k0; at < min(k0 + kSegment, k); at += 16) {
      const bool inside = at + 4 * g < k;                  // (k is a multiple of 4: a group of four is whole or absent)
      const floats4 a = inside ? *reinterpret_cast<const floats4*>(w + at + 4 * g) : zero;
      const floats4 v = inside ? *reinterpret_cast<const floats4*>(x + at + 4 * g) : zero;
#pragma unroll
      for (int j = 0; j < 4; ++j) sums = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], v[j], sums, 0, 0, 0);
    }
    total += sums;
  }
  return total;
}

// The sums of segments 0, 4, 8 ..., of 1, 5, 9 ... and so on, four side by side in LDS (`stride` apart), take `count` more (a multiple
// of four) in their order; in LDS because a kernel's waves need their registers for loads.
__device__ __forceinline__ void add_fourths(floats4* total, const floats4* pieces, int count, int stride, bool begins) {
  floats4 of[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) of[n] = begins ? floats4{0.f, 0.f, 0.f, 0.f} : total[n * stride];
  for (int s = 0; s < count; s += 4) {
#pragma unroll
    for (int n = 0; n < 4; ++n) of[n] += pieces[(s + n) * stride];
  }
#pragma unroll
  for (int n = 0; n < 4; ++n) total[n * stride] = of[n];
}
__device__ __forceinline__ floats4 all_fourths(const floats4* total, int stride) {
  return (total[0] + total[2 * stride]) - (total[stride] + total[3 * stride]);
}

__device__ __forceinline__ bool finite(float v) { return fabsf(v) < INFINITY; }
__device__ __forceinline__ bool finite(const floats4 v) { return finite(v[0]) && finite(v[1]) && finite(v[2]) && finite(v[3]); }

// The sums of a wave's tile of 16 x 16 as results, those that are no finite numbers formed anew.  All lanes of the wave call it.
__device__ __forceinline__ floats4 settled(floats4 sums, const float* __restrict__ w, const float* __restrict__ x, int k, int g) {
  sums *= kLowered;
  if (!__any(!finite(sums))) return sums;
  const floats4 again = redo_f32(w, x, k, g);
#pragma unroll
  for (int j = 0; j < 4; ++j) sums[j] = finite(sums[j]) ? sums[j] : again[j];
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

__device__ __forceinline__ floats4 load_at(const char* from, uint32_t offset) {
  asm("" : "+v"(offset));            // (known to have 32 bits where it is used: a scalar address and an offset, no pair of registers)
  return *reinterpret_cast<const floats4*>(from + offset);
}

// GATED: y = silu(x Wgate^T) * (x Wup^T) of a matrix whose first half is the gate's, in steps of up to 16 rows, where a launch costs as
// much as it does: a block owns as many outputs of either half and forms what the activation's kernel forms from the stored
// product, the same bits (3 rows, us: 6144 x 2048 and the activation's kernel 12.3 + 4.6, gated 13.2).
__device__ __forceinline__ float silu(float v) { return v / (1.f + expf(-v)); }

// Up to 32 rows: the matrix is read once and its reads are what the product waits for.  A block owns 16 outputs and all of
// k; its waves take a segment each (a second round where k has more than 16), with the whole segment's loads in flight - 8 KB
// a wave, 128 KB a block -, and leave their sums in LDS, where the first waves add them in order.  Rows lie in cache and
// are read by every wave in operand order, without LDS, NT tiles of 16 rows - a single one before the weights (loads return in
// order), so that it is split while those are on their way (1 row of 6144 x 2048: 13.8 -> 11.8 us).
template <int NT, bool GATED>
__global__ __launch_bounds__(1024) void linear_f32_few_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             float* __restrict__ y, int rows, int outs, int k, int segments,
                                                             const float* __restrict__ bias, bool wide_stores) {
  static_assert(NT == 1 || !GATED, "");
  extern __shared__ floats4 pieces[];                      // [waves][NT][64], then the sums of every fourth
  floats4* total = pieces + (blockDim.x >> 6) * NT * 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  constexpr int kOuts = GATED ? 8 : 16;                    // (of the result; with the gate's half of the matrix eight and eight)
  const int out0 = blockIdx.x * kOuts;
  const float* wp = w + static_cast<long>(GATED && r >= 8 ? outs + min(out0 + r - 8, outs - 1) : min(out0 + (GATED ? r & 7 : r), outs - 1)) * k;
  const float* xp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) xp[t] = x + static_cast<long>(min(16 * t + r, rows - 1)) * k;
  const floats4 zero = {0.f, 0.f, 0.f, 0.f};
  for (int first = 0; first < segments; first += waves) {
    const int segment = first + wave;
    if (segment >= segments) {
#pragma unroll
      for (int t = 0; t < NT; ++t) pieces[(wave * NT + t) * 64 + lane] = zero;
    } else {
      const int at = segment * kSegment + 4 * g;
      floats4 a[kSegmentBlocks], v[NT][kSegmentBlocks];
      auto fetch = [&](const float* from, floats4 (&to)[kSegmentBlocks]) {
        // (beyond k - a multiple of 4: a group of four is whole or absent - the last elements once more, which count as zeros)
#pragma unroll
        for (int b = 0; b < kSegmentBlocks; ++b) to[b] = *reinterpret_cast<const floats4*>(from + min(at + 16 * b, k - 4));
      };
      if (NT == 1) fetch(xp[0], v[0]);
      fetch(wp, a);
      if (NT > 1) {
#pragma unroll
        for (int t = 0; t < NT; ++t) fetch(xp[t], v[t]);
      }
      __builtin_amdgcn_sched_barrier(0);                   // (else the loads are moved down to where they are used)
      floats4 sums[NT];
      auto of_x = [&](int t, int b) {
        return split8(at + 32 * b < k ? v[t][2 * b] : zero, at + 32 * b + 16 < k ? v[t][2 * b + 1] : zero, raised_in(segment));
      };
      if constexpr (NT == 1) {
        Parts8 held[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) held[b] = of_x(0, b);
        sums[0] = zero;
#pragma unroll
        for (int b = 0; b < 4; ++b) sums[0] = products(split8(a[2 * b], a[2 * b + 1]), held[b], sums[0]);
      } else {
#pragma unroll
        for (int t = 0; t < NT; ++t) sums[t] = zero;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const Parts8 of_w = split8(a[2 * b], a[2 * b + 1]);
#pragma unroll
          for (int t = 0; t < NT; ++t) sums[t] = products(of_w, of_x(t, b), sums[t]);
        }
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) pieces[(wave * NT + t) * 64 + lane] = sums[t];
    }
    __syncthreads();
    if (wave < NT) add_fourths(total + wave * 64 + lane, pieces + wave * 64 + lane, waves, NT * 64, first == 0);
    __syncthreads();
  }
  // (a block has a multiple of four waves: the launch sees to it)
  if (wave >= NT) return;
  floats4 sums = settled(all_fourths(total + wave * 64 + lane, NT * 64), wp, x + static_cast<long>(min(16 * wave + r, rows - 1)) * k, k, g);
  if constexpr (GATED) {
    floats4 up;
#pragma unroll
    for (int n = 0; n < 4; ++n) up[n] = __shfl_xor(sums[n], 32, 64);       // lane (row, g + 2)
#pragma unroll
    for (int n = 0; n < 4; ++n) sums[n] = silu(sums[n]) * up[n];
    if (g >= 2) return;
  }
  if (16 * wave + r < rows) store_f32(y, 16 * wave + r, out0 + 4 * g, outs, sums, bias, wide_stores);
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
  extern __shared__ floats4 pieces[];                      // [2 waves][16], then the sums of every fourth
  floats4* total = pieces + (blockDim.x >> 6) * 32;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int r = lane & 7, second = lane >> 3 & 1, g = lane >> 4;
  constexpr int kOuts = GATED ? 4 : 8;                     // (of the result; with the gate's half of the matrix four and four)
  const int out0 = blockIdx.x * kOuts;
  const float* wp = w + static_cast<long>(GATED && r >= 4 ? outs + min(out0 + r - 4, outs - 1) : min(out0 + (GATED ? r & 3 : r), outs - 1)) * k;
  const float* xp = x + static_cast<long>(min(r, rows - 1)) * k;
  const floats4 zero = {0.f, 0.f, 0.f, 0.f};
  for (int first = 0; first < segments; first += 2 * waves) {
    const int segment = first + 2 * wave + second, at = segment * kSegment + 4 * g;
    floats4 a[kSegmentBlocks], v[kSegmentBlocks];
    // (the rows first: they lie in cache and are split while the weights are on their way; loads return in order.  Beyond k - a
    // multiple of 4: a group of four is whole or absent - the last elements once more, which count as zeros)
#pragma unroll
    for (int b = 0; b < kSegmentBlocks; ++b) v[b] = *reinterpret_cast<const floats4*>(xp + min(at + 16 * b, k - 4));
#pragma unroll
    for (int b = 0; b < kSegmentBlocks; ++b) a[b] = *reinterpret_cast<const floats4*>(wp + min(at + 16 * b, k - 4));
    __builtin_amdgcn_sched_barrier(0);                     // (else the loads are moved down to where they are used)
    Parts8 of_x[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
      of_x[b] = split8(at + 32 * b < k ? v[2 * b] : zero, at + 32 * b + 16 < k ? v[2 * b + 1] : zero, raised_in(segment));
    __builtin_amdgcn_sched_barrier(0);
    floats4 sums = zero;
#pragma unroll
    for (int b = 0; b < 4; ++b) sums = products(split8(a[2 * b], a[2 * b + 1]), of_x[b], sums);
    // lane (column, g) holds the sums of instruction rows 4 g .. 4 g + 3: of outputs 4 (g & 1) .. + 3 and segment g / 2
    if (second == g >> 1) pieces[(2 * wave + second) * 16 + (g & 1) * 8 + r] = sums;
    __syncthreads();
    // (a segment beyond the last: zeros; a block has an even number of waves)
    if (threadIdx.x < 16) add_fourths(total + threadIdx.x, pieces + threadIdx.x, 2 * waves, 16, first == 0);
    __syncthreads();
  }
  if (wave > 0) return;
  floats4 sums = zero;                                     // (lanes 16 and more: zeros)
  if (lane < 16) sums = all_fourths(total + lane, 16) * kLowered;
  if (__any(!finite(sums))) {
    const floats4 again = redo_f32(wp, xp, k, g);          // lane (row, g): outputs 4 g .. 4 g + 3
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float other = __shfl(again[j], second * 16 + r, 64);
      sums[j] = finite(sums[j]) ? sums[j] : other;
    }
  }
  if constexpr (GATED) {
#pragma unroll
    for (int n = 0; n < 4; ++n) sums[n] = silu(sums[n]) * __shfl_xor(sums[n], 8, 64);      // lane (row, second): the up's four
    if (lane < 8 && r < rows) store_f32(y, r, out0, outs, sums, bias, wide_stores);
    return;
  }
  if (lane < 16 && r < rows) store_f32(y, r, out0 + 4 * second, outs, sums, bias, wide_stores && out0 + 8 <= outs);
}

// More rows: a block has G groups of OW waves.  A wave owns 16 TM outputs by the block's 16 TN rows; a group takes every G-th
// segment of k, and the groups' sums are added through LDS at the end, so that a vector unit has two waves and more where tiles
// are one a unit, and few rows' products have short chains.  A step is 32 of k: eight lanes read a row's 128 bytes, kAhead steps
// ahead into registers.  A wave's weights turn into operand order through LDS of its own, pieces of 16 bytes exchanged by the row's
// number against bank conflicts, and are split when they come back; the rows are split as they come, each by one wave of its group,
// and lie in LDS as parts in operand order.
// What bounds it: of a step's 1.35 us where a unit has one block of 128 x 64, 0.7 are its matrix instructions, and the splitting,
// the trips through LDS and the reads of parts add up to the rest (two waves a vector unit that wait for one barrier overlap
// little; written orders of the instructions, groups half a step apart and waves of three tiles gave the same 50 to 55 us, weights
// read in operand order, whose loads name sixteen lines for sixteen lanes, 52 to 57).
template <int TM, int TN, int OW, int G>
__global__ __launch_bounds__(64 * G * OW, TM * TN * OW > 16 ? 2 : 4) void linear_f32_wide_kernel(
    const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ y, int rows, int outs, int k,
    const float* __restrict__ bias, bool wide_stores) {
  constexpr int kAhead = OW == 2 ? 4 : 2;                  // steps on their way (few blocks: nothing else covers a read)
  constexpr int kRuns = 2 * TN / OW;                       // runs of 8 rows that a wave splits a step
  constexpr int kTotals = 4 / G;
  static_assert(2 * TN % OW == 0 && 4 % kAhead == 0 && (G == 2 || G == 4), "");
  __shared__ __align__(16) uints4 x_parts[2][G][TN][3][64];            // [buffer][group][tile of rows][part][lane]
  __shared__ __align__(16) floats4 w_rows[G * OW][16 * TM * 8];        // a wave's rows of 32 elements
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int of_run = lane >> 3, piece = lane & 7;          // what the lane fetches: 16 bytes of a row of eight
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), column = wave % OW, group = wave / OW;
  const int out0 = (blockIdx.x * OW + column) * 16 * TM, row0 = blockIdx.y * 16 * TN;
  const int first_out = min(out0, outs - 1);
  const char* w_bytes = reinterpret_cast<const char*>(w + static_cast<long>(first_out) * k);
  const char* x_bytes = reinterpret_cast<const char*>(x + static_cast<long>(row0) * k);
  uint32_t w_from[2 * TM], x_from[kRuns];                  // (k is less than 2^24)
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i) w_from[i] = static_cast<uint32_t>(min(out0 + 8 * i + of_run, outs - 1) - first_out) * k * 4u;
#pragma unroll
  for (int i = 0; i < kRuns; ++i) x_from[i] = static_cast<uint32_t>(min(row0 + 8 * (column * kRuns + i) + of_run, rows - 1) - row0) * k * 4u;
  const floats4 zero = {0.f, 0.f, 0.f, 0.f};
  floats4 sums[TM][TN], total[kTotals][TM][TN], next_w[kAhead][2 * TM], next_x[kAhead][kRuns];
  Parts8 a[2][TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      sums[i][j] = zero;
#pragma unroll
      for (int n = 0; n < kTotals; ++n) total[n][i][j] = zero;
    }
  auto k_of = [&](int step) { return ((step >> 2) * G + group) * kSegment + (step & 3) * 32 + 4 * piece; };
  auto fetch = [&](int slot, int step) {                   // (beyond k the last elements once more; the rows' count as zeros)
    const uint32_t at = static_cast<uint32_t>(min(k_of(step), k - 4)) * 4u;
#pragma unroll
    for (int i = 0; i < kRuns; ++i) next_x[slot][i] = load_at(x_bytes, x_from[i] + at);
#pragma unroll
    for (int i = 0; i < 2 * TM; ++i) next_w[slot][i] = load_at(w_bytes, w_from[i] + at);
  };
  auto file_x = [&](int slot, int buffer, int step) {      // four elements: half of the operand of lane (row, piece % 4)
    const bool inside = k_of(step) < k;
#pragma unroll
    for (int i = 0; i < kRuns; ++i) {
      const Parts4 s = split4(inside ? next_x[slot][i] : zero, raised_in(group));     // (segments that differ by G, an even number)
      const int run = column * kRuns + i, row = (run & 1) * 8 + of_run, h = piece & 3;
      const int place = (h * 16 + (row ^ 2 * h)) * 2 + (piece >> 2);
#pragma unroll
      for (int p = 0; p < 3; ++p) reinterpret_cast<uint2*>(x_parts[buffer][group][run >> 1][p])[place] = s.p[p];
    }
  };
  auto turn_w = [&](int slot, int which) {
#pragma unroll
    for (int i = 0; i < 2 * TM; ++i) w_rows[wave][(8 * i + of_run) * 8 + (piece ^ of_run)] = next_w[slot][i];
#pragma unroll
    for (int i = 0; i < TM; ++i)
      a[which][i] = split8(w_rows[wave][(16 * i + r) * 8 + (g ^ (r & 7))], w_rows[wave][(16 * i + r) * 8 + ((g + 4) ^ (r & 7))]);
  };
  const int segments = (k + kSegment - 1) / kSegment, steps = (segments + G - 1) / G * 4;
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(i, i);
  file_x(0, 0, 0);
  turn_w(0, 0);
  __syncthreads();
  for (int first = 0; first < steps;) {
#pragma unroll
    for (int n = 0; n < kTotals; ++n) {                    // a segment
      if (n > 0 && first >= steps) break;
#pragma unroll
      for (int turn = 0; turn < 4; ++turn) {
        const int buffer = turn & 1;
        fetch(turn % kAhead, first + turn + kAhead);
        __builtin_amdgcn_sched_barrier(0);                 // (else the loads are moved down to where they are used)
        turn_w((turn + 1) % kAhead, buffer ^ 1);
        file_x((turn + 1) % kAhead, buffer ^ 1, first + turn + 1);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          uints4 v[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) v[p] = x_parts[buffer][group][j][p][g * 16 + (r ^ 2 * g)];
#pragma unroll
          for (int m = 0; m < kProducts; ++m)
#pragma unroll
            for (int i = 0; i < TM; ++i) sums[i][j] = mfma32(a[buffer][i].p[kPartOfW[m]], v[kPartOfX[m]], sums[i][j]);
        }
        if (turn == 3) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              total[n][i][j] += sums[i][j];
              sums[i][j] = zero;
            }
        }
        __syncthreads();
      }
      first += 4;
    }
  }
  // the groups' sums to the first one
  constexpr int kTile = TM * TN * 64;
  floats4* pass = reinterpret_cast<floats4*>(&x_parts[0][0][0][0][0]) + column * kTile;
  static_assert((G - 1) * OW * kTile <= 2 * G * TN * 3 * 64, "the sums fit where the rows lay");
  if (group > 0) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        pass[(group - 1) * OW * kTile + (i * TN + j) * 64 + lane] = G == 2 ? total[0][i][j] + total[kTotals - 1][i][j] : total[0][i][j];
  }
  __syncthreads();
  if (group > 0) return;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int row = row0 + 16 * j + r;
    const float* x_row = x + static_cast<long>(min(row, rows - 1)) * k;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const float* w_row = w + static_cast<long>(min(out0 + 16 * i + r, outs - 1)) * k;
      auto other = [&](int n) { return pass[(n - 1) * OW * kTile + (i * TN + j) * 64 + lane]; };
      const floats4 all = G == 2 ? (total[0][i][j] + total[kTotals - 1][i][j]) - other(1) : (total[0][i][j] + other(2)) - (other(1) + other(3));
      const floats4 result = settled(all, w_row, x_row, k, g);
      if (row < rows) store_f32(y, row, out0 + 16 * i + 4 * g, outs, result, bias, wide_stores);
    }
  }
}

template <int NT, bool GATED = false>
int launch_f32_few(const float* x, const float* w, float* y, int rows, int outs, int k, const float* bias, bool wide_stores,
                   hipStream_t stream) {
  constexpr int kOuts = GATED ? 8 : 16;
  const int segments = (k + kSegment - 1) / kSegment, rounds = (segments + 15) / 16;
  const int waves = ((segments + rounds - 1) / rounds + 3) / 4 * 4;
  const size_t lds = static_cast<size_t>(waves + 4) * NT * 64 * sizeof(floats4);     // 40 KB at most
  linear_f32_few_kernel<NT, GATED><<<(outs + kOuts - 1) / kOuts, waves * 64, lds, stream>>>(x, w, y, rows, outs, k, segments, bias, wide_stores);
  return AKV_LAUNCH_STATUS();
}

template <bool GATED>
int launch_f32_pairs(const float* x, const float* w, float* y, int rows, int outs, int k, const float* bias, bool wide_stores,
                     hipStream_t stream) {
  constexpr int kOuts = GATED ? 4 : 8;
  const int segments = (k + kSegment - 1) / kSegment, pairs = (segments + 1) / 2, rounds = (pairs + 15) / 16;
  const int waves = ((pairs + rounds - 1) / rounds + 1) / 2 * 2;
  linear_f32_pairs_kernel<GATED><<<(outs + kOuts - 1) / kOuts, waves * 64, (2 * waves + 4) * 16 * sizeof(floats4), stream>>>(
      x, w, y, rows, outs, k, segments, bias, wide_stores);
  return AKV_LAUNCH_STATUS();
}

template <int TM, int TN, int OW, int G>
int launch_f32_wide(const float* x, const float* w, float* y, int rows, int outs, int k, const float* bias, bool wide_stores,
                    hipStream_t stream) {
  dim3 grid((outs + 16 * TM * OW - 1) / (16 * TM * OW), (rows + 16 * TN - 1) / (16 * TN));
  linear_f32_wide_kernel<TM, TN, OW, G><<<grid, 64 * G * OW, 0, stream>>>(x, w, y, rows, outs, k, bias, wide_stores);
  return AKV_LAUNCH_STATUS();
}

// Whether up to 16 rows go to blocks of 8 outputs (pairs) rather than 16 (few): see `launch_f32`.
bool takes_pairs(int rows, long outs, int k) {
  const long units = device_facts().compute_units, tiles = (outs + 15) / 16;
  return k > kSegment && (rows <= 4 || (rows <= 8 && ((outs + 7) / 8 <= units || tiles > units)));
}

// Up to 16 rows by blocks of few outputs; gated: `outs` of the result.
template <bool GATED>
int launch_f32_few_rows(const float* x, const float* w, float* y, int rows, int outs, int k, const float* bias, hipStream_t stream) {
  const bool wide_stores = outs % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
  if (takes_pairs(rows, GATED ? 2l * outs : outs, k)) return launch_f32_pairs<GATED>(x, w, y, rows, outs, k, bias, wide_stores, stream);
  return launch_f32_few<1, GATED>(x, w, y, rows, outs, k, bias, wide_stores, stream);
}

// float32 operands whose rows are 16-byte aligned, k less than 2^24.  Which kernel takes a product is a matter of time alone (the bits
// are the same).  Measured, us, on weights that no cache holds (outs x k = 2048 x 2048 / 3072 x 2048 / 6144 x 2048 / 2048 x 3072 /
// 32768 x 2048), before (the float32 instruction, its best kernel) and as chosen here:
//      1 row:  8.6 / 8.8 / 11.9 / 8.3 / 48  ->  8.4 / 8.6 / 11.9 / 8.4 / 47     (pairs)
//     16 rows: 10.0 / 11.2 / 20.4 / 15.8 / 74  ->  10.1 / 11.0 / 20.5 / 15.2 / 56   (few; 32768: 64 x 32)
//     32 rows: 13.5 / 15.2 / 20.0 / 21.4 / 64  ->  15.2 / 16.5 / 19.9 / 23.5 / 57   (few; 6144: 32 x 32; 32768: 64 x 32)
//     64 rows: 19.1 / 19.6 / 30.0 / 28.0 / 89  ->  17.1 / 18.5 / 23.0 / 24.6 / 76   (32 x 32, 64 x 32)
//    200 rows: 29.5 / 38.3 / 65.3 / 43.2 / 314  ->  20.9 / 30.7 / 52.7 / 30.0 / 255
//    333 rows: 37.3 / 56.1 / 98.2 / 54.3 / 467  ->  29.8 / 52.3 / 87.3 / 44.3 / 370
//    999 rows: 82.8 / 121 / 236 / 122 / 1218  ->  55.1 / 91.9 / 161 / 81.7 / 965   (128 x 64: 152 to 156 TFLOP/s; the float32 one 101)
// Tiles of outputs x rows, us by rounds of blocks on the units, k 2,048: 128 x 64 51 / 102 / 161, 64 x 64 in four groups 29 / 58 / 92,
// 64 x 32 in four groups 21, in two 23 / 38 / 56 / 74, 32 x 32 in four 17 / 26 / 37 / 47: the tile whose rounds cost least.  Few rows
// stay with the kernels that read the matrix once, from 17 on only where blocks of 16 outputs are one a unit, and from 5 on not
// where they are more than four (32768 x 2048, 8 rows: pairs 63, few 63, 64 x 32 56).
// Up to 8 rows, blocks of 8 outputs (pairs) against blocks of 16 (few): 1 to 4 rows pairs (3 rows of 2048 x 3072: 8.3 / 12.2); from 5
// on where they are one block a unit, or where blocks of 16 are several a unit (8 rows of 4096 x 12288 56 / 50, 3072 x 2048 10.4 /
// 9.8).  Never where k is one segment: an instruction's second would be empty.
int launch_f32(const float* x, const float* w, float* y, int rows, int outs, int k, const float* bias, hipStream_t stream) {
  const bool wide_stores = outs % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
  const long units = device_facts().compute_units;
  const auto rounds = [&](int out_tile, int row_tile) {
    const long blocks = static_cast<long>((outs + out_tile - 1) / out_tile) * ((rows + row_tile - 1) / row_tile);
    return (blocks + units - 1) / units;
  };
  const long tiles = (outs + 15) / 16;
  if (rows <= 4 || tiles <= 4 * units) {
    if (rows <= 16) return launch_f32_few_rows<false>(x, w, y, rows, outs, k, bias, stream);
    if (rows <= 32 && tiles <= units) return launch_f32_few<2>(x, w, y, rows, outs, k, bias, wide_stores, stream);
  }
  // (The caller counts the grid's limit in tiles of 64 rows: where tiles of 32 would pass it they are not taken.)
  const bool many = (rows + 31) / 32 > 65535;
  const long a = rounds(128, 64), b = rounds(64, 64), c = rounds(64, 32), d = rounds(32, 32);
  const long cost_a = 530 * a, cost_b = 295 * b, cost_c = c == 1 ? 210 : 182 * c + 10, cost_d = d == 1 ? 175 : 112 * d + 30;
  if (cost_a <= cost_b && (many || (cost_a <= cost_c && cost_a <= cost_d))) return launch_f32_wide<2, 4, 4, 2>(x, w, y, rows, outs, k, bias, wide_stores, stream);
  if (many || (cost_b <= cost_c && cost_b <= cost_d)) return launch_f32_wide<1, 4, 4, 4>(x, w, y, rows, outs, k, bias, wide_stores, stream);
  if (cost_c <= cost_d) {
    if (c == 1) return launch_f32_wide<1, 2, 4, 4>(x, w, y, rows, outs, k, bias, wide_stores, stream);
    return launch_f32_wide<1, 2, 4, 2>(x, w, y, rows, outs, k, bias, wide_stores, stream);
  }
  return launch_f32_wide<1, 2, 2, 4>(x, w, y, rows, outs, k, bias, wide_stores, stream);
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
      if (k > 0 && k % 4 == 0 && k < (1 << 24) && (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0)
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

// y [rows, inter] = silu(x W[:inter]^T) * (x W[inter:]^T), w [2 inter, k]: float32 throughout, up to 16 rows, k a multiple of 4 below
// 2^24, x and w on 16-byte boundaries (else -2).
extern "C" int akv_linear_f32_gated(const float* x, const float* w, float* y, int rows, int inter, int k, hipStream_t stream) {
  if (rows <= 0 || inter <= 0) return 0;
  if (rows > 16 || k <= 0 || k % 4 != 0 || k >= (1 << 24) || inter >= (1 << 30) ||
      (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 != 0)
    return -2;
  return launch_f32_few_rows<true>(x, w, y, rows, inter, k, nullptr, stream);
}
