// Grouped-query attention for designs whose scores and weights are float32 and whose keys and values may differ in
// width: unit norm of queries and keys with the cache write, and the attention itself with an optional softcap on the
// scores, a bias that grows with the distance, chunks of positions, a window, a sink in the softmax's denominator and a gate
// per head.
//
// Keys lie [pages, kv_heads, page, dim], values [pages, kv_heads, vdim, page].  `gated_attention_rows` is the plain path:
// one wave per (token, query head); keys are visited in tiles of 64 aligned to absolute key positions, so the order of
// every sum depends on the token's own position only - not on how the request was cut into steps or on what else is in
// the batch.  Scores, the softmax and the weighted sum are float32.

#include "common.h"
#include "api_parts.h"

using namespace akv;

namespace {

__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One wave per (token, item): the token's query heads (normed into q_out), its key heads (normed into the token's slot
// of the key pages) and its value heads (copied into the value pages).  projected rows: [q | k | v | ...].
// With `maps` > 1 a head's queries and keys are `maps` vectors of `dim` side by side: the token has q_heads * maps query
// vectors and kv_heads * maps key vectors, each normed and rotated for itself, and a key head's record in the pages is
// its `maps` vectors one after the other.  With `table` [positions, rot_dims / 2, 2] (cos, sin) a vector's first rot_dims
// dimensions are rotated by the token's position, dimension i with i + rot_dims / 2 - or, with `interleaved`, dimension 2 i
// with 2 i + 1.  With `whole` the root mean square is taken over all of the token's query vectors at once (and over all of
// its key vectors): every wave sums its side's whole projection for itself.  `q_weight` [q vectors x dim] and `k_weight`
// [k vectors x dim] (float32, either may be null) multiply the normed values, before the rotation.  With `temp_every` > 0 a
// query is multiplied by 1 + temp_coef ln(floor((p + 1) / temp_every) + 1) at its position p; with `value_eps` >= 0 a value
// head is divided by its root mean square (value_eps inside the root) before it is written.  The value heads lie from column
// `values_at` of a row on: behind the keys, or - values that are the keys as they were projected - where the keys lie.
// One (token, item): `which` < q_vectors is a query vector, then the key vectors, then the value heads.  `given` > 0: the
// factor 1 / rms of the item's side, formed by the caller over the whole projection; else the vector norms itself.
template <typename T>
__device__ __forceinline__ void unit_norm_item(const T* __restrict__ row, long n, int which, int lane, int q_heads, int kv_heads,
                                               int dim, int vdim, float eps, int normed, float given,
                                               const int* __restrict__ slot_map, T* __restrict__ k_pages, T* __restrict__ v_pages,
                                               int page_size, long num_pages, T* __restrict__ q_out, int maps,
                                               const float* __restrict__ table, int table_positions, int rot_dims,
                                               const int* __restrict__ positions, const float* __restrict__ q_weight,
                                               const float* __restrict__ k_weight, int interleaved, float value_eps,
                                               float temp_coef, int temp_every, int values_at) {
  const int q_vectors = q_heads * maps, k_vectors = kv_heads * maps;
  if (which < q_vectors + k_vectors) {
    const bool is_q = which < q_vectors;
    const T* x = row + static_cast<long>(which) * dim;       // (key vectors follow the query vectors at the same width)
    T* y;
    if (is_q) {
      y = q_out + (n * q_vectors + which) * dim;
    } else {
      if (slot_map == nullptr) return;
      const long slot = slot_map[n];
      const long page = slot / page_size;
      if (slot < 0 || page >= num_pages) return;
      const int vector = which - q_vectors;
      y = k_pages + (((page * kv_heads + vector / maps) * page_size + slot % page_size) * maps + vector % maps) * dim;
    }
    float scale = 1.f;
    if (normed && given > 0.f) {
      scale = given;
    } else if (normed) {
      float squares = 0.f;
      for (int i = lane; i < dim; i += kWave) {
        const float v = to_float(x[i]);
        squares += v * v;
      }
      scale = rsqrtf(wave_sum(squares) / static_cast<float>(dim) + eps);
    }
    // a temperature on queries that grows with their position
    if (is_q && temp_every > 0) scale *= 1.f + temp_coef * logf(static_cast<float>((positions[n] + 1) / temp_every + 1));
    const float* gain = is_q ? q_weight : k_weight;
    if (gain != nullptr) gain += static_cast<long>(is_q ? which : which - q_vectors) * dim;
    if (table == nullptr || rot_dims <= 0) {
      for (int i = lane; i < dim; i += kWave) y[i] = from_float<T>(to_float(x[i]) * scale * (gain != nullptr ? gain[i] : 1.f));
    } else {
      const int half = rot_dims / 2;
      const int pos = positions[n];
      const bool known = pos >= 0 && pos < table_positions;      // (a position beyond the table poisons the vector)
      const float* angles = table + static_cast<long>(known ? pos : 0) * half * 2;
      for (int i = lane; i < dim; i += kWave) {
        float v = to_float(x[i]) * scale * (gain != nullptr ? gain[i] : 1.f);
        if (i < rot_dims) {
          const bool low = interleaved ? (i & 1) == 0 : i < half;
          const int pair = interleaved ? i >> 1 : (low ? i : i - half);
          const int mate = interleaved ? i ^ 1 : (low ? i + half : i - half);
          const float c = angles[2 * pair], s = angles[2 * pair + 1];
          const float other = to_float(x[mate]) * scale * (gain != nullptr ? gain[mate] : 1.f);
          v = low ? v * c - other * s : v * c + other * s;
          if (!known) v = __uint_as_float(0x7fc00000u);
        }
        y[i] = from_float<T>(v);
      }
    }
  } else {
    if (slot_map == nullptr) return;
    const int h = which - q_vectors - k_vectors;
    const long slot = slot_map[n];
    const long page = slot / page_size;
    if (slot < 0 || page >= num_pages) return;
    const T* x = row + values_at + static_cast<long>(h) * vdim;
    T* y = v_pages + (page * kv_heads + h) * vdim * page_size + slot % page_size;
    if (value_eps >= 0.f) {      // values divided by their root mean square per head
      float squares = 0.f;
      for (int i = lane; i < vdim; i += kWave) {
        const float v = to_float(x[i]);
        squares += v * v;
      }
      const float scale = rsqrtf(wave_sum(squares) / static_cast<float>(vdim) + value_eps);
      for (int i = lane; i < vdim; i += kWave) y[static_cast<long>(i) * page_size] = from_float<T>(to_float(x[i]) * scale);
      return;
    }
    for (int i = lane; i < vdim; i += kWave) y[static_cast<long>(i) * page_size] = x[i];
  }
}

template <typename T>
__global__ __launch_bounds__(256) void unit_norm_write_kernel(const T* __restrict__ projected, long stride, long tokens,
                                                              int q_heads, int kv_heads, int dim, int vdim, float eps,
                                                              int normed, const int* __restrict__ slot_map,
                                                              T* __restrict__ k_pages, T* __restrict__ v_pages, int page_size,
                                                              long num_pages, T* __restrict__ q_out, int maps,
                                                              const float* __restrict__ table, int table_positions,
                                                              int rot_dims, const int* __restrict__ positions,
                                                              const float* __restrict__ q_weight,
                                                              const float* __restrict__ k_weight, int interleaved,
                                                              float value_eps, float temp_coef, int temp_every, int values_at) {
  const int waves = blockDim.x / kWave, wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  const int items = (q_heads + kv_heads) * maps + kv_heads;
  const long item = static_cast<long>(blockIdx.x) * waves + wave;
  if (item >= tokens * items) return;
  const long n = item / items;
  unit_norm_item<T>(projected + n * stride, n, static_cast<int>(item % items), lane, q_heads, kv_heads, dim, vdim, eps, normed,
                    0.f, slot_map, k_pages, v_pages, page_size, num_pages, q_out, maps, table, table_positions, rot_dims,
                    positions, q_weight, k_weight, interleaved, value_eps, temp_coef, temp_every, values_at);
}

// Eight bfloat16 (or float32) values from 16-byte aligned memory, widened.
__device__ __forceinline__ void load8(const bf16_t* p, float (&v)[8]) {
  const uint4 raw = *reinterpret_cast<const uint4*>(p);
  const uint32_t words[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[2 * k] = __uint_as_float(words[k] << 16);
    v[2 * k + 1] = __uint_as_float(words[k] & 0xffff0000u);
  }
}
__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

// bfloat16 vectors whose widths come in eights, unscaled but for the norm: a thread takes eight neighbouring elements of a
// vector with 16-byte reads and writes (a norm's sum meets over the dim / 8 lanes of its vector, a power of two), and a wave
// takes 64 dimensions of a value head for eight tokens, which it turns through LDS: where the eight slots are a run of one
// page from a multiple of eight on - a prompt's are -, every lane writes its dimension's eight tokens as 16 bytes.  Bound by
// memory; what is not is the reads of single elements and the writes of two bytes each that the kernel above makes (a wave a
// vector).  2,000 tokens of 16 query, 4 key and 4 value heads of 128 (25 MB): 18.9 us there, of 32 query and 8 key vectors of 64
// and 4 values of 128 27.8; here 10.1 both (2.5 TB/s: a thread has one 16-byte group or two on their way).  8 tokens 4 us both.
template <bool NORMED>
__global__ __launch_bounds__(256) void unit_norm_write_eights_kernel(const bf16_t* __restrict__ projected, long stride, int tokens,
                                                                     int q_vectors, int kv_heads, int dim, int vdim, float eps,
                                                                     const int* __restrict__ slot_map,
                                                                     bf16_t* __restrict__ k_pages, bf16_t* __restrict__ v_pages,
                                                                     int page_size, long num_pages, bf16_t* __restrict__ q_out,
                                                                     int maps, const float* __restrict__ table,
                                                                     int table_positions, int rot_dims,
                                                                     const int* __restrict__ positions, int values_at,
                                                                     unsigned vector_blocks) {
  __shared__ __align__(16) bf16_t turned[4][8][72];        // (a row of 144 bytes: 16-byte writes, reads along a column)
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  if (blockIdx.x < vector_blocks) {
    const unsigned eights = dim / 8, per_token = (q_vectors + (slot_map != nullptr ? kv_heads * maps : 0)) * eights;
    const unsigned index = blockIdx.x * 256 + threadIdx.x, token = index / per_token, at = index % per_token;
    if (token >= static_cast<unsigned>(tokens)) return;    // (whole vectors: a vector's lanes leave together)
    const int which = at / eights, i = (at % eights) * 8;
    const bf16_t* x = projected + token * stride + static_cast<long>(which) * dim;
    float v[8];
    load8(x + i, v);
    float scale = 1.f;
    if constexpr (NORMED) {
      float squares = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) squares += v[j] * v[j];
      for (unsigned reach = 1; reach < eights; reach *= 2) squares += __shfl_xor(squares, reach);
      scale = rsqrtf(squares / static_cast<float>(dim) + eps);
    }
    bf16_t* y = q_out + (static_cast<long>(token) * q_vectors + which) * dim;
    if (which >= q_vectors) {
      const int slot = slot_map[token], page = slot / page_size, vector = which - q_vectors;
      if (slot < 0 || page >= num_pages) return;
      y = k_pages + (((static_cast<long>(page) * kv_heads + vector / maps) * page_size + slot % page_size) * maps + vector % maps) * dim;
    }
    if (NORMED) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] *= scale;
    }
    if (i < rot_dims) {
      const int half = rot_dims / 2;
      const bool low = i < half;
      const int pos = positions[token];
      const bool known = pos >= 0 && pos < table_positions;      // (a position beyond the table poisons the vector)
      const float* angles = table + (static_cast<long>(known ? pos : 0) * half + (low ? i : i - half)) * 2;
      float other[8];
      load8(x + (low ? i + half : i - half), other);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float c = angles[2 * j], s = angles[2 * j + 1], o = other[j] * scale;
        v[j] = low ? v[j] * c - o * s : v[j] * c + o * s;
        if (!known) v[j] = __uint_as_float(0x7fc00000u);
      }
    }
    alignas(16) bf16_t packed[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) packed[j] = from_float<bf16_t>(v[j]);
    *reinterpret_cast<uint4*>(y + i) = *reinterpret_cast<const uint4*>(packed);
    return;
  }
  // values: a wave's item is eight tokens, a head and 64 of its dimensions
  const int pieces = (vdim + 63) / 64, per_group = kv_heads * pieces;
  const unsigned item = (blockIdx.x - vector_blocks) * 4 + wave;
  const int first = item / per_group * 8, h = item % per_group / pieces, d0 = item % pieces * 64;
  const int token = first + lane / 8, d = d0 + lane % 8 * 8;
  const bool there = token < tokens && d < vdim;
  const int slot = token < tokens ? slot_map[token] : -1;
  uint4 raw = make_uint4(0, 0, 0, 0);
  if (there) raw = *reinterpret_cast<const uint4*>(projected + token * stride + values_at + static_cast<long>(h) * vdim + d);
  const int start = __shfl(slot, 0);
  const bool run = first + 8 <= tokens && start >= 0 && start % 8 == 0;
  // (page_size is a multiple of eight: a run from a multiple of eight on stays in its page)
  if (__all(run && slot == start + lane / 8)) {
    *reinterpret_cast<uint4*>(&turned[wave][lane / 8][lane % 8 * 8]) = raw;
    wave_sync_lds();
    alignas(16) bf16_t packed[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) packed[t] = turned[wave][t][lane];
    const long page = start / page_size;
    if (page < num_pages && d0 + lane < vdim)
      *reinterpret_cast<uint4*>(v_pages + ((page * kv_heads + h) * vdim + d0 + lane) * page_size + start % page_size) =
          *reinterpret_cast<const uint4*>(packed);
    return;
  }
  if (!there || slot < 0 || slot / page_size >= num_pages) return;
  alignas(16) bf16_t own[8];
  *reinterpret_cast<uint4*>(own) = raw;
  bf16_t* y = v_pages + ((static_cast<long>(slot / page_size) * kv_heads + h) * vdim + d) * page_size + slot % page_size;
#pragma unroll
  for (int j = 0; j < 8; ++j) y[static_cast<long>(j) * page_size] = own[j];
}

// The same with the root mean square taken over all of a token's query vectors at once, and over all its key vectors: a
// block is a token, sums both sides' squares once, and its waves then take the token's items in turn.
template <typename T>
__global__ __launch_bounds__(1024) void unit_norm_write_whole_kernel(const T* __restrict__ projected, long stride, int q_heads,
                                                                    int kv_heads, int dim, int vdim, float eps,
                                                                    const int* __restrict__ slot_map, T* __restrict__ k_pages,
                                                                    T* __restrict__ v_pages, int page_size, long num_pages,
                                                                    T* __restrict__ q_out, int maps,
                                                                    const float* __restrict__ table, int table_positions,
                                                                    int rot_dims, const int* __restrict__ positions,
                                                                    const float* __restrict__ q_weight,
                                                                    const float* __restrict__ k_weight, int interleaved,
                                                                    float value_eps, float temp_coef, int temp_every, int values_at) {
  __shared__ float scratch[16];
  const int waves = blockDim.x / kWave, wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  const long n = blockIdx.x;
  const T* row = projected + n * stride;
  const int q_count = q_heads * maps * dim, k_count = kv_heads * maps * dim;
  float q_squares = 0.f, k_squares = 0.f;
  for (int i = threadIdx.x; i < q_count + k_count; i += blockDim.x) {
    const float v = to_float(row[i]);
    if (i < q_count) q_squares += v * v;
    else k_squares += v * v;
  }
  const float q_scale = rsqrtf(block_sum(q_squares, scratch) / static_cast<float>(q_count) + eps);
  const float k_scale = rsqrtf(block_sum(k_squares, scratch) / static_cast<float>(k_count) + eps);
  const int q_vectors = q_heads * maps, items = (q_heads + kv_heads) * maps + kv_heads;
  for (int which = wave; which < items; which += waves)
    unit_norm_item<T>(row, n, which, lane, q_heads, kv_heads, dim, vdim, eps, 1, which < q_vectors ? q_scale : k_scale, slot_map,
                      k_pages, v_pages, page_size, num_pages, q_out, maps, table, table_positions, rot_dims, positions, q_weight,
                      k_weight, interleaved, value_eps, temp_coef, temp_every, values_at);
}

constexpr int kMaxValueRegs = 4;  // value widths up to 256: each lane owns dims lane, lane + 64, ...
constexpr int kMaxRowWaves = 16;  // the most waves that share a (token, head): wave w of W takes the key tiles w, w + W, ...

// A block is a token and G query heads that read the same key head (G = 1: a single head); its waves (1 to 16, the
// caller's choice) take the row's tiles of 64 keys in turn and their shares - maximum, sum of weights, weighted values,
// per head - meet in LDS in the order of the waves.  Inside a tile a lane scores one key for all G heads from one read of
// it (VEC: its dimensions eight at a time) and then owns value dimensions, for which it reads eight neighbouring keys'
// values at a time (the value pages lie [vdim, page]) - once for the G heads.  VEC needs key rows and groups of eight
// values that are 16-byte aligned.
template <typename T, bool VEC, int G>
__global__ __launch_bounds__(kMaxRowWaves * kWave) void gated_attention_rows_kernel(
    const T* __restrict__ q, const T* __restrict__ k_pages, const T* __restrict__ v_pages, const T* __restrict__ gates,
    long gate_stride, int gate_at, const int* __restrict__ seq_of_token, const int* __restrict__ positions,
    const int* __restrict__ block_table, const int* __restrict__ table_rows, int table_width, T* __restrict__ out,
    long tokens, int q_heads, int kv_heads, int dim, int vdim, int page_size, long num_pages, float scale, float softcap,
    int chunk, int window, int sink, long out_stride, float out_scale, const float* __restrict__ sink_logits, int maps,
    int keep_first, const float* __restrict__ distance_bias) {
  // (`q_heads` counts query vectors: with `maps` > 1 a head has `maps` of them, which read the `maps` vectors of their key
  // head's record in turn and the same values; vector v's key head is still v / (q_heads / kv_heads))
  extern __shared__ unsigned char lds_raw[];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1), kRowWaves = blockDim.x / kWave;
  // blocks go to the XCDs in turn: neighbouring rows - which read the same or neighbouring keys and values - are given to
  // blocks of one XCD
  const long row = static_cast<long>(blockIdx.x % kXcds) * (gridDim.x / kXcds) + blockIdx.x / kXcds;
  const int bundles = q_heads / G;           // rows of a token
  if (row >= tokens * bundles) return;
  // the block: G x dim floats of q; per wave G x 64 weights and 64 value-row offsets; then the waves' shares
  float* qs = reinterpret_cast<float*>(lds_raw);
  const size_t q_bytes = (static_cast<size_t>(G) * dim * 4 + 7) / 8 * 8;
  float* ps = reinterpret_cast<float*>(lds_raw + q_bytes) + wave * G * kWave;
  long* offs = reinterpret_cast<long*>(lds_raw + q_bytes + static_cast<size_t>(kRowWaves) * G * kWave * 4) + wave * kWave;
  float* shares = reinterpret_cast<float*>(lds_raw + q_bytes + static_cast<size_t>(kRowWaves) * kWave * (G * 4 + 8));

  const long n = row / bundles;
  const int h0 = static_cast<int>(row % bundles) * G;
  const int kvh = h0 / (q_heads / kv_heads);
  const int r = table_rows != nullptr ? table_rows[seq_of_token[n]] : seq_of_token[n];
  const int pos = positions[n];
  int lowest = window > 0 ? max(0, pos - window + 1) : 0;
  if (chunk > 0) lowest = max(lowest, pos / chunk * chunk);
  for (int i = threadIdx.x; i < G * dim; i += blockDim.x) qs[i] = to_float(q[(n * q_heads + h0) * dim + i]);
  __syncthreads();

  // with a sink the sums start as if a key of score 0 and no value had been seen (in the first wave's share)
  // (a learned sink: the term is exp(sink_logits[head]) instead of exp(0))
  float m[G], l[G], acc[G][kMaxValueRegs];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = sink && wave == 0 ? (sink_logits != nullptr ? sink_logits[h0 + g] : 0.f) : -INFINITY;
    l[g] = sink && wave == 0 ? 1.f : 0.f;
#pragma unroll
    for (int c = 0; c < kMaxValueRegs; ++c) acc[g][c] = 0.f;
  }
  // the request's first `keep_first` keys stay visible behind the window: their tiles come first, then the window's
  const int first_tile = lowest / kWave, kept_tiles = min((keep_first + kWave - 1) / kWave, first_tile);
  const int all_tiles = kept_tiles + pos / kWave - first_tile + 1;
  for (int turn = wave; turn < all_tiles; turn += kRowWaves) {
    const int tile = turn < kept_tiles ? turn : first_tile + turn - kept_tiles;
    const int j = tile * kWave + lane;
    const bool valid = (j >= lowest || j < keep_first) && j <= pos;
    float s[G];
#pragma unroll
    for (int g = 0; g < G; ++g) s[g] = -INFINITY;
    long value_at = -1;
    if (valid) {
      const long page = block_table[static_cast<long>(r) * table_width + j / page_size];
      if (page < 0 || page >= num_pages) {
#pragma unroll
        for (int g = 0; g < G; ++g) s[g] = __uint_as_float(0x7fc00000u);  // a page that is not the request's: poison
      } else {
        const T* kp = k_pages + (((page * kv_heads + kvh) * page_size + j % page_size) * maps + h0 % maps) * dim;
        float dot[G];
#pragma unroll
        for (int g = 0; g < G; ++g) dot[g] = 0.f;
        int i = 0;
        if (VEC) {
          for (; i + 16 <= dim; i += 16) {       // two loads are asked for before the first is used
            float kv[2][8];
#pragma unroll
            for (int u = 0; u < 2; ++u) load8(kp + i + 8 * u, kv[u]);
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
              for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int g = 0; g < G; ++g) dot[g] = fmaf(qs[g * dim + i + 8 * u + e], kv[u][e], dot[g]);
          }
          for (; i + 8 <= dim; i += 8) {
            float kv[8];
            load8(kp + i, kv);
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
              for (int g = 0; g < G; ++g) dot[g] = fmaf(qs[g * dim + i + e], kv[e], dot[g]);
          }
        }
        for (; i < dim; ++i) {
          const float kv = to_float(kp[i]);
#pragma unroll
          for (int g = 0; g < G; ++g) dot[g] = fmaf(qs[g * dim + i], kv, dot[g]);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          s[g] = dot[g] * scale;
          if (softcap > 0.f) s[g] = softcap * tanhf(s[g] / softcap);
          if (distance_bias != nullptr)
            s[g] -= distance_bias[h0 + g] * log1pf(distance_bias[q_heads + h0 + g] * static_cast<float>(pos - j));
        }
        value_at = (page * kv_heads + kvh) * vdim * page_size + j % page_size;  // values are [vdim, page_size]
      }
    }
    float correction[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float m_new = fmaxf(m[g], wave_max(s[g]));
      const float p = valid ? expf(s[g] - m_new) : 0.f;
      correction[g] = m_new == m[g] ? 1.f : expf(m[g] - m_new);
      l[g] = l[g] * correction[g] + wave_sum(p);
      m[g] = m_new;
      ps[g * kWave + lane] = value_at >= 0 || !VEC ? p : 0.f;
    }
    offs[lane] = value_at;
    wave_sync_lds();
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int c = 0; c < kMaxValueRegs; ++c) acc[g][c] *= correction[g];
    if (VEC) {
      // a group of eight keys shares a page: its first key that counts tells where the group's values lie
#pragma unroll 2
      for (int k = 0; k < 8; ++k) {
        long at = -1;
#pragma unroll
        for (int e = 7; e >= 0; --e)
          if (offs[8 * k + e] >= 0) at = offs[8 * k + e] - e;
        if (at < 0) continue;  // uniform over the wave
        float weights[G][8];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int e = 0; e < 8; ++e) weights[g][e] = ps[g * kWave + 8 * k + e];
#pragma unroll
        for (int c = 0; c < kMaxValueRegs; ++c) {
          const int i = lane + c * kWave;
          if (i < vdim) {
            float values[8];
            load8(v_pages + at + static_cast<long>(i) * page_size, values);
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
              for (int g = 0; g < G; ++g) acc[g][c] += weights[g][e] != 0.f ? weights[g][e] * values[e] : 0.f;
          }
        }
      }
    } else {
      for (int jj = 0; jj < kWave; ++jj) {
        const long at = offs[jj];
        if (at < 0) continue;  // uniform over the wave
#pragma unroll
        for (int c = 0; c < kMaxValueRegs; ++c) {
          const int i = lane + c * kWave;
          if (i < vdim) {
            const float value = to_float(v_pages[at + static_cast<long>(i) * page_size]);
#pragma unroll
            for (int g = 0; g < G; ++g) acc[g][c] = fmaf(ps[g * kWave + jj], value, acc[g][c]);
          }
        }
      }
    }
    wave_sync_lds();
  }
  const int share = 2 + vdim;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float* mine = shares + static_cast<size_t>(wave * G + g) * share;
    if (lane == 0) mine[0] = m[g], mine[1] = l[g];
#pragma unroll
    for (int c = 0; c < kMaxValueRegs; ++c) {
      const int i = lane + c * kWave;
      if (i < vdim) mine[2 + i] = acc[g][c];
    }
  }
  __syncthreads();
  for (int g = 0; g < G; ++g) {
    float highest = -INFINITY;
    for (int w = 0; w < kRowWaves; ++w) highest = fmaxf(highest, shares[static_cast<size_t>(w * G + g) * share]);
    float total = 0.f, factors[kMaxRowWaves];
#pragma unroll
    for (int w = 0; w < kMaxRowWaves; ++w) {
      const float m_w = w < kRowWaves ? shares[static_cast<size_t>(w * G + g) * share] : -INFINITY;
      factors[w] = m_w == -INFINITY ? 0.f : expf(m_w - highest);
      total += w < kRowWaves ? shares[static_cast<size_t>(w * G + g) * share + 1] * factors[w] : 0.f;
    }
    const int h = h0 + g;
    float gate = out_scale;
    if (gates != nullptr) gate = out_scale / (1.f + expf(-to_float(gates[n * gate_stride + gate_at + h])));
    for (int i = threadIdx.x; i < vdim; i += blockDim.x) {
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < kMaxRowWaves; ++w)
        if (w < kRowWaves) sum += shares[static_cast<size_t>(w * G + g) * share + 2 + i] * factors[w];
      out[n * out_stride + static_cast<long>(h) * vdim + i] = from_float<T>(sum / total * gate);
    }
  }
}

}  // namespace

namespace {

// ---- prompt portions on the matrix cores ----------------------------------------------------------------------------
// bfloat16, keys 16 DT and values 16 VT wide, pages of a multiple of 16 tokens.  A wave is 16 neighbouring rows of the
// step and one query head.  S^T = K Q^T (16 keys x 16 queries a step, the keys as A operand straight from the page) leaves
// lane (c = l % 16, g = l / 16) with the scores of keys 4 g .. 4 g + 3 for query c - which is where the B operand of
// O^T = V^T P^T wants the weights, so they never leave the registers; the values, [vdim, page] in the page, are its A
// operand as they lie.  Scores, softcap, maxima, weights and sums are float32; a weight enters the second product as
// two bfloat16 (its rounding and what the rounding left).  Rows of one tile may belong to several requests (the end of
// one portion and the start of the next): the wave then takes the requests one after the other, each over its own keys,
// with the other requests' columns switched off.  Key tiles lie at absolute positions.
typedef __attribute__((ext_vector_type(4))) short short4_t;
typedef __attribute__((ext_vector_type(4))) float float4_t;

__device__ __forceinline__ short4_t load_bf16x4(const bf16_t* p) {
  return __builtin_bit_cast(short4_t, *reinterpret_cast<const uint2*>(p));
}

// What the matrix-core kernels read 16 bytes and write 8 bytes at a time.
inline bool aligned_for_tiles(const void* q, const void* k_pages, const void* v_pages, const void* out, long out_stride) {
  return ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_pages) | reinterpret_cast<uintptr_t>(v_pages)) % 16 == 0) &&
         reinterpret_cast<uintptr_t>(out) % 8 == 0 && out_stride % 4 == 0;
}

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;

__device__ __forceinline__ uint4 load_bf16x8(const bf16_t* p) { return *reinterpret_cast<const uint4*>(p); }

// DT: key width / 32 (the first product runs in steps of 32 dimensions), VT: value width / 16.
template <int DT, int VT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu((DT + VT <= 12 ? 3 : 2), 4))) void gated_attention_tiles_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_pages, const bf16_t* __restrict__ v_pages,
    const bf16_t* __restrict__ gates, long gate_stride, int gate_at, const int* __restrict__ seq_of_token,
    const int* __restrict__ q_start, const int* __restrict__ positions, const int* __restrict__ block_table,
    const int* __restrict__ table_rows, int table_width, bf16_t* __restrict__ out, int first_row, int tokens, int q_heads,
    int kv_heads, int page_size, long num_pages, float scale, float softcap, int chunk, int window, int sink,
    long out_stride, float out_scale, const float* __restrict__ sink_logits, int maps, int keep_first,
    const float* __restrict__ distance_bias) {
  constexpr int DIM = 32 * DT, VDIM = 16 * VT;
  extern __shared__ float tile_shares[];      // [waves][2 + 4 VT][64]: what the block's waves found over their keys
  // a block is 16 rows and a head; its waves take the steps of 16 keys in turn
  const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1), waves = blockDim.x / kWave;
  // blocks go to the XCDs in turn: the heads of a tile, which share keys and values, are given to blocks of one XCD, the
  // tiles to the XCDs in turn, and the tiles with the most keys before them - the last of a portion - start first
  const int tiles = (tokens - first_row + 15) / 16;
  const int slot = blockIdx.x / kXcds;
  const int head = slot % q_heads, turned = slot / q_heads * kXcds + blockIdx.x % kXcds;
  if (turned >= tiles) return;
  const int tile = tiles - 1 - turned;
  const int kvh = head / (q_heads / kv_heads);
  const int col = lane & 15, grp = lane >> 4;
  const int row0 = first_row + tile * 16, row_end = min(row0 + 16, tokens);
  const int my_row = row0 + col;
  const bool have = my_row < row_end;
  int my_pos = -1, my_lowest = 0;
  uint4 qb[DT];
  if (have) {
    my_pos = positions[my_row];
    my_lowest = window > 0 ? max(0, my_pos - window + 1) : 0;
    if (chunk > 0) my_lowest = max(my_lowest, my_pos / chunk * chunk);
    const bf16_t* qp = q + (static_cast<long>(my_row) * q_heads + head) * DIM + grp * 8;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) qb[dt] = load_bf16x8(qp + dt * 32);
  } else {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) qb[dt] = make_uint4(0u, 0u, 0u, 0u);
  }
  float m = sink && wave == 0 ? (sink_logits != nullptr ? sink_logits[head] : 0.f) : -INFINITY, l = sink && wave == 0 ? 1.f : 0.f;
  const float inverse_cap = softcap > 0.f ? 1.f / softcap : 0.f;
  // (the logarithm in the hardware's base)
  const float bias_size = distance_bias != nullptr ? distance_bias[head] * 0.6931471805599453f : 0.f;
  const float bias_rate = distance_bias != nullptr ? distance_bias[q_heads + head] : 0.f;
  float4_t o[VT];
#pragma unroll
  for (int vt = 0; vt < VT; ++vt) o[vt] = float4_t{0.f, 0.f, 0.f, 0.f};

  int row = row0;
  while (row < row_end) {
    const int r = seq_of_token[row];
    const int run_end = min(row_end, q_start[r + 1]);
    const int p_first = positions[row], p_last = p_first + (run_end - row - 1);
    int lo_run = window > 0 ? max(0, p_first - window + 1) : 0;
    if (chunk > 0) lo_run = max(lo_run, p_first / chunk * chunk);
    const long table_at = static_cast<long>(table_rows != nullptr ? table_rows[r] : r) * table_width;
    const bool in_run = have && my_row >= row && my_row < run_end;
    // a step's keys and values are asked for while the step before is worked on
    uint4 keys[DT], keys_next[DT];
    short4_t values[VT], values_next[VT];
    bool there = false, there_next = false;
    auto fetch = [&](int j0, uint4 (&ks)[DT], short4_t (&vs)[VT]) -> bool {
      const long page = block_table[table_at + j0 / page_size];
      if (page < 0 || page >= num_pages) return false;      // (uniform; a page that is not the request's is never read)
      const int o0 = j0 % page_size;
      const bf16_t* kp = k_pages + (((page * kv_heads + kvh) * page_size + o0 + col) * maps + head % maps) * DIM + grp * 8;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) ks[dt] = load_bf16x8(kp + dt * 32);
      const bf16_t* vp = v_pages + ((page * kv_heads + kvh) * VDIM + col) * page_size + o0 + grp * 4;
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) vs[vt] = load_bf16x4(vp + static_cast<long>(vt) * 16 * page_size);
      return true;
    };
    // steps of 16 keys: those of the request's first `keep_first` keys that lie before the window, then the window's
    const int first_step = lo_run >> 4, kept_steps = min((keep_first + 15) >> 4, first_step);
    const int all_steps = kept_steps + (p_last >> 4) - first_step + 1;
    auto keys_of = [&](int turn) { return (turn < kept_steps ? turn : first_step + turn - kept_steps) << 4; };
    if (wave < all_steps) there = fetch(keys_of(wave), keys, values);
    for (int turn = wave; turn < all_steps; turn += waves) {
      const int j0 = keys_of(turn);
      there_next = turn + waves < all_steps ? fetch(keys_of(turn + waves), keys_next, values_next) : false;
      if (there) {
        float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, keys[dt]),
                                                        __builtin_bit_cast(bf16x8_t, qb[dt]), acc, 0, 0, 0);
        float s[4];
        float highest = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = j0 + grp * 4 + i;
          float v = acc[i] * scale;
          if (softcap > 0.f) {      // tanh(x) = 1 - 2 / (exp(2 x) + 1), with the hardware's exponential and reciprocal
            const float e = __expf(2.f * fabsf(v) * inverse_cap);
            v = copysignf(softcap * (1.f - 2.f * __frcp_rn(e + 1.f)), v);
          }
          if (distance_bias != nullptr)      // (keys behind the query are masked below: their logarithm is taken of 1)
            v -= bias_size * __builtin_amdgcn_logf(fmaf(bias_rate, static_cast<float>(max(my_pos - j, 0)), 1.f));
          s[i] = (in_run && (j >= my_lowest || j < keep_first) && j <= my_pos) ? v : -INFINITY;
          highest = fmaxf(highest, s[i]);
        }
        highest = fmaxf(highest, __shfl_xor(highest, 16, kWave));
        highest = fmaxf(highest, __shfl_xor(highest, 32, kWave));
        const float m_new = fmaxf(m, highest);
        const float correction = m_new == m ? 1.f : __expf(m - m_new);
        float p[4], added = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[i] = s[i] == -INFINITY ? 0.f : __expf(s[i] - m_new);
          added += p[i];
        }
        added += __shfl_xor(added, 16, kWave);
        added += __shfl_xor(added, 32, kWave);
        l = l * correction + added;
        m = m_new;
        short4_t p_high, p_low;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint16_t high = bf16_bits(p[i]);
          p_high[i] = static_cast<short>(high);
          p_low[i] = static_cast<short>(bf16_bits(p[i] - __uint_as_float(static_cast<uint32_t>(high) << 16)));
        }
        const int beyond = j0 + grp * 4 + 3 - p_last;      // this many of the lane's four keys are not written yet
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          short4_t operand = values[vt];
          if (beyond > 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (i > 3 - beyond) operand[i] = 0;
          }
          float4_t sum = o[vt];
#pragma unroll
          for (int i = 0; i < 4; ++i) sum[i] *= correction;
          sum = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(operand, p_high, sum, 0, 0, 0);
          o[vt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(operand, p_low, sum, 0, 0, 0);
        }
      }
      there = there_next;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) keys[dt] = keys_next[dt];
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) values[vt] = values_next[vt];
    }
    row = run_end;
  }
  if (waves > 1) {      // the waves' shares meet in LDS and the first wave adds them in the order of the waves
    float* mine = tile_shares + static_cast<size_t>(wave) * (2 + 4 * VT) * kWave + lane;
    mine[0] = m;
    mine[kWave] = l;
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int i = 0; i < 4; ++i) mine[(2 + 4 * vt + i) * kWave] = o[vt][i];
    __syncthreads();
    if (wave != 0) return;
    float highest = m;
    for (int w = 1; w < waves; ++w) highest = fmaxf(highest, tile_shares[static_cast<size_t>(w) * (2 + 4 * VT) * kWave + lane]);
    const float own = m == -INFINITY ? 0.f : expf(m - highest);
    l *= own;
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[vt][i] *= own;
    for (int w = 1; w < waves; ++w) {
      const float* other = tile_shares + static_cast<size_t>(w) * (2 + 4 * VT) * kWave + lane;
      const float factor = other[0] == -INFINITY ? 0.f : expf(other[0] - highest);
      l += other[kWave] * factor;
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[vt][i] += other[(2 + 4 * vt + i) * kWave] * factor;
    }
  }
  if (!have) return;
  float gate = out_scale;
  if (gates != nullptr) gate = out_scale / (1.f + expf(-to_float(gates[static_cast<long>(my_row) * gate_stride + gate_at + head])));
  const float factor = gate / l;
  bf16_t* dst = out + static_cast<long>(my_row) * out_stride + head * VDIM + grp * 4;
#pragma unroll
  for (int vt = 0; vt < VT; ++vt) {
    uint2 packed;
    packed.x = bf16_pair(o[vt][0] * factor, o[vt][1] * factor);
    packed.y = bf16_pair(o[vt][2] * factor, o[vt][3] * factor);
    *reinterpret_cast<uint2*>(dst + vt * 16) = packed;
  }
}

}  // namespace

extern "C" {

// The same for rows first_row .. tokens - 1 of a bfloat16 step on the matrix cores: keys and values of 32, 64, 128 or 256,
// pages of a multiple of 16 tokens (-2 otherwise).  Rows of a request follow each other in the order of their positions.
int akv_gated_attention_tiles(const void* q, const void* k_pages, const void* v_pages, const void* gates, long gate_stride,
                              int gate_at, const int* seq_of_token, const int* q_start, const int* positions,
                              const int* block_table, const int* table_rows, int table_width, void* out, int first_row,
                              int tokens, int q_heads, int kv_heads, int dim, int vdim, int page_size, long num_pages,
                              float scale, float softcap, int chunk, int window, int sink, long out_stride, float out_scale,
                              const float* sink_logits, int maps, int keep_first, const float* distance_bias,
                              hipStream_t stream) {
  if (tokens <= first_row) return 0;
  if (page_size % 16 != 0 || q_heads % kv_heads != 0 || maps < 1) return -2;
  if (!aligned_for_tiles(q, k_pages, v_pages, out, out_stride)) return -2;
  const long items = static_cast<long>((tokens - first_row + 15) / 16) * q_heads;
  const unsigned grid = static_cast<unsigned>(((tokens - first_row + 15) / 16 + kXcds - 1) / kXcds * kXcds * q_heads);
  const int waves = vdim > 128 ? 2 : 4;       // (their shares must fit into 64 KB of LDS)
  const size_t lds = static_cast<size_t>(waves) * (2 + vdim / 4) * kWave * 4;
#define AKV_TILES(DT, VT)                                                                                              \
  gated_attention_tiles_kernel<DT, VT><<<grid, waves * kWave, lds, stream>>>(                                                    \
      static_cast<const bf16_t*>(q), static_cast<const bf16_t*>(k_pages), static_cast<const bf16_t*>(v_pages),         \
      static_cast<const bf16_t*>(gates), gate_stride, gate_at, seq_of_token, q_start, positions, block_table, table_rows, \
      table_width, static_cast<bf16_t*>(out), first_row, tokens, q_heads, kv_heads, page_size, num_pages, scale, softcap, \
      chunk, window, sink, out_stride, out_scale, sink_logits, maps, keep_first, distance_bias)
#define AKV_TILES_V(DT)                    \
  switch (vdim) {                          \
    case 32: AKV_TILES(DT, 2); break;      \
    case 64: AKV_TILES(DT, 4); break;      \
    case 128: AKV_TILES(DT, 8); break;     \
    case 256: AKV_TILES(DT, 16); break;    \
    default: return -2;                    \
  }
  switch (dim) {
    case 32: AKV_TILES_V(1); break;
    case 64: AKV_TILES_V(2); break;
    case 128: AKV_TILES_V(4); break;
    case 256: AKV_TILES_V(8); break;
    default: return -2;
  }
#undef AKV_TILES_V
#undef AKV_TILES
  return AKV_LAUNCH_STATUS();
}

int akv_unit_norm_write(const void* projected, long stride, int dtype, long tokens, int q_heads, int kv_heads, int dim,
                        int vdim, float eps, int normed, const int* slot_map, void* k_pages, void* v_pages, int page_size,
                        long num_pages, void* q_out, int maps, const float* table, int table_positions, int rot_dims,
                        const int* positions, const float* q_weight, const float* k_weight, int whole, int interleaved,
                        float value_eps, float temp_coef, int temp_every, int keyed_values, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (q_heads <= 0 || kv_heads <= 0 || dim <= 0 || vdim <= 0 || page_size <= 0 || maps < 1) return -2;
  if (table != nullptr && (rot_dims < 0 || rot_dims % 2 != 0 || rot_dims > dim || positions == nullptr)) return -2;
  if (temp_every > 0 && positions == nullptr) return -2;
  if (keyed_values && (vdim != dim || maps != 1)) return -2;
  const int values_at = keyed_values ? q_heads * dim : (q_heads + kv_heads) * maps * dim;
  const long items = tokens * ((q_heads + kv_heads) * maps + kv_heads);
  if (whole && normed) {
    // (few tokens: sixteen waves a token share its items; many: four, and the tokens fill the device)
    const int threads = tokens <= 256 ? 1024 : 256;
    AKV_DISPATCH(dtype, T, unit_norm_write_whole_kernel<T><<<static_cast<unsigned>(tokens), threads, 0, stream>>>(
                               static_cast<const T*>(projected), stride, q_heads, kv_heads, dim, vdim, eps, slot_map,
                               static_cast<T*>(k_pages), static_cast<T*>(v_pages), page_size, num_pages, static_cast<T*>(q_out),
                               maps, table, table_positions, rot_dims, positions, q_weight, k_weight, interleaved, value_eps,
                               temp_coef, temp_every, values_at));
    return AKV_LAUNCH_STATUS();
  }
  // Eights: nothing but a norm and a rotation of halves, and every 16-byte group of a vector, a rotated half or a page row is
  // whole and aligned - of all numbers of tokens, so that a token's bits do not depend on how its request was cut (2,000
  // tokens 10 us against 19 to 28, 8 tokens 4 us either way).
  const auto aligned = [](const void* at) { return reinterpret_cast<uintptr_t>(at) % 16 == 0; };
  const int eights = dim / 8;
  const bool rotates = table != nullptr && rot_dims > 0;
  if (dtype == 1 && dim % 8 == 0 && vdim % 8 == 0 && stride % 8 == 0 && page_size % 8 == 0 &&
      (q_heads + kv_heads) * static_cast<long>(maps) * eights * tokens < (1L << 31) && q_weight == nullptr &&
      k_weight == nullptr && value_eps < 0.f && temp_every <= 0 &&
      (!rotates || (rot_dims % 16 == 0 && !interleaved)) && (!normed || ((eights & (eights - 1)) == 0 && eights <= kWave)) &&
      aligned(projected) && aligned(q_out) && aligned(k_pages) && aligned(v_pages)) {
    const long vectors = (q_heads + (slot_map != nullptr ? kv_heads : 0)) * static_cast<long>(maps);
    const long value_items = slot_map != nullptr ? (tokens + 7) / 8 * kv_heads * ((vdim + 63) / 64) : 0;
    const unsigned vector_blocks = static_cast<unsigned>((vectors * eights * tokens + 255) / 256);
    const unsigned blocks = vector_blocks + static_cast<unsigned>((value_items + 3) / 4);
    const auto kernel = normed ? unit_norm_write_eights_kernel<true> : unit_norm_write_eights_kernel<false>;
    kernel<<<blocks, 256, 0, stream>>>(static_cast<const bf16_t*>(projected), stride, static_cast<int>(tokens), q_heads * maps,
                                       kv_heads, dim, vdim, eps, slot_map, static_cast<bf16_t*>(k_pages),
                                       static_cast<bf16_t*>(v_pages), page_size, num_pages, static_cast<bf16_t*>(q_out), maps,
                                       table, table_positions, rotates ? rot_dims : 0, positions, values_at, vector_blocks);
    return AKV_LAUNCH_STATUS();
  }
  AKV_DISPATCH(dtype, T, unit_norm_write_kernel<T><<<static_cast<unsigned>((items + 3) / 4), 256, 0, stream>>>(
                             static_cast<const T*>(projected), stride, tokens, q_heads, kv_heads, dim, vdim, eps, normed,
                             slot_map, static_cast<T*>(k_pages), static_cast<T*>(v_pages), page_size, num_pages,
                             static_cast<T*>(q_out), maps, table, table_positions, rot_dims, positions, q_weight,
                             k_weight, interleaved, value_eps, temp_coef, temp_every, values_at));
  return AKV_LAUNCH_STATUS();
}

int akv_gated_attention_rows(const void* q, const void* k_pages, const void* v_pages, const void* gates, long gate_stride,
                             int gate_at, const int* seq_of_token, const int* positions, const int* block_table,
                             const int* table_rows, int table_width, void* out, int dtype, long tokens, int q_heads,
                             int kv_heads, int dim, int vdim, int page_size, long num_pages, float scale, float softcap,
                             int chunk, int window, int sink, long out_stride, float out_scale, int row_waves,
                             const float* sink_logits, int maps, int keep_first, const float* distance_bias,
                             hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (maps < 1) return -2;
  const int kRowWaves = row_waves;
  if (row_waves < 1 || row_waves > kMaxRowWaves) return -2;
  if (vdim > kMaxValueRegs * kWave || dim <= 0 || q_heads % kv_heads != 0) return -2;
  // A block a head.  (The kernel can take 2 or 4 query heads of a key head in one block, reading keys and values once
  // for them; with a quarter of the blocks at its register count that was slower at 8 requests of 2,048 keys, 16 query
  // and 4 key heads - 66 us against 39 - and is not chosen.)
  int bundle = 1;
  int waves = kRowWaves;
  auto lds_of = [&](int g, int w) {
    return (static_cast<size_t>(g) * dim * 4 + 7) / 8 * 8 + static_cast<size_t>(w) * kWave * (g * 4 + 8) +
           static_cast<size_t>(w) * g * (2 + vdim) * 4;
  };
  while (lds_of(bundle, waves) > 64 * 1024 && waves > 1) waves /= 2;
  while (lds_of(bundle, waves) > 64 * 1024 && bundle > 1) bundle /= 2;
  const size_t lds = lds_of(bundle, waves);
  if (lds > 64 * 1024) return -2;
  const long rows = tokens * (q_heads / bundle);
  const size_t element = dtype == kBF16 ? 2 : 4;
  // 16-byte loads: key rows and groups of eight neighbouring keys' values must be aligned
  const bool vec = (dim * element) % 16 == 0 && page_size % 8 == 0 &&
                   (static_cast<size_t>(page_size) * element) % 16 == 0 && reinterpret_cast<uintptr_t>(k_pages) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(v_pages) % 16 == 0;
  const unsigned grid = static_cast<unsigned>((rows + kXcds - 1) / kXcds * kXcds);
#define AKV_ROWS(VEC, G)                                                                                                \
  AKV_DISPATCH(dtype, T,                                                                                                \
               gated_attention_rows_kernel<T, VEC, G><<<grid, waves * kWave, lds, stream>>>(                           \
                   static_cast<const T*>(q), static_cast<const T*>(k_pages), static_cast<const T*>(v_pages),            \
                   static_cast<const T*>(gates), gate_stride, gate_at, seq_of_token, positions, block_table, table_rows, \
                   table_width, static_cast<T*>(out), tokens, q_heads, kv_heads, dim, vdim, page_size, num_pages, scale, \
                   softcap, chunk, window, sink, out_stride, out_scale, sink_logits, maps, keep_first, distance_bias))
#define AKV_ROWS_G(VEC)          \
  switch (bundle) {              \
    case 4: AKV_ROWS(VEC, 4); break; \
    case 2: AKV_ROWS(VEC, 2); break; \
    default: AKV_ROWS(VEC, 1); break; \
  }
  if (vec) AKV_ROWS_G(true)
  else AKV_ROWS_G(false)
#undef AKV_ROWS_G
#undef AKV_ROWS
  return AKV_LAUNCH_STATUS();
}
}

namespace {

// ---- single tokens on the matrix cores ---------------------------------------------------------------------------------
// bfloat16, the sizes of the tiles above.  What a single token waits for is its keys and values: a block that walks them all
// for one query head asks for them a tile after the other, and the heads of a group ask for the same ones again.  Here a
// block is a token, a vector of a key head with all query vectors that read it as the columns of a tile, and ONE segment of 16
// steps of 16 keys at absolute positions; its four waves take four steps each and ask for all of their keys and values
// before the first score: one trip to the block table, one to the pages.  A wave's 64 keys have one maximum; waves and
// segments are folded in their order.  A token of one segment is finished by its block; of more, the segments' sums are left
// in `partial` ([token][query vector][segment][vdim + 4], as many of the step's tokens at once as the caller has room for) and
// added by `gated_attention_fold_kernel`.  How a token's keys are cut depends on its position alone.  Scores, maxima, weights and sums are float32; a weight enters the second product as
// three bfloat16 numbers that add up to it.
// What bounds it: trips to memory in a row (positions, table, keys and values, then the fold's launch).  8 tokens of 2,048 keys
// (34 MB), 16 query and 4 key heads of 128, us: 39 with a block of sixteen waves per (token, query head) in `rows`, 14 + 7 for
// the fold here; two maps of 64 over a window of 1,024: 26.5 -> 12 + 5.  (With the loads behind tests, which the compiler
// waits for one by one, and the softcap's and the bias's code in every kernel: 33.)  Where tokens and key heads are many, blocks
// beside each other on a unit hide the trips: up to four, where registers allow them (64 tokens of 2,048 keys, 16 heads of 64 of
// their own: 119 us, 139 with two at most).
struct Steps {
  int lowest, first, kept, all;      // the window's first key; its step, the steps of the kept first keys, all steps
  __device__ __forceinline__ Steps(int pos, int window, int chunk, int keep_first) {
    lowest = window > 0 ? max(0, pos - window + 1) : 0;
    if (chunk > 0) lowest = max(lowest, pos / chunk * chunk);
    first = lowest >> 4;
    kept = min((keep_first + 15) >> 4, first);
    all = kept + (pos >> 4) - first + 1;
  }
  __device__ __forceinline__ int key(int turn) const { return (turn < kept ? turn : first + turn - kept) << 4; }
};
constexpr int kSegmentSteps = 16;

// What a running (maximum, sum of weights, weighted sums) and a later part of it are multiplied by when they are added.
struct Fold {
  float kept, added;
  __device__ __forceinline__ Fold(float& maximum, float other) {
    const float m = fmaxf(maximum, other);
    const float shift = m == -INFINITY ? 0.f : m;          // (of a part of no keys the factor is exp(-inf))
    kept = expf(maximum - shift);
    added = expf(other - shift);
    maximum = m;
  }
  __device__ __forceinline__ float operator()(float total, float part) const { return fmaf(total, kept, part * added); }
};

struct SingleArgs {
  const bf16_t *q, *k_pages, *v_pages, *gates;
  const int *seq_of_token, *positions, *block_table, *table_rows;
  const float *sink_logits, *distance_bias;
  bf16_t* out;
  float* partial;
  long gate_stride, num_pages, out_stride;
  float scale, softcap, out_scale;
  int gate_at, table_width, q_heads, kv_heads, page_size, chunk, window, sink, maps, keep_first, segments;
  int share, groups;                 // query vectors of a key vector, tiles of 16 of them
  Divider by_segments, by_page, by_maps_and_groups, by_groups, by_heads;   // (a block's divisions stand before its first load)
};

__device__ __forceinline__ float gate_of(const SingleArgs& a, long n, int vector) {
  if (a.gates == nullptr) return a.out_scale;
  return a.out_scale / (1.f + expf(-to_float(a.gates[n * a.gate_stride + a.gate_at + vector])));
}
__device__ __forceinline__ float sink_of(const SingleArgs& a, int vector) {
  return !a.sink ? -INFINITY : a.sink_logits != nullptr ? a.sink_logits[vector] : 0.f;
}

// SHAPED: scores have a softcap or a distance bias (their code, in every kernel, would be most of what a block fetches).
// SHORT: one segment holds all keys that a token can see.  A wave that has one step of 16 keys takes that one alone, and one that
// has none leaves zeros for the fold: 256 tokens of 30 keys, 16 heads of 64 of their own, 52 -> 20 us, of 128 77 -> 37 (14 and 21 in
// `gated_attention_rows`, a wave per token and head), 16 / 4 heads of 128 24.5 -> 12.6 (17).  Of several segments most are whole, and
// a look at the steps first would stand before their loads.
template <int DT, int VT, bool SHAPED, bool SHORT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 4))) void gated_attention_singles_kernel(const SingleArgs a) {
  constexpr int DIM = 32 * DT, VDIM = 16 * VT, kOwn = (VT + 3) / 4;      // tiles of values whose totals a wave keeps
  __shared__ float4_t sums_of[4][VT][kWave];
  __shared__ float top_of[4][16], weight_of[4][16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  const int col = lane & 15, grp = lane >> 4;
  const long n = a.by_segments.quotient(blockIdx.x);
  const int segment = a.by_segments.rest(blockIdx.x, static_cast<int>(n));
  const int share = a.share, kvh = a.by_maps_and_groups.quotient(blockIdx.y), of_key = a.by_maps_and_groups.rest(blockIdx.y, kvh);
  const int map = a.by_groups.quotient(of_key), of_group = a.by_groups.rest(of_key, map) * 16 + col;
  const int vector = (kvh * share + min(of_group, share - 1)) * a.maps + map;
  const int r = a.table_rows != nullptr ? a.table_rows[a.seq_of_token[n]] : a.seq_of_token[n];
  const int pos = a.positions[n];
  const Steps steps(pos, a.window, a.chunk, a.keep_first);
  const int first = segment * kSegmentSteps;
  if (first >= steps.all) return;

  const int* table = a.block_table + static_cast<long>(r) * a.table_width;
  float4_t sums[VT];
#pragma unroll
  for (int v = 0; v < VT; ++v) sums[v] = float4_t{0.f, 0.f, 0.f, 0.f};
  float top = -INFINITY, weight = 0.f;
  // a wave's first STEPS steps: scores, their maximum, weights and weighted sums
  const auto take = [&](auto count) {
    constexpr int STEPS = decltype(count)::value;
    uint4 q[DT], keys[STEPS][DT];
    uint2 values[STEPS][VT];
    int at_key[STEPS], offset[STEPS];
    long page[STEPS];
    bool foreign[STEPS];
    // (no load stands behind a test: the compiler would wait for it before the next; a step beyond the last asks for the last)
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int turn = first + wave + 4 * i;
      const int key = steps.key(min(turn, steps.all - 1));
      const int nth = a.by_page.quotient(key);
      page[i] = table[nth];
      offset[i] = a.by_page.rest(key, nth);
      at_key[i] = turn < steps.all ? key : pos + 1;                  // (none of a step beyond the last counts)
    }
    const bf16_t* qp = a.q + (n * a.q_heads + vector) * DIM + grp * 8;
#pragma unroll
    for (int d = 0; d < DT; ++d) q[d] = load_bf16x8(qp + d * 32);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      foreign[i] = page[i] < 0 || page[i] >= a.num_pages;            // (a page that is not the request's is never read: its
      const long from = (foreign[i] ? 0 : page[i]) * a.kv_heads + kvh;                                 // scores are NaN)
      const bf16_t* kp = a.k_pages + ((from * a.page_size + offset[i] + col) * a.maps + map) * DIM + grp * 8;
#pragma unroll
      for (int d = 0; d < DT; ++d) keys[i][d] = load_bf16x8(kp + d * 32);
    }
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const long from = (foreign[i] ? 0 : page[i]) * a.kv_heads + kvh;
      const bf16_t* vp = a.v_pages + (from * VDIM + col) * a.page_size + offset[i] + grp * 4;
#pragma unroll
      for (int v = 0; v < VT; ++v) values[i][v] = *reinterpret_cast<const uint2*>(vp + static_cast<long>(v) * 16 * a.page_size);
    }
    __builtin_amdgcn_sched_barrier(0);             // (else the loads are moved down to where they are used)

    const auto counts = [&](int i, int e) {
      const int j = at_key[i] + 4 * grp + e;
      return ((j >= steps.lowest) | (j < a.keep_first)) & (j <= pos);
    };
    const float bias_size = SHAPED && a.distance_bias != nullptr ? a.distance_bias[vector] : 0.f;
    const float bias_rate = SHAPED && a.distance_bias != nullptr ? a.distance_bias[a.q_heads + vector] : 0.f;
    float s[STEPS][4];
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < DT; ++d)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, keys[i][d]), __builtin_bit_cast(bf16x8_t, q[d]),
                                                      acc, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = acc[e] * a.scale;
        if constexpr (SHAPED) {
          if (a.softcap > 0.f) v = a.softcap * tanhf(v / a.softcap);
          if (a.distance_bias != nullptr)
            v -= bias_size * log1pf(bias_rate * static_cast<float>(max(pos - at_key[i] - 4 * grp - e, 0)));
        }
        if (foreign[i]) v = __uint_as_float(0x7fc00000u);
        s[i][e] = counts(i, e) ? v : -INFINITY;
        top = fmaxf(top, s[i][e]);
      }
    }
    top = fmaxf(top, __shfl_xor(top, 16, kWave));
    top = fmaxf(top, __shfl_xor(top, 32, kWave));
    const float shift = top == -INFINITY ? 0.f : top;
    bool fine = true;
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      uint32_t kept[2] = {0u, 0u};                 // slots that nobody has written hold anything: what does not count is zero
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool counted = counts(i, e);
        s[i][e] = expf(s[i][e] - shift);           // (exp(-inf) where the key does not count)
        weight += s[i][e];
        kept[e >> 1] |= counted & !foreign[i] ? 0xffffu << (16 * (e & 1)) : 0u;
      }
#pragma unroll
      for (int v = 0; v < VT; ++v) {
        values[i][v].x &= kept[0];
        values[i][v].y &= kept[1];
        fine = fine & ((values[i][v].x & 0x7f80u) != 0x7f80u) & ((values[i][v].x & 0x7f800000u) != 0x7f800000u) &
               ((values[i][v].y & 0x7f80u) != 0x7f80u) & ((values[i][v].y & 0x7f800000u) != 0x7f800000u);
      }
    }
    weight += __shfl_xor(weight, 16, kWave);
    weight += __shfl_xor(weight, 32, kWave);

    if (__builtin_expect(__all(fine), 1)) {
      // two steps of 16 keys are one product over 32: a lane's eight are keys 4 grp .. + 3 of the one and of the other
#pragma unroll
      for (int i = 0; i < STEPS; i += 2) {
        float left[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) left[e] = i + (e >> 2) < STEPS ? s[min(i + (e >> 2), STEPS - 1)][e & 3] : 0.f;
#pragma unroll
        for (int part = 0; part < 3; ++part) {
          uint32_t words[4];
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            words[w] = bf16_pair(left[2 * w], left[2 * w + 1]);
            left[2 * w] -= __uint_as_float(words[w] << 16);
            left[2 * w + 1] -= __uint_as_float(words[w] & 0xffff0000u);
          }
          const bf16x8_t weights = __builtin_bit_cast(bf16x8_t, make_uint4(words[0], words[1], words[2], words[3]));
#pragma unroll
          for (int v = 0; v < VT; ++v)
            sums[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8_t, make_uint4(values[i][v].x, values[i][v].y, i + 1 < STEPS ? values[min(i + 1, STEPS - 1)][v].x : 0u,
                                                        i + 1 < STEPS ? values[min(i + 1, STEPS - 1)][v].y : 0u)),
                weights, sums[v], 0, 0, 0);
        }
      }
    } else {
      // an infinite or undefined value: a weight of zero takes nothing from it (zero times infinity is not zero), so the keys
      // are added one by one - of step i the one that lies in element e of group `four` - where their weight is not zero
#pragma unroll
      for (int i = 0; i < STEPS; ++i)
#pragma unroll 1
        for (int one = 0; one < 16; ++one) {
          const int four = one >> 2, e = one & 3;
          const float own = e == 0 ? s[i][0] : e == 1 ? s[i][1] : e == 2 ? s[i][2] : s[i][3];
          const bool taken = __shfl(own, 16 * four + col, kWave) != 0.f;
          const uint32_t place = grp == four ? 0xffffu << (16 * (e & 1)) : 0u;
          const uint2 only = make_uint2(e < 2 ? place : 0u, e < 2 ? 0u : place);
          short4_t part[3];
          float left = own;
#pragma unroll
          for (int t = 0; t < 3; ++t) {
            const uint32_t bits = bf16_bits(left);
            left -= __uint_as_float(bits << 16);
            part[t] = __builtin_bit_cast(short4_t, make_uint2((bits | bits << 16) & only.x, (bits | bits << 16) & only.y));
          }
#pragma unroll
          for (int v = 0; v < VT; ++v) {
            const short4_t value = __builtin_bit_cast(short4_t, make_uint2(values[i][v].x & only.x, values[i][v].y & only.y));
            float4_t with = sums[v];
#pragma unroll
            for (int t = 0; t < 3; ++t) with = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(value, part[t], with, 0, 0, 0);
            if (taken) sums[v] = with;
          }
        }
    }
  };
  const int own = (steps.all - first - wave + 3) >> 2;               // (steps of the wave, four at most)
  if (!SHORT || own > 1)
    take(std::integral_constant<int, 4>());
  else if (own == 1)
    take(std::integral_constant<int, 1>());

  // the four waves' parts, in their order; a token of one segment starts from its sink
#pragma unroll
  for (int v = 0; v < VT; ++v) sums_of[wave][v][lane] = sums[v];
  if (grp == 0) {
    top_of[wave][col] = top;
    weight_of[wave][col] = weight;
  }
  __syncthreads();
  const bool whole = steps.all <= kSegmentSteps;
  float total_top = whole ? sink_of(a, vector) : -INFINITY, total_weight = total_top == -INFINITY ? 0.f : 1.f;
  float4_t total[kOwn];
#pragma unroll
  for (int i = 0; i < kOwn; ++i) total[i] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const Fold f(total_top, top_of[w][col]);
    total_weight = f(total_weight, weight_of[w][col]);
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      if (wave + 4 * i >= VT) continue;
      const float4_t part = sums_of[w][wave + 4 * i][lane];
#pragma unroll
      for (int d = 0; d < 4; ++d) total[i][d] = f(total[i][d], part[d]);
    }
  }
  if (of_group >= share) return;
  if (!whole) {
    float* at = a.partial + ((n * a.q_heads + vector) * a.segments + segment) * (VDIM + 4);
#pragma unroll
    for (int i = 0; i < kOwn; ++i)
      if (wave + 4 * i < VT) *reinterpret_cast<float4_t*>(at + 16 * (wave + 4 * i) + 4 * grp) = total[i];
    if (wave == 0 && grp == 0) {
      at[VDIM] = total_top;
      at[VDIM + 1] = total_weight;
    }
    return;
  }
  const float factor = gate_of(a, n, vector) / total_weight;
  bf16_t* at = a.out + n * a.out_stride + static_cast<long>(vector) * VDIM + 4 * grp;
#pragma unroll
  for (int i = 0; i < kOwn; ++i) {
    if (wave + 4 * i >= VT) continue;
    uint2 packed;
    packed.x = bf16_pair(total[i][0] * factor, total[i][1] * factor);
    packed.y = bf16_pair(total[i][2] * factor, total[i][3] * factor);
    *reinterpret_cast<uint2*>(at + 16 * (wave + 4 * i)) = packed;
  }
}

// The segments of every (token, query vector) that has more than one, in their order: a wave a row, four values a lane.
__global__ __launch_bounds__(256) void gated_attention_fold_kernel(const SingleArgs a, int vdim, long rows) {
  const int lane = threadIdx.x & (kWave - 1);
  const long row = static_cast<long>(blockIdx.x) * 4 + threadIdx.x / kWave;
  if (row >= rows) return;
  const long n = a.by_heads.quotient(static_cast<int>(row));
  const int vector = a.by_heads.rest(static_cast<int>(row), static_cast<int>(n));
  const Steps steps(a.positions[n], a.window, a.chunk, a.keep_first);
  if (steps.all <= kSegmentSteps || 4 * lane >= vdim) return;
  const int count = min((steps.all + kSegmentSteps - 1) / kSegmentSteps, a.segments);
  const float* at = a.partial + row * a.segments * (vdim + 4);
  float total_top = sink_of(a, vector), total_weight = total_top == -INFINITY ? 0.f : 1.f;
  float4_t total = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int segment = 0; segment < count; ++segment) {
    const float* part = at + static_cast<long>(segment) * (vdim + 4);
    const float4_t sums = *reinterpret_cast<const float4_t*>(part + 4 * lane);
    const Fold f(total_top, part[vdim]);
    total_weight = f(total_weight, part[vdim + 1]);
#pragma unroll
    for (int d = 0; d < 4; ++d) total[d] = f(total[d], sums[d]);
  }
  const float factor = gate_of(a, n, vector) / total_weight;
  uint2 packed;
  packed.x = bf16_pair(total[0] * factor, total[1] * factor);
  packed.y = bf16_pair(total[2] * factor, total[3] * factor);
  *reinterpret_cast<uint2*>(a.out + n * a.out_stride + static_cast<long>(vector) * vdim + 4 * lane) = packed;
}

}  // namespace

extern "C" {

int akv_gated_attention_singles(const void* q, const void* k_pages, const void* v_pages, const void* gates, long gate_stride,
                                int gate_at, const int* seq_of_token, const int* positions, const int* block_table,
                                const int* table_rows, int table_width, void* out, float* partial, int segments, int at_once,
                                int tokens, int q_heads, int kv_heads, int dim, int vdim, int page_size, long num_pages, float scale,
                                float softcap, int chunk, int window, int sink, long out_stride, float out_scale,
                                const float* sink_logits, int maps, int keep_first, const float* distance_bias,
                                hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (page_size % 16 != 0 || maps < 1 || kv_heads <= 0 || q_heads % (kv_heads * maps) != 0 || segments < 1 || at_once < 1 ||
      static_cast<long>(at_once) * segments > 0x7fffffffL || (segments > 1 && partial == nullptr))
    return -2;
  SingleArgs a{static_cast<const bf16_t*>(q), static_cast<const bf16_t*>(k_pages), static_cast<const bf16_t*>(v_pages),
                     static_cast<const bf16_t*>(gates), seq_of_token, positions, block_table, table_rows, sink_logits,
                     distance_bias, static_cast<bf16_t*>(out), partial, gate_stride, num_pages, out_stride, scale, softcap,
                     out_scale, gate_at, table_width, q_heads, kv_heads, page_size, chunk, window, sink, maps, keep_first, segments};
  a.share = q_heads / kv_heads / maps, a.groups = (a.share + 15) / 16;
  if (a.share < 1 || page_size < 1) return -2;
  at_once = min(at_once, 0x7fffffff / q_heads);      // (a launch's rows of the fold are counted in 31 bits)
  a.by_segments = Divider::of(segments), a.by_page = Divider::of(page_size), a.by_groups = Divider::of(a.groups);
  a.by_maps_and_groups = Divider::of(maps * a.groups), a.by_heads = Divider::of(q_heads);
  const long columns = static_cast<long>(kv_heads) * maps * a.groups;
  if (!aligned_for_tiles(q, k_pages, v_pages, out, out_stride)) return -2;
  if (columns > 65535) return -2;
  // (a launch's partial sums are folded before the next one, on the same stream, writes its own)
  for (int first = 0; first < tokens; first += at_once) {
    const int count = min(at_once, tokens - first);
    const dim3 grid(static_cast<unsigned>(static_cast<long>(count) * segments), static_cast<unsigned>(columns));
    const bool shaped = softcap > 0.f || distance_bias != nullptr;
#define AKV_SINGLES(DT, VT)                                                                        \
  if (segments > 1 && shaped)                                                                      \
    gated_attention_singles_kernel<DT, VT, true, false><<<grid, 256, 0, stream>>>(a);               \
  else if (segments > 1)                                                                           \
    gated_attention_singles_kernel<DT, VT, false, false><<<grid, 256, 0, stream>>>(a);              \
  else if (shaped)                                                                                 \
    gated_attention_singles_kernel<DT, VT, true, true><<<grid, 256, 0, stream>>>(a);                \
  else                                                                                             \
    gated_attention_singles_kernel<DT, VT, false, true><<<grid, 256, 0, stream>>>(a)
#define AKV_SINGLES_V(DT)                  \
  switch (vdim) {                          \
    case 32: AKV_SINGLES(DT, 2); break;    \
    case 64: AKV_SINGLES(DT, 4); break;    \
    case 128: AKV_SINGLES(DT, 8); break;   \
    case 256: AKV_SINGLES(DT, 16); break;  \
    default: return -2;                    \
  }
    switch (dim) {
      case 32: AKV_SINGLES_V(1); break;
      case 64: AKV_SINGLES_V(2); break;
      case 128: AKV_SINGLES_V(4); break;
      case 256: AKV_SINGLES_V(8); break;
      default: return -2;
    }
#undef AKV_SINGLES_V
#undef AKV_SINGLES
    if (segments > 1) {
      const long rows = static_cast<long>(count) * q_heads;
      gated_attention_fold_kernel<<<static_cast<unsigned>((rows + 3) / 4), 256, 0, stream>>>(a, vdim, rows);
    }
    a.q += static_cast<long>(count) * q_heads * dim;
    a.out += count * out_stride;
    a.seq_of_token += count;
    a.positions += count;
    if (a.gates != nullptr) a.gates += count * gate_stride;
  }
  return AKV_LAUNCH_STATUS();
}

}

namespace {

// ---- prompt portions, keys and values shared through LDS ------------------------------------------------------------------
// bfloat16, keys and values of 32, 64 or 128, where the portions make enough blocks to fill the device.  The tiles above
// have every wave fetch its own keys and values: 2,000 tokens of 16 heads ask the L2 for a gigabyte, and a step of 16 keys
// pays the softmax's bookkeeping for four scores a lane.  Here a block is 64 columns - consecutive (token, query vector)
// pairs of one request whose vectors read one vector of one key head -, a wave 16 of them; a step is 32 keys at absolute
// positions, fetched once by the block two steps ahead and filed in two LDS buffers in turn (one barrier a step): keys by rows of the
// head's width, values by rows of 32 keys in the order of the second product's operand (a lane's eight are keys 4 g .. 4 g + 3
// of the step's two sixteens, where the first product leaves their scores).  Rows are padded by 16 bytes, so that a 16-byte
// read of sixteen rows meets no bank twice.  A wave passes over steps that none of its columns sees.  Scores, maxima,
// weights and sums are float32 (base 2); a weight enters the second product as two bfloat16; the exponentials' reference
// point trails the maximum by at most 2^8, so that sums are rescaled a few times a prompt and not once a step.
// A key that one column sees and another does not has weight zero for the other, and zero times an infinity is not zero: where a
// step is masked for some column of the block, the threads that file its values file zeros for what is not finite and say so,
// and the waves then add it, one value at a time, to the columns that see its key (finite values pay for the look in a few
// steps a block: 2,048 tokens of 16 heads of 64 of their own 56.5 -> 59.0 us, of 16 / 4 heads of 128 76.7 -> 74.6).
// What bounds it: a step's chain of dependent instructions (products, maximum, exponentials, products: 1.2 us with one wave a
// SIMD), as often as the longest block has steps; two blocks a unit fill each other's gaps.  2,000 tokens of 16 / 4 heads of
// 128, us: 116 with the tiles above, 102 here with pages and keys asked for a step ahead, 85 two steps ahead, 75 with the
// place in the page moved on by additions (a division a page and sixteen: 40 instructions of a step's 500).
constexpr int kSharedColumns = 64;

// The maximum over the four lanes c, c + 16, c + 32 and c + 48, in all four: lane swaps inside the vector unit.
__device__ __forceinline__ float max_over_groups(float v) {
  const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(halves[0]), __uint_as_float(halves[1]));
  const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(rows[0]), __uint_as_float(rows[1]));
}
constexpr float kTrail = 8.f;

struct SharedArgs {
  const bf16_t *q, *k_pages, *v_pages, *gates;
  const int *q_start, *seq_lens, *block_table, *table_rows;
  const float *sink_logits, *distance_bias;
  bf16_t* out;
  long gate_stride, num_pages, out_stride;
  float scale, softcap, out_scale;
  int first_seq, seqs, tiles, gate_at, table_width, q_heads, kv_heads, page_size, chunk, window, sink, maps, keep_first;
};

template <int DT, int VT, bool SHAPED>
__global__ __launch_bounds__(256, 2) void gated_attention_shared_kernel(const SharedArgs a) {
  constexpr int DIM = 32 * DT, VDIM = 16 * VT, kKeyRow = DIM + 8, kValueRow = 32 + 8;
  constexpr int kKeyLoads = (32 * DIM / 8 + 255) / 256, kValueLoads = (VDIM * 4 + 255) / 256;     // 16 bytes a thread each
  __shared__ __attribute__((aligned(16))) bf16_t filed_keys[2][32 * kKeyRow];
  __shared__ __attribute__((aligned(16))) bf16_t filed_values[2][VDIM * kValueRow];
  __shared__ __attribute__((aligned(4))) unsigned char filed_infinite[2][4];     // by wave: what it was to file is not all finite
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  const int col = lane & 15, grp = lane >> 4;
  const int share = a.q_heads / a.kv_heads / a.maps, columns = a.kv_heads * a.maps;
  const int kvh = blockIdx.x % columns / a.maps, map = blockIdx.x % a.maps;
  // whose tile this is: numbered request by request; the last ones - those with the most keys before them - start first
  int request = -1, tile = a.tiles - 1 - static_cast<int>(blockIdx.x) / columns;
  for (int first = a.first_seq; first < a.seqs && request < 0; first += kWave) {
    const int r = first + lane;
    const int count = r < a.seqs ? ((a.q_start[r + 1] - a.q_start[r]) * share + kSharedColumns - 1) / kSharedColumns : 0;
    int upto = count;
#pragma unroll
    for (int step = 1; step < kWave; step <<= 1) {
      const int other = __shfl_up(upto, step, kWave);
      if (lane >= step) upto += other;
    }
    const unsigned long long here = __ballot(tile < upto);
    if (here != 0) {
      const int at = __ffsll(here) - 1;
      request = first + at;
      tile -= __shfl(upto - count, at, kWave);
    } else {
      tile -= __shfl(upto, kWave - 1, kWave);
    }
  }
  if (request < 0) return;
  request = __builtin_amdgcn_readfirstlane(request);             // (the same in every lane: what follows is scalar)
  tile = __builtin_amdgcn_readfirstlane(tile);
  const int token0 = a.q_start[request], tokens = a.q_start[request + 1] - token0, history = a.seq_lens[request] - tokens;
  const int rows = tokens * share, row0 = tile * kSharedColumns, row_end = min(row0 + kSharedColumns, rows);
  const auto low_of = [&](int pos) {
    int low = a.window > 0 ? max(0, pos - a.window + 1) : 0;
    if (a.chunk > 0) low = max(low, pos / a.chunk * a.chunk);
    return low;
  };
  const int my_row = min(row0 + wave * 16 + col, rows - 1);      // (columns beyond the request's repeat its last, unstored)
  const int token = token0 + my_row / share, vector = (kvh * share + my_row % share) * a.maps + map;
  const int pos = history + my_row / share, low = low_of(pos);
  // what the block's and the wave's columns see: positions first .. last
  const int block_first = history + row0 / share, block_last = history + (row_end - 1) / share;
  const int block_low = low_of(block_first), block_low_last = low_of(block_last);
  const int wave_first = history + min(row0 + wave * 16, rows - 1) / share, wave_last = history + min(row0 + wave * 16 + 15, rows - 1) / share;
  const int wave_low = low_of(wave_first);

  uint4 q[DT];
  const bf16_t* qp = a.q + (static_cast<long>(token) * a.q_heads + vector) * DIM + grp * 8;
#pragma unroll
  for (int d = 0; d < DT; ++d) q[d] = load_bf16x8(qp + d * 32);
  constexpr float kLog2e = 1.4426950408889634f;
  const float scale = SHAPED ? a.scale : a.scale * kLog2e;
  const float cap = SHAPED ? a.softcap : 0.f, inverse_cap = SHAPED && a.softcap > 0.f ? 1.f / a.softcap : 0.f;
  const float bias_size = SHAPED && a.distance_bias != nullptr ? a.distance_bias[vector] : 0.f;
  const float bias_rate = SHAPED && a.distance_bias != nullptr ? a.distance_bias[a.q_heads + vector] : 0.f;
  float m = !a.sink ? -INFINITY : a.sink_logits != nullptr ? a.sink_logits[vector] * kLog2e : 0.f;
  float l = a.sink && grp == 0 ? 1.f : 0.f;                      // (a lane's own keys; added over the groups at the end)
  float4_t o[VT];
#pragma unroll
  for (int v = 0; v < VT; ++v) o[v] = float4_t{0.f, 0.f, 0.f, 0.f};

  // steps of 32 keys: those of the request's first `keep_first` that lie before the window's, then the window's
  const int first_step = block_low >> 5, kept_steps = min((a.keep_first + 31) >> 5, first_step);
  const int steps = kept_steps + (block_last >> 5) - first_step + 1;
  const auto key_of = [&](int turn) { return (turn < kept_steps ? turn : first_step + turn - kept_steps) << 5; };
  const int* table = a.block_table + static_cast<long>(a.table_rows != nullptr ? a.table_rows[request] : request) * a.table_width;
  const auto known = [&](int page) -> bool { return (page >= 0) & (page < a.num_pages); };
  // Where the step to fetch next lies: the table entry and the place in the page of each of its two sixteens (a page holds a
  // multiple of sixteen).  It moves on with additions: a division a step and sixteen cost more than the step's products.
  int entry[2], place[2], pages[2];
  const int last_entry = block_last / a.page_size;
  const auto stand_at = [&](int key) {
    entry[0] = key / a.page_size;
    place[0] = key - entry[0] * a.page_size;
  };
  const auto ask_pages = [&]() {
    entry[1] = entry[0];
    place[1] = place[0] + 16;
    if (place[1] >= a.page_size) {
      place[1] -= a.page_size;
      ++entry[1];
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) pages[half] = table[min(entry[half], last_entry)];    // (beyond the last: the last)
  };
  // what a step's keys and values come through: two sets in turn, asked for two steps ahead; their pages three steps ahead
  struct Ahead {
    uint4 keys[kKeyLoads], values[kValueLoads];
    bool there[2];
  } even, odd;
  // thread t fetches 16 bytes of key t / (DIM / 8) and, for values, keys 8 (t & 3) .. + 7 of dimension t / 4, and so on;
  // then the pages of the step after are asked for
  const auto fetch = [&](int turn, Ahead& to) {
    const bf16_t* key_half[2];
    const bf16_t* value_half[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      to.there[half] = known(pages[half]);
      const long head = (to.there[half] ? pages[half] : 0) * static_cast<long>(a.kv_heads) + kvh;
      key_half[half] = a.k_pages + ((head * a.page_size + place[half]) * a.maps + map) * DIM;
      value_half[half] = a.v_pages + head * VDIM * a.page_size + place[half];
    }
#pragma unroll
    for (int i = 0; i < kKeyLoads; ++i) {
      const int at = min(i * 256 + static_cast<int>(threadIdx.x), 32 * DIM / 8 - 1), key = at / (DIM / 8);
      to.keys[i] = load_bf16x8((key < 16 ? key_half[0] : key_half[1]) + (key & 15) * a.maps * DIM + at % (DIM / 8) * 8);
    }
#pragma unroll
    for (int i = 0; i < kValueLoads; ++i) {
      const int at = min(i * 256 + static_cast<int>(threadIdx.x), VDIM * 4 - 1), eight = at & 3;
      to.values[i] = load_bf16x8((eight < 2 ? value_half[0] : value_half[1]) + at / 4 * a.page_size + 8 * (eight & 1));
    }
    if (turn + 1 == kept_steps) {
      stand_at(first_step << 5);
    } else {
      place[0] += 32;
      while (place[0] >= a.page_size) {
        place[0] -= a.page_size;
        ++entry[0];
      }
    }
    ask_pages();
  };
  stand_at(key_of(0));
  ask_pages();
  const auto work = [&](int turn, Ahead& from, int buffer) {
    bf16_t *keys = filed_keys[buffer], *values = filed_values[buffer];
    const int j0 = key_of(turn);
    const bool here0 = from.there[0], here1 = from.there[1];
#pragma unroll
    for (int i = 0; i < kKeyLoads; ++i) {
      const int at = i * 256 + threadIdx.x;
      if (32 * DIM / 8 % 256 == 0 || at < 32 * DIM / 8)
        *reinterpret_cast<uint4*>(keys + at / (DIM / 8) * kKeyRow + at % (DIM / 8) * 8) = from.keys[i];
    }
    // (the same for the whole block: some column does not see some key of the step)
    const bool partly = j0 + 31 > block_first || (j0 < block_low_last && j0 + 31 >= a.keep_first) || !here0 || !here1;
    if (partly) {
      // slots that nobody has written, or of a page that is not the request's, hold anything: zeros - and zeros for what is not
      // finite (an exponent of all ones), which is said to the waves
      bool finite = true;
#pragma unroll
      for (int i = 0; i < kValueLoads; ++i) {
        const int eight = (i * 256 + static_cast<int>(threadIdx.x)) & 3;
        const int left = (eight < 2 ? here0 : here1) ? block_last - (j0 + 8 * eight) + 1 : 0;
        uint32_t words[4] = {from.values[i].x, from.values[i].y, from.values[i].z, from.values[i].w};
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          words[w] &= (2 * w < left ? 0xffffu : 0u) | (2 * w + 1 < left ? 0xffff0000u : 0u);
          const uint32_t kept = ((words[w] & 0x7f80u) != 0x7f80u ? 0xffffu : 0u) |
                                ((words[w] & 0x7f800000u) != 0x7f800000u ? 0xffff0000u : 0u);
          finite = finite & (kept == 0xffffffffu);
          words[w] &= kept;
        }
        from.values[i] = make_uint4(words[0], words[1], words[2], words[3]);
      }
      const bool any = __any(!finite);
      if (lane == 0) filed_infinite[buffer][wave] = any;
    }
#pragma unroll
    for (int i = 0; i < kValueLoads; ++i) {
      const int at = i * 256 + threadIdx.x, eight = at & 3;
      const uint4 v = from.values[i];
      if (VDIM * 4 % 256 == 0 || at < VDIM * 4) {
        // keys 8 eight .. + 3 are group 2 (eight & 1)'s of sixteen number eight / 2, the next four the group after's
        bf16_t* to = values + at / 4 * kValueRow + (eight & 1) * 16 + (eight >> 1) * 4;
        *reinterpret_cast<uint2*>(to) = make_uint2(v.x, v.y);
        *reinterpret_cast<uint2*>(to + 8) = make_uint2(v.z, v.w);
      }
    }
    __syncthreads();
    fetch(turn + 2, from);
    // (the same for the whole wave: none of its columns sees a key of the step)
    if (j0 > wave_last || (j0 + 31 < wave_low && j0 >= a.keep_first)) return;
    float4_t acc[2] = {float4_t{0.f, 0.f, 0.f, 0.f}, float4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int half = 0; half < 2; ++half)
        acc[half] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8_t, load_bf16x8(keys + (16 * half + col) * kKeyRow + d * 32 + grp * 8)),
            __builtin_bit_cast(bf16x8_t, q[d]), acc[half], 0, 0, 0);
    float s[8], top = -INFINITY;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      s[e] = acc[e >> 2][e & 3] * scale;
      if constexpr (SHAPED) {
        if (cap > 0.f) {      // tanh(x) = 1 - 2 / (exp(2 x) + 1), with the hardware's exponential and reciprocal
          const float x = __expf(2.f * fabsf(s[e]) * inverse_cap);
          s[e] = copysignf(cap * (1.f - 2.f * __frcp_rn(x + 1.f)), s[e]);
        }
        s[e] *= kLog2e;
        if (a.distance_bias != nullptr) {        // (keys behind the query are masked below: their logarithm is taken of 1)
          const int j = j0 + 16 * (e >> 2) + 4 * grp + (e & 3);
          s[e] -= bias_size * __builtin_amdgcn_logf(fmaf(bias_rate, static_cast<float>(max(pos - j, 0)), 1.f));
        }
      }
    }
    const auto sees = [&](int j, bool here) -> bool { return ((j >= low) | (j < a.keep_first)) & (j <= pos) & here; };
    int infinite = 0;
    if (partly) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        s[e] = sees(j0 + 16 * (e >> 2) + 4 * grp + (e & 3), e < 4 ? here0 : here1) ? s[e] : -INFINITY;
      infinite = __builtin_amdgcn_readfirstlane(*reinterpret_cast<const int*>(filed_infinite[buffer]));
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) top = fmaxf(top, s[e]);
    top = max_over_groups(top);
    if (__any(top > m + kTrail) || infinite != 0) {
      const float moved = fmaxf(m, top), shift = moved == -INFINITY ? 0.f : moved;
      const float correction = __builtin_amdgcn_exp2f(m - shift);
      l *= correction;
#pragma unroll
      for (int v = 0; v < VT; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[v][i] *= correction;
      m = moved;
      if (infinite != 0) {       // the values that were filed as zeros
#pragma unroll 1
        for (int one = 0; one < 32; ++one) {
          const int j = j0 + one, page = table[min(j / a.page_size, last_entry)];
          float own = s[0];      // the key's score lies in element 4 (one / 16) + one % 4 of group one / 4 % 4
#pragma unroll
          for (int e = 1; e < 8; ++e) own = e == (one >> 4) * 4 + (one & 3) ? s[e] : own;
          const float weight = __builtin_amdgcn_exp2f(__shfl(own, (one & 12) * 4 + col, kWave) - shift);
          if (!sees(j, known(page))) continue;
          const bf16_t* at = a.v_pages + ((page * static_cast<long>(a.kv_heads) + kvh) * VDIM + grp * 4) * a.page_size + j % a.page_size;
#pragma unroll
          for (int v = 0; v < VT; ++v)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float value = to_float(at[static_cast<long>(16 * v + i) * a.page_size]);
              if (!(fabsf(value) < INFINITY)) o[v][i] = fmaf(weight, value, o[v][i]);
              __builtin_amdgcn_sched_barrier(0); // (else all loads are asked for first: a third more registers in the kernel)
            }
        }
      }
    }
    const float reference = m == -INFINITY ? 0.f : m;
    uint32_t high[4], rest[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float p0 = __builtin_amdgcn_exp2f(s[2 * w] - reference), p1 = __builtin_amdgcn_exp2f(s[2 * w + 1] - reference);
      l += p0 + p1;
      high[w] = bf16_pair(p0, p1);
      rest[w] = bf16_pair(p0 - __uint_as_float(high[w] << 16), p1 - __uint_as_float(high[w] & 0xffff0000u));
    }
    const bf16x8_t p_high = __builtin_bit_cast(bf16x8_t, make_uint4(high[0], high[1], high[2], high[3]));
    const bf16x8_t p_rest = __builtin_bit_cast(bf16x8_t, make_uint4(rest[0], rest[1], rest[2], rest[3]));
#pragma unroll
    for (int v = 0; v < VT; ++v) {
      const bf16x8_t operand = __builtin_bit_cast(bf16x8_t, load_bf16x8(values + (16 * v + col) * kValueRow + grp * 8));
      o[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(operand, p_high, o[v], 0, 0, 0);
      o[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(operand, p_rest, o[v], 0, 0, 0);
    }
  };
  fetch(0, even);
  fetch(1, odd);
  for (int turn = 0; turn < steps; turn += 2) {
    work(turn, even, 0);
    if (turn + 1 < steps) work(turn + 1, odd, 1);
  }
  l += __shfl_xor(l, 16, kWave);
  l += __shfl_xor(l, 32, kWave);
  if (row0 + wave * 16 + col >= rows) return;
  float gate = a.out_scale;
  if (a.gates != nullptr) gate = a.out_scale / (1.f + expf(-to_float(a.gates[static_cast<long>(token) * a.gate_stride + a.gate_at + vector])));
  const float factor = gate / l;
  bf16_t* to = a.out + static_cast<long>(token) * a.out_stride + static_cast<long>(vector) * VDIM + grp * 4;
#pragma unroll
  for (int v = 0; v < VT; ++v) {
    uint2 packed;
    packed.x = bf16_pair(o[v][0] * factor, o[v][1] * factor);
    packed.y = bf16_pair(o[v][2] * factor, o[v][3] * factor);
    *reinterpret_cast<uint2*>(to + v * 16) = packed;
  }
}

}  // namespace

extern "C" int akv_gated_attention_shared(const void* q, const void* k_pages, const void* v_pages, const void* gates,
                                          long gate_stride, int gate_at, const int* q_start, const int* seq_lens,
                                          const int* block_table, const int* table_rows, int table_width, void* out, int first_seq,
                                          int seqs, int tiles, int q_heads, int kv_heads, int dim, int vdim, int page_size,
                                          long num_pages, float scale, float softcap, int chunk, int window, int sink,
                                          long out_stride, float out_scale, const float* sink_logits, int maps, int keep_first,
                                          const float* distance_bias, hipStream_t stream) {
  if (seqs <= first_seq || tiles <= 0) return 0;
  if (page_size % 16 != 0 || maps < 1 || kv_heads <= 0 || q_heads % (kv_heads * maps) != 0) return -2;
  if (!aligned_for_tiles(q, k_pages, v_pages, out, out_stride)) return -2;
  const long blocks = static_cast<long>(tiles) * kv_heads * maps;
  if (blocks > 0x7fffffffL) return -2;
  const SharedArgs a{static_cast<const bf16_t*>(q), static_cast<const bf16_t*>(k_pages), static_cast<const bf16_t*>(v_pages),
                     static_cast<const bf16_t*>(gates), q_start, seq_lens, block_table, table_rows, sink_logits, distance_bias,
                     static_cast<bf16_t*>(out), gate_stride, num_pages, out_stride, scale, softcap, out_scale, first_seq, seqs,
                     tiles, gate_at, table_width, q_heads, kv_heads, page_size, chunk, window, sink, maps, keep_first};
#define AKV_SHARED(DT, VT)                                                                                                  \
  if (softcap > 0.f || distance_bias != nullptr)                                                                            \
    gated_attention_shared_kernel<DT, VT, true><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(a);                      \
  else                                                                                                                      \
    gated_attention_shared_kernel<DT, VT, false><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(a)
#define AKV_SHARED_V(DT)                  \
  switch (vdim) {                         \
    case 32: AKV_SHARED(DT, 2); break;    \
    case 64: AKV_SHARED(DT, 4); break;    \
    case 128: AKV_SHARED(DT, 8); break;   \
    default: return -2;                   \
  }
  switch (dim) {
    case 32: AKV_SHARED_V(1); break;
    case 64: AKV_SHARED_V(2); break;
    case 128: AKV_SHARED_V(4); break;
    default: return -2;
  }
#undef AKV_SHARED_V
#undef AKV_SHARED
  return AKV_LAUNCH_STATUS();
}
