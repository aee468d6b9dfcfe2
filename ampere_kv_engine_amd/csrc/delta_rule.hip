// The gated delta rule, its decay per key channel or per head.  Per request and head, token after token, with S [dim, vdim]:
//     S <- g * S (row d times g_d, or all of it times g_h);  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
// where q and k are unit vectors per head (q also times dim^(-1/2)), beta = sigmoid(.), g = exp(-rate_h softplus(. + bias)).
// Everything after the projections and the short convolutions is float32: the unit norms, sigmoid, softplus, the
// exponentials, the state and its sums, the norm of the outputs.
//
// Three kernels.  `delta_prepare` is token-wise: the unit vectors, decays, betas and k . q of every token, float32, into a
// workspace.  The walk over a request's tokens is state_walk.h's with the rule kDelta.  (For the requests that bring many
// tokens two others stand in the place of these: below.)
// `state_finish_kernel` is token-wise again: o / rms(o) times a weight per value channel and a gate.

#include <type_traits>

#include "api_parts.h"
#include "state_walk.h"

using namespace akv;

namespace {

// A wave is a token's unit of work: units 0 .. groups - 1 are a q / k pair (sums of squares and the product from one pass
// over the raw vectors: k . q of the unit vectors follows without reading them back; the scalars of the pair's heads go
// along), every further unit 256 decays of channels.  conv rows: [q (groups x dim) | k (groups x dim) | v ...] after
// convolution and activation; beta_logits at `beta_stride` per token; decay logits (TD) at `decay_stride` per token.
template <typename T, typename TD, bool HEAD_DECAY>
__global__ __launch_bounds__(256) void delta_prepare_kernel(const T* __restrict__ conv, long conv_stride,
                                                            const T* __restrict__ beta_logits, long beta_stride,
                                                            const TD* __restrict__ decay_logits, long decay_stride,
                                                            const float* __restrict__ decay_bias,
                                                            const float* __restrict__ rate, float unit_eps, float q_scale,
                                                            float* __restrict__ prepared, int heads, int groups, int dim) {
  const long n = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1);
  const int unit = blockIdx.y * (blockDim.x / kWave) + threadIdx.x / kWave;
  const long width = prepared_width(heads, groups, dim, HEAD_DECAY);
  float* row = prepared + n * width;
  float* g = row + 2L * groups * dim;
  float* beta = row + prepared_scalars_at(heads, groups, dim, HEAD_DECAY);
  const TD* logits = decay_logits + n * decay_stride;
  const int share = heads / groups;
  if (unit < groups) {
    const T* qs = conv + n * conv_stride + static_cast<long>(unit) * dim;
    const T* ks = qs + static_cast<long>(groups) * dim;
    float qq = 0.f, kk = 0.f, qk = 0.f;
    for (int i = lane; i < dim; i += kWave) {
      const float a = to_float(qs[i]), b = to_float(ks[i]);
      qq = fmaf(a, a, qq), kk = fmaf(b, b, kk), qk = fmaf(a, b, qk);
    }
    const float q_unit = q_scale / sqrtf(wave_sum(qq) + unit_eps), k_unit = 1.f / sqrtf(wave_sum(kk) + unit_eps);
    const float dot = wave_sum(qk) * q_unit * k_unit;
    for (int i = lane; i < dim; i += kWave) {
      row[static_cast<long>(unit) * dim + i] = to_float(qs[i]) * q_unit;
      row[static_cast<long>(groups + unit) * dim + i] = to_float(ks[i]) * k_unit;
    }
    for (int j = lane; j < share; j += kWave) {
      const int h = unit * share + j;
      beta[h] = sigmoid_of(to_float(beta_logits[n * beta_stride + h]));
      beta[heads + h] = dot;
      if constexpr (HEAD_DECAY) beta[2 * heads + h] = expf(-rate[h] * softplus_of(to_float(logits[h]) + decay_bias[h]));
    }
    return;
  }
  if constexpr (!HEAD_DECAY) {
    const int first = (unit - groups) * 256;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = first + e * kWave + lane;
      if (i < heads * dim) g[i] = expf(-rate[i / dim] * softplus_of(to_float(logits[i]) + decay_bias[i]));
    }
  }
}

// The same for vectors of 4 L elements, L a power of two up to 64: L lanes take a q / k pair, four elements of each a lane, and
// behind the pairs (from a multiple of a wave on) a lane takes four decays.  Memory and the exponentials bound it: 2,000 tokens
// of 16 heads of 128 with decays per channel, 82 MB: 24.4 us, 33.5 with single elements; 8 tokens 4.2 and 5.1.
template <typename T, typename TD, bool HEAD_DECAY>
__global__ __launch_bounds__(256) void delta_prepare_fours_kernel(const T* __restrict__ conv, long conv_stride,
                                                                  const T* __restrict__ beta_logits, long beta_stride,
                                                                  const TD* __restrict__ decay_logits, long decay_stride,
                                                                  const float* __restrict__ decay_bias,
                                                                  const float* __restrict__ rate, float unit_eps, float q_scale,
                                                                  float* __restrict__ prepared, int heads, int groups, int dim) {
  const long n = blockIdx.x;
  const int lanes = dim / 4, pairs = groups * lanes, at = blockIdx.y * 256 + threadIdx.x;
  const long width = prepared_width(heads, groups, dim, HEAD_DECAY);
  float* row = prepared + n * width;
  float* beta = row + prepared_scalars_at(heads, groups, dim, HEAD_DECAY);
  const TD* logits = decay_logits + n * decay_stride;
  if (at < pairs) {                                        // (a pair's lanes come together)
    const T* from = conv + n * conv_stride + at * 4;
    const float4 q = four_of(from), k = four_of(from + static_cast<long>(groups) * dim);
    const float qq = lanes_sum(four_squares(q), lanes), kk = lanes_sum(four_squares(k), lanes);
    const float q_unit = q_scale / sqrtf(qq + unit_eps), k_unit = 1.f / sqrtf(kk + unit_eps);
    const float dot = lanes_sum(fmaf(q.z, k.z, q.x * k.x) + fmaf(q.w, k.w, q.y * k.y), lanes) * q_unit * k_unit;
    put_four(row + at * 4, make_float4(q.x * q_unit, q.y * q_unit, q.z * q_unit, q.w * q_unit));
    put_four(row + static_cast<long>(groups) * dim + at * 4, make_float4(k.x * k_unit, k.y * k_unit, k.z * k_unit, k.w * k_unit));
    const int unit = at / lanes, share = heads / groups;
    for (int j = at % lanes; j < share; j += lanes) {
      const int h = unit * share + j;
      beta[h] = sigmoid_of(to_float(beta_logits[n * beta_stride + h]));
      beta[heads + h] = dot;
      if constexpr (HEAD_DECAY) beta[2 * heads + h] = expf(-rate[h] * softplus_of(to_float(logits[h]) + decay_bias[h]));
    }
    return;
  }
  if constexpr (!HEAD_DECAY) {
    const int i = (at - (pairs + kWave - 1) / kWave * kWave) * 4;
    if (i < 0 || i >= heads * dim) return;
    const float4 z = four_of(logits + i), bias = four_of(decay_bias + i);
    const float fall = -rate[i / dim];
    put_four(row + 2L * groups * dim + i, make_float4(expf(fall * softplus_of(z.x + bias.x)), expf(fall * softplus_of(z.y + bias.y)),
                                                      expf(fall * softplus_of(z.z + bias.z)), expf(fall * softplus_of(z.w + bias.w))));
  }
}

// ---- many tokens of a request: the walk in chunks of 16 tokens on the matrix cores ------------------------------------------
// The chunkwise form of Yang et al., "Parallelizing Linear Transformers with the Delta Rule over Sequence Length" (2024).
// Over a chunk the recurrence is a linear system.  With S0 the state before it, cum_t the product of the decays of its tokens
// up to t and fall_st that of the decays behind token s up to t (all products of decays forward in time: nothing is divided,
// and what underflows is what has decayed away):
//     A_ts = k_s . (fall_st k_t), s < t;   B_ts = k_s . (fall_st q_t), s <= t
//     U = T (V - (cum k) S0),  T = (1 + diag(beta) A)^-1 diag(beta)          the u of every token
//     O = (cum q) S0 + B U;    S <- cum_15 S0 + sum_t fall_t,15 k_t u_t
// Everything but S0 is known for all chunks beforehand: `delta_chunks_kernel` makes cum k, cum q, the last chunk's decay, the
// k that enter the next state, T and B of every (chunk, head) in parallel - T's rows by substitution, as the walk would have
// -, and `delta_chunk_walk_kernel` is left with four products on the float32 matrix instruction per chunk, a chain of
// 16 tokens at a time.  All of it is float32.
// Chunks count from a request's first token of the step; chunk c of request r has slot q_start[r] / 16 + r + c of the
// workspace, which no other request's chunks reach.
// Bound by the chain: per chunk (dim 128) 20 matrix instructions of 32 cycles that wait for each other, an exchange of sums
// through LDS (160 ns alone) and their way between registers; 0.92 us as measured.  One request of 16 heads of 128 x 128, whole
// rule (prepare, walk, finish), token by token / in chunks: decays per channel 171 tokens 35.5 / 29.4 us, 512 78.8 / 55.8, 2,000 257 /
// 154; a decay per head 32.3 / 26.7, 70.0 / 52.9, 229 / 146.  Against 64 bits both are 2e-7 off (relative, outputs and states, 64
// to 2,000 tokens).  With the outputs in the chain's own waves the walk of 2,000 tokens took 149 us, with them beside it 116.
constexpr int kChunk = 16;
typedef __attribute__((ext_vector_type(4))) float floatx4;

inline long chunk_slots(int tokens, int seqs) { return tokens / kChunk + static_cast<long>(seqs) + 1; }
// [cum k | cum q | k for the next state] in the order the matrix instruction's lanes read them, [cum_15], [T], [B]
__host__ __device__ inline long chunk_floats(int dim) { return 3L * kChunk * dim + dim + 2L * kChunk * kChunk; }
// The fewest tokens of a request that goes in chunks.  Which form a request takes hangs on its own tokens and the head's size
// alone, so that its bits do not change with what else is in the step (fewer than kTilesFrom walk in small tiles, others in
// large ones: a step of all three kinds has three launches).  32 single tokens beside 171, 16 heads of 128 x 128: 60 us, where
// the single ones went in chunks too 113, where all walked in large tiles 162.  Of 64 and 128 the lines lie where one request
// alone breaks even (batches would from fewer on), of 192 and 256, whose large tiles take most of a unit's LDS, at the large
// tiles' own: a request alone loses a little there and several gain much.  Whole rule, walk / chunks us, decays per channel: 16
// heads of 64 x 64 64 tokens 14.9 / 15.5, 80 18.1 / 16.1; 16 of 128 x 128 96 tokens 21.6 / 24.2, 128 25.8 / 25.9, 160 30.4 / 28.4
// (four requests of 80 43.0 / 36.6; a decay per head 96 21.2 / 21.5, 128 25.0 / 23.5); 8 of 256 x 256 24 tokens 21.3 / 27.2, 48
// 32.2 / 29.6, four requests of 24 60.7 / 35.6; 6 of 192 x 192 24 tokens 22.1 / 23.9, four requests 41.9 / 29.8.
__host__ __device__ inline int chunks_from(int dim) {
  return dim == 64 ? 65 : dim == 128 ? 128 : dim == 192 || dim == 256 ? kTilesFrom : 0x7fffffff;
}

// Products over the 16 lanes of a row: of lanes up to this one (SHR), of this one and those behind it (SHL).
template <int CTRL> __device__ __forceinline__ float times_lane(float v) {
  return v * __int_as_float(__builtin_amdgcn_update_dpp(0x3f800000, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float product_upto(float v) { return times_lane<0x118>(times_lane<0x114>(times_lane<0x112>(times_lane<0x111>(v)))); }
__device__ __forceinline__ float product_from(float v) { return times_lane<0x108>(times_lane<0x104>(times_lane<0x102>(times_lane<0x101>(v)))); }

// A block is a chunk of one request and a head.  TILES: dim / 64.
template <typename T, typename TD, bool HEAD_DECAY, int TILES>
__global__ __launch_bounds__(256) void delta_chunks_kernel(const T* __restrict__ conv, long conv_stride,
                                                           const T* __restrict__ beta_logits, long beta_stride,
                                                           const TD* __restrict__ decay_logits, long decay_stride,
                                                           const float* __restrict__ decay_bias, const float* __restrict__ rate,
                                                           float unit_eps, float q_scale, const int* __restrict__ q_start,
                                                           int seqs, float* __restrict__ chunks, int heads, int groups) {
  constexpr int dim = 64 * TILES, kRow = dim + 4, kPair = 20;
  __shared__ __align__(16) float k_of[kChunk * kRow], q_of[kChunk * kRow], g_of[kChunk * kRow];
  __shared__ __align__(16) float a_of[kChunk * kPair], b_of[kChunk * kPair], t_of[kChunk * kPair], beta[kChunk];
  const int slot = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int r = 0;
  for (int low = 1, high = seqs - 1; low <= high;) {       // the last request whose first slot is not beyond this one
    const int middle = (low + high) / 2;
    if (q_start[middle] / kChunk + middle <= slot) r = middle, low = middle + 1;
    else high = middle - 1;
  }
  const int t0 = q_start[r] + (slot - (q_start[r] / kChunk + r)) * kChunk, count = min(kChunk, q_start[r + 1] - t0);
  if (count <= 0 || q_start[r + 1] - q_start[r] < chunks_from(dim)) return;   // (the same in every thread)
  float* to = chunks + (static_cast<long>(slot) * heads + h) * chunk_floats(dim);

  // unit vectors and decays, thread (token, 16 parts of four elements 64 apart); a token that does not exist changes nothing
  {
    const int t = tid >> 4, part = tid & 15, share = heads / groups;
    const long n = t0 + min(t, count - 1);
    const bool there = t < count;
    const T* qs = conv + n * conv_stride + static_cast<long>(h / share) * dim + part * 4;
    const T* ks = qs + static_cast<long>(groups) * dim;
    float4 q[TILES], k[TILES];
    float qq = 0.f, kk = 0.f;
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      q[j] = four_of(qs + j * 64), k[j] = four_of(ks + j * 64);
      qq += four_squares(q[j]), kk += four_squares(k[j]);
    }
    const float q_unit = there ? q_scale / sqrtf(column_sum<16>(qq) + unit_eps) : 0.f;
    const float k_unit = there ? 1.f / sqrtf(column_sum<16>(kk) + unit_eps) : 0.f;
    const float fall = -rate[h];
    float head_decay = 1.f;
    if (HEAD_DECAY && there) head_decay = expf(fall * softplus_of(to_float(decay_logits[n * decay_stride + h]) + decay_bias[h]));
    const auto kept = [&](float v, float unit) { return there ? v * unit : 0.f; };
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const int at = t * kRow + part * 4 + j * 64;
      put_four(q_of + at, make_float4(kept(q[j].x, q_unit), kept(q[j].y, q_unit), kept(q[j].z, q_unit), kept(q[j].w, q_unit)));
      put_four(k_of + at, make_float4(kept(k[j].x, k_unit), kept(k[j].y, k_unit), kept(k[j].z, k_unit), kept(k[j].w, k_unit)));
      float4 g = make_float4(head_decay, head_decay, head_decay, head_decay);
      if constexpr (!HEAD_DECAY) {
        const long i = static_cast<long>(h) * dim + part * 4 + j * 64;
        const float4 z = four_of(decay_logits + n * decay_stride + i), bias = four_of(decay_bias + i);
        const auto decay = [&](float v, float b) { return there ? expf(fall * softplus_of(v + b)) : 1.f; };
        g = make_float4(decay(z.x, bias.x), decay(z.y, bias.y), decay(z.z, bias.z), decay(z.w, bias.w));
      }
      put_four(g_of + at, g);
    }
    if (part == 0) beta[t] = there ? sigmoid_of(to_float(beta_logits[n * beta_stride + h])) : 0.f;
  }
  __syncthreads();

  // the decayed vectors: a lane is (token lane % 16, four elements of a tile of 16), a row of lanes multiplies along the tokens
  {
    const int t = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const int tile = wave + j * 4, at = t * kRow + tile * 16 + g * 4;
      const float4 q = four_of(q_of + at), k = four_of(k_of + at), d = four_of(g_of + at);
      const float decays[4] = {d.x, d.y, d.z, d.w}, keys[4] = {k.x, k.y, k.z, k.w};
      float upto[4], next[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        upto[e] = product_upto(decays[e]);
        const float behind = __int_as_float(__builtin_amdgcn_update_dpp(0x3f800000, __float_as_int(decays[e]), 0x101, 0xF, 0xF, false));
        next[e] = keys[e] * product_from(behind);
      }
      put_four(to + (tile * 64 + lane) * 4, make_float4(k.x * upto[0], k.y * upto[1], k.z * upto[2], k.w * upto[3]));
      put_four(to + kChunk * dim + (tile * 64 + lane) * 4, make_float4(q.x * upto[0], q.y * upto[1], q.z * upto[2], q.w * upto[3]));
      // (the next state's product runs over tokens: lane d % 16 + 16 (t / 4), element t % 4)
#pragma unroll
      for (int e = 0; e < 4; ++e) to[2 * kChunk * dim + (tile * 64 + (t >> 2) * 16 + g * 4 + e) * 4 + (t & 3)] = next[e];
      if (t == kChunk - 1) put_four(to + 3 * kChunk * dim + tile * 16 + g * 4, make_float4(upto[0], upto[1], upto[2], upto[3]));
    }
  }

  // A and B: thread (token s, 16 parts); its k_s decays token by token while it meets the later tokens
  {
    const int s = tid >> 4, part = tid & 15;
    float4 k[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j) k[j] = four_of(k_of + s * kRow + part * 4 + j * 64);
    float a_mine = 0.f, b_mine = 0.f;
#pragma unroll
    for (int t = 0; t < kChunk; ++t) {
      float a = 0.f, b = 0.f;
#pragma unroll
      for (int j = 0; j < TILES; ++j) {
        const int at = t * kRow + part * 4 + j * 64;
        const float4 kt = four_of(k_of + at), qt = four_of(q_of + at), d = four_of(g_of + at);
        const bool later = t > s;
        k[j] = make_float4(later ? k[j].x * d.x : k[j].x, later ? k[j].y * d.y : k[j].y, later ? k[j].z * d.z : k[j].z,
                           later ? k[j].w * d.w : k[j].w);
        a += fmaf(k[j].z, kt.z, k[j].x * kt.x) + fmaf(k[j].w, kt.w, k[j].y * kt.y);
        b += fmaf(k[j].z, qt.z, k[j].x * qt.x) + fmaf(k[j].w, qt.w, k[j].y * qt.y);
      }
      a = column_sum<16>(a), b = column_sum<16>(b);
      if (part == t) a_mine = t > s ? a : 0.f, b_mine = t >= s ? b : 0.f;
    }
    a_of[part * kPair + s] = a_mine, b_of[part * kPair + s] = b_mine;
  }
  __syncthreads();
  if (tid < kChunk) {                                      // column tid of T: (1 + diag(beta) A) x = beta_tid e_tid
    float x[kChunk];
#pragma unroll
    for (int t = 0; t < kChunk; ++t) {
      float sum = 0.f;
#pragma unroll
      for (int s = 0; s < t; ++s) sum = fmaf(a_of[t * kPair + s], x[s], sum);
      x[t] = beta[t] * ((t == tid ? 1.f : 0.f) - sum);
      if (t < tid) x[t] = 0.f;
      t_of[t * kPair + tid] = x[t];
    }
  }
  __syncthreads();
  if (tid < 128) {
    const float* from = (tid < 64 ? t_of : b_of) + (lane & 15) * kPair + (lane >> 4) * 4;
    put_four(to + 3 * kChunk * dim + dim + tid * 4, four_of(from));
  }
}

// A block: one request, one head, 16 columns of S, eight waves.  Four are the chain: each holds dim / 4 rows of S as the matrix
// instruction's operand (lane: column lane % 16, rows 4 (lane / 16) .. + 3 of each tile of 16) and takes V - (cum k) S0 to U and
// S to the next chunk.  The other four stand beside them on the same vector units and make the outputs from the S0 and U that
// the chain leaves in LDS, one phase later: what is not on the way from one state to the next runs while the chain waits.
// There is one barrier a chunk.  Before barrier p the chain has left S0 and its parts of (cum k) S0 of chunk p, and U of chunk
// p - 1; the output waves have left their parts of the outputs of chunk p - 2.  Barriers wait for LDS alone: the operands of
// three chunks on their way from memory and the stores of finished outputs pass them.
// A column whose V - (cum k) S0 or u is not finite at some token gets NaN from that token on, and the tokens before keep what
// they have: the products would have spread it to them (0 times it).  (In S it spreads to the whole column, as it should.)
// (chunks and token_values are not __restrict__: with it the compiler moves a chunk's loads past the barriers to where they are
// used, three chunks later.)
template <typename T, int TILES>
__global__ __launch_bounds__(512) void delta_chunk_walk_kernel(const float* chunks, const T* token_values,
                                                               long value_stride, float* __restrict__ state, long state_stride,
                                                               const int* __restrict__ q_start, const int* __restrict__ seq_slots,
                                                               float* __restrict__ raw_out, int seqs, int heads, int vdim) {
  constexpr int dim = 64 * TILES;
  __shared__ __align__(16) float w_parts[2][4 * 256], o_parts[2][4 * 256], s_parts[2][4 * TILES * 256], u_whole[2][256], x_whole[2][256];
  const WalkUnit unit = walk_unit(seqs, heads, (vdim + 15) / 16);
  if (unit.request >= seqs) return;
  const int r = unit.request, h = unit.head, col0 = unit.column_block * 16;
  const int first = q_start[r], last = q_start[r + 1];
  if (last - first < chunks_from(dim)) return;             // (it walks)
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4;
  const bool chain = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) == 0;
  const int total = (last - first + kChunk - 1) / kChunk;
  // What a chunk reads lies at addresses that are the same for the whole wave, plus a constant offset of the lane: address
  // arithmetic per lane would be a good part of a wave's instructions.
  constexpr int kArray = kChunk * dim * 4;                 // bytes of one of a chunk's three arrays of vectors
  const long step = static_cast<long>(heads) * chunk_floats(dim) * 4;
  const char* base = reinterpret_cast<const char*>(chunks) + (static_cast<long>(first / kChunk + r) * heads + h) * chunk_floats(dim) * 4;
  const uint32_t lane16 = lane * 16u, g16 = g * 16u;
  auto product = [](float a, float b, floatx4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); };
  auto meet = []() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  const float nan = __uint_as_float(0x7fc00000u);

  if (chain) {
    const int col = min(col0 + (lane & 15), vdim - 1);
    float* kept = state + static_cast<long>(seq_slots[r]) * state_stride + (static_cast<long>(h) * vdim + col) * dim + wave * 16 * TILES + g * 4;
    floatx4 S[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j) S[j] = *reinterpret_cast<const floatx4*>(kept + j * 16);
    const char* value_rows = reinterpret_cast<const char*>(token_values + static_cast<long>(first) * value_stride + static_cast<long>(h) * vdim + col0);
    const uint32_t row_bytes = static_cast<uint32_t>(value_stride) * static_cast<uint32_t>(sizeof(T));
    const int left = last - first - (total - 1) * kChunk;  // tokens of the last chunk (rows behind them are not read; what
    uint32_t value_at[4], last_at[4];                      // stands for them meets columns of T that are zero)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t in_row = static_cast<uint32_t>(col - col0) * static_cast<uint32_t>(sizeof(T));
      value_at[i] = static_cast<uint32_t>(g * 4 + i) * row_bytes + in_row;
      last_at[i] = static_cast<uint32_t>(min(g * 4 + i, left - 1)) * row_bytes + in_row;
    }
    struct Operands {
      floatx4 kk[TILES], kd[TILES], fall[TILES], t;
      uint32_t v[4];                                       // (the values' bits)
    } held[3];
    typedef typename std::conditional<sizeof(T) == 2, uint16_t, uint32_t>::type Bits;
    auto fetch = [&](Operands& into, int chunk) {
      const int c = min(chunk, total - 1);                 // (beyond the last: read and not used)
      const char* from = base + c * step;
      const char* tiles = from + wave * (TILES * 1024);
      const char* rows = value_rows + static_cast<long>(c) * kChunk * row_bytes;
      const bool whole = c + 1 < total;
#pragma unroll
      for (int j = 0; j < TILES; ++j) into.kk[j] = *reinterpret_cast<const floatx4*>(tiles + j * 1024 + lane16);
#pragma unroll
      for (int i = 0; i < 4; ++i) into.v[i] = *reinterpret_cast<const Bits*>(rows + (whole ? value_at[i] : last_at[i]));
      into.t = *reinterpret_cast<const floatx4*>(from + 3 * kArray + dim * 4 + lane16);
#pragma unroll
      for (int j = 0; j < TILES; ++j) {
        into.fall[j] = *reinterpret_cast<const floatx4*>(from + 3 * kArray + (wave * TILES + j) * 64 + g16);
        into.kd[j] = *reinterpret_cast<const floatx4*>(tiles + 2 * kArray + j * 1024 + lane16);
      }
    };
    auto leave_state = [&](int chunk) {
#pragma unroll
      for (int j = 0; j < TILES; ++j) *reinterpret_cast<floatx4*>(&s_parts[chunk & 1][(wave * TILES + j) * 256 + lane * 4]) = S[j];
    };
    auto walk = [&](Operands& now, int chunk) {
      floatx4 w[TILES];
#pragma unroll
      for (int j = 0; j < TILES; ++j) w[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < TILES; ++j) w[j] = product(now.kk[j][i], S[j][i], w[j]);
      leave_state(chunk);
#pragma unroll
      for (int j = 0; j < TILES; ++j) S[j] *= now.fall[j];
#pragma unroll
      for (int j = 1; j < TILES; ++j) w[0] += w[j];
      *reinterpret_cast<floatx4*>(&w_parts[chunk & 1][wave * 256 + lane * 4]) = w[0];
      meet();
      const float* parts = w_parts[chunk & 1] + lane * 4;
      const floatx4 sum = ((*reinterpret_cast<const floatx4*>(parts) + *reinterpret_cast<const floatx4*>(parts + 256)) +
                           *reinterpret_cast<const floatx4*>(parts + 512)) + *reinterpret_cast<const floatx4*>(parts + 768);
      floatx4 x, u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = __uint_as_float(sizeof(T) == 2 ? now.v[i] << 16 : now.v[i]) - sum[i];
#pragma unroll
      for (int i = 0; i < 4; ++i) u = product(now.t[i], x[i], u);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < TILES; ++j) S[j] = product(now.kd[j][i], u[i], S[j]);
      // (the four waves hold the same u and x and write the same)
      *reinterpret_cast<floatx4*>(&u_whole[chunk & 1][lane * 4]) = u;
      *reinterpret_cast<floatx4*>(&x_whole[chunk & 1][lane * 4]) = x;
      fetch(now, chunk + 3);
    };
#pragma unroll
    for (int i = 0; i < 3; ++i) fetch(held[i], i);
    // (the first loads end here: see `settle`)
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      asm volatile("" : "+v"(S[j]));
#pragma unroll
      for (int i = 0; i < 3; ++i) asm volatile("" : "+v"(held[i].kk[j]), "+v"(held[i].kd[j]), "+v"(held[i].fall[j]));
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
      asm volatile("" : "+v"(held[i].t), "+v"(held[i].v[0]), "+v"(held[i].v[1]), "+v"(held[i].v[2]), "+v"(held[i].v[3]));
    int chunk = 0;
    for (; chunk + 3 <= total; chunk += 3) {               // (no test inside: the compiler counts the loads on their way)
      walk(held[0], chunk);
      walk(held[1], chunk + 1);
      walk(held[2], chunk + 2);
    }
    if (chunk < total) walk(held[0], chunk);
    if (chunk + 1 < total) walk(held[1], chunk + 1);
    meet();
    meet();
    if (col0 + (lane & 15) < vdim) {
#pragma unroll
      for (int j = 0; j < TILES; ++j) *reinterpret_cast<floatx4*>(kept + j * 16) = S[j];
    }
    return;
  }

  // ---- the outputs ----------------------------------------------------------------------------------------------------------
  struct Operands {
    floatx4 qq[TILES];
    float b;
  } held[3];
  auto fetch = [&](Operands& into, int chunk) {
    const char* from = base + min(chunk, total - 1) * step;
#pragma unroll
    for (int j = 0; j < TILES; ++j) into.qq[j] = *reinterpret_cast<const floatx4*>(from + kArray + (wave * TILES + j) * 1024 + lane16);
    into.b = *reinterpret_cast<const float*>(from + 3 * kArray + (dim + kChunk * kChunk + wave) * 4 + lane16);
  };
  // thread (token tid / 16, column tid % 16) stores: the four waves' parts in their order
  const int out_at = (((tid >> 4) >> 2) * 16 + (tid & 15)) * 4 + ((tid >> 4) & 3);
  const bool stores = col0 + (tid & 15) < vdim;
  char* out_rows = reinterpret_cast<char*>(raw_out + (static_cast<long>(first) * heads + h) * vdim + col0);
  const long out_step = static_cast<long>(kChunk) * heads * vdim * 4;
  const uint32_t out_lane = static_cast<uint32_t>((tid >> 4) * heads * vdim + (tid & 15)) * 4u;
  auto store_outputs = [&](int chunk) {
    const float* parts = o_parts[chunk & 1] + out_at;
    const float sum = ((parts[0] + parts[256]) + parts[512]) + parts[768];
    if (stores && (tid >> 4) < last - first - chunk * kChunk) *reinterpret_cast<float*>(out_rows + chunk * out_step + out_lane) = sum;
  };
  floatx4 out = {0.f, 0.f, 0.f, 0.f};                      // (cum q) S0 of the chunk before
  float b = 0.f;
  auto finish = [&](int chunk) {                           // + B U, the wave's quarter of the tokens
    // (step i of the product takes tokens 4 (lane / 16) + i: this wave is step `wave`)
    floatx4 u = *reinterpret_cast<const floatx4*>(&u_whole[chunk & 1][lane * 4]);
    const floatx4 before = out;
    out = product(b, u_whole[chunk & 1][lane * 4 + wave], before);
    const float whole = (u[0] - u[0]) + (u[1] - u[1]) + (u[2] - u[2]) + (u[3] - u[3]);   // 0, or not a number
    if (__any(whole != 0.f)) {
      const floatx4 x = *reinterpret_cast<const floatx4*>(&x_whole[chunk & 1][lane * 4]);
      const floatx4 t = *reinterpret_cast<const floatx4*>(base + chunk * step + 3 * kArray + dim * 4 + lane16);
      u = floatx4{0.f, 0.f, 0.f, 0.f};
      int from = kChunk;
#pragma unroll
      for (int i = 0; i < 4; ++i) u = product(t[i], x[i] - x[i] != 0.f ? 0.f : x[i], u);
#pragma unroll
      for (int i = 3; i >= 0; --i) from = x[i] - x[i] != 0.f || u[i] - u[i] != 0.f ? g * 4 + i : from;
      from = min(from, __shfl_xor(from, 16)), from = min(from, __shfl_xor(from, 32));
      float mine = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (wave == i && g * 4 + i < from) mine = u[i];
      const floatx4 again = product(b, mine, before);
#pragma unroll
      for (int i = 0; i < 4; ++i) out[i] = from == kChunk ? out[i] : g * 4 + i < from ? again[i] : nan;
    }
    *reinterpret_cast<floatx4*>(&o_parts[chunk & 1][wave * 256 + lane * 4]) = out;
  };
  auto follow = [&](Operands& now, int chunk) {
    meet();
    floatx4 next = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const floatx4 S = *reinterpret_cast<const floatx4*>(&s_parts[chunk & 1][(wave * TILES + j) * 256 + lane * 4]);
#pragma unroll
      for (int i = 0; i < 4; ++i) next = product(now.qq[j][i], S[i], next);
    }
    if (chunk > 0) finish(chunk - 1);
    if (chunk > 1) store_outputs(chunk - 2);
    out = next, b = now.b;
    fetch(now, chunk + 3);
  };
#pragma unroll
  for (int i = 0; i < 3; ++i) fetch(held[i], i);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    asm volatile("" : "+v"(held[i].b));
#pragma unroll
    for (int j = 0; j < TILES; ++j) asm volatile("" : "+v"(held[i].qq[j]));
  }
  int chunk = 0;
  for (; chunk + 3 <= total; chunk += 3) {               // (no test inside: the compiler counts the loads on their way)
    follow(held[0], chunk);
    follow(held[1], chunk + 1);
    follow(held[2], chunk + 2);
  }
  if (chunk < total) follow(held[0], chunk);
  if (chunk + 1 < total) follow(held[1], chunk + 1);
  meet();
  finish(total - 1);
  if (total > 1) store_outputs(total - 2);
  meet();
  store_outputs(total - 1);
}

template <typename T, typename TD, bool HEAD_DECAY, int TILES>
void launch_chunks(const T* conv, long conv_stride, const T* beta_logits, long beta_stride, const TD* decay_logits,
                   long decay_stride, const float* decay_bias, const float* rate, float unit_eps, float q_scale, float* state,
                   long state_stride, const int* q_start, const int* seq_slots, float* chunks, float* raw, int tokens, int seqs,
                   int heads, int groups, int vdim, hipStream_t stream) {
  delta_chunks_kernel<T, TD, HEAD_DECAY, TILES><<<dim3(static_cast<unsigned>(chunk_slots(tokens, seqs)), heads), 256, 0, stream>>>(
      conv, conv_stride, beta_logits, beta_stride, decay_logits, decay_stride, decay_bias, rate, unit_eps, q_scale, q_start, seqs,
      chunks, heads, groups);
  delta_chunk_walk_kernel<T, TILES><<<walk_grid(seqs, heads, (vdim + 15) / 16), 512, 0, stream>>>(
      chunks, conv + 2L * groups * 64 * TILES, conv_stride, state, state_stride, q_start, seq_slots, raw, seqs, heads, vdim);
}

// Unit vectors, decays, betas and k . q of the first `tokens` tokens.
template <typename T, typename TD, bool HEAD_DECAY>
void launch_prepare(const T* conv, long conv_stride, const T* beta_logits, long beta_stride, const TD* decay_logits, long decay_stride,
                    const float* decay_bias, const float* rate, float unit_eps, float q_scale, float* prepared, int tokens, int heads,
                    int groups, int dim, hipStream_t stream) {
  if (lanes_of_fours(dim) && conv_stride % 4 == 0 && in_fours(conv) && in_fours(prepared) &&
      (HEAD_DECAY || (decay_stride % 4 == 0 && in_fours(decay_logits) && in_fours(decay_bias)))) {
    const int pairs = (groups * dim / 4 + kWave - 1) / kWave * kWave, threads = pairs + (HEAD_DECAY ? 0 : heads * dim / 4);
    delta_prepare_fours_kernel<T, TD, HEAD_DECAY><<<dim3(tokens, (threads + 255) / 256), 256, 0, stream>>>(
        conv, conv_stride, beta_logits, beta_stride, decay_logits, decay_stride, decay_bias, rate, unit_eps, q_scale, prepared,
        heads, groups, dim);
  } else {
    const int units = groups + (HEAD_DECAY ? 0 : (heads * dim + 255) / 256);
    delta_prepare_kernel<T, TD, HEAD_DECAY><<<dim3(tokens, (units + 3) / 4), 256, 0, stream>>>(
        conv, conv_stride, beta_logits, beta_stride, decay_logits, decay_stride, decay_bias, rate, unit_eps, q_scale, prepared,
        heads, groups, dim);
  }
}

// The workspace: [chunks][rows of the tokens that walk][outputs], the first part only where some request goes in chunks.
struct Parts {
  long rows, raw, total;      // floats before the rows, before the outputs, in all
};
inline Parts parts_of(int tokens, int seqs, int heads, int groups, int dim, int vdim, bool head_decay, bool chunks, int walked_tokens) {
  Parts p;
  p.rows = chunks ? chunk_slots(tokens, seqs) * heads * chunk_floats(dim) : 0;
  p.raw = p.rows + (walked_tokens > 0 ? (static_cast<long>(walked_tokens) + kRowsBehind) * prepared_width(heads, groups, dim, head_decay) : 0);
  p.total = p.raw + (static_cast<long>(tokens) + kRowsBehind) * heads * vdim;
  return p;
}

template <typename T, typename TD, typename TG, bool HEAD_DECAY>
int delta_rule(const T* conv, long conv_stride, const T* beta_logits, long beta_stride, const TD* decay_logits,
               long decay_stride, const float* decay_bias, const float* rate, const TG* gates, long gate_stride, int gate_act,
               const float* norm_weight, float unit_eps, float norm_eps, float q_scale, float* state, long state_stride,
               const int* q_start, const int* seq_slots, float* workspace, T* out, int tokens, int seqs, int heads, int groups,
               int dim, int vdim, int longest, int walked_tokens, bool shorts, bool longer, hipStream_t stream) {
  const bool chunks = longest >= chunks_from(dim) && conv_stride % 4 == 0 && in_fours(conv) && in_fours(workspace) &&
                      state_stride % 4 == 0 && in_fours(state) &&
                      (HEAD_DECAY || (decay_stride % 4 == 0 && in_fours(decay_logits) && in_fours(decay_bias)));
  if (!chunks) walked_tokens = tokens, longer = longest >= kTilesFrom;
  const Parts parts = parts_of(tokens, seqs, heads, groups, dim, vdim, HEAD_DECAY, chunks, walked_tokens);
  float* raw = workspace + parts.raw;
  if (chunks) {
#define AKV_CHUNKS(TILES)                                                                                                      \
  launch_chunks<T, TD, HEAD_DECAY, TILES>(conv, conv_stride, beta_logits, beta_stride, decay_logits, decay_stride, decay_bias, \
                                          rate, unit_eps, q_scale, state, state_stride, q_start, seq_slots, workspace, raw,    \
                                          tokens, seqs, heads, groups, vdim, stream)
    if (dim == 64) AKV_CHUNKS(1);
    else if (dim == 128) AKV_CHUNKS(2);
    else if (dim == 192) AKV_CHUNKS(3);
    else AKV_CHUNKS(4);
#undef AKV_CHUNKS
  }
  if (walked_tokens > 0) {
    float* prepared = workspace + parts.rows;
    launch_prepare<T, TD, HEAD_DECAY>(conv, conv_stride, beta_logits, beta_stride, decay_logits, decay_stride, decay_bias, rate,
                                      unit_eps, q_scale, prepared, walked_tokens, heads, groups, dim, stream);
    auto walk = [&](int longest, int least, int most) {
      return launch_state_walk<T, kDelta, HEAD_DECAY>(prepared, conv + 2L * groups * dim, conv_stride, state, state_stride, q_start,
                                                      seq_slots, raw, seqs, heads, groups, dim, vdim, 0, longest, stream, least, most);
    };
    const int short_status = shorts ? walk(kTilesFrom - 1, 0, kTilesFrom - 1) : 0;
    const int status = longer && short_status == 0 ? walk(longest, kTilesFrom, chunks ? chunks_from(dim) - 1 : 0x7fffffff) : short_status;
    if (status != 0) return status;
  }
  launch_state_finish<T, TG>(raw, nullptr, 0.f, norm_weight, 0, gates, gate_stride, gate_act, norm_eps, out, tokens, heads, vdim,
                             0, stream);
  return 0;
}

}  // namespace

extern "C" {

void akv_delta_rule_forms(int dim, int* from) { from[0] = kTilesFrom, from[1] = chunks_from(dim); }

long akv_delta_rule_workspace(int tokens, int seqs, int heads, int groups, int dim, int vdim, int decay_per_head, int longest,
                              int walked_tokens) {
  const bool head_decay = decay_per_head != 0;
  const long walked = parts_of(tokens, seqs, heads, groups, dim, vdim, head_decay, false, tokens).total;
  if (longest < chunks_from(dim)) return walked;
  const long in_chunks = parts_of(tokens, seqs, heads, groups, dim, vdim, head_decay, true, walked_tokens).total;
  return in_chunks > walked ? in_chunks : walked;
}

int akv_delta_rule(const void* conv, long conv_stride, int dtype, const void* beta_logits, long beta_stride,
                   const void* decay_logits, int decay_dtype, long decay_stride, const float* decay_bias, const float* rate,
                   int decay_per_head, const void* gates, int gate_dtype, long gate_stride, int gate_act,
                   const float* norm_weight, float unit_eps, float norm_eps, float q_scale, float* state, long state_stride,
                   const int* q_start, const int* seq_slots, float* workspace, void* out, int tokens, int seqs, int heads,
                   int groups, int dim, int vdim, int longest, int walked_tokens, int walked_forms, hipStream_t stream) {
  if (tokens <= 0 || seqs <= 0) return 0;
  if (heads <= 0 || groups <= 0 || heads % groups != 0 || dim <= 0 || vdim <= 0 || dim > 2048) return -2;
  if (gate_act != 1 && gate_act != 2) return -2;
  if (walked_tokens < 0 || walked_tokens > tokens) return -2;
  // decays per channel come from a product of their own with float32 sums, as do their gates; decays per head and their
  // gates are columns of the layer's first product
  const int own = decay_per_head ? dtype : static_cast<int>(kF32);
  if (decay_dtype != own || gate_dtype != own) return -1;
  int status = 0;
#define AKV_DELTA(TD, HEAD)                                                                                                    \
  status = delta_rule<T, TD, TD, HEAD>(static_cast<const T*>(conv), conv_stride, static_cast<const T*>(beta_logits), beta_stride, \
                                       static_cast<const TD*>(decay_logits), decay_stride, decay_bias, rate,                    \
                                       static_cast<const TD*>(gates), gate_stride, gate_act, norm_weight, unit_eps, norm_eps,   \
                                       q_scale, state, state_stride, q_start, seq_slots, workspace, static_cast<T*>(out), tokens, \
                                       seqs, heads, groups, dim, vdim, longest, walked_tokens, walked_forms & 1, walked_forms & 2, stream)
  AKV_DISPATCH(dtype, T, {
    if (decay_per_head) AKV_DELTA(T, true);
    else AKV_DELTA(float, false);
  });
#undef AKV_DELTA
  if (status != 0) return status;
  return AKV_LAUNCH_STATUS();
}
}
