// Attention over the paged cache in float32, on the matrix cores.
//
// v_mfma_f32_16x16x4_f32 takes float32 operands as they are and adds in float32.  A wave works on a tile of 16 query rows -
// consecutive (token, head) pairs of one request whose heads read the same kv head - and 16 keys at a time:
//   scores  S^T [keys x rows]  = K [keys x dim] Q^T:   a lane's operand of four instructions is 16 bytes of a key's record;
//   sums    O^T [dim x rows]   = V^T [dim x keys] P^T: 16 bytes of a value row (pages hold values [dim, page]); what a lane
//           has of S^T - keys 4 g .. 4 g + 3 of row lane & 15 - is its operand P^T as it stands, no exchange between lanes.
// The order of every sum depends on the token's own position only - not on how a request was cut into steps, on what else
// is in the batch, or on which blocks did the work: keys are cut at absolute positions into segments of 256; the four waves
// of a block take tiles w, w + 4, w + 8, w + 12 of a segment's sixteen under ONE maximum per wave (no running rescaling
// inside a segment), the waves' sums are folded in their order, then the segments' in theirs, always by `Fold`.  A tile or
// segment that a row does not see folds as the identity, bit for bit.  Where a step has fewer tiles than would fill the
// device, blocks take (tile, segment) items, leave the segments' sums in memory - counted from the first segment that a row sees,
// so that a window bounds them - and a second kernel folds them: the same folds, the same bits.  Such a launch may take a part
// of the step's tokens, as many as the caller has room for.
//
// Rows of one tile have different positions: a key that one row sees and another does not gets weight zero for the
// other, and zero times an infinity is not zero.  So where a tile of keys is masked for some rows and its values are not
// all finite, the sums are taken key by key and kept only for the rows that see the key.
//
// What bounds it: single tokens wait for their keys - a trip to the block table, one to the records, one to the values, then
// the fold's launch; prompts run at the matrix cores' rate (64 instructions of 32 cycles per 16 x 16 scores at dim 128) where
// their tiles fill the device.  Measured, us a layer, 16 heads over 4 of 128, against one wave per (token, head) in plain
// float32 (`attention_rows`): 3 single tokens after 64 to 700 keys 298 -> 13.4 + 4.6 for the fold; 3 prompts of 333 tokens
// 811 -> 47.

#include <type_traits>

#include "common.h"
#include "api.h"

using namespace akv;

namespace {

typedef float floats4 __attribute__((ext_vector_type(4)));

constexpr int kRows = 16;         // query rows of a tile
constexpr int kSegment = 256;     // keys of a segment
constexpr int kTiles = 4;         // tiles of 16 keys a wave takes of a segment

struct Args {
  const float* q;
  const float* k_pages;
  const float* v_pages;
  float* out;
  float* partial;                 // [(token_end - first_token) * q_heads][segments][dim + 4], or null: a block folds all of its tile's
  const int* q_start;
  const int* seq_lens;
  const int* block_table;
  const int* table_rows;
  int table_width, seqs, q_heads, kv_heads, page_size, window, segments, splits;
  int first_tile, first_token, token_end;      // what the launch takes of the step's tokens (all of them where `partial` is null)
  long num_pages;
  float scale;
  int share;                      // query heads of a key head
  Divider by_share, by_page;      // (a dozen divisions stand before a tile's loads: a step of 3 requests, 8 layers, 615 -> 604 us)
};

// What a running (maximum, sum of weights, weighted sums) and a later part of it are multiplied by when they are added; the
// maximum becomes that of both.  A part of no keys has maximum -inf and sums of zero.
struct Fold {
  float kept, added;
  __device__ __forceinline__ Fold(float& maximum, float other) {
    const float m = fmaxf(maximum, other);
    const float shift = m == -INFINITY ? 0.f : m;          // (of a part of no keys the factor is exp(-inf))
    kept = expf(maximum - shift);
    added = expf(other - shift);
    maximum = m;
  }
  // (written as one fused operation: left to the compiler, two kernels could fuse the two products differently)
  __device__ __forceinline__ float operator()(float total, float part) const { return fmaf(total, kept, part * added); }
};

__device__ __forceinline__ bool all_finite(const floats4 v) {
  bool fine = true;              // (an exponent of all ones: infinity or NaN)
#pragma unroll
  for (int j = 0; j < 4; ++j) fine = fine & ((__float_as_uint(v[j]) & 0x7f800000u) != 0x7f800000u);
  return fine;
}

// Whose tile this is: tiles are numbered request by request, and a lane counts those of EACH requests in a row (four: one turn for
// 256).  Sets `request`, which is -1 before, and leaves `tile` its number in the request; the same for all lanes of a wave.  With
// four that is said to the compiler, which keeps what follows from it in scalar registers; a block of SPLIT, which waits for each
// load in turn, finds the next numbers of the step sooner where the vector loads left them (a decode step of 3 requests and 8
// layers: 632 us with scalar loads, 624 without).
template <int EACH>
__device__ __forceinline__ void find_request(const Args& a, int share, int lane, int& request, int& tile) {
  for (int first = 0; first < a.seqs && request < 0; first += EACH * kWave) {
    int upto[EACH], count = 0, start = a.q_start[min(first + EACH * lane, a.seqs)];
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int end = a.q_start[min(first + EACH * lane + i + 1, a.seqs)];
      upto[i] = count += ((end - start) * share + kRows - 1) / kRows;
      start = end;
    }
    int all = count;
#pragma unroll
    for (int step = 1; step < kWave; step <<= 1) {
      const int other = __shfl_up(all, step, kWave);
      if (lane >= step) all += other;
    }
    const unsigned long long here = __ballot(tile < all);
    if (here != 0) {
      const int at = __ffsll(here) - 1, own = tile - (all - count);
      int of_lane = 0, before = 0;
#pragma unroll
      for (int i = 0; i + 1 < EACH; ++i) {
        of_lane += own >= upto[i];
        before = own >= upto[i] ? upto[i] : before;
      }
      request = first + EACH * at + (EACH > 1 ? __builtin_amdgcn_readlane(of_lane, at) : 0);
      tile = EACH > 1 ? __builtin_amdgcn_readlane(own - before, at) : __shfl(own, at, kWave);
    } else {
      tile -= __shfl(all, kWave - 1, kWave);
    }
  }
}

// FEW: there are fewer blocks than compute units, and a block waits for its loads: a tile's values are asked for a tile ahead,
// with the registers of one wave a SIMD.  Otherwise two waves a SIMD hide each other's waits, three or four of narrow heads.
// A wave that has one tile of a segment - short contexts, windows, a request's last segment - takes that one alone, with its
// values asked for beside its records, and one that has none goes straight to the fold: 256 tokens of 30 keys, 16 heads of
// 64 of their own, 73 us with four tiles always and 34 now (31 in `attention_rows`), a window of 100 of 300 keys 130 -> 65 (79),
// 5 tokens of 16 / 4 heads of 128 12.4 -> 8.6 (11.1).  SPLIT: the segments are blocks of their own, most of them whole, and waves
// take four tiles always.
template <int NT, bool FEW, bool SPLIT>
__global__ __launch_bounds__(256, FEW || NT > 8 ? 1 : NT > 4 ? 2 : NT > 2 ? 3 : 4) void attention_f32_kernel(const Args a) {
  constexpr int kDim = 16 * NT;
  constexpr int kOwn = (NT + 3) / 4;             // tiles of 16 dims whose totals a wave keeps: w, w + 4, ...
  constexpr int kGroup = NT <= 6 ? kTiles : 2;   // tiles of keys whose records are asked for together (registers)
  __shared__ floats4 sums_of[4][NT][64];
  __shared__ float top_of[4][kRows], weight_of[4][kRows];
  const int lane = threadIdx.x & 63, wave = SPLIT ? threadIdx.x >> 6 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;        // the row (or key, or dim) of a tile, and the lane's group of four
  const int share = a.share, kvh = blockIdx.y;

  int request = -1, tile = a.first_tile + static_cast<int>(blockIdx.x);
  find_request<SPLIT ? 1 : 4>(a, share, lane, request, tile);
  if (request < 0) return;
  if constexpr (!SPLIT) request = __builtin_amdgcn_readfirstlane(request), tile = __builtin_amdgcn_readfirstlane(tile);
  const int token0 = a.q_start[request], tokens = a.q_start[request + 1] - token0;
  const int rows = tokens * share, row0 = tile * kRows;
  const int history = a.seq_lens[request] - tokens;
  const int* table = a.block_table + static_cast<long>(a.table_rows != nullptr ? a.table_rows[request] : request) * a.table_width;
  const int row = min(row0 + c, rows - 1);       // (rows beyond the request's repeat its last and are not stored)
  const int of_token = a.by_share.quotient(row), token = token0 + of_token, head = kvh * share + a.by_share.rest(row, of_token);
  const int pos = history + of_token;
  const int low = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  // keys that some row of the tile sees: lowest .. pos_max; that every row sees: low_max .. pos_min
  const int pos_min = history + a.by_share.quotient(row0), pos_max = history + a.by_share.quotient(min(row0 + kRows - 1, rows - 1));
  const int lowest = a.window > 0 ? max(0, pos_min - a.window + 1) : 0;
  const int low_max = a.window > 0 ? max(0, pos_max - a.window + 1) : 0;
  const int first_segment = lowest / kSegment, last_segment = pos_max / kSegment;

  const int stride = SPLIT ? a.splits : 1, first_own = first_segment + (SPLIT ? static_cast<int>(blockIdx.z) : 0);
  if (first_own > last_segment) return;

  floats4 q[NT];
  {
    const float* qp = a.q + (static_cast<long>(token) * a.q_heads + head) * kDim + 4 * g;
#pragma unroll
    for (int b = 0; b < NT; ++b) q[b] = *reinterpret_cast<const floats4*>(qp + 16 * b);
  }
  const floats4 zero = {0.f, 0.f, 0.f, 0.f};
  float total_top = -INFINITY, total_weight = 0.f;
  floats4 total[kOwn];
#pragma unroll
  for (int i = 0; i < kOwn; ++i) total[i] = zero;

  for (int segment = first_own; segment <= last_segment; segment += stride) {
    // A wave's tiles that some row sees lie side by side: the first and how many (the same for the whole wave)
    const auto first_tile_of = [&](int w) { return max(0, (lowest - 15 - (segment * kSegment + 16 * w) + 63) >> 6); };
    const auto tiles_of = [&](int w) {
      return min(kTiles - 1, (pos_max - (segment * kSegment + 16 * w)) >> 6) - first_tile_of(w) + 1;
    };
    floats4 sums[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) sums[n] = zero;
    float top = -INFINITY, weight = 0.f;
    // The scores of a wave's TILES tiles from `base` on, their maximum, weights and weighted sums.
    const auto take = [&](auto count, const int base) {
      constexpr int TILES = decltype(count)::value;
      constexpr int kTogether = TILES < kGroup ? TILES : kGroup;
      constexpr bool kAtOnce = TILES == 1;       // the values are asked for with the records
      // ---- scores of the wave's tiles
      // (no load stands behind a test: the compiler would wait for it before the next.  A key that no row sees asks for the
      // nearest that one does)
      floats4 s[TILES], v[NT];
      const float* vp[TILES];                    // the lane's four keys in their page's first value row
      bool there[TILES];
      const auto values = [&](int t, floats4* to) {
#pragma unroll
        for (int n = 0; n < NT; ++n) to[n] = *reinterpret_cast<const floats4*>(vp[t] + static_cast<long>(16 * n + c) * a.page_size);
      };
#pragma unroll
      for (int t0 = 0; t0 < TILES; t0 += kTogether) {
        floats4 k[kTogether][NT];
        bool known[kTogether];
        int key[kTogether], four[kTogether], page[kTogether], vpage[kTogether], nth[kTogether], vnth[kTogether];
#pragma unroll
        for (int t = 0; t < kTogether; ++t) {
          key[t] = min(max(base + 64 * (t0 + t) + c, lowest), pos_max);
          four[t] = min(max(base + 64 * (t0 + t) + 4 * g, lowest & ~3), pos_max & ~3);      // (pages hold a multiple of four)
          nth[t] = a.by_page.quotient(key[t]);
          vnth[t] = a.by_page.quotient(four[t]);
          page[t] = table[nth[t]];
          vpage[t] = table[vnth[t]];
        }
#pragma unroll
        for (int t = 0; t < kTogether; ++t) {
          known[t] = (page[t] >= 0) & (page[t] < a.num_pages);       // (a page that is not the request's is never read: its scores
          there[t0 + t] = (vpage[t] >= 0) & (vpage[t] < a.num_pages);                                              // are NaN)
          const long record = ((known[t] ? page[t] : 0) * static_cast<long>(a.kv_heads) + kvh) * a.page_size + a.by_page.rest(key[t], nth[t]);
          const float* kp = a.k_pages + record * kDim + 4 * g;
#pragma unroll
          for (int b = 0; b < NT; ++b) k[t][b] = *reinterpret_cast<const floats4*>(kp + 16 * b);
          vp[t0 + t] = a.v_pages + ((there[t0 + t] ? vpage[t] : 0) * static_cast<long>(a.kv_heads) + kvh) * kDim * a.page_size +
                       a.by_page.rest(four[t], vnth[t]);
        }
        if constexpr (kAtOnce) values(0, v);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < kTogether; ++t) {
          floats4 scores = zero;
#pragma unroll
          for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) scores = __builtin_amdgcn_mfma_f32_16x16x4f32(k[t][b][e], q[b][e], scores, 0, 0, 0);
          // lane (c, g) now has row c's scores of keys 4 g .. 4 g + 3
          const unsigned unknown = static_cast<unsigned>(__ballot(!known[t]) & 0xffffu);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int key = base + 64 * (t0 + t) + 4 * g + j;
            const float score = (unknown >> (4 * g + j)) & 1u ? __uint_as_float(0x7fc00000u) : scores[j] * a.scale;
            s[t0 + t][j] = (key >= low) & (key <= pos) ? score : -INFINITY;
          }
        }
      }
      // ---- one maximum for the wave's tiles, weights, their sum
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) top = fmaxf(top, s[t][j]);
      top = fmaxf(top, __shfl_xor(top, 16, kWave));
      top = fmaxf(top, __shfl_xor(top, 32, kWave));
      const float shift = top == -INFINITY ? 0.f : top;
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          s[t][j] = expf(s[t][j] - shift);         // (exp(-inf) of a key that the row does not see)
          weight += s[t][j];
        }
      weight += __shfl_xor(weight, 16, kWave);
      weight += __shfl_xor(weight, 32, kWave);
      // ---- weighted sums
      constexpr bool kAhead = FEW && NT <= 8 && !kAtOnce;
      floats4 next[kAhead ? NT : 1];
      if constexpr (kAhead) values(0, next);
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
        const int first_key = base + 64 * t;
        if constexpr (kAhead) {
#pragma unroll
          for (int n = 0; n < NT; ++n) v[n] = next[n];
          if (t + 1 < TILES) values(t + 1, next);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (first_key > pos_max || first_key + 15 < lowest) continue;        // (the same for the whole wave)
        if constexpr (!kAhead && !kAtOnce) values(t, v);
        bool fine = true;
        if (first_key < low_max || first_key + 15 > pos_min || !__all(there[t])) {
          // some row does not see some key of the tile.  Slots that nobody has written, or that are not the request's, hold
          // anything: no row sees them, and they count as zero
#pragma unroll
          for (int n = 0; n < NT; ++n) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int key = first_key + 4 * g + j;
              v[n][j] = there[t] & (key >= lowest) & (key <= pos_max) ? v[n][j] : 0.f;
            }
            fine = fine & all_finite(v[n]);
          }
        }
        if (__all(fine)) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int n = 0; n < NT; ++n) sums[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[n][e], s[t][e], sums[n], 0, 0, 0);
        } else {                                   // key by key, for the rows that see it
#pragma unroll 1
          for (int four = 0; four < 4; ++four)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int key = first_key + 4 * four + e;
              const bool seen = key >= low && key <= pos, mine = four == g;
#pragma unroll
              for (int n = 0; n < NT; ++n) {
                const floats4 with = __builtin_amdgcn_mfma_f32_16x16x4f32(mine ? v[n][e] : 0.f, mine ? s[t][e] : 0.f, sums[n], 0, 0, 0);
                if (seen) sums[n] = with;
              }
            }
        }
      }
    };
    const int own_tiles = tiles_of(wave);
    if (!SPLIT && own_tiles == 1)
      take(std::integral_constant<int, 1>(), segment * kSegment + wave * 16 + 64 * first_tile_of(wave));
    else if (SPLIT || own_tiles > 1)
      take(std::integral_constant<int, kTiles>(), segment * kSegment + wave * 16);
    // ---- the four waves' parts, in their order; one of no keys changes nothing (and is passed over where no latency hangs on it)
    if (FEW || own_tiles > 0) {
#pragma unroll
      for (int n = 0; n < NT; ++n) sums_of[wave][n][lane] = sums[n];
      if (g == 0) {
        top_of[wave][c] = top;
        weight_of[wave][c] = weight;
      }
    }
    __syncthreads();
    float segment_top = -INFINITY, segment_weight = 0.f;
    floats4 segment_sums[kOwn];
#pragma unroll
    for (int i = 0; i < kOwn; ++i) segment_sums[i] = zero;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (!FEW && tiles_of(w) <= 0) continue;
      const Fold f(segment_top, top_of[w][c]);
      segment_weight = f(segment_weight, weight_of[w][c]);
#pragma unroll
      for (int i = 0; i < kOwn; ++i) {
        if (wave + 4 * i >= NT) continue;
        const floats4 part = sums_of[w][wave + 4 * i][lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) segment_sums[i][j] = f(segment_sums[i][j], part[j]);
      }
    }
    __syncthreads();                             // (the next segment writes LDS again)
    if constexpr (SPLIT) {
      const int of_row = segment - low / kSegment;         // (segments that the row does not see are nobody's to fold)
      if (row0 + c < rows && token >= a.first_token && token < a.token_end && of_row >= 0 && of_row < a.segments) {
        float* at = a.partial + ((static_cast<long>(token - a.first_token) * a.q_heads + head) * a.segments + of_row) * (kDim + 4);
#pragma unroll
        for (int i = 0; i < kOwn; ++i)
          if (wave + 4 * i < NT) *reinterpret_cast<floats4*>(at + 16 * (wave + 4 * i) + 4 * g) = segment_sums[i];
        if (wave == 0 && g == 0) {
          at[kDim] = segment_top;
          at[kDim + 1] = segment_weight;
        }
      }
      continue;
    }
    const Fold f(total_top, segment_top);
    total_weight = f(total_weight, segment_weight);
#pragma unroll
    for (int i = 0; i < kOwn; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) total[i][j] = f(total[i][j], segment_sums[i][j]);
  }
  if (SPLIT || row0 + c >= rows) return;
  float* at = a.out + (static_cast<long>(token) * a.q_heads + head) * kDim + 4 * g;
#pragma unroll
  for (int i = 0; i < kOwn; ++i) {
    if (wave + 4 * i >= NT) continue;
    floats4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = total[i][j] / total_weight;
    *reinterpret_cast<floats4*>(at + 16 * (wave + 4 * i)) = o;
  }
}

// The segments' sums of one (token, head), in their order: a wave a row, four values of dim a lane.
__global__ __launch_bounds__(256) void attention_f32_fold_kernel(const Args a, const int* __restrict__ positions, int dim, long rows) {
  const int lane = threadIdx.x & 63;
  const long row = static_cast<long>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int pos = positions[a.first_token + row / a.q_heads];
  const int low = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  const int d = min(4 * lane, dim - 4);
  const float* at = a.partial + row * a.segments * (dim + 4);
  float total_top = -INFINITY, total_weight = 0.f;
  floats4 total = {0.f, 0.f, 0.f, 0.f};
  const int last = min(pos / kSegment - low / kSegment, a.segments - 1);
#pragma unroll 4
  for (int segment = 0; segment <= last; ++segment) {
    const float* part = at + static_cast<long>(segment) * (dim + 4);
    const floats4 sums = *reinterpret_cast<const floats4*>(part + d);
    const float top = part[dim], weight = part[dim + 1];
    const Fold f(total_top, top);
    total_weight = f(total_weight, weight);
#pragma unroll
    for (int j = 0; j < 4; ++j) total[j] = f(total[j], sums[j]);
  }
  if (4 * lane >= dim) return;
#pragma unroll
  for (int j = 0; j < 4; ++j) total[j] /= total_weight;
  *reinterpret_cast<floats4*>(a.out + (static_cast<long>(a.first_token) * a.q_heads + row) * dim + d) = total;
}

}  // namespace

extern "C" int akv_attention_f32_fits(int dim, int page_size) {
  const int nt = dim / 16;
  return dim % 16 == 0 && page_size > 0 && page_size % 4 == 0 &&
         ((nt >= 1 && nt <= 6) || nt == 8 || nt == 12 || nt == 16);
}

extern "C" int akv_attention_f32_segments(long tiles, int longest, int window, int kv_heads) {
  int segments = (longest + kSegment - 1) / kSegment;
  // (a row's keys are `window` in a row: they touch one segment more than they fill where they begin inside one)
  if (window > 0) segments = min(segments, (window + kSegment - 2) / kSegment + 1);
  return segments <= 1 || tiles * kv_heads >= device_facts().compute_units ? 1 : segments;
}

extern "C" int akv_attention_f32(const float* q, const float* k_pages, const float* v_pages, const int* q_start, const int* seq_lens,
                                 const int* positions, const int* block_table, const int* table_rows, int table_width, float* out,
                                 float* partial, int first_token, int token_end, int seqs, int first_tile, long tiles, int segments,
                                 int q_heads, int kv_heads, int dim, int page_size, long num_pages, float scale, int window,
                                 hipStream_t stream) {
  if (token_end <= first_token || seqs <= 0 || tiles <= 0) return 0;
  if (!akv_attention_f32_fits(dim, page_size) || first_token < 0 || first_tile < 0 || first_tile + tiles > 0x7fffffffL ||
      kv_heads <= 0 || kv_heads > 65535 || q_heads < kv_heads || segments < 1 ||
      (partial == nullptr) != (segments == 1) ||
      (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_pages) | reinterpret_cast<uintptr_t>(v_pages) |
       reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(partial)) % 16 != 0)      // (what is read and written 16 bytes at a time)
    return -2;
  Args a{q, k_pages, v_pages, out, partial, q_start, seq_lens, block_table, table_rows, table_width, seqs, q_heads, kv_heads,
         page_size, window, segments, 1, first_tile, first_token, token_end, num_pages, scale, q_heads / kv_heads,
         Divider::of(q_heads / kv_heads), Divider::of(page_size)};
  if (partial != nullptr) {
    const long blocks = tiles * kv_heads, wanted = (2L * device_facts().compute_units + blocks - 1) / blocks;
    a.splits = static_cast<int>(wanted < segments ? wanted : segments);
  }
  const dim3 grid(static_cast<unsigned>(tiles), kv_heads, a.splits);
  const bool few = tiles * kv_heads < device_facts().compute_units;
  switch (dim / 16) {
#define AKV_CASE(n)                                                                            \
  case n:                                                                                      \
    if (partial != nullptr) attention_f32_kernel<n, true, true><<<grid, 256, 0, stream>>>(a); \
    else if (few) attention_f32_kernel<n, true, false><<<grid, 256, 0, stream>>>(a);           \
    else attention_f32_kernel<n, false, false><<<grid, 256, 0, stream>>>(a);                   \
    break
    AKV_CASE(1); AKV_CASE(2); AKV_CASE(3); AKV_CASE(4); AKV_CASE(5); AKV_CASE(6); AKV_CASE(8); AKV_CASE(12); AKV_CASE(16);
#undef AKV_CASE
  }
  if (partial != nullptr) {
    const long rows = static_cast<long>(token_end - first_token) * q_heads;
    attention_f32_fold_kernel<<<static_cast<unsigned>((rows + 3) / 4), 256, 0, stream>>>(a, positions, dim, rows);
  }
  return AKV_LAUNCH_STATUS();
}
