// Prefill attention of a layer over its cached rows: the prologue (per-head norm, rotation,
// cache write) and a tiled attention with the softmax kept on chip.
//
// Arithmetic of the Core chain (core/kernels/attention/default.py:85-156), rounding point
// by rounding point up to the order of the fp32 sums:
//   n = bf16(w * bf16(x * inv)), inv = 1 / sqrt(mean(x^2) + eps)      (heads with a gain)
//   a, b = bf16(n_p * bf16(mscale)), bf16(n_{p+P} * bf16(mscale)), rotated in fp32 and
//   rounded once; scores = (q . k) * scale, softmax and probabilities x values in fp32,
//   the sink logit (if any) in the denominator only, one bf16 rounding at the end.
// A row that attends nothing gives 0 / 0, as the softmax over -inf alone does there.
#include <cfloat>

#include "common.hpp"
#include "host.hpp"

namespace omnia {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4_lds __attribute__((ext_vector_type(4)));

// ---- prologue -------------------------------------------------------------------------

struct ProjectArgs {
  const uint16_t* raw[3];   // queries, keys, values: rows of heads x D, `stride` apart
  int64_t stride[3];
  const uint16_t* gain[2];  // query and key norm weights [D], or null
  const float* cos;         // [length, pairs] rows `table_stride` floats apart
  const float* sin;
  int64_t table_stride;
  uint16_t* out[3];         // head h, token t at h * head_stride + t * D
  int64_t head_stride[3];
  int heads, kv_heads, length, pairs;
  float mscale, eps;
};

// One head vector of one token per D / 8 lanes, 16 bytes a lane: any token count from one
// (80 vectors for 64 + 2 x 8 heads) up. Bound by its launch at one token and by memory at a
// prompt; it stands for about twenty elementwise launches (a sink layer's decode step over
// 4,096 rows: 268 -> 77 us a call, all of it the launches' host time).
template <int D>
__global__ __launch_bounds__(256) void attention_project_kernel(ProjectArgs a) {
  constexpr int kLanes = D / 8;
  const int64_t item = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) / kLanes;
  const int lane = threadIdx.x % kLanes;
  const int slots = a.heads + 2 * a.kv_heads;
  const int64_t token = item / slots;
  int head = static_cast<int>(item % slots);
  if (token >= a.length) return;   // whole groups of lanes: their shuffles stay inside
  const int part = head < a.heads ? 0 : head < a.heads + a.kv_heads ? 1 : 2;
  head -= part == 0 ? 0 : part == 1 ? a.heads : a.heads + a.kv_heads;
  u32x4 v = *reinterpret_cast<const u32x4*>(a.raw[part] + token * a.stride[part] + head * D + lane * 8);
  if (part < 2) {
    float x[8];
    unpack8(v, x);
    const uint16_t* gain = a.gain[part];
    if (gain != nullptr) {
      float sum = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += x[i] * x[i];
      sum = group_sum<kLanes>(sum);
      const float inv = 1.0f / sqrtf(sum / static_cast<float>(D) + a.eps);
      float w[8];
      unpack8(*reinterpret_cast<const u32x4*>(gain + lane * 8), w);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = round_bf16(w[i] * round_bf16(x[i] * inv));
    }
    if (a.pairs > 0) {
      const int half = a.pairs / 8;   // lanes of one half of the rotated block
      const int first = lane < half ? lane : lane - half;
      const int partner = lane < half ? lane + half : lane - half;
      const float factor = round_bf16(a.mscale);
      // Lanes past the rotated block read row 0 of the block and keep their values.
      const int at = lane < 2 * half ? first * 8 : 0;
      float c[8], s[8];
      *reinterpret_cast<f32x4*>(c) = *reinterpret_cast<const f32x4*>(a.cos + token * a.table_stride + at);
      *reinterpret_cast<f32x4*>(c + 4) = *reinterpret_cast<const f32x4*>(a.cos + token * a.table_stride + at + 4);
      *reinterpret_cast<f32x4*>(s) = *reinterpret_cast<const f32x4*>(a.sin + token * a.table_stride + at);
      *reinterpret_cast<f32x4*>(s + 4) = *reinterpret_cast<const f32x4*>(a.sin + token * a.table_stride + at + 4);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float mine = round_bf16(x[i] * factor);
        const float other = __shfl(mine, partner < kLanes ? partner : lane, kLanes);
        const float turned = lane < half ? mine * c[i] - other * s[i] : other * s[i] + mine * c[i];
        x[i] = lane < 2 * half ? turned : x[i];
      }
    }
    v = pack8(x);
  }
  *reinterpret_cast<u32x4*>(a.out[part] + head * a.head_stride[part] + token * D + lane * 8) = v;
}

// ---- attention ------------------------------------------------------------------------

struct PrefillArgs {
  const uint16_t* q;        // [heads, length, D]
  const uint16_t* keys;     // kv head h, row r at h * head_stride + r * D
  const uint16_t* values;
  int64_t key_stride, value_stride;
  const uint8_t* mask;      // [length, rows] bytes (true attends), rows `mask_stride` apart, or null
  int64_t mask_stride;
  const uint16_t* sinks;    // [heads] or null
  uint16_t* out;            // [heads, length, D]
  float* partial;           // splits > 1: [splits, heads, length, D] unnormalised contexts, then
                            // [splits, heads, length, 2] running maxima and sums
  int heads, group, share, length, rows, causal, splits;
  float scale_log2, sink_log2;
};

constexpr int kWaveQueries = 32, kTileKeys = 64, kWaves = 4;
constexpr int kTargetBlocks = 256, kMinSplitTiles = 4, kMaxSplits = 16;
constexpr int kWindow = 64;   // tiles whose masks are looked through at a time

// 4 mask bytes of any alignment (global memory reads need none on this target).
__device__ __forceinline__ uint32_t mask_word(const uint8_t* at) {
  uint32_t word;
  __builtin_memcpy(&word, at, 4);
  return word;
}

// `rows` rows of D values as a buffer, whose loads check their offset against its bytes and
// bring zeros past them (below 2^24 rows of 256 bytes: an offset is 32 bits).
template <int D>
__device__ __forceinline__ auto row_buffer(const uint16_t* first, int rows) {
  constexpr int kRawDword = 0x00027000;   // the resource's last word: 32-bit data, no swizzle
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(first), 0, static_cast<uint32_t>(rows) * (2u * D),
                                           kRawDword);
}

// A workgroup's four waves take 32 queries each: `share` heads of one kv head (the largest
// of 1, 2, 4 dividing the group, so that the waves read the same keys), 4 / share runs of
// queries. It walks the attended rows in tiles of 64 through two LDS buffers, the next
// tile's rows in registers while this one's are multiplied.
//
// Scores are taken transposed, S^T = K Q^T on 32x32x16 MFMA: a lane then holds 32 scores of
// one query (column lane % 32), so the softmax needs one cross-lane step (the other half of
// the wave), its state is a scalar per lane, and P^T is the B operand of O^T = V^T P^T as it
// stands: the MFMA's k index of lane half h, element j names key 8 (j / 4) + 4 h + j % 4,
// for both operands. V^T comes out of LDS by the transposing read.
//
// The probabilities keep their 24 bits: P = p1 + p2 + p3, each the bf16 of what is left, so
// P V is three MFMAs whose products are exact. The scores' products are exact as well.
//
// Bound by the matrix cores and the softmax's VALU work about equally. The torch chain it
// replaces wrote and read the fp32 scores five times and widened and repeated K and V:
// 4,096 tokens, 32 heads over 4, D = 128, causal: 6,181 -> 293 us a call (470 TFLOP/s of the
// products counted once, twice that on the matrix cores); 777 tokens after 1,500, 64 heads
// over 8, D = 64, sinks: 1,962 -> 80 us.
template <int D, bool kMasked>
__global__ __launch_bounds__(256, 2) void attention_prefill_kernel(PrefillArgs a) {
  constexpr int kSteps = D / 16, kBlocks = D / 32, kChunks = D / 8;
  constexpr int kLoads = kTileKeys * kChunks / 256;   // 16-byte vectors a thread stages, each of K and V
  constexpr int kTile = kTileKeys * D;                // elements of one tile
  __shared__ __attribute__((aligned(16))) uint16_t lds[4 * kTile];   // K, V of two stages
  __shared__ unsigned long long window_flags[kMasked ? 2 : 1];

  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int column = lane % 32, half = lane / 32;
  const int head_groups = a.heads / a.share;
  const int tiles_of_queries = static_cast<int>(gridDim.x) / head_groups;
  const int head_group = static_cast<int>(blockIdx.x) % head_groups;
  // The longest tiles of a causal prefill start first.
  const int tile_index = static_cast<int>(blockIdx.x) / head_groups;
  const int query_tile = a.causal ? tiles_of_queries - 1 - tile_index : tile_index;
  const int head = head_group * a.share + wave % a.share;
  const int kv_head = head_group * a.share / a.group;   // of every wave
  const int tile_queries = kWaveQueries * (kWaves / a.share);
  const int first_query = query_tile * tile_queries + (wave / a.share) * kWaveQueries;
  const int query = first_query + column;
  const int query_row = min(query, a.length - 1);
  const int past = a.rows - a.length;
  const int last_query = min((query_tile + 1) * tile_queries, a.length) - 1;
  const int row_end = a.causal ? past + last_query + 1 : a.rows;
  // This workgroup's share of the attended tiles.
  const int split = blockIdx.y;
  const int all_tiles = (row_end + kTileKeys - 1) / kTileKeys;
  const int split_tiles = (all_tiles + a.splits - 1) / a.splits;
  const int first_tile = split * split_tiles;
  const int tiles = min(first_tile + split_tiles, all_tiles);   // past the last
  // Buffers of the head's rows: past the last row a load brings zeros. (The last row again
  // in their place would do for K, whose scores are masked. For V it would not: it has no
  // weight, but zero times an infinity is a NaN.)
  const auto keys = row_buffer<D>(a.keys + kv_head * a.key_stride, a.rows);
  const auto values = row_buffer<D>(a.values + kv_head * a.value_stride, a.rows);

  // Q^T as the B operand: column = query, k = 8 half + j of each 16-wide step.
  s16x8 q[kSteps];
  {
    const uint16_t* row = a.q + (static_cast<int64_t>(head) * a.length + query_row) * D + 8 * half;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) q[s] = *reinterpret_cast<const s16x8*>(row + 16 * s);
  }

  // Staging: thread t's vector i is row (t + 256 i) / kChunks, chunk t % kChunks of the tile.
  // Chunks are permuted in LDS so that both operands' reads touch every bank once: K's 16
  // rows of one chunk, V's four rows of one 64-byte group.
  const int chunk = threadIdx.x % kChunks;
  u32x4 stage_k[kLoads], stage_v[kLoads];
  auto load_tile = [&](int tile) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int row = min(tile * kTileKeys + (static_cast<int>(threadIdx.x) + 256 * i) / kChunks, a.rows);
      const int at = static_cast<int>(static_cast<uint32_t>(row) * (2u * D) + chunk * 16u);   // bytes
      stage_k[i] = __builtin_amdgcn_raw_buffer_load_b128(keys, at, 0, 0);
      stage_v[i] = __builtin_amdgcn_raw_buffer_load_b128(values, at, 0, 0);
    }
  };
  auto store_tile = [&](int stage) {
    uint16_t* tile_k = lds + stage * 2 * kTile;
    uint16_t* tile_v = tile_k + kTile;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int row = (static_cast<int>(threadIdx.x) + 256 * i) / kChunks;
      const int turn_k = D == 128 ? row & 15 : (row >> 1) & 7;
      const int turn_v = D == 128 ? (row & 3) << 2 : (row & 2) << 1;
      *reinterpret_cast<u32x4*>(tile_k + row * D + (chunk ^ turn_k) * 8) = stage_k[i];
      *reinterpret_cast<u32x4*>(tile_v + row * D + (chunk ^ turn_v) * 8) = stage_v[i];
    }
  };

  // Where this lane reads: K row `column`, chunk 2 s + half; V keys 4 half + sub / 4, 4
  // values from 16 (lane / 16 % 2) + 4 (sub % 4) of each 32-wide block.
  const int turn_k = D == 128 ? column & 15 : (column >> 1) & 7;
  const int key_at = column * D + ((half ^ turn_k) * 8);
  const int sub = lane % 16;
  int value_at[kBlocks];
#pragma unroll
  for (int b = 0; b < kBlocks; ++b) {
    const int r = sub / 4;
    const int turn = D == 128 ? r << 2 : (r & 2) << 1;
    const int piece = (b * 4 + 2 * (lane / 16 % 2) + (sub % 4) / 2) ^ turn;
    value_at[b] = (4 * half + r) * D + piece * 8 + (sub % 2) * 4;
  }

  f32x16 out[kBlocks];
#pragma unroll
  for (int b = 0; b < kBlocks; ++b) out[b] = f32x16{};
  const bool sink = a.sinks != nullptr && split == 0;
  const float sink_logit = sink ? bf16_to_f32(a.sinks[head]) : -INFINITY;
  float top = sink ? fminf(fmaxf(sink_logit * a.sink_log2, -FLT_MAX), FLT_MAX) : -INFINITY;
  // The sink's own weight: 1, or 0 where it is -inf, or NaN where it is +inf or a NaN. (Its
  // maximum stays finite, so that it compares and cancels.)
  float total = half == 0 ? __builtin_amdgcn_exp2f(sink_logit - fmaxf(sink_logit, -FLT_MAX)) : 0.0f;

  // With a mask, the tiles in which any of the workgroup's queries attends anything: the
  // masks of 64 tiles at a time are read 256 keys a load, so that the tiles outside a band
  // cost their mask bytes and no more (2,000 tokens, 64 heads over 8, D = 64, a band of 128:
  // 434 -> 86 us; 777 after 1,500: 217 -> 42).
  uint64_t flags = ~uint64_t{0};
  int window = -1;
  auto look = [&](int w) {   // uniform over the workgroup, barriers inside
    if (threadIdx.x == 0) window_flags[w & 1] = 0;
    lds_barrier();
    uint64_t found = 0;
    const int queries = min(tile_queries, a.length - query_tile * tile_queries);
    const int end = min(tiles, (w + 1) * kWindow) * kTileKeys;
    for (int r = wave; r < queries; r += kWaves) {
      const uint8_t* row = a.mask + static_cast<int64_t>(query_tile * tile_queries + r) * a.mask_stride;
#pragma unroll 4
      for (int key0 = w * kWindow * kTileKeys; key0 < end; key0 += 4 * kWave) {
        const int key = key0 + 4 * lane;
        uint32_t word = 0;
        if (key + 4 <= a.rows) {
          word = mask_word(row + key);
        } else {
          for (int i = key; i < a.rows; ++i) word |= row[i];
        }
        const uint64_t lanes = __ballot(word != 0);
        const int at = key0 / kTileKeys - w * kWindow;
#pragma unroll
        for (int i = 0; i < 4; ++i) found |= ((lanes >> (16 * i)) & 0xFFFF) != 0 ? uint64_t{1} << (at + i) : 0;
      }
    }
    if (lane == 0 && found != 0) atomicOr(&window_flags[w & 1], static_cast<unsigned long long>(found));
    lds_barrier();
    flags = window_flags[w & 1];
    window = w;
  };
  auto next_tile = [&](int tile) {   // the first tile from `tile` on to walk, or `tiles`
    if constexpr (!kMasked) return tile;
    while (tile < tiles) {
      if (tile / kWindow != window) look(tile / kWindow);
      const uint64_t rest = flags >> (tile % kWindow);
      if (rest != 0) return min(tile + __builtin_ctzll(rest), tiles);
      tile = (window + 1) * kWindow;
    }
    return tiles;
  };

  int tile = next_tile(first_tile);
  if (tile < tiles) {
    load_tile(tile);
    store_tile(0);
  }
  // Nothing is in flight when the walk begins (the compiler cannot tell the first products'
  // operand from the tile asked for meanwhile, and waited for both).
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  lds_barrier();
  for (int turn = 0; tile < tiles; turn ^= 1) {
    const int following = next_tile(tile + 1);
    const bool more = following < tiles;
    if (more) load_tile(following);
    const int key0 = tile * kTileKeys;
    bool active = first_query < a.length && !(a.causal && key0 > past + first_query + kWaveQueries - 1);
    uint32_t allowed = 0xFFFFFFFFu;
    if (kMasked && active) {
      const uint8_t* row = a.mask + query_row * a.mask_stride;
      allowed = 0;
#pragma unroll
      for (int e = 0; e < 32; e += 4) {   // runs of 4 keys
        const int key = key0 + (e / 16) * 32 + 8 * ((e % 16) / 4) + 4 * half;
        const bool whole = key + 4 <= a.rows;
        const uint32_t word = whole ? mask_word(row + key) : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t byte = whole ? (word >> (8 * i)) & 0xFFu : key + i < a.rows ? row[key + i] : 0;
          allowed |= (byte != 0 ? 1u : 0u) << (e + i);
        }
      }
      active = __ballot(allowed != 0) != 0;
    }
    if (active) {   // the same for the whole wave
      const uint16_t* tile_k = lds + turn * 2 * kTile;
      const uint16_t* tile_v = tile_k + kTile;
      f32x16 s[2] = {f32x16{}, f32x16{}};
#pragma unroll
      for (int step = 0; step < kSteps; ++step) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const s16x8 k = *reinterpret_cast<const s16x8*>(tile_k + kb * 32 * D + (key_at ^ (step * 16)));
          s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, k),
                                                          __builtin_bit_cast(bf16x8, q[step]), s[kb], 0, 0, 0);
        }
      }
      const bool edge = key0 + kTileKeys > a.rows ||
                        (a.causal && key0 + kTileKeys - 1 > past + first_query) || kMasked;
      if (edge) {
        const int bound = a.causal ? min(a.rows - 1, past + query) : a.rows - 1;
#pragma unroll
        for (int e = 0; e < 32; ++e) {
          const int key = key0 + (e / 16) * 32 + 8 * ((e % 16) / 4) + 4 * half + e % 4;
          const bool keep = key <= bound && (!kMasked || ((allowed >> e) & 1u) != 0);
          s[e / 16][e % 16] = keep ? s[e / 16][e % 16] : -INFINITY;
        }
      }
      float best = s[0][0];
#pragma unroll
      for (int e = 1; e < 32; ++e) best = fmaxf(best, s[e / 16][e % 16]);
      uint32_t low, high;
      half_pair(__float_as_uint(best), low, high);
      best = fmaxf(__uint_as_float(low), __uint_as_float(high)) * a.scale_log2;
      const float next = fmaxf(top, best);
      const float base = next == -INFINITY ? 0.0f : next;
      if (__ballot(next > top) != 0) {
        const float shrink = __builtin_amdgcn_exp2f(top - base);
        total *= shrink;
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) out[b] *= shrink;
        top = next;
      }
      float sums[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int step = 0; step < 4; ++step) {   // 16 keys each
        float p[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          p[j] = __builtin_amdgcn_exp2f(
              __builtin_fmaf(s[step / 2][(step % 2) * 8 + j], a.scale_log2, -base));
          sums[j % 4] += p[j];
        }
        u32x4 parts[3];
        split_weights(p, parts);
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
          typedef __attribute__((address_space(3))) s16x4_lds* LdsPtr;
          const uint16_t* at = tile_v + step * 16 * D + value_at[b];
          const s16x4_lds v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsPtr)(at));
          const s16x4_lds v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsPtr)(at + 8 * D));
          const s16x8 v = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
          for (int part = 0; part < 3; ++part) {
            out[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, v),
                                                             __builtin_bit_cast(bf16x8, parts[part]), out[b], 0, 0, 0);
          }
        }
      }
      total += (sums[0] + sums[1]) + (sums[2] + sums[3]);
    }
    if (more) store_tile(turn ^ 1);
    lds_barrier();
    tile = following;
  }

  uint32_t low, high;
  half_pair(__float_as_uint(total), low, high);
  total = __uint_as_float(low) + __uint_as_float(high);
  if (query >= a.length) return;
  if (a.splits > 1) {
    const int64_t at = (static_cast<int64_t>(split) * a.heads + head) * a.length + query;
    float* row = a.partial + at * D + 4 * half;
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        *reinterpret_cast<f32x4*>(row + b * 32 + 8 * i) =
            f32x4{out[b][4 * i], out[b][4 * i + 1], out[b][4 * i + 2], out[b][4 * i + 3]};
      }
    }
    if (half == 0) {
      float* state = a.partial + static_cast<int64_t>(a.splits) * a.heads * a.length * D + 2 * at;
      state[0] = top;
      state[1] = total;
    }
    return;
  }
  const float inverse = 1.0f / total;
  uint16_t* row = a.out + (static_cast<int64_t>(head) * a.length + query) * D + 4 * half;
#pragma unroll
  for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint2 packed;
      packed.x = pack_bf16(out[b][4 * i] * inverse, out[b][4 * i + 1] * inverse);
      packed.y = pack_bf16(out[b][4 * i + 2] * inverse, out[b][4 * i + 3] * inverse);
      *reinterpret_cast<uint2*>(row + b * 32 + 8 * i) = packed;
    }
  }
}

// Merges the splits' states: 4 columns a thread.
template <int D>
__global__ __launch_bounds__(256) void attention_prefill_combine_kernel(const float* partial, uint16_t* out,
                                                                        int64_t rows, int splits) {
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t row = item / (D / 4);   // head * length + token
  if (row >= rows) return;
  const int column = static_cast<int>(item % (D / 4)) * 4;
  const float2* states = reinterpret_cast<const float2*>(partial + splits * rows * D);
  float top = -INFINITY;
  for (int s = 0; s < splits; ++s) top = fmaxf(top, states[s * rows + row].x);
  const float base = top == -INFINITY ? 0.0f : top;
  float total = 0.0f;
  f32x4 sum = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    const float2 state = states[s * rows + row];
    const f32x4 part = *reinterpret_cast<const f32x4*>(partial + (s * rows + row) * D + column);
    const float factor = __builtin_amdgcn_exp2f(state.x - base);
    total = __builtin_fmaf(state.y, factor, total);
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] = __builtin_fmaf(part[i], factor, sum[i]);
  }
  const float inverse = 1.0f / total;
  uint2 packed;
  packed.x = pack_bf16(sum[0] * inverse, sum[1] * inverse);
  packed.y = pack_bf16(sum[2] * inverse, sum[3] * inverse);
  *reinterpret_cast<uint2*>(out + row * D + column) = packed;
}

int64_t head_share(int64_t group) { return group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1; }

int64_t query_blocks(int64_t heads, int64_t group, int64_t length) {
  const int64_t tile = kWaveQueries * (kWaves / head_share(group));
  return heads / head_share(group) * ((length + tile - 1) / tile);
}

// Where the queries' tiles leave CUs without a workgroup, each walks its keys in several, of
// at least four tiles: 64 tokens after 2,000, 32 heads over 8, D = 128: 72.3 -> 24.4 us; 8
// after 2,500: 82.9 -> 18.3; 20 after 2,000, 64 over 8, D = 64: 48.3 -> 14.9. Two for every
// CU cost 1,024 tokens of 32 heads 48.3 us, where one does with 42.5, and two tiles each
// cost 200 tokens 15.2 us for 12.2.
int64_t key_splits(int64_t heads, int64_t kv_heads, int64_t length, int64_t rows) {
  const int64_t blocks = query_blocks(heads, heads / kv_heads, length);
  if (blocks >= kTargetBlocks) return 1;
  const int64_t by_blocks = (kTargetBlocks + blocks - 1) / blocks;
  const int64_t by_tiles = (rows + kTileKeys - 1) / kTileKeys / kMinSplitTiles;
  const int64_t splits = by_blocks < by_tiles ? by_blocks : by_tiles;
  return splits < 1 ? 1 : splits > kMaxSplits ? kMaxSplits : splits;
}

}  // namespace
}  // namespace omnia

extern "C" int64_t omnia_attention_prefill_workspace_bytes(int64_t heads, int64_t kv_heads, int64_t head_dim,
                                                           int64_t length, int64_t rows) {
  using namespace omnia;
  if ((head_dim != 64 && head_dim != 128) || heads <= 0 || kv_heads <= 0 || heads > 4096 || heads % kv_heads != 0 ||
      length < 0 || rows < length || rows >= (int64_t{1} << 24)) {
    return -EINVAL;
  }
  if (length == 0) return 0;
  const int64_t splits = key_splits(heads, kv_heads, length, rows);
  return splits == 1 ? 0 : splits * heads * length * (head_dim + 2) * static_cast<int64_t>(sizeof(float));
}

extern "C" int32_t omnia_attention_project(const uint16_t* raw_queries, int64_t query_stride,
                                           const uint16_t* raw_keys, int64_t key_stride,
                                           const uint16_t* raw_values, int64_t value_stride,
                                           const uint16_t* query_weight, const uint16_t* key_weight,
                                           const float* cos_rows, const float* sin_rows, int64_t table_stride,
                                           int64_t rotary_pairs, float mscale, float eps, int64_t length,
                                           int64_t heads, int64_t kv_heads, int64_t head_dim, uint16_t* queries,
                                           uint16_t* key_rows, int64_t key_head_stride, uint16_t* value_rows,
                                           int64_t value_head_stride, hipStream_t stream) {
  using namespace omnia;
  OMNIA_REQUIRE(head_dim == 64 || head_dim == 128, "attention_project: head_dim must be 64 or 128");
  OMNIA_REQUIRE(heads > 0 && kv_heads > 0 && heads <= 4096 && kv_heads <= 4096, "attention_project: bad head count");
  OMNIA_REQUIRE(length >= 0 && length < (int64_t{1} << 24), "attention_project: bad length");
  OMNIA_REQUIRE(rotary_pairs >= 0 && rotary_pairs % 8 == 0 && 2 * rotary_pairs <= head_dim,
                "attention_project: rotary_pairs must be a multiple of 8 within the head");
  if (length == 0) return 0;
  OMNIA_REQUIRE(raw_queries && raw_keys && raw_values && queries && key_rows && value_rows,
                "attention_project: null pointer");
  OMNIA_REQUIRE(aligned16(raw_queries) && aligned16(raw_keys) && aligned16(raw_values) && aligned16(queries) &&
                    aligned16(key_rows) && aligned16(value_rows) && aligned16(query_weight) && aligned16(key_weight),
                "attention_project: pointers must be 16-byte aligned");
  OMNIA_REQUIRE(query_stride % 8 == 0 && key_stride % 8 == 0 && value_stride % 8 == 0 &&
                    query_stride >= heads * head_dim && key_stride >= kv_heads * head_dim &&
                    value_stride >= kv_heads * head_dim,
                "attention_project: row strides must be multiples of 8 covering the heads");
  OMNIA_REQUIRE(key_head_stride % 8 == 0 && value_head_stride % 8 == 0 && key_head_stride >= length * head_dim &&
                    value_head_stride >= length * head_dim,
                "attention_project: head strides must be multiples of 8 covering the rows");
  OMNIA_REQUIRE(rotary_pairs == 0 || (cos_rows && sin_rows && aligned16(cos_rows) && aligned16(sin_rows) &&
                                      table_stride % 4 == 0 && table_stride >= rotary_pairs),
                "attention_project: angle rows must be 16-byte aligned and cover the pairs");
  int32_t rc = check_device(stream);
  if (rc != 0) return rc;
  ProjectArgs a{{raw_queries, raw_keys, raw_values}, {query_stride, key_stride, value_stride},
                {query_weight, key_weight}, cos_rows, sin_rows, table_stride,
                {queries, key_rows, value_rows}, {length * head_dim, key_head_stride, value_head_stride},
                static_cast<int>(heads), static_cast<int>(kv_heads), static_cast<int>(length),
                static_cast<int>(rotary_pairs), mscale, eps};
  const int64_t threads = length * (heads + 2 * kv_heads) * (head_dim / 8);
  const dim3 grid(static_cast<unsigned>((threads + 255) / 256));
  if (head_dim == 64) {
    attention_project_kernel<64><<<grid, 256, 0, stream>>>(a);
  } else {
    attention_project_kernel<128><<<grid, 256, 0, stream>>>(a);
  }
  return launched("attention_project");
}

extern "C" int32_t omnia_attention_prefill(const uint16_t* queries, const uint16_t* keys, const uint16_t* values,
                                           int64_t key_head_stride, int64_t value_head_stride, int64_t heads,
                                           int64_t kv_heads, int64_t head_dim, int64_t length, int64_t rows,
                                           int32_t causal, const uint8_t* mask, int64_t mask_stride,
                                           const uint16_t* sinks, float scale, void* workspace, int64_t workspace_bytes,
                                           uint16_t* out, hipStream_t stream) {
  using namespace omnia;
  OMNIA_REQUIRE(head_dim == 64 || head_dim == 128, "attention_prefill: head_dim must be 64 or 128");
  OMNIA_REQUIRE(heads > 0 && kv_heads > 0 && heads <= 4096 && heads % kv_heads == 0,
                "attention_prefill: heads must be a multiple of kv_heads");
  OMNIA_REQUIRE(length >= 0 && rows >= length && rows < (int64_t{1} << 24), "attention_prefill: bad lengths");
  OMNIA_REQUIRE(scale > 0.0f && scale < INFINITY, "attention_prefill: the scale must be positive");
  if (length == 0) return 0;
  OMNIA_REQUIRE(queries && keys && values && out, "attention_prefill: null pointer");
  OMNIA_REQUIRE(aligned16(queries) && aligned16(keys) && aligned16(values) && aligned16(out),
                "attention_prefill: pointers must be 16-byte aligned");
  OMNIA_REQUIRE(key_head_stride % 8 == 0 && value_head_stride % 8 == 0 && key_head_stride >= rows * head_dim &&
                    value_head_stride >= rows * head_dim,
                "attention_prefill: head strides must be multiples of 8 covering the rows");
  OMNIA_REQUIRE(mask == nullptr || mask_stride >= rows, "attention_prefill: the mask must cover the rows");
  const int64_t need = omnia_attention_prefill_workspace_bytes(heads, kv_heads, head_dim, length, rows);
  OMNIA_REQUIRE(need == 0 || (workspace && workspace_bytes >= need && aligned16(workspace)),
                "attention_prefill: workspace too small (omnia_attention_prefill_workspace_bytes) or not aligned");
  int32_t rc = check_device(stream);
  if (rc != 0) return rc;
  const int64_t group = heads / kv_heads;
  const int64_t blocks = query_blocks(heads, group, length);
  OMNIA_REQUIRE(blocks < (int64_t{1} << 31), "attention_prefill: too many tiles");
  const int64_t splits = key_splits(heads, kv_heads, length, rows);
  constexpr float kLog2e = 1.4426950408889634f;
  PrefillArgs a{queries, keys, values, key_head_stride, value_head_stride, mask, mask_stride, sinks, out,
                static_cast<float*>(workspace), static_cast<int>(heads), static_cast<int>(group),
                static_cast<int>(head_share(group)), static_cast<int>(length), static_cast<int>(rows),
                causal != 0 ? 1 : 0, static_cast<int>(splits), scale * kLog2e, kLog2e};
  const dim3 grid(static_cast<unsigned>(blocks), static_cast<unsigned>(splits));
  const int64_t merged = heads * length;
  const dim3 merge_grid(static_cast<unsigned>((merged * (head_dim / 4) + 255) / 256));
  const auto kernel = head_dim == 64 ? (mask ? attention_prefill_kernel<64, true> : attention_prefill_kernel<64, false>)
                                     : (mask ? attention_prefill_kernel<128, true> : attention_prefill_kernel<128, false>);
  kernel<<<grid, 256, 0, stream>>>(a);
  if (splits > 1) {
    const auto merge = head_dim == 64 ? attention_prefill_combine_kernel<64> : attention_prefill_combine_kernel<128>;
    merge<<<merge_grid, 256, 0, stream>>>(a.partial, out, merged, a.splits);
  }
  return launched("attention_prefill");
}
