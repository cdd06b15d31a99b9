// The packed NVFP4 down/combine (moe_fp4.hip, moe_down_nvfp4_shared_kernel) over a prompt:
// the same results with the tokens grouped by expert, so that each expert's matrix is read
// and decoded once for all of its tokens and the products run on the matrix cores.
//
//   1. expert_plan_kernel lists every expert's (token, slot) pairs;
//   2. grouped_down_kernel: d[t, s, n] = bf16(sum_i act[t, s, i] W_e[n, i]) into scratch, a
//      workgroup per (expert, 128 output rows), and per (run of tokens, 128 rows) for the
//      shared stack;
//   3. grouped_combine_kernel: the bf16 epilogue of the per-token kernel, in slot order.
//
// A weight is an e2m1 code (2 significant bits) times an e4m3 scale (4 bits): at most 6
// significant bits, so the product is a bf16 exactly and every product with a bf16
// activation is exact in fp32, as in the per-token kernel; only the order of the fp32 sum
// differs.
//
// The per-token kernel reads a token's 11 matrices anew and multiplies on the vector units:
// bound by that work, 1.6 us a token. Here the floor is the stacks' bytes, or with many
// tokens per expert the products. Top-10 of 512 experts plus the shared one, hidden 2048:
// 818 -> 103 us at 512 tokens (the stacks' 302 MB: 47 us at a copy's rate; under tracing 87 in
// grouped_down_kernel, 9 in the combine, 6 in the plan), 6,471 -> 385 at 4,096.
#include <cmath>

#include "common.hpp"
#include "fp4.hpp"
#include "host.hpp"

namespace omnia {
namespace {

constexpr int kInner = 512;             // the packed form's contraction
constexpr int kChunks = kInner / 32;    // 16-byte vectors of codes per row
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * kWave;
constexpr int kRowsPerBlock = kWaves * 32;
constexpr int kLdsRow = kInner + 8;     // padded: 16 rows of one 16-byte column on distinct banks
constexpr int kPlanThreads = 512;
constexpr int64_t kScratchBytes = int64_t{256} << 20;   // d of one pass over some of the tokens

// offsets[e] = the pairs whose expert is below e (invalid ids excluded), entries[offsets[e]
// ..] = expert e's pairs (token * top_k + slot), those of one thread after another. One
// workgroup per expert, each reading all ids (they stay in cache): no atomics, nothing to
// clear.
__global__ __launch_bounds__(kPlanThreads) void expert_plan_kernel(const int32_t* chosen, int pairs, int experts,
                                                                   int32_t* offsets, int32_t* entries) {
  constexpr int kPlanWaves = kPlanThreads / kWave;
  __shared__ int wave_less[kPlanWaves], wave_equal[kPlanWaves];
  const int expert = blockIdx.x;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  int less = 0, equal = 0;
#pragma unroll 4
  for (int i = threadIdx.x; i < pairs; i += kPlanThreads) {
    const int id = chosen[i];
    less += id >= 0 && id < expert ? 1 : 0;
    equal += id == expert ? 1 : 0;
  }
  int before = equal;   // inclusive scan of `equal` over the wave
#pragma unroll
  for (int step = 1; step < kWave; step *= 2) {
    const int below = __shfl_up(before, step, kWave);
    before += lane >= step ? below : 0;
  }
  less = group_sum<kWave>(less);
  if (lane == kWave - 1) {
    wave_less[wave] = less;
    wave_equal[wave] = before;
  }
  __syncthreads();
  int base = 0, total = 0, at = before - equal;
#pragma unroll
  for (int w = 0; w < kPlanWaves; ++w) {
    base += wave_less[w];
    total += wave_equal[w];
    at += w < wave ? wave_equal[w] : 0;
  }
  if (threadIdx.x == 0) {
    offsets[expert] = base;
    if (expert == experts - 1) offsets[experts] = base + total;
  }
  if (total == 0) return;
  at += base;
#pragma unroll 4
  for (int i = threadIdx.x; i < pairs; i += kPlanThreads) {
    if (chosen[i] == expert) entries[at++] = i;
  }
}

struct GroupedArgs {
  const uint16_t* act;       // [tokens, top_k + 1, 512]
  const u32x4* weight;       // [experts, hidden, 16] chunks of 32 codes
  const uint16_t* scales;    // [experts, hidden, 16] pairs of e4m3 bytes
  const u32x4* shared_weight;
  const uint16_t* shared_scales;
  const int32_t* offsets;
  const int32_t* entries;
  uint16_t* d;               // [tokens, top_k + 1, stride] bf16
  int tokens, top_k, hidden, stride;
  int shared_blocks;         // workgroups (per row tile) over the shared stack's tokens
  int splits;                // workgroups (per row tile) over one expert's tokens
  int row_tiles;             // tiles of 128 rows per workgroup
};

// What a workgroup works on: `count` tokens' pairs of one expert, or the shared stack's
// tokens, in tiles first_tile, first_tile + tile_step, ...
struct Run {
  const int32_t* entries;   // null for the shared stack
  const u32x4* codes;       // of the matrix' first row
  const uint16_t* scales;
  int first_tile, tile_step, count, slots, top_k;
  // The activation (and d) row of the run's `at`-th pair (at most the last): a lane each,
  // from one load, read ahead of the loads that wait for nothing.
  __device__ __forceinline__ int pair(int at) const {
    at = min(at, count - 1);
    const int entry = entries != nullptr ? entries[at] : 0;
    return entries != nullptr ? entry / top_k * slots + entry % top_k : at * slots + top_k;
  }
};

__device__ __forceinline__ int of_lane(int value, int lane) { return __builtin_amdgcn_readlane(value, lane); }

__device__ __forceinline__ Run run_of(const GroupedArgs& a, int unit) {
  Run r;
  r.slots = a.top_k + 1;
  r.top_k = a.top_k;
  if (unit < a.shared_blocks) {   // the longest runs start first
    r.entries = nullptr;
    r.codes = a.shared_weight;
    r.scales = a.shared_scales;
    r.first_tile = unit;
    r.tile_step = a.shared_blocks;
    r.count = a.tokens;
    return r;
  }
  const int expert = (unit - a.shared_blocks) / a.splits;
  const int begin = a.offsets[expert];
  const int64_t first = static_cast<int64_t>(expert) * a.hidden * kChunks;
  r.entries = a.entries + begin;
  r.codes = a.weight + first;
  r.scales = a.scales + first;
  r.first_tile = (unit - a.shared_blocks) % a.splits;
  r.tile_step = a.splits;
  r.count = a.offsets[expert + 1] - begin;
  return r;
}

// The bf16 operand of one word of codes: 8 weights, exactly.
__device__ __forceinline__ bf16x8 decode(uint32_t word, float s) {
  const f32x2 v0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 0);
  const f32x2 v1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 1);
  const f32x2 v2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 2);
  const f32x2 v3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 3);
  u32x4 packed;
  packed.x = pack_bf16(v0.x * s, v0.y * s);
  packed.y = pack_bf16(v1.x * s, v1.y * s);
  packed.z = pack_bf16(v2.x * s, v2.y * s);
  packed.w = pack_bf16(v3.x * s, v3.y * s);
  return __builtin_bit_cast(bf16x8, packed);
}

typedef const __attribute__((address_space(1))) void* GlobalPtr;
typedef __attribute__((address_space(3))) void* LdsPtr;

// Few tokens per expert: the codes' stream from HBM is the bound. A workgroup stages 16
// tokens and walks `row_tiles` tiles of 128 rows, a wave 32 of them as two 16-row operands
// that share the activations' LDS reads. A wave's codes come through its own piece of LDS, a
// load bringing four whole rows (1 KiB): loads in operand order took 64 bytes of 16 rows each
// and fetched lines twice once a CU's waves outgrew its L1. The next tile's codes are under
// way while this one's, moved to registers, are multiplied. The k index is free as long as
// both operands share it: lane group g takes chunk 4 i + g, i < 4.
__global__ __launch_bounds__(kThreads, 3) void grouped_down_kernel(GroupedArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t codes_lds[kRowsPerBlock * kInner / 4];
  __shared__ __attribute__((aligned(16))) uint16_t tile[16 * kLdsRow];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  const int column = lane % 16, group = lane / 16;
  const Run run = run_of(a, blockIdx.y);
  const int tiles = (run.count + 15) / 16;
  if (run.first_tile >= tiles) return;   // the same for the whole workgroup
  const int first_row = blockIdx.x * a.row_tiles * kRowsPerBlock + wave * 32;
  uint16_t* wave_codes = codes_lds + wave * (32 * kInner / 4);
  // Position p of row r holds chunk p ^ (r % 16), so that 16 rows' reads of one chunk touch
  // every bank once. Rows past the last re-read the last and are not stored.
  auto load_codes = [&](int row0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 4 * i + group;
      const int64_t at = static_cast<int64_t>(min(row0 + r, a.hidden - 1)) * kChunks + (column ^ (r % 16));
      __builtin_amdgcn_global_load_lds((GlobalPtr)(run.codes + at), (LdsPtr)(wave_codes + i * 512), 16, 0, 0);
    }
  };
  uint32_t scale[2][4];
  auto load_scales = [&](int row0) {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int64_t at = static_cast<int64_t>(min(row0 + 16 * sub + column, a.hidden - 1)) * kChunks + group;
#pragma unroll
      for (int i = 0; i < 4; ++i) scale[sub][i] = run.scales[at + 4 * i];
    }
  };
  int pair = run.pair(run.first_tile * 16 + column);
  load_codes(first_row);
  load_scales(first_row);

  for (int t = run.first_tile; t < tiles; t += run.tile_step) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {   // one activation row (1 KiB) per load of a wave
      const int64_t from = of_lane(pair, 4 * i + wave);
      __builtin_amdgcn_global_load_lds((GlobalPtr)(a.act + from * kInner + lane * 8),
                                       (LdsPtr)(tile + (4 * i + wave) * kLdsRow), 16, 0, 0);
    }
    const int at = t * 16 + column;
    const int64_t to = static_cast<int64_t>(pair) * a.stride;
    pair = run.pair((t + run.tile_step) * 16 + column);
    __syncthreads();   // waits for every wave's loads
    for (int r = 0; r < a.row_tiles; ++r) {
      const int row0 = first_row + r * kRowsPerBlock;
      u32x4 raw[2][4];
      float factor[2][4][2];
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          raw[sub][i] = *reinterpret_cast<const u32x4*>(wave_codes + (16 * sub + column) * (kInner / 4) +
                                                        ((4 * i + group) ^ column) * 8);
          factor[sub][i][0] = e4m3(scale[sub][i] & 0xFFu);
          factor[sub][i][1] = e4m3(scale[sub][i] >> 8);
        }
      }
      // The wave's own reads are done before its piece is written again.
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
      __builtin_amdgcn_sched_barrier(0);
      const bool last = r + 1 == a.row_tiles;
      if (!last || t + run.tile_step < tiles) {
        const int next = last ? first_row : row0 + kRowsPerBlock;
        load_codes(next);
        load_scales(next);
      }
      f32x4 sum[2] = {f32x4{}, f32x4{}};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {   // 8 codes each; a scale covers 16
          const bf16x8 x = *reinterpret_cast<const bf16x8*>(tile + column * kLdsRow + (4 * i + group) * 32 + j * 8);
#pragma unroll
          for (int sub = 0; sub < 2; ++sub) {
            sum[sub] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(decode(raw[sub][i][j], factor[sub][i][j / 2]), x,
                                                               sum[sub], 0, 0, 0);
          }
        }
      }
      const int n = row0 + 4 * group;   // four rows of token `column`, of either operand
      if (at < run.count) {
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
          if (n + 16 * sub < a.hidden) {   // the stride covers a short tail
            uint2 packed;
            packed.x = pack_bf16(sum[sub][0], sum[sub][1]);
            packed.y = pack_bf16(sum[sub][2], sum[sub][3]);
            *reinterpret_cast<uint2*>(a.d + to + n + 16 * sub) = packed;
          }
        }
      }
      // The next tile's codes have arrived before they are read.
      __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();   // the tile is read before the next one arrives
  }
}

// More tokens per expert: the matrix cores and the decoding are the bound. A wave decodes 32
// rows from registers, step by step, against 64 tokens in LDS: a step's 16 vector
// instructions and its two 32x32x16 MFMAs take as long. Lane half h takes chunk 2 i + h.
__global__ __launch_bounds__(kThreads, 2) void grouped_down_wide_kernel(GroupedArgs a) {
  constexpr int kTile = 64;
  typedef float f32x16 __attribute__((ext_vector_type(16)));
  __shared__ __attribute__((aligned(16))) uint16_t tile[kTile * kLdsRow];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  const int column = lane % 32, half = lane / 32;
  const Run run = run_of(a, blockIdx.y);
  const int tiles = (run.count + kTile - 1) / kTile;
  if (run.first_tile >= tiles) return;   // the same for the whole workgroup
  const int row0 = blockIdx.x * kRowsPerBlock + wave * 32;
  const int64_t at_row = static_cast<int64_t>(min(row0 + column, a.hidden - 1)) * kChunks + half;
  int pair = run.pair(run.first_tile * kTile + lane);
  u32x4 raw[8];
  uint32_t scale[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    raw[i] = run.codes[at_row + 2 * i];
    scale[i] = run.scales[at_row + 2 * i];
  }
  for (int t = run.first_tile; t < tiles; t += run.tile_step) {
#pragma unroll
    for (int i = 0; i < kTile / kWaves; ++i) {
      const int64_t from = of_lane(pair, kWaves * i + wave);
      __builtin_amdgcn_global_load_lds((GlobalPtr)(a.act + from * kInner + lane * 8),
                                       (LdsPtr)(tile + (kWaves * i + wave) * kLdsRow), 16, 0, 0);
    }
    const int here = pair;
    pair = run.pair((t + run.tile_step) * kTile + lane);
    __syncthreads();   // waits for every wave's loads
    f32x16 sum[2] = {f32x16{}, f32x16{}};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float low = e4m3(scale[i] & 0xFFu), high = e4m3(scale[i] >> 8);
#pragma unroll
      for (int j = 0; j < 4; ++j) {   // 8 codes each; a scale covers 16
        const bf16x8 w = decode(raw[i][j], j < 2 ? low : high);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const bf16x8 x =
              *reinterpret_cast<const bf16x8*>(tile + (c * 32 + column) * kLdsRow + (2 * i + half) * 32 + j * 8);
          sum[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, sum[c], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int at = t * kTile + c * 32 + column;
      const int n = row0 + 4 * half;   // of token `column`, four rows and every eighth four after
      uint16_t* to = a.d + static_cast<int64_t>(__shfl(here, c * 32 + column, kWave)) * a.stride + n;
      if (at < run.count) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (n + 8 * q < a.hidden) {   // the stride covers a short tail
            uint2 packed;
            packed.x = pack_bf16(sum[c][4 * q], sum[c][4 * q + 1]);
            packed.y = pack_bf16(sum[c][4 * q + 2], sum[c][4 * q + 3]);
            *reinterpret_cast<uint2*>(to + 8 * q) = packed;
          }
        }
      }
    }
    __syncthreads();   // the tile is read before the next one arrives
  }
}

// V output columns per thread (8, or 1 where rows of out and residual are not 16-byte
// vectors).
template <int V>
__global__ __launch_bounds__(256) void grouped_combine_kernel(const uint16_t* d, const int32_t* chosen,
                                                              const float* weights, const uint16_t* residual,
                                                              uint16_t* out, int tokens, int top_k, int hidden,
                                                              int stride, int64_t experts) {
  const int per_token = hidden / V;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t token = item / per_token;
  if (token >= tokens) return;
  const int n = static_cast<int>(item % per_token) * V;
  const uint16_t* rows = d + token * (top_k + 1) * stride + n;
  auto load = [&](const uint16_t* at, float (&v)[V]) {
    if constexpr (V == 8) {
      unpack8(*reinterpret_cast<const u32x4*>(at), v);
    } else {
      v[0] = bf16_to_f32(*at);
    }
  };
  float total[V];
#pragma unroll
  for (int i = 0; i < V; ++i) total[i] = 0.0f;
#pragma unroll 4
  for (int j = 0; j < top_k; ++j) {
    const int64_t pair = token * top_k + j;
    const int id = chosen[pair];
    const float weight = round_bf16(weights[pair]);
    const bool valid = id >= 0 && id < experts;
    float v[V];
    load(rows + static_cast<int64_t>(j) * stride, v);
#pragma unroll
    for (int i = 0; i < V; ++i) total[i] = round_bf16(round_bf16((valid ? v[i] : 0.0f) * weight) + total[i]);
  }
  float last[V], joined[V];
  load(rows + static_cast<int64_t>(top_k) * stride, last);
  load(residual + token * hidden + n, joined);
#pragma unroll
  for (int i = 0; i < V; ++i) joined[i] = joined[i] + round_bf16(total[i] + last[i]);
  if constexpr (V == 8) {
    *reinterpret_cast<u32x4*>(out + token * hidden + n) = pack8(joined);
  } else {
    out[token * hidden + n] = f32_to_bf16(joined[0]);
  }
}

int64_t row_stride(int64_t hidden) { return (hidden + 7) / 8 * 8; }

// Tokens of one pass: their d fits the scratch.
int64_t pass_tokens(int64_t hidden, int64_t tokens, int64_t top_k) {
  const int64_t most = kScratchBytes / ((top_k + 1) * row_stride(hidden) * 2);
  return most < tokens ? (most < 1 ? 1 : most) : tokens;
}

// What either form takes the device, in us, as fitted to 16 to 512 experts, top-1 to top-31,
// hidden 1024 and 2048 and 100 thousand to a million rows of slots (tokens x (top_k + 1) x
// hidden) in a graph: within 9% of the per-token kernel's times and, but for a few, 8% of
// these kernels'. The per-token kernel takes so long per row of a slot, less with few waves
// or whole groups of them a workgroup (3, 8, 16 slots), more where the matrices of the chosen
// experts outgrow the L2s. This one reads each of those matrices once.
// Top-7 of 16 experts, hidden 1024: 22.0 against 18.3 us at 38 tokens, 16.2 against 16.7 at
// 25; top-10 of 512, hidden 2048: 37 against 43 at 19, 55 against 53 at 30; top-31 of 512: 54
// against 73 at 13.
double chosen_rows(int64_t experts, int64_t hidden, int64_t tokens, int64_t top_k) {
  const double share = static_cast<double>(tokens) * top_k / experts;
  return experts * -std::expm1(-share) * hidden;   // as many experts as routes drawn evenly choose
}

double per_token_us(int64_t experts, int64_t hidden, int64_t tokens, int64_t top_k) {
  const bool far = chosen_rows(experts, hidden, tokens, top_k) > 80e3;   // 23 MB of codes and scales
  const double ps = top_k < 3 ? (far ? 49 : 45) : top_k < 8 ? (far ? 59 : 50) : top_k < 16 ? (far ? 68 : 57) : far ? 57 : 52;
  return 6.5 + ps * 1e-6 * (static_cast<double>(tokens) * (top_k + 1) * hidden);
}

double grouped_us(int64_t experts, int64_t hidden, int64_t tokens, int64_t top_k) {
  return 12.5 + 0.5 * top_k + 0.0135 * experts + 52.5e-6 * chosen_rows(experts, hidden, tokens, top_k) +
         5e-6 * (static_cast<double>(tokens) * (top_k + 1) * hidden);
}

int64_t plan_bytes(int64_t experts, int64_t pairs) {
  return ((experts + 1 + pairs) * 4 + 15) / 16 * 16;
}

}  // namespace
}  // namespace omnia

extern "C" int64_t omnia_moe_nvfp4_shared_workspace_bytes(int64_t experts, int64_t hidden, int64_t inner,
                                                          int64_t tokens, int64_t top_k) {
  using namespace omnia;
  if (experts <= 0 || hidden <= 0 || inner <= 0 || tokens < 0 || top_k < 0) return -EINVAL;
  // The grouped form takes the packed form's own contraction, and grids that a launch holds.
  if (inner != kInner || tokens > 65535 || top_k < 1 || top_k > 31 || experts > 16384 ||
      hidden >= (int64_t{1} << 24)) {
    return 0;
  }
  if (per_token_us(experts, hidden, tokens, top_k) < grouped_us(experts, hidden, tokens, top_k)) return 0;
  const int64_t pass = pass_tokens(hidden, tokens, top_k);
  return plan_bytes(experts, pass * top_k) + pass * (top_k + 1) * row_stride(hidden) * 2;
}

extern "C" int64_t omnia_moe_nvfp4_shared_per_token_ns(int64_t experts, int64_t hidden, int64_t tokens,
                                                       int64_t top_k) {
  using namespace omnia;
  if (experts <= 0 || hidden <= 0 || tokens < 0 || top_k < 0) return -EINVAL;
  return static_cast<int64_t>(1e3 * per_token_us(experts, hidden, tokens, top_k));
}

extern "C" int32_t omnia_moe_down_combine_nvfp4_shared_grouped(
    const uint16_t* act, const uint32_t* weight, const uint8_t* scales, int64_t experts,
    const uint32_t* shared_weight, const uint8_t* shared_scales, int64_t hidden, int64_t inner,
    const int32_t* chosen, const float* weights, int64_t tokens, int64_t top_k, const uint16_t* residual,
    void* workspace, int64_t workspace_bytes, uint16_t* out, hipStream_t stream) {
  using namespace omnia;
  const int64_t need = omnia_moe_nvfp4_shared_workspace_bytes(experts, hidden, inner, tokens, top_k);
  OMNIA_REQUIRE(need >= 0, "moe_down_combine_nvfp4_shared_grouped: bad geometry");
  if (need == 0) {   // too few tokens, or a shape of the per-token kernel's only
    return omnia_moe_down_combine_nvfp4_shared(act, weight, scales, experts, shared_weight, shared_scales, hidden,
                                               inner, chosen, weights, tokens, top_k, residual, out, stream);
  }
  OMNIA_REQUIRE(act && weight && scales && shared_weight && shared_scales && chosen && weights && residual && out,
                "moe_down_combine_nvfp4_shared_grouped: null pointer");
  OMNIA_REQUIRE(workspace && workspace_bytes >= need && aligned16(workspace),
                "moe_down_combine_nvfp4_shared_grouped: workspace too small or not 16-byte aligned");
  OMNIA_REQUIRE(aligned16(act) && aligned16(weight) && aligned16(shared_weight),
                "moe_down_combine_nvfp4_shared_grouped: act and the weights must be 16-byte aligned");
  OMNIA_REQUIRE(reinterpret_cast<uintptr_t>(scales) % 2 == 0 && reinterpret_cast<uintptr_t>(shared_scales) % 2 == 0,
                "moe_down_combine_nvfp4_shared_grouped: the scales must be 2-byte aligned");
  int32_t rc = check_device(stream);
  if (rc != 0) return rc;
  const int64_t pass = pass_tokens(hidden, tokens, top_k);
  int32_t* offsets = static_cast<int32_t*>(workspace);
  int32_t* entries = offsets + experts + 1;
  uint16_t* d = reinterpret_cast<uint16_t*>(static_cast<char*>(workspace) + plan_bytes(experts, pass * top_k));
  const int stride = static_cast<int>(row_stride(hidden));
  const bool vectors = hidden % 8 == 0 && aligned16(residual) && aligned16(out);
  for (int64_t first = 0; first < tokens; first += pass) {
    const int64_t now = tokens - first < pass ? tokens - first : pass;
    const int pairs = static_cast<int>(now * top_k);
    const int32_t* ids = chosen + first * top_k;
    expert_plan_kernel<<<dim3(static_cast<unsigned>(experts)), kPlanThreads, 0, stream>>>(
        ids, pairs, static_cast<int>(experts), offsets, entries);
    // The wide kernel from 13 pairs per expert on average: 64 experts, hidden 1504, top-6: 26.6
    // against 26.9 us at 12, 34.7 against 28.7 at 24; 128 experts, hidden 2048, top-8: 32.9
    // against 46.3 at 8, 69.0 against 52.4 at 32. As many workgroups per expert as its average
    // run has tiles.
    const bool wide = pairs / experts > 12;
    const int64_t run = wide ? 64 : 16;
    const int64_t shared_blocks = (now + run - 1) / run;
    int64_t splits = (pairs / experts + run - 1) / run;
    if (splits < 1 || shared_blocks + experts * splits > 65535) splits = 1;
    // Two row tiles a workgroup where that leaves enough of them: 512 experts 102.6 -> 97.2
    // us at 512 tokens, but 128 experts 31.5 -> 32.9 at 128.
    const int64_t row_blocks = (hidden + kRowsPerBlock - 1) / kRowsPerBlock;
    const int row_tiles = !wide && row_blocks * (shared_blocks + experts * splits) >= 4096 ? 2 : 1;
    GroupedArgs a{act + first * (top_k + 1) * kInner, reinterpret_cast<const u32x4*>(weight),
                  reinterpret_cast<const uint16_t*>(scales), reinterpret_cast<const u32x4*>(shared_weight),
                  reinterpret_cast<const uint16_t*>(shared_scales), offsets, entries, d, static_cast<int>(now),
                  static_cast<int>(top_k), static_cast<int>(hidden), stride, static_cast<int>(shared_blocks),
                  static_cast<int>(splits), row_tiles};
    const int64_t rows = static_cast<int64_t>(a.row_tiles) * kRowsPerBlock;
    const dim3 tiles(static_cast<unsigned>((hidden + rows - 1) / rows),
                     static_cast<unsigned>(shared_blocks + experts * splits));
    if (wide) {
      grouped_down_wide_kernel<<<tiles, kThreads, 0, stream>>>(a);
    } else {
      grouped_down_kernel<<<tiles, kThreads, 0, stream>>>(a);
    }
    const int64_t items = now * (vectors ? hidden / 8 : hidden);
    const dim3 grid(static_cast<unsigned>((items + 255) / 256));
    if (vectors) {
      grouped_combine_kernel<8><<<grid, 256, 0, stream>>>(d, ids, weights + first * top_k, residual + first * hidden,
                                                          out + first * hidden, static_cast<int>(now),
                                                          static_cast<int>(top_k), static_cast<int>(hidden), stride,
                                                          experts);
    } else {
      grouped_combine_kernel<1><<<grid, 256, 0, stream>>>(d, ids, weights + first * top_k, residual + first * hidden,
                                                          out + first * hidden, static_cast<int>(now),
                                                          static_cast<int>(top_k), static_cast<int>(hidden), stride,
                                                          experts);
    }
  }
  return launched("moe_down_combine_nvfp4_shared_grouped");
}
