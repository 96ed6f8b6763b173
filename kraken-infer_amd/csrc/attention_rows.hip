// Decode attention over several query tokens of one sequence (a prompt's last
// chunk of up to 63 tokens, drafted tokens to verify): head_dim 256, f16 cache,
// up to 4 query heads per KV head.  Semantics as attention_decode.hip
// (mps_backend.mm:2943-3008): f32 query, token t attends keys 0 .. start + t.
//
// One workgroup per token read the whole K/V stream again for each of them.  Here
// the 16 columns of the S^T = K Q^T tile are 16 query rows: 16 / G consecutive
// tokens x G heads.  A workgroup owns one such row group, one KV head and one key
// split; its four waves take the split's 16-key tiles w, w + 4, ...  As in
// attention_decode_mfma_kernel: each wave copies its tiles straight into two LDS
// stages of its own, query and probabilities are split into f16 hi + lo, the S^T
// accumulator is the A operand of O += P V, V^T comes through the transposing LDS
// read, the denominator is compensated.  Every lane has scores of its own
// column here, with the column's own causal limit and reference max; a rescale
// of O (rare: the max moves only by more than 2^8) fetches the rows' factors from
// the lanes of their columns.
//
// A tile is 48 MFMAs and about 270 other instructions; what bounded the first
// form was the wait for each of its 24 LDS reads in turn (1.6 us a tile).  All of
// a tile's K fragments are requested before the first is used, and all of its V
// fragments before the softmax: 37 tokens after 6144 keys (8 / 2 heads, with
// prologue and merge) 33.4 -> 25.8 us, from 59.7 with one workgroup per token.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "attention_decode_internal.hpp"
#include "device_common.hpp"

namespace kraken {
namespace decode {
namespace {

constexpr int kWaves = 4;
constexpr int kStages = 2;            // tiles in flight per wave
constexpr int kOStride = kMD + 4;     // floats: the four row groups of a store hit 16 banks each

template <int G>
__global__ __launch_bounds__(64 * kWaves) void attention_rows_kernel(DecodeParams p) {
  constexpr uint32_t kTokens = kRowsPerGroup / G;
  constexpr int kRows = kRowsPerGroup;
  __shared__ __attribute__((aligned(16))) half_t s_kv[kWaves][kStages][2][kMTileHalfs];
  __shared__ float s_m[kWaves][kRows];
  __shared__ float s_l[kWaves][kRows];
  static_assert(sizeof(float) * kWaves * kRows * kOStride <= sizeof(s_kv), "merge area");
  float(*s_o)[kRows][kOStride] = reinterpret_cast<float(*)[kRows][kOStride]>(&s_kv[0][0][0][0]);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15;
  const int kq = lane >> 4;
  const uint32_t groups = (p.tokens + kTokens - 1u) / kTokens;
  const RowsPlace at_grid = place_rows(p.splits * p.kv_heads, groups);
  const uint32_t split = at_grid.unit / p.kv_heads;
  const uint32_t kvh = at_grid.unit % p.kv_heads;
  const uint32_t first_token = at_grid.order * kTokens;
  const uint32_t last_token = min(first_token + kTokens, p.tokens) - 1u;
  const uint32_t key_begin = split * p.keys_per_split;
  const uint32_t most_keys = p.start_position + last_token + 1u;
  if (key_begin >= most_keys) {
    return;  // empty split (whole workgroup)
  }
  const uint32_t count = min(most_keys, key_begin + p.keys_per_split) - key_begin;

  const size_t row_stride = (size_t)p.kv_heads * kMD;
  const uint32_t row_bytes = (uint32_t)(row_stride * sizeof(half_t));
  const uint64_t first_elem = ((uint64_t)p.layer * p.capacity_tokens + key_begin) * row_stride +
                              (uint64_t)kvh * kMD;
  const i32x4_t krs =
    rsrc_words(static_cast<const half_t*>(p.key_cache) + first_elem, count * row_bytes);
  const i32x4_t vrs =
    rsrc_words(static_cast<const half_t*>(p.value_cache) + first_elem, count * row_bytes);

  // Copies tile t of K and V into stage st of this wave (as attention_decode.hip);
  // rows at or past the split's end read as zeros.
  const uint32_t copy_row = (uint32_t)(lane >> 5);
  const uint32_t chunk = (uint32_t)(lane & 31);
  auto issue_tile = [&](uint32_t t, int st) __attribute__((always_inline)) {
    half_t* kdst = &s_kv[wave][st][0][0];
    half_t* vdst = &s_kv[wave][st][1][0];
#pragma unroll
    for (int c = 0; c < kMTile / 2; ++c) {
      const uint32_t row = 2u * c + copy_row;
      const uint32_t base = (kMTile * t + row) * row_bytes;
      copy16_to_lds(krs, base + 16u * (chunk ^ (row & 7u)), kdst + c * 2 * kMD);
      copy16_to_lds(vrs, base + 16u * (chunk ^ (2u * (row & 3u))), vdst + c * 2 * kMD);
    }
  };
  issue_tile((uint32_t)wave, 0);
  issue_tile((uint32_t)wave + kWaves, 1);

  // Column r16: token first_token + r16 / G, head kvh G + r16 % G; `limit` counts
  // its visible keys in the split (none for a column past the tokens).
  const uint32_t token = first_token + (uint32_t)r16 / G;
  const uint32_t keys = p.start_position + token + 1u;
  const uint32_t limit = token < p.tokens && keys > key_begin ? min(keys - key_begin, count) : 0u;
  // The keys from the split's first that the first token sees (negative before
  // them); token j after it sees j more.
  const int64_t first_seen = (int64_t)p.start_position + first_token + 1 - (int64_t)key_begin;
  half8_t qhi[8], qlo[8];
  {
    const float* qh =
      p.query + ((size_t)min(token, last_token) * p.heads + kvh * G + r16 % G) * kMD + 8 * kq;
    float4 raw[8][2];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      raw[s][0] = *reinterpret_cast<const float4*>(qh + 32 * s);
      raw[s][1] = *reinterpret_cast<const float4*>(qh + 32 * s + 4);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const float4 a = raw[s][0];
      const float4 b = raw[s][1];
      const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        half_t hi, lo;
        split_f16(v[j] * p.scale_log2, hi, lo);
        qhi[s][j] = hi;
        qlo[s][j] = lo;
      }
    }
  }

  float m = -INFINITY;  // reference max of this lane's column (log2 domain)
  float lpart = 0.0f, lcomp = 0.0f;
  float4v_t o[16], olo[16];
#pragma unroll
  for (int d = 0; d < 16; ++d) {
    o[d] = float4v_t{0.f, 0.f, 0.f, 0.f};
    olo[d] = float4v_t{0.f, 0.f, 0.f, 0.f};
  }
  const int vrow = 4 * kq + (r16 >> 2);
  const int vq = r16 & 3;
  const int vswz = 2 * (vrow & 3);

  const uint32_t ntiles = (count + kMTile - 1) / kMTile;
  // One tile; kDiagonal: some of its keys are not the group's first token's.
  auto tile = [&](uint32_t t, int st, auto diagonal) __attribute__((always_inline)) {
    constexpr bool kDiagonal = decltype(diagonal)::value;
    // Stage st holds tile t once only the other stage's copies are in flight.
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kMTile) : "memory");
    const half_t* ks = &s_kv[wave][st][0][0] + r16 * kMD;
    const half_t* vs = &s_kv[wave][st][1][0] + vrow * kMD + 4 * (vq & 1);
    half8_t kf[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      kf[s] = *reinterpret_cast<const half8_t*>(ks + 8 * ((4 * s + kq) ^ (r16 & 7)));
    }
    __builtin_amdgcn_sched_barrier(0);
    float4v_t shi = {0.f, 0.f, 0.f, 0.f};
    float4v_t slo = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      shi = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[s], qhi[s], shi, 0, 0, 0);
      slo = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[s], qlo[s], slo, 0, 0, 0);
    }
    half4_t vf[16];
#pragma unroll
    for (int d = 0; d < 16; ++d) {
      vf[d] = read_tr16(vs + 8 * ((2 * d + (vq >> 1)) ^ vswz));
    }
    __builtin_amdgcn_sched_barrier(0);

    // Softmax: the lane holds keys 16 t + 4 kq + r of its column.
    float sc[4];
    bool valid[4];
    float cmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      valid[r] = kMTile * t + 4u * kq + r < limit;
      sc[r] = valid[r] ? fmaf(slo[r], kLoUnscale, shi[r]) : -INFINITY;
      cmax = fmaxf(cmax, sc[r]);
    }
    cmax = xor32_max(xor16_max(cmax));
    const bool moves = cmax > m + kRescaleSlack;
    if (__builtin_amdgcn_ballot_w64(moves) != 0) {
      // 0 on the column's first visible tile; a column that stays keeps 1.
      const float corr = moves ? fast_exp2(m - cmax) : 1.0f;
      m = moves ? cmax : m;
      lpart *= corr;
      lcomp *= corr;
      float f[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        f[r] = __shfl(corr, 4 * kq + r, 64);
      }
#pragma unroll
      for (int d = 0; d < 16; ++d) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          o[d][r] *= f[r];
          olo[d][r] *= f[r];
        }
      }
    }
    half4_t phi, plo;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float pr = valid[r] ? fast_exp2(sc[r] - m) : 0.0f;
      kahan_add(lpart, lcomp, pr);
      half_t h, l;
      split_f16(pr, h, l);
      phi[r] = h;
      plo[r] = l;
    }
    // The V reads above have returned by the time their values are used; the
    // stage is free for tile t + 8 then.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    issue_tile(t + kStages * kWaves, st);
    // A NaN or an infinity in a later token's value row must not reach an earlier
    // one through 0 x V.
    bool per_token = false;
    if constexpr (kDiagonal) {
      bool bad = false;
#pragma unroll
      for (int d = 0; d < 16; ++d) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          bad |= !(__builtin_fabsf(static_cast<float>(vf[d][r])) < INFINITY);
        }
      }
      per_token = __builtin_amdgcn_ballot_w64(bad) != 0;
    }
    if (!per_token) {
#pragma unroll
      for (int d = 0; d < 16; ++d) {
        o[d] = __builtin_amdgcn_mfma_f32_16x16x16f16(phi, vf[d], o[d], 0, 0, 0);
        olo[d] = __builtin_amdgcn_mfma_f32_16x16x16f16(plo, vf[d], olo[d], 0, 0, 0);
      }
    } else {
      // One token at a time against the values that it sees, kept for its rows.
      const float4v_t none = {0.f, 0.f, 0.f, 0.f};
      for (uint32_t j = 0; j < kTokens; ++j) {
#pragma unroll
        for (int d = 0; d < 16; ++d) {
          half4_t v = vf[d];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v[r] = (int64_t)(kMTile * t + 4u * kq + r) < first_seen + j ? v[r] : static_cast<half_t>(0.0f);
          }
          const float4v_t hi = __builtin_amdgcn_mfma_f32_16x16x16f16(phi, v, none, 0, 0, 0);
          const float4v_t lo = __builtin_amdgcn_mfma_f32_16x16x16f16(plo, v, none, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool own = (4u * kq + r) / G == j;
            o[d][r] = own ? o[d][r] + hi[r] : o[d][r];
            olo[d][r] = own ? olo[d][r] + lo[r] : olo[d][r];
          }
        }
      }
    }
  };
  uint32_t t = (uint32_t)wave;
  int st = 0;
  for (; t < ntiles && (int64_t)(kMTile * (t + 1u)) <= first_seen; t += kWaves, st ^= 1) {
    tile(t, st, std::false_type{});
  }
  for (; t < ntiles; t += kWaves, st ^= 1) {
    tile(t, st, std::true_type{});
  }
  // No copy may land in a stage after the stages are reused below.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();  // every wave is done with its stages
  const float lw = xor32_sum(xor16_sum(lpart - lcomp));
  if (lane < 16) {
    s_m[wave][lane] = m;
    s_l[wave][lane] = lw;
  }
#pragma unroll
  for (int d = 0; d < 16; ++d) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s_o[wave][4 * kq + r][16 * d + r16] = fmaf(olo[d][r], kLoUnscale, o[d][r]);
    }
  }
  __syncthreads();

  // Workgroup merge of the wave partials: wave w takes rows 4 w .. 4 w + 3, a
  // lane the dims lane + 64 j.  A row is written if its token exists and has keys
  // in this split.
  constexpr int kR = kRows / kWaves;
  constexpr int kJ = kMD / 64;
  float acc[kR][kJ], den[kR], mx[kR];
  uint32_t tk[kR];
  bool live[kR];
#pragma unroll
  for (int i = 0; i < kR; ++i) {
    const int row = kR * wave + i;
    tk[i] = first_token + (uint32_t)row / G;
    live[i] = tk[i] <= last_token && p.start_position + tk[i] + 1u > key_begin;
    mx[i] = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      mx[i] = fmaxf(mx[i], s_m[w][row]);
    }
    den[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      acc[i][j] = 0.0f;
    }
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float wt = s_m[w][row] == -INFINITY ? 0.0f : fast_exp2(s_m[w][row] - mx[i]);
      den[i] = fmaf(wt, s_l[w][row], den[i]);
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        acc[i][j] = fmaf(wt, s_o[w][row][lane + 64 * j], acc[i][j]);
      }
    }
  }
  if (p.splits != 1) {
#pragma unroll
    for (int i = 0; i < kR; ++i) {
      if (live[i]) {
        const int g = (kR * wave + i) % G;
        const size_t at = ((size_t)tk[i] * p.kv_heads + kvh) * p.splits + split;
#pragma unroll
        for (int j = 0; j < kJ; ++j) {
          store_through(&p.part_o[(at * G + g) * kMD + lane + 64 * j], acc[i][j]);
        }
        if (lane == 0) {
          store_through(&p.part_ml[(at * G + g) * 2 + 0], mx[i]);
          store_through(&p.part_ml[(at * G + g) * 2 + 1], den[i]);
        }
      }
    }
    return;
  }
  // One split: the output itself, all of its gate values requested first.
  float gate[kR][kJ];
#pragma unroll
  for (int i = 0; i < kR; ++i) {
    const size_t at =
      ((size_t)min(tk[i], last_token) * p.heads + kvh * G + (kR * wave + i) % G) * kMD + lane;
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      gate[i][j] = p.gate != nullptr ? p.gate[at + 64 * j] : 0.0f;
    }
  }
#pragma unroll
  for (int i = 0; i < kR; ++i) {
    if (live[i]) {
      const size_t at =
        ((size_t)tk[i] * p.heads + kvh * G + (kR * wave + i) % G) * kMD + lane;
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        float r = den[i] == 0.0f ? 0.0f : acc[i][j] / den[i];
        if (p.gate != nullptr) {
          r *= sigmoidf_acc(gate[i][j]);
        }
        p.output[at + 64 * j] = r;
      }
    }
  }
}

}  // namespace

hipError_t launch_decode_rows(const DecodeParams& p, uint32_t group, hipStream_t stream) {
  const uint32_t tokens = kRowsPerGroup / group;
  const uint32_t groups = (p.tokens + tokens - 1u) / tokens;
  const dim3 grid = rows_grid(p.splits * p.kv_heads, groups);
  switch (group) {
    case 1: attention_rows_kernel<1><<<grid, 64 * kWaves, 0, stream>>>(p); break;
    case 2: attention_rows_kernel<2><<<grid, 64 * kWaves, 0, stream>>>(p); break;
    case 4: attention_rows_kernel<4><<<grid, 64 * kWaves, 0, stream>>>(p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace decode
}  // namespace kraken
