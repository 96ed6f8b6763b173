// Causal attention of several query tokens over an F32 cache (the legacy layer's
// prefill chunk and its tail): semantics of attention_f32_batched
// (mps_backend.mm:2879-2941), head_dim 64 or 128, 1, 2, 4 or 8 query heads per KV
// head, every product in f32 on v_mfma_f32_16x16x4_f32.
//
// One workgroup per token read its whole K/V range for one token's heads: 512
// tokens (16 / 8 heads of 128) read 1 GB through the caches in 67 us.  Here a
// workgroup owns 16 query rows (16 / G consecutive tokens x G heads), a KV head
// and a key split; its four waves take the split's 16-key tiles w, w + 4, ...
//  * S^T = K Q^T: the MFMA's k index kq of step 4 j + e stands for dim
//    16 j + 4 kq + e, so that a lane's operands are float4s of its key's (or query
//    row's) row and the four lanes of a row load 64 consecutive bytes.
//  * The accumulator (lane: row l % 16, keys 4 (l / 16) + r) is the A operand of
//    O += P V for step r as it is.  O's tile n holds dim 64 (n / 4) + 4 (l % 16) +
//    n % 4, so a lane's V operands are float4s too, 256 consecutive bytes per key.
//  * No operand goes through LDS; the next tile's loads are in flight while a tile
//    computes (range-checked buffer loads: rows past the split read zeros).
// A 16 x 16 tile is D / 4 MFMAs for K Q^T and D / 4 for P V, of 32 cycles each; what
// bounds the 512-token chunk is that rate (1.1 GFLOP, 7 us at the card's f32 matrix
// peak) and the causal imbalance, so a heavy row group and a light one share a CU:
// 67.1 -> 22.1 us as a node of a graph, 168 -> 41.9 us after 500 tokens.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "attention_decode_internal.hpp"
#include "device_common.hpp"

namespace kraken {
namespace decode {
namespace {

constexpr int kWaves = 4;
constexpr int kTile = 16;

__device__ __forceinline__ float at4(const float4& v, int e) {
  return e == 0 ? v.x : (e == 1 ? v.y : (e == 2 ? v.z : v.w));
}

template <int D, int G>
__global__ __launch_bounds__(64 * kWaves, 2) void attention_rows_f32_kernel(DecodeParams p) {
  constexpr uint32_t kTokens = kRowsPerGroup / G;
  constexpr int kRows = kRowsPerGroup;
  constexpr int KJ = D / 16;  // float4s of a lane's K (or query) operands
  constexpr int VH = D / 64;  // float4s of a lane's V operands per key
  constexpr int kStride = D + 4;
  __shared__ float s_m[kWaves][kRows];
  __shared__ float s_l[kWaves][kRows];
  __shared__ __attribute__((aligned(16))) float s_o[kWaves][kRows][kStride];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15;
  const int kq = lane >> 4;
  // The row groups run from the last to the middle, then from the first: the two
  // workgroups of a CU (half the grid apart) add up to about the same number of keys.
  const uint32_t groups = (p.tokens + kTokens - 1u) / kTokens;
  const RowsPlace at_grid = place_rows(p.splits * p.kv_heads, groups);
  const uint32_t order = at_grid.order, half = groups / 2u;
  const uint32_t group = order < groups - half ? groups - 1u - order : order - (groups - half);
  const uint32_t split = at_grid.unit / p.kv_heads;
  const uint32_t kvh = at_grid.unit % p.kv_heads;
  const uint32_t first_token = group * kTokens;
  const uint32_t last_token = min(first_token + kTokens, p.tokens) - 1u;
  const uint32_t key_begin = split * p.keys_per_split;
  const uint32_t most_keys = p.start_position + last_token + 1u;
  if (key_begin >= most_keys) {
    return;  // empty split (whole workgroup)
  }
  const uint32_t count = min(most_keys, key_begin + p.keys_per_split) - key_begin;

  const size_t row_stride = (size_t)p.kv_heads * D;
  const uint32_t row_bytes = (uint32_t)(row_stride * sizeof(float));
  const uint64_t first_elem =
    ((uint64_t)p.layer * p.capacity_tokens + key_begin) * row_stride + (uint64_t)kvh * D;
  const __amdgpu_buffer_rsrc_t krs =
    make_buffer_rsrc(static_cast<const float*>(p.key_cache) + first_elem, count * row_bytes);
  const __amdgpu_buffer_rsrc_t vrs =
    make_buffer_rsrc(static_cast<const float*>(p.value_cache) + first_elem, count * row_bytes);

  const uint32_t token = first_token + (uint32_t)r16 / G;
  const uint32_t keys = p.start_position + token + 1u;
  const uint32_t limit = token < p.tokens && keys > key_begin ? min(keys - key_begin, count) : 0u;
  // The keys from the split's first that the first token sees (negative before
  // them); token j after it sees j more.
  const int64_t first_seen = (int64_t)p.start_position + first_token + 1 - (int64_t)key_begin;

  struct Tile {
    float4 k[KJ], v[4][VH];
  };
  auto load_tile = [&](uint32_t t, Tile& x) __attribute__((always_inline)) {
    const uint32_t krow = (kTile * t + (uint32_t)r16) * row_bytes + 16u * kq;
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      x.k[j] = __builtin_bit_cast(
        float4, __builtin_amdgcn_raw_buffer_load_b128(krs, (int)(krow + 64u * j), 0, 0));
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t vrow = (kTile * t + 4u * kq + r) * row_bytes + 16u * r16;
#pragma unroll
      for (int h = 0; h < VH; ++h) {
        x.v[r][h] = __builtin_bit_cast(
          float4, __builtin_amdgcn_raw_buffer_load_b128(vrs, (int)(vrow + 256u * h), 0, 0));
      }
    }
  };
  float4 q[KJ];
  {
    const float* qh =
      p.query + ((size_t)min(token, last_token) * p.heads + kvh * G + r16 % G) * D + 4 * kq;
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      q[j] = *reinterpret_cast<const float4*>(qh + 16 * j);
    }
  }
  Tile x[2];
  load_tile((uint32_t)wave, x[0]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < KJ; ++j) {
    q[j] = make_float4(q[j].x * p.scale_log2, q[j].y * p.scale_log2, q[j].z * p.scale_log2,
                       q[j].w * p.scale_log2);
  }

  float m = -INFINITY;  // reference max of this lane's column (log2 domain)
  float lpart = 0.0f, lcomp = 0.0f;
  float4v_t o[4 * VH];
#pragma unroll
  for (int n = 0; n < 4 * VH; ++n) {
    o[n] = float4v_t{0.f, 0.f, 0.f, 0.f};
  }

  auto compute = [&](uint32_t t, const Tile& c) __attribute__((always_inline)) {
    // Four chains of D / 32 steps, twice, added in pairs: short sums, so that the
    // scores are as exact as the one-token kernel's.
    float4v_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      float4v_t s[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[e] = float4v_t{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int j = part * KJ / 2; j < (part + 1) * KJ / 2; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(at4(c.k[j], e), at4(q[j], e), s[e], 0, 0, 0);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sum[r] += (s[0][r] + s[1][r]) + (s[2][r] + s[3][r]);
      }
    }
    float sc[4];
    bool valid[4];
    float cmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      valid[r] = kTile * t + 4u * kq + r < limit;
      sc[r] = valid[r] ? sum[r] : -INFINITY;
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
      for (int n = 0; n < 4 * VH; ++n) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          o[n][r] *= f[r];
        }
      }
    }
    float pr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      pr[r] = valid[r] ? fast_exp2(sc[r] - m) : 0.0f;
      kahan_add(lpart, lcomp, pr[r]);
    }
    // A NaN or an infinity in a later token's value row must not reach an earlier
    // one through 0 x V.
    bool per_token = false;
    if ((int64_t)(kTile * (t + 1u)) > first_seen) {  // keys that not all tokens see
      bool bad = false;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int h = 0; h < VH; ++h) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            bad |= !(__builtin_fabsf(at4(c.v[r][h], e)) < INFINITY);
          }
        }
      }
      per_token = __builtin_amdgcn_ballot_w64(bad) != 0;
    }
    if (!per_token) {
      // A tile's 16 products are summed on their own before they join O.
#pragma unroll
      for (int n = 0; n < 4 * VH; ++n) {
        float4v_t part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          part = __builtin_amdgcn_mfma_f32_16x16x4f32(pr[r], at4(c.v[r][n / 4], n % 4), part, 0, 0,
                                                      0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          o[n][r] += part[r];
        }
      }
    } else {
      // One token at a time against the values that it sees, kept for its rows.
      for (uint32_t j = 0; j < kTokens; ++j) {
#pragma unroll
        for (int n = 0; n < 4 * VH; ++n) {
          float4v_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool seen = (int64_t)(kTile * t + 4u * kq + r) < first_seen + j;
            const float v = seen ? at4(c.v[r][n / 4], n % 4) : 0.0f;
            sum = __builtin_amdgcn_mfma_f32_16x16x4f32(pr[r], v, sum, 0, 0, 0);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            o[n][r] = (4u * kq + r) / G == j ? o[n][r] + sum[r] : o[n][r];
          }
        }
      }
    }
  };
  const uint32_t ntiles = (count + kTile - 1) / kTile;
  for (uint32_t t = (uint32_t)wave; t < ntiles; t += 2 * kWaves) {
    load_tile(t + kWaves, x[1]);
    __builtin_amdgcn_sched_barrier(0);
    compute(t, x[0]);
    __builtin_amdgcn_sched_barrier(0);
    load_tile(t + 2 * kWaves, x[0]);
    __builtin_amdgcn_sched_barrier(0);
    if (t + kWaves < ntiles) {
      compute(t + kWaves, x[1]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  const float lw = xor32_sum(xor16_sum(lpart - lcomp));
  if (lane < 16) {
    s_m[wave][lane] = m;
    s_l[wave][lane] = lw;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int h = 0; h < VH; ++h) {
      *reinterpret_cast<float4*>(&s_o[wave][4 * kq + r][64 * h + 4 * r16]) =
        make_float4(o[4 * h][r], o[4 * h + 1][r], o[4 * h + 2][r], o[4 * h + 3][r]);
    }
  }
  __syncthreads();

  // Workgroup merge of the wave partials: wave w takes rows 4 w .. 4 w + 3, a
  // lane the dims lane + 64 j.  A row is written if its token exists and has keys
  // in this split.
  constexpr int kR = kRows / kWaves;
#pragma unroll
  for (int i = 0; i < kR; ++i) {
    const int row = kR * wave + i;
    const uint32_t tk = first_token + (uint32_t)row / G;
    const int g = row % G;
    const bool live = tk <= last_token && p.start_position + tk + 1u > key_begin;
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      mx = fmaxf(mx, s_m[w][row]);
    }
    float wt[kWaves];
    float den = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      wt[w] = s_m[w][row] == -INFINITY ? 0.0f : fast_exp2(s_m[w][row] - mx);
      den = fmaf(wt[w], s_l[w][row], den);
    }
    const size_t at = ((size_t)tk * p.kv_heads + kvh) * p.splits + split;
#pragma unroll
    for (int j = 0; j < VH; ++j) {
      const int d = lane + 64 * j;
      float acc = 0.0f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        acc = fmaf(wt[w], s_o[w][row][d], acc);
      }
      if (live) {
        if (p.splits == 1) {
          write_final<D, G>(p, tk, kvh, g * D + d, den, acc);
        } else {
          store_through(&p.part_o[(at * G + g) * D + d], acc);
        }
      }
    }
    if (live && p.splits != 1 && lane == 0) {
      store_through(&p.part_ml[(at * G + g) * 2 + 0], mx);
      store_through(&p.part_ml[(at * G + g) * 2 + 1], den);
    }
  }
}

template <int D>
hipError_t launch_dim(const DecodeParams& p, uint32_t group, dim3 grid, hipStream_t stream) {
  switch (group) {
    case 1: attention_rows_f32_kernel<D, 1><<<grid, 64 * kWaves, 0, stream>>>(p); break;
    case 2: attention_rows_f32_kernel<D, 2><<<grid, 64 * kWaves, 0, stream>>>(p); break;
    case 4: attention_rows_f32_kernel<D, 4><<<grid, 64 * kWaves, 0, stream>>>(p); break;
    case 8: attention_rows_f32_kernel<D, 8><<<grid, 64 * kWaves, 0, stream>>>(p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_decode_rows_f32(const DecodeParams& p, uint32_t head_dim, uint32_t group,
                                  hipStream_t stream) {
  const uint32_t tokens = kRowsPerGroup / group;
  const uint32_t groups = (p.tokens + tokens - 1u) / tokens;
  const dim3 grid = rows_grid(p.splits * p.kv_heads, groups);
  switch (head_dim) {
    case 64: return launch_dim<64>(p, group, grid, stream);
    case 128: return launch_dim<128>(p, group, grid, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace decode
}  // namespace kraken
