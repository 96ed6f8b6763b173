// The full-attention prologue of run_qwen35_full_attention_layer_chunk
// (qwen35_runtime.cpp:3229-3326) as one kernel:
//   copy_f32_rows x2           split of the joint Q/gate projection
//   qk_norm_f32_f32_batched x2 RMSNorm of q (q_norm) and k (k_norm)
//   mrope_f32_in_place x2      MRoPE of q and k
//   copy_f32_rows_to_f16 x2    K and V rows appended to the F16 cache
// One wave per token and run of head slots: slots 0 .. heads-1 are query heads,
// then the key heads, then the value heads.  The arithmetic is that of
// rms_norm_heads_kernel and mrope_kernel (same element-to-lane layout, same
// reduction order, the angle in double), so the result equals the unfused
// chain's bit for bit.
#include <hip/hip_runtime.h>

#include "attention_prologue_common.hpp"
#include "context_internal.hpp"
#include "device_common.hpp"

namespace kraken {
namespace {

constexpr int kWaves = 4;

// A wave per token and head.
__global__ __launch_bounds__(256) void attention_prologue_head_kernel(PrologueArgs a) {
  const int lane = threadIdx.x & 63;
  const uint32_t slots = a.heads + 2u * a.kv_heads;
  const size_t item = (size_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
  if (item >= (size_t)a.tokens * slots) {
    return;  // whole wave
  }
  const uint32_t t = (uint32_t)(item / slots);
  const uint32_t slot = (uint32_t)(item % slots);
  const uint32_t d_head = a.head_dim;
  const size_t kv_dim = (size_t)a.kv_heads * d_head;

  if (slot >= a.heads + a.kv_heads) {  // value head: f32 -> f16 append
    const uint32_t kh = slot - a.heads - a.kv_heads;
    const float* src = a.value + (size_t)t * kv_dim + (size_t)kh * d_head;
    half_t* dst = a.value_cache + a.cache_offset + (size_t)t * kv_dim + (size_t)kh * d_head;
    for (uint32_t d = lane; d < d_head; d += 64) {
      dst[d] = static_cast<half_t>(src[d]);
    }
    return;
  }

  const bool is_q = slot < a.heads;
  const uint32_t head = is_q ? slot : slot - a.heads;
  const float* src = is_q ? a.q_gate + ((size_t)t * a.heads + head) * 2u * d_head
                          : a.key + (size_t)t * kv_dim + (size_t)head * d_head;
  const float* weight = is_q ? a.q_norm : a.k_norm;
  const RopeArgs rope{a.positions, a.mrope_start, a.tokens, a.n_dims, a.s0, a.s1, a.s2, a.s3,
                      a.theta};
  float v[4], w[4], g[4];
  load_head(src, weight, d_head, lane, v, w);
  // The gate half of a q_gate head is copied out; its loads go out with the rest.
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t d = lane + 64u * i;
    g[i] = is_q && d < d_head ? src[d_head + d] : 0.0f;
  }
  int32_t pos[4];
  rope_positions(rope, t, pos);
  double sn[4], cs[4];
  rope_angles(rope, pos, lane, sn, cs);
  float r[4];
  norm_rope(v, w, d_head, a.eps, a.n_dims, sn, cs, lane, r);

  if (is_q) {
    float* q_out = a.query_out + ((size_t)t * a.heads + head) * d_head;
    float* g_out = a.gate_out + ((size_t)t * a.heads + head) * d_head;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t d = lane + 64u * i;
      if (d < d_head) {
        q_out[d] = r[i];
        g_out[d] = g[i];
      }
    }
  } else {
    half_t* dst = a.key_cache + a.cache_offset + (size_t)t * kv_dim + (size_t)head * d_head;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t d = lane + 64u * i;
      if (d < d_head) {
        dst[d] = static_cast<half_t>(r[i]);
      }
    }
  }
}

// A wave takes H consecutive heads of one token (query, then key, then value
// heads); the token's rotation angles (a pow and a sincos in double per pair) are
// computed once for them.
template <int H>
__global__ __launch_bounds__(256) void attention_prologue_kernel(PrologueArgs a) {
  const int lane = threadIdx.x & 63;
  const uint32_t slots = a.heads + 2u * a.kv_heads;
  const uint32_t groups = (slots + H - 1u) / H;
  const size_t item = (size_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
  if (item >= (size_t)a.tokens * groups) {
    return;  // whole wave
  }
  const uint32_t t = (uint32_t)(item / groups);
  const uint32_t first = (uint32_t)(item % groups) * H;
  const uint32_t last = min(first + H, slots);
  const uint32_t d_head = a.head_dim;
  const size_t kv_dim = (size_t)a.kv_heads * d_head;
  const uint32_t keys_at = a.heads;
  const uint32_t values_at = a.heads + a.kv_heads;

  // Every load first: the heads' values, the gate half of the q_gate heads (copied
  // out) and the norm weights that apply.
  float v[H][4], g[H][4], wq[4], wk[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t d = lane + 64u * i;
    wq[i] = first < keys_at && d < d_head ? a.q_norm[d] : 0.0f;
    wk[i] = first < values_at && last > keys_at && d < d_head ? a.k_norm[d] : 0.0f;
  }
#pragma unroll
  for (int h = 0; h < H; ++h) {
    // Past the last slot: its loads again, so that none is behind a branch.
    const uint32_t slot = min(first + h, last - 1u);
    const float* src = slot < keys_at
                         ? a.q_gate + ((size_t)t * a.heads + slot) * 2u * d_head
                         : (slot < values_at
                              ? a.key + (size_t)t * kv_dim + (size_t)(slot - keys_at) * d_head
                              : a.value + (size_t)t * kv_dim + (size_t)(slot - values_at) * d_head);
    const uint32_t gate_at = slot < keys_at ? d_head : 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t d = lane + 64u * i;
      v[h][i] = d < d_head ? src[d] : 0.0f;
      g[h][i] = d < d_head ? src[gate_at + d] : 0.0f;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  double sn[4], cs[4];
  if (first < values_at) {
    const RopeArgs rope{a.positions, a.mrope_start, a.tokens, a.n_dims, a.s0, a.s1, a.s2, a.s3,
                        a.theta};
    int32_t pos[4];
    rope_positions(rope, t, pos);
    rope_angles(rope, pos, lane, sn, cs);
  }
  // All loads have returned (vmcnt 0): a wait that the compiler would place at a
  // value's use further down would count the stores of the heads before it too.
  __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const uint32_t slot = first + h;
    if (slot >= last) {
      break;
    }
    float r[4];
    if (slot < values_at) {
      norm_rope(v[h], slot < keys_at ? wq : wk, d_head, a.eps, a.n_dims, sn, cs, lane, r);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r[i] = v[h][i];
      }
    }
    if (slot < keys_at) {
      float* q_out = a.query_out + ((size_t)t * a.heads + slot) * d_head;
      float* g_out = a.gate_out + ((size_t)t * a.heads + slot) * d_head;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t d = lane + 64u * i;
        if (d < d_head) {
          q_out[d] = r[i];
          g_out[d] = g[h][i];
        }
      }
    } else {
      half_t* dst = (slot < values_at ? a.key_cache : a.value_cache) + a.cache_offset +
                    (size_t)t * kv_dim +
                    (size_t)(slot - (slot < values_at ? keys_at : values_at)) * d_head;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t d = lane + 64u * i;
        if (d < d_head) {
          dst[d] = static_cast<half_t>(r[i]);
        }
      }
    }
  }
}

template <int H>
void launch_heads(const PrologueArgs& a, hipStream_t stream) {
  const size_t groups = (a.heads + 2u * (size_t)a.kv_heads + H - 1u) / H;
  const size_t blocks = (a.tokens * groups + kWaves - 1) / kWaves;
  attention_prologue_kernel<H><<<dim3((uint32_t)blocks), 256, 0, stream>>>(a);
}

}  // namespace

hipError_t launch_attention_prologue(const PrologueArgs& a, hipStream_t stream) {
  if (a.tokens == 0) {
    return hipSuccess;
  }
  // Heads per wave: one where few waves run, whose latency then counts; from 256
  // tokens and 4096 heads on (3072 where more than 64 elements rotate) up to four, so
  // that the angles are formed less often.  Three where that divides a token's heads
  // over one workgroup's waves.  Measured, us, one / several heads per wave (q + k + v
  // heads of 256, n_dims 64):
  //   8 + 2 + 2  300 tokens 6.3 / 6.6   400 7.5 / 6.9   1024 14.6 / 11.3
  //   4 + 2 + 2  300 tokens 5.5 / 5.6   512 6.5 / 6.7    700  8.6 /  8.1
  //   4 + 1 + 1  512 tokens 5.5 / 5.8   700 7.1 / 6.7
  //   1 + 1 + 1  512 tokens 4.3 / 5.3  1024 5.4 / 5.7   2048  8.0 /  6.9
  //   8 + 4 + 4  128 tokens 4.5 / 6.2   256 6.8 / 6.7   1024 18.2 / 12.7
  //   8 + 2 + 2, n_dims 256  128 tokens 8.8 / 8.7  256 11.7 / 9.1
  const size_t slots = a.heads + 2u * (size_t)a.kv_heads;
  if (a.tokens < 256u || a.tokens * slots < (a.n_dims <= 64u ? 4096u : 3072u)) {
    const size_t blocks = (a.tokens * slots + kWaves - 1) / kWaves;
    attention_prologue_head_kernel<<<dim3((uint32_t)blocks), 256, 0, stream>>>(a);
  } else if (slots <= 12u) {
    launch_heads<3>(a, stream);
  } else {
    launch_heads<4>(a, stream);
  }
  return hipGetLastError();
}

}  // namespace kraken
