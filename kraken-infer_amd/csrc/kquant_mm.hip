// K-quant matrix products for more than 8 tokens: C[t][r] = sum_k W[r][k] X[t][k]
// with W in GGUF Q4_K / Q5_K / Q6_K blocks and X in f32, both rounded to fp16
// (RNE, the weights after the exact f32 dequantization) and accumulated in f32
// (v_mfma_f32_32x32x16_f16), as the reference's tiled kernels do
// (mps_backend.mm:1082-1266).
//
// Two launches.  kq_pack_x_kernel rounds the inputs (or silu(gate) * up) to
// fp16 once and writes them in the order in which the MFMA reads them: 1 KB
// pieces [32 tokens][16 k], lane l's eight values at 16 l.  kq_mm_kernel then
// needs no LDS for its operands and no barrier in its loop: a wave loads a
// piece of X with one coalesced instruction straight into its fragment
// registers, loads its own weight rows' blocks as they are, and decodes them in
// registers into the other fragment.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "context_internal.hpp"
#include "device_common.hpp"

namespace kraken {
namespace {

typedef float float2v_t __attribute__((ext_vector_type(2)));
typedef float float16v_t __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(1))) uint8_t* gbytes_t;
typedef uint32_t u32x4_even_t __attribute__((ext_vector_type(4), aligned(2)));

template <int F>
struct BlockBytes;
template <>
struct BlockBytes<0> {
  static constexpr uint32_t value = 144;
};
template <>
struct BlockBytes<1> {
  static constexpr uint32_t value = 176;
};
template <>
struct BlockBytes<2> {
  static constexpr uint32_t value = 210;
};

__device__ __forceinline__ u32x4_t load16(gbytes_t p) {
  return *reinterpret_cast<const __attribute__((address_space(1))) u32x4_t*>(p);
}

// 16 bytes from an even address (Q6_K's 210-byte blocks): one load in the
// unaligned access mode that amdhsa programs run in.
__device__ __forceinline__ u32x4_t load16_even(gbytes_t p) {
  return *reinterpret_cast<const __attribute__((address_space(1))) u32x4_even_t*>(p);
}

// Lane l and lane l + 32 hold the two 16-byte halves of a 32-byte group; after
// this the lower lane holds bytes 0..7 and 16..23, the upper one 8..15 and
// 24..31: the eight consecutive k of each of its two MFMA fragments.
__device__ __forceinline__ void split_group(u32x4_t& w) {
  const auto a = __builtin_amdgcn_permlane32_swap(w.x, w.z, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(w.y, w.w, false, false);
  w.x = a[0];
  w.y = b[0];
  w.z = a[1];
  w.w = b[1];
}

// One lane's share of a weight row's super-block: half of its quants, and its
// scales.
template <int F>
struct RawBlock {
  u32x4_t head;   // Q4_K/Q5_K: d, dmin and the packed scales; Q6_K: the 16 scales
  u32x4_t q[4];   // the 4-bit quants of 64 k each (after split_group, this lane's)
  u32x4_t hi[2];  // Q5_K: the fifth bits ([0]); Q6_K: the high pairs of each half
  uint32_t d;     // Q6_K: f16 d

  // The lane's row of the block at `base` starts `row` bytes in.
  __device__ __forceinline__ void load_head(gbytes_t base, uint32_t row) {
    if constexpr (F == 2) {
      head = load16_even(base + row + 192u);
      d = *reinterpret_cast<const __attribute__((address_space(1))) uint16_t*>(base + row + 208u);
    } else {
      head = load16(base + row);
    }
  }
  __device__ __forceinline__ void load_hi(gbytes_t base, uint32_t row, uint32_t kh, int h) {
    const gbytes_t part = base + (row + 16u * kh);
    if constexpr (F == 2) {
      hi[h] = load16_even(part + 128u + 32u * h);
    } else if constexpr (F == 1) {
      hi[0] = load16(part + 16u);
    }
  }
  __device__ __forceinline__ void load_q(gbytes_t base, uint32_t row, uint32_t kh, int j) {
    const gbytes_t part = base + (row + 16u * kh);
    if constexpr (F == 2) {
      q[j] = load16_even(part + 32u * j);
    } else {
      q[j] = load16(part + (F == 1 ? 48u : 16u) + 32u * j);
    }
  }
  __device__ __forceinline__ void load(gbytes_t base, uint32_t row, uint32_t kh) {
    load_head(base, row);
    load_hi(base, row, kh, 0);
    if constexpr (F == 2) {
      load_hi(base, row, kh, 1);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      load_q(base, row, kh, j);
    }
  }
};

__device__ __forceinline__ float f16_low(uint32_t w) {
  return static_cast<float>(__builtin_bit_cast(half_t, static_cast<uint16_t>(w)));
}

__device__ __forceinline__ uint32_t word_of(const u32x4_t& v, int i) {
  return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w));
}

// Byte i (a constant) of the 16.
__device__ __forceinline__ uint32_t byte_at(const u32x4_t& v, int i) {
  return (word_of(v, i >> 2) >> (8 * (i & 3))) & 0xFFu;
}

// The scale and min of sub-block j (a constant) of a Q4_K/Q5_K header
// (mps_backend.mm:284-293).
__device__ __forceinline__ void sub_block(const u32x4_t& head, int j, uint32_t& sc, uint32_t& m) {
  if (j < 4) {
    sc = byte_at(head, 4 + j) & 63u;
    m = byte_at(head, 8 + j) & 63u;
  } else {
    sc = (byte_at(head, 8 + j) & 15u) | ((byte_at(head, j) >> 6) << 4);
    m = (byte_at(head, 8 + j) >> 4) | ((byte_at(head, 4 + j) >> 6) << 4);
  }
}

// Two quants as f16 denormals (q 2^-24, in each half of `pair`) times `scale`
// (their weight scale times 2^24) plus `offset`: v_fma_mix reads the f16
// operands as they are, so no conversion is needed.  The product has at most
// 24 significant bits and is exact, so the one rounding of the FMA is the
// rounding of (d sc) q - dmin m, and of (d sc) (q - 32).
__device__ __forceinline__ void fma_pair(uint32_t pair, float scale, float offset, float& a,
                                         float& b) {
  const half2_t q = __builtin_bit_cast(half2_t, pair);
  a = fmaf(static_cast<float>(q.x), scale, offset);
  b = fmaf(static_cast<float>(q.y), scale, offset);
  // The f32 values kept as such: their rounding to f16 is a second one.
  asm("" : "+v"(a), "+v"(b));
}

__device__ __forceinline__ half8_t round8(const float v[8]) {
  half8_t r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const half2_t h = __builtin_convertvector((float2v_t{v[2 * i], v[2 * i + 1]}), half2_t);
    r[2 * i] = h.x;
    r[2 * i + 1] = h.y;
  }
  return r;
}

// The lane's eight weights of step m (a constant, 0..15: k = 16 m + 8 kh ..) of
// a block, rounded to fp16.  split_group has been applied to the raw words.
template <int F>
__device__ __forceinline__ half8_t decode_step(const RawBlock<F>& b, int m, float scale,
                                               float offset) {
  uint32_t w[2], x[2];
  bool high;   // the quants are the high nibbles: masked in place, 16 q
  if constexpr (F == 2) {
    const int h = m >> 3, g = (m & 7) >> 1;
    const u32x4_t& q = b.q[2 * h + (g & 1)];
    high = g >= 2;
    w[0] = (m & 1) ? q.z : q.x;
    w[1] = (m & 1) ? q.w : q.y;
    x[0] = (m & 1) ? b.hi[h].z : b.hi[h].x;
    x[1] = (m & 1) ? b.hi[h].w : b.hi[h].y;
  } else {
    const u32x4_t& q = b.q[m >> 2];
    high = (m & 2) != 0;
    w[0] = (m & 1) ? q.z : q.x;
    w[1] = (m & 1) ? q.w : q.y;
    x[0] = (m & 1) ? b.hi[0].z : b.hi[0].x;
    x[1] = (m & 1) ? b.hi[0].w : b.hi[0].y;
  }
  const uint32_t mask = high ? 0x00F000F0u : 0x000F000Fu;
  float v[8];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint32_t even = w[i] & mask;
    uint32_t odd = (w[i] >> 8) & mask;
    if constexpr (F != 0) {
      // The bits above the nibble: bit m / 2 of the fifth-bit byte, or pair g of
      // the high-pair byte, brought to bit 4 (or 8).
      const uint32_t top = F == 1 ? (high ? 0x01000100u : 0x00100010u)
                                  : (high ? 0x03000300u : 0x00300030u);
      const int from = F == 1 ? m >> 1 : m & 6;
      const int to = high ? 8 : 4;
      const uint32_t xe = to >= from ? x[i] << (to - from) : x[i] >> (from - to);
      const int odd_from = from + 8;
      const uint32_t xo = to >= odd_from ? x[i] << (to - odd_from) : x[i] >> (odd_from - to);
      even |= xe & top;
      odd |= xo & top;
    }
    fma_pair(even, scale, offset, v[4 * i], v[4 * i + 2]);
    fma_pair(odd, scale, offset, v[4 * i + 1], v[4 * i + 3]);
  }
  return round8(v);
}

// One lane's weight row on its way through a block: decode(m), m = 0 .. 15 in
// order, gives the fragment of step m.
template <int F>
struct WeightStream {
  RawBlock<F> raw;
  float d, dmin, scale, offset;

  __device__ __forceinline__ half8_t decode(int m) {
    if (m == 0) {
      d = f16_low(F == 2 ? raw.d : raw.head.x);
      dmin = F == 2 ? 0.0f : f16_low(raw.head.x >> 16);
      if constexpr (F == 1) {
        split_group(raw.hi[0]);
      }
    }
    // The quants stay where the mask leaves them: 16 q in steps with high nibbles.
    if constexpr (F == 2) {
      if (m % 8 == 0) {
        split_group(raw.hi[m / 8]);
        split_group(raw.q[2 * (m / 8)]);
        split_group(raw.q[2 * (m / 8) + 1]);
      }
      const int s8 = (int)(int8_t)byte_at(raw.head, m);
      const float ds = d * (float)s8;
      scale = ds * ((m & 4) ? 0x1p20f : 0x1p24f);
      offset = ds * -32.0f;
    } else {
      if (m % 4 == 0) {
        split_group(raw.q[m / 4]);
      }
      if (m % 2 == 0) {
        uint32_t sc, mn;
        sub_block(raw.head, m / 2, sc, mn);
        scale = (d * (float)sc) * ((m & 2) ? 0x1p20f : 0x1p24f);
        offset = -(dmin * (float)mn);
      }
    }
    return decode_step<F>(raw, m, scale, offset);
  }
};

constexpr int kMmGroupMax = kKquantGroupMax;

struct MmArgs {
  const uint8_t* w[kMmGroupMax];
  float* c[kMmGroupMax];
  const float* residual;  // one matrix only
  uint32_t rows[kMmGroupMax];
  uint32_t tile_end[kMmGroupMax];  // row tiles of matrices 0 .. i
  uint32_t count;
  const half_t* x;  // packed
  uint32_t tokens, cols;
  uint32_t token_tiles;
};

// A workgroup's matrix and the first row and token of its tile.  Consecutive
// workgroups go to consecutive XCDs: each XCD takes a run of tiles, token tiles
// fastest, so its L2 holds a run of weight rows once.
struct MmTile {
  uint32_t matrix, row, token;
};
template <int kRows, int kTokens>
__device__ __forceinline__ MmTile locate_tile(const MmArgs& a) {
  const uint32_t per = gridDim.x / 8u, rest = gridDim.x % 8u;
  const uint32_t xcd = blockIdx.x % 8u;
  const uint32_t id = xcd * per + min(xcd, rest) + blockIdx.x / 8u;
  uint32_t tile = id / a.token_tiles;
  uint32_t g = 0;
  while (g + 1 < a.count && tile >= a.tile_end[g]) {
    ++g;
  }
  tile -= g == 0 ? 0u : a.tile_end[g - 1];
  return MmTile{g, tile * kRows, id % a.token_tiles * kTokens};
}

// Few tokens, or few rows: the KW waves of a workgroup split the K blocks of one
// tile of 32 RA rows x 32 TB tokens and add their sums through LDS in wave order.
// No wave waits for another before that, and each has a whole stage of pieces
// and the next block's weights in flight.
template <int RA, int TB, int KW>
struct MmShape {
  static constexpr int kRows = 32 * RA;
  static constexpr int kTokens = 32 * TB;
  static constexpr int kRegs = RA * TB * 16;
  static constexpr int kXSteps = RA * TB >= 4 ? 4 : 8;  // X pieces per prefetch stage
};

template <int F, int RA, int TB, int KW>
__global__ __launch_bounds__(64 * KW, 2) void kq_mm_kernel(MmArgs a) {
  using S = MmShape<RA, TB, KW>;
  const int lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t r32 = lane & 31;
  const uint32_t kh = lane >> 5;
  const MmTile at = locate_tile<S::kRows, S::kTokens>(a);
  const uint32_t g = at.matrix;
  const uint32_t n = a.rows[g];
  const uint32_t n0 = at.row;
  const uint32_t t0 = at.token;
  const uint32_t nb = a.cols / 256u;
  const uint32_t b0 = wave * nb / KW;
  const uint32_t b1 = (wave + 1u) * nb / KW;
  const uint32_t row_bytes = nb * BlockBytes<F>::value;

  float16v_t acc[RA][TB];
#pragma unroll
  for (int r = 0; r < RA; ++r) {
#pragma unroll
    for (int t = 0; t < TB; ++t) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[r][t][e] = 0.0f;
      }
    }
  }

  // Rows past the matrix read its last row and token groups past the input read
  // its last group; neither is stored.  A wave-uniform base and a 32-bit lane
  // offset per operand.
  const uint32_t base_row = min(n0, n - 1u);
  const gbytes_t wbase = (gbytes_t)a.w[g] + (uint64_t)base_row * row_bytes;
  uint32_t woff[RA];
#pragma unroll
  for (int r = 0; r < RA; ++r) {
    woff[r] = (min(n0 + 32u * r + r32, n - 1u) - base_row) * row_bytes;
  }
  const uint32_t groups = (a.tokens + 31u) / 32u;
  gbytes_t xbase[TB];
#pragma unroll
  for (int t = 0; t < TB; ++t) {
    xbase[t] = (gbytes_t)a.x + (uint64_t)min(t0 / 32u + t, groups - 1u) * a.cols * 64u;
  }
  const uint32_t xoff = 16u * lane;

  if (b0 < b1) {
    constexpr int XS = S::kXSteps;
    WeightStream<F> w[RA];
    half8_t x[2][XS][TB];
    // The X pieces of phase ph (XS steps) of block b into stage ph % 2.
    auto load_x = [&](uint32_t b, int ph) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < XS; ++s) {
#pragma unroll
        for (int t = 0; t < TB; ++t) {
          const gbytes_t piece = xbase[t] + (uint64_t)b * 16384u + 1024u * (XS * ph + s);
          x[ph & 1][s][t] = __builtin_bit_cast(half8_t, load16(piece + xoff));
        }
      }
    };
#pragma unroll
    for (int r = 0; r < RA; ++r) {
      w[r].raw.load(wbase + (uint64_t)b0 * BlockBytes<F>::value, woff[r], kh);
    }
    load_x(b0, 0);
    __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of their uses
    for (uint32_t b = b0; b < b1; ++b) {
      const uint32_t bn = min(b + 1u, b1 - 1u);
      load_x(b, 1);
      // The next block's headers; its quants replace this block's as those are
      // used up (three quarters of a block ahead).
      const gbytes_t wn = wbase + (uint64_t)bn * BlockBytes<F>::value;
      RawBlock<F> next[RA];
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        next[r].load_head(wn, woff[r]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        if (m > 0 && m % XS == 0) {
          const int ph = m / XS + 1;
          load_x(ph * XS < 16 ? b : bn, ph * XS < 16 ? ph : 0);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int r = 0; r < RA; ++r) {
          const half8_t wf = w[r].decode(m);
#pragma unroll
          for (int t = 0; t < TB; ++t) {
            acc[r][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[(m / XS) & 1][m % XS][t], wf,
                                                               acc[r][t], 0, 0, 0);
          }
          if constexpr (F == 2) {
            if (m % 8 == 5) {
              w[r].raw.load_q(wn, woff[r], kh, m / 8 * 2);
            }
            if (m % 8 == 7) {
              w[r].raw.load_q(wn, woff[r], kh, m / 8 * 2 + 1);
              w[r].raw.load_hi(wn, woff[r], kh, m / 8);
            }
          } else {
            if (m % 4 == 3) {
              w[r].raw.load_q(wn, woff[r], kh, m / 4);
            }
            if (F == 1 && m == 15) {
              w[r].raw.load_hi(wn, woff[r], kh, 0);
            }
          }
        }
      }
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        w[r].raw.head = next[r].head;
        w[r].raw.d = next[r].d;
      }
    }
  }

  __shared__ float s_sum[KW][S::kRegs][64];
#pragma unroll
  for (int r = 0; r < RA; ++r) {
#pragma unroll
    for (int t = 0; t < TB; ++t) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s_sum[wave][(r * TB + t) * 16 + e][lane] = acc[r][t][e];
      }
    }
  }
  __syncthreads();
  // A wave's share of the sums: registers of one 32-row block.
  constexpr int kShare = S::kRegs / KW;
  static_assert(16 * TB % kShare == 0, "a share within 32 rows");
  float v[kShare];
#pragma unroll
  for (int i = 0; i < kShare; ++i) {
    const uint32_t reg = wave * kShare + i;
    v[i] = s_sum[0][reg][lane];
#pragma unroll
    for (int k = 1; k < KW; ++k) {
      v[i] += s_sum[k][reg][lane];
    }
  }
  store_sums(a.c[g], a.residual, n, n0 + 32u * (wave * kShare / (16u * TB)) + r32, a.tokens, [&](int i) {
    const uint32_t reg = wave * kShare + i;
    const uint32_t e = reg % 16u, t = reg / 16u % TB;
    return t0 + 32u * t + 8u * (e / 4u) + 4u * kh + (e % 4u);
  }, v);
}

// Many tokens: RW waves along the rows, each holding 32 rows x 128 tokens over
// the whole of K, so a decoded weight fragment feeds four MFMAs and an X piece
// feeds RW of them.  X goes through four LDS stages of 64 k; the pieces of stage
// s + 3 are written while stage s computes (from registers loaded four stages
// before that), and each step's fragments are read and decoded under the MFMAs
// of the step before (sched_group_barrier), across the one barrier per stage.
template <int RW>
struct LdsShape {
  static constexpr int kThreads = 64 * RW;
  static constexpr int kRows = 32 * RW;
  static constexpr int kTokens = 128;
  static constexpr int kPieces = 16 / RW;  // X pieces per wave and stage
};

template <int F, int RW>
__global__ __launch_bounds__(LdsShape<RW>::kThreads, (RW == 2 ? 1 : 2))
void kq_mm_lds_kernel(MmArgs a) {
  using S = LdsShape<RW>;
  constexpr int NP = S::kPieces;
  __shared__ __attribute__((aligned(16))) half_t s_x[4][16][512];  // [stage][piece]
  const int lane = threadIdx.x & 63;
  const uint32_t rw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t r32 = lane & 31;
  const uint32_t kh = lane >> 5;
  const MmTile at = locate_tile<S::kRows, S::kTokens>(a);
  const uint32_t g = at.matrix;
  const uint32_t n = a.rows[g];
  const uint32_t n0 = at.row + 32u * rw;
  const uint32_t t0 = at.token;
  const uint32_t nb = a.cols / 256u;
  const uint32_t row_bytes = nb * BlockBytes<F>::value;

  float16v_t acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      acc[t][e] = 0.0f;
    }
  }
  const uint32_t base_row = min(n0, n - 1u);
  const gbytes_t wbase = (gbytes_t)a.w[g] + (uint64_t)base_row * row_bytes;
  const uint32_t woff = (min(n0 + r32, n - 1u) - base_row) * row_bytes;
  const uint32_t groups = (a.tokens + 31u) / 32u;
  // Piece i of this wave's share of a stage is piece rw + RW i: k step
  // piece / 4, token group piece % 4.
  gbytes_t xbase[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const uint32_t piece = rw + RW * i;
    xbase[i] = (gbytes_t)a.x +
               (uint64_t)min(t0 / 32u + piece % 4u, groups - 1u) * a.cols * 64u +
               (piece / 4u) * 1024u;
  }
  const uint32_t xoff = 16u * lane;

  const uint32_t last_stage = 4u * nb - 1u;
  u32x4_t xr[4][NP];
  auto load_x = [&](uint32_t stage, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      xr[slot][i] = load16(xbase[i] + (uint64_t)min(stage, last_stage) * 4096u + xoff);
    }
  };
  auto write_x = [&](int buf, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      *reinterpret_cast<u32x4_t*>(&s_x[buf][rw + RW * i][8 * lane]) = xr[slot][i];
    }
  };
  half8_t xf[2][4], wf[2];
  auto read_x = [&](int buf, int ms, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      xf[slot][t] = *reinterpret_cast<const half8_t*>(&s_x[buf][4 * ms + t][8 * lane]);
    }
  };

  WeightStream<F> w;
  uint32_t stage = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    load_x(stage + i, i);
  }
  w.raw.load(wbase, woff, kh);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    write_x(i, i);
    load_x(stage + 4u + i, i);
  }
  __syncthreads();
  read_x(0, 0, 0);
  wf[0] = w.decode(0);
  for (uint32_t b = 0; b < nb; ++b) {
    const gbytes_t wn = wbase + (uint64_t)min(b + 1u, nb - 1u) * BlockBytes<F>::value;
    RawBlock<F> next;
    next.load_head(wn, woff);
    if constexpr (F == 1) {
      next.load_hi(wn, woff, kh, 0);
    }
#pragma unroll
    for (int st = 0; st < 4; ++st, ++stage) {
      write_x((st + 3) % 4, (st + 3) % 4);  // stage + 3
      load_x(stage + 7u, (st + 3) % 4);
#pragma unroll
      for (int ms = 0; ms < 4; ++ms) {
        const int m = 4 * st + ms;
        read_x(ms < 3 ? st : (st + 1) % 4, (ms + 1) % 4, (m + 1) % 2);
        if (m == 15) {
          w.raw.head = next.head;
          w.raw.d = next.d;
          if constexpr (F == 1) {
            w.raw.hi[0] = next.hi[0];
          }
        }
        wf[(m + 1) % 2] = w.decode((m + 1) % 16);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[m % 2][t], wf[m % 2], acc[t], 0, 0, 0);
        }
        if (ms == 2) {
          // The stage's quants are decoded: the next block's take their place.
          if constexpr (F == 2) {
            if (st & 1) {
              w.raw.load_q(wn, woff, kh, st - 1);
              w.raw.load_q(wn, woff, kh, st);
              w.raw.load_hi(wn, woff, kh, st / 2);
            }
          } else {
            w.raw.load_q(wn, woff, kh, st);
          }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA,
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
          __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);  // and decode under it
        }
      }
      __syncthreads();
    }
  }

#pragma unroll
  for (int t = 0; t < 4; ++t) {
    float v[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      v[e] = acc[t][e];
    }
    store_sums(a.c[g], a.residual, n, n0 + r32, a.tokens, [&](int e) {
      return t0 + 32u * t + 8u * (e / 4) + 4u * kh + (e % 4);
    }, v);
  }
}

// X [tokens][cols] f32 -> fp16 pieces [token group of 32][k / 16][lane][8]:
// lane l holds token l % 32 and k = 16 s + 8 (l / 32) .. + 7; tokens past the
// input are zero.  With up, X is silu(x) * up (silu_mul_f32_in_place's
// arithmetic).  One wave per piece: bound by latency, so that with four pieces per
// wave the products took 0.4 to 0.8 us longer, and 2.0 to 2.4 us with up, whose
// exponentials then form one chain (48 tokens x 1024, Q4_K 3584 rows: 6.9 -> 6.2
// us, with up 9.0 -> 6.6).
template <bool kSwiglu>
__global__ __launch_bounds__(256) void kq_pack_x_kernel(const float* x, const float* up,
                                                        half_t* out, uint32_t tokens,
                                                        uint32_t cols, uint32_t pieces) {
#pragma clang fp contract(off)
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t piece = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (piece >= pieces) {
    return;
  }
  const uint32_t per_group = cols / 16u;
  const uint32_t token = piece / per_group * 32u + (lane & 31u);
  const uint32_t k = piece % per_group * 16u + 8u * (lane >> 5);
  float4 v[2], u[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    u[i] = v[i];
    if (token < tokens) {
      const uint64_t at = ((uint64_t)token * cols + k + 4u * i) / 4u;
      v[i] = reinterpret_cast<const float4*>(x)[at];
      if constexpr (kSwiglu) {
        u[i] = reinterpret_cast<const float4*>(up)[at];
      }
    }
  }
  half8_t h;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float f[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
    const float q[4] = {u[i].x, u[i].y, u[i].z, u[i].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float y = f[e];
      if constexpr (kSwiglu) {
        // The f32 product kept as such before its rounding to fp16.
        y = (y / (1.0f + expf(-y))) * q[e];
        asm("" : "+v"(y));
      }
      h[4 * i + e] = static_cast<half_t>(y);
    }
  }
  reinterpret_cast<half8_t*>(out)[(uint64_t)piece * 64u + lane] = h;
}

template <class S>
uint32_t tile_grid(MmArgs& a) {
  uint32_t tiles = 0;
  for (uint32_t i = 0; i < a.count; ++i) {
    tiles += (a.rows[i] + S::kRows - 1u) / S::kRows;
    a.tile_end[i] = tiles;
  }
  a.token_tiles = (a.tokens + S::kTokens - 1u) / S::kTokens;
  return tiles * a.token_tiles;
}

template <int F, int RA, int TB>
void launch_split(MmArgs a, hipStream_t stream) {
  const uint32_t grid = tile_grid<MmShape<RA, TB, 4>>(a);
  kq_mm_kernel<F, RA, TB, 4><<<grid, 256, 0, stream>>>(a);
}

template <int F, int RW>
void launch_lds(MmArgs a, hipStream_t stream) {
  const uint32_t grid = tile_grid<LdsShape<RW>>(a);
  kq_mm_lds_kernel<F, RW><<<grid, LdsShape<RW>::kThreads, 0, stream>>>(a);
}

// The tile shapes, smallest first.  Whether they or the older forms run: mm_us.
enum class MmForm { two_pass, split_32x32, split_32x64, split_64x64, lds_64, lds_128, lds_256 };

// The smallest tile whose workgroups do not exceed the chip's 256 CUs (about two
// each for the 64 x 64 tile), counted for one matrix of `rows` rows (the largest of a
// group: only matrices of that size get the same tiles, and the same bits, in a group
// and on their own).  Measured at 1024 columns, us per call with the packing launch,
// 32x32 / 32x64 / 64x64 / 128x128 / 256x128 tiles:
//   Q4_K 6144 rows   32 tokens   7.1 /  8.2 /  9.3 / 15.6 / 19.6   (192 of 32x32)
//                   128 tokens  10.8 / 10.8 /  9.9 / 16.0 / 20.2   (192 of 64x64)
//                   256 tokens  16.3 / 14.6 / 14.1 / 16.3 / 20.5   (384 of 64x64)
//                   384 tokens  22.0 / 19.8 / 19.0 / 16.9 / 20.8   (576 of 64x64)
//                   768 tokens  37.9 / 32.0 / 28.1 / 26.9 / 23.3   (144 of 256x128)
//                  1024 tokens  48.6 / 39.3 / 33.1 / 28.0 / 26.5
//   Q4_K 3584 rows 1024 tokens  32.4 / 27.2 / 24.4 / 19.9 / 23.6   (112 of 256x128)
//   Q5_K 6144 rows  256 tokens  17.5 / 15.1 / 14.9 / 17.2 / 21.7
//                   768 tokens  42.5 / 33.6 / 29.9 / 27.7 / 24.4
// Q6_K decodes at twice the cost per weight, so that its 64x64 tile loses to
// 64x128 (one decode per four MFMAs) beyond 256 workgroups (2048 rows, 768
// tokens: 22.1 against 19.5 us), and with many column blocks, where 64x128 tiles
// are too few, to dequantizing the matrix once (1024 x 3584, 768 tokens: 32.4
// against 25.3 us).
MmForm mm_form(int format, uint64_t rows, uint64_t cols, uint64_t tokens) {
  auto grid = [&](uint64_t r, uint64_t t) { return (rows + r - 1) / r * ((tokens + t - 1) / t); };
  if (grid(32, 32) <= 256) {
    return MmForm::split_32x32;
  }
  if (grid(32, 64) <= 256) {
    return MmForm::split_32x64;
  }
  if (format == 2) {
    if (cols > 1536) {
      return MmForm::two_pass;
    }
    if (grid(64, 64) <= 256) {
      return MmForm::split_64x64;
    }
    if (grid(64, 128) <= 256) {
      return MmForm::lds_64;
    }
  } else if (grid(64, 64) <= 512) {
    return MmForm::split_64x64;
  }
  return grid(256, 128) > 128 ? MmForm::lds_256 : MmForm::lds_128;
}

// The estimated time of the two launches in us, for the forms of more than 256 tiles
// of 32 x 64: packing, the output, and per round of 256 workgroups the K blocks that
// a wave walks.  Fitted to 3855 products (512 to 24576 rows, 256 to 12288 columns, 65
// to 2048 tokens): 8% off (rms), kquant_matmul_us 5%.  Where many tokens share the
// weights, decoding them once per 64 or 128 tokens costs more than dequantizing them
// first or than the B tile's decode; those forms / these tiles, us:
//   Q6_K 6144 x 1024, 1024 tokens  28.3 / 31.1     2048 x 1024, 1024  18.8 / 19.8
//   Q5_K 6144 x 2048, 1024 tokens  43.2 / 44.1     2048 x 6144,  700  49.1 / 53.5
//   Q4_K 8192 x 256,   512 tokens (B tile)  9.0 / 10.9
// By this rule 38 of the 3855 take these tiles where they are more than 3% slower, at
// most 17%; without it 647 did, at most 48%.
double mm_us(MmForm form, int format, size_t count, const size_t* rows, size_t cols,
             size_t tokens) {
  struct Cost {
    uint64_t rows, tokens;
    double block[3];  // per K block (per four, split over the waves), by format
    double round;
  };
  const Cost c = form == MmForm::split_64x64 ? Cost{64, 64, {2.7, 3.1, 6.25}, 0.0}
                 : form == MmForm::lds_64    ? Cost{64, 128, {0.0, 0.0, 2.3}, 1.8}
                 : form == MmForm::lds_128   ? Cost{128, 128, {1.85, 2.2, 2.9}, 0.65}
                                             : Cost{256, 128, {3.25, 3.8, 4.95}, 0.5};
  uint64_t tiles = 0;
  double outputs = 0.0;
  for (size_t i = 0; i < count; ++i) {
    tiles += (rows[i] + c.rows - 1) / c.rows;
    outputs += 1e-6 * (double)rows[i] * (double)tokens;
  }
  const double rounds = (double)((tiles * ((tokens + c.tokens - 1) / c.tokens) + 255) / 256);
  const uint64_t nb = cols / 256;
  // Fewer blocks than waves, or than the pipeline of a Q6_K chain needs to fill.
  double walk = nb == 1 && format == 2 ? 1.3 : (double)nb;
  if (form == MmForm::split_64x64) {
    walk = nb < 4 ? (double)(nb + 3) / 7.0 : (double)((nb + 3) / 4);
  }
  return 5.0 + 2.6e-6 * (double)tokens * (double)cols + 0.82 * outputs +
         rounds * (walk * c.block[format] + c.round);
}

template <int F>
hipError_t launch_form(MmForm form, const MmArgs& a, hipStream_t stream) {
  switch (form) {
    case MmForm::split_32x32: launch_split<F, 1, 1>(a, stream); break;
    case MmForm::split_32x64: launch_split<F, 1, 2>(a, stream); break;
    case MmForm::split_64x64: launch_split<F, 2, 2>(a, stream); break;
    case MmForm::lds_64:
      if constexpr (F == 2) {
        launch_lds<F, 2>(a, stream);
        break;
      }
      return hipErrorInvalidValue;
    case MmForm::lds_128: launch_lds<F, 4>(a, stream); break;
    case MmForm::lds_256: launch_lds<F, 8>(a, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

bool kquant_mm_supported(int format, size_t count, const size_t* rows, size_t cols,
                         size_t tokens) {
  // 32-bit lane offsets within a tile's rows.
  if (tokens <= kKquantGemvMaxTokens ||
      (uint64_t)cols / 256u * kquant_block_bytes(format) * 256u >= (1ull << 31)) {
    return false;
  }
  const MmForm form = mm_form(format, *std::max_element(rows, rows + count), cols, tokens);
  if (form == MmForm::split_32x32 || form == MmForm::split_32x64) {
    return true;
  }
  return form != MmForm::two_pass && mm_us(form, format, count, rows, cols, tokens) <=
                                       0.98 * kquant_matmul_us(format, count, rows, cols, tokens);
}

size_t kquant_mm_workspace_bytes(size_t cols, size_t tokens) {
  return (tokens + 31u) / 32u * 32u * cols * sizeof(half_t);
}

hipError_t launch_kquant_mm(int format, size_t count, const void* const* weights,
                            const size_t* rows, size_t cols, size_t tokens, const float* input,
                            const float* up, const float* residual, float* const* outputs,
                            void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (count == 0 || count > kKquantGroupMax || (residual != nullptr && count != 1) ||
      workspace == nullptr || workspace_bytes < kquant_mm_workspace_bytes(cols, tokens)) {
    return hipErrorInvalidValue;
  }
  MmArgs a{};
  size_t most_rows = 0;
  for (size_t i = 0; i < count; ++i) {
    most_rows = std::max(most_rows, rows[i]);
    a.w[i] = static_cast<const uint8_t*>(weights[i]);
    a.c[i] = outputs[i];
    a.rows[i] = (uint32_t)rows[i];
  }
  a.residual = residual;
  a.count = (uint32_t)count;
  a.x = static_cast<const half_t*>(workspace);
  a.tokens = (uint32_t)tokens;
  a.cols = (uint32_t)cols;
  const MmForm form = mm_form(format, most_rows, cols, tokens);
  const uint32_t pieces = (uint32_t)((tokens + 31u) / 32u * (cols / 16u));
  const dim3 grid((pieces + 3u) / 4u);
  half_t* packed = static_cast<half_t*>(workspace);
  if (up != nullptr) {
    kq_pack_x_kernel<true><<<grid, 256, 0, stream>>>(input, up, packed, a.tokens, a.cols, pieces);
  } else {
    kq_pack_x_kernel<false><<<grid, 256, 0, stream>>>(input, up, packed, a.tokens, a.cols, pieces);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    return e;
  }
  switch (format) {
    case 0: return launch_form<0>(form, a, stream);
    case 1: return launch_form<1>(form, a, stream);
    case 2: return launch_form<2>(form, a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace kraken
