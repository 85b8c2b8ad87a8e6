// Sixteen consecutive channels of one row, from any page format to fp32.
//
// A lane reads the raw words of its own token's 16-channel chunk (1 to 16
// words, loaded as wide as the format allows, neighbouring tokens at
// neighbouring addresses) and turns them into values s * code + b in a few
// instructions per channel: byte conversions (v_cvt_f32_ubyteN) of masked
// words for 2-, 4- and 8-bit codes, bit fields for 3-bit ones.  Symmetric
// pages take b = -zero_point * s, which is exact (fp16 scale times an
// integer below 128), so s * code + b rounds once, as s * (code - zero_point)
// does.  Chunks never straddle a group: group_size and head_dim are
// multiples of 16 (chunk16_geometry).
#pragma once

#include <type_traits>
#include <utility>

#include "dc_common.h"

namespace dc {

enum ChunkKind { CK_B2 = 0, CK_B3, CK_B4, CK_B8, CK_F16, CK_F32, CK_I8, CK_NONE };

__host__ __device__ inline int chunk_kind(int32_t fmt, int32_t bits) {
  if (fmt == DC_FMT_M0_AFFINE || fmt == DC_FMT_M0_SYMMETRIC)
    return bits == 2 ? CK_B2 : bits == 3 ? CK_B3 : bits == 4 ? CK_B4 : bits == 8 ? CK_B8 : CK_NONE;
  return fmt == DC_FMT_M3_F16 ? CK_F16 : fmt == DC_FMT_M3_F32 ? CK_F32 : fmt == DC_FMT_M3_I8 ? CK_I8 : CK_NONE;
}

// Whether 16-channel chunks tile this geometry's groups and rows, with every
// offset inside a blob a 32-bit number.
__host__ __device__ inline bool chunk16_geometry(const dc_page_geometry& g) {
  return g.head_dim % 16 == 0 && g.group_size % 16 == 0 && int64_t(g.page_capacity) * num_groups(g) * g.group_size < (1 << 28);
}

// Where a chunk's words, scale and bias sit in its blob, in bytes.  Every
// field is linear in the token: add t times the step.
struct Chunk16 {
  uint32_t word, word_step;    // first raw word
  uint32_t scale, scale_step;  // fp16 scale (M0, int8 rows)
  uint32_t bias;               // fp16 bias (affine; same step as the scale)
  int shift;                   // 3-bit codes: bit of channel 0 in the first word (0 or 16)
};

__device__ __forceinline__ Chunk16 chunk16_at(int32_t fmt, int32_t bits, const dc_page_geometry& geo, const BlobLayout& L,
                                              int32_t c0) {
  Chunk16 k{};
  if (is_m0(fmt)) {
    const int32_t g = c0 / geo.group_size, bit = (c0 - g * geo.group_size) * bits;
    const uint32_t row = L.words * 4;
    k.word = (geo.layout == 0 ? uint32_t(g) * geo.page_capacity * row : g * row) + (bit >> 5) * 4;
    k.word_step = geo.layout == 0 ? row : L.groups * row;
    k.shift = bit & 31;
    k.scale = uint32_t(L.scales_off) + 2 * g;
    k.bias = uint32_t(L.bias_off) + 2 * g;
    k.scale_step = 2 * L.groups;
    return k;
  }
  const uint32_t es = fmt == DC_FMT_M3_F16 ? 2 : fmt == DC_FMT_M3_F32 ? 4 : 1;
  k.word = c0 * es;
  k.word_step = geo.head_dim * es;
  k.scale = uint32_t(L.scales_off);
  k.scale_step = 2;
  return k;
}

// The chunk's raw words.  p is 4-byte aligned for 2- and 3-bit codes, 8 for
// 4-bit codes and 16 otherwise (rows of 16-channel multiples in a 256-byte
// aligned blob).
__device__ __forceinline__ void load_chunk16(int kind, const uint8_t* p, uint32_t (&r)[16]) {
  auto put4 = [&](int i, uint4 x) { r[i] = x.x; r[i + 1] = x.y; r[i + 2] = x.z; r[i + 3] = x.w; };
  const uint32_t* w = reinterpret_cast<const uint32_t*>(p);
  const uint4* w4 = reinterpret_cast<const uint4*>(p);
  switch (kind) {
    case CK_B2: r[0] = w[0]; break;
    case CK_B3: r[0] = w[0]; r[1] = w[1]; break;
    case CK_B4: {
      const uint2 x = *reinterpret_cast<const uint2*>(p);
      r[0] = x.x; r[1] = x.y;
      break;
    }
    case CK_B8: case CK_I8: put4(0, w4[0]); break;
    case CK_F16: put4(0, w4[0]); put4(4, w4[1]); break;
    case CK_F32: put4(0, w4[0]); put4(4, w4[1]); put4(8, w4[2]); put4(12, w4[3]); break;
    default: break;
  }
}

__device__ __forceinline__ float half_bits(uint32_t w, int hi) {
  return float(__builtin_bit_cast(_Float16, uint16_t(hi ? w >> 16 : w & 0xffffu)));
}

// Values of the chunk's channels.  s and b: the scale and bias (1 and 0 for
// fp16 / fp32 rows, the row scale and 0 for int8 rows).
template <int KIND>
__device__ __forceinline__ void values16(const uint32_t (&r)[16], int shift, float s, float b, float (&v)[16]) {
  if constexpr (KIND == CK_B2) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {  // byte j of the masked word is code 4 j + k
      const uint32_t m = (r[0] >> (2 * k)) & 0x03030303u;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * j + k] = fmaf(float((m >> (8 * j)) & 0xffu), s, b);
    }
  } else if constexpr (KIND == CK_B3) {
    const uint64_t x = (uint64_t(r[1]) << 32 | r[0]) >> shift;
    const uint32_t lo = uint32_t(x), hi = uint32_t(x >> 24);  // channels 0 .. 7, 8 .. 15
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = fmaf(float((lo >> (3 * j)) & 7u), s, b);
      v[8 + j] = fmaf(float((hi >> (3 * j)) & 7u), s, b);
    }
  } else if constexpr (KIND == CK_B4) {
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const uint32_t e = r[w] & 0x0f0f0f0fu, o = (r[w] >> 4) & 0x0f0f0f0fu;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[8 * w + 2 * j] = fmaf(float((e >> (8 * j)) & 0xffu), s, b);
        v[8 * w + 2 * j + 1] = fmaf(float((o >> (8 * j)) & 0xffu), s, b);
      }
    }
  } else if constexpr (KIND == CK_B8) {
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = fmaf(float((r[j >> 2] >> (8 * (j & 3))) & 0xffu), s, b);
  } else if constexpr (KIND == CK_I8) {
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = float(int32_t(r[j >> 2] << (24 - 8 * (j & 3))) >> 24) * s;
  } else if constexpr (KIND == CK_F16) {
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = half_bits(r[j >> 1], j & 1);
  } else {
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = __builtin_bit_cast(float, r[j]);
  }
}

typedef float f32x4v __attribute__((ext_vector_type(4)));

// d[i] += a[i] * b per lane for the four rows i of block J of a (lanes 4 J ..
// 4 J + 3, one row each), read by every lane: one fp32 multiply-add per
// (row, lane), in 8 cycles (v_mfma_f32_4x4x1, A block J broadcast to all 16).
template <int J>
__device__ __forceinline__ f32x4v mfma4_bcast(float a, float b, f32x4v d) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, d, 4, J, 0);
}

// d += sum over i < 16 of block i of a times v[i]: 16 channels (or tokens) of
// four rows against this lane's 16 values, in two chains (even i in d0, odd
// in d1) so that no product waits for the one before it.
template <int... I>
__device__ __forceinline__ void dot16(float a, const float (&v)[16], f32x4v& d0, f32x4v& d1,
                                      std::integer_sequence<int, I...>) {
  ((I % 2 == 0 ? void(d0 = mfma4_bcast<I>(a, v[I], d0)) : void(d1 = mfma4_bcast<I>(a, v[I], d1))), ...);
}
__device__ __forceinline__ void dot16(float a, const float (&v)[16], f32x4v& d0, f32x4v& d1) {
  dot16(a, v, d0, d1, std::make_integer_sequence<int, 16>{});
}

// fn(std::integral_constant<int, KIND>) for a wave-uniform kind.
template <typename F>
__device__ __forceinline__ void for_chunk_kind(int kind, F&& fn) {
  switch (kind) {
    case CK_B2: fn(std::integral_constant<int, CK_B2>{}); break;
    case CK_B3: fn(std::integral_constant<int, CK_B3>{}); break;
    case CK_B4: fn(std::integral_constant<int, CK_B4>{}); break;
    case CK_B8: fn(std::integral_constant<int, CK_B8>{}); break;
    case CK_I8: fn(std::integral_constant<int, CK_I8>{}); break;
    case CK_F16: fn(std::integral_constant<int, CK_F16>{}); break;
    case CK_F32: fn(std::integral_constant<int, CK_F32>{}); break;
    default: break;
  }
}

}  // namespace dc
