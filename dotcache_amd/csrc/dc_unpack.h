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

// blob_layout in 32 bits, for geometries chunk16_geometry accepts (their
// blobs stay below 2^30 bytes): a page's layout costs a few instructions.
struct Blob32 {
  uint32_t groups, words, scales_off, bias_off, total;
};

__host__ __device__ inline Blob32 blob32(int32_t fmt, int32_t bits, const dc_page_geometry& g, uint32_t groups) {
  const uint32_t C = g.page_capacity;
  auto up16 = [](uint32_t x) { return (x + 15u) & ~15u; };
  Blob32 L{};
  L.groups = groups;
  const bool m0 = is_m0(fmt);
  L.words = m0 ? (uint32_t(g.group_size) * bits + 31) / 32 : 0;
  const uint32_t es = fmt == DC_FMT_M3_F16 ? 2 : fmt == DC_FMT_M3_F32 ? 4 : 1;
  L.scales_off = up16(m0 ? groups * C * L.words * 4 : C * uint32_t(g.head_dim) * es);
  const uint32_t per = m0 ? up16(C * groups * 2) : fmt == DC_FMT_M3_I8 ? up16(C * 2) : 0;
  L.bias_off = L.scales_off + per;
  L.total = fmt == DC_FMT_M0_AFFINE ? L.bias_off + per : L.bias_off;
  return L;
}

// A walk over a page's 16-channel chunks: where the current one's words,
// scale and bias sit in the blob, in bytes.  Every offset is linear in the
// token: add t times the step.  next() moves on without a division.
struct Chunk16 {
  uint32_t word_step, scale_step;  // per token
  uint32_t base, bit;              // first word of the group (escapes: of the row), bit of the chunk from there
  uint32_t scale, bias;
  uint32_t chunk_bits, group_bits, group_step;  // (escapes: one group that never ends)

  __device__ __forceinline__ uint32_t word() const { return base + (bit >> 5) * 4; }
  __device__ __forceinline__ int shift() const { return int(bit & 31); }  // nonzero (16) for 3-bit codes only
  __device__ __forceinline__ void next() {
    bit += chunk_bits;
    if (bit == group_bits) {
      bit = 0;
      base += group_step;
      scale += 2;
      bias += 2;
    }
  }
};

__device__ __forceinline__ Chunk16 chunk16_at(int32_t fmt, int32_t bits, const dc_page_geometry& geo, const Blob32& L,
                                              uint32_t c0) {
  Chunk16 k{};
  k.scale = L.scales_off;
  k.bias = L.bias_off;
  if (is_m0(fmt)) {
    const uint32_t gs = geo.group_size, row = L.words * 4;
    k.chunk_bits = 16 * bits;
    k.group_bits = gs * bits;
    k.group_step = geo.layout == 0 ? uint32_t(geo.page_capacity) * row : row;
    k.word_step = geo.layout == 0 ? row : L.groups * row;
    k.scale_step = 2 * L.groups;
    if (c0 != 0) {
      const uint32_t g = c0 / gs;
      k.bit = (c0 - g * gs) * bits;
      k.base = g * k.group_step;
      k.scale += 2 * g;
      k.bias += 2 * g;
    }
    return k;
  }
  const uint32_t es = fmt == DC_FMT_M3_F16 ? 2 : fmt == DC_FMT_M3_F32 ? 4 : 1;
  k.chunk_bits = 128 * es;
  k.group_bits = ~0u;
  k.bit = c0 * 8 * es;
  k.word_step = geo.head_dim * es;
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

// s0[n] + s1[n]: dot products of this lane's row (token t of the page d
// describes) with the four queries of each register block n < NB, over hd
// channels.  get_q(c0, n) is block n's query register of channels c0 .. c0 +
// 15 (lane (b, r): channel c0 + b of its query r).  Two chunks in flight.
template <int NB, typename GetQ>
__device__ __forceinline__ void score_row(const dc_page_desc& d, const dc_page_geometry& geo, const Blob32& L,
                                          const uint8_t* blob, uint32_t t, GetQ&& get_q, f32x4v (&s0)[NB],
                                          f32x4v (&s1)[NB]) {
  const int32_t hd = geo.head_dim;
  // (a chunk holds what its loads return; conversions wait until it is used,
  // or every load would be waited for where it was issued)
  struct Chunk {
    uint32_t r[16];
    uint16_t s, b;
    float q[NB];
    int shift;
  };
  const bool affine = d.format == DC_FMT_M0_AFFINE;
  Chunk16 ck = chunk16_at(d.format, d.bits, geo, L, 0);
  const uint8_t* row = blob + t * ck.word_step;
  const uint8_t* scales = blob + t * ck.scale_step;
  for_chunk_kind(chunk_kind(d.format, d.bits), [&](auto kind) __attribute__((always_inline)) {
    constexpr int K = decltype(kind)::value;
    constexpr int D = K == CK_F32 ? 2 : 4;  // chunks in flight
    auto load = [&](int32_t c0, Chunk& x) __attribute__((always_inline)) {
      load_chunk16(K, row + ck.word(), x.r);
      x.shift = ck.shift();
      if constexpr (K != CK_F16 && K != CK_F32) {
        x.s = *reinterpret_cast<const uint16_t*>(scales + ck.scale);
        // (no bias: the scale again, unused)
        x.b = *reinterpret_cast<const uint16_t*>(scales + (affine ? ck.bias : ck.scale));
      }
#pragma unroll
      for (int n = 0; n < NB; ++n) x.q[n] = get_q(c0, n);
      ck.next();
    };
    auto dot = [&](const Chunk& x) __attribute__((always_inline)) {
      float v[16], s = 1.f, b = 0.f;
      if constexpr (K != CK_F16 && K != CK_F32) {
        constexpr float zp = K == CK_B2 ? -1.f : K == CK_B3 ? -3.f : K == CK_B4 ? -7.f : K == CK_B8 ? -127.f : 0.f;
        s = half_bits(x.s, 0);
        b = affine ? half_bits(x.b, 0) : K == CK_I8 ? 0.f : zp * s;
      }
      values16<K>(x.r, x.shift, s, b, v);
#pragma unroll
      for (int n = 0; n < NB; ++n) dot16(x.q[n], v, s0[n], s1[n]);
    };
    // whole rounds of D chunks without a branch, then the rest
    Chunk X[D];
    const int32_t n_chunks = hd / 16, whole = n_chunks / D * D;
    if (whole > 0) {
#pragma unroll
      for (int j = 0; j < D; ++j) load(16 * j, X[j]);
      for (int32_t c = D; c < whole; c += D)
#pragma unroll
        for (int j = 0; j < D; ++j) {
          dot(X[j]);
          load(16 * (c + j), X[j]);
        }
#pragma unroll
      for (int j = 0; j < D; ++j) dot(X[j]);
    }
    for (int32_t c = whole; c < n_chunks; ++c) {
      load(16 * c, X[0]);
      dot(X[0]);
    }
  });
}

}  // namespace dc
