// Fused paged decode for the page formats the MFMA kernel
// (dc_decode_mfma.hip) does not take: 2- and 3-bit codes, int8 and fp32
// escapes, other group sizes, head_dims and layouts, pools of several code
// widths.  Everything is fp32: values are s * code + b as read, products and
// sums v_mfma_f32_4x4x1.
//
// A block of four wavefronts runs one work item.  The item's tokens are cut
// into units of 64; each wave takes every fourth unit and keeps its own
// running (max, sum, output), which the block combines at the end, so the
// waves never wait for each other.  Per unit:
//   score  one token per lane: the lane unpacks its key row 16 channels at a
//          time (score_row; neighbouring lanes read neighbouring words) and
//          the queries come as the matrix instruction's broadcast operand,
//          four heads per register.  Logits stay in the token's lane.
//   softmax  per head one maximum over the wave; weights go to LDS as
//          [token][head].
//   mix    NS consecutive channels per lane, one token at a time: the
//          token's weights are the broadcast operand (16 tokens x 4 heads
//          per register), the lane unpacks its NS values.  M0 codes, scales
//          and biases of the unit come to LDS by DMA, issued before the
//          score so that they fly under it, and lie there token by token, so
//          that one 16-byte read gives a lane four tokens' code words or
//          eight tokens' scales; escape rows are read 4 or 8 tokens ahead.
// Registers hold 4 heads x NS channels of output per head block and no
// per-format state, so one instance serves every format.
//
// Bound by instruction issue at long contexts (a token costs a wave about 11
// vector instructions and 2 NB NS matrix instructions in the mix) and by one
// unit's chain of loads, score and mix at short ones.  Against the
// one-thread-per-token kernel of dc_decode.hip: 4 x 8192 tokens x 4 KV heads,
// int8 keys and 3-bit values at head_dim 128, 4 queries per head: 237.7 ->
// 21.7 us; 3 x 2901 tokens x 6 KV heads at head_dim 96, 4-bit: 112.3 -> 16.3
// us.  (Values read from LDS one token at a time, with a branch per token:
// 43.2 and 32.2 us.)
#include "dc_decode.h"
#include "dc_unpack.h"

namespace dc {

namespace {

constexpr int kTileWaves = 4;
constexpr int kTile = 64;  // tokens per unit

// LDS of one unit's M0 values: code word w of group g as a row of 64 tokens
// (G W rows), scales as they come ([64][G] fp16) and as one row of 64 tokens
// per group, biases likewise.  Rows are padded by 16 bytes, so the rows that
// the lanes of one read touch start in different banks.
constexpr uint32_t kCodeRow = (kTile + 4) * 4, kScaleRow = (kTile + 8) * 2;
__host__ __device__ inline uint32_t raw_scale_bytes(uint32_t groups) { return (kTile * groups * 2 + 1023u) & ~1023u; }
__host__ __device__ inline uint32_t unit_bytes(uint32_t groups, uint32_t words, bool affine) {
  return groups * (words + 1) * kCodeRow + (raw_scale_bytes(groups) + groups * kScaleRow) * (affine ? 2u : 1u);
}

template <int N>
__device__ __forceinline__ float row_ror_max(float x) {
  return fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + N, 0xf,
                                                                        0xf, false)));
}

// Maximum over the wavefront, the same value in every lane.
__device__ __forceinline__ float wave_max_all(float x) {
  x = row_ror_max<8>(row_ror_max<4>(row_ror_max<2>(row_ror_max<1>(x))));
  auto at = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l)); };
  return fmaxf(fmaxf(at(0), at(16)), fmaxf(at(32), at(48)));
}

template <int N>
__device__ __forceinline__ float row_ror_add(float x) {
  return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + N, 0xf, 0xf, false));
}

// Sum over the wavefront, the same value in every lane.
__device__ __forceinline__ float wave_sum_all(float x) {
  x = row_ror_add<8>(row_ror_add<4>(row_ror_add<2>(row_ror_add<1>(x))));
  auto at = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l)); };
  return (at(0) + at(16)) + (at(32) + at(48));
}

// acc[n][c] += weights of token J (block J of a[n]) times v[c].
template <int J, int NB, int NS>
__device__ __forceinline__ void mix_token(const float (&a)[NB], const float (&v)[NS], f32x4v (&acc)[NB][NS]) {
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int c = 0; c < NS; ++c) acc[n][c] = mfma4_bcast<J>(a[n], v[c], acc[n][c]);
}

// fn(std::integral_constant<int, J>) for every J of the sequence.
template <typename F, int... J>
__device__ __forceinline__ void each(F&& fn, std::integer_sequence<int, J...>) {
  (fn(std::integral_constant<int, J>{}), ...);
}

typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

}  // namespace

template <int NB, int NS>
__global__ void __launch_bounds__(64 * kTileWaves, NB * NS <= 2 ? 4 : NB == 4 ? 2 : NB * NS <= 4 ? 3 : 2) decode_tiles_kernel(DecodeArgs a, uint32_t v_bytes) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ float ml[kTileWaves][4 * NB][2];
  // page records are indexed by the block alone: lane j's (page j of the
  // item) is loaded together with the item
  dc_page_record rec{};
  if (a.recs != nullptr) {
    const int slot = int(threadIdx.x & 63) < a.rec_stride ? int(threadIdx.x & 63) : a.rec_stride - 1;
    rec = a.recs[int64_t(blockIdx.x) * a.rec_stride + slot];
  }
  const dc_work_item it = a.items[blockIdx.x];
  if (!item_in_bounds(it, a)) return;
  const dc_page_geometry geo = a.kpool.geometry, vgeo = a.vpool.geometry;
  const int hd = geo.head_dim, C = geo.page_capacity, nq = a.n_q;
  const uint32_t kgroups = num_groups(geo), vgroups = num_groups(vgeo);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // LDS: query registers [hd / 16][NB][64], then per wave weights [64][4 NB]
  // and the unit's M0 values; the combine reuses all of it as [nq][hd]
  float* const qreg = reinterpret_cast<float*>(lds);
  const uint32_t q_bytes = uint32_t(hd) * NB * 16, p_bytes = kTile * 4 * NB * 4;
  uint8_t* const mine = lds + q_bytes + wave * (p_bytes + v_bytes);
  float* const prob = reinterpret_cast<float*>(mine);
  uint8_t* const vlds = mine + p_bytes;

  const int64_t stream = int64_t(it.seq) * a.n_kv_heads + it.kv_head, qbase = stream * nq * hd;
  for (int i = tid; i < hd * NB * 4; i += 64 * kTileWaves) {
    const int l = i & 63, n = (i >> 6) % NB, k = (i >> 6) / NB;
    const int j = 4 * n + (l & 3), c = 16 * k + (l >> 2);
    qreg[i] = j < nq ? load_value(a.queries, a.queries_dtype, qbase + int64_t(j) * hd + c) * a.q_scale : 0.f;
  }

  f32x4v acc[NB][NS];
  float m_ref[NB][4], l_sum[NB][4];
#pragma unroll
  for (int n = 0; n < NB; ++n) {
#pragma unroll
    for (int c = 0; c < NS; ++c) acc[n][c] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      m_ref[n][r] = -INFINITY;
      l_sum[n][r] = 0.f;
    }
  }
  // this lane's output channels c0 .. c0 + NS - 1 and their value group
  const bool ch_live = lane * NS < hd;
  const int c0 = ch_live ? lane * NS : 0, vg = c0 / vgeo.group_size, vk = c0 - vg * vgeo.group_size;
  __syncthreads();

  const int np = it.page_end - it.page_begin;
  int counter = 0;  // units walked so far, over the whole item
  for (int base = 0; base < np; base += 64) {
    // lane j: descriptors of page base + j of the item, its tokens [lo, hi)
    const int nb = np - base < 64 ? np - base : 64;
    uint32_t kblock = 0, vblock = 0;
    int fmts = 0, range = 0;
    if (lane < nb) {
      const int p = it.page_begin + base + lane;
      dc_page_desc kd{}, vd{};
      bool ok = true;
      if (a.recs != nullptr && np <= a.rec_stride) {
        kd = rec.key;  // (rec_stride <= 64: one batch)
        vd = rec.value;
      } else {
        const int32_t kid = a.k_table[stream * a.table_stride + p], vid = a.v_table[stream * a.table_stride + p];
        ok = kid >= 0 && kid < a.kpool.n_descs && vid >= 0 && vid < a.vpool.n_descs;
        if (ok) {
          kd = a.kpool.descs[kid];
          vd = a.vpool.descs[vid];
        }
      }
      const Blob32 KL = blob32(kd.format, kd.bits, geo, kgroups), VL = blob32(vd.format, vd.bits, vgeo, vgroups);
      ok = ok && (int64_t(kd.block) << 8) + KL.total <= a.kpool.arena_bytes &&
           (int64_t(vd.block) << 8) + VL.total <= a.vpool.arena_bytes &&
           (!is_m0(vd.format) || unit_bytes(VL.groups, VL.words, vd.format == DC_FMT_M0_AFFINE) <= v_bytes);
      int T = min(min(int(kd.tokens), int(vd.tokens)), C);
      // (the item may start and end inside a page, on 32-token chunks)
      const int lo = base + lane == 0 ? 32 * it.chunk_begin : 0;
      if (base + lane == np - 1 && it.chunk_end > 0) T = min(T, 32 * it.chunk_end);
      range = ok && T > lo ? lo | T << 16 : 0;
      kblock = kd.block;
      vblock = vd.block;
      fmts = int(kd.format) | int(kd.bits) << 8 | int(vd.format) << 16 | int(vd.bits) << 24;
    }
    for (int i = 0; i < nb; ++i) {
      const int rg = __builtin_amdgcn_readlane(range, i), hi = rg >> 16;
      for (int t0 = rg & 0xffff; t0 < hi; t0 += kTile) {
        if ((counter++ & (kTileWaves - 1)) != wave) continue;
        const int T = min(hi - t0, kTile);
        const uint32_t fm = uint32_t(__builtin_amdgcn_readlane(fmts, i));
        dc_page_desc kd{}, vd{};
        kd.block = uint32_t(__builtin_amdgcn_readlane(int(kblock), i));
        vd.block = uint32_t(__builtin_amdgcn_readlane(int(vblock), i));
        kd.format = uint8_t(fm);
        kd.bits = uint8_t(fm >> 8);
        vd.format = uint8_t(fm >> 16);
        vd.bits = uint8_t(fm >> 24);
        const Blob32 KL = blob32(kd.format, kd.bits, geo, kgroups), VL = blob32(vd.format, vd.bits, vgeo, vgroups);
        const uint8_t* kb = blob_ptr(a.kpool.arena, kd);
        const uint8_t* vb = blob_ptr(a.vpool.arena, vd);
        const bool vm0 = is_m0(vd.format), vaff = vd.format == DC_FMT_M0_AFFINE;
        const uint32_t G = vgroups, W = VL.words;
        // scales and biases: as they come, then by group
        uint8_t* const sraw = vlds + G * (W + 1) * kCodeRow;
        uint8_t* const srow = sraw + raw_scale_bytes(G);
        uint8_t* const braw = srow + G * kScaleRow;
        uint8_t* const brow = braw + raw_scale_bytes(G);

        // ---- the unit's M0 values -> LDS ----
        if (vm0) {
          const __amdgpu_buffer_rsrc_t rs =
              __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(vb), 0, int(VL.total), 0x00020000);
          const uint32_t row = W * 4, tstep = vgeo.layout == 0 ? row : G * row,
                         gstep = vgeo.layout == 0 ? uint32_t(C) * row : row;
          const int tok = int(uint32_t(t0 + lane) * tstep);  // (past the page: zeros, or another group's words)
          // (the previous unit's LDS reads are done before its buffer is refilled)
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          uint8_t* to = vlds;
          for (uint32_t g = 0; g < G; ++g)
            for (uint32_t w = 0; w < W; ++w, to += kCodeRow) {
              const int off = int(g * gstep + w * 4);
              __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)to, 4, tok, off, 0, 0);
            }
          for (uint32_t e0 = 0; e0 < kTile * G * 2; e0 += 1024) {
            const uint32_t e = e0 + 16 * lane;
            const int in = e < kTile * G * 2 ? int(uint32_t(t0) * G * 2 + e) : 0x7f000000;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(sraw + e0), 16, in,
                                                     int(VL.scales_off), 0, 0);
            if (vaff)
              __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(braw + e0), 16, in,
                                                       int(VL.bias_off), 0, 0);
          }
        }

        // ---- score and softmax: one token per lane ----
        const uint32_t tl = uint32_t(t0 + (lane < T ? lane : T - 1));
        f32x4v s0[NB], s1[NB];
#pragma unroll
        for (int n = 0; n < NB; ++n) s0[n] = s1[n] = f32x4v{0.f, 0.f, 0.f, 0.f};
        score_row<NB>(kd, geo, KL, kb, tl, [&](int32_t c, int n) { return qreg[(c / 16 * NB + n) * 64 + lane]; }, s0, s1);
        // (int8 value rows: their scale joins the weight)
        float vscale = 1.f;
        if (vd.format == DC_FMT_M3_I8) vscale = __half2float(reinterpret_cast<const __half*>(vb + VL.scales_off)[tl]);
        float lg[NB][4], m_new[NB][4];
        bool moved = false;
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            lg[n][r] = lane < T ? (s0[n][r] + s1[n][r]) * kLog2e : -INFINITY;
            m_new[n][r] = 4 * n + r < nq ? fmaxf(m_ref[n][r], wave_max_all(lg[n][r])) : m_ref[n][r];
            moved = moved || m_new[n][r] > m_ref[n][r];
          }
        if (moved) {
#pragma unroll
          for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float alpha = m_ref[n][r] == m_new[n][r] ? 1.f : exp2f(m_ref[n][r] - m_new[n][r]);
              m_ref[n][r] = m_new[n][r];
              l_sum[n][r] *= alpha;
#pragma unroll
              for (int c = 0; c < NS; ++c) acc[n][c][r] *= alpha;
            }
        }
#pragma unroll
        for (int n = 0; n < NB; ++n) {
          f32x4v p;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float w = 4 * n + r < nq && lane < T ? exp2f(lg[n][r] - m_ref[n][r]) : 0.f;
            l_sum[n][r] += w;
            p[r] = w * vscale;
          }
          *reinterpret_cast<f32x4v*>(prob + (lane * NB + n) * 4) = p;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        // weight register of tokens 16 r .. 16 r + 15: lane (b, i) = token 16 r + b, head i of block n
        auto weights = [&](int r, float (&w)[NB]) __attribute__((always_inline)) {
#pragma unroll
          for (int n = 0; n < NB; ++n) w[n] = prob[((16 * r + (lane >> 2)) * NB + n) * 4 + (lane & 3)];
        };

        // ---- mix: NS channels per lane, token by token ----
        if (vm0) {
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the DMA has landed
          // scales and biases by group; tokens past the unit get zeros, so
          // that whatever their codes are they add 0 x 0
          auto by_group = [&](const uint8_t* raw, uint8_t* rows) __attribute__((always_inline)) {
            const uint16_t* in = reinterpret_cast<const uint16_t*>(raw) + lane * G;
            uint16_t* out = reinterpret_cast<uint16_t*>(rows) + lane;
            for (uint32_t g = 0; g < G; g += 4) {
              uint16_t x[4];
#pragma unroll
              for (uint32_t i = 0; i < 4; ++i) x[i] = in[g + i < G ? g + i : G - 1];
#pragma unroll
              for (uint32_t i = 0; i < 4; ++i)
                if (g + i < G) out[(g + i) * (kScaleRow / 2)] = lane < T ? x[i] : uint16_t(0);
            }
          };
          by_group(sraw, srow);
          if (vaff) by_group(braw, brow);
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          const int bits = vd.bits, bit = vk * bits, shift = bit & 31;
          const uint8_t* cw = vlds + (vg * W + (bit >> 5)) * kCodeRow;
          const uint8_t* sp = srow + vg * kScaleRow;
          const uint8_t* bp = brow + vg * kScaleRow;
          const float zp = -float((1 << (bits - 1)) - 1);
          auto walk = [&](auto bits_c, auto aff) __attribute__((always_inline)) {
            constexpr int BITS = decltype(bits_c)::value;
            constexpr bool AFF = decltype(aff)::value;
            for (int r = 0; 16 * r < T; ++r) {
              float w[NB];
              weights(r, w);
              // 16 tokens: code words (two rows for 3-bit codes, whose
              // channels may straddle words), scales, biases
              u32x4v x[4], y[BITS == 3 ? 4 : 1], s[2], b[AFF ? 2 : 1];
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                x[i] = *reinterpret_cast<const u32x4v*>(cw + 64 * r + 16 * i);
                if constexpr (BITS == 3) y[i] = *reinterpret_cast<const u32x4v*>(cw + kCodeRow + 64 * r + 16 * i);
              }
#pragma unroll
              for (int i = 0; i < 2; ++i) {
                s[i] = *reinterpret_cast<const u32x4v*>(sp + 32 * r + 16 * i);
                if constexpr (AFF) b[i] = *reinterpret_cast<const u32x4v*>(bp + 32 * r + 16 * i);
              }
              each([&](auto j) __attribute__((always_inline)) {
                constexpr int J = decltype(j)::value;
                uint32_t c = x[J / 4][J % 4];
                if constexpr (BITS == 3)
                  c = __builtin_amdgcn_alignbit(y[J / 4][J % 4], c, shift);
                else
                  c >>= shift;
                const float sc = half_bits(s[J / 8][J % 8 / 2], J & 1);
                const float bs = AFF ? half_bits(b[AFF ? J / 8 : 0][J % 8 / 2], J & 1) : zp * sc;
                float v[NS];
#pragma unroll
                for (int k = 0; k < NS; ++k) v[k] = fmaf(float((c >> (BITS * k)) & ((1u << BITS) - 1u)), sc, bs);
                mix_token<J>(w, v, acc);
              }, std::make_integer_sequence<int, 16>{});
            }
          };
          auto by_bits = [&](auto aff) __attribute__((always_inline)) {
            if (bits == 4)
              walk(std::integral_constant<int, 4>{}, aff);
            else if (bits == 8)
              walk(std::integral_constant<int, 8>{}, aff);
            else if (bits == 3)
              walk(std::integral_constant<int, 3>{}, aff);
            else
              walk(std::integral_constant<int, 2>{}, aff);
          };
          if (vaff)
            by_bits(std::true_type{});
          else
            by_bits(std::false_type{});
        } else {
          // escape rows: NS elements per lane, the next S tokens' loads in
          // flight while S are summed (a token past the unit reloads its
          // last one and counts as zeros)
          auto walk = [&](auto elem) __attribute__((always_inline)) {
            using E = decltype(elem);
            struct alignas(sizeof(E) * NS) Piece {
              E e[NS];
            };
            constexpr int S = sizeof(Piece) > 8 ? 4 : 8;
            const E* rows = reinterpret_cast<const E*>(vb) + int64_t(t0) * hd + c0;
            Piece x[2][S];
            auto load = [&](int first, Piece (&to)[S]) __attribute__((always_inline)) {
#pragma unroll
              for (int j = 0; j < S; ++j) to[j] = *reinterpret_cast<const Piece*>(rows + int64_t(min(first + j, T - 1)) * hd);
            };
            load(0, x[0]);
            for (int r = 0; 16 * r < T; ++r) {
              float w[NB];
              weights(r, w);
              each([&](auto h) __attribute__((always_inline)) {
                constexpr int H = decltype(h)::value;
                const int left = T - 16 * r - S * H;
                if (left <= 0) return;
                if (left > S) load(16 * r + S * H + S, x[1 - H % 2]);
                each([&](auto j) __attribute__((always_inline)) {
                  constexpr int J = decltype(j)::value;
                  float v[NS];
#pragma unroll
                  for (int c = 0; c < NS; ++c) v[c] = J < left ? float(x[H % 2][J].e[c]) : 0.f;
                  mix_token<S * H + J>(w, v, acc);
                }, std::make_integer_sequence<int, S>{});
              }, std::make_integer_sequence<int, 16 / S>{});
            }
          };
          if (vd.format == DC_FMT_M3_F16)
            walk(_Float16{});
          else if (vd.format == DC_FMT_M3_F32)
            walk(float{});
          else
            walk(int8_t{});
        }
      }
    }
  }

  const int used = counter < kTileWaves ? counter : kTileWaves;  // waves that had a unit
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) l_sum[n][r] = wave_sum_all(l_sum[n][r]);
  if (it.partial >= a.max_partials) return;
  float* const dst = it.partial < 0 ? a.out + qbase : a.part_o + int64_t(it.partial) * nq * hd;
  float* const dst_ml = a.part_ml + int64_t(it.partial) * nq * 2;
  if (used <= 1) {  // one unit (or none): wave 0 holds the item's result
    if (wave != 0) return;
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = 4 * n + r;
        if (j >= nq) continue;
        const float den = it.partial < 0 ? fmaxf(l_sum[n][r], 1e-30f) : 1.f;
#pragma unroll
        for (int c = 0; c < NS; ++c)
          if (ch_live) dst[j * hd + c0 + c] = acc[n][c][r] / den;
        if (it.partial >= 0 && lane == 0) {
          dst_ml[2 * j] = m_ref[n][r];
          dst_ml[2 * j + 1] = l_sum[n][r];
        }
      }
    return;
  }

  // ---- the waves' (m, l, o) -> one ----
  if (lane == 0) {
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ml[wave][4 * n + r][0] = m_ref[n][r];
        ml[wave][4 * n + r][1] = l_sum[n][r];
      }
  }
  __syncthreads();  // (every wave is past its unit's LDS)
  // each wave scales its output to the common maximum and adds it in LDS in
  // wave order
  float* const red = reinterpret_cast<float*>(lds);
  float scale[NB][4];
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float M = ml[0][4 * n + r][0];
#pragma unroll
      for (int u = 1; u < kTileWaves; ++u) M = fmaxf(M, ml[u][4 * n + r][0]);
      scale[n][r] = m_ref[n][r] == M ? 1.f : exp2f(m_ref[n][r] - M);
    }
  for (int w = 0; w < used; ++w) {
    if (w == wave && ch_live) {
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (4 * n + r >= nq) continue;
#pragma unroll
          for (int c = 0; c < NS; ++c) {
            float* o = red + (4 * n + r) * hd + c0 + c;
            const float x = acc[n][c][r] * scale[n][r];
            *o = w == 0 ? x : *o + x;
          }
        }
    }
    __syncthreads();
  }
  for (int j = wave; j < nq; j += kTileWaves) {
    float M = ml[0][j][0], l = 0.f;
#pragma unroll
    for (int u = 1; u < kTileWaves; ++u) M = fmaxf(M, ml[u][j][0]);
#pragma unroll
    for (int u = 0; u < kTileWaves; ++u) l += u < used ? ml[u][j][1] * (ml[u][j][0] == M ? 1.f : exp2f(ml[u][j][0] - M)) : 0.f;
    const float den = it.partial < 0 ? fmaxf(l, 1e-30f) : 1.f;
    for (int c = lane; c < hd; c += 64) dst[j * hd + c] = red[j * hd + c] / den;
    if (it.partial >= 0 && lane == 0) {
      dst_ml[2 * j] = M;
      dst_ml[2 * j + 1] = l;
    }
  }
}

// Takes every geometry that 16-channel chunks tile in both pools.  *launched
// tells the caller whether to fall back to the one-thread-per-token kernel.
int launch_decode_tiles(const DecodeArgs& a, hipStream_t stream, bool* launched) {
  *launched = false;
  const dc_page_geometry& g = a.kpool.geometry;
  const dc_page_geometry& vg = a.vpool.geometry;
  if (!chunk16_geometry(g) || !chunk16_geometry(vg)) return DC_OK;
  // LDS for the widest M0 values the pool may hold
  uint32_t v_bytes = 0;
  for (int bits : {2, 3, 4, 8})
    for (int fmt : {DC_FMT_M0_AFFINE, DC_FMT_M0_SYMMETRIC})
      if (a.vpool.format_mask == 0 || (a.vpool.format_mask >> (fmt * 9 + bits) & 1)) {
        const uint32_t n = unit_bytes(num_groups(vg), words_per_group(vg.group_size, bits), fmt == DC_FMT_M0_AFFINE);
        v_bytes = n > v_bytes ? n : v_bytes;
      }
  const int hd = g.head_dim, nb = a.n_q <= 4 ? 1 : a.n_q <= 8 ? 2 : 4;
  uint32_t lds = uint32_t(hd) * nb * 16 + kTileWaves * (kTile * 16 * nb + v_bytes);
  if (lds < uint32_t(a.n_q) * hd * 4) lds = uint32_t(a.n_q) * hd * 4;
  if (lds > 150 * 1024) return DC_OK;
#define DC_TILES(NB_, NS_) \
  hipLaunchKernelGGL((decode_tiles_kernel<NB_, NS_>), dim3(uint32_t(a.n_items)), dim3(64 * kTileWaves), lds, stream, a, v_bytes)
#define DC_TILES_NS(NB_)  \
  if (hd <= 64)           \
    DC_TILES(NB_, 1);     \
  else if (hd <= 128)     \
    DC_TILES(NB_, 2);     \
  else                    \
    DC_TILES(NB_, 4)
  if (nb == 1) {
    DC_TILES_NS(1);
  } else if (nb == 2) {
    DC_TILES_NS(2);
  } else {
    DC_TILES_NS(4);
  }
#undef DC_TILES_NS
#undef DC_TILES
  *launched = true;
  return check_hip(hipGetLastError(), "decode_tiles_kernel launch");
}

}  // namespace dc
