// Per-page score and mix entry points (the score_page / mix_page surface).
//
// These serve the reference's page-at-a-time API and its parity tests; the
// fused decode kernel (dc_decode.hip) is the throughput path.  The
// arithmetic follows the reference's streaming form
// (dotcache/attention_reference.py:97-126, :165-192): per group,
// s * (codes . q_g) + b * sum(q_g) for affine pages, s * ((codes - zp) . q_g)
// for symmetric pages, fp32 escape rows for M3 pages.
#include "dc_common.h"
#include "dc_unpack.h"

namespace dc {

constexpr int kScoreQ = 8;  // queries scored per pass

// Geometries that 16-channel chunks do not tile: grid.x = page index, grid.y
// = query chunk; one thread per token.  With
// page_group, page i is scored against the queries of group page_group[i]
// (queries [n_groups][n_queries][hd]) into logits rows
// group * n_queries + q; without it every page belongs to group 0.
__global__ void __launch_bounds__(256) score_pages_kernel(dc_pool pool, const int32_t* __restrict__ page_ids,
                                                          const int32_t* __restrict__ token_offsets,
                                                          const int32_t* __restrict__ page_group, int32_t n_groups,
                                                          const float* __restrict__ queries_all, int32_t n_queries,
                                                          float* __restrict__ logits_all, int64_t logits_stride) {
  const int32_t i = blockIdx.x;
  const int32_t q0 = blockIdx.y * kScoreQ;
  const int32_t grp = page_group ? page_group[i] : 0;
  if (grp < 0 || grp >= n_groups) return;
  const float* queries = queries_all + int64_t(grp) * n_queries * pool.geometry.head_dim;
  float* logits = logits_all + int64_t(grp) * n_queries * logits_stride;
  const int32_t pid = page_ids[i];
  if (pid < 0 || pid >= pool.n_descs) return;
  const dc_page_desc d = pool.descs[pid];
  const dc_page_geometry geo = pool.geometry;
  const BlobLayout L = blob_layout(d.format, d.bits, geo);
  if ((int64_t(d.block) << 8) + L.total > pool.arena_bytes) return;
  const uint8_t* blob = blob_ptr(pool.arena, d);
  const int32_t off = token_offsets[i];
  const int32_t T = d.tokens < geo.page_capacity ? d.tokens : geo.page_capacity;
  const int32_t nq = n_queries - q0 < kScoreQ ? n_queries - q0 : kScoreQ;
  const int32_t G = L.groups, gs = geo.group_size, hd = geo.head_dim;

  for (int32_t t = threadIdx.x; t < T; t += blockDim.x) {
    float acc[kScoreQ];
#pragma unroll
    for (int j = 0; j < kScoreQ; ++j) acc[j] = 0.f;
    if (is_m0(d.format)) {
      const uint32_t* payload = reinterpret_cast<const uint32_t*>(blob);
      const __half* sc = reinterpret_cast<const __half*>(blob + L.scales_off);
      const __half* bs = reinterpret_cast<const __half*>(blob + L.bias_off);
      const float zp = float((1 << (d.bits - 1)) - 1);
      for (int32_t g = 0; g < G; ++g) {
        float dot[kScoreQ], qs[kScoreQ];
#pragma unroll
        for (int j = 0; j < kScoreQ; ++j) dot[j] = qs[j] = 0.f;
        for (int32_t k = 0; k < gs; ++k) {
          const int32_t c = g * gs + k;
          if (c >= hd) break;  // padded channels meet zero-padded queries
          float code = float(m0_code(payload, t, g, k, d.bits, L.words, G, geo.page_capacity, geo.layout));
          if (d.format == DC_FMT_M0_SYMMETRIC) code -= zp;
#pragma unroll
          for (int j = 0; j < kScoreQ; ++j) {
            if (j < nq) {
              const float qv = queries[int64_t(q0 + j) * hd + c];
              dot[j] += code * qv;
              qs[j] += qv;
            }
          }
        }
        const float s = __half2float(sc[t * G + g]);
        const float b = d.format == DC_FMT_M0_AFFINE ? __half2float(bs[t * G + g]) : 0.f;
#pragma unroll
        for (int j = 0; j < kScoreQ; ++j) acc[j] += s * dot[j] + b * qs[j];
      }
    } else {
      for (int32_t c = 0; c < hd; ++c) {
        const float v = page_value(blob, d, L, geo, t, c);
#pragma unroll
        for (int j = 0; j < kScoreQ; ++j)
          if (j < nq) acc[j] += v * queries[int64_t(q0 + j) * hd + c];
      }
    }
#pragma unroll
    for (int j = 0; j < kScoreQ; ++j)
      if (j < nq) logits[int64_t(q0 + j) * logits_stride + off + t] = acc[j];
  }
}

// ---- score over 64-token tiles --------------------------------------------
//
// One wavefront scores 64 tokens of a page, one per lane, for 4 NB queries:
// the lane unpacks its token's 16-channel chunks (contiguous words across
// the lanes) and v_mfma_f32_4x4x1 multiplies each channel with four queries
// at once, the queries (one chunk of four per register) broadcast from the A
// operand's blocks.  No value crosses lanes and the logits leave in token
// order.  Products and sums are fp32.  A page's words are read once for 4 NB
// queries; the next chunks' words fly while one is multiplied.  A launch of a
// few thousand tokens is bound by its chain of dependent loads (id,
// descriptor, words).  4096 tokens of 4-bit pages at head_dim 128: one query
// 36.6 -> 4.6 us, 8 groups of 3 queries 51.8 -> 5.0 (a third slower with scales
// converted where they are loaded, which waits for each load).
template <int NB>
__global__ void __launch_bounds__(64) score_tiles_kernel(dc_pool pool, const int32_t* __restrict__ page_ids,
                                                         const int32_t* __restrict__ token_offsets,
                                                         const int32_t* __restrict__ page_group, int32_t n_groups,
                                                         const float* __restrict__ queries_all, int32_t n_queries,
                                                         float* __restrict__ logits_all, int64_t logits_stride,
                                                         int32_t units_per_page) {
  const dc_page_geometry geo = pool.geometry;
  const int32_t i = blockIdx.x / units_per_page, t0 = int32_t(blockIdx.x - uint32_t(i) * units_per_page) * 64;
  const int32_t q0 = blockIdx.y * 4 * NB, hd = geo.head_dim;
  const int lane = threadIdx.x;
  const int32_t grp = page_group ? page_group[i] : 0, pid = page_ids[i], off = token_offsets[i];
  if (grp < 0 || grp >= n_groups || pid < 0 || pid >= pool.n_descs) return;
  const dc_page_desc d = pool.descs[pid];
  const Blob32 L = blob32(d.format, d.bits, geo, num_groups(geo));
  if ((int64_t(d.block) << 8) + L.total > pool.arena_bytes) return;
  const int32_t T = (d.tokens < geo.page_capacity ? d.tokens : geo.page_capacity) - t0;
  if (T <= 0) return;
  const uint8_t* blob = blob_ptr(pool.arena, d);
  const uint32_t t = uint32_t(t0 + (lane < T ? lane : T - 1));  // (lanes past the page repeat its last token)

  // lane (b, r) of a query register: channel 16 k + b of query q0 + 4 n + r
  const float* qp[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const int32_t q = q0 + 4 * n + (lane & 3);
    // (a head past the last repeats the block's first: its sums are not stored)
    qp[n] = queries_all + (int64_t(grp) * n_queries + (q < n_queries ? q : q0)) * hd + (lane >> 2);
  }
  f32x4v s0[NB], s1[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) s0[n] = s1[n] = f32x4v{0.f, 0.f, 0.f, 0.f};

  score_row<NB>(d, geo, L, blob, t, [&](int32_t c0, int n) { return qp[n][c0]; }, s0, s1);
  if (lane >= T) return;
  float* logits = logits_all + (int64_t(grp) * n_queries + q0) * logits_stride + off + t0 + lane;
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (q0 + 4 * n + r < n_queries) logits[int64_t(4 * n + r) * logits_stride] = s0[n][r] + s1[n][r];
}

// ---- mix over 16-channel slices -------------------------------------------
//
// out[q, c] (+)= sum over tokens of w[q, t] V[t, c] for 16 channels c0 ..
// c0 + 15 and QB queries per block of kMixWaves wavefronts.  The tokens of
// the group's pages are cut into units of 64; wave w takes units w, w +
// kMixWaves, ..., one token per lane, so code words and weights are read
// contiguously and every lane keeps QB x 16 sums in registers.  The lanes'
// sums meet in a butterfly that halves them at each step, the waves' in LDS,
// in a fixed order.  What bounds it at these sizes is latency: the chain page
// id -> descriptor -> words is walked once per 64 units (lane j holds unit
// j's page), and unit j + 1's words are in flight while unit j is summed.
// One block per slice rather than per query head: a single query's 128
// channels run on 8 CUs instead of one, 1024 tokens at a time.  4096 tokens of
// 4-bit pages at head_dim 128: one query 1135 -> 9.5 us, 8 groups of 3
// queries 1146 -> 10.8 us (14.2 in 8 waves, 16.6 in blocks of 4 queries; a
// third unit in flight does not fit 1024 threads' registers).
template <int QB, int kMixWaves>
__global__ void __launch_bounds__(64 * kMixWaves) mix_slices_kernel(
    dc_pool pool, const int32_t* __restrict__ page_ids, const int32_t* __restrict__ token_offsets, int32_t n_pages,
    const int32_t* __restrict__ group_pages, int32_t n_queries, const float* __restrict__ weights,
    int64_t weights_stride, float* out, int32_t accumulate) {
  __shared__ float part[kMixWaves][QB * 16];
  const dc_page_geometry geo = pool.geometry;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int32_t grp = blockIdx.z, q0 = blockIdx.y * QB, c0 = blockIdx.x * 16, C = geo.page_capacity;
  const uint32_t groups = num_groups(geo);
  const int nq = n_queries - q0 < QB ? n_queries - q0 : QB;
  int32_t i0 = 0, i1 = n_pages;
  if (group_pages) {
    i0 = group_pages[grp] < 0 ? 0 : group_pages[grp];
    i1 = group_pages[grp + 1] > n_pages ? n_pages : group_pages[grp + 1];
  }
  const float* w0 = weights + (int64_t(grp) * n_queries + q0) * weights_stride;
  const int32_t upp = (C + 63) >> 6;  // units per page
  const int64_t units = i1 > i0 ? int64_t(i1 - i0) * upp : 0;

  float acc[QB][16];
#pragma unroll
  for (int q = 0; q < QB; ++q)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[q][i] = 0.f;

  struct Unit {  // one unit's loads: raw words, scale, bias, weights of this lane's token
    uint32_t r[16];
    uint16_t s, b;
    float w[QB];
    int kind, format, bits, shift;
    bool live;
  };
  for (int64_t base = wave; base < units; base += 64 * kMixWaves) {
    // lane j: the page of unit base + kMixWaves j
    const int64_t u = base + int64_t(kMixWaves) * lane;
    int32_t block = 0, info = 0, off = 0, sub = 0;
    if (u < units) {
      const int32_t i = i0 + int32_t(u / upp);
      sub = int32_t(u - int64_t(i - i0) * upp) * 64;
      const int32_t pid = page_ids[i];
      off = token_offsets[i] + sub;
      if (pid >= 0 && pid < pool.n_descs) {
        const dc_page_desc d = pool.descs[pid];
        const Blob32 L = blob32(d.format, d.bits, geo, groups);
        const int32_t T = (d.tokens < C ? d.tokens : C) - sub;
        if ((int64_t(d.block) << 8) + L.total <= pool.arena_bytes && T > 0) {
          block = int32_t(d.block);
          info = (T < 64 ? T : 64) | int32_t(d.format) << 8 | int32_t(d.bits) << 16;
        }
      }
    }
    const int64_t left = (units - base + kMixWaves - 1) / kMixWaves;
    const int n = left < 64 ? int(left) : 64;

    auto load = [&](int j, Unit& x) __attribute__((always_inline)) {
      const int32_t inf = __builtin_amdgcn_readlane(info, j);
      dc_page_desc d{};
      d.block = uint32_t(__builtin_amdgcn_readlane(block, j));
      d.format = uint8_t(inf >> 8);
      d.bits = uint8_t(inf >> 16);
      const int32_t T = inf & 0xff, o = __builtin_amdgcn_readlane(off, j), t0 = __builtin_amdgcn_readlane(sub, j);
      x.kind = T > 0 ? chunk_kind(d.format, d.bits) : CK_NONE;
      x.format = d.format;
      x.bits = d.bits;
      if (x.kind == CK_NONE) return;
      const Blob32 L = blob32(d.format, d.bits, geo, groups);
      const Chunk16 ck = chunk16_at(d.format, d.bits, geo, L, c0);
      x.shift = ck.shift();
      // (a lane past the page's tokens reads its last token, and adds nothing)
      x.live = lane < T;
      const uint32_t tok = x.live ? lane : T - 1, t = uint32_t(t0) + tok;
      const uint8_t* blob = blob_ptr(pool.arena, d);
      // Loads only: conversions wait until the unit is summed, or each load
      // would be waited for where it was issued.
      load_chunk16(x.kind, blob + ck.word() + t * ck.word_step, x.r);
      if (x.kind != CK_F16 && x.kind != CK_F32) {
        x.s = *reinterpret_cast<const uint16_t*>(blob + ck.scale + t * ck.scale_step);
        // (no bias: the scale again, unused)
        x.b = *reinterpret_cast<const uint16_t*>(blob + (d.format == DC_FMT_M0_AFFINE ? ck.bias : ck.scale) + t * ck.scale_step);
      }
#pragma unroll
      for (int q = 0; q < QB; ++q) x.w[q] = w0[int64_t(q < nq ? q : 0) * weights_stride + o + int32_t(tok)];
    };
    auto sum = [&](const Unit& x) __attribute__((always_inline)) {
      for_chunk_kind(x.kind, [&](auto k) __attribute__((always_inline)) {
        constexpr int K = decltype(k)::value;
        float v[16], s = 1.f, b = 0.f;
        if constexpr (K != CK_F16 && K != CK_F32) {
          s = half_bits(x.s, 0);
          b = x.format == DC_FMT_M0_AFFINE ? half_bits(x.b, 0) : K == CK_I8 ? 0.f : -float((1 << (x.bits - 1)) - 1) * s;
        }
        values16<K>(x.r, x.shift, s, b, v);
        if (!x.live) return;
#pragma unroll
        for (int q = 0; q < QB; ++q)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[q][i] = fmaf(x.w[q], v[i], acc[q][i]);
      });
    };
    Unit A, B;
    load(0, A);
    for (int j = 0; j < n; j += 2) {
      if (j + 1 < n) load(j + 1, B);
      sum(A);
      if (j + 1 >= n) break;
      if (j + 2 < n) load(j + 2, A);
      sum(B);
    }
  }

  // Lanes: at each step a lane keeps one half of its sums and adds its
  // partner's copy of that half, so N sums take N - 1 exchanges; once one
  // sum is left the remaining steps add whole copies.  With N = 16 QB sums
  // the lane's sum is number (lane >> (6 - log2 N)) counted from the top bit.
  float* f = &acc[0][0];
  int idx = 0;
#pragma unroll
  for (int step = 0; step < 6; ++step) {
    const int o = 32 >> step, n = (16 * QB) >> step;  // sums before this step
    if (n > 1) {
      const bool up = (lane & o) != 0;
      idx = 2 * idx + (up ? 1 : 0);
#pragma unroll
      for (int i = 0; i < n / 2; ++i) {
        const float send = up ? f[i] : f[i + n / 2];
        const float keep = up ? f[i + n / 2] : f[i];
        f[i] = keep + __shfl_xor(send, o, 64);
      }
    } else {
      f[0] += __shfl_xor(f[0], o, 64);
    }
  }
  part[wave][idx] = f[0];  // (lanes that share a sum write the same value)
  __syncthreads();
  const int k = threadIdx.x;
  if (k < 16 * QB && k / 16 < nq) {
    float total = part[0][k];
#pragma unroll
    for (int w = 1; w < kMixWaves; ++w) total += part[w][k];
    float* o = out + (int64_t(grp) * n_queries + q0 + k / 16) * geo.head_dim + c0 + k % 16;
    *o = accumulate ? *o + total : total;
  }
}

// Geometries whose groups or rows are no multiple of 16 channels: grid.x =
// query row (group * n_queries + q), grid.y = channel block; one thread per
// channel, looping over the pages of the row's group
// [group_pages[g], group_pages[g + 1]) (every page without group_pages) and
// their tokens.
__global__ void __launch_bounds__(256) mix_pages_kernel(dc_pool pool, const int32_t* __restrict__ page_ids,
                                                        const int32_t* __restrict__ token_offsets, int32_t n_pages,
                                                        const int32_t* __restrict__ group_pages, int32_t n_queries,
                                                        const float* __restrict__ weights, int64_t weights_stride,
                                                        float* __restrict__ out, int32_t accumulate) {
  const int32_t q = blockIdx.x;
  const int32_t c = blockIdx.y * blockDim.x + threadIdx.x;
  const dc_page_geometry geo = pool.geometry;
  if (c >= geo.head_dim) return;
  const float* w = weights + int64_t(q) * weights_stride;
  int32_t i0 = 0, i1 = n_pages;
  if (group_pages) {
    const int32_t g = q / n_queries;
    i0 = group_pages[g] < 0 ? 0 : group_pages[g];
    i1 = group_pages[g + 1] > n_pages ? n_pages : group_pages[g + 1];
  }
  float acc = 0.f;
  for (int32_t i = i0; i < i1; ++i) {
    const int32_t pid = page_ids[i];
    if (pid < 0 || pid >= pool.n_descs) continue;
    const dc_page_desc d = pool.descs[pid];
    const BlobLayout L = blob_layout(d.format, d.bits, geo);
    if ((int64_t(d.block) << 8) + L.total > pool.arena_bytes) continue;
    const uint8_t* blob = blob_ptr(pool.arena, d);
    const int32_t off = token_offsets[i];
    const int32_t T = d.tokens < geo.page_capacity ? d.tokens : geo.page_capacity;
    for (int32_t t = 0; t < T; ++t) acc += w[off + t] * page_value(blob, d, L, geo, t, c);
  }
  float* o = out + int64_t(q) * geo.head_dim + c;
  *o = accumulate ? *o + acc : acc;
}

}  // namespace dc

static int score_launch(const dc_pool& pool, const int32_t* page_ids, const int32_t* token_offsets,
                        const int32_t* page_group, int32_t n_groups, int32_t n_pages, const float* queries,
                        int32_t n_queries, float* logits, int64_t logits_stride, hipStream_t stream, const char* who) {
  if (int rc = dc::validate_geometry(pool.geometry)) return rc;
  if (n_pages < 0 || n_queries < 0 || n_groups <= 0) return dc::fail(DC_EINVAL, "%s: bad counts", who);
  if (n_pages == 0 || n_queries == 0) return DC_OK;
  if (!page_ids || !token_offsets || !queries || !logits || !pool.arena || !pool.descs)
    return dc::fail(DC_EINVAL, "%s: null pointer", who);
  const int32_t upp = (pool.geometry.page_capacity + 63) / 64;
  if (dc::chunk16_geometry(pool.geometry) && int64_t(n_pages) * upp < (int64_t(1) << 31) && n_queries <= 65535) {
    // (queries per pass over the words: as many as there are, up to 16)
    const int nb = n_queries <= 4 ? 1 : n_queries <= 8 ? 2 : 4;
    const dim3 grid(uint32_t(n_pages * upp), uint32_t((n_queries + 4 * nb - 1) / (4 * nb)));
#define DC_SCORE(NB_)                                                                                              \
  hipLaunchKernelGGL((dc::score_tiles_kernel<NB_>), grid, dim3(64), 0, stream, pool, page_ids, token_offsets, page_group, \
                     n_groups, queries, n_queries, logits, logits_stride, upp)
    if (nb == 1)
      DC_SCORE(1);
    else if (nb == 2)
      DC_SCORE(2);
    else
      DC_SCORE(4);
#undef DC_SCORE
    return dc::check_hip(hipGetLastError(), who);
  }
  const uint32_t qchunks = uint32_t((n_queries + dc::kScoreQ - 1) / dc::kScoreQ);
  hipLaunchKernelGGL(dc::score_pages_kernel, dim3(uint32_t(n_pages), qchunks), dim3(128), 0, stream, pool, page_ids,
                     token_offsets, page_group, n_groups, queries, n_queries, logits, logits_stride);
  return dc::check_hip(hipGetLastError(), who);
}

static int mix_launch(const dc_pool& pool, const int32_t* page_ids, const int32_t* token_offsets, int32_t n_pages,
                      const int32_t* group_pages, int32_t n_groups, const float* weights, int32_t n_queries,
                      int64_t weights_stride, float* out, int32_t accumulate, hipStream_t stream, const char* who) {
  if (int rc = dc::validate_geometry(pool.geometry)) return rc;
  if (n_pages < 0 || n_queries < 0 || n_groups <= 0) return dc::fail(DC_EINVAL, "%s: bad counts", who);
  if (n_queries == 0) return DC_OK;
  if (!weights || !out || (n_pages > 0 && (!page_ids || !token_offsets || !pool.arena || !pool.descs)))
    return dc::fail(DC_EINVAL, "%s: null pointer", who);
  if (dc::chunk16_geometry(pool.geometry) && n_groups <= 65535 && n_queries <= 65535) {
    // blocks of 2 queries (32 sums per lane) where there are two
    const int qb = n_queries >= 2 ? 2 : 1;
    const dim3 grid(uint32_t(pool.geometry.head_dim / 16), uint32_t((n_queries + qb - 1) / qb), uint32_t(n_groups));
#define DC_MIX(QB_, W_)                                                                                              \
  hipLaunchKernelGGL((dc::mix_slices_kernel<QB_, W_>), grid, dim3(64 * W_), 0, stream, pool, page_ids,               \
                     token_offsets, n_pages, group_pages, n_queries, weights, weights_stride, out, accumulate)
    if (qb == 1)
      DC_MIX(1, 16);
    else
      DC_MIX(2, 16);
#undef DC_MIX
    return dc::check_hip(hipGetLastError(), who);
  }
  const uint32_t cblocks = uint32_t((pool.geometry.head_dim + 255) / 256);
  hipLaunchKernelGGL(dc::mix_pages_kernel, dim3(uint32_t(n_groups) * uint32_t(n_queries), cblocks), dim3(256), 0,
                     stream, pool, page_ids, token_offsets, n_pages, group_pages, n_queries, weights, weights_stride,
                     out, accumulate);
  return dc::check_hip(hipGetLastError(), who);
}

extern "C" int dc_score_pages(dc_pool pool, const int32_t* page_ids, const int32_t* token_offsets, int32_t n_pages,
                              const float* queries, int32_t n_queries, float* logits, int64_t logits_stride,
                              dc_stream_t stream) {
  return score_launch(pool, page_ids, token_offsets, nullptr, 1, n_pages, queries, n_queries, logits, logits_stride,
                      hipStream_t(stream), "dc_score_pages");
}

extern "C" int dc_mix_pages(dc_pool pool, const int32_t* page_ids, const int32_t* token_offsets, int32_t n_pages,
                            const float* weights, int32_t n_queries, int64_t weights_stride, float* out,
                            int32_t accumulate, dc_stream_t stream) {
  return mix_launch(pool, page_ids, token_offsets, n_pages, nullptr, 1, weights, n_queries, weights_stride, out,
                    accumulate, hipStream_t(stream), "dc_mix_pages");
}

extern "C" int dc_score_pages_grouped(dc_pool pool, const int32_t* page_ids, const int32_t* token_offsets,
                                      const int32_t* page_group, int32_t n_groups, int32_t n_pages,
                                      const float* queries, int32_t n_queries, float* logits, int64_t logits_stride,
                                      dc_stream_t stream) {
  if (n_pages > 0 && !page_group) return dc::fail(DC_EINVAL, "dc_score_pages_grouped: null page_group");
  return score_launch(pool, page_ids, token_offsets, page_group, n_groups, n_pages, queries, n_queries, logits,
                      logits_stride, hipStream_t(stream), "dc_score_pages_grouped");
}

extern "C" int dc_mix_pages_grouped(dc_pool pool, const int32_t* page_ids, const int32_t* token_offsets,
                                    const int32_t* group_pages, int32_t n_groups, int32_t n_pages,
                                    const float* weights, int32_t n_queries, int64_t weights_stride, float* out,
                                    int32_t accumulate, dc_stream_t stream) {
  if (!group_pages) return dc::fail(DC_EINVAL, "dc_mix_pages_grouped: null group_pages");
  return mix_launch(pool, page_ids, token_offsets, n_pages, group_pages, n_groups, weights, n_queries, weights_stride,
                    out, accumulate, hipStream_t(stream), "dc_mix_pages_grouped");
}

namespace dc {

// Softmax of each row (reference attention_reference.py:27-31): exp(x - max)
// / sum, fp32, one block of T threads per row, from src to dst (which may be
// the same row).  Up to kSoftmaxRegs columns per thread stay in registers
// between the passes (SKIP: columns past the row's end cost no instructions;
// rows that fill the registers run faster without the branches, 1024 rows of
// 8192 columns 13.5 us against 14.5); longer rows are read again (from dst
// once the exponentials are there).  Bound by latency: one load round, two
// block reductions (24 rows of 4096: 9.9 -> 3.9 us, 8192 rows of 200: 10.2 ->
// 6.3; 256 threads walked the row three times).
constexpr int kSoftmaxRegs = 8;
template <int T, bool SKIP>
__global__ void __launch_bounds__(T) softmax_rows_kernel(const float* src, int64_t src_stride, float* dst,
                                                         int64_t dst_stride, int32_t n_cols) {
  const float* x = src + int64_t(blockIdx.x) * src_stride;
  float* y = dst + int64_t(blockIdx.x) * dst_stride;
  constexpr int kWaves = T / 64;
  __shared__ float red[2][kWaves];
  const int tid = threadIdx.x;
  float v[kSoftmaxRegs];
  // (every load of the row in flight: a clamped column, masked)
#pragma unroll
  for (int k = 0; k < kSoftmaxRegs; ++k) {
    if (SKIP && T * k >= n_cols) break;
    const int32_t i = tid + T * k;
    v[k] = x[i < n_cols ? i : n_cols - 1];
  }
  float mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < kSoftmaxRegs; ++k) {
    if (SKIP && T * k >= n_cols) break;
    mx = tid + T * k < n_cols ? fmaxf(mx, v[k]) : mx;
  }
  for (int32_t i = tid + T * kSoftmaxRegs; i < n_cols; i += T) mx = fmaxf(mx, x[i]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if (tid % 64 == 0) red[0][tid / 64] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, red[0][w]);
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < kSoftmaxRegs; ++k) {
    if (SKIP && T * k >= n_cols) break;
    v[k] = expf(v[k] - mx);
    sum += tid + T * k < n_cols ? v[k] : 0.f;
  }
  for (int32_t i = tid + T * kSoftmaxRegs; i < n_cols; i += T) {
    const float e = expf(x[i] - mx);
    y[i] = e;
    sum += e;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  if (tid % 64 == 0) red[1][tid / 64] = sum;
  __syncthreads();
  sum = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) sum += red[1][w];
#pragma unroll
  for (int k = 0; k < kSoftmaxRegs; ++k)
    if (tid + T * k < n_cols) y[tid + T * k] = v[k] / sum;
  for (int32_t i = tid + T * kSoftmaxRegs; i < n_cols; i += T) y[i] = y[i] / sum;
}

}  // namespace dc

static int softmax_launch(const float* src, int64_t src_stride, float* dst, int64_t dst_stride, int32_t n_rows,
                          int32_t n_cols, dc_stream_t stream, const char* who) {
  if (n_rows < 0 || n_cols < 0 || (n_rows > 0 && (src_stride < n_cols || dst_stride < n_cols)))
    return dc::fail(DC_EINVAL, "%s: bad shape", who);
  if (n_rows == 0 || n_cols == 0) return DC_OK;
  if (!src || !dst) return dc::fail(DC_EINVAL, "%s: null pointer", who);
#define DC_SOFTMAX(T_, SKIP_)                                                                                        \
  hipLaunchKernelGGL((dc::softmax_rows_kernel<T_, SKIP_>), dim3(uint32_t(n_rows)), dim3(T_), 0, hipStream_t(stream), \
                     src, src_stride, dst, dst_stride, n_cols)
  // The smallest block that loses nothing on few rows: 1024 threads on short
  // rows leave most of their lanes idle (8192 rows of 200 columns: 34.3 us,
  // 6.1 in blocks of 64; 4096 of 1000: 21.1, 9.6 in 256; 512 of 2048: 5.2,
  // 4.3 in 512), and fewer threads wait on more columns each (24 rows of 500:
  // 3.5 us in 64, 3.0 in 256; of 2048: 3.7 in 256, 3.3 in 512; of 4096: 4.1
  // in 512, 3.9 in 1024).
  if (n_cols <= 256)
    DC_SOFTMAX(64, true);
  else if (n_cols <= 1024)
    DC_SOFTMAX(256, true);
  else if (n_cols <= 2048)
    DC_SOFTMAX(512, true);
  else if (n_cols <= 1024 * (dc::kSoftmaxRegs - 1))
    DC_SOFTMAX(1024, true);
  else
    DC_SOFTMAX(1024, false);
#undef DC_SOFTMAX
  return dc::check_hip(hipGetLastError(), who);
}

extern "C" int dc_softmax_rows(float* x, int32_t n_rows, int32_t n_cols, int64_t stride, dc_stream_t stream) {
  return softmax_launch(x, stride, x, stride, n_rows, n_cols, stream, "dc_softmax_rows");
}

extern "C" int dc_softmax_rows_to(const float* x, int64_t x_stride, float* y, int64_t y_stride, int32_t n_rows,
                                  int32_t n_cols, dc_stream_t stream) {
  return softmax_launch(x, x_stride, y, y_stride, n_rows, n_cols, stream, "dc_softmax_rows_to");
}
