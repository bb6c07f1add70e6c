// TopK backward: latent-major segment reduction producing dW (written once, no atomics) and
// dvals, from the pair list and the forward residual.
#pragma once

#include "common.hpp"
#include "segment_kernels.hpp"

#ifndef FLEXSAE_TOPK_NT
#define FLEXSAE_TOPK_NT true
#endif

namespace flexsae {

// For the slots [s_begin, s_end) of latent f (W row tile in w[]), over the lane's VEC columns:
//   acc      += vals[p] * scale * resid[b_p]          (dW contribution)
//   dv_tile[slot] = scale * <resid[b_p], W[f]>        (this tile's share of dvals[p]; the lane that
//                                                      owns the slot stores it, so stores coalesce;
//                                                      topk_epilogue_kernel adds the tiles up)
// resid rows (element type RT) are read through the caches: the waves in flight share one
// B x tile slice of the [B,D] matrix, which has to stay in the 4 MB L2 of every XCD.
template <typename RT, int VEC>
__device__ __forceinline__ void topk_accumulate_slots(
    const vec_t<uint32_t, 2> *__restrict__ slot_bv,
    const void *__restrict__ resid, float scale, float *__restrict__ dv_tile, const float (&w)[VEC],
    uint32_t s_begin, uint32_t s_end, int D, int dsafe, float (&acc)[VEC]) {
  using S = typename Traits<RT>::store_t;
  const int lane = lane_id();
  // row address = scalar base of the row + the lane's fixed byte offset
  const uint32_t lane_off = static_cast<uint32_t>(dsafe) * sizeof(S);
  const size_t row_bytes = static_cast<size_t>(D) * sizeof(S);
  for (uint32_t s = s_begin; s < s_end; s += kWave) {
    const uint32_t slot = s + lane;
    int my_b = 0;
    float v = 0.f;
    if (slot < s_end) {  // the pair's (batch row, val) record; the val of an out-of-range index is zero there
      const vec_t<uint32_t, 2> bv = slot_bv[slot];
      my_b = static_cast<int>(bv[0]);
      v = __uint_as_float(bv[1]) * scale;
    }
    const int n = (s_end - s) < static_cast<uint32_t>(kWave) ? static_cast<int>(s_end - s) : kWave;
    float my_dot = 0.f;
    // eight gathers in flight; a group reaching past the end re-reads the last row (a cache hit);
    // the eight dot products of a group share one transposed wave reduction
    for (int j = 0; j < n; j += 8) {
      raw_vec_t<RT, VEC> buf[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int jj = (j + u) < n ? (j + u) : (n - 1);
        const char *row = static_cast<const char *>(resid) +
                          static_cast<size_t>(static_cast<uint32_t>(bcast_i32(my_b, jj))) * row_bytes;
        buf[u] = *reinterpret_cast<const raw_vec_t<RT, VEC> *>(row + lane_off);
      }
      float dots[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        dots[u] = 0.f;
        if (j + u < n) {  // uniform
          float x[VEC];
          unpack_raw<RT, VEC>(buf[u], x);
          const float vj = bcast_f32(v, j + u);
          float dot = 0.f;
#pragma unroll
          for (int i = 0; i < VEC; ++i) {
            acc[i] = fmaf(vj, x[i], acc[i]);
            dot = fmaf(x[i], w[i], dot);
          }
          dots[u] = dot;
        }
      }
      const float tot = wave_sum8_transposed(dots);  // lane L: total of slot s + j + (L & 7)
      if ((lane >> 3) == (j >> 3)) my_dot = tot;
    }
    if (slot < s_end) dv_tile[slot] = my_dot * scale;
  }
}

// A wavefront's W pieces, one per latent of its group, and in their places the finished pieces of dW.
template <typename WT, typename GT, int VEC>
union LatentPiece {
  raw_vec_t<WT, VEC> w;
  raw_vec_t<GT, VEC> g;
};
// Latents per wavefront: eight; four where a piece takes more than 16 bytes of LDS per lane (32 KB per block either way).
template <typename WT, typename GT, int VEC>
constexpr int topk_group() {
  return sizeof(LatentPiece<WT, GT, VEC>) > 16 ? 4 : 8;
}

// Stores of dW take the streaming hint but for rows stored two bytes per lane, whose runs of 128 bytes begin and end inside lines,
// and, where nearly all rows are zeros (`plain`), for rows stored four bytes per lane.  us with / without it, uniform and skewed
// indices: D=1001 bf16 B=128, K=32, F=131072 159 / 113, 160 / 113, B=1024 169 / 155, 182 / 145; D=1938 B=128 239 / 207, 239 / 187,
// D=778 fp16 156 / 130, 156 / 121; not B=1024 D=1938 252 / 273, 257 / 271, B=4096, F=65536 266 / 268, 268 / 306, and
// not with eight bytes and more (B=1024, F=131072, D=1764 bf16 189 / 271, D=2304 215 / 274).
template <bool STREAM, typename V>
__device__ __forceinline__ void store_dw(V *to, V x, bool plain) {
  if constexpr (STREAM && sizeof(V) == 4) {
    if (plain) {  // uniform
      asm volatile("");  // (two stores that differ in the hint alone would become one without it)
      *to = x;
      asm volatile("");
      return;
    }
  }
  if constexpr (STREAM && sizeof(V) >= 4) __builtin_nontemporal_store(x, to);
  else *to = x;
}

// The short latents (at most kSegChunk pairs) of a group of L neighbours, one tile: their pairs are one run of slots but for
// the long latents among them, so a wavefront walks them as one stream.  The chain of trips to memory at the head of a
// latent (its bounds, its records and W row, the first residual rows) is paid once per group, and the batches of eight rows
// are full whatever the latents' counts.  The W pieces wait in the LDS, each finished piece of dW takes the place of its W
// piece, and all of them are stored at the end: the memory counter retires in order, so a store among the gathers would be
// waited for by the batch behind it.  Residual rows are gathered through a buffer descriptor (no vector ALU work for
// addresses), each batch requested while other wavefronts work on theirs, and its dot products share one transposed wave
// reduction.  With bf16 weights and a bf16 residual copy the products run on packed pairs (dot2) without unpacking.
// What bounds it: the L2s' row gathers (14 of 18 TB/s at B=4096, K=128, F=65536, D=2304 bf16, W and dW beside them), for fp32
// the W and dW streams.  Against one latent per wavefront (us; the kernel there 265 -> 245) the whole backward: K=128 340 ->
// 320, K=64 247 -> 224, K=32 214 -> 180; F=262144, K=64 650 -> 463; B=2048, K=64, F=131072, D=1024 fp32 241 -> 192; two or four
// latents, or two batches in flight (fewer wavefronts per SIMD): 2-20 % slower.
//
// EV < VEC: rows of W and dW that only vectors of EV elements divide (the residual copy's rows are padded to VEC with zeros).
// They pass through the LDS in such vectors, neighbouring lanes on neighbouring ones, so that every access is one run of
// lines as with narrow tiles, while the gathers keep their 16 bytes per lane.
template <typename WT, typename GT, typename RT, int VEC, int EV, int L>
__device__ __forceinline__ void topk_short_latents(
    const uint32_t *__restrict__ begin, const vec_t<uint32_t, 2> *__restrict__ slot_bv, const void *__restrict__ weight,
    int vals_dtype, const GatherSource &rows_src, uint32_t row_stride, float scale, void *__restrict__ dW,
    float *__restrict__ dv_tile, int64_t f0, int per_wave, int64_t F, int d0, int D,
    LatentPiece<WT, GT, VEC> *__restrict__ pieces, bool plain) {
  using S = typename Traits<RT>::store_t;
  using S_w = typename Traits<WT>::store_t;
  static_assert(L <= 8, "the counts of a wavefront's latents are scanned inside eight lanes");
  const int lane = lane_id();
  const bool active = d0 < D;
  const int dsafe = active ? d0 : 0;
  const uint32_t lane_off = static_cast<uint32_t>(dsafe) * sizeof(S);
  constexpr bool kDot2 = Traits<WT>::dtype == FLEXSAE_BF16 && Traits<RT>::dtype == FLEXSAE_BF16 && VEC % 2 == 0;
  // bf16 vals enter the dot2 as they are, beside a zero for the pair's other column.  Not in rows of odd length: a residual
  // that is infinite or NaN stays in its own column of dW there, as with the narrow tiles (and the products in fp32 are the
  // faster ones: the backward at B=4096, K=128, F=65536, D=2305 394 -> 377 us; at D=2304 302 -> 311).
  const bool late_scale = kDot2 && EV != 1 && vals_dtype == FLEXSAE_BF16;

  // lane l: first slot of latent f0 + l (of the one after the last for l >= per_wave, and wherever F cuts the group short)
  const int64_t fl = f0 + (lane < per_wave ? lane : per_wave);
  const uint32_t first = begin[fl < F ? fl : F];
  const uint32_t past = static_cast<uint32_t>(__shfl_down(static_cast<int>(first), 1));  // (of all lanes: lane L is read)
  const uint32_t n_all = lane < per_wave ? past - first : 0u;
  const bool is_long = n_all > static_cast<uint32_t>(kSegChunk);  // chunk role
  const uint32_t n_mine = is_long ? 0u : n_all;
  uint32_t upto = n_mine;  // pairs of latents f0 .. f0 + lane
#pragma unroll
  for (int d = 1; d < L; d *= 2) {
    const uint32_t o = static_cast<uint32_t>(__shfl_up(static_cast<int>(upto), d));
    if (lane >= d) upto += o;
  }
  const int M = bcast_i32(static_cast<int>(upto), L - 1);
  const uint32_t s0 = static_cast<uint32_t>(bcast_i32(static_cast<int>(first), 0));
  const uint64_t any_long = __ballot(is_long);

  int at = -1, end = 0;  // the latent being summed and the place in the stream where its pairs end
  vec_t<uint32_t, 2> bv{0u, 0u};
  auto slot_of = [&](int p) {
    uint32_t slot = s0 + static_cast<uint32_t>(p);
    if (any_long) {
#pragma unroll
      for (int l = 0; l < L; ++l)
        if (any_long >> l & 1)
          slot += p >= bcast_i32(static_cast<int>(upto), l) ? static_cast<uint32_t>(bcast_i32(static_cast<int>(n_all), l)) : 0u;
    }
    return slot;
  };
  uint32_t slot = slot_of(lane);
  // W rows: for a latent without pairs here a descriptor of no bytes, which reads zeros and no memory (so do lanes beyond D)
  constexpr int kParts = VEC / EV;
  auto w_row = [&](int l) {
    const uint32_t bytes = bcast_i32(static_cast<int>(n_mine), l) != 0 ? static_cast<uint32_t>(D) * sizeof(S_w) : 0u;
    return make_gather_source(static_cast<const S_w *>(weight) + (f0 + l) * D, bytes);
  };
  if constexpr (kParts == 1) {
    raw_vec_t<WT, VEC> wraw[L];
#pragma unroll
    for (int l = 0; l < L; ++l)
      wraw[l] = gather_raw<WT, VEC, FLEXSAE_TOPK_NT>(w_row(l), static_cast<uint32_t>(d0) * sizeof(S_w), 0u);
    if (lane < M) bv = __builtin_nontemporal_load(slot_bv + slot);
#pragma unroll
    for (int l = 0; l < L; ++l) pieces[l * kWave + lane].w = wraw[l];
  } else {
    const int tile0 = d0 - lane * VEC;
    if (lane < M) bv = __builtin_nontemporal_load(slot_bv + slot);
    constexpr int kAtOnce = kParts == 8 && L == 8 ? L / 2 : L;  // 32 registers
#pragma unroll
    for (int l0 = 0; l0 < L; l0 += kAtOnce) {
      raw_vec_t<WT, EV> part[kAtOnce][kParts];
#pragma unroll
      for (int l = 0; l < kAtOnce; ++l) {
        const GatherSource row = w_row(l0 + l);
#pragma unroll
        for (int k = 0; k < kParts; ++k)
          part[l][k] = gather_raw<WT, EV>(row, static_cast<uint32_t>(tile0 + (k * kWave + lane) * EV) * sizeof(S_w), 0u);
      }
#pragma unroll
      for (int l = 0; l < kAtOnce; ++l)
#pragma unroll
        for (int k = 0; k < kParts; ++k) {
          const int c = (k * kWave + lane) * EV;
          auto *const w_at = reinterpret_cast<S_w *>(&pieces[(l0 + l) * kWave + c / VEC].w) + c % VEC;
          *reinterpret_cast<raw_vec_t<WT, EV> *>(w_at) = part[l][k];
        }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();

  float w[kDot2 ? 1 : VEC], acc[VEC];
  uint32_t ww[(VEC + 1) / 2];  // the W piece as packed pairs (dot2 path)
  auto next_latent = [&]() {
    do {
      ++at;
      end = bcast_i32(static_cast<int>(upto), at);
    } while (bcast_i32(static_cast<int>(n_mine), at) == 0 && at < L - 1);
    const raw_vec_t<WT, VEC> x = pieces[at * kWave + lane].w;
    if constexpr (kDot2) __builtin_memcpy(ww, &x, sizeof(x));
    else unpack_raw<WT, VEC>(x, w);
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
  };
  auto flush = [&]() {
    if (late_scale) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] *= scale;
    }
    raw_vec_t<GT, VEC> x;
    store_vec<GT, VEC>(&x, 0, acc);
    pieces[at * kWave + lane].g = x;
  };
  if (M > 0) next_latent();
  // late: vals are bf16 and enter the dot2 as they are (kDot2 only)
  auto walk = [&](auto late) {
    constexpr bool kLate = decltype(late)::value;
#pragma unroll 1
    for (int p0 = 0; p0 < M; p0 += kWave) {
      const int n = M - p0 < kWave ? M - p0 : kWave;  // uniform
      if (p0 > 0) {
        slot = slot_of(p0 + lane);
        bv = vec_t<uint32_t, 2>{0u, 0u};
        if (lane < n) bv = __builtin_nontemporal_load(slot_bv + slot);
      }
      const uint32_t my_off = bv[0] * row_stride;
      const uint32_t vbits = kLate ? bv[1] : __float_as_uint(__uint_as_float(bv[1]) * scale);
      float my_dot = 0.f;
      raw_vec_t<RT, VEC> rows[8];
      auto issue = [&](int j) {  // past the end: the last row once more, not consumed
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int jj = (j + u) < n ? (j + u) : (n - 1);
          rows[u] = gather_raw<RT, VEC>(rows_src, lane_off, static_cast<uint32_t>(bcast_i32(static_cast<int>(my_off), jj)));
        }
      };
      auto consume = [&](auto full, int j) {
        constexpr bool kFull = decltype(full)::value;
        float dots[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          dots[u] = 0.f;
          if (!kFull && j + u >= n) continue;  // uniform
          if (p0 + j + u == end) {
            flush();
            next_latent();
          }
          const uint32_t vj = static_cast<uint32_t>(bcast_i32(static_cast<int>(vbits), j + u));
          float dot = 0.f;
          if constexpr (kDot2) {
            uint32_t xw[VEC / 2];
            __builtin_memcpy(xw, &rows[u], sizeof(xw));
#pragma unroll
            for (int i = 0; i < VEC / 2; ++i) dot = dot2_bf16(xw[i], ww[i], dot);
            if constexpr (kLate) {
              // a bf16 val widened to fp32 keeps its 16 bits in the upper half
              const uint32_t v_lo = vj >> 16;
#pragma unroll
              for (int i = 0; i < VEC / 2; ++i) {
                acc[2 * i] = dot2_bf16(xw[i], v_lo, acc[2 * i]);
                acc[2 * i + 1] = dot2_bf16(xw[i], vj, acc[2 * i + 1]);
              }
            } else {
              float x[VEC];
              unpack_raw<RT, VEC>(rows[u], x);
#pragma unroll
              for (int i = 0; i < VEC; ++i) acc[i] = fmaf(__uint_as_float(vj), x[i], acc[i]);
            }
          } else {
            float x[VEC];
            unpack_raw<RT, VEC>(rows[u], x);
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
              acc[i] = fmaf(__uint_as_float(vj), x[i], acc[i]);
              dot = fmaf(x[i], w[i], dot);
            }
          }
          dots[u] = dot;
        }
        const float tot = wave_sum8_transposed(dots);  // lane L: total of place j + (L & 7)
        if ((lane >> 3) == (j >> 3)) my_dot = tot;
      };
      issue(0);
#pragma unroll 1
      for (int j = 0; j < n; j += 8) {
        if (j + 8 <= n) consume(std::true_type{}, j);
        else consume(std::false_type{}, j);
        if (j + 8 < n) issue(j + 8);
      }
      if (lane < n) dv_tile[slot] = my_dot * scale;
    }
  };
  if constexpr (kDot2 && EV != 1) {
    if (late_scale) walk(std::true_type{});
    else walk(std::false_type{});
  } else {
    walk(std::false_type{});
  }
  if (M > 0) flush();
  if constexpr (kParts > 1) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int l = 0; l < L; ++l) {
    const uint32_t n = static_cast<uint32_t>(bcast_i32(static_cast<int>(n_all), l));
    if (l < per_wave && f0 + l < F && n <= static_cast<uint32_t>(kSegChunk)) {  // uniform
      using G = typename Traits<GT>::store_t;
#pragma unroll
      for (int k = 0; k < kParts; ++k) {
        const int c = kParts == 1 ? lane * VEC : (k * kWave + lane) * EV;  // column in the tile
        const int d = d0 - lane * VEC + c;
        raw_vec_t<GT, EV> x =
            *reinterpret_cast<const raw_vec_t<GT, EV> *>(reinterpret_cast<const G *>(&pieces[l * kWave + c / VEC].g) + c % VEC);
        if (n == 0) x = raw_vec_t<GT, EV>{};
        if (d < D) {
          auto *const to = reinterpret_cast<raw_vec_t<GT, EV> *>(static_cast<G *>(dW) + (f0 + l) * D + d);
          store_dw<FLEXSAE_TOPK_NT>(to, x, plain);
        }
      }
    }
  }
}

// One short latent (1 to kSegChunk pairs) for one tile, the fewer registers where latents have many pairs (which sizes take
// it: one_latent_per_wave): the pair records of the latent are one
// contiguous load, the residual rows are gathered through a buffer descriptor (no vector ALU work
// for addresses) eight at a time (with the next eight already requested when registers allow),
// and each group of eight shares one transposed wave reduction for the dvals dot products.  Inside a
// group, rows are requested and consumed two at a time under one uniform test, so a latent with
// nine pairs costs ten rows, not sixteen (a test per row costs more than it saves; the odd slot
// past the end re-reads the last row, a cache hit, with a val of zero).  With bf16 weights and a
// bf16 residual copy the products run on packed pairs (dot2) without unpacking.
template <typename WT, typename GT, typename RT, int VEC>
__device__ __forceinline__ void topk_short_latent(
    const vec_t<uint32_t, 2> *__restrict__ slot_bv, const void *__restrict__ weight, int vals_dtype,
    const GatherSource &rows_src, uint32_t row_stride, float scale, void *__restrict__ dW,
    float *__restrict__ dv_tile, int64_t f, uint32_t b0, int n, int d0, int D) {
  using S = typename Traits<RT>::store_t;
  const int lane = lane_id();
  const bool active = d0 < D;
  const uint32_t lane_off = static_cast<uint32_t>(active ? d0 : 0) * sizeof(S);
  constexpr bool kDot2 = Traits<WT>::dtype == FLEXSAE_BF16 && Traits<RT>::dtype == FLEXSAE_BF16 && VEC % 2 == 0;
  const bool late_scale = kDot2 && vals_dtype == FLEXSAE_BF16;  // vals enter the dot2 as they are

  const raw_vec_t<WT, VEC> wraw = load_raw<WT, VEC, FLEXSAE_TOPK_NT>(weight, f * D + (active ? d0 : 0));
  // lanes past the end hold row 0 and a val of zero
  const vec_t<uint32_t, 2> bv = lane < n ? __builtin_nontemporal_load(slot_bv + b0 + lane) : vec_t<uint32_t, 2>{0u, 0u};
  const int my_b = static_cast<int>(bv[0]);
  const uint32_t vbits = bv[1];

  // two groups of eight rows in flight, or one when a group alone takes 32 registers: the
  // kernel gains more from another wavefront per SIMD than from the deeper prefetch
  constexpr int kRowsPerTest = 2;  // rows of a group of eight that share one uniform "are there rows left" test
  constexpr bool kTwoGroups = sizeof(raw_vec_t<RT, VEC>) * 8 <= 64;
  raw_vec_t<RT, VEC> buf_a[8], buf_b[kTwoGroups ? 8 : 1];
  auto issue = [&](raw_vec_t<RT, VEC>(&buf)[8], int j) {
#pragma unroll
    for (int h = 0; h < 8; h += kRowsPerTest) {
      if (h == 0 || j + h < n) {  // uniform: the second half of a group only when it has rows
#pragma unroll
        for (int u = h; u < h + kRowsPerTest; ++u) {
          const int jj = (j + u) < n ? (j + u) : (n - 1);
          buf[u] = gather_raw<RT, VEC>(rows_src, lane_off, static_cast<uint32_t>(bcast_i32(my_b, jj)) * row_stride);
        }
      }
    }
  };
  issue(buf_a, 0);
  if constexpr (kTwoGroups) {
    if (n > 8) issue(buf_b, 8);
  }

  float w[VEC], acc[VEC];
  unpack_raw<WT, VEC>(wraw, w);
#pragma unroll
  for (int i = 0; i < VEC; ++i) {
    acc[i] = 0.f;
    if (!active) w[i] = 0.f;
  }
  uint32_t ww[(VEC + 1) / 2] = {};  // the W piece as packed pairs (dot2 path)
  if constexpr (kDot2) {
    __builtin_memcpy(ww, &wraw, sizeof(raw_vec_t<WT, VEC>));
#pragma unroll
    for (int i = 0; i < VEC / 2; ++i)
      if (!active) ww[i] = 0u;
  }
  const float v = __uint_as_float(vbits) * (late_scale ? 1.f : scale);
  float my_dot = 0.f;
  auto consume = [&](const raw_vec_t<RT, VEC>(&rows)[8], int j) {  // slots j .. j+7 of the latent
    float dots[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) dots[u] = 0.f;
#pragma unroll
    for (int h = 0; h < 8; h += kRowsPerTest) {
      if (h != 0 && j + h >= n) continue;  // uniform
#pragma unroll
      for (int u = h; u < h + kRowsPerTest; ++u) {
        float dot = 0.f;
        if constexpr (kDot2) {
          uint32_t xw[VEC / 2];
          __builtin_memcpy(xw, &rows[u], sizeof(xw));
#pragma unroll
          for (int i = 0; i < VEC / 2; ++i) dot = dot2_bf16(xw[i], ww[i], dot);
          if (late_scale) {  // uniform
            // a bf16 val widened to fp32 keeps its 16 bits in the upper half
            const uint32_t v_hi = static_cast<uint32_t>(bcast_i32(static_cast<int>(vbits), j + u));
            const uint32_t v_lo = v_hi >> 16;
#pragma unroll
            for (int i = 0; i < VEC / 2; ++i) {
              acc[2 * i] = dot2_bf16(xw[i], v_lo, acc[2 * i]);
              acc[2 * i + 1] = dot2_bf16(xw[i], v_hi, acc[2 * i + 1]);
            }
          } else {
            float x[VEC];
            unpack_raw<RT, VEC>(rows[u], x);
            const float vj = bcast_f32(v, j + u);
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc[i] = fmaf(vj, x[i], acc[i]);
          }
        } else {
          float x[VEC];
          unpack_raw<RT, VEC>(rows[u], x);
          const float vj = bcast_f32(v, j + u);
#pragma unroll
          for (int i = 0; i < VEC; ++i) {
            acc[i] = fmaf(vj, x[i], acc[i]);
            dot = fmaf(x[i], w[i], dot);
          }
        }
        dots[u] = dot;
      }
    }
    const float tot = wave_sum8_transposed(dots);  // lane L: total of slot j + (L & 7)
    if ((lane >> 3) == (j >> 3)) my_dot = tot;
  };
  if constexpr (kTwoGroups) {
    for (int j = 0; j < n; j += 16) {
      consume(buf_a, j);
      if (j + 16 < n) issue(buf_a, j + 16);
      if (j + 8 < n) {
        consume(buf_b, j + 8);
        if (j + 24 < n) issue(buf_b, j + 24);
      }
    }
  } else {
    for (int j = 0; j < n; j += 8) {
      consume(buf_a, j);
      if (j + 8 < n) issue(buf_a, j + 8);
    }
  }
  if (late_scale) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] *= scale;
  }
  if (active) store_vec<GT, VEC, FLEXSAE_TOPK_NT && sizeof(raw_vec_t<GT, VEC>) >= 4>(dW, f * D + d0, acc);
  if (lane < n) dv_tile[b0 + lane] = my_dot * scale;
}

// TopK backward of one slice.  scale = grad_out * 2/(B*D).
// Blocks [0, n_long_blocks), a multiple of eight: long latents, one wavefront per (64-pair chunk, tile): stores its
// dvals shares, leaves its dW contribution in partial[chunk, slice column] (fp32) for
// seg_reduce_long_finalize_kernel (next launch).  They come first so hot latents start at once.
// Remaining blocks: one wavefront per (tile of the slice, group of per_wave latents), see topk_short_latents, or with ONE per
// (tile, latent), see topk_short_latent; tile = 64*VEC columns,
// lane l owning VEC consecutive columns.  The n_groups blocks of each of the first n_full tiles, tiles
// outermost, are cut into eight runs of xcd_span, one per XCD (blocks go round the XCDs): an L2 holds the B x tile slice of
// resid that its own wavefronts gather from, instead of every L2 fetching every slice (B=2048, K=256, F=131072, D=1024 fp32
// 327 -> 301 us for the whole backward, K=64 249 -> 192; bf16 the same either way).  A last tile with few columns follows in
// eight runs of its own: among the others' it leaves the XCDs that hold it idle for much of the time.
// dW[f, tile] is written exactly once, in the gradient's final dtype; latents without pairs
// get zeros.
// resid_ld: elements from one row of resid to the next.  EV: elements of a vector that divides the rows of W and dW.
template <typename WT, typename GT, typename RT, int VEC, int EV, bool ONE>
__global__ __launch_bounds__(256) void topk_bwd_kernel(
    const uint32_t *__restrict__ begin, const uint32_t *__restrict__ map,
    const uint32_t *__restrict__ long_ctrl, const uint32_t *__restrict__ long_list,
    const uint32_t *__restrict__ chunk_begin, const vec_t<uint32_t, 2> *__restrict__ slot_bv,
    const void *__restrict__ weight, const void *__restrict__ vals, int vals_dtype,
    const void *__restrict__ resid, const float *__restrict__ grad_out, float coef,
    void *__restrict__ dW, float *__restrict__ dv_part, int64_t n_pairs, float *__restrict__ partial,
    unsigned n_long_blocks, uint32_t n_groups, uint32_t xcd_span, uint32_t n_full, int per_wave, int tps, int col0, int slice_w,
    int64_t F, int K, int D, int resid_ld, uint32_t resid_bytes) {
  const int lane = lane_id();
  const float scale = coef * grad_out[0];
  if (blockIdx.x >= n_long_blocks) {
    // (in 32 bits: a launch holds fewer than 2^24 blocks)
    const uint32_t i = (blockIdx.x - n_long_blocks) >> 3;
    const bool in_full = i < xcd_span;
    const uint32_t item = in_full ? (blockIdx.x & 7) * xcd_span + i
                                  : n_groups * n_full + (blockIdx.x & 7) * ((n_groups + 7) >> 3) + i - xcd_span;
    const uint32_t t = item / n_groups;
    if (t >= (in_full ? n_full : static_cast<uint32_t>(tps))) return;
    const int64_t f0 = static_cast<int64_t>((item - t * n_groups) * (blockDim.x >> 6) + wave_in_block()) * per_wave;
    if (f0 >= F) return;  // uniform per wavefront
    const GatherSource rows_src = make_gather_source(resid, resid_bytes);
    if constexpr (ONE) {
      const uint32_t b0 = begin[f0];
      const uint32_t n = begin[f0 + 1] - b0;
      if (n > static_cast<uint32_t>(kSegChunk)) return;  // chunk role
      const int d0 = col0 + static_cast<int>(t) * (kWave * VEC) + lane * VEC;
      if (n == 0) {  // unused latent: zeros
        const float zero[VEC] = {};
        if (d0 < D) store_vec<GT, VEC, FLEXSAE_TOPK_NT && sizeof(raw_vec_t<GT, VEC>) >= 4>(dW, f0 * D + d0, zero);
        return;
      }
      topk_short_latent<WT, GT, RT, VEC>(
          slot_bv, weight, vals_dtype, rows_src, static_cast<uint32_t>(resid_ld) * sizeof(typename Traits<RT>::store_t), scale,
          dW, dv_part + (col0 / (kWave * VEC) + t) * n_pairs, f0, b0, static_cast<int>(n), d0, D);
    } else {
      constexpr int L = topk_group<WT, GT, VEC>();
      __shared__ LatentPiece<WT, GT, VEC> pieces[256 / kWave][L * kWave];
      topk_short_latents<WT, GT, RT, VEC, EV, L>(
          begin, slot_bv, weight, vals_dtype, rows_src, static_cast<uint32_t>(resid_ld) * sizeof(typename Traits<RT>::store_t), scale,
          dW, dv_part + (col0 / (kWave * VEC) + t) * n_pairs, f0, per_wave, F,
          col0 + static_cast<int>(t) * (kWave * VEC) + lane * VEC, D, pieces[wave_in_block()],
          16 * n_pairs < F);
    }
    return;
  }
  const uint32_t n_long = long_ctrl[kLongCount];
  if (n_long == 0) return;
  const uint32_t n_chunks = long_ctrl[kLongChunks];
  const int64_t total = static_cast<int64_t>(n_chunks) * tps;
  const int64_t n_waves = static_cast<int64_t>(n_long_blocks) * (blockDim.x >> 6);
  for (int64_t wk = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + wave_in_block();
       wk < total; wk += n_waves) {
    // tile-major over the work list as well
    const int t = static_cast<int>(wk / n_chunks);
    const uint32_t chunk = static_cast<uint32_t>(wk - static_cast<int64_t>(t) * n_chunks);
    const LongChunk c = seg_decode_chunk(begin, long_list, chunk_begin, n_long, chunk);
    const int pc = t * (kWave * VEC) + lane * VEC;
    const int d0 = col0 + pc;
    const bool active = d0 < D;
    const int dsafe = active ? d0 : 0;
    float w[VEC], acc[VEC];
#pragma unroll
    for (int i = 0; i < VEC; i += EV) {
      float part[EV];
      const int d = d0 + i < D ? d0 + i : 0;
      load_vec<WT, EV>(weight, c.f * D + d, part);
#pragma unroll
      for (int k = 0; k < EV; ++k) {
        acc[i + k] = 0.f;
        w[i + k] = d0 + i < D ? part[k] : 0.f;
      }
    }
    topk_accumulate_slots<RT, VEC>(slot_bv, resid, scale, dv_part + (col0 / (kWave * VEC) + t) * n_pairs, w, c.s0,
                                   c.s1, resid_ld, dsafe, acc);
    store_vec<float, VEC>(partial, static_cast<int64_t>(chunk) * slice_w + pc, acc);
  }
}

// x (fp32) rounded to run-time type `dtype`
__device__ __forceinline__ void store_scalar(void *base, int dtype, int64_t i, float x) {
  const float v[1] = {x};
  if (dtype == FLEXSAE_F32) store_vec<float, 1>(base, i, v);
  else if (dtype == FLEXSAE_BF16) store_vec<bf16_t, 1>(base, i, v);
  else store_vec<f16_t, 1>(base, i, v);
}

// Gradients of vals and bias in the leaves' types.
struct LeafGrads {
  void *dvals, *dbias;
  int dvals_dtype, dbias_dtype;
};

// What follows the (last) slice of a TopK backward, in one launch of 256-thread blocks; the parts are independent:
//   the first n_long_blocks  second step of the slice's long latents (seg_long_finalize_body);
//   the next n_col_blocks    dbias = coef * grad_out * column sums of resid: stage 2 (colsum_final_one);
//   the rest                 dvals[map[slot]] = sum over the column tiles of dv_part[tile, slot], in tile order (every
//                            pair sits in exactly one slot, so dvals is written once and needs no zero-fill).
// A launch costs 4-5 us in a busy stream: with the preparation (below) four launches instead of eight around the pair
// list and the backward: B=4096, K=128, F=65536, D=2304 bf16 618 -> 610 us, B=64, K=32, F=4096, D=256 250 -> 239.
template <typename GT, int VEC>
__global__ __launch_bounds__(256) void topk_epilogue_kernel(
    const uint32_t *__restrict__ long_ctrl, const uint32_t *__restrict__ long_list,
    const uint32_t *__restrict__ chunk_begin, const float *__restrict__ partial, void *__restrict__ dW, int tps, int col0,
    int slice_w, int D, unsigned n_long_blocks, const float *__restrict__ colsum_part, int n_chunks,
    const float *__restrict__ grad_out, float coef, unsigned n_col_blocks,
    const uint32_t *__restrict__ map, const float *__restrict__ dv_part, int n_tiles, int64_t n_pairs, LeafGrads leaf) {
  if (blockIdx.x < n_long_blocks) {
    seg_long_finalize_body<GT, VEC, 8>(long_ctrl, long_list, chunk_begin, partial, dW, nullptr, tps, col0, slice_w, D,
                                       blockIdx.x, n_long_blocks);
    return;
  }
  unsigned blk = blockIdx.x - n_long_blocks;
  if (blk < n_col_blocks) {
    const int c = static_cast<int>(blk * blockDim.x + threadIdx.x);
    if (c < D) store_scalar(leaf.dbias, leaf.dbias_dtype, c, colsum_final_value(colsum_part, n_chunks, D, grad_out, coef, c));
    return;
  }
  blk -= n_col_blocks;
  const int64_t stride = static_cast<int64_t>(gridDim.x - n_long_blocks - n_col_blocks) * blockDim.x;
  for (int64_t s = static_cast<int64_t>(blk) * blockDim.x + threadIdx.x; s < n_pairs; s += stride) {
    float acc = 0.f;
    for (int t = 0; t < n_tiles; ++t) acc += dv_part[t * n_pairs + s];
    store_scalar(leaf.dvals, leaf.dvals_dtype, map[s], acc);
  }
}

// For the kColsumRows rows of a chunk and 64 * V columns, by one block of four wavefronts: resid16[b, c] = bf16(resid[b, c])
// (resid16 null: no copy; ld16 >= cols elements a row, zeros past cols; V divides cols and ld16) and stage 1 of the column sums
// of resid, both from one read.  A wavefront has sixteen rows, all in flight at once; the sums are colsum_partial_one's: a
// wavefront adds its rows to the sums of the rows before.
template <int V>
__device__ __forceinline__ void resid_block(const float *__restrict__ resid, int64_t rows, int cols, int ld16,
                                            void *__restrict__ resid16, float *__restrict__ colsum_part, unsigned block,
                                            float *__restrict__ sums) {
  constexpr int kBlockWaves = kChunkThreads / kWave, U = kColsumRows / kBlockWaves;
  const int width = resid16 ? ld16 : cols;
  const unsigned across = static_cast<unsigned>((width + kWave * V - 1) / (kWave * V));
  const unsigned chunk = block / across;
  const int lane = lane_id(), wv = wave_in_block();
  const int c = static_cast<int>((block - chunk * across) * (kWave * V)) + lane * V;
  const int64_t r0 = static_cast<int64_t>(chunk) * kColsumRows + wv * U;
  const bool inside = c < cols;
  float x[U][V];
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int i = 0; i < V; ++i) x[u][i] = 0.f;
    if (inside && r0 + u < rows) load_vec<float, V>(resid, (r0 + u) * cols + c, x[u]);
  }
  for (int w = 0; w < kBlockWaves; ++w) {
    if (w == wv) {  // uniform
      float s[V];
#pragma unroll
      for (int i = 0; i < V; ++i) s[i] = w == 0 ? 0.f : sums[lane * V + i];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (r0 + u < rows) {  // uniform
#pragma unroll
          for (int i = 0; i < V; ++i) s[i] += x[u][i];
        }
#pragma unroll
      for (int i = 0; i < V; ++i) sums[lane * V + i] = s[i];
      if (w == kBlockWaves - 1 && inside) store_vec<float, V>(colsum_part, static_cast<int64_t>(chunk) * cols + c, s);
    }
    __syncthreads();
  }
  if (!resid16 || c >= ld16) return;
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (r0 + u < rows) store_vec<bf16_t, V>(resid16, (r0 + u) * ld16 + c, x[u]);
}

// Blocks of resid_block for a residual of `cols` columns
inline int64_t resid_blocks(int64_t rows, int cols, int width) {
  const int v = cols % 4 == 0 ? 4 : cols % 2 == 0 ? 2 : 1;
  return ((rows + kColsumRows - 1) / kColsumRows) * ((width + kWave * v - 1) / (kWave * v));
}

// First launch of a TopK backward that makes its own pair list: the first n_chunks blocks order the list's chunks
// (csr_chunk_sort_kernel), the others are resid_block; the records come with the second launch (csr_bucket_sort_kernel).
// The chunks are a chain of trips to memory on a few wavefronts per compute unit and the residual streams beside them.  B=4096,
// K=128, F=65536, D=2304 bf16: the two launches take 15.7 + 18.8 us; chunks, buckets, topk_prepare_kernel and pair_lists_kernel
// 9.4 + 12.6 + 23.2 + 4.7 (fp32 B=2048, K=256, F=131072, D=1024 9.7 + 19.2 against 9.2 + 13.0 + 13.3 + 4.7; B=64, K=32, F=4096,
// D=256 5.3 + 9.5 against 5.2 + 7.6 + 4.0 + 2.9).
__global__ __launch_bounds__(kChunkThreads) void topk_front_kernel(
    const int64_t *__restrict__ indices, int64_t n_pairs, int64_t F, int shift, int pack_shift, uint32_t n_buckets, int n_bits,
    int64_t chunk, uint32_t n_chunks, uint32_t *__restrict__ table, uint32_t *__restrict__ tmp, uint32_t *__restrict__ ctrl,
    int *status_flag, const float *__restrict__ resid, int64_t rows, int cols, int ld16, void *__restrict__ resid16,
    float *__restrict__ colsum_part) {
  if (blockIdx.x < n_chunks) {
    chunk_sort_block(indices, n_pairs, F, shift, pack_shift, n_buckets, n_bits, chunk, n_chunks, table, tmp, ctrl, status_flag);
    return;
  }
  __shared__ float sums[kWave * 4];
  const unsigned block = blockIdx.x - n_chunks;
  if (cols % 4 == 0) resid_block<4>(resid, rows, cols, ld16, resid16, colsum_part, block, sums);
  else if (cols % 2 == 0) resid_block<2>(resid, rows, cols, ld16, resid16, colsum_part, block, sums);
  else resid_block<1>(resid, rows, cols, ld16, resid16, colsum_part, block, sums);
}

// Preparation of a TopK backward on a given pair list, one launch:
//   slot_bv[s] = (batch row, val as fp32 bits) of the pair in slot s of the latent-major list: what
//     the backward reads per pair, contiguous per latent instead of scattered over vals; a pair
//     whose index lies outside [0, F) gets a val of zero, as in the forward (the pair list files it
//     under latent 0), so that it adds nothing to dW (`indices` may be null: every val is kept);
//   resid16[b, d] = bf16(resid[b, d]), rows of ld16 >= cols elements with zeros past cols (ld16 a multiple of four, or
//     cols; n_resid = rows * ld16, 0: no copy wanted);
//   ctrl[] = 0: the control words of the lists that the next launch fills;
//   in the first n_col_blocks blocks, stage 1 of the column sums of resid (for dbias).
__global__ __launch_bounds__(256) void topk_prepare_kernel(const uint32_t *__restrict__ map, const int64_t *__restrict__ indices,
                                    int64_t F, const void *__restrict__ vals,
                                    int vals_dtype, int64_t n_pairs, int K,
                                    vec_t<uint32_t, 2> *__restrict__ slot_bv, const float *__restrict__ resid,
                                    int64_t n_resid, void *__restrict__ resid16, uint32_t *__restrict__ ctrl,
                                    int64_t rows, int cols, int ld16, float *__restrict__ colsum_part, unsigned n_col_blocks) {
  if (blockIdx.x < n_col_blocks) {
    const unsigned across = static_cast<unsigned>((cols + 255) / 256);
    colsum_partial_one(resid, rows, cols, cols, colsum_part, static_cast<int>(blockIdx.x % across * 256 + threadIdx.x),
                       static_cast<int64_t>(blockIdx.x / across));
    return;
  }
  if (blockIdx.x == n_col_blocks && threadIdx.x < kCtrlWords) ctrl[threadIdx.x] = 0u;
  const int64_t stride = static_cast<int64_t>(gridDim.x - n_col_blocks) * blockDim.x;
  const int64_t tid = static_cast<int64_t>(blockIdx.x - n_col_blocks) * blockDim.x + threadIdx.x;
  for (int64_t s = tid; s < n_pairs; s += stride) {
    const uint32_t p = map[s];
    vec_t<uint32_t, 2> r;
    r[0] = p / static_cast<uint32_t>(K);
    float v = load_scalar(vals, vals_dtype, p);
    if (indices && static_cast<uint64_t>(indices[p]) >= static_cast<uint64_t>(F)) v = 0.f;
    r[1] = __float_as_uint(v);
    slot_bv[s] = r;
  }
  const int64_t n4 = n_resid >> 2;
  if (ld16 != cols) {
    const uint32_t per_row = static_cast<uint32_t>(ld16) >> 2;
    for (int64_t i = tid; i < n4; i += stride) {
      const uint32_t row = static_cast<uint32_t>(i) / per_row;
      const int c = static_cast<int>((static_cast<uint32_t>(i) - row * per_row) * 4);
      const float *const from = resid + static_cast<int64_t>(row) * cols;
      float x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = c + k < cols ? from[c + k] : 0.f;
      store_vec<bf16_t, 4>(resid16, i * 4, x);
    }
    return;
  }
  for (int64_t i = tid; i < n4; i += stride) {
    float x[4];
    load_vec<float, 4>(resid, i * 4, x);
    store_vec<bf16_t, 4>(resid16, i * 4, x);
  }
  for (int64_t i = (n4 << 2) + tid; i < n_resid; i += stride) {
    float x[1] = {resid[i]};
    store_vec<bf16_t, 1>(resid16, i, x);
  }
}

}  // namespace flexsae
