// Latent-major segment reduction: out[f, slice] = sum of the rows [begin[f], begin[f+1]) of
// P[., slice] (rows of one latent are adjacent), with fp32 accumulation and one write per
// output element.  Short groups (<= 64 rows) are reduced by one wavefront; long ones are cut
// into chunks of 64 rows whose fp32 partial sums are combined in chunk order, so a hot latent is
// spread over many wavefronts and the summation order stays fixed (deterministic).
#pragma once

#include <type_traits>

#include "common.hpp"
#include "csr_kernels.hpp"

#ifndef FLEXSAE_REDUCE_NT
#define FLEXSAE_REDUCE_NT true
#endif

namespace flexsae {

constexpr int kSegChunk = 64;  // rows per chunk; groups longer than this count as "long"
static_assert(kSegChunk == static_cast<int>(kListLong), "the long latents of a pair list are the ones reduced in chunks");

// acc += sum of rows [r0, r0+n) of X (row stride `ld` elements) over the lane's VEC columns at pc.
// Rows are fetched up to U at a time; n is uniform over the wavefront, so the tests around the
// loads are scalar branches and a short group issues exactly its own loads, all in flight at once.
template <typename PT, int VEC, int U, bool NT = false>
__device__ __forceinline__ void accumulate_rows(const void *__restrict__ X, int64_t r0, int n,
                                                int64_t ld, int pc, float (&acc)[VEC]) {
  for (int j = 0; j < n; j += U) {
    raw_vec_t<PT, VEC> raw[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (j + u < n) raw[u] = load_raw<PT, VEC, NT>(X, (r0 + j + u) * ld + pc);  // uniform
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (j + u < n) {  // uniform
        float x[VEC];
        unpack_raw<PT, VEC>(raw[u], x);
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] += x[i];
      }
    }
  }
}

// The same sum in the order of the reduction by pieces (below), so that both reductions give the
// same bits for long latents: four running sums, row j goes to sum j % 4, combined as
// (s0 + s1) + (s2 + s3).
template <typename PT, int VEC, int U, bool NT = false>
__device__ __forceinline__ void accumulate_rows_by4(const void *__restrict__ X, int64_t r0, int n,
                                                    int64_t ld, int pc, float (&acc)[VEC]) {
  static_assert(U % 4 == 0, "rows are dealt to four sums");
  float part[4][VEC];
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int i = 0; i < VEC; ++i) part[g][i] = 0.f;
  for (int j = 0; j < n; j += U) {
    raw_vec_t<PT, VEC> raw[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (j + u < n) raw[u] = load_raw<PT, VEC, NT>(X, (r0 + j + u) * ld + pc);  // uniform
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (j + u < n) {  // uniform
        float x[VEC];
        unpack_raw<PT, VEC>(raw[u], x);
#pragma unroll
        for (int i = 0; i < VEC; ++i) part[u & 3][i] += x[i];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < VEC; ++i) acc[i] = (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]);
}

// The long latents a reduction serves: a pair list's (see PairLists), or those of them that the
// hot-latent accumulators have not taken.
struct LongList {
  const uint32_t *ctrl;  // [kLongChunks], [kLongCount]
  const uint32_t *list;
  const uint32_t *chunk_begin;
};

// Decode work item `chunk` of the long-latent work list: which latent, which rows.
struct LongChunk {
  uint32_t long_slot;
  int64_t f;
  uint32_t s0, s1;  // rows [s0, s1) of the pair list
};
__device__ __forceinline__ LongChunk seg_decode_chunk(const uint32_t *__restrict__ begin,
                                                      const uint32_t *__restrict__ long_list,
                                                      const uint32_t *__restrict__ chunk_begin,
                                                      uint32_t n_long, uint32_t chunk) {
  uint32_t lo = 0, hi = n_long;  // largest i with chunk_begin[i] <= chunk
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (chunk_begin[mid] <= chunk) lo = mid; else hi = mid;
  }
  LongChunk c;
  c.long_slot = lo;
  c.f = long_list[lo];
  c.s0 = begin[c.f] + (chunk - chunk_begin[lo]) * kSegChunk;
  const uint32_t s_lim = begin[c.f + 1];
  c.s1 = (s_lim - c.s0) < static_cast<uint32_t>(kSegChunk) ? s_lim : c.s0 + kSegChunk;
  return c;
}

// Segment reduction of one slice.
// Blocks [0, n_long_blocks): long latents.  Every (64-row chunk, tile) is reduced by one
// wavefront into partial[chunk, slice column] (fp32); the wavefronts stride over the work list,
// whose length is only known on the device.  seg_reduce_long_finalize_kernel (next launch)
// combines the partials in chunk order.  These blocks come first so that hot latents start
// at once and overlap with the bulk of the work.
// Remaining blocks: one wavefront per (latent, tile of 64*VEC columns of the slice); latents
// without rows get zeros; latents with more than kSegChunk rows are skipped, and with skip_solo those of
// one row (the training step has written them: see kSoloSlotBit).
template <typename PT, typename GT, int VEC, int U>
__global__ __launch_bounds__(256) void seg_reduce_kernel(
    const uint32_t *__restrict__ begin, const uint32_t *__restrict__ long_ctrl,
    const uint32_t *__restrict__ long_list, const uint32_t *__restrict__ chunk_begin,
    const void *__restrict__ P, float *__restrict__ partial, void *__restrict__ out,
    const float *__restrict__ scale, int64_t F, unsigned n_long_blocks, int tps_and_solo, int col0,
    int slice_w, int D) {
  // tiles per slice << 1 | skip_solo: one word, loaded with the first arguments, so that a latent without rows waits
  // for no further one
  const int tps = tps_and_solo >> 1;
  const bool skip_solo = (tps_and_solo & 1) != 0;
  const int lane = lane_id();
  if (blockIdx.x >= n_long_blocks) {
    // one wavefront per (latent, tile), tiles of a latent adjacent: the launch reads P front to back
    const int64_t item = static_cast<int64_t>(blockIdx.x - n_long_blocks) * (blockDim.x >> 6) + wave_in_block();
    const int64_t f = item / tps;
    if (f >= F) return;  // uniform per wavefront
    const int t = static_cast<int>(item - f * tps);
    const uint32_t s0 = begin[f];
    const uint32_t n = begin[f + 1] - s0;
    const int pc = t * (kWave * VEC) + lane * VEC;
    const int d0 = col0 + pc;
    float acc[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
    if (n != 0) {  // (first of all: a launch over mostly empty latents is bound by its scalar instructions)
      if (n > static_cast<uint32_t>(kSegChunk)) return;
      if (n == 1 && skip_solo) return;
      accumulate_rows<PT, VEC, U, FLEXSAE_REDUCE_NT>(P, s0, static_cast<int>(n), slice_w, pc, acc);
    }
    if (scale) {  // the rows were produced for a unit upstream gradient
      const float g = scale[0];
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] *= g;
    }
    if (d0 < D) store_vec<GT, VEC, FLEXSAE_REDUCE_NT>(out, f * D + d0, acc);
    return;
  }
  const uint32_t n_long = long_ctrl[kLongCount];
  if (n_long == 0) return;
  const int64_t total = static_cast<int64_t>(long_ctrl[kLongChunks]) * tps;
  const int64_t n_waves = static_cast<int64_t>(n_long_blocks) * (blockDim.x >> 6);
  for (int64_t w = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + wave_in_block(); w < total;
       w += n_waves) {
    const uint32_t chunk = static_cast<uint32_t>(w / tps);
    const int t = static_cast<int>(w - static_cast<int64_t>(chunk) * tps);
    const LongChunk c = seg_decode_chunk(begin, long_list, chunk_begin, n_long, chunk);
    const int pc = t * (kWave * VEC) + lane * VEC;
    float acc[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
    accumulate_rows_by4<PT, VEC, 8, FLEXSAE_REDUCE_NT>(P, c.s0, static_cast<int>(c.s1 - c.s0), slice_w, pc, acc);
    store_vec<float, VEC>(partial, static_cast<int64_t>(chunk) * slice_w + pc, acc);
  }
}

// Same reduction with a finer work item: sixteen lanes (a quarter of a wavefront), 16 bytes each,
// serve one (latent, 256-byte piece of the slice's rows of P) -- 128 columns of bf16 contributions,
// 64 of fp32 -- so that a slice may be any whole number of such pieces wide.  A narrow slice is what
// keeps the contributions of one slice in the memory-side cache between the launch that writes them
// and this one.  The four latents (or pieces) of a wavefront have different row counts: the loop
// runs to the longest, loads beyond a group's own count are masked off.  Work order: pieces of a
// latent adjacent, latents ascending, so the launch still reads P front to back.  G > 1: a group
// serves G latents taken from the lists of latents by row count (chosen by the caller where most
// latents have no or few rows), and latents without rows are not written here.
// The rows of `out` may start and end anywhere (store_vec_upto): 24571 latents of 1538 bf16 columns, 3.6 rows each,
// took 13.6 us per 256 columns at 4 bytes per lane (one wavefront per latent and 128 columns), 11.1 by pieces.
__device__ __forceinline__ int64_t ceil_div_u32(uint32_t a, int b) { return (static_cast<int64_t>(a) + b - 1) / b; }

constexpr int kPieceLanes = 16;
constexpr int kPieceBytes = kPieceLanes * 16;
// What a reduction by pieces is told in one word: the blocks of a launch over mostly empty latents are so short that
// every further load of an argument shows (387930 latents of 2240 fp32 columns: the step 592 us with a word each and a test
// against the number of items, 557 without).
enum { kReduceUpdate = 1, kReduceSkipSolo = 2, kReduceDwords = 4 };
// The lists of a reduction that works from them; a launch that does not is not handed their addresses.
struct NoLists {};
template <int G>
using PieceLists = std::conditional_t<(G > 1), PairLists, NoLists>;

template <typename PT, typename GT, int U, int G>
__global__ __launch_bounds__(256) void seg_reduce_piece_kernel(
    const uint32_t *__restrict__ begin, const uint32_t *__restrict__ long_ctrl,
    const uint32_t *__restrict__ long_list, const uint32_t *__restrict__ chunk_begin,
    const void *__restrict__ P, float *__restrict__ partial, void *__restrict__ out,
    const float *__restrict__ scale, int64_t F, unsigned n_long_blocks, int pps, int pps_shift, int col0,
    int slice_w, int D, int how, PieceLists<G> lists) {
  const bool update = (how & kReduceUpdate) != 0, skip_solo = (how & kReduceSkipSolo) != 0, dwords = (how & kReduceDwords) != 0;
  using S = typename Traits<PT>::store_t;
  constexpr int EV = 16 / static_cast<int>(sizeof(S));  // columns per lane
  constexpr int kGroupsPerBlock = 256 / kPieceLanes;
  const int sub = static_cast<int>(threadIdx.x) & (kPieceLanes - 1);
  const int group = static_cast<int>(threadIdx.x) / kPieceLanes;
  const S *__restrict__ Pp = static_cast<const S *>(P);

  // acc += rows r0, r0+step, ... (n of them) of P at the lane's columns; n differs between the
  // groups of a wavefront
  auto accumulate = [&](int64_t r0, int n, int step, int pc, float (&acc)[EV]) {
    const S *row = Pp + r0 * slice_w + pc;
    const int64_t stride = static_cast<int64_t>(step) * slice_w;
    for (int j = 0; __any(j < n); j += U) {
      raw_vec_t<PT, EV> raw[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        raw[u] = raw_vec_t<PT, EV>{};
        if (j + u < n)
          raw[u] = __builtin_nontemporal_load(reinterpret_cast<const raw_vec_t<PT, EV> *>(row + (j + u) * stride));
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float x[EV];
        unpack_raw<PT, EV>(raw[u], x);
#pragma unroll
        for (int i = 0; i < EV; ++i) acc[i] += x[i];  // masked-off loads left zeros
      }
    }
  };

  // A latent's finished sum goes to out[f, d0..]; in update mode it is subtracted from what is there
  // (out is then the weight matrix, the sum arrives scaled by the step size, and latents without
  // rows are left alone).
  auto emit = [&](int64_t f, int d0, float (&acc)[EV]) {
    if (d0 >= D) return;
    if (update) {
      float w[EV];
      load_vec<GT, EV>(out, f * D + d0, w);
#pragma unroll
      for (int i = 0; i < EV; ++i) acc[i] = w[i] - acc[i];
    }
    store_vec_upto<GT, EV, FLEXSAE_REDUCE_NT>(out, f * D + d0, acc, D - d0, dwords);
  };

  if (blockIdx.x >= n_long_blocks) {
    // (latent block, piece) of this group of lanes; a latent block is G consecutive latents.  How many
    // there are is only known on the device where they come from the lists: a bounded number of blocks strides
    // over them (a block for every group there could be is four times as many, most of them empty: 69 instead of
    // 64 us for 75 750 latents of 1 to 8 and 4 252 of 9 to 64 rows of 512 columns).  A block's first item is split with one wave-uniform division; the sixteen groups then only
    // divide a number below pps + 16 (a 64-bit division per lane would cost more instructions than
    // the rest of a short item)
    int64_t n_items = 0;
    int64_t item0 = static_cast<int64_t>(blockIdx.x - n_long_blocks) * kGroupsPerBlock;
    if constexpr (G > 1) {
#pragma unroll
      for (int i = 0; i < kClasses; ++i)
        n_items += i == 0 && skip_solo ? 0 : ceil_div_u32(lists.ctrl[kClassCount + i], i < kClassSolo ? G : 1);
      n_items *= pps;
      if (item0 >= n_items) return;
    }
    const int64_t item_stride = static_cast<int64_t>(gridDim.x - n_long_blocks) * kGroupsPerBlock;
    do {
      int64_t fb;
      int t;
      if (pps_shift >= 0) {  // pps is a power of two (the usual slice widths): shifts only
        const int64_t item = item0 + group;
        fb = item >> pps_shift;
        t = static_cast<int>(item & ((1 << pps_shift) - 1));
      } else {
        const int64_t f_first = item0 / pps;
        const uint32_t rem = static_cast<uint32_t>(item0 - f_first * pps) + static_cast<uint32_t>(group);
        const uint32_t q = rem / static_cast<uint32_t>(pps);
        fb = f_first + q;
        t = static_cast<int>(rem - q * static_cast<uint32_t>(pps));
      }
      const int pc = t * (kPieceLanes * EV) + sub * EV;
      const int d0 = col0 + pc;
      const float g = scale ? scale[0] : 1.0f;  // the rows were produced for a unit upstream gradient
      float acc[EV];
#pragma unroll
      for (int i = 0; i < EV; ++i) acc[i] = 0.f;
      if constexpr (G == 1) {
        const int64_t f = fb;
        uint32_t s0 = 0, n = 0;
        if (f < F) {
          s0 = begin[f];
          n = begin[f + 1] - s0;
        }
        // longer ones: chunked below
        const bool mine = f < F && n <= static_cast<uint32_t>(kSegChunk) && !(skip_solo && n == 1);
        accumulate(s0, mine ? static_cast<int>(n) : 0, 1, pc, acc);
        if (scale) {
#pragma unroll
          for (int i = 0; i < EV; ++i) acc[i] *= g;
        }
        if (mine && !(update && n == 0)) emit(f, d0, acc);
      } else {
        // Few rows per latent and most latents without any: the latents come from the lists of the pair
        // list (those without rows are zeroed by seg_zero_rows_kernel and skipped here; those with more
        // than kSegChunk rows are in neither list).  A group serves G consecutive entries, i.e. G latents
        // of nearly always the same row count, so the four groups of a wavefront finish together; their
        // rows are fetched U at a time regardless of where one latent ends and the next begins, and a
        // latent's sum is stored when its last row has been added.  The order of the additions of a
        // latent is the same as with G = 1.  Work items: the classes in descending order, so that the heaviest
        // groups start first, those of kClassSolo on one latent per group (a group that had four of them
        // would still be running long after the rest of the launch), the others G per group.
        const uint32_t *list = nullptr;  // first entry of this group
        int count = 0;                   // entries it serves
        int64_t at = fb;
#pragma unroll
        for (int i = kClasses - 1; i >= 0; --i) {
          const int64_t n_cls = static_cast<int64_t>(lists.ctrl[kClassCount + i]);
          const int per = i < kClassSolo ? G : 1;
          const int64_t groups = ceil_div_u32(lists.ctrl[kClassCount + i], per);
          if (at >= 0 && at < groups && !(i == 0 && skip_solo)) {
            list = lists.cls_list[i] + at * per;
            const int64_t left = n_cls - at * per;
            count = left < per ? static_cast<int>(left) : per;
          }
          at -= groups;
        }
        uint32_t fv = 0, b0v = 0, b1v = 0;  // lane j < count of the group: entry j, its latent and rows
        if (sub < count) {
          fv = list[sub];
          b0v = begin[fv];
          b1v = begin[fv + 1];
        }
        uint32_t c[G + 1], off[G], fid[G];  // row i of the group's list, c[j] <= i < c[j+1], is row i + off[j] of P
        c[0] = 0;
#pragma unroll
        for (int j = 0; j < G; ++j) {
          const uint32_t b0 = static_cast<uint32_t>(__shfl(static_cast<int>(b0v), j, kPieceLanes));
          const uint32_t b1 = static_cast<uint32_t>(__shfl(static_cast<int>(b1v), j, kPieceLanes));
          fid[j] = static_cast<uint32_t>(__shfl(static_cast<int>(fv), j, kPieceLanes));
          c[j + 1] = c[j] + (b1 - b0);  // nothing for entries beyond the list
          off[j] = b0 - c[j];
        }
        const uint32_t total = c[G];
        for (uint32_t i0 = 0; __any(i0 < total); i0 += U) {
          raw_vec_t<PT, EV> raw[U];
          uint32_t whose[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + u;
            raw[u] = raw_vec_t<PT, EV>{};
            whose[u] = fid[0];
            uint32_t o = off[0];
#pragma unroll
            for (int j = 1; j < G; ++j)
              if (i >= c[j]) {
                whose[u] = fid[j];
                o = off[j];
              }
            if (i < total)
              raw[u] = __builtin_nontemporal_load(reinterpret_cast<const raw_vec_t<PT, EV> *>(
                  Pp + static_cast<int64_t>(i + o) * slice_w + pc));
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + u;
            float x[EV];
            unpack_raw<PT, EV>(raw[u], x);
#pragma unroll
            for (int k = 0; k < EV; ++k) acc[k] += x[k];  // masked-off loads left zeros
            bool last = false;  // the last row of its latent
#pragma unroll
            for (int j = 1; j <= G; ++j) last |= i + 1 == c[j];
            if (i < total && last) {
              if (scale) {
#pragma unroll
                for (int k = 0; k < EV; ++k) acc[k] *= g;
              }
              emit(static_cast<int64_t>(whose[u]), d0, acc);
#pragma unroll
              for (int k = 0; k < EV; ++k) acc[k] = 0.f;
            }
          }
        }
      }
      // (without the lists the grid covers every item: no loop around the short body, whose loads would wait for
      // the loop's bookkeeping; 131072 latents of 64 fp32 columns, four rows each: 27.6 us looped, 26.8 not)
      if constexpr (G == 1) return;
      item0 += item_stride;
    } while (item0 < n_items);
    return;
  }
  // Long latents: one wavefront per (64-row chunk, piece); its four groups take every fourth row
  // (sixteen rows in flight per wavefront) and their sums are added across the groups in a fixed
  // order.  A hot latent's chunks are spread over many wavefronts.
  const uint32_t n_long = long_ctrl[kLongCount];
  if (n_long == 0) return;
  constexpr int kGroups = kWave / kPieceLanes;
  const int64_t total = static_cast<int64_t>(long_ctrl[kLongChunks]) * pps;
  const int64_t n_waves = static_cast<int64_t>(n_long_blocks) * (blockDim.x >> 6);
  const int g = (static_cast<int>(threadIdx.x) & (kWave - 1)) / kPieceLanes;
  for (int64_t w = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + wave_in_block(); w < total; w += n_waves) {
    const uint32_t chunk = static_cast<uint32_t>(w / pps);
    const int t = static_cast<int>(w - static_cast<int64_t>(chunk) * pps);
    const LongChunk c = seg_decode_chunk(begin, long_list, chunk_begin, n_long, chunk);
    const int rows = static_cast<int>(c.s1 - c.s0);
    const int pc = t * (kPieceLanes * EV) + sub * EV;
    float acc[EV];
#pragma unroll
    for (int i = 0; i < EV; ++i) acc[i] = 0.f;
    accumulate(static_cast<int64_t>(c.s0) + g, (rows - g + kGroups - 1) / kGroups, kGroups, pc, acc);
#pragma unroll
    for (int i = 0; i < EV; ++i) acc[i] = add_across_rows(acc[i]);
    if (g == 0) store_vec<float, EV>(partial, static_cast<int64_t>(chunk) * slice_w + pc, acc);
  }
}

// Long latents of the piece reduction, second step: out[f, slice] = sum of the latent's chunk
// partials in a fixed order.  One wavefront per (long latent, 64-column piece of the fp32
// partials); its four groups take every fourth chunk and are added up as above.  `block` of
// `n_blocks` blocks of 256 threads share the work (a launch of its own, or the leading blocks of
// the next slice's training-step launch).
template <typename GT>
__device__ __forceinline__ void seg_piece_finalize_body(
    const uint32_t *__restrict__ long_ctrl, const uint32_t *__restrict__ long_list,
    const uint32_t *__restrict__ chunk_begin, const float *__restrict__ partial,
    void *__restrict__ out, const float *__restrict__ scale, int pieces, int col0, int slice_w, int D,
    int update, int dwords, unsigned block, unsigned n_blocks) {
  constexpr int EV = 4, U = 4, kGroups = kWave / kPieceLanes;
  const int lane = lane_id();
  const int sub = lane & (kPieceLanes - 1), g = lane / kPieceLanes;
  const uint32_t n_long = long_ctrl[kLongCount];
  const int64_t total = static_cast<int64_t>(n_long) * pieces;
  const int64_t n_waves = static_cast<int64_t>(n_blocks) * (blockDim.x >> 6);
  for (int64_t w = static_cast<int64_t>(block) * (blockDim.x >> 6) + wave_in_block(); w < total; w += n_waves) {
    const uint32_t i = static_cast<uint32_t>(w / pieces);
    const int t = static_cast<int>(w - static_cast<int64_t>(i) * pieces);
    const int pc = t * (kPieceLanes * EV) + sub * EV;
    const int d0 = col0 + pc;
    const uint32_t c0 = chunk_begin[i], c1 = i + 1 < n_long ? chunk_begin[i + 1] : long_ctrl[kLongChunks];
    const int n = (static_cast<int>(c1 - c0) - g + kGroups - 1) / kGroups;
    const float *row = partial + (static_cast<int64_t>(c0) + g) * slice_w + pc;
    const int64_t stride = static_cast<int64_t>(kGroups) * slice_w;
    float acc[EV] = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; __any(j < n); j += U) {
      vec_t<float, EV> raw[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        raw[u] = vec_t<float, EV>{};
        if (j + u < n) raw[u] = *reinterpret_cast<const vec_t<float, EV> *>(row + (j + u) * stride);
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int k = 0; k < EV; ++k) acc[k] += raw[u][k];
    }
#pragma unroll
    for (int k = 0; k < EV; ++k) acc[k] = add_across_rows(acc[k]);
    if (scale) {
      const float gs = scale[0];
#pragma unroll
      for (int k = 0; k < EV; ++k) acc[k] *= gs;
    }
    if (g == 0 && d0 < D) {
      const int64_t o = static_cast<int64_t>(long_list[i]) * D + d0;
      if (update) {  // out is the weight matrix: subtract the (scaled) sum from it
        float w[EV];
        load_vec<GT, EV>(out, o, w);
#pragma unroll
        for (int k = 0; k < EV; ++k) acc[k] = w[k] - acc[k];
      }
      store_vec_upto<GT, EV>(out, o, acc, D - d0, dwords);
    }
  }
}

// Long latents, second step of the reduction by tiles: out[f, slice] = sum of the latent's chunk
// partials, in chunk order.
template <typename GT, int VEC, int U>
__device__ __forceinline__ void seg_long_finalize_body(
    const uint32_t *__restrict__ long_ctrl, const uint32_t *__restrict__ long_list,
    const uint32_t *__restrict__ chunk_begin, const float *__restrict__ partial,
    void *__restrict__ out, const float *__restrict__ scale, int tps, int col0, int slice_w, int D,
    unsigned block, unsigned n_blocks) {
  const int lane = lane_id();
  const uint32_t n_long = long_ctrl[kLongCount];
  const int64_t total = static_cast<int64_t>(n_long) * tps;
  const int64_t n_waves = static_cast<int64_t>(n_blocks) * (blockDim.x >> 6);
  for (int64_t w = static_cast<int64_t>(block) * (blockDim.x >> 6) + wave_in_block(); w < total;
       w += n_waves) {
    const uint32_t i = static_cast<uint32_t>(w / tps);
    const int t = static_cast<int>(w - static_cast<int64_t>(i) * tps);
    const int pc = t * (kWave * VEC) + lane * VEC;
    const int d0 = col0 + pc;
    const uint32_t c0 = chunk_begin[i], c1 = i + 1 < n_long ? chunk_begin[i + 1] : long_ctrl[kLongChunks];
    float acc[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) acc[k] = 0.f;
    accumulate_rows_by4<float, VEC, U>(partial, c0, static_cast<int>(c1 - c0), slice_w, pc, acc);
    if (scale) {
      const float g = scale[0];
#pragma unroll
      for (int k = 0; k < VEC; ++k) acc[k] *= g;
    }
    if (d0 < D) store_vec<GT, VEC>(out, static_cast<int64_t>(long_list[i]) * D + d0, acc);
  }
}

template <typename GT, int VEC, int U>
__global__ __launch_bounds__(256) void seg_reduce_long_finalize_kernel(
    const uint32_t *__restrict__ long_ctrl, const uint32_t *__restrict__ long_list,
    const uint32_t *__restrict__ chunk_begin, const float *__restrict__ partial,
    void *__restrict__ out, const float *__restrict__ scale, int tps, int col0, int slice_w, int D) {
  seg_long_finalize_body<GT, VEC, U>(long_ctrl, long_list, chunk_begin, partial, out, scale, tps, col0, slice_w, D,
                                     blockIdx.x, gridDim.x);
}

// The second step of a slice's hot latents as a parcel that another launch can carry: the
// training-step kernel of the next slice runs it in its leading blocks (it touches neither the
// contributions nor the partial sums, and the reduction that overwrites the partial sums comes after
// it in the stream), which saves a launch per slice.
struct HotFinalize {
  const uint32_t *long_ctrl;
  const uint32_t *long_list;
  const uint32_t *chunk_begin;
  const float *partial;
  void *out;
  const float *scale;
  int mode;   // 0: nothing, 1: pieces of 64 columns, 2: tiles of 256 columns, 3: tiles of 128 columns
  int units;  // pieces or tiles per slice
  int col0, slice_w, D, update;
  int dwords;  // rows of `out` start at multiples of four bytes (mode 1)
  int weight_typed;  // `out` has the weight's type where CarriedGrad's is another (mode 1; so it does with update)
  unsigned n_blocks;  // blocks of 256 threads that share it
};

template <typename GT>
__device__ __forceinline__ void hot_finalize_run(const HotFinalize &h, unsigned block) {
  if (h.mode == 1)
    seg_piece_finalize_body<GT>(h.long_ctrl, h.long_list, h.chunk_begin, h.partial, h.out, h.scale, h.units, h.col0,
                                h.slice_w, h.D, h.update, h.dwords, block, h.n_blocks);
  else if (h.mode == 2)
    seg_long_finalize_body<GT, 4, 8>(h.long_ctrl, h.long_list, h.chunk_begin, h.partial, h.out, h.scale, h.units,
                                     h.col0, h.slice_w, h.D, block, h.n_blocks);
  else if (h.mode == 3)
    seg_long_finalize_body<GT, 2, 8>(h.long_ctrl, h.long_list, h.chunk_begin, h.partial, h.out, h.scale, h.units,
                                     h.col0, h.slice_w, h.D, block, h.n_blocks);
}

// Gradient type of the finalize work that a training-step launch carries: the weight's own, or fp32 for fp16 weights (whose
// unit gradient would underflow); by pieces also the weight's type there: the in-place update, and a gradient that is
// scaled before its only rounding.
template <typename WT>
struct CarriedGrad {
  using type = WT;
};
template <>
struct CarriedGrad<f16_t> {
  using type = float;
};

template <typename WT>
__device__ __forceinline__ void hot_finalize_carried(const HotFinalize &h, unsigned block) {
  if constexpr (!std::is_same<WT, typename CarriedGrad<WT>::type>::value) {
    if (h.weight_typed) {
      if (h.mode == 1)
        seg_piece_finalize_body<WT>(h.long_ctrl, h.long_list, h.chunk_begin, h.partial, h.out, h.scale, h.units, h.col0,
                                    h.slice_w, h.D, h.update, h.dwords, block, h.n_blocks);
      return;
    }
  }
  hot_finalize_run<typename CarriedGrad<WT>::type>(h, block);
}

template <typename GT>
__global__ __launch_bounds__(256) void hot_finalize_kernel(HotFinalize h) {
  hot_finalize_run<GT>(h, blockIdx.x);
}

// out[f, 0..D) = 0 for the latents without rows: kZeroRows rows of the list per wavefront, 16 bytes per lane.  Bound by
// the memory's write rate.  A wavefront's rows are neighbours in the (ascending) list, their numbers one load, and the
// stores carry no streaming hint: rows that do not end on a line share it with the next one, and a hint sends the two
// parts of the line to memory one by one.  693763 rows of 382 fp32 columns (1.06 GB): 281 us with a hint and the wavefronts
// of the launch taking every 8192nd row each, 238 with neighbouring rows, 199 without the hint; 250000 rows of 4096 bf16
// columns: 295 and 257 with and without.
constexpr int kZeroRows = 8;
template <typename GT>
__device__ __forceinline__ void zero_rows_block(const uint32_t *__restrict__ ctrl, const uint32_t *__restrict__ empty_list,
                                                void *__restrict__ out, int D, int dwords, unsigned block) {
  constexpr int EV = 16 / static_cast<int>(sizeof(typename Traits<GT>::store_t));
  const uint32_t n = ctrl[kListed] ? ctrl[kEmptyCount] : 0u;
  const int lane = lane_id();
  const int64_t w0 = (static_cast<int64_t>(block) * (blockDim.x >> 6) + wave_in_block()) * kZeroRows;
  if (w0 >= n) return;  // uniform per wavefront
  const int rows = static_cast<int>((n - w0) < kZeroRows ? (n - w0) : kZeroRows);
  const int mine = lane < rows ? static_cast<int>(empty_list[w0 + lane]) : 0;
  float zero[EV];
#pragma unroll
  for (int i = 0; i < EV; ++i) zero[i] = 0.f;
  for (int r = 0; r < rows; ++r) {
    const int64_t row = static_cast<int64_t>(static_cast<uint32_t>(bcast_i32(mine, r))) * D;
    for (int d = lane * EV; d < D; d += kWave * EV) store_vec_upto<GT, EV>(out, row + d, zero, D - d, dwords);
  }
}

template <typename GT>
__global__ __launch_bounds__(256) void seg_zero_rows_kernel(const uint32_t *__restrict__ ctrl,
                                                            const uint32_t *__restrict__ empty_list,
                                                            void *__restrict__ out, int D, int dwords) {
  zero_rows_block<GT>(ctrl, empty_list, out, D, dwords, blockIdx.x);
}

// The same for blocks of another launch (n_blocks of them; 0: none): zero is zero in every type, so rows of 16-bit elements
// are bf16 here.
struct ZeroRows {
  const uint32_t *ctrl, *empty_list;
  void *out;
  int wide;  // 32-bit elements
  int dwords;
  unsigned n_blocks;
};

__device__ __forceinline__ void zero_rows_carried(const ZeroRows &z, int D, unsigned block) {
  if (z.wide) zero_rows_block<float>(z.ctrl, z.empty_list, z.out, D, z.dwords, block);
  else zero_rows_block<bf16_t>(z.ctrl, z.empty_list, z.out, D, z.dwords, block);
}

}  // namespace flexsae
