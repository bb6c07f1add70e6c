// Forward kernels: fused embedding-bag + bias - target + squared error, for the TopK loss
// (one squared error at the end of the row) and the HierarchicalTopK loss (one after
// every prefix), without ever materialising the [B,K,D] reconstruction.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace flexsae {

// Work decomposition: a block of four wavefronts walks 4 * R rows of one narrow column tile.  LPR lanes
// serve a row piece of LPR * VEC columns, so a wavefront has R = 64 / LPR rows and one vector load
// fetches R row pieces.  Every step's row number and val are read from the LDS, where the
// wavefront has put those of kFwdChunk steps of its R rows with coalesced loads (a broadcast read:
// all lanes of a piece read the same entry).  U independent gathers are issued before the first one
// is consumed.
//
// What bounds it: the gathered bytes.  The weight matrix is read once per pair, and how fast depends on
// which cache answers.  Three orders of the (tile, row block) items, picked by plan_fwd:
//   xcd_span > 0   the items, tiles outermost, are cut into eight equal runs, one per L2 (blocks
//                  go round the eight XCDs): an L2 sees F pieces of one narrow tile at a time instead of
//                  whole rows.  65536 pieces of 128 bytes are 8.4 MB against 4 MB of L2: about half of the
//                  gathers hit.  128 bytes is the L2's line; 64-byte pieces fetch the whole line anyway
//                  (twice as slow).
//   xcd_span == 0  items in order, tiles outermost, wide tiles: all XCDs gather from the same column
//                  tile, which the memory-side cache (256 MB) holds where the L2s cannot help.
//   xcd_span < 0   wavefronts in order, the -xcd_span tiles of a row next to each other: where no cache
//                  holds a tile long enough for its pieces to be asked for again, and where rows do not
//                  start on a 128-byte line and neighbouring pieces share lines.
// Against one wavefront per (row, 256 columns) in row order, which no cache but the memory-side one served:
// B=4096, K=128, F=65536, D=2304 bf16 (2.42 GB gathered) 328 -> 275 us (8.8 TB/s), K=64 172 -> 143 us; B=2048,
// K=256, F=131072, D=1024 fp32 292 -> 273 us; B=16384, K=128, F=524288, D=8192 bf16 6.3 -> 4.8 ms (7.2 TB/s).
// Where the L2s serve nearly all of it (skewed indices, few latents) it runs at their 18 TB/s.  Streaming hints
// on the index loads cost 5-10 % (the eight XCDs share those lines in the memory-side cache); 32-bit
// offsets through a buffer descriptor change nothing.
//
// Per item the block writes resid[b, tile] = r_{b,K-1} - target_b (fp32) and one partial sum of squares;
// loss_finalize_kernel adds the partials in a fixed order, so the loss is bit-reproducible from
// run to run.  Everything beyond a lane's own column of a row is added in double.
constexpr int kFwdChunk = 64;  // steps per LDS fill

// Bits of a pair's position in a row of at most 64 * C pairs (topk_order_kernel).
constexpr int order_pos_bits(int C) { return C == 1 ? 6 : C == 2 ? 7 : C == 4 ? 8 : 9; }

template <typename WT, int VEC, int LPR, bool HIER, int U>
__global__ __launch_bounds__(256) void sae_fwd_kernel(
    const int64_t *__restrict__ indices, const void *__restrict__ weight,
    const void *__restrict__ vals, int vals_dtype, const void *__restrict__ bias, int bias_dtype,
    const void *__restrict__ target, int target_dtype, float *__restrict__ resid,
    double *__restrict__ partial, int *status_flag, int64_t B, int64_t n_row_blocks, int64_t n_items,
    int64_t xcd_span, int K, int64_t F, int D) {
  constexpr int R = kWave / LPR;  // rows per wavefront
  constexpr int kWaves = 256 / kWave;
  static_assert(kFwdChunk == kWave && kFwdChunk % U == 0, "one lane per step of a chunk");
  __shared__ vec_t<uint32_t, 2> steps[kWaves][R][kFwdChunk];  // (row of the weight matrix, val bits)
  __shared__ double wave_loss[kWaves];
  const int lane = lane_id();
  const int wv = wave_in_block();
  int64_t item = blockIdx.x;
  if (xcd_span > 0) {
    const int64_t i = item >> 3;
    item = (item & 7) * xcd_span + i;
    if (i >= xcd_span) return;  // uniform per block
  }
  if (item >= n_items) return;  // uniform per block
  int64_t tile, b0;  // of the wavefront: its tile, its first row
  bool idle = false;
  if (xcd_span >= 0) {
    tile = item / n_row_blocks;
    b0 = ((item - tile * n_row_blocks) * kWaves + wv) * R;
  } else {
    const int64_t n_tiles = -xcd_span;
    const int64_t at = item * kWaves + wv;
    b0 = at / n_tiles;
    tile = at - b0 * n_tiles;
    b0 *= R;
    idle = b0 >= B;  // uniform per wavefront
    if (idle) b0 = 0;
  }
  const int64_t b = b0 + lane / LPR;
  const int d0 = static_cast<int>(tile) * (LPR * VEC) + (lane % LPR) * VEC;
  const bool active = d0 < D && b < B && !idle;  // D % VEC == 0 is checked on the host
  const int dsafe = d0 < D ? d0 : 0;
  const int64_t bsafe = b < B ? b : B - 1;

  // e = reconstruction error, starting from bias - target
  float e[VEC], acc[VEC];
  {
    float t[VEC];
    load_vec_dyn<WT, VEC>(bias, bias_dtype, dsafe, e);
    load_vec_dyn<WT, VEC>(target, target_dtype, bsafe * D + dsafe, t);
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      e[i] -= t[i];
      acc[i] = 0.f;
    }
  }
  using S = typename Traits<WT>::store_t;
  const S *__restrict__ wbase = static_cast<const S *>(weight) + dsafe;
  const uint32_t d_elems = static_cast<uint32_t>(D);
  const vec_t<uint32_t, 2> *my_steps = &steps[wv][lane / LPR][0];

  auto consume = [&](const raw_vec_t<WT, VEC> &raw, float v) {
    float w[VEC];
    unpack_raw<WT, VEC>(raw, w);
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      e[i] = fmaf(w[i], v, e[i]);
      if constexpr (HIER) acc[i] = fmaf(e[i], e[i], acc[i]);
    }
  };
  auto gather = [&](uint32_t row) {
    return *reinterpret_cast<const raw_vec_t<WT, VEC> *>(wbase + static_cast<uint64_t>(row) * d_elems);
  };

  for (int k0 = idle ? K : 0; k0 < K; k0 += kFwdChunk) {
    const int n = (K - k0) < kFwdChunk ? (K - k0) : kFwdChunk;  // uniform
    // lane j: step k0 + j of every row of the wavefront
    {
      int64_t idx[R];
      uint32_t vbits[R];
      const int kk = k0 + (lane < n ? lane : 0);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int64_t p = (b0 + r < B ? b0 + r : B - 1) * K + kk;
        idx[r] = indices[p];
        vbits[r] = load_scalar_bits(vals, vals_dtype, p);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float v = scalar_from_bits(vbits[r], vals_dtype);
        if (static_cast<uint64_t>(idx[r]) >= static_cast<uint64_t>(F)) {
          if (status_flag) atomicOr(status_flag, FLEXSAE_FLAG_INDEX_RANGE);
          idx[r] = 0;
          v = 0.f;
        }
        vec_t<uint32_t, 2> s;
        s[0] = static_cast<uint32_t>(idx[r]);
        s[1] = __float_as_uint(v);
        steps[wv][r][lane] = s;
      }
      // (the wavefront's own LDS accesses are served in order; this keeps the compiler from moving them)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    int j = 0;
    for (; j + U <= n; j += U) {
      raw_vec_t<WT, VEC> raw[U];
      float v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const vec_t<uint32_t, 2> s = my_steps[j + u];
        v[u] = __uint_as_float(s[1]);
        raw[u] = gather(s[0]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) consume(raw[u], v[u]);
    }
    for (; j + 4 <= n; j += 4) {
      raw_vec_t<WT, VEC> raw[4];
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const vec_t<uint32_t, 2> s = my_steps[j + u];
        v[u] = __uint_as_float(s[1]);
        raw[u] = gather(s[0]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) consume(raw[u], v[u]);
    }
    for (; j < n; ++j) {
      const vec_t<uint32_t, 2> s = my_steps[j];
      consume(gather(s[0]), __uint_as_float(s[1]));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }

  double lsum = 0.0;
#pragma unroll
  for (int i = 0; i < VEC; ++i) {
    if constexpr (HIER) {
      lsum += static_cast<double>(acc[i]);
    } else {
      lsum = fma(static_cast<double>(e[i]), static_cast<double>(e[i]), lsum);
    }
  }
  if (active) {
    store_vec<float, VEC>(resid, b * D + d0, e);
  } else {
    lsum = 0.0;
  }
  lsum = wave_sum_lane63(lsum);
  if (lane == kWave - 1) wave_loss[wv] = lsum;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s += wave_loss[w];
    partial[item] = s;
  }
}

// ---- TopK forward in latent order ---------------------------------------------------------
// The TopK loss adds a row's pairs up in any order, so every row can walk them by ascending latent.  The wavefronts that
// an XCD runs at a time then sweep the latents of their column tile together, and a row piece that one of them gathers is
// still in the L2 when the others ask for it: where one tile's pieces are several times the L2, the misses fall to about
// the weights once (B=4096, K=128, F=65536, D=2304 bf16: 16.3 -> 6.3 million lines, 2.1 -> 0.8 GB; the least is 2.4).

// (row of the weight matrix, val bits) of every pair, each row's pairs by ascending latent (and by position where two are
// equal: the order, and so every sum, is the same on every run).  One wavefront per row of at most 64 * C pairs: a bitonic
// sort of one key per pair, the latent over the pair's position (fewer than 2^20 latents).  An index outside [0, F) becomes
// latent 0 with a val of zero, as in the kernels that read indices themselves.  5-6 us for half a million pairs, most of it
// the launch (ranks by counting, a comparison per pair of pairs: 9 us at K=128, 19 at K=256).
template <int C>
__global__ __launch_bounds__(256) void topk_order_kernel(const int64_t *__restrict__ indices, const void *__restrict__ vals,
                                                         int vals_dtype, int64_t B, int K, int64_t F,
                                                         vec_t<uint32_t, 2> *__restrict__ steps, int *status_flag) {
  constexpr int N = kWave * C;
  constexpr int kPosBits = order_pos_bits(C);
  static_assert(N == 1 << kPosBits, "a key holds the position of a pair in its row");
  __shared__ vec_t<uint32_t, 2> rows[256 / kWave][N];
  const int lane = lane_id();
  vec_t<uint32_t, 2> *const mine = rows[wave_in_block()];
  const int64_t b = static_cast<int64_t>(blockIdx.x) * (256 / kWave) + wave_in_block();
  if (b >= B) return;  // uniform per wavefront
  // element e = lane * C + c of the row
  uint32_t key[C], vbits[C];
  int64_t idx[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int k = lane * C + c;
    const int64_t p = b * K + (k < K ? k : 0);
    idx[c] = indices[p];
    vbits[c] = load_scalar_bits(vals, vals_dtype, p);
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int k = lane * C + c;
    float v = scalar_from_bits(vbits[c], vals_dtype);
    if (static_cast<uint64_t>(idx[c]) >= static_cast<uint64_t>(F)) {
      if (status_flag) atomicOr(status_flag, FLEXSAE_FLAG_INDEX_RANGE);
      idx[c] = 0;
      v = 0.f;
    }
    vec_t<uint32_t, 2> s;
    s[0] = static_cast<uint32_t>(idx[c]);
    s[1] = __float_as_uint(v);
    mine[k] = s;
    // elements past the row's end sort behind all others
    key[c] = k < K ? static_cast<uint32_t>(idx[c]) << kPosBits | static_cast<uint32_t>(k) : 0xffffffffu;
  }
#pragma unroll
  for (int size = 2; size <= N; size *= 2) {
#pragma unroll
    for (int stride = size / 2; stride > 0; stride /= 2) {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const bool up = size == N || ((lane * C + c) & size) == 0;  // this run ascends
        if (stride >= C) {
          const uint32_t other = __shfl_xor(key[c], stride / C);
          const bool low = (lane & (stride / C)) == 0;
          key[c] = (low == up) == (key[c] < other) ? key[c] : other;
        } else if ((c & stride) == 0) {
          const uint32_t a = key[c], z = key[c | stride];
          key[c] = up == (a < z) ? a : z;
          key[c | stride] = up == (a < z) ? z : a;
        }
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int e = lane * C + c;
    if (e < K) steps[b * K + e] = mine[key[c] & (N - 1)];
  }
}

// sae_fwd_kernel for rows in latent order: NW wavefronts per block, the tiles cut into runs, one per XCD.
// At most four wavefronts per SIMD and eight gathers in flight, sixteen of 256-byte pieces (16-byte lanes): with more of either
// the wavefronts of a tile drift further apart than the L2 covers, and those of the next tile join them.  What bounds it: the
// L2s, at 13-14 of the 18 TB/s they give to row gathers, and the misses beside them (5-6 TB/s).  Ordering included: B=4096,
// K=128, F=65536, D=2304 bf16 286 -> 188 us (128-byte pieces), B=2048, K=256, F=131072, D=1024 fp32 275 -> 181 us (256-byte
// pieces).
template <typename WT, int VEC, int LPR, int U, int NW>
__global__ __launch_bounds__(NW *kWave) __attribute__((amdgpu_waves_per_eu(1, 4))) void topk_ordered_fwd_kernel(
    const vec_t<uint32_t, 2> *__restrict__ ordered, const void *__restrict__ weight, const void *__restrict__ bias,
    int bias_dtype, const void *__restrict__ target, int target_dtype, float *__restrict__ resid,
    double *__restrict__ partial, int64_t B, int64_t n_row_blocks, int64_t n_items, int64_t xcd_span, int K, int D) {
  constexpr int R = kWave / LPR;  // rows per wavefront
  static_assert(kFwdChunk == kWave, "one lane per step of a chunk");
  __shared__ vec_t<uint32_t, 2> steps[NW][R][kFwdChunk];
  __shared__ double wave_loss[NW];
  const int lane = lane_id();
  const int wv = wave_in_block();
  const int64_t i = blockIdx.x >> 3;
  const int64_t item = (blockIdx.x & 7) * xcd_span + i;
  if (i >= xcd_span || item >= n_items) return;  // uniform per block
  const int64_t tile = item / n_row_blocks;
  const int64_t b0 = ((item - tile * n_row_blocks) * NW + wv) * R;
  const int64_t b = b0 + lane / LPR;
  const int d0 = static_cast<int>(tile) * (LPR * VEC) + (lane % LPR) * VEC;
  const bool active = d0 < D && b < B;  // D % VEC == 0 is checked on the host
  const int dsafe = d0 < D ? d0 : 0;
  const int64_t bsafe = b < B ? b : B - 1;
  float e[VEC];
  {
    float t[VEC];
    load_vec_dyn<WT, VEC>(bias, bias_dtype, dsafe, e);
    load_vec_dyn<WT, VEC>(target, target_dtype, bsafe * D + dsafe, t);
#pragma unroll
    for (int k = 0; k < VEC; ++k) e[k] -= t[k];
  }
  using S = typename Traits<WT>::store_t;
  const S *__restrict__ wbase = static_cast<const S *>(weight) + dsafe;
  const uint32_t d_elems = static_cast<uint32_t>(D);
  const vec_t<uint32_t, 2> *my_steps = &steps[wv][lane / LPR][0];
  for (int k0 = 0; k0 < K; k0 += kFwdChunk) {
    const int n = (K - k0) < kFwdChunk ? (K - k0) : kFwdChunk;  // uniform
    {
      vec_t<uint32_t, 2> s[R];
      const int kk = k0 + (lane < n ? lane : 0);
#pragma unroll
      for (int r = 0; r < R; ++r) s[r] = ordered[(b0 + r < B ? b0 + r : B - 1) * K + kk];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int r = 0; r < R; ++r) steps[wv][r][lane] = s[r];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    auto group = [&](auto count, int j) {
      constexpr int N = decltype(count)::value;
      raw_vec_t<WT, VEC> raw[N];
      float v[N];
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const vec_t<uint32_t, 2> s = my_steps[j + u];
        v[u] = __uint_as_float(s[1]);
        raw[u] = *reinterpret_cast<const raw_vec_t<WT, VEC> *>(wbase + static_cast<uint64_t>(s[0]) * d_elems);
      }
#pragma unroll
      for (int u = 0; u < N; ++u) {
        float w[VEC];
        unpack_raw<WT, VEC>(raw[u], w);
#pragma unroll
        for (int k = 0; k < VEC; ++k) e[k] = fmaf(w[k], v[u], e[k]);
      }
    };
    int j = 0;
#pragma unroll 1
    for (; j + U <= n; j += U) group(std::integral_constant<int, U>{}, j);
#pragma unroll 1
    for (; j + 4 <= n; j += 4) group(std::integral_constant<int, 4>{}, j);
#pragma unroll 1
    for (; j < n; ++j) group(std::integral_constant<int, 1>{}, j);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  double lsum = 0.0;
#pragma unroll
  for (int k = 0; k < VEC; ++k) lsum = fma(static_cast<double>(e[k]), static_cast<double>(e[k]), lsum);
  if (active)
    store_vec<float, VEC>(resid, b * D + d0, e);
  else
    lsum = 0.0;
  lsum = wave_sum_lane63(lsum);
  if (lane == kWave - 1) wave_loss[wv] = lsum;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) s += wave_loss[w];
    partial[item] = s;
  }
}

// loss[0] = inv_count * sum(partial[0..n)), one block, fixed summation order, double
// accumulation (n up to a few million).
// (the body, for a block of 1024 threads; `red` is 1024 doubles of LDS; PT: float or double partials)
template <typename PT>
__device__ __forceinline__ void loss_finalize_block(const PT *__restrict__ partial, int64_t n, double inv_count,
                                                    float *__restrict__ loss, double *red) {
  double s = 0.0;
  int64_t i = threadIdx.x;
  if constexpr (sizeof(PT) == 8) {  // two at a time (partial starts at a multiple of 16 bytes)
    const auto *const two = reinterpret_cast<const vec_t<PT, 2> *>(partial);
    const int64_t n2 = n / 2;
    for (; i + 7 * 1024 < n2; i += 8 * 1024) {
      vec_t<PT, 2> x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = two[i + u * 1024];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += x[u][0] + x[u][1];
    }
    for (; i < n2; i += 1024) s += two[i][0] + two[i][1];
    i = n2 * 2 + threadIdx.x;  // the last one of an odd number
  }
  for (; i + 7 * 1024 < n; i += 8 * 1024) {  // eight independent loads in flight
    PT x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = partial[i + u * 1024];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += static_cast<double>(x[u]);
  }
  for (; i < n; i += 1024) s += static_cast<double>(partial[i]);
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (static_cast<int>(threadIdx.x) < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[0] = static_cast<float>(red[0] * inv_count);
}

__global__ __launch_bounds__(1024) void loss_finalize_kernel(const double *__restrict__ partial,
                                                             int64_t n, double inv_count,
                                                             float *__restrict__ loss) {
  __shared__ double red[1024];
  loss_finalize_block(partial, n, inv_count, loss, red);
}

}  // namespace flexsae
