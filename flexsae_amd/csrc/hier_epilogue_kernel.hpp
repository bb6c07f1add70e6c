// The end of a hierarchical step: everything that follows its slices, in one launch.
#pragma once

#include "common.hpp"
#include "csr_kernels.hpp"
#include "fwd_kernels.hpp"
#include "hier_hot_kernel.hpp"
#include "segment_kernels.hpp"

namespace flexsae {

// The most rows whose column sums it finishes: D / 32 blocks are few, and each walks all rows.  Beyond, stage 1 is spread over
// a block per 256 columns and 256 rows and stage 2 is a launch of its own (us of the step with one and with two launches: B=64,
// K=32, F=4096, D=256 fp32 185 and 193; B=1777, K=50, F=24571, D=1538 bf16 209 and 212; B=4096, K=32, F=65536, D=2304 fp16 728
// and 718; with one launch for all sizes and K=128 there 1223 against 1214, B=16384, D=8192 19340 against 19270).
constexpr int64_t kEndRows = 2048;
constexpr int kEndSlots = static_cast<int>(kEndRows / kColsumRows);  // chunks of rows, one thread per column and chunk
constexpr int kEndCols = 1024 / kEndSlots;                           // 32: the 128-byte line of a row
// out[c] = column sums of x [rows <= kEndRows, ld] for the kEndCols columns from c0 on, by one block of 1024 threads: the same
// sums in the same order as colsum_partial_one and colsum_final_one (chunks of kColsumRows rows, added in order), with the
// chunks' sums in the LDS instead of in memory, so that no second launch has to wait for the first.  Bound by its chain of
// loads: sixteen in flight per thread, four trips to memory.
__device__ __forceinline__ void colsum_whole_block(const float *__restrict__ x, int64_t rows, int64_t ld, int cols,
                                                   float *__restrict__ out, int c0, float *__restrict__ sums) {
  static_assert(kEndRows % kColsumRows == 0 && 1024 % kEndSlots == 0, "a thread per column and chunk");
  const int c = c0 + static_cast<int>(threadIdx.x % kEndCols);
  const int64_t r0 = static_cast<int64_t>(threadIdx.x / kEndCols) * kColsumRows;
  const int64_t r1 = (r0 + kColsumRows) < rows ? (r0 + kColsumRows) : rows;
  float s = 0.f;
  if (c < cols) {
    int64_t r = r0;
    for (; r + 16 <= r1; r += 16) {
      float v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = x[(r + u) * ld + c];
#pragma unroll
      for (int u = 0; u < 16; ++u) s += v[u];
    }
    for (; r < r1; ++r) s += x[r * ld + c];
  }
  sums[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x >= kEndCols || c >= cols) return;
  const int n = static_cast<int>((rows + kColsumRows - 1) / kColsumRows);
  float total = 0.f;
  for (int j = 0; j < n; ++j) total += sums[j * kEndCols + threadIdx.x];
  out[c] = total;
}

// What follows the slices of a hierarchical step, in one launch of 1024-thread blocks.  The parts are independent:
//   block 0                   the loss from the per-(tile, row) partials (loss_finalize_kernel), when loss_partial is given, and
//                             what the pair list says about the indices, where that is wanted;
//   the next fin.n_blocks     the second step of the last slice's frequent latents (hot_finalize_run);
//   the next n_hot_blocks     the last slice's accumulator rows (hot_block_finalize_run);
//   the next n_col_blocks     dbias: column sums of s_final, kEndCols columns per block (n_parts = 0), or of more than kEndRows
//                             rows stage 1 of them (n_parts < 0; a block takes 256 columns of four chunks), or, where the
//                             walk formed stage 1 on chip, stage 2 from n_parts partial sums, 1024 columns per block;
//   the rest                  dvals[p] = sum over the column tiles of dv_part[tile, p], in tile order (deterministic),
//                             eight loads in flight.
// As launches of their own the second steps, and dbias's where one block can wait for no other, cost 3-5 us each, whether
// they had work or not: B=1024, K=64, F=32768, D=1024 bf16 Zipf SGD step 127.5 -> 121 us, B=8192, K=64, F=262144, D=4096
// bf16 Zipf 2130 -> 2097 (a third of it from the loads in flight), B=1777, K=50, F=24571, D=1538 bf16 213 -> 209, B=4096,
// K=128, F=65536, D=2304 bf16 1218 -> 1216.
template <typename GT>
__global__ __launch_bounds__(1024) void hier_epilogue_kernel(
    const float *__restrict__ loss_partial, int64_t n_loss_partials, double inv_count, float *__restrict__ loss,
    HotFinalize fin, HotBlockFinalize hfin, unsigned n_hot_blocks, const float *__restrict__ s_final, int64_t rows,
    int64_t ld, int cols, float *__restrict__ colsum_part, int n_parts, float *__restrict__ dbias,
    unsigned n_col_blocks, const float *__restrict__ dv_part, int n_tiles, int64_t n_pairs, float *__restrict__ dvals,
    PairStats stats) {
  __shared__ double red[1024];
  unsigned blk = blockIdx.x;
  if (blk == 0) {
    if (stats.out && threadIdx.x == 0) write_pair_stats(stats);
    if (loss_partial) loss_finalize_block(loss_partial, n_loss_partials, inv_count, loss, red);
    return;
  }
  blk -= 1;
  if (blk < fin.n_blocks) {
    hot_finalize_run<GT>(fin, blk);
    return;
  }
  blk -= fin.n_blocks;
  if (blk < n_hot_blocks) {
    hot_block_finalize_run<GT>(hfin, blk, n_hot_blocks);
    return;
  }
  blk -= n_hot_blocks;
  if (blk < n_col_blocks) {
    if (n_parts < 0) {
      const unsigned across = static_cast<unsigned>((cols + 255) / 256);
      colsum_partial_one(s_final, rows, ld, cols, colsum_part, static_cast<int>(blk % across * 256 + (threadIdx.x & 255)),
                         static_cast<int64_t>(blk / across) * 4 + (threadIdx.x >> 8));
    } else if (n_parts == 0) {
      colsum_whole_block(s_final, rows, ld, cols, dbias, static_cast<int>(blk * kEndCols), reinterpret_cast<float *>(red));
    } else {
      colsum_final_one(colsum_part, n_parts, cols, nullptr, 1.0f, dbias, static_cast<int>(blk * 1024 + threadIdx.x));
    }
    return;
  }
  blk -= n_col_blocks;
  const int64_t stride = (static_cast<int64_t>(gridDim.x) - (blockIdx.x - blk)) * 1024;
  for (int64_t p = static_cast<int64_t>(blk) * 1024 + threadIdx.x; p < n_pairs; p += stride) {
    float acc = 0.f;
    int t = 0;
    for (; t + 8 <= n_tiles; t += 8) {  // eight independent loads in flight
      float x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = dv_part[(t + u) * n_pairs + p];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += x[u];
    }
    for (; t < n_tiles; ++t) acc += dv_part[t * n_pairs + p];
    dvals[p] = acc;
  }
}

}  // namespace flexsae
