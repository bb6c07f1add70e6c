// Latent-major pair list (CSR over latents) construction, plus small utility kernels
// (column sums, fills, casts).
#pragma once

#include "common.hpp"

namespace flexsae {

// ---------------------------------------------------------------------------------
// What comes with a pair list besides begin[] and map[]: counters (`ctrl`) and lists of latents by
// their number of pairs, appended to by the kernels below (the order of a list's entries is that of
// the atomics; nothing that reads the lists depends on it):
//   long latents (more than kListLong pairs): long_list[0 .. ctrl[kLongCount]) and, for the reduction in
//     chunks of kListLong pairs, chunk_begin[i] = chunks of the latents before entry i.  Count and chunks
//     are advanced by one 64-bit atomic, so chunk_begin ascends with i;
//   latents without pairs: ctrl[kEmptyCount] of them;
// and, only for a reduction that works from them (they cost 4 bytes per latent and a second pass over the counts:
// a training step of B=31, K=1, F=576929, D=88 bf16 that reads none of them 60 us with, 54 without):
//   latents without pairs: empty_list[0 .. ctrl[kEmptyCount]);
//   latents with 1, 2, 3-4, 5-8, 9-16, 17-32, 33-64 pairs: cls_list[i][0 .. ctrl[kClassCount + i]), i = 0 .. 6.
// A block of the list kernels appends its latents ordered by their number of pairs, with one atomic per list.
// ---------------------------------------------------------------------------------
constexpr int kClasses = 7;  // class i: more than 2^(i-1), at most 2^i pairs
// (kListed: 1 if the lists by number of pairs are there, so that a reduction asked to work from a pair list without them
// writes nothing instead of following what the workspace held before)
enum { kLongChunks = 0, kLongCount = 1, kEmptyCount = 2, kClassCount = 3, kListed = kClassCount + kClasses, kCtrlWords = 64 };
constexpr uint32_t kListLong = 64;  // a wavefront's worth of pairs
constexpr int kClassSolo = 4;       // from this class on (9 pairs) a latent gets a group of lanes to itself in the reduction

struct PairLists {
  uint32_t *ctrl;         // kCtrlWords words, zero before the list kernels run
  uint32_t *long_list;    // n_pairs / 65 + 1 entries
  uint32_t *chunk_begin;  // n_pairs / 65 + 1 entries, or null: no lists at all
  uint32_t *empty_list;   // F entries, or null: no lists by number of pairs
  uint32_t *cls_list[kClasses];  // min(F, n_pairs / (smallest number of pairs of the class)) + 1 entries
};

constexpr int kListThreads = 1024;  // threads of a block that appends

// Scratch of append_latents, shared by the block.
struct AppendScratch {
  unsigned long long long_at;      // long latents << 32 | their chunks, then the next place
  uint32_t cursor[kListLong + 1];  // latents per number of pairs, then the next place in the list
  uint32_t empty[kListThreads / kWave];  // per wavefront: its latents without pairs, then their first place
};

// class of a latent with 1 .. kListLong pairs
__device__ __forceinline__ int class_of(uint32_t pairs) { return pairs <= 1 ? 0 : 32 - __builtin_clz(pairs - 1); }

// Appends the block's latents to the lists: the thread's are f .. f + n - 1 (n <= PER, n may differ or be zero), latent
// f + i has count[i] pairs.  Run by a whole block of kListThreads; begins with a barrier, leaves sh in use.
template <int PER>
__device__ __forceinline__ void append_latents(const PairLists &ls, int64_t f, int n, const uint32_t (&count)[PER],
                                               AppendScratch &sh) {
  constexpr int kWaves = kListThreads / kWave;
  const int lane = lane_id(), wv = wave_in_block();
  const bool classes = ls.empty_list != nullptr;
  auto long_step = [&](uint32_t c) { return (1ull << 32) | static_cast<unsigned long long>((c + kListLong - 1) / kListLong); };
  for (uint32_t k = threadIdx.x; k <= kListLong; k += kListThreads) sh.cursor[k] = 0u;
  if (threadIdx.x == 0) sh.long_at = 0ull;
  __syncthreads();
  bool any_long = false;
  {
    uint32_t empty = 0;  // of the wavefront (most latents of a sparse batch: counted without an atomic)
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const bool have = i < n;
      empty += static_cast<uint32_t>(__popcll(__ballot(have && count[i] == 0u)));
      if (have && count[i] > kListLong) {
        any_long = true;
        atomicAdd(&sh.long_at, long_step(count[i]));
      } else if (classes && have && count[i] != 0u) {
        atomicAdd(&sh.cursor[count[i]], 1u);
      }
    }
    if (lane == 0) sh.empty[wv] = empty;
  }
  if (classes && blockIdx.x == 0 && threadIdx.x == 0) ls.ctrl[kListed] = 1u;
  const bool places = __syncthreads_or(any_long) != 0 || classes;  // uniform: something to be written
  if (wv == 0) {  // totals of the lists, a place in each, first place of every class
    const uint32_t own = lane < kWaves ? sh.empty[lane] : 0u;
    uint32_t upto = own;  // inclusive prefix over the wavefronts
#pragma unroll
    for (int off = 1; off < kWaves; off <<= 1) {
      const uint32_t y = __shfl_up(upto, off, kWave);
      if (lane >= off) upto += y;
    }
    const uint32_t n_empty = static_cast<uint32_t>(__shfl(static_cast<int>(upto), kWaves - 1, kWave));
    const uint32_t c = static_cast<uint32_t>(lane) + 1;  // class of this lane: 1 .. 64 pairs
    const uint32_t mine = sh.cursor[c];
    uint32_t inc = mine;  // inclusive prefix over the classes 1 .. c
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off, kWave);
      if (lane >= off) inc += y;
    }
    // lane l: the number of latents in list l (0: empty, 1 + i: class i)
    const int hi = 1 << (lane > 0 && lane <= kClasses ? lane - 1 : 0), lo = hi >> 1;
    const uint32_t upto_hi = static_cast<uint32_t>(__shfl(static_cast<int>(inc), hi - 1, kWave));
    const uint32_t upto_lo = static_cast<uint32_t>(__shfl(static_cast<int>(inc), lo > 0 ? lo - 1 : 0, kWave));
    const uint32_t add = lane == 0 ? n_empty : upto_hi - (lo > 0 ? upto_lo : 0u);
    uint32_t at = 0;
    if (lane <= kClasses && add) at = atomicAdd(&ls.ctrl[kEmptyCount + lane], add);
    if (lane == kClasses + 1 && sh.long_at)
      sh.long_at = atomicAdd(reinterpret_cast<unsigned long long *>(ls.ctrl), sh.long_at);
    static_assert(kClassCount == kEmptyCount + 1, "the counters of the lists follow each other");
    const int cls = class_of(c);
    const int below_cls = (1 << cls) >> 1;  // pairs of the classes before
    const uint32_t below = static_cast<uint32_t>(__shfl(static_cast<int>(inc), below_cls > 0 ? below_cls - 1 : 0, kWave));
    const uint32_t base = static_cast<uint32_t>(__shfl(static_cast<int>(at), 1 + cls, kWave));
    sh.cursor[c] = base + (inc - mine - (below_cls > 0 ? below : 0u));
    const uint32_t empty_at = static_cast<uint32_t>(__shfl(static_cast<int>(at), 0, kWave));
    if (lane < kWaves) sh.empty[lane] = empty_at + (upto - own);
  }
  if (!places) return;
  __syncthreads();
  // (the wavefront's empty latents in ascending order: their rows are cleared in the order of the list)
  uint32_t empty_at = sh.empty[wv];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const unsigned long long with = __ballot(i < n && count[i] == 0u);
    empty_at += __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(with >> 32),
                                          __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(with), 0u));
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (i >= n) continue;
    const uint32_t at_f = static_cast<uint32_t>(f + i);
    if (count[i] > kListLong) {
      const unsigned long long at = atomicAdd(&sh.long_at, long_step(count[i]));
      ls.long_list[at >> 32] = at_f;
      ls.chunk_begin[at >> 32] = static_cast<uint32_t>(at);
    } else if (classes && count[i] == 0u) {
      ls.empty_list[empty_at++] = at_f;
    } else if (classes) {
      ls.cls_list[class_of(count[i])][atomicAdd(&sh.cursor[count[i]], 1u)] = at_f;
    }
  }
}

// The lists of a pair list whose begin[] is given (one that was imported or built elsewhere); ctrl zero on entry.
constexpr int kListPer = 2;                           // latents per thread
constexpr int kListLatents = kListPer * kListThreads;  // per block
__global__ __launch_bounds__(kListThreads) void pair_lists_kernel(const uint32_t *__restrict__ begin, int64_t F, PairLists ls) {
  __shared__ AppendScratch sh;
  const int64_t f = (static_cast<int64_t>(blockIdx.x) * kListThreads + threadIdx.x) * kListPer;
  const int n = (F - f) >= kListPer ? kListPer : F > f ? static_cast<int>(F - f) : 0;
  uint32_t count[kListPer];
#pragma unroll
  for (int i = 0; i < kListPer; ++i) count[i] = i < n ? begin[f + i + 1] - begin[f + i] : 0u;
  append_latents(ls, f, n, count, sh);
}

// ---------------------------------------------------------------------------------
// Pair list with one memory atomic per pair, for more latents than the bucketed construction below takes:
// count (keeping each pair's rank in its group) -> exclusive scan -> fill -> sort each group ascending.
// ---------------------------------------------------------------------------------

__global__ void fill_u32_kernel(uint32_t *__restrict__ p, int64_t n, uint32_t value) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    p[i] = value;
}

// Start of a pair-list build with memory atomics: zero the per-latent counters and the control words.
__global__ void csr_init_kernel(uint32_t *__restrict__ counts, int64_t n, uint32_t *__restrict__ ctrl) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    counts[i] = 0u;
  if (blockIdx.x == 0 && threadIdx.x < kCtrlWords) ctrl[threadIdx.x] = 0u;
}

// counts[f] += 1 for every pair, and rank[p] = the value the counter had before: a position
// inside the latent's group that is unique but depends on the order the atomics were served in
// (the groups are sorted afterwards).  Out-of-range indices are flagged and counted as latent 0.
__global__ void csr_count_kernel(const int64_t *__restrict__ indices, int64_t n_pairs, int64_t F,
                                 uint32_t *__restrict__ counts, uint32_t *__restrict__ rank,
                                 int *status_flag) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; p < n_pairs;
       p += stride) {
    int64_t f = indices[p];
    if (static_cast<uint64_t>(f) >= static_cast<uint64_t>(F)) {
      if (status_flag) atomicOr(status_flag, FLEXSAE_FLAG_INDEX_RANGE);
      f = 0;
    }
    rank[p] = atomicAdd(counts + f, 1u);
  }
}

// Exclusive scan of the per-latent counts in two launches.  Every block owns kScanBlockElems
// consecutive latents: csr_scan_sums_kernel writes the block totals, csr_scan_apply_kernel
// adds up the totals of the blocks before it (a few hundred values at most), scans its own
// elements and writes begin[]; the last block writes begin[F].
constexpr int kScanThreads = 256;
constexpr int kScanPerThread = 8;
constexpr int kScanBlockElems = kScanThreads * kScanPerThread;

__device__ __forceinline__ uint32_t block_sum_u32(uint32_t v, uint32_t *smem /*[kScanThreads/64]*/) {
  // all threads receive the block total
  for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  const int wv = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0) smem[wv] = v;
  __syncthreads();
  uint32_t t = 0;
  for (int w = 0; w < kScanThreads / kWave; ++w) t += smem[w];
  return t;
}

__global__ __launch_bounds__(kScanThreads) void csr_scan_sums_kernel(const uint32_t *__restrict__ counts,
                                                                     int64_t F,
                                                                     uint32_t *__restrict__ block_sums) {
  __shared__ uint32_t smem[kScanThreads / kWave];
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kScanBlockElems +
                     static_cast<int64_t>(threadIdx.x) * kScanPerThread;
  uint32_t tsum = 0;
#pragma unroll
  for (int i = 0; i < kScanPerThread; ++i) tsum += (i0 + i < F) ? counts[i0 + i] : 0u;
  const uint32_t tot = block_sum_u32(tsum, smem);
  if (threadIdx.x == 0) block_sums[blockIdx.x] = tot;
}

__global__ __launch_bounds__(kScanThreads) void csr_scan_apply_kernel(uint32_t *__restrict__ begin,
                                                                      int64_t F,
                                                                      const uint32_t *__restrict__ block_sums) {
  __shared__ uint32_t smem[kScanThreads / kWave];
  __shared__ uint32_t wave_tot[kScanThreads / kWave];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid >> 6;
  // offset of this block = sum of the totals of all earlier blocks
  uint32_t part = 0;
  for (uint32_t j = tid; j < blockIdx.x; j += kScanThreads) part += block_sums[j];
  const uint32_t block_off = block_sum_u32(part, smem);

  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kScanBlockElems +
                     static_cast<int64_t>(tid) * kScanPerThread;
  uint32_t x[kScanPerThread];
  uint32_t tsum = 0;
#pragma unroll
  for (int i = 0; i < kScanPerThread; ++i) {
    x[i] = (i0 + i < F) ? begin[i0 + i] : 0u;
    tsum += x[i];
  }
  uint32_t inc = tsum;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t y = __shfl_up(inc, off, kWave);
    if (lane >= off) inc += y;
  }
  if (lane == kWave - 1) wave_tot[wv] = inc;
  __syncthreads();
  uint32_t wave_off = 0;
  for (int w = 0; w < wv; ++w) wave_off += wave_tot[w];
  uint32_t run = block_off + wave_off + (inc - tsum);
#pragma unroll
  for (int i = 0; i < kScanPerThread; ++i) {
    if (i0 + i < F) begin[i0 + i] = run;
    run += x[i];
  }
  if (blockIdx.x == gridDim.x - 1 && tid == kScanThreads - 1) begin[F] = run;
}

// map[begin[f] + rank[p]] = p: every pair goes to its group without any further atomic.
__global__ void csr_fill_kernel(const int64_t *__restrict__ indices, int64_t n_pairs, int64_t F,
                                const uint32_t *__restrict__ begin, const uint32_t *__restrict__ rank,
                                uint32_t *__restrict__ map) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; p < n_pairs;
       p += stride) {
    int64_t f = indices[p];
    if (static_cast<uint64_t>(f) >= static_cast<uint64_t>(F)) f = 0;
    map[begin[f] + rank[p]] = static_cast<uint32_t>(p);
  }
}

// Sort every group ascending so that the list does not depend on the order in which the
// count kernel's atomics happened to be served.  One wavefront per latent: groups of up to
// 64 pairs are rank-sorted in registers (pair ids are distinct); longer ones are appended
// to long_list for csr_sort_long_kernel.
__global__ __launch_bounds__(256) void csr_sort_short_kernel(const uint32_t *__restrict__ begin,
                                                             uint32_t *__restrict__ map, int64_t F,
                                                             uint32_t *__restrict__ long_count,
                                                             uint32_t *__restrict__ long_list) {
  const int lane = lane_id();
  const int64_t f = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + wave_in_block();
  if (f >= F) return;
  const uint32_t s0 = begin[f];
  const uint32_t n = begin[f + 1] - s0;
  if (n <= 1) return;
  if (n > static_cast<uint32_t>(kWave)) {
    if (lane == 0) long_list[atomicAdd(long_count, 1u)] = static_cast<uint32_t>(f);
    return;
  }
  const bool have = static_cast<uint32_t>(lane) < n;
  const uint32_t x = have ? map[s0 + lane] : 0xffffffffu;
  uint32_t rank = 0;
  for (uint32_t j = 0; j < n; ++j) {
    const uint32_t y = static_cast<uint32_t>(bcast_i32(static_cast<int>(x), static_cast<int>(j)));
    rank += (y < x) ? 1u : 0u;
  }
  if (have) map[s0 + rank] = x;  // every lane read its element before any lane writes
}

// Bitonic network in which every comparator points the same way (first sub-step of each merge
// mirrors, the rest are plain strides), so a length that is not a power of two is handled by
// skipping comparators whose partner lies beyond the end.  Run by one whole block on a[0..n).
template <typename Ptr>
__device__ __forceinline__ void block_bitonic_sort(Ptr a, uint32_t n) {
  uint32_t np2 = 1;
  while (np2 < n) np2 <<= 1;
  for (uint32_t k = 2; k <= np2; k <<= 1) {
    // mirrored sub-step: inside each block of k, position i pairs with (k-1-i)
    for (uint32_t t = threadIdx.x; t < np2 / 2; t += blockDim.x) {
      const uint32_t blk = t / (k / 2), i = t % (k / 2);
      const uint32_t lo = blk * k + i, hi = blk * k + (k - 1 - i);
      if (hi < n) {
        const uint32_t x = a[lo], y = a[hi];
        if (x > y) {
          a[lo] = y;
          a[hi] = x;
        }
      }
    }
    __syncthreads();
    for (uint32_t j = k / 4; j > 0; j >>= 1) {
      for (uint32_t t = threadIdx.x; t < np2 / 2; t += blockDim.x) {
        const uint32_t lo = (t / j) * (2 * j) + (t % j), hi = lo + j;
        if (hi < n) {
          const uint32_t x = a[lo], y = a[hi];
          if (x > y) {
            a[lo] = y;
            a[hi] = x;
          }
        }
      }
      __syncthreads();
    }
  }
}

// Long groups (more than 64 pairs): one block per group, striding over the list.  Groups of up
// to kSortLdsElems pairs are sorted in LDS, longer ones in place in global memory.
// A latent that is in a large share of the rows (thousands of pairs) is not compared at all: a
// pair id is row * K + step, so counting the group's pairs per row and scanning the counts places
// every pair (a counting sort over the rows, O(pairs + rows) instead of the network's
// O(pairs log^2 pairs)); pairs of the same row, if a row holds the latent more than once, are
// ranked among themselves afterwards.  Taken when the rows fit the LDS counters and the network
// would cost several times more.
constexpr uint32_t kSortLdsElems = 8192;
constexpr uint32_t kSortRowsMax = 8192;  // rows (B) the counting sort has LDS counters for
// buf + rowcnt + wave_tot come to 65 600 bytes of LDS per block: more than the 64 KiB of earlier gfx9
// parts, within the 160 KiB a workgroup may use on gfx950 (the only target of this library)
static_assert((kSortLdsElems + kSortRowsMax + 1024 / kWave) * 4 <= 160 * 1024, "LDS of csr_sort_long_kernel");
__global__ __launch_bounds__(1024) void csr_sort_long_kernel(const uint32_t *__restrict__ begin,
                                                            uint32_t *__restrict__ map,
                                                            const uint32_t *__restrict__ long_count,
                                                            const uint32_t *__restrict__ long_list,
                                                            uint32_t n_rows, uint32_t K) {
  __shared__ uint32_t buf[kSortLdsElems];  // the group (network), or its pairs grouped by row (counting sort)
  __shared__ uint32_t rowcnt[kSortRowsMax];
  __shared__ uint32_t wave_tot[1024 / kWave];
  const uint32_t n_long = *long_count;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid >> 6;
  for (uint32_t w = blockIdx.x; w < n_long; w += gridDim.x) {
    const uint32_t f = long_list[w];
    const uint32_t base = begin[f];
    uint32_t *a = map + base;
    const uint32_t n = begin[f + 1] - base;
    if (n <= kSortLdsElems) {
      uint32_t lg = 1;
      while ((1u << lg) < n) ++lg;
      // network: about n/2 * lg*(lg+1)/2 comparators; counting: a few passes over n pairs and n_rows counters
      const bool by_rows = n_rows <= kSortRowsMax && K > 0 &&
                           static_cast<uint64_t>(n) * lg * (lg + 1) > 4ull * (static_cast<uint64_t>(n) + n_rows);
      if (by_rows) {  // uniform over the block
        for (uint32_t r = tid; r < n_rows; r += blockDim.x) rowcnt[r] = 0u;
        __syncthreads();
        for (uint32_t i = tid; i < n; i += blockDim.x) atomicAdd(&rowcnt[a[i] / K], 1u);
        __syncthreads();
        // exclusive scan of rowcnt[0..n_rows): every thread owns eight consecutive counters
        {
          constexpr uint32_t PER = kSortRowsMax / 1024;
          uint32_t x[PER], tsum = 0;
#pragma unroll
          for (uint32_t i = 0; i < PER; ++i) {
            const uint32_t r = static_cast<uint32_t>(tid) * PER + i;
            x[i] = r < n_rows ? rowcnt[r] : 0u;
            tsum += x[i];
          }
          uint32_t inc = tsum;
#pragma unroll
          for (int off = 1; off < kWave; off <<= 1) {
            const uint32_t y = __shfl_up(inc, off, kWave);
            if (lane >= off) inc += y;
          }
          if (lane == kWave - 1) wave_tot[wv] = inc;
          __syncthreads();
          uint32_t run = inc - tsum;
          for (int q = 0; q < wv; ++q) run += wave_tot[q];
#pragma unroll
          for (uint32_t i = 0; i < PER; ++i) {
            const uint32_t r = static_cast<uint32_t>(tid) * PER + i;
            if (r < n_rows) rowcnt[r] = run;
            run += x[i];
          }
          __syncthreads();
        }
        // placement by row; the atomics leave rowcnt[r] at the end of row r's pairs
        for (uint32_t i = tid; i < n; i += blockDim.x) {
          const uint32_t id = a[i];
          buf[atomicAdd(&rowcnt[id / K], 1u)] = id;
        }
        __syncthreads();
        // pairs of one row are in the order of the atomics: rank them among themselves on the way out
        for (uint32_t i = tid; i < n; i += blockDim.x) {
          const uint32_t id = buf[i], r = id / K;
          const uint32_t s0 = r ? rowcnt[r - 1] : 0u, s1 = rowcnt[r];
          uint32_t rank = 0;
          for (uint32_t j = s0; j < s1; ++j) rank += (buf[j] < id) ? 1u : 0u;
          a[s0 + rank] = id;
        }
        __syncthreads();
        continue;
      }
      for (uint32_t i = tid; i < n; i += blockDim.x) buf[i] = a[i];
      __syncthreads();
      block_bitonic_sort(buf, n);
      for (uint32_t i = tid; i < n; i += blockDim.x) a[i] = buf[i];
      __syncthreads();
    } else {
      block_bitonic_sort(a, n);  // ends with a barrier
    }
  }
}

// ---------------------------------------------------------------------------------
// Bucketed construction (the default), two launches.  The latents are cut into buckets of 2^shift
// consecutive ids, sized so that a bucket holds a few thousand pairs.
//   csr_chunk_sort_kernel   one block per chunk of consecutive pairs: the chunk's pairs ordered by bucket, ties
//                           by pair id, and the first place of every bucket in it (table[bucket][chunk]).
//   csr_bucket_sort_kernel  one block per bucket: collects the bucket's pieces from all chunks.  The sum
//                           over the chunks of the bucket's first place is the number of pairs in earlier
//                           buckets, so no scan over the table is needed in between.  Per-latent counts
//                           -> begin[], the lists, and map[] ascending inside every latent.
// Bound by latency (a few dependent passes over a megabyte) and by launches, which cost 4-5 us each in a
// busy stream; where frequent latents share a bucket, by the instructions of that bucket's one block.
// ---------------------------------------------------------------------------------
constexpr int kChunkThreads = 256;
constexpr int kChunkWaves = kChunkThreads / kWave;
constexpr int kBucketMaxBuckets = 8192;  // LDS cursors of the chunk kernel: 4 bytes per wavefront and bucket
constexpr int kSortThreads = kListThreads;
constexpr int kSortMaxShift = 12;
constexpr int kSortMaxLatents = 1 << kSortMaxShift;  // latents per bucket at most
constexpr int kSortCap = 4096;                       // pairs of a bucket that its block keeps in registers
constexpr int kSortChunks = 2048;                    // chunks at most
constexpr int kRunLatents = 512;                     // latents of a larger bucket that are placed together
static_assert((kBucketMaxBuckets * kChunkWaves + kChunkWaves) * 4 <= 160 * 1024, "LDS of csr_chunk_sort_kernel");
constexpr int64_t kBucketBlocks = 512;  // blocks of the bucket kernel on the chip at once (77 KB of LDS: two per compute unit)

// A pair inside its chunk is one word: latent within its bucket << pack_shift | place in the chunk.
inline int csr_pack_shift(int shift) { return 32 - (shift > 11 ? shift : 11); }

// Chunk blockIdx.x.  Dynamic LDS: (n_buckets rounded up to four + 1) * kChunkWaves words.  n_bits: bits of a bucket number.
__device__ __forceinline__ void chunk_sort_block(
    const int64_t *__restrict__ indices, int64_t n_pairs, int64_t F, int shift, int pack_shift, uint32_t n_buckets, int n_bits,
    int64_t chunk, uint32_t n_chunks, uint32_t *__restrict__ table, uint32_t *__restrict__ tmp,
    uint32_t *__restrict__ ctrl, int *status_flag) {
  extern __shared__ __align__(16) uint32_t chunk_lds[];
  using four_t = vec_t<uint32_t, 4>;
  const uint32_t n_cursors = (n_buckets + 3u) & ~3u;
  uint32_t *const cursor = chunk_lds;                            // [wavefront][bucket]
  uint32_t *const wave_tot = chunk_lds + kChunkWaves * n_cursors;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = wave_in_block();
  if (blockIdx.x == 0 && tid < kCtrlWords) ctrl[tid] = 0u;
  for (uint32_t q = tid; q < kChunkWaves * n_cursors / 4; q += kChunkThreads) reinterpret_cast<four_t *>(cursor)[q] = four_t{};
  __syncthreads();
  const int64_t p0 = static_cast<int64_t>(blockIdx.x) * chunk;
  const int64_t n = (n_pairs - p0) < chunk ? (n_pairs - p0) : chunk;
  // every wavefront owns a run of the chunk (chunk is a multiple of kChunkThreads)
  const int64_t run = chunk / kChunkWaves;
  const int64_t r0 = wv * run, r1 = (r0 + run) < n ? (r0 + run) : n;
  constexpr int U = 8;  // rounds of 64 pairs whose loads are in flight together
  auto load = [&](int64_t at, int64_t(&f)[U], bool flag) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t i = at + u * kWave + lane;
      f[u] = i < r1 ? indices[p0 + i] : 0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (static_cast<uint64_t>(f[u]) >= static_cast<uint64_t>(F)) {
        if (flag && status_flag) atomicOr(status_flag, FLEXSAE_FLAG_INDEX_RANGE);
        f[u] = 0;
      }
  };
  uint32_t *const mine = cursor + wv * n_cursors;
  for (int64_t at = r0; at < r1; at += U * kWave) {
    int64_t f[U];
    load(at, f, true);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (at + u * kWave + lane < r1) atomicAdd(&mine[f[u] >> shift], 1u);
  }
  __syncthreads();
  // exclusive scan over (bucket, wavefront), four buckets per thread and round
  uint32_t earlier = 0;  // pairs of the buckets of earlier rounds
  for (uint32_t q0 = 0; q0 < n_buckets; q0 += 4 * kChunkThreads) {
    const uint32_t q = q0 + 4 * tid;
    four_t c[kChunkWaves];
    uint32_t sum = 0;
#pragma unroll
    for (int w = 0; w < kChunkWaves; ++w) {
      c[w] = four_t{};
      if (q < n_buckets) c[w] = *reinterpret_cast<const four_t *>(cursor + w * n_cursors + q);
      sum += c[w][0] + c[w][1] + c[w][2] + c[w][3];
    }
    uint32_t inc = sum;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off, kWave);
      if (lane >= off) inc += y;
    }
    if (lane == kWave - 1) wave_tot[wv] = inc;
    __syncthreads();
    uint32_t at = earlier + inc - sum;
#pragma unroll
    for (int w = 0; w < kChunkWaves; ++w) {
      if (w < wv) at += wave_tot[w];
      earlier += wave_tot[w];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (q + i < n_buckets) table[static_cast<size_t>(q + i) * n_chunks + blockIdx.x] = at;
#pragma unroll
      for (int w = 0; w < kChunkWaves; ++w) {
        const uint32_t mine_c = c[w][i];
        c[w][i] = at;
        at += mine_c;
      }
    }
    if (q < n_buckets) {
#pragma unroll
      for (int w = 0; w < kChunkWaves; ++w) *reinterpret_cast<four_t *>(cursor + w * n_cursors + q) = c[w];
    }
    __syncthreads();
  }
  if (tid == 0) table[static_cast<size_t>(n_buckets) * n_chunks + blockIdx.x] = static_cast<uint32_t>(n);
  const int64_t mask = (static_cast<int64_t>(1) << shift) - 1;
  for (int64_t at = r0; at < r1; at += U * kWave) {
    int64_t f[U];
    load(at, f, false);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t i = at + u * kWave + lane;
      const bool have = i < r1;
      const uint32_t q = static_cast<uint32_t>(f[u] >> shift);
      // the lanes with the same bucket
      unsigned long long same = __ballot(have);
      for (int b = 0; b < n_bits; ++b) {
        const unsigned long long ones = __ballot((q >> b) & 1u);
        same &= ((q >> b) & 1u) ? ones : ~ones;
      }
      const uint32_t rank = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(same >> 32),
                                                      __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(same), 0u));
      if (have) {
        const uint32_t place = mine[q] + rank;
        tmp[p0 + place] = (static_cast<uint32_t>(f[u] & mask) << pack_shift) | static_cast<uint32_t>(i);
        // (LDS accesses of a wavefront are served in order: all lanes have read the cursor)
        if (rank == 0) mine[q] = place + static_cast<uint32_t>(__popcll(same));
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

__global__ __launch_bounds__(kChunkThreads) void csr_chunk_sort_kernel(
    const int64_t *__restrict__ indices, int64_t n_pairs, int64_t F, int shift, int pack_shift, uint32_t n_buckets, int n_bits,
    int64_t chunk, uint32_t n_chunks, uint32_t *__restrict__ table, uint32_t *__restrict__ tmp,
    uint32_t *__restrict__ ctrl, int *status_flag) {
  chunk_sort_block(indices, n_pairs, F, shift, pack_shift, n_buckets, n_bits, chunk, n_chunks, table, tmp, ctrl, status_flag);
}

// Records of the pairs in the order of the list: out[place] = (batch row, val as fp32 bits), what a backward reads per pair,
// contiguous per latent instead of scattered over vals.  A pair whose index lies outside [0, F) gets a val of zero, as in the
// forward (the list files it under latent 0, so only that latent's pairs are looked up in indices).
struct PairRecords {
  const void *vals;
  const int64_t *indices;
  vec_t<uint32_t, 2> *out;
  int vals_dtype;
  uint32_t K;
};

// counter[at] += 1 for every lane with `have`, in the LDS.  The lanes that agree with the first one add up
// beforehand (ROUNDS times over): adds to one address are served one lane after the other, and a frequent latent
// is most of its bucket.
template <int ROUNDS>
__device__ __forceinline__ void count_in_lds(uint32_t *counter, uint32_t at, bool have) {
#pragma unroll
  for (int round = 0; round < ROUNDS; ++round) {
    const unsigned long long left = __ballot(have);
    if (left == 0) return;  // uniform
    const int leader = __builtin_ctzll(left);
    const uint32_t key = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(at), leader));
    const bool same = have && at == key;
    const unsigned long long with = __ballot(same);
    if (lane_id() == leader) atomicAdd(&counter[key], static_cast<uint32_t>(__popcll(with)));
    have = have && !same;
  }
  if (have) atomicAdd(&counter[at], 1u);
}

// One block per bucket.  hslot: a second copy of slot[] (null: none).  solo_bit: marks in both the only pair of
// its latent (0: no marks).  RECORDS: writes the pairs' records (rec) instead of slot[] and hslot[].
// The pieces of a bucket, one from every chunk, hold its pairs in pair order: pair i of the bucket is found by a search
// for its chunk in first[].
//   Up to kSortCap pairs: four to a thread, kept in registers.  Groups of up to kListLong pairs are gathered in the LDS in
//     any order, and every pair counts the smaller ids of its group.  Pairs of longer groups (frequent latents) are placed
//     by wavefront: a round of a wavefront is 64 consecutive pairs, and goes behind the rounds before it.
//   More pairs (frequent latents among them): every wavefront walks a run of the bucket's pairs twice, kRunLatents
//     latents at a time; first it counts its pairs of every latent, then it places them behind those of the wavefronts
//     before it.  Nothing is searched for within a piece of 64 pairs or more.  The blocks of a bucket (gridDim.y) share
//     the batches of latents, where there is room for more blocks than buckets.  What bounds it are the instructions of
//     one compute unit (and a line per pair of the stores, where every pair goes to another group).
// Pair list, us; in brackets with every pair searched for, separate passes for long and short groups and the latter in
// batches that fit the LDS: 524288 pairs of 65536 latents, uniform: 21 (24); 262144 of 262144, skewed, latents in any
// order: 75 (96), latents by frequency: 298 (3336), half of the pairs on the first 32 latents: 144 (317); 64 latents in
// every one of 16384 rows: 1329 (2584).
// WAVES: wavefronts per SIMD that its registers leave room for: eight, two blocks per compute unit, spill 13 (with records 30)
// registers; four do not, where there are no more buckets than compute units (with records, us: 26.9 -> 18.8 for 524288 pairs of
// 65536 latents, 13.7 -> 9.5 for 2048 of 4096, 19.5 -> 10.7 for 4710 of 262144; without 11.1 -> 10.2 for the second and the same
// for the first).
template <bool RECORDS, int WAVES>
__global__ __launch_bounds__(kSortThreads, WAVES) void csr_bucket_sort_kernel(
    const uint32_t *__restrict__ tmp, const uint32_t *__restrict__ table, uint32_t n_chunks, int64_t chunk, int shift,
    int pack_shift, int64_t F, uint32_t *__restrict__ begin, uint32_t *__restrict__ map, uint32_t *__restrict__ slot,
    uint32_t *__restrict__ hslot, uint32_t solo_bit, PairLists ls, PairRecords rec) {
  constexpr int kWaves = kSortThreads / kWave;
  constexpr int PER = kSortMaxLatents / kSortThreads;  // latents per thread
  constexpr int kPairs = kSortCap / kSortThreads;      // pairs per thread
  constexpr int CPER = kSortChunks / kSortThreads;     // chunks per thread
  __shared__ __align__(16) uint32_t cnt[kSortMaxLatents + 4];  // pairs per latent, then their exclusive scan
  __shared__ uint8_t lid[kSortMaxLatents];        // number of a frequent latent
  // up to kSortCap pairs: first half cursors [frequent latent][round], then the pair ids of short groups; second half
  // the next place of every latent.  More: cursors [wavefront][latent of the batch]
  __shared__ __align__(16) uint32_t ids[kWaves * kRunLatents];
  __shared__ uint32_t first[kSortChunks + 1];     // first pair of each chunk's piece; the number of pairs beyond the last
  __shared__ uint32_t from[kSortChunks];          // what to add to the number of a pair of that piece for its place in tmp[]
  __shared__ uint32_t wave_tot[kWaves], wave_tot2[kWaves];
  __shared__ unsigned long long agree[kWaves][kWave];
  __shared__ uint32_t n_long_s;
  __shared__ AppendScratch sh;
  static_assert(kWaves * kRunLatents >= kSortCap + kSortMaxLatents, "ids and next places");
  constexpr uint32_t kRounds = kSortCap / kWave;
  static_assert(kRounds == kWave && (kSortCap / (kListLong + 1)) * kRounds <= kSortCap && kSortCap / (kListLong + 1) <= 64,
                "a lane per round, cursors of all frequent latents, six bits for the number of one");
  uint32_t *const next_place = ids + kSortCap;
  using latents_t = vec_t<uint32_t, PER>;
  const int tid = threadIdx.x, lane = lane_id(), wv = wave_in_block();
  const uint32_t q = blockIdx.x;
  const uint32_t lpb = 1u << shift;
  const int64_t f0 = static_cast<int64_t>(q) << shift;
  const uint32_t nlat = (F - f0) < static_cast<int64_t>(lpb) ? static_cast<uint32_t>(F - f0) : lpb;
  const uint32_t place_mask = (1u << pack_shift) - 1u;
  const uint32_t chunk_w = static_cast<uint32_t>(chunk);
  const uint32_t my_k = static_cast<uint32_t>(tid) * PER;

  // base = pairs in earlier buckets, n = pairs in this one; the table of the pieces
  uint32_t base = 0, n = 0;
  {
    const uint32_t *const row0 = table + static_cast<size_t>(q) * n_chunks;
    uint32_t at[CPER], len[CPER], s0 = 0, s1 = 0;
#pragma unroll
    for (int j = 0; j < CPER; ++j) {
      const uint32_t c = static_cast<uint32_t>(tid) * CPER + j;
      at[j] = len[j] = 0;
      if (c < n_chunks) {
        at[j] = row0[c];
        len[j] = row0[n_chunks + c] - at[j];
      }
      s0 += at[j];
      s1 += len[j];
    }
    uint32_t inc = s1;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off, kWave);
      if (lane >= off) inc += y;
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) s0 += static_cast<uint32_t>(__shfl_xor(static_cast<int>(s0), off, kWave));
    if (lane == kWave - 1) {
      wave_tot[wv] = inc;
      wave_tot2[wv] = s0;
    }
    for (uint32_t k = my_k; k <= lpb; k += kSortThreads * PER) *reinterpret_cast<latents_t *>(cnt + k) = latents_t{};
    agree[wv][lane] = 0ull;
    if (tid == 0) n_long_s = 0u;
    __syncthreads();
    uint32_t start = inc - s1;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      base += wave_tot2[w];
      if (w < wv) start += wave_tot[w];
      n += wave_tot[w];
    }
#pragma unroll
    for (int j = 0; j < CPER; ++j) {
      const uint32_t c = static_cast<uint32_t>(tid) * CPER + j;
      first[c] = start;
      from[c] = c * chunk_w + at[j] - start;  // (modulo 2^32, as the sum with a pair's number: fewer than 2^32 pairs)
      start += len[j];
    }
    if (tid == 0) first[kSortChunks] = n;
    __syncthreads();
  }
  uint32_t probes = 1;  // a power of two, at least the number of chunks
  while (probes < n_chunks) probes <<= 1;
  // largest chunk with first[chunk] <= i (an empty piece repeats its successor's place)
  auto chunk_of = [&](uint32_t i) {
    uint32_t c = 0;
    for (uint32_t step = probes >> 1; step > 0; step >>= 1) c += first[c + step] <= i ? step : 0u;
    return c;
  };
  // the bits of a pair's val, where records are written
  auto val_bits = [&](uint32_t id) {
    uint32_t bits = 0;
    if constexpr (RECORDS) bits = load_scalar_bits(rec.vals, rec.vals_dtype, id);
    return bits;
  };
  auto put = [&](uint32_t place, uint32_t key, uint32_t id, uint32_t mark, uint32_t bits) {
    map[place] = id;
    if constexpr (RECORDS) {
      float v = scalar_from_bits(bits, rec.vals_dtype);
      if (f0 + key == 0 && static_cast<uint64_t>(rec.indices[id]) >= static_cast<uint64_t>(F)) v = 0.f;
      rec.out[place] = vec_t<uint32_t, 2>{id / rec.K, __float_as_uint(v)};
    } else {
      if (slot) slot[id] = place | mark;
      if (hslot) hslot[id] = place | mark;
    }
  };
  // the lanes (of those with `have`, at least one) that agree with this one in the low `bits` bits of key: the first
  // lane's followers by a ballot (a frequent latent), the others by their marks in the LDS under the key's low six bits
  // and a ballot for each bit above.  Seven vector operations for each of nine bits cost the walk below a fifth more.
  auto agreeing = [&](uint32_t key, bool have, uint32_t bits) {
    const int leader = __builtin_ctzll(__ballot(have));
    const bool led = have && key == static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(key), leader));
    unsigned long long same = __ballot(led);
    if (have && !led) {
      // (LDS accesses of a wavefront are served in order)
      unsigned long long *const mark = &agree[wv][key & (kWave - 1)];
      atomicOr(mark, 1ull << lane);
      same = *mark;
      *mark = 0ull;
    }
    for (uint32_t b = 6; b < bits; ++b) {
      const unsigned long long ones = __ballot((key >> b) & 1u);
      if (!led) same &= ((key >> b) & 1u) ? ones : ~ones;
    }
    return same;
  };
  auto lanes_before = [](unsigned long long with) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(with >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(with), 0u));
  };

  if (n <= static_cast<uint32_t>(kSortCap)) {  // uniform
    if (blockIdx.y != 0) return;
    uint32_t x[PER] = {};  // pairs of the thread's latents
    const int my_n = nlat >= my_k + PER ? PER : nlat > my_k ? static_cast<int>(nlat - my_k) : 0;
    if (n == 0) {
      for (uint32_t k = tid; k < nlat; k += kSortThreads) begin[f0 + k] = base;
      if (tid == 0 && q == gridDim.x - 1) begin[F] = base;
      if (ls.chunk_begin) append_latents(ls, f0 + my_k, my_n, x, sh);
      return;
    }
    uint32_t key[kPairs], id[kPairs], bits_of[kPairs];
    const int rounds = static_cast<int>((n + kSortThreads - 1) / kSortThreads);
    {
      uint32_t c[kPairs], v[kPairs];
#pragma unroll
      for (int u = 0; u < kPairs; ++u) {
        if (u < rounds) {  // uniform
          const uint32_t i = static_cast<uint32_t>(tid) + u * kSortThreads;
          const uint32_t at = i < n ? i : 0u;
          c[u] = chunk_of(at);
          v[u] = tmp[from[c[u]] + at];
        }
      }
#pragma unroll
      for (int u = 0; u < kPairs; ++u) {
        key[u] = id[u] = bits_of[u] = 0;
        if (u < rounds) {
          key[u] = v[u] >> pack_shift;
          id[u] = c[u] * chunk_w + (v[u] & place_mask);
          bits_of[u] = val_bits(id[u]);
          count_in_lds<2>(cnt, key[u], static_cast<uint32_t>(tid) + u * kSortThreads < n);
        }
      }
    }
    __syncthreads();
    {  // exclusive scan over the latents
      uint32_t xs = 0;
      latents_t own = {};
      if (my_k < lpb) own = *reinterpret_cast<const latents_t *>(cnt + my_k);
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        x[i] = my_k + i < lpb ? own[i] : 0u;
        if (x[i] > kListLong) lid[my_k + i] = static_cast<uint8_t>(atomicAdd(&n_long_s, 1u));
        xs += x[i];
      }
      uint32_t xi = xs;
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t y = __shfl_up(xi, off, kWave);
        if (lane >= off) xi += y;
      }
      if (lane == kWave - 1) wave_tot[wv] = xi;
      __syncthreads();
      uint32_t run = xi - xs;
#pragma unroll
      for (int w = 0; w < kWaves; ++w)
        if (w < wv) run += wave_tot[w];
      latents_t at;
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        at[i] = run;
        run += x[i];
      }
      if (my_k <= lpb) *reinterpret_cast<latents_t *>(cnt + my_k) = at;  // (n beyond the last latent)
      if (my_k < lpb) *reinterpret_cast<latents_t *>(next_place + my_k) = at;
      if (lpb == kSortMaxLatents && tid == 0) cnt[lpb] = n;
    }
    __syncthreads();
    for (uint32_t k = tid; k < nlat; k += kSortThreads) begin[f0 + k] = base + cnt[k];
    const uint32_t n_long = n_long_s;
    if (n_long != 0) {  // uniform
      uint32_t bits = 0;
      while ((1u << bits) < n_long) ++bits;
      for (uint32_t l = tid; l < n_long * kRounds; l += kSortThreads) ids[l] = 0u;
      __syncthreads();
      auto is_long = [&](int u) {
        return static_cast<uint32_t>(tid) + u * kSortThreads < n && cnt[key[u] + 1] - cnt[key[u]] > kListLong;
      };
#pragma unroll
      for (int u = 0; u < kPairs; ++u)
        if (u < rounds) {
          const bool have = is_long(u);
          count_in_lds<2>(ids, have ? lid[key[u]] * kRounds + u * kWaves + wv : 0u, have);
        }
      __syncthreads();
      for (uint32_t l = wv; l < n_long; l += kWaves) {  // a wavefront per latent, a lane per round
        const uint32_t own = ids[l * kRounds + lane];
        uint32_t inc = own;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
          const uint32_t y = __shfl_up(inc, off, kWave);
          if (lane >= off) inc += y;
        }
        ids[l * kRounds + lane] = inc - own;
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < kPairs; ++u)
        if (u < rounds) {
          const bool have = is_long(u);
          if (!__any(have)) continue;
          const uint32_t l = have ? lid[key[u]] : 0u;
          const unsigned long long same = agreeing(l, have, bits);
          if (have) put(base + cnt[key[u]] + ids[l * kRounds + u * kWaves + wv] + lanes_before(same), key[u], id[u], 0u, bits_of[u]);
        }
      __syncthreads();
    }
    // short groups: placed in the order of the atomics, then ranked
#pragma unroll
    for (int u = 0; u < kPairs; ++u)
      if (static_cast<uint32_t>(tid) + u * kSortThreads < n && cnt[key[u] + 1] - cnt[key[u]] <= kListLong)
        ids[atomicAdd(&next_place[key[u]], 1u)] = id[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPairs; ++u) {
      if (static_cast<uint32_t>(tid) + u * kSortThreads >= n) continue;
      const uint32_t start = cnt[key[u]], len = cnt[key[u] + 1] - start;
      if (len > kListLong) continue;
      const uint32_t *const group = ids + start;
      uint32_t rank = 0, j = 0;
      for (; j + 8 <= len; j += 8) {
        uint32_t y[8];
#pragma unroll
        for (int w = 0; w < 8; ++w) y[w] = group[j + w];
#pragma unroll
        for (int w = 0; w < 8; ++w) rank += (y[w] < id[u]) ? 1u : 0u;
      }
      for (; j < len; ++j) rank += (group[j] < id[u]) ? 1u : 0u;
      put(base + start + rank, key[u], id[u], len == 1 ? solo_bit : 0u, bits_of[u]);
    }
    if (ls.chunk_begin) append_latents(ls, f0 + my_k, my_n, x, sh);
  } else {
    uint32_t run = (n + kWaves - 1) / kWaves;
    run = (run + kWave - 1) / kWave * kWave;
    const uint32_t r0 = wv * run, r1 = (r0 + run) < n ? (r0 + run) : n;
    // body(key, id, valid, fetch(key, id, valid)) for the wavefront's pairs in order, 64 at a time; what is fetched for several
    // of them is in flight together
    auto walk = [&](auto fetch, auto body) {
      constexpr int U = 8;
      uint32_t hi = 0, off = 0, id0 = 0;  // pairs from the last one looked at to hi lie in one piece
      for (uint32_t i0 = r0; i0 < r1; i0 += U * kWave) {
        uint32_t v[U], idb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t at = i0 + u * kWave;  // uniform
          v[u] = idb[u] = 0;
          if (at >= r1) continue;
          const uint32_t i = at + lane < n ? at + lane : n - 1;
          if (at + kWave <= hi) {
            v[u] = tmp[off + i];
            idb[u] = id0;
          } else {
            const uint32_t c = chunk_of(i);
            v[u] = tmp[from[c] + i];
            idb[u] = c * chunk_w;
            const uint32_t last = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(c), kWave - 1));
            hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(first[last + 1])));
            off = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(from[last])));
            id0 = last * chunk_w;
          }
        }
        uint32_t x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          idb[u] += v[u] & place_mask;
          x[u] = fetch(v[u] >> pack_shift, idb[u], i0 + u * kWave + lane < r1);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t at = i0 + u * kWave;
          if (at < r1) body(v[u] >> pack_shift, idb[u], at + lane < r1, x[u]);
        }
      }
    };
    uint32_t *const mine = ids + wv * kRunLatents;
    const uint32_t batch = lpb < static_cast<uint32_t>(kRunLatents) ? lpb : static_cast<uint32_t>(kRunLatents);
    uint32_t bits = 0;
    while ((1u << bits) < batch) ++bits;
    for (uint32_t k0 = blockIdx.y * batch; k0 < nlat; k0 += gridDim.y * batch) {  // uniform
      for (uint32_t l = tid; l < kWaves * kRunLatents; l += kSortThreads) ids[l] = 0u;
      __syncthreads();
      uint32_t before = 0;  // this lane's pairs of the latents before the batch
      walk([](uint32_t, uint32_t, bool) { return 0u; }, [&](uint32_t key, uint32_t, bool valid, uint32_t) {
        before += valid && key < k0 ? 1u : 0u;
        count_in_lds<1>(mine, key - k0, valid && key - k0 < batch);
      });
#pragma unroll
      for (int off = kWave / 2; off > 0; off >>= 1) before += static_cast<uint32_t>(__shfl_xor(static_cast<int>(before), off, kWave));
      if (lane == 0) wave_tot2[wv] = before;
      __syncthreads();
      uint32_t total[1] = {0};  // of latent k0 + tid
      if (static_cast<uint32_t>(tid) < batch) {
        uint32_t c[kWaves];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) c[w] = ids[w * kRunLatents + tid];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          ids[w * kRunLatents + tid] = total[0];
          total[0] += c[w];
        }
      }
      uint32_t inc = total[0];
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t y = __shfl_up(inc, off, kWave);
        if (lane >= off) inc += y;
      }
      if (lane == kWave - 1) wave_tot[wv] = inc;
      __syncthreads();
      uint32_t start = inc - total[0];
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        start += wave_tot2[w];
        if (w < wv) start += wave_tot[w];
      }
      const bool mine_too = static_cast<uint32_t>(tid) < batch && k0 + tid < nlat;
      if (static_cast<uint32_t>(tid) < batch) cnt[tid] = start;
      if (tid == static_cast<int>(batch) - 1) cnt[batch] = start + total[0];
      if (mine_too) begin[f0 + k0 + tid] = base + start;
      if (ls.chunk_begin) append_latents(ls, f0 + k0 + tid, mine_too ? 1 : 0, total, sh);
      __syncthreads();
      walk([&](uint32_t key, uint32_t id, bool valid) { return valid && key - k0 < batch ? val_bits(id) : 0u; },
           [&](uint32_t key, uint32_t id, bool valid, uint32_t bits_of) {
        const uint32_t l = key - k0;
        const bool have = valid && l < batch;
        if (!__any(have)) return;
        const unsigned long long same = agreeing(l, have, bits);
        const uint32_t rank = lanes_before(same);
        if (have) {
          const uint32_t place = mine[l] + rank, at = cnt[l];
          put(base + at + place, key, id, cnt[l + 1] - at == 1u ? solo_bit : 0u, bits_of);
          // (LDS accesses of a wavefront are served in order: all lanes have read the cursor)
          if (rank == 0) mine[l] = place + static_cast<uint32_t>(__popcll(same));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      });
      __syncthreads();
    }
  }
  if (tid == 0 && blockIdx.y == 0 && q == gridDim.x - 1) begin[F] = base + n;
}

__global__ void copy_u32_kernel(uint32_t *__restrict__ dst, const uint32_t *__restrict__ src, int64_t n) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    dst[i] = src[i];
}

// slot[map[s]] = s: position of every pair in the latent-major list (and a second copy in hslot).
__global__ void csr_inverse_kernel(const uint32_t *__restrict__ map, int64_t n_pairs,
                                   uint32_t *__restrict__ slot, uint32_t *__restrict__ hslot) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t s = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; s < n_pairs; s += stride) {
    slot[map[s]] = static_cast<uint32_t>(s);
    if (hslot) hslot[map[s]] = static_cast<uint32_t>(s);
  }
}

// Column sums of a row-major [rows, ld] fp32 matrix over `cols` columns, in two stages with a
// fixed summation order (deterministic): stage 1 sums kColsumRows rows per block into
// partial[chunk, cols]; stage 2 adds the chunks in order and writes
// out[c] = scale * sum  with  scale = coef * (grad_out ? grad_out[0] : 1).
constexpr int kColsumRows = 64;

// stage 1 for column c and row chunk `chunk`
__device__ __forceinline__ void colsum_partial_one(const float *__restrict__ x, int64_t rows, int64_t ld, int cols,
                                                   float *__restrict__ partial, int c, int64_t chunk) {
  if (c >= cols) return;
  const int64_t r0 = chunk * kColsumRows;
  if (r0 >= rows) return;
  const int64_t r1 = (r0 + kColsumRows) < rows ? (r0 + kColsumRows) : rows;
  float s = 0.f;
  int64_t r = r0;
  for (; r + 8 <= r1; r += 8) {  // eight independent loads in flight
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = x[(r + u) * ld + c];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; r < r1; ++r) s += x[r * ld + c];
  partial[chunk * cols + c] = s;
}

// stage 2 for column c < cols
__device__ __forceinline__ float colsum_final_value(const float *__restrict__ partial, int n_chunks, int cols,
                                                    const float *__restrict__ grad_out, float coef, int c) {
  float s = 0.f;
  int k = 0;
  for (; k + 8 <= n_chunks; k += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = partial[static_cast<int64_t>(k + u) * cols + c];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; k < n_chunks; ++k) s += partial[static_cast<int64_t>(k) * cols + c];
  return s * coef * (grad_out ? grad_out[0] : 1.f);
}

__device__ __forceinline__ void colsum_final_one(const float *__restrict__ partial, int n_chunks, int cols,
                                                 const float *__restrict__ grad_out, float coef,
                                                 float *__restrict__ out, int c) {
  if (c < cols) out[c] = colsum_final_value(partial, n_chunks, cols, grad_out, coef, c);
}

__global__ __launch_bounds__(256) void colsum_final_kernel(const float *__restrict__ partial,
                                                           int n_chunks, int cols,
                                                           const float *__restrict__ grad_out, float coef,
                                                           float *__restrict__ out) {
  colsum_final_one(partial, n_chunks, cols, grad_out, coef, out, static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x));
}

__global__ void fill_f32_kernel(float *__restrict__ p, int64_t n) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  const int64_t n4 = n >> 2;
  float4 *p4 = reinterpret_cast<float4 *>(p);
  const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n4; i += stride)
    p4[i] = z;
  for (int64_t i = (n4 << 2) + static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += stride)
    p[i] = 0.f;
}

// dst = GT(src * scale[0]) (scale null: a plain cast)
template <typename GT>
__global__ void cast_from_f32_kernel(void *__restrict__ dst, const float *__restrict__ src,
                                     int64_t n, const float *__restrict__ scale = nullptr) {
  const float g = scale ? scale[0] : 1.0f;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  const int64_t n4 = n >> 2;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n4; i += stride) {
    float x[4];
    load_vec<float, 4>(src, i * 4, x);
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] *= g;
    store_vec<GT, 4>(dst, i * 4, x);
  }
  for (int64_t i = (n4 << 2) + static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += stride) {
    float x[1] = {src[i] * g};
    store_vec<GT, 1>(dst, i, x);
  }
}

// dst[0..n) (run-time type) = src * g, four elements at a time by the threads of `n_blocks` blocks
__device__ __forceinline__ void scale_to_dyn(void *__restrict__ dst, int dtype, const float *__restrict__ src, int64_t n,
                                             float g, unsigned block, unsigned n_blocks) {
  const int64_t stride = static_cast<int64_t>(n_blocks) * blockDim.x;
  const int64_t n4 = n >> 2;
  const int64_t tid = static_cast<int64_t>(block) * blockDim.x + threadIdx.x;
  for (int64_t i = tid; i < n4; i += stride) {
    float x[4];
    load_vec<float, 4>(src, i * 4, x);
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] *= g;
    if (dtype == FLEXSAE_F32) store_vec<float, 4>(dst, i * 4, x);
    else if (dtype == FLEXSAE_BF16) store_vec<bf16_t, 4>(dst, i * 4, x);
    else store_vec<f16_t, 4>(dst, i * 4, x);
  }
  for (int64_t i = (n4 << 2) + tid; i < n; i += stride) {
    const float x[1] = {src[i] * g};
    if (dtype == FLEXSAE_F32) store_vec<float, 1>(dst, i, x);
    else if (dtype == FLEXSAE_BF16) store_vec<bf16_t, 1>(dst, i, x);
    else store_vec<f16_t, 1>(dst, i, x);
  }
}

// What follows a step in its backward, one launch: dvals and dbias = their fp32 values times scale[0] (null: one) in the
// leaves' types, in the first n_small blocks (one eighth of them, at least one, for dbias); dW = dW_unit times scale[0],
// rounded once, in the rest; in place with a scale of exactly one those return at once.  Five launches of torch (two
// products, two casts, dW) otherwise, 4-5 us each: B=4096, K=128, F=65536, D=2304 bf16 the step
// 1235 -> 1223.
template <typename UT, typename GT>
__global__ __launch_bounds__(256) void finish_grads_kernel(void *dW, const void *dW_unit, int64_t n_dw,
                                                           void *__restrict__ dvals, int dvals_dtype,
                                                           const float *__restrict__ dvals_unit, int64_t n_dvals,
                                                           void *__restrict__ dbias, int dbias_dtype,
                                                           const float *__restrict__ dbias_unit, int64_t n_dbias,
                                                           const float *__restrict__ scale, unsigned n_small) {
  const float g = scale ? scale[0] : 1.0f;
  const unsigned n_bias_blocks = n_small > 8 ? n_small / 8 : 1;
  if (blockIdx.x < n_bias_blocks) {
    scale_to_dyn(dbias, dbias_dtype, dbias_unit, n_dbias, g, blockIdx.x, n_bias_blocks);
    return;
  }
  if (blockIdx.x < n_small) {
    scale_to_dyn(dvals, dvals_dtype, dvals_unit, n_dvals, g, blockIdx.x - n_bias_blocks, n_small - n_bias_blocks);
    return;
  }
  if (dW == dW_unit && g == 1.0f) return;
  const int64_t stride = static_cast<int64_t>(gridDim.x - n_small) * blockDim.x;
  const int64_t tid = static_cast<int64_t>(blockIdx.x - n_small) * blockDim.x + threadIdx.x;
  const int64_t n4 = n_dw >> 2;
  for (int64_t i = tid; i < n4; i += stride) {
    float x[4];
    load_vec<UT, 4>(dW_unit, i * 4, x);
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] *= g;
    store_vec<GT, 4>(dW, i * 4, x);
  }
  for (int64_t i = (n4 << 2) + tid; i < n_dw; i += stride) {
    float x[1];
    load_vec<UT, 1>(dW_unit, i, x);
    x[0] *= g;
    store_vec<GT, 1>(dW, i, x);
  }
}

}  // namespace flexsae
