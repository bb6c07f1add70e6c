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
  uint32_t empty_at = sh.empty[wv];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const bool have = i < n;
    const uint32_t at_f = static_cast<uint32_t>(f + i);
    const unsigned long long with = __ballot(have && count[i] == 0u);
    if (!have) continue;
    if (count[i] > kListLong) {
      const unsigned long long at = atomicAdd(&sh.long_at, long_step(count[i]));
      ls.long_list[at >> 32] = at_f;
      ls.chunk_begin[at >> 32] = static_cast<uint32_t>(at);
    } else if (classes && count[i] == 0u) {
      ls.empty_list[empty_at + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(with >> 32),
                                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(with), 0u))] = at_f;
    } else if (classes) {
      ls.cls_list[class_of(count[i])][atomicAdd(&sh.cursor[count[i]], 1u)] = at_f;
    }
    empty_at += static_cast<uint32_t>(__popcll(with));
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
// busy stream.  B*K = 524288 over 65536 latents: 8 + 15 us; 524288 Zipf pairs over 262144 latents: 9 + 56 us
// (count, two scan launches, scatter, bucket sort, long-group sort, chunk table and, for sparse shapes, two
// launches for the lists before: 41 and 115 us).
// ---------------------------------------------------------------------------------
constexpr int kChunkThreads = 256;
constexpr int kChunkWaves = kChunkThreads / kWave;
constexpr int kBucketMaxBuckets = 8192;  // LDS cursors of the chunk kernel: 4 bytes per wavefront and bucket
constexpr int kSortThreads = kListThreads;
constexpr int kSortMaxShift = 11;
constexpr int kSortMaxLatents = 1 << kSortMaxShift;  // latents per bucket at most
constexpr int kSortCap = 4096;                       // pairs of a bucket that are kept in the LDS
constexpr int kSortWindow = 1024;                    // chunks whose pieces are collected together
constexpr int kPackShift = 32 - kSortMaxShift;       // a pair inside its chunk: latent within bucket | place in the chunk
constexpr int64_t kMaxChunk = int64_t{1} << kPackShift;
static_assert((kBucketMaxBuckets * kChunkWaves + kChunkWaves) * 4 <= 160 * 1024, "LDS of csr_chunk_sort_kernel");
// (the bucket kernel's arrays come to 71 KB: two blocks per compute unit)

// Dynamic LDS: kChunkWaves * n_buckets + kChunkWaves words.  n_bits: bits of a bucket number.
__global__ __launch_bounds__(kChunkThreads) void csr_chunk_sort_kernel(
    const int64_t *__restrict__ indices, int64_t n_pairs, int64_t F, int shift, uint32_t n_buckets, int n_bits,
    int64_t chunk, uint32_t n_chunks, uint32_t *__restrict__ table, uint32_t *__restrict__ tmp,
    uint32_t *__restrict__ ctrl, int *status_flag) {
  extern __shared__ uint32_t chunk_lds[];
  uint32_t *const cursor = chunk_lds;                            // [wavefront][bucket]
  uint32_t *const wave_tot = chunk_lds + kChunkWaves * n_buckets;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = wave_in_block();
  if (blockIdx.x == 0 && tid < kCtrlWords) ctrl[tid] = 0u;
  for (uint32_t q = tid; q < kChunkWaves * n_buckets; q += kChunkThreads) cursor[q] = 0u;
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
  uint32_t *const mine = cursor + wv * n_buckets;
  for (int64_t at = r0; at < r1; at += U * kWave) {
    int64_t f[U];
    load(at, f, true);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (at + u * kWave + lane < r1) atomicAdd(&mine[f[u] >> shift], 1u);
  }
  __syncthreads();
  {  // exclusive scan over (bucket, wavefront): every thread owns `per` consecutive buckets
    const uint32_t per = (n_buckets + kChunkThreads - 1) / kChunkThreads;
    const uint32_t q0 = tid * per, q1 = (q0 + per) < n_buckets ? (q0 + per) : n_buckets;
    uint32_t sum = 0;
    for (uint32_t q = q0; q < q1; ++q)
#pragma unroll
      for (int w = 0; w < kChunkWaves; ++w) sum += cursor[w * n_buckets + q];
    uint32_t inc = sum;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off, kWave);
      if (lane >= off) inc += y;
    }
    if (lane == kWave - 1) wave_tot[wv] = inc;
    __syncthreads();
    uint32_t at = inc - sum;
    for (int w = 0; w < wv; ++w) at += wave_tot[w];
    for (uint32_t q = q0; q < q1; ++q) {
      table[static_cast<size_t>(q) * n_chunks + blockIdx.x] = at;
#pragma unroll
      for (int w = 0; w < kChunkWaves; ++w) {
        const uint32_t c = cursor[w * n_buckets + q];
        cursor[w * n_buckets + q] = at;
        at += c;
      }
    }
    if (tid == 0) table[static_cast<size_t>(n_buckets) * n_chunks + blockIdx.x] = static_cast<uint32_t>(n);
  }
  __syncthreads();
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
        tmp[p0 + place] = (static_cast<uint32_t>(f[u] & mask) << kPackShift) | static_cast<uint32_t>(i);
        // (LDS accesses of a wavefront are served in order: all lanes have read the cursor)
        if (rank == 0) mine[q] = place + static_cast<uint32_t>(__popcll(same));
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// counter[at] += 1 for every lane with `have`, in the LDS.  The lanes that agree with the first one add up
// beforehand (twice over): adds to one address are served one lane after the other, and a frequent latent
// is most of its bucket.
__device__ __forceinline__ void count_in_lds(uint32_t *counter, uint32_t at, bool have) {
#pragma unroll
  for (int round = 0; round < 2; ++round) {
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
// its latent (0: no marks).
// Groups of more than kListLong pairs (frequent latents) are placed by walking the bucket's pairs in order:
// every wavefront takes a run of them, counts its pairs of every such latent, and places them behind those
// of the wavefronts before it.  The others are gathered in the LDS in any order, and every pair counts
// the smaller ids of its group.
__global__ __launch_bounds__(kSortThreads, 8) void csr_bucket_sort_kernel(
    const uint32_t *__restrict__ tmp, const uint32_t *__restrict__ table, uint32_t n_chunks, int64_t chunk, int shift,
    int64_t F, uint32_t *__restrict__ begin, uint32_t *__restrict__ map, uint32_t *__restrict__ slot,
    uint32_t *__restrict__ hslot, uint32_t solo_bit, PairLists ls) {
  constexpr int kWaves = kSortThreads / kWave;
  constexpr int PER = kSortMaxLatents / kSortThreads;
  constexpr uint32_t kRunLatents = kSortCap / kWaves;  // frequent latents counted per wavefront at a time
  constexpr uint32_t kShort = 0xffffu;
  __shared__ uint32_t cnt[kSortMaxLatents + 1];    // pairs per latent, then their exclusive scan
  __shared__ uint32_t shorts[kSortMaxLatents + 1]; // the same over the groups of up to kListLong pairs
  __shared__ uint16_t lid[kSortMaxLatents];        // number of a frequent latent, or kShort
  __shared__ uint32_t ids[kSortCap];               // cursors [wavefront][frequent latent], then short groups' pair ids
  __shared__ uint32_t list_id[kSortCap];           // the bucket's pairs in pair order, where they fit
  __shared__ uint16_t list_key[kSortCap];          //   and their latents
  __shared__ uint32_t first[kSortWindow + 1];      // window of chunks: first place of each chunk's piece in the list
  __shared__ uint32_t from[kSortWindow + 1];       //   and its place inside the chunk
  __shared__ uint32_t wave_tot[kWaves], wave_tot2[kWaves];
  __shared__ uint32_t n_long_s, n_short_s;
  __shared__ AppendScratch sh;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = wave_in_block();
  const uint32_t q = blockIdx.x;
  const uint32_t lpb = 1u << shift;
  const int64_t f0 = static_cast<int64_t>(q) << shift;
  const uint32_t nlat = (F - f0) < static_cast<int64_t>(lpb) ? static_cast<uint32_t>(F - f0) : lpb;
  const uint32_t *const row0 = table + static_cast<size_t>(q) * n_chunks;
  const uint32_t *const row1 = row0 + n_chunks;

  // base = pairs in earlier buckets, n = pairs in this one
  uint32_t base = 0, n = 0;
  {
    uint32_t s0 = 0, s1 = 0;
    for (uint32_t c = tid; c < n_chunks; c += kSortThreads) {
      s0 += row0[c];
      s1 += row1[c];
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
      s0 += static_cast<uint32_t>(__shfl_xor(static_cast<int>(s0), off, kWave));
      s1 += static_cast<uint32_t>(__shfl_xor(static_cast<int>(s1), off, kWave));
    }
    if (lane == 0) {
      wave_tot[wv] = s0;
      wave_tot2[wv] = s1;
    }
    for (uint32_t k = tid; k <= lpb; k += kSortThreads) cnt[k] = 0u;
    if (tid == 0) n_long_s = n_short_s = 0u;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      base += wave_tot[w];
      n += wave_tot2[w];
    }
    n -= base;
  }
  const bool listed = n <= static_cast<uint32_t>(kSortCap) && n_chunks <= static_cast<uint32_t>(kSortWindow);

  // The pieces of the window of chunks that begins at c0: fills first[] and from[], returns the number of pairs.
  auto open_window = [&](uint32_t c0) {
    static_assert(kSortWindow == kSortThreads, "one chunk per thread");
    const uint32_t c = c0 + tid;
    uint32_t len = 0, at = 0;
    if (c < n_chunks) {
      at = row0[c];
      len = row1[c] - at;
    }
    uint32_t inc = len;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off, kWave);
      if (lane >= off) inc += y;
    }
    __syncthreads();  // the window before has been read by everybody
    if (lane == kWave - 1) wave_tot[wv] = inc;
    __syncthreads();
    uint32_t start = inc - len, m = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      if (w < wv) start += wave_tot[w];
      m += wave_tot[w];
    }
    first[tid] = start;
    from[tid] = at;
    __syncthreads();
    return m;
  };
  // U pairs of that window at once, from the chunks or from the list where there is one: i[u], any pair where i[u] >= m
  uint32_t probes = 1;  // a power of two, at least the number of chunks in a window
  while (probes < n_chunks && probes < static_cast<uint32_t>(kSortWindow)) probes <<= 1;
  auto fetch = [&](uint32_t c0, uint32_t m, bool from_list, const auto &i, auto &key, auto &id) {
    constexpr int U = sizeof(i) / sizeof(i[0]);
    if (from_list) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t at = i[u] < m ? i[u] : 0u;
        key[u] = list_key[at];
        id[u] = list_id[at];
      }
      return;
    }
    uint32_t at[U], c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      at[u] = i[u] < m ? i[u] : 0u;
      c[u] = 0;
    }
    // largest chunk with first[chunk] <= i (an empty chunk repeats its successor's place; past the last one: m)
    for (uint32_t step = probes >> 1; step > 0; step >>= 1)
#pragma unroll
      for (int u = 0; u < U; ++u) c[u] += first[c[u] + step] <= at[u] ? step : 0u;
    uint32_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      v[u] = tmp[static_cast<int64_t>(c0 + c[u]) * chunk + from[c[u]] + (at[u] - first[c[u]])];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      key[u] = v[u] >> kPackShift;
      id[u] = static_cast<uint32_t>(static_cast<int64_t>(c0 + c[u]) * chunk) + (v[u] & static_cast<uint32_t>(kMaxChunk - 1));
    }
  };
  // body(i, key, id, valid) for the pairs begin, begin + stride, ... of the window, U of them requested together; called
  // by all lanes of a wavefront alike, valid: below end
  auto for_pairs = [&](uint32_t c0, uint32_t m, bool from_list, uint32_t begin_i, uint32_t end_i, uint32_t stride, auto body) {
    constexpr int U = 4;
    for (uint32_t i0 = begin_i; __any(i0 < end_i); i0 += U * stride) {
      uint32_t i[U], key[U], id[U];
#pragma unroll
      for (int u = 0; u < U; ++u) i[u] = i0 + u * stride;
      fetch(c0, m, from_list, i, key, id);
#pragma unroll
      for (int u = 0; u < U; ++u)
        body(i[u], key[u], id[u], i[u] < end_i);
    }
  };
  // body(c0, m) for every window of chunks; a single window stays open
  uint32_t open_m = 0;
  const bool one_window = n_chunks <= static_cast<uint32_t>(kSortWindow);
  if (one_window) open_m = open_window(0);
  auto for_windows = [&](auto body) {
    for (uint32_t c0 = 0; c0 < n_chunks; c0 += kSortWindow) body(c0, one_window ? open_m : open_window(c0));
  };

  for_windows([&](uint32_t c0, uint32_t m) {
    for_pairs(c0, m, false, tid, m, kSortThreads, [&](uint32_t i, uint32_t key, uint32_t id, bool valid) {
      if (listed && valid) {
        list_id[i] = id;
        list_key[i] = static_cast<uint16_t>(key);
      }
      count_in_lds(cnt, key, valid);
    });
  });
  __syncthreads();
  uint32_t x[PER];  // pairs of the thread's latents
  {  // exclusive scans of all groups and of the short ones
    uint32_t y[PER], xs = 0, ys = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const uint32_t k = static_cast<uint32_t>(tid) * PER + i;
      x[i] = (k < lpb) ? cnt[k] : 0u;
      y[i] = x[i] > kListLong ? 0u : x[i];
      if (k < lpb) lid[k] = static_cast<uint16_t>(x[i] > kListLong ? atomicAdd(&n_long_s, 1u) : kShort);
      xs += x[i];
      ys += y[i];
    }
    uint32_t xi = xs, yi = ys;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t a = __shfl_up(xi, off, kWave), b = __shfl_up(yi, off, kWave);
      if (lane >= off) {
        xi += a;
        yi += b;
      }
    }
    if (lane == kWave - 1) {
      wave_tot[wv] = xi;
      wave_tot2[wv] = yi;
    }
    __syncthreads();
    uint32_t xr = xi - xs, yr = yi - ys;
    for (int w = 0; w < wv; ++w) {
      xr += wave_tot[w];
      yr += wave_tot2[w];
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const uint32_t k = static_cast<uint32_t>(tid) * PER + i;
      if (k < nlat) begin[f0 + k] = base + xr;
      if (k < lpb) {
        cnt[k] = xr;
        shorts[k] = yr;
      }
      xr += x[i];
      yr += y[i];
    }
    if (tid == kSortThreads - 1) {
      cnt[lpb] = xr;
      shorts[lpb] = yr;
      if (q == gridDim.x - 1) begin[F] = base + n;
    }
  }
  if (ls.chunk_begin) {  // uniform
    const uint32_t k = static_cast<uint32_t>(tid) * PER;
    append_latents(ls, f0 + k, nlat >= k + PER ? PER : nlat > k ? static_cast<int>(nlat - k) : 0, x, sh);
  }
  __syncthreads();

  auto put = [&](uint32_t place, uint32_t id, uint32_t mark) {
    map[place] = id;
    if (slot) slot[id] = place | mark;
    if (hslot) hslot[id] = place | mark;
  };
  // frequent latents, kRunLatents of them at a time; where the bucket's list did not fit the LDS but its other
  // pairs do, those are listed on the way
  const uint32_t n_long = n_long_s;
  const bool collect = !listed && n_long != 0 && shorts[nlat] <= static_cast<uint32_t>(kSortCap);
  for (uint32_t l0 = 0; l0 < n_long; l0 += kRunLatents) {
    const uint32_t nl = (n_long - l0) < kRunLatents ? (n_long - l0) : kRunLatents;
    uint32_t bits = 0;
    while ((1u << bits) < nl) ++bits;
    uint32_t *const mine = ids + wv * kRunLatents;
    bool opened = false;
    for_windows([&](uint32_t c0, uint32_t m) {
      uint32_t run = (m + kWaves - 1) / kWaves;
      run = (run + kWave - 1) / kWave * kWave;
      const uint32_t r0 = wv * run, r1 = (r0 + run) < m ? (r0 + run) : m;
      // wavefront 0's cursors go on from the window before; the others' hold counts until the scan below
      for (uint32_t l = lane; l < nl; l += kWave)
        if (wv != 0 || !opened) mine[l] = 0u;
      __syncthreads();
      if (!opened)
        for (uint32_t k = tid; k < nlat; k += kSortThreads) {
          const uint32_t l = lid[k] - l0;
          if (lid[k] != kShort && l < nl) ids[l] = base + cnt[k];
        }
      opened = true;
      __syncthreads();
      // wavefront w counts into the cursors of wavefront w + 1
      if (wv + 1 < kWaves) {
        for_pairs(c0, m, listed, r0 + lane, r1, kWave, [&](uint32_t, uint32_t key, uint32_t, bool valid) {
          const uint32_t l = lid[key] - l0;
          count_in_lds(mine + kRunLatents, l, valid && lid[key] != kShort && l < nl);
        });
      }
      __syncthreads();
      for (uint32_t l = tid; l < nl; l += kSortThreads) {
        uint32_t at = ids[l];
        for (int w = 1; w < kWaves; ++w) {
          at += ids[w * kRunLatents + l];
          ids[w * kRunLatents + l] = at;
        }
      }
      __syncthreads();
      constexpr int U = 4;
      for (uint32_t i0 = r0; i0 < r1; i0 += U * kWave) {
        uint32_t i[U], key[U], id[U];
#pragma unroll
        for (int u = 0; u < U; ++u) i[u] = i0 + u * kWave + lane;
        fetch(c0, m, listed, i, key, id);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t l = lid[key[u]] - l0;
          const bool have = i[u] < r1 && lid[key[u]] != kShort && l < nl;
          if (collect && l0 == 0) {  // uniform
            const bool is_short = i[u] < r1 && lid[key[u]] == kShort;
            const unsigned long long with = __ballot(is_short);
            uint32_t at = 0;
            if (lane == 0 && with) at = atomicAdd(&n_short_s, static_cast<uint32_t>(__popcll(with)));
            at = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(at)));
            if (is_short) {
              at += __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(with >> 32),
                                              __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(with), 0u));
              list_id[at] = id[u];
              list_key[at] = static_cast<uint16_t>(key[u]);
            }
          }
          unsigned long long same = __ballot(have);
          if (same == 0) continue;
          for (uint32_t b = 0; b < bits; ++b) {
            const unsigned long long ones = __ballot((l >> b) & 1u);
            same &= ((l >> b) & 1u) ? ones : ~ones;
          }
          const uint32_t rank = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(same >> 32),
                                                          __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(same), 0u));
          if (have) {
            const uint32_t place = mine[l] + rank;
            put(place, id[u], 0u);
            if (rank == 0) mine[l] = place + static_cast<uint32_t>(__popcll(same));
          }
          __builtin_amdgcn_wave_barrier();
        }
      }
      __syncthreads();
      // the last wavefront's cursors are where the next window goes on
      for (uint32_t l = tid; l < nl; l += kSortThreads) ids[l] = ids[(kWaves - 1) * kRunLatents + l];
      __syncthreads();
    });
  }

  // short groups, as many consecutive latents at a time as the LDS holds the pairs of (usually all)
  auto for_shorts = [&](auto body) {
    if (collect) for_pairs(0, n_short_s, true, tid, n_short_s, kSortThreads, body);
    else for_windows([&](uint32_t c0, uint32_t m) { for_pairs(c0, m, listed, tid, m, kSortThreads, body); });
  };
  for (uint32_t k0 = 0; k0 < nlat;) {  // uniform
    const uint32_t s0 = shorts[k0];
    uint32_t k1 = nlat;
    if (shorts[nlat] - s0 > static_cast<uint32_t>(kSortCap)) {
      uint32_t lo = k0 + 1, hi = nlat;  // largest k1 with shorts[k1] - s0 <= kSortCap
      while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (shorts[mid] - s0 <= static_cast<uint32_t>(kSortCap)) lo = mid; else hi = mid - 1;
      }
      k1 = lo;
    }
    __syncthreads();  // everybody has read shorts[] and is done with ids[]
    // placed in the order of the atomics, which leave shorts[k] at the end of group k
    for_shorts([&](uint32_t, uint32_t key, uint32_t id, bool valid) {
      if (valid && key >= k0 && key < k1 && lid[key] == kShort) ids[atomicAdd(&shorts[key], 1u) - s0] = id;
    });
    __syncthreads();
    for_shorts([&](uint32_t, uint32_t key, uint32_t id, bool valid) {
      if (!valid || key < k0 || key >= k1 || lid[key] != kShort) return;
      const uint32_t len = cnt[key + 1] - cnt[key];
      const uint32_t *const group = ids + (shorts[key] - len - s0);
      uint32_t rank = 0, j = 0;
      for (; j + 8 <= len; j += 8) {
        uint32_t x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = group[j + u];
#pragma unroll
        for (int u = 0; u < 8; ++u) rank += (x[u] < id) ? 1u : 0u;
      }
      for (; j < len; ++j) rank += (group[j] < id) ? 1u : 0u;
      put(base + cnt[key] + rank, id, len == 1 ? solo_bit : 0u);
    });
    k0 = k1;
  }
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

// stage 2 for column c
__device__ __forceinline__ void colsum_final_one(const float *__restrict__ partial, int n_chunks, int cols,
                                                 const float *__restrict__ grad_out, float coef,
                                                 float *__restrict__ out, int c) {
  if (c >= cols) return;
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
  out[c] = s * coef * (grad_out ? grad_out[0] : 1.f);
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

}  // namespace flexsae
