// C-ABI entry points (include/flexsae_amd.h): argument validation, kernel selection and
// launches.  No allocation, no synchronisation, no global state.
#include <hip/hip_runtime.h>
#include <stdlib.h>

#include <mutex>

#include "common.hpp"
#include "fwd_kernels.hpp"
#include "csr_kernels.hpp"
#include "hier_bwd_kernels.hpp"
#include "hier_train_kernel.hpp"
#include "hier_hot_kernel.hpp"
#include "hier_epilogue_kernel.hpp"
#include "segment_kernels.hpp"
#include "topk_bwd_kernels.hpp"

using namespace flexsae;

// Device memory of flexsae_hier_fwd_static, the one entry point that takes no workspace: the
// forward kernels' per-(row, tile) loss partials live here.  Every GPU the library runs on holds
// its own copy of the array until the process ends.  Host code never uses the array's name as an
// address: the per-device address comes from hipGetSymbolAddress (static_scratch_for_current_device).
constexpr size_t kStaticScratchBytes = FLEXSAE_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

// gathers in flight per wavefront before the first one is consumed
#ifndef FLEXSAE_SWEEP_U
#define FLEXSAE_SWEEP_U 16
#endif
#ifndef FLEXSAE_REDUCE_U
#define FLEXSAE_REDUCE_U 4
#endif
#ifndef FLEXSAE_PIECE_U
#define FLEXSAE_PIECE_U 4
#endif
#ifndef FLEXSAE_FWD_U
#define FLEXSAE_FWD_U 8
#endif
#ifndef FLEXSAE_TOPK_VEC8
#define FLEXSAE_TOPK_VEC8 1
#endif
#ifndef FLEXSAE_TOPK_RESID16
#define FLEXSAE_TOPK_RESID16 1
#endif

namespace {

constexpr int kBlock = 256;              // threads per block of the wave-per-item kernels
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr size_t kAlign = 256;
constexpr int kBwdSgdUpdate = 1 << 20;  // internal flag of the slice loop: dW is the weight matrix, updated in place
constexpr int kBwdSolo = 1 << 22;       // internal flag of the slice loop: slot[] marks the only pairs of their latents
constexpr int kBwdScaled = 1 << 23;  // internal flag of the slice loop: dW is multiplied by grad_out[0] before it is rounded
constexpr int kBwdHot = 1 << 21;        // internal flag of the slice loop: hot latents are accumulated in the LDS
constexpr unsigned kLongBlocks = 1024;    // leading blocks of a reduction launch that serve hot latents
constexpr int64_t kListBlocks = 8192;     // blocks of a reduction launch that work from the lists of latents

inline bool valid_dtype(int d) { return d == FLEXSAE_F32 || d == FLEXSAE_BF16 || d == FLEXSAE_F16; }
inline size_t dtype_size(int d) { return d == FLEXSAE_F32 ? 4 : 2; }
inline bool aligned(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
inline size_t round_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

int check_shape(const flexsae_shape *s) {
  if (!s) return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (s->B <= 0 || s->K <= 0 || s->F <= 0 || s->D <= 0) return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (!valid_dtype(s->weight_dtype) || !valid_dtype(s->vals_dtype) || !valid_dtype(s->bias_dtype) ||
      !valid_dtype(s->target_dtype))
    return FLEXSAE_ERR_INVALID_ARGUMENT;
  // D < 2^29: a row of any matrix here (at most 4 bytes per element) fits a buffer descriptor
  if (s->F >= (1LL << 31) || s->D >= (1LL << 29) || s->K >= (1LL << 31)) return FLEXSAE_ERR_UNSUPPORTED;
  if (s->B > ((1LL << 32) - 1) / s->K) return FLEXSAE_ERR_UNSUPPORTED;  // B*K < 2^32
  return FLEXSAE_OK;
}

int launch_status() { return hipGetLastError() == hipSuccess ? FLEXSAE_OK : FLEXSAE_ERR_LAUNCH; }

// Address of `scratch` on the current device, looked up once per device and kept.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {};

int static_scratch_for_current_device(void **out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return FLEXSAE_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
      (void)hipGetLastError();
      return FLEXSAE_ERR_LAUNCH;
    }
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return FLEXSAE_OK;
}

// Largest vector width (elements per lane) the row layout allows: every row start and
// every lane offset must be aligned to the vector, and wider than 16 bytes gains nothing.
int pick_vec(int64_t D, size_t elem_size, const void *base, int max_vec) {
  for (int v = max_vec; v > 1; v >>= 1) {
    if (static_cast<size_t>(v) * elem_size > 16) continue;
    if (D % v == 0 && aligned(base, v * elem_size)) return v;
  }
  return 1;
}

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

inline unsigned grid_for(int64_t n_threads, int block, int64_t cap) {
  int64_t g = ceil_div(n_threads, block);
  if (g > cap) g = cap;
  if (g < 1) g = 1;
  return static_cast<unsigned>(g);
}

struct FwdPlan {
  int vec;
  int lpr;  // lanes per row piece
  int64_t n_row_blocks;
  int64_t n_items;   // blocks with work, each leaves one loss partial
  int64_t xcd_span;  // items per XCD; 0: items in order; -n_tiles: wavefronts in row order
  unsigned grid;
};

FwdPlan plan_fwd(const flexsae_shape *s, const void *weight, const void *target, const void *bias,
                 const float *resid) {
  const size_t es = dtype_size(s->weight_dtype);
  int vec = pick_vec(s->D, es, weight, 8);
  // resid is stored with fp32 vectors of the same width, target/bias are read with the
  // weight's vector type when they share its dtype
  if (s->target_dtype == s->weight_dtype && !aligned(target, vec * es)) vec = 1;
  if (s->bias_dtype == s->weight_dtype && !aligned(bias, vec * es)) vec = 1;
  if (!aligned(resid, 16)) vec = 1;
  const uint64_t row_bytes = static_cast<uint64_t>(s->D) * es;
  // Eight bytes per lane where sixteen leave fewer than five wavefronts for every four SIMDs.  us with sixteen / eight (K=64,
  // bf16; uniform, skewed indices): 512 wavefronts (B=512, D=512, F=65536) 14.4 / 10.4, 10.0 / 8.6; 1024 (B=451, D=1160,
  // F=16384) 18.0 / 15.4, 14.1 / 12.4; 1152 (B=256, D=2304, F=16384) 16.8 / 14.1, 12.8 / 12.7; above it depends on the
  // shape: 1536 (B=768, D=1024, F=65536) 18.2 / 17.1, 14.0 / 12.7, (B=677, D=1160, F=65536) 21.2 / 24.5, 16.0 / 15.3; from
  // 2048 on the wider ones (B=1024, D=1024, F=65536) 21.2 / 21.7, 15.2 / 16.1.
  if (vec == 8 && static_cast<uint64_t>(s->B) * row_bytes < 1280 * 1024) vec = 4;
  FwdPlan p;
  p.vec = vec;
  // Bytes of a row piece, and whether every L2 works on a tile of its own.  Measured (us; uniform / skewed
  // indices; B=4096, K=64, D=2304 bf16):
  //   F            128 B per L2    256 B per L2    512 B, all L2s on one tile
  //   16384          68 / 62         72 / 59         135 / 63
  //   32768          93 / 64        114 / 61         152 / 66
  //   49152         124 / 66        133 / 62         166 / 69
  //   65536         139 / 72        145 / 67         162 / 72
  //   131072        168 / 87        161 / 82         167 / 83
  //   196608        175 / 93        179 / 87         173 / 87
  // (from 65536 on the narrow pieces gain less on uniform indices than they lose on skewed ones) and fp32
  // (B=2048, K=64, D=1024): 256 B beats 128 B from 32768 rows on (65536: 65 / 31 against 73 / 32, 131072:
  // 73 / 32 against 83 / 34; 512 B 78 / 37) and equals it below.  Eight-byte lanes gain 5 % on uniform
  // indices around 65536 rows and lose 25 % on skewed ones: 16 bytes per lane wherever rows allow it.
  // The narrow pieces want the blocks of one tile (B / 32) to be about as many as an XCD runs at a time; with fewer it
  // works on several tiles at once (F=32768, D=2304, 128 B against 256 B: B=1024 45.0 / 25.4 against 41.4 / 22.0, B=2048
  // 64.4 / 39.3 against 70.9 / 36.4; F=16384, D=8192: B=256 43.9 / 20.8 against 40.5 / 19.6).
  //
  // Rows that do not start on a line: a piece reaches into one line more than its own, which the L2 has to hold and to
  // fetch; in row order the pieces of a row share them.  The tiles pay while an L2 (4 MB) holds about two fifths of one
  // tile's lines (F * 384 B = 10 MB); latents up to which they are the faster ones on uniform indices (B=4096, K=64; on
  // skewed ones the two orders are within 6 %): D=1538 bf16 31000, 1540 29700, 2305 33000, 3004 32500, 4100 32500, fp32
  // (B=2048) D=1002 27500, 1700 26800.  Rows of a few pieces are close together in row order too and lose the most to a
  // last piece that is nearly empty: D=264 bf16 15000, 520 fp16 18500, 772 bf16 20000, 300 fp32 19000.
  //
  // Tiles that all L2s walk together pay where latents repeat within the batch.  Pairs per latent, then the time with
  // tiles and in row order (K=64, bf16):
  //   1/8   F=262144, D=4096  46.6 / 23.8    45.3 / 21.8      F=524288, D=8192  216.9 / 92.8   212.7 / 83.2
  //   1/4   F=262144, D=4096  102.7 / 42.9   98.3 / 39.8      F=524288, D=2304  114.7 / 43.5   112.0 / 45.5
  //   1/2   F=262144, D=4096  183.9 / 79.8   194.2 / 73.1     F=524288, D=2304  208.7 / 85.9   220.4 / 91.4
  //   1     F=262144, D=4096  325.9 / 157.8  384.4 / 150.4    F=262144, D=8184  1464 / 654     1673 / 649
  // (the last one two pairs per latent).  Where rows do not start on a line: only for weights of 4 GiB and more (D=3004,
  // F=262144, one pair per latent: 281 / 144 against 281 / 142), not where one tile's lines are far more than the
  // memory-side cache holds (B=16384, D=3004, F=800000: 1211 / 611 against 1238 / 587; D=1004, F=2000000: 491 / 205
  // against 427 / 195), and not where a lane's four bytes halve the pieces (B=1346, K=256, F=524288, D=4966: 737
  // against 640, uniform).
  const bool lines = row_bytes % 128 == 0;
  const uint64_t F = static_cast<uint64_t>(s->F);
  const uint64_t n_256 = (row_bytes + 255) / 256;
  const bool by_xcd = s->B > 1 && (lines ? F <= 131072 : n_256 < 8 ? F * n_256 * 256 <= 24576 * row_bytes : F <= 26624);
  const bool repeats = 8 * static_cast<uint64_t>(s->B) * static_cast<uint64_t>(s->K) > 3 * F;
  // (A single row: a block per narrow tile would leave more partials than the workspace has room for, see forward().)
  const bool by_row = !by_xcd && (s->B == 1 || !repeats ||
                                  (!lines && (F * row_bytes < (uint64_t{1} << 32) || F > (uint64_t{1} << 20) || vec * es < 8)));
  const size_t piece_bytes = by_row ? 1024 : !by_xcd ? 512 : (es == 2 && F <= 49152 && lines && s->B >= 2048) ? 128 : 256;
  p.lpr = static_cast<int>(piece_bytes / (static_cast<size_t>(vec) * es));
  if (p.lpr > kWave) p.lpr = kWave;
  const int64_t rows = kWave / p.lpr;
  const int64_t n_tiles = ceil_div(s->D, static_cast<int64_t>(p.lpr) * vec);
  p.n_row_blocks = ceil_div(s->B, rows * kWavesPerBlock);
  p.n_items = by_row ? ceil_div(n_tiles * ceil_div(s->B, rows), static_cast<int64_t>(kWavesPerBlock)) : n_tiles * p.n_row_blocks;
  p.xcd_span = by_xcd ? ceil_div(p.n_items, 8) : by_row ? -n_tiles : 0;
  p.grid = static_cast<unsigned>(by_xcd ? p.xcd_span * 8 : p.n_items);
  return p;
}

template <typename WT, bool HIER>
void launch_fwd(const flexsae_shape *s, const FwdPlan &p, const int64_t *indices,
                const void *weight, const void *vals, const void *bias, const void *target,
                float *resid, double *partial, int *status_flag, hipStream_t st) {
#define FLEXSAE_LAUNCH_FWD(VEC, LPR)                                                                       \
  hipLaunchKernelGGL((sae_fwd_kernel<WT, VEC, LPR, HIER, FLEXSAE_FWD_U>), dim3(p.grid), dim3(kBlock), 0, st, \
                     indices, weight, vals, s->vals_dtype, bias, s->bias_dtype, target, s->target_dtype,   \
                     resid, partial, status_flag, s->B, p.n_row_blocks, p.n_items, p.xcd_span,             \
                     static_cast<int>(s->K), s->F, static_cast<int>(s->D))
  constexpr int E = static_cast<int>(sizeof(typename Traits<WT>::store_t));
  constexpr int V16 = 16 / E, V8 = 8 / E, V4 = 4 / E;  // columns per lane
  constexpr bool kNarrow = E == 2;  // 128-byte pieces: 16-bit weights only
#define FLEXSAE_LAUNCH_FWD_V(VEC, LPR128, LPR256, LPR512)  \
  do {                                                     \
    if (kNarrow && p.lpr == LPR128) {                      \
      FLEXSAE_LAUNCH_FWD(VEC, (kNarrow ? LPR128 : LPR256)); \
    } else if (p.lpr == LPR256) {                          \
      FLEXSAE_LAUNCH_FWD(VEC, LPR256);                     \
    } else if (p.lpr == LPR512) {                          \
      FLEXSAE_LAUNCH_FWD(VEC, LPR512);                     \
    } else {                                               \
      FLEXSAE_LAUNCH_FWD(VEC, 64);                         \
    }                                                      \
  } while (0)
  if (p.vec == V16) {
    FLEXSAE_LAUNCH_FWD_V(V16, 8, 16, 32);
  } else if (p.vec == V8) {
    FLEXSAE_LAUNCH_FWD_V(V8, 16, 32, 64);
  } else if (p.vec == V4) {
    FLEXSAE_LAUNCH_FWD_V(V4, 32, 64, 64);
  } else if constexpr (kNarrow) {
    FLEXSAE_LAUNCH_FWD_V(1, 64, 64, 64);
  }
#undef FLEXSAE_LAUNCH_FWD_V
#undef FLEXSAE_LAUNCH_FWD
}

// ---- TopK forward in latent order ---------------------------------------------------------
// Rows of at most 512 pairs.  `waves` wavefronts per block, lpr lanes per row piece; waves == 0: not in latent order.
struct OrderedPlan {
  int waves, lpr;
  int64_t n_row_blocks, n_items, xcd_span;
  size_t steps_bytes;  // (row, val) of every pair, after the loss partials
};

// What the ordered walk takes (whether it pays: order_pays): 64 to 512 pairs per row and 512 batch rows or more, rows that
// start on a line, pieces of one tile that do not fit an L2 (4 MB), gathers of 128 MiB and more, half a GiB below 128 pairs per
// row; forward_ordered() also asks for whole 16-byte vectors and room for the steps.  Fewer than 2^20 latents: a latent and
// a position in its row fit a dword.
// 128-byte pieces (16-bit weights, eight rows per wavefront) beat 256-byte ones from more than 2048 rows on (B=4096, K=64,
// D=2304, F=131072 149 / 161; at B=2048, K=256, D=1024 96 / 87, at B=512 143 / 114).  As many wavefronts per block as
// leave 32 blocks, one per compute unit of an XCD, for a tile: fp32, K=256, D=4096, F=65536, B=512 blocks of 16 / 8 / 4
// wavefronts 236 / 237 / 228, B=1024 (D=1024) 85 / 76 / 88, B=2048 181 / 210 / 235; 16-bit pieces of 128 bytes always
// eight (they leave a last round of blocks that is not full otherwise).
OrderedPlan plan_ordered(const flexsae_shape *s) {
  OrderedPlan p = {};
  const size_t es = dtype_size(s->weight_dtype);
  const uint64_t row_bytes = static_cast<uint64_t>(s->D) * es;
  const uint64_t F = static_cast<uint64_t>(s->F);
  if (s->K < 64 || s->K > 512 || s->B < 512 || F >= (uint64_t{1} << 20) || row_bytes % 128 != 0) return p;
  if (static_cast<uint64_t>(s->B) * s->K * row_bytes < (s->K < 128 ? uint64_t{512} << 20 : uint64_t{128} << 20)) return p;
  const bool narrow = es == 2 && s->B > 2048;
  const uint64_t piece_bytes = narrow ? 128 : 256;
  if (F * piece_bytes < (uint64_t{4} << 20)) return p;
  p.lpr = static_cast<int>(piece_bytes / 16);
  const int64_t rows = kWave / p.lpr;
  p.waves = narrow ? 8 : s->B >= 2048 ? 16 : s->B >= 1024 ? 8 : 4;
  if (es == 2 && p.waves == 16) p.waves = 8;
  p.n_row_blocks = ceil_div(s->B, rows * p.waves);
  p.n_items = ceil_div(static_cast<int64_t>(row_bytes), static_cast<int64_t>(piece_bytes)) * p.n_row_blocks;
  p.xcd_span = ceil_div(p.n_items, 8);
  p.steps_bytes = round_up(static_cast<size_t>(s->B) * static_cast<size_t>(s->K) * 8, kAlign);
  return p;
}

// Whether it is the better walk of such a shape.  A call does not know how its indices repeat: uniform ones gain by the order,
// skewed ones (Zipf 1.1), most of whose gathers hit an L2 either way, pay a sort of 5-6 us and mostly gain little.  The lines lie
// where the gain of the first is most, a loss of the second counted three times; two things decide:
//   reuse   pairs per latent among the rows that an XCD walks at a time (32 compute units of sixteen wavefronts): what a piece
//           fetched once is used for.  From two with 128-byte pieces, more than 0.75 with 256-byte ones, with more and with fewer
//           latents than 131072 alike.
//   work    the gathered MiB: 800 with 128-byte pieces; with 256-byte ones 1200, or 500 where the last round of blocks (up to
//           sixteen wavefronts each) leaves no more than a quarter of the rounds empty, and 80 pairs per row or 1000 MiB.
// us without / with the ordering, uniform and skewed indices:
//   bf16, 128 B   B=4096, D=2304: K=128, F=65536 286 / 188, 150 / 149; K=64, F=65536 150 / 116, 69 / 77, F=131072 169 / 149,
//                 83 / 90; K=256, F=262144 673 / 487, 359 / 315;  B=16384, K=64, F=52516, D=1024 247 / 158, 116 / 125;  not
//                 B=8041, K=128, F=524288, D=512 153 / 183, 72 / 88 (fp16), nor B=4096, K=134, F=131072, D=256 41 / 36, 24 / 32
//   bf16, 256 B   B=2048, D=4096: K=128, F=32768 264 / 149, 127 / 120; K=256, F=262144 604 / 510, 364 / 298;  B=1016, K=195,
//                 F=65536, D=2048 108 / 83, 51 / 61;  not B=1024, K=128, D=2304, F=131072 93 / 96, 43 / 53
//   fp32, 256 B   B=2048, D=1024: K=256, F=131072 275 / 181, 144 / 133; K=96, F=65536 100 / 66, 45 / 44;  B=8192, K=109,
//                 F=65536, D=704 293 / 166, 121 / 125;  not B=2048, K=64, F=65536, D=1024 69 / 50, 32 / 34, B=1024, K=192,
//                 D=1152, F=32768 103 / 72, 52 / 59 or B=512, K=256, F=65536, D=256 24 / 26, 22 / 22
// Of 230 shapes (F 16384 to 524288) it takes 157: uniform indices are 1.34 times as fast there, none slower by 5 %, skewed ones 1.01,
// 30 of them 5 % slower or more (the most B=8192, K=66, F=32768, D=672 fp32: 139 / 104, 74 / 89).
bool order_pays(const flexsae_shape *s, const OrderedPlan &p) {
  const uint64_t B = static_cast<uint64_t>(s->B), K = static_cast<uint64_t>(s->K), F = static_cast<uint64_t>(s->F);
  const uint64_t mib = B * K * static_cast<uint64_t>(s->D) * dtype_size(s->weight_dtype) >> 20;
  const bool narrow = p.lpr == 8;
  const uint64_t at_a_time = 32 * 16 * (narrow ? 8 : 4);
  const uint64_t reused = (B < at_a_time ? B : at_a_time) * K;
  if (narrow) return reused >= 2 * F && mib >= 800;
  if (4 * reused <= 3 * F || (K < 80 && mib < 1000)) return false;
  const int64_t round = 32 * 16 / p.waves;  // blocks of an XCD at a time
  return mib >= 1200 || (mib >= 500 && 4 * p.xcd_span >= 3 * round * ceil_div(p.xcd_span, round));
}

void launch_order(const flexsae_shape *s, const int64_t *indices, const void *vals, vec_t<uint32_t, 2> *steps,
                  int *status_flag, hipStream_t st) {
  const int K = static_cast<int>(s->K);
  const int C = K <= 64 ? 1 : K <= 128 ? 2 : K <= 256 ? 4 : 8;
  const dim3 grid(static_cast<unsigned>(ceil_div(s->B, kWavesPerBlock)));
  const auto kernel = C == 1 ? topk_order_kernel<1> : C == 2 ? topk_order_kernel<2> : C == 4 ? topk_order_kernel<4> : topk_order_kernel<8>;
  hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, st, indices, vals, s->vals_dtype, s->B, K, s->F, steps, status_flag);
}

template <typename WT>
void launch_ordered_fwd(const flexsae_shape *s, const OrderedPlan &p, const vec_t<uint32_t, 2> *steps, const void *weight,
                        const void *bias, const void *target, float *resid, double *partial, hipStream_t st) {
  constexpr int VEC = 16 / static_cast<int>(sizeof(typename Traits<WT>::store_t));
#define FLEXSAE_ORDERED(LPR, U, NW)                                                                                          \
  hipLaunchKernelGGL((topk_ordered_fwd_kernel<WT, VEC, LPR, U, NW>), dim3(static_cast<unsigned>(p.xcd_span * 8)),            \
                     dim3(NW * kWave), 0, st, steps, weight, bias, s->bias_dtype, target, s->target_dtype, resid, partial, \
                     s->B, p.n_row_blocks, p.n_items, p.xcd_span, static_cast<int>(s->K), static_cast<int>(s->D))
  if constexpr (VEC == 8) {
    if (p.lpr == 8) {
      FLEXSAE_ORDERED(8, 8, 8);
    } else if (p.waves == 8) {
      FLEXSAE_ORDERED(16, 16, 8);
    } else {
      FLEXSAE_ORDERED(16, 16, 4);
    }
  } else {
    if (p.waves == 16) {
      FLEXSAE_ORDERED(16, 16, 16);
    } else if (p.waves == 8) {
      FLEXSAE_ORDERED(16, 16, 8);
    } else {
      FLEXSAE_ORDERED(16, 16, 4);
    }
  }
#undef FLEXSAE_ORDERED
}

// The TopK forward in latent order, where the shape and the rows allow it and the workspace has room behind the partials
// (flexsae_topk_fwd_workspace_bytes).  Returns the number of loss partials, 0 if nothing was launched.
int64_t forward_ordered(const flexsae_shape *s, const int64_t *indices, const void *weight, const void *vals,
                        const void *bias, const void *target, float *resid, void *workspace, size_t workspace_bytes,
                        int *status_flag, hipStream_t st) {
  const OrderedPlan p = plan_ordered(s);
  const size_t base = flexsae_fwd_workspace_bytes(s);
  if (p.waves == 0 || workspace_bytes < base + p.steps_bytes || !aligned(weight, 16) ||
      static_cast<size_t>(p.n_items) * sizeof(double) > base)
    return 0;
  if ((s->target_dtype == s->weight_dtype && !aligned(target, 16)) || (s->bias_dtype == s->weight_dtype && !aligned(bias, 16)))
    return 0;
  auto *const steps = reinterpret_cast<vec_t<uint32_t, 2> *>(static_cast<uint8_t *>(workspace) + base);
  double *const partial = static_cast<double *>(workspace);
  launch_order(s, indices, vals, steps, status_flag, st);
  switch (s->weight_dtype) {
    case FLEXSAE_F32:
      launch_ordered_fwd<float>(s, p, steps, weight, bias, target, resid, partial, st);
      break;
    case FLEXSAE_BF16:
      launch_ordered_fwd<bf16_t>(s, p, steps, weight, bias, target, resid, partial, st);
      break;
    default:
      launch_ordered_fwd<f16_t>(s, p, steps, weight, bias, target, resid, partial, st);
  }
  return p.n_items;
}

template <bool HIER>
int forward(const flexsae_shape *s, const int64_t *indices, const void *weight, const void *vals,
            const void *bias, const void *target, float *loss, float *resid, void *workspace,
            size_t workspace_bytes, int *status_flag, void *stream) {
  int rc = check_shape(s);
  if (rc != FLEXSAE_OK) return rc;
  if (!indices || !weight || !vals || !bias || !target || !loss || !resid)
    return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (!aligned(indices, 8) || !aligned(weight, dtype_size(s->weight_dtype)) ||
      !aligned(vals, dtype_size(s->vals_dtype)) || !aligned(bias, dtype_size(s->bias_dtype)) ||
      !aligned(target, dtype_size(s->target_dtype)) || !aligned(loss, 4) || !aligned(resid, 16))
    return FLEXSAE_ERR_ALIGNMENT;
  if (!workspace || workspace_bytes < flexsae_fwd_workspace_bytes(s) || !aligned(workspace, kAlign))
    return FLEXSAE_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  int64_t n_partials = 0;
  if constexpr (!HIER)
    n_partials = forward_ordered(s, indices, weight, vals, bias, target, resid, workspace, workspace_bytes, status_flag, st);
  double *partial = static_cast<double *>(workspace);
  if (n_partials == 0) {
    const FwdPlan p = plan_fwd(s, weight, target, bias, resid);
    // One double per block.  A tile has at least 64 columns and a block four rows (two or more rows are at least twice as
    // many as blocks of them; a single row goes by row, four tiles to a block): no more than the workspace's four bytes
    // per row and 64 columns, to which it is rounded up.
    if (static_cast<size_t>(p.n_items) * sizeof(double) > workspace_bytes) return FLEXSAE_ERR_WORKSPACE;
    switch (s->weight_dtype) {
      case FLEXSAE_F32:
        launch_fwd<float, HIER>(s, p, indices, weight, vals, bias, target, resid, partial,
                                  status_flag, st);
        break;
      case FLEXSAE_BF16:
        launch_fwd<bf16_t, HIER>(s, p, indices, weight, vals, bias, target, resid, partial,
                                   status_flag, st);
        break;
      default:
        launch_fwd<f16_t, HIER>(s, p, indices, weight, vals, bias, target, resid, partial,
                                  status_flag, st);
    }
    n_partials = p.n_items;
  }
  rc = launch_status();
  if (rc != FLEXSAE_OK) return rc;
  const double count = static_cast<double>(s->B) * static_cast<double>(s->D) *
                       (HIER ? static_cast<double>(s->K) : 1.0);
  hipLaunchKernelGGL(loss_finalize_kernel, dim3(1), dim3(1024), 0, st, partial, n_partials,
                     1.0 / count, loss);
  return launch_status();
}

template <typename WT>
void launch_hier_bwd_t(const flexsae_shape *s, const int64_t *indices, const void *weight,
                       const void *vals, const float *resid, const float *grad_out, float coef,
                       float *dW, float *dvals, float *dbias, int *status_flag, hipStream_t st) {
  const int K = static_cast<int>(s->K), D = static_cast<int>(s->D);
  // widest tile that the row length fills without padding (C columns per lane)
  const int C = (D % 256 == 0) ? 4 : (D % 128 == 0) ? 2 : 1;
  const int ntiles = static_cast<int>(ceil_div(D, static_cast<int64_t>(kWave) * C));
  const int64_t n_items = s->B * ntiles;
  const unsigned grid = static_cast<unsigned>(ceil_div(n_items, kWavesPerBlock));
#define FLEXSAE_LAUNCH_HB(CC)                                                                    \
  hipLaunchKernelGGL((hier_bwd_kernel<WT, CC, 4>), dim3(grid), dim3(kBlock), 0, st, indices,     \
                     weight, vals, s->vals_dtype, resid, grad_out, coef, dW, dvals, dbias,       \
                     status_flag, n_items, ntiles, K, s->F, D)
  if (C == 4) {
    FLEXSAE_LAUNCH_HB(4);
  } else if (C == 2) {
    FLEXSAE_LAUNCH_HB(2);
  } else {
    FLEXSAE_LAUNCH_HB(1);
  }
#undef FLEXSAE_LAUNCH_HB
}

void zero_f32(float *p, int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(fill_f32_kernel, dim3(grid_for(ceil_div(n, 4), 256, 1 << 16)), dim3(256), 0, st,
                     p, n);
}

// How a pair list is built for a given problem size.  The bucketed construction serves every
// size whose bucket count fits the LDS cursors of its chunk kernel; beyond that (more than
// kBucketMaxBuckets * kSortMaxLatents latents) the list is built with one memory atomic per pair.
struct CsrPlan {
  bool bucketed;
  int shift;           // a bucket is 2^shift consecutive latents
  int pack_shift;
  uint32_t n_batches;  // blocks per bucket, which share the batches of latents of a large one
  uint32_t n_buckets;
  int n_bits;          // bits of a bucket number
  int64_t chunk;       // consecutive pairs ordered by one block
  uint32_t n_chunks;
  size_t table_len;    // (n_buckets + 1) * n_chunks
};

CsrPlan plan_csr(int64_t n_pairs, int64_t F) {
  CsrPlan p;
  // latents per bucket: about 2048 pairs per bucket on average, a power of two (see below for fewer); more than 2048 latents only where buckets
  // of 2048 are more than the chip holds at once (2097152 latents, 262144 pairs: 29 us that way and 21 with 4096 latents;
  // 1048576 latents fit and are as fast either way)
  int shift = 0;
  while (shift < kSortMaxShift && (static_cast<int64_t>(2) << shift) * n_pairs <= 2048 * F &&
         (shift < 11 || ceil_div(F, static_cast<int64_t>(1) << shift) > kBucketBlocks))
    ++shift;
  while (shift < kSortMaxShift && ceil_div(F, static_cast<int64_t>(1) << shift) > kBucketMaxBuckets) ++shift;
  // Half as many where every compute unit still has at most one block (kBucketBlocks is two for each; with the batches below): a
  // block with fewer pairs is done sooner, one with frequent latents above all, which is what the rule is for: uniform indices gain
  // less or, once, lose 1 %.  us of the pair list, uniform and skewed (distinct in a row), before / with this:
  // B=1024, K=64, F=32768 18.1 / 17.1, 27.6 / 25.6; B=4096, K=64, F=65536 22.5 / 22.8, 33.8 / 31.5; B=404, K=50, F=12953 16.9 /
  // 15.9, 23.8 / 21.3; not with more blocks than that: B=2435, K=128, F=24332 in 381 buckets 23.1 / 24.5, 31.3 / 36.2, B=2048,
  // K=64, F=262144 in 256 of two batches 21.4 / 24.5; nor a quarter, whose chunks take longer to order (B=1777, K=50, F=24571,
  // D=1538 bf16, the step: 183.6 us with 2048 pairs, 181.9 with 1024, 186.7 with 512).
  while (shift > 0 && (n_pairs << shift) > 1024 * F &&
         ceil_div(F, int64_t{1} << (shift - 1)) * ceil_div(int64_t{1} << (shift - 1), kRunLatents) <= kBucketBlocks / 2)
    --shift;
  p.shift = shift;
  p.pack_shift = csr_pack_shift(shift);
  const int64_t n_buckets = ceil_div(F, static_cast<int64_t>(1) << shift);
  p.n_batches = 1;
  while ((p.n_batches * kRunLatents) >> shift == 0 && 2 * p.n_batches * n_buckets <= kBucketBlocks) p.n_batches *= 2;
  p.bucketed = n_buckets <= kBucketMaxBuckets;
  p.n_bits = 0;
  while (p.bucketed && (static_cast<int64_t>(1) << p.n_bits) < n_buckets) ++p.n_bits;
  p.chunk = 2048;
  while (p.bucketed && p.chunk < (int64_t{1} << p.pack_shift) &&
         (ceil_div(n_pairs, p.chunk) > kSortChunks || ceil_div(n_pairs, p.chunk) * n_buckets > (static_cast<int64_t>(1) << 22)))
    p.chunk *= 2;
  p.n_chunks = static_cast<uint32_t>(ceil_div(n_pairs, p.chunk));
  if (p.n_chunks > static_cast<uint32_t>(kSortChunks)) p.bucketed = false;  // (more than 2^31 pairs over more than 2^24 latents)
  p.n_buckets = static_cast<uint32_t>(p.bucketed ? n_buckets : 0);
  p.table_len = p.bucketed ? static_cast<size_t>(n_buckets + 1) * p.n_chunks : 0;
  return p;
}

// Scratch of the pair-list construction, carved out of one workspace:
//   bucketed: tmp[B*K] u32 | table[table_len] | ctrl (kCtrlWords) | long_list[B*K/65 + 1]
//   atomic:   rank[B*K] u32 | scan block sums[ceil(F/kScanBlockElems)] | ctrl | long_list
// The lists besides long_list (chunk_begin, empty_list, cls_list) belong to the caller's workspace.
struct CsrScratch {
  CsrPlan plan;
  uint32_t *tmp;
  uint32_t *table;
  uint32_t *rank;
  uint32_t *block_sums;
  PairLists lists;
};

size_t csr_scan_sums_bytes(int64_t n) {
  return round_up(static_cast<size_t>(ceil_div(n, kScanBlockElems)) * 4, kAlign);
}

size_t csr_scratch_bytes(int64_t n_pairs, int64_t F, CsrScratch *sc, uint8_t *ws) {
  CsrScratch local = {};
  CsrScratch &c = sc ? *sc : local;
  c = CsrScratch{};
  c.plan = plan_csr(n_pairs, F);
  size_t off = 0;
  auto take = [&](auto *&ptr, size_t bytes) {
    ptr = reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(ws + off);
    off += round_up(bytes, kAlign);
  };
  if (c.plan.bucketed) {
    take(c.tmp, static_cast<size_t>(n_pairs) * 4);
    take(c.table, c.plan.table_len * 4);
  } else {
    take(c.rank, static_cast<size_t>(n_pairs) * 4);
    take(c.block_sums, csr_scan_sums_bytes(F));
  }
  static_assert(kCtrlWords * 4 <= kAlign, "the control words are one aligned slot");
  take(c.lists.ctrl, kCtrlWords * 4);
  take(c.lists.long_list, (static_cast<size_t>(n_pairs) / 65 + 1) * 4);
  return off;
}

CsrScratch carve_csr_scratch(void *workspace, int64_t F, int64_t n_pairs) {
  CsrScratch sc;
  csr_scratch_bytes(n_pairs, F, &sc, static_cast<uint8_t *>(workspace));
  return sc;
}

// cleared: the control words are zero already
void launch_pair_lists(const uint32_t *begin, int64_t F, const PairLists &lists, hipStream_t st, bool cleared = false) {
  if (!cleared)
    hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(64), 0, st, lists.ctrl, static_cast<int64_t>(kCtrlWords), 0u);
  hipLaunchKernelGGL(pair_lists_kernel, dim3(static_cast<unsigned>(ceil_div(F, kListLatents))), dim3(1024), 0, st, begin,
                     F, lists);
}

template <bool RECORDS>
void launch_bucket_sort(const CsrScratch &sc, int64_t F, uint32_t *begin, uint32_t *map, uint32_t *slot, uint32_t *hslot,
                        uint32_t solo_bit, const PairLists &lists, const PairRecords &rec, hipStream_t st) {
  const CsrPlan &pl = sc.plan;
  // (of the blocks that share a bucket most return at once)
  const auto kernel =
      pl.n_buckets <= kBucketBlocks / 2 ? csr_bucket_sort_kernel<RECORDS, 4> : csr_bucket_sort_kernel<RECORDS, 8>;
  hipLaunchKernelGGL(kernel, dim3(pl.n_buckets, pl.n_batches), dim3(kSortThreads), 0, st, sc.tmp, sc.table, pl.n_chunks,
                     pl.chunk, pl.shift, pl.pack_shift, F, begin, map, slot, hslot, solo_bit, lists, rec);
}

// begin[F+1], map[B*K] and, when `slot` is given, its inverse slot[B*K] (and a second copy of it in
// `hslot`); fills the lists of sc.lists.
void csr_build_launch(const int64_t *indices, int64_t B, int64_t K, int64_t F, uint32_t *begin,
                      uint32_t *map, uint32_t *slot, uint32_t *hslot, const CsrScratch &sc, int *status_flag,
                      hipStream_t st, uint32_t solo_bit = 0u) {
  const int64_t n_pairs = B * K;
  const CsrPlan &pl = sc.plan;
  if (pl.bucketed) {
    const size_t lds = (round_up(pl.n_buckets, 4) + 1) * kChunkWaves * 4;
    hipLaunchKernelGGL(csr_chunk_sort_kernel, dim3(pl.n_chunks), dim3(kChunkThreads), lds, st, indices, n_pairs, F,
                       pl.shift, pl.pack_shift, pl.n_buckets, pl.n_bits, pl.chunk, pl.n_chunks, sc.table, sc.tmp, sc.lists.ctrl,
                       status_flag);
    launch_bucket_sort<false>(sc, F, begin, map, slot, hslot, solo_bit, sc.lists, PairRecords{}, st);
    return;
  }
  hipLaunchKernelGGL(csr_init_kernel, dim3(grid_for(F + 1, 256, 4096)), dim3(256), 0, st, begin, F + 1,
                     sc.lists.ctrl);
  hipLaunchKernelGGL(csr_count_kernel, dim3(grid_for(n_pairs, 256, 8192)), dim3(256), 0, st,
                     indices, n_pairs, F, begin, sc.rank, status_flag);
  const unsigned scan_blocks = static_cast<unsigned>(ceil_div(F, kScanBlockElems));
  hipLaunchKernelGGL(csr_scan_sums_kernel, dim3(scan_blocks), dim3(kScanThreads), 0, st, begin, F,
                     sc.block_sums);
  hipLaunchKernelGGL(csr_scan_apply_kernel, dim3(scan_blocks), dim3(kScanThreads), 0, st, begin, F,
                     sc.block_sums);
  hipLaunchKernelGGL(csr_fill_kernel, dim3(grid_for(n_pairs, 256, 8192)), dim3(256), 0, st, indices,
                     n_pairs, F, begin, sc.rank, map);
  hipLaunchKernelGGL(csr_sort_short_kernel,
                     dim3(static_cast<unsigned>(ceil_div(F, kWavesPerBlock))), dim3(kBlock), 0, st,
                     begin, map, F, sc.lists.ctrl + kLongCount, sc.lists.long_list);
  hipLaunchKernelGGL(csr_sort_long_kernel, dim3(1024), dim3(1024), 0, st, begin, map, sc.lists.ctrl + kLongCount,
                     sc.lists.long_list, static_cast<uint32_t>(B < (1LL << 31) ? B : 0xffffffffLL),
                     static_cast<uint32_t>(K));
  if (slot)
    hipLaunchKernelGGL(csr_inverse_kernel, dim3(grid_for(n_pairs, 256, 8192)), dim3(256), 0, st, map, n_pairs,
                       slot, hslot);
  if (sc.lists.chunk_begin) launch_pair_lists(begin, F, sc.lists, st);
}

// The lists of a pair list that belong to the caller's workspace (everything but ctrl and long_list): their bytes, and
// their places in `base` if that is given.  classes: the lists by number of pairs too.
size_t carve_pair_lists(size_t n_pairs, size_t F, bool classes, void *base, PairLists *ls) {
  size_t off = 0;
  auto take = [&](uint32_t *&ptr, size_t entries) {
    if (base) ptr = reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(base) + off);
    off += round_up(entries * 4, kAlign);
  };
  PairLists none = {};
  PairLists &l = ls ? *ls : none;
  take(l.chunk_begin, n_pairs / 65 + 1);
  if (!classes) return off;
  take(l.empty_list, F);
  for (int i = 0; i < kClasses; ++i) {
    const size_t most = n_pairs / ((size_t{1} << i) / 2 + 1);
    take(l.cls_list[i], (most < F ? most : F) + 1);
  }
  return off;
}

// Columns per tile of the training-step kernel: one register per gathered row piece, so 16-bit
// weights take two columns per lane (128-column tiles) and fp32 weights one once K exceeds 64.
inline int64_t train_tile_cols(const flexsae_shape *s) {
  return (s->weight_dtype == FLEXSAE_F32 && s->K > 64) ? 64 : 128;
}

// ---- two-phase hierarchical backward: workspace plan -----------------------------------

// Most latents without a pair, the rest with few: the reduction by pieces then works from the lists
// of latents by row count and the rows of latents without pairs are zeroed in one pass.
// Whether that pays depends on how many latents really are without a pair: with two pairs per latent
// on average it does for skewed indices (two thirds of the latents empty: the step a sixth faster) and
// does not for uniform ones (an eighth of them empty: the step 8 % slower).  Only the caller can know,
// from an earlier step: FLEXSAE_BWD_DENSE_LATENTS says "most latents have pairs".
inline bool sparse_latents(const flexsae_shape *s, int flags = 0) {
  return !(flags & FLEXSAE_BWD_DENSE_LATENTS) && s->B * s->K <= 2 * s->F;
}

struct HierBwdPlan {
  int vec;                 // columns per lane
  int tile;                // 64 * vec columns per wavefront
  size_t p_size;           // bytes per element of the contribution matrix P
  int64_t d_pad;           // D rounded up to a whole number of tiles
  size_t n_pairs;          // B * K
  size_t n_rows;           // B
  size_t n_partial_rows;   // upper bound on the number of 64-pair chunks of long latents
  size_t off_begin, off_map, off_slot, off_csr, off_lists, off_sfinal, off_colsum, off_loss, off_dvpart, off_partial;  // per-slice buffers follow
  size_t n_loss_partials;  // training-step kernel: one per (tile of 64 or 128 columns, row)
  size_t fixed_bytes;      // everything that does not depend on the slice width
  // hot-latent tables (only with `hot`): slots with the hot pairs marked, control words, the hot
  // latents, the candidates and what became of them, the long latents that stayed cold and their
  // chunk table
  bool hot;
  size_t off_hslot, off_hot_steps, off_hot_ctrl, off_hot_list, off_cand_list, off_long2, off_chunk2;
  int hot_rows;            // rows per block of the accumulator kernel
  size_t n_row_blocks;     // blocks of that many rows
};

// Hot-latent accumulators: 16-bit weights of at most 64 steps (one register per row piece, four
// wavefronts per SIMD next to 144 KiB of accumulators) whose slices the piece reduction serves, and
// pair numbers below the walk's mark of a latent's only pair (kSoloSlotBit).
inline bool hot_supported(const flexsae_shape *s) {
  return s->D % 4 == 0 && s->K <= 64 && s->weight_dtype != FLEXSAE_F32 &&
         s->D % (s->weight_dtype == FLEXSAE_BF16 ? 8 : 4) == 0 && s->B * s->K < (1LL << 30);
}

HierBwdPlan plan_hier_bwd(const flexsae_shape *s, bool hot = false, int flags = 0) {
  HierBwdPlan p;
  p.vec = (s->D % 4 == 0) ? 4 : (s->D % 2 == 0) ? 2 : 1;
  p.tile = kWave * p.vec;
  p.p_size = (s->weight_dtype == FLEXSAE_BF16) ? 2 : 4;  // bf16 weights: bf16 contributions
  p.d_pad = ceil_div(s->D, p.tile) * p.tile;
  p.n_pairs = static_cast<size_t>(s->B) * static_cast<size_t>(s->K);
  p.n_rows = static_cast<size_t>(s->B);
  p.n_partial_rows = p.n_pairs / kSegChunk + p.n_pairs / 65 + 2;
  size_t off = 0;
  p.off_begin = off;
  off += round_up(static_cast<size_t>(s->F + 1) * 4, kAlign);
  p.off_map = off;
  off += round_up(p.n_pairs * 4, kAlign);
  p.off_slot = off;
  off += round_up(p.n_pairs * 4, kAlign);
  p.off_csr = off;
  off += flexsae_csr_workspace_bytes(s->B, s->K, s->F);
  p.off_lists = off;
  off += carve_pair_lists(p.n_pairs, static_cast<size_t>(s->F), sparse_latents(s), nullptr, nullptr);
  p.off_sfinal = off;  // S_{b,0} of every row, [B, d_pad] fp32: dbias is its column sum
  off += round_up(p.n_rows * static_cast<size_t>(p.d_pad) * 4, kAlign);
  p.off_colsum = off;  // partial column sums, [ceil(B/64), D] fp32
  // (with hot latents one per row block, however small the flags make those)
  off += round_up(static_cast<size_t>(ceil_div(s->B, hot ? kHotMinRowsPerBlock : kColsumRows)) * static_cast<size_t>(s->D) * 4,
                  kAlign);
  p.off_loss = off;
  p.n_loss_partials = p.n_rows * static_cast<size_t>(p.d_pad / 64 + 1);
  off += round_up(p.n_loss_partials * 4, kAlign);
  // per-tile shares of dvals, [number of tiles, B*K] fp32, added up in tile order afterwards
  // (tiles are 64 or 128 columns in the training-step kernel, 64*vec in the sweep kernel)
  p.off_dvpart = off;
  const int64_t tt = train_tile_cols(s);
  off += round_up(static_cast<size_t>(p.d_pad / (p.tile < tt ? p.tile : tt)) * p.n_pairs * 4, kAlign);
  p.hot = hot;
  p.hot_rows = kHotRowsPerBlock >> hot_halvings(flags);
  p.n_row_blocks = static_cast<size_t>(ceil_div(s->B, p.hot_rows));
  if (hot) {
    const size_t n_long_max = p.n_pairs / 65 + 2;
    p.off_hslot = off;
    off += round_up(p.n_pairs * 4, kAlign);
    p.off_hot_steps = off;  // what the walk reads of a row: hot_row_words words
    off += round_up(p.n_rows * hot_row_words(hot_kmax(s->K)) * 4, kAlign);
    p.off_hot_ctrl = off;
    off += round_up(kHotCtrlWords * 4, kAlign);
    p.off_hot_list = off;
    off += round_up(kHotMax * 4, kAlign);
    p.off_cand_list = off;
    off += round_up(kHotMax * 4, kAlign);
    p.off_long2 = off;
    off += round_up(n_long_max * 4, kAlign);
    p.off_chunk2 = off;
    off += round_up(n_long_max * 4, kAlign);
  }
  p.off_partial = off;
  p.fixed_bytes = off;
  return p;
}

// The pair-list scratch and lists of a hierarchical workspace, the lists by number of pairs only where a call with
// these flags reduces from them.
CsrScratch carve_hier_lists(const flexsae_shape *s, const HierBwdPlan &pl, uint8_t *ws, int flags = 0) {
  CsrScratch sc = carve_csr_scratch(ws + pl.off_csr, s->F, s->B * s->K);
  carve_pair_lists(pl.n_pairs, static_cast<size_t>(s->F), sparse_latents(s, flags), ws + pl.off_lists, &sc.lists);
  return sc;
}

// Slice granule (columns) of the training step.  The training-step kernel works on tiles of
// train_tile_cols(); when dW rows can be written 16 bytes per lane, the reduction works on
// 256-byte pieces of P (seg_reduce_piece_kernel) and a slice may be any number of training tiles
// wide; otherwise slices are whole reduction tiles (64 * vec columns).
inline int64_t piece_cols(const HierBwdPlan &p) { return kPieceBytes / static_cast<int64_t>(p.p_size); }

inline bool piece_reduce_ok(const flexsae_shape *s, const HierBwdPlan &p, const void *dW, int dW_dtype) {
  const int64_t ev = 16 / static_cast<int64_t>(p.p_size);  // columns per lane of the piece reduction
  return s->D % ev == 0 && train_tile_cols(s) % piece_cols(p) == 0 &&
         (dW == nullptr || aligned(dW, static_cast<size_t>(ev) * dtype_size(dW_dtype)));
}

// The same for the training step: rows that allow no 8- or 16-byte access of their own elements are reduced by pieces, which
// are read 16 bytes per lane whatever D is and written in dword-aligned vectors or by elements.
inline bool train_piece_ok(const flexsae_shape *s, const HierBwdPlan &p, const void *dW, int dW_dtype) {
  return p.vec < 4 ? train_tile_cols(s) % piece_cols(p) == 0 : piece_reduce_ok(s, p, dW, dW_dtype);
}

// Columns the slice loop works on: D rounded up to whole reduction tiles, or to whole training tiles
// when the piece reduction lets slices end there.
inline int64_t hier_cols_used(const flexsae_shape *s, const HierBwdPlan &p, bool train, bool piece) {
  if (!(train && piece)) return p.d_pad;
  const int64_t tt = train_tile_cols(s);
  return ceil_div(s->D, tt) * tt;
}

// Forward-only inputs of the training-step variant of the slice loop (null = plain backward).
struct TrainArgs {
  const void *bias;
  const void *target;
  float *loss;              // finished by the epilogue from the per-(tile, row) partials
  int64_t n_loss_partials;
  double inv_count;         // 1 / (B*K*D)
  PairStats stats;          // likewise
};

// what of slot[] is the slot: all of it, or all but the mark of a latent's only pair
inline bool solo_marks(const flexsae_shape *s) { return s->B * s->K < (1LL << 30); }
inline uint32_t slot_mask(const flexsae_shape *s) { return solo_marks(s) ? kSoloSlotBit - 1u : 0xffffffffu; }

// largest K the training-step kernel holds in registers
inline bool train_supported(const flexsae_shape *s, int flags = 0) {
  if (s->K > 256) return false;
  // FLEXSAE_BWD_RAGGED_ROWS: any row that a lane's columns divide (two, or one for fp32 rows of more than 64 steps)
  if (flags & FLEXSAE_BWD_RAGGED_ROWS) return s->D % 2 == 0 || train_tile_cols(s) == kWave;
  return s->D % 4 == 0;
}

// Row pieces the training-step kernel keeps in the LDS instead of registers (one dword per lane
// and row: 16-bit weights with two columns per lane, fp32 with one), chosen so that one more
// wavefront fits each SIMD: 256 steps 222-224 registers, two wavefronts (280-284 and one with all pieces in
// registers; 16 KB of LDS each), 128 steps 120-122, four (146-150, three; 8 KB each), 64 steps 63, eight
// (80, six).
#ifndef FLEXSAE_LDS_256
#define FLEXSAE_LDS_256 64
#endif
#ifndef FLEXSAE_LDS_128
#define FLEXSAE_LDS_128 32
#endif
#ifndef FLEXSAE_LDS_64
#define FLEXSAE_LDS_64 16
#endif
template <typename WT, int KMAX, int VEC>
constexpr int train_lds_rows() {
  if (VEC * sizeof(typename Traits<WT>::store_t) != 4) return 0;
  return KMAX == 256 ? FLEXSAE_LDS_256 : KMAX == 128 ? FLEXSAE_LDS_128 : KMAX == 64 ? FLEXSAE_LDS_64 : 0;
}

template <typename WT, typename PT, int KMAX, int VEC = 2>
void launch_train_kernel(const flexsae_shape *s, const TrainArgs &ta, const int64_t *indices,
                         const void *weight, const void *vals, float coef, const uint32_t *slot, void *P,
                         float *dvals, float *s_final, int d_pad, float *loss_partial, int *status_flag,
                         int64_t cols, int col0, int slice_w, hipStream_t st, const HotFinalize &fin, void *dW_solo,
                         const ZeroRows &zero) {
  constexpr int LDSROWS = train_lds_rows<WT, KMAX, VEC>();
  const int64_t n_items = s->B * (cols / (kWave * VEC));
  // K == KMAX (the usual powers of two) runs the variant without per-step bound tests, part of its
  // row pieces in the LDS
  const bool stream = slice_w >= d_pad;  // all of P in one launch: streaming stores
  // Tiles of a row one after the other where there are too few rows for the wavefronts on the chip (4096) to share the pieces
  // of one tile anyway: what is gathered and stored of a row then lies side by side.  us of the step by tile / by row: B=1024,
  // K=64, F=65536, D=4096 bf16 407 / 387, B=128, K=128, F=16384, D=2048 73 / 66, B=512, K=64, F=65536, D=2048 fp32 274 / 255,
  // B=207, K=90, F=68238, D=2348 fp16 228 / 224, B=1777, K=50, F=24571, D=1538 193 / 187; not B=2048, K=64, F=32768, D=1024 bf16
  // 165 / 167, B=4096, K=128, F=65536, D=2304 1224 / 1257, nor in slices where latents repeat, B=1024, K=100, F=40000, D=2304
  // 318 / 323.
  const bool by_row = s->B < 2048 && (slice_w >= s->D || s->B * s->K <= s->F);
  const int row_tiles = by_row ? static_cast<int>(cols / (kWave * VEC)) : 0;
  const auto kernel = s->K == KMAX
                          ? (stream ? hier_train_kernel<WT, PT, KMAX, true, true, VEC, LDSROWS>
                                    : hier_train_kernel<WT, PT, KMAX, true, false, VEC, LDSROWS>)
                          : (stream ? hier_train_kernel<WT, PT, KMAX, false, true, VEC, 0>
                                    : hier_train_kernel<WT, PT, KMAX, false, false, VEC, 0>);
  hipLaunchKernelGGL(kernel, dim3(fin.n_blocks + static_cast<unsigned>(ceil_div(n_items, kWavesPerBlock)) + zero.n_blocks),
                     dim3(kBlock), 0, st, indices, weight, vals, s->vals_dtype, ta.bias, s->bias_dtype, ta.target, s->target_dtype,
                     coef, slot, P, dvals, s_final, d_pad, loss_partial, status_flag, n_items, s->B, row_tiles, col0,
                     slice_w, static_cast<int>(s->K), s->F, static_cast<int>(s->D), slot_mask(s), dW_solo, fin, zero);
}

template <typename WT, typename PT>
void launch_train_kernel_k(const flexsae_shape *s, const TrainArgs &ta, const int64_t *indices,
                           const void *weight, const void *vals, float coef, const uint32_t *slot, void *P,
                           float *dvals, float *s_final, int d_pad, float *loss_partial,
                           int *status_flag, int64_t cols, int col0, int slice_w, hipStream_t st,
                           const HotFinalize &fin, void *dW_solo, const ZeroRows &zero) {
#define FLEXSAE_TRAIN(KM)                                                                              \
  launch_train_kernel<WT, PT, KM>(s, ta, indices, weight, vals, coef, slot, P, dvals, s_final, d_pad,  \
                                  loss_partial, status_flag, cols, col0, slice_w, st, fin, dW_solo, zero)
  // (the fp32 16-step instantiation allocates registers badly; 32 covers it)
  if (s->K <= 16 && sizeof(typename Traits<WT>::store_t) == 2) {
    FLEXSAE_TRAIN(16);
  } else if (s->K <= 32) {
    FLEXSAE_TRAIN(32);
  } else if (s->K <= 64) {
    FLEXSAE_TRAIN(64);
  } else if constexpr (sizeof(typename Traits<WT>::store_t) == 2) {
    if (s->K <= 128) {
      FLEXSAE_TRAIN(128);
    } else {  // 129..256 steps: two wavefronts per SIMD with 64 rows in the LDS (K = 256), else one
      FLEXSAE_TRAIN(256);
    }
  } else if (s->K <= 128) {  // fp32 rows of 65..128 steps: one column per lane
    launch_train_kernel<WT, PT, 128, 1>(s, ta, indices, weight, vals, coef, slot, P, dvals, s_final, d_pad,
                                        loss_partial, status_flag, cols, col0, slice_w, st, fin, dW_solo, zero);
  } else {
    launch_train_kernel<WT, PT, 256, 1>(s, ta, indices, weight, vals, coef, slot, P, dvals, s_final, d_pad,
                                        loss_partial, status_flag, cols, col0, slice_w, st, fin, dW_solo, zero);
  }
#undef FLEXSAE_TRAIN
}

// The training-step kernel with hot-latent accumulators (16-bit weights, K <= 64): one block per
// (row block, 128-column tile); every block first takes its share of the previous slice's second steps.
template <typename WT, typename PT>
void launch_train_hot_kernel(const flexsae_shape *s, const TrainArgs &ta, const uint32_t *steps, bool off32,
                             const void *weight, float coef, void *P, float *dvals, float *colsum_part, float *loss_partial,
                             int64_t cols, int col0, int slice_w, hipStream_t st, HotFinalize fin,
                             const HotBlockFinalize &hfin, uint32_t *ctrl, float *hot_partial,
                             int hot_rows, int n_row_blocks, int headroom, void *dW_solo) {
  if constexpr (sizeof(typename Traits<WT>::store_t) == 2) {
    const int n_tiles = static_cast<int>(cols / kHotCols);
    const unsigned grid = static_cast<unsigned>(n_tiles) * static_cast<unsigned>(n_row_blocks);
    if (fin.mode != 0) fin.n_blocks = grid;  // every block takes a share
#define FLEXSAE_TRAIN_HOT(KM)                                                                                   \
  do {                                                                                                          \
    const auto kernel = s->K == KM ? (off32 ? hier_train_hot_kernel<WT, PT, KM, true, true>                     \
                                            : hier_train_hot_kernel<WT, PT, KM, true, false>)                   \
                                   : (off32 ? hier_train_hot_kernel<WT, PT, KM, false, true>                    \
                                            : hier_train_hot_kernel<WT, PT, KM, false, false>);                 \
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kHotThreads), 0, st, steps, weight, ta.bias, s->bias_dtype, ta.target, \
                       s->target_dtype, coef, P, dvals, colsum_part, loss_partial, s->B, n_tiles, n_row_blocks, col0, \
                       slice_w, static_cast<int>(s->K), s->F, static_cast<int>(s->D), ctrl, hot_partial, headroom, \
                       hot_rows / kHotWaves, dW_solo, fin, hfin);                                               \
  } while (0)
    if (s->K <= 16) {
      FLEXSAE_TRAIN_HOT(16);
    } else if (s->K <= 32) {
      FLEXSAE_TRAIN_HOT(32);
    } else {
      FLEXSAE_TRAIN_HOT(64);
    }
#undef FLEXSAE_TRAIN_HOT
  }
}

// per-slice buffers after the fixed part: chunk partials[n_partial_rows, w] | P[B*K, w]
size_t hier_partial_bytes(const HierBwdPlan &p, int64_t slice_w) {
  return round_up(p.n_partial_rows * static_cast<size_t>(slice_w) * 4, kAlign);
}

size_t hier_p_bytes(const HierBwdPlan &p, int64_t slice_w) {
  return round_up(p.n_pairs * static_cast<size_t>(slice_w) * p.p_size, kAlign);
}

// one buffer of block partials of the hot latents: [tiles of the slice][row blocks][kHotMax][128] fp32
size_t hier_hot_partial_bytes(const HierBwdPlan &p, int64_t slice_w) {
  return round_up(static_cast<size_t>(ceil_div(slice_w, kHotCols)) * p.n_row_blocks * kHotMax * kHotCols * 4, kAlign);
}

// ... | chunk partials | P | (hot: two buffers of block partials, used by alternate slices)
size_t hier_bwd_bytes(const HierBwdPlan &p, int64_t slice_w) {
  return p.fixed_bytes + hier_partial_bytes(p, slice_w) + hier_p_bytes(p, slice_w) +
         (p.hot ? 2 * hier_hot_partial_bytes(p, slice_w) : 0);
}

// every row starts at a multiple of four bytes
inline int rows_on_dwords(const void *rows, int64_t D, size_t elem) { return aligned(rows, 4) && D * elem % 4 == 0; }

// Segment reduction of one slice plus the finalize step of its hot latents.  fp32 contributions
// are read 16 bytes per lane (256-column tiles), or, when `narrow`, 8 bytes per lane (128-column
// tiles, twice the wavefronts): faster once a latent has about four rows or more, slower for
// shorter groups.
template <typename PT, typename GT, int VEC>
void launch_seg_reduce(bool narrow, const uint32_t *begin, const LongList &ll, const PairLists &ls,
                       const void *P, float *partial, void *dW, const float *dw_scale, int64_t F, int tps,
                       int col0, int sw, int D, hipStream_t st, int piece_cols = 0, int64_t cols = 0, int64_t n_pairs = 0,
                       int update = 0, bool by_count = false, HotFinalize *defer = nullptr, int skip_solo = 0) {
  const int dwords = rows_on_dwords(dW, D, sizeof(typename Traits<GT>::store_t));
  // the second step of the hot latents: launched here, or handed back through `defer` for the next
  // training-step launch to carry
  auto finalize = [&](int mode, int units) {
    HotFinalize h = {ll.ctrl, ll.list, ll.chunk_begin, partial, dW, dw_scale, mode, units, col0, sw, D, update, dwords, 0, 256u};
    if (defer) {
      h.n_blocks = 64u;  // riding along with a long launch: few blocks, so that they cost little where there is nothing to do
      *defer = h;
    }
    else
      hipLaunchKernelGGL((hot_finalize_kernel<GT>), dim3(h.n_blocks), dim3(kBlock), 0, st, h);
  };
  if (piece_cols > 0) {  // 256-byte pieces, sixteen lanes each
    const int how = (update ? kReduceUpdate : 0) | (skip_solo ? kReduceSkipSolo : 0) | (dwords ? kReduceDwords : 0);
    const int pps = static_cast<int>(ceil_div(cols, piece_cols));
    int pps_shift = -1;  // log2(pps) when pps is a power of two
    for (int sh = 0; sh < 16; ++sh)
      if (pps == (1 << sh)) pps_shift = sh;
    // latents per group of lanes: four, taken from the lists by row count, where most latents
    // have no or few rows (with four rows per latent on average the bookkeeping already costs more
    // than the shorter launch saves); the lists hold at most min(F, pairs) latents with rows
#define FLEXSAE_PIECE_REDUCE(G, N_BLOCKS, LISTS)                                                                       \
  hipLaunchKernelGGL((seg_reduce_piece_kernel<PT, GT, FLEXSAE_PIECE_U, G>),                                        \
                     dim3(kLongBlocks + static_cast<unsigned>(N_BLOCKS)), dim3(kBlock), 0, st, begin, ll.ctrl, ll.list, \
                     ll.chunk_begin, P, partial, dW, dw_scale, F, kLongBlocks, pps, pps_shift, col0, sw, D, how, LISTS)
    constexpr int64_t kGroups = kBlock / kPieceLanes;
    if (by_count) {
      // work items: one per latent with nine rows or more, one per four others of a class
      const int64_t n_listed_max = F < n_pairs ? F : n_pairs;
      const int64_t n_items_max = (n_pairs / 9 + ceil_div(n_listed_max, 4) + kClasses) * pps;
      const int64_t n_blocks = ceil_div(n_items_max, kGroups);
      FLEXSAE_PIECE_REDUCE(4, (n_blocks < kListBlocks ? n_blocks : kListBlocks), ls);
    } else {
      FLEXSAE_PIECE_REDUCE(1, ceil_div(F * pps, kGroups), NoLists{});
    }
#undef FLEXSAE_PIECE_REDUCE
    // the chunk partials of hot latents are combined per 64-column piece
    finalize(1, static_cast<int>(cols / kWave));
    return;
  }
  constexpr bool kCanNarrow = sizeof(typename Traits<PT>::store_t) == 4 && VEC == 4;
  if (kCanNarrow && narrow) {
    constexpr int RV = kCanNarrow ? 2 : VEC;
    const int rtps = tps * (VEC / RV);
    const unsigned n_short_blocks = static_cast<unsigned>(ceil_div(F * rtps, kWavesPerBlock));
    hipLaunchKernelGGL((seg_reduce_kernel<PT, GT, RV, FLEXSAE_REDUCE_U>), dim3(kLongBlocks + n_short_blocks),
                       dim3(kBlock), 0, st, begin, ll.ctrl, ll.list, ll.chunk_begin, P, partial, dW, dw_scale,
                       F, kLongBlocks, rtps << 1 | skip_solo, col0, sw, D);
    static_assert(RV == 2 || !kCanNarrow, "the narrow reduction works on tiles of 128 columns");
    finalize(3, rtps);
    return;
  }
  const unsigned n_short_blocks = static_cast<unsigned>(ceil_div(F * tps, kWavesPerBlock));
  hipLaunchKernelGGL((seg_reduce_kernel<PT, GT, VEC, FLEXSAE_REDUCE_U>), dim3(kLongBlocks + n_short_blocks),
                     dim3(kBlock), 0, st, begin, ll.ctrl, ll.list, ll.chunk_begin, P, partial, dW, dw_scale, F,
                     kLongBlocks, tps << 1 | skip_solo, col0, sw, D);
  if constexpr (VEC == 4) {
    finalize(2, tps);
  } else {
    hipLaunchKernelGGL((seg_reduce_long_finalize_kernel<GT, VEC, 8>), dim3(256), dim3(kBlock), 0, st, ll.ctrl,
                       ll.list, ll.chunk_begin, partial, dW, dw_scale, tps, col0, sw, D);
  }
}

template <typename WT, typename PT, typename GT, int VEC>
void launch_hier_slices(const flexsae_shape *s, const HierBwdPlan &pl, int64_t slice_w,
                        const int64_t *indices, const void *weight, const void *vals,
                        const float *resid, const float *grad_out, float coef, void *dW,
                        float *dvals, float *dbias, uint8_t *ws, int flags, int *status_flag,
                        hipStream_t st, const TrainArgs *train = nullptr, int piece = 0) {
  const bool do_sweep = !(flags & FLEXSAE_BWD_REDUCE_ONLY);
  const bool do_reduce = !(flags & FLEXSAE_BWD_SWEEP_ONLY);
  // in-place weight update: `grad_out` is the step size and dW the weight matrix (piece reduction only)
  const int update = (flags & kBwdSgdUpdate) ? 1 : 0;
  const float *dw_scale = (flags & (FLEXSAE_BWD_SCALE_BY_GRAD_OUT | kBwdSgdUpdate | kBwdScaled)) ? grad_out : nullptr;
  const uint32_t *begin = reinterpret_cast<const uint32_t *>(ws + pl.off_begin);
  const uint32_t *slot = reinterpret_cast<const uint32_t *>(ws + pl.off_slot);
  const CsrScratch sc = carve_hier_lists(s, pl, ws);
  float *s_final = reinterpret_cast<float *>(ws + pl.off_sfinal);
  float *dv_part = reinterpret_cast<float *>(ws + pl.off_dvpart);
  float *colsum_part = reinterpret_cast<float *>(ws + pl.off_colsum);
  const int d_pad = static_cast<int>(pl.d_pad);
  const int K = static_cast<int>(s->K), D = static_cast<int>(s->D);
  const int sw = static_cast<int>(slice_w);
  const bool narrow_reduce = s->B * s->K >= 4 * s->F;
  float *partial = reinterpret_cast<float *>(ws + pl.off_partial);
  void *P = ws + pl.off_partial + hier_partial_bytes(pl, slice_w);
  // Hot latents (training step only): their pairs are marked in hslot and accumulated by the
  // training-step kernel; the chunked part of the reduction then serves the long latents that stayed
  // cold, from a list and a chunk table of their own.
  const bool hot = (flags & kBwdHot) != 0 && pl.hot && train != nullptr;
  uint32_t *hot_ctrl = hot ? reinterpret_cast<uint32_t *>(ws + pl.off_hot_ctrl) : nullptr;
  const uint32_t *hot_list = hot ? reinterpret_cast<const uint32_t *>(ws + pl.off_hot_list) : nullptr;
  float *hot_partial[2] = {nullptr, nullptr};
  // the long latents the reduction serves
  LongList reduce_long = {sc.lists.ctrl, sc.lists.long_list, sc.lists.chunk_begin};
  if (hot) {
    uint8_t *base = static_cast<uint8_t *>(P) + hier_p_bytes(pl, slice_w);
    hot_partial[0] = reinterpret_cast<float *>(base);
    hot_partial[1] = reinterpret_cast<float *>(base + hier_hot_partial_bytes(pl, slice_w));
    reduce_long = {hot_ctrl + kHotLong2, reinterpret_cast<uint32_t *>(ws + pl.off_long2),
                   reinterpret_cast<uint32_t *>(ws + pl.off_chunk2)};
  }
  const int hot_headroom = (flags & FLEXSAE_BWD_HOT_NO_HEADROOM) ? -6 : 2;
  // columns that are worked on: whole reduction tiles, or, with the piece reduction, whole training
  // tiles (tiles that lie entirely beyond column D are left out, and so are their shares below)
  const int64_t d_used = hier_cols_used(s, pl, train != nullptr, piece != 0);
  // The sweep kernel's tile (64 * sweep_vec columns per wavefront): narrower than the reduction's
  // when a slice would otherwise hold too few wavefronts to cover the memory latency (small B).
  // (not below the tile width the per-tile dvals shares of the workspace are laid out for)
  int sweep_vec = VEC;
  const int min_sweep_vec = static_cast<int>((pl.tile < train_tile_cols(s) ? pl.tile : train_tile_cols(s)) / kWave);
  while (sweep_vec > 1 && sweep_vec > min_sweep_vec && s->B * (slice_w / (kWave * sweep_vec)) < 6144) sweep_vec >>= 1;
  // Sparse shapes reduce every slice by pieces from the lists of latents by row count; the
  // rows of latents without pairs are zeroed here, whole rows in one pass (the in-place update leaves
  // them alone).
  const bool sparse = piece != 0 && sparse_latents(s, flags);
  // (by the first blocks of the first walk, where that is hier_train_kernel)
  ZeroRows zero = {};
  if (sparse && do_reduce && !update) {
    const unsigned n_zero_blocks = static_cast<unsigned>(ceil_div(s->F, kZeroRows * kWavesPerBlock));
    const int dwords = rows_on_dwords(dW, D, sizeof(typename Traits<GT>::store_t));
    if (train && do_sweep && !hot)
      zero = {sc.lists.ctrl, sc.lists.empty_list, dW, sizeof(typename Traits<GT>::store_t) == 4, dwords, n_zero_blocks};
    else
      hipLaunchKernelGGL((seg_zero_rows_kernel<GT>), dim3(n_zero_blocks), dim3(kBlock), 0, st, sc.lists.ctrl,
                         sc.lists.empty_list, dW, D, dwords);
  }
  // In the training step the second step of a slice's hot latents travels with the next slice's
  // training-step launch (a gradient of CarriedGrad's type; by pieces, the weight's: that is what that kernel
  // writes; a launch of its own costs 4.7 us a slice); the last slice's gets one.
  HotFinalize pending = {};
  HotBlockFinalize pending_hot = {};
  // (the sweep of the plain backward carries it for a gradient of the weight's type)
  constexpr bool carried = std::is_same<GT, typename CarriedGrad<WT>::type>::value;
  constexpr bool weight_typed = std::is_same<GT, WT>::value && !carried;
  const bool fold = (train && !update ? carried || weight_typed : std::is_same<GT, WT>::value) && do_sweep && do_reduce;
  // Only pairs of their latents write dW themselves where its type is the contributions' own.
  void *const dW_solo = (flags & kBwdSolo) && std::is_same<GT, PT>::value && train != nullptr && do_sweep && do_reduce &&
                                !update && !dw_scale
                            ? dW
                            : nullptr;
  // 32-bit byte offsets from one descriptor per matrix where the matrices allow it
  const bool hot_off32 = s->D % kHotCols == 0 && sw % kHotCols == 0 &&
                         static_cast<uint64_t>(s->F) * s->D * sizeof(typename Traits<WT>::store_t) < (uint64_t{1} << 32) &&
                         static_cast<uint64_t>(s->B) * s->K * slice_w * sizeof(typename Traits<PT>::store_t) < (uint64_t{1} << 31);
  if (hot && do_sweep)
    hipLaunchKernelGGL(hot_steps_kernel, dim3(static_cast<unsigned>(ceil_div(s->B, kWavesPerBlock))), dim3(kBlock), 0, st, indices,
                       vals, s->vals_dtype, reinterpret_cast<const uint32_t *>(ws + pl.off_hslot), s->B, K, hot_kmax(s->K), s->F,
                       slot_mask(s), dW_solo != nullptr, hot_off32,
                       static_cast<uint32_t>(s->D * sizeof(typename Traits<WT>::store_t)),
                       static_cast<uint32_t>(slice_w * sizeof(typename Traits<PT>::store_t)),
                       reinterpret_cast<uint32_t *>(ws + pl.off_hot_steps), status_flag);
  int slice_no = 0;
  for (int64_t col0 = 0; col0 < s->D; col0 += slice_w, ++slice_no) {
    const int64_t cols = (d_used - col0) < slice_w ? (d_used - col0) : slice_w;
    const int tps = static_cast<int>(cols / pl.tile);
    if (train && do_sweep && hot) {
      launch_train_hot_kernel<WT, PT>(s, *train, reinterpret_cast<const uint32_t *>(ws + pl.off_hot_steps), hot_off32, weight,
                                      coef, P, dv_part, colsum_part, reinterpret_cast<float *>(ws + pl.off_loss), cols,
                                      static_cast<int>(col0), sw, st, pending, pending_hot, hot_ctrl,
                                      hot_partial[slice_no & 1], pl.hot_rows, static_cast<int>(pl.n_row_blocks), hot_headroom,
                                      dW_solo);
      pending = HotFinalize{};
      pending_hot = HotBlockFinalize{};
    } else if (train && do_sweep) {
      launch_train_kernel_k<WT, PT>(s, *train, indices, weight, vals, coef, slot, P, dv_part, s_final, d_pad,
                                    reinterpret_cast<float *>(ws + pl.off_loss), status_flag, cols,
                                    static_cast<int>(col0), sw, st, pending, dW_solo, zero);
      pending = HotFinalize{};
      zero = ZeroRows{};
    } else if (do_sweep) {
#define FLEXSAE_SWEEP(SV)                                                                                      \
  hipLaunchKernelGGL((hier_sweep_kernel<WT, PT, SV, FLEXSAE_SWEEP_U>),                                         \
                     dim3(pending.n_blocks +                                                                   \
                          static_cast<unsigned>(ceil_div(s->B * (cols / (kWave * SV)), kWavesPerBlock))),      \
                     dim3(kBlock), 0, st, indices, weight, vals, s->vals_dtype, resid, grad_out, coef, slot, P, \
                     dv_part, s_final, d_pad, status_flag, s->B * (cols / (kWave * SV)), s->B,                 \
                     static_cast<int>(col0), sw, K, s->F, D, slot_mask(s), pending)
      if (sweep_vec == VEC) {
        FLEXSAE_SWEEP(VEC);
      } else if (sweep_vec == (VEC >= 2 ? VEC / 2 : 1)) {
        FLEXSAE_SWEEP((VEC >= 2 ? VEC / 2 : 1));
      } else {
        FLEXSAE_SWEEP(1);
      }
#undef FLEXSAE_SWEEP
      pending = HotFinalize{};
    }
    if (!do_reduce) continue;
    // Pieces where rows allow no 8- or 16-byte access of their own elements (a piece of contributions is read 16
    // bytes per lane whatever D is), where the slice is not made of whole reduction tiles, where most latents are empty
    // (four latents per group of lanes), for the in-place update, and where a slice of
    // contributions is about the size of the memory-side cache (measured 1 % faster there); else one
    // wavefront per (latent, reduction tile), which wastes no load slots on the unequal row counts
    // of the four latents a wavefront would otherwise share (4 % faster on slices read from HBM).
    const bool cache_sized = static_cast<size_t>(s->B * s->K) * static_cast<size_t>(sw) * pl.p_size <= (size_t{384} << 20);
    const bool by_pieces =
        piece != 0 && (update || pl.vec < 4 || cols % pl.tile != 0 || sparse_latents(s, flags) || cache_sized);
    launch_seg_reduce<PT, GT, VEC>(narrow_reduce, begin, reduce_long, sc.lists, P, partial, dW, dw_scale, s->F, tps,
                                   static_cast<int>(col0), sw, D, st, by_pieces ? piece : 0, cols, s->B * s->K, update,
                                   sparse, fold && (!train || carried || by_pieces) ? &pending : nullptr, dW_solo != nullptr);
    pending.weight_typed = weight_typed;
    if (hot) {
      // the block partials of the slice's hot latents are added up by the next training-step launch
      // (they live in the buffer that launch does not write), or here
      const HotBlockFinalize h = {hot_ctrl, hot_list, hot_partial[slice_no & 1], dW, dw_scale,
                                  static_cast<int>(cols / kHotCols), static_cast<int>(pl.n_row_blocks),
                                  static_cast<int>(col0), D, update, weight_typed};
      if (fold)
        pending_hot = h;
      else
        hipLaunchKernelGGL((hot_block_finalize_kernel<GT>), dim3(256), dim3(kBlock), 0, st, h);
    }
  }
  // What is left goes into one launch, unless this call ends with its reductions.
  const bool with_epilogue = do_sweep && (do_reduce || train) && !(flags & FLEXSAE_BWD_SKIP_EPILOGUE);
  if (!with_epilogue) {
    if (pending.n_blocks != 0) {
      pending.n_blocks = 256u;
      hipLaunchKernelGGL((hot_finalize_kernel<GT>), dim3(pending.n_blocks), dim3(kBlock), 0, st, pending);
    }
    if (pending_hot.ctrl != nullptr)
      hipLaunchKernelGGL((hot_block_finalize_kernel<GT>), dim3(256), dim3(kBlock), 0, st, pending_hot);
    return;  // (with !do_reduce && !train a measurement aid of the plain backward: sweep kernels only)
  }
  if (pending.n_blocks != 0) pending.n_blocks = 64u;  // of 1024 threads
  const unsigned n_hot_blocks = pending_hot.ctrl != nullptr ? 64u : 0u;
  // (the hot-latent training step has formed stage 1 of the column sums on chip, one partial per row block)
  const int n_chunks = static_cast<int>(ceil_div(s->B, kColsumRows));
  const bool two_launches = !hot && s->B > kEndRows;
  const unsigned n_col_blocks =
      hot ? static_cast<unsigned>(ceil_div(D, 1024))
          : static_cast<unsigned>(two_launches ? ceil_div(D, 256) * ceil_div(n_chunks, 4) : ceil_div(D, kEndCols));
  const unsigned n_dvals_blocks = grid_for(s->B * s->K, 1024, 2048);
  hipLaunchKernelGGL((hier_epilogue_kernel<GT>), dim3(1 + pending.n_blocks + n_hot_blocks + n_col_blocks + n_dvals_blocks),
                     dim3(1024), 0, st,
                     train ? reinterpret_cast<const float *>(ws + pl.off_loss) : static_cast<const float *>(nullptr),
                     train ? train->n_loss_partials : 0, train ? train->inv_count : 0.0,
                     train ? train->loss : static_cast<float *>(nullptr), pending, pending_hot, n_hot_blocks,
                     s_final, s->B, static_cast<int64_t>(d_pad), D, colsum_part,
                     hot ? static_cast<int>(pl.n_row_blocks) : two_launches ? -1 : 0, dbias, n_col_blocks, dv_part,
                     static_cast<int>(d_used / (train ? train_tile_cols(s) : kWave * sweep_vec)), s->B * s->K, dvals,
                     train ? train->stats : PairStats{});
  if (two_launches)
    hipLaunchKernelGGL(colsum_final_kernel, dim3(static_cast<unsigned>(ceil_div(D, 256))), dim3(256), 0, st, colsum_part,
                       n_chunks, D, static_cast<const float *>(nullptr), 1.0f, dbias);
}

template <typename WT, typename PT, int VEC>
void launch_hier_slices_g(const flexsae_shape *s, const HierBwdPlan &pl, int64_t slice_w,
                          const int64_t *indices, const void *weight, const void *vals,
                          const float *resid, const float *grad_out, float coef, void *dW,
                          int dW_dtype, float *dvals, float *dbias, uint8_t *ws, int flags,
                          int *status_flag, hipStream_t st, const TrainArgs *train, int piece) {
  switch (dW_dtype) {
    case FLEXSAE_F32:
      launch_hier_slices<WT, PT, float, VEC>(s, pl, slice_w, indices, weight, vals, resid, grad_out,
                                             coef, dW, dvals, dbias, ws, flags, status_flag, st, train, piece);
      break;
    case FLEXSAE_BF16:
      launch_hier_slices<WT, PT, bf16_t, VEC>(s, pl, slice_w, indices, weight, vals, resid, grad_out,
                                              coef, dW, dvals, dbias, ws, flags, status_flag, st, train, piece);
      break;
    default:
      launch_hier_slices<WT, PT, f16_t, VEC>(s, pl, slice_w, indices, weight, vals, resid, grad_out,
                                             coef, dW, dvals, dbias, ws, flags, status_flag, st, train, piece);
  }
}

template <int VEC>
void launch_hier_slices_w(const flexsae_shape *s, const HierBwdPlan &pl, int64_t slice_w,
                          const int64_t *indices, const void *weight, const void *vals,
                          const float *resid, const float *grad_out, float coef, void *dW,
                          int dW_dtype, float *dvals, float *dbias, uint8_t *ws, int flags,
                          int *status_flag, hipStream_t st, const TrainArgs *train = nullptr, int piece = 0) {
  switch (s->weight_dtype) {
    case FLEXSAE_F32:
      launch_hier_slices_g<float, float, VEC>(s, pl, slice_w, indices, weight, vals, resid, grad_out,
                                              coef, dW, dW_dtype, dvals, dbias, ws, flags, status_flag, st, train, piece);
      break;
    case FLEXSAE_BF16:
      launch_hier_slices_g<bf16_t, bf16_t, VEC>(s, pl, slice_w, indices, weight, vals, resid, grad_out,
                                                coef, dW, dW_dtype, dvals, dbias, ws, flags, status_flag, st, train, piece);
      break;
    default:
      launch_hier_slices_g<f16_t, float, VEC>(s, pl, slice_w, indices, weight, vals, resid, grad_out,
                                              coef, dW, dW_dtype, dvals, dbias, ws, flags, status_flag, st, train, piece);
  }
}

// Hot-latent tables of a workspace whose pair list is complete: the slots with the hot pairs marked,
// the hot latents, the long latents that stayed cold and their chunk table.  have_hslot: hslot[] already
// holds a copy of slot[].
void build_hot_tables(const flexsae_shape *s, const HierBwdPlan &pl, uint8_t *ws, const CsrScratch &sc, bool have_hslot,
                      hipStream_t st) {
  const uint32_t *begin = reinterpret_cast<const uint32_t *>(ws + pl.off_begin);
  const uint32_t *map = reinterpret_cast<const uint32_t *>(ws + pl.off_map);
  uint32_t *hslot = reinterpret_cast<uint32_t *>(ws + pl.off_hslot);
  uint32_t *ctrl = reinterpret_cast<uint32_t *>(ws + pl.off_hot_ctrl);
  uint32_t *hot_list = reinterpret_cast<uint32_t *>(ws + pl.off_hot_list);
  uint32_t *cand_list = reinterpret_cast<uint32_t *>(ws + pl.off_cand_list);
  uint32_t *long2 = reinterpret_cast<uint32_t *>(ws + pl.off_long2);
  if (!have_hslot) {
    const int64_t n_pairs = s->B * s->K;
    hipLaunchKernelGGL(copy_u32_kernel, dim3(grid_for(n_pairs, 256, 8192)), dim3(256), 0, st, hslot,
                       reinterpret_cast<const uint32_t *>(ws + pl.off_slot), n_pairs);
  }
  uint32_t *chunk2 = reinterpret_cast<uint32_t *>(ws + pl.off_chunk2);
  hipLaunchKernelGGL(hot_select_kernel, dim3(1), dim3(1024), 0, st, begin, sc.lists.ctrl, sc.lists.long_list, ctrl,
                     cand_list, long2, chunk2, static_cast<uint32_t>(kHotMax));
  hipLaunchKernelGGL(hot_mark_kernel, dim3(kHotMax), dim3(1024), 0, st, begin, map, ctrl, cand_list, hot_list, hslot,
                     static_cast<uint32_t>(s->K), long2, chunk2);
}

// ---- TopK backward: workspace plan and slice loop ---------------------------------------

struct TopkBwdPlan {
  int vec, tile;
  int row_vec;      // elements of a vector that divides the rows of W and dW: vec, or less where the residual copy is padded
  int resid_ld;     // elements from one gathered row to the next
  int64_t d_pad;
  size_t n_pairs, n_partial_rows;
  size_t off_colsum, off_ctrl, off_long_list, off_lists, off_resid16, off_dvpart, off_slotbv, off_partial, fixed_bytes;
  bool resid16;  // gather a bf16 copy of the residual (bf16 weights): half the cache footprint
  bool whole_groups;  // as many latents per wavefront as it takes, whatever the size
};

// Whether a bf16 copy of the residual with padded rows (16 bytes per lane, tiles of 512 columns) beats one whose rows are read
// in the vectors of `vec` elements that divide them (tiles of 64 * vec).  By 1120 shapes of both kinds of indices; the backward
// in us with narrow / padded rows, uniform and skewed:
//   vec 1, 160 columns and more, or more than 128 and at least 65536 latents: B=4096, K=128, F=65536, D=2305 695 / 374,
//       834 / 477, D=129 101 / 94, 135 / 134;  B=1024, K=64, F=32768, D=129 44 / 43, 58 / 60
//   vec 2, more than 256 columns: B=8192, K=64, F=262144, D=1026 491 / 440, 551 / 490.  From 12000 batch rows on, whose tile of
//       the copy is three L2s (1 KB per row), only where the tiles are full to 0.68: B=14886, K=43, F=73564, D=2154 607 / 587,
//       776 / 685; not B=12288, K=32, F=16384, D=1026 187 / 224, 243 / 251
//   vec 4, more than 256 columns in one tile and 1024 batch rows; in several tiles where there is enough to do for half the
//       wavefronts (38000 latents in all tiles, four tiles, or three and 100000 pairs: B=2716, K=123, F=8124, D=1324 144 / 127,
//       170 / 160; not B=700, K=159, F=7689, D=556 58 / 64, 75 / 85), and beyond 4096 batch rows, an L2, where few pairs gather
//       from it: five per latent, or thirteen up to 6144 rows (B=6189, K=89, F=256085, D=828 345 / 321, 366 / 325; not B=8192,
//       K=64, F=16384, D=1028 186 / 239, 237 / 272)
// Where it takes them, padded rows are on average 60 % ahead with vec 1 and 12 % with the others, at most 6 % behind on one kind
// of indices.
// (Pairs in chunks of long latents, most of them with skewed indices, load their W piece in vectors of `vec` elements either way;
// that is in the figures.)
bool padding_pays(const flexsae_shape *s, int vec) {
  const int64_t tiles = ceil_div(s->D, kWave * 8), pairs = s->B * s->K;
  if (vec == 1) return s->D >= 160 || (s->D > 128 && s->F >= 65536);
  if (s->D <= 256) return false;
  if (vec == 2) return tiles == 1 || s->B <= 12000 || 100 * s->D >= 68 * kWave * 8 * tiles;
  if (tiles == 1) return s->B >= 1024;
  if (s->F * tiles < 38000 && tiles < 4 && !(tiles == 3 && pairs >= 100000)) return false;
  return s->B <= 4096 || pairs <= 5 * s->F || (s->B <= 6144 && pairs <= 13 * s->F);
}

TopkBwdPlan plan_topk_bwd(const flexsae_shape *s, int flags = 0) {
  TopkBwdPlan p;
  // The reference hands its backward the residual gradient in the weight dtype
  // (topk_kernels.py:52,221); for bf16 weights the gathers here read a bf16 copy as well, unless
  // the caller asks for the fp32 residual (no copy, but narrower tiles and so more per-tile dvals
  // shares: flexsae_topk_bwd_workspace_bytes returns the larger of the two layouts).
  p.resid16 = FLEXSAE_TOPK_RESID16 && s->weight_dtype == FLEXSAE_BF16 && !(flags & FLEXSAE_TOPK_BWD_FP32_RESIDUAL);
  p.whole_groups = (flags & FLEXSAE_TOPK_BWD_AS_LARGE) != 0;
  p.vec = (s->D % 4 == 0) ? 4 : (s->D % 2 == 0) ? 2 : 1;
  p.row_vec = p.vec;
  p.resid_ld = static_cast<int>(s->D);
  // all-bf16: 16 bytes per lane (512-column tiles) halve the per-tile overheads
  if (FLEXSAE_TOPK_VEC8 && p.resid16 && s->D % 8 == 0) p.vec = p.row_vec = 8;
  // Rows that eight does not divide: the copy's rows are padded, so that its gathers are as wide.
  if (FLEXSAE_TOPK_VEC8 && p.resid16 && p.vec != 8 &&
      ((flags & FLEXSAE_TOPK_BWD_AS_LARGE) ? s->D > kWave * p.vec : padding_pays(s, p.vec))) {
    p.vec = 8;
    p.resid_ld = static_cast<int>(round_up(static_cast<size_t>(s->D), 8));
  }
  p.tile = kWave * p.vec;
  p.d_pad = ceil_div(s->D, p.tile) * p.tile;
  p.n_pairs = static_cast<size_t>(s->B) * static_cast<size_t>(s->K);
  p.n_partial_rows = p.n_pairs / kSegChunk + p.n_pairs / 65 + 2;
  size_t off = 0;
  p.off_colsum = off;
  off += round_up(static_cast<size_t>(ceil_div(s->B, kColsumRows)) * static_cast<size_t>(s->D) * 4, kAlign);
  p.off_ctrl = off;
  off += round_up(kCtrlWords * 4, kAlign);
  p.off_long_list = off;
  off += round_up((p.n_pairs / 65 + 1) * 4, kAlign);
  p.off_lists = off;
  off += carve_pair_lists(p.n_pairs, static_cast<size_t>(s->F), false, nullptr, nullptr);
  p.off_resid16 = off;
  if (p.resid16) off += round_up(static_cast<size_t>(s->B) * static_cast<size_t>(p.resid_ld) * 2, kAlign);
  p.off_dvpart = off;  // per-tile shares of dvals: [d_pad / tile, B*K] fp32
  off += round_up(static_cast<size_t>(p.d_pad / p.tile) * p.n_pairs * 4, kAlign);
  p.off_slotbv = off;  // (batch row, val) of every pair in pair-list order
  off += round_up(p.n_pairs * 8, kAlign);
  p.off_partial = off;
  p.fixed_bytes = off;
  return p;
}

PairLists carve_topk_lists(const flexsae_shape *s, const TopkBwdPlan &pl, uint8_t *ws) {
  PairLists ls = {};
  ls.ctrl = reinterpret_cast<uint32_t *>(ws + pl.off_ctrl);
  ls.long_list = reinterpret_cast<uint32_t *>(ws + pl.off_long_list);
  carve_pair_lists(pl.n_pairs, static_cast<size_t>(s->F), false, ws + pl.off_lists, &ls);
  return ls;
}

// Neighbouring latents per wavefront, a power of two up to `most`: a wavefront walks their pairs one after the other, so
// groups pay while there are wavefronts enough with them.  The fewest wavefronts (the chip holds 5120), by pairs per latent;
// us of the backward with eight / four / two / one latents per wavefront, uniform and skewed (Zipf 1.1) indices:
//   from 12 pairs on 8192: the walk is long and wants wavefronts to spread over
//          B=2048, K=109, F=4096, D=336 bf16 108 / 88 / 73 / 67, 92 / 81 / 78 / 76;  8192 to 16384 wavefronts with eight, 16 to
//          48 pairs: 1.01 / 1.00 / 0.93 and 1.00 / 0.97 / 0.88 times as fast with four / two / one
//   from 2 on 3072, below 1024: what a wavefront waits for is the head of a latent (its bounds, its records, its W row), and
//          a group pays it once: 4096 to 6144 wavefronts with eight, 1 to 4 pairs: 0.96 / 0.85 / 0.68, 0.96 / 0.87 / 0.75
// Over 320 shapes (F 4096 to 131072) 0.6 % behind the best of the four on average, and 5 % at most behind eight.
int latents_per_wave(const flexsae_shape *s, const TopkBwdPlan &pl, int most) {
  const int64_t tiles = pl.d_pad / pl.tile, pairs = s->B * s->K;
  const int64_t least = pairs >= 12 * s->F ? 8192 : pairs >= 2 * s->F ? 3072 : 1024;
  int n = most;
  while (n > 1 && ceil_div(s->F, static_cast<int64_t>(n)) * tiles < least) n /= 2;
  return n;
}

// The kernel of one latent per wavefront (topk_short_latent): 54 to 73 registers against 92 to 117 leave two or three more
// wavefronts per SIMD to gather with, and a head per latent, which a group pays once.  Times as fast as the groups, geometric
// mean over 300 shapes, uniform and skewed indices: 12 to 72 pairs per latent 1.04 and 1.04 (B=8192, K=63, F=16384, D=296
// fp16 126 -> 117 us), with more than 140000 latents in all tiles 0.96; 8 to 12 1.04 and 1.03 with fewer than 65536, 0.99 and
// 0.97 with more; 4 to 8 0.98 and 0.97; below 4 0.87 and 0.91; above 72 (nearly all pairs in chunks of long latents) 1.00 and
// 1.01.
// And with less than one pair for 32 latents, pieces of 16 bytes per lane (`wide`): all but zero rows of dW, which a group
// stores a row apart (groups / one, us, uniform and skewed: B=64, K=16, F=131072, fp32 D=8192 861 / 759, 866 / 722, D=4096
// 446 / 388, 438 / 369, bf16 D=8192 469 / 420, 462 / 397; fp16, 8 bytes, 550 / 629, 468 / 615).
bool one_latent_per_wave(const flexsae_shape *s, const TopkBwdPlan &pl, bool wide) {
  const int64_t pairs = s->B * s->K;
  const int64_t latents = s->F * (pl.d_pad / pl.tile);  // of all tiles
  if (pl.whole_groups) return false;
  if (wide && 32 * pairs < s->F) return true;
  return latents < 140000 && pairs >= (latents < 65536 ? 8 : 12) * s->F && pairs < 72 * s->F;
}

size_t topk_bwd_bytes(const TopkBwdPlan &p, int64_t slice_w) {
  return p.fixed_bytes + round_up(p.n_partial_rows * static_cast<size_t>(slice_w) * 4, kAlign);
}

template <typename WT, typename GT, typename RT, int VEC, int EV>
void launch_topk_slices(const flexsae_shape *s, const TopkBwdPlan &pl, int64_t slice_w,
                        const uint32_t *begin, const uint32_t *map, const void *weight,
                        const void *vals, const void *resid, const float *grad_out, float coef,
                        void *dW, const LeafGrads &leaf, uint8_t *ws, hipStream_t st) {
  const PairLists ls = carve_topk_lists(s, pl, ws);
  const uint32_t *long_ctrl = ls.ctrl, *long_list = ls.long_list, *chunk_begin = ls.chunk_begin;
  float *partial = reinterpret_cast<float *>(ws + pl.off_partial);
  float *dv_part = reinterpret_cast<float *>(ws + pl.off_dvpart);
  const int64_t n_pairs = static_cast<int64_t>(pl.n_pairs);
  const bool one = EV == VEC && one_latent_per_wave(s, pl, sizeof(LatentPiece<WT, GT, VEC>) == 16 &&
                                                               sizeof(raw_vec_t<WT, VEC>) == sizeof(raw_vec_t<GT, VEC>));
  const int per_wave = one ? 1 : pl.whole_groups ? topk_group<WT, GT, VEC>() : latents_per_wave(s, pl, topk_group<WT, GT, VEC>());
  const int64_t n_groups = ceil_div(s->F, static_cast<int64_t>(kWavesPerBlock) * per_wave);
  // a launch holds fewer than 2^32 threads, 2^24 blocks: narrower slices where all tiles would be more
  const int64_t most_tiles = (int64_t{1} << 23) / (n_groups + kLongBlocks);
  if (slice_w / pl.tile > most_tiles) slice_w = (most_tiles < 1 ? 1 : most_tiles) * pl.tile;
  const int K = static_cast<int>(s->K), D = static_cast<int>(s->D), sw = static_cast<int>(slice_w);
  for (int64_t col0 = 0; col0 < s->D; col0 += slice_w) {
    const int64_t cols = (pl.d_pad - col0) < slice_w ? (pl.d_pad - col0) : slice_w;
    const int tps = static_cast<int>(cols / pl.tile);
    // A last tile of less than two thirds of the columns apart from the others (us with it among them / apart, uniform
    // indices: D=296 of 256-column tiles, B=11147, K=62, F=50975 fp32 227 / 192; D=2304 of 512, B=4096, K=128, F=65536 bf16
    // 296 / 289; with more columns it fetches its slice into all L2s for little: D=1992, B=2048, K=44, F=32768 bf16 102 / 106).
    // Not of an even number of tiles, four or more, with less than two pairs per latent, where W and dW are what moves: the runs
    // of several XCDs then begin at the same latents and write a row's pieces at one time (four tiles, B=1721, K=23, F=343189,
    // D=1576 bf16 354 / 369, skewed 341 / 398; sixteen, B=1458, K=55, F=89752, D=3844 fp32 557 / 591; an odd number has no such
    // order to lose: nine, B=388, K=167, F=159036, D=2084 478 / 459).
    const int64_t last_cols = s->D - (col0 + cols - pl.tile);
    const bool in_step = tps >= 4 && tps % 2 == 0 && n_pairs < 2 * s->F;
    const int n_full = 3 * last_cols < 2 * static_cast<int64_t>(pl.tile) && !in_step ? tps - 1 : tps;
    const int64_t xcd_span = ceil_div(n_groups * n_full, 8);
    const int64_t last_span = n_full < tps ? ceil_div(n_groups, 8) : 0;
    // no more leading blocks than chunks of long latents there can be (a multiple of eight)
    const int64_t most_long = (ceil_div(static_cast<int64_t>(pl.n_partial_rows) * tps, kWavesPerBlock) + 7) & ~int64_t{7};
    const int64_t all_long = static_cast<int64_t>(kLongBlocks) * tps;
    const unsigned n_long = static_cast<unsigned>(most_long < all_long ? most_long : all_long);
    const size_t resid_bytes =
        static_cast<size_t>(s->B) * static_cast<size_t>(pl.resid_ld) * sizeof(typename Traits<RT>::store_t);
    constexpr int kEndTiles = VEC / EV;  // tiles of the long latents' second step per tile
    const auto kernel = one ? topk_bwd_kernel<WT, GT, RT, VEC, EV, EV == VEC> : topk_bwd_kernel<WT, GT, RT, VEC, EV, false>;
    hipLaunchKernelGGL(kernel,
                       dim3(n_long + static_cast<unsigned>((xcd_span + last_span) * 8)),
                       dim3(kBlock), 0, st, begin, map, long_ctrl, long_list, chunk_begin,
                       reinterpret_cast<const vec_t<uint32_t, 2> *>(ws + pl.off_slotbv), weight, vals,
                       s->vals_dtype, resid, grad_out, coef, dW, dv_part, n_pairs, partial, n_long, static_cast<uint32_t>(n_groups),
                       static_cast<uint32_t>(xcd_span), static_cast<uint32_t>(n_full),
                       per_wave, tps,
                       static_cast<int>(col0), sw, s->F, K, D, pl.resid_ld, static_cast<uint32_t>(resid_bytes));
    if (col0 + slice_w < s->D) {
      hipLaunchKernelGGL((seg_reduce_long_finalize_kernel<GT, EV, 8>), dim3(256), dim3(kBlock), 0, st,
                         long_ctrl, long_list, chunk_begin, partial, dW, static_cast<const float *>(nullptr), tps * kEndTiles,
                         static_cast<int>(col0), sw, D);
      continue;
    }
    constexpr unsigned n_long_blocks = 256;
    const unsigned n_col_blocks = static_cast<unsigned>(ceil_div(D, kBlock));
    hipLaunchKernelGGL((topk_epilogue_kernel<GT, EV>),
                       dim3(n_long_blocks + n_col_blocks + grid_for(n_pairs, kBlock, 8192)), dim3(kBlock), 0, st, long_ctrl,
                       long_list, chunk_begin, partial, dW, tps * kEndTiles, static_cast<int>(col0), sw, D, n_long_blocks,
                       reinterpret_cast<const float *>(ws + pl.off_colsum), static_cast<int>(ceil_div(s->B, kColsumRows)),
                       grad_out, coef, n_col_blocks, map, dv_part, static_cast<int>(pl.d_pad / pl.tile), n_pairs, leaf);
  }
}

template <typename WT, typename RT, int VEC, int EV = VEC>
void launch_topk_slices_g(const flexsae_shape *s, const TopkBwdPlan &pl, int64_t slice_w,
                          const uint32_t *begin, const uint32_t *map, const void *weight,
                          const void *vals, const void *resid, const float *grad_out, float coef,
                          void *dW, int dW_dtype, const LeafGrads &leaf, uint8_t *ws, hipStream_t st) {
  switch (dW_dtype) {
    case FLEXSAE_F32:
      launch_topk_slices<WT, float, RT, VEC, EV>(s, pl, slice_w, begin, map, weight, vals, resid, grad_out,
                                             coef, dW, leaf, ws, st);
      break;
    case FLEXSAE_BF16:
      launch_topk_slices<WT, bf16_t, RT, VEC, EV>(s, pl, slice_w, begin, map, weight, vals, resid, grad_out,
                                              coef, dW, leaf, ws, st);
      break;
    default:
      launch_topk_slices<WT, f16_t, RT, VEC, EV>(s, pl, slice_w, begin, map, weight, vals, resid, grad_out,
                                             coef, dW, leaf, ws, st);
  }
}

// `resid` is the fp32 residual, or its bf16 copy when the plan says so (bf16 weights only)
template <int VEC>
void launch_topk_slices_w(const flexsae_shape *s, const TopkBwdPlan &pl, int64_t slice_w,
                          const uint32_t *begin, const uint32_t *map, const void *weight,
                          const void *vals, const void *resid, const float *grad_out, float coef,
                          void *dW, int dW_dtype, const LeafGrads &leaf, uint8_t *ws, hipStream_t st) {
  switch (s->weight_dtype) {
    case FLEXSAE_F32:
      launch_topk_slices_g<float, float, VEC>(s, pl, slice_w, begin, map, weight, vals, resid, grad_out,
                                              coef, dW, dW_dtype, leaf, ws, st);
      break;
    case FLEXSAE_BF16:
      if (pl.resid16)
        launch_topk_slices_g<bf16_t, bf16_t, VEC>(s, pl, slice_w, begin, map, weight, vals, resid, grad_out,
                                                  coef, dW, dW_dtype, leaf, ws, st);
      else
        launch_topk_slices_g<bf16_t, float, VEC>(s, pl, slice_w, begin, map, weight, vals, resid, grad_out,
                                                 coef, dW, dW_dtype, leaf, ws, st);
      break;
    default:
      launch_topk_slices_g<f16_t, float, VEC>(s, pl, slice_w, begin, map, weight, vals, resid, grad_out,
                                              coef, dW, dW_dtype, leaf, ws, st);
  }
}

size_t least_topk_bwd_bytes(const TopkBwdPlan &pl) { return topk_bwd_bytes(pl, pl.tile); }

// What a backward checks besides the pair list.
int check_topk_bwd(const flexsae_shape *s, const TopkBwdPlan &pl, const int64_t *indices, const void *weight, const void *vals,
                   const float *resid, const float *grad_out, const void *dW, int dW_dtype) {
  if ((indices && !aligned(indices, 8)) || !aligned(weight, pl.row_vec * dtype_size(s->weight_dtype)) ||
      !aligned(vals, dtype_size(s->vals_dtype)) || !aligned(resid, pl.resid16 ? 16 : pl.vec * 4) || !aligned(grad_out, 4) ||
      !aligned(dW, pl.row_vec * dtype_size(dW_dtype)))
    return FLEXSAE_ERR_ALIGNMENT;
  return FLEXSAE_OK;
}

// The backward proper, with the records, the lists, the copy of the residual and stage 1 of dbias in the workspace.
void launch_topk_bwd(const flexsae_shape *s, const TopkBwdPlan &pl, const uint32_t *begin, const uint32_t *map,
                     const void *weight, const void *vals, const float *resid, const float *grad_out, void *dW, int dW_dtype,
                     const LeafGrads &leaf, uint8_t *ws, size_t ws_bytes, hipStream_t st) {
  int64_t slice_w = pl.tile;
  while (slice_w + pl.tile <= pl.d_pad && topk_bwd_bytes(pl, slice_w + pl.tile) <= ws_bytes) slice_w += pl.tile;
  const float coef =
      static_cast<float>(2.0 / (static_cast<double>(s->B) * static_cast<double>(s->D)));
  const void *gather_src = pl.resid16 ? static_cast<const void *>(ws + pl.off_resid16) : resid;
  if (pl.vec == 8) {
    const auto slices = pl.row_vec == 8   ? launch_topk_slices_g<bf16_t, bf16_t, 8>
                        : pl.row_vec == 4 ? launch_topk_slices_g<bf16_t, bf16_t, 8, 4>
                        : pl.row_vec == 2 ? launch_topk_slices_g<bf16_t, bf16_t, 8, 2>
                                          : launch_topk_slices_g<bf16_t, bf16_t, 8, 1>;
    slices(s, pl, slice_w, begin, map, weight, vals, gather_src, grad_out, coef, dW, dW_dtype, leaf, ws, st);
    return;
  }
  const auto slices = pl.vec == 4 ? launch_topk_slices_w<4> : pl.vec == 2 ? launch_topk_slices_w<2> : launch_topk_slices_w<1>;
  slices(s, pl, slice_w, begin, map, weight, vals, gather_src, grad_out, coef, dW, dW_dtype, leaf, ws, st);
}

// The preparation on a given pair list (topk_prepare_kernel) and the lists of its long latents.
void launch_topk_prepare(const flexsae_shape *s, const TopkBwdPlan &pl, const uint32_t *begin, const uint32_t *map,
                         const int64_t *indices, const void *vals, const float *resid, uint8_t *ws, hipStream_t st) {
  const PairLists lists = carve_topk_lists(s, pl, ws);
  const int64_t n_resid = pl.resid16 ? s->B * pl.resid_ld : 0;
  const int64_t work = s->B * s->K > ceil_div(n_resid, 4) ? s->B * s->K : ceil_div(n_resid, 4);
  const unsigned n_col_blocks = static_cast<unsigned>(ceil_div(s->D, 256) * ceil_div(s->B, kColsumRows));
  hipLaunchKernelGGL(topk_prepare_kernel, dim3(n_col_blocks + grid_for(work, 256, 1 << 16)), dim3(256), 0, st, map, indices,
                     s->F, vals, s->vals_dtype, s->B * s->K, static_cast<int>(s->K),
                     reinterpret_cast<vec_t<uint32_t, 2> *>(ws + pl.off_slotbv), resid, n_resid,
                     pl.resid16 ? static_cast<void *>(ws + pl.off_resid16) : nullptr, lists.ctrl, s->B,
                     static_cast<int>(s->D), pl.resid_ld, reinterpret_cast<float *>(ws + pl.off_colsum), n_col_blocks);
  launch_pair_lists(begin, s->F, lists, st, true);
}

// A pair list made for one TopK backward, in front of its workspace: begin[F+1] | map[B*K] | scratch.
struct TopkListPlan {
  size_t off_map, off_csr, bytes;
};

TopkListPlan plan_topk_list(const flexsae_shape *s) {
  TopkListPlan p;
  p.off_map = round_up(static_cast<size_t>(s->F + 1) * 4, kAlign);
  p.off_csr = p.off_map + round_up(static_cast<size_t>(s->B) * static_cast<size_t>(s->K) * 4, kAlign);
  p.bytes = p.off_csr + round_up(flexsae_csr_workspace_bytes(s->B, s->K, s->F), kAlign);
  return p;
}

}  // namespace

extern "C" {

int flexsae_abi_version(void) { return FLEXSAE_ABI_VERSION; }

#ifndef FLEXSAE_BUILD_ID
#define FLEXSAE_BUILD_ID "unknown"
#endif
const char *flexsae_build_id(void) { return FLEXSAE_BUILD_ID; }

const char *flexsae_status_string(int status) {
  switch (status) {
    case FLEXSAE_OK:
      return "ok";
    case FLEXSAE_ERR_INVALID_ARGUMENT:
      return "invalid argument (null pointer, non-positive size or unknown dtype)";
    case FLEXSAE_ERR_UNSUPPORTED:
      return "unsupported size (need F, K < 2^31, D < 2^29 and B*K < 2^32)";
    case FLEXSAE_ERR_WORKSPACE:
      return "workspace missing, too small or not 256-byte aligned";
    case FLEXSAE_ERR_LAUNCH:
      return "HIP kernel launch failed";
    case FLEXSAE_ERR_ALIGNMENT:
      return "tensor pointer not aligned to its element size";
    case FLEXSAE_ERR_SCRATCH_LIMIT:
      return "problem too large for the static scratch of this entry point (use the variant that takes a workspace)";
    default:
      return "unknown status";
  }
}

size_t flexsae_fwd_workspace_bytes(const flexsae_shape *s) {
  if (check_shape(s) != FLEXSAE_OK) return 0;
  // one fp32 partial per (row, tile); the narrowest tile is 64 columns
  return round_up(static_cast<size_t>(s->B) * static_cast<size_t>(ceil_div(s->D, kWave)) * 4, kAlign);
}

size_t flexsae_topk_fwd_workspace_bytes(const flexsae_shape *s) {
  const size_t base = flexsae_fwd_workspace_bytes(s);
  return base == 0 ? 0 : base + plan_ordered(s).steps_bytes;
}

size_t flexsae_topk_fwd_best_workspace_bytes(const flexsae_shape *s) {
  const size_t base = flexsae_fwd_workspace_bytes(s);
  if (base == 0) return 0;
  const OrderedPlan p = plan_ordered(s);
  return base + (p.waves != 0 && order_pays(s, p) ? p.steps_bytes : 0);
}

int flexsae_hier_fwd(const flexsae_shape *shape, const int64_t *indices, const void *weight,
                     const void *vals, const void *bias, const void *target, float *loss,
                     float *resid, void *workspace, size_t workspace_bytes, int *status_flag,
                     void *stream) {
  return forward<true>(shape, indices, weight, vals, bias, target, loss, resid, workspace,
                       workspace_bytes, status_flag, stream);
}

int flexsae_hier_fwd_static(const flexsae_shape *shape, const int64_t *indices, const void *weight,
                            const void *vals, const void *bias, const void *target, float *loss,
                            float *resid, int *status_flag, void *stream) {
  const int rc = check_shape(shape);
  if (rc != FLEXSAE_OK) return rc;
  if (flexsae_fwd_workspace_bytes(shape) > kStaticScratchBytes) return FLEXSAE_ERR_SCRATCH_LIMIT;
  void *ptr = nullptr;
  const int src = static_scratch_for_current_device(&ptr);
  if (src != FLEXSAE_OK) return src;
  // every partial the finalize kernel reads is written by the forward kernel of the same call:
  // nothing in the array has to start at zero
  return forward<true>(shape, indices, weight, vals, bias, target, loss, resid, ptr, kStaticScratchBytes,
                       status_flag, stream);
}

int flexsae_topk_fwd(const flexsae_shape *shape, const int64_t *indices, const void *weight,
                     const void *vals, const void *bias, const void *target, float *loss,
                     float *resid, void *workspace, size_t workspace_bytes, int *status_flag,
                     void *stream) {
  return forward<false>(shape, indices, weight, vals, bias, target, loss, resid, workspace,
                        workspace_bytes, status_flag, stream);
}

int flexsae_hier_bwd_atomic(const flexsae_shape *s, const int64_t *indices, const void *weight,
                            const void *vals, const float *resid, const float *grad_out,
                            float *dW_acc, float *dvals, float *dbias, int flags, int *status_flag,
                            void *stream) {
  int rc = check_shape(s);
  if (rc != FLEXSAE_OK) return rc;
  if (!indices || !weight || !vals || !resid || !grad_out || !dW_acc || !dvals || !dbias)
    return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (!aligned(indices, 8) || !aligned(weight, dtype_size(s->weight_dtype)) ||
      !aligned(vals, dtype_size(s->vals_dtype)) || !aligned(resid, 4) || !aligned(grad_out, 4) ||
      !aligned(dW_acc, 16) || !aligned(dvals, 16) || !aligned(dbias, 16))
    return FLEXSAE_ERR_ALIGNMENT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (!(flags & FLEXSAE_BWD_OUTPUTS_PREZEROED)) {
    zero_f32(dW_acc, s->F * s->D, st);
    zero_f32(dvals, s->B * s->K, st);
    zero_f32(dbias, s->D, st);
  }
  const float coef = static_cast<float>(
      2.0 / (static_cast<double>(s->B) * static_cast<double>(s->K) * static_cast<double>(s->D)));
  switch (s->weight_dtype) {
    case FLEXSAE_F32:
      launch_hier_bwd_t<float>(s, indices, weight, vals, resid, grad_out, coef, dW_acc, dvals,
                               dbias, status_flag, st);
      break;
    case FLEXSAE_BF16:
      launch_hier_bwd_t<bf16_t>(s, indices, weight, vals, resid, grad_out, coef, dW_acc, dvals,
                                dbias, status_flag, st);
      break;
    default:
      launch_hier_bwd_t<f16_t>(s, indices, weight, vals, resid, grad_out, coef, dW_acc, dvals,
                               dbias, status_flag, st);
  }
  return launch_status();
}

size_t flexsae_hier_bwd_workspace_bytes(const flexsae_shape *s, int64_t slice_cols) {
  if (check_shape(s) != FLEXSAE_OK) return 0;
  const HierBwdPlan pl = plan_hier_bwd(s);
  int64_t sw = slice_cols <= 0 ? pl.tile : ceil_div(slice_cols, pl.tile) * pl.tile;
  if (sw > pl.d_pad) sw = pl.d_pad;
  return hier_bwd_bytes(pl, sw);
}

size_t flexsae_hier_fwd_bwd_workspace_bytes_flags(const flexsae_shape *s, int64_t slice_cols, int flags) {
  if (check_shape(s) != FLEXSAE_OK || !train_supported(s, flags)) return 0;
  const bool hot = (flags & FLEXSAE_BWD_HOT_LATENTS) && hot_supported(s);
  const HierBwdPlan pl = plan_hier_bwd(s, hot, flags);
  const int64_t granule = train_piece_ok(s, pl, nullptr, s->weight_dtype) ? train_tile_cols(s) : pl.tile;
  int64_t sw = slice_cols <= 0 ? granule : ceil_div(slice_cols, granule) * granule;
  if (sw > pl.d_pad) sw = pl.d_pad;
  return hier_bwd_bytes(pl, sw);
}

size_t flexsae_hier_fwd_bwd_workspace_bytes(const flexsae_shape *s, int64_t slice_cols) {
  return flexsae_hier_fwd_bwd_workspace_bytes_flags(s, slice_cols, 0);
}

int flexsae_hier_hot_latents_supported(const flexsae_shape *s) {
  return check_shape(s) == FLEXSAE_OK && train_supported(s) && hot_supported(s) ? 1 : 0;
}

int flexsae_hier_pair_stats(const flexsae_shape *s, const void *workspace, uint32_t *stats, void *stream) {
  const int rc = check_shape(s);
  if (rc != FLEXSAE_OK) return rc;
  if (!workspace || !stats) return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (!aligned(workspace, kAlign) || !aligned(stats, 4)) return FLEXSAE_ERR_ALIGNMENT;
  const HierBwdPlan pl = plan_hier_bwd(s);  // the part of the layout every hierarchical workspace shares
  uint8_t *ws = static_cast<uint8_t *>(const_cast<void *>(workspace));
  const CsrScratch sc = carve_hier_lists(s, pl, ws);
  hipLaunchKernelGGL(pair_stats_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                     PairStats{sc.lists.ctrl, stats, 0u, 0});
  return launch_status();
}

int flexsae_hier_hot_stats(const flexsae_shape *s, const void *workspace, uint32_t *stats, void *stream) {
  const int rc = check_shape(s);
  if (rc != FLEXSAE_OK) return rc;
  if (!workspace || !stats) return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (!train_supported(s) || !hot_supported(s)) return FLEXSAE_ERR_UNSUPPORTED;
  if (!aligned(workspace, kAlign) || !aligned(stats, 4)) return FLEXSAE_ERR_ALIGNMENT;
  const HierBwdPlan pl = plan_hier_bwd(s, true);
  const uint32_t *ctrl = reinterpret_cast<const uint32_t *>(static_cast<const uint8_t *>(workspace) + pl.off_hot_ctrl);
  static_assert(kHotNHot == 0 && kHotNCand == 1 && kHotLong2Count == 2 && kHotThreshold == 3 && kHotDeferred == 4,
                "flexsae_hier_hot_stats hands out the first five control words");
  hipLaunchKernelGGL(copy_u32_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream), stats, ctrl,
                     static_cast<int64_t>(5));
  return launch_status();
}

int flexsae_hier_bwd(const flexsae_shape *s, const int64_t *indices, const void *weight,
                     const void *vals, const float *resid, const float *grad_out, void *dW,
                     int dW_dtype, float *dvals, float *dbias, void *workspace,
                     size_t workspace_bytes, int flags, int *status_flag, void *stream) {
  int rc = check_shape(s);
  if (rc != FLEXSAE_OK) return rc;
  if (!grad_out || !dW || !valid_dtype(dW_dtype)) return FLEXSAE_ERR_INVALID_ARGUMENT;
  const HierBwdPlan pl = plan_hier_bwd(s);
  if (!workspace || !aligned(workspace, kAlign) || workspace_bytes < hier_bwd_bytes(pl, pl.tile))
    return FLEXSAE_ERR_WORKSPACE;
  // widest slice (whole tiles) the workspace can hold
  int64_t slice_w = pl.tile;
  while (slice_w + pl.tile <= pl.d_pad && hier_bwd_bytes(pl, slice_w + pl.tile) <= workspace_bytes)
    slice_w += pl.tile;
  // REDUCE_ONLY on a kept pair list: with a single-slice workspace this is the deferred reduction
  // of staged contributions, which only reads the workspace and writes dW; on a sliced workspace
  // it is the reduction phase of every slice (profiling), which still needs the other arguments
  const bool reduce_only = (flags & FLEXSAE_BWD_REDUCE_ONLY) && (flags & FLEXSAE_BWD_REUSE_PAIR_LIST) &&
                           slice_w >= pl.d_pad;
  if (!reduce_only && (!indices || !weight || !vals || !resid || !dvals || !dbias))
    return (flags & FLEXSAE_BWD_SCALE_BY_GRAD_OUT) ? FLEXSAE_ERR_WORKSPACE : FLEXSAE_ERR_INVALID_ARGUMENT;
  if ((flags & FLEXSAE_BWD_SCALE_BY_GRAD_OUT) && !reduce_only)
    return slice_w < pl.d_pad ? FLEXSAE_ERR_WORKSPACE : FLEXSAE_ERR_INVALID_ARGUMENT;
  if (!aligned(grad_out, 4) || !aligned(dW, pl.vec * dtype_size(dW_dtype))) return FLEXSAE_ERR_ALIGNMENT;
  if (!reduce_only &&
      (!aligned(indices, 8) || !aligned(weight, pl.vec * dtype_size(s->weight_dtype)) ||
       !aligned(vals, dtype_size(s->vals_dtype)) || !aligned(resid, pl.vec * 4) || !aligned(dvals, 16) ||
       !aligned(dbias, 16)))
    return FLEXSAE_ERR_ALIGNMENT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint8_t *ws = static_cast<uint8_t *>(workspace);
  uint32_t *begin = reinterpret_cast<uint32_t *>(ws + pl.off_begin);
  uint32_t *map = reinterpret_cast<uint32_t *>(ws + pl.off_map);
  if (!(flags & FLEXSAE_BWD_REUSE_PAIR_LIST))
    csr_build_launch(indices, s->B, s->K, s->F, begin, map, reinterpret_cast<uint32_t *>(ws + pl.off_slot), nullptr,
                     carve_hier_lists(s, pl, ws, flags), status_flag, st);
  const float coef = static_cast<float>(
      2.0 / (static_cast<double>(s->B) * static_cast<double>(s->K) * static_cast<double>(s->D)));
  if (pl.vec == 4) {
    launch_hier_slices_w<4>(s, pl, slice_w, indices, weight, vals, resid, grad_out, coef, dW, dW_dtype,
                            dvals, dbias, ws, flags, status_flag, st);
  } else {
    // rows that allow no more than 8 bytes of their own elements at a time are reduced by pieces where a slice is
    // whole pieces
    const int64_t pc = piece_cols(pl);
    if (slice_w % pc != 0 && slice_w > pc && s->F * s->D >= (6 << 20) &&
        !(flags & (FLEXSAE_BWD_SWEEP_ONLY | FLEXSAE_BWD_REDUCE_ONLY))) {
      // as many slices of whole pieces as are needed, of about the same width (bf16 rows of odd length; us of the step in one
      // slice by elements / in two by pieces: B=287, K=32, F=14239, D=4099 237 / 187, B=4096, K=64, F=65536, D=129 171 / 144;
      // small dW only pays for the launches: B=300, K=20, F=8000, D=513 61 / 73)
      const int64_t n_slices = ceil_div(pl.d_pad, slice_w - slice_w % pc);
      slice_w = ceil_div(ceil_div(pl.d_pad, n_slices), pc) * pc;
    }
    const int piece = slice_w % pc == 0 ? static_cast<int>(pc) : 0;
    if (pl.vec == 2)
      launch_hier_slices_w<2>(s, pl, slice_w, indices, weight, vals, resid, grad_out, coef, dW, dW_dtype,
                              dvals, dbias, ws, flags, status_flag, st, nullptr, piece);
    else
      launch_hier_slices_w<1>(s, pl, slice_w, indices, weight, vals, resid, grad_out, coef, dW, dW_dtype,
                              dvals, dbias, ws, flags, status_flag, st, nullptr, piece);
  }
  return launch_status();
}

int flexsae_hier_pair_list_layout(const flexsae_shape *s, size_t *begin_offset, size_t *map_offset) {
  const int rc = check_shape(s);
  if (rc != FLEXSAE_OK) return rc;
  if (!begin_offset || !map_offset) return FLEXSAE_ERR_INVALID_ARGUMENT;
  const HierBwdPlan pl = plan_hier_bwd(s);
  *begin_offset = pl.off_begin;
  *map_offset = pl.off_map;
  return FLEXSAE_OK;
}

int flexsae_hier_import_pair_list(const flexsae_shape *s, const uint32_t *begin, const uint32_t *map,
                                  void *workspace, size_t workspace_bytes, void *stream) {
  const int rc = check_shape(s);
  if (rc != FLEXSAE_OK) return rc;
  if (!begin || !map) return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (!aligned(begin, 4) || !aligned(map, 4)) return FLEXSAE_ERR_ALIGNMENT;
  const HierBwdPlan pl = plan_hier_bwd(s);
  if (!workspace || !aligned(workspace, kAlign) || workspace_bytes < hier_bwd_bytes(pl, pl.tile))
    return FLEXSAE_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint8_t *ws = static_cast<uint8_t *>(workspace);
  uint32_t *ws_begin = reinterpret_cast<uint32_t *>(ws + pl.off_begin);
  uint32_t *ws_map = reinterpret_cast<uint32_t *>(ws + pl.off_map);
  const int64_t n_pairs = s->B * s->K;
  if (ws_begin != begin)
    hipLaunchKernelGGL(copy_u32_kernel, dim3(grid_for(s->F + 1, 256, 4096)), dim3(256), 0, st, ws_begin, begin,
                       s->F + 1);
  if (ws_map != map)
    hipLaunchKernelGGL(copy_u32_kernel, dim3(grid_for(n_pairs, 256, 8192)), dim3(256), 0, st, ws_map, map, n_pairs);
  hipLaunchKernelGGL(csr_inverse_kernel, dim3(grid_for(n_pairs, 256, 8192)), dim3(256), 0, st, ws_map, n_pairs,
                     reinterpret_cast<uint32_t *>(ws + pl.off_slot), static_cast<uint32_t *>(nullptr));
  launch_pair_lists(ws_begin, s->F, carve_hier_lists(s, pl, ws).lists, st);
  return launch_status();
}

int flexsae_hier_fwd_bwd_supported(const flexsae_shape *s) {
  return check_shape(s) == FLEXSAE_OK && train_supported(s) ? 1 : 0;
}

}  // extern "C"

namespace {

// flexsae_hier_fwd_bwd, or with `sgd_step` (a device scalar) flexsae_hier_sgd_step: dW is then the
// weight matrix itself and every touched row has step * (its unit-gradient row) subtracted.
int hier_fwd_bwd_impl(const flexsae_shape *s, const int64_t *indices, const void *weight,
                      const void *vals, const void *bias, const void *target, float *loss,
                      void *dW, int dW_dtype, float *dvals, float *dbias, void *workspace,
                      size_t workspace_bytes, int flags, int *status_flag, void *stream,
                      const float *sgd_step, const float *dw_scale = nullptr, uint32_t *stats = nullptr,
                      uint32_t stats_tag = 0) {
  int rc = check_shape(s);
  if (rc != FLEXSAE_OK) return rc;
  if (sgd_step || dw_scale) {
    if (flags & (FLEXSAE_BWD_NO_DW | FLEXSAE_BWD_SWEEP_ONLY | FLEXSAE_BWD_REDUCE_ONLY | FLEXSAE_BWD_SKIP_EPILOGUE))
      return FLEXSAE_ERR_INVALID_ARGUMENT;
    if (!aligned(sgd_step, 4) || !aligned(dw_scale, 4)) return FLEXSAE_ERR_ALIGNMENT;
  }
  const bool no_dw = (flags & FLEXSAE_BWD_NO_DW) != 0;
  const bool defer_reduce = (flags & FLEXSAE_BWD_SWEEP_ONLY) != 0 && !no_dw;
  if (!indices || !weight || !vals || !bias || !target || !loss || !dvals || !dbias ||
      (!defer_reduce && !no_dw && (!dW || !valid_dtype(dW_dtype))))
    return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (!train_supported(s, flags)) return FLEXSAE_ERR_UNSUPPORTED;
  if (s->D % 4 != 0 && defer_reduce) return FLEXSAE_ERR_UNSUPPORTED;
  // hot-latent accumulators: a hint, taken where the shape allows them, the reductions run in this
  // call and every pointer is aligned for the piece reduction (the workspace layout depends on it)
  const bool hot = (flags & FLEXSAE_BWD_HOT_LATENTS) && hot_supported(s) && !defer_reduce &&
                   piece_reduce_ok(s, plan_hier_bwd(s), (defer_reduce || no_dw) ? nullptr : dW, dW_dtype);
  const HierBwdPlan pl = plan_hier_bwd(s, hot, flags);
  if (!aligned(indices, 8) || !aligned(weight, 4 * dtype_size(s->weight_dtype)) ||
      !aligned(vals, dtype_size(s->vals_dtype)) || !aligned(bias, 2 * dtype_size(s->bias_dtype)) ||
      !aligned(target, 2 * dtype_size(s->target_dtype)) || !aligned(loss, 4) ||
      (!defer_reduce && !no_dw && !aligned(dW, 4 * dtype_size(dW_dtype))) || !aligned(dvals, 16) ||
      !aligned(dbias, 16))
    return FLEXSAE_ERR_ALIGNMENT;
  // slices are whole training tiles when the reduction can work on 256-byte pieces, else whole
  // reduction tiles
  const bool piece = train_piece_ok(s, pl, (defer_reduce || no_dw) ? nullptr : dW, dW_dtype);
  if (sgd_step && !piece) return FLEXSAE_ERR_UNSUPPORTED;  // only the piece reduction updates in place
  const int64_t granule = piece ? train_tile_cols(s) : pl.tile;
  if (!workspace || !aligned(workspace, kAlign) || workspace_bytes < hier_bwd_bytes(pl, granule))
    return FLEXSAE_ERR_WORKSPACE;
  int64_t slice_w = granule;
  while (slice_w + granule <= pl.d_pad && hier_bwd_bytes(pl, slice_w + granule) <= workspace_bytes)
    slice_w += granule;
  if (defer_reduce && slice_w < pl.d_pad) return FLEXSAE_ERR_WORKSPACE;  // contributions must all fit
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint8_t *ws = static_cast<uint8_t *>(workspace);
  uint32_t *begin = reinterpret_cast<uint32_t *>(ws + pl.off_begin);
  uint32_t *map = reinterpret_cast<uint32_t *>(ws + pl.off_map);
  const CsrScratch sc = carve_hier_lists(s, pl, ws, flags);
  const bool build = !(flags & FLEXSAE_BWD_REUSE_PAIR_LIST);
  // Latents of one pair: their contribution is their gradient (kSoloSlotBit), where this call builds the list that
  // marks them.  (Whatever the number of pairs per latent: see hier_train_kernel.)
  const bool solo = build && !defer_reduce && !no_dw && !sgd_step && solo_marks(s) && sc.plan.bucketed;
  if (build)
    csr_build_launch(indices, s->B, s->K, s->F, begin, map, reinterpret_cast<uint32_t *>(ws + pl.off_slot),
                     hot ? reinterpret_cast<uint32_t *>(ws + pl.off_hslot) : nullptr, sc, status_flag, st,
                     solo ? kSoloSlotBit : 0u);
  if (hot && !((flags & FLEXSAE_BWD_REUSE_PAIR_LIST) && (flags & FLEXSAE_BWD_REUSE_HOT_TABLES)))
    build_hot_tables(s, pl, ws, sc, build, st);
  const double count = static_cast<double>(s->B) * static_cast<double>(s->K) * static_cast<double>(s->D);
  const float coef = static_cast<float>(2.0 / count);
  const TrainArgs ta = {bias, target, loss, s->B * (hier_cols_used(s, pl, true, piece) / train_tile_cols(s)),
                        1.0 / count, PairStats{sc.lists.ctrl, stats, stats_tag, 1}};
  // without dW the reductions are left out like in the deferred case (dW_dtype only selects a template then)
  const auto slices = pl.vec == 4 ? launch_hier_slices_w<4> : pl.vec == 2 ? launch_hier_slices_w<2> : launch_hier_slices_w<1>;
  slices(s, pl, slice_w, indices, weight, vals, nullptr, sgd_step ? sgd_step : dw_scale, coef, dW,
         no_dw ? s->weight_dtype : dW_dtype, dvals, dbias, ws,
         (flags & (FLEXSAE_BWD_SWEEP_ONLY | FLEXSAE_BWD_REDUCE_ONLY | FLEXSAE_BWD_SKIP_EPILOGUE |
                   FLEXSAE_BWD_HOT_NO_HEADROOM | FLEXSAE_BWD_DENSE_LATENTS)) |
             (no_dw ? FLEXSAE_BWD_SWEEP_ONLY : 0) | (sgd_step ? kBwdSgdUpdate : dw_scale ? kBwdScaled : 0) |
             (hot ? kBwdHot : 0) | (solo ? kBwdSolo : 0),
         status_flag, st, &ta, piece ? static_cast<int>(piece_cols(pl)) : 0);
  return launch_status();
}

}  // namespace

extern "C" {

int flexsae_hier_fwd_bwd(const flexsae_shape *s, const int64_t *indices, const void *weight,
                         const void *vals, const void *bias, const void *target, float *loss,
                         void *dW, int dW_dtype, float *dvals, float *dbias, void *workspace,
                         size_t workspace_bytes, int flags, int *status_flag, void *stream) {
  return hier_fwd_bwd_impl(s, indices, weight, vals, bias, target, loss, dW, dW_dtype, dvals, dbias, workspace,
                           workspace_bytes, flags & ~(kBwdSgdUpdate | kBwdHot | kBwdSolo | kBwdScaled), status_flag, stream, nullptr);
}

int flexsae_hier_fwd_bwd_scaled(const flexsae_shape *s, const int64_t *indices, const void *weight, const void *vals,
                                const void *bias, const void *target, const float *grad_out, float *loss, void *dW,
                                int dW_dtype, float *dvals, float *dbias, void *workspace, size_t workspace_bytes,
                                int flags, int *status_flag, void *stream) {
  if (!grad_out) return FLEXSAE_ERR_INVALID_ARGUMENT;
  return hier_fwd_bwd_impl(s, indices, weight, vals, bias, target, loss, dW, dW_dtype, dvals, dbias, workspace,
                           workspace_bytes, flags & ~(kBwdSgdUpdate | kBwdHot | kBwdSolo | kBwdScaled), status_flag, stream,
                           nullptr, grad_out);
}

int flexsae_hier_sgd_step(const flexsae_shape *s, const int64_t *indices, void *weight, const void *vals,
                          const void *bias, const void *target, const float *step, float *loss,
                          float *dvals, float *dbias, void *workspace, size_t workspace_bytes, int flags,
                          int *status_flag, void *stream) {
  if (!step || !s) return FLEXSAE_ERR_INVALID_ARGUMENT;
  return hier_fwd_bwd_impl(s, indices, weight, vals, bias, target, loss, weight, s->weight_dtype, dvals, dbias,
                           workspace, workspace_bytes,
                           flags & (FLEXSAE_BWD_REUSE_PAIR_LIST | FLEXSAE_BWD_HOT_LATENTS | FLEXSAE_BWD_REUSE_HOT_TABLES |
                                    FLEXSAE_BWD_HOT_NO_HEADROOM | FLEXSAE_BWD_DENSE_LATENTS | FLEXSAE_BWD_HOT_BLOCKS_64 |
                                    FLEXSAE_BWD_HOT_BLOCKS_32),
                           status_flag, stream, step);
}

int flexsae_hier_step(const flexsae_shape *s, const int64_t *indices, void *weight, const void *vals, const void *bias,
                      const void *target, const float *grad_out, const float *step, float *loss, void *dW, int dW_dtype,
                      float *dvals, float *dbias, void *workspace, size_t workspace_bytes, int flags, uint32_t *stats,
                      uint32_t stats_tag, int *status_flag, void *stream) {
  if (!s || (step && (grad_out || dW)) ||
      (flags & (FLEXSAE_BWD_SWEEP_ONLY | FLEXSAE_BWD_REDUCE_ONLY | FLEXSAE_BWD_SKIP_EPILOGUE)))
    return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (!aligned(stats, 4)) return FLEXSAE_ERR_ALIGNMENT;
  return hier_fwd_bwd_impl(s, indices, weight, vals, bias, target, loss, step ? weight : dW, step ? s->weight_dtype : dW_dtype,
                           dvals, dbias, workspace, workspace_bytes,
                           flags & ~(kBwdSgdUpdate | kBwdHot | kBwdSolo | kBwdScaled | (step ? FLEXSAE_BWD_RAGGED_ROWS : 0)),
                           status_flag, stream, step, grad_out, stats, stats_tag);
}

int flexsae_scale(void *dst, const void *src, int dtype, int64_t n, const float *scale, void *stream) {
  if (!dst || !src || !scale || n < 0 || !valid_dtype(dtype)) return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (n == 0) return FLEXSAE_OK;
  if (!aligned(src, 4 * dtype_size(dtype)) || !aligned(dst, 4 * dtype_size(dtype)) || !aligned(scale, 4))
    return FLEXSAE_ERR_ALIGNMENT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid(grid_for(ceil_div(n, 4), 256, 4096));  // few blocks: in place by one they all return at once
  switch (dtype) {
    case FLEXSAE_F32:
      hipLaunchKernelGGL(scale_kernel<float>, grid, dim3(256), 0, st, dst, src, n, scale);
      break;
    case FLEXSAE_BF16:
      hipLaunchKernelGGL(scale_kernel<bf16_t>, grid, dim3(256), 0, st, dst, src, n, scale);
      break;
    default:
      hipLaunchKernelGGL(scale_kernel<f16_t>, grid, dim3(256), 0, st, dst, src, n, scale);
  }
  return launch_status();
}

size_t flexsae_csr_workspace_bytes(int64_t B, int64_t K, int64_t F) {
  if (B <= 0 || K <= 0 || F <= 0) return 0;
  if (B > ((1LL << 32) - 1) / K) return 0;
  return csr_scratch_bytes(B * K, F, nullptr, nullptr);
}

int flexsae_csr_build(const int64_t *indices, int64_t B, int64_t K, int64_t F, uint32_t *begin,
                      uint32_t *map, void *workspace, size_t workspace_bytes, int *status_flag,
                      void *stream) {
  if (!indices || !begin || !map || B <= 0 || K <= 0 || F <= 0) return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (F >= (1LL << 31) || B > ((1LL << 32) - 1) / K) return FLEXSAE_ERR_UNSUPPORTED;
  if (!aligned(indices, 8) || !aligned(begin, 4) || !aligned(map, 4)) return FLEXSAE_ERR_ALIGNMENT;
  if (!workspace || workspace_bytes < flexsae_csr_workspace_bytes(B, K, F) ||
      !aligned(workspace, kAlign))
    return FLEXSAE_ERR_WORKSPACE;
  const CsrScratch sc = carve_csr_scratch(workspace, F, B * K);
  csr_build_launch(indices, B, K, F, begin, map, nullptr, nullptr, sc, status_flag, static_cast<hipStream_t>(stream));
  return launch_status();
}

size_t flexsae_topk_bwd_workspace_bytes(const flexsae_shape *s, int64_t slice_cols) {
  if (check_shape(s) != FLEXSAE_OK) return 0;
  // The query takes no flags, so it covers both layouts of the call: the bf16-residual one (wide
  // tiles plus the bf16 copy of the residual) and the FLEXSAE_TOPK_BWD_FP32_RESIDUAL one (narrower
  // tiles: twice the per-tile dvals shares, which outweighs the copy once K exceeds 256).
  size_t need = 0;
  for (const int flags : {0, static_cast<int>(FLEXSAE_TOPK_BWD_FP32_RESIDUAL), static_cast<int>(FLEXSAE_TOPK_BWD_AS_LARGE)}) {
    const TopkBwdPlan pl = plan_topk_bwd(s, flags);
    int64_t sw = slice_cols <= 0 ? pl.tile : ceil_div(slice_cols, pl.tile) * pl.tile;
    if (sw > pl.d_pad) sw = pl.d_pad;
    const size_t bytes = topk_bwd_bytes(pl, sw);
    if (bytes > need) need = bytes;
  }
  return need;
}

int flexsae_topk_bwd(const flexsae_shape *s, const uint32_t *begin, const uint32_t *map,
                     const int64_t *indices, const void *weight, const void *vals, const float *resid,
                     const float *grad_out, void *dW, int dW_dtype, float *dvals, float *dbias,
                     void *workspace, size_t workspace_bytes, int flags, void *stream) {
  int rc = check_shape(s);
  if (rc != FLEXSAE_OK) return rc;
  if (!begin || !map || !weight || !vals || !resid || !grad_out || !dW || !dvals || !dbias ||
      !valid_dtype(dW_dtype))
    return FLEXSAE_ERR_INVALID_ARGUMENT;
  // the residual rows are gathered through a 32-bit buffer descriptor
  if (static_cast<size_t>(s->B) * static_cast<size_t>(s->D) * 4 > 0xffffffffull) return FLEXSAE_ERR_UNSUPPORTED;
  const TopkBwdPlan pl = plan_topk_bwd(s, flags);
  if (!aligned(begin, 4) || !aligned(map, 4) || !aligned(dvals, 16) || !aligned(dbias, 4)) return FLEXSAE_ERR_ALIGNMENT;
  rc = check_topk_bwd(s, pl, indices, weight, vals, resid, grad_out, dW, dW_dtype);
  if (rc != FLEXSAE_OK) return rc;
  if (!workspace || !aligned(workspace, kAlign) || workspace_bytes < least_topk_bwd_bytes(pl)) return FLEXSAE_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint8_t *ws = static_cast<uint8_t *>(workspace);
  // (every output element is written exactly once: nothing needs a zero-fill, whatever `flags` says)
  launch_topk_prepare(s, pl, begin, map, indices, vals, resid, ws, st);
  launch_topk_bwd(s, pl, begin, map, weight, vals, resid, grad_out, dW, dW_dtype,
                  LeafGrads{dvals, dbias, FLEXSAE_F32, FLEXSAE_F32}, ws, workspace_bytes, st);
  return launch_status();
}

size_t flexsae_topk_bwd_from_indices_workspace_bytes(const flexsae_shape *s, int64_t slice_cols) {
  if (check_shape(s) != FLEXSAE_OK) return 0;
  return plan_topk_list(s).bytes + flexsae_topk_bwd_workspace_bytes(s, slice_cols);
}

int flexsae_topk_bwd_from_indices(const flexsae_shape *s, const int64_t *indices, const void *weight, const void *vals,
                                  const float *resid, const float *grad_out, void *dW, int dW_dtype, void *dvals,
                                  int dvals_dtype, void *dbias, int dbias_dtype, void *workspace, size_t workspace_bytes,
                                  int flags, int *status_flag, void *stream) {
  int rc = check_shape(s);
  if (rc != FLEXSAE_OK) return rc;
  if (!indices || !weight || !vals || !resid || !grad_out || !dW || !dvals || !dbias || !valid_dtype(dW_dtype) ||
      !valid_dtype(dvals_dtype) || !valid_dtype(dbias_dtype))
    return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (static_cast<size_t>(s->B) * static_cast<size_t>(s->D) * 4 > 0xffffffffull) return FLEXSAE_ERR_UNSUPPORTED;
  const TopkBwdPlan pl = plan_topk_bwd(s, flags);
  if (!aligned(dvals, dtype_size(dvals_dtype)) || !aligned(dbias, dtype_size(dbias_dtype)) || !aligned(status_flag, 4))
    return FLEXSAE_ERR_ALIGNMENT;
  rc = check_topk_bwd(s, pl, indices, weight, vals, resid, grad_out, dW, dW_dtype);
  if (rc != FLEXSAE_OK) return rc;
  const TopkListPlan lp = plan_topk_list(s);
  if (!workspace || !aligned(workspace, kAlign) || workspace_bytes < lp.bytes + least_topk_bwd_bytes(pl))
    return FLEXSAE_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint32_t *begin = static_cast<uint32_t *>(workspace);
  uint32_t *map = reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(workspace) + lp.off_map);
  uint8_t *ws = static_cast<uint8_t *>(workspace) + lp.bytes;
  CsrScratch sc = carve_csr_scratch(static_cast<uint8_t *>(workspace) + lp.off_csr, s->F, s->B * s->K);
  const CsrPlan &cp = sc.plan;
  if (cp.bucketed) {
    const size_t lds = (round_up(cp.n_buckets, 4) + 1) * kChunkWaves * 4;
    const int cols = static_cast<int>(s->D);
    const int64_t n_resid_blocks = resid_blocks(s->B, cols, pl.resid16 ? pl.resid_ld : cols);
    const PairLists lists = carve_topk_lists(s, pl, ws);
    hipLaunchKernelGGL(topk_front_kernel, dim3(cp.n_chunks + static_cast<unsigned>(n_resid_blocks)),
                       dim3(kChunkThreads), lds, st, indices, s->B * s->K, s->F, cp.shift, cp.pack_shift, cp.n_buckets,
                       cp.n_bits, cp.chunk, cp.n_chunks, sc.table, sc.tmp, lists.ctrl, status_flag, resid, s->B, cols,
                       pl.resid_ld, pl.resid16 ? static_cast<void *>(ws + pl.off_resid16) : nullptr,
                       reinterpret_cast<float *>(ws + pl.off_colsum));
    const PairRecords rec = {vals, indices, reinterpret_cast<vec_t<uint32_t, 2> *>(ws + pl.off_slotbv), s->vals_dtype,
                             static_cast<uint32_t>(s->K)};
    launch_bucket_sort<true>(sc, s->F, begin, map, nullptr, nullptr, 0u, lists, rec, st);
  } else {
    csr_build_launch(indices, s->B, s->K, s->F, begin, map, nullptr, nullptr, sc, status_flag, st);
    launch_topk_prepare(s, pl, begin, map, indices, vals, resid, ws, st);
  }
  launch_topk_bwd(s, pl, begin, map, weight, vals, resid, grad_out, dW, dW_dtype,
                  LeafGrads{dvals, dbias, dvals_dtype, dbias_dtype}, ws, workspace_bytes - lp.bytes, st);
  return launch_status();
}

int flexsae_scale_from_f32(void *dst, int dst_dtype, const float *src, int64_t n, const float *scale,
                           void *stream) {
  if (!dst || !src || n < 0 || !valid_dtype(dst_dtype)) return FLEXSAE_ERR_INVALID_ARGUMENT;
  if (n == 0) return FLEXSAE_OK;
  if (!aligned(src, 16) || !aligned(dst, 4 * dtype_size(dst_dtype)) || !aligned(scale, 4)) return FLEXSAE_ERR_ALIGNMENT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid(grid_for(ceil_div(n, 4), 256, 1 << 16));
  switch (dst_dtype) {
    case FLEXSAE_F32:
      hipLaunchKernelGGL(cast_from_f32_kernel<float>, grid, dim3(256), 0, st, dst, src, n, scale);
      break;
    case FLEXSAE_BF16:
      hipLaunchKernelGGL(cast_from_f32_kernel<bf16_t>, grid, dim3(256), 0, st, dst, src, n, scale);
      break;
    default:
      hipLaunchKernelGGL(cast_from_f32_kernel<f16_t>, grid, dim3(256), 0, st, dst, src, n, scale);
  }
  return launch_status();
}

int flexsae_finish_grads(void *dW, int dW_dtype, const void *dW_unit, int dW_unit_dtype, int64_t n_dw, void *dvals,
                         int dvals_dtype, const float *dvals_unit, int64_t n_dvals, void *dbias, int dbias_dtype,
                         const float *dbias_unit, int64_t n_dbias, const float *scale, void *stream) {
  if (n_dw < 0 || n_dvals < 0 || n_dbias < 0 || (n_dw > 0 && (!dW || !dW_unit)) || (n_dvals > 0 && (!dvals || !dvals_unit)) ||
      (n_dbias > 0 && (!dbias || !dbias_unit)) || !valid_dtype(dW_dtype) || !valid_dtype(dW_unit_dtype) ||
      !valid_dtype(dvals_dtype) || !valid_dtype(dbias_dtype) ||
      (dW_unit_dtype != dW_dtype && (dW_unit_dtype != FLEXSAE_F32 || dW == dW_unit)))
    return FLEXSAE_ERR_INVALID_ARGUMENT;
  if ((n_dw > 0 && (!aligned(dW, 4 * dtype_size(dW_dtype)) || !aligned(dW_unit, 4 * dtype_size(dW_unit_dtype)))) ||
      (n_dvals > 0 && (!aligned(dvals, 4 * dtype_size(dvals_dtype)) || !aligned(dvals_unit, 16))) ||
      (n_dbias > 0 && (!aligned(dbias, 4 * dtype_size(dbias_dtype)) || !aligned(dbias_unit, 16))) || !aligned(scale, 4))
    return FLEXSAE_ERR_ALIGNMENT;
  if (n_dw + n_dvals + n_dbias == 0) return FLEXSAE_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const unsigned n_small = 1 + grid_for(ceil_div(n_dvals, 4), 256, 1024);
  // in place: few blocks, since by one they all return at once
  const unsigned n_large = n_dw == 0 ? 0 : grid_for(ceil_div(n_dw, 4), 256, dW == dW_unit ? 2048 : 1 << 16);
#define FLEXSAE_FINISH(UT, GT)                                                                                             \
  hipLaunchKernelGGL((finish_grads_kernel<UT, GT>), dim3(n_small + n_large), dim3(256), 0, st, dW, dW_unit, n_dw, dvals,   \
                     dvals_dtype, dvals_unit, n_dvals, dbias, dbias_dtype, dbias_unit, n_dbias, scale, n_small)
  if (dW_unit_dtype == FLEXSAE_F32) {
    if (dW_dtype == FLEXSAE_F32) FLEXSAE_FINISH(float, float);
    else if (dW_dtype == FLEXSAE_BF16) FLEXSAE_FINISH(float, bf16_t);
    else FLEXSAE_FINISH(float, f16_t);
  } else if (dW_unit_dtype == FLEXSAE_BF16) {
    FLEXSAE_FINISH(bf16_t, bf16_t);
  } else {
    FLEXSAE_FINISH(f16_t, f16_t);
  }
#undef FLEXSAE_FINISH
  return launch_status();
}

int flexsae_cast_from_f32(void *dst, int dst_dtype, const float *src, int64_t n, void *stream) {
  return flexsae_scale_from_f32(dst, dst_dtype, src, n, nullptr, stream);
}

}  // extern "C"
