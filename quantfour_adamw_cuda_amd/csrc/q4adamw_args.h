// Launch arguments of the kernels (passed by value in the kernarg segment) and the constant
// tables they read.  Shared by the kernels and the host launchers of q4adamw.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/q4adamw.h"
#include "q4adamw_tables.h"

namespace q4 {


constexpr int kWaves = 4;                  // waves per workgroup
constexpr int kThreads = kWaves * 64;
constexpr int kMaxTensors = 61;            // tensors per fused launch: as many as 4 KiB of arguments hold
constexpr int kSmallChunk = 1024;          // elements per workgroup, non-quantized kernel
// As many as 4 KiB of arguments hold.  A launch costs 4 to 5 us of device time however little it
// does, so a batch of one launch instead of two is worth a denser descriptor: GPT-2-small's 98 small and 50
// quantized tensors took two launches of each kind with 80 and 48, 358.6 us a clipped step
// against 350.9 with one of each.
constexpr int kMaxSmallTensors = 103;

// derived on the host exactly as optim/cuda_adamw_kernels.cu:435-440
struct StepConsts {
  float b1, b2, r1, r2;  // beta1, beta2, 1-beta1, 1-beta2
  float wdu, ss;         // 1 - lr*wd, lr / (1 - beta1^t)
  float c2s;             // sqrt(1 - beta2^t)
  float eps;
  // the fused kernel's parameter update in its folded form, p*wdu - m'/(sqrt(v')*den_scale +
  // den_eps), the step size folded into the denominator: 1/(c2s*ss) and eps/ss
  float den_scale, den_eps;
  // For the correctly rounded form of the update: RN(1 / c2s), which sqrt(v') is divided by
  // c2s with (div_by_reciprocal), and whether eps and c2s lie where that form's short
  // sequences hold (non-zero: 2^-60 <= eps <= 2^60, 2^-13 <= c2s <= 1; otherwise every lane
  // takes the general expansions).
  float c2s_rcp;
  uint32_t exact_short;
};

// (float)(1.0 / (double)c) is RN(1/c): rounding a quotient twice is harmless when the wide
// format has at least 2 * 24 + 2 bits (host and device: fp64 division is IEEE on both).
__host__ __device__ inline void make_exact_consts(StepConsts *sc) {
  sc->c2s_rcp = (float)(1.0 / (double)sc->c2s);
  sc->exact_short = (sc->eps >= 8.673617379884035e-19f && sc->eps <= 1.152921504606847e+18f &&
                     sc->c2s >= 1.220703125e-4f && sc->c2s <= 1.0f) ? 1u : 0u;
}

// What a launch does to the gradients besides reading them (kernels with EXT only).
struct GradOps {
  float scale;             // host part of the multiplier
  uint32_t zero;           // non-zero: overwrite the gradients with zeros once they are read
  const float *scale_dev;  // device part of the multiplier, or null
  const float *skip;       // device flag, or null: non-zero turns the launch into a no-op
  const StepConsts *sc_dev;  // the step's derived scalars in device memory (device_step_kernel), or null
};

// Which chunk of a grid a workgroup takes.  Workgroups are dealt to the 8 XCDs in turn; with runs
// of 2^shift consecutive chunks per XCD (the first `grouped` workgroups; the rest take the chunk of
// their own number) neighbouring blocks' 4-byte scales meet in one L2, and all XCDs still
// work through the same stretch of memory together.  One eighth of the grid per XCD, as this
// was before, serves the scales as well but keeps eight far-apart stretches open at once and
// leaves XCDs idle when the work is uneven: one fp32 4096 x 4096 tensor 41.3-43.6 us against
// 37.8 with runs of 64, GPT-2-small's large launch 273-285 against 261-279, Llama-2-13B layers
// (bf16) 2066-2090 against 2030, Llama-3-8B layers and tables with half of the embedding's rows
// never touched 4200 against 3825.  Runs of 1, 4, 16, 64, 128, 256, 1024 on the last: 3887, 4012,
// 3943, 3825, 3857, 3841, 3839; on the 4096 x 4096 tensor: 40.4, 40.4, 38.3, 37.8, 38.2, 39.8, 41.0.
struct ChunkRuns {
  uint32_t shift;
  uint32_t grouped;   // a multiple of 8 << shift
};

// Runs of 1024 chunks in grids where every XCD gets 64 of them (2^19 chunks), otherwise of 64 or, in grids too
// small for 64 of those, the longest that leave every XCD 64.  Both sides of the line, medians of ten rounds in
// turn in one process, the range over four cards, us a step with runs of 64 / 1024 / one eighth of the grid per
// XCD; fp32 parameters and bf16 gradients, Llama-3-8B's layers:
//     426000 chunks   838-854      841-856      847-855
//     852000 chunks   1694-1718    1686-1710    1694-1711
//    1704000 chunks   3407-3453    3373-3439    3391-3438
//    7842048 chunks   15744-16004  15642-15871  15719-15904   (the whole set)
// i.e. 0.5 to 0.8 % on the whole set, on every card.  All in fp32 or in bf16 the line could lie higher: 852000
// chunks 1888-1909 / 1897-1909 / 1926-1935 and 2189-2200 / 2206-2210 / 2250-2269.  The 4096 x 4096 tensor in
// fp32 (runs of 32): 38.5, 38.3 with runs of 64, 37.9 with 256, 41.5 with one eighth.
__host__ inline ChunkRuns make_chunk_runs(uint32_t count) {
  ChunkRuns r = {(count >> 13) >= 64u ? 10u : 6u, 0u};
  while (r.shift > 0u && (count >> (r.shift + 3u)) < 64u) --r.shift;
  r.grouped = (count >> (r.shift + 3u)) << (r.shift + 3u);
  return r;
}

__device__ __forceinline__ uint32_t run_chunk(const ChunkRuns &r, uint32_t workgroup) {
  const uint32_t turn = workgroup >> 3, run = ((turn >> r.shift) << 3) + (workgroup & 7u);
  const uint32_t chunk = (run << r.shift) + (turn & ((1u << r.shift) - 1u));
  return workgroup < r.grouped ? chunk : workgroup;
}

struct TensorDesc {  // 56 bytes
  void *p;
  const void *g;
  uint8_t *m;
  uint8_t *v;
  float *sm;
  float *sv;
  int64_t numel;
};

// Kernel arguments of one fused launch (nearly 4 KiB, passed by value).
// first_chunk[i] = index of tensor i's first chunk; entries past ntensors hold
// 0x7fffffff (more than any chunk index).  pivot[k] = first_chunk[8k] lets a workgroup find its tensor with two
// wide scalar loads.
struct FusedArgs {
  static constexpr int kCapacity = kMaxTensors;
  static constexpr int kPivots = (kMaxTensors + 7) / 8;
  StepConsts sc;
  GradOps go;
  int ntensors;
  // A batch's chunks run in one grid or, beyond what a grid may hold, in several: this grid
  // takes the chunks from chunk_base on, one per workgroup.
  uint32_t chunk_base;
  ChunkRuns runs;
  uint32_t pivot[kPivots];
  uint32_t first_chunk[kPivots * 8];
  TensorDesc desc[kMaxTensors];
  // stochastic rounding: the tensors' noise salts of this step; with a step number on the
  // device (go.sc_dev) the hash of each tensor's own salt, which the kernel carries on
  // through step number and seed
  uint32_t sr_salt[kMaxTensors];
  uint32_t seed_lo, seed_hi;
};

struct SmallDesc {  // 32 bytes
  void *p;
  const void *g;
  float *m;
  float *v;
};

struct SmallArgs {
  static constexpr int kCapacity = kMaxSmallTensors;
  static constexpr int kPivots = (kMaxSmallTensors + 1 + 7) / 8;   // first_chunk[ntensors] is there too
  StepConsts sc;
  GradOps go;
  int ntensors;
  uint32_t chunk_base;     // this grid's first chunk (workgroup 0)
  uint32_t pivot[kPivots];
  uint32_t first_chunk[kPivots * 8];
  SmallDesc desc[kMaxSmallTensors];
  uint16_t last[kMaxSmallTensors];   // elements of the tensor's last chunk, 1 .. kSmallChunk
};

// One tensor whose second moment is rank-1 scaled (a rows x cols matrix, row-major).
struct Rank1Desc {  // 104 bytes
  void *p;
  const void *g;
  uint8_t *m;
  uint8_t *v;
  float *sm;          // block scales of the first moment
  float *rmax;        // current statistics of the second moment: rows, cols floats
  float *cmax;
  float *rmax_next;   // the step's new statistics (all zero between steps)
  float *cmax_next;
  int64_t numel;      // rows * cols
  int64_t rows;
  int64_t cols;
  // division of a 32-bit number by cols / 8 (rows form of the update kernel: by the number
  // of tiles in a row) as multiply-high, add and shifts
  // (round-up method: exact for every 32-bit dividend)
  uint32_t div_magic;
  uint32_t div_shift;
};

struct FastDiv {
  uint32_t magic, shift;
};

// n / d for the divisor the pair was made for
__host__ __device__ __forceinline__ uint32_t fast_div(uint32_t n, uint32_t magic, uint32_t shift) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t t = __umulhi(n, magic);
#else
  const uint32_t t = (uint32_t)(((uint64_t)n * magic) >> 32);
#endif
  return (t + ((n - t) >> 1)) >> shift;
}

// divisors from 1 on (a size of 1 has the magic number 0, which no other has)
__host__ __device__ __forceinline__ uint32_t fast_div_any(uint32_t n, uint32_t magic, uint32_t shift) {
  return magic == 0u ? n : fast_div(n, magic, shift);
}

static FastDiv make_fast_div(uint32_t d) {  // d >= 2
  uint32_t l = 0;
  while ((1ull << l) < d) ++l;                     // ceil(log2 d) >= 1
  FastDiv f;
  f.magic = (uint32_t)((((1ull << l) - d) << 32) / d + 1);
  f.shift = l - 1;
  return f;
}

constexpr int kMaxRank1Tensors = 32;

// Kernel arguments of the rank-1 launches.  The update kernel indexes chunks of
// kChunk flat elements like FusedArgs.
struct Rank1Args {
  static constexpr int kCapacity = kMaxRank1Tensors;
  static constexpr int kPivots = (kMaxRank1Tensors + 7) / 8;
  StepConsts sc;
  GradOps go;
  int ntensors;
  uint32_t chunk_base;     // as FusedArgs
  ChunkRuns runs;
  uint32_t pivot[kPivots];
  uint32_t first_chunk[kPivots * 8];
  uint32_t sr_salt[kMaxRank1Tensors];   // stochastic rounding: as FusedArgs::sr_salt
  uint32_t seed_lo, seed_hi;
  Rank1Desc desc[kMaxRank1Tensors];
};

// The same for tensors with several leading dimensions and short rows, of fewer than 2^32 elements, whose update
// reads the leading dimensions' statistics themselves.
constexpr int kMaxShortTensors = 25;
constexpr uint32_t kShortMaxCols = 64;

struct ShortDesc {  // 144 bytes
  void *p;
  const void *g;
  uint8_t *m;
  uint8_t *v;
  float *sm;
  float *rmax;              // rows' scales, written
  const float *cmax;
  const float *cmax_next;
  // statistics of the last leading dimension, the one before it and the first of three (of two: the first again)
  const float *last, *before, *outer;
  const float *last_next, *before_next, *outer_next;
  uint32_t numel;
  uint32_t last_size, before_size;
  uint32_t cols_magic, last_magic, before_magic;   // divisions by cols and by the two sizes (fast_div)
  uint16_t cols;
  uint8_t cols_shift, last_shift, before_shift;
  uint8_t lead_dims;        // 2 or 3
};

struct ShortArgs {
  static constexpr int kCapacity = kMaxShortTensors;
  static constexpr int kPivots = (kMaxShortTensors + 7) / 8;
  StepConsts sc;
  GradOps go;
  int ntensors;
  uint32_t chunk_base;     // as FusedArgs
  ChunkRuns runs;
  uint32_t pivot[kPivots];
  uint32_t first_chunk[kPivots * 8];
  uint32_t sr_salt[kMaxShortTensors];
  uint32_t seed_lo, seed_hi;
  ShortDesc desc[kMaxShortTensors];
};

// The statistics kernels index tiles of a matrix (rank1_stat_chunks).  A tensor with two or
// three leading dimensions is the matrix [their product, last dimension]; its rows' maxima go
// straight into one statistic per leading dimension (lead_next) and `rmax_next` is left alone.
// Row and column counts fit 32 bits (2^35 - 1 elements, at least 16 columns above 2^32).
struct Rank1StatArgs {
  static constexpr int kCapacity = kMaxRank1Tensors;
  static constexpr int kPivots = (kMaxRank1Tensors + 7) / 8;
  float b2, r2;
  GradOps go;
  uint32_t chunk_base;     // this grid's first tile (workgroup 0)
  ChunkRuns runs;          // wide forms: which tile a workgroup takes
  // rows of a workgroup (flat form: at most, but for one tile; lead form: indices of the first dimension): 32, 64, 128 or 256
  uint32_t stat_rows;
  uint32_t lead_runs;      // lead form: runs of a workgroup, at most
  uint32_t pivot[kPivots];
  uint32_t first_chunk[kPivots * 8];
  struct Desc {  // 120 bytes
    const void *g;
    const uint8_t *v;
    const float *rmax;
    const float *cmax;
    float *rmax_next;
    float *cmax_next;
    float *lead_next[3];
    const float *lead_old[3];
    uint32_t lead_shape[3];
    uint32_t lead_dims;    // 0, 2 or 3
    uint32_t rows;
    uint32_t cols;
  } desc[kMaxRank1Tensors];
};

// Between statistics and update of tensors with several leading dimensions: the rows' new
// scales, each the minimum over its leading statistics.  Chunks of kRowScaleChunk rows.
constexpr int kRowScaleChunk = 2048;

struct RowScaleArgs {
  static constexpr int kCapacity = kMaxRank1Tensors;
  static constexpr int kPivots = (kMaxRank1Tensors + 7) / 8;
  GradOps go;
  uint32_t pivot[kPivots];
  uint32_t first_chunk[kPivots * 8];
  struct Desc {  // 64 bytes
    float *row_next;
    const float *lead_next[3];
    uint32_t lead_shape[3];
    uint32_t lead_dims;
    uint32_t rows;
    uint32_t pad_;
  } desc[kMaxRank1Tensors];
};

// After the update: every new statistic (rows, columns, leading dimensions) becomes the current
// one and its buffer returns to zero.  Chunks of kCommitChunk floats, each in one of a tensor's
// vectors.
constexpr int kCommitChunk = 2048;

struct CommitArgs {
  static constexpr int kCapacity = kMaxRank1Tensors;
  static constexpr int kPivots = (kMaxRank1Tensors + 7) / 8;
  GradOps go;
  uint32_t pivot[kPivots];
  uint32_t first_chunk[kPivots * 8];
  struct Desc {  // 104 bytes
    float *cur[5];    // rows, columns, leading dimensions (unused ones have size 0)
    float *next[5];
    uint32_t size[5];
    uint32_t pad_;
  } desc[kMaxRank1Tensors];
};

// Gradient-norm launch: every workgroup walks chunks of 32 KiB with a grid stride.
constexpr int kMaxNormTensors = 160;
constexpr int kNormPartials = Q4ADAMW_NORM_WORKSPACE_BYTES / 8;  // workgroups = fp64 partial sums
constexpr int kNormChunkBytes = 32768;                          // 8 16-byte loads per thread

struct NormDesc {
  const void *g;
  int64_t numel;
};

struct NormArgs {
  static constexpr int kCapacity = kMaxNormTensors;
  static constexpr int kPivots = (kMaxNormTensors + 7) / 8;
  double *partials;   // kNormPartials sums, one per workgroup
  uint32_t nchunks;
  uint32_t first;     // non-zero: the partial sums are overwritten, otherwise added to
  int ntensors;
  uint32_t pivot[kPivots];
  uint32_t first_chunk[kPivots * 8];
  NormDesc desc[kMaxNormTensors];
};

static_assert(sizeof(StepConsts) <= Q4ADAMW_STEP_CONSTS_BYTES, "the device copy of a step's scalars");
static_assert(sizeof(FusedArgs) <= 4096 && sizeof(SmallArgs) <= 4096 && sizeof(NormArgs) <= 4096 &&
                  sizeof(Rank1Args) <= 4096 && sizeof(ShortDesc) == 144 && sizeof(ShortArgs) <= 4096 && sizeof(Rank1StatArgs) <= 4096 && sizeof(RowScaleArgs) <= 4096 &&
                  sizeof(CommitArgs) <= 4096,
              "kernel arguments are limited to 4 KiB");

// the first-moment bucket table (see q4adamw_tables.h), copied into LDS by every
// workgroup at start-up, one entry per thread
__device__ const HalfTable kHalfTable = make_half_table();
// stochastic rounding: code-book entries per bucket and the 17 intervals between them
__device__ const SrHalfTable kSrHalfTable = make_sr_half_table();
__device__ const SrIntervalTable kSrIntervals = make_sr_interval_table();
__device__ const SrAffineTable kSrFixed = make_sr_fixed_table();
// first-moment code book for kernels that index it per lane
__device__ const uint32_t kQmapMDev[16] = {
    0xbf633333u, 0xbf29999au, 0xbee00000u, 0xbe59999au, 0xbd9eb852u, 0xbd051eb8u,
    0xbbb43958u, 0x00000000u, 0x3bb43958u, 0x3d051eb8u, 0x3d9eb852u, 0x3e59999au,
    0x3ee00000u, 0x3f29999au, 0x3f633333u, 0x3f800000u};

}  // namespace q4
