// Rank-1 scaling of the second moment, the launches around the update kernels of
// q4adamw_step.h: statistics (new second moments reduced to row and column maxima, or to one
// statistic per dimension for tensors with several leading dimensions), those tensors' row
// scales, and the commit.
#pragma once
#include "q4adamw_device.h"

namespace q4 {

// Raises a statistic to u (a non-negative float's bits).  Maxima settle early, so most calls
// find the statistic already there: a value read too early is only too small, and then the
// atomic decides.  Unconditional atomics on statistics that many workgroups share are what such
// a launch waits for: 786432 rows x 3 leading statistics one by one took 4.6 ms.
__device__ __forceinline__ void raise_max(float *addr, uint32_t u) {
  unsigned int *const a = reinterpret_cast<unsigned int *>(addr);
  if (u > __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(a, u);
}

// The same without the look.  In the wide statistics form the atomic, for which nothing waits, costs less
// than the load that every workgroup would end with, from 16 workgroups for a column's statistic (4096 x
// 14336 fp32, four of them: 191 us against 195; 4000 x 512: 8.6 against 11.0) to 3906 (1000000 x 264: 253
// against 270).
__device__ __forceinline__ void atomic_max_bits(float *addr, uint32_t u) {
  atomicMax(reinterpret_cast<unsigned int *>(addr), u);
}

// A workgroup's share of the leading statistics: rows [row0, row0 + n) with their maxima in
// row_bits.  The rows are consecutive, so dimension j meets at most min(shape[j], n / stride + 2)
// of its indices: one LDS slot for each of them, all dimensions side by side (at most 2 n + 4
// words), then one update per slot, all of them in flight together.
template <typename Desc>
__device__ __forceinline__ void fold_rows(const Desc &T, uint32_t row0, uint32_t n, const uint32_t *row_bits,
                                          uint32_t *slots) {
  uint32_t first[3], count[3];   // per dimension: index of slot 0 (before the wrap at shape), slots
  uint32_t stride = 1, total = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {  // from the last leading dimension to the first
    const int j = (int)T.lead_dims - 1 - k;
    const uint32_t shape = j >= 0 ? T.lead_shape[j] : 1u;
    first[k] = row0 / stride;
    const uint32_t span = (row0 + n - 1) / stride - first[k] + 1;
    count[k] = j < 0 ? 0u : span < shape ? span : shape;
    total += count[k];
    stride *= shape;
  }
  for (uint32_t i = threadIdx.x; i < total; i += kThreads) slots[i] = 0u;
  __syncthreads();
  for (uint32_t r = threadIdx.x; r < n; r += kThreads) {
    const uint32_t u = row_bits[r];
    uint32_t q = row0 + r, base = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if (count[k] != 0u) {
        uint32_t slot = q - first[k];
        const uint32_t shape = T.lead_shape[(int)T.lead_dims - 1 - k], next = q / shape;
        if (count[k] == shape) slot %= shape;
        if (u > slots[base + slot]) atomicMax(&slots[base + slot], u);
        base += count[k];
        q = next;
      }
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < total; i += kThreads) {
    uint32_t slot = i;
    int k = 0;
    if (slot >= count[0]) { slot -= count[0]; k = 1; }
    if (k == 1 && slot >= count[1]) { slot -= count[1]; k = 2; }
    const int j = (int)T.lead_dims - 1 - k;
    const uint32_t base = k == 0 ? first[0] : k == 1 ? first[1] : first[2];
    if (slots[i] != 0u) raise_max(T.lead_next[j] + (base + slot) % T.lead_shape[j], slots[i]);
  }
}

// GT = kAbsValues: the statistics of |g| itself (fp32, no codes): what the checkpoint quantizer
// needs of a second moment it is handed.
constexpr int kAbsValues = 3;

constexpr int kStatRowsPerWave = 64;     // rows a wave walks, at most
constexpr int kStatRows = kStatRowsPerWave * kWaves;   // rows per workgroup of the statistics kernel, at most
constexpr int kStatCols = 512;           // columns per workgroup: 8 per lane

// The packed codes of PER (4 or 8) consecutive elements from element `elem` of a run whose first code is at
// the low (odd = 0) or high nibble of byte 0.  ANY: elem + odd may be odd, and the codes end in one byte more.
template <uint32_t PER, bool ANY>
__device__ __forceinline__ uint32_t load_part_codes(const void *run, uint32_t odd, uint32_t elem) {
  const uint32_t nibble = ANY ? odd + elem : elem;
  uint32_t w = PER == 8 ? __builtin_amdgcn_raw_buffer_load_b32(tile_rsrc(run), nibble >> 1, 0, kNtReadOnly)
                        : (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(tile_rsrc(run), nibble >> 1, 0, kNtReadOnly);
  if (ANY && (nibble & 1u) != 0u)
    w = (w >> 4) | (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(tile_rsrc(run), (nibble >> 1) + PER / 2, 0, kNtReadOnly) << (4 * PER - 4);
  return w;
}

// The codes of 4 elements in a matrix whose rows may begin at either nibble, in two steps: a load whose result nothing looks
// at before all loads of a group of rows are under way, and their place in it.  With load_part_codes the byte after
// an odd start is in a branch of its own, behind which every part of every odd row waited: a step of 97 x 511 fp32 elements took
// 17.7 us (now 13.5), 15.8 before gradients were read in parts, of 30000 x 1001 123 (103).  The 4 bytes of the window end with the codes'
// last byte; those of the matrix' first 4 elements, before which nothing may be read, begin with the first.
__device__ __forceinline__ uint32_t load_window(const uint8_t *run, int64_t run_first, uint32_t elem) {
  const uint32_t nibble = ((uint32_t)run_first & 1u) + elem, at_start = run_first == 0 && elem == 0u ? 2u : 0u;
  return __builtin_amdgcn_raw_buffer_load_b32(tile_rsrc(run - 2), (nibble >> 1) + (nibble & 1u) + at_start, 0, kNtReadOnly);
}

__device__ __forceinline__ uint32_t window_codes(uint32_t window, int64_t run_first, uint32_t elem) {
  const uint32_t odd = ((uint32_t)run_first + elem) & 1u;
  return window >> (run_first == 0 && elem == 0u ? 0u : 16u - 4u * odd);
}

// New second moments of a tile of stat_rows x kStatCols elements, reduced to row and
// column maxima (get_variance_tensor_statistics, adamw_fourbit_triton.py:738-746).  The
// arithmetic is the update kernel's, operation for operation, so the maxima are maxima
// of exactly the values that kernel quantizes.  The four waves of a workgroup share the
// columns and split the rows: every lane keeps 8 columns over its wave's rows, the waves'
// column maxima meet in LDS, and the tile issues one atomic per column and one per row
// (atomics on the column vector are what this kernel's time depends on most: a tile of
// 64 rows with four times as many of them took 1.25 to 2 times as long).  A wave walks 64 rows
// where the launch has workgroups enough for the chip (args.stat_rows = 256) and fewer in a
// small launch, which would otherwise wait for one wave's 16 rounds of loads (one 1000 x 512
// matrix: 30 us with 64 rows per wave); how many rows, and why, is said where the launch decides.
// ANY: rows of any length (at least 8).  A row may then start at either nibble of a byte of the
// codes, and the lane that would run past the row's end works on the row's last 8 columns
// instead: maxima do not mind columns seen twice.
template <int GT_, bool EXT, bool ANY>
__global__ __launch_bounds__(kThreads) void rank1_stats_kernel(const Rank1StatArgs args) {
  constexpr bool kAbs = GT_ == kAbsValues;
  constexpr int GT = kAbs ? Q4ADAMW_FP32 : GT_;
  constexpr int kAhead = 4;  // rows whose loads are in flight together
  // A lane's 8 columns.  Of 16-bit gradients they are consecutive, one 16-byte access; of fp32 ones two parts of 4
  // columns half a tile apart, so that a wave's access is one run of bytes: with 8 consecutive columns, two
  // accesses of every other 16 bytes, GPT-2-small in fp32 took 412 us a step against 391, a 4-bit encoding of
  // 14336 x 4096 elements 133 against 128, a step of 8000 x 9001 elements 327 against 314.
  constexpr int kParts = GT ? 1 : 2;
  constexpr uint32_t kPer = 8 / kParts;
  constexpr bool kWindow = ANY && kPer == 4;
  __shared__ uint32_t row_bits[4][kStatRows];       // row maxima of each 16-lane quarter of the row's wave
  __shared__ uint32_t col_bits[kWaves][kStatCols];  // column maxima of each wave
  const uint32_t chunk = args.chunk_base + run_chunk(args.runs, blockIdx.x);
  float gscale = 1.0f;
  if (EXT && !grad_ops_begin(args.go, gscale)) return;
  const int t = find_tensor(args, chunk);
  const auto &T = args.desc[t];
  const uint32_t local = chunk - args.first_chunk[t];
  const uint32_t groups = (T.cols + kStatCols - 1) / kStatCols;
  const uint32_t rg = local / groups, cg = local - rg * groups;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the tile's first column, and the lane's parts counted from there: all columns of a part are in the row
  uint32_t col0 = cg * kStatCols, part_elem[kParts];
  bool active[kParts];
#pragma unroll
  for (int h = 0; h < kParts; ++h) {
    part_elem[h] = (uint32_t)(h * (kStatCols / kParts) + lane * kPer);
    active[h] = col0 + part_elem[h] < T.cols;
  }
  if (ANY) {
    col0 = col0 < T.cols - kPer ? col0 : T.cols - kPer;
    const uint32_t last = T.cols - kPer - col0;
#pragma unroll
    for (int h = 0; h < kParts; ++h) part_elem[h] = part_elem[h] < last ? part_elem[h] : last;
  }
  const uint32_t stat_rows = args.stat_rows;
  const uint32_t tile_row0 = rg * stat_rows;
  const int tile_rows = (int)(T.rows - tile_row0 < stat_rows ? T.rows - tile_row0 : stat_rows);
  const int rows_per_wave = (int)(stat_rows / kWaves);
  const int wave_row0 = wave * rows_per_wave;                            // within the tile
  int nrows = tile_rows - wave_row0;                                      // rows of this wave
  nrows = nrows < 0 ? 0 : (nrows > rows_per_wave ? rows_per_wave : nrows);
  // lanes past the last column work on zeros: code 0 under a zero scale and a zero
  // gradient give a zero second moment, which leaves every maximum alone
  float c_old[8], c_max[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    c_old[k] = active[k / kPer] && !kAbs ? as_global<const float>(T.cmax)[col0 + part_elem[k / kPer] + k % kPer] : 0.0f;
    c_max[k] = 0.0f;
  }
  const uint32_t quarter = (uint32_t)lane >> 4;
  for (int r0 = 0; r0 < nrows; r0 += kAhead) {
    // a group past the wave's last row repeats that row: maxima do not mind
    u32x4 gw[kAhead][kParts];
    uint32_t vw[kAhead][kParts];
    float r_old[kAhead];
    int64_t run_first[kAhead];   // uniform
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int r = r0 + i < nrows ? r0 + i : nrows - 1;
      const uint32_t row = tile_row0 + wave_row0 + r;
      r_old[i] = kAbs ? 0.0f : as_global<const float>(T.rmax)[row];
      // row bases are uniform; the lane's column is a 32-bit offset
      const int64_t row_first = run_first[i] = (int64_t)row * T.cols + col0;
      const void *g_row = static_cast<const char *>(T.g) + row_first * (GT ? 2 : 4);
      const uint8_t *v_row = T.v + (row_first >> 1);
#pragma unroll
      for (int h = 0; h < kParts; ++h) {
        vw[i][h] = 0u;
        gw[i][h] = u32x4{0u, 0u, 0u, 0u};
        if (active[h]) {
          if (!kAbs)
            vw[i][h] = kWindow ? load_window(v_row, row_first, part_elem[h]) : load_part_codes<kPer, ANY>(v_row, (uint32_t)row_first & 1u, part_elem[h]);
          gw[i][h] = __builtin_amdgcn_raw_buffer_load_b128(tile_rsrc(g_row), part_elem[h] * (GT ? 2u : 4u), 0, kNtReadOnly);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      float g[8], code[8];   // codes as numbers, 0 .. 15
#pragma unroll
      for (int h = 0; h < kParts; ++h) {
        const u32x4 w = gw[i][h];
        if constexpr (GT != 0) {
          widen_pair<GT>(w.x, g[0], g[1]);
          widen_pair<GT>(w.y, g[2], g[3]);
          widen_pair<GT>(w.z, g[4], g[5]);
          widen_pair<GT>(w.w, g[6], g[7]);
        } else {
          g[4 * h] = bits2f(w.x); g[4 * h + 1] = bits2f(w.y); g[4 * h + 2] = bits2f(w.z); g[4 * h + 3] = bits2f(w.w);
        }
        const uint32_t codes = kWindow ? window_codes(vw[i][h], run_first[i], part_elem[h]) : vw[i][h];
        const uint32_t even = codes & 0x0F0F0F0Fu, odd = (codes >> 4) & 0x0F0F0F0Fu;  // one code per byte
#pragma unroll
        for (uint32_t k = 0; k < kPer; ++k) code[kPer * h + k] = (float)(((k & 1 ? odd : even) >> (8 * (k >> 1))) & 0xffu);
      }
      float r_max = 0.0f;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float gk = EXT ? g[k] * gscale : g[k];
        const float code_value = __builtin_fmaf(code[k], 0.0625f, 0.0625f);  // (code + 1) / 16, exact
        const float v_old = code_value * min_nonneg(r_old[i], c_old[k]);
        const float v = kAbs ? __builtin_fabsf(gk) : args.b2 * v_old + args.r2 * (gk * gk);
        c_max[k] = __builtin_fmaxf(c_max[k], v);
        r_max = __builtin_fmaxf(r_max, v);
      }
      uint32_t u = f2bits(r_max);
      u = dpp_umax<0xB1>(u);
      u = dpp_umax<0x4E>(u);
      u = dpp_umax<0x141>(u);
      u = dpp_umax<0x140>(u);           // maximum of each 16-lane quarter, in all its lanes
      if ((lane & 15) == 0) row_bits[quarter][wave_row0 + r0 + i] = u;   // slots past the last row are not read
    }
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) col_bits[wave][k / kPer * (kStatCols / kParts) + lane * kPer + k % kPer] = f2bits(c_max[k]);
  __syncthreads();
  // one update per column of the tile, and one per row or per leading index of its rows
#pragma unroll
  for (int h = 0; h < kStatCols / kThreads; ++h) {
    const uint32_t c = (uint32_t)(tid + h * kThreads);
    uint32_t u = col_bits[0][c];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) u = u > col_bits[w][c] ? u : col_bits[w][c];
    const bool there = cg * kStatCols + (ANY ? c & ~(kPer - 1u) : c) < T.cols;
    uint32_t cc = cg * kStatCols + c;
    if (ANY) {   // the column that slot c's lane worked on
      const uint32_t first = c & ~(kPer - 1u), last = T.cols - kPer - col0;
      cc = col0 + (first < last ? first : last) + (c & (kPer - 1u));
    }
    if (there && u != 0u) atomic_max_bits(T.cmax_next + cc, u);
  }
  static_assert(kStatRows == kThreads, "one row per thread below");
  uint32_t u = row_bits[0][tid];
#pragma unroll
  for (int qi = 1; qi < 4; ++qi) u = u > row_bits[qi][tid] ? u : row_bits[qi][tid];
  if (T.lead_dims == 0u) {
    if (tid < tile_rows && u != 0u) {
      // A few rows of very many columns: what the launch waits for is the atomics on these rows' statistics, and once
      // the first tiles are through, nearly all of them find the maximum there.  With few tiles most of them start together, find
      // less and pay for the look as well.  us a step, atomics / with the look, in fp32 and bf16: 4 rows of 1024 tiles
      // 29.1 / 34.7 and 31.8 / 32.7, 8 of 1536 49.8 / 55.0 and 49.5 / 51.5, 3 of 2560 54.9 / 57.0 and 58.1 / 63.5; 1 row of 3072
      // 60.4 / 53.0 and 60.6 / 56.5, 3 of 3073 68.1 / 64.3 and 65.9 / 66.3, 8 of 3073 91.2 / 85.3 and 82.2 / 81.0, 4 of 9766
      // 194 / 128 and 179 / 120.  More rows share fewer updates each: 24 rows of 1024 tiles 59 / 69 and 48 / 53.
      if (T.rows <= 8u && groups > 3072u) raise_max(T.rmax_next + tile_row0 + tid, u);
      else atomic_max_bits(T.rmax_next + tile_row0 + tid, u);
    }
    return;
  }
  __syncthreads();          // every thread has read its row's quarters
  row_bits[0][tid] = u;
  __syncthreads();
  fold_rows(T, tile_row0, (uint32_t)tile_rows, row_bits[0], row_bits[1]);
}

// The same statistics for matrices of up to kFlatMaxCols columns: a tile is as many whole rows as fit
// kFlatWords elements (an odd row pitch, so that a walk along rows and one across them meet all
// banks), read as one run of consecutive elements: thread t's elements are t, t + k * cols,
// t + 2 * k * cols, ... (k rows a time), all of
// one column, whose maximum stays in a register.  The second moments meet the rows in LDS:
// a thread per row, or several where the tile has fewer than 256 rows.  A row lies in one
// workgroup, so its maximum is stored without an atomic.
// The forms it replaces here gave a lane to every column or to every 8th of them: with 3 columns
// (the last dimension of a 3x3 convolution kernel) 3 of 256 threads had work.
// In tall matrices a workgroup takes one tile after another until it has the rows of a wide form's tile
// (stat_rows), for the same reason, the updates of the columns' statistics: of an fp32 matrix of 100000 x 64
// 41 us with one tile, 26 with four; of four of 50000 x 64 75 and 38; of one of 1000000 x 100 154 and 143.
// Same arithmetic, operation for operation.
constexpr uint32_t kFlatMaxCols = 256, kFlatMaxCols8 = 88;   // the latter for multiples of 8
constexpr uint32_t kFlatWords = 4096;
constexpr uint32_t kFlatMaxRows = kFlatWords / 3;     // up to 3 columns: a pitch of 3 words

__host__ __device__ __forceinline__ uint32_t flat_tile_rows(uint32_t cols) { return cols < 3u ? kFlatMaxRows : kFlatWords / (cols | 1u); }

// tiles of a workgroup (one in short matrices, where they would only wait for each other: 1000 x 255 7.2 us
// with one, 9.8 with two)
__host__ __device__ __forceinline__ uint32_t flat_tiles(uint32_t cols, uint32_t stat_rows) {
  const uint32_t tiles = stat_rows / flat_tile_rows(cols);
  return stat_rows > 32u && tiles > 1u ? tiles : 1u;
}

template <int GT_, bool EXT>
__global__ __launch_bounds__(kThreads) void rank1_stats_flat_kernel(const Rank1StatArgs args) {
  constexpr bool kAbs = GT_ == kAbsValues;
  constexpr int GT = kAbs ? Q4ADAMW_FP32 : GT_;
  constexpr int kAhead = 8;   // elements of a thread whose loads are in flight together
  __shared__ float tile[kFlatWords];
  __shared__ uint32_t row_bits[kFlatMaxRows];
  __shared__ uint32_t col_bits[kFlatMaxCols];
  const uint32_t chunk = args.chunk_base + blockIdx.x;
  float gscale = 1.0f;
  if (EXT && !grad_ops_begin(args.go, gscale)) return;
  const int t = find_tensor(args, chunk);
  const auto &T = args.desc[t];
  const uint32_t tid = threadIdx.x, cols = T.cols, pitch = cols | 1u, tile_rows = flat_tile_rows(cols);
  const uint32_t tiles = flat_tiles(cols, args.stat_rows), tile0 = (chunk - args.first_chunk[t]) * tiles;
  if (tid < cols) col_bits[tid] = 0u;

  const uint32_t rows_per_pass = (uint32_t)kThreads / cols;
  const uint32_t r_first = tid / cols, col = tid - r_first * cols;
  float c_max = 0.0f;
  const float c_old = kAbs ? 0.0f : as_global<const float>(T.cmax)[col];
  for (uint32_t k = 0; k < tiles; ++k) {
    const uint32_t row0 = (tile0 + k) * tile_rows;
    if (row0 >= T.rows) break;                                // the first tile is always there
    const uint32_t n = T.rows - row0 < tile_rows ? T.rows - row0 : tile_rows;
    const uint32_t parts = n >= (uint32_t)kThreads ? 1u : (uint32_t)kThreads / n;   // threads per row
    if (k != 0u) __syncthreads();                             // the last tile's row maxima have been read
    if (parts > 1u && tid < n) row_bits[tid] = 0u;
    const int64_t first = (int64_t)row0 * cols;               // the tile's first element
    const void *g_tile = static_cast<const char *>(T.g) + first * (GT ? 2 : 4);
    const uint8_t *v_tile = T.v + (first >> 1);
    const uint32_t odd = (uint32_t)first & 1u;
    if (r_first < rows_per_pass) {
      for (uint32_t r0 = r_first; r0 < n; r0 += kAhead * rows_per_pass) {
        float g[kAhead], r_old[kAhead];
        uint32_t byte[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
          uint32_t r = r0 + (uint32_t)i * rows_per_pass;
          r = r < n ? r : r0;                                  // past the tile: a row seen already
          const uint32_t e = r * cols + col;
          g[i] = load_scalar<GT>(g_tile, e);
          byte[i] = kAbs ? 0u : as_global<const uint8_t>(v_tile)[(e + odd) >> 1];
          r_old[i] = kAbs ? 0.0f : as_global<const float>(T.rmax)[row0 + r];
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
          uint32_t r = r0 + (uint32_t)i * rows_per_pass;
          r = r < n ? r : r0;
          const float gi = EXT ? g[i] * gscale : g[i];
          const uint32_t code = (byte[i] >> (4u * ((r * cols + col + odd) & 1u))) & 15u;
          const float code_value = __builtin_fmaf((float)code, 0.0625f, 0.0625f);  // (code + 1) / 16, exact
          const float v_old = code_value * min_nonneg(r_old[i], c_old);
          const float v = __builtin_fmaxf(kAbs ? __builtin_fabsf(gi) : args.b2 * v_old + args.r2 * (gi * gi), 0.0f);   // a NaN never becomes a maximum
          c_max = __builtin_fmaxf(c_max, v);
          tile[r * pitch + col] = v;
        }
      }
    }
    __syncthreads();
    for (uint32_t i = tid; i < n * parts; i += kThreads) {
      const uint32_t r = i / parts, part = i - r * parts;
      float r_max = 0.0f;
      for (uint32_t c = part; c < cols; c += parts) r_max = __builtin_fmaxf(r_max, tile[r * pitch + c]);
      if (parts == 1u) row_bits[r] = f2bits(r_max);
      else if (r_max != 0.0f) atomicMax(&row_bits[r], f2bits(r_max));
    }
    __syncthreads();
    for (uint32_t r = tid; r < n; r += kThreads) as_global<uint32_t>(T.rmax_next)[row0 + r] = row_bits[r];
  }
  if (r_first < rows_per_pass && c_max != 0.0f) atomicMax(&col_bits[col], f2bits(c_max));
  __syncthreads();
  if (tid < cols && col_bits[tid] != 0u) raise_max(T.cmax_next + tid, col_bits[tid]);
}

// The same for tensors with several leading dimensions and at most kFlatMaxCols columns (a
// stack of 3x3 convolution kernels: [out, in, 3, 3]), straight to one statistic per dimension.
// What bounds such a kernel is not its bytes but the updates of statistics that every
// workgroup shares, which the memory side takes one after another: tiles of consecutive rows meet
// nearly all of the second dimension each (on 20 such stacks, 11 million elements, a kernel
// with those tiles took 23 us without its updates and 64 us with them).  So a tile is
// two-dimensional: indices of the first dimension (args.stat_rows, 32 to 256: lead_stat_outer) times a run of whole rows
// below it, which meets as many statistics of the first dimension and a few dozen of the second.
// A lane keeps N consecutive elements of the run, 16 bytes of gradients, and the workgroup's waves share the first
// dimension's indices.  Under one index after another the elements' other statistics stay the same, so a lane takes
// their minimum once and the first dimension's is one number for the wave; the maxima stay in registers until the end.
// With one element per lane, a load of each row's scale (4 bytes for every row of three elements) and 32 indices, steps
// of residual networks took, us, 64 wide in fp32 88 (now 79), 96 wide in bf16 174 (133), of [256, n, 64] with 41 million
// elements in fp32 213 (157), in bf16 166 (102).  With fewer elements below an index than a lane's N, every lane takes one
// (those past the end the first one again): all N of them in each lane, one load after another, made a step of [300000, 2, 3]
// with bf16 gradients 119 us (now 69; 84 with one element per lane everywhere).
constexpr uint32_t kLeadOuter = 32, kLeadMostOuter = 256;    // a round's indices; the most
constexpr uint32_t kLeadMostRows = 256, kLeadMostRuns = 16;  // rows and runs of a workgroup, at most

// elements of a run, at most (16 bytes of gradients per lane)
__host__ __device__ __forceinline__ constexpr uint32_t lead_run(bool half) { return half ? 512u : 256u; }

struct LeadTiles {
  uint32_t inner_rows;   // rows below one index of the first dimension
  uint32_t rows;         // of them in a run; the last run begins early enough to have as many
  uint32_t runs;         // along them
  uint32_t each;         // of a workgroup, one after another: so many that their rows are at most 256
  uint32_t inner;        // workgroups along them
};

__host__ __device__ __forceinline__ LeadTiles lead_tiles(uint32_t rows, uint32_t outer, uint32_t cols, uint32_t run, uint32_t each) {
  LeadTiles l;
  l.inner_rows = rows / outer;
  const uint32_t most = run / cols;
  l.runs = (l.inner_rows + most - 1u) / most;
  l.rows = (l.inner_rows + l.runs - 1u) / l.runs;   // evenly
  l.each = each == 1u || each * l.rows <= kLeadMostRows ? each : kLeadMostRows / l.rows;
  l.inner = (l.runs + l.each - 1u) / l.each;
  return l;
}

// RUNS: a workgroup takes several runs (lead_split), which cost the form with one of them 3 to 10 %.
template <int GT, bool EXT, bool RUNS>
__global__ __launch_bounds__(kThreads) void rank1_stats_lead_kernel(const Rank1StatArgs args) {
  constexpr uint32_t N = GT ? 8 : 4, kRun = lead_run(GT != 0), kSlots = 258;   // more than the rows, and than columns
  constexpr int kPerWave = kLeadOuter / kWaves;                // indices of the first dimension, all in flight together
  __shared__ uint32_t outer_bits[4][kLeadMostOuter];           // first dimension: each 16 lanes' maxima
  __shared__ float run_max[kWaves][kRun];                      // the run's elements
  __shared__ uint32_t slots[3][kSlots];                        // second and third dimension, columns
  const uint32_t chunk = args.chunk_base + blockIdx.x;
  float gscale = 1.0f;
  if (EXT && !grad_ops_begin(args.go, gscale)) return;
  const int t = find_tensor(args, chunk);
  const auto &T = args.desc[t];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, cols = T.cols, outer = T.lead_shape[0];
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const LeadTiles L = lead_tiles(T.rows, outer, cols, kRun, RUNS ? args.lead_runs : 1u);
  const uint32_t local = chunk - args.first_chunk[t], ot = local / L.inner, run0 = (local - ot * L.inner) * L.each;
  const uint32_t o0 = ot * args.stat_rows, no = outer - o0 < args.stat_rows ? outer - o0 : args.stat_rows;
  const uint32_t nruns = !RUNS ? 1u : L.runs - run0 < L.each ? L.runs - run0 : L.each;
  // maxima do not mind rows seen twice
  auto first_row = [&](uint32_t run) { return run * L.rows < L.inner_rows - L.rows ? run * L.rows : L.inner_rows - L.rows; };
  const uint32_t len = L.rows * cols;                          // elements of the run
  for (uint32_t i = tid; i < kSlots; i += kThreads) slots[0][i] = slots[1][i] = slots[2][i] = 0u;

  // this lane's elements, the same under every index of the first dimension: the last ones of the run for lanes
  // that would reach past its end, and of a run shorter than that a single one
  const bool whole = len >= N;
  const uint32_t elem = !whole ? (lane < len ? lane : 0u) : lane * N < len - N ? lane * N : len - N;
  const uint32_t shape2 = T.lead_dims == 3u ? T.lead_shape[2] : 1u;
  const gptr<const float> before = as_global<const float>(T.lead_old[1]), last = as_global<const float>(T.lead_old[2]);
  const uint32_t row0 = first_row(run0), first1 = row0 / shape2;   // the workgroup's first row and index of the second dimension
  for (uint32_t run = 0; run < nruns; ++run) {
    const uint32_t r0 = first_row(run0 + run);
    float s_old[N], x_max[N];
    {
      const uint32_t row = elem / cols;
      uint32_t col = elem - row * cols, i1 = (r0 + row) / shape2, i2 = r0 + row - i1 * shape2;
#pragma unroll
      for (uint32_t k = 0; k < N; ++k) {
        float s = 0.0f;
        if (whole || k == 0u) {
          s = min_nonneg(as_global<const float>(T.cmax)[col], before[i1]);
          if (T.lead_dims == 3u) s = min_nonneg(s, last[i2]);
        }
        s_old[k] = s;
        x_max[k] = 0.0f;
        const bool row_ends = ++col == cols;
        col = row_ends ? 0u : col;
        i2 += row_ends ? 1u : 0u;
        const bool wraps = i2 == shape2;
        i2 = wraps ? 0u : i2;
        i1 += wraps ? 1u : 0u;
      }
    }
    const int64_t below = (int64_t)L.inner_rows * cols;          // elements below one index
    const int64_t first = (int64_t)o0 * below + (int64_t)r0 * cols;
    u32x4 gw[kPerWave];
    uint32_t vw[kPerWave];
    float o_old[kPerWave];
    auto load = [&](uint32_t base, int i) {
      // past the first dimension's end: its last index once more
      const uint32_t mine = base + wave + (uint32_t)i * kWaves, o = mine < no ? mine : no - 1u;
      const int64_t e = first + (int64_t)o * below;              // uniform
      const void *g_run = static_cast<const char *>(T.g) + e * (GT ? 2 : 4);
      const void *v_run = T.v + (e >> 1);
      o_old[i] = as_constant<const float>(T.lead_old[0])[o0 + o];
      if (whole) {
        gw[i] = __builtin_amdgcn_raw_buffer_load_b128(tile_rsrc(g_run), elem * (GT ? 2u : 4u), 0, 0);
        vw[i] = load_part_codes<N, true>(v_run, (uint32_t)e & 1u, elem);
      } else {
        const uint32_t g_bits = GT != 0 ? (uint32_t)as_global<const uint16_t>(g_run)[elem] : as_global<const uint32_t>(g_run)[elem];
        gw[i] = u32x4{g_bits, 0u, 0u, 0u};
        vw[i] = as_global<const uint8_t>(v_run)[(((uint32_t)e & 1u) + elem) >> 1];
      }
    };
    auto reduce = [&](uint32_t base, int i) {
      float g[8];
      const u32x4 w = gw[i];
      if constexpr (GT != 0) {
        widen_pair<GT>(w.x, g[0], g[1]);
        widen_pair<GT>(w.y, g[2], g[3]);
        widen_pair<GT>(w.z, g[4], g[5]);
        widen_pair<GT>(w.w, g[6], g[7]);
      } else {
        g[0] = bits2f(w.x); g[1] = bits2f(w.y); g[2] = bits2f(w.z); g[3] = bits2f(w.w);
      }
      const uint32_t mine = base + wave + (uint32_t)i * kWaves, o = mine < no ? mine : no - 1u;
      // a single element's code is the low or the high half of its byte
      const uint32_t codes = whole ? vw[i] : vw[i] >> ((((uint32_t)(first + (int64_t)o * below) + elem) & 1u) * 4u);
      const uint32_t even = codes & 0x0F0F0F0Fu, odd = (codes >> 4) & 0x0F0F0F0Fu;  // one code per byte
      float o_max = 0.0f;
#pragma unroll
      for (uint32_t k = 0; k < N; ++k) {
        const float gk = EXT ? g[k] * gscale : g[k];
        const float code_value = __builtin_fmaf((float)(((k & 1 ? odd : even) >> (8 * (k >> 1))) & 0xffu), 0.0625f, 0.0625f);  // (code + 1) / 16, exact
        const float v_old = code_value * min_nonneg(o_old[i], s_old[k]);
        const float v = args.b2 * v_old + args.r2 * (gk * gk);     // a NaN never becomes a maximum
        x_max[k] = __builtin_fmaxf(x_max[k], v);
        if (whole || k == 0u) o_max = __builtin_fmaxf(o_max, v);
      }
      o_max = row_max16(o_max);
      if ((lane & 15u) == 0u) {
        uint32_t &slot = outer_bits[lane >> 4][mine];   // this lane's in every run
        slot = run != 0u && slot > f2bits(o_max) ? slot : f2bits(o_max);
      }
    };
    for (uint32_t base = 0; base < no; base += kLeadOuter) {
      if (no - base > kLeadOuter / 2) {
#pragma unroll
        for (int i = 0; i < kPerWave; ++i) load(base, i);
#pragma unroll
        for (int i = 0; i < kPerWave; ++i) reduce(base, i);
      } else {   // few indices are left: half as many rounds
#pragma unroll
        for (int i = 0; i < kPerWave / 2; ++i) load(base, i);
#pragma unroll
        for (int i = 0; i < kPerWave / 2; ++i) reduce(base, i);
      }
    }
#pragma unroll
    for (uint32_t k = 0; k < N; ++k) {
      if (whole || k == 0u) run_max[wave][elem + k] = x_max[k];
    }
    __syncthreads();
    for (uint32_t x = tid; x < len; x += kThreads) {
      float u = run_max[0][x];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) u = __builtin_fmaxf(u, run_max[w][x]);
      const uint32_t row = x / cols, i1 = (r0 + row) / shape2, i2 = r0 + row - i1 * shape2;
      auto raise_slot = [&](uint32_t &slot) {
        if (f2bits(u) > slot) atomicMax(&slot, f2bits(u));
      };
      raise_slot(slots[0][i1 - first1]);
      // the third dimension's indices of consecutive rows: there are fewer rows than slots, so rows that
      // share a slot share the index
      if (T.lead_dims == 3u) raise_slot(slots[1][shape2 < kSlots ? i2 : r0 - row0 + row]);
      raise_slot(slots[2][x - row * cols]);
    }
    __syncthreads();
  }
  static_assert(kLeadMostOuter <= kThreads, "one index per thread below");
  if (tid < no) {
    uint32_t u = outer_bits[0][tid];
#pragma unroll
    for (int k = 1; k < 4; ++k) u = u > outer_bits[k][tid] ? u : outer_bits[k][tid];
    if (u != 0u) raise_max(T.lead_next[0] + o0 + tid, u);
  }
  for (uint32_t i = tid; i < kSlots; i += kThreads) {
    if (slots[0][i] != 0u) raise_max(T.lead_next[1] + first1 + i, slots[0][i]);
    if (slots[1][i] != 0u) raise_max(T.lead_next[2] + (shape2 < kSlots ? i : (row0 + i) % shape2), slots[1][i]);
    if (slots[2][i] != 0u) raise_max(T.cmax_next + i, slots[2][i]);
  }
}

// Tensors with several leading dimensions, between statistics and update: every row's new scale
// is the minimum over its leading statistics.  A thread takes four consecutive rows a time: one
// division per dimension for the first, the others by counting on.
__global__ __launch_bounds__(256) void rank1_row_scale_kernel(const RowScaleArgs args) {
  float gscale;
  if (!grad_ops_begin(args.go, gscale)) return;
  const int t = find_tensor(args, blockIdx.x);
  const auto &T = args.desc[t];
  const uint32_t row0 = (blockIdx.x - args.first_chunk[t]) * kRowScaleChunk;
  const uint32_t n = T.rows - row0 < (uint32_t)kRowScaleChunk ? T.rows - row0 : (uint32_t)kRowScaleChunk;
  const gptr<float> out = as_global<float>(T.row_next) + row0;
  // the last two leading dimensions, and the first of three (or a dimension of one index)
  const uint32_t d = T.lead_dims, s2 = T.lead_shape[d - 1], s1 = T.lead_shape[d - 2], s0 = d == 3u ? T.lead_shape[0] : 1u;
  const gptr<const float> x2 = as_global<const float>(T.lead_next[d - 1]), x1 = as_global<const float>(T.lead_next[d - 2]);
  const gptr<const float> x0 = as_global<const float>(d == 3u ? T.lead_next[0] : T.lead_next[d - 2]);
#pragma unroll
  for (int pass = 0; pass < kRowScaleChunk / 1024; ++pass) {
    const uint32_t r = (uint32_t)pass * 1024u + threadIdx.x * 4u;
    if (r >= n) return;
    uint32_t q = row0 + r, i2, i1, i0;
    i2 = q % s2; q /= s2;
    i1 = q % s1; i0 = q / s1;
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = min_nonneg(x2[i2], x1[i1]);
      if (d == 3u) v[k] = min_nonneg(v[k], x0[i0]);
      if (++i2 == s2) {
        i2 = 0u;
        if (++i1 == s1) { i1 = 0u; i0 = i0 + 1u < s0 ? i0 + 1u : i0; }   // past the last row: stay in bounds
      }
    }
    if (r + 4u <= n) {
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{f2bits(v[0]), f2bits(v[1]), f2bits(v[2]), f2bits(v[3])},
                                             tile_rsrc(T.row_next + row0), r * 4u, 0, 0);
    } else {
      for (uint32_t k = 0; r + k < n; ++k) out[r + k] = k == 0u ? v[0] : k == 1u ? v[1] : v[2];
    }
  }
}

// After the update: the new statistics become the current ones and the buffers that
// received them go back to zero for the next step's maxima.  A workgroup's chunk lies in one of
// the tensor's vectors (rows, columns, leading dimensions); all its loads are in flight
// together.
__global__ __launch_bounds__(256) void rank1_commit_kernel(const CommitArgs args) {
  constexpr int kPer = kCommitChunk / 256;
  float gscale;
  if (!grad_ops_begin(args.go, gscale)) return;
  const int t = find_tensor(args, blockIdx.x);
  const auto &T = args.desc[t];
  uint32_t local = blockIdx.x - args.first_chunk[t];
  int k = 0;
  while (k < 4 && local >= (T.size[k] + kCommitChunk - 1) / kCommitChunk) {
    local -= (T.size[k] + kCommitChunk - 1) / kCommitChunk;
    ++k;
  }
  const uint32_t i0 = local * kCommitChunk + threadIdx.x, size = T.size[k];
  const gptr<float> cur = as_global<float>(T.cur[k]), next = as_global<float>(T.next[k]);
  float x[kPer];
#pragma unroll
  for (int h = 0; h < kPer; ++h) x[h] = i0 + h * 256u < size ? next[i0 + h * 256u] : 0.0f;
#pragma unroll
  for (int h = 0; h < kPer; ++h) {
    if (i0 + h * 256u < size) {
      cur[i0 + h * 256u] = x[h];
      next[i0 + h * 256u] = 0.0f;
    }
  }
}

}  // namespace q4
