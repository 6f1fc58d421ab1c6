// Kernels around the fused step: the non-quantized step of small tensors, the global
// gradient norm, stand-alone quantize / dequantize for checkpoint interchange.
#pragma once
#include "q4adamw_device.h"

namespace q4 {

// Non-quantized step for small tensors (cuda_adamw_kernels.cu:100-133): fp32
// moments in place, same derived scalars and operation order as the fused path.
template <int PT, int GT, bool EXT>
__global__ __launch_bounds__(256) void single_tensor_kernel(const SmallArgs args) {
  const uint32_t chunk = args.chunk_base + blockIdx.x;
  float gscale = 1.0f;
  const bool cancelled = EXT && !grad_ops_begin(args.go, gscale);
  const bool zero_g = EXT && args.go.zero != 0u;
  if (cancelled && !zero_g) return;
  const int t = find_tensor(args, chunk);
  const SmallDesc &T = args.desc[t];
  const StepConsts sc = EXT ? step_consts(args.sc, args.go) : args.sc;
  const int64_t base = (int64_t)(chunk - args.first_chunk[t]) * kSmallChunk;
  const int64_t end = base + (chunk + 1u == args.first_chunk[t + 1] ? args.last[t] : kSmallChunk);
  small_elements<PT, GT, EXT>(T.p, T.g, T.m, T.v, base, end, sc, gscale, zero_g, cancelled);
}

// ---------------------------------------------------------------------------
// a step whose number lives on the device
// ---------------------------------------------------------------------------
// One thread: advances the step counter and derives the step's scalars exactly as the
// host does for a step it knows (make_consts; optim/cuda_adamw_kernels.cu:435-440), from
// the bias-correction pair the host tabulated for that step number: every operation
// below is the IEEE operation the host performs, so the scalars agree bit for bit.  A
// set overflow flag leaves counter and scalars alone (the step's launches do nothing then).
__global__ void device_step_kernel(float *counter_, const float *table_, int64_t first_step, int64_t table_steps,
                                   const float *lr_dev, float beta1, float beta2, float lr, float wd, float eps,
                                   const float *skip, StepConsts *out_) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  if (skip && *as_global<const float>(skip) != 0.0f) return;
  const gptr<float> counter = as_global<float>(counter_);
  const float t = *counter + 1.0f;
  *counter = t;
  int64_t k = (int64_t)t - first_step;
  k = k < 0 ? 0 : (k >= table_steps ? table_steps - 1 : k);   // past the table: its last, converged entry
  const float c1 = as_global<const float>(table_)[2 * k], c2s = as_global<const float>(table_)[2 * k + 1];
  const float lrv = lr_dev ? *as_global<const float>(lr_dev) : lr;
  StepConsts sc;
  sc.b1 = beta1;
  sc.b2 = beta2;
  sc.r1 = 1.0f - beta1;
  sc.r2 = 1.0f - beta2;
  const float lrwd = lrv * wd;
  sc.wdu = 1.0f - lrwd;
  sc.ss = lrv / c1;
  sc.c2s = c2s;
  sc.eps = eps;
  const double den_scale = 1.0 / ((double)c2s * (double)sc.ss), den_eps = (double)eps / (double)sc.ss;
  const bool fits = den_scale <= (double)FLT_MAX && den_eps <= (double)FLT_MAX;
  sc.den_scale = fits ? (float)den_scale : 0.0f;
  sc.den_eps = fits ? (float)den_eps : __builtin_inff();
  const gptr<float> o = as_global<float>(out_);   // the order step_consts() reads
  o[0] = sc.b1; o[1] = sc.b2; o[2] = sc.r1; o[3] = sc.r2; o[4] = sc.wdu;
  o[5] = sc.ss; o[6] = sc.c2s; o[7] = sc.eps; o[8] = sc.den_scale; o[9] = sc.den_eps;
  as_global<uint32_t>(out_)[10] = (uint32_t)t;   // the step number, for the rounding noise's salt
  make_exact_consts(&sc);
  o[11] = sc.c2s_rcp;
  as_global<uint32_t>(out_)[12] = sc.exact_short;
}

// ---------------------------------------------------------------------------
// self-check of the exact parameter update's short forms on the running GPU
// ---------------------------------------------------------------------------
// Walks every fp32 pattern of the short forms' domains through them and counts disagreements
// with the correctly rounded results, taken in fp64 and rounded to fp32 (for a square root, a
// reciprocal and a quotient the second rounding is harmless: 53 >= 2 * 24 + 2 bits):
//   out[0]  sqrt_rn(x) != RN(sqrt x)                      x in [2^-96, 2^90]
//   out[1]  estimate + one Newton step != RN(1 / d)       d in [2^-60, 2^60]
//   out[2]  div_rn(m, d) != RN(m / d)                     every such d with three numerators:
//           1, and two of either sign with a mantissa and exponent (2^-60 .. 2^59) hashed from d
//   out[3]  the compiler's general sqrtf != RN(sqrt x)    (what lanes outside the domains take)
//   out[4]  the compiler's general m / d != RN(m / d)
//   out[5]  patterns walked
// out[1] is a property of the hardware's reciprocal estimate: arithmetic alone promises it only
// for divisors whose mantissa is not all ones.
__global__ __launch_bounds__(256) void rounding_selfcheck_kernel(unsigned long long *out_) {
  const gptr<unsigned long long> out = as_global<unsigned long long>(out_);
  unsigned long long bad[5] = {0, 0, 0, 0, 0}, walked = 0;
  const uint32_t first = (blockIdx.x * 256u + threadIdx.x) << 11;   // 2^21 threads x 2^11 patterns = 2^32
  for (uint32_t k = 0; k < 2048u; ++k) {
    const uint32_t u = first + k;
    const float x = bits2f(u);
    if (x >= kExactVLo && x <= kExactVHi) {
      const float want = (float)__builtin_sqrt((double)x);
      bad[0] += f2bits(sqrt_rn(x)) != f2bits(want);
      bad[3] += f2bits(__builtin_sqrtf(x)) != f2bits(want);
      ++walked;
    }
    if (x >= kExactLo && x <= kExactHi) {
      const float y0 = __builtin_amdgcn_rcpf(x);
      const float y = __builtin_fmaf(__builtin_fmaf(-x, y0, 1.0f), y0, y0);
      bad[1] += f2bits(y) != f2bits((float)(1.0 / (double)x));
      const uint32_t h = lowbias32(u);
      const float m1 = bits2f((h & 0x807fffffu) | ((67u + (h >> 23) % 120u) << 23));
      const float ms[3] = {1.0f, m1, -m1 * 0.75f};
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const float want = (float)((double)ms[j] / (double)x);
        bad[2] += f2bits(div_rn(ms[j], x)) != f2bits(want);
        bad[4] += f2bits(ms[j] / x) != f2bits(want);
      }
      ++walked;
    }
  }
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    if (bad[j]) atomicAdd(out_ + j, bad[j]);
  }
  atomicAdd(out_ + 5, walked);
  (void)out;
}

// ---------------------------------------------------------------------------
// global gradient norm (what a caller computes before it clips)
// ---------------------------------------------------------------------------
// Sum over a 256-thread workgroup in a fixed order; the result is valid in thread 0.
__device__ __forceinline__ double workgroup_sum(double x, double *lds4) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  if ((threadIdx.x & 63) == 0) lds4[threadIdx.x >> 6] = x;
  __syncthreads();
  return (lds4[0] + lds4[1]) + (lds4[2] + lds4[3]);
}

// Squares are exact in fp64 and summed there: four accumulators per thread, chunks in
// grid-stride order, so the sum depends on the tensor list only, not on scheduling.
template <int GT>
__global__ __launch_bounds__(256) void grad_sumsq_kernel(const NormArgs args) {
  constexpr int kElemBytes = GT ? 2 : 4;
  constexpr int64_t kChunkElems = kNormChunkBytes / kElemBytes;
  __shared__ double lds4[4];
  const int tid = threadIdx.x;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (uint32_t chunk = blockIdx.x; chunk < args.nchunks; chunk += kNormPartials) {
    const int t = find_tensor(args, chunk);
    const NormDesc &T = args.desc[t];
    const int64_t base = (int64_t)(chunk - args.first_chunk[t]) * kChunkElems;
    const void *cb = static_cast<const char *>(T.g) + base * kElemBytes;
    const int64_t rem = T.numel - base;
    if (rem >= kChunkElems) {
      u32x4 w[8];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        w[k] = __builtin_amdgcn_raw_buffer_load_b128(tile_rsrc(cb), (uint32_t)(k * 256 + tid) * 16u, 0, kNtReadOnly);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t u[4] = {w[k].x, w[k].y, w[k].z, w[k].w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if constexpr (GT != 0) {
            float lo, hi;
            widen_pair<GT>(u[c], lo, hi);
            acc[c] = __builtin_fma((double)lo, (double)lo, acc[c]);
            acc[c] = __builtin_fma((double)hi, (double)hi, acc[c]);
          } else {
            const double x = (double)bits2f(u[c]);
            acc[c] = __builtin_fma(x, x, acc[c]);
          }
        }
      }
    } else {
      for (int64_t i = tid; i < rem; i += 256) {
        const double x = (double)load_scalar<GT>(cb, i);
        acc[0] = __builtin_fma(x, x, acc[0]);
      }
    }
  }
  const double total = workgroup_sum((acc[0] + acc[1]) + (acc[2] + acc[3]), lds4);
  if (tid == 0) {
    const gptr<double> out = as_global<double>(args.partials) + blockIdx.x;
    *out = args.first ? total : *out + total;
  }
}

__global__ __launch_bounds__(256) void grad_norm_finish_kernel(const double *partials_, float scale,
                                                               const float *scale_dev, float max_norm,
                                                               float *out3_) {
  __shared__ double lds4[4];
  const gptr<const double> partials = as_global<const double>(partials_);
  double a = 0.0;
#pragma unroll
  for (int k = 0; k < kNormPartials / 256; ++k) a += partials[threadIdx.x * (kNormPartials / 256) + k];
  const double total = workgroup_sum(a, lds4);
  if (threadIdx.x == 0) {
    float s = scale;
    if (scale_dev) s *= *as_global<const float>(scale_dev);
    const float norm = __builtin_fabsf(s) * (float)__builtin_sqrt(total);
    // torch.nn.utils.clip_grad_norm_: max_norm / (total_norm + 1e-6), clamped to 1
    // (a NaN stays a NaN)
    float coef = 1.0f;
    if (max_norm > 0.0f) {
      coef = max_norm / (norm + 1e-6f);
      coef = coef > 1.0f ? 1.0f : coef;
    }
    const gptr<float> out3 = as_global<float>(out3_);
    out3[0] = norm;
    out3[1] = coef;
    out3[2] = s * coef;
  }
}

// ---------------------------------------------------------------------------
// stand-alone quantize / dequantize of moments (checkpoint interchange)
// ---------------------------------------------------------------------------
// fp32 on one side and 4-bit codes on the other: 4.03 bytes per element one way and 0.5 the
// other, so these are streams, bound by HBM.  A wave takes two (encoding) or four (decoding)
// tiles of 256 consecutive elements, a lane four elements of each: one 16-byte access on the
// fp32 side and one 2-byte access on the codes' per tile, all tiles' loads in flight together.
// Tiles per wave measured on 14336 x 4096 elements, first / second moment, us: encoding one
// 53 / 51, two 41.8 / 40.0, four 42.2 / 42.6, eight 44.0 / 44.4; decoding one 64 / 53, two
// 49 / 46, four 45.8 / 44.0, eight 48.6 / 49.6.
constexpr int kEncodeTiles = 2, kDecodeTiles = 4;
constexpr int64_t kEncodeChunk = 256 * kEncodeTiles * kWaves, kDecodeChunk = 256 * kDecodeTiles * kWaves;   // elements per workgroup

__device__ __forceinline__ int wave_number() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

// Four consecutive elements from e on (e a multiple of 4) of x, and how many of them exist.
__device__ __forceinline__ int load_four(const float *x, int64_t e, int64_t numel, float (&v)[4]) {
  const int64_t rem = numel - e;
  if (rem >= 4) {
    const f32x4 w = __builtin_nontemporal_load((gptr<const f32x4u>)(uintptr_t)(x + e));
    v[0] = w.x; v[1] = w.y; v[2] = w.z; v[3] = w.w;
    return 4;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = j < rem ? as_global<const float>(x)[e + j] : 0.0f;
  return rem > 0 ? (int)rem : 0;
}

// The codes of n of four elements from e on, a nibble each.
__device__ __forceinline__ void store_four_codes(uint8_t *codes, int64_t e, int n, uint32_t word, bool even) {
  const gptr<uint8_t> out = as_global<uint8_t>(codes) + (e >> 1);
  if (n == 4 && even) {
    __builtin_nontemporal_store((uint16_t)word, (gptr<uint16_t>)(uintptr_t)(codes + (e >> 1)));
    return;
  }
  word &= (1u << (4 * n)) - 1u;          // an odd element count: the last byte's high nibble stays 0
  if (n > 0) out[0] = (uint8_t)word;
  if (n > 2) out[1] = (uint8_t)(word >> 8);
}

__device__ __forceinline__ uint32_t load_four_codes(const uint8_t *codes, int64_t e, int64_t numel, bool even) {
  const int64_t rem = numel - e;
  if (rem >= 4 && even) return __builtin_nontemporal_load((gptr<const uint16_t>)(uintptr_t)(codes + (e >> 1)));
  uint32_t word = 0;
  if (rem > 0) word = as_global<const uint8_t>(codes)[e >> 1];
  if (rem > 2) word |= (uint32_t)as_global<const uint8_t>(codes)[(e >> 1) + 1] << 8;
  return word;
}

// v to the four elements of the lane in the tile (uniform) at tile0.  The streamed stores' policy
// (kNt) measures 2 to 4 % faster here than the non-temporal hint alone.
__device__ __forceinline__ void store_four(float *out, int64_t tile0, int64_t numel, const float (&v)[4]) {
  const uint32_t lane4 = (threadIdx.x & 63u) * 4u;
  const int64_t e = tile0 + lane4, rem = numel - e;
  if (rem >= 4) {
    store_b128<kNt>(u32x4{f2bits(v[0]), f2bits(v[1]), f2bits(v[2]), f2bits(v[3])}, out + tile0, lane4 * 4u);
    return;
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    if (j < rem) as_global<float>(out)[e + j] = v[j];
  }
}

// Second moment: the codes of four values under scales whose 16 / scale are inv16; the step's fast path
// (q4adamw_step.h) for values of either sign.  near: raised where a quotient is within the guard
// band of a threshold.
__device__ __forceinline__ uint32_t fast_codes_v(const float (&x)[4], const float (&inv16)[4], float &near) {
  uint32_t word = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float t = __builtin_fmaxf(__builtin_fmaf(x[j], inv16[j], kVGuard - 0.5f), 0.0f);   // a NaN: code 0
    t = __builtin_fminf(t, 15.5f);         // scales may be given, and smaller than the values
    near = __builtin_fminf(near, t == 0.0f ? 1.0f : __builtin_amdgcn_fractf(t));
    word |= (uint32_t)(int)t << (4 * j);
  }
  return word;
}

// Per-128 abs-max and nearest codes (optim/adamw_fourbit_triton.py:618-630,
// cuda_adamw_kernels.cu:167-194).  The quotients are the step kernel's: a refined reciprocal, the
// half-indexed bucket table for the first moment, one multiply-add for the second; blocks
// whose scale is out of range and values within the guard band of a threshold take IEEE
// division and the 15-compare count.  even: codes starts at an even address.
// 14336 x 4096 elements: 123 us (one wave per block, 8 bytes per lane, every quotient divided)
// -> 41 us = 6.5 TB/s.
template <bool SECOND>
__global__ __launch_bounds__(kThreads) void quantize_kernel(const float *__restrict__ x_, int64_t numel,
                                                            uint8_t *__restrict__ codes_,
                                                            float *__restrict__ scale_, int64_t group0, bool even) {
  __shared__ uint2 table[SECOND ? 1 : kHalfTableEntries];
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t wave0 = ((group0 + blockIdx.x) * kWaves + wave_number()) * (256 * kEncodeTiles);
  float x[kEncodeTiles][4];
  int n[kEncodeTiles];
#pragma unroll
  for (int k = 0; k < kEncodeTiles; ++k) n[k] = load_four(x_, wave0 + k * 256 + lane * 4, numel, x[k]);
  if (!SECOND) {
    const MtabEntry e = kHalfTable.e[tid];
    table[tid] = make_uint2(e.lo, e.hi);
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < kEncodeTiles; ++k) {
    const int64_t e = wave0 + k * 256 + lane * 4;
    // fmaxf drops a NaN next to a number; from 0 on a NaN never becomes the scale
    float am = 0.0f, unused = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) am = __builtin_fmaxf(am, __builtin_fabsf(x[k][j]));
    block_max32_pair(am, unused);
    if (n[k] > 0 && (lane & 31) == 0) as_global<float>(scale_)[e / Q4ADAMW_BLOCK] = am;
    const bool safe = am >= kScaleLo && am <= kScaleHi;
    const float r = safe ? refined_rcp(am) : 0.0f;
    bool redo = !safe && am != 0.0f;
    uint32_t word = 0;
    if (SECOND) {
      const float inv = r * 16.0f, inv16[4] = {inv, inv, inv, inv};
      float near = 1.0f;
      word = fast_codes_v(x[k], inv16, near);
      redo |= near < 2.0f * kVGuard;
    } else {
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const float q0 = x[k][j] * r, q1 = x[k][j + 1] * r;
        const uint32_t halves = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(q0, q1));
        const uint2 e0 = table[(halves >> 8) & 255u], e1 = table[halves >> 24];
        const bool hi0 = q0 > bits2f(e0.y), hi1 = q1 > bits2f(e1.y);
        redo |= hi0 != (q0 > bits2f(e0.x));
        redo |= hi1 != (q1 > bits2f(e1.x));
        word = __builtin_amdgcn_alignbit(e0.x + (hi0 ? 1u : 0u), word, 4);
        word = __builtin_amdgcn_alignbit(e1.x + (hi1 ? 1u : 0u), word, 4);
      }
      word >>= 16;
    }
    if (__builtin_expect(redo, 0)) {
      Vals<4> v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v.x[j] = x[k][j];
      word = quantize_exact<SECOND, 4>(v, am);
    }
    if (am == 0.0f) word = 0;     // 0/0: code 0 for the whole block
    store_four_codes(codes_, e, n[k], word, even);
  }
}

// cuda_adamw_kernels.cu:329-343: code -> code-book entry * block scale
// 14336 x 4096 elements: 116 us for a first, 87 us for a second moment (one byte of codes per
// thread) -> 43 us = 6.1 TB/s.
template <bool SECOND>
__global__ __launch_bounds__(kThreads) void dequantize_kernel(const uint8_t *__restrict__ codes_,
                                                              const float *__restrict__ scale_,
                                                              int64_t numel, float *__restrict__ out_, int64_t group0,
                                                              bool even) {
  __shared__ float book[16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t wave0 = ((group0 + blockIdx.x) * kWaves + wave_number()) * (256 * kDecodeTiles);
  uint32_t word[kDecodeTiles];
  float s[kDecodeTiles];
#pragma unroll
  for (int k = 0; k < kDecodeTiles; ++k) {
    const int64_t e = wave0 + k * 256 + lane * 4;
    word[k] = load_four_codes(codes_, e, numel, even);
    s[k] = e < numel ? as_global<const float>(scale_)[e / Q4ADAMW_BLOCK] : 0.0f;
  }
  if (!SECOND) {
    if (tid < 16) book[tid] = bits2f(kQmapMDev[tid]);
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < kDecodeTiles; ++k) {
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t c = (word[k] >> (4 * j)) & 15u;
      v[j] = (SECOND ? qmap_v((int)c) : book[c]) * s[k];
    }
    store_four(out_, wave0 + k * 256, numel, v);
  }
}

// ---------------------------------------------------------------------------
// rank-1 forms for the second moment of a rows x cols matrix
// ---------------------------------------------------------------------------
// Zeros over two vectors (a matrix's row and column maxima before their statistics launch).
__global__ __launch_bounds__(256) void fill_zero_kernel(float *x_, int64_t nx, float *y_, int64_t ny) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nx + ny; i += (int64_t)gridDim.x * 256) {
    if (i < nx) as_global<float>(x_)[i] = 0.0f;
    else as_global<float>(y_)[i - nx] = 0.0f;
  }
}

// Row and column of element e.  div: by cols, where the matrix has fewer than 2^32 elements and two
// columns or more (BIG, everything else: a 64-bit division).
template <bool BIG>
__device__ __forceinline__ void row_and_column(int64_t e, int64_t cols, FastDiv div, int64_t &i, int64_t &j) {
  if (BIG) {
    i = e / cols;
    j = e - i * cols;
  } else {
    const uint32_t q = fast_div((uint32_t)e, div.magic, div.shift);
    i = q;
    j = (uint32_t)e - q * (uint32_t)cols;
  }
}

// The lesser of two scales as patterns, signed: of two without a sign it is the lesser number (a NaN
// gives way), and where one has a sign the result has it too.
__device__ __forceinline__ float min_signed(float a, float b) {
  const int32_t x = (int32_t)f2bits(a), y = (int32_t)f2bits(b);
  return bits2f((uint32_t)(x < y ? x : y));
}

// The scales min(row maximum, column maximum) of four consecutive elements from e on (those
// past the matrix's end get the last row's).  The statistics may be a caller's: where a scale has a
// sign (-0.0, below zero, such a NaN), the caller of this takes number_scale instead.  Floating-point
// minima here, whose operands the compiler makes quiet first, cost 57 us instead of 48 (quantizing
// 14336 x 4096 elements).
template <bool BIG>
__device__ __forceinline__ void four_scales(int64_t e, int64_t rows, int64_t cols, FastDiv div, const float *row_max,
                                            const float *col_max, float (&s)[4]) {
  const gptr<const float> rm = as_global<const float>(row_max), cm = as_global<const float>(col_max);
  int64_t i, j;
  row_and_column<BIG>(e, cols, div, i, j);
  if (j + 4 <= cols) {
    const float r = rm[i];
    const f32x4 c = *(gptr<const f32x4u>)(uintptr_t)(col_max + j);
    s[0] = min_signed(r, c.x); s[1] = min_signed(r, c.y); s[2] = min_signed(r, c.z); s[3] = min_signed(r, c.w);
    return;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    s[k] = min_signed(rm[i], cm[j]);
    if (++j == cols) {
      j = 0;
      i = i + 1 < rows ? i + 1 : i;
    }
  }
}

// One element's scale, the lesser of any two numbers.
template <bool BIG>
__device__ __forceinline__ float number_scale(int64_t e, int64_t rows, int64_t cols, FastDiv div, const float *row_max,
                                              const float *col_max) {
  int64_t i, j;
  row_and_column<BIG>(e < rows * cols ? e : rows * cols - 1, cols, div, i, j);
  return __builtin_fminf(as_global<const float>(row_max)[i], as_global<const float>(col_max)[j]);
}

// x / min(row maximum, column maximum), nearest code (optim/adamw_fourbit_triton.py:834-863).
// As quantize_kernel, the scales from the (cached) statistics; an element whose scale is out of
// the reciprocal's range sends its lane to the exact path unless it is a zero (code 0 both ways).
template <bool BIG>
__global__ __launch_bounds__(kThreads) void quantize_rank1_kernel(const float *x_, int64_t rows, int64_t cols, FastDiv div,
                                                                  const float *row_max, const float *col_max,
                                                                  uint8_t *codes_, int64_t group0, bool even) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t numel = rows * cols;
  const int64_t wave0 = ((group0 + blockIdx.x) * kWaves + wave_number()) * (256 * kEncodeTiles);
  float x[kEncodeTiles][4];
  int n[kEncodeTiles];
#pragma unroll
  for (int k = 0; k < kEncodeTiles; ++k) n[k] = load_four(x_, wave0 + k * 256 + lane * 4, numel, x[k]);
#pragma unroll
  for (int k = 0; k < kEncodeTiles; ++k) {
    const int64_t e = wave0 + k * 256 + lane * 4;
    if (e >= numel) return;
    float s[4], inv16[4], near = 1.0f;
    four_scales<BIG>(e, rows, cols, div, row_max, col_max, s);
    bool redo = false;   // a scale with a sign is out of range too
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      redo |= !(s[j] >= kScaleLo && s[j] <= kScaleHi) && x[k][j] != 0.0f;
      inv16[j] = refined_rcp(max_nonneg(s[j], kScaleLo)) * 16.0f;
    }
    uint32_t word = fast_codes_v(x[k], inv16, near);
    redo |= near < 2.0f * kVGuard;
    if (__builtin_expect(redo, 0)) {
      Vals<4> v, sc;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v.x[j] = x[k][j];
        sc.x[j] = number_scale<BIG>(e + j, rows, cols, div, row_max, col_max);
      }
      word = quantize_exact_scales<4>(v, sc);
    }
    store_four_codes(codes_, e, n[k], word, even);
  }
}

// optim/adamw_fourbit_triton.py:520-527: code-book entry times min(row, column maximum)
template <bool BIG>
__global__ __launch_bounds__(kThreads) void dequantize_rank1_kernel(const uint8_t *codes_, const float *row_max,
                                                                    const float *col_max, int64_t rows, int64_t cols,
                                                                    FastDiv div, float *out_, int64_t group0, bool even) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t numel = rows * cols;
  const int64_t wave0 = ((group0 + blockIdx.x) * kWaves + wave_number()) * (256 * kDecodeTiles);
  uint32_t word[kDecodeTiles];
#pragma unroll
  for (int k = 0; k < kDecodeTiles; ++k) word[k] = load_four_codes(codes_, wave0 + k * 256 + lane * 4, numel, even);
#pragma unroll
  for (int k = 0; k < kDecodeTiles; ++k) {
    const int64_t e = wave0 + k * 256 + lane * 4;
    if (e >= numel) return;
    float s[4], v[4];
    four_scales<BIG>(e, rows, cols, div, row_max, col_max, s);
    if (__builtin_expect((int32_t)(f2bits(s[0]) | f2bits(s[1]) | f2bits(s[2]) | f2bits(s[3])) < 0, 0)) {
#pragma unroll
      for (int j = 0; j < 4; ++j) s[j] = number_scale<BIG>(e + j, rows, cols, div, row_max, col_max);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = qmap_v((int)((word[k] >> (4 * j)) & 15u)) * s[j];
    store_four(out_, wave0 + k * 256, numel, v);
  }
}

}  // namespace q4
