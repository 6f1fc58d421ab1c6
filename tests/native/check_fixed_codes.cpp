// Host model of the step's fixed-point codes (csrc/q4adamw_device.h): the float operations with
// std::fmaf, the integer ones as they are, the tables from csrc/q4adamw_tables.h.  Built and run by
// tests/test_abi_and_tables.py with g++ -fopenmp; prints one line per check, "ok" last.
//
// For scales of every mantissa class and values at, around and between all decision points it
// checks, with the scale's reciprocal off by whole units in the last place,
//   1. the code wherever the fast path decides, against the exactly divided quotient's;
//   2. the error bounds that the undecided band is sized for: z before its own rounding lies within
//      0.13 (block scale: reciprocal correctly rounded), 0.31 (rank-1: one unit off) and 0.65
//      (first moment, stochastic) units of 2^-16 of the exact position's;
//   3. that few values are undecided;
// and for every upper half and the lower halves at its ends that a NaN gets code 0, whatever the noise.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <initializer_list>

#include "../../quantfour_adamw_cuda_amd/csrc/q4adamw_tables.h"

using namespace q4;

static inline uint64_t mix(uint64_t x) {   // splitmix64
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

static inline float nudge(float x, int d) { return bits2f(f2bits(x) + (uint32_t)d); }   // away from zero for d > 0

// high byte of q converted to half precision toward zero (v_cvt_pkrtz_f16_f32)
static inline uint32_t half_index(float q) {
  const uint32_t b = f2bits(q), sign = b >> 31, mag = b & 0x7fffffffu, e8 = mag >> 23;
  if (e8 >= 113u) return (sign << 7) | ((e8 - 112u) << 2) | ((mag >> 21) & 3u);
  const uint32_t m = (uint32_t)std::floor(std::fabs((double)q) * 16777216.0);
  return (sign << 7) | (m >> 8);
}

// clamped_halves and collect_codes, one element
static inline uint32_t code_of(uint32_t g) {
  uint32_t h = g >> 16;
  h = h < 0x431fu ? h : 0x431fu;
  return 15u - (h & 15u);
}

static inline uint32_t add_noise(uint32_t g, uint32_t n16) {
  const uint32_t s = g + n16;
  return s < g ? 0xffffffffu : s;
}

constexpr uint32_t kNearRn = 1u, kNearSr = 2u;

static int exact_nearest_v(float q) {
  int c = 0;
  for (int k = 0; k < 15; ++k) c += qmid_v(k) < q;
  return c;
}

static int exact_sr(bool second, float q, float noise, int *interval) {
  int k = 0;
  for (int j = 0; j < 16; ++j) k += (second ? qmap_v(j) : bits2f(kQmapMBits[j])) <= q;
  *interval = k;
  float lower, width;
  if (second) {
    lower = k == 0 ? 0.0f : (float)k * 0.0625f;
    width = 0.0625f;
    if (k == 0) return 0;
  } else {
    lower = sr_interval_m((uint32_t)k).lower;
    width = sr_interval_m((uint32_t)k).width;
  }
  const int c = k - 1 + (noise * width < q - lower ? 1 : 0);
  return c < 0 ? 0 : c > 15 ? 15 : c;
}

struct Tally {
  long long decided = 0, undecided = 0, wrong = 0;
  double worst = 0.0;
  void add(bool is_decided, bool right, double e) {
    if (is_decided) { ++decided; wrong += !right; }
    else ++undecided;
    worst = e > worst ? e : worst;
  }
  void join(const Tally &o) {
    decided += o.decided; undecided += o.undecided; wrong += o.wrong;
    worst = o.worst > worst ? o.worst : worst;
  }
};

int main() {
  static SrEntry sr[256];
  for (uint32_t h = 0; h < 256; ++h) sr[h] = sr_entry(h);
  constexpr int kScales = 20000, kSpread = 24;   // scales; values spread over (0, 1] for each
  Tally near_rn, near_sr_v, near_sr_m, far_rn, far_sr_v, far_sr_m;   // around decision points, and spread
  double worst_block = 0.0, worst_rank1 = 0.0;
#pragma omp parallel
  {
    Tally a, b, c, d, e, f;
    double wb = 0.0, wr = 0.0;
#pragma omp for schedule(static)
    for (int i = 0; i < kScales; ++i) {
      const uint64_t h = mix((uint64_t)i);
      uint32_t mant = (uint32_t)h & 0x7fffffu;
      if (i % 8 == 0) mant = (uint32_t)(i / 8) & 0x3ffu;                 // just above a power of two
      if (i % 8 == 1) mant = 0x7fffffu - ((uint32_t)(i / 8) & 0x3ffu);   // just below one
      const float s = bits2f(((40u + (uint32_t)(h >> 32) % 170u) << 23) | mant);   // 2^-87 .. 2^82
      const float r0 = (float)(1.0 / (double)s);
      for (int dr = -2; dr <= 2; ++dr) {
        const float r = nudge(r0, dr), neg_inv16 = r * -16.0f;
        // second moment, nearest: around the 15 thresholds, then spread
        for (int k = 0; k < 15 + kSpread; ++k) {
          const bool near = k < 15;
          const float t = near ? qmid_v(k) * s : (float)((mix(h + (uint64_t)k) >> 40) + 1) * 0x1p-24f * s;
          for (int o = near ? -40 : 0; o <= (near ? 40 : 0); ++o) {
            float x = nudge(t, o);
            if (x > s) x = s;
            const float q = x / s;
            const double z = (double)x * (double)neg_inv16 + 160.5;
            const double err = std::fabs(z - (160.5 - 16.0 * (double)q)) * 65536.0;
            const uint32_t g = f2bits(std::fmaf(x, neg_inv16, bits2f(0x43208000u)));
            (near ? a : d).add((g & 0xffffu) >= kNearRn, (int)code_of(g) == exact_nearest_v(q), 0.0);
            if (dr == 0 && err > wb) wb = err;
            if (dr >= -1 && dr <= 1 && err > wr) wr = err;
          }
        }
        // stochastic: both moments, positions within a few units of the noise, then spread
        for (int k = 0; k < 32 + kSpread; ++k) {
          const bool near = k < 32;
          const uint64_t hk = mix(h ^ ((uint64_t)k << 20) ^ (uint64_t)(dr + 2));
          const uint32_t n = near && k % 16 == 0 ? 0u : near && k % 16 == 1 ? 65535u : (uint32_t)hk & 0xffffu;
          const float noise = (float)(2u * n + 1u) * 0x1p-17f;
          const double off = near ? (double)((int)((hk >> 16) % 33u) - 16) * 0x1p-18 : 0.0;   // +-4 units
          {
            const int at = (int)((hk >> 24) % 16u);                                     // between entries at and at + 1
            double pos = near ? (double)at + (double)noise + off : 16.0 * (double)((hk >> 40) + 1) * 0x1p-24;
            float x = (float)(pos / 16.0 * (double)s);
            if (!(x > 0.0f)) x = s * 0x1p-20f;
            if (x > s) x = s;
            int interval;
            const int want = exact_sr(true, x / s, noise, &interval);
            const uint32_t g = add_noise(f2bits(std::fmaf(x, neg_inv16, bits2f(0x43200001u))), n);
            (near ? b : e).add((g & 0xffffu) >= kNearSr, (int)code_of(g) == want, 0.0);
          }
          if (dr >= -1 && dr <= 1) {
            const uint32_t at = 1u + (uint32_t)((hk >> 24) % 15u);                      // interval 1..15
            const double lower = bits2f(kQmapMBits[at - 1]), width = (double)bits2f(kQmapMBits[at]) - lower;
            double target = near ? lower + ((double)noise + off) * width : 2.0 * (double)((hk >> 40) + 1) * 0x1p-24 - 1.0;
            float x = (float)(target * (double)s);
            if (x > s) x = s;
            if (x < -s) x = -s;
            int interval;
            const float q_exact = x / s, q = x * r;
            const int want = exact_sr(false, q_exact, noise, &interval);
            const uint32_t hi = half_index(q), k_raw = sr[hi].base + (q >= bits2f(sr[hi].thr) ? 1u : 0u);
            const SrAffine af = sr_fixed_m(k_raw);
            const uint32_t g = add_noise(f2bits(std::fmaf(q, af.a, af.c)), n);
            double err = 0.0;
            if (k_raw == (uint32_t)interval && k_raw > 0u && k_raw < 16u) {
              const SrInterval iv = sr_interval_m(k_raw);
              const double w = (double)bits2f(kQmapMBits[k_raw]) - (double)iv.lower;
              const double y = (double)k_raw + ((double)q_exact - (double)iv.lower) / w;
              err = std::fabs((double)q * (double)af.a + (double)af.c - (160.0 + 0x1p-16 - y)) * 65536.0;
            }
            if (dr != 0) err = 0.0;   // the block scale's reciprocal is refined
            (near ? c : f).add((g & 0xffffu) >= kNearSr, (int)code_of(g) == want, err);
          }
        }
      }
    }
#pragma omp critical
    {
      near_rn.join(a); near_sr_v.join(b); near_sr_m.join(c); far_rn.join(d); far_sr_v.join(e); far_sr_m.join(f);
      worst_block = wb > worst_block ? wb : worst_block;
      worst_rank1 = wr > worst_rank1 ? wr : worst_rank1;
    }
  }
  long long bad = 0;
  const struct { const char *name; const Tally *near, *far; } lines[3] = {
      {"second moment, nearest", &near_rn, &far_rn}, {"second moment, stochastic", &near_sr_v, &far_sr_v}, {"first moment, stochastic", &near_sr_m, &far_sr_m}};
  for (const auto &l : lines) {
    std::printf("%s: %lld decided, %lld undecided, %lld wrong around decision points; %lld, %lld, %lld spread\n", l.name, l.near->decided,
                l.near->undecided, l.near->wrong, l.far->decided, l.far->undecided, l.far->wrong);
    bad += l.near->wrong + l.far->wrong;
    bad += l.near->undecided <= 0 || l.near->undecided > 2 * l.near->decided || l.far->undecided * 5000 > l.far->decided;
  }
  const double worst_m = near_sr_m.worst > far_sr_m.worst ? near_sr_m.worst : far_sr_m.worst;
  std::printf("errors before rounding, units of 2^-16: %.4f block scale, %.4f rank-1, %.4f first moment\n", worst_block, worst_rank1, worst_m);
  bad += worst_block > 0.13 || worst_rank1 > 0.31 || worst_m > 0.65;

  // NaN: fma keeps its pattern (quiet), the noise must not carry it out of the word
  long long bad_nan = 0, seen = 0;
  for (uint32_t top = 0; top < 0x10000u; ++top) {
    for (uint32_t low : {0u, 1u, 2u, 0x7fffu, 0x8000u, 0x8001u, 0xe000u, 0xfffeu, 0xffffu}) {
      const uint32_t b = top << 16 | low;
      if (bits2f(b) == bits2f(b)) continue;
      for (uint32_t n : {0u, 1u, 2u, 0x1fffu, 0x2000u, 0x7fffu, 0x8000u, 0xfffeu, 0xffffu}) {
        const uint32_t g = add_noise(b | 0x400000u, n);
        bad_nan += code_of(g) != 0u;   // undecided or not: the exact path gives 0 as well
        ++seen;
      }
    }
  }
  std::printf("NaN: %lld patterns and noises, %lld with another code than 0\n", seen, bad_nan);
  if (bad || bad_nan) return 1;
  std::printf("ok\n");
  return 0;
}
