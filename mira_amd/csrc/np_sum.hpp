// NumPy's float32 pairwise summation, shared by every kernel that reproduces
// an f32 add-reduce (np.sum / np.mean along an axis).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mr {

// NumPy's float32 pairwise summation (numpy/_core/src/umath/loops_utils.h.src,
// @TYPE@_pairwise_sum, PW_BLOCKSIZE 128) of the n values elem(0..n), where
// elem(i) loads (or computes) the i-th summand.  A block of fewer than 8 values
// is summed in order from -0.0; a block of 8..128 values runs 8 interleaved
// accumulators, combines them as ((r0+r1)+(r2+r3))+((r4+r5)+(r6+r7)) and adds
// the n % 8 trailing values in order.
template <class Elem>
__device__ inline float pairwise_block_of(Elem elem, int64_t off, int64_t n) {
  if (n < 8) {
    float res = -0.0f;
    for (int64_t i = 0; i < n; ++i) res = __fadd_rn(res, elem(off + i));
    return res;
  }
  float r[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = elem(off + j);
  int64_t i = 8;
  for (; i < n - (n % 8); i += 8) {
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = __fadd_rn(r[j], elem(off + i + j));
  }
  float res = __fadd_rn(__fadd_rn(__fadd_rn(r[0], r[1]), __fadd_rn(r[2], r[3])),
                        __fadd_rn(__fadd_rn(r[4], r[5]), __fadd_rn(r[6], r[7])));
  for (; i < n; ++i) res = __fadd_rn(res, elem(off + i));
  return res;
}

// Above 128 values NumPy splits at n/2 rounded down to a multiple of 8 and
// adds the two halves' sums.  The recursion runs with an explicit stack; its
// depth is about log2(n / 128) + 1, so 40 levels cover n < 2^46.
template <class Elem>
__device__ inline float pairwise_sum_of(Elem elem, int64_t n) {
  if (n <= 128) return pairwise_block_of(elem, 0, n);
  int64_t off[40], cnt[40];
  float left[40];
  int state[40];
  int sp = 0;
  off[0] = 0;
  cnt[0] = n;
  state[0] = 0;
  float ret = 0.0f;
  while (true) {
    if (cnt[sp] <= 128) {
      ret = pairwise_block_of(elem, off[sp], cnt[sp]);
      --sp;
      // unwind: finished children return into their parents
      while (sp >= 0) {
        if (state[sp] == 0) {
          left[sp] = ret;
          state[sp] = 1;
          int64_t n2 = cnt[sp] / 2;
          n2 -= n2 % 8;
          off[sp + 1] = off[sp] + n2;
          cnt[sp + 1] = cnt[sp] - n2;
          state[sp + 1] = 0;
          ++sp;
          break;
        }
        ret = __fadd_rn(left[sp], ret);
        --sp;
      }
      if (sp < 0) return ret;
      continue;
    }
    int64_t n2 = cnt[sp] / 2;
    n2 -= n2 % 8;
    state[sp] = 0;
    off[sp + 1] = off[sp];
    cnt[sp + 1] = n2;
    state[sp + 1] = 0;
    ++sp;
  }
}

// The pairwise sum of n values spaced `stride` apart in memory.
__device__ inline float pairwise_sum(const float* a, int64_t n, int64_t stride) {
  return pairwise_sum_of([=](int64_t i) { return a[i * stride]; }, n);
}

// Butterfly steps as DPP moves and row swaps, a few clocks each where __shfl_xor is a trip
// through LDS.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E;              // quad_perm [1, 0, 3, 2], [2, 3, 0, 1]
constexpr int DPP_MIRROR8 = 0x141, DPP_ROR4 = 0x124, DPP_ROR8 = 0x128, DPP_SHR1 = 0x111;

template <class F>
__device__ __forceinline__ float fold_xor16(float v, F f) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
template <class F>
__device__ __forceinline__ float fold_xor32(float v, F f) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(a[0]), __uint_as_float(a[1]));
}

// All 64 lanes combined in the order of `for (o = 32; o; o >>= 1) v = f(v, __shfl_xor(v, o))`;
// every lane gets the result.  Past the step of 8, lanes 8 apart agree, so the rotation by 4
// brings the value of lane ^ 4.
template <class F>
__device__ __forceinline__ float wave_fold(float v, F f) {
  v = fold_xor16(fold_xor32(v, f), f);
  v = f(v, dpp<DPP_ROR8>(v));
  v = f(v, dpp<DPP_ROR4>(v));
  v = f(v, dpp<DPP_XOR2>(v));
  return f(v, dpp<DPP_XOR1>(v));
}

__device__ __forceinline__ float add_rn(float a, float b) { return __fadd_rn(a, b); }

// The same sum computed by one 64-lane wave, for n <= WAVE_SUM_MAX: the recursion has at most
// 8 blocks (three halvings: 512 -> at most 264 -> 136 -> 72 values), and the 8 lanes of group
// g run the block that g's bits, the first halving's highest, lead to (bit 0 left, 1 right; a
// range of at most 128 values is a block already and only 0 bits lead on).  Lane j of a group
// holds the block's elements j, j + 8, ... in registers, loaded together: loads inside the sum
// would be a chain of memory latencies.
constexpr int WAVE_SUM_MAX = 512;

struct WaveValues {
  float v[16];      // elements j, j + 8, ... of the block, below the last multiple of 8
  float t;          // element j of the block's last cnt % 8
  int cnt;          // the block's elements; 0 in a group without one
  bool split[3];    // this group's range was halved at level l
};

template <class Elem>
__device__ inline void wave_load(Elem elem, int n, int lane, WaveValues& w) {
  const int j = lane & 7, g = lane >> 3;
  int off = 0, cnt = n;
  bool on = true;
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    const bool right = (g >> (2 - l)) & 1;
    w.split[l] = on && cnt > 128;
    if (w.split[l]) {
      const int n2 = (cnt / 2) & ~7;
      off += right ? n2 : 0;
      cnt = right ? cnt - n2 : n2;
    } else if (right) {
      on = false;
    }
  }
  w.cnt = on ? cnt : 0;
  const int body = w.cnt & ~7;
#pragma unroll
  for (int i = 0; i < 16; ++i) w.v[i] = 8 * i < body ? elem(off + 8 * i + j) : 0.0f;
  w.t = j < w.cnt - body ? elem(off + body + j) : 0.0f;
}

// Lane j runs accumulator r[j] over its elements in order, the combine tree is three butterfly
// steps (additions commute exactly), the tail is added in order, and the blocks meet as the
// recursion adds its halves.  Every lane calls it (n: the row's length) and gets the result.
__device__ inline float wave_pairwise_sum(const WaveValues& w, int n, int lane) {
  const int body = w.cnt & ~7;
  float r = w.v[0];
#pragma unroll
  for (int i = 1; i < 16; ++i) r = 8 * i < body ? __fadd_rn(r, w.v[i]) : r;
  r = __fadd_rn(r, dpp<DPP_XOR1>(r));
  r = __fadd_rn(r, dpp<DPP_XOR2>(r));
  r = __fadd_rn(r, dpp<DPP_MIRROR8>(r));     // the quads agree by now: the other quad's sum
  float res = body ? r : -0.0f;       // fewer than 8 values: in order from -0
  if (n & 7) {                        // else every block is a multiple of 8
#pragma unroll
    for (int i = 0; i < 7; ++i) {
      const float t = __shfl(w.t, (lane & ~7) + i);
      res = i < w.cnt - body ? __fadd_rn(res, t) : res;
    }
  }
  // a group adds its right-hand partner's sum where its range was halved; the groups whose
  // lower bits are 0 hold the sums that count
  if (n > 128) {
#pragma unroll
    for (int l = 2; l >= 0; --l) {
      const float other = __shfl_xor(res, 32 >> l);
      if (w.split[l]) res = __fadd_rn(res, other);
    }
  }
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(res)));
}

// ---------------------------------------------------------------- layer normalisation of one row

// Correctly rounded f32 square root (NumPy's np.sqrt), whatever the compiler lowers sqrtf to
// (clang's __fsqrt_rn is the hardware approximation, within 1 ulp).  Rounding to nearest
// picks s when the true root lies between the midpoints m- and m+ to s's neighbours; a
// midpoint has at most 25 significant bits, so m*m is exact in double and the comparison
// with v is exact (never equal: m*m has more bits than a float).  A faithful first guess
// is off by at most one ulp, so one correction suffices.
__device__ inline float sqrt_rn(float v) {
  float s = sqrtf(v);
  if (!(v > 0.0f) || !(v < __builtin_inff())) return s;     // +-0, negative, NaN, inf: exact cases
  const float dn = __int_as_float(__float_as_int(s) - 1), up = __int_as_float(__float_as_int(s) + 1);  // s > 0
  const double x = static_cast<double>(v);
  const double lo = 0.5 * (static_cast<double>(s) + static_cast<double>(dn));
  const double hi = 0.5 * (static_cast<double>(s) + static_cast<double>(up));
  if (__dmul_rn(lo, lo) > x) return dn;
  if (__dmul_rn(hi, hi) < x) return up;
  return s;
}

__device__ inline float mean_of_sum(float s, int d) {
  return static_cast<float>(__ddiv_rn(static_cast<double>(__fadd_rn(0.0f, s)), static_cast<double>(d)));
}

// The same with rd = fl64(1 / d) in place of the f64 division (about 400 clocks).  s / d of a
// 24-bit s and an integer d <= WAVE_SUM_MAX is never a midpoint m of two normal floats (m has 25
// bits, m * d at least as many) and misses the nearest by at least 2^-35 of itself, so the two
// f64 roundings here, 2^-52 together, give the float the correctly rounded quotient gives.
// Results at or below the smallest normal floats are divided.
__device__ inline float mean_of_sum_rcp(float s, int d, double rd) {
  const float m = static_cast<float>(__dmul_rn(static_cast<double>(__fadd_rn(0.0f, s)), rd));
  return fabsf(m) < 2.4e-38f ? mean_of_sum(s, d) : m;
}

// mira/ops.py:356-360 for one row of d elements (read through elem) by one 64-lane wave:
// mu = mean(x), sd = sqrt(mean((x - mu)^2) + eps).  NumPy's mean is an add-reduce seeded
// with +0 over the pairwise f32 sum, then the division of that f32 sum by the count in
// double precision, rounded back to f32; eps is added in f32; the square root is IEEE.
// Rows of at most WAVE_SUM_MAX elements split the pairwise accumulators over the lanes, longer
// ones run the pairwise recursion on lane 0.  Every lane ends with mu and sd.
template <class Elem, class Mean>
__device__ inline void layernorm_wave_stats(Elem elem, int d, int lane, float eps, Mean mean, float& mu, float& sd) {
  WaveValues w;
  wave_load(elem, d, lane, w);
  mu = mean(wave_pairwise_sum(w, d, lane));
#pragma unroll
  for (int i = 0; i < 17; ++i) {
    float& v = i < 16 ? w.v[i] : w.t;
    const float t = __fsub_rn(v, mu);
    v = __fmul_rn(t, t);
  }
  sd = sqrt_rn(__fadd_rn(mean(wave_pairwise_sum(w, d, lane)), eps));
}

// The same for a row x whose pairwise sum has 1, 2 or 4 blocks of 8 N values each: the 8 lanes
// of group g hold block g modulo their number, and the blocks meet in one or two butterfly
// steps.  Fewer instructions than the general split: they are what a lone wave waits for.
template <int N, class Ptr, class Mean>
__device__ __forceinline__ void layernorm_even_stats(Ptr x, int d, int lane, float eps, Mean mean, float& mu, float& sd) {
  const int blocks = d / (8 * N);
  const Ptr p = x + ((lane >> 3) & (blocks - 1)) * (8 * N) + (lane & 7);
  float v[N];
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = p[8 * i];
  auto sum = [&]() __attribute__((always_inline)) {
    float r = v[0];
#pragma unroll
    for (int i = 1; i < N; ++i) r = __fadd_rn(r, v[i]);
    r = __fadd_rn(r, dpp<DPP_XOR1>(r));
    r = __fadd_rn(r, dpp<DPP_XOR2>(r));
    r = __fadd_rn(r, dpp<DPP_MIRROR8>(r));
    if (blocks > 1) r = __fadd_rn(r, dpp<DPP_ROR8>(r));
    if (blocks > 2) r = fold_xor16(r, add_rn);
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(r)));
  };
  mu = mean(sum());
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float t = __fsub_rn(v[i], mu);
    v[i] = __fmul_rn(t, t);
  }
  sd = sqrt_rn(__fadd_rn(mean(sum()), eps));
}

template <class Elem>
__device__ inline void layernorm_row_stats(Elem elem, int d, int lane, float eps, float& mu, float& sd) {
  if (d <= WAVE_SUM_MAX)
    return layernorm_wave_stats(elem, d, lane, eps, [=](float s) { return mean_of_sum(s, d); }, mu, sd);
  float s = 0.0f;
  if (lane == 0) s = pairwise_sum_of(elem, d);
  mu = mean_of_sum(__shfl(s, 0), d);
  const float m = mu;
  s = 0.0f;
  if (lane == 0)
    s = pairwise_sum_of([=](int64_t i) {
      const float t = __fsub_rn(elem(i), m);
      return __fmul_rn(t, t);
    }, d);
  sd = sqrt_rn(__fadd_rn(mean_of_sum(__shfl(s, 0), d), eps));
}

// (x - mu) / sd * g + b, each operation rounded once (before any f16 rounding of the result)
__device__ inline float layernorm_value(float x, float mu, float sd, float g, float b) {
  return __fadd_rn(__fmul_rn(__fdiv_rn(__fsub_rn(x, mu), sd), g), b);
}

}  // namespace mr
