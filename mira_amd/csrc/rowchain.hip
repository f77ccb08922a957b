// A run of row-local ops as one launch: quantize_activation (mira/ops.py:602-603),
// layernorm (mira/ops.py:356-360), qmatmul with its epilogue (mira/ops.py:616-620, 192-199)
// and decode attention (mira/ops.py:217-219, 310-313 over a cache).  Row r of each of these
// results depends on row r of its inputs only (sequence r, for the attention), so a workgroup
// that owns a few rows can run the whole run of ops on them, one after another, with a
// workgroup barrier where separate launches had a kernel boundary.
//
// What bounds it: at decode shapes a launch of a few rows takes 4-11 us, nearly all of it
// launch, drain and first-touch latency (a 512-row x 64 x 64 projection took 9.9 us).  Here an
// op is a barrier and its own instructions: 16 waves (W) share 4 SIMDs, so an instruction that all
// of them run costs 16 clocks, and a stage's time is its instruction count as much as its
// loads.  The price is that each workgroup reads every weight byte of the run through its own
// CU, so the caller keeps runs to weights that are small next to a launch
// (RocmExecutable._plan_row_chains).
//
//  * Stages read their rows from LDS, where the stage that made them left them; rows that come
//    from outside the run are brought in first.  Only values that something else reads are
//    stored to memory: loads and stores leave one counter in order, so a wave's next load would
//    wait for its last store's way there.
//  * Stage descriptors are uniform and read by scalar loads; the last wave touches the next
//    stage's while a stage runs, so that they hit the scalar cache.
//  * The constants of a stage (a q-op's first weights, its scale and bias, a layernorm's gain)
//    are loaded before the barrier in front of it.
//
// Measured, against the launches: the 16 of a two-layer D = 64 decode step over 272 keys for 512
// sequences 140.4 -> 56.8 us; one sequence's greedy decode of it 69.0 -> 44.0 us a token, 31 of
// them here (1.2-2 us a stage, 5.5 us an attention); one attention half (layernorm,
// projections, attention) of 512 sequences, 71 MB of cache, 23.7 -> 19.4; a quantize and a
// 256 x 64 x 10 dense layer 10.8 -> 5.7.
#include "mr_common.hpp"
#include "np_sum.hpp"

#include <algorithm>
#include <cstring>
#include <new>
#include <vector>

namespace mr {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
#define MR_GLOBAL __attribute__((address_space(1)))
#define MR_LDS __attribute__((address_space(3)))

// An epilogue step's operand: one value per column in memory, or rows in LDS.
struct RowStep {
  int32_t fn, swapped, mode, at, ld, reserved;
  const float* ptr;
};

// *_at: byte offsets in LDS (-1: not there); strides in elements, the same in LDS and in memory.
struct RowStage {
  int32_t kind;
  int32_t flags;
  int32_t d;             // load: words per row; quantize / layernorm: elements per row; qmatmul: N
  int32_t k_tiles;       // qmatmul: k_pad / 64
  int32_t n_pad, n_steps;
  int32_t x_at, ldx;     // quantize / layernorm / attention (query): f32 rows
  int32_t a_at, lda;     // qmatmul: int8 rows
  int32_t y_at, ldy;     // f32 result
  int32_t q_at, ldq;     // int8 result
  int32_t H, hd, T, c_ld;
  int32_t kn_at, ldkn, vn_at, ldvn;
  int32_t even;          // layernorm: values per lane when the pairwise sum's blocks are alike, or 0
  float eps, xs, scale;
  float* y;              // results in memory, where something outside the run reads them
  int8_t* q;
  double rxs, rd;        // fl64(1 / xs), fl64(1 / d)
  const float* x;        // load / quantize: rows in memory
  int64_t ld_x;          // their stride in bytes
  const float* gamma;
  const float* beta;
  const int8_t* b;
  const double* col_scale;
  const float* kc;
  const float* vc;
  int64_t c_bs;
  const float* mask;
  int32_t pad[10];
  RowStep steps[MR_MAX_EPI];
};
static_assert(sizeof(RowStage) % 64 == 0, "whole lines of the scalar cache");
// read through the constant address space: uniform scalar loads
typedef const __attribute__((address_space(4))) RowStage* RowStageP;

enum { ROW_LOAD = 0, ROW_F16 = 1, ROW_NO_BARRIER = 2 };   // a kind of the library's own; flags

constexpr int ROW_BATCH = 5;     // attention: key rows a lane has in flight (5 x 16 bytes of K and of V)
constexpr int ROW_AHEAD = 2;     // qmatmul: epilogue steps whose column operands are loaded ahead

// The workgroup: its LDS, rows r0 .. r0 + nr - 1, and this thread's place.
struct RowGroup {
  MR_LDS char* lds;
  int64_t r0;
  int nr, rpw, wave, lane;
  template <class T>
  __device__ __forceinline__ MR_LDS T* at(int offset) const { return reinterpret_cast<MR_LDS T*>(lds + offset); }
};

// Where a stage's result elements go.
struct RowOut {
  MR_GLOBAL float* y;
  MR_GLOBAL int8_t* q;
  MR_LDS float* ly;
  MR_LDS int8_t* lq;
  int ldy, ldq;
  double rxs;
  bool f32_lds, i8, i8_lds, f16;
  __device__ __forceinline__ RowOut(const RowStage& st, const RowGroup& g)
      : y(st.y ? reinterpret_cast<MR_GLOBAL float*>(reinterpret_cast<uint64_t>(st.y + g.r0 * st.ldy)) : nullptr),
        q(st.q ? reinterpret_cast<MR_GLOBAL int8_t*>(reinterpret_cast<uint64_t>(st.q + g.r0 * st.ldq)) : nullptr),
        ly(g.at<float>(st.y_at)), lq(g.at<int8_t>(st.q_at)), ldy(st.ldy), ldq(st.ldq), rxs(st.rxs),
        f32_lds(st.y_at >= 0), i8(st.q || st.q_at >= 0), i8_lds(st.q_at >= 0), f16(st.flags & ROW_F16) {}
  __device__ __forceinline__ void put8(int r, int c, int8_t v) const {
    const uint32_t i = static_cast<uint32_t>(r * ldq + c);
    if (i8_lds) lq[i] = v;
    if (q) q[i] = v;
  }
  __device__ __forceinline__ void put(int r, int c, float v) const {
    if (f16) v = round_f16(v);
    const uint32_t i = static_cast<uint32_t>(r * ldy + c);
    if (f32_lds) ly[i] = v;
    if (y) y[i] = v;
    if (i8) put8(r, c, quantize_rcp(v, rxs));
  }
};

// What a wave loads for the next stage before the barrier in front of it.
//   qmatmul: its first column block's weights (4 steps of K), scale and per-column operands
//   layernorm: gain (w[0]) and bias (w[1]) of elements lane, lane + 64, lane + 128, lane + 192
struct Ahead {
  v4i w[4];
  double scale;
  float col[ROW_AHEAD];
};

template <class T>
__device__ __forceinline__ const MR_GLOBAL T* in_memory(const T* p) {
  return reinterpret_cast<const MR_GLOBAL T*>(reinterpret_cast<uint64_t>(p));
}

__device__ __forceinline__ bool per_column(const RowStep& s) {
  return s.fn != MR_EPI_RELU && s.fn < MR_EPI_GELU && (s.mode == MR_BC_SCALAR || s.mode == MR_BC_COL);
}
__device__ __forceinline__ float column_operand(const RowStep& s, int col) {
  return in_memory(s.ptr)[s.mode == MR_BC_COL ? col : 0];
}

// weights of row n (a column of the result), bytes kg * 16 .. +15 of step k
__device__ __forceinline__ v4i row_weights(const RowStage& st, int n, int kg, int k) {
  const uint32_t off = static_cast<uint32_t>(k) * (static_cast<uint32_t>(st.n_pad) * 64u) +
                       static_cast<uint32_t>(n * 64 + kg * 16);     // packed weights are under 2 GiB
  return *reinterpret_cast<const MR_GLOBAL v4i*>(in_memory(st.b) + off);
}

template <int W>
__device__ __forceinline__ void look_ahead(const RowStage& st, const RowGroup& g, Ahead& a) {
  if (st.kind == MR_ROW_QMATMUL) {
    if (g.wave * 16 >= st.d) return;
    const int n = g.wave * 16 + (g.lane & 15), col = min(n, st.d - 1);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k < st.k_tiles) a.w[k] = row_weights(st, n, g.lane >> 4, k);
    a.scale = in_memory(st.col_scale)[col];
#pragma unroll
    for (int s = 0; s < ROW_AHEAD; ++s)
      if (s < st.n_steps && per_column(st.steps[s])) a.col[s] = column_operand(st.steps[s], col);
  } else if (st.kind == MR_ROW_LAYERNORM) {
    if (g.wave >= g.nr) return;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (64 * k < st.d) {
        const int i = min(g.lane + 64 * k, st.d - 1);
        a.w[0][k] = __float_as_int(in_memory(st.gamma)[i]);
        a.w[1][k] = __float_as_int(in_memory(st.beta)[i]);
      }
  }
}

// the workgroup's rows of a value made outside the run, d words each
template <int W>
__device__ __forceinline__ void row_load(const RowStage& st, const RowGroup& g) {
  for (int r = 0; r < g.nr; ++r) {
    const MR_GLOBAL int* src = reinterpret_cast<const MR_GLOBAL int*>(reinterpret_cast<uint64_t>(st.x) + (g.r0 + r) * st.ld_x);
    MR_LDS int* dst = g.at<int>(st.y_at + r * st.ldy);
    for (int c = g.wave * 64 + g.lane; c < st.d; c += W * 64) dst[c] = src[c];
  }
}

// clip(rint(x / xs)) of the workgroup's rows, the bytes up to the row stride zeroed
template <int W>
__device__ __forceinline__ void row_quantize(const RowStage& st, const RowGroup& g) {
  const RowOut out(st, g);
  for (int r = 0; r < g.nr; ++r) {
    const MR_GLOBAL float* src =
        reinterpret_cast<const MR_GLOBAL float*>(reinterpret_cast<uint64_t>(st.x) + (g.r0 + r) * st.ld_x);
    for (int c = g.wave * 64 + g.lane; c < st.ldq; c += W * 64) {
      int8_t v = 0;
      if (c < st.d) v = quantize_one(st.x_at >= 0 ? g.at<float>(st.x_at)[r * st.ldx + c] : src[c], st.xs);
      out.put8(r, c, v);
    }
  }
}

// one wave per row (at most as many rows as waves), as layernorm_kernel
__device__ __forceinline__ void row_layernorm(const RowStage& st, const RowGroup& g, const Ahead& ahead) {
  const int r = g.wave, d = st.d;
  if (r >= g.nr) return;
  const double rd = st.rd;
  const float eps = st.eps;
  auto mean = [=](float s) { return mean_of_sum_rcp(s, d, rd); };
  const MR_LDS float* x = g.at<float>(st.x_at) + r * st.ldx;
  const RowOut out(st, g);
  float mu, sd;
  switch (st.even) {            // values per lane when the pairwise sum's blocks are alike
    case 2: layernorm_even_stats<2>(x, d, g.lane, eps, mean, mu, sd); break;
    case 4: layernorm_even_stats<4>(x, d, g.lane, eps, mean, mu, sd); break;
    case 6: layernorm_even_stats<6>(x, d, g.lane, eps, mean, mu, sd); break;
    case 8: layernorm_even_stats<8>(x, d, g.lane, eps, mean, mu, sd); break;
    case 12: layernorm_even_stats<12>(x, d, g.lane, eps, mean, mu, sd); break;
    case 16: layernorm_even_stats<16>(x, d, g.lane, eps, mean, mu, sd); break;
    default: layernorm_wave_stats([=](int i) { return x[i]; }, d, g.lane, eps, mean, mu, sd);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (64 * k < d) {
      const int i = g.lane + 64 * k;
      if (i < d)
        out.put(r, i, layernorm_value(x[i], mu, sd, __int_as_float(ahead.w[0][k]), __int_as_float(ahead.w[1][k])));
    }
  for (int i = g.lane + 256; i < d; i += 64)
    out.put(r, i, layernorm_value(x[i], mu, sd, in_memory(st.gamma)[i], in_memory(st.beta)[i]));
}

// 16 result columns per wave and turn on v_mfma_i32_16x16x64_i8: lane (l16, kg) holds bytes
// 16 kg .. +15 of each 64-byte step, of input row l16 (any row past the workgroup's) and of
// weight row n0 + l16 (1 KB contiguous per wave and step); its results are column l16, rows
// 4 kg .. +3.  Bytes past the end of an input row meet zero weights.
template <int W>
__device__ __forceinline__ void row_qmatmul(const RowStage& st, const RowGroup& g, Ahead& ahead) {
  const int N = st.d, KT = st.k_tiles;
  if (g.wave * 16 >= N) return;
  const RowOut out(st, g);
  const int l16 = g.lane & 15, kg = g.lane >> 4;
  const MR_LDS int8_t* a = g.at<int8_t>(st.a_at) + min(l16, g.nr - 1) * st.lda + kg * 16;
  for (int n0 = g.wave * 16; n0 < N; n0 += W * 16) {
    const int col = min(n0 + l16, N - 1);
    if (n0 != g.wave * 16) {                  // past what look_ahead loaded
      ahead.scale = in_memory(st.col_scale)[col];
#pragma unroll
      for (int s = 0; s < ROW_AHEAD; ++s)
        if (s < st.n_steps && per_column(st.steps[s])) ahead.col[s] = column_operand(st.steps[s], col);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < KT) ahead.w[k] = row_weights(st, n0 + l16, kg, k);
    }
    v4i acc = {0, 0, 0, 0};
    for (int kt = 0; kt < KT; kt += 4) {
      v4i av[4], wv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        wv[u] = ahead.w[u];
        if (kt + u < KT) av[u] = *reinterpret_cast<const MR_LDS v4i*>(a + (kt + u) * 64);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (kt + 4 + u < KT) ahead.w[u] = row_weights(st, n0 + l16, kg, kt + 4 + u);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (kt + u < KT) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[u], wv[u], acc, 0, 0, 0);
    }
#pragma unroll 1
    for (int r = 0; r < min(4, g.nr); ++r) {
      const int row = 4 * kg + r, at_row = min(row, g.nr - 1);
      float y = dequant(acc[0], ahead.scale);
      acc = v4i{acc[1], acc[2], acc[3], acc[0]};
#pragma unroll 1
      for (int s = 0; s < st.n_steps; ++s) {
        const RowStep& e = st.steps[s];
        if (e.fn == MR_EPI_RELU) {
          y = np_maximum(y, 0.0f);
        } else if (e.fn >= MR_EPI_GELU) {
          y = epi_unary_approx(e.fn, y);
        } else {
          float o;
          if (e.mode == MR_BC_ROW || e.mode == MR_BC_FULL) o = g.at<float>(e.at)[at_row * e.ld + (e.mode == MR_BC_FULL ? col : 0)];
          else if (s < ROW_AHEAD) o = s ? ahead.col[1] : ahead.col[0];
          else o = column_operand(e, col);
          y = e.swapped ? epi_binary(e.fn, o, y) : epi_binary(e.fn, y, o);
        }
      }
      if (row < g.nr && n0 + l16 < N) out.put(row, n0 + l16, y);
    }
  }
}

// Decode attention of the workgroup's sequences, W / rpw waves each, bit for bit
// attention_decode_kernel's arithmetic: a score is one chain of multiply-adds over the head's
// columns, value rows l, l + 64, ... are one chain per l, and the 64 chains meet in a butterfly
// from 32 down (an int8 step behind it may flip with any other order, and with it a greedy
// decode's tokens).  A key or value row is D consecutive floats, read by D / 4 neighbouring
// lanes of LP (the next power of two); lane (slot, c) of 64 / LP slots takes chain
// l = slot * LP + m, m running over the sequence's waves and then over up to 4 passes.  So a
// wave's loads are whole rows, the butterfly's first steps stay in the wave (slots), the next
// in registers (passes), and the rest meet in LDS (waves).  Scores pass along the HD / 4 lanes
// of a head, each adding its 4 columns.
//   work: [rpw][H][T + 1] scores, then [W][64] float4 partial sums
template <int W, int HD>
__device__ __forceinline__ void row_attention(const RowStage& st, const RowGroup& g, MR_LDS float* work) {
  const RowOut out(st, g);
  constexpr int HL = HD / 4;                       // lanes that share a head's part of a row
  const int H = st.H, T = st.T, D = H * HD, L = D / 4, nj = T + 1, lane = g.lane;
  const int lp_log2 = L <= 1 ? 0 : 32 - __builtin_clz(L - 1), LP = 1 << lp_log2;
  const int slot = lane >> lp_log2, c = lane & (LP - 1), h = c / HL;
  const int wps = W / g.rpw;               // waves per sequence
  const int s = g.wave / wps, ws = g.wave - s * wps;
  const int passes = LP > wps ? LP / wps : 1;
  const bool on = c < L && s < g.nr && ws < LP;
  const int sr = s < g.nr ? s : 0;                 // its row (a partial last workgroup: any valid one)
  const uint32_t c_ld = st.c_ld;                   // a sequence's cache is under 2 GiB: 32-bit offsets
  const MR_GLOBAL float* kc = in_memory(st.kc) + (g.r0 + sr) * st.c_bs;
  const MR_GLOBAL float* vc = in_memory(st.vc) + (g.r0 + sr) * st.c_bs;
  MR_LDS float* sc = work + (s * H + h) * nj;
  MR_LDS float* part = work + ((g.rpw * H * nj + 3) & ~3);
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  auto cached = [&](const MR_GLOBAL float* cache, int j) __attribute__((always_inline)) {
    return *reinterpret_cast<const MR_GLOBAL v4f*>(cache + (j * c_ld + c * 4u));
  };
  auto own = [&](int at, int ld) __attribute__((always_inline)) {
    return *reinterpret_cast<const MR_LDS v4f*>(g.at<float>(at) + sr * ld + c * 4);
  };
  const v4f q = on ? own(st.x_at, st.ldx) : zero;
  auto chain = [&](const v4f& k, float a) __attribute__((always_inline)) {
    a = fmaf(q.x, k.x, a);
    a = fmaf(q.y, k.y, a);
    a = fmaf(q.z, k.z, a);
    return fmaf(q.w, k.w, a);
  };
  const bool last = on && c % HL == HL - 1;        // the lane a head's score ends in

  v4f vv[ROW_BATCH];                               // the first pass's first value rows, loaded beside its keys
  for (int p = 0; p < passes; ++p) {
    const int l = slot * LP + p * wps + ws;
    for (int base = 0; base < nj; base += 64 * ROW_BATCH) {
      v4f kv[ROW_BATCH];
      float a[ROW_BATCH], mk[ROW_BATCH];
#pragma unroll
      for (int u = 0; u < ROW_BATCH; ++u) {
        const int j = base + l + 64 * u;
        kv[u] = on && j < T ? cached(kc, j) : zero;
        if (on && j == T) kv[u] = own(st.kn_at, st.ldkn);
        mk[u] = last && j < nj ? in_memory(st.mask)[j] : 0.0f;
      }
      if (p == 0 && base == 0) {
#pragma unroll
        for (int u = 0; u < ROW_BATCH; ++u) vv[u] = on && l + 64 * u < T ? cached(vc, l + 64 * u) : zero;
      }
#pragma unroll
      for (int u = 0; u < ROW_BATCH; ++u) a[u] = chain(kv[u], 0.0f);
#pragma unroll
      for (int t = 1; t < HL; ++t)                 // lane t of a head is right from step t on
#pragma unroll
        for (int u = 0; u < ROW_BATCH; ++u) a[u] = chain(kv[u], dpp<DPP_SHR1>(a[u]));
#pragma unroll
      for (int u = 0; u < ROW_BATCH; ++u) {
        const int j = base + l + 64 * u;
        if (last && j < nj) sc[j] = __fadd_rn(__fmul_rn(a[u], st.scale), mk[u]);
      }
    }
  }
  lds_store_barrier();
  for (int job = g.wave; job < g.nr * H; job += W) {
    MR_LDS float* row = work + job * nj;
    float m = -__builtin_inff(), sum = 0.0f, e[ROW_BATCH];
#pragma unroll
    for (int u = 0; u < ROW_BATCH; ++u) {
      e[u] = row[min(lane + 64 * u, T)];           // past the end: the last one again
      m = np_maximum(m, e[u]);
    }
    for (int j = lane + 64 * ROW_BATCH; j < nj; j += 64) m = np_maximum(m, row[j]);
    m = wave_fold(m, np_maximum);
#pragma unroll
    for (int u = 0; u < ROW_BATCH; ++u) {
      e[u] = expf(__fsub_rn(e[u], m));
      sum = lane + 64 * u < nj ? __fadd_rn(sum, e[u]) : sum;
    }
    for (int j = lane + 64 * ROW_BATCH; j < nj; j += 64) {
      const float x = expf(__fsub_rn(row[j], m));
      row[j] = x;
      sum = __fadd_rn(sum, x);
    }
    sum = wave_fold(sum, add_rn);
#pragma unroll
    for (int u = 0; u < ROW_BATCH; ++u)
      if (lane + 64 * u < nj) row[lane + 64 * u] = __fdiv_rn(e[u], sum);
    for (int j = lane + 64 * ROW_BATCH; j < nj; j += 64) row[j] = __fdiv_rn(row[j], sum);
  }
  lds_store_barrier();
  // the chains of each pass, then the butterfly over l: slots (its bits from 32 down to LP) in
  // the wave, passes in registers, waves in LDS
  v4f o = zero, o1 = zero, o2 = zero;
#pragma unroll 1
  for (int p = 0; p < passes; ++p) {
    v4f acc = zero;
    const int l = slot * LP + p * wps + ws;
    for (int base = 0; base < nj; base += 64 * ROW_BATCH) {
      if (p || base) {
#pragma unroll
        for (int u = 0; u < ROW_BATCH; ++u) {
          const int j = base + l + 64 * u;
          vv[u] = on && j < T ? cached(vc, j) : zero;
        }
      }
#pragma unroll
      for (int u = 0; u < ROW_BATCH; ++u) {
        const int j = base + l + 64 * u;
        if (on && j < nj) {
          if (j == T) vv[u] = own(st.vn_at, st.ldvn);
          const float pj = sc[j];
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[i] = fmaf(pj, vv[u][i], acc[i]);
        }
      }
    }
    if (LP <= 32)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fold_xor32(float(acc[i]), add_rn);
    if (LP <= 16)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fold_xor16(float(acc[i]), add_rn);
    if (LP <= 8)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = __fadd_rn(acc[i], dpp<DPP_ROR8>(acc[i]));
    if (LP <= 4)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = __fadd_rn(acc[i], dpp<DPP_ROR4>(acc[i]));
    // passes p and p + passes / 2 are the butterfly's next pairs: (0 + 2) + (1 + 3), or 0 + 1
    if (p == 0) o = acc;
    else if (passes == 2) o = o + acc;
    else if (p == 1) o1 = acc;
    else if (p == 2) o2 = o + acc;
    else o = o2 + (o1 + acc);
  }
  if (slot == 0 && on) *reinterpret_cast<MR_LDS v4f*>(part + (g.wave * L + c) * 4) = o;
  lds_store_barrier();
  const int n = min(wps, LP);
  for (int t = g.wave * 64 + lane; t < g.nr * D; t += W * 64) {
    const int sq = t >= D ? 1 : 0, d = t - sq * D;   // at most 2 sequences
    const MR_LDS float* p = part + sq * wps * D + d;
    float v[W];
#pragma unroll
    for (int i = 0; i < W; ++i) v[i] = p[min(i, n - 1) * D];
#pragma unroll
    for (int k = W / 2; k > 0; k >>= 1)
      if (k < n)
#pragma unroll
        for (int i = 0; i < k; ++i) v[i] = __fadd_rn(v[i], v[i + k]);
    out.put(sq, d, v[0]);
  }
}

// work_at: LDS offset of the attention's own part, behind the rows
template <int W>
__global__ void __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu(4))) row_chain_kernel(uint64_t stages, int32_t n, int64_t rows, int32_t rpw,
                                                                  int32_t work_at) {
  extern __shared__ __attribute__((aligned(16))) char row_lds[];
  RowGroup g;
  g.lds = (MR_LDS char*)row_lds;
  g.lane = threadIdx.x & 63;
  g.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  g.r0 = int64_t(blockIdx.x) * rpw;
  g.nr = static_cast<int>(min(int64_t(rpw), rows - g.r0));
  g.rpw = rpw;
  const RowStageP first = reinterpret_cast<RowStageP>(stages);
  Ahead ahead;
  for (int i = 0; i < n; ++i) {
    const RowStage& st = *(const RowStage*)(first + i);
    look_ahead<W>(st, g, ahead);
    if (!(st.flags & ROW_NO_BARRIER)) lds_store_barrier();
    if (g.wave == W - 1 && i + 1 < n) {
      const __attribute__((address_space(4))) int* next =
          reinterpret_cast<const __attribute__((address_space(4))) int*>(stages + (i + 1) * sizeof(RowStage));
      int any = 0;
#pragma unroll
      for (int k = 0; k < 5; ++k) any |= next[k * 16];      // its fields and first steps, a word per line
      asm volatile("" ::"s"(any));                          // read: the loads stay
    }
    // what a stage derives from the lane is worked out in that stage: kept over the loop for all
    // the kinds, it takes the registers past 128 and spills
    asm volatile("" : "+v"(g.lane));
    switch (st.kind) {
      case ROW_LOAD: row_load<W>(st, g); break;
      case MR_ROW_QUANTIZE: row_quantize<W>(st, g); break;
      case MR_ROW_LAYERNORM: row_layernorm(st, g, ahead); break;
      case MR_ROW_QMATMUL: row_qmatmul<W>(st, g, ahead); break;
      default:
        if (st.hd == 16) row_attention<W, 16>(st, g, reinterpret_cast<MR_LDS float*>(g.lds + work_at));
        else if (st.hd == 32) row_attention<W, 32>(st, g, reinterpret_cast<MR_LDS float*>(g.lds + work_at));
        else row_attention<W, 64>(st, g, reinterpret_cast<MR_LDS float*>(g.lds + work_at));
    }
  }
}

constexpr int ROW_MAX_ROWS = 16;          // rows per workgroup: the MFMA's row block
constexpr int ROW_MAX_LDS = 64 * 1024;
constexpr int ROW_LDS_PAD = 64;           // a q-op's last step may read this far past its row
constexpr int ROW_MAX_LN = WAVE_SUM_MAX;

static bool al(const void* p, int bytes) { return reinterpret_cast<uintptr_t>(p) % bytes == 0; }

// Rows in LDS: a result of the run, or (made == -1) rows from outside it.
struct RowValue {
  const char* base;
  int64_t ld;           // stride in memory, bytes
  int64_t width;        // bytes per row in LDS
  int64_t need;         // rows from outside: the bytes read of each
  int made, last;       // the stages that write it and that read it last (-1: none)
  bool only_here;       // nothing outside the run reads it
  int64_t at;           // its place, or -1
};

static int64_t chain_bytes(int32_t n) { return n > 0 && n < (1 << 20) ? int64_t(2 * n + 8) * sizeof(RowStage) : -1; }

static int chain_prepare(const mr_row_stage* stages, int32_t n, int64_t rows, void* descriptors, int64_t bytes,
                         int32_t* plan) {
  MR_REQUIRE(stages && descriptors && plan && n > 0 && n < (1 << 20), "mr_row_chain_prepare: NULL argument or no stage");
  MR_REQUIRE(rows >= 0 && rows < (int64_t(1) << 31), "mr_row_chain_prepare: bad row count %lld", (long long)rows);
  MR_REQUIRE(bytes >= chain_bytes(n), "mr_row_chain_prepare: descriptors need %lld bytes",
             (long long)chain_bytes(n));
  std::vector<RowStage> out(n);
  std::memset(out.data(), 0, n * sizeof(RowStage));
  int64_t score_floats = 0, wide = 0;     // per row, the largest attention's scores; its columns
  std::vector<RowValue> values;
  struct Input {
    int stage;
    const char* p;
    int64_t ld, width;      // bytes
    int32_t *at, *stride;   // the stage's words
    int size;               // of an element
  };
  std::vector<Input> inputs;
  bool fits = true;
  auto fit = [&](int64_t v, int64_t most) { fits = fits && v < most; return static_cast<int32_t>(v); };
  for (int i = 0; i < n; ++i) {
    const mr_row_stage& s = stages[i];
    RowStage& d = out[i];
    auto input = [&](int32_t* at, int32_t* stride, const void* p, int64_t ld, int64_t cols, int size) {
      inputs.push_back({i, static_cast<const char*>(p), ld * size, cols * size, at, stride, size});
    };
    auto output_f32 = [&](float* p, int64_t ld) {
      d.y = p;
      d.ldy = fit(ld, 1 << 27);
      if (p) values.push_back({reinterpret_cast<const char*>(p), ld * 4, ld * 4, 0, i, -1, (s.flags & MR_ROW_ONLY_HERE_F32) != 0, -1});
    };
    auto output_i8 = [&](int8_t* p, int64_t ld) {
      d.q = p;
      d.ldq = fit(ld, 1 << 29);
      if (p) values.push_back({reinterpret_cast<const char*>(p), ld, ld, 0, i, -1, (s.flags & MR_ROW_ONLY_HERE_I8) != 0, -1});
    };
    d.kind = s.kind;
    d.d = s.d;
    d.x_at = d.a_at = d.y_at = d.q_at = d.kn_at = d.vn_at = -1;
    d.flags = s.round_f16 ? ROW_F16 : 0;
    d.xs = s.xs;
    d.rxs = s.xs > 0.0f ? 1.0 / static_cast<double>(s.xs) : 0.0;
    d.rd = s.d > 0 ? 1.0 / s.d : 0.0;
    switch (s.kind) {
      case MR_ROW_QUANTIZE:
        MR_REQUIRE(s.x && s.yq && s.d > 0 && s.ldx >= s.d && s.ldq >= s.d && s.xs > 0.0f,
                   "mr_row_chain_prepare: bad quantize stage %d", i);
        d.x = s.x;
        d.ld_x = s.ldx * 4;
        input(&d.x_at, &d.ldx, s.x, s.ldx, s.d, 4);
        output_i8(s.yq, s.ldq);
        break;
      case MR_ROW_LAYERNORM: {
        MR_REQUIRE(s.x && s.gamma && s.beta && s.d > 0 && s.ldx >= s.d && (s.y || s.yq) && (!s.y || s.ldy >= s.d) &&
                   (!s.yq || (s.ldq >= s.d && s.xs > 0.0f)), "mr_row_chain_prepare: bad layernorm stage %d", i);
        if (s.d > ROW_MAX_LN) {
          set_error("mr_row_chain_prepare: layernorm rows of %d elements (at most %d)", s.d, ROW_MAX_LN);
          return MR_EUNSUPPORTED;
        }
        int size = s.d;                  // halved as the pairwise sum halves it, while that is even
        while (size > 128 && size % 16 == 0) size /= 2;
        d.even = size <= 128 && size % 8 == 0 ? size / 8 : 0;
        d.eps = s.eps;
        d.gamma = s.gamma;
        d.beta = s.beta;
        input(&d.x_at, &d.ldx, s.x, s.ldx, s.d, 4);
        output_f32(s.y, s.ldy);
        output_i8(s.yq, s.ldq);
        break;
      }
      case MR_ROW_QMATMUL: {
        MR_REQUIRE(s.a && s.b && s.epi && s.d > 0 && s.K > 0 && s.K <= MAX_EXACT_K && s.lda >= s.K &&
                   s.lda % 16 == 0 && s.k_pad >= s.K && s.k_pad % 64 == 0 && s.n_pad >= s.d && s.n_pad % 32 == 0 &&
                   al(s.a, 16) && al(s.b, 16), "mr_row_chain_prepare: bad qmatmul stage %d", i);
        EpiDev e;
        const int rc = make_epi(s.epi, s.d, true, &e);
        if (rc != MR_OK) return rc;
        if (e.out_acc) {
          set_error("mr_row_chain_prepare: no int32 accumulators");
          return MR_EUNSUPPORTED;
        }
        fits = fits && s.k_pad * s.n_pad < (int64_t(1) << 31);
        d.k_tiles = static_cast<int32_t>(s.k_pad / 64);
        d.n_pad = static_cast<int32_t>(s.n_pad);
        d.n_steps = e.n_steps;
        d.flags = e.f16 ? ROW_F16 : 0;
        d.b = s.b;
        d.col_scale = e.scale;
        d.rxs = e.out_rxs;
        // whole 16-byte chunks of the row, up to k_pad
        input(&d.a_at, &d.lda, s.a, s.lda, std::min(s.lda, s.k_pad), 1);
        for (int k = 0; k < e.n_steps; ++k) {
          RowStep& o = d.steps[k];
          o.fn = e.steps[k].fn;
          o.swapped = e.steps[k].swapped;
          o.mode = e.steps[k].mode;
          o.ptr = e.steps[k].ptr;
          const bool unary = o.fn == MR_EPI_RELU || o.fn >= MR_EPI_GELU;
          if (!unary && (o.mode == MR_BC_ROW || o.mode == MR_BC_FULL))
            input(&o.at, &o.ld, o.ptr, e.steps[k].ld, o.mode == MR_BC_FULL ? s.d : 1, 4);
        }
        output_f32(e.out_f32, e.ldo);
        output_i8(e.out_i8, e.ldq);
        break;
      }
      case MR_ROW_ATTENTION: {
        const int64_t wd = int64_t(s.heads) * s.head_dim;
        MR_REQUIRE(s.x && s.k_new && s.v_new && s.mask && (s.keys == 0 || (s.k_cache && s.v_cache)) && (s.y || s.yq) &&
                   s.heads > 0 && s.keys >= 0 && (s.head_dim == 16 || s.head_dim == 32 || s.head_dim == 64),
                   "mr_row_chain_prepare: bad attention stage %d", i);
        MR_REQUIRE(s.ldx >= wd && s.ld_kn >= wd && s.ld_vn >= wd && s.c_ld >= wd && s.c_bs >= int64_t(s.keys) * s.c_ld &&
                   s.ldx % 4 == 0 && s.ld_kn % 4 == 0 && s.ld_vn % 4 == 0 && s.c_ld % 4 == 0 && s.c_bs % 4 == 0 &&
                   (!s.y || s.ldy >= wd) && (!s.yq || (s.ldq >= wd && s.xs > 0.0f)),
                   "mr_row_chain_prepare: bad attention strides in stage %d", i);
        MR_REQUIRE(al(s.x, 16) && al(s.k_new, 16) && al(s.v_new, 16) &&
                   (s.keys == 0 || (al(s.k_cache, 16) && al(s.v_cache, 16))),
                   "mr_row_chain_prepare: attention operands of stage %d must be 16-byte aligned", i);
        if (wd > 256 || s.keys + 1 > 1024) {
          set_error("mr_row_chain_prepare: attention over %lld columns and %d keys (at most 256 and 1024)",
                    (long long)wd, s.keys + 1);
          return MR_EUNSUPPORTED;
        }
        score_floats = std::max(score_floats, int64_t(s.heads) * (s.keys + 1));
        wide = std::max(wide, wd);
        d.d = static_cast<int32_t>(wd);
        d.H = s.heads;
        d.hd = s.head_dim;
        d.T = s.keys;
        d.scale = s.scale;
        // the caches and the mask are read in memory: they come from outside the run
        d.kc = s.k_cache;
        d.vc = s.v_cache;
        fits = fits && (int64_t(s.keys) + 1) * s.c_ld < (int64_t(1) << 29);
        d.c_ld = fit(s.c_ld, 1 << 29);
        d.c_bs = s.c_bs;
        d.mask = s.mask;
        input(&d.x_at, &d.ldx, s.x, s.ldx, wd, 4);
        input(&d.kn_at, &d.ldkn, s.k_new, s.ld_kn, wd, 4);
        input(&d.vn_at, &d.ldvn, s.v_new, s.ld_vn, wd, 4);
        output_f32(s.y, s.ldy);
        output_i8(s.yq, s.ldq);
        break;
      }
      default: MR_REQUIRE(false, "mr_row_chain_prepare: unknown kind %d of stage %d", s.kind, i);
    }
  }

  // one workgroup per CU while the rows allow it, with at most 2 sequences of an attention each
  // (its waves split the keys: at most 4 passes) or 16 rows without one
  const int64_t cus = device_cu_count();
  int most = !score_floats ? ROW_MAX_ROWS : wide <= 128 ? 2 : 1;
  int rpw = 1, waves = 16;
  if (score_floats && rows > cus && wide <= 128) {
    // two workgroups of 8 waves and one sequence share a CU, so that one's cache loads run under
    // the other's short stages (512 sequences, D = 64: a two-layer step 59.9 -> 56.8 us, an
    // attention half 20.1 -> 19.4); wider rows would take more than 4 passes
    waves = 8;
    most = 1;
  }
  auto work = [&](int r) { return score_floats ? (((r * score_floats + 3) & ~int64_t(3)) + waves * 64 * 4) * 4 : 0; };
  while (rpw < most && (rows + rpw - 1) / rpw > cus && work(2 * rpw) <= ROW_MAX_LDS) rpw *= 2;

  // which value each input is: rows an earlier stage wrote last, at the same stride (a column
  // slice of them), or rows from outside the run
  std::vector<int> source(inputs.size());
  const size_t made_here = values.size();
  for (size_t k = 0; k < inputs.size(); ++k) {
    const Input& in = inputs[k];
    int found = -1;
    for (size_t v = 0; v < made_here; ++v)
      if (values[v].made < in.stage && in.p < values[v].base + values[v].ld * std::max<int64_t>(rows, 1) &&
          values[v].base < in.p + in.ld * std::max<int64_t>(rows - 1, 0) + in.width)
        found = static_cast<int>(v);
    if (found >= 0) {
      const int64_t off = in.p - values[found].base;
      if (in.ld != values[found].ld || off < 0 || off + in.width > values[found].ld || off % 16 != 0) {
        set_error("mr_row_chain_prepare: stage %d reads stage %d's result in another layout", in.stage, values[found].made);
        return MR_EUNSUPPORTED;
      }
    } else {
      if (stages[in.stage].kind == MR_ROW_QUANTIZE) {       // quantizes straight from memory
        source[k] = -1;
        continue;
      }
      for (size_t v = made_here; v < values.size() && found < 0; ++v)
        if (values[v].base == in.p && values[v].ld == in.ld) found = static_cast<int>(v);
      if (found < 0) {
        values.push_back({in.p, in.ld, 0, 0, -1, -1, true, -1});
        found = static_cast<int>(values.size()) - 1;
      }
      values[found].need = std::max(values[found].need, in.width);
      values[found].width = (values[found].need + 15) & ~int64_t(15);
    }
    values[found].last = std::max(values[found].last, in.stage);
    source[k] = found;
  }
  // first fit, a place free again after its value's last reader
  int64_t kept = 0;
  auto size_of = [&](const RowValue& v) { return (v.width * rpw + 15) & ~int64_t(15); };
  for (size_t v = 0; v < values.size(); ++v) {
    RowValue& x = values[v];
    if (x.last < 0) continue;
    int64_t at = 0;
    for (bool moved = true; moved;) {
      moved = false;
      for (const RowValue& u : values)
        if (u.at >= 0 && u.last >= x.made && x.last >= u.made && at < u.at + size_of(u) && u.at < at + size_of(x)) {
          at = u.at + size_of(u);
          moved = true;
        }
    }
    x.at = at;
    kept = std::max(kept, at + size_of(x));
  }
  kept += ROW_LDS_PAD;
  if (!fits || kept + work(rpw) > ROW_MAX_LDS) {
    set_error(fits ? "mr_row_chain_prepare: the run's rows need %lld bytes of LDS"
                   : "mr_row_chain_prepare: a stride or size does not fit 32 bits", (long long)(kept + work(rpw)));
    return MR_EUNSUPPORTED;
  }
  for (size_t k = 0; k < inputs.size(); ++k) {
    if (source[k] < 0) continue;
    const RowValue& v = values[source[k]];
    *inputs[k].at = static_cast<int32_t>(v.at + (v.made >= 0 ? inputs[k].p - v.base : 0));
    *inputs[k].stride = static_cast<int32_t>(v.width / inputs[k].size);
  }
  for (const RowValue& v : values) {
    if (v.made < 0) continue;
    RowStage& d = out[v.made];
    const bool f32 = reinterpret_cast<const char*>(d.y) == v.base;
    (f32 ? d.y_at : d.q_at) = static_cast<int32_t>(v.at);
  }
  for (const RowValue& v : values)       // every reader has it in LDS
    if (v.made >= 0 && v.only_here && v.at >= 0) {
      RowStage& d = out[v.made];
      if (reinterpret_cast<const char*>(d.y) == v.base) d.y = nullptr;
      else d.q = nullptr;
    }
  std::vector<RowStage> all;
  for (const RowValue& v : values) {
    if (v.made >= 0) continue;
    RowStage d;
    std::memset(&d, 0, sizeof(d));
    d.kind = ROW_LOAD;
    d.flags = ROW_NO_BARRIER;            // the first of a run, or beside another one
    d.d = static_cast<int32_t>(v.need / 4);
    d.y_at = static_cast<int32_t>(v.at);
    d.ldy = static_cast<int32_t>(v.width);
    d.x = reinterpret_cast<const float*>(v.base);
    d.ld_x = v.ld;
    all.push_back(d);
  }
  if (all.empty()) out[0].flags |= ROW_NO_BARRIER;
  all.insert(all.end(), out.begin(), out.end());
  if (int64_t(all.size() * sizeof(RowStage)) > bytes) {
    set_error("mr_row_chain_prepare: %lld values from outside the run", (long long)(all.size() - out.size()));
    return MR_EUNSUPPORTED;
  }
  std::memcpy(descriptors, all.data(), all.size() * sizeof(RowStage));
  plan[0] = rpw;
  plan[1] = static_cast<int32_t>(kept);
  plan[2] = static_cast<int32_t>(kept + work(rpw));
  plan[3] = static_cast<int32_t>(all.size());
  plan[4] = waves;
  return MR_OK;
}

}  // namespace mr

extern "C" {

int64_t mr_row_chain_bytes(int32_t n) { return mr::chain_bytes(n); }

int mr_row_chain_prepare(const mr_row_stage* stages, int32_t n, int64_t rows, void* descriptors, int64_t bytes,
                         int32_t* plan) {
  try {
    return mr::chain_prepare(stages, n, rows, descriptors, bytes, plan);
  } catch (const std::bad_alloc&) {
    mr::set_error("mr_row_chain_prepare: out of host memory");
    return MR_EUNSUPPORTED;
  }
}

int mr_row_chain(const void* descriptors, int64_t rows, const int32_t* plan, void* stream) {
  MR_REQUIRE(descriptors && plan && rows >= 0, "mr_row_chain: bad argument");
  MR_REQUIRE(plan[0] >= 1 && plan[0] <= mr::ROW_MAX_ROWS && plan[1] >= 0 && plan[1] <= plan[2] &&
             plan[2] <= mr::ROW_MAX_LDS && plan[3] > 0 &&
             (plan[4] == 16 || (plan[4] == 8 && plan[0] <= 8)), "mr_row_chain: not a plan of mr_row_chain_prepare");
  if (rows == 0) return MR_OK;
  const unsigned grid = static_cast<unsigned>((rows + plan[0] - 1) / plan[0]);
  auto* kernel = plan[4] == 8 ? mr::row_chain_kernel<8> : mr::row_chain_kernel<16>;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(plan[4] * 64), static_cast<unsigned>(plan[2]),
                     static_cast<hipStream_t>(stream), reinterpret_cast<uint64_t>(descriptors), plan[3], rows, plan[0],
                     plan[1]);
  MR_LAUNCH_CHECK("row_chain");
  return MR_OK;
}

}  // extern "C"
