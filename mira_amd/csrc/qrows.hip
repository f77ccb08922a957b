// int8 x int8 -> int32 matmul / convolution of a small result (mira/ops.py:616-620, 630-634,
// with the fused epilogue): batch-1 convolutions, layers of a few hundred rows.
//
// What bounds it: such a result has fewer 64 x 32 tiles than the GPU has CUs, and a workgroup of
// qgemm_kernel walks all of K alone, stage after stage, each waiting for its loads (a 3x3
// convolution of 512 channels on 7 x 7 pixels: 16 workgroups, 36 stages, 17.5 us; its 2.4 MB of
// weights take 0.5 us to read).  Here a workgroup owns a 16- or 32-row by 16- or 32-column tile
// and its 8 waves split K: wave w takes the 64-byte steps w, w + 8, ..., four in flight and the
// next four behind them, straight from memory into the MFMA operand registers (no two waves
// read the same bytes, so LDS has nothing to share); the int32 partial tiles meet in LDS, and
// integer sums are exact in any order.
//
// Measured, us per launch, qgemm_kernel -> this one: ResNet-18 at batch 1, 3x3 convolutions of
// layers 1 / 2 / 3 / 4 8.5 / 12.2 / 12.4 / 17.5 -> 6.5 / 5.4 / 5.2 / 6.5 (the whole image on the
// device 221 -> 121); MobileNetV2's projections from 576 / 960 channels at 14 x 14 / 7 x 7
// 5.5 / 6.7 -> 4.2 / 4.1; dense, 64 rows: 512 x 512 5.6 -> 4.0, 4096 x 1000 13.2 -> 6.1.
#include "mr_common.hpp"

namespace mr {

typedef int v4i __attribute__((ext_vector_type(4)));

struct RowsArgs {
  const int8_t* a;
  const int8_t* b;          // packed weights [k_pad / 64][n_pad][64]
  uint32_t a_bytes, b_bytes;
  int32_t M, N, n_pad, k_tiles, tiles_m;
  // A's 16-byte chunk c of K is chunk c % cpt of tap c / cpt (a matmul row: one tap of lda / 16)
  int32_t cpt, taps, C_pad;
  uint32_t cpt_magic, kw_magic;       // ceil(2^32 / d); 0: d == 1
  int32_t H, W, OH, OW, KW, SH, SW, PH, PW, DH, DW;
};

constexpr uint32_t ROWS_OOB = 0x80000000u;     // past every buffer (each under 2 GiB): loads zeros
constexpr int ROWS_WAVES = 8, ROWS_U = 4;

__device__ __forceinline__ int magic_div(int n, uint32_t magic) {
  return magic ? static_cast<int>(__umulhi(static_cast<uint32_t>(n), magic)) : n;
}

template <int RB, int CB>
__global__ void __launch_bounds__(ROWS_WAVES * 64) qrows_kernel(const RowsArgs g, const EpiDev e) {
  constexpr int LD = CB * 16 + 4;
  __shared__ int32_t part[ROWS_WAVES][RB * 16][LD];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kg = lane >> 4;
  const int tile_n = blockIdx.x / g.tiles_m;
  const int m0 = (blockIdx.x - tile_n * g.tiles_m) * RB * 16, n0 = tile_n * CB * 16;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(g.a), 0, g.a_bytes, BUF_DWORD3);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(g.b), 0, g.b_bytes, BUF_DWORD3);

  // this lane's input rows: the byte offset of tap (0, 0) (negative above / left of the image) and its pixel
  int32_t a_off[RB], ih0[RB], iw0[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int m = m0 + i * 16 + l16;
    const int img = m / (g.OH * g.OW), rem = m - img * g.OH * g.OW, oh = rem / g.OW;
    ih0[i] = m < g.M ? oh * g.SH - g.PH : -(1 << 28);        // a row past M is outside at every tap
    iw0[i] = (rem - oh * g.OW) * g.SW - g.PW;
    a_off[i] = ((img * g.H + (m < g.M ? ih0[i] : 0)) * g.W + iw0[i]) * g.C_pad;
  }
  uint32_t b_off[CB];
#pragma unroll
  for (int j = 0; j < CB; ++j) b_off[j] = static_cast<uint32_t>((n0 + j * 16 + l16) * 64 + kg * 16);

  v4i acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) acc[i][j] = v4i{0, 0, 0, 0};

  struct Steps {
    v4i a[ROWS_U][RB], b[ROWS_U][CB];
  };
  auto fetch = [&](Steps& t, int kt0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < ROWS_U; ++u) {
      const int kt = kt0 + u * ROWS_WAVES;
      const uint32_t soff = static_cast<uint32_t>(kt) * static_cast<uint32_t>(g.n_pad) * 64u;
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const bool in = kt < g.k_tiles && n0 + j * 16 + l16 < g.n_pad;
        t.b[u][j] = __builtin_amdgcn_raw_buffer_load_b128(rb, in ? b_off[j] + soff : ROWS_OOB, 0, 0);
      }
      const int c = kt * 4 + kg, tap = magic_div(c, g.cpt_magic);
      const int kh = magic_div(tap, g.kw_magic), kw = tap - kh * g.KW;
      const int dh = kh * g.DH, dw = kw * g.DW;
      const int rel = (dh * g.W + dw) * g.C_pad + (c - tap * g.cpt) * 16;
      const bool in = kt < g.k_tiles && tap < g.taps;
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const bool ok = in && unsigned(ih0[i] + dh) < unsigned(g.H) && unsigned(iw0[i] + dw) < unsigned(g.W);
        t.a[u][i] = __builtin_amdgcn_raw_buffer_load_b128(ra, ok ? static_cast<uint32_t>(a_off[i] + rel) : ROWS_OOB, 0, 0);
      }
    }
  };
  auto multiply = [&](const Steps& t) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < ROWS_U; ++u)
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(t.a[u][i], t.b[u][j], acc[i][j], 0, 0, 0);
  };
  constexpr int STRIDE = ROWS_WAVES * ROWS_U;
  Steps s0, s1;
  int kt = wave;
  if (kt < g.k_tiles) fetch(s0, kt);
  for (; kt < g.k_tiles; kt += 2 * STRIDE) {
    if (kt + STRIDE < g.k_tiles) fetch(s1, kt + STRIDE);
    multiply(s0);
    if (kt + STRIDE >= g.k_tiles) break;
    if (kt + 2 * STRIDE < g.k_tiles) fetch(s0, kt + 2 * STRIDE);
    multiply(s1);
  }
  // lane holds column l16 and rows 4 * kg .. + 3 of each block
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wave][i * 16 + 4 * kg + r][j * 16 + l16] = acc[i][j][r];
  lds_store_barrier();
  for (int o = threadIdx.x; o < RB * 16 * CB * 16; o += ROWS_WAVES * 64) {
    const int r = o / (CB * 16), c = o % (CB * 16);
    const int64_t row = m0 + r;
    const int col = n0 + c;
    if (row >= g.M || col >= g.N) continue;
    int32_t sum = 0;
#pragma unroll
    for (int w = 0; w < ROWS_WAVES; ++w) sum += part[w][r][c];
    if (e.out_acc) e.out_acc[row * e.ldacc + col] = sum;
    epi_store(e, epi_steps(e, dequant(sum, e.scale[col]), row, col), row, col);
  }
}

template <int RB, int CB>
static void qrows_start(const RowsArgs& g, const EpiDev& e, hipStream_t stream) {
  RowsArgs a = g;
  a.tiles_m = (g.M + RB * 16 - 1) / (RB * 16);
  const unsigned grid = static_cast<unsigned>(a.tiles_m) * static_cast<unsigned>((g.N + CB * 16 - 1) / (CB * 16));
  hipLaunchKernelGGL((qrows_kernel<RB, CB>), dim3(grid), dim3(ROWS_WAVES * 64), 0, stream, a, e);
}

// How many 64 x 32 tiles of qgemm_kernel a result may have, by the length of K in 64-byte steps:
// its launch takes as long for one tile as for one per CU, this one's grows with the tiles.
// us, qgemm_kernel / this one:
//   64 steps   4096 x 4096, 128 tiles 12.8 / 10.4, 256 13.4 / 18.9;  4096 x 1000, 96 tiles 12.8 / 12.5
//   36         layer 3, 104 tiles 12.6 / 9.5, 152 12.7 / 12.6
//   9          layer 1, 98 tiles 8.5 / 6.5, 196 8.5 / 8.5;  stride 2 to 128 channels, 148 7.3 / 8.4
//   8          512 x 512, 48 tiles 5.7 / 4.8, 80 5.8 / 6.4
//   5 - 6      8 tiles 4.7 / 4.2, 38 4.8 / 5.0, 80 4.5 / 5.8
//   2          32 tiles 4.3 / 3.7, 80 4.4 / 5.6
static bool qrows_pays(int64_t M, int64_t N, int64_t k_tiles) {
  const int64_t tiles = (M + 63) / 64 * ((N + 31) / 32), most = device_cu_count() / (k_tiles >= 9 ? 2 : k_tiles >= 8 ? 4 : 8);
  return k_tiles >= 2 && tiles <= most;
}

int qrows_launch(const int8_t* x, int64_t lda, const mr_conv_geom* cg, const int8_t* b, int64_t k_pad, int64_t n_pad,
                 int64_t M, int64_t N, const EpiDev& e, hipStream_t stream) {
  RowsArgs g = {};
  int64_t a_bytes;
  int32_t cpt;
  if (cg) {
    if (cg->c_pad % 16 != 0) return MR_EUNSUPPORTED;       // the 4-channel stem layout
    a_bytes = int64_t(cg->n) * cg->h * cg->w * cg->c_pad;
    cpt = cg->c_pad / 16;
    g.taps = cg->kh * cg->kw;
    g.C_pad = cg->c_pad;
    g.H = cg->h; g.W = cg->w; g.OH = cg->oh; g.OW = cg->ow; g.KW = cg->kw;
    g.SH = cg->sh; g.SW = cg->sw; g.PH = cg->ph; g.PW = cg->pw; g.DH = cg->dh; g.DW = cg->dw;
  } else {       // M images of one pixel of lda channels
    a_bytes = M * lda;
    cpt = static_cast<int32_t>(lda / 16);
    g.taps = 1;
    g.C_pad = static_cast<int32_t>(lda);
    g.H = g.W = g.OH = g.OW = g.KW = g.SH = g.SW = g.DH = g.DW = 1;
  }
  // magic divisions are exact for n * d < 2^32
  const int64_t chunks = k_pad / 16 + 4 * ROWS_WAVES * ROWS_U;
  if (!qrows_pays(M, N, k_pad / 64) || a_bytes >= (int64_t(1) << 31) || k_pad * n_pad >= (int64_t(1) << 31) ||
      lda >= (int64_t(1) << 31) || chunks * cpt >= (int64_t(1) << 32) || chunks * g.KW >= (int64_t(1) << 32))
    return MR_EUNSUPPORTED;
  auto magic = [](uint32_t d) { return d <= 1 ? 0u : static_cast<uint32_t>(((uint64_t(1) << 32) + d - 1) / d); };
  g.a = x;
  g.b = b;
  g.a_bytes = static_cast<uint32_t>(a_bytes);
  g.b_bytes = static_cast<uint32_t>(k_pad * n_pad);
  g.M = static_cast<int32_t>(M);
  g.N = static_cast<int32_t>(N);
  g.n_pad = static_cast<int32_t>(n_pad);
  g.k_tiles = static_cast<int32_t>(k_pad / 64);
  g.cpt = cpt;
  g.cpt_magic = magic(static_cast<uint32_t>(cpt));
  g.kw_magic = magic(static_cast<uint32_t>(g.KW));
  // the widest tile (fewest loads per product) that still gives every CU a workgroup
  const int64_t cus = device_cu_count();
  auto grid = [&](int rb, int cb) { return (M + rb * 16 - 1) / (rb * 16) * ((N + cb * 16 - 1) / (cb * 16)); };
  if (grid(2, 2) >= cus) qrows_start<2, 2>(g, e, stream);
  else if (grid(1, 2) >= cus) qrows_start<1, 2>(g, e, stream);
  else qrows_start<1, 1>(g, e, stream);
  MR_LAUNCH_CHECK("qrows");
  return MR_OK;
}

}  // namespace mr
