// Bias-free linear layers of the model's sublayers for inference: up to three that
// share an input in one launch (q, k, v), and gate and up with silu(gate) * up.
// 16-bit tensors (bf16 or fp16), fp32 sums, one rounding.
#include "mhc_gemm.hpp"

namespace mhc {
namespace {

// Which weight a column tile belongs to, and its first row there.
struct Segment {
  const char* w;
  uint16_t* out;
  int n0, N;
};
template <int COLS>
__device__ __forceinline__ Segment segment(const LinearArgs& a, int tile) {
  int i = 0;
  for (; i + 1 < a.count; ++i) {
    const int t = (a.n[i] + COLS - 1) / COLS;
    if (tile < t) break;
    tile -= t;
  }
  return {static_cast<const char*>(a.w[i]), static_cast<uint16_t*>(a.out[i]), tile * COLS, a.n[i]};
}

// ------------------------------------------------------------------- few rows
// Few rows (a decode step) leave a product bound by the latency of one pass over
// the weights, so each 16 x 16 tile of the output is a workgroup, its K split over
// NW waves that issue U steps' loads at once and meet in LDS.  GLU: the gate and
// the up tile.  64 rows, K = 768: 1536 columns 5.4 us, 768 columns 3.9 us; the
// 64 x 64 tiles below 5.8 and 6.2.
template <bool F16, int NW, bool GLU>
__global__ __launch_bounds__(NW * 64) void skinny_kernel(LinearArgs a) {
  constexpr int WT = GLU ? 2 : 1;  // weight tiles
  constexpr int U = 3;             // steps in flight
  __shared__ __align__(16) f32x4_t red[NW][WT][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const Segment s = segment<16>(a, blockIdx.x);
  const int64_t m0 = (int64_t)blockIdx.y * 16;
  const int64_t kb = (int64_t)a.K * 2;
  const int64_t wrow = min(s.n0 + r, s.N - 1);
  const char* wp[WT];
  wp[0] = s.w + wrow * kb + 16 * g;
  if constexpr (GLU) wp[1] = static_cast<const char*>(a.w[1]) + wrow * kb + 16 * g;
  const char* xp = static_cast<const char*>(a.x) + min(m0 + r, a.M - 1) * kb + 16 * g;
  f32x4_t acc[WT];
#pragma unroll
  for (int w = 0; w < WT; ++w) acc[w] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int steps = a.K / 32;
  for (int k0 = wave; k0 < steps; k0 += NW * U) {  // uniform
    U32x4 wv[U][WT], xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * NW;
      if (k >= steps) break;  // uniform
#pragma unroll
      for (int w = 0; w < WT; ++w) wv[u][w] = *reinterpret_cast<const U32x4*>(wp[w] + k * 64);
      xv[u] = *reinterpret_cast<const U32x4*>(xp + k * 64);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k0 + u * NW >= steps) break;
#pragma unroll
      for (int w = 0; w < WT; ++w) acc[w] = mfma16<F16>(wv[u][w], xv[u], acc[w]);
    }
  }
#pragma unroll
  for (int w = 0; w < WT; ++w) red[wave][w][lane] = acc[w];
  __syncthreads();
  if (tid >= 64) return;
  f32x4_t v[WT];
#pragma unroll
  for (int w = 0; w < WT; ++w) {
    v[w] = red[0][w][lane];
#pragma unroll
    for (int k = 1; k < NW; ++k) v[w] += red[k][w][lane];
  }
  const int64_t row = m0 + r;
  const int col = s.n0 + 4 * g;
  if (row >= a.M || col >= s.N) return;
  if constexpr (GLU)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[0][i] = silu_mul(v[0][i], v[1][i]);
  store4<F16>(s.out + row * s.N + col, v[0]);
}

// ------------------------------------------------------------------ many rows
// gemm_tile over BM x BN tiles; workgroups of one XCD take neighbouring tiles.
template <bool F16, typename G, bool GLU>
__global__ __launch_bounds__(G::THREADS, G::WAVES) void linear_kernel(LinearArgs a, int col_tiles) {
  __shared__ __align__(16) char lds[G::LDS];
  constexpr int BM = G::BM, BN = G::BN;
  constexpr int kCols = GLU ? BN / 2 : BN;
  const int work = gridDim.x, chunk = (work + 7) / 8;
  // the last chunks of a count that 8 does not divide are shorter
  const int xcd = blockIdx.x % 8, full = work % 8 == 0 ? 8 : work % 8;
  const int logical = xcd * chunk - max(0, xcd - full) + blockIdx.x / 8;
  const Segment s = segment<kCols>(a, logical % col_tiles);
  const int64_t row0 = (int64_t)(logical / col_tiles) * BM;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % G::WGM, wn = wave / G::WGM;
  const int64_t kb = (int64_t)a.K * 2;
  auto a_row = [&](int i) { return (uint32_t)(min(row0 + i, a.M - 1) - row0) * (uint32_t)kb; };
  auto b_base = [&](int n) { return (GLU && n >= kCols ? static_cast<const char*>(a.w[1]) : s.w) + s.n0 * kb; };
  auto b_row = [&](int n) { return (uint32_t)min(n % kCols, s.N - 1 - s.n0) * (uint32_t)kb; };
  constexpr int HALF = G::NT / 2;
  auto col_tile = [&](int n) {
    return GLU ? wn * HALF + (n >= HALF ? n - HALF + BN / 32 : n) : wn * G::NT + n;
  };
  f32x4_t acc[G::NT][G::MT];
  gemm_tile<F16, G>(lds, a.K, static_cast<const char*>(a.x) + row0 * kb, a_row, b_base, b_row, col_tile, acc);
  const int64_t row = row0 + wm * G::WM;
  const int col = s.n0 + wn * (GLU ? G::WN / 2 : G::WN);
  if constexpr (GLU)
#pragma unroll
    for (int n = 0; n < HALF; ++n)
#pragma unroll
      for (int m = 0; m < G::MT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[n][m][i] = silu_mul(acc[n][m][i], acc[n + HALF][m][i]);
  store_tile<F16, G, GLU ? G::WN / 2 : G::WN>(lds, s.out + row * s.N + col, s.N, a.M - row, s.N - col,
                                              [&](int n, int m) { return acc[n][m]; });
}

template <bool F16, bool GLU, typename G>
hipError_t launch_tiles(const LinearArgs& a, int64_t work, int col_tiles, hipStream_t s) {
  linear_kernel<F16, G, GLU><<<dim3((unsigned)work), G::THREADS, 0, s>>>(a, col_tiles);
  return hipGetLastError();
}

// 16 x 16 tiles up to 448 of them (K = 768 unless noted, us): 384 (64 rows x 1536) 5.4
// against 5.8 for 64 x 64 tiles, 384 (128 x 768, K = 2048) 9.4 against 11.1; 512 (64 x
// 2048, GLU) 7.9 against 6.8, 768 (256 x 768) 7.6 against 6.4.  Above, pick_tile's:
// 8192 rows: 1536 columns 22.2 us (868 TFLOP/s; 28.4 with 128 x 128 tiles of 32-column
// slices and stores from the accumulators, the three library products 39.0), GLU 2048
// columns 52.1 us (990 TFLOP/s; 64.2 before, two library products, silu and the
// multiplication 83.3).
struct Choice {
  Tile tile;
  int64_t work;   // tiles
  int col_tiles;
};
Choice choose(const LinearArgs& a) {
  auto tiles = [&](int width) {
    int t = 0;
    for (int i = 0; i < (a.glu ? 1 : a.count); ++i) t += (a.n[i] + width - 1) / width;
    return t;
  };
  auto rows = [&](int height) { return (a.M + height - 1) / height; };
  if (tiles(16) * rows(16) <= 448) return {Tile::k16x16, tiles(16) * rows(16), tiles(16)};
  auto cols = [&](int width) { return tiles(a.glu ? width / 2 : width); };  // GLU: half gate, half up
  const Tile t = pick_tile(rows, cols, a.glu);
  switch (t) {
    case Tile::k256x256: return {t, rows(256) * cols(256), cols(256)};
    case Tile::k128x192: return {t, rows(128) * cols(192), cols(192)};
    case Tile::k128x128: return {t, rows(128) * cols(128), cols(128)};
    case Tile::k128x64: return {t, rows(128) * cols(64), cols(64)};
    default: return {t, rows(64) * cols(64), cols(64)};
  }
}

template <bool F16, bool GLU>
hipError_t launch(const LinearArgs& a, hipStream_t s) {
  const Choice c = choose(a);
  switch (c.tile) {
    case Tile::k16x16: {
      const dim3 grid((unsigned)c.col_tiles, (unsigned)((a.M + 15) / 16));
      if (a.K >= 1536) skinny_kernel<F16, 16, GLU><<<grid, 16 * 64, 0, s>>>(a);
      else skinny_kernel<F16, 8, GLU><<<grid, 8 * 64, 0, s>>>(a);
      return hipGetLastError();
    }
    case Tile::k256x256: return launch_tiles<F16, GLU, GemmTile<256, 256, 4, 2, 2>>(a, c.work, c.col_tiles, s);
    case Tile::k128x192:
      if constexpr (!GLU) return launch_tiles<F16, GLU, GemmTile<128, 192, 4, 2, 2>>(a, c.work, c.col_tiles, s);
      [[fallthrough]];
    case Tile::k128x128: return launch_tiles<F16, GLU, GemmTile<128, 128, 4, 2, 2>>(a, c.work, c.col_tiles, s);
    case Tile::k128x64: return launch_tiles<F16, GLU, GemmTile<128, 64, 4, 1, 2>>(a, c.work, c.col_tiles, s);
    default: return launch_tiles<F16, GLU, GemmTile<64, 64, 2, 2, 4>>(a, c.work, c.col_tiles, s);
  }
}

}  // namespace

// Where the kernels are no slower than the library's (torch 2.10; GPU times of graph
// replays over 1907, 202 and 480 sizes, M 1 to 65536, K 256 to 8192; a round fills the
// chip: two workgroups a CU, one of the 256 x 256 tiles).  The kernels keep K in one
// workgroup, so a long K makes a long tile; the library's own splits it.
//   One layer: a kernel's gain is the host's (a call costs 11 us, the library's 20), so
//     it pays while the host bounds the call: kernels of up to some 13 us.  16 x 16 tiles
//     to K = 6464 in one tile a CU (M x K x N: 64 x 3264 x 1024 7.9 us against the library's
//     10.6, 64 x 6464 x 1024 13.2 and 16.4, 128 x 4096 x 64 8.9 and 7.6), 2560 past that
//     (128 x 2048 x 768 9.1 and 6.0, 128 x 4096 x 768 16.0 and 7.4), 64 x 64 ones to 2048 in one
//     a CU (512 x 2048 x 2048 12.7 and 10.8), to 1024 past that (512 x 1536 x 2432 15.8 and
//     11.7), 128 x 64 to K = 768 (512 x 768 x 6400 11.9 and 10.6; at 1024 half the sizes are
//     9% slower or more, up to 15.0).  Larger tiles pay where they win by themselves:
//     128 x 128 to K = 512 in one round (8192 x 512 x 1024 12.9 and 15.0; two rounds, 2048 x
//     512 x 6400, 24.1 and 20.1), 128 x 192 to K = 1024 (8192 x 768 x 768 14.1 and 14.9,
//     8192 x 1024 x 768 16.8 and 17.9, 12000 x 1536 x 768 32.8 and 28.7).  256 x 256 ones
//     mostly lose (4096 x 768 x 6400 50 and 42).
//   q, k, v: two launches less.  128 x 128 tiles while rounds x K is up to 4096 (2048
//     rows, hidden 2048, 30.7 and 42.4; 12000 rows 157 and 141), 128 x 192 up to 3072 (two
//     rounds: 8192 x 2304 at K = 1536 54 and 71, 2051 x 8064 at K = 1984 84 and 74), 256 x
//     256 up to 2560
//     (16384 rows, hidden 768, 49.1 and 54.4; 65536 rows 187 and 167; 16384 x 3072 at K =
//     1024, three rounds, 7% slower), the rest to K = 4096 (never slower).
//   Gate and up: also two passes less.  128 x 128 to K = 1536 (1 to 170% faster, 5400 rows
//     of 4864 or more columns 3% slower), past that by the same rounds x K (2048 columns,
//     two rounds 5% faster, three 6% slower); the rest to K = 3072 (2% faster and more).
bool linear_pays(const LinearArgs& a) {
  const Choice c = choose(a);
  const int64_t cus = device_cus(), chip = c.tile == Tile::k256x256 ? cus : 2 * cus;
  const int64_t rounds = (c.work + chip - 1) / chip;
  if (a.glu) return c.tile == Tile::k128x128 && a.K > 1536 ? rounds * a.K <= 4096 : a.K <= 3072;
  if (a.count > 1) {
    if (c.tile == Tile::k128x128) return rounds * a.K <= 4096;
    if (c.tile == Tile::k128x192) return rounds * a.K <= 3072;
    return c.tile == Tile::k256x256 ? rounds * a.K <= 2560 : a.K <= 4096;
  }
  switch (c.tile) {
    case Tile::k16x16: return a.K <= (c.work <= cus ? 6464 : 2560);
    case Tile::k64x64: return a.K <= (c.work <= cus ? 2048 : 1024);
    case Tile::k128x64: return a.K <= 768;
    case Tile::k128x128: return a.K <= 512 && rounds == 1;
    case Tile::k128x192: return a.K <= 1024;
    default: return false;
  }
}

hipError_t launch_linear(const LinearArgs& a, hipStream_t s) {
  if (a.glu) return a.f16 ? launch<true, true>(a, s) : launch<false, true>(a, s);
  return a.f16 ? launch<true, false>(a, s) : launch<false, false>(a, s);
}

}  // namespace mhc
