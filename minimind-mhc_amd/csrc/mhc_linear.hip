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
template <bool F16, bool GLU>
hipError_t launch(const LinearArgs& a, hipStream_t s) {
  auto tiles = [&](int width) {
    int t = 0;
    for (int i = 0; i < (GLU ? 1 : a.count); ++i) t += (a.n[i] + width - 1) / width;
    return t;
  };
  auto rows = [&](int height) { return (a.M + height - 1) / height; };
  if (tiles(16) * rows(16) <= 448) {
    const dim3 grid((unsigned)tiles(16), (unsigned)rows(16));
    if (a.K >= 1536) skinny_kernel<F16, 16, GLU><<<grid, 16 * 64, 0, s>>>(a);
    else skinny_kernel<F16, 8, GLU><<<grid, 8 * 64, 0, s>>>(a);
    return hipGetLastError();
  }
  auto cols = [&](int width) { return tiles(GLU ? width / 2 : width); };  // GLU: half gate, half up
  switch (pick_tile(rows, cols, GLU)) {
    case Tile::k256x256: return launch_tiles<F16, GLU, GemmTile<256, 256, 4, 2, 2>>(a, rows(256) * cols(256), cols(256), s);
    case Tile::k128x192:
      if constexpr (!GLU) return launch_tiles<F16, GLU, GemmTile<128, 192, 4, 2, 2>>(a, rows(128) * cols(192), cols(192), s);
      [[fallthrough]];
    case Tile::k128x128: return launch_tiles<F16, GLU, GemmTile<128, 128, 4, 2, 2>>(a, rows(128) * cols(128), cols(128), s);
    case Tile::k128x64: return launch_tiles<F16, GLU, GemmTile<128, 64, 4, 1, 2>>(a, rows(128) * cols(64), cols(64), s);
    default: return launch_tiles<F16, GLU, GemmTile<64, 64, 2, 2, 4>>(a, rows(64) * cols(64), cols(64), s);
  }
}

}  // namespace

hipError_t launch_linear(const LinearArgs& a, hipStream_t s) {
  if (a.glu) return a.f16 ? launch<true, true>(a, s) : launch<false, true>(a, s);
  return a.f16 ? launch<true, false>(a, s) : launch<false, false>(a, s);
}

}  // namespace mhc
