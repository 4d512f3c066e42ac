// Routed-expert feed-forward layer for inference (model/model_minimind.py:270-298):
// top-k selection, grouping of the tokens by expert, the experts' SwiGLU products on
// MFMA and the weighted sum, with no host synchronisation.  16-bit tensors (bf16 or
// fp16), fp32 sums.
#include "mhc_gemm.hpp"

namespace mhc {
namespace {

template <bool F16>
__device__ __forceinline__ float to_f32(uint16_t b) {
  return F16 ? f16_bits_to_f32(b) : bf16_bits_to_f32(b);
}
template <bool F16>
__device__ __forceinline__ float rounded(float v) {
  return round_to(v, F16 ? kF16 : kBF16);
}

// ------------------------------------------------------------------- grouping
constexpr int kRouteTok = 256;  // tokens a workgroup of the two grouping launches takes

// One token a thread: its top-k experts (the largest probability first, the lower
// index where two are equal) and their weights, rounded as the torch ops round
// them; per workgroup, how many tokens each expert got.
template <bool F16>
__global__ __launch_bounds__(kRouteTok) void moe_route_kernel(MoeArgs a) {
  __shared__ int count[kMoeMaxExperts];
  const int tid = threadIdx.x;
  if (tid < a.experts) count[tid] = 0;
  __syncthreads();
  const int64_t tok = (int64_t)blockIdx.x * kRouteTok + tid;
  if (tok < a.M) {
    const uint16_t* p = static_cast<const uint16_t*>(a.probs) + tok * a.experts;
    uint32_t used = 0;
    float w[kMoeMaxTopk], sum = 0.f;
    int id[kMoeMaxTopk];
#pragma unroll
    for (int k = 0; k < kMoeMaxTopk; ++k) {
      if (k >= a.topk) break;
      int best = -1;
      float bv = 0.f;
      for (int e = 0; e < a.experts; ++e) {
        const float v = to_f32<F16>(p[e]);
        if (!(used >> e & 1) && (best < 0 || v > bv)) {
          best = e;
          bv = v;
        }
      }
      used |= 1u << best;
      id[k] = best;
      w[k] = bv;
      sum += bv;
    }
    if (a.norm_topk) sum = rounded<F16>(rounded<F16>(sum) + rounded<F16>(1e-20f));
#pragma unroll
    for (int k = 0; k < kMoeMaxTopk; ++k) {
      if (k >= a.topk) break;
      a.pick[tok * a.topk + k] = id[k];
      a.pick_w[tok * a.topk + k] = a.norm_topk ? rounded<F16>(__fdiv_rn(w[k], sum)) : w[k];
      atomicAdd(&count[id[k]], 1);
    }
  }
  __syncthreads();
  if (tid < a.experts) a.counts[(int64_t)blockIdx.x * a.experts + tid] = count[tid];
}

// Gives each (token, expert) pair its row among the expert's rows.  A row's place
// in its expert's group depends on the order of LDS atomics; its value does not
// depend on its place.
__global__ __launch_bounds__(kRouteTok) void moe_group_kernel(MoeArgs a) {
  __shared__ int total[kMoeMaxExperts], before[kMoeMaxExperts], next[kMoeMaxExperts];
  const int tid = threadIdx.x;
  if (tid < a.experts) total[tid] = before[tid] = 0;
  __syncthreads();
  // 256 threads stride over [workgroups][experts]
  for (int64_t i = tid; i < (int64_t)gridDim.x * a.experts; i += kRouteTok) {
    const int blk = (int)(i / a.experts), e = (int)(i % a.experts), n = a.counts[i];
    if (n) {
      atomicAdd(&total[e], n);
      if (blk < (int)blockIdx.x) atomicAdd(&before[e], n);
    }
  }
  __syncthreads();
  if (tid < a.experts) {
    int base = 0;
    for (int e = 0; e < tid; ++e) base += total[e];
    next[tid] = base + before[tid];
    if (blockIdx.x == 0) {
      a.offsets[tid] = base;
      if (tid == a.experts - 1) a.offsets[a.experts] = base + total[tid];
    }
  }
  __syncthreads();
  const int64_t tok = (int64_t)blockIdx.x * kRouteTok + tid;
  if (tok >= a.M) return;
  for (int k = 0; k < a.topk; ++k) {
    const int64_t i = tok * a.topk + k;
    const int slot = atomicAdd(&next[a.pick[i]], 1);
    a.slot_of[i] = slot;
    a.row_tok[slot] = (int)tok;
    a.row_w[slot] = a.pick_w[i];
  }
}

// ------------------------------------------------------------ grouped products
// C[row][n] of one expert's rows, a BM x BN tile (gemm_tile) a workgroup.
//   * GLU: BN / 2 gate and the matching BN / 2 up columns; stores silu(gate) * up.
//     Otherwise: BN columns of the down projection, scaled by the row's weight.
//   * Workgroups of one XCD take neighbouring tiles (the same expert's weights stay
//     in its L2).
// 8192 tokens, 8 experts, top 2, 768 x 1024: 71 us for gate and up (128 x 128 tiles, 51.5
// GFLOP, 725 TFLOP/s; 77 with 32-column slices and stores from the accumulators), 41 us
// for down (128 x 192 tiles, 25.8 GFLOP, 629 TFLOP/s; 47 before).  As many rows of a dense
// layer take 56 and 27 us, on 512 whole tiles each.  The experts' part-filled last tiles
// are 3% of the operations, but they take gate and up just past whole rounds of the chip
// (2112 tiles, 4.1 rounds of two a CU; 544 of 256 x 256, 2.1 rounds, 72 us); the gathered
// rows cost no more traffic (113 MB read either way).
// The layer's loop over experts took 1.6 ms, of which library products were 290 us.
template <bool F16, typename G, bool GLU>
__global__ __launch_bounds__(G::THREADS, G::WAVES) void moe_gemm_kernel(MoeArgs a) {
  constexpr int BM = G::BM, BN = G::BN;
  __shared__ __align__(16) char lds[G::LDS];
  const int N = GLU ? a.inter : a.hidden;
  const int K = GLU ? a.hidden : a.inter;
  constexpr int kCols = GLU ? BN / 2 : BN;
  const int ntn = (N + kCols - 1) / kCols;
  // this workgroup's tile: count the row tiles of every expert
  int tiles = 0;
  for (int e = 0; e < a.experts; ++e) tiles += (a.offsets[e + 1] - a.offsets[e] + BM - 1) / BM;
  const int work = tiles * ntn, chunk = (work + 7) / 8;
  const int at = blockIdx.x / 8, logical = (blockIdx.x % 8) * chunk + at;
  if (at >= chunk || logical >= work) return;
  int mt = logical / ntn, e = 0;
  const int n0 = logical % ntn * kCols;
  for (; e < a.experts; ++e) {
    const int t = (a.offsets[e + 1] - a.offsets[e] + BM - 1) / BM;
    if (mt < t) break;
    mt -= t;
  }
  const int row_end = a.offsets[e + 1], row0 = a.offsets[e] + mt * BM;

  const int r = threadIdx.x & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % G::WGM, wn = wave / G::WGM;
  const uint32_t kb = (uint32_t)K * 2;
  const char* x = GLU ? static_cast<const char*>(a.x) : static_cast<const char*>(a.h) + (int64_t)row0 * kb;
  auto a_row = [&](int i) {
    const int row = min(row0 + i, row_end - 1);
    return GLU ? (uint32_t)a.row_tok[row] * kb : (uint32_t)(row - row0) * kb;
  };
  auto b_base = [&](int n) {
    const void* w = GLU ? (n < kCols ? a.gate_w[e] : a.up_w[e]) : a.down_w[e];
    return static_cast<const char*>(w) + (int64_t)n0 * kb;
  };
  auto b_row = [&](int n) { return (uint32_t)min(n % kCols, N - 1 - n0) * kb; };
  // GLU: this wave's gate columns, then its up columns
  constexpr int HALF = G::NT / 2;
  auto col_tile = [&](int n) {
    return GLU ? wn * HALF + (n >= HALF ? n - HALF + BN / 32 : n) : wn * G::NT + n;
  };
  f32x4_t acc[G::NT][G::MT];
  gemm_tile<F16, G>(lds, K, x, a_row, b_base, b_row, col_tile, acc);
  const int row = row0 + wm * G::WM, col = n0 + wn * (GLU ? G::WN / 2 : G::WN);
  float w[G::MT];
  if constexpr (!GLU)
#pragma unroll
    for (int m = 0; m < G::MT; ++m) w[m] = a.row_w[min(row + m * 16 + r, row_end - 1)];
  uint16_t* out = static_cast<uint16_t*>(GLU ? a.h : a.y) + (int64_t)row * N + col;
#pragma unroll
  for (int n = 0; n < (GLU ? HALF : G::NT); ++n)
#pragma unroll
    for (int m = 0; m < G::MT; ++m) {
      if constexpr (GLU) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[n][m][i] = silu_mul(acc[n][m][i], acc[n + HALF][m][i]);
      } else {
        acc[n][m] *= w[m];
      }
    }
  store_tile<F16, G, GLU ? G::WN / 2 : G::WN>(lds, out, N, row_end - row, N - col,
                                              [&](int n, int m) { return acc[n][m]; });
}

// out[token] = the sum of its experts' rows, 8 columns a thread; and a.zero = 0, which
// took a 4.5 us launch of its own.
template <bool F16>
__global__ __launch_bounds__(256) void moe_combine_kernel(MoeArgs a) {
  const int per = a.hidden / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i == 0 && a.zero) *static_cast<uint16_t*>(a.zero) = 0;
  if (i >= a.M * per) return;
  const int64_t tok = i / per;
  const int col = (int)(i - tok * per) * 8;
  float s[8] = {};
  for (int k = 0; k < a.topk; ++k) {
    const int64_t slot = a.slot_of[tok * a.topk + k];
    const U32x4 v = *reinterpret_cast<const U32x4*>(static_cast<const uint16_t*>(a.y) + slot * a.hidden + col);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s[2 * j] += to_f32<F16>((uint16_t)(v.v[j] & 0xffffu));
      s[2 * j + 1] += to_f32<F16>((uint16_t)(v.v[j] >> 16));
    }
  }
  U32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o.v[j] = pack2<F16>(s[2 * j], s[2 * j + 1]);
  *reinterpret_cast<U32x4*>(static_cast<uint16_t*>(a.out) + tok * a.hidden + col) = o;
}

template <bool F16, bool GLU, typename G>
hipError_t launch_tiles(const MoeArgs& a, hipStream_t s) {
  // most row tiles: every expert's last one may be partly filled
  const int64_t rows = a.M * a.topk, tiles = rows / G::BM + (rows < a.experts ? rows : a.experts);
  constexpr int cols = GLU ? G::BN / 2 : G::BN;
  const int64_t work = tiles * (((GLU ? a.inter : a.hidden) + cols - 1) / cols);
  moe_gemm_kernel<F16, G, GLU><<<dim3((unsigned)((work + 7) / 8 * 8)), G::THREADS, 0, s>>>(a);
  return hipGetLastError();
}

// The dense layers' rule; half an expert's last row tile is padding on average.
template <bool F16, bool GLU>
hipError_t launch_gemm(const MoeArgs& a, hipStream_t s) {
  auto rows = [&](int height) { return a.M * a.topk / height + (a.experts + 1) / 2; };
  auto cols = [&](int width) {
    const int w = GLU ? width / 2 : width;
    return ((GLU ? a.inter : a.hidden) + w - 1) / w;
  };
  switch (pick_tile(rows, cols, GLU)) {
    case Tile::k256x256: return launch_tiles<F16, GLU, GemmTile<256, 256, 4, 2, 2>>(a, s);
    case Tile::k128x192:
      if constexpr (!GLU) return launch_tiles<F16, GLU, GemmTile<128, 192, 4, 2, 2>>(a, s);
      [[fallthrough]];
    case Tile::k128x128: return launch_tiles<F16, GLU, GemmTile<128, 128, 4, 2, 2>>(a, s);
    case Tile::k128x64: return launch_tiles<F16, GLU, GemmTile<128, 64, 4, 1, 2>>(a, s);
    default: return launch_tiles<F16, GLU, GemmTile<64, 64, 2, 2, 4>>(a, s);
  }
}

template <bool F16>
hipError_t launch(const MoeArgs& a, hipStream_t s) {
  const unsigned route = (unsigned)((a.M + kRouteTok - 1) / kRouteTok);
  moe_route_kernel<F16><<<dim3(route), kRouteTok, 0, s>>>(a);
  moe_group_kernel<<<dim3(route), kRouteTok, 0, s>>>(a);
  if (hipError_t e = launch_gemm<F16, true>(a, s); e != hipSuccess) return e;
  if (hipError_t e = launch_gemm<F16, false>(a, s); e != hipSuccess) return e;
  const int64_t vec = a.M * (a.hidden / 8);
  moe_combine_kernel<F16><<<dim3((unsigned)((vec + 255) / 256)), 256, 0, s>>>(a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_moe(const MoeArgs& a, hipStream_t s) { return a.f16 ? launch<true>(a, s) : launch<false>(a, s); }

// counts, offsets, pick, pick_w, slot_of, row_tok, row_w, then h and y, each piece
// 16-byte aligned.
static int64_t pad16(int64_t b) { return (b + 15) / 16 * 16; }
int64_t moe_workspace(MoeArgs& a, char* base) {
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    char* p = base ? base + at : nullptr;
    at += pad16(bytes);
    return p;
  };
  const int64_t blocks = (a.M + kRouteTok - 1) / kRouteTok, rows = a.M * a.topk;
  a.counts = reinterpret_cast<int*>(take(blocks * a.experts * 4));
  a.offsets = reinterpret_cast<int*>(take((a.experts + 1) * 4));
  a.pick = reinterpret_cast<int*>(take(rows * 4));
  a.pick_w = reinterpret_cast<float*>(take(rows * 4));
  a.slot_of = reinterpret_cast<int*>(take(rows * 4));
  a.row_tok = reinterpret_cast<int*>(take(rows * 4));
  a.row_w = reinterpret_cast<float*>(take(rows * 4));
  a.h = take(rows * a.inter * 2);
  a.y = take(rows * a.hidden * 2);
  return at;
}

}  // namespace mhc
