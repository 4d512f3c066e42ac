// Routed-expert feed-forward layer for inference (model/model_minimind.py:270-298):
// top-k selection, grouping of the tokens by expert, the experts' SwiGLU products on
// MFMA and the weighted sum, with no host synchronisation.  16-bit tensors (bf16 or
// fp16), fp32 sums.
#include "mhc_internal.hpp"

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
// C[row][n] of one expert's rows: 128 rows x 256 weight rows a 4-wave workgroup,
// K in steps of 32 through a ring of three LDS stages filled by direct-to-LDS
// loads (two steps ahead).  Each wave holds 64 rows x 128 columns: 128
// accumulator registers, 12 LDS reads for 32 MFMAs.
//   * Both operands lie K-contiguous in memory, so a lane's 16 bytes are the MFMA
//     operand.  A stage row is 64 bytes; its four 16-byte slots are permuted by the
//     row's bits 2 and 3 (on the global side), so 16 rows hit all 64 banks.
//   * The product is formed as W x^T, so a lane ends with four neighbouring columns
//     of one row.
//   * GLU: 128 gate and the matching 128 up columns; stores silu(gate) * up.
//     Otherwise: 256 columns of the down projection, scaled by the row's weight.
//   * Workgroups of one XCD take neighbouring tiles (the same expert's weights stay
//     in its L2).
// 8192 tokens, 8 experts, top 2, 768 x 1024: 84 us for gate and up (51.5 GFLOP, 613
// TFLOP/s), 48 us for down (25.8 GFLOP, 535 TFLOP/s); bound by the LDS reads beside
// the MFMAs (12 reads of 1 KiB against 512 MFMA cycles a wave and step).  The layer's
// loop over experts took 1.6 ms, of which library products were 290 us.
template <bool F16, bool GLU>
__global__ __launch_bounds__(256, 2) void moe_gemm_kernel(MoeArgs a) {
  constexpr int BM = 128, BN = 256, STAGES = 3;
  constexpr int kStageBytes = (BM + BN) * 64;
  __shared__ __align__(16) char lds[STAGES * kStageBytes];
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

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1;

  // stage pieces of 16 rows x 64 bytes: 8 of x rows, then 16 of weight rows
  constexpr int PIECES = (BM + BN) / 16 / 4;
  const char* src[PIECES];
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int piece = wave * PIECES + i;
    const int prow = lane >> 2, slot = (lane & 3) ^ ((prow >> 2) & 3);
    const char* base;
    if (piece < BM / 16) {
      const int row = min(row0 + piece * 16 + prow, row_end - 1);
      base = GLU ? static_cast<const char*>(a.x) + (int64_t)a.row_tok[row] * K * 2
                 : static_cast<const char*>(a.h) + (int64_t)row * K * 2;
    } else {
      const int n = (piece - BM / 16) * 16 + prow;
      const void* w = GLU ? (n < kCols ? a.gate_w[e] : a.up_w[e]) : a.down_w[e];
      base = static_cast<const char*>(w) + (int64_t)min(n0 + n % kCols, N - 1) * K * 2;
    }
    src[i] = base + slot * 16;
  }
  auto issue = [&](int stage) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)src[i],
          (__attribute__((address_space(3))) void*)(lds + stage * kStageBytes + (wave * PIECES + i) * 1024),
          16, 0, 0);
      src[i] += 64;
    }
  };
  f32x4_t acc[8][4];
#pragma unroll
  for (int n = 0; n < 8; ++n)
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int steps = K / 32;
  issue(0);
  if (steps > 1) issue(1);
  const int off = r * 64 + ((g ^ (r >> 2)) & 3) * 16;
  int stage = 0;
  for (int kt = 0; kt < steps; ++kt) {
    // this step's pieces have landed when at most the next step's are in flight
    if (kt + 1 < steps)
      asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + 2 < steps) issue(stage == 0 ? 2 : stage - 1);
    const char* sa = lds + stage * kStageBytes + wm * 64 * 64 + off;
    // GLU: this wave's 64 gate columns, then its 64 up columns
    const char* sb = lds + stage * kStageBytes + BM * 64 + wn * (GLU ? 64 : 128) * 64 + off;
    U32x4 xa[4], wb[8];
#pragma unroll
    for (int m = 0; m < 4; ++m) xa[m] = *reinterpret_cast<const U32x4*>(sa + m * 1024);
#pragma unroll
    for (int n = 0; n < 8; ++n)
      wb[n] = *reinterpret_cast<const U32x4*>(sb + (GLU && n >= 4 ? n - 4 + 8 : n) * 1024);
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[n][m] = mfma16<F16>(wb[n], xa[m], acc[n][m]);
    stage = stage == 2 ? 0 : stage + 1;
  }
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int row = row0 + wm * 64 + m * 16 + r;
    if (row >= row_end) continue;
    if constexpr (GLU) {
      uint16_t* out = static_cast<uint16_t*>(a.h) + (int64_t)row * N;
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const int col = n0 + wn * 64 + n * 16 + 4 * g;
        if (col >= N) continue;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float z = acc[n][m][i];
          v[i] = z / (1.f + expf(-z)) * acc[n + 4][m][i];
        }
        *reinterpret_cast<uint2*>(out + col) = make_uint2(pack2<F16>(v[0], v[1]), pack2<F16>(v[2], v[3]));
      }
    } else {
      uint16_t* out = static_cast<uint16_t*>(a.y) + (int64_t)row * N;
      const float w = a.row_w[row];
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        const int col = n0 + wn * 128 + n * 16 + 4 * g;
        if (col >= N) continue;
        *reinterpret_cast<uint2*>(out + col) =
            make_uint2(pack2<F16>(acc[n][m][0] * w, acc[n][m][1] * w),
                       pack2<F16>(acc[n][m][2] * w, acc[n][m][3] * w));
      }
    }
  }
}

// out[token] = the sum of its experts' rows, 8 columns a thread.
template <bool F16>
__global__ __launch_bounds__(256) void moe_combine_kernel(MoeArgs a) {
  const int per = a.hidden / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
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

template <bool F16>
hipError_t launch(const MoeArgs& a, hipStream_t s) {
  const unsigned route = (unsigned)((a.M + kRouteTok - 1) / kRouteTok);
  moe_route_kernel<F16><<<dim3(route), kRouteTok, 0, s>>>(a);
  moe_group_kernel<<<dim3(route), kRouteTok, 0, s>>>(a);
  // most row tiles: every expert's last one may be partly filled
  const int64_t rows = a.M * a.topk;
  const int64_t tiles = rows / 128 + (rows < a.experts ? rows : a.experts);
  auto grid = [&](int64_t ntn) { return dim3((unsigned)((tiles * ntn + 7) / 8 * 8)); };
  moe_gemm_kernel<F16, true><<<grid((a.inter + 127) / 128), 256, 0, s>>>(a);
  moe_gemm_kernel<F16, false><<<grid((a.hidden + 255) / 256), 256, 0, s>>>(a);
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
