// The 16-bit product tile shared by the dense and the grouped layers: BM rows of x
// times BN rows of weights, both K-contiguous, on v_mfma 16x16x32 (fp32 sums).
#pragma once

#include "mhc_internal.hpp"

namespace mhc {

// BM x BN over WGM x WGN waves, STAGES stages of KB 32-column slices in LDS.
template <int BM_, int BN_, int WGM_, int WGN_, int STAGES_, int KB_ = 1>
struct GemmTile {
  static constexpr int KB = KB_;
  static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, STAGES = STAGES_;
  static constexpr int NW = WGM * WGN, THREADS = NW * 64;
  static constexpr int SLICE = (BM + BN) * 64;        // bytes of a slice, of a stage
  static constexpr int STAGE = KB * SLICE;
  static constexpr int LDS = STAGES * STAGE;
  static constexpr int PIECES = (BM + BN) / 16 / NW;  // 16-row pieces a wave loads a stage
  static constexpr int WM = BM / WGM, WN = BN / WGN;  // a wave's rows and columns
  static constexpr int MT = WM / 16, NT = WN / 16;
  static_assert((BM + BN) % (16 * NW) == 0, "whole pieces per wave");
};

// At most N vector-memory operations of this wave in flight, and no LDS one.
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(N) : "memory");
}

// acc[nt][mt] of this wave (wave % WGM: row part, wave / WGM: column part): lane
// (r, g) ends with columns 16 nt + 4 g .. + 3 of row 16 mt + r, since the product is
// formed as W x^T.
//   * K goes in steps of 32 KB through a ring of LDS stages, filled STAGES - 1 steps
//     ahead by direct-to-LDS loads.
//   * A slice's row is 64 bytes; its four 16-byte slots are permuted by the row's bits
//     2 and 3 (on the global side), so 16 rows hit all 64 banks.
//   * a_row(i) / b_row(i): byte pointer of x row i < BM / weight row i < BN.  col_tile
//     maps a wave's column tile to the stage's weight tile.
template <bool F16, typename G, typename ARow, typename BRow, typename ColTile>
__device__ __forceinline__ void gemm_tile(char* lds, int K, ARow a_row, BRow b_row, ColTile col_tile,
                                          f32x4_t (&acc)[G::NT][G::MT]) {
  constexpr int S = G::STAGES;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wm = wave % G::WGM;
  const char* src[G::PIECES];
#pragma unroll
  for (int i = 0; i < G::PIECES; ++i) {
    const int piece = wave * G::PIECES + i;
    const int prow = lane >> 2, slot = (lane & 3) ^ ((prow >> 2) & 3);
    src[i] = (piece < G::BM / 16 ? a_row(piece * 16 + prow) : b_row((piece - G::BM / 16) * 16 + prow)) + slot * 16;
  }
  auto issue = [&](int stage) {
#pragma unroll
    for (int i = 0; i < G::PIECES; ++i) {
#pragma unroll
      for (int q = 0; q < G::KB; ++q)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(src[i] + q * 64),
            (__attribute__((address_space(3))) void*)(lds + stage * G::STAGE + q * G::SLICE + (wave * G::PIECES + i) * 1024),
            16, 0, 0);
      src[i] += 64 * G::KB;
    }
  };
#pragma unroll
  for (int n = 0; n < G::NT; ++n)
#pragma unroll
    for (int m = 0; m < G::MT; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int steps = K / (32 * G::KB);
#pragma unroll
  for (int p = 0; p < S - 1; ++p)
    if (p < steps) issue(p);
  const int off = r * 64 + ((g ^ (r >> 2)) & 3) * 16;
  int stage = 0;
  for (int kt = 0; kt < steps; ++kt) {
    // S - 1 steps are in flight until the last ones: this step's pieces have landed
    // when only those of the S - 2 after it are left
    if (kt + S - 2 < steps) wait_loads<G::PIECES * G::KB * (S - 2)>();
    else wait_loads<0>();
    __builtin_amdgcn_s_barrier();  // every wave's pieces, and every wave is done with the stage issued next
    asm volatile("" ::: "memory");
    if (kt + S - 1 < steps) issue(stage == 0 ? S - 1 : stage - 1);
    const char* sa = lds + stage * G::STAGE + wm * G::WM * 64 + off;
    const char* sb = lds + stage * G::STAGE + G::BM * 64 + off;
    U32x4 xa[G::KB][G::MT], wb[G::KB][G::NT];
#pragma unroll
    for (int q = 0; q < G::KB; ++q) {
#pragma unroll
      for (int m = 0; m < G::MT; ++m) xa[q][m] = *reinterpret_cast<const U32x4*>(sa + q * G::SLICE + m * 1024);
#pragma unroll
      for (int n = 0; n < G::NT; ++n)
        wb[q][n] = *reinterpret_cast<const U32x4*>(sb + q * G::SLICE + col_tile(n) * 1024);
    }
#pragma unroll
    for (int q = 0; q < G::KB; ++q)
#pragma unroll
      for (int n = 0; n < G::NT; ++n)
#pragma unroll
        for (int m = 0; m < G::MT; ++m) acc[n][m] = mfma16<F16>(wb[q][n], xa[q][m], acc[n][m]);
    stage = stage == S - 1 ? 0 : stage + 1;
  }
}

// silu(z) * u in fp32.
__device__ __forceinline__ float silu_mul(float z, float u) { return z / (1.f + expf(-z)) * u; }

// Four neighbouring outputs, rounded.
template <bool F16>
__device__ __forceinline__ void store4(uint16_t* out, const f32x4_t& v) {
  *reinterpret_cast<uint2*>(out) = make_uint2(pack2<F16>(v[0], v[1]), pack2<F16>(v[2], v[3]));
}

}  // namespace mhc
