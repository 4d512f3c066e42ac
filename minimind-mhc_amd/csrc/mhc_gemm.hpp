// The 16-bit product tile shared by the dense and the grouped layers: BM rows of x
// times BN rows of weights, both K-contiguous, on v_mfma 16x16x32 (fp32 sums).
#pragma once

#include "mhc_internal.hpp"

namespace mhc {

// BM x BN over WGM x WGN waves, STAGES 64-column slices of both in LDS.
template <int BM_, int BN_, int WGM_, int WGN_, int STAGES_>
struct GemmTile {
  static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, STAGES = STAGES_;
  static constexpr int NW = WGM * WGN, THREADS = NW * 64;
  static constexpr int SLICE = (BM + BN) * 128;      // bytes of a slice
  static constexpr int LDS = STAGES * SLICE;
  static constexpr int PIECES = (BM + BN) / 8 / NW;  // 8-row pieces a wave loads a slice
  static constexpr int WM = BM / WGM, WN = BN / WGN;  // a wave's rows and columns
  static constexpr int MT = WM / 16, NT = WN / 16;
  // waves a SIMD: two workgroups a CU where their LDS allows
  static constexpr int WAVES = (LDS > 80 * 1024 ? 1 : 2) * NW / 4;
  static_assert((BM + BN) % (8 * NW) == 0, "whole pieces per wave");
  static_assert(STAGES >= 2, "a slice is read while the next one lands");
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
//   * K goes in slices of 64 (whole 128-byte lines of each row) through a ring of LDS
//     stages filled by direct-to-LDS loads.  A half slice's operands are read to
//     registers while the products of the half before run, so a stage is free again
//     (and refilled) before its last products begin.
//   * A slice's row is 128 bytes; its eight 16-byte slots are permuted by the row's
//     bits 1 to 3 (on the global side), so 16 rows hit all 64 banks.
//   * K % 64 == 32: the last slice is moved back by 32 columns (at K = 32 the columns
//     are taken twice) and only its upper half used.
//   * a_row(i) / b_row(i): byte offset of x row i < BM / weight row i < BN from a /
//     b_base(j), the base of the 8 rows around weight row j (uniform: it stays in
//     scalar registers).  col_tile maps a wave's column tile to the slice's weight tile.
template <bool F16, typename G, typename ARow, typename BBase, typename BRow, typename ColTile>
__device__ __forceinline__ void gemm_tile(char* lds, int K, const char* a, ARow a_row, BBase b_base, BRow b_row,
                                          ColTile col_tile, f32x4_t (&acc)[G::NT][G::MT]) {
  constexpr int S = G::STAGES;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wm = wave % G::WGM;
  const int slices = (K + 63) / 64;
  const bool odd = K % 64 != 0;
  const char* base[G::PIECES];
  uint32_t src[G::PIECES];
#pragma unroll
  for (int i = 0; i < G::PIECES; ++i) {
    const int row0 = (wave * G::PIECES + i) * 8, row = row0 + (lane >> 3);
    const int slot = ((lane & 7) ^ ((row >> 1) & 7)) & (K < 64 ? 3 : 7);
    base[i] = row0 < G::BM ? a : b_base(row0 - G::BM);
    src[i] = (row0 < G::BM ? a_row(row) : b_row(row - G::BM)) + slot * 16;
  }
  auto issue = [&](int stage, int slice) {
    const int64_t at = (int64_t)slice * 128 - (odd && K > 64 && slice == slices - 1 ? 64 : 0);  // uniform
#pragma unroll
    for (int i = 0; i < G::PIECES; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(base[i] + at + src[i]),
          (__attribute__((address_space(3))) void*)(lds + stage * G::SLICE + (wave * G::PIECES + i) * 1024), 16, 0, 0);
  };
  auto read = [&](int stage, int half, U32x4(&xa)[G::MT], U32x4(&wb)[G::NT]) {
    const int off = r * 128 + (((half * 4 + g) ^ (r >> 1)) & 7) * 16;
    const char* sa = lds + stage * G::SLICE + wm * G::WM * 128 + off;
    const char* sb = lds + stage * G::SLICE + G::BM * 128 + off;
#pragma unroll
    for (int m = 0; m < G::MT; ++m) xa[m] = *reinterpret_cast<const U32x4*>(sa + m * 2048);
#pragma unroll
    for (int n = 0; n < G::NT; ++n) wb[n] = *reinterpret_cast<const U32x4*>(sb + col_tile(n) * 2048);
  };
#pragma unroll
  for (int n = 0; n < G::NT; ++n)
#pragma unroll
    for (int m = 0; m < G::MT; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int p = 0; p < S; ++p)
    if (p < slices) issue(p, p);
  if (slices >= S) wait_loads<G::PIECES * (S - 1)>();
  else wait_loads<0>();
  __builtin_amdgcn_s_barrier();  // every wave's pieces of the first slice
  asm volatile("" ::: "memory");
  U32x4 xa[2][G::MT], wb[2][G::NT];
  auto products = [&](int set) {
#pragma unroll
    for (int n = 0; n < G::NT; ++n)
#pragma unroll
      for (int m = 0; m < G::MT; ++m) acc[n][m] = mfma16<F16>(wb[set][n], xa[set][m], acc[n][m]);
  };
  read(0, 0, xa[0], wb[0]);
  int stage = 0;
  for (int ks = 0; ks < slices; ++ks) {
    // lgkmcnt(0) in a form the compiler counts with: at the products it would otherwise
    // wait for the next half's operands too
    __builtin_amdgcn_s_waitcnt(0xc07f);
    read(stage, 1, xa[1], wb[1]);
    if (!odd || ks + 1 < slices) products(0);  // uniform
    __builtin_amdgcn_s_waitcnt(0xc07f);
    if (ks + 1 < slices) {  // uniform
      // slices up to ks + S - 1 are issued: the next one has landed when only the
      // S - 2 after it are in flight
      if (S > 2 && ks + S <= slices) wait_loads<G::PIECES * (S - 2)>();
      else wait_loads<0>();
      __builtin_amdgcn_s_barrier();  // every wave's pieces, and every wave has read slice ks
      asm volatile("" ::: "memory");
      if (ks + S < slices) issue(stage, ks + S);
      stage = stage == S - 1 ? 0 : stage + 1;
      read(stage, 0, xa[0], wb[0]);
    }
    products(1);
  }
}

// silu(z) * u in fp32, on the hardware's exponential and reciprocal (1 ulp each): expf
// and the division are some 25 instructions more, 10 of the 62 us of gate and up at
// 8192 rows, 768 x 2048.
__device__ __forceinline__ float silu_mul(float z, float u) {
  constexpr float kLog2e = 1.44269504088896340736f;
  return z * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-kLog2e * z)) * u;
}

// Which tile a product of that many rows and columns takes: BM x BN of GemmTile.  The
// lines come from these sizes; the counts 192 and (linear layers) 448 are tiles on the
// 256 CUs they were measured on.
//   256 x 256: one workgroup a CU, so only for rounds of the chip that are nearly full.
//     8192 x 6400, K = 768 (800 tiles, 3.1 of 4 rounds): 97 us, 128 x 192 tiles 107;
//     gate and up of 8192 x 2048 (512 tiles): 52.1, 128 x 128 tiles 61.0; of 8 routed
//     experts (16384 rows x 1024, 544 tiles, 2.1 of 3 rounds): 72.4 and 70.8; 8192 x 1536
//     (192 tiles, under one round): 26.0 against 22.2 for 128 x 192.
//   128 x 192: where a tile a CU is left and no column is padding that 128 would not
//     have.  8192 x 1536: 22.2 us, 128 x 128 tiles 24.7; 8192 x 768 (256 tiles) 14.6
//     and 15.6; 2048 x 1536 (128 tiles) 12.1 and 10.3.  Gate and up gain little from it
//     (59.0 and 61.0).
//   128 x 64 up to one 128 x 128 tile a CU: 512 x 6400 (200) 11.9 and 12.6 us, gate and
//     up of 1024 x 2048 (256) 12.0 and 13.3; of 2048 x 2048 (512) 22.6 and 17.4.
//   64 x 64 while 128 x 64 ones would be fewer than 192: 1024 x 1536 (192) 7.5 us
//     either way, 512 x 6400 (400) 17.9 and 11.9.
enum class Tile { k16x16, k64x64, k128x64, k128x128, k128x192, k256x256 };  // 16 x 16: linear layers only
template <typename Rows, typename Cols>
Tile pick_tile(Rows rows, Cols cols, bool glu) {
  const int64_t cus = device_cus();
  const int64_t t256 = rows(256) * cols(256), full = (t256 + cus - 1) / cus * cus;
  if (t256 > cus && t256 * 8 >= full * (glu ? 7 : 6)) return Tile::k256x256;
  if (!glu && rows(128) * cols(192) >= cus && cols(192) * 3 <= cols(128) * 2) return Tile::k128x192;
  if (rows(128) * cols(128) > cus) return Tile::k128x128;
  return rows(128) * cols(64) < 192 ? Tile::k64x64 : Tile::k128x64;
}

// Four neighbouring outputs, rounded.
template <bool F16>
__device__ __forceinline__ void store4(uint16_t* out, const f32x4_t& v) {
  *reinterpret_cast<uint2*>(out) = make_uint2(pack2<F16>(v[0], v[1]), pack2<F16>(v[2], v[3]));
}

// A wave's columns (COLS of them: 16 nt + 4 g .. of value(nt, mt)) of its G::WM rows, 16
// rows at a time through LDS, so that a row leaves in whole 16-byte pieces next to each
// other.  Stored from the accumulators, a launch writes 32-byte segments of 16 rows.
// out: the wave's first row and column; rows, cols: how many there are.
template <bool F16, typename G, int COLS, typename Value>
__device__ __forceinline__ void store_tile(char* lds, uint16_t* out, int64_t stride, int64_t rows, int cols, Value value) {
  constexpr int ST = COLS + 8;  // 16 rows on distinct banks
  static_assert(G::NW * 16 * ST * 2 <= G::LDS, "a row block of every wave");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  uint16_t* buf = reinterpret_cast<uint16_t*>(lds) + wave * 16 * ST;
  __syncthreads();  // every wave has read its last operands
#pragma unroll
  for (int m = 0; m < G::MT; ++m) {
#pragma unroll
    for (int n = 0; n < COLS / 16; ++n) store4<F16>(buf + r * ST + n * 16 + 4 * g, value(n, m));
    asm volatile("" ::: "memory");  // the wave's LDS operations run in order
#pragma unroll
    for (int p = 0; p < (2 * COLS + 63) / 64; ++p) {
      const int piece = p * 64 + lane, row = piece / (COLS / 8), col = piece % (COLS / 8) * 8;
      if (row >= 16) continue;
      const U32x4 v = *reinterpret_cast<const U32x4*>(buf + row * ST + col);
      if (m * 16 + row >= rows) continue;
      uint16_t* o = out + (m * 16 + row) * stride + col;
      if (stride % 8 == 0) {
        if (col < cols) *reinterpret_cast<U32x4*>(o) = v;
      } else {  // rows 8-byte aligned, a last piece of four
        if (col < cols) *reinterpret_cast<uint2*>(o) = make_uint2(v.v[0], v.v[1]);
        if (col + 4 < cols) *reinterpret_cast<uint2*>(o + 4) = make_uint2(v.v[2], v.v[3]);
      }
    }
    asm volatile("" ::: "memory");
  }
}

}  // namespace mhc
