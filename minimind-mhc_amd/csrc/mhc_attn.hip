// Attention of the model's sublayer for inference (model/model_minimind.py:161-256):
// per-head RMSNorm and rotary embedding of q and k, causal prefill attention, and
// the decode step over a KV cache.  16-bit tensors (bf16 or fp16), fp32 sums,
// head_dim in {64, 96, 128}, grouped query heads without expanded copies of k, v.
#include "mhc_internal.hpp"

namespace mhc {
namespace {

typedef short s16x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ U32x4 ld16(const void* p) { return *static_cast<const U32x4*>(p); }

// Eight consecutive elements of one head: RMSNorm over the head (inv, gain w)
// and the rotary embedding, whose partner elements (half a head away) are xp
// with gain wp.  fp32 throughout, one rounding at the end.
template <bool F16>
__device__ __forceinline__ U32x4 norm_rope8(const U32x4& x, const U32x4& xp, const U32x4& w,
                                            const U32x4& wp, const U32x4& cs, const U32x4& sn,
                                            float inv, bool upper) {
  U32x4 o;
  const float sgn = upper ? 1.f : -1.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float a0 = elem_lo<F16>(x.v[j]) * inv * elem_lo<F16>(w.v[j]);
    const float a1 = elem_hi<F16>(x.v[j]) * inv * elem_hi<F16>(w.v[j]);
    const float b0 = elem_lo<F16>(xp.v[j]) * inv * elem_lo<F16>(wp.v[j]);
    const float b1 = elem_hi<F16>(xp.v[j]) * inv * elem_hi<F16>(wp.v[j]);
    o.v[j] = pack2<F16>(a0 * elem_lo<F16>(cs.v[j]) + sgn * b0 * elem_lo<F16>(sn.v[j]),
                        a1 * elem_hi<F16>(cs.v[j]) + sgn * b1 * elem_hi<F16>(sn.v[j]));
  }
  return o;
}

template <bool F16>
__device__ __forceinline__ float sumsq8(const U32x4& x) {
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float a = elem_lo<F16>(x.v[j]);
    const float b = elem_hi<F16>(x.v[j]);
    s += a * a + b * b;
  }
  return s;
}

// One head's row as an MFMA operand: lane group g's 16 bytes of each 32-column
// block, normed and rotated (four lanes, 16 apart, share the row).
template <bool F16, int HD>
__device__ __forceinline__ void norm_rope_operand(const uint16_t* x, const void* gain, const void* cos,
                                                  const void* sin, float eps, int g,
                                                  U32x4 (&o)[HD / 32]) {
  const uint16_t* w = static_cast<const uint16_t*>(gain);
  const uint16_t* cs = static_cast<const uint16_t*>(cos);
  const uint16_t* sn = static_cast<const uint16_t*>(sin);
  U32x4 xv[HD / 32], xp[HD / 32];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < HD / 32; ++c) {
    const int d = 32 * c + 8 * g;
    xv[c] = ld16(x + d);
    xp[c] = ld16(x + (d < HD / 2 ? d + HD / 2 : d - HD / 2));
    ss += sumsq8<F16>(xv[c]);
  }
  ss += xor_lane16(ss);
  ss += xor_lane32(ss);
  const float inv = 1.0f / sqrtf(ss / HD + eps);
#pragma unroll
  for (int c = 0; c < HD / 32; ++c) {
    const int d = 32 * c + 8 * g;
    const int p = d < HD / 2 ? d + HD / 2 : d - HD / 2;
    o[c] = norm_rope8<F16>(xv[c], xp[c], ld16(w + d), ld16(w + p), ld16(cs + d), ld16(sn + d), inv,
                           d >= HD / 2);
  }
}

// ------------------------------------------------------- norm + rotary of k, prefill
// G lanes per (token, kv head): lane j < HD / 16 holds elements 8j.. and their
// rotary partners HD / 2 + 8j.., so one load of each gives both halves.  k is
// read by many workgroups of the attention kernel and is the cache's content, so
// it is formed once, here; q is formed where it is used.
template <bool F16, int HD>
__global__ __launch_bounds__(256) void k_norm_rope_kernel(KRopeArgs a) {
  constexpr int G = HD <= 64 ? 4 : 8;
  constexpr int L = HD / 16;  // lanes that hold data
  const int lane = threadIdx.x & (G - 1);
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / G;
  const bool live = row < a.M * a.kv_heads && lane < L;
  const int64_t off = live ? row * HD + 8 * lane : 0;
  const uint16_t* in = static_cast<const uint16_t*>(a.k) + off;
  const int64_t po = live ? (row / a.kv_heads % a.T) * HD + 8 * lane : 0;
  const uint16_t* gain = static_cast<const uint16_t*>(a.gain) + (live ? 8 * lane : 0);
  const uint16_t* cs = static_cast<const uint16_t*>(a.cos) + po;
  const uint16_t* sn = static_cast<const uint16_t*>(a.sin) + po;
  const U32x4 x0 = ld16(in), x1 = ld16(in + HD / 2);
  const U32x4 w0 = ld16(gain), w1 = ld16(gain + HD / 2);
  const U32x4 c0 = ld16(cs), c1 = ld16(cs + HD / 2);
  const U32x4 s0 = ld16(sn), s1 = ld16(sn + HD / 2);
  const float ss = live ? sumsq8<F16>(x0) + sumsq8<F16>(x1) : 0.f;
  const float inv = 1.0f / sqrtf(row_reduce<G, OpAdd>(ss) / HD + a.eps);
  if (!live) return;
  uint16_t* out = static_cast<uint16_t*>(a.out) + off;
  *reinterpret_cast<U32x4*>(out) = norm_rope8<F16>(x0, x1, w0, w1, c0, s0, inv, false);
  *reinterpret_cast<U32x4*>(out + HD / 2) = norm_rope8<F16>(x1, x0, w1, w0, c1, s1, inv, true);
}

// ------------------------------------------------------------------ decode step
// One query token per sequence over S cached positions and the new one.  The
// step is bound by the cache's bytes (and, when a grown cache is returned, by
// writing them back), so each K and V row is read once, serves all REP query heads
// of its kv head, and is stored to the grown cache on the way.
//   * q, and in the range that ends with the new position k, are normed
//     and rotated here: the raw projections are the inputs.
//   * Scores on v_mfma 16x16x32: A rows 4g + i all hold query head i, so lane
//     (r, g) gets its REP scores of position r without a shuffle; B is the K row
//     straight from memory (16 bytes a lane).
//   * Each lane keeps its own running maximum, sum and output columns (8 per
//     32-column chunk) of the positions r mod 16 it saw: no cross-lane step in
//     the loop.  The 16 lanes merge at the end, the ranges in a second launch.
//   * A workgroup takes four waves' worth of rows (a tile): 4, 2 or 1 kv heads of 16,
//     32 or 64 positions, loaded (non-temporal: read once) and stored as their bytes
//     run, whole lines across the workgroup, and regrouped through LDS.  64
//     sequences, 4 kv heads of 96, S = 2048, grown cache, 403 MB: 72.6 us, 5.55 TB/s
//     (a 1 GiB torch copy runs at 5.07); the same over eight caches in turn (1.6 GB)
//     and with eight grown ones kept, 85 between the model's other launches.  Each
//     wave loading and storing its own head's rows 80 us (cached loads 97,
//     non-temporal stores 101), in the operand layout (16 rows x 64 bytes) 94; here
//     non-temporal stores 85.  The torch ops (cat, two expanded copies, SDPA, norms
//     and rotary) took 670 us.
//   * The maximum is raised (and the sums rescaled) only when some score exceeds
//     it by more than 2^8 in the exponent; fp32 sums lose nothing by that.
constexpr float kLazyMax = 8.f;
constexpr float kNegBig = -1e30f;
constexpr float kLog2e = 1.44269504088896340736f;

__device__ __forceinline__ float exp2_f(float x) { return __builtin_amdgcn_exp2f(x); }

template <int CTRL>
__device__ __forceinline__ float dpp_max(float v) { return fmaxf(v, dpp_f<CTRL>(v)); }
__device__ __forceinline__ float row16_max(float v) {
  return dpp_max<kDppRowMirror>(dpp_max<kDppHalfMirror>(dpp_max<kDppXor2>(dpp_max<kDppXor1>(v))));
}

template <bool F16, int HD, int REP>
__global__ __launch_bounds__(256) void attn_decode_kernel(AttnDecodeArgs a) {
  constexpr int NC = HD / 32;
  constexpr int LST = HD + 8;  // 16 rows on distinct banks
  __shared__ __align__(16) uint16_t kl[2][4 * 16 * LST];
  __shared__ __align__(16) uint16_t vl[2][4 * 16 * LST];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int r = lane & 15, g = lane >> 4;
  // the workgroup's kv heads (1, 2 or 4), its waves' rows: wave = sub * G + head
  const int G = a.group, rows = 64 / G;  // positions a tile
  const int hg = blockIdx.x % (a.kv_heads / G);
  const int64_t bs = blockIdx.x / (a.kv_heads / G);
  const int split = (int)(bs % a.splits);
  const int64_t b = bs / a.splits;
  const int kvh = hg * G + wave % G;
  const int sub = wave / G * 16;
  const int t0 = split * a.tiles_per_split;
  const int t1 = min(t0 + a.tiles_per_split, (a.S + rows - 1) / rows);
  const bool has_new = split == a.splits - 1 && wave < G;

  // A tile is loaded and stored as its bytes run in the cache (whole lines across the
  // workgroup: the heads of a position are neighbours), piece p * 256 + tid, and
  // reaches the waves' operand layout through LDS.
  const uint16_t* kb = static_cast<const uint16_t*>(a.k_past) + b * a.ks_b + hg * G * a.ks_h;
  const uint16_t* vb = static_cast<const uint16_t*>(a.v_past) + b * a.vs_b + hg * G * a.vs_h;
  const int64_t orow = (int64_t)a.kv_heads * HD;  // grown cache: contiguous [B, S + 1, kv, HD]
  uint16_t* ko = static_cast<uint16_t*>(a.k_out);
  uint16_t* vo = static_cast<uint16_t*>(a.v_out);
  const int64_t obase = b * (a.S + 1) * orow;
  const uint16_t* kp[NC];
  const uint16_t* vp[NC];
  int prow[NC], ocol[NC], lpos[NC];
#pragma unroll
  for (int p = 0; p < NC; ++p) {
    const int piece = p * 256 + tid, per = G * (HD / 8);
    prow[p] = piece / per;
    const int in_row = piece - prow[p] * per;
    const int head = in_row / (HD / 8), col = in_row % (HD / 8) * 8;
    kp[p] = kb + head * a.ks_h + col;
    vp[p] = vb + head * a.vs_h + col;
    ocol[p] = (hg * G + head) * HD + col;
    lpos[p] = ((prow[p] / 16 * G + head) * 16 + prow[p] % 16) * LST + col;
  }
  U32x4 kn[NC], vn[NC];  // next tile
  auto load = [&](int t) {
#pragma unroll
    for (int p = 0; p < NC; ++p) kn[p] = ld16_nt(kp[p] + (int64_t)min(t * rows + prow[p], a.S - 1) * a.ks_s);
#pragma unroll
    for (int p = 0; p < NC; ++p) vn[p] = ld16_nt(vp[p] + (int64_t)min(t * rows + prow[p], a.S - 1) * a.vs_s);
  };
  if (t0 < t1) load(t0);

  // A operand: q head (r & 3) of this kv head, normed and rotated.
  U32x4 qa[NC];
  const int qh = kvh * REP + min(r & 3, REP - 1);
  norm_rope_operand<F16, HD>(static_cast<const uint16_t*>(a.q) + (b * a.heads + qh) * HD, a.q_gain, a.cos,
                             a.sin, a.q_eps, g, qa);

  const float scale = kLog2e / sqrtf((float)HD);
  float m[REP], l[REP], acc[REP][NC][8];
#pragma unroll
  for (int i = 0; i < REP; ++i) {
    m[i] = kNegBig;
    l[i] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[i][c][e] = 0.f;
  }
  auto step = [&](const U32x4(&kc)[NC], const U32x4(&vc)[NC], bool ok) {
    f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NC; ++c) s = mfma16<F16>(qa[c], kc[c], s);
    float z[REP];
    bool raise = false;
#pragma unroll
    for (int i = 0; i < REP; ++i) {
      z[i] = ok ? s[i] * scale : -__builtin_inff();
      raise = raise || z[i] > m[i] + kLazyMax;
    }
    if (__any(raise)) {
#pragma unroll
      for (int i = 0; i < REP; ++i) {
        const float mn = fmaxf(m[i], z[i]);
        const float f = exp2_f(m[i] - mn);
        m[i] = mn;
        l[i] *= f;
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[i][c][e] *= f;
      }
    }
    float p[REP];
#pragma unroll
    for (int i = 0; i < REP; ++i) {
      p[i] = exp2_f(z[i] - m[i]);
      l[i] += p[i];
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float v0 = elem_lo<F16>(vc[c].v[j]);
        const float v1 = elem_hi<F16>(vc[c].v[j]);
#pragma unroll
        for (int i = 0; i < REP; ++i) {
          acc[i][c][2 * j] += p[i] * v0;
          acc[i][c][2 * j + 1] += p[i] * v1;
        }
      }
  };
  for (int t = t0; t < t1; ++t) {  // uniform: two buffers, so one barrier a tile
    const int buf = (t - t0) & 1;
#pragma unroll
    for (int p = 0; p < NC; ++p) {
      *reinterpret_cast<U32x4*>(&kl[buf][lpos[p]]) = kn[p];
      *reinterpret_cast<U32x4*>(&vl[buf][lpos[p]]) = vn[p];
      const int row = t * rows + prow[p];
      if (ko && row < a.S) {
        *reinterpret_cast<U32x4*>(ko + obase + row * orow + ocol[p]) = kn[p];
        *reinterpret_cast<U32x4*>(vo + obase + row * orow + ocol[p]) = vn[p];
      }
    }
    // rows that are not there: 0 x infinity would be NaN (here and not as a select on vc: 176
    // registers instead of 160 at head_dim 96 cost the third wave a SIMD, 5 us a launch)
    if ((t + 1) * rows > a.S)
#pragma unroll
      for (int p = 0; p < NC; ++p)
        if (t * rows + prow[p] >= a.S) *reinterpret_cast<U32x4*>(&vl[buf][lpos[p]]) = U32x4{};
    if (t + 1 < t1) load(t + 1);
    __syncthreads();
    U32x4 kc[NC], vc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      kc[c] = *reinterpret_cast<const U32x4*>(&kl[buf][(wave * 16 + r) * LST + 32 * c + 8 * g]);
      vc[c] = *reinterpret_cast<const U32x4*>(&vl[buf][(wave * 16 + r) * LST + 32 * c + 8 * g]);
    }
    step(kc, vc, t * rows + sub + r < a.S);
  }
  if (has_new) {  // the new position: one row, in the lanes with r == 0
    U32x4 kc[NC], vc[NC];
    norm_rope_operand<F16, HD>(static_cast<const uint16_t*>(a.k) + (b * a.kv_heads + kvh) * HD, a.k_gain,
                               a.cos, a.sin, a.k_eps, g, kc);
    const uint16_t* vp = static_cast<const uint16_t*>(a.v) + (b * a.kv_heads + kvh) * HD + 8 * g;
#pragma unroll
    for (int c = 0; c < NC; ++c) vc[c] = ld16(vp + 32 * c);
    if (ko && r == 0) {
      const int64_t o = obase + a.S * orow + kvh * HD + 8 * g;
#pragma unroll
      for (int c = 0; c < NC; ++c) *reinterpret_cast<U32x4*>(ko + o + 32 * c) = kc[c];
#pragma unroll
      for (int c = 0; c < NC; ++c) *reinterpret_cast<U32x4*>(vo + o + 32 * c) = vc[c];
    }
    const uint32_t keep = r == 0 ? ~0u : 0u;  // the other lanes hold no position
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) vc[c].v[j] &= keep;
    step(kc, vc, r == 0);
  }
  // merge the 16 positions of the row
#pragma unroll
  for (int i = 0; i < REP; ++i) {
    const float mx = row16_max(m[i]);
    const float f = exp2_f(m[i] - mx);
    const float ls = row16_sum(l[i] * f);
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[i][c][e] = row16_sum(acc[i][c][e] * f);
    if (r != 0) continue;
    const int64_t row = b * a.heads + kvh * REP + i;
    if (a.parts == 1) {
      uint16_t* o = static_cast<uint16_t*>(a.out) + row * HD + 8 * g;
      const float inv = 1.f / ls;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        U32x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w.v[j] = pack2<F16>(acc[i][c][2 * j] * inv, acc[i][c][2 * j + 1] * inv);
        *reinterpret_cast<U32x4*>(o + 32 * c) = w;
      }
    } else {
      const int64_t part = row * a.parts + split * (4 / G) + wave / G;
      float* o = a.work + part * HD + 8 * g;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int e = 0; e < 8; e += 4)
          *reinterpret_cast<f32x4_t*>(o + 32 * c + e) =
              f32x4_t{acc[i][c][e], acc[i][c][e + 1], acc[i][c][e + 2], acc[i][c][e + 3]};
      if (g == 0) {
        float* ml = a.work + a.B * a.heads * a.parts * HD + 2 * part;
        ml[0] = mx;
        ml[1] = ls;
      }
    }
  }
}

// Sums the ranges of one (sequence, head): HD / 4 lanes hold four columns each,
// the wave's other lane groups every second (fourth) range.
template <bool F16, int HD>
__global__ __launch_bounds__(64) void attn_merge_kernel(AttnDecodeArgs a) {
  constexpr int LPR = HD <= 64 ? 16 : 32;  // lanes a range takes (HD / 4 of them hold data)
  constexpr int PAR = 64 / LPR;
  const int lane = threadIdx.x & (LPR - 1);
  const int sub = threadIdx.x / LPR;
  const int64_t row = blockIdx.x;
  const bool live = lane < HD / 4;
  const float* part = a.work + row * a.parts * HD + (live ? 4 * lane : 0);
  const float* ml = a.work + a.B * a.heads * a.parts * HD + 2 * row * a.parts;
  float mx = kNegBig;
  for (int s = threadIdx.x; s < a.parts; s += 64) mx = fmaxf(mx, ml[2 * s]);
  mx = row16_max(mx);
  mx = fmaxf(mx, xor_lane16(mx));
  mx = fmaxf(mx, xor_lane32(mx));
  float l = 0.f;
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = sub; s < a.parts; s += PAR) {
    const float f = exp2_f(ml[2 * s] - mx);
    l += f * ml[2 * s + 1];
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(part + (int64_t)s * HD);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] += f * v[e];
  }
  if constexpr (PAR == 4) {
    l += xor_lane16(l);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] += xor_lane16(o[e]);
  }
  l += xor_lane32(l);
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] += xor_lane32(o[e]);
  if (sub != 0 || !live) return;
  const float inv = 1.f / l;
  uint32_t* out = reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(a.out) + row * HD + 4 * lane);
  out[0] = pack2<F16>(o[0] * inv, o[1] * inv);
  out[1] = pack2<F16>(o[2] * inv, o[3] * inv);
}

// --------------------------------------------------------------- causal prefill
// One 4-wave workgroup per (sequence, 128 query rows of one kv head): HP query
// heads of it (two where the group has an even count) times 128 / HP positions,
// 32 rows a wave.  K and V tiles of 64 positions go through LDS (double
// buffered, the next tile's loads in registers meanwhile).
//   * S^T = K Q^T and O^T = V^T P^T on v_mfma 16x16x32, so a lane holds scores
//     and outputs of one query row: the softmax needs no LDS, the rescaling no
//     shuffle, and S^T's registers, rounded, are P^T's operand as they are (the
//     contraction runs over positions 16 (j / 4) + 4 g + j % 4 of each 32).
//   * V^T is read from the row-major tile by the transposing LDS load
//     (ds_read_b64_tr_b16: a 16-lane group gets columns of 4 rows x 16).
//   * Row strides of HD + 8 (K) and HD + 16 (V) elements spread the 16 rows of a read
//     over all 64 banks; with the tile's stores, 31% of the LDS cycles are conflicts.
//   * Tiles above the diagonal are skipped; the workgroups with the longest rows
//     start first.  The maximum is raised lazily as in the decode step.
//   * Each wave norms and rotates its own q rows (a pass over q less).
//   * Only the tiles on the diagonal compare positions (a uniform branch: as selects on
//     every score 37 us, a fifth of the loop's VALU work).
// 8 sequences of 1024, 8 query / 4 kv heads of 96: 34 us with the norms and rotary of
// q (matrix cores busy 22% of the time, the VALU 48%), and 5 us for k; torch took 92 us
// for SDPA (with expanded k, v) and 200 us for the norms, rotary and expanded copies.
template <bool F16, int HD, int HP>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(AttnPrefillArgs a) {
  constexpr int NC = HD / 32, ND = HD / 16, KT = 64;
  constexpr int PW = 128 / HP;
  constexpr int KST = HD + 8, VST = HD + 16;
  constexpr int PPT = KT * (HD / 8) / 256;  // 16-byte pieces a thread moves per tile
  __shared__ __align__(16) uint16_t ks[2][KT * KST];
  __shared__ __align__(16) uint16_t vs[2][KT * VST];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r = lane & 15, g = lane >> 4;
  const int groups = a.B * (a.heads / HP);
  // every second round of one workgroup per CU runs the other way, so a CU's
  // workgroups add up to about the same number of tiles
  const int round = blockIdx.x / a.cus, at = blockIdx.x % a.cus;
  const int idx = (round & 1) ? round * a.cus + min(a.cus, (int)gridDim.x - round * a.cus) - 1 - at : (int)blockIdx.x;
  const int qt = a.qtiles - 1 - idx / groups;
  const int grp = idx % groups;
  const int b = grp / (a.heads / HP);
  const int h = (grp % (a.heads / HP)) * HP + (HP == 2 ? wave >> 1 : 0);
  const int kvh = ((grp % (a.heads / HP)) * HP) / (a.heads / a.kv_heads);
  const int q0 = qt * PW;
  const int pb = q0 + (HP == 2 ? (wave & 1) * 32 : wave * 32);
  const int T = a.T;

  const uint16_t* kg = static_cast<const uint16_t*>(a.k) + ((int64_t)b * T * a.kv_heads + kvh) * HD;
  const uint16_t* vg = static_cast<const uint16_t*>(a.v) + ((int64_t)b * T * a.kv_heads + kvh) * HD;
  const int64_t rs = (int64_t)a.kv_heads * HD;

  U32x4 kr[PPT], vr[PPT];
  auto load = [&](int s0) {
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      const int piece = p * 256 + tid;
      const int row = min(s0 + piece / (HD / 8), T - 1);
      const int col = (piece % (HD / 8)) * 8;
      kr[p] = ld16(kg + row * rs + col);
      vr[p] = ld16(vg + row * rs + col);
    }
  };
  auto stash = [&](int buf, int s0) {
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      const int piece = p * 256 + tid;
      const int row = piece / (HD / 8);
      const int col = (piece % (HD / 8)) * 8;
      *reinterpret_cast<U32x4*>(&ks[buf][row * KST + col]) = kr[p];
      *reinterpret_cast<U32x4*>(&vs[buf][row * VST + col]) = vr[p];
    }
    // rows that are not there: 0 x infinity would be NaN (stores in a uniform branch: as
    // selects on every tile's registers 1.7% of the layer)
    if (s0 + KT > T)
#pragma unroll
      for (int p = 0; p < PPT; ++p) {
        const int piece = p * 256 + tid;
        const int row = piece / (HD / 8);
        if (s0 + row >= T) *reinterpret_cast<U32x4*>(&vs[buf][row * VST + (piece % (HD / 8)) * 8]) = U32x4{};
      }
  };
  load(0);
  U32x4 qb[2][NC];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int pos = min(pb + u * 16 + r, T - 1);
    norm_rope_operand<F16, HD>(static_cast<const uint16_t*>(a.q) + (((int64_t)b * T + pos) * a.heads + h) * HD,
                               a.q_gain, static_cast<const uint16_t*>(a.cos) + (int64_t)pos * HD,
                               static_cast<const uint16_t*>(a.sin) + (int64_t)pos * HD, a.q_eps, g, qb[u]);
  }
  const float scale = kLog2e / sqrtf((float)HD);
  float m[2] = {kNegBig, kNegBig}, l[2] = {0.f, 0.f};
  f32x4_t o[2][ND];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int d = 0; d < ND; ++d) o[u][d] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int last = min(q0 + PW, T);  // positions any row of the workgroup sees
  const int nt = (last + KT - 1) / KT;
  for (int t = 0; t < nt; ++t) {
    const int buf = t & 1;
    stash(buf, t * KT);
    __syncthreads();
    if (t + 1 < nt) load((t + 1) * KT);
    const int s0 = t * KT;
    if (s0 > pb + 31) continue;  // wholly above this wave's diagonal
    f32x4_t s[2][4];
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      s[0][st] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      s[1][st] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const U32x4 ka = *reinterpret_cast<const U32x4*>(&ks[buf][(st * 16 + r) * KST + 32 * c + 8 * g]);
        s[0][st] = mfma16<F16>(ka, qb[0][c], s[0][st]);
        s[1][st] = mfma16<F16>(ka, qb[1][c], s[1][st]);
      }
    }
    if (s0 + KT - 1 > pb) {  // uniform: only the tiles on the diagonal are compared
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (s0 + st * 16 + 4 * g + i > pb + u * 16 + r) s[u][st][i] = -__builtin_inff();
    }
    U32x4 pf[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float mx = kNegBig;
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[u][st][i]);
      mx *= scale;
      if (__any(!(mx <= m[u] + kLazyMax))) {
        mx = fmaxf(mx, xor_lane16(mx));
        mx = fmaxf(mx, xor_lane32(mx));
        mx = fmaxf(mx, m[u]);
        const float f = exp2_f(m[u] - mx);
        m[u] = mx;
        l[u] *= f;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[u][d][i] *= f;
      }
      float sum = 0.f;
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[i] = exp2_f(fmaf(s[u][st][i], scale, -m[u]));
          sum += p[i];
        }
        pf[u][st >> 1].v[2 * (st & 1)] = pack2<F16>(p[0], p[1]);
        pf[u][st >> 1].v[2 * (st & 1) + 1] = pack2<F16>(p[2], p[3]);
      }
      l[u] += sum;
    }
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        U32x4 va;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const uint16_t* src = &vs[buf][(hh * 32 + q * 16 + 4 * g + (r >> 2)) * VST + 16 * d + 4 * (r & 3)];
          const s16x4_t w = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) s16x4_t*)const_cast<uint16_t*>(src));
          typedef uint32_t u32x2_v __attribute__((ext_vector_type(2)));
          const u32x2_v w2 = __builtin_bit_cast(u32x2_v, w);
          va.v[2 * q] = w2.x;
          va.v[2 * q + 1] = w2.y;
        }
        o[0][d] = mfma16<F16>(va, pf[0][hh], o[0][d]);
        o[1][d] = mfma16<F16>(va, pf[1][hh], o[1][d]);
      }
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    float ls = l[u];
    ls += xor_lane16(ls);
    ls += xor_lane32(ls);
    const float inv = 1.f / ls;
    const int pos = pb + u * 16 + r;
    if (pos >= T) continue;
    uint16_t* out = static_cast<uint16_t*>(a.out) + (((int64_t)b * T + pos) * a.heads + h) * HD + 4 * g;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      uint2 w;
      w.x = pack2<F16>(o[u][d][0] * inv, o[u][d][1] * inv);
      w.y = pack2<F16>(o[u][d][2] * inv, o[u][d][3] * inv);
      *reinterpret_cast<uint2*>(out + 16 * d) = w;
    }
  }
}

template <bool F16, int HD>
hipError_t rope_hd(const KRopeArgs& a, hipStream_t s) {
  constexpr int G = HD <= 64 ? 4 : 8;
  const int64_t blocks = (a.M * a.kv_heads * G + 255) / 256;
  k_norm_rope_kernel<F16, HD><<<dim3((unsigned)blocks), 256, 0, s>>>(a);
  return hipGetLastError();
}

template <bool F16, int HD>
hipError_t decode_hd(const AttnDecodeArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(a.B * a.splits * (a.kv_heads / a.group)));
  switch (a.heads / a.kv_heads) {
    case 1: attn_decode_kernel<F16, HD, 1><<<grid, 256, 0, s>>>(a); break;
    case 2: attn_decode_kernel<F16, HD, 2><<<grid, 256, 0, s>>>(a); break;
    case 3: attn_decode_kernel<F16, HD, 3><<<grid, 256, 0, s>>>(a); break;
    case 4: attn_decode_kernel<F16, HD, 4><<<grid, 256, 0, s>>>(a); break;
    default: return hipErrorInvalidValue;
  }
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  if (a.parts > 1) attn_merge_kernel<F16, HD><<<dim3((unsigned)(a.B * a.heads)), 64, 0, s>>>(a);
  return hipGetLastError();
}

template <bool F16, int HD>
hipError_t prefill_hd(AttnPrefillArgs a, hipStream_t s) {
  a.cus = device_cus();
  if ((a.heads / a.kv_heads) % 2 == 0) {
    a.qtiles = (a.T + 63) / 64;
    attn_prefill_kernel<F16, HD, 2><<<dim3((unsigned)(a.qtiles * a.B * (a.heads / 2))), 256, 0, s>>>(a);
  } else {
    a.qtiles = (a.T + 127) / 128;
    attn_prefill_kernel<F16, HD, 1><<<dim3((unsigned)(a.qtiles * a.B * a.heads)), 256, 0, s>>>(a);
  }
  return hipGetLastError();
}

}  // namespace

// Cuts a decode step into ranges of the cache, one workgroup for each and for each
// group of 4, 2 or 1 kv heads.  Two fit a CU at once;
// with eight (four rounds) the ends even out: the step above took 75 us with four a
// CU, 72.6 with eight, 81 with sixteen.  A range of under two tiles would spend more
// on its own set-up and on the merge than on its rows.
void attn_decode_plan(AttnDecodeArgs& a) {
  a.group = a.kv_heads % 4 == 0 ? 4 : a.kv_heads % 2 == 0 ? 2 : 1;
  const int tiles = (a.S + 64 / a.group - 1) / (64 / a.group);
  const int64_t units = a.B * (a.kv_heads / a.group);
  int64_t want = ((int64_t)device_cus() * 8 + units - 1) / units;
  if (want > tiles / 2) want = tiles / 2;
  if (want < 1) want = 1;
  a.tiles_per_split = (int)((tiles + want - 1) / want);
  a.splits = (tiles + a.tiles_per_split - 1) / a.tiles_per_split;
  a.parts = a.splits * (4 / a.group);
}

#define MHC_ATTN_HD(fn, a, s)                                      \
  switch (a.head_dim) {                                            \
    case 64: return a.f16 ? fn<true, 64>(a, s) : fn<false, 64>(a, s);    \
    case 96: return a.f16 ? fn<true, 96>(a, s) : fn<false, 96>(a, s);    \
    case 128: return a.f16 ? fn<true, 128>(a, s) : fn<false, 128>(a, s); \
    default: return hipErrorInvalidValue;                          \
  }

hipError_t launch_k_norm_rope(const KRopeArgs& a, hipStream_t s) { MHC_ATTN_HD(rope_hd, a, s) }
hipError_t launch_attn_decode(const AttnDecodeArgs& a, hipStream_t s) { MHC_ATTN_HD(decode_hd, a, s) }
hipError_t launch_attn_prefill(const AttnPrefillArgs& a, hipStream_t s) { MHC_ATTN_HD(prefill_hd, a, s) }

}  // namespace mhc
