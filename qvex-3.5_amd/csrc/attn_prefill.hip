// Attention of prompt chunks: the same split-K flash attention over the tiled
// caches as attn_mfma_partial_kernel (mx.fast.scaled_dot_product_attention with
// the sigmoid gate, engine/model.py:221-232), for calls of many rows.
//
// The decode-side kernel gives a block 16 rows, so every key and value byte goes
// from L2 to a CU once per 4 prompt positions (2.1 GB for 512 positions at 4096
// keys: 137 us, 15 TB/s). Here a block is 64 rows of one kv head (4 of the 16-row
// tiles, one per wave; 16 positions of 4 query heads), and blocks of 32 keys go
// through LDS by DMA, double-buffered.
//
// Both products are transposed, so that P never leaves its lanes:
//   S^T[keys x rows] = K Q^T: the K operand's row i of key tile h is key
//     8 (i / 4) + 4 h + i % 4 of the block, so that lane (lg, li) ends with keys
//     8 lg + 4 h + j of q row li: as bf16 pairs the B operand of
//   O^T[dims x rows] += V^T P^T, whose A operand is 8 consecutive keys of one dim:
//     the V cache's own layout.
// A lane owns one q row: its m and l are scalars. Scores are kept in base 2; the
// reference m of a row moves only when a score exceeds it by more than 8 (P up to
// 256, fp32 sums), so nearly all blocks need no reduction across lanes and no pass
// over O. P is the sum of two bf16 terms, the second product on the V operand
// already in registers: with one term the largest weights, exact when every
// 32 keys have their own maximum, would lose their last bits (error of the output
// 2.3e-3 of its norm, 2.1e-3 with per-wave maxima, 1.66e-3 with two terms, which
// is the output's own rounding).
//
// A row's bits depend on nothing else of the call it comes in: m, l and O start afresh
// at every unit of keys (ATT_UNIT, counted from key 0), units are folded in key order into groups of ATT_GROUP, groups into the row, and a unit or a
// block of keys that a row does not see adds exactly nothing. Who folds is free: a
// block takes one unit, and the merge folds them, or a whole group, folded in
// registers (a second m, l, O; so one tile per wave, not two). One unit per block
// keeps a call of few rows wide; a group per block writes and merges a quarter of the
// records (us at 256 keys a unit, unit | group per block: 16 positions at 4096 keys
// 20 | 45, 128 40 | 54, 256 67 | 58, 512 112 | 90, 512 at 16384 498 | 260).
// LDS: 16-byte units in the caches' order, the K rows of odd 8-dim groups with
// rows r ^ 4, a dim's four V units XORed by (0, 2, 3, 1)[dim / 4 % 4], so that the
// 16 lanes of one pass of a read hit 16 bank groups (the permutation is in the
// DMA's per-lane source).
// us with the merge, against a block per 16-row tile with its combine and 512 keys a
// split (16 query and 4 kv heads of 256): 512 positions at 0 keys 25 (57), at 1024 46 (90),
// at 4096 90 (180), at 16384 260 (573); 128 at 4096 40 (51), at 1024 20 (26); 32 at
// 4096 23 (20), 16 at 256 17 (13), at 16384 31 (30). Bound by the LDS reads (32 of 16
// bytes per lane, wave and key block, a third more cycles than its 48 MFMAs) beside
// the exponentials at 2 waves per SIMD; few rows by the chain of a key block, 0.95 us.
#include "attn_prefill.h"

#include <math.h>

#include "lds_dma.h"

namespace {

typedef __bf16 ap_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 ap_bf16x2 __attribute__((ext_vector_type(2)));
typedef float ap_f32x4 __attribute__((ext_vector_type(4)));
typedef float ap_f32x2 __attribute__((ext_vector_type(2)));

constexpr float AP_NONE = -3.0e38f;    // m before any visible key
constexpr float AP_SLACK = 8.0f;

__device__ __forceinline__ ap_bf16x8 as_ap8(const u32x4 v) { return __builtin_bit_cast(ap_bf16x8, v); }
__device__ __forceinline__ uint32_t ap_pack(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((ap_f32x2{lo, hi}), ap_bf16x2));
}

// (m, l, o) of a row and of later keys of it, m in base 2: the same arithmetic in
// both kernels, from (AP_NONE, 0, 0), so that who folds does not show in the bits.
struct Fold {
  float a, b;
  __device__ __forceinline__ Fold(float& m, float& l, float m1, float l1) {
    const float mn = fmaxf(m, m1);
    a = __builtin_amdgcn_exp2f(m - mn);
    b = __builtin_amdgcn_exp2f(m1 - mn);
    m = mn;
    l = fmaf(l1, b, l * a);
  }
  __device__ __forceinline__ void operator()(float& o, float o1) const { o = fmaf(o1, b, o * a); }
};

template <int D>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache, const uint16_t* __restrict__ v_cache,
    const int32_t* __restrict__ pos0, int L, int Hq, int Hkv, int cap, int ntile, int QT, int unit, int units,
    float scale, float* __restrict__ ws) {
#pragma clang fp contract(off)
  constexpr int KS = D / 32;           // MFMA steps over head dims
  constexpr int NT = D / 16;           // 16-dim tiles of O
  constexpr int HALF = 64 * D;         // bytes of 32 keys of K, and of V
  __shared__ __align__(1024) uint8_t lds[2][2 * HALF];
  const int kh = blockIdx.x, split = blockIdx.z;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 15, lg = lane >> 4;
  const int GQ = Hq / Hkv;
  const int p0 = *pos0;
  const int k_lo = split * unit * units;
  const int first = blockIdx.y * qvex::ATT_BLOCK_TILES;                        // tiles of the block
  const int keys = p0 + min(L, (first + qvex::ATT_BLOCK_TILES) * QT);
  if (k_lo >= keys) return;            // the merge reads only splits that hold visible keys
  const int k_hi = k_lo + min(unit * units, keys - k_lo);
  const int tile = first + wave;

  // B operand: q row li of the tile; the row's last visible key
  u32x4 qa[KS];
  const int g = li / QT, lq = tile * QT + li % QT;
  const bool used = g < GQ && lq < L;
  const int rlim = used ? p0 + lq : -1;
  const uint16_t* qp = q + ((size_t)(used ? lq : 0) * Hq + kh * GQ + (used ? g : 0)) * D + 8 * lg;
#pragma unroll
  for (int s = 0; s < KS; ++s) qa[s] = used ? load16(qp + 32 * s) : u32x4{0, 0, 0, 0};
  // keys up to full_hi are visible to every row of the tile that is used, keys from wave_hi on to none
  const int full_hi = p0 + tile * QT, wave_hi = tile < ntile ? min(k_hi, p0 + min(L, (tile + 1) * QT)) : 0;

  const uint8_t* kb8 = reinterpret_cast<const uint8_t*>(k_cache + (size_t)kh * cap * D);
  const uint8_t* vb8 = reinterpret_cast<const uint8_t*>(v_cache + (size_t)kh * D * cap);
  const uint32_t base = lds_offset(lds);
  const int perm_d = (0x78 >> (2 * lg)) & 3;                      // lane / 16 -> 0, 2, 3, 1
  const uint32_t k_src = (lane ^ ((lg & 1) << 2)) * 16, v_src = (lane ^ perm_d) * 16;
  auto fetch = [&](int kb, int buf) __attribute__((always_inline)) {
    kb = min(kb, cap - 32);
    const uint8_t* ks = kb8 + (size_t)kb * (2 * D);
    const uint8_t* vs = vb8 + (size_t)kb * (2 * D);
#pragma unroll
    for (int i = 0; i < HALF / 4096; ++i) {
      const int at = (wave + 4 * i) * 1024;
      dma16(base + buf * 2 * HALF + at, k_src, ks + at);
      dma16(base + buf * 2 * HALF + HALF + at, v_src, vs + at);
    }
  };
  int k_at[2];                                                    // K operand of key tile h, step 0
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = 8 * ((li >> 2) & 1) + 4 * h + (li & 3);
    k_at[h] = (li >> 3) * KS * 1024 + lg * 256 + (r ^ ((lg & 1) << 2)) * 16;
  }
  const int v_at = HALF + li * 64 + (lg ^ ((0x78 >> (2 * ((li >> 2) & 3))) & 3)) * 16;

  const float c = scale * 1.44269504088896340736f;                // scores in base 2
  const ap_f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  float m = AP_NONE, l = 0.0f, mf = AP_NONE, lf = 0.0f;           // of the unit; of the units before it
  ap_f32x4 o[NT], of[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) o[t] = of[t] = zero;

  fetch(k_lo, 0);
  int buf = 0, unit_hi = k_lo + min(unit, k_hi - k_lo);
#pragma unroll 1
  for (int kb = k_lo; kb < k_hi; kb += 32, buf ^= 1) {
    arrive<0>();                       // this block has landed, and every wave has read the one before
    if (kb + 32 < k_hi) fetch(kb + 32, buf ^ 1);
    if (kb >= wave_hi) continue;       // uniform over the wave; the barrier above is reached all the same
    const uint8_t* from = lds[buf];

    ap_f32x4 sc[2] = {zero, zero};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        sc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_ap8(load16(from + k_at[h] + s * 1024)), as_ap8(qa[s]),
                                                        sc[h], 0, 0, 0);
    if (kb + 32 > min(full_hi + 1, k_hi)) {                       // some keys are not visible to some rows
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int key = kb + 8 * lg + 4 * h + j;
          if (key >= k_hi || key > rlim) sc[h][j] = -INFINITY;
        }
    }
    float top = sc[0][0];
#pragma unroll
    for (int e = 1; e < 8; ++e) top = fmaxf(top, sc[e >> 2][e & 3]);
    top *= c;
    if (__any(top - m > AP_SLACK)) {
      float x = fmaxf(top, __shfl_xor(top, 16, 64));
      x = fmaxf(x, __shfl_xor(x, 32, 64));                        // of the row, in its four lanes
      const float mn = x - m > AP_SLACK ? x : m;
      const float f = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= f;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) o[t][j] *= f;
    }
    u32x4 p, p_lo;                     // P and what its rounding left
    float e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      e[i] = __builtin_amdgcn_exp2f(fmaf(sc[i >> 2][i & 3], c, -m));
      l += e[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t hi = ap_pack(e[2 * i], e[2 * i + 1]);
      p[i] = hi;
      p_lo[i] = ap_pack(e[2 * i] - bf16_lo(hi), e[2 * i + 1] - bf16_hi(hi));
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const ap_bf16x8 vf = as_ap8(load16(from + v_at + t * 1024));
      o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, as_ap8(p), o[t], 0, 0, 0);
      o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, as_ap8(p_lo), o[t], 0, 0, 0);
    }
    if (kb + 32 >= min(unit_hi, wave_hi)) {                       // the tile's last block of the unit
      float sum = l + __shfl_xor(l, 16, 64);
      sum += __shfl_xor(sum, 32, 64);
      const Fold fold(mf, lf, m, sum);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float x = of[t][j];
          fold(x, o[t][j]);
          of[t][j] = x;
        }
        o[t] = zero;
      }
      m = AP_NONE;
      l = 0.0f;
      unit_hi += min(unit, k_hi - unit_hi);
    }
  }

  // one record per tile and split: ([16 rows][m, l], [16 rows][O[D]])
  if (tile >= ntile) return;
  float* rec = ws + (((size_t)kh * ntile + tile) * gridDim.z + split) * 16 * (D + 2);
  if (lg == 0) *reinterpret_cast<float2*>(rec + 2 * li) = make_float2(mf, lf);
#pragma unroll
  for (int t = 0; t < NT; ++t) *reinterpret_cast<ap_f32x4*>(rec + 32 + (size_t)li * D + 16 * t + 4 * lg) = of[t];
}

// out[lq, h D + d] = bf16(sigmoid(gate) * O / l), the records of the splits that hold keys visible
// to the row's tile folded in key order: units into groups of ATT_GROUP, groups into
// the row (a record is a unit or, units > 1, a whole group). D / 4 lanes per row, four
// dims each, eight records requested at a time (attn_combine_kernel gives a row to
// four blocks, which only a handful of rows needs).
template <int D>
__global__ __launch_bounds__(256) void attn_prefill_merge_kernel(const float* __restrict__ ws, int nsplit, int ntile,
                                                                 int unit, int units,
                                                                 const int32_t* __restrict__ pos0, int L, int Hq,
                                                                 int Hkv, int QT, const uint16_t* __restrict__ gate,
                                                                 long g_stride, uint16_t* __restrict__ out, int vec) {
#pragma clang fp contract(off)
  constexpr int LANES = D / 4, B = 8, G = qvex::ATT_GROUP;
  static_assert(B % G == 0, "a batch holds whole groups");
  const int row = blockIdx.x * (256 / LANES) + (int)threadIdx.x / LANES, j = (int)threadIdx.x % LANES;
  if (row >= L * Hq) return;
  const int lq = row / Hq, h = row - lq * Hq, GQ = Hq / Hkv, kh = h / GQ, tile = lq / QT;
  const int r = (h - kh * GQ) * QT + lq % QT;
  const size_t rec = (size_t)16 * (D + 2);
  const float* base = ws + ((size_t)kh * ntile + tile) * nsplit * rec;
  const uint16_t* gp = gate + (size_t)lq * g_stride + (size_t)h * 2 * D + D + 4 * j;
  float gt[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) gt[i] = bf16_to_f32(gp[i]);
  const int keys = *pos0 + min(L, (tile + 1) * QT), nact = min(nsplit, (keys - 1) / (unit * units) + 1);

  float m = AP_NONE, l = 0.0f, mg = AP_NONE, lg = 0.0f;           // of the row; of the group so far
  float o[4] = {0.0f, 0.0f, 0.0f, 0.0f}, og[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = 0; s0 < nact; s0 += B) {
    float2 ml[B];
    ap_f32x4 os[B];
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const float* rp = base + (size_t)min(s0 + i, nact - 1) * rec;
      ml[i] = *reinterpret_cast<const float2*>(rp + 2 * r);
      os[i] = *reinterpret_cast<const ap_f32x4*>(rp + 32 + (size_t)r * D + 4 * j);
    }
#pragma unroll
    for (int i = 0; i < B; ++i) {
      if (s0 + i >= nact) break;
      const Fold f(mg, lg, ml[i].x, ml[i].y);
#pragma unroll
      for (int e = 0; e < 4; ++e) f(og[e], os[i][e]);
      if (units == 1 && i % G != G - 1 && s0 + i + 1 < nact) continue;
      const Fold t(m, l, mg, lg);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        t(o[e], og[e]);
        og[e] = 0.0f;
      }
      mg = AP_NONE;
      lg = 0.0f;
    }
  }
  const float invl = l > 0.0f ? 1.0f / l : 0.0f;
  uint16_t b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = f32_to_bf16(o[i] * invl / (1.0f + expf(-gt[i])));
  uint16_t* op = out + (size_t)lq * Hq * D + (size_t)h * D + 4 * j;
  if (vec) {
    *reinterpret_cast<u32x2*>(op) = u32x2{(uint32_t)b[0] | (uint32_t)b[1] << 16, (uint32_t)b[2] | (uint32_t)b[3] << 16};
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) op[i] = b[i];
  }
}

template <int D>
void launch(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, const int32_t* pos0, int L, int Hq,
            int Hkv, int cap, int ntile, int nsplit, int QT, int unit, int units, float scale, const uint16_t* gate,
            long g_stride, uint16_t* out, float* ws, hipStream_t st) {
  constexpr int BT = qvex::ATT_BLOCK_TILES;
  hipLaunchKernelGGL(attn_prefill_kernel<D>, dim3(Hkv, (ntile + BT - 1) / BT, nsplit), dim3(64 * BT), 0, st, q, k_cache,
                     v_cache, pos0, L, Hq, Hkv, cap, ntile, QT, unit, units, scale, ws);
  const long rows = (long)L * Hq;
  const int per = 256 / (D / 4);
  hipLaunchKernelGGL(attn_prefill_merge_kernel<D>, dim3((unsigned)((rows + per - 1) / per)), dim3(256), 0, st, ws,
                     nsplit, ntile, unit, units, pos0, L, Hq, Hkv, QT, gate, g_stride, out,
                     (int)qvex_aligned(out, 8));
}

}  // namespace

void qvex::attention_prefill(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, const int32_t* pos0,
                             int L, int Hq, int Hkv, int D, int cap, int ntile, int nsplit, int QT, int unit,
                             int units, float scale, const uint16_t* gate, long gate_stride, uint16_t* out, float* ws,
                             void* stream) {
  const auto go = D == 256 ? &launch<256> : &launch<128>;
  go(q, k_cache, v_cache, pos0, L, Hq, Hkv, cap, ntile, nsplit, QT, unit, units, scale, gate, gate_stride, out, ws,
     (hipStream_t)stream);
}
