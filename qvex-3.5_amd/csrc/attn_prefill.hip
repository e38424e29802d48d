// Attention of prompt chunks: the same split-K flash attention over the tiled
// caches as attn_mfma_partial_kernel (mx.fast.scaled_dot_product_attention with
// the sigmoid gate, engine/model.py:221-232), for calls of many rows.
//
// The decode-side kernel gives a block 16 rows, so every key and value byte goes
// from L2 to a CU once per 4 prompt positions (2.1 GB for 512 positions at 4096
// keys: 137 us, 15 TB/s). Here a block is 128 rows of one kv head (8 of the 16-row
// tiles; 32 positions of 4 query heads), each of its 4 waves owns two tiles, and
// blocks of 32 keys go through LDS by DMA, double-buffered.
//
// Both products are transposed, so that P never leaves its lanes:
//   S^T[keys x rows] = K Q^T: the K operand's row i of key tile h is key
//     8 (i / 4) + 4 h + i % 4 of the block, so that lane (lg, li) ends with keys
//     8 lg + 4 h + j of q row li: as bf16 pairs the B operand of
//   O^T[dims x rows] += V^T P^T, whose A operand is 8 consecutive keys of one dim:
//     the V cache's own layout.
// A lane owns one q row of each tile: its m and l are scalars. Scores are kept in
// base 2; the reference m of a row moves only when a score exceeds it by more than 8
// (P up to 256, fp32 sums), so nearly all blocks need no reduction across lanes and
// no pass over O. Each row decides for itself, so its bits do not depend on the
// rows beside it. P is the sum of two bf16 terms, the second product on the V
// operand already in registers: with one term the largest weights, exact when every
// 32 keys have their own maximum, would lose their last bits (error of the output
// 2.3e-3 of its norm, 2.1e-3 with per-wave maxima, 1.66e-3 with two terms, which
// is the output's own rounding; 57 us against 68 below).
// LDS: 16-byte units in the caches' order, the K rows of odd 8-dim groups with
// rows r ^ 4, a dim's four V units XORed by (0, 2, 3, 1)[dim / 4 % 4], so that the
// 16 lanes of one pass of a read hit 16 bank groups (the permutation is in the
// DMA's per-lane source).
// us with the merge, against a block per 16-row tile with its combine (16 query and
// 4 kv heads of 256): 512 positions at 0 keys 27 (57), at 1024 45 (90), at 3584 68
// (163), at 16384 204 (576); 128 at 4096 37 (49). Bound by the MFMAs (96 per wave
// and key block) and as many cycles of LDS reads (32 of 16 bytes per lane) beside
// the exponentials, at 2 waves per SIMD.
#include "attn_prefill.h"

#include <math.h>

#include "lds_dma.h"

namespace {

typedef __bf16 ap_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 ap_bf16x2 __attribute__((ext_vector_type(2)));
typedef float ap_f32x4 __attribute__((ext_vector_type(4)));
typedef float ap_f32x2 __attribute__((ext_vector_type(2)));

constexpr int AP_TILES = 8;            // 16-row tiles per block
constexpr int AP_RT = 2;               // per wave
constexpr float AP_NONE = -3.0e38f;    // m before any visible key
constexpr float AP_SLACK = 8.0f;

__device__ __forceinline__ ap_bf16x8 as_ap8(const u32x4 v) { return __builtin_bit_cast(ap_bf16x8, v); }
__device__ __forceinline__ uint32_t ap_pack(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((ap_f32x2{lo, hi}), ap_bf16x2));
}

template <int D>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache, const uint16_t* __restrict__ v_cache,
    const int32_t* __restrict__ pos0, int L, int Hq, int Hkv, int cap, int ntile, int QT, int keys_per_split,
    float scale, float* __restrict__ ws) {
  constexpr int KS = D / 32;           // MFMA steps over head dims
  constexpr int NT = D / 16;           // 16-dim tiles of O
  constexpr int HALF = 64 * D;         // bytes of 32 keys of K, and of V
  __shared__ __align__(1024) uint8_t lds[2][2 * HALF];
  const int kh = blockIdx.x, split = blockIdx.z;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 15, lg = lane >> 4;
  const int GQ = Hq / Hkv;
  const int p0 = *pos0;
  const int k_lo = split * keys_per_split;
  const int first = blockIdx.y * AP_TILES;                        // tiles of the block
  const int k_hi = min(k_lo + keys_per_split, p0 + min(L, (first + AP_TILES) * QT));
  if (k_lo >= k_hi) return;            // the merge reads only splits that hold visible keys
  const int tile0 = first + AP_RT * wave;

  // B operand: q row li of each tile; the row's last visible key
  u32x4 qa[AP_RT][KS];
  int rlim[AP_RT];
#pragma unroll
  for (int rt = 0; rt < AP_RT; ++rt) {
    const int g = li / QT, lq = (tile0 + rt) * QT + li % QT;
    const bool ok = g < GQ && lq < L;
    rlim[rt] = ok ? p0 + lq : -1;
    const uint16_t* qp = q + ((size_t)(ok ? lq : 0) * Hq + kh * GQ + (ok ? g : 0)) * D + 8 * lg;
#pragma unroll
    for (int s = 0; s < KS; ++s) qa[rt][s] = ok ? load16(qp + 32 * s) : u32x4{0, 0, 0, 0};
  }
  // keys up to full_hi are visible to every row of the wave that is used, keys from wave_hi on to none
  const int full_hi = p0 + tile0 * QT, wave_hi = tile0 < ntile ? p0 + min(L, (tile0 + AP_RT) * QT) : 0;

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
  float m[AP_RT], l[AP_RT];
  ap_f32x4 o[AP_RT][NT];
#pragma unroll
  for (int rt = 0; rt < AP_RT; ++rt) {
    m[rt] = AP_NONE;
    l[rt] = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t) o[rt][t] = ap_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }

  fetch(k_lo, 0);
  int buf = 0;
#pragma unroll 1
  for (int kb = k_lo; kb < k_hi; kb += 32, buf ^= 1) {
    arrive<0>();                       // this block has landed, and every wave has read the one before
    if (kb + 32 < k_hi) fetch(kb + 32, buf ^ 1);
    if (kb >= wave_hi) continue;       // uniform over the wave; the barrier above is reached all the same
    const uint8_t* from = lds[buf];

    ap_f32x4 sc[AP_RT][2];
#pragma unroll
    for (int rt = 0; rt < AP_RT; ++rt)
#pragma unroll
      for (int h = 0; h < 2; ++h) sc[rt][h] = ap_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const ap_bf16x8 kf = as_ap8(load16(from + k_at[h] + s * 1024));
#pragma unroll
        for (int rt = 0; rt < AP_RT; ++rt)
          sc[rt][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, as_ap8(qa[rt][s]), sc[rt][h], 0, 0, 0);
      }
    if (kb + 32 > min(full_hi + 1, k_hi)) {                       // some keys are not visible to some rows
#pragma unroll
      for (int rt = 0; rt < AP_RT; ++rt)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int key = kb + 8 * lg + 4 * h + j;
            if (key >= k_hi || key > rlim[rt]) sc[rt][h][j] = -INFINITY;
          }
    }
    float top[AP_RT];
    bool moves = false;
#pragma unroll
    for (int rt = 0; rt < AP_RT; ++rt) {
      top[rt] = sc[rt][0][0];
#pragma unroll
      for (int e = 1; e < 8; ++e) top[rt] = fmaxf(top[rt], sc[rt][e >> 2][e & 3]);
      top[rt] *= c;
      moves |= top[rt] - m[rt] > AP_SLACK;
    }
    if (__any(moves)) {
#pragma unroll
      for (int rt = 0; rt < AP_RT; ++rt) {
        float x = fmaxf(top[rt], __shfl_xor(top[rt], 16, 64));
        x = fmaxf(x, __shfl_xor(x, 32, 64));                      // of the row, in its four lanes
        const float mn = x - m[rt] > AP_SLACK ? x : m[rt];
        const float f = __builtin_amdgcn_exp2f(m[rt] - mn);
        m[rt] = mn;
        l[rt] *= f;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int j = 0; j < 4; ++j) o[rt][t][j] *= f;
      }
    }
    u32x4 p[AP_RT], p_lo[AP_RT];       // P and what its rounding left
#pragma unroll
    for (int rt = 0; rt < AP_RT; ++rt) {
      float e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        e[i] = __builtin_amdgcn_exp2f(fmaf(sc[rt][i >> 2][i & 3], c, -m[rt]));
        l[rt] += e[i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t hi = ap_pack(e[2 * i], e[2 * i + 1]);
        p[rt][i] = hi;
        p_lo[rt][i] = ap_pack(e[2 * i] - bf16_lo(hi), e[2 * i + 1] - bf16_hi(hi));
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const ap_bf16x8 vf = as_ap8(load16(from + v_at + t * 1024));
#pragma unroll
      for (int rt = 0; rt < AP_RT; ++rt)
        o[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, as_ap8(p[rt]), o[rt][t], 0, 0, 0);
#pragma unroll
      for (int rt = 0; rt < AP_RT; ++rt)
        o[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, as_ap8(p_lo[rt]), o[rt][t], 0, 0, 0);
    }
  }

  // one record per tile and split: ([16 rows][m, l], [16 rows][O[D]]), m in base e
#pragma unroll
  for (int rt = 0; rt < AP_RT; ++rt) {
    if (tile0 + rt >= ntile) continue;
    float* rec = ws + (((size_t)kh * ntile + tile0 + rt) * gridDim.z + split) * 16 * (D + 2);
    float sum = l[rt] + __shfl_xor(l[rt], 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (lg == 0)
      *reinterpret_cast<float2*>(rec + 2 * li) =
          make_float2(m[rt] == AP_NONE ? -INFINITY : m[rt] * 0.693147180559945309417f, sum);
#pragma unroll
    for (int t = 0; t < NT; ++t) *reinterpret_cast<ap_f32x4*>(rec + 32 + (size_t)li * D + 16 * t + 4 * lg) = o[rt][t];
  }
}

// out[lq, h D + d] = bf16(sigmoid(gate) * sum_s O_s e^{m_s - m} / sum_s l_s e^{m_s - m})
// over the splits that hold keys visible to the row's tile. D / 4 lanes per row,
// four dims each, eight splits requested at a time (attn_combine_kernel gives a row
// to four blocks, which only a handful of rows needs).
template <int D>
__global__ __launch_bounds__(256) void attn_prefill_merge_kernel(const float* __restrict__ ws, int nsplit, int ntile,
                                                                 int keys_per_split, const int32_t* __restrict__ pos0,
                                                                 int L, int Hq, int Hkv, int QT,
                                                                 const uint16_t* __restrict__ gate, long g_stride,
                                                                 uint16_t* __restrict__ out, int vec) {
  constexpr int LANES = D / 4, B = 8;
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
  const int nact = min(nsplit, (*pos0 + min(L, (tile + 1) * QT) + keys_per_split - 1) / keys_per_split);

  float m = -INFINITY, l = 0.0f;
  float4 o = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = 0; s0 < nact; s0 += B) {
    float2 ml[B];
    float4 os[B];
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const float* rp = base + (size_t)min(s0 + i, nact - 1) * rec;
      ml[i] = *reinterpret_cast<const float2*>(rp + 2 * r);
      os[i] = *reinterpret_cast<const float4*>(rp + 32 + (size_t)r * D + 4 * j);
    }
    float mb = m;
#pragma unroll
    for (int i = 0; i < B; ++i) mb = fmaxf(mb, ml[i].x);
    if (mb == -INFINITY) continue;
    const float f0 = m == -INFINITY ? 0.0f : expf(m - mb);
    l *= f0;
    o.x *= f0; o.y *= f0; o.z *= f0; o.w *= f0;
#pragma unroll
    for (int i = 0; i < B; ++i) {
      if (s0 + i >= nact || ml[i].x == -INFINITY) continue;
      const float f = expf(ml[i].x - mb);
      l = fmaf(ml[i].y, f, l);
      o.x = fmaf(os[i].x, f, o.x);
      o.y = fmaf(os[i].y, f, o.y);
      o.z = fmaf(os[i].z, f, o.z);
      o.w = fmaf(os[i].w, f, o.w);
    }
    m = mb;
  }
  const float invl = l > 0.0f ? 1.0f / l : 0.0f;
  const float y[4] = {o.x, o.y, o.z, o.w};
  uint16_t b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = f32_to_bf16(y[i] * invl / (1.0f + expf(-gt[i])));
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
            int Hkv, int cap, int ntile, int nsplit, int QT, int kps, float scale, const uint16_t* gate, long g_stride,
            uint16_t* out, float* ws, hipStream_t st) {
  hipLaunchKernelGGL(attn_prefill_kernel<D>, dim3(Hkv, (ntile + AP_TILES - 1) / AP_TILES, nsplit), dim3(256), 0, st, q,
                     k_cache, v_cache, pos0, L, Hq, Hkv, cap, ntile, QT, kps, scale, ws);
  const long rows = (long)L * Hq;
  const int per = 256 / (D / 4);
  hipLaunchKernelGGL(attn_prefill_merge_kernel<D>, dim3((unsigned)((rows + per - 1) / per)), dim3(256), 0, st, ws,
                     nsplit, ntile, kps, pos0, L, Hq, Hkv, QT, gate, g_stride, out, (int)qvex_aligned(out, 8));
}

}  // namespace

void qvex::attention_prefill(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, const int32_t* pos0,
                             int L, int Hq, int Hkv, int D, int cap, int ntile, int nsplit, int QT, int keys_per_split,
                             float scale, const uint16_t* gate, long gate_stride, uint16_t* out, float* ws,
                             void* stream) {
  const auto go = D == 256 ? &launch<256> : &launch<128>;
  go(q, k_cache, v_cache, pos0, L, Hq, Hkv, cap, ntile, nsplit, QT, keys_per_split, scale, gate, gate_stride, out, ws,
     (hipStream_t)stream);
}
