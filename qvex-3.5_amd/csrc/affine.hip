// MLX affine quantization of any supported width: bits 2, 3, 4, 5, 6, 8 and
// groups of 32, 64 or 128 codes (the per-module overrides of Config.qparams,
// engine/model.py:68-71, fed to mx.quantized_matmul / mx.dequantize at
// engine/model.py:87-91, 127-130).
//
// Layout (quant/quantize.py:71-75): each weight row is one little-endian bit
// stream, code k at stream bits [k*bits, (k+1)*bits), read as uint32 words; a
// row of K codes is K*bits/32 words. Per (row, group): a bf16 scale s and bias
// b, w = s*q + b.
//
// Four kernels:
//   * qmv_affine_kernel: y = x W^T for 1..8 activation rows, VALU only. A chunk
//     is 32 consecutive codes of one row = `bits` words (K % 32 == 0 and the
//     group is a multiple of 32, so a chunk lies in one group). Each lane
//     extracts its chunk's 32 codes once per weight row (compile-time bit
//     offsets: one v_bfe per code, an alignbit first where a code straddles two
//     words), then accumulates d = sum q*x and X = sum x per activation row in
//     fp32 and folds acc += s*d + b*X. R weight rows per wave share the
//     activation chunk; lanes stride over the chunks; one wave sum per output.
//   * affine_gemm_kernel: the same product for any number of rows (prompt
//     chunks) on the matrix cores.
//   * embed_affine_kernel: the rows of an embedding table, bf16(s*q + b).
//   * widen_w4_kernel: lossless re-encoding of a width <= 4, group % 64 == 0
//     weight as 4-bit group-64 (codes widened to nibbles, a group-128 scale and
//     bias repeated for both 64-code halves), so such layers run the packed
//     MFMA products and every fused epilogue of the 4-bit path unchanged.
#include "lds_dma.h"
#include "qvex_common.h"

namespace {

// Code j (0..31) of a chunk held as BITS words: compile-time offsets after unrolling.
template <int BITS>
__device__ __forceinline__ uint32_t chunk_code(const uint32_t (&wv)[BITS], int j) {
  const int o = j * BITS;
  const int wi = o >> 5, sh = o & 31;
  const uint32_t mask = (1u << BITS) - 1u;
  if (sh + BITS <= 32) return (wv[wi] >> sh) & mask;
  return __builtin_amdgcn_alignbit(wv[wi + 1], wv[wi], sh) & mask;
}

// The BITS words of one chunk: the widest vector load the chunk's alignment
// allows (a chunk starts at a multiple of 4*BITS bytes of a 16-byte aligned row
// stream): x4 for 4 and 8 bits, x2 for 2 and 6, single words for 3 and 5.
template <int BITS>
__device__ __forceinline__ void load_chunk(const uint32_t* __restrict__ p, uint32_t (&wv)[BITS]) {
  if constexpr (BITS % 4 == 0) {
#pragma unroll
    for (int i = 0; i < BITS / 4; ++i) {
      const u32x4 v = load_nt16(p + 4 * i);
      wv[4 * i] = v.x; wv[4 * i + 1] = v.y; wv[4 * i + 2] = v.z; wv[4 * i + 3] = v.w;
    }
  } else if constexpr (BITS % 2 == 0) {
#pragma unroll
    for (int i = 0; i < BITS / 2; ++i) {
      const u32x2 v = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p + 2 * i));
      wv[2 * i] = v.x; wv[2 * i + 1] = v.y;
    }
  } else {
#pragma unroll
    for (int i = 0; i < BITS; ++i) wv[i] = __builtin_nontemporal_load(p + i);
  }
}

constexpr int AFF_MAXM = 8;    // activation rows per launch
constexpr long AFF_GEMM_TALL = 512;    // blocks of 64 rows from which the GEMM takes them

// AFF_R weight rows per wave share each activation chunk: 1 for one or two
// activation rows (81 VGPRs, more waves in flight: 12.6 against 13.6 us for a
// 5-bit 12,288 x 4,096 product at one row), 2 above (the dequantized codes serve
// twice as many products: 25 against 28.5 us at four rows).
template <int BITS, int AFF_R>
__global__ __launch_bounds__(256) void qmv_affine_kernel(const uint16_t* __restrict__ x,
                                                         const uint32_t* __restrict__ w,
                                                         const uint16_t* __restrict__ scales,
                                                         const uint16_t* __restrict__ biases,
                                                         uint16_t* __restrict__ y, int M, int N, int K,
                                                         int gshift) {
  const int lane = threadIdx.x & 63;
  const int row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * AFF_R;
  const int nchunk = K >> 5;
  const int KW = nchunk * BITS;        // words per row
  const int G = K >> gshift;           // groups per row

  float acc[AFF_R][AFF_MAXM];
#pragma unroll
  for (int r = 0; r < AFF_R; ++r)
#pragma unroll
    for (int m = 0; m < AFF_MAXM; ++m) acc[r][m] = 0.0f;

  for (int c = lane; c < nchunk; c += 64) {
    // rows past N re-read row N-1 (never stored)
    float q[AFF_R][32];
    float s[AFF_R], b[AFF_R];
#pragma unroll
    for (int r = 0; r < AFF_R; ++r) {
      const int row = min(row0 + r, N - 1);
      uint32_t wv[BITS];
      load_chunk<BITS>(w + (size_t)row * KW + (size_t)c * BITS, wv);
      const int g = (c << 5) >> gshift;
      s[r] = bf16_to_f32(scales[(size_t)row * G + g]);
      b[r] = bf16_to_f32(biases[(size_t)row * G + g]);
#pragma unroll
      for (int j = 0; j < 32; ++j) q[r][j] = (float)chunk_code<BITS>(wv, j);
    }
#pragma unroll
    for (int m = 0; m < AFF_MAXM; ++m) {
      if (m >= M) break;
      const uint16_t* xr = x + (size_t)m * K + (size_t)c * 32;
      float xs = 0.0f;
      float d[AFF_R];
#pragma unroll
      for (int r = 0; r < AFF_R; ++r) d[r] = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const u32x4 v = load16(xr + 8 * i);
        const uint32_t pr[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const float x0 = bf16_lo(pr[h]), x1 = bf16_hi(pr[h]);
          xs += x0;
          xs += x1;
#pragma unroll
          for (int r = 0; r < AFF_R; ++r) {
            d[r] = fmaf(q[r][8 * i + 2 * h], x0, d[r]);
            d[r] = fmaf(q[r][8 * i + 2 * h + 1], x1, d[r]);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < AFF_R; ++r) acc[r][m] = fmaf(s[r], d[r], fmaf(b[r], xs, acc[r][m]));
    }
  }

#pragma unroll
  for (int r = 0; r < AFF_R; ++r)
#pragma unroll
    for (int m = 0; m < AFF_MAXM; ++m)
      if (m < M) acc[r][m] = wave_sum_to_lane63(acc[r][m]);
  if (lane == 63) {
#pragma unroll
    for (int r = 0; r < AFF_R; ++r) {
      const int row = row0 + r;
      if (row >= N) continue;
#pragma unroll
      for (int m = 0; m < AFF_MAXM; ++m)
        if (m < M) y[(size_t)m * N + row] = f32_to_bf16(acc[r][m]);
    }
  }
}

// ---------------------------------------------------------------- prompt chunks
//
// y = x W^T on the matrix cores without rounding a weight: the codes themselves
// are bf16 numbers (integers up to 255 are exact), so a group's d = sum q*x comes
// from MFMAs on the raw codes, X = sum x from an MFMA against ones (it lands in
// d's lanes), both in fp32, and acc += s*d + b*X folds the group as the VALU
// kernel does. A row's order of sums depends on neither M nor the block shape.
//
// A block is 4 waves, 16 MT rows x 64 outputs, one 16-output tile per wave; a
// stage of the k loop is 128 codes (4 MFMA steps of 32). Activations go through
// LDS (16-byte chunk ch of a row at ch ^ row_swizzle(row): the 16 lanes of one
// pass of a 16-byte read hit 16 bank groups). A wave's weights go through LDS of
// its own: whole 16 BITS-byte row pieces by 16-byte loads, then BITS bytes (8
// codes) per lane and step. (Taken from global memory by the lanes that use them,
// 8 bytes of each of 16 rows per load, a stage cost about 1 us whatever MT.)
// (scale, bias) pairs: one load per lane serves four stages, broadcast by a lane
// permute per group. Bound by issue: a step's extraction (12 VALU instructions
// for 8 bits), 8 fmas per row tile and group, 2 MFMAs per row tile.
// us, against chunks of 8 rows through the VALU kernel: 200 rows of 4096 x 4096 at
// 8 bits 30.5 (368; replays of a graph 34.4), 512 rows of 12288 x 4096 at 6 bits 155,
// 1024 rows of 24576 x 4096 at 8 bits 484.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// the 8 codes at bit `sh` (a multiple of 8) of the words (lo, hi), as bf16
template <int BITS>
__device__ __forceinline__ bf16x8_t codes8(uint32_t lo, uint32_t hi, int sh) {
  constexpr uint32_t mask = (1u << BITS) - 1u;
  uint32_t v[2] = {lo, hi};
  if constexpr (BITS != 4 && BITS != 8) {
    v[0] = __builtin_amdgcn_alignbit(hi, lo, sh);
    v[1] = hi >> sh;
  }
  float f[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int o = j * BITS, wi = o >> 5, s = o & 31;
    const uint32_t q = s + BITS <= 32 ? v[wi] >> s : __builtin_amdgcn_alignbit(v[1], v[0], s);
    f[j] = (float)(q & mask);
  }
  u32x4 r;      // the high halves: exact
#pragma unroll
  for (int j = 0; j < 4; ++j)
    r[j] = __builtin_amdgcn_perm(__float_as_uint(f[2 * j + 1]), __float_as_uint(f[2 * j]), 0x07060302u);
  return __builtin_bit_cast(bf16x8_t, r);
}

template <int BITS, int G32, int MT>     // G32: 32-code steps per group
__global__ __launch_bounds__(256) void affine_gemm_kernel(const uint16_t* __restrict__ x,
                                                          const uint32_t* __restrict__ w,
                                                          const uint16_t* __restrict__ scales,
                                                          const uint16_t* __restrict__ biases,
                                                          uint16_t* __restrict__ y, int M, int N, int K) {
  constexpr int NG = 4 / G32;                      // groups per stage, and of four stages per lane
  constexpr int NW = (16 * BITS + 63) / 64;        // 16-byte weight loads per lane and stage
  constexpr int PITCH = 16 * BITS + 16;            // bytes of a weight row of one stage in LDS
  __shared__ u32x4 xs[2][MT * 256];
  __shared__ __align__(16) uint8_t ws[2][4][16 * PITCH];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane >> 4, i16 = lane & 15;
  // consecutive blocks of one XCD (dispatch is round-robin over 8) share their weights
  const int row_blocks = (M + 16 * MT - 1) / (16 * MT), columns = (N + 63) / 64;
  const int at = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
  const int column = at / row_blocks, m0 = (at - column * row_blocks) * 16 * MT;
  if (column >= columns) return;
  const int n0 = column * 64 + wave * 16, n = n0 + i16;
  const int chunks = K >> 5, groups = chunks / G32, stages = (chunks + 3) >> 2;
  const int words = chunks * BITS;                 // of a weight row

  struct Stage {
    u32x4 x[MT], w[NW];
  };
  const uint16_t* xp[MT];
  int xl[MT], wl[NW], wo[NW];
  const uint32_t* wp[NW];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int row = (tid >> 4) + 16 * i;
    xp[i] = x + (size_t)min(m0 + row, M - 1) * K;
    xl[i] = row * 16 + ((tid & 15) ^ row_swizzle(row));
  }
#pragma unroll
  for (int i = 0; i < NW; ++i) {                   // 16 rows x BITS pieces; rows past N repeat the last
    const int id = min(lane + 64 * i, 16 * BITS - 1), row = id / BITS, piece = id - row * BITS;
    wp[i] = w + (size_t)min(n0 + row, N - 1) * words;
    wo[i] = 4 * piece;
    wl[i] = row * PITCH + 16 * piece;
  }
  // stages past the last repeat it; what lies past K is never used
  auto load = [&](Stage& t, int st) __attribute__((always_inline)) {
    st = min(st, stages - 1);
#pragma unroll
    for (int i = 0; i < MT; ++i) t.x[i] = load16(xp[i] + min(st * 128 + (tid & 15) * 8, K - 8));
    if (G32 == 4 || st * 4 + 4 <= chunks) {
#pragma unroll
      for (int i = 0; i < NW; ++i) t.w[i] = *reinterpret_cast<const u32x4_a4*>(wp[i] + st * 4 * BITS + wo[i]);
    } else {
#pragma unroll
      for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) t.w[i][e] = wp[i][min(st * 4 * BITS + wo[i] + e, words - 1)];
    }
  };
  auto stage_to_lds = [&](const Stage& t, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; ++i) xs[buf][xl[i]] = t.x[i];
#pragma unroll
    for (int i = 0; i < NW; ++i)
      if (16 * BITS % 64 == 0 || lane + 64 * i < 16 * BITS) *reinterpret_cast<u32x4*>(&ws[buf][wave][wl[i]]) = t.w[i];
  };
  // (scale, bias) of four stages: lane (c, i) holds row i's groups NG c .. NG c + NG - 1 of the 4 NG
  const uint16_t* sr = scales + (size_t)min(n, N - 1) * groups;
  const uint16_t* br = biases + (size_t)min(n, N - 1) * groups;
  auto load_scales = [&](uint32_t (&sb)[NG], int st0) __attribute__((always_inline)) {
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int at_g = min(st0 * NG + NG * c + g, groups - 1);
      sb[g] = (uint32_t)sr[at_g] | (uint32_t)br[at_g] << 16;
    }
  };

  f32x4_t acc[MT], d[MT], X[MT];
  const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = d[mt] = X[mt] = zero;
  const bf16x8_t ones = __builtin_bit_cast(bf16x8_t, u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});
  const int a_at = i16 * 16, swz = row_swizzle(i16), w_at = i16 * PITCH + ((c * BITS) >> 2) * 4;
  const int sh = ((c * BITS) & 3) * 8;
  // step j of a stage, u its place among the four that sb covers
  auto step = [&](int buf, int j, const uint32_t (&sb)[NG], int u) __attribute__((always_inline)) {
    // a lane's 8 codes: BITS bytes, at most two words (the row's padding follows the last piece)
    const uint8_t* from = &ws[buf][wave][w_at + j * 4 * BITS];
    uint32_t lo, hi = 0;
    if constexpr (BITS == 8) {
      const u32x2 v = *reinterpret_cast<const u32x2*>(from);
      lo = v.x;
      hi = v.y;
    } else {
      lo = reinterpret_cast<const uint32_t*>(from)[0];
      if constexpr (BITS != 2 && BITS != 4) hi = reinterpret_cast<const uint32_t*>(from)[1];
    }
    const bf16x8_t q = codes8<BITS>(lo, hi, sh);
    const bool first = j % G32 == 0, last = j % G32 == G32 - 1;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const bf16x8_t a = __builtin_bit_cast(bf16x8_t, xs[buf][mt * 256 + a_at + ((4 * j + c) ^ swz)]);
      d[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, q, first ? zero : d[mt], 0, 0, 0);
      X[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ones, first ? zero : X[mt], 0, 0, 0);
    }
    if (!last) return;
    const uint32_t v = (uint32_t)__shfl((int)sb[j / G32], 16 * u + i16, 64);   // group NG u + j / G32
    const float s = bf16_lo(v), b = bf16_hi(v);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[mt][r] = fmaf(s, d[mt][r], fmaf(b, X[mt][r], acc[mt][r]));
  };

  // stage st is computed from LDS, st + 1 and st + 2 are in registers or on their way
  Stage t[2];
  uint32_t sb[NG], sb_next[NG];
  load(t[0], 0);
  load_scales(sb, 0);
  load(t[1], 1);
  stage_to_lds(t[0], 0);
  load(t[0], 2);
  __syncthreads();
#pragma unroll 1
  for (int st0 = 0; st0 < stages; st0 += 4) {
    load_scales(sb_next, min(st0 + 4, stages - 1));
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int st = st0 + u, buf = u & 1;
      if (st >= stages) break;
      const int steps = chunks - st * 4;
      if (G32 == 4 || steps >= 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) step(buf, j, sb, u);
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (j < steps) step(buf, j, sb, u);
      }
      stage_to_lds(t[buf ^ 1], buf ^ 1);
      load(t[buf ^ 1], st + 3);
      __syncthreads();
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) sb[g] = sb_next[g];
  }

  if (n >= N) return;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + 16 * mt + 4 * c + r;
      if (m < M) y[(size_t)m * N + n] = f32_to_bf16(acc[mt][r]);
    }
}

// One block per gathered row; a thread per 32-code chunk writes 64 bytes.
template <int BITS>
__global__ __launch_bounds__(256) void embed_affine_kernel(const int32_t* __restrict__ ids,
                                                           const uint32_t* __restrict__ w,
                                                           const uint16_t* __restrict__ sc,
                                                           const uint16_t* __restrict__ bi,
                                                           uint16_t* __restrict__ out, int V, int H, int gshift) {
  const int l = blockIdx.x;
  int id = ids[l];
  id = id < 0 ? 0 : (id >= V ? V - 1 : id);          // clamped like the 4-bit gather
  const int nchunk = H >> 5, G = H >> gshift;
  const uint32_t* wr = w + (size_t)id * nchunk * BITS;
  for (int c = threadIdx.x; c < nchunk; c += blockDim.x) {
    uint32_t wv[BITS];
    load_chunk<BITS>(wr + (size_t)c * BITS, wv);
    const int g = (c << 5) >> gshift;
    const float s = bf16_to_f32(sc[(size_t)id * G + g]);
    const float b = bf16_to_f32(bi[(size_t)id * G + g]);
    uint16_t* o = out + (size_t)l * H + (size_t)c * 32;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t pk[4];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const int j = 8 * i + 2 * h;
        pk[h] = pack_bf16x2(fmaf(s, (float)chunk_code<BITS>(wv, j), b),
                            fmaf(s, (float)chunk_code<BITS>(wv, j + 1), b));
      }
      u32x4 v;
      v.x = pk[0]; v.y = pk[1]; v.z = pk[2]; v.w = pk[3];
      *reinterpret_cast<u32x4*>(o + 8 * i) = v;
    }
  }
}

// One thread per 32-code chunk: four nibble words out; the first chunk of each
// 64-code group also writes that group's scale and bias.
template <int BITS>
__global__ __launch_bounds__(256) void widen_w4_kernel(const uint32_t* __restrict__ w,
                                                       const uint16_t* __restrict__ sc,
                                                       const uint16_t* __restrict__ bi, uint32_t* __restrict__ w4,
                                                       uint16_t* __restrict__ sc4, uint16_t* __restrict__ bi4,
                                                       long chunks, int K, int gshift) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= chunks) return;
  const int nchunk = K >> 5;
  const long n = t / nchunk;
  const int c = (int)(t - n * nchunk);
  uint32_t wv[BITS];
  load_chunk<BITS>(w + (size_t)t * BITS, wv);
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t v = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) v |= chunk_code<BITS>(wv, 8 * i + j) << (4 * j);
    o[i] = v;
  }
  u32x4 v;
  v.x = o[0]; v.y = o[1]; v.z = o[2]; v.w = o[3];
  *reinterpret_cast<u32x4*>(w4 + (size_t)t * 4) = v;
  if ((c & 1) == 0) {
    const int g = (c << 5) >> gshift;
    sc4[n * (K >> 6) + (c >> 1)] = sc[n * (K >> gshift) + g];
    bi4[n * (K >> 6) + (c >> 1)] = bi[n * (K >> gshift) + g];
  }
}

int group_shift(int group_size) {
  switch (group_size) {
    case 32: return 5;
    case 64: return 6;
    case 128: return 7;
  }
  return -1;
}

bool width_ok(int bits) { return bits == 2 || bits == 3 || bits == 4 || bits == 5 || bits == 6 || bits == 8; }

#define AFFINE_BITS_SWITCH(bits, KERNEL, ...)          \
  switch (bits) {                                      \
    case 2: KERNEL<2>(__VA_ARGS__); break;             \
    case 3: KERNEL<3>(__VA_ARGS__); break;             \
    case 4: KERNEL<4>(__VA_ARGS__); break;             \
    case 5: KERNEL<5>(__VA_ARGS__); break;             \
    case 6: KERNEL<6>(__VA_ARGS__); break;             \
    case 8: KERNEL<8>(__VA_ARGS__); break;             \
  }

template <int BITS>
void launch_qmv(hipStream_t st, const uint16_t* x, const uint32_t* w, const uint16_t* s, const uint16_t* b,
                uint16_t* y, int M, int N, int K, int gs) {
  if (M <= 2)
    hipLaunchKernelGGL((qmv_affine_kernel<BITS, 1>), dim3((unsigned)((N + 3) / 4)), dim3(256), 0, st, x, w, s, b, y,
                       M, N, K, gs);
  else
    hipLaunchKernelGGL((qmv_affine_kernel<BITS, 2>), dim3((unsigned)((N + 7) / 8)), dim3(256), 0, st, x, w, s, b, y,
                       M, N, K, gs);
}

template <int BITS, int G32>
void launch_gemm_group(hipStream_t st, const uint16_t* x, const uint32_t* w, const uint16_t* s, const uint16_t* b,
                       uint16_t* y, int M, int N, int K) {
  const long columns = (N + 63) / 64;
  auto go = [&](auto kernel, int rows) {
    const long blocks = columns * ((M + rows - 1) / rows);
    hipLaunchKernelGGL(kernel, dim3((unsigned)((blocks + 7) / 8 * 8)), dim3(256), 0, st, x, w, s, b, y, M, N, K);
  };
  // Tall blocks extract each code for more rows; below AFF_GEMM_TALL of them the
  // chip is not full and shorter ones finish sooner (us, 8 bits, K = 4096, blocks of
  // 64 | 32 rows: 64 x 4096 34 | 25, 200 x 4096 37 | 34, 512 x 4096 51 | 63,
  // 100 x 24576 65 | 86; 20 x 24576 at 5 bits, half of 64 rows empty, 49 | 38)
  if (M <= 16)
    go(affine_gemm_kernel<BITS, G32, 1>, 16);
  else if (M <= 32 || columns * ((M + 63) / 64) < AFF_GEMM_TALL)
    go(affine_gemm_kernel<BITS, G32, 2>, 32);
  else
    go(affine_gemm_kernel<BITS, G32, 4>, 64);
}

template <int BITS>
void launch_affine_gemm(hipStream_t st, const uint16_t* x, const uint32_t* w, const uint16_t* s, const uint16_t* b,
                        uint16_t* y, int M, int N, int K, int gs) {
  if (gs == 5) launch_gemm_group<BITS, 1>(st, x, w, s, b, y, M, N, K);
  if (gs == 6) launch_gemm_group<BITS, 2>(st, x, w, s, b, y, M, N, K);
  if (gs == 7) launch_gemm_group<BITS, 4>(st, x, w, s, b, y, M, N, K);
}

template <int BITS>
void launch_embed(dim3 grid, hipStream_t st, const int32_t* ids, const uint32_t* w, const uint16_t* s,
                  const uint16_t* b, uint16_t* out, int V, int H, int gs) {
  hipLaunchKernelGGL(embed_affine_kernel<BITS>, grid, dim3(256), 0, st, ids, w, s, b, out, V, H, gs);
}

template <int BITS>
void launch_widen(dim3 grid, hipStream_t st, const uint32_t* w, const uint16_t* s, const uint16_t* b, uint32_t* w4,
                  uint16_t* s4, uint16_t* b4, long chunks, int K, int gs) {
  hipLaunchKernelGGL(widen_w4_kernel<BITS>, grid, dim3(256), 0, st, w, s, b, w4, s4, b4, chunks, K, gs);
}

}  // namespace

extern "C" int qvex_qmv_affine(const uint16_t* x, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                               uint16_t* y, int M, int N, int K, int bits, int group_size, void* stream) {
  QVEX_CHECK_ARG(x && w && scales && biases && y, "qvex_qmv_affine: null pointer");
  const int gs = group_shift(group_size);
  QVEX_CHECK_ARG(width_ok(bits) && gs > 0, "qvex_qmv_affine: bits=%d group_size=%d (bits 2,3,4,5,6,8; groups 32,64,128)",
                 bits, group_size);
  QVEX_CHECK_ARG(M >= 1 && M <= AFF_MAXM && N >= 1 && K >= group_size && K % group_size == 0,
                 "qvex_qmv_affine: M=%d N=%d K=%d (1 <= M <= 8, K a positive multiple of the group size %d)", M, N,
                 K, group_size);
  QVEX_CHECK_ARG(qvex_aligned(x, 16) && qvex_aligned(w, 16), "qvex_qmv_affine: x and w must be 16-byte aligned");
  AFFINE_BITS_SWITCH(bits, launch_qmv, (hipStream_t)stream, x, w, scales, biases, y, M, N, K, gs);
  QVEX_CHECK_LAUNCH("qvex_qmv_affine");
  return QVEX_OK;
}

extern "C" int qvex_affine_gemm(const uint16_t* x, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                                uint16_t* y, int M, int N, int K, int bits, int group_size, void* stream) {
  QVEX_CHECK_ARG(x && w && scales && biases && y, "qvex_affine_gemm: null pointer");
  const int gs = group_shift(group_size);
  QVEX_CHECK_ARG(width_ok(bits) && gs > 0, "qvex_affine_gemm: bits=%d group_size=%d (bits 2,3,4,5,6,8; groups 32,64,128)",
                 bits, group_size);
  QVEX_CHECK_ARG(M >= 1 && N >= 1 && K >= group_size && K % group_size == 0,
                 "qvex_affine_gemm: M=%d N=%d K=%d (K a positive multiple of the group size %d)", M, N, K, group_size);
  QVEX_CHECK_ARG(((M + 15L) / 16) * ((N + 63L) / 64) <= (1L << 30), "qvex_affine_gemm: M=%d N=%d too large", M, N);
  QVEX_CHECK_ARG(qvex_aligned(x, 16) && qvex_aligned(w, 16), "qvex_affine_gemm: x and w must be 16-byte aligned");
  AFFINE_BITS_SWITCH(bits, launch_affine_gemm, (hipStream_t)stream, x, w, scales, biases, y, M, N, K, gs);
  QVEX_CHECK_LAUNCH("qvex_affine_gemm");
  return QVEX_OK;
}

extern "C" int qvex_embed_affine(const int32_t* ids, int L, const uint32_t* w, const uint16_t* scales,
                                 const uint16_t* biases, int V, int H, int bits, int group_size, uint16_t* out,
                                 void* stream) {
  QVEX_CHECK_ARG(ids && w && scales && biases && out, "qvex_embed_affine: null pointer");
  const int gs = group_shift(group_size);
  QVEX_CHECK_ARG(width_ok(bits) && gs > 0,
                 "qvex_embed_affine: bits=%d group_size=%d (bits 2,3,4,5,6,8; groups 32,64,128)", bits, group_size);
  QVEX_CHECK_ARG(L >= 1 && V >= 1 && H >= group_size && H % group_size == 0,
                 "qvex_embed_affine: L=%d V=%d H=%d (H a positive multiple of the group size)", L, V, H);
  QVEX_CHECK_ARG(qvex_aligned(out, 16) && qvex_aligned(w, 16), "qvex_embed_affine: w and out must be 16-byte aligned");
  AFFINE_BITS_SWITCH(bits, launch_embed, dim3(L), (hipStream_t)stream, ids, w, scales, biases, out, V, H, gs);
  QVEX_CHECK_LAUNCH("qvex_embed_affine");
  return QVEX_OK;
}

extern "C" int qvex_affine_widen_w4g64(const uint32_t* w, const uint16_t* scales, const uint16_t* biases, int N,
                                       int K, int bits, int group_size, uint32_t* w4, uint16_t* scales4,
                                       uint16_t* biases4, void* stream) {
  QVEX_CHECK_ARG(w && scales && biases && w4 && scales4 && biases4, "qvex_affine_widen_w4g64: null pointer");
  const int gs = group_shift(group_size);
  QVEX_CHECK_ARG((bits == 2 || bits == 3 || bits == 4) && (group_size == 64 || group_size == 128),
                 "qvex_affine_widen_w4g64: bits=%d group_size=%d (bits 2..4, groups 64 or 128 widen losslessly)",
                 bits, group_size);
  QVEX_CHECK_ARG(N >= 1 && K >= group_size && K % group_size == 0,
                 "qvex_affine_widen_w4g64: N=%d K=%d (K a positive multiple of the group size)", N, K);
  QVEX_CHECK_ARG(qvex_aligned(w, 16) && qvex_aligned(w4, 16), "qvex_affine_widen_w4g64: w and w4 must be 16-byte aligned");
  const long chunks = (long)N * (K / 32);
  QVEX_CHECK_ARG(chunks / 256 < 0x7fffffffL, "qvex_affine_widen_w4g64: too large");
  const dim3 grid((unsigned)((chunks + 255) / 256));
  if (bits == 2) launch_widen<2>(grid, (hipStream_t)stream, w, scales, biases, w4, scales4, biases4, chunks, K, gs);
  if (bits == 3) launch_widen<3>(grid, (hipStream_t)stream, w, scales, biases, w4, scales4, biases4, chunks, K, gs);
  if (bits == 4) launch_widen<4>(grid, (hipStream_t)stream, w, scales, biases, w4, scales4, biases4, chunks, K, gs);
  QVEX_CHECK_LAUNCH("qvex_affine_widen_w4g64");
  return QVEX_OK;
}
