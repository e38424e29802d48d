// Prefill products: y[M, N] = x[M, K] @ W^T for prompt chunks (M >= 16 rows),
// read straight from the tile-packed 4-bit copy of the weight.
//
// Reference semantics: mx.quantized_matmul(transpose=True, group_size=64,
// bits=4) in QLinear.__call__ (engine/model.py:87-91) on a prefill chunk
// (engine/engine.py:232-248). Each weight is dequantized in registers to
// bf16(s * q + b) (the value an fp32 fma gives, rounded once to bf16) and the
// products accumulate in fp32 on the matrix cores, so the result equals a bf16
// GEMM on the dequantized weight up to the summation order. That order depends
// on neither M nor the tile shape: a row's result is the same in every call.
//
// Operands. The packed record (tile t of 16 rows, set s of 256 k; see
// qmv_packed.hip) holds, for group g = 0..3 and row i, eight words of eight
// codes and the group's (scale, bias). A stage of the k loop is half a set, the
// groups 2h and 2h + 1: 128 consecutive k, so that a row's slice of the
// activations is two whole 128-byte lines (slices of 64 bytes move every line
// twice through L2: 24576 x 4096 at 1024 rows took 211 us against 198). Lane
// (c, i) = 16 c + i takes the words 4 (c & 1) + j (j = 0..3) of group
// 2h + c / 2: its eight codes of step j are k = 128 h + 32 c + 8 j .. + 7 of
// row i, one v_mfma_f32_16x16x32_bf16 operand, and the other operand is the
// same k of 16 activation rows. The weights are the first operand, so that a
// lane ends with four consecutive outputs of one row (8-byte stores).
//
// Dequantization. A masked word is a pair of fp16 subnormals, codes at bits 0
// and 16 (q * 2^-24) or at bits 4 and 20 (q * 2^-20): v_fma_mix_f32 reads either
// half, so s * 2^24 (or 2^20) and b give s * q + b in one instruction per code
// and 17 VALU instructions per 8 codes (27 with bf16 pairs unpacked to fp32). Where
// |s| is 2^104 or more s * 2^24 overflows and every sum it enters is infinite or NaN:
// a wave that ends with such a sum makes its tiles again from s * q + b itself, in
// the same order (no instruction more in the loop).
//
// Staging. Activations and weights both go from global memory to LDS by DMA
// into rings of stages, the stage that a wave reads first waited for with one
// counted vmcnt and one barrier: no staging registers, and loads two stages
// ahead. The DMAs are written as asm since the compiler otherwise makes LDS
// reads wait for DMAs into other ring slots (and drains all of them).
// Activation rows in LDS are 256 bytes, their 16-byte chunk ch at position
// ch ^ row_swizzle(row): the 16 lanes that one pass of ds_read_b128 serves
// (0-3, 12-15 of one quarter, 4-11 of the next) then hit 16 different bank
// groups (SQ_LDS_BANK_CONFLICT 0; half of the LDS cycles with ch ^ (row & 15)).
//
// Two kernels: packed_gemm_kernel for 65 rows and more (bound by the matrix
// cores together with the LDS and DMA traffic beside them: 1040 TFLOP/s at
// 1024 x 24576 x 4096, where the same loop without dequantization, LDS reads and
// DMA reaches 1600), packed_gemm_small_kernel for a few dozen rows (bound by
// the weights' way in and each wave's latency chain).
//
// us per product, against the 64 x 128 blocks with register-staged double
// buffers that these replace: 512 rows of 24576 x 4096 101 (255), 4096 x 12288 78
// (195), 12352 x 4096 64 (156), 10240 x 4096 59 (138), 4096 x 4096 29 (67); 37 rows
// of 10240 x 4096 15 (64).
#include "lds_dma.h"
#include "qvex_common.h"
#include "w4_dequant.h"

namespace {

constexpr int QG_TILE = 16;
constexpr int QG_SET = 256;                 // k per record
constexpr int QG_RECORD = 2304;             // bytes per (tile, set) record
constexpr int QG_WBYTES = 2048;
constexpr int QG_WSLOT = 1024 + 256;        // a tile's codes and (scale, bias) pairs of one stage in LDS

typedef _Float16 f16x2v __attribute__((ext_vector_type(2)));
typedef float f32x2v __attribute__((ext_vector_type(2)));

// the scale (for either code position) and bias of one weight row's group
struct GroupScale {
  float s0, s1, b;
  __device__ __forceinline__ void set(uint32_t sb) {
    const float s = bf16_lo(sb);
    s0 = s * 16777216.0f;
    s1 = s * 1048576.0f;
    b = bf16_hi(sb);
  }
};

__device__ __forceinline__ void mix2(uint32_t pair, float s, float b, float& lo, float& hi) {
  const f16x2v q = __builtin_bit_cast(f16x2v, pair);
  lo = __builtin_fmaf((float)q.x, s, b);
  hi = __builtin_fmaf((float)q.y, s, b);
}
__device__ __forceinline__ uint32_t cvt2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v){lo, hi}, bf16x2_t));
}

// the eight codes of a packed word as bf16(s * q + b); the conversions come
// last, away from the fmas they depend on (a hazard nop each otherwise)
__device__ __forceinline__ bf16x8_t dequant8(uint32_t w, const GroupScale& g) {
  const uint32_t m0 = 0x000F000Fu, m1 = 0x00F000F0u, wh = w >> 8;
  float lo[4], hi[4];
  mix2(w & m0, g.s0, g.b, lo[0], hi[0]);
  mix2(w & m1, g.s1, g.b, lo[1], hi[1]);
  mix2(wh & m0, g.s0, g.b, lo[2], hi[2]);
  mix2(wh & m1, g.s1, g.b, lo[3], hi[3]);
  return as_bf16x8(cvt2(lo[0], hi[0]), cvt2(lo[1], hi[1]), cvt2(lo[2], hi[2]), cvt2(lo[3], hi[3]));
}

// Workgroup -> (column group, row block): consecutive blocks of one XCD (the
// dispatch order is round-robin over 8) share a column group, so that its
// weights come from HBM once. Blocks past the last pair get column >= columns.
__device__ __forceinline__ void block_place(int row_blocks, int columns, int& column, int& row) {
  const int per = gridDim.x >> 3;
  const int at = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  column = at / row_blocks;
  row = at - column * row_blocks;
}

// Per-lane DMA sources of a block's activation rows and weight tiles.
template <int BM, int TPW, int NW>
struct Source {
  static constexpr int NLD = BM / 4 / NW;      // DMAs (4 rows each) per wave and stage
  static constexpr int ASZ = BM * 256;         // bytes of a stage's activations
  static constexpr int WSZ = NW * TPW * QG_WSLOT;
  static constexpr int PER_STAGE = NLD + 2 * TPW;
  const uint8_t* xb;
  const uint8_t* packed;
  uint32_t off, off_last, w_off, s_off, lds;
  int K, GS, tile0, tiles, last, h_last, wave;

  __device__ __forceinline__ void init(const uint16_t* x, const uint8_t* packed_, uint32_t lds_, int M, int K_,
                                       int m0, int tile0_, int tiles_, int wave_, int lane, int h_last_) {
    K = K_, GS = K / QG_SET, packed = packed_, lds = lds_, tile0 = tile0_, tiles = tiles_, wave = wave_;
    h_last = h_last_;
    const int c = lane >> 4, r4 = c, ch = (lane & 15) ^ row_swizzle(4 * wave + r4);
    const int lim = min(M - m0, BM) - 1;       // last row of the block; rows past it repeat rows of its group of 4
    last = lim & ~3;
    off = (uint32_t)(r4 * K + ch * 8) * 2u;
    off_last = (uint32_t)(min(r4, lim & 3) * K + ch * 8) * 2u;
    xb = reinterpret_cast<const uint8_t*>(x + (size_t)m0 * K);
    w_off = (c & 1) * 1024 + ((c >> 1) * 16 + (lane & 15)) * 16;
    s_off = ((c >> 1) * 16 + (lane & 15)) * 4;
  }
  // stages past the last re-read it: every stage issues the same number of DMAs
  __device__ __forceinline__ void activations(int h, uint32_t slot) const {
    const uint8_t* base = xb + (size_t)min(h, h_last) * 256;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int row = 4 * (wave + NW * i), g = min(row, last);
      dma16(lds + slot + row * 256, g == last ? off_last : off, base + (size_t)g * K * 2);
    }
  }
  // tiles past the end re-read the last one (their outputs are never stored)
  __device__ __forceinline__ void weights(int h, uint32_t slot) const {
    h = min(h, h_last);
#pragma unroll
    for (int p = 0; p < TPW; ++p) {
      const uint8_t* rec = packed + ((size_t)min(tile0 + p, tiles - 1) * GS + (h >> 1)) * QG_RECORD;
      const uint32_t to = lds + slot + (wave * TPW + p) * QG_WSLOT;
      dma16_nt(to, w_off, rec + (h & 1) * 512);
      dma4(to + 1024, s_off, rec + QG_WBYTES + (h & 1) * 128);
    }
  }
};

// Outputs of one 16 x 16 tile: lane (c, i) holds weight rows 4c .. 4c + 3 of
// activation row m. SWIGLU: interleaved tile, rows 0-7 gate rows 8 tile + i,
// rows 8-15 the matching up rows.
template <bool SWIGLU>
__device__ __forceinline__ void store_tile(uint16_t* __restrict__ y, f32x4_t v, int tile, int m, int c, int M, int N,
                                           bool vec) {
  if constexpr (SWIGLU) {
    const int half = N / 2, n = 8 * tile + 4 * c;
    float o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float u = __shfl_xor(v[r], 32, 64);
      const float gv = bf16_to_f32(f32_to_bf16(v[r])), uv = bf16_to_f32(f32_to_bf16(u));
      o[r] = gv / (1.0f + expf(-gv)) * uv;
    }
    if (c >= 2 || m >= M || n >= half) return;
    uint16_t* yp = y + (size_t)m * half + n;
    if (vec) {
      *reinterpret_cast<u32x2*>(yp) = u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) yp[r] = f32_to_bf16(o[r]);     // half is a multiple of 8
    }
  } else {
    const int n = tile * QG_TILE + 4 * c;
    if (m >= M || n >= N) return;
    uint16_t* yp = y + (size_t)m * N + n;
    if (vec) {
      *reinterpret_cast<u32x2*>(yp) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < N) yp[r] = f32_to_bf16(v[r]);
    }
  }
}

// The sums of one tile and 16 activation rows again, without the scaled scales: the
// same weights and the same order, so the same bits wherever those do not overflow.
__device__ __forceinline__ f32x4_t plain_tile(const uint16_t* __restrict__ x, const uint8_t* __restrict__ packed,
                                              int tile, int row, int K, int h_last) {
  const int lane = threadIdx.x & 63, c = lane >> 4, i16 = lane & 15;
  const uint16_t* xr = x + (size_t)row * K + 32 * c;
  const uint8_t* rec = packed + (size_t)tile * (K / QG_SET) * QG_RECORD;
  f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
  for (int h = 0; h <= h_last; ++h) {
    const uint8_t* r = rec + (size_t)(h >> 1) * QG_RECORD;
    const u32x4 w = load16(r + (h & 1) * 512 + (c & 1) * 1024 + ((c >> 1) * 16 + i16) * 16);
    const uint32_t sb = *reinterpret_cast<const uint32_t*>(r + QG_WBYTES + (h & 1) * 128 + ((c >> 1) * 16 + i16) * 4);
    const float s = bf16_lo(sb), b = bf16_hi(sb);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = cvt2(fmaf((float)(w[j] >> (4 * e) & 15u), s, b), fmaf((float)(w[j] >> (4 * e + 16) & 15u), s, b));
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v[0], v[1], v[2], v[3]),
                                                    __builtin_bit_cast(bf16x8_t, load16(xr + 128 * h + 8 * j)), acc, 0,
                                                    0, 0);
    }
  }
  return acc;
}

// v * 0 added: NaN from the first infinity or NaN on
__device__ __forceinline__ void note_overflow(float& seen, f32x4_t v) {
#pragma unroll
  for (int r = 0; r < 4; ++r) seen = fmaf(v[r], 0.0f, seen);
}

// ---------------------------------------------------------------- 65 rows and more
//
// A block of NW waves owns 16 MT rows x 16 TPW NW outputs, wave w the weight
// tiles TPW w .. of all its rows (so that each weight is dequantized by one
// wave per row block). Within a step the MFMAs run tile by tile; meanwhile the
// previous tile's next operand is dequantized and, in the last tile's pass, each
// activation fragment is replaced by the next step's as soon as its product is
// issued (sched_group_barrier: one MFMA, then two or three VALU instructions).
// The barrier stands before a stage's last step, so that the next stage's
// first fragments are read behind that step's products. AD, WD: ring depths.
template <int MT, int TPW, int NW, int AD, int WD, int PER_CU, bool SWIGLU>
__global__ __launch_bounds__(64 * NW, PER_CU) void packed_gemm_kernel(const uint16_t* __restrict__ x,
                                                                      const uint8_t* __restrict__ packed,
                                                                      uint16_t* __restrict__ y, int M, int N, int K,
                                                                      int vec) {
  constexpr int BM = MT * 16;
  typedef Source<BM, TPW, NW> Src;
  constexpr int ASZ = Src::ASZ, WSZ = Src::WSZ;
  // DMAs issued after the stage that arrive() waits for: stage h + 1's weights
  // go out WD stages ahead, its activations AD >= WD stages ahead
  constexpr int AHEAD = (WD - 2) * Src::PER_STAGE + (AD > WD ? Src::NLD : 0);
  static_assert(BM / 4 % NW == 0 && AD >= WD && WD >= 2, "ring");
  __shared__ __align__(1024) uint8_t lds[AD * ASZ + WD * WSZ];
  const int lane = threadIdx.x & 63, c = lane >> 4, i16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = (N + QG_TILE - 1) / QG_TILE;
  const int columns = (tiles + TPW * NW - 1) / (TPW * NW);
  int column, row;
  block_place((M + BM - 1) / BM, columns, column, row);
  if (column >= columns) return;
  const int m0 = row * BM, tile0 = (column * NW + wave) * TPW;
  const int h_last = 2 * (K / QG_SET) - 1;
  Src src;
  src.init(x, packed, lds_offset(lds), M, K, m0, tile0, tiles, wave,
           lane, h_last);

  f32x4_t acc[MT][TPW];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int p = 0; p < TPW; ++p) acc[mt][p] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  int a_off[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) a_off[j] = i16 * 256 + ((4 * c + j) ^ row_swizzle(i16)) * 16;

  u32x4 wc[TPW], wn[TPW];      // the current and the next stage's words
  uint32_t sn[TPW];
  GroupScale g[TPW];
  auto read_words = [&](u32x4* w, int slot) __attribute__((always_inline)) {
    const uint8_t* from = lds + AD * ASZ + slot * WSZ + wave * TPW * QG_WSLOT;
#pragma unroll
    for (int p = 0; p < TPW; ++p) {
      w[p] = load16(from + p * QG_WSLOT + lane * 16);
      sn[p] = *reinterpret_cast<const uint32_t*>(from + p * QG_WSLOT + 1024 + lane * 4);
    }
  };
  auto read_a = [&](int slot, int j, int mt) __attribute__((always_inline)) {
    return __builtin_bit_cast(bf16x8_t, load16(lds + slot * ASZ + a_off[j] + mt * 4096));
  };
  bf16x8_t a[MT], b[TPW];
  auto step = [&](const u32x4* w, int j, const u32x4* w_next, int j_next, int slot, bool new_stage)
      __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < TPW; ++p) {
      if (TPW > 1 && p == 0) b[TPW - 1] = dequant8(w[TPW - 1][j], g[TPW - 1]);
      if (p > 0) {
        if (new_stage) g[p - 1].set(sn[p - 1]);
        b[p - 1] = dequant8(w_next[p - 1][j_next], g[p - 1]);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        acc[mt][p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[p], a[mt], acc[mt][p], 0, 0, 0);
        if (p == TPW - 1) a[mt] = read_a(slot, j_next, mt);
      }
      if (p == TPW - 1 && new_stage) g[p].set(sn[p]);
      if (TPW == 1) b[0] = dequant8(w_next[0][j_next], g[0]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                      // MFMA
        __builtin_amdgcn_sched_group_barrier(0x2, (17 + MT - 1) / MT, 0);     // VALU
        if (p == TPW - 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

#pragma unroll
  for (int k = 0; k < AD; ++k) {
    if (k - AD + WD >= 0) src.weights(k - AD + WD, AD * ASZ + (k - AD + WD) * WSZ);
    src.activations(k, k * ASZ);
  }
  arrive<AHEAD>();
  read_words(wc, 0);
#pragma unroll
  for (int p = 0; p < TPW; ++p) g[p].set(sn[p]);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) a[mt] = read_a(0, 0, mt);
#pragma unroll
  for (int p = 0; p < (TPW > 1 ? TPW - 1 : 1); ++p) b[p] = dequant8(wc[p][0], g[p]);
  __builtin_amdgcn_sched_barrier(0);
  int as = 0, ws = 0;          // ring slots of the current stage
#pragma unroll 1
  for (int h = 0; h <= h_last; ++h) {
    step(wc, 0, wc, 1, as, false);
    step(wc, 1, wc, 2, as, false);
    step(wc, 2, wc, 3, as, false);
    // stage h + 1 has landed, and every wave has read all of stage h
    arrive<AHEAD>();
    const int an = as + 1 == AD ? 0 : as + 1, wsn = ws + 1 == WD ? 0 : ws + 1;
    read_words(wn, wsn);
    src.weights(h + WD, AD * ASZ + ws * WSZ);
    src.activations(h + AD, as * ASZ);
    __builtin_amdgcn_sched_barrier(0);
    step(wc, 3, wn, 0, an, true);
#pragma unroll
    for (int p = 0; p < TPW; ++p) wc[p] = wn[p];
    as = an;
    ws = wsn;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the LDS is given back with no DMA in flight

  float seen = 0.0f;
#pragma unroll
  for (int p = 0; p < TPW; ++p)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) note_overflow(seen, acc[mt][p]);
  if (__any(seen != 0.0f)) {
#pragma unroll 1
    for (int e = 0; e < TPW * MT; ++e) {
      const int tile = tile0 + e / MT, m = m0 + 16 * (e % MT) + i16;
      if (tile >= tiles) break;
      store_tile<SWIGLU>(y, plain_tile(x, packed, tile, min(m, M - 1), K, h_last), tile, m, c, M, N, vec);
    }
    return;
  }
#pragma unroll
  for (int p = 0; p < TPW; ++p) {
    if (tile0 + p >= tiles) continue;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) store_tile<SWIGLU>(y, acc[mt][p], tile0 + p, m0 + 16 * mt + i16, c, M, N, vec);
  }
}

// ---------------------------------------------------------------- up to 64 rows
//
// One weight tile per wave, 4 waves, all rows in one block: few MFMAs, so a
// wave's time is its chain of waits. A whole stage's fragments (4 MT) and words
// are read behind the products of the stage before, one round trip to LDS per
// stage, and the rings are as deep as two blocks per CU allow.
template <int MT, bool SWIGLU>
__global__ __launch_bounds__(256, 2) void packed_gemm_small_kernel(const uint16_t* __restrict__ x,
                                                                   const uint8_t* __restrict__ packed,
                                                                   uint16_t* __restrict__ y, int M, int N, int K,
                                                                   int vec) {
  constexpr int NW = 4, BM = MT * 16;
  typedef Source<BM, 1, NW> Src;
  constexpr int STAGE = Src::ASZ + Src::WSZ;
  constexpr int D = 81920 / STAGE > 8 ? 8 : 81920 / STAGE;
  constexpr int AHEAD = (D - 2) * Src::PER_STAGE;
  static_assert(D >= 3 && BM / 4 % NW == 0, "ring");
  __shared__ __align__(1024) uint8_t lds[D * STAGE];
  const int lane = threadIdx.x & 63, c = lane >> 4, i16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = (N + QG_TILE - 1) / QG_TILE;
  const int tile = blockIdx.x * NW + wave;
  const int h_last = 2 * (K / QG_SET) - 1;
  Src src;
  src.init(x, packed, lds_offset(lds), M, K, 0, tile, tiles, wave,
           lane, h_last);
  f32x4_t acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  int a_off[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) a_off[j] = i16 * 256 + ((4 * c + j) ^ row_swizzle(i16)) * 16;

  struct Frags {
    bf16x8_t a[4][MT];
    u32x4 w;
    uint32_t sb;
  };
  auto read = [&](Frags& f, int slot) __attribute__((always_inline)) {
    const uint8_t* from = lds + slot * STAGE;
    f.w = load16(from + Src::ASZ + wave * QG_WSLOT + lane * 16);
    f.sb = *reinterpret_cast<const uint32_t*>(from + Src::ASZ + wave * QG_WSLOT + 1024 + lane * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) f.a[j][mt] = __builtin_bit_cast(bf16x8_t, load16(from + a_off[j] + mt * 4096));
  };
  auto products = [&](const Frags& f) __attribute__((always_inline)) {
    GroupScale g;
    g.set(f.sb);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bf16x8_t b = dequant8(f.w[j], g);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, f.a[j][mt], acc[mt], 0, 0, 0);
    }
  };
#pragma unroll
  for (int k = 0; k < D; ++k) {
    src.weights(k, k * STAGE + Src::ASZ);
    src.activations(k, k * STAGE);
  }
  Frags f0, f1;
  arrive<AHEAD + Src::PER_STAGE>();
  read(f0, 0);
  // Stage h's slot is refilled once every wave has read it: by the barrier in
  // stage h, which also waits for stage h + 1.
  int slot = 0;
  auto stage = [&](int h, const Frags& cur, Frags& next) __attribute__((always_inline)) {
    arrive<AHEAD>();
    const int sn = slot + 1 == D ? 0 : slot + 1;
    read(next, sn);
    src.weights(h + D, slot * STAGE + Src::ASZ);
    src.activations(h + D, slot * STAGE);
    __builtin_amdgcn_sched_barrier(0);
    products(cur);
    __builtin_amdgcn_sched_barrier(0);
    slot = sn;
  };
#pragma unroll 1
  for (int h = 0; h <= h_last; h += 2) {       // two stages per set
    stage(h, f0, f1);
    stage(h + 1, f1, f0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (tile >= tiles) return;
  float seen = 0.0f;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) note_overflow(seen, acc[mt]);
  if (__any(seen != 0.0f)) {
#pragma unroll 1
    for (int mt = 0; mt < MT; ++mt)
      store_tile<SWIGLU>(y, plain_tile(x, packed, tile, min(16 * mt + i16, M - 1), K, h_last), tile, 16 * mt + i16, c,
                         M, N, vec);
    return;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) store_tile<SWIGLU>(y, acc[mt], tile, 16 * mt + i16, c, M, N, vec);
}

// ---------------------------------------------------------------- launch

typedef void (*gemm_fn)(const uint16_t*, const uint8_t*, uint16_t*, int, int, int, int);

// The block shapes of packed_gemm_kernel, and what one round of blocks (as many
// as the chip holds) takes relative to the others. Measured, K = 4096: 128 rows x
// 384 outputs 97 us a round of 256, x 256 65 us, x 128 38 us, and 64 rows x 64
// outputs 28 us a round of 512 (20 us for 256 or fewer; 128 x 64 took 29 us a round of
// 256, never less than the 64 x 64 blocks of the same outputs).
struct GemmShape {
  int rows, tiles;       // per block
  int threads;
  int round;             // blocks in one round
  float cost, cost_half; // of a round, and of one at most half full
  gemm_fn fn[2];         // plain, SwiGLU
};
#define GEMM_SHAPE(MT, TPW, NW, AD, WD, PER_CU, COST, HALF)                        \
  {16 * MT, TPW * NW, 64 * NW, 256 * PER_CU, COST, HALF,                           \
   {packed_gemm_kernel<MT, TPW, NW, AD, WD, PER_CU, false>, packed_gemm_kernel<MT, TPW, NW, AD, WD, PER_CU, true>}}
const GemmShape kShapes[] = {
    GEMM_SHAPE(8, 3, 8, 3, 2, 1, 97.0f, 80.0f), GEMM_SHAPE(8, 2, 8, 3, 3, 1, 65.0f, 58.0f),
    GEMM_SHAPE(8, 1, 8, 3, 3, 1, 38.0f, 37.0f), GEMM_SHAPE(4, 1, 4, 3, 3, 2, 28.0f, 20.0f),
};

// The shape whose rounds cost least: tall tiles of many outputs move the fewest
// activation bytes per product, but leave the last round (or the only one) with
// idle CUs.
const GemmShape* pick_shape(int M, int tiles, long* blocks) {
  const GemmShape* best = nullptr;
  float best_cost = 0.0f;
  for (const GemmShape& s : kShapes) {
    const long b = (long)((M + s.rows - 1) / s.rows) * ((tiles + s.tiles - 1) / s.tiles);
    const long full = b / s.round, rest = b - full * s.round;
    const float cost = full * s.cost + (rest == 0 ? 0.0f : 2 * rest <= s.round ? s.cost_half : s.cost);
    if (best == nullptr || cost < best_cost) {
      best = &s;
      best_cost = cost;
      *blocks = b;
    }
  }
  return best;
}

constexpr int QG_SMALL_ROWS = 64;

gemm_fn small_kernel(int M, bool swiglu) {
  switch ((M + 15) / 16) {
    case 1: return swiglu ? packed_gemm_small_kernel<1, true> : packed_gemm_small_kernel<1, false>;
    case 2: return swiglu ? packed_gemm_small_kernel<2, true> : packed_gemm_small_kernel<2, false>;
    case 3: return swiglu ? packed_gemm_small_kernel<3, true> : packed_gemm_small_kernel<3, false>;
    default: return swiglu ? packed_gemm_small_kernel<4, true> : packed_gemm_small_kernel<4, false>;
  }
}

int launch_gemm(const uint16_t* x, const void* packed, uint16_t* y, int M, int N, int K, bool swiglu,
                void* stream, const char* name) {
  QVEX_CHECK_ARG(x && packed && y, "%s: null pointer", name);
  QVEX_CHECK_ARG(M >= 1 && N >= 1 && K >= QG_SET && K % QG_SET == 0, "%s: M=%d N=%d K=%d (K a multiple of 256)",
                 name, M, N, K);
  QVEX_CHECK_ARG(!swiglu || N % 16 == 0, "%s: N=%d must be a multiple of 16 for the gate/up interleave", name, N);
  QVEX_CHECK_ARG(qvex_aligned(x, 16) && qvex_aligned(packed, 16), "%s: x and packed must be 16-byte aligned", name);
  QVEX_CHECK_ARG((M + 63) / 64 <= 65535, "%s: M=%d too large", name, M);
  const int tiles = (N + QG_TILE - 1) / QG_TILE;
  const int vec = qvex_aligned(y, 8) && (swiglu || N % 4 == 0);     // 8-byte stores
  gemm_fn fn;
  unsigned grid, threads;
  if (M <= QG_SMALL_ROWS) {
    fn = small_kernel(M, swiglu);
    grid = (tiles + 3) / 4;
    threads = 256;
  } else {
    long blocks;
    const GemmShape* s = pick_shape(M, tiles, &blocks);
    QVEX_CHECK_ARG(blocks <= (1L << 30), "%s: M=%d N=%d too large", name, M, N);
    fn = s->fn[swiglu];
    grid = (unsigned)((blocks + 7) / 8 * 8);      // block_place: 8 equal runs
    threads = s->threads;
  }
  hipLaunchKernelGGL(fn, dim3(grid), dim3(threads), 0, (hipStream_t)stream, x, (const uint8_t*)packed, y, M, N, K, vec);
  QVEX_CHECK_LAUNCH(name);
  return QVEX_OK;
}

}  // namespace

extern "C" int qvex_w4g64_packed_gemm(const uint16_t* x, const void* packed, uint16_t* y, int M, int N, int K,
                                      void* stream) {
  return launch_gemm(x, packed, y, M, N, K, false, stream, "qvex_w4g64_packed_gemm");
}

extern "C" int qvex_w4g64_packed_gemm_swiglu(const uint16_t* x, const void* packed, uint16_t* y, int M, int N,
                                             int K, void* stream) {
  return launch_gemm(x, packed, y, M, N, K, true, stream, "qvex_w4g64_packed_gemm_swiglu");
}
