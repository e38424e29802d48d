// The prompt-chunk path of qvex_attention (attn_prefill.hip).
#pragma once
#include <stdint.h>

namespace qvex {

constexpr int ATT_PROMPT_ROWS = 9;     // positions of a call from which the path is taken
// Keys after which a row's sums start afresh (fewer if keys_per_split is): one
// length for every call, so that a row's bits depend on no other. us for 512 positions
// at 0 | 1024 | 4096 | 16384 keys, 16 query and 4 kv heads of 256: units of 128 24 | 45 | 107 | 384,
// 256 25 | 46 | 90 | 260, 512 32 | 41 | 99 | 365; 16 positions at 256 | 1024 | 4096: 13 | 14 | 19,
// 17 | 17 | 20, 18 | 25 | 31.
constexpr int ATT_UNIT = 256;
constexpr int ATT_GROUP = 4;           // units in a group
constexpr int ATT_BLOCK_TILES = 4;     // 16-row tiles per block, one per wave

// Blocks up to which each takes one unit: two rounds of what the chip holds (2 per CU
// by LDS and registers, 4 for D = 128); more take a group each. us, unit | group, at
// 780 blocks 53 | 59, 1024 47 | 63, 1040 62 | 62, 1088 67 | 58, 1560 83 | 71; D = 128 at
// 1152 39 | 43, 4224 93 | 76.
constexpr long att_unit_blocks(int D) { return D == 256 ? 1024 : 2048; }

// Units that a block takes (and a record holds) in a call of `units` units of keys.
constexpr int attention_units(int Hkv, int ntile, int D, int units) {
  const long blocks = (long)Hkv * ((ntile + ATT_BLOCK_TILES - 1) / ATT_BLOCK_TILES) * units;
  return blocks <= att_unit_blocks(D) ? 1 : units < ATT_GROUP ? units : ATT_GROUP;
}

// Launches both kernels on arguments that qvex_attention has checked (D 128 or 256):
// nsplit blocks along the keys, each of `units` units of `unit` keys.
void attention_prefill(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, const int32_t* pos0, int L,
                       int Hq, int Hkv, int D, int cap, int ntile, int nsplit, int QT, int unit, int units,
                       float scale, const uint16_t* gate, long gate_stride, uint16_t* out, float* ws, void* stream);

}  // namespace qvex
