// The prompt-chunk path of qvex_attention (attn_prefill.hip).
#pragma once
#include <stdint.h>

namespace qvex {

// Tiles of 16 rows (as qvex_attention's workspace has them) from which the path
// is taken: three blocks of 128 rows. us, one block per tile | 128-row blocks, 16
// query and 4 kv heads of 256: 32 positions at 4096 keys 20 | 26, 64 at 4096 30 | 32,
// 128 at 0 18 | 17, 128 at 4096 49 | 37.
constexpr int ATT_PREFILL_TILES = 24;

// Launches both kernels on arguments that qvex_attention has checked (D 128 or 256).
void attention_prefill(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, const int32_t* pos0, int L,
                       int Hq, int Hkv, int D, int cap, int ntile, int nsplit, int QT, int keys_per_split, float scale,
                       const uint16_t* gate, long gate_stride, uint16_t* out, float* ws, void* stream);

}  // namespace qvex
