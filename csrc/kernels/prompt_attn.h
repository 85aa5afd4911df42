// Attention of several query rows per sequence over a bf16 cache (prompt_attn.hip), called by decode_attn.
#pragma once
#include "common.h"
#include <algorithm>
#include <type_traits>

namespace penroz {

// whether it is faster than decode_kernel for Tq query rows per sequence at the given number of keys
bool prompt_attn_applies(int64_t B, int64_t Tq, int64_t H, int64_t Hkv, int64_t D, int64_t keys);

// parts that the keys are split into for `rows` query rows (tokens x heads of a group) of each of `items` KV heads;
// part_keys: keys of a part, 0 for the measured number
int prompt_attn_splits(int64_t items, int64_t rows, int64_t keys, int D, int part_keys);

// D 64, 128, 256 or 512; q rows of stride q_rs (16-byte aligned), caches [B, Hkv, cap, D], out [B, Tq, H, D]; with
// splits > 1 the parts go to ws_o [splits, B, Tq, H, D] and ws_ml [.., 2] (maximum in powers of two, sum)
void prompt_attn_launch(const bf16* q, const bf16* kc, const bf16* vc, bf16* out, float* ws_o, float* ws_ml, int B,
                        int Tq, int H, int Hkv, int D, int cap, int q_offset, int splits, float scale, int64_t q_rs,
                        hipStream_t stream);

}  // namespace penroz
