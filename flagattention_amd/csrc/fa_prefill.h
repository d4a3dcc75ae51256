// The many-row attention kernel (fa_prefill.hip) behind fa_gqa_decode.
#pragma once

#include "fa_common.h"

namespace fa {

constexpr int kPrefillRows = 128;    // query rows per work-group
constexpr int kPrefillMinRows = 16;  // up to these rows per KV head the 16-row kernel reads K/V once too

// Up to 256 keys the 16-row kernel's four waves take 128 keys side by side and need two turns
// at most, where a work-group here walks 64 (32 at head dim 256) at a time.  That is faster at
// head dim 64 past one tile while its work-groups run all at once (256 CUs): 8 KV heads x 64
// rows, 97 / 256 keys 5.5 / 6.2 us against 6.1 / 7.7; of 578 shapes 517 by 2% to 29%, 21 slower.
// At 128 and 256, whose products weigh more, only past 192 keys with a few work-groups (64
// shapes each, 193 .. 256 keys: 0.79 .. 1.04 of the time here).
constexpr int kFewKeysMax = 256;
constexpr int few_keys_min(int d) { return d == 64 ? 64 : 192; }
constexpr int few_keys_wgs(int d) { return d == 64 ? 256 : 16; }

// Whether launch_prefill runs this (already checked) call.
bool prefill_takes(const fa_gqa_decode_args* a);
int launch_prefill(const fa_gqa_decode_args* a, void* stream);

}  // namespace fa
