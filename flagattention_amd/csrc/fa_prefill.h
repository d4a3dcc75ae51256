// The many-row attention kernel (fa_prefill.hip) behind fa_gqa_decode.
#pragma once

#include "fa_common.h"

namespace fa {

constexpr int kPrefillRows = 128;    // query rows per work-group
constexpr int kPrefillMinRows = 16;  // up to these rows per KV head the 16-row kernel reads K/V once too

// Whether launch_prefill runs this (already checked) call.
bool prefill_takes(const fa_gqa_decode_args* a);
int launch_prefill(const fa_gqa_decode_args* a, void* stream);

}  // namespace fa
