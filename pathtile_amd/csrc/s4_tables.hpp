// s4_tables.hpp — dispatch tables of the S4ConvD block's kernels by H / 32 - 1,
// each defined in its own translation unit (inst_s4_*.hip).
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace pt {

constexpr int kNumS4H = 8;  // H = 32, 64, ..., 256

using ConvClFn = void (*)(const float*, const float*, const float*, const uint8_t*, float, float*,
                          float*, int, int, int);
using TailFwdFn = void (*)(const float*, const float*, const __bf16*, const float*, const float*,
                           float*, float*, uint32_t, uint32_t);
using TailBwdFn = void (*)(const float*, const float*, const float*, const uint8_t*, float,
                           const __bf16*, const float*, float*, float*, uint32_t, uint32_t, uint32_t,
                           uint32_t);
using DwFn = void (*)(const float*, const float*, float*, uint32_t, uint32_t, uint32_t);

// [forward, dx, forward with mask, with copy, with both][row bucket 8, ..., 48]
extern const ConvClFn kConvCl[5][6];
extern const TailFwdFn kTailFwd[kNumS4H];
extern const TailBwdFn kTailBwd[2][kNumS4H];  // [dropout mask]
extern const DwFn kDw[kNumS4H];

}  // namespace pt
