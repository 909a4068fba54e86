// Instantiates the one-pass backward for BF16 tensors by row bucket 16, 32, 48.
#include "dwconv1d_bwd.hpp"
#include "dwconv1d_tables.hpp"

namespace pt {
// [non-temporal loads][row bucket]
const BwdBf16Fn kBwdBf16[2][3] = {
    {&dwconv_bwd_bf16_kernel<16, kCpolNone>, &dwconv_bwd_bf16_kernel<32, kCpolNone>,
     &dwconv_bwd_bf16_kernel<48, kCpolNone>},
    {&dwconv_bwd_bf16_kernel<16, kCpolNT>, &dwconv_bwd_bf16_kernel<32, kCpolNT>,
     &dwconv_bwd_bf16_kernel<48, kCpolNT>}};
}  // namespace pt
