// Instantiates the one-pass backward by row bucket 16, 32, 48.
#include "dwconv1d_bwd.hpp"
#include "dwconv1d_tables.hpp"

namespace pt {
// [non-temporal loads][whole float4 rows][row bucket]
const BwdCgFn kBwdCg[2][2][3] = {
    {{&dwconv_bwd_cg_kernel<16, kCpolNone, false>, &dwconv_bwd_cg_kernel<32, kCpolNone, false>,
      &dwconv_bwd_cg_kernel<48, kCpolNone, false>},
     {&dwconv_bwd_cg_kernel<16, kCpolNone, true>, &dwconv_bwd_cg_kernel<32, kCpolNone, true>,
      &dwconv_bwd_cg_kernel<48, kCpolNone, true>}},
    {{&dwconv_bwd_cg_kernel<16, kCpolNT, false>, &dwconv_bwd_cg_kernel<32, kCpolNT, false>,
      &dwconv_bwd_cg_kernel<48, kCpolNT, false>},
     {&dwconv_bwd_cg_kernel<16, kCpolNT, true>, &dwconv_bwd_cg_kernel<32, kCpolNT, true>,
      &dwconv_bwd_cg_kernel<48, kCpolNT, true>}}};
}  // namespace pt
