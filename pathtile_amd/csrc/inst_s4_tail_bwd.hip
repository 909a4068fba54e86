// Instantiates the S4ConvD tail's bwd kernels.
#include "s4_kernels.hpp"
#include "s4_tables.hpp"

namespace pt {
const TailBwdFn kTailBwd[2][kNumS4H] = {
    {&s4_tail_bwd_kernel<2, false>, &s4_tail_bwd_kernel<4, false>, &s4_tail_bwd_kernel<6, false>,
     &s4_tail_bwd_kernel<8, false>, &s4_tail_bwd_kernel<10, false>, &s4_tail_bwd_kernel<12, false>,
     &s4_tail_bwd_kernel<14, false>, &s4_tail_bwd_kernel<16, false>},
    {&s4_tail_bwd_kernel<2, true>, &s4_tail_bwd_kernel<4, true>, &s4_tail_bwd_kernel<6, true>,
     &s4_tail_bwd_kernel<8, true>, &s4_tail_bwd_kernel<10, true>, &s4_tail_bwd_kernel<12, true>,
     &s4_tail_bwd_kernel<14, true>, &s4_tail_bwd_kernel<16, true>}};
}  // namespace pt
