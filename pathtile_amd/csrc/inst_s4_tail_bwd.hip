// Instantiates the S4ConvD tail's bwd kernels.
#include "s4_kernels.hpp"
#include "s4_tables.hpp"

namespace pt {
const TailBwdFn kTailBwd[kNumS4H] = {
    &s4_tail_bwd_kernel<2>,  &s4_tail_bwd_kernel<4>,  &s4_tail_bwd_kernel<6>,
    &s4_tail_bwd_kernel<8>,  &s4_tail_bwd_kernel<10>, &s4_tail_bwd_kernel<12>,
    &s4_tail_bwd_kernel<14>, &s4_tail_bwd_kernel<16>};
}  // namespace pt
