// Instantiates the S4ConvD tail's fwd kernels.
#include "s4_kernels.hpp"
#include "s4_tables.hpp"

namespace pt {
const TailFwdFn kTailFwd[kNumS4H] = {
    &s4_tail_fwd_kernel<2>,  &s4_tail_fwd_kernel<4>,  &s4_tail_fwd_kernel<6>,
    &s4_tail_fwd_kernel<8>,  &s4_tail_fwd_kernel<10>, &s4_tail_fwd_kernel<12>,
    &s4_tail_fwd_kernel<14>, &s4_tail_fwd_kernel<16>};
}  // namespace pt
