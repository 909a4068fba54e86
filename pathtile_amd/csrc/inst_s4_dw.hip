// Instantiates the S4ConvD projection's weight gradient.
#include "s4_kernels.hpp"
#include "s4_tables.hpp"

namespace pt {
const DwFn kDw[kNumS4H] = {&s4_dw_kernel<2>,  &s4_dw_kernel<4>,  &s4_dw_kernel<6>,
                           &s4_dw_kernel<8>,  &s4_dw_kernel<10>, &s4_dw_kernel<12>,
                           &s4_dw_kernel<14>, &s4_dw_kernel<16>};
}  // namespace pt
