// Instantiates the S4ConvD projection's weight gradient.
#include "s4_kernels.hpp"
#include "s4_tables.hpp"

namespace pt {
const DwFn kDw[kNumS4H][2] = {
    {&s4_dw_kernel<2, false>, &s4_dw_kernel<2, true>},
    {&s4_dw_kernel<4, false>, &s4_dw_kernel<4, true>},
    {&s4_dw_kernel<6, false>, &s4_dw_kernel<6, true>},
    {&s4_dw_kernel<8, false>, &s4_dw_kernel<8, true>},
    {&s4_dw_kernel<10, false>, &s4_dw_kernel<10, true>},
    {&s4_dw_kernel<12, false>, &s4_dw_kernel<12, true>},
    {&s4_dw_kernel<14, false>, &s4_dw_kernel<14, true>},
    {&s4_dw_kernel<16, false>, &s4_dw_kernel<16, true>}};
}  // namespace pt
