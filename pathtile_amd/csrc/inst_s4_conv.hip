// Instantiates the [B, L, H] convolution by row bucket 8, 16, ..., 48.
#include "s4_conv.hpp"
#include "s4_tables.hpp"

namespace pt {
const ConvClFn kConvCl[3][6] = {
    {&s4_conv_cl_kernel<8, false, false>, &s4_conv_cl_kernel<16, false, false>,
     &s4_conv_cl_kernel<24, false, false>, &s4_conv_cl_kernel<32, false, false>,
     &s4_conv_cl_kernel<40, false, false>, &s4_conv_cl_kernel<48, false, false>},
    {&s4_conv_cl_kernel<8, true, false>, &s4_conv_cl_kernel<16, true, false>,
     &s4_conv_cl_kernel<24, true, false>, &s4_conv_cl_kernel<32, true, false>,
     &s4_conv_cl_kernel<40, true, false>, &s4_conv_cl_kernel<48, true, false>},
    {&s4_conv_cl_kernel<8, false, true>, &s4_conv_cl_kernel<16, false, true>,
     &s4_conv_cl_kernel<24, false, true>, &s4_conv_cl_kernel<32, false, true>,
     &s4_conv_cl_kernel<40, false, true>, &s4_conv_cl_kernel<48, false, true>}};
}  // namespace pt
