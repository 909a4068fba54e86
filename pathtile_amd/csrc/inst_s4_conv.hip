// Instantiates the [B, L, H] convolution by row bucket 8, 16, ..., 48.
#include "s4_conv.hpp"
#include "s4_tables.hpp"

namespace pt {
const ConvClFn kConvCl[5][6] = {
    {&s4_conv_cl_kernel<8, false, false, false>, &s4_conv_cl_kernel<16, false, false, false>,
     &s4_conv_cl_kernel<24, false, false, false>, &s4_conv_cl_kernel<32, false, false, false>,
     &s4_conv_cl_kernel<40, false, false, false>, &s4_conv_cl_kernel<48, false, false, false>},
    {&s4_conv_cl_kernel<8, true, false, false>, &s4_conv_cl_kernel<16, true, false, false>,
     &s4_conv_cl_kernel<24, true, false, false>, &s4_conv_cl_kernel<32, true, false, false>,
     &s4_conv_cl_kernel<40, true, false, false>, &s4_conv_cl_kernel<48, true, false, false>},
    {&s4_conv_cl_kernel<8, false, true, false>, &s4_conv_cl_kernel<16, false, true, false>,
     &s4_conv_cl_kernel<24, false, true, false>, &s4_conv_cl_kernel<32, false, true, false>,
     &s4_conv_cl_kernel<40, false, true, false>, &s4_conv_cl_kernel<48, false, true, false>},
    {&s4_conv_cl_kernel<8, false, false, true>, &s4_conv_cl_kernel<16, false, false, true>,
     &s4_conv_cl_kernel<24, false, false, true>, &s4_conv_cl_kernel<32, false, false, true>,
     &s4_conv_cl_kernel<40, false, false, true>, &s4_conv_cl_kernel<48, false, false, true>},
    {&s4_conv_cl_kernel<8, false, true, true>, &s4_conv_cl_kernel<16, false, true, true>,
     &s4_conv_cl_kernel<24, false, true, true>, &s4_conv_cl_kernel<32, false, true, true>,
     &s4_conv_cl_kernel<40, false, true, true>, &s4_conv_cl_kernel<48, false, true, true>}};
}  // namespace pt
