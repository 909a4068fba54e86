// Instantiates the channels-last DK kernels ([B, L, H] tensors, [K, H] dw).
#include "dwconv1d_kernels.hpp"
#include "dwconv1d_tables.hpp"

namespace pt {
// [deterministic][row bucket]: 16 waves of two channels for rows up to 32
// columns, 8 waves of four channels with two steps of loads in registers for 48.
const DkClFn kDkClTable[2][3] = {{&dwconv_dk_cl_kernel<16, kCgChannelsPerWave, 1, false>,
                                  &dwconv_dk_cl_kernel<32, kCgChannelsPerWave, 1, false>,
                                  &dwconv_dk_cl_kernel<48, kClWideChannels, 2, false>},
                                 {&dwconv_dk_cl_kernel<16, kCgChannelsPerWave, 1, true>,
                                  &dwconv_dk_cl_kernel<32, kCgChannelsPerWave, 1, true>,
                                  &dwconv_dk_cl_kernel<48, kClWideChannels, 2, true>}};
}  // namespace pt
