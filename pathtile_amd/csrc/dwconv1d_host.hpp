// dwconv1d_host.hpp — host helpers of dwconv1d_abi.hip that other translation
// units launch through.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace pt {

// Launches `fn` on `stream`; PT_OK or PT_ERR_HIP (the error is consumed).
int launch(const void* fn, uint32_t grid, uint32_t block, size_t lds, void* stream, void** args);
// Compute units of the current device.
int num_cus();
// Resident workgroups per CU for (kernel, block size, dynamic LDS), at least 1.
int blocks_per_cu(const void* fn, int block, size_t lds);

}  // namespace pt
