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

// Channels-last DK of dwconv1d_kernels.hpp: its sample ranges on the current
// device (0: not served), and the deterministic form, dk [H, K] from
// H * K * nranges floats of partials (B > 0, H % 32 == 0, 16-byte aligned).
int dk_cl_ranges(int B, int H, int L);
int dk_cl_det(const float* x, const float* dy, float* dk, float* partials, int B, int H, int L,
              int K, int nranges, void* stream);

}  // namespace pt
