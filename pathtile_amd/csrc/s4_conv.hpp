// s4_conv.hpp — the depthwise convolution on [B, L, H] tensors, for the
// S4ConvD block, which keeps its activations in that layout.
#pragma once

#include "dwconv1d_kernels.hpp"

namespace pt {

constexpr int kConvClThreads = 256;

// Threads of a workgroup: whole samples' channels, at most kConvClThreads.
__host__ __device__ constexpr int conv_cl_threads(int H) {
  return H >= kConvClThreads ? H : kConvClThreads / H * H;
}

// FWD y[b,t,h] = sum_j w[h][j] x[b, t + j - L / 2, h], DX the transposed sum
// plus `add` [B, L, H], for H channels in the last dimension and K = L taps.
// A lane owns one channel: its taps stay in registers over a persistent walk
// of samples, the L values of a sample load as whole lines of consecutive
// channels, and the outputs leave the same way, so nothing passes through
// LDS; the [B, H, L] kernels would need a transpose on each side (142 and
// 210 us at B16384 L48 H128 beside their own 140 us). Each output is the
// reference's fmaf chain in its tap order (FWD j ascending, DX j ascending,
// that is from the largest column down), four outputs as independent chains.
// The unrolled window of LMAX columns has zero taps beyond the call's K;
// where such a tap meets a value that is not finite the chain is repeated
// without them. MASK: the output times a dropout mask [B, H, L], whose row a
// lane reads as whole dwords, and scale. COPY: x as it was read, for a
// backward that must not depend on what becomes of x, stored with the outputs
// (one block's forward and backward at B2048 L48 H128 368 -> 377 us; stored
// before the products, where the loads then have to be waited for at once, 389;
// a separate copy 379). 36 FMAs per output on average at 48 taps are 92 us of
// issue at B16384 L48 H128, beside two tensor passes (128 us at the rate of a
// large copy): FWD 176 us (4.6 TB/s), 231 with the mask, DX, three passes, 241
// (5.0 TB/s), VALU 45 to 47% busy, against 305 and 366 with the transposes.
template <int LMAX, bool DX, bool MASK, bool COPY>
__global__ __launch_bounds__(kConvClThreads, LMAX > 40 ? 3 : 4) void s4_conv_cl_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ add,
    const uint8_t* __restrict__ mask, float scale, float* __restrict__ y,
    float* __restrict__ xcopy, int B, int H, int L) {
  static_assert(!(DX && (MASK || COPY)), "mask and copy belong to the forward");
  constexpr int LO = DX ? -(LMAX / 2 - 1) : -(LMAX / 2);  // smallest column offset s - t
  const int h = threadIdx.x % H, sub = threadIdx.x / H, per = blockDim.x / H, p = L / 2;
  float tap[LMAX];  // of offset LO + i
#pragma unroll
  for (int i = 0; i < LMAX; ++i) {
    const int j = DX ? p - (LO + i) : p + LO + i;
    tap[i] = j >= 0 && j < L ? w[h * L + j] : 0.0f;
  }
  // byte offset of (column t, this lane) from the workgroup's first sample;
  // columns past L and samples past B fall outside the buffers
  const uint32_t lane_off = 4u * (uint32_t)(sub * L * H + h);
  auto off = [&](uint32_t lane, int t) {
    return lane + (t < L ? 4u * (uint32_t)(t * H) : kOob);
  };
  // An opaque copy, so that an offset is an addition where it is used and not
  // LMAX registers kept over the samples.
  auto copy = [](uint32_t o) {
    asm volatile("" : "+v"(o));
    return o;
  };
  for (int b0 = blockIdx.x * per; b0 < B; b0 += gridDim.x * per) {
    const size_t base = (size_t)b0 * L * H;
    const uint32_t bytes = 4u * (uint32_t)((B - b0 < per ? B - b0 : per) * L * H);
    const __amdgpu_buffer_rsrc_t rx = make_rsrc_n(x + base, bytes);
    const __amdgpu_buffer_rsrc_t ry = make_rsrc_n(y + base, bytes);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc_n(DX ? add + base : x, DX ? bytes : 0);
    const __amdgpu_buffer_rsrc_t rc = make_rsrc_n(COPY ? xcopy + base : y, COPY ? bytes : 0);
    float v[LMAX];
    const uint32_t lane = copy(lane_off);
#pragma unroll
    for (int s = 0; s < LMAX; ++s) v[s] = buf_load1(rx, off(lane, s), 0);
    uint32_t keep[MASK ? LMAX / 4 : 1];  // the mask bytes of four columns each
    if constexpr (MASK) {
      const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint8_t*>(mask) + base, 0, (int)(bytes / 4), kRsrcWord3);
      const uint32_t row = (uint32_t)((sub * H + h) * L);
      if (L % 4 == 0) {
#pragma unroll
        for (int i = 0; i < LMAX / 4; ++i)
          keep[i] = __builtin_amdgcn_raw_buffer_load_b32(rm, 4 * i < L ? row + 4 * i : kOob, 0, 0);
      } else {
#pragma unroll
        for (int i = 0; i < LMAX / 4; ++i) {
          uint32_t k[4];
#pragma unroll
          for (int r = 0; r < 4; ++r)
            k[r] = __builtin_amdgcn_raw_buffer_load_b8(rm, 4 * i + r < L ? row + 4 * i + r : kOob,
                                                       0, 0);
          keep[i] = k[0] | k[1] << 8 | k[2] << 16 | k[3] << 24;
        }
      }
    }
    static_for<0, LMAX / 4>([&](auto group) {
      constexpr int t0 = 4 * decltype(group)::value;
      if (t0 < L) {
        float o[4] = {0.f, 0.f, 0.f, 0.f}, e[4] = {0.f, 0.f, 0.f, 0.f};
        const uint32_t at = copy(lane_off);
        if constexpr (DX) {  // on their way during the chains
#pragma unroll
          for (int r = 0; r < 4; ++r) e[r] = buf_load1(ra, off(at, t0 + r), 0);
        }
        static_for<0, LMAX>([&](auto step) {
          constexpr int i = DX ? LMAX - 1 - decltype(step)::value : decltype(step)::value;
          constexpr int s = t0 + LO + i;
          if constexpr (s >= 0 && s < LMAX) o[0] = fmaf(tap[i], v[s], o[0]);
          if constexpr (s + 1 >= 0 && s + 1 < LMAX) o[1] = fmaf(tap[i], v[s + 1], o[1]);
          if constexpr (s + 2 >= 0 && s + 2 < LMAX) o[2] = fmaf(tap[i], v[s + 2], o[2]);
          if constexpr (s + 3 >= 0 && s + 3 < LMAX) o[3] = fmaf(tap[i], v[s + 3], o[3]);
        });
        if (__builtin_expect(!(fabsf(o[0]) + fabsf(o[1]) + fabsf(o[2]) + fabsf(o[3]) < INFINITY), 0)) {
          const float* const src = x + base + (size_t)sub * L * H + h;
#pragma unroll 1
          for (int r = 0; r < 4 && b0 + sub < B; ++r) {
            float a = 0.0f;
#pragma unroll 1
            for (int j = 0; j < L; ++j) {
              const int s = DX ? t0 + r - j + p : t0 + r + j - p;
              if (s >= 0 && s < L) a = fmaf(w[h * L + j], src[s * H], a);
            }
            o[0] = r == 0 ? a : o[0];
            o[1] = r == 1 ? a : o[1];
            o[2] = r == 2 ? a : o[2];
            o[3] = r == 3 ? a : o[3];
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if constexpr (DX) o[r] += e[r];
          if constexpr (MASK) o[r] = o[r] * (float)((keep[t0 / 4] >> (8 * r)) & 0xffu) * scale;
          buf_store1(o[r], ry, off(at, t0 + r));
          if constexpr (COPY) buf_store1(v[t0 + r], rc, off(at, t0 + r));
        }
      }
    });
  }
}

}  // namespace pt
