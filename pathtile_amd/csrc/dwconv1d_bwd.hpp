// dwconv1d_bwd.hpp — dX and dK of the depthwise Conv1D in one pass over dY
// and x.
#pragma once

#include "dwconv1d_kernels.hpp"

namespace pt {

__host__ __device__ constexpr size_t bwd_cg_lds_bytes(int L, int lmax) {
  // two stages of dY and of x, two output stages, 16 samples x (8 L + 4) floats
  const size_t stages = (size_t)6 * kRowsCgStep * (kRowsCgWaves * L + 4) * sizeof(float);
  const size_t dtile = (size_t)kRowsCgWaves * lmax * (lmax + 1) * sizeof(float);
  return stages > dtile ? stages : dtile;
}

// The separate kernels move four tensor passes (dX: dY in, dX out; dK: dY and
// x in) where three suffice; this one reads dY once. It is
// dwconv_rows_cg_kernel's dX (8 channels, one per wave, 16-sample steps, band
// matrix of the taps in registers, outputs through LDS) with x staged beside
// dY and the step's dK contraction D += dY^T x after the dX products: MFMA i of
// a tile takes samples 4 kk + i of the step in its four K slots (both operands
// alike), so the lanes of the four slots read rows 4 sample strides apart
// (16 mod 64 floats at every L: disjoint banks), and kChain MFMAs sum from
// zero before they join D, so a range's longer sums round less often (dK's
// error against FP64 at B16384 H128 L48 K48: 5.7e-7 straight into D, 4.1e-7 in
// the separate kernel, 1.9e-7 here; chains of 2 at 48 columns spill, and cost
// 2% in a rolled loop). The epilogue is, with eight sums a diagonal,
// dwconv_dk_cg_kernel's: one partial per (h, j, range) for dk_reduce_kernel.
// Per 16 samples and channel 72 FP32 MFMAs of 32 cycles at 48 columns (dX 36,
// dK 36); at B16384 H128 L48 K48 the matrix cores need 140 us of the 192 us
// that its 1.2 GB take at the rate of a large copy; 216-230 us against 256-264
// for the two kernels, and 843 against 1021 at B32768 H256 L48 K4.
// A column past L reads the channel's last one; rows and columns of D there
// are never summed. nranges: ranges of samples, as in dwconv_rows_cg_kernel.
template <int LMAX, int LOAD_CPOL, bool A4>
__global__ __launch_bounds__(kRowsCgWaves* kWave, LMAX <= 16 ? 4 : 2) void dwconv_bwd_cg_kernel(
    const float* __restrict__ gy, const float* __restrict__ x, const float* __restrict__ w,
    float* __restrict__ out, float* __restrict__ partials, int B, int H, int L, int K, int nranges,
    uint32_t nblocks) {
  constexpr int HC = kRowsCgWaves;
  constexpr int NT = LMAX / 16;  // 16-wide tiles
  constexpr int NU = LMAX / 4;   // dX: MFMA steps over the input columns
  constexpr int TH = HC * kWave;
  constexpr int kChain = NT == 3 ? 4 : 2;  // MFMAs that sum from zero
  constexpr int kNpt = (HC * LMAX * kRowsCgStep / 4 + TH - 1) / TH;
  extern __shared__ float lds[];

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int ngroups = H / HC;
  const uint32_t blk = xcd_remap(blockIdx.x, nblocks);
  const int g = (int)(blk % (uint32_t)ngroups);
  const int r = (int)(blk / (uint32_t)ngroups);
  const int tsteps = (B + kRowsCgStep - 1) / kRowsCgStep;
  const int nsteps = r < tsteps ? (tsteps - 1 - r) / nranges + 1 : 0;

  const int seg = HC * L, segc = seg / 4;  // floats, 16-byte chunks per sample
  const int sk = seg + 4;                  // LDS stride between samples
  const int sz = kRowsCgStep * sk;         // one stage of one tensor
  const int per = kRowsCgStep * segc;      // chunks per stage
  const uint32_t row_bytes = (uint32_t)H * (uint32_t)L * 4u;
  const uint32_t grp_bytes = (uint32_t)g * (uint32_t)seg * 4u;
  float* const outl = lds + 4 * sz;  // stage b: dY at 2 b sz, x at (2 b + 1) sz

  int ek[kNpt];
  uint32_t eoff[kNpt], elds[kNpt];
#pragma unroll
  for (int i = 0; i < kNpt; ++i) {
    const int e = i * TH + (int)threadIdx.x;
    const int k = e < per ? e / segc : kRowsCgStep;
    const int q = e - (e / segc) * segc;
    ek[i] = k;
    eoff[i] = (uint32_t)k * row_bytes + grp_bytes + 16u * (uint32_t)q;
    elds[i] = (uint32_t)(k * sk + 4 * q);
  }
  u32x4 stg[2][2][kNpt];  // [step parity][dY, x]
  auto load_step = [&](int s, u32x4 (&st)[2][kNpt]) {
    const int bs = (r + s * nranges) * kRowsCgStep;
    const size_t at = (size_t)bs * (size_t)H * (size_t)L;
    const __amdgpu_buffer_rsrc_t rg = make_rsrc(gy + at), rx = make_rsrc(x + at);
    const int klim = min(kRowsCgStep, B - bs);
#pragma unroll
    for (int i = 0; i < kNpt; ++i) {
      const uint32_t o = ek[i] < klim ? eoff[i] : kOob;
      st[0][i] = buf_load_chunk<LOAD_CPOL>(rg, o);
      st[1][i] = buf_load_chunk<LOAD_CPOL>(rx, o);
    }
  };
  auto store_stage = [&](int buf, const u32x4 (&st)[2][kNpt]) {
    float* const base = lds + 2 * buf * sz;
#pragma unroll
    for (int i = 0; i < kNpt; ++i)
      if (ek[i] < kRowsCgStep) {
        chunk_to_lds(base + elds[i], st[0][i]);
        chunk_to_lds(base + sz + elds[i], st[1][i]);
      }
  };
  auto flush_out = [&](int s) {
    const float* o = outl + (s & 1) * sz;
    const int bs = (r + s * nranges) * kRowsCgStep;
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(out + (size_t)bs * (size_t)H * (size_t)L);
    const int klim = min(kRowsCgStep, B - bs);
#pragma unroll
    for (int i = 0; i < kNpt; ++i) {
      const u32x4 v = lds_to_chunk(o + (ek[i] < kRowsCgStep ? elds[i] : 0u));
      buf_store_chunk<kCpolNT>(v, ro, ek[i] < klim ? eoff[i] : kOob);
    }
  };

  const int kk = lane >> 4, jj = lane & 15;
  const int p = K >> 1;
  const int h = g * HC + wave;
  const float* wh = w + (size_t)h * K;
  float bt[NU][NT];
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
      const int sc = u + NU * kk, tc = 16 * tt + jj;
      const int j = tc - sc + p;
      const bool ok = j >= 0 && j < K && sc < L && tc < L;
      bt[u][tt] = ok ? wh[j] : 0.0f;
    }

  const int rq = 4 * kk;
  const int cb = wave * L;
  int dcol[NT];  // this lane's column of each tile
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) dcol[tt] = cb + min(16 * tt + jj, L - 1);
  f32x4 acc[1][NT][NT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[0][a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto mfma_step = [&](int s) {
    const float* const sgy = lds + 2 * (s & 1) * sz;
    const float* const sx = sgy + sz;
    const float* row = sgy + jj * sk + cb;  // sample jj, this channel
    const float* src = row + NU * kk;
    float* orow = outl + (s & 1) * sz + jj * sk + cb;
    float a[NU];
    if constexpr (A4) {
#pragma unroll
      for (int q = 0; q < NU / 4; ++q) {
        const float4 v = *reinterpret_cast<const float4*>(src + 4 * q);
        a[4 * q + 0] = v.x;
        a[4 * q + 1] = v.y;
        a[4 * q + 2] = v.z;
        a[4 * q + 3] = v.w;
      }
      if (L != LMAX) {  // columns >= L belong to the next channel: zero them
#pragma unroll
        for (int u = 0; u < NU; ++u) a[u] = u + NU * kk < L ? a[u] : 0.0f;
      }
    } else {  // read in place (the stages of x follow those of dY) and zeroed
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const float v = src[u];
        a[u] = u + NU * kk < L ? v : 0.0f;
      }
    }
    bool bad = false;
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
      f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < NU; ++u)
        d = __builtin_amdgcn_mfma_f32_16x16x4f32(bt[u][tt], a[u], d, 0, 0, 0);
      if (tt == 0) bad = !__builtin_isfinite(d[0]);
      const int t = 16 * tt + rq;
      if constexpr (A4) {
        if (t < L) *reinterpret_cast<f32x4*>(orow + t) = d;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (t + e < L) orow[t + e] = d[e];
      }
    }
#pragma unroll
    for (int i0 = 0; i0 < 4; i0 += kChain) {
      float bv[kChain][NT];
#pragma unroll
      for (int i = 0; i < kChain; ++i)
#pragma unroll
        for (int tb = 0; tb < NT; ++tb) bv[i][tb] = sx[(4 * kk + i0 + i) * sk + dcol[tb]];
#pragma unroll
      for (int ta = 0; ta < NT; ++ta) {
        f32x4 d[NT];
#pragma unroll
        for (int tb = 0; tb < NT; ++tb) d[tb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kChain; ++i) {
          const float av = sgy[(4 * kk + i0 + i) * sk + dcol[ta]];
#pragma unroll
          for (int tb = 0; tb < NT; ++tb)
            d[tb] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv[i][tb], d[tb], 0, 0, 0);
        }
#pragma unroll
        for (int tb = 0; tb < NT; ++tb) acc[0][ta][tb] += d[tb];
      }
    }
    if (__builtin_amdgcn_ballot_w64(bad)) {  // as in dwconv_rows_cg_kernel
      if (bad) {
#pragma unroll 1
        for (int q = 0; q < 4 * NT; ++q) {
          const int t = 16 * (q >> 2) + rq + (q & 3);
          if (t < L) {
            float v = 0.0f;
#pragma unroll 1
            for (int j = 0; j < K; ++j) {
              const int e = t - j + p;
              if ((unsigned)e < (unsigned)L) v = fmaf(row[e], wh[j], v);
            }
            orow[t] = v;
          }
        }
      }
    }
  };

  if (nsteps > 0) {
    load_step(0, stg[0]);
    if (1 < nsteps) load_step(1, stg[1]);
    store_stage(0, stg[0]);
    if (2 < nsteps) load_step(2, stg[0]);
    __syncthreads();
    for (int s0 = 0; s0 < nsteps; s0 += 2) {
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const int s = s0 + d;
        if (s < nsteps) {
          // stages as in dwconv_rows_cg_kernel: step s + 1's input goes to
          // LDS and the loads after it are issued before the matrix work
          if (s + 1 < nsteps) {
            store_stage((s + 1) & 1, stg[(d + 1) & 1]);
            if (s + 3 < nsteps) load_step(s + 3, stg[(d + 1) & 1]);
          }
          mfma_step(s);
          __syncthreads();
          flush_out(s);
        }
      }
    }
    __syncthreads();  // the epilogue's tiles take the stages' place
  }
  dk_cg_epilogue<LMAX, false, 1, 8>(acc, lds, partials, wave, HC, g, r, HC, L, K, nranges, 1);
}

__host__ __device__ constexpr size_t bwd_bf16_lds_bytes(int L, int lmax) {
  // two stages of dY and of x, two output stages, 16 samples x (8 L + 8) values
  const size_t stages = (size_t)6 * kRowsCgStep * (kRowsCgWaves * L + 8) * sizeof(uint16_t);
  const size_t dtile = (size_t)kRowsCgWaves * lmax * (lmax + 1) * sizeof(float);
  return stages > dtile ? stages : dtile;
}

// The same for BF16 tensors: dwconv_rows_bf16mma_kernel's dX (its operands and
// order, so its bits) and D += dY^T x of the step's 16 samples, the K of one
// BF16 MFMA, from one read of dY. K slots 4 kk + i of both operands take
// sample 4 kk + i: rows 4 sample strides apart are 16 mod 64 dwords at every
// L, disjoint banks for the four lane groups. Each step's products sum from
// zero and join D by a rounded addition (dK's error against FP64 at B22016 H128
// L48 K40: 2.3e-7 in the separate kernel, 1.5e-7 here). Bound by memory: three
// tensor passes instead of four, 132 us against 147-156 at B16384 H128 L48 K48
// (96 us at the rate of a large copy) and 478 against 520 at B32768 H256 L48.
// L % 4 == 0.
template <int LMAX, int LOAD_CPOL>
__global__ __launch_bounds__(kRowsCgWaves* kWave, 4) void dwconv_bwd_bf16_kernel(
    const uint16_t* __restrict__ gy, const uint16_t* __restrict__ x, const float* __restrict__ w,
    uint16_t* __restrict__ out, float* __restrict__ partials, int B, int H, int L, int K,
    int nranges, uint32_t nblocks) {
  constexpr int HC = kRowsCgWaves;
  constexpr int NT = LMAX / 16;   // 16-wide tiles
  constexpr int NUB = LMAX / 4;   // input columns per K group of a lane
  constexpr int NG = NUB / 4;     // MFMAs (16 input columns) per dX tile
  constexpr int TH = HC * kWave;
  constexpr int kNpt = (HC * LMAX * kRowsCgStep / 8 + TH - 1) / TH;
  extern __shared__ float lds[];

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int ngroups = H / HC;
  const uint32_t blk = xcd_remap(blockIdx.x, nblocks);
  const int g = (int)(blk % (uint32_t)ngroups);
  const int r = (int)(blk / (uint32_t)ngroups);
  const int tsteps = (B + kRowsCgStep - 1) / kRowsCgStep;
  const int nsteps = r < tsteps ? (tsteps - 1 - r) / nranges + 1 : 0;

  const int seg = HC * L, segc = seg / 8;  // BF16 values, 16-byte chunks
  const int sk = seg + 8;                  // LDS stride between samples (values)
  const int sz = kRowsCgStep * sk;         // one stage of one tensor
  const int per = kRowsCgStep * segc;      // chunks per stage
  const uint32_t row_bytes = (uint32_t)H * (uint32_t)L * 2u;
  const uint32_t grp_bytes = (uint32_t)g * (uint32_t)seg * 2u;
  uint16_t* const inl = reinterpret_cast<uint16_t*>(lds);  // stage b: dY at 2 b sz, x after it
  uint16_t* const outl = inl + 4 * sz;

  int ek[kNpt];
  uint32_t eoff[kNpt], elds[kNpt];
#pragma unroll
  for (int i = 0; i < kNpt; ++i) {
    const int e = i * TH + (int)threadIdx.x;
    const int k = e < per ? e / segc : kRowsCgStep;
    const int q = e - (e / segc) * segc;
    ek[i] = k;
    eoff[i] = (uint32_t)k * row_bytes + grp_bytes + 16u * (uint32_t)q;
    elds[i] = (uint32_t)(k * sk + 8 * q);
  }
  u32x4 stg[2][kNpt];  // dY, x of the step in flight
  auto load_step = [&](int s, u32x4 (&st)[2][kNpt]) {
    const int bs = (r + s * nranges) * kRowsCgStep;
    const size_t at = (size_t)bs * (size_t)H * (size_t)L;
    const __amdgpu_buffer_rsrc_t rg = make_rsrc_t(gy + at), rx = make_rsrc_t(x + at);
    const int klim = min(kRowsCgStep, B - bs);
#pragma unroll
    for (int i = 0; i < kNpt; ++i) {
      const uint32_t o = ek[i] < klim ? eoff[i] : kOob;
      st[0][i] = buf_load_chunk<LOAD_CPOL>(rg, o);
      st[1][i] = buf_load_chunk<LOAD_CPOL>(rx, o);
    }
  };
  auto store_stage = [&](int buf, const u32x4 (&st)[2][kNpt]) {
    uint16_t* const base = inl + 2 * buf * sz;
#pragma unroll
    for (int i = 0; i < kNpt; ++i)
      if (ek[i] < kRowsCgStep) {
        *reinterpret_cast<u32x4*>(base + elds[i]) = st[0][i];
        *reinterpret_cast<u32x4*>(base + sz + elds[i]) = st[1][i];
      }
  };
  auto flush_out = [&](int s) {
    const uint16_t* o = outl + (s & 1) * sz;
    const int bs = (r + s * nranges) * kRowsCgStep;
    const __amdgpu_buffer_rsrc_t ro = make_rsrc_t(out + (size_t)bs * (size_t)H * (size_t)L);
    const int klim = min(kRowsCgStep, B - bs);
#pragma unroll
    for (int i = 0; i < kNpt; ++i) {
      const u32x4 v =
          *reinterpret_cast<const u32x4*>(o + (ek[i] < kRowsCgStep ? elds[i] : 0u));
      buf_store_chunk<kCpolNT>(v, ro, ek[i] < klim ? eoff[i] : kOob);
    }
  };

  const int kk = lane >> 4, jj = lane & 15;
  const int p = K >> 1;
  const int h = g * HC + wave;
  s16x4 bh[NG][NT], bl[NG][NT];  // the taps' band, split as in the dX kernel
#pragma unroll
  for (int u = 0; u < NG; ++u)
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int sc = NUB * kk + 4 * u + i, tc = 16 * tt + jj;
        const int j = tc - sc + p;
        const bool ok = j >= 0 && j < K && sc < L && tc < L;
        const float wv = ok ? w[(size_t)h * K + j] : 0.0f;
        const uint32_t hi = bf16_bits_rne(wv);
        const uint32_t lo = bf16_bits_rne(wv - __uint_as_float(hi << 16));
        bh[u][tt][i] = (short)hi;
        bl[u][tt][i] = (short)lo;
      }

  const int cb = wave * L;
  int dcol[NT];  // first sample's offset of this lane's column of each tile
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) dcol[tt] = 4 * kk * sk + cb + min(16 * tt + jj, L - 1);
  f32x4 acc[1][NT][NT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[0][a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto mfma_step = [&](int s) {
    const uint16_t* const sgy = inl + 2 * (s & 1) * sz;
    const uint16_t* const sx = sgy + sz;
    const uint16_t* src = sgy + jj * sk + cb + NUB * kk;  // sample jj, this channel
    uint16_t* o = outl + (s & 1) * sz;
    s16x4 a[NG];
#pragma unroll
    for (int u = 0; u < NG; ++u) {  // past L: read in place (x's stage follows) and zeroed
      a[u] = *reinterpret_cast<const s16x4*>(src + 4 * u);
      if (L != LMAX && NUB * kk + 4 * u >= L) a[u] = s16x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
      f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < NG; ++u) {
        d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bh[u][tt], a[u], d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bl[u][tt], a[u], d, 0, 0, 0);
      }
      const int t = 16 * tt + 4 * kk;  // L % 4 == 0: all four columns or none
      if (t < L) {
        u32x2 v;
        v.x = bf16_pack2(d[0], d[1]);
        v.y = bf16_pack2(d[2], d[3]);
        *reinterpret_cast<u32x2*>(o + jj * sk + cb + t) = v;
      }
    }
    s16x4 bv[NT];
#pragma unroll
    for (int tb = 0; tb < NT; ++tb)
#pragma unroll
      for (int i = 0; i < 4; ++i) bv[tb][i] = (short)sx[dcol[tb] + i * sk];
#pragma unroll
    for (int ta = 0; ta < NT; ++ta) {
      s16x4 av;
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = (short)sgy[dcol[ta] + i * sk];
#pragma unroll
      for (int tb = 0; tb < NT; ++tb)
        acc[0][ta][tb] += __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
            av, bv[tb], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    }
  };

  if (nsteps > 0) {
    load_step(0, stg);
    store_stage(0, stg);
    if (1 < nsteps) load_step(1, stg);
    __syncthreads();
    for (int s = 0; s < nsteps; ++s) {
      if (s + 1 < nsteps) {
        store_stage((s + 1) & 1, stg);
        if (s + 2 < nsteps) load_step(s + 2, stg);
      }
      mfma_step(s);
      __syncthreads();
      flush_out(s);
    }
    __syncthreads();  // the epilogue's tiles take the stages' place
  }
  dk_cg_epilogue<LMAX, false, 1, 8>(acc, lds, partials, wave, HC, g, r, HC, L, K, nranges, 1);
}

}  // namespace pt
