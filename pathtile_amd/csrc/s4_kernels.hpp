// s4_kernels.hpp — device code of the S4ConvD block around the depthwise
// Conv1D (kernels/warp_tiled_ampere.py:1122-1190 in the reference), FP32,
// for MI355X (gfx950, wave64).
//
// One block computes, for x [B, L, H] and N2 complex states per channel,
//   taps[h][t] = 2 Re sum_n C_eff[h,n] exp(dt[h] A[h,n] t)  (+ skip at L / 2)
//   u [b,h,t]  = conv(x^T, taps),  v = dropout(u),  g = gelu(v)
//   P [b,c,t]  = sum_h W[c][h] g[b,h,t] + bias[c],  c < 2 H
//   y [b,t,c]  = P[c] sigmoid(P[H + c]) + x[b,t,c],  c < H
// The convolution runs on the kernels of dwconv1d_kernels.hpp. Here are the
// taps and their gradient, the [B,L,H] <-> [B,H,L] transposes, and the tail
// (GELU, projection, GLU, residual) with its backward, each one pass over
// its tensors. The tail treats the B L columns as one list of tokens
// (token = b L + t), so its tiles do not depend on L.
//
// The projection runs on the BF16 matrix cores with both operands split into
// three BF16 parts (split3_bf16x8; six of the nine part products, dropped
// terms at most about 2^-22 of a product), which keeps FP32 accuracy at
// 1.55x the FP32 matrix instructions' rate.

#pragma once

#include "dwconv1d_kernels.hpp"

namespace pt {

constexpr int kTailTok = 64;     // tokens per tile of the tail's forward
constexpr int kS4MaxH = 256;     // largest H of the fused block (H % 32 == 0)
constexpr int kDwTok = 32;       // tokens per step of the weight gradient

// Waves of a tail workgroup for CT = H / 16 channel tiles: WPC waves side by
// side on channels (MT tiles each, every tile with its gate tile H channels
// further) and WPT on tokens, so that each weight fragment is read by as few
// waves as possible and small H still fills eight waves.
template <int CT>
struct TailGeo {
  static_assert(CT % 2 == 0 && CT >= 2 && CT <= 16, "H = 32 .. 256 in steps of 32");
  static constexpr int H = 16 * CT;
  static constexpr int KS = H / 32;                       // contraction steps over H
  static constexpr int WPC = CT <= 8 ? CT : CT / 2;
  static constexpr int WPT = CT == 2 ? 4 : CT == 4 ? 2 : 1;
  static constexpr int MT = CT / WPC;
  static constexpr int NW = WPC * WPT;
  static constexpr int GS = H + 8;       // BF16 values per token row of a g part
  static constexpr int PS = 2 * H + 8;   // the same for a dP part
  static constexpr int OS = H + 4;       // floats per token row of the output stage
  // tokens per backward tile: the dP parts of 64 tokens fit the LDS up to H = 128
  static constexpr int BT = CT <= 8 ? 64 : 32;
};

__host__ __device__ constexpr size_t tail_fwd_lds(int H) {
  const size_t g = (size_t)3 * kTailTok * (H + 8) * 2;
  const size_t o = (size_t)kTailTok * (H + 4) * 4;
  return g > o ? g : o;
}
__host__ __device__ constexpr size_t tail_bwd_lds(int H) {
  const size_t bt = H <= 128 ? 64 : 32;
  return (size_t)3 * bt * (2 * H + 8) * 2;  // dP parts, over the g parts
}

// Values of the split weights in the workspace: W as A operands of the
// forward product, then W^T as A operands of the backward one.
__host__ __device__ constexpr size_t wfrag_values(int H) { return (size_t)3 * 2 * H * H; }

__device__ __forceinline__ float gelu_f(float x) {
  return x * 0.5f * (1.0f + erff(x * 0.70710678118654752f));
}

__device__ __forceinline__ float gelu_grad_f(float x) {
  const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
  const float pdf = expf(-0.5f * x * x) * 0.39894228040143268f;
  return cdf + x * pdf;
}

__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }

__device__ __forceinline__ bool finite4(float a, float b, float c, float d) {
  return fabsf(a) + fabsf(b) + fabsf(c) + fabsf(d) < INFINITY;
}

__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The six part products of one 16x16 tile, small ones first.
__device__ __forceinline__ f32x4 mfma_split6(const bf16x8 (&a)[3], const bf16x8 (&b)[3], f32x4 c) {
  c = mfma_bf16(a[2], b[0], c);
  c = mfma_bf16(a[0], b[2], c);
  c = mfma_bf16(a[1], b[1], c);
  c = mfma_bf16(a[1], b[0], c);
  c = mfma_bf16(a[0], b[1], c);
  return mfma_bf16(a[0], b[0], c);
}

// The matrix instruction's internal sum rounds towards minus infinity
// (measured on this product: a mean error of -8.5e-9 of the mean |sum|, where
// FP32 instructions have none). A shift of one sign in du adds up over the
// B L columns of the skip gradient, so the contraction steps of a product
// alternate in sign (odd bit counts of the step number: the balanced order
// + - - + - + + -): those steps' weight fragments are stored negated and the
// accumulators change sign in between, so the shifts cancel.
__host__ __device__ constexpr bool step_negated(int ks) { return __builtin_popcount(ks) & 1; }

template <int N>
__device__ __forceinline__ void negate(f32x4 (&acc)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] = -acc[i];
}

// ---------------------------------------------------------------------------
// Preparation: taps and split weights, one launch per block and pass.
// Blocks 0 .. H - 1 compute the taps of one channel; the others split W
// [2 H][H] into A-operand fragments of 64 lanes x 8 values (lane l holds row
// l % 16, contraction values 8 (l / 16) .. + 7), three parts each:
//   wf[((ct * 2 + half) * KS + ks) * 3 + part][lane][8]   rows of W
//   wt[(ct * 2 KS + ks) * 3 + part][lane][8]              rows of W^T
// so that a wave's fragment is one contiguous 1 KiB read.
// The taps are the reference's formula in FP32 with exp(dt A) - 1 from
// expm1 and sin^2 (no cancellation at small dt A).
// ---------------------------------------------------------------------------
struct Cf { float re, im; };
__device__ __forceinline__ Cf cmul(Cf a, Cf b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ __forceinline__ Cf cdiv(Cf a, Cf b) {
  const float d = 1.0f / (b.re * b.re + b.im * b.im);
  return {(a.re * b.re + a.im * b.im) * d, (a.im * b.re - a.re * b.im) * d};
}
__device__ __forceinline__ Cf cexpm1(Cf a) {
  float s, c;
  sincosf(a.im, &s, &c);
  const float h = sinf(0.5f * a.im);
  return {expm1f(a.re) * c - 2.0f * h * h, expf(a.re) * s};
}
__device__ __forceinline__ Cf cexp_at(Cf a, float t) {
  float s, c;
  sincosf(a.im * t, &s, &c);
  const float e = expf(a.re * t);
  return {e * c, e * s};
}

constexpr int kPrepThreads = 256;
constexpr int kPrepStates = 32;  // states per LDS pass

__global__ __launch_bounds__(kPrepThreads) void s4_prep_kernel(
    const float* __restrict__ log_dt, const float* __restrict__ c_re,
    const float* __restrict__ c_im, const float* __restrict__ log_a_re,
    const float* __restrict__ a_im, const float* __restrict__ skip,
    const float* __restrict__ w, float* __restrict__ taps, __bf16* __restrict__ wf,
    int H, int L, int N2, int transposed) {
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < H) {
    const int h = blockIdx.x;
    __shared__ float ce[2][kPrepStates], da[2][kPrepStates];
    __shared__ float part[kMaxL][kPrepStates + 1];
    const float dt = expf(log_dt[h]);
    float acc = 0.0f;  // thread t < L: taps[h][t]
    for (int n0 = 0; n0 < N2; n0 += kPrepStates) {
      const int nn = N2 - n0 < kPrepStates ? N2 - n0 : kPrepStates;
      if (tid < nn) {
        const int i = h * N2 + n0 + tid;
        const Cf A = {-expf(log_a_re[i]), a_im[i]};
        const Cf dA = {A.re * dt, A.im * dt};
        const Cf e = cdiv(cmul(Cf{c_re[i], c_im[i]}, cexpm1(dA)), A);
        ce[0][tid] = e.re;
        ce[1][tid] = e.im;
        da[0][tid] = dA.re;
        da[1][tid] = dA.im;
      }
      __syncthreads();
      for (int q = tid; q < nn * L; q += kPrepThreads) {
        const int t = q / nn, n = q - t * nn;
        const Cf z = cexp_at(Cf{da[0][n], da[1][n]}, (float)t);
        part[t][n] = ce[0][n] * z.re - ce[1][n] * z.im;
      }
      __syncthreads();
      if (tid < L)
        for (int n = 0; n < nn; ++n) acc += part[tid][n];
      __syncthreads();
    }
    if (tid < L) taps[h * L + tid] = 2.0f * acc + (tid == L / 2 ? skip[h] : 0.0f);
    return;
  }
  // one fragment lane (8 values) per thread
  const int KS = H / 32, nf = 2 * H * H / 8;
  int q = ((int)blockIdx.x - H) * kPrepThreads + tid;
  const bool back = q >= nf;
  if (back) q -= nf;
  if (q >= nf || (back && !transposed)) return;
  const int lane = q & 63, f = q >> 6;
  const int row = lane & 15, k0 = 8 * (lane >> 4);
  float v[8];
  __bf16* dst;
  const int ks = f % (back ? 2 * KS : KS);
  if (!back) {
    const int tile = f / KS;  // tile = ct * 2 + half
    const float* src = w + (size_t)((tile & 1) * H + 16 * (tile >> 1) + row) * H + 32 * ks + k0;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = src[i];
    dst = wf + (size_t)f * 3 * 512;
  } else {
    const int ct = f / (2 * KS);
    const float* src = w + (size_t)(32 * ks + k0) * H + 16 * ct + row;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = src[(size_t)i * H];
    dst = wf + wfrag_values(H) + (size_t)f * 3 * 512;
  }
  if (step_negated(ks)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = -v[i];
  }
  bf16x8 hi, mid, lo;
  split3_bf16x8(v, hi, mid, lo);
  *reinterpret_cast<bf16x8*>(dst + 0 * 512 + lane * 8) = hi;
  *reinterpret_cast<bf16x8*>(dst + 1 * 512 + lane * 8) = mid;
  *reinterpret_cast<bf16x8*>(dst + 2 * 512 + lane * 8) = lo;
}

// ---------------------------------------------------------------------------
// Gradient of the taps with respect to the kernel's parameters, from
// dk [H][L]: with z = exp(dt A), E = z - 1, S0 = sum_t dk[t] z^t,
// S1 = sum_t t dk[t] z^t per state,
//   dL = 2 Re sum_n ( S0 E / A dC + R dA + (S0 C z + C_eff A S1) ddt ),
//   R  = S0 C / A^2 (z dt A - E) + dt C_eff S1,
// one workgroup per channel. z dt A - E cancels to second order in dt A, so
// that factor and E are computed in FP64 (a handful of operations per state).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kPrepThreads) void s4_taps_grad_kernel(
    const float* __restrict__ dk, const float* __restrict__ log_dt,
    const float* __restrict__ c_re, const float* __restrict__ c_im,
    const float* __restrict__ log_a_re, const float* __restrict__ a_im,
    float* __restrict__ d_log_dt, float* __restrict__ d_c_re, float* __restrict__ d_c_im,
    float* __restrict__ d_log_a_re, float* __restrict__ d_a_im, float* __restrict__ d_skip,
    int L, int N2) {
  constexpr int kChunks = 8;  // threads per state
  __shared__ float sdk[kMaxL];
  __shared__ float s0r[kPrepStates][kChunks], s0i[kPrepStates][kChunks];
  __shared__ float s1r[kPrepStates][kChunks], s1i[kPrepStates][kChunks];
  __shared__ float ddt[kPrepStates];
  const int h = blockIdx.x, tid = threadIdx.x;
  if (tid < L) sdk[tid] = dk[h * L + tid];
  __syncthreads();
  const float dt = expf(log_dt[h]);
  float ddt_sum = 0.0f;  // thread 0
  for (int n0 = 0; n0 < N2; n0 += kPrepStates) {
    const int nn = N2 - n0 < kPrepStates ? N2 - n0 : kPrepStates;
    const int n = tid / kChunks, q = tid % kChunks;
    if (n < nn) {
      const int i = h * N2 + n0 + n;
      const Cf dA = {-expf(log_a_re[i]) * dt, a_im[i] * dt};
      Cf s0 = {0.f, 0.f}, s1 = {0.f, 0.f};
      for (int t = q; t < L; t += kChunks) {
        const Cf z = cexp_at(dA, (float)t);
        const float d = sdk[t], td = d * (float)t;
        s0.re += d * z.re;
        s0.im += d * z.im;
        s1.re += td * z.re;
        s1.im += td * z.im;
      }
      s0r[n][q] = s0.re;
      s0i[n][q] = s0.im;
      s1r[n][q] = s1.re;
      s1i[n][q] = s1.im;
    }
    __syncthreads();
    if (tid < nn) {
      const int i = h * N2 + n0 + tid;
      double S0r = 0, S0i = 0, S1r = 0, S1i = 0;
      for (int k = 0; k < kChunks; ++k) {
        S0r += s0r[tid][k];
        S0i += s0i[tid][k];
        S1r += s1r[tid][k];
        S1i += s1i[tid][k];
      }
      const double ar = -(double)expf(log_a_re[i]), ai = a_im[i], d = dt;
      const double cr = c_re[i], ci = c_im[i];
      const double xr = ar * d, xi = ai * d;
      double sn, cs;
      sincos(xi, &sn, &cs);
      const double ex = exp(xr), zr = ex * cs, zi = ex * sn;
      const double hs = sin(0.5 * xi);
      const double Er = expm1(xr) * cs - 2.0 * hs * hs, Ei = zi;
      const double inv = 1.0 / (ar * ar + ai * ai);
      // E / A
      const double er = (Er * ar + Ei * ai) * inv, ei = (Ei * ar - Er * ai) * inv;
      // dC: S0 E / A
      const double gr = S0r * er - S0i * ei, gi = S0r * ei + S0i * er;
      // C_eff = C E / A
      const double fr = cr * er - ci * ei, fi = cr * ei + ci * er;
      // C_eff S1
      const double pr = fr * S1r - fi * S1i, pi = fr * S1i + fi * S1r;
      // S0 C
      const double qr = S0r * cr - S0i * ci, qi = S0r * ci + S0i * cr;
      // (z dt A - E) / A^2
      const double mr = zr * xr - zi * xi - Er, mi = zr * xi + zi * xr - Ei;
      const double a1r = (mr * ar + mi * ai) * inv, a1i = (mi * ar - mr * ai) * inv;
      const double a2r = (a1r * ar + a1i * ai) * inv, a2i = (a1i * ar - a1r * ai) * inv;
      const double Rr = qr * a2r - qi * a2i + d * pr, Ri = qr * a2i + qi * a2r + d * pi;
      // ddt: S0 C z + C_eff S1 A
      const double Dr = qr * zr - qi * zi + pr * ar - pi * ai;
      d_c_re[i] = (float)(2.0 * gr);
      d_c_im[i] = (float)(-2.0 * gi);
      d_log_a_re[i] = (float)(2.0 * Rr * ar);
      d_a_im[i] = (float)(-2.0 * Ri);
      ddt[tid] = (float)(2.0 * Dr * d);
    }
    __syncthreads();
    if (tid == 0)
      for (int k = 0; k < nn; ++k) ddt_sum += ddt[k];
    __syncthreads();
  }
  if (tid == 0) {
    d_log_dt[h] = ddt_sum;
    d_skip[h] = sdk[L / 2];
  }
}

// ---------------------------------------------------------------------------
// Transposes of whole samples, [L][H] <-> [H][L]; both sides move 16-byte
// pieces (dwords where L % 4 != 0) through one LDS tile per workgroup with an
// odd row stride. ADD: the [L][H] result also gets `add` (the residual
// gradient). Bound by HBM: one read and one write of the tensor.
// ---------------------------------------------------------------------------
constexpr int kTransThreads = 256;

template <bool VEC>
__global__ __launch_bounds__(kTransThreads) void s4_transpose_kernel(
    const float* __restrict__ x, float* __restrict__ out, int B, int H, int L) {
  extern __shared__ float tile[];  // [L][S]
  const int S = H + 1, n4 = L * H / 4, h4 = H / 4;
  for (int b = blockIdx.x; b < B; b += gridDim.x) {
    const float* src = x + (size_t)b * L * H;
    float* dst = out + (size_t)b * L * H;
    for (int i = threadIdx.x; i < n4; i += kTransThreads) {
      const float4 v = reinterpret_cast<const float4*>(src)[i];
      const int t = i / h4, c = 4 * (i - t * h4);
      float* p = tile + t * S + c;
      p[0] = v.x;
      p[1] = v.y;
      p[2] = v.z;
      p[3] = v.w;
    }
    __syncthreads();
    if constexpr (VEC) {
      const int l4 = L / 4;
      for (int i = threadIdx.x; i < n4; i += kTransThreads) {
        const int c = i / l4, t = 4 * (i - c * l4);
        const float* p = tile + t * S + c;
        reinterpret_cast<float4*>(dst)[i] = float4{p[0], p[S], p[2 * S], p[3 * S]};
      }
    } else {
      for (int i = threadIdx.x; i < L * H; i += kTransThreads) {
        const int c = i / L, t = i - c * L;
        dst[i] = tile[t * S + c];
      }
    }
    __syncthreads();
  }
}

template <bool VEC>
__global__ __launch_bounds__(kTransThreads) void s4_transpose_add_kernel(
    const float* __restrict__ d, const float* __restrict__ add, float* __restrict__ out, int B,
    int H, int L) {
  extern __shared__ float tile[];
  const int S = H + 1, n4 = L * H / 4, h4 = H / 4;
  for (int b = blockIdx.x; b < B; b += gridDim.x) {
    const float* src = d + (size_t)b * L * H;
    if constexpr (VEC) {
      const int l4 = L / 4;
      for (int i = threadIdx.x; i < n4; i += kTransThreads) {
        const float4 v = reinterpret_cast<const float4*>(src)[i];
        const int c = i / l4, t = 4 * (i - c * l4);
        float* p = tile + t * S + c;
        p[0] = v.x;
        p[S] = v.y;
        p[2 * S] = v.z;
        p[3 * S] = v.w;
      }
    } else {
      for (int i = threadIdx.x; i < L * H; i += kTransThreads) {
        const int c = i / L, t = i - c * L;
        tile[t * S + c] = src[i];
      }
    }
    __syncthreads();
    const float4* a4 = reinterpret_cast<const float4*>(add + (size_t)b * L * H);
    float4* o4 = reinterpret_cast<float4*>(out + (size_t)b * L * H);
    for (int i = threadIdx.x; i < n4; i += kTransThreads) {
      const int t = i / h4, c = 4 * (i - t * h4);
      const float* p = tile + t * S + c;
      const float4 a = a4[i];
      o4[i] = float4{p[0] + a.x, p[1] + a.y, p[2] + a.z, p[3] + a.w};
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Tail, shared pieces
// ---------------------------------------------------------------------------
// Element offset of (token n, channel 0) in a [B, H, L] tensor.
__device__ __forceinline__ uint32_t token_base(uint32_t n, uint32_t H, uint32_t L) {
  const uint32_t b = n / L;
  return b * H * L + (n - b * L);
}

// gelu(v) of TOK tokens from token n0 on, split into the three parts of the
// LDS stage [part][token][GS]: a lane takes one token and eight channels, so
// a wave's loads run along the tokens of one channel.
template <int CT, int TOK>
__device__ __forceinline__ void stage_gelu(__bf16* sg, const float* __restrict__ v, uint32_t n0,
                                           uint32_t ntok, uint32_t L) {
  using G = TailGeo<CT>;
  constexpr int kUnits = TOK * (G::H / 8);
  for (int u = threadIdx.x; u < kUnits; u += G::NW * kWave) {
    const int tk = u % TOK, c = 8 * (u / TOK);
    float g[8];
    const uint32_t n = n0 + tk;
    if (n < ntok) {
      const float* src = v + token_base(n, G::H, L) + (size_t)c * L;
#pragma unroll
      for (int i = 0; i < 8; ++i) g[i] = src[i * L];
#pragma unroll
      for (int i = 0; i < 8; ++i) g[i] = gelu_f(g[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) g[i] = 0.0f;
    }
    bf16x8 hi, mid, lo;
    split3_bf16x8(g, hi, mid, lo);
    __bf16* d = sg + tk * G::GS + c;
    *reinterpret_cast<bf16x8*>(d) = hi;
    *reinterpret_cast<bf16x8*>(d + TOK * G::GS) = mid;
    *reinterpret_cast<bf16x8*>(d + 2 * TOK * G::GS) = lo;
  }
}

// Weight fragments of N row tiles `steps` contraction steps apart.
template <int N>
__device__ __forceinline__ void load_frags(bf16x8 (&a)[N][3], const __bf16* __restrict__ w,
                                           int steps) {
#pragma unroll
  for (int m = 0; m < N; ++m)
#pragma unroll
    for (int p = 0; p < 3; ++p)
      a[m][p] = *reinterpret_cast<const bf16x8*>(w + ((size_t)m * steps * 3 + p) * 512);
}

// P tiles of this wave: acc[m][half][nt] = W rows (16 (ct0 + m) .. of half)
// times the staged tokens 16 (nt0 + nt) .. .
template <int CT, int TOK, int NT>
__device__ __forceinline__ void project(f32x4 (&acc)[TailGeo<CT>::MT][2][NT], const __bf16* sg,
                                        const __bf16* __restrict__ wf, int ct0, int nt0, int lane) {
  using G = TailGeo<CT>;
#pragma unroll
  for (int m = 0; m < G::MT; ++m)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[m][hf][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const __bf16* const b0 = sg + (16 * nt0 + (lane & 15)) * G::GS + 8 * (lane >> 4);
  const __bf16* const a0 = wf + (size_t)ct0 * 2 * G::KS * 3 * 512 + lane * 8;
  bf16x8 a[G::MT][2][3];
  load_frags<G::MT * 2>(reinterpret_cast<bf16x8(&)[G::MT * 2][3]>(a), a0, G::KS);
#pragma unroll 1
  for (int ks = 0; ks < G::KS; ++ks) {
    // the next step's weight fragments are on their way during this step
    bf16x8 an[G::MT][2][3];
    load_frags<G::MT * 2>(reinterpret_cast<bf16x8(&)[G::MT * 2][3]>(an),
                          a0 + (ks + 1 < G::KS ? ks + 1 : 0) * 3 * 512, G::KS);
    if (ks > 0 && step_negated(ks) != step_negated(ks - 1))
      negate(reinterpret_cast<f32x4(&)[G::MT * 2 * NT]>(acc));
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      bf16x8 b[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        b[p] = *reinterpret_cast<const bf16x8*>(b0 + (p * TOK + 16 * nt) * G::GS + 32 * ks);
#pragma unroll
      for (int m = 0; m < G::MT; ++m)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) acc[m][hf][nt] = mfma_split6(a[m][hf], b, acc[m][hf][nt]);
    }
#pragma unroll
    for (int m = 0; m < G::MT; ++m)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int p = 0; p < 3; ++p) a[m][hf][p] = an[m][hf][p];
  }
  if (step_negated(G::KS - 1)) negate(reinterpret_cast<f32x4(&)[G::MT * 2 * NT]>(acc));
}

// One pre-activation of one token by the FP32 chain, for values that the
// split cannot carry (Inf, NaN, or rounding past BF16's largest value).
__device__ __forceinline__ float project_one(const float* __restrict__ v, const float* __restrict__ w,
                                             uint32_t base, int row, int H, int L) {
  float s = 0.0f;
#pragma unroll 1
  for (int h = 0; h < H; ++h) s = fmaf(w[(size_t)row * H + h], gelu_f(v[base + (uint32_t)(h * L)]), s);
  return s;
}

// Recomputes a lane's four value and gate sums where one is not finite.
__device__ __forceinline__ void project_fix(f32x4& a, f32x4& b, const float* __restrict__ v,
                                            const float* __restrict__ w, uint32_t n, int c, int H,
                                            uint32_t L) {
  const uint32_t base = token_base(n, H, L);
#pragma unroll 1
  for (int r = 0; r < 4; ++r) {
    const float pa = project_one(v, w, base, c + r, H, L);
    const float pb = project_one(v, w, base, H + c + r, H, L);
    a[0] = r == 0 ? pa : a[0];
    a[1] = r == 1 ? pa : a[1];
    a[2] = r == 2 ? pa : a[2];
    a[3] = r == 3 ? pa : a[3];
    b[0] = r == 0 ? pb : b[0];
    b[1] = r == 1 ? pb : b[1];
    b[2] = r == 2 ? pb : b[2];
    b[3] = r == 3 ? pb : b[3];
  }
}

// ---------------------------------------------------------------------------
// Tail forward: y = GLU(W gelu(v) + bias) + x, v [B,H,L], x and y [B,L,H].
// A persistent workgroup takes tiles of 64 tokens: gelu and split into LDS,
// the projection (the weight fragments stream from the L2, the token parts
// from LDS), GLU into an FP32 stage over the same LDS, then flat 16-byte rows
// with the residual. Two workgroups per CU at H <= 128, so that one's gelu
// (VALU) runs beside the other's matrix work.
// ---------------------------------------------------------------------------
template <int CT>
__global__ __launch_bounds__(TailGeo<CT>::NW* kWave, CT <= 8 ? 4 : 2) void s4_tail_fwd_kernel(
    const float* __restrict__ v, const float* __restrict__ x, const __bf16* __restrict__ wf,
    const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ y,
    uint32_t ntok, uint32_t L, uint32_t ntiles) {
  using G = TailGeo<CT>;
  constexpr int NT = kTailTok / 16 / G::WPT;
  extern __shared__ __align__(16) char smem[];
  __bf16* const sg = reinterpret_cast<__bf16*>(smem);
  float* const so = reinterpret_cast<float*>(smem);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ct0 = (wave % G::WPC) * G::MT, nt0 = (wave / G::WPC) * NT;
  for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const uint32_t n0 = tile * kTailTok;
    stage_gelu<CT, kTailTok>(sg, v, n0, ntok, L);
    __syncthreads();
    f32x4 acc[G::MT][2][NT];
    project<CT, kTailTok, NT>(acc, sg, wf, ct0, nt0, lane);
    __syncthreads();  // the stage is read; the output stage takes its place
#pragma unroll
    for (int m = 0; m < G::MT; ++m) {
      const int c = 16 * (ct0 + m) + 4 * (lane >> 4);
      const float4 ba = *reinterpret_cast<const float4*>(bias + c);
      const float4 bb = *reinterpret_cast<const float4*>(bias + G::H + c);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int tk = 16 * (nt0 + nt) + (lane & 15);
        f32x4 a = acc[m][0][nt], b = acc[m][1][nt];
        if (__builtin_expect(!(finite4(a[0], a[1], a[2], a[3]) && finite4(b[0], b[1], b[2], b[3])), 0)) {
          if (n0 + tk < ntok) project_fix(a, b, v, w, n0 + tk, c, G::H, L);
        }
        float4 o;
        o.x = (a[0] + ba.x) * sigmoid_f(b[0] + bb.x);
        o.y = (a[1] + ba.y) * sigmoid_f(b[1] + bb.y);
        o.z = (a[2] + ba.z) * sigmoid_f(b[2] + bb.z);
        o.w = (a[3] + ba.w) * sigmoid_f(b[3] + bb.w);
        *reinterpret_cast<float4*>(so + tk * G::OS + c) = o;
      }
    }
    __syncthreads();
    const float4* const x4 = reinterpret_cast<const float4*>(x + (size_t)n0 * G::H);
    float4* const y4 = reinterpret_cast<float4*>(y + (size_t)n0 * G::H);
    const uint32_t left = ntok - n0 < kTailTok ? ntok - n0 : kTailTok;
    for (uint32_t i = threadIdx.x; i < left * (G::H / 4); i += G::NW * kWave) {
      const uint32_t tk = i / (G::H / 4), c = 4 * (i % (G::H / 4));
      const float4 o = *reinterpret_cast<const float4*>(so + tk * G::OS + c);
      const float4 r = x4[i];
      y4[i] = float4{o.x + r.x, o.y + r.y, o.z + r.z, o.w + r.w};
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Tail backward with respect to its input: from gy [B,L,H], du = dL/du
// [B,H,L] (through GLU, projection, gelu and the dropout mask) and
// dP [2 H][np] (token-contiguous rows, zero past the last token) for the
// weight gradient. The pre-activations are recomputed. The dP parts
// [part][token][PS] are the B operands of W^T dP and lie over the g parts.
// ---------------------------------------------------------------------------
template <int CT>
__global__ __launch_bounds__(TailGeo<CT>::NW* kWave, 2) void s4_tail_bwd_kernel(
    const float* __restrict__ gy, const float* __restrict__ v, const uint8_t* __restrict__ mask,
    float scale, const __bf16* __restrict__ wf, const float* __restrict__ w,
    const float* __restrict__ bias, float* __restrict__ du, float* __restrict__ dp, uint32_t ntok,
    uint32_t L, uint32_t ntiles, uint32_t np) {
  using G = TailGeo<CT>;
  constexpr int TOK = G::BT;
  constexpr int WPT = G::WPT < TOK / 16 ? G::WPT : TOK / 16;
  static_assert(WPT == G::WPT, "every wave has tokens");
  constexpr int NT = TOK / 16 / G::WPT;
  extern __shared__ __align__(16) char smem[];
  __bf16* const sg = reinterpret_cast<__bf16*>(smem);
  __bf16* const sp = sg;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ct0 = (wave % G::WPC) * G::MT, nt0 = (wave / G::WPC) * NT;
  const __bf16* const wt = wf + wfrag_values(G::H);
  for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const uint32_t n0 = tile * TOK;
    stage_gelu<CT, TOK>(sg, v, n0, ntok, L);
    __syncthreads();
    f32x4 acc[G::MT][2][NT];
    project<CT, TOK, NT>(acc, sg, wf, ct0, nt0, lane);
    __syncthreads();  // the g parts are read; the dP parts take their place
#pragma unroll
    for (int m = 0; m < G::MT; ++m) {
      const int c = 16 * (ct0 + m) + 4 * (lane >> 4);
      const float4 ba = *reinterpret_cast<const float4*>(bias + c);
      const float4 bb = *reinterpret_cast<const float4*>(bias + G::H + c);
      const float vba[4] = {ba.x, ba.y, ba.z, ba.w}, vbb[4] = {bb.x, bb.y, bb.z, bb.w};
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int tk = 16 * (nt0 + nt) + (lane & 15);
        const bool in = n0 + tk < ntok;
        f32x4 a = acc[m][0][nt], b = acc[m][1][nt];
        float4 g4 = {0.f, 0.f, 0.f, 0.f};
        if (in) g4 = *reinterpret_cast<const float4*>(gy + (size_t)(n0 + tk) * G::H + c);
        if (__builtin_expect(!(finite4(a[0], a[1], a[2], a[3]) && finite4(b[0], b[1], b[2], b[3])), 0)) {
          if (in) project_fix(a, b, v, w, n0 + tk, c, G::H, L);
        }
        const float g[4] = {g4.x, g4.y, g4.z, g4.w};
        float pa[8];  // four value and four gate gradients
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float s = sigmoid_f(b[r] + vbb[r]);
          const float da = s * g[r];
          const float db = (1.0f - s) * s * g[r] * (a[r] + vba[r]);
          pa[r] = in ? da : 0.0f;
          pa[4 + r] = in ? db : 0.0f;
          dp[(size_t)(c + r) * np + n0 + tk] = pa[r];
          dp[(size_t)(G::H + c + r) * np + n0 + tk] = pa[4 + r];
        }
        bf16x8 hi, mid, lo;
        split3_bf16x8(pa, hi, mid, lo);
        const bf16x8 parts[3] = {hi, mid, lo};
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          typedef __bf16 bf16x4v __attribute__((ext_vector_type(4)));
          __bf16* d = sp + (p * TOK + tk) * G::PS + c;
          *reinterpret_cast<bf16x4v*>(d) =
              bf16x4v{parts[p][0], parts[p][1], parts[p][2], parts[p][3]};
          *reinterpret_cast<bf16x4v*>(d + G::H) =
              bf16x4v{parts[p][4], parts[p][5], parts[p][6], parts[p][7]};
        }
      }
    }
    __threadfence_block();
    __syncthreads();
    // dg = W^T dP
    f32x4 dg[G::MT][NT];
#pragma unroll
    for (int m = 0; m < G::MT; ++m)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) dg[m][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __bf16* const b0 = sp + (16 * nt0 + (lane & 15)) * G::PS + 8 * (lane >> 4);
    const __bf16* const a0 = wt + (size_t)ct0 * 2 * G::KS * 3 * 512 + lane * 8;
    bf16x8 a[G::MT][3];
    load_frags<G::MT>(a, a0, 2 * G::KS);
#pragma unroll 1
    for (int ks = 0; ks < 2 * G::KS; ++ks) {
      bf16x8 an[G::MT][3];
      load_frags<G::MT>(an, a0 + (ks + 1 < 2 * G::KS ? ks + 1 : 0) * 3 * 512, 2 * G::KS);
      if (ks > 0 && step_negated(ks) != step_negated(ks - 1))
        negate(reinterpret_cast<f32x4(&)[G::MT * NT]>(dg));
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        bf16x8 b[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          b[p] = *reinterpret_cast<const bf16x8*>(b0 + (p * TOK + 16 * nt) * G::PS + 32 * ks);
#pragma unroll
        for (int m = 0; m < G::MT; ++m) dg[m][nt] = mfma_split6(a[m], b, dg[m][nt]);
      }
#pragma unroll
      for (int m = 0; m < G::MT; ++m)
#pragma unroll
        for (int p = 0; p < 3; ++p) a[m][p] = an[m][p];
    }
    if (step_negated(2 * G::KS - 1)) negate(reinterpret_cast<f32x4(&)[G::MT * NT]>(dg));
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const uint32_t tk = 16 * (nt0 + nt) + (lane & 15), n = n0 + tk;
      if (n < ntok) {
        const uint32_t base = token_base(n, G::H, L);
#pragma unroll
        for (int m = 0; m < G::MT; ++m) {
          const int c = 16 * (ct0 + m) + 4 * (lane >> 4);
          f32x4 d = dg[m][nt];
          if (__builtin_expect(!finite4(d[0], d[1], d[2], d[3]), 0)) {
#pragma unroll 1
            for (int r = 0; r < 4; ++r) {
              float s = 0.0f;
#pragma unroll 1
              for (int o = 0; o < 2 * G::H; ++o)
                s = fmaf(w[(size_t)o * G::H + c + r], dp[(size_t)o * np + n], s);
              d[0] = r == 0 ? s : d[0];
              d[1] = r == 1 ? s : d[1];
              d[2] = r == 2 ? s : d[2];
              d[3] = r == 3 ? s : d[3];
            }
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const uint32_t at = base + (uint32_t)(c + r) * L;
            float o = d[r] * gelu_grad_f(v[at]);
            if (mask) o = o * (float)mask[at] * scale;
            du[at] = o;
          }
        }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Weight gradient of the projection: dW[c][h] = sum_tok dP[c][tok] g[h][tok]
// and dbias[c] = sum_tok dP[c][tok], split over the tokens. A workgroup takes
// a contiguous run of 32-token steps and NB channels (columns); its waves own
// rows of dP, read straight from memory in the A layout (each row's 32 tokens
// are one 128-byte line) and split in registers; g is computed, split and
// shared through LDS [part][channel][40]. Partials [range][2 H H + 2 H] go to
// the workspace for a fixed-order reduction.
// ---------------------------------------------------------------------------
template <int CT>
struct DwGeo {
  static constexpr int RT = 2 * CT;  // row tiles
  static constexpr int NW = RT % 8 == 0 ? 8 : RT == 4 ? 4 : RT == 12 ? 6 : RT / 4;
  static constexpr int MT = RT / NW;
  static constexpr int NB = CT <= 8 ? CT : CT / 2;  // column tiles per workgroup
  static constexpr int SPLIT = CT / NB;
  static constexpr int CS = kDwTok + 8;  // BF16 values per channel row of a part
  static constexpr size_t lds = (size_t)2 * 3 * NB * 16 * CS * 2;
};

template <int CT, bool VEC>
__global__ __launch_bounds__(DwGeo<CT>::NW* kWave, 2) void s4_dw_kernel(
    const float* __restrict__ dp, const float* __restrict__ v, float* __restrict__ part,
    uint32_t ntok, uint32_t L, uint32_t nsteps, uint32_t steps_per, uint32_t np) {
  using D = DwGeo<CT>;
  constexpr int H = 16 * CT, NC = 16 * D::NB, TH = D::NW * kWave;
  constexpr int kUnits = NC * (kDwTok / 8);  // (channel, eight tokens)
  constexpr int U = (kUnits + TH - 1) / TH;
  constexpr int SZ = 3 * NC * D::CS;
  extern __shared__ __align__(16) char smem[];
  __bf16* const sg = reinterpret_cast<__bf16*>(smem);  // two stages
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int range = blockIdx.x / D::SPLIT, nb = blockIdx.x % D::SPLIT;
  const uint32_t s0 = range * steps_per;
  const uint32_t s1 = s0 + steps_per < nsteps ? s0 + steps_per : nsteps;
  f32x4 acc[D::MT][D::NB];
  float rows[D::MT];
#pragma unroll
  for (int m = 0; m < D::MT; ++m) {
    rows[m] = 0.0f;
#pragma unroll
    for (int n = 0; n < D::NB; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float* const a0 =
      dp + (size_t)(16 * wave * D::MT + (lane & 15)) * np + 8 * (lane >> 4);
  float vr[U][8];
  float ar[D::MT][8];
  auto load_v = [&](uint32_t s) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int u = threadIdx.x + i * TH;
      const int c = u >> 2, q = u & 3;
      const uint32_t n = s * kDwTok + 8 * q;
      const bool on = u < kUnits;
#pragma unroll
      for (int e = 0; e < 8; ++e) vr[i][e] = 0.0f;
      if constexpr (VEC) {  // L % 4 == 0: four tokens from a multiple of four lie in one row
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
          if (on && n + e < ntok) {
            const float4 f = *reinterpret_cast<const float4*>(
                v + token_base(n + e, H, L) + (size_t)(nb * NC + c) * L);
            vr[i][e] = f.x;
            vr[i][e + 1] = f.y;
            vr[i][e + 2] = f.z;
            vr[i][e + 3] = f.w;
          }
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (on && n + e < ntok) vr[i][e] = v[token_base(n + e, H, L) + (size_t)(nb * NC + c) * L];
      }
    }
  };
  auto load_a = [&](uint32_t s) {
#pragma unroll
    for (int m = 0; m < D::MT; ++m) {
      const float* p = a0 + (size_t)16 * m * np + (size_t)s * kDwTok;
      const float4 f0 = *reinterpret_cast<const float4*>(p);
      const float4 f1 = *reinterpret_cast<const float4*>(p + 4);
      ar[m][0] = f0.x;
      ar[m][1] = f0.y;
      ar[m][2] = f0.z;
      ar[m][3] = f0.w;
      ar[m][4] = f1.x;
      ar[m][5] = f1.y;
      ar[m][6] = f1.z;
      ar[m][7] = f1.w;
    }
  };
  if (s0 < s1) {
    load_v(s0);
    load_a(s0);
  }
  for (uint32_t s = s0; s < s1; ++s) {
    __bf16* const st = sg + ((s - s0) & 1) * SZ;
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int u = threadIdx.x + i * TH;
      if (u < kUnits) {
        float g[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) g[e] = gelu_f(vr[i][e]);  // gelu(0) = 0 past the end
        bf16x8 hi, mid, lo;
        split3_bf16x8(g, hi, mid, lo);
        __bf16* d = st + (u >> 2) * D::CS + 8 * (u & 3);
        *reinterpret_cast<bf16x8*>(d) = hi;
        *reinterpret_cast<bf16x8*>(d + NC * D::CS) = mid;
        *reinterpret_cast<bf16x8*>(d + 2 * NC * D::CS) = lo;
      }
    }
    bf16x8 a[D::MT][3];
#pragma unroll
    for (int m = 0; m < D::MT; ++m) {
#pragma unroll
      for (int e = 0; e < 8; ++e) rows[m] += ar[m][e];
      split3_bf16x8(ar[m], a[m][0], a[m][1], a[m][2]);
    }
    if (s + 1 < s1) {
      load_v(s + 1);
      load_a(s + 1);
    }
    __syncthreads();  // one per step: the stages alternate
    const __bf16* const b0 = st + (lane & 15) * D::CS + 8 * (lane >> 4);
#pragma unroll
    for (int n = 0; n < D::NB; ++n) {
      bf16x8 b[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        b[p] = *reinterpret_cast<const bf16x8*>(b0 + (p * NC + 16 * n) * D::CS);
#pragma unroll
      for (int m = 0; m < D::MT; ++m) acc[m][n] = mfma_split6(a[m], b, acc[m][n]);
    }
  }
  float* const dst = part + (size_t)range * (2 * H * H + 2 * H);
#pragma unroll
  for (int m = 0; m < D::MT; ++m) {
    const int r0 = 16 * (wave * D::MT + m);
#pragma unroll
    for (int n = 0; n < D::NB; ++n) {
      const int h = nb * NC + 16 * n + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = r0 + 4 * (lane >> 4) + r;
        float s = acc[m][n][r];
        if (__builtin_expect(!(fabsf(s) < INFINITY), 0)) {  // values the split cannot carry
          s = 0.0f;
          const uint32_t e1 = s1 * kDwTok < ntok ? s1 * kDwTok : ntok;
#pragma unroll 1
          for (uint32_t k = s0 * kDwTok; k < e1; ++k)
            s = fmaf(dp[(size_t)c * np + k], gelu_f(v[token_base(k, H, L) + (uint32_t)h * L]), s);
        }
        dst[(size_t)c * H + h] = s;
      }
    }
    float t = rows[m];
    t += __shfl_xor(t, 16);
    t += __shfl_xor(t, 32);
    if (nb == 0 && lane < 16) dst[(size_t)2 * H * H + r0 + lane] = t;
  }
}

// Sums the ranges in a fixed order: 16 threads per element take every 16th
// range, then a tree over them.
__global__ __launch_bounds__(256) void s4_dw_reduce_kernel(const float* __restrict__ part,
                                                           float* __restrict__ dw,
                                                           float* __restrict__ dbias, int nw, int nb,
                                                           int nranges) {
  __shared__ float s[16][17];
  const int e = threadIdx.x & 15, q = threadIdx.x >> 4;
  const int i = blockIdx.x * 16 + e, n = nw + nb;
  float acc = 0.0f;
  if (i < n)
    for (int r = q; r < nranges; r += 16) acc += part[(size_t)r * n + i];
  s[q][e] = acc;
  __syncthreads();
  if (q == 0 && i < n) {
    float t = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += s[k][e];
    if (i < nw) dw[i] = t;
    else dbias[i - nw] = t;
  }
}

}  // namespace pt
