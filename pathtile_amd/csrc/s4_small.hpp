// s4_small.hpp — the S4ConvD block's kernels besides the tail: taps and split
// weights, the taps' gradient, the reduction of the weight gradient's partials,
// and the model's ends. Included by s4_block.hip alone.

#pragma once

#include "s4_kernels.hpp"

namespace pt {

// ---------------------------------------------------------------------------
// Preparation: taps and split weights, one launch per block and pass.
// Blocks 0 .. H - 1 compute the taps of one channel; the others split W
// [2 H][H] into A-operand fragments of 64 lanes x 8 values (lane l holds row
// l % 16, contraction values 8 (l / 16) .. + 7), three parts each:
//   wf[((ct * 2 + half) * KS + ks) * 3 + part][lane][8]   rows of W
//   wt[(ct * 2 KS + ks) * 3 + part][lane][8]              rows of W^T
// so that a wave's fragment is one contiguous 1 KiB read. poles: dt [H], then
// Re A [H][N2], which the taps' gradient reads.
// The taps are the reference's formula in FP32 with exp(dt A) - 1 from
// expm1 and sin^2 (no cancellation at small dt A).
// ---------------------------------------------------------------------------
struct Cf { float re, im; };
__device__ __forceinline__ Cf cmul(Cf a, Cf b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
// b scaled by a power of two to about 1 first: |b|^2 would leave FP32's range
// where b itself is an ordinary value (below 1e-19 or above 1e19).
__device__ __forceinline__ Cf cdiv(Cf a, Cf b) {
  const float m = fmaxf(fabsf(b.re), fabsf(b.im));
  int e = 0;
  frexpf(m, &e);
  e = m > 0.0f && m < INFINITY ? -e : 0;
  b = {ldexpf(b.re, e), ldexpf(b.im, e)};
  const float d = 1.0f / (b.re * b.re + b.im * b.im);
  return {ldexpf((a.re * b.re + a.im * b.im) * d, e), ldexpf((a.im * b.re - a.re * b.im) * d, e)};
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
    float* __restrict__ poles, int H, int L, int N2, int transposed) {
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < H) {
    const int h = blockIdx.x;
    __shared__ float ce[2][kPrepStates], da[2][kPrepStates];
    __shared__ float part[kMaxL][kPrepStates + 1];
    const float dt = expf(log_dt[h]);
    if (tid == 0) poles[h] = dt;
    float acc = 0.0f;  // thread t < L: taps[h][t]
    for (int n0 = 0; n0 < N2; n0 += kPrepStates) {
      const int nn = N2 - n0 < kPrepStates ? N2 - n0 : kPrepStates;
      if (tid < nn) {
        const int i = h * N2 + n0 + tid;
        const Cf A = {-expf(log_a_re[i]), a_im[i]};
        poles[H + i] = A.re;
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
// dk [H][L] and the preparation's poles: with z = exp(dt A), E = z - 1,
// S0 = sum_t dk[t] z^t,
// S1 = sum_t t dk[t] z^t per state,
//   dL = 2 Re sum_n ( S0 E / A dC + R dA + (S0 C z + C_eff A S1) ddt ),
//   R  = S0 C / A^2 (z dt A - E) + dt C_eff S1,
// one workgroup per channel. z dt A - E cancels to second order in dt A, so
// that factor and E are computed in FP64 (a handful of operations per state).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kPrepThreads) void s4_taps_grad_kernel(
    const float* __restrict__ dk, const float* __restrict__ poles,
    const float* __restrict__ c_re, const float* __restrict__ c_im, const float* __restrict__ a_im,
    float* __restrict__ d_log_dt, float* __restrict__ d_c_re, float* __restrict__ d_c_im,
    float* __restrict__ d_log_a_re, float* __restrict__ d_a_im, float* __restrict__ d_skip,
    int L, int N2) {
  constexpr int kChunks = 8;  // threads per state
  __shared__ float sdk[kMaxL];
  __shared__ float s0r[kPrepStates][kChunks], s0i[kPrepStates][kChunks];
  __shared__ float s1r[kPrepStates][kChunks], s1i[kPrepStates][kChunks];
  __shared__ float ddt[kPrepStates];
  const int h = blockIdx.x, tid = threadIdx.x;
  const float* const a_re = poles + gridDim.x;  // after dt, one per channel
  if (tid < L) sdk[tid] = dk[h * L + tid];
  __syncthreads();
  const float dt = poles[h];
  float ddt_sum = 0.0f;  // thread 0
  for (int n0 = 0; n0 < N2; n0 += kPrepStates) {
    const int nn = N2 - n0 < kPrepStates ? N2 - n0 : kPrepStates;
    const int n = tid / kChunks, q = tid % kChunks;
    if (n < nn) {
      const int i = h * N2 + n0 + n;
      const Cf dA = {a_re[i] * dt, a_im[i] * dt};
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
      const double ar = a_re[i], ai = a_im[i], d = dt;
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


// ---------------------------------------------------------------------------
// The model's ends. Encoder: y[n][h] = sum_i x[n][i] w[h][i] + bias[h] over
// NI <= 8 input features; bound by the write of y and, backward, by the read
// of gy, which one pass turns into the gradients of w and bias. A thread keeps
// four channels (their weights or sums in registers) and walks tokens.
// ---------------------------------------------------------------------------
constexpr int kEndThreads = 256;
constexpr int kEncMaxIn = 8;
constexpr int kHeadMaxOut = 4;

template <int NI>
__global__ __launch_bounds__(kEndThreads) void s4_encode_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ y, uint32_t ntok, int H) {
  const int h4 = H / 4, c = threadIdx.x % h4, per = blockDim.x / h4;
  float wr[4][NI];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int i = 0; i < NI; ++i) wr[r][i] = w[(4 * c + r) * NI + i];
  const float4 b = reinterpret_cast<const float4*>(bias)[c];
  const uint32_t step = gridDim.x * per;
  for (uint32_t n = blockIdx.x * per + threadIdx.x / h4; n < ntok; n += step) {
    float xi[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) xi[i] = x[(size_t)n * NI + i];
    float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < NI; ++i) o[r] = fmaf(xi[i], wr[r][i], o[r]);
    reinterpret_cast<float4*>(y)[(size_t)n * h4 + c] =
        float4{o[0] + b.x, o[1] + b.y, o[2] + b.z, o[3] + b.w};
  }
}

// Partials [block][H NI + H] for s4_dw_reduce_kernel.
template <int NI>
__global__ __launch_bounds__(kEndThreads) void s4_encode_grad_kernel(
    const float* __restrict__ x, const float* __restrict__ gy, float* __restrict__ part,
    uint32_t ntok, int H) {
  __shared__ float red[kEndThreads][4 * (NI + 1) + 1];
  const int h4 = H / 4, c = threadIdx.x % h4, row = threadIdx.x / h4, per = blockDim.x / h4;
  float acc[4][NI + 1];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int i = 0; i <= NI; ++i) acc[r][i] = 0.0f;
  const uint32_t step = gridDim.x * per;
#pragma unroll 4
  for (uint32_t n = blockIdx.x * per + row; n < ntok; n += step) {
    const float4 g = reinterpret_cast<const float4*>(gy)[(size_t)n * h4 + c];
    const float gv[4] = {g.x, g.y, g.z, g.w};
    float xi[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) xi[i] = x[(size_t)n * NI + i];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int i = 0; i < NI; ++i) acc[r][i] = fmaf(gv[r], xi[i], acc[r][i]);
      acc[r][NI] += gv[r];
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int i = 0; i <= NI; ++i) red[threadIdx.x][r * (NI + 1) + i] = acc[r][i];
  __syncthreads();
  float* const dst = part + (size_t)blockIdx.x * (H * NI + H);
  for (int q = threadIdx.x; q < H * (NI + 1); q += blockDim.x) {
    const int h = q / (NI + 1), i = q % (NI + 1);
    float s = 0.0f;
    for (int k = 0; k < per; ++k) s += red[k * h4 + h / 4][(h % 4) * (NI + 1) + i];
    dst[i < NI ? h * NI + i : H * NI + h] = s;
  }
}

// Head: out[b][o] = sum_h w[o][h] x[b][L-1][h] + bias[o], one wave per sample
// (NO <= 4 outputs).
__global__ __launch_bounds__(kEndThreads) void s4_head_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ out, int B, int H, int L, int NO) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b = blockIdx.x * (kEndThreads / kWave) + wave;
  if (b >= B) return;
  const float* row = x + ((size_t)b * L + L - 1) * H;
  for (int o = 0; o < NO; ++o) {
    float s = 0.0f;
    for (int h = lane; h < H; h += kWave) s = fmaf(row[h], w[o * H + h], s);
    s = wave_sum(s);
    if (lane == 0) out[b * NO + o] = s + bias[o];
  }
}

// Its gradients: gx is gy w in the last column and zero elsewhere (the write
// of gx bounds it), with the partials [block][NO H + NO] of the weight and
// bias gradients on the way.
__global__ __launch_bounds__(kEndThreads) void s4_head_grad_kernel(
    const float* __restrict__ x, const float* __restrict__ gy, const float* __restrict__ w,
    float* __restrict__ gx, float* __restrict__ part, int B, int H, int L, int NO, int per) {
  const int h4 = H / 4, n4 = L * h4;
  const int b0 = blockIdx.x * per, b1 = b0 + per < B ? b0 + per : B;
  const int c = threadIdx.x;  // channels 4 c .. of the weight gradient
  float acc[kHeadMaxOut][4], accb[kHeadMaxOut];
#pragma unroll
  for (int o = 0; o < kHeadMaxOut; ++o) {
    accb[o] = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[o][r] = 0.0f;
  }
  for (int b = b0; b < b1; ++b) {
    float g[kHeadMaxOut];
#pragma unroll
    for (int o = 0; o < kHeadMaxOut; ++o) g[o] = o < NO ? gy[b * NO + o] : 0.0f;
    if (gx) {
      float4* dst = reinterpret_cast<float4*>(gx) + (size_t)b * n4;
      for (int i = threadIdx.x; i < n4 - h4; i += kEndThreads) dst[i] = float4{0.f, 0.f, 0.f, 0.f};
      if (c < h4) {
        float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int o = 0; o < kHeadMaxOut; ++o)
          if (o < NO)
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = fmaf(g[o], w[o * H + 4 * c + r], v[r]);
        dst[n4 - h4 + c] = float4{v[0], v[1], v[2], v[3]};
      }
    }
    if (c < h4) {
      const float4 xv = reinterpret_cast<const float4*>(x)[(size_t)b * n4 + n4 - h4 + c];
#pragma unroll
      for (int o = 0; o < kHeadMaxOut; ++o) {
        acc[o][0] = fmaf(g[o], xv.x, acc[o][0]);
        acc[o][1] = fmaf(g[o], xv.y, acc[o][1]);
        acc[o][2] = fmaf(g[o], xv.z, acc[o][2]);
        acc[o][3] = fmaf(g[o], xv.w, acc[o][3]);
        accb[o] += g[o];
      }
    }
  }
  float* const dst = part + (size_t)blockIdx.x * (NO * H + NO);
#pragma unroll
  for (int o = 0; o < kHeadMaxOut; ++o)
    if (o < NO) {
      if (c < h4)
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[o * H + 4 * c + r] = acc[o][r];
      if (c == 0) dst[NO * H + o] = accb[o];
    }
}

}  // namespace pt
