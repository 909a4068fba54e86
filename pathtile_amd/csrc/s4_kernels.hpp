// s4_kernels.hpp — device code of the S4ConvD block around the depthwise
// Conv1D (kernels/warp_tiled_ampere.py:1122-1190 in the reference), FP32,
// for MI355X (gfx950, wave64).
//
// One block computes, for x [B, L, H] and N2 complex states per channel,
//   taps[h][t] = 2 Re sum_n C_eff[h,n] exp(dt[h] A[h,n] t)  (+ skip at L / 2)
//   u [b,t,h]  = conv(x, taps) over t,  v = dropout(u),  g = gelu(v)
//   P [b,t,c]  = sum_h W[c][h] g[b,t,h] + bias[c],  c < 2 H
//   y [b,t,c]  = P[c] sigmoid(P[H + c]) + x[b,t,c],  c < H
// in [B, L, H] throughout. The convolution and its input gradient are in
// s4_conv.hpp, its weight gradient is the channels-last DK of
// dwconv1d_kernels.hpp, taps, their gradient and the model's ends are in
// s4_small.hpp. Here is the tail (GELU, projection, GLU, residual) with its
// backward, each one pass over its tensors. The tail treats the B L columns as
// one list of tokens (token = b L + t), so its tiles do not depend on L.
//
// The projection runs on the BF16 matrix cores with both operands split into
// three BF16 parts (split3_bf16x8; six of the nine part products, dropped
// terms at most about 2^-22 of a product), which keeps FP32 accuracy at
// 1.55x the FP32 matrix instructions' rate.

#pragma once

#include "dwconv1d_kernels.hpp"

namespace pt {

constexpr int kS4MaxH = 256;     // largest H of the fused block (H % 32 == 0)
constexpr int kDwTok = 32;       // tokens per block of dP and step of the weight gradient

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
  // tokens per forward tile: the LDS holds the stages of 64 tokens up to H = 128
  static constexpr int TOK = CT <= 8 ? 64 : 32;
  // tokens per backward tile, and whether the LDS holds two dP stages of them
  static constexpr int BTOK = 16 * WPT > 32 ? 16 * WPT : 32;
  static constexpr bool TWO = CT <= 8;
};

__host__ __device__ constexpr int tail_tok(int H) { return H <= 128 ? 64 : 32; }
__host__ __device__ constexpr size_t tail_fwd_lds(int H) {  // two g stages, the output stage
  return (size_t)tail_tok(H) * (2 * 3 * (H + 8) * 2 + (H + 4) * 4);
}
// Byte offset of dP's (token, row) from the tile's first block of 32 tokens.
template <int H>
__device__ __forceinline__ uint32_t dp_offset(uint32_t tk, uint32_t row) {
  return 4 * ((tk / kDwTok) * (2 * H * kDwTok) + row * kDwTok + tk % kDwTok);
}

template <int CT>
constexpr size_t tail_bwd_lds() {  // dP parts
  return (size_t)(TailGeo<CT>::TWO ? 2 : 1) * 3 * TailGeo<CT>::BTOK * TailGeo<CT>::PS * 2;
}

// Values of the split weights in the workspace: W as A operands of the
// forward product, then W^T as A operands of the backward one.
__host__ __device__ constexpr size_t wfrag_values(int H) { return (size_t)3 * 2 * H * H; }

// The normal distribution function without branches: for a = |x|,
// Q(a) = 1 - cdf(a) = exp(-a^2 / 2) R(a) with R(a) = erfcx(a / sqrt 2) / 2 as
// t times a polynomial of degree 7 in t = 1 / (1 + 9/32 a); 20 instructions
// where erff takes about 75 on both of its branches. The fit minimises the
// largest max(1, a) |error of Q| over 0 <= a <= 8 (Lawson's weighted least
// squares), its coefficients rounded to FP32 from the constant up with the
// others fitted again: 3.9e-10 of the cdf and of gelu, of which 2.1e-10 before
// the rounding (the CPU tests fit it anew). The
// exponential also gives the density. a is cut at 20, where Q underflows, so
// that infinities keep the formula's values (gelu(-inf) = NaN).
struct NormalCdf {
  float cdf, e;  // e = exp(-x^2 / 2)
};
__device__ __forceinline__ NormalCdf normal_cdf(float x) {
  const float a = fminf(fabsf(x), 20.0f);
  const float d = fmaf(0.28125f, a, 1.0f);
  float t = __builtin_amdgcn_rcpf(d);
  t = fmaf(t, fmaf(-d, t, 1.0f), t);
  const float s = a * a;
  const float e = __builtin_amdgcn_exp2f(-fmaf(s, 0.72134751081466675f, s * 9.6298152e-09f));
  float r = 0.0391756147146225f;
  r = fmaf(r, t, -0.20986095070838928f);
  r = fmaf(r, t, 0.37282636761665344f);
  r = fmaf(r, t, -0.21809245645999908f);
  r = fmaf(r, t, 0.22155848145484924f);
  r = fmaf(r, t, 0.06441713869571686f);
  r = fmaf(r, t, 0.11812617629766464f);
  r = fmaf(r, t, 0.11184962838888168f);
  const float q = r * t * e;
  return {x < 0.0f ? q : 1.0f - q, e};
}

__device__ __forceinline__ float gelu_f(float x) { return x * normal_cdf(x).cdf; }

__device__ __forceinline__ float gelu_grad_f(float x) {
  const NormalCdf n = normal_cdf(x);
  return fmaf(x, n.e * 0.39894228040143268f, n.cdf);
}

// 1 / (1 + exp(-x)), NaN kept; above 87 the result is 1, and 0 where exp(-x)
// is past FP32's range (an infinite value times such a gate is NaN).
__device__ __forceinline__ float sigmoid_f(float x) {
  const float c = x > 87.0f ? 87.0f : x < -87.0f ? -87.0f : x;
  const float d =
      1.0f + __builtin_amdgcn_exp2f(-fmaf(c, 1.44269502162933349609375f, c * 1.92596303e-08f));
  const float t = __builtin_amdgcn_rcpf(d);
  return x < -88.7228394f ? 0.0f : fmaf(t, fmaf(-d, t, 1.0f), t);
}

__device__ __forceinline__ bool finite4(float a, float b, float c, float d) {
  return fabsf(a) + fabsf(b) + fabsf(c) + fabsf(d) < INFINITY;
}

__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
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
// Tail, shared pieces
// ---------------------------------------------------------------------------
// Element offset of (token n, channel 0) in a [B, H, L] tensor. magic =
// floor(2^32 / L) + 1 (0 at L = 1): umulhi(n, magic) = n / L for every
// n < 2^32 / L, and there are at most 2^31 / 32 tokens.
__device__ __forceinline__ uint32_t token_sample(uint32_t n, uint32_t magic) {
  return magic ? __umulhi(n, magic) : n;
}
__device__ __forceinline__ uint32_t token_base(uint32_t n, uint32_t H, uint32_t L, uint32_t magic) {
  const uint32_t b = token_sample(n, magic);
  return b * (H * L) + (n - b * L);
}

// A [B, H, L] tensor (elements of `size` bytes) from the sample of token n0
// on, as a buffer that ends with the tensor: loads of later tokens read 0 and
// stores to them are dropped, without a branch. Byte offsets within a tile
// stay far below 2 GiB (64 tokens touch at most 65 samples at L = 1).
struct Slab {
  __amdgpu_buffer_rsrc_t r;
  uint32_t first;  // element offset of the slab
};
template <int SIZE = 4>
__device__ __forceinline__ Slab make_slab(const void* t, uint32_t n0, uint32_t ntok, uint32_t H,
                                          uint32_t L, uint32_t magic) {
  const uint32_t first = token_sample(n0, magic) * (H * L), all = ntok * H;
  const uint64_t left = first < all ? (uint64_t)(all - first) * SIZE : 0;
  const uint32_t bytes = left < (uint64_t)kNumRecords ? (uint32_t)left : (uint32_t)kNumRecords;
  return {__builtin_amdgcn_make_buffer_rsrc(
              const_cast<char*>(static_cast<const char*>(t)) + (size_t)first * SIZE, 0, (int)bytes,
              kRsrcWord3),
          first};
}
// Rows n0 .. of a [tokens, H] tensor.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_token_rows(const float* t, uint32_t n0,
                                                                  uint32_t ntok, uint32_t H) {
  const uint64_t left = n0 < ntok ? (uint64_t)(ntok - n0) * H * 4 : 0;
  const uint32_t bytes = left < (uint64_t)kNumRecords ? (uint32_t)left : (uint32_t)kNumRecords;
  return make_rsrc_n(t + (size_t)n0 * H, bytes);
}

// gelu of TOK tokens' values, split into the three parts of the LDS stage
// [part][token][GS]: a lane takes eight channels of one token, 32 consecutive
// bytes. store<I, N> does the I-th of N slices of the work.
template <int CT, int TOK>
struct GeluStage {
  using G = TailGeo<CT>;
  static constexpr int TH = G::NW * kWave, kUnits = TOK * (G::H / 8), CPT = G::H / 8;
  static constexpr int U = (kUnits + TH - 1) / TH;
  float x[U][8];

  __device__ __forceinline__ void load(const float* __restrict__ v, uint32_t n0, uint32_t ntok) {
    const __amdgpu_buffer_rsrc_t r = make_token_rows(v, n0, ntok, G::H);
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int u = threadIdx.x + i * TH;
      const uint32_t o = kUnits % TH == 0 || u < kUnits ? 32 * u : kOob;
      const float4 a = buf_load4(r, o, 0), b = buf_load4(r, o + 16, 0);
      x[i][0] = a.x;
      x[i][1] = a.y;
      x[i][2] = a.z;
      x[i][3] = a.w;
      x[i][4] = b.x;
      x[i][5] = b.y;
      x[i][6] = b.z;
      x[i][7] = b.w;
    }
  }

  template <int I, int N>
  __device__ __forceinline__ void store(__bf16* sg) {
#pragma unroll
    for (int e = 8 * U * I / N; e < 8 * U * (I + 1) / N; ++e) {
      const int i = e / 8, u = threadIdx.x + i * TH;
      const bool on = kUnits % TH == 0 || u < kUnits;
      x[i][e % 8] = gelu_f(x[i][e % 8]);  // 0 past the last token
      if (e % 8 == 7) {
        bf16x8 hi, mid, lo;
        split3_bf16x8(x[i], hi, mid, lo);
        // units past the end write to a row padding that nothing reads
        __bf16* d = sg + (on ? (u / CPT) * G::GS + 8 * (u % CPT) : (u % TOK) * G::GS + G::H);
        *reinterpret_cast<bf16x8*>(d) = hi;
        *reinterpret_cast<bf16x8*>(d + TOK * G::GS) = mid;
        *reinterpret_cast<bf16x8*>(d + 2 * TOK * G::GS) = lo;
      }
    }
  }
};

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

// Weight fragments of M row tiles and KS contraction steps, streamed from the
// L2 (the next step's load while a step multiplies) or kept in registers.
template <int M, int KS>
struct StreamedFrags {
  const __bf16* w0;
  const __bf16* w;
  bf16x8 a[2][M][3];
  __device__ __forceinline__ explicit StreamedFrags(const __bf16* p) : w0(p), w(p) {}
  __device__ __forceinline__ void begin() {
    // Opaque to the compiler, which would otherwise keep every fragment in
    // registers over the tile loop and spill.
    uint32_t zero = 0;
    asm volatile("" : "+s"(zero));
    w = w0 + zero;
    load_frags<M>(a[0], w, KS);
  }
  template <int ks>
  __device__ __forceinline__ void ahead() {
    if constexpr (ks + 1 < KS) load_frags<M>(a[(ks + 1) & 1], w + (ks + 1) * 3 * 512, KS);
  }
  template <int ks>
  __device__ __forceinline__ bf16x8 frag(int m, int p) const { return a[ks & 1][m][p]; }
};
template <int M, int KS>
struct ResidentFrags {
  bf16x8 a[KS][M][3];
  __device__ __forceinline__ explicit ResidentFrags(const __bf16* p) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) load_frags<M>(a[ks], p + ks * 3 * 512, KS);
  }
  __device__ __forceinline__ void begin() {}
  template <int ks>
  __device__ __forceinline__ void ahead() {}
  template <int ks>
  __device__ __forceinline__ bf16x8 frag(int m, int p) const { return a[ks][m][p]; }
};

// acc[m][nt] = M row tiles of the weights (fragments from w0, KS steps) times
// NT token tiles of the stage from b0 on (row stride RS, parts TOK * RS
// apart). The next step's fragments load while a step multiplies, and
// shadow(step) adds vector work that runs beside the step's products.
template <int M, int NT, int KS, int RS, int TOK, typename W, typename F>
__device__ __forceinline__ void multiply(f32x4 (&acc)[M][NT], W& w, const __bf16* b0, F&& shadow) {
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[m][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  static_for<0, KS>([&](auto step) {
    constexpr int ks = decltype(step)::value;
    w.template ahead<ks>();
    if constexpr (ks > 0 && step_negated(ks) != step_negated(ks - 1))
      negate(reinterpret_cast<f32x4(&)[M * NT]>(acc));
    bf16x8 b[NT][3];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        b[nt][p] = *reinterpret_cast<const bf16x8*>(b0 + (p * TOK + 16 * nt) * RS + 32 * ks);
    // after the reads in program order: its LDS writes cannot pass them
    shadow(step);
    // one product of every tile after the other: an accumulator's next
    // product waits for its last
    constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};  // small ones first
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int m = 0; m < M; ++m)
          acc[m][nt] = mfma_bf16(w.template frag<ks>(m, pa[q]), b[nt][pb[q]], acc[m][nt]);
    __builtin_amdgcn_sched_barrier(0);
  });
  if constexpr (step_negated(KS - 1)) negate(reinterpret_cast<f32x4(&)[M * NT]>(acc));
}

// One pre-activation of one token by the FP32 chain, for values that the
// split cannot carry (Inf, NaN, or rounding past BF16's largest value).
__device__ __forceinline__ float project_one(const float* v, const float* __restrict__ w, int row,
                                             int H) {
  float s = 0.0f;
#pragma unroll 1
  for (int h = 0; h < H; ++h) s = fmaf(w[(size_t)row * H + h], gelu_f(v[h]), s);
  return s;
}

__device__ __forceinline__ void set_elem(f32x4& a, int r, float v) {
  a[0] = r == 0 ? v : a[0];
  a[1] = r == 1 ? v : a[1];
  a[2] = r == 2 ? v : a[2];
  a[3] = r == 3 ? v : a[3];
}

// Recomputes a lane's four value and gate sums where one is not finite; v are
// the token's values.
__device__ __forceinline__ void project_fix(f32x4& a, f32x4& b, const float* v,
                                            const float* __restrict__ w, int c, int H) {
#pragma unroll 1
  for (int r = 0; r < 4; ++r) {
    set_elem(a, r, project_one(v, w, c + r, H));
    set_elem(b, r, project_one(v, w, H + c + r, H));
  }
}

// ---------------------------------------------------------------------------
// Tail forward: y = GLU(W gelu(v) + bias) + x, all [tokens][H].
// A persistent workgroup, one per CU, walks tiles of 64 tokens (32 above
// H = 128, what the LDS holds). gelu is as much vector work as the products
// are matrix work, and both kinds from one wave overlap where they are
// interleaved in one stretch of code (two workgroups that share a CU fall
// into step instead and add the two up: 452 us at B16384 L48 H128 against 388),
// so tile t + 1's gelu and split run in the shadow of tile t's products, into
// the other of two stages. The weight fragments stay in registers up to H = 128
// (streamed from the L2 they cost 511 us) and stream above. For a later backward, q [2][tokens][H] gets
// the values P[c] + bias and the gates' sigmoids. GLU results pass through an
// FP32 stage to flat 16-byte rows with the residual. Averages of a trace at
// B16384 L48 H128: 442 us, 459 with q (4.4 TB/s, matrix cores 32% and VALU 45%
// busy).
// ---------------------------------------------------------------------------
template <int CT>
__global__ __launch_bounds__(TailGeo<CT>::NW* kWave, 2) void s4_tail_fwd_kernel(
    const float* __restrict__ v, const float* __restrict__ x, const __bf16* __restrict__ wf,
    const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ y,
    float* __restrict__ q, uint32_t ntok, uint32_t ntiles) {
  using G = TailGeo<CT>;
  constexpr int TOK = G::TOK, NT = TOK / 16 / G::WPT, SZ = 3 * TOK * G::GS, TH = G::NW * kWave;
  constexpr int R4 = TOK * G::H / 4 / TH;  // 16-byte pieces of a tile's rows per thread
  static_assert(TOK * G::H / 4 % TH == 0 && NT >= 1, "whole pieces and token tiles");
  extern __shared__ __align__(16) char smem[];
  __bf16* const sg = reinterpret_cast<__bf16*>(smem);
  float* const so = reinterpret_cast<float*>(smem + (size_t)2 * SZ * 2);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ct0 = (wave % G::WPC) * G::MT, nt0 = (wave / G::WPC) * NT;
  const int tk0 = 16 * nt0 + (lane & 15);     // this lane's token of tile nt: tk0 + 16 nt
  const int c0 = 16 * ct0 + 4 * (lane >> 4);  // this lane's channels: c0 + 16 m + r
  const __bf16* const w0 = wf + (size_t)ct0 * 2 * G::KS * 3 * 512 + lane * 8;
  std::conditional_t<CT <= 8, ResidentFrags<2 * G::MT, G::KS>, StreamedFrags<2 * G::MT, G::KS>>
      frags(w0);
  GeluStage<CT, TOK> stage;
  stage.load(v, blockIdx.x * TOK, ntok);
  stage.template store<0, 1>(sg);
  stage.load(v, (blockIdx.x + gridDim.x) * TOK, ntok);
  uint32_t cur = 0;
  for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x, cur ^= 1) {
    const uint32_t n0 = tile * TOK;
    __syncthreads();  // stage `cur` is written, the output stage read
    const __amdgpu_buffer_rsrc_t xr = make_token_rows(x, n0, ntok, G::H);
    float4 res[R4];
#pragma unroll
    for (int i = 0; i < R4; ++i) res[i] = buf_load4(xr, 16 * (threadIdx.x + i * TH), 0);
    f32x4 acc[2 * G::MT][NT];
    frags.begin();
    multiply<2 * G::MT, NT, G::KS, G::GS, TOK>(
        acc, frags, sg + cur * SZ + tk0 * G::GS + 8 * (lane >> 4), [&](auto ks) {
          stage.template store<decltype(ks)::value, G::KS>(sg + (cur ^ 1) * SZ);
        });
    stage.load(v, (tile + 2 * gridDim.x) * TOK, ntok);
#pragma unroll
    for (int m = 0; m < G::MT; ++m) {
      const int c = c0 + 16 * m;
      const float4 ba = *reinterpret_cast<const float4*>(bias + c);
      const float4 bb = *reinterpret_cast<const float4*>(bias + G::H + c);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int tk = tk0 + 16 * nt;
        f32x4 a = acc[2 * m][nt], b = acc[2 * m + 1][nt];
        if (__builtin_expect(!(finite4(a[0], a[1], a[2], a[3]) && finite4(b[0], b[1], b[2], b[3])), 0)) {
          if (n0 + tk < ntok) project_fix(a, b, v + (size_t)(n0 + tk) * G::H, w, c, G::H);
        }
        const float4 pa = {a[0] + ba.x, a[1] + ba.y, a[2] + ba.z, a[3] + ba.w};
        const float4 ps = {sigmoid_f(b[0] + bb.x), sigmoid_f(b[1] + bb.y), sigmoid_f(b[2] + bb.z),
                           sigmoid_f(b[3] + bb.w)};
        *reinterpret_cast<float4*>(so + tk * G::OS + c) =
            float4{pa.x * ps.x, pa.y * ps.y, pa.z * ps.z, pa.w * ps.w};
        if (q) {
          const uint32_t o = 4 * (tk * G::H + c);
          buf_store4(pa, make_token_rows(q, n0, ntok, G::H), o);
          buf_store4(ps, make_token_rows(q + (size_t)ntok * G::H, n0, ntok, G::H), o);
        }
      }
    }
    __syncthreads();
    const __amdgpu_buffer_rsrc_t yr = make_token_rows(y, n0, ntok, G::H);
#pragma unroll
    for (int i = 0; i < R4; ++i) {
      const int q = threadIdx.x + i * TH, tk = q / (G::H / 4), c = 4 * (q % (G::H / 4));
      const float4 o = *reinterpret_cast<const float4*>(so + tk * G::OS + c);
      buf_store4(float4{o.x + res[i].x, o.y + res[i].y, o.z + res[i].z, o.w + res[i].w}, yr, 16 * q);
    }
  }
}

// ---------------------------------------------------------------------------
// Tail backward with respect to its input: from gy [tokens][H] and the
// forward's q and v, du = dL/du [tokens][H] (through GLU, projection, gelu and the dropout mask)
// and dP [blocks of 32 tokens][2 H][32] (zero past the last token) for the
// weight gradient, whose loads it makes whole lines. A persistent workgroup walks tiles of 32 tokens (64 at
// H = 32): tile t's product W^T dP from LDS, the weight fragments resident up
// to H = 128, and in its shadow tile t + 1's GLU gradient into the other of
// two dP stages and tile t - 1's gelu gradient; one barrier per tile. Above
// H = 128 the LDS holds one stage, the GLU gradient comes before the product
// and the fragments stream. Seven tensor passes of HBM bound it; recomputing
// the pre-activations instead of reading q took 5 passes but 975 us at B16384
// L48 H128 on the sum of its matrix and vector work, 698 with q read (the
// forward, which writes it, 388 -> 483 then). Now 632 us in a trace (4.5 TB/s,
// matrix cores 22% and VALU 33% busy).
// ---------------------------------------------------------------------------
template <int CT, bool MASK>
__global__ __launch_bounds__(TailGeo<CT>::NW* kWave, 2) void s4_tail_bwd_kernel(
    const float* __restrict__ gy, const float* __restrict__ q, const float* __restrict__ v,
    const uint8_t* __restrict__ mask, float scale, const __bf16* __restrict__ wf,
    const float* __restrict__ w, float* __restrict__ du, float* __restrict__ dp, uint32_t ntok,
    uint32_t L, uint32_t magic, uint32_t ntiles) {
  using G = TailGeo<CT>;
  constexpr int TOK = G::BTOK, NT = TOK / 16 / G::WPT, SZ = 3 * TOK * G::PS, KS = 2 * G::KS;
  static_assert(NT >= 1, "every wave has tokens");
  typedef __bf16 bf16x4v __attribute__((ext_vector_type(4)));
  extern __shared__ __align__(16) char smem[];
  __bf16* const sp = reinterpret_cast<__bf16*>(smem);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ct0 = (wave % G::WPC) * G::MT, nt0 = (wave / G::WPC) * NT;
  const int tk0 = 16 * nt0 + (lane & 15);
  const int c0 = 16 * ct0 + 4 * (lane >> 4);
  std::conditional_t<G::TWO, ResidentFrags<G::MT, KS>, StreamedFrags<G::MT, KS>> frags(
      wf + wfrag_values(G::H) + (size_t)ct0 * KS * 3 * 512 + lane * 8);
  constexpr int E = G::MT * NT * 4;  // du values per lane and tile: (m, nt, r)

  // GLU gradient of the tile whose q and gy are loaded
  struct Glu {
    float4 q1[G::MT][NT], q2[G::MT][NT], g4[G::MT][NT];
  };
  Glu ga, gb;
  auto load_glu = [&](Glu& s, uint32_t n0) {
    const __amdgpu_buffer_rsrc_t r1 = make_token_rows(q, n0, ntok, G::H);
    const __amdgpu_buffer_rsrc_t r2 = make_token_rows(q + (size_t)ntok * G::H, n0, ntok, G::H);
    const __amdgpu_buffer_rsrc_t rg = make_token_rows(gy, n0, ntok, G::H);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int m = 0; m < G::MT; ++m) {
        const uint32_t o = 4 * ((tk0 + 16 * nt) * G::H + c0 + 16 * m);
        s.q1[m][nt] = buf_load4(r1, o, 0);
        s.q2[m][nt] = buf_load4(r2, o, 0);
        s.g4[m][nt] = buf_load4(rg, o, 0);
      }
  };
  float pa[8];  // four value and four gate gradients
  auto glu = [&](const Glu& in_, auto slice, auto slices, uint32_t n0, __bf16* st) {
    constexpr int I = decltype(slice)::value, N = decltype(slices)::value;
    // past the last tile the stores are dropped
    const __amdgpu_buffer_rsrc_t dr =
        make_rsrc_n(dp + (size_t)n0 * (2 * G::H), n0 < ntok ? 2 * G::H * TOK * 4 : 0);
#pragma unroll
    for (int e = E * I / N; e < E * (I + 1) / N; ++e) {
      const int r = e % 4, m = e / 4 % G::MT, nt = e / 4 / G::MT;
      const int tk = tk0 + 16 * nt, c = c0 + 16 * m;
      const bool in = n0 + tk < ntok;
      const float a = (&in_.q1[m][nt].x)[r], s = (&in_.q2[m][nt].x)[r];
      const float g = (&in_.g4[m][nt].x)[r];
      pa[r] = in ? s * g : 0.0f;
      pa[4 + r] = in ? (1.0f - s) * s * g * a : 0.0f;
      buf_store1(pa[r], dr, dp_offset<G::H>(tk, c + r));
      buf_store1(pa[4 + r], dr, dp_offset<G::H>(tk, G::H + c + r));
      if (r == 3) {
        bf16x8 parts[3];
        split3_bf16x8(pa, parts[0], parts[1], parts[2]);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          __bf16* d = st + (p * TOK + tk) * G::PS + c;
          *reinterpret_cast<bf16x4v*>(d) =
              bf16x4v{parts[p][0], parts[p][1], parts[p][2], parts[p][3]};
          *reinterpret_cast<bf16x4v*>(d + G::H) =
              bf16x4v{parts[p][4], parts[p][5], parts[p][6], parts[p][7]};
        }
      }
    }
  };

  // gelu gradient of a finished product: its values, mask and where du goes
  // (nowhere before the first tile)
  f32x4 dg[G::MT][NT];
  struct Vals {
    float4 vv[G::MT][NT];
    uint32_t mk[MASK ? G::MT : 1][MASK ? NT : 1][4];
  };
  Vals la, lb;
  __amdgpu_buffer_rsrc_t out = make_token_rows(du, ntok, ntok, G::H);
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
    for (int m = 0; m < G::MT; ++m) {
      dg[m][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
      lb.vv[m][nt] = float4{0.f, 0.f, 0.f, 0.f};
      if constexpr (MASK) {
#pragma unroll
        for (int r = 0; r < 4; ++r) lb.mk[m][nt][r] = 0;
      }
    }
  }
  float o4[4];
  auto finish = [&](const Vals& l, auto slice, auto slices) {
    constexpr int I = decltype(slice)::value, N = decltype(slices)::value;
#pragma unroll
    for (int e = E * I / N; e < E * (I + 1) / N; ++e) {
      const int r = e % 4, m = e / 4 % G::MT, nt = e / 4 / G::MT;
      o4[r] = dg[m][nt][r] * gelu_grad_f((&l.vv[m][nt].x)[r]);
      if constexpr (MASK) o4[r] = o4[r] * (float)l.mk[m][nt][r] * scale;
      if (r == 3)
        buf_store4(float4{o4[0], o4[1], o4[2], o4[3]}, out,
                   4 * ((tk0 + 16 * nt) * G::H + c0 + 16 * m));
    }
  };
  using All = std::integral_constant<int, 1>;
  using Steps = std::integral_constant<int, KS>;
  using Zero = std::integral_constant<int, 0>;

  uint32_t cur = 0;
  // One tile. `now` holds the GLU inputs of the tile that this call's shadow
  // (or, with one stage, its start) works on; `then` is loaded for the call
  // after, a whole tile ahead of its use, as are `vals` for the tile's own
  // gelu gradient, which runs in the next call's shadow.
  auto body = [&](uint32_t tile, const Glu& now, Glu& then, Vals& vals, const Vals& before) {
    const uint32_t n0 = tile * TOK, next = (tile + gridDim.x) * TOK;
    if constexpr (!G::TWO) {
      __syncthreads();  // the stage is read
      glu(now, Zero{}, All{}, n0, sp);
    }
    __threadfence_block();
    __syncthreads();  // tile t's dP parts are written
    frags.begin();
    load_glu(then, G::TWO ? next + gridDim.x * TOK : next);
    const __amdgpu_buffer_rsrc_t in = make_token_rows(v, n0, ntok, G::H);
    const Slab ms = make_slab<1>(mask, n0, ntok, G::H, L, magic);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int m = 0; m < G::MT; ++m) {
        vals.vv[m][nt] = buf_load4(in, 4 * ((tk0 + 16 * nt) * G::H + c0 + 16 * m), 0);
        if constexpr (MASK) {
          const uint32_t at = token_base(n0 + tk0 + 16 * nt, G::H, L, magic) - ms.first +
                              (uint32_t)(c0 + 16 * m) * L;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            vals.mk[m][nt][r] = __builtin_amdgcn_raw_buffer_load_b8(ms.r, at + r * L, 0, 0);
        }
      }
    f32x4 dgn[G::MT][NT];
    multiply<G::MT, NT, KS, G::PS, TOK>(
        dgn, frags, sp + cur * SZ + tk0 * G::PS + 8 * (lane >> 4), [&](auto ks) {
          finish(before, ks, Steps{});
          if constexpr (G::TWO) glu(now, ks, Steps{}, next, sp + (cur ^ 1) * SZ);
        });
    out = make_token_rows(du, n0, ntok, G::H);
    cur ^= G::TWO;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const uint32_t n = n0 + tk0 + 16 * nt;
#pragma unroll
      for (int m = 0; m < G::MT; ++m) {
        f32x4 d = dgn[m][nt];
        if (__builtin_expect(!finite4(d[0], d[1], d[2], d[3]), 0)) {
          if (n < ntok) {
#pragma unroll 1
            for (int r = 0; r < 4; ++r) {
              const int c = c0 + 16 * m + r;
              float s = 0.0f;
#pragma unroll 1
              for (int o = 0; o < 2 * G::H; ++o)
                s = fmaf(w[(size_t)o * G::H + c],
                         dp[(size_t)n0 * (2 * G::H) + dp_offset<G::H>(n - n0, o) / 4], s);
              set_elem(d, r, s);
            }
          }
        }
        dg[m][nt] = d;
      }
    }
  };

  load_glu(ga, blockIdx.x * TOK);
  if constexpr (G::TWO) {
    glu(ga, Zero{}, All{}, blockIdx.x * TOK, sp);
    load_glu(ga, (blockIdx.x + gridDim.x) * TOK);
  }
  uint32_t tile = blockIdx.x;
  while (true) {
    if (tile >= ntiles) {
      finish(lb, Zero{}, All{});
      break;
    }
    body(tile, ga, gb, la, lb);
    tile += gridDim.x;
    if (tile >= ntiles) {
      finish(la, Zero{}, All{});
      break;
    }
    body(tile, gb, ga, lb, la);
    tile += gridDim.x;
  }
}

// ---------------------------------------------------------------------------
// Weight gradient of the projection: dW[c][h] = sum_tok dP[c][tok] g[h][tok]
// and dbias[c] = sum_tok dP[c][tok], split over the tokens. A workgroup takes
// a contiguous run of 32-token steps and NB channels (columns); its waves own
// rows of dP, read straight from memory in the A layout (a step's block is
// contiguous) and split in registers; g is computed, split and
// shared through LDS [part][channel][40]. Partials [range][2 H H + 2 H] go to
// the workspace for a fixed-order reduction. Step s + 1's gelu and splits run
// in the shadow of step s's products: 354 us at B16384 L48 H128, 430 with them
// ahead of the products; with two sets of loads in flight 315 (matrix cores 47%
// and VALU 55% busy). The matrix instruction's rounding towards minus infinity
// (step_negated) is not cancelled here: it moves dW by -2.8e-6 of its mean
// magnitude there, of an error against FP64 of 2.3e-6 (7.4e-6 as a library FP32
// product; B2048 L48 H128 4.3e-7 against 3.5e-6).
// ---------------------------------------------------------------------------
template <int CT>
struct DwGeo {
  static constexpr int RT = 2 * CT;  // row tiles
  static constexpr int NW = RT % 8 == 0 ? 8 : RT == 4 ? 4 : RT == 12 ? 6 : RT / 4;
  static constexpr int MT = RT / NW;
  // column tiles per workgroup, so that the accumulators leave room for the loads
  static constexpr int NB = CT <= 8 ? CT : CT % 4 == 0 ? CT / 4 : CT / 2;
  static constexpr bool DEEP = CT <= 8 || CT == 12;     // two sets of loads in flight
  static constexpr bool AHEAD = CT <= 8 || CT % 4 == 0;  // rows split a step ahead
  static constexpr int SPLIT = CT / NB;
  static constexpr int CS = kDwTok + 8;  // BF16 values per channel row of a part
  static constexpr size_t lds = (size_t)2 * 3 * NB * 16 * CS * 2;
};

template <int CT>
__global__ __launch_bounds__(DwGeo<CT>::NW* kWave, 2) void s4_dw_kernel(
    const float* __restrict__ dp, const float* __restrict__ v, float* __restrict__ part,
    uint32_t ntok, uint32_t nsteps, uint32_t steps_per) {
  using D = DwGeo<CT>;
  constexpr int H = 16 * CT, NC = 16 * D::NB, TH = D::NW * kWave;
  constexpr int kUnits = NC * (kDwTok / 8);  // (channel, eight tokens)
  constexpr int U = (kUnits + TH - 1) / TH;
  constexpr int SZ = 3 * NC * D::CS;
  extern __shared__ __align__(16) char smem[];
  __bf16* const sg = reinterpret_cast<__bf16*>(smem);  // two stages
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // the workgroups of one range, which read the same rows, on one XCD
  int range = blockIdx.x / D::SPLIT, nb = blockIdx.x % D::SPLIT;
  if (D::SPLIT > 1 && gridDim.x % (kNumXcd * D::SPLIT) == 0) {
    const int q = blockIdx.x / (kNumXcd * D::SPLIT), r = blockIdx.x % (kNumXcd * D::SPLIT);
    range = q * kNumXcd + r % kNumXcd;
    nb = r / kNumXcd;
  }
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
      dp + (16 * wave * D::MT + (lane & 15)) * kDwTok + 8 * (lane >> 4);
  // Two sets of a step's operands where the registers allow: the loads of step
  // s + 3 are issued after step s and first used after step s + 1.
  float va[U][8], vb[U][8], ra[D::MT][8], rb[D::MT][8];
  auto load_v = [&](float (&vr)[U][8], uint32_t s) {  // a lane takes one channel: whole lines
    const __amdgpu_buffer_rsrc_t in = make_token_rows(v, s * kDwTok, ntok, H);
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int u = threadIdx.x + i * TH;
      const uint32_t o =
          kUnits % TH == 0 || u < kUnits ? 4 * (8 * (u / NC) * H + nb * NC + u % NC) : kOob;
#pragma unroll
      for (int e = 0; e < 8; ++e) vr[i][e] = buf_load1(in, o, 4 * e * H);
    }
  };
  auto load_a = [&](float (&ar)[D::MT][8], uint32_t s) {
#pragma unroll
    for (int m = 0; m < D::MT; ++m) {
      const float* p = a0 + 16 * m * kDwTok + (size_t)s * (2 * H * kDwTok);
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
  // gelu and split of a set's values into a stage
  auto store_v = [&](const float (&vr)[U][8], __bf16* st) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int u = threadIdx.x + i * TH;
      float g[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) g[e] = gelu_f(vr[i][e]);  // gelu(0) = 0 past the end
      bf16x8 hi, mid, lo;
      split3_bf16x8(g, hi, mid, lo);
      if (kUnits % TH == 0 || u < kUnits) {
        __bf16* d = st + (u % NC) * D::CS + 8 * (u / NC);
        *reinterpret_cast<bf16x8*>(d) = hi;
        *reinterpret_cast<bf16x8*>(d + NC * D::CS) = mid;
        *reinterpret_cast<bf16x8*>(d + 2 * NC * D::CS) = lo;
      }
    }
  };
  bf16x8 a[D::MT][3], an[D::MT][3];
  auto split_a = [&](const float (&ar)[D::MT][8], bf16x8 (&o)[D::MT][3]) {
#pragma unroll
    for (int m = 0; m < D::MT; ++m) {
#pragma unroll
      for (int e = 0; e < 8; ++e) rows[m] += ar[m][e];
      split3_bf16x8(ar[m], o[m][0], o[m][1], o[m][2]);
    }
  };
  auto last = [&](uint32_t s) { return s < s1 ? s : s1 - 1; };
  if (s0 < s1) {
    load_v(va, s0);
    load_a(ra, s0);
    store_v(va, sg);
    load_v(va, last(s0 + 1));
    if constexpr (D::AHEAD) {
      split_a(ra, a);
      load_a(ra, last(s0 + 1));
    }
    if constexpr (D::DEEP) {
      load_v(vb, last(s0 + 2));
      load_a(rb, last(s0 + 2));
    }
  }
  auto products = [&](const __bf16* st) {
    const __bf16* const b0 = st + (lane & 15) * D::CS + 8 * (lane >> 4);
    constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};  // small ones first
    constexpr int NG = D::NB % 4 == 0 ? 4 : D::NB % 3 == 0 ? 3 : D::NB % 5 == 0 ? 5 : D::NB;
#pragma unroll
    for (int n0 = 0; n0 < D::NB; n0 += NG) {
      bf16x8 b[NG][3];
#pragma unroll
      for (int n = 0; n < NG; ++n)
#pragma unroll
        for (int p = 0; p < 3; ++p)
          b[n][p] = *reinterpret_cast<const bf16x8*>(b0 + (p * NC + 16 * (n0 + n)) * D::CS);
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int n = 0; n < NG; ++n)
#pragma unroll
          for (int m = 0; m < D::MT; ++m)
            acc[m][n0 + n] = mfma_bf16(a[m][pa[q]], b[n][pb[q]], acc[m][n0 + n]);
    }
  };
  uint32_t s = s0;
  auto step = [&](float (&vr)[U][8], float (&ar)[D::MT][8]) {
    __syncthreads();  // one per step: the stages alternate
    if constexpr (!D::AHEAD) {
      split_a(ar, a);
      load_a(ar, s + 1);
    }
    // step s's products, and in their shadow step s + 1's gelu and splits
    // (after them in program order: LDS writes cannot pass the products' reads)
    products(sg + ((s - s0) & 1) * SZ);
    store_v(vr, sg + ((s + 1 - s0) & 1) * SZ);
    if constexpr (D::AHEAD) split_a(ar, an);
    __builtin_amdgcn_sched_barrier(0);
    load_v(vr, last(s + (D::DEEP ? 3 : 2)));
    if constexpr (D::AHEAD) {
      load_a(ar, last(s + (D::DEEP ? 3 : 2)));
#pragma unroll
      for (int m = 0; m < D::MT; ++m)
#pragma unroll
        for (int p = 0; p < 3; ++p) a[m][p] = an[m][p];
    }
    ++s;
  };
  while (s + 1 < s1) {
    step(va, ra);
    if constexpr (D::DEEP) {
      if (s + 1 >= s1) break;
      step(vb, rb);
    }
  }
  if (s < s1) {
    __syncthreads();
    if constexpr (!D::AHEAD) split_a(ra, a);
    products(sg + ((s - s0) & 1) * SZ);
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
            s = fmaf(dp[(size_t)(k / kDwTok) * (2 * H * kDwTok) + c * kDwTok + k % kDwTok],
                     gelu_f(v[(size_t)k * H + h]), s);
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

}  // namespace pt
