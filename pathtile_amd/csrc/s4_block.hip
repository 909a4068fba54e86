// s4_block.hip — the S4ConvD block's entry points: argument checks, workspace
// layout and the launches of the s4 kernels around the convolution's own.

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "dwconv1d_host.hpp"
#include "pathtile_hip.h"
#include "s4_conv.hpp"
#include "s4_small.hpp"
#include "s4_tables.hpp"

namespace pt {

struct TailGeometry {
  int nw, tok, btok, dw_nw, dw_split;
  size_t bwd_lds, dw_lds;
};

template <int CT>
constexpr TailGeometry tail_geometry() {
  return {TailGeo<CT>::NW,  TailGeo<CT>::TOK,   TailGeo<CT>::BTOK, DwGeo<CT>::NW,
          DwGeo<CT>::SPLIT, tail_bwd_lds<CT>(), DwGeo<CT>::lds};
}

static constexpr TailGeometry kTail[kNumS4H] = {
    tail_geometry<2>(),  tail_geometry<4>(),  tail_geometry<6>(),  tail_geometry<8>(),
    tail_geometry<10>(), tail_geometry<12>(), tail_geometry<14>(), tail_geometry<16>()};

static int check_block(int B, int H, int L, int states) {
  if (B < 1 || H < 32 || H > kS4MaxH || H % 32 != 0 || L < 1 || L > kMaxL || states < 1)
    return PT_ERR_SHAPE;
  if ((long long)B * H * L >= (1LL << 31) || (long long)H * states >= (1LL << 28))
    return PT_ERR_SHAPE;
  return PT_OK;
}

static bool aligned(const void* p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; }
static bool aligned16(const void* p) { return aligned(p, 16); }

// token_base's multiplier for n / L.
static uint32_t token_magic(int L) { return L == 1 ? 0u : (uint32_t)((1ULL << 32) / (unsigned)L) + 1u; }

static size_t round_up(size_t n, size_t q) { return (n + q - 1) / q * q; }

// prep, in floats: taps, the split weights, the poles.
static size_t prep_weights(int H, int L) { return round_up((size_t)H * L, 64); }
static size_t prep_poles(int H, int L) { return prep_weights(H, L) + wfrag_values(H); }

// Token ranges of the weight gradient: one workgroup on each of 256 CUs (its
// accumulators and fragments take half of the registers), at least four
// 32-token steps each. The count depends on the shape alone, so that dW's bits
// do; the whole workspace also on the device, through dk_cl_ranges.
static uint32_t dw_steps_per_range(uint32_t nsteps, int split) {
  const uint32_t ranges = 256u / (uint32_t)split;
  const uint32_t per = (nsteps + ranges - 1) / ranges;
  return per < 4 ? 4 : per;
}

// Workspace of the backward, in floats: dP (blocks of 32 tokens), du, the
// weight gradient's partials, dk [H][L] and its partials.
struct BwdLayout {
  size_t du, part, dk, dkp, total;
  uint32_t nsteps, per, ranges;
  int dk_ranges;
};

static int bwd_layout(int B, int H, int L, BwdLayout* o) {
  const TailGeometry& k = kTail[H / 32 - 1];
  const size_t ntok = (size_t)B * L;
  o->nsteps = (uint32_t)((ntok + kDwTok - 1) / kDwTok);
  o->per = dw_steps_per_range(o->nsteps, k.dw_split);
  o->ranges = (o->nsteps + o->per - 1) / o->per;
  o->dk_ranges = dk_cl_ranges(B, H, L);
  if (o->dk_ranges < 1) return PT_ERR_CONFIG;
  o->du = (size_t)2 * H * round_up(ntok, 64);
  o->part = o->du + ntok * H;
  o->dk = o->part + round_up((size_t)o->ranges * (2 * H * H + 2 * H), 64);
  o->dkp = o->dk + round_up((size_t)H * L, 64);
  o->total = (o->dkp + (size_t)H * L * o->dk_ranges) * sizeof(float);
  return PT_OK;
}

static uint32_t resident_grid(const void* fn, int block, size_t lds, uint32_t work) {
  const uint32_t n = (uint32_t)(blocks_per_cu(fn, block, lds) * num_cus());
  return n < work ? n : work;
}

// add: the input gradient plus that tensor; else the forward, with or without
// a mask and a copy of x.
static int conv_cl_launch(const float* x, const float* w, const float* add,
                          const unsigned char* mask, float scale, float* y, float* xcopy, int B,
                          int H, int L, void* stream) {
  const int form = add ? 1 : xcopy ? (mask ? 4 : 3) : mask ? 2 : 0;
  const void* fn = (const void*)kConvCl[form][(L + 7) / 8 - 1];
  const int block = conv_cl_threads(H), per = block / H;
  void* args[] = {&x, &w, &add, &mask, &scale, &y, &xcopy, &B, &H, &L};
  return launch(fn, resident_grid(fn, block, 0, (uint32_t)((B + per - 1) / per)), (uint32_t)block, 0,
                stream, args);
}

// --- the model's ends ---------------------------------------------------------
constexpr int kEndRanges = 1024;  // partials of the ends' weight gradients

static int check_ends(int B, int H, int L, int n, int most) {
  if (B < 1 || L < 1 || H < 4 || H > 4 * kEndThreads || H % 4 != 0 || n < 1 || n > most)
    return PT_ERR_SHAPE;
  if ((long long)B * H * L >= (1LL << 31)) return PT_ERR_SHAPE;
  return PT_OK;
}

static uint32_t encode_grid(uint32_t ntok, int H) {
  const uint32_t per = (uint32_t)(kEndThreads / (H / 4));
  const uint32_t n = (ntok + per - 1) / per;
  return n < (uint32_t)kEndRanges ? n : (uint32_t)kEndRanges;
}

template <int NI>
static const void* encode_fn(int ni, bool grad) {
  if constexpr (NI <= kEncMaxIn) {
    if (ni == NI)
      return grad ? (const void*)&s4_encode_grad_kernel<NI> : (const void*)&s4_encode_kernel<NI>;
    return encode_fn<NI + 1>(ni, grad);
  }
  return nullptr;
}

static int reduce_launch(const float* part, float* dw, float* db, int nw, int nb, int nr,
                         void* stream) {
  void* args[] = {&part, &dw, &db, &nw, &nb, &nr};
  return launch((const void*)&s4_dw_reduce_kernel, (uint32_t)((nw + nb + 15) / 16), 256, 0, stream,
                args);
}

}  // namespace pt

extern "C" {

int pt_s4_block_prep_values(int H, int L, int states, size_t* floats) {
  if (!floats) return PT_ERR_NULL;
  const int st = pt::check_block(1, H, L, states);
  if (st != PT_OK) return st;
  *floats = pt::prep_poles(H, L) + (size_t)H * (1 + (size_t)states);
  return PT_OK;
}

int pt_s4_block_mix_f32(const float* x, const float* log_dt, const float* c_re, const float* c_im,
                        const float* log_a_re, const float* a_im, const float* skip,
                        const float* w, const unsigned char* mask, float scale, float* prep,
                        float* v, float* x_copy, int B, int H, int L, int states, int backward,
                        void* stream) {
  int st = pt::check_block(B, H, L, states);
  if (st != PT_OK) return st;
  if (!x || !log_dt || !c_re || !c_im || !log_a_re || !a_im || !skip || !w || !prep || !v)
    return PT_ERR_NULL;
  if (!pt::aligned16(x) || !pt::aligned16(prep) || !pt::aligned16(v) ||
      !pt::aligned16(x_copy) || !pt::aligned(mask, 4))
    return PT_ERR_ALIGN;
  float *taps = prep, *poles = prep + pt::prep_poles(H, L);
  __bf16* wf = reinterpret_cast<__bf16*>(prep + pt::prep_weights(H, L));
  const int frags = 2 * H * H / 8 * (backward ? 2 : 1);
  const uint32_t grid = (uint32_t)(H + (frags + pt::kPrepThreads - 1) / pt::kPrepThreads);
  void* args[] = {&log_dt, &c_re, &c_im, &log_a_re, &a_im, &skip, &w, &taps, &wf,
                  &poles, &H, &L, &states, &backward};
  st = pt::launch((const void*)&pt::s4_prep_kernel, grid, pt::kPrepThreads, 0, stream, args);
  if (st != PT_OK) return st;
  return pt::conv_cl_launch(x, taps, nullptr, mask, scale, v, x_copy, B, H, L, stream);
}

int pt_s4_block_tail_f32(const float* v, const float* x, const float* prep, const float* w,
                         const float* bias, float* y, float* q, int B, int H, int L,
                         void* stream) {
  const int st = pt::check_block(B, H, L, 1);
  if (st != PT_OK) return st;
  if (!v || !x || !prep || !w || !bias || !y) return PT_ERR_NULL;
  if (!pt::aligned16(v) || !pt::aligned16(x) || !pt::aligned16(prep) || !pt::aligned16(bias) ||
      !pt::aligned16(y) || !pt::aligned16(q))
    return PT_ERR_ALIGN;
  const pt::TailGeometry& k = pt::kTail[H / 32 - 1];
  const __bf16* wf = reinterpret_cast<const __bf16*>(prep + pt::prep_weights(H, L));
  uint32_t ntok = (uint32_t)B * (uint32_t)L;
  uint32_t ntiles = (ntok + k.tok - 1) / k.tok;
  const size_t lds = pt::tail_fwd_lds(H);
  const int block = k.nw * pt::kWave;
  void* args[] = {&v, &x, &wf, &w, &bias, &y, &q, &ntok, &ntiles};
  const void* fn = (const void*)pt::kTailFwd[H / 32 - 1];
  return pt::launch(fn, pt::resident_grid(fn, block, lds, ntiles), (uint32_t)block, lds, stream,
                    args);
}

int pt_s4_block_bwd_workspace_bytes(int B, int H, int L, size_t* bytes) {
  if (!bytes) return PT_ERR_NULL;
  int st = pt::check_block(B, H, L, 1);
  if (st != PT_OK) return st;
  pt::BwdLayout o;
  st = pt::bwd_layout(B, H, L, &o);
  if (st == PT_OK) *bytes = o.total;
  return st;
}

int pt_s4_block_bwd_f32(const float* gy, const float* x, const float* v, const float* q,
                        const unsigned char* mask, float scale, const float* prep, const float* w,
                        const float* c_re, const float* c_im, const float* a_im, float* gx,
                        float* d_log_dt, float* d_c_re, float* d_c_im, float* d_log_a_re,
                        float* d_a_im, float* d_skip, float* dw, float* dbias, void* workspace,
                        size_t workspace_bytes, int B, int H, int L, int states, void* stream) {
  int st = pt::check_block(B, H, L, states);
  if (st != PT_OK) return st;
  if (!gy || !x || !v || !q || !prep || !w) return PT_ERR_NULL;
  const bool taps_grad = d_skip != nullptr;
  if (taps_grad && (!c_re || !c_im || !a_im || !d_log_dt || !d_c_re || !d_c_im || !d_log_a_re ||
                    !d_a_im))
    return PT_ERR_NULL;
  if ((dw == nullptr) != (dbias == nullptr)) return PT_ERR_NULL;
  if (!pt::aligned16(gy) || !pt::aligned16(x) || !pt::aligned16(v) || !pt::aligned16(prep) ||
      !pt::aligned16(q) || !pt::aligned16(workspace) || (gx && !pt::aligned16(gx)))
    return PT_ERR_ALIGN;
  pt::BwdLayout o;
  st = pt::bwd_layout(B, H, L, &o);
  if (st != PT_OK) return st;
  if (!workspace || workspace_bytes < o.total) return PT_ERR_WORKSPACE;
  const pt::TailGeometry& k = pt::kTail[H / 32 - 1];
  float* const ws = static_cast<float*>(workspace);
  float *dp = ws, *du = ws + o.du, *part = ws + o.part, *dk = ws + o.dk;
  const float *taps = prep, *poles = prep + pt::prep_poles(H, L);
  const __bf16* wf = reinterpret_cast<const __bf16*>(prep + pt::prep_weights(H, L));
  uint32_t ntok = (uint32_t)B * (uint32_t)L, uL = (uint32_t)L, magic = pt::token_magic(L);
  {
    uint32_t ntiles = (ntok + k.btok - 1) / k.btok;
    const int block = k.nw * pt::kWave;
    void* args[] = {&gy, &q, &v, &mask, &scale, &wf, &w, &du, &dp, &ntok, &uL, &magic, &ntiles};
    const void* fn = (const void*)pt::kTailBwd[mask != nullptr][H / 32 - 1];
    st = pt::launch(fn, pt::resident_grid(fn, block, k.bwd_lds, ntiles), (uint32_t)block,
                    k.bwd_lds, stream, args);
    if (st != PT_OK) return st;
  }
  if (dw) {
    const float* cdp = dp;
    void* args[] = {&cdp, &v, &part, &ntok, &o.nsteps, &o.per};
    st = pt::launch((const void*)pt::kDw[H / 32 - 1], o.ranges * (uint32_t)k.dw_split,
                    (uint32_t)(k.dw_nw * pt::kWave), k.dw_lds, stream, args);
    if (st != PT_OK) return st;
    st = pt::reduce_launch(part, dw, dbias, 2 * H * H, 2 * H, (int)o.ranges, stream);
    if (st != PT_OK) return st;
  }
  if (gx) {
    st = pt::conv_cl_launch(du, taps, gy, nullptr, 0.0f, gx, nullptr, B, H, L, stream);
    if (st != PT_OK) return st;
  }
  if (!taps_grad) return PT_OK;
  st = pt::dk_cl_det(x, du, dk, ws + o.dkp, B, H, L, L, o.dk_ranges, stream);
  if (st != PT_OK) return st;
  const float* cdk = dk;
  void* targs[] = {&cdk, &poles, &c_re, &c_im, &a_im, &d_log_dt, &d_c_re, &d_c_im, &d_log_a_re,
                   &d_a_im, &d_skip, &L, &states};
  return pt::launch((const void*)&pt::s4_taps_grad_kernel, (uint32_t)H, pt::kPrepThreads, 0, stream,
                    targs);
}

int pt_s4_encode_f32(const float* x, const float* w, const float* bias, float* y, int B, int L,
                     int inputs, int H, void* stream) {
  const int st = pt::check_ends(B, H, L, inputs, pt::kEncMaxIn);
  if (st != PT_OK) return st;
  if (!x || !w || !bias || !y) return PT_ERR_NULL;
  if (!pt::aligned16(bias) || !pt::aligned16(y)) return PT_ERR_ALIGN;
  uint32_t ntok = (uint32_t)B * (uint32_t)L;
  const uint32_t per = (uint32_t)(pt::kEndThreads / (H / 4));
  const void* fn = pt::encode_fn<1>(inputs, false);
  void* args[] = {&x, &w, &bias, &y, &ntok, &H};
  return pt::launch(fn, pt::resident_grid(fn, pt::kEndThreads, 0, (ntok + per - 1) / per),
                    per * (uint32_t)(H / 4), 0, stream, args);
}

int pt_s4_encode_grad_workspace_bytes(int B, int L, int inputs, int H, size_t* bytes) {
  if (!bytes) return PT_ERR_NULL;
  const int st = pt::check_ends(B, H, L, inputs, pt::kEncMaxIn);
  if (st == PT_OK)
    *bytes = (size_t)pt::encode_grid((uint32_t)B * (uint32_t)L, H) * (H * inputs + H) * 4;
  return st;
}

int pt_s4_encode_grad_f32(const float* x, const float* gy, float* dw, float* dbias,
                          void* workspace, size_t workspace_bytes, int B, int L, int inputs, int H,
                          void* stream) {
  size_t need = 0;
  int st = pt_s4_encode_grad_workspace_bytes(B, L, inputs, H, &need);
  if (st != PT_OK) return st;
  if (!x || !gy || !dw || !dbias) return PT_ERR_NULL;
  if (!pt::aligned16(gy)) return PT_ERR_ALIGN;
  if (!workspace || workspace_bytes < need) return PT_ERR_WORKSPACE;
  uint32_t ntok = (uint32_t)B * (uint32_t)L;
  const uint32_t grid = pt::encode_grid(ntok, H), per = (uint32_t)(pt::kEndThreads / (H / 4));
  float* part = static_cast<float*>(workspace);
  void* args[] = {&x, &gy, &part, &ntok, &H};
  st = pt::launch(pt::encode_fn<1>(inputs, true), grid, per * (uint32_t)(H / 4), 0, stream, args);
  if (st != PT_OK) return st;
  return pt::reduce_launch(part, dw, dbias, H * inputs, H, (int)grid, stream);
}

int pt_s4_head_f32(const float* x, const float* w, const float* bias, float* out, int B, int H,
                   int L, int outputs, void* stream) {
  const int st = pt::check_ends(B, H, L, outputs, pt::kHeadMaxOut);
  if (st != PT_OK) return st;
  if (!x || !w || !bias || !out) return PT_ERR_NULL;
  void* args[] = {&x, &w, &bias, &out, &B, &H, &L, &outputs};
  const uint32_t per = pt::kEndThreads / pt::kWave;
  return pt::launch((const void*)&pt::s4_head_kernel, ((uint32_t)B + per - 1) / per,
                    pt::kEndThreads, 0, stream, args);
}

int pt_s4_head_grad_workspace_bytes(int B, int H, int L, int outputs, size_t* bytes) {
  if (!bytes) return PT_ERR_NULL;
  const int st = pt::check_ends(B, H, L, outputs, pt::kHeadMaxOut);
  const int n = B < pt::kEndRanges ? B : pt::kEndRanges;
  if (st == PT_OK) *bytes = (size_t)n * (outputs * H + outputs) * 4;
  return st;
}

int pt_s4_head_grad_f32(const float* x, const float* gy, const float* w, float* gx, float* dw,
                        float* dbias, void* workspace, size_t workspace_bytes, int B, int H, int L,
                        int outputs, void* stream) {
  size_t need = 0;
  int st = pt_s4_head_grad_workspace_bytes(B, H, L, outputs, &need);
  if (st != PT_OK) return st;
  if (!x || !gy || (gx && !w) || !dw || !dbias) return PT_ERR_NULL;
  if (!pt::aligned16(x) || (gx && !pt::aligned16(gx))) return PT_ERR_ALIGN;
  if (!workspace || workspace_bytes < need) return PT_ERR_WORKSPACE;
  int per = (B + pt::kEndRanges - 1) / pt::kEndRanges;
  const int grid = (B + per - 1) / per;
  float* part = static_cast<float*>(workspace);
  void* args[] = {&x, &gy, &w, &gx, &part, &B, &H, &L, &outputs, &per};
  st = pt::launch((const void*)&pt::s4_head_grad_kernel, (uint32_t)grid, pt::kEndThreads, 0, stream,
                  args);
  if (st != PT_OK) return st;
  return pt::reduce_launch(part, dw, dbias, outputs * H, outputs, grid, stream);
}

}  // extern "C"
