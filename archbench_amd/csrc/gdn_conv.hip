// Short causal depthwise convolution + SiLU (+ optional L2 normalisation per head), forward and backward: the
// ShortConvolution in front of the gated DeltaNet op (archbench/layers/nsgdn.py:420-470, the causal_conv1d
// kernels behind fla's GatedDeltaNet; normalisation of q and k per head as in nsgdn.py:527-528).
//
//   z[t,c] = bias[c] + sum_i w[c,i] x[t - (W-1) + i, c]      (x at t < 0 comes from the conv state)
//   y[t,c] = silu(z[t,c]);  with normalisation over each group of NG channels: y / max(||y||_group, 1e-12)
//
// Layout: y, dy [B, T, D] token-major (channel-last); x and dx [B, T] rows of D channels ldx / lddx elements apart
// (= D, or larger to read or write a column slice of a wider tensor in place); w [D, W] fp32 (used rounded to the
// activation dtype; dw is the fp32 gradient of those rounded taps), bias [D] fp32, conv states
// [B, D, W-1] in the activation dtype (the previous W-1 inputs, oldest first).
// Mapping: one wave per (256 channels, chunk of 8 to 128 tokens, b); each lane holds 4 consecutive channels, so every
// token row is one 8-byte (bf16) or 16-byte (fp32) access per lane and a wave covers 512 B / 1 KB contiguous.  The W-1
// inputs before a chunk are re-read.  A normalisation group of NG channels spans NG/4 lanes and is reduced with lane
// shuffles.  One launch covers up to three column groups of x (ConvGroups): the mixer's q, k and v, whose three launches
// of 2 to 8 waves per CU left the memory half idle (B64 T1024 H4: forward 153 -> 96 us, 5.6 TB/s; backward 252 -> 172
// us, 4.7 TB/s, with the rolling row slots below).  The forward is HBM-bound (x read once, y written once); the backward
// is near both its HBM and its VALU bound (about 37 issue slots per element, 126 us at that size).
// Backward: each wave recomputes z for its chunk plus W-1 tokens of look-ahead, forms dz and emits dx with a
// W-token delay; dw and dbias are summed per wave into a per-chunk partial and reduced over chunks in a fixed
// order by column_sum_kernel (deterministic, no atomics).
#include <type_traits>

#include "gdn_common.h"
#include "gdn_launch.h"

namespace gdn {

// Tokens per wave, a multiple of the rows in flight.  64 on a grid of ordinary size.  The backward takes 128 once that
// leaves 8 waves per CU: the set-up, the look-ahead recompute and the dw partial of a wave are then amortised over twice
// the tokens (D = 2048 without normalisation: 94.5 -> 76.6 us at B8 T4096, but 47.8 -> 58.9 at B4 T4000, 4 waves per CU;
// the 65m mixer's input stage, B64 T1024, 182 -> 172 us).  A small grid is cut finer until it has 10 waves per CU in
// the forward and 6 in the backward, whose dw partials grow with the cut (input stage, forward / backward at 64, 32, 16
// and 8 tokens: B6 T777 H8 30.1 / 51.6, 23.9 / 46.0, 22.5 / 52.0, 24.4 / 70.3 us; B2 T1000 H4 20.5 / 37.2, 13.5 / 25.6,
// 12.4 / 23.4, 9.5 / 23.9 us; B12 T1024 H8, 12 waves per CU at 64 tokens, 42.7 / 74.0, 46.0 / 85.7 us), the backward
// below 16 tokens only when even that leaves CUs without a wave (B1 T200 H3: 19.0 -> 13.4 us).
constexpr int CONV_L = 64, CONV_L_LONG = 128, CONV_L_MIN = 8, CONV_L_MIN_BWD = 16;
constexpr int CONV_LONG_WAVES_PER_CU = 8, CONV_FWD_WAVES_PER_CU = 10, CONV_BWD_WAVES_PER_CU = 6;
constexpr int CONV_CPL = 4;  // consecutive channels per lane
constexpr int CONV_CW = 64 * CONV_CPL;  // channels per wave
constexpr int CONV_WAVES = 4;  // waves per workgroup, on adjacent channel blocks of the same chunk
constexpr int CONV_UF = 8;  // token rows per load batch, forward
constexpr int CONV_UB = 8;  // token rows of x and of dy in flight, backward (4: 180 against 172 us)
static_assert(CONV_L_MIN % CONV_UB == 0 && CONV_L_MIN_BWD % CONV_UB == 0, "whole batches in every chunk but the last");

// CONV_CPL = 4 consecutive channels of one token row as loaded (8 B in bf16, 16 B in fp32), converted at use so
// that a whole batch of loads is in flight at once.  The backward reads x and dy and writes dx once each through
// buffer resources with the nontemporal hint (load_buf_nt / store4_buf_nt: 7-17% faster than ordinary global
// accesses, and 32-bit offsets spare it the 64-bit address arithmetic of a VALU-bound loop); the forward, whose
// workgroups re-read a few halo rows of their neighbours, runs slower with the hint and keeps ordinary loads.
template <typename T>
struct Row4;
template <>
struct Row4<bf16> {
  bf16x4 r;
  __device__ __forceinline__ void load(const bf16* p) { r = *reinterpret_cast<const bf16x4*>(p); }
  // nontemporal buffer read at byte offset off
  __device__ __forceinline__ void load_buf_nt(__amdgpu_buffer_rsrc_t rs, int off) {
    r = __builtin_bit_cast(bf16x4, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 2));
  }
  __device__ __forceinline__ void get(float (&v)[4]) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = static_cast<float>(r[j]);
  }
};
template <>
struct Row4<float> {
  f32x4 r;
  __device__ __forceinline__ void load(const float* p) { r = *reinterpret_cast<const f32x4*>(p); }
  __device__ __forceinline__ void load_buf_nt(__amdgpu_buffer_rsrc_t rs, int off) {
    r = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 2));
  }
  __device__ __forceinline__ void get(float (&v)[4]) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = r[j];
  }
};

template <typename T>
__device__ __forceinline__ void store4(T* p, const float (&v)[4]) {
  if constexpr (sizeof(T) == 2) {
    *reinterpret_cast<bf16x4*>(p) =
        bf16x4{static_cast<bf16>(v[0]), static_cast<bf16>(v[1]), static_cast<bf16>(v[2]), static_cast<bf16>(v[3])};
  } else {
    *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
  }
}
// nontemporal buffer write of 4 consecutive channels at byte offset off
template <typename T>
__device__ __forceinline__ void store4_buf_nt(__amdgpu_buffer_rsrc_t rs, int off, const float (&v)[4]) {
  if constexpr (sizeof(T) == 2) {
    const bf16x4 r{static_cast<bf16>(v[0]), static_cast<bf16>(v[1]), static_cast<bf16>(v[2]), static_cast<bf16>(v[3])};
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, r), rs, off, 0, 2);
  } else {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, f32x4{v[0], v[1], v[2], v[3]}), rs, off, 0, 2);
  }
}
// A tap weight at the activation dtype's precision: the reference's conv runs under bf16 autocast, which casts its
// fp32 weight to bf16 (archbench/layers/nsgdn.py:464); rounding here spares the caller two cast passes each way.
template <typename T>
__device__ __forceinline__ float act_round(float x) {
  if constexpr (sizeof(T) == 2) return static_cast<float>(static_cast<bf16>(x));
  return x;
}
// sum over the NG / CONV_CPL lanes of a normalisation group (aligned runs of lanes), the same value in every lane
template <int NG>
__device__ __forceinline__ float group_sum(float s) {
  return lane_group_sum<NG / CONV_CPL>(s);
}
constexpr float NORM_EPS = 1e-12f;  // F.normalize's eps

template <typename T, int W>
__device__ __forceinline__ void load_window(const T* xl, const T* state_in, int64_t srow, int ldx, int t0,
                                            float (&win)[W - 1][CONV_CPL]) {
  // inputs at t0 - (W-1) .. t0 - 1; negative positions from the conv state (zero if none)
#pragma unroll
  for (int i = 0; i < W - 1; ++i) {
    const int t = t0 - (W - 1) + i;
    if (t >= 0) {
      Row4<T> r;
      r.load(xl + (int64_t)t * ldx);
      r.get(win[i]);
    } else if (state_in) {
#pragma unroll
      for (int j = 0; j < CONV_CPL; ++j) win[i][j] = to_f(state_in[srow + (int64_t)j * (W - 1) + (W - 1) + t]);
    } else {
#pragma unroll
      for (int j = 0; j < CONV_CPL; ++j) win[i][j] = 0.f;
    }
  }
}

// The channels of x in up to three consecutive column groups (plain convolutions: one), each with a contiguous tensor
// of its own on the other side (y in the forward, dy in the backward: [B, T, n]); the first `normed` groups are
// L2-normalised.
template <typename T>
struct ConvGroups {
  T* p[3];
  int n[3];
  int normed;
};
// Work items: (part = b * nchunk + chunk, 256-channel block of one group), blocks fastest; wave w of workgroup x takes
// item x * CONV_WAVES + w, so the waves of a workgroup, each independent, cover adjacent channel blocks of the same
// token rows (and, when there are fewer than CONV_WAVES blocks, the next chunk's: no wave idles).  The whole item is
// uniform over the wave.
template <typename T>
struct ConvItem {
  int part, b, t0, t1, cw0, xc0, n;  // cw0: first channel inside the group, xc0: the group's first column of x
  bool norm;
  T* p;
  __device__ __forceinline__ bool init(const ConvGroups<T>& g, int Tn, int L, int nchunk, int nparts) {
    const int nb0 = (g.n[0] + CONV_CW - 1) / CONV_CW, nb1 = nb0 + (g.n[1] + CONV_CW - 1) / CONV_CW;
    const int ncb = nb1 + (g.n[2] + CONV_CW - 1) / CONV_CW;
    const int item = (int)blockIdx.x * CONV_WAVES + __builtin_amdgcn_readfirstlane(wave_id());
    part = item / ncb;
    const int blk = item - part * ncb, gi = (blk >= nb0) + (blk >= nb1);
    cw0 = (blk - (gi == 0 ? 0 : gi == 1 ? nb0 : nb1)) * CONV_CW;
    xc0 = gi == 0 ? 0 : gi == 1 ? g.n[0] : g.n[0] + g.n[1];
    n = gi == 0 ? g.n[0] : gi == 1 ? g.n[1] : g.n[2];
    p = gi == 0 ? g.p[0] : gi == 1 ? g.p[1] : g.p[2];
    norm = gi < g.normed;
    b = part / nchunk;
    t0 = (part - b * nchunk) * L;
    t1 = min(Tn, t0 + L);
    return part < nparts;
  }
};
// Forward: grid ceil(B * nchunk * blocks / CONV_WAVES), CONV_WAVES waves.  Rows are loaded in batches of CONV_UF with
// the next batch in flight while the current one is computed; the prefetch of the last batch re-reads it (start clamped
// to t1 - CONV_UF) so every load stays inside the chunk.  D: all channels (those of w and the states).
template <typename T, int W, int NG, typename WT>
__device__ __forceinline__ void conv_fwd_wave(const ConvItem<T>& it, const T* __restrict__ x,
                                              const WT* __restrict__ w, const float* __restrict__ bias,
                                              const T* __restrict__ state_in, T* __restrict__ state_out, int Tn, int D,
                                              int ldx) {
  constexpr int CPL = CONV_CPL, U = CONV_UF;
  const int c = it.cw0 + CPL * lane_id();
  const int b = it.b, t0 = it.t0, t1 = it.t1;
  const bool on = c < it.n;
  const int cg = on ? c : 0;      // channel inside the group; clamped: lanes past it compute on its first channel and
  const int cc = it.xc0 + cg;     // store nothing.  cc: the same channel of x, w, bias and the states
  const T* xl = x + (int64_t)b * Tn * ldx + cc;  // token t of x at xl + t * ldx
  const int ldy = it.n;
  T* yl = it.p + (int64_t)b * Tn * ldy + cg;
  const int64_t srow = ((int64_t)b * D + cc) * (W - 1);
  float wk[CPL][W], bk[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
#pragma unroll
    for (int i = 0; i < W; ++i) wk[j][i] = act_round<T>(to_f(w[(cc + j) * W + i]));
    bk[j] = bias ? bias[cc + j] : 0.f;
  }
  float win[W - 1][CPL];
  load_window<T, W>(xl, state_in, srow, ldx, t0, win);
  auto step = [&](int t, const Row4<T>& row) {
    float xt[CPL], yt[CPL];
    row.get(xt);
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      float z = bk[j] + wk[j][W - 1] * xt[j];
#pragma unroll
      for (int i = 0; i < W - 1; ++i) z += wk[j][i] * win[i][j];
      yt[j] = z * fast_sigmoid(z);
      ss += yt[j] * yt[j];
    }
    if constexpr (NG > 0) {
      const float inv = fast_rcp(fmaxf(sqrtf(group_sum<NG>(ss)), NORM_EPS));
#pragma unroll
      for (int j = 0; j < CPL; ++j) yt[j] *= inv;
    }
    if (on) store4(yl + (int64_t)t * ldy, yt);
#pragma unroll
    for (int i = 0; i + 1 < W - 1; ++i)
#pragma unroll
      for (int j = 0; j < CPL; ++j) win[i][j] = win[i + 1][j];
#pragma unroll
    for (int j = 0; j < CPL; ++j) win[W - 2][j] = xt[j];
  };
  const int nfull = (t1 - t0) / U;
  int t = t0;
  if (nfull > 0) {
    Row4<T> buf[U];
#pragma unroll
    for (int u = 0; u < U; ++u) buf[u].load(xl + (int64_t)(t0 + u) * ldx);
    for (int n = 0; n < nfull; ++n, t += U) {
      Row4<T> cur[U];
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = buf[u];
      const int tn = min(t + U, t1 - U);
#pragma unroll
      for (int u = 0; u < U; ++u) buf[u].load(xl + (int64_t)(tn + u) * ldx);
#pragma unroll
      for (int u = 0; u < U; ++u) step(t + u, cur[u]);
    }
  }
  for (; t < t1; ++t) {
    Row4<T> row;
    row.load(xl + (int64_t)t * ldx);
    step(t, row);
  }
  // the last W-1 inputs become the new conv state (written by the chunk that holds the sequence end; for
  // Tn < W-1 part of it still comes from the old state, which must not be the same buffer)
  if (state_out && on && t1 == Tn) {
    float last[W - 1][CPL];
    load_window<T, W>(xl, state_in, srow, ldx, Tn, last);
#pragma unroll
    for (int i = 0; i < W - 1; ++i)
#pragma unroll
      for (int j = 0; j < CPL; ++j) state_out[srow + (int64_t)j * (W - 1) + i] = from_f<T>(last[i][j]);
  }
}

// NG: the normalisation group of the groups that have one (0: none has)
template <typename T, int W, int NG>
__global__ __launch_bounds__(64 * CONV_WAVES) void conv_silu_fwd_kernel(const T* __restrict__ x,
                                                                        const float* __restrict__ w,
                                                                        const float* __restrict__ bias,
                                                                        const T* __restrict__ state_in,
                                                                        ConvGroups<T> y, T* __restrict__ state_out,
                                                                        int Tn, int D, int ldx, int L, int nchunk,
                                                                        int nparts) {
  ConvItem<T> it;
  if (!it.init(y, Tn, L, nchunk, nparts)) return;  // past the last item (waves never synchronise)
  if constexpr (NG > 0) {
    if (it.norm) return conv_fwd_wave<T, W, NG>(it, x, w, bias, state_in, state_out, Tn, D, ldx);
  }
  conv_fwd_wave<T, W, 0>(it, x, w, bias, state_in, state_out, Tn, D, ldx);
}

// One decoded token per sequence: a wave per (b, 256-channel block of q, k or v), each convolution with its own taps and
// states, then the workgroups of the gates, an element per thread.  Latency-bound: 4.0 us at B8 H8, where three
// convolutions, the gates and the copies and casts in front of them took 25 us in eleven launches.
struct DecodeParam {
  const void* p;
  bool half;
  __device__ __forceinline__ float operator[](int i) const {
    return half ? to_f(static_cast<const bf16*>(p)[i]) : static_cast<const float*>(p)[i];
  }
};
template <typename WT, int NG>
__global__ __launch_bounds__(64 * CONV_WAVES) void decode_stage_kernel(DecodeStageArgs a, int conv_wgs) {
  if ((int)blockIdx.x >= conv_wgs) {
    const int e = ((int)blockIdx.x - conv_wgs) * 64 * CONV_WAVES + threadIdx.x;
    if (e < a.B * a.H) {
      const int b = e / a.H, h = e - b * a.H;
      const bf16* ab = static_cast<const bf16*>(a.ab) + (int64_t)b * 2 * a.H;
      const bool half = a.gate_dtype == DT_BF16;
      a.g[e] = gate_g(to_f(ab[h]) + DecodeParam{a.dt_bias, half}[h], DecodeParam{a.A_log, half}[h], a.g_min);
      a.beta[e] = gate_beta(to_f(ab[a.H + h]), a.beta_scale);
    }
    return;
  }
  const int nb0 = (a.n[0] + CONV_CW - 1) / CONV_CW, nb1 = nb0 + (a.n[1] + CONV_CW - 1) / CONV_CW;
  const int ncb = nb1 + (a.n[2] + CONV_CW - 1) / CONV_CW;
  const int item = (int)blockIdx.x * CONV_WAVES + __builtin_amdgcn_readfirstlane(wave_id());
  if (item >= a.B * ncb) return;
  auto pick = [&](int gi, auto x0, auto x1, auto x2) { return gi == 0 ? x0 : gi == 1 ? x1 : x2; };
  ConvItem<bf16> it;
  it.part = it.b = item / ncb;
  const int blk = item - it.b * ncb, gi = (blk >= nb0) + (blk >= nb1);
  it.t0 = 0, it.t1 = 1;
  it.cw0 = (blk - pick(gi, 0, nb0, nb1)) * CONV_CW;
  it.xc0 = 0;
  it.n = pick(gi, a.n[0], a.n[1], a.n[2]);
  it.norm = gi < 2;
  it.p = static_cast<bf16*>(pick(gi, a.out[0], a.out[1], a.out[2]));
  const bf16* y = static_cast<const bf16*>(a.y) + pick(gi, 0, a.n[0], a.n[0] + a.n[1]);
  const WT* w = static_cast<const WT*>(pick(gi, a.w[0], a.w[1], a.w[2]));
  const bf16* sin = static_cast<const bf16*>(pick(gi, a.state_in[0], a.state_in[1], a.state_in[2]));
  bf16* sout = static_cast<bf16*>(pick(gi, a.state_out[0], a.state_out[1], a.state_out[2]));
  const int ldx = a.n[0] + a.n[1] + a.n[2];
  if (it.norm) return conv_fwd_wave<bf16, 4, NG>(it, y, w, nullptr, sin, sout, 1, it.n, ldx);
  conv_fwd_wave<bf16, 4, 0>(it, y, w, nullptr, sin, sout, 1, it.n, ldx);
}

// grid and waves as in the forward; partial sums of dw and dbias per (b, chunk) = part.
// Each wave recomputes z over its chunk plus W-1 tokens of look-ahead, forms dz, and emits dx with a W-1 token
// delay; CONV_UB rows of x and dy are in flight.
template <typename T, int W, int NG, bool BIAS>
__device__ __forceinline__ void conv_bwd_wave(const ConvItem<const T>& it, const T* __restrict__ x,
                                              const float* __restrict__ w, const float* __restrict__ bias,
                                              const T* __restrict__ state_in, T* __restrict__ dx,
                                              T* __restrict__ dstate_in, float* __restrict__ part_out, int ldp,
                                              int Tn, int D, int ldx, int lddx) {
  constexpr int CPL = CONV_CPL, U = CONV_UB;
  const int c = it.cw0 + CPL * lane_id();
  const int b = it.b, t0 = it.t0, t1 = it.t1;
  const bool on = c < it.n;
  const int cg = on ? c : 0, cc = it.xc0 + cg;  // as in the forward
  const T* xl = x + (int64_t)b * Tn * ldx + cc;
  const int64_t srow = ((int64_t)b * D + cc) * (W - 1);
  // the batch element's rows of x ([Tn] rows ldx apart), dy ([Tn][n]) and dx (rows lddx apart) as buffer resources
  // (uniform base, 32-bit offsets: the host keeps Tn * ldx * sizeof(T) under 2 GiB); token t, this lane's channels at
  // byte offset xoff(t) in x, boff(t) in dy and dxoff(t) in dx
  const int ldy = it.n;
  const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(x + (int64_t)b * Tn * ldx), 0,
                                                    Tn * ldx * (int)sizeof(T), BUF_RSRC_WORD3);
  const auto rdy = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(it.p + (int64_t)b * Tn * ldy), 0,
                                                     Tn * ldy * (int)sizeof(T), BUF_RSRC_WORD3);
  const auto rdx = __builtin_amdgcn_make_buffer_rsrc(dx + (int64_t)b * Tn * lddx, 0, Tn * lddx * (int)sizeof(T),
                                                     BUF_RSRC_WORD3);
  auto boff = [&](int t) { return (t * ldy + cg) * (int)sizeof(T); };
  auto xoff = [&](int t) { return (t * ldx + cc) * (int)sizeof(T); };
  auto dxoff = [&](int t) { return (t * lddx + cc) * (int)sizeof(T); };
  float wk[CPL][W], bk[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
#pragma unroll
    for (int i = 0; i < W; ++i) wk[j][i] = act_round<T>(w[(cc + j) * W + i]);
    bk[j] = BIAS && bias ? bias[cc + j] : 0.f;
  }
  float win[W - 1][CPL], dzw[W - 1][CPL], dwa[CPL][W], dba[CPL];
  load_window<T, W>(xl, state_in, srow, ldx, t0, win);
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    dba[j] = 0.f;
#pragma unroll
    for (int i = 0; i < W; ++i) dwa[j][i] = 0.f;
#pragma unroll
    for (int i = 0; i < W - 1; ++i) dzw[i][j] = 0.f;
  }
  // dx[p] = sum_i w[i] dz[p + W-1 - i]: emitted at s = p + W-1 from dz[s] and the W-1 dz before it (dzw).  This
  // wave emits dx for its own tokens, and for chunk 0 also the state gradient (p = -(W-1) .. -1).
  auto emit = [&](int s, const float (&dz)[CPL], bool have_dz) {
    const int p = s - (W - 1);
    if (p >= t0 || (t0 == 0 && p >= -(W - 1))) {
      float o[CPL];
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        o[j] = have_dz ? wk[j][0] * dz[j] : 0.f;
#pragma unroll
        for (int i = 1; i < W; ++i) o[j] += wk[j][i] * dzw[W - 1 - i][j];
      }
      if (on) {
        if (p >= 0) {
          store4_buf_nt<T>(rdx, dxoff(p), o);
        } else if (dstate_in) {
#pragma unroll
          for (int j = 0; j < CPL; ++j) dstate_in[srow + (int64_t)j * (W - 1) + (W - 1) + p] = from_f<T>(o[j]);
        }
      }
    }
  };
  // own = the chunk's own tokens, which carry dw and dbias (the W-1 look-ahead tokens only feed dx)
  auto step = [&](int s, const Row4<T>& xrow, const Row4<T>& dyrow, auto own) {
    float xs[CPL], ds[CPL], dz[CPL];
    xrow.get(xs);
    dyrow.get(ds);
    float z[CPL], sg[CPL], ysl[CPL], ss = 0.f;
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      z[j] = bk[j] + wk[j][W - 1] * xs[j];
#pragma unroll
      for (int i = 0; i < W - 1; ++i) z[j] += wk[j][i] * win[i][j];
      sg[j] = fast_sigmoid(z[j]);
      ysl[j] = z[j] * sg[j];
      ss += ysl[j] * ysl[j];
    }
    if constexpr (NG > 0) {
      const float nrm = sqrtf(group_sum<NG>(ss));
      const float inv = fast_rcp(fmaxf(nrm, NORM_EPS));
      float dot = 0.f;
#pragma unroll
      for (int j = 0; j < CPL; ++j) dot += ysl[j] * inv * ds[j];
      dot = group_sum<NG>(dot);
      const bool big = nrm > NORM_EPS;
#pragma unroll
      for (int j = 0; j < CPL; ++j) ds[j] = big ? (ds[j] - ysl[j] * inv * dot) * inv : ds[j] * inv;
    }
#pragma unroll
    for (int j = 0; j < CPL; ++j) dz[j] = ds[j] * sg[j] * (1.f + z[j] * (1.f - sg[j]));
    if constexpr (decltype(own)::value) {
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        if constexpr (BIAS) dba[j] += dz[j];
        dwa[j][W - 1] += dz[j] * xs[j];
#pragma unroll
        for (int i = 0; i < W - 1; ++i) dwa[j][i] += dz[j] * win[i][j];
      }
    }
    emit(s, dz, true);
#pragma unroll
    for (int i = 0; i + 1 < W - 1; ++i)
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        win[i][j] = win[i + 1][j];
        dzw[i][j] = dzw[i + 1][j];
      }
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      win[W - 2][j] = xs[j];
      dzw[W - 2][j] = dz[j];
    }
  };
  using Own = std::true_type;
  using LookAhead = std::false_type;
  // Rows U tokens ahead, one register slot per row modulo U, reloaded as soon as it is consumed (a second set of slots
  // for the next batch took 32 more registers, one wave per SIMD fewer).  Loads past the sequence's end read its last row.
  Row4<T> bx[U], bd[U];
  auto load = [&](int u, int t) {
    const int tc = min(t, Tn - 1);
    bx[u].load_buf_nt(rx, xoff(tc));
    bd[u].load_buf_nt(rdy, boff(tc));
  };
#pragma unroll
  for (int u = 0; u < U; ++u) load(u, t0 + u);
  int s = t0;
  for (const int full = t0 + (t1 - t0) / U * U; s < full; s += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const Row4<T> cx = bx[u], cd = bd[u];
      load(u, s + u + U);
      step(s + u, cx, cd, Own{});
    }
  }
  // Only the sequence's last chunk can hold a partial batch (the host keeps chunks whole multiples of U), only the
  // others look ahead; either way the rows are in the slots already.
  if (t1 == Tn) {
#pragma unroll
    for (int u = 0; u < U - 1; ++u)
      if (s + u < t1) step(s + u, bx[u], bd[u], Own{});
    s = t1;
  } else {
#pragma unroll
    for (int u = 0; u < W - 1; ++u)
      if (t1 + u < Tn) step(t1 + u, bx[u], bd[u], LookAhead{});
    s = min(Tn, t1 + W - 1);
  }
  // past the sequence end dz = 0: flush the remaining dx of the chunk's tail (and of the state when Tn is short)
  for (; s < t1 + W - 1; ++s) {
    const float zero[CPL] = {};
    emit(s, zero, false);
#pragma unroll
    for (int i = 0; i + 1 < W - 1; ++i)
#pragma unroll
      for (int j = 0; j < CPL; ++j) dzw[i][j] = dzw[i + 1][j];
#pragma unroll
    for (int j = 0; j < CPL; ++j) dzw[W - 2][j] = 0.f;
  }
  if (on) {
    float* row = part_out + (int64_t)it.part * ldp;  // [dw (D x W) | dbias (D) if wanted] of this (b, chunk)
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
#pragma unroll
      for (int i = 0; i < W; ++i) row[(cc + j) * W + i] = dwa[j][i];
      if constexpr (BIAS) row[D * W + cc + j] = dba[j];
    }
  }
}

// BIAS: there is a bias or its gradient is wanted
template <typename T, int W, int NG, bool BIAS>
__global__ __launch_bounds__(64 * CONV_WAVES) void conv_silu_bwd_kernel(const T* __restrict__ x,
                                                                        const float* __restrict__ w,
                                                                        const float* __restrict__ bias,
                                                                        const T* __restrict__ state_in,
                                                                        ConvGroups<const T> dy, T* __restrict__ dx,
                                                                        T* __restrict__ dstate_in,
                                                                        float* __restrict__ part_out, int ldp, int Tn,
                                                                        int D, int ldx, int lddx, int L, int nchunk,
                                                                        int nparts) {
  ConvItem<const T> it;
  if (!it.init(dy, Tn, L, nchunk, nparts)) return;  // past the last item (waves never synchronise)
  if constexpr (NG > 0) {
    if (it.norm)
      return conv_bwd_wave<T, W, NG, BIAS>(it, x, w, bias, state_in, dx, dstate_in, part_out, ldp, Tn, D, ldx, lddx);
  }
  conv_bwd_wave<T, W, 0, BIAS>(it, x, w, bias, state_in, dx, dstate_in, part_out, ldp, Tn, D, ldx, lddx);
}

// ---------------------------------------------------------------------------------------------------------
static int conv_blocks(const int (&n)[3]) {
  int ncb = 0;
  for (int i = 0; i < 3; ++i) ncb += (n[i] + CONV_CW - 1) / CONV_CW;
  return ncb;
}

// tokens per wave (see CONV_L)
static int conv_len(int B, int T, int ncb, bool backward) {
  const int64_t cus = device_cu_count();
  auto waves = [&](int L) { return (int64_t)ncb * B * ((T + L - 1) / L); };
  if (backward && waves(CONV_L_LONG) >= CONV_LONG_WAVES_PER_CU * cus) return CONV_L_LONG;
  int L = CONV_L;
  while (L > (backward ? CONV_L_MIN_BWD : CONV_L_MIN) &&
         waves(L) < (backward ? CONV_BWD_WAVES_PER_CU : CONV_FWD_WAVES_PER_CU) * cus)
    L /= 2;
  return backward && waves(L) < cus ? CONV_L_MIN : L;
}

size_t conv_ws_bytes(int B, int T, const int (&n)[3], int W) {
  // partial rows of the backward: one per (b, chunk)
  const int D = n[0] + n[1] + n[2];
  const int L = conv_len(B, T, conv_blocks(n), true);
  const size_t nparts = (size_t)B * ((T + L - 1) / L);
  return (nparts * (size_t)(D * W + D) * 4 + 255) & ~size_t(255);
}

static bool conv_width_ok(int n, int norm_group) {
  return n > 0 && n % CONV_CPL == 0 &&
         (norm_group == 0 || ((norm_group == 64 || norm_group == 128 || norm_group == 256) && n % norm_group == 0));
}
bool conv_shape_supported(int D, int W, int norm_group) { return W == 4 && conv_width_ok(D, norm_group); }

// workgroups for every (part, 256-channel block) item, CONV_WAVES items each
static dim3 conv_grid(int ncb, int nparts) {
  return dim3((unsigned)(((int64_t)ncb * nparts + CONV_WAVES - 1) / CONV_WAVES));
}

template <typename T, int NG>
static hipError_t conv_fwd_k(const ConvArgs& a) {
  const int ncb = conv_blocks(a.n), D = a.n[0] + a.n[1] + a.n[2];
  const int L = conv_len(a.B, a.T, ncb, false), nchunk = (a.T + L - 1) / L, nparts = a.B * nchunk;
  ConvGroups<T> g;
  for (int i = 0; i < 3; ++i) g.p[i] = static_cast<T*>(a.y[i]), g.n[i] = a.n[i];
  g.normed = NG > 0 ? a.normed : 0;
  conv_silu_fwd_kernel<T, 4, NG><<<conv_grid(ncb, nparts), 64 * CONV_WAVES, 0, a.stream>>>(
      static_cast<const T*>(a.x), a.w, a.bias, static_cast<const T*>(a.state_in), g, static_cast<T*>(a.state_out),
      a.T, D, (int)a.ldx, L, nchunk, nparts);
  return hipGetLastError();
}

template <typename T, int NG, bool BIAS>
static hipError_t conv_bwd_k(const ConvArgs& a) {
  const int ncb = conv_blocks(a.n), D = a.n[0] + a.n[1] + a.n[2];
  const int L = conv_len(a.B, a.T, ncb, true), nchunk = (a.T + L - 1) / L, nparts = a.B * nchunk;
  ConvGroups<const T> g;
  for (int i = 0; i < 3; ++i) g.p[i] = static_cast<const T*>(a.dy[i]), g.n[i] = a.n[i];
  g.normed = NG > 0 ? a.normed : 0;
  float* part = static_cast<float*>(a.ws);
  const int ldp = D * 4 + (BIAS ? D : 0);
  conv_silu_bwd_kernel<T, 4, NG, BIAS><<<conv_grid(ncb, nparts), 64 * CONV_WAVES, 0, a.stream>>>(
      static_cast<const T*>(a.x), a.w, a.bias, static_cast<const T*>(a.state_in), g, static_cast<T*>(a.dx),
      static_cast<T*>(a.dstate_in), part, ldp, a.T, D, (int)a.ldx, (int)a.lddx, L, nchunk, nparts);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_column_sum(part, nparts, ldp, ColumnOut{{a.dw, a.dbias, nullptr}, {D * 4, ldp - D * 4, 0}}, a.stream);
}

template <typename T, int NG>
static hipError_t conv_k(const ConvArgs& a, bool backward) {
  if (!backward) return conv_fwd_k<T, NG>(a);
  return a.bias || a.dbias ? conv_bwd_k<T, NG, true>(a) : conv_bwd_k<T, NG, false>(a);
}

template <typename T>
static hipError_t conv_dispatch(const ConvArgs& a, bool backward) {
  switch (a.norm_group) {
    case 0: return conv_k<T, 0>(a, backward);
    case 64: return conv_k<T, 64>(a, backward);
    case 128: return conv_k<T, 128>(a, backward);
    case 256: return conv_k<T, 256>(a, backward);
  }
  return hipErrorInvalidValue;
}

template <typename WT>
static hipError_t decode_stage_w(const DecodeStageArgs& a) {
  const int wgs = (int)conv_grid(conv_blocks(a.n), a.B).x, gate_wgs = (a.B * a.H + 64 * CONV_WAVES - 1) / (64 * CONV_WAVES);
  const dim3 grid(wgs + gate_wgs), block(64 * CONV_WAVES);
  switch (a.norm_group) {
    case 64: decode_stage_kernel<WT, 64><<<grid, block, 0, a.stream>>>(a, wgs); break;
    case 128: decode_stage_kernel<WT, 128><<<grid, block, 0, a.stream>>>(a, wgs); break;
    case 256: decode_stage_kernel<WT, 256><<<grid, block, 0, a.stream>>>(a, wgs); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
hipError_t launch_decode_stage(const DecodeStageArgs& a) {
  return a.w_dtype == DT_BF16 ? decode_stage_w<bf16>(a) : decode_stage_w<float>(a);
}

hipError_t launch_conv(const ConvArgs& a, bool backward) {
  return a.dtype == DT_BF16 ? conv_dispatch<bf16>(a, backward) : conv_dispatch<float>(a, backward);
}

}  // namespace gdn
