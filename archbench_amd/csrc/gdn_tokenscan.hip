// Exact fp32 token scan of the n-step gated DeltaNet, forward and reverse-time backward: the reference's
// "triton" / "ref" scan (archbench/layers/nsgdn.py:80-154, ops :162-216; the recurrence of nsgdn_ref, :408-417).
// Per token t of a (b, h) sequence, with the state S [V, K] fp32 from zero (or from an initial state):
//     S <- e^{la_t} S;   r_t = v_t - S k_t;   S <- S + r_t u_t^T;   y_t = S q_t.
// Rows of S are independent given the token stream.  Sixteen lanes (one DPP row) share RL rows of S, lane part
// p = l & 15 holding K / 16 entries of each in registers, so a row's dot products (S k, S q, G u) are a partial sum per
// lane and four DPP steps.  k, u, q of a token are workgroup-uniform and reach the lanes through LDS, staged a block of
// tokens at a time (double-buffered: the next block is staged while one computes, one barrier per block).  A row's
// per-token scalars (v; r and dy in the backward) are loaded once per block, one token per lane, and broadcast inside
// the DPP row (row_newbcast); e^{la} is computed by one lane per token and read with readlane; a block's results are
// kept by the lane of their token and leave in one store.  So the chain from token to token is a handful of
// arithmetic steps: no load, store, transcendental or branch stands in it.
// Every CT tokens the forward stores S (the checkpoint the backward restarts from) in [K][V] order.
// The backward walks the checkpoints in reverse and each chunk in groups of four tokens, last first: it recomputes
// a group's states forward from the state entering the group (stored by a forward pass over the chunk from its
// checkpoint), keeping e^{la} S before each token's update in registers and accumulating dq = sum_rows S_t^T dy_t,
// then runs the group's tokens backward with the state gradient G [V, K] in registers beside S:
//     G += dy_t q_t^T;  dv_t = G u_t;  du_t = sum_rows G r_t;  G -= dv_t k_t^T;
//     dk_t = -sum_rows (e^{la} S_{t-1}) dv_t;  dla_t = sum (G o e^{la} S_{t-1});  G <- e^{la_t} G.
// Sums over rows are formed over a lane's own rows, then a reduce-scatter over the wave's four row groups (lane swaps,
// no LDS crossbar), then over the waves through LDS (a fixed order, no atomics), then over a head's workgroups through
// partial rows that are added afterwards.
// Only G needs the tokens in reverse order one by one: S restarts from any checkpoint.  With few sequences the backward
// is therefore split (ts_bwd_plan): token_scan_gstate_kernel runs G's recurrence alone, at the forward's pace, leaving dv
// and G at every chunk's end, and the rest runs with the chunks in parallel.
// Bound: the forward and G's recurrence by the chain (per token at K = 128 about 0.24 and 0.21 us: a dot product and its
// row sum, the update and the reads between them) until a SIMD holds two waves or more, the rest of the backward by its
// arithmetic (its row sums over the state's rows included, about 330 instructions per token and wave) at two waves per
// SIMD, a 64-row chunk of 32 tokens in 57 us.  B4 T1024 H4 K128 V256: forward 507 -> 235 us (eight lanes per row with the
// token's loads, stores, expf and LDS row sums in the chain before), backward 1916 -> 908 (as one chain) -> 216 + 459 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "gdn_common.h"
#include "gdn_launch.h"

namespace gdn {

constexpr int TS_CT = 32;   // tokens between checkpoints
constexpr int TS_GS = 4;    // tokens per group of the backward (decayed states held in registers)
constexpr int TS_TB = 8;    // tokens per block of the forward
constexpr int TS_LPR = 16;  // lanes per row: one DPP row
static_assert(TS_CT % TS_TB == 0, "checkpoints fall on block starts");

// A workgroup's share of the state: RL rows per lane, four row groups per wave
template <int RL_, int WAVES_>
struct TsShape {
  static constexpr int RL = RL_, WAVES = WAVES_, THREADS = 64 * WAVES, WROWS = 4 * RL, ROWS = WROWS * WAVES;
  static_assert(RL == 1 || RL == 2, "a group's row scalars fit the sixteen lanes of a row");
  static_assert((WAVES & (WAVES - 1)) == 0, "the waves' sums are added as a binary tree");
};

// The block / group barrier orders LDS only (the staged vectors and the row sums): __syncthreads() would also wait
// for every global load in flight, the next block's included, and so expose a memory latency per barrier.
__device__ __forceinline__ void ts_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// f(integral_constant<0>), ..., f(integral_constant<N - 1>): DPP and readlane patterns need constant indexes
template <typename F, int... I>
__device__ __forceinline__ void ts_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void ts_for(F&& f) {
  ts_for_impl(f, std::make_integer_sequence<int, N>{});
}

// lane I's value of each 16-lane row, in every lane of the row (row_newbcast:I)
template <int I>
__device__ __forceinline__ float ts_row_bcast(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x150 + I, 0xf, 0xf, true));
}
template <int I>
__device__ __forceinline__ float ts_lane(float x) {  // lane I's value, uniform over the wave
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), I));
}

// `x` is kept as computed here: a select on a lane index would otherwise sink x's last steps under an exec-mask branch
__device__ __forceinline__ float ts_pin(float x) {
  asm volatile("" : "+v"(x));
  return x;
}

// Reduce-scatter over a wave's four row groups: N values per lane (its part's columns, already summed over the lane's
// rows), summed over the lanes that share l & 15.  With R = N / 4, lane l ends with the sums of columns
// m + R (l >> 4), m < R, in a[0 .. R).  Each round pairs lanes that differ in one bit and hold the same column set: one
// keeps the lower half of its set, the other the upper half, and each adds what its partner sends
// (v_permlane32_swap of (a[m], a[m + N/2]) gives the lower half-wave its partner's a[m] and the upper half its partner's
// a[m + N/2], each keeping its own in the other result, so one add finishes the round; v_permlane16_swap likewise
// between even and odd 16-lane rows).
template <int N>
__device__ __forceinline__ void ts_rows_rs(float (&a)[N]) {
#pragma unroll
  for (int m = 0; m < N / 2; ++m) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[m]), __float_as_uint(a[m + N / 2]), false, false);
    a[m] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
#pragma unroll
  for (int m = 0; m < N / 4; ++m) {
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a[m]), __float_as_uint(a[m + N / 4]), false, false);
    a[m] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
}

// Row sums of RL values at once (left in every lane of the row): a DPP step may read its source only two instructions
// after it was written, so each of the four steps is followed by a quarter of the RL * N independent instructions that
// `fill` issues (fill(j), j < N: at least two per step) instead of idling; the scheduling barriers keep them there.
template <int RL, int N, typename F>
__device__ __forceinline__ void ts_row_sums(float (&d)[RL], F&& fill) {
  ts_for<4>([&](auto S) {
    constexpr int s = decltype(S)::value, CTRL = s == 0 ? 0xb1 : s == 1 ? 0x4e : s == 2 ? 0x141 : 0x140;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < RL; ++i) d[i] = dpp_sum_step<CTRL>(d[i]);
#pragma unroll
    for (int j = s * N / 4; j < (s + 1) * N / 4; ++j) fill(j);
  });
  __builtin_amdgcn_sched_barrier(0);
}
// One round of a reduce-scatter over a row's lanes: a[0 .. 2N) -> a[0 .. N); the lane whose bit is clear keeps a[k] and
// sends a[k + N] to its partner under CTRL, which has the bit set and does the reverse.
template <int N, int CTRL>
__device__ __forceinline__ void ts_lane_rs(float* a, bool hi) {
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const float keep = hi ? a[k + N] : a[k], send = hi ? a[k] : a[k + N];
    a[k] = keep + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(send), CTRL, 0xf, 0xf, true));
  }
}

// sum of a lane's products, in four chains
template <int N>
__device__ __forceinline__ float ts_dot(const float (&a)[N], const float (&b)[N]) {
  float d[4] = {a[0] * b[0], a[1] * b[1], a[2] * b[2], a[3] * b[3]};
#pragma unroll
  for (int j = 4; j < N; ++j) d[j & 3] = fmaf(a[j], b[j], d[j & 3]);
  return (d[0] + d[1]) + (d[2] + d[3]);
}

// A token's k, u, q in LDS: per vector sixteen parts of K / 16 floats, padded so that the lanes of a row (one per part)
// read different banks with 16-byte reads (K = 64: one piece each, contiguous).  Piece p < 3 K / 4 of a token is one
// float4, loaded into a register well ahead of its token and stored here before it.
template <int K>
struct TokStage {
  static constexpr int KQ = K / TS_LPR, K4 = K / 4, LD = KQ == 4 ? 4 : KQ + 4, VEC = TS_LPR * LD, SIZE = 3 * VEC;
  static constexpr int PER = 3 * K4;  // pieces per token
  static_assert(KQ % 4 == 0, "a lane's part of a vector is read in 16-byte pieces");
  static __device__ __forceinline__ f32x4 load(const float* kp, const float* up, const float* qp, int64_t t, int piece) {
    const int vec = piece / K4, e4 = piece - vec * K4;
    const float* src = vec == 0 ? kp : vec == 1 ? up : qp;
    return *reinterpret_cast<const f32x4*>(src + t * K + 4 * e4);
  }
  static __device__ __forceinline__ void stage(float* sv, int piece, const f32x4& x) {
    const int vec = piece / K4, c = 4 * (piece - vec * K4), qd = c / KQ;
    *reinterpret_cast<f32x4*>(sv + vec * VEC + qd * LD + c - qd * KQ) = x;
  }
  // this lane's part of staged vector vec
  static __device__ __forceinline__ void read(const float* sv, int vec, int part, float (&o)[KQ]) {
    const f32x4* p = reinterpret_cast<const f32x4*>(sv + vec * VEC + part * LD);
#pragma unroll
    for (int m = 0; m < KQ / 4; ++m) {
      const f32x4 t = p[m];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[4 * m + e] = t[e];
    }
  }
};

// grid B * H * NB (NB = ceil(V / ROWS)) workgroups: workgroup x -> (b h, row block vb).  Tokens past the end of the
// sequence in the last block are identity tokens (zero vectors, v = 0, la = 0), which leave a finite S as it is; nothing
// is stored for them.
// FIN: the final state is wanted (its epilogue in the other calls' kernel cost them 1%).
template <int K, typename SH, bool FIN>
__global__ __launch_bounds__(SH::THREADS) void token_scan_fwd_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ u, const float* __restrict__ v,
    const float* __restrict__ la, const float* __restrict__ h0, float* __restrict__ y, float* __restrict__ r,
    float* __restrict__ st, float* __restrict__ hT, int T_, int H, int V, int NCH, int NB) {
  using TS = TokStage<K>;
  constexpr int KQ = TS::KQ, RL = SH::RL, NL = (TS_TB * TS::PER + SH::THREADS - 1) / SH::THREADS;
  __shared__ __attribute__((aligned(16))) float sv[2][TS_TB][TS::SIZE];
  const int tid = threadIdx.x, l = lane_id(), p = l & 15;
  const int pid = blockIdx.x, bh = pid / NB, vb = pid - bh * NB;
  const int b = bh / H, h = bh - b * H;
  const int v0 = vb * SH::ROWS + wave_id() * SH::WROWS + (l >> 4) * RL;  // this lane's rows v0 .. v0 + RL - 1
  // states [B, H, K, V] (fla's layout): entry (row v0 + i, column p KQ + j) at cb + j V + i
  const int64_t cb = (int64_t)bh * K * V + (int64_t)p * KQ * V + v0;
  float S[RL][KQ];
#pragma unroll
  for (int i = 0; i < RL; ++i)
#pragma unroll
    for (int j = 0; j < KQ; ++j) S[i][j] = h0 && v0 + i < V ? h0[cb + (int64_t)j * V + i] : 0.f;
  float* stb = st + (int64_t)bh * NCH * K * V;  // uniform; this lane's entries at st_off + j V + i of a checkpoint
  const int64_t st_off = (int64_t)p * KQ * V + v0;
  const int64_t tok_first = (int64_t)b * T_ * H + h;
  // block t0's row scalars: this lane loads v of token p >> 1 for its row (RL = 2: row p & 1), and la of that token; the
  // block's vectors: piece e < TB * PER is float4 e % PER of token t0 + e / PER
  const int ti = p >> 1, vs = v0 + (RL == 2 ? p & 1 : 0);
  f32x4 xr[NL];
  float vn = 0.f, ln = 0.f;
  auto load_block = [&](int t0) {
#pragma unroll
    for (int m = 0; m < NL; ++m) {
      const int e = tid + m * SH::THREADS, i = e / TS::PER;
      xr[m] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (e < TS_TB * TS::PER && t0 + i < T_)
        xr[m] = TS::load(k, u, q, tok_first + (int64_t)(t0 + i) * H, e - i * TS::PER);
    }
    const bool in = t0 + ti < T_;
    const int64_t tk = tok_first + (int64_t)(t0 + ti) * H;
    vn = in && vs < V ? v[tk * V + vs] : 0.f;
    ln = in ? la[tk] : 0.f;
  };
  auto stage_block = [&](float (*dst)[TS::SIZE]) {
#pragma unroll
    for (int m = 0; m < NL; ++m) {
      const int e = tid + m * SH::THREADS, i = e / TS::PER;
      if (e < TS_TB * TS::PER) TS::stage(dst[i], e - i * TS::PER, xr[m]);
    }
  };
  load_block(0);  // T_ >= 1 here (the host returns before launching an empty scan)
  stage_block(sv[0]);
  float vc = vn, ac = expf(ln);
  if (TS_TB < T_) load_block(TS_TB);
  ts_barrier();
  for (int t0 = 0, blk = 0; t0 < T_; t0 += TS_TB, ++blk) {
    if (t0 % TS_CT == 0) {
      const int64_t c = t0 / TS_CT;
#pragma unroll
      for (int i = 0; i < RL; ++i)
        if (v0 + i < V) {
#pragma unroll
          for (int j = 0; j < KQ; ++j) stb[c * K * V + (int64_t)j * V + (st_off + i)] = S[i][j];
        }
    }
    const float(*sb)[TS::SIZE] = sv[blk & 1];
    float rout[RL] = {}, ypart[RL][TS_TB];  // lane 2 i + 1: r of token i; this lane's part of each token's y
    // the next token's vectors are read from LDS before this token's arithmetic, so their latency is off the chain
    float vec[2][3][KQ];
    auto read3 = [&](int i, float (&d)[3][KQ]) {
      TS::read(sb[i], 0, p, d[0]);
      TS::read(sb[i], 1, p, d[1]);
      TS::read(sb[i], 2, p, d[2]);
    };
    read3(0, vec[0]);
    ts_for<TS_TB>([&](auto I) {
      constexpr int i = decltype(I)::value;
      if constexpr (i + 1 < TS_TB) read3(i + 1, vec[(i + 1) & 1]);
      const auto& kk = vec[i & 1][0];
      const auto& uu = vec[i & 1][1];
      const auto& qq = vec[i & 1][2];
      const float a = ts_lane<2 * i>(ac);
      float d[RL], vr[RL];
      ts_for<RL>([&](auto RI) {
        constexpr int rr = decltype(RI)::value;
        d[rr] = ts_dot(S[rr], kk);
        vr[rr] = ts_row_bcast<2 * i + (RL == 2 ? rr : 0)>(vc);
      });
      // r = v - a (S k), with the decay of S in the gaps of the row sum
      ts_row_sums<RL, KQ>(d, [&](int j) {
#pragma unroll
        for (int rr = 0; rr < RL; ++rr) S[rr][j] *= a;
      });
#pragma unroll
      for (int rr = 0; rr < RL; ++rr) {
        const float res = fmaf(-a, d[rr], vr[rr]);
#pragma unroll
        for (int j = 0; j < KQ; ++j) S[rr][j] = fmaf(res, uu[j], S[rr][j]);
        rout[rr] = p == 2 * i + 1 ? res : rout[rr];
        ypart[rr][i] = ts_dot(S[rr], qq);
      }
    });
    // y: the block's eight partials reduce-scattered over the row's lanes (bits 3, 2, 1 of p select the token, bit 0 is
    // summed), so lane p ends with token p >> 1's
    static_assert(TS_TB == 8, "three rounds scatter the block's tokens");
    float out[RL];
#pragma unroll
    for (int i = 0; i < RL; ++i) {
      float* a = ypart[i];
      ts_lane_rs<4, 0x140>(a, p & 8);
      ts_lane_rs<2, 0x141>(a, p & 4);
      ts_lane_rs<1, 0x4e>(a, p & 2);
      const float yy = ts_pin(dpp_sum_step<0xb1>(a[0]));
      out[i] = p & 1 ? rout[i] : yy;
    }
    if (t0 + TS_TB < T_) {  // stage the next block (loaded a block ago); before the stores below, whose way to memory
      stage_block(sv[(blk + 1) & 1]);  // the wait for these loads would otherwise include
      vc = vn;
      ac = expf(ln);
    }
    if (t0 + ti < T_) {
      const int64_t tok = tok_first + (int64_t)(t0 + ti) * H;
      float* dst = (p & 1 ? r : y) + tok * V + v0;
#pragma unroll
      for (int i = 0; i < RL; ++i)
        if (v0 + i < V) dst[i] = out[i];
    }
    if (t0 + 2 * TS_TB < T_) load_block(t0 + 2 * TS_TB);
    ts_barrier();  // the block's vectors read by every lane; the next block's staged
  }
  if constexpr (FIN) {
    // an infinite entry of S has become a NaN at the identity tokens (their S k is inf 0): such a wave steps from the last
    // checkpoint to the end again with the r it stored
    bool nan = false;
#pragma unroll
    for (int i = 0; i < RL; ++i)
#pragma unroll
      for (int j = 0; j < KQ; ++j) nan |= S[i][j] != S[i][j];
    if (T_ % TS_TB != 0 && __any(nan)) {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      const int64_t c = (T_ - 1) / TS_CT;
      for (int i = 0; i < RL; ++i)
        if (v0 + i < V)
          for (int j = 0; j < KQ; ++j) {
            float s = stb[c * K * V + (int64_t)j * V + (st_off + i)];
            for (int t = (int)c * TS_CT; t < T_; ++t) {
              const int64_t tok = tok_first + (int64_t)t * H;
              s = fmaf(r[tok * V + v0 + i], u[tok * K + p * KQ + j], s * expf(la[tok]));
            }
            hT[cb + (int64_t)j * V + i] = s;
          }
      return;
    }
#pragma unroll
    for (int i = 0; i < RL; ++i)
      if (v0 + i < V) {
#pragma unroll
        for (int j = 0; j < KQ; ++j) hT[cb + (int64_t)j * V + i] = S[i][j];
      }
  }
}

// The row sums of a group's steps: each wave's column sums (after ts_rows_rs) and its dla go to LDS slots of their
// own (vector, token), and after the group's barrier the waves are added in a fixed order and stored as the
// workgroup's partial rows (double-buffered by group parity).
template <int K, typename SH>
struct TokSums {
  static constexpr int KQ = K / TS_LPR, R = KQ / 4;
  float col[2][3][TS_GS][SH::WAVES][K];  // [parity][dq, du, dk][token][wave][column]
  float sca[2][SH::WAVES][TS_GS];        // [parity][wave][token]: dla
  // this wave's reduce-scattered sums into slot (vec, i)
  __device__ __forceinline__ void put(int par, int vec, int i, const float (&a)[KQ], int l) {
    float* d = &col[par][vec][i][wave_id()][(l & 15) * KQ + R * (l >> 4)];
#pragma unroll
    for (int m = 0; m < R; ++m) d[m] = a[m];
  }
  // the waves' values added as a pairwise tree (a fixed order)
  template <typename X, typename F>
  static __device__ __forceinline__ X tree(F&& x) {
    X a[SH::WAVES];
#pragma unroll
    for (int w = 0; w < SH::WAVES; ++w) a[w] = x(w);
#pragma unroll
    for (int h = SH::WAVES / 2; h >= 1; h /= 2) {
#pragma unroll
      for (int w = 0; w < h; ++w) a[w] = a[2 * w] + a[2 * w + 1];
    }
    return a[0];
  }
  __device__ __forceinline__ f32x4 col_sum4(int par, int vec, int i, int c) const {
    return tree<f32x4>([&](int w) { return *reinterpret_cast<const f32x4*>(&col[par][vec][i][w][c]); });
  }
  __device__ __forceinline__ float sca_sum(int par, int i) const {
    return tree<float>([&](int w) { return sca[par][w][i]; });
  }
};

// Partials: gqp, gup, gkp [NB][B*T*H][K], glap [NB][B*T*H]; sc [B*H*NB][TS_CT / TS_GS][THREADS][RL K / 16] scratch of
// the chunk's group-start states.
// Per chunk (last first), in groups of TS_GS tokens: a forward pass from the checkpoint stores the state entering each
// group but the first and last (the last stays in registers); then, group by group from the last, the group's tokens
// are recomputed forward from its start state with each decayed state e^{la} S_{t-1} kept in registers (and dq
// accumulated), and walked backward.  A short last group is padded with identity tokens (la = 0, zero vectors and
// row values), which change neither S nor G, and whose sums are not stored.  The forward pass has the chunk's u in LDS
// at once; the groups' vectors are staged (and their row values loaded) a group ahead: one barrier per group.
// SPLIT: G at each chunk's end (gst, [BH][NCH][K][V]) and dv come from token_scan_gstate_kernel, so that the chunks are
// independent: nitems = BH NCH NB (bh, chunk, row block) items, walked by the grid's workgroups (scratch per workgroup).
// Otherwise a workgroup is a (bh, row block) and carries G through its chunks, computing dv and dh0.
template <int K, typename SH, bool SPLIT>
__global__ __launch_bounds__(SH::THREADS) __attribute__((amdgpu_waves_per_eu(2))) void token_scan_bwd_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ u, const float* __restrict__ la,
    const float* __restrict__ r, const float* __restrict__ st, const float* __restrict__ gy,
    const float* __restrict__ dhT, float* __restrict__ gv, float* __restrict__ gqp, float* __restrict__ gup,
    float* __restrict__ gkp, float* __restrict__ glap, float* __restrict__ dh0, float* __restrict__ sc,
    const float* __restrict__ gst, int nitems, int T_, int H, int V, int NCH, int NB, int64_t ntok) {
  using TS = TokStage<K>;
  constexpr int KQ = TS::KQ, RL = SH::RL, THREADS = SH::THREADS, NGS = TS_CT / TS_GS;
  constexpr int NL = (TS_GS * TS::PER + THREADS - 1) / THREADS;
  __shared__ __attribute__((aligned(16))) float sv[2][TS_GS][TS::SIZE];
  __shared__ __attribute__((aligned(16))) TokSums<K, SH> sums;
  const int tid = threadIdx.x, l = lane_id(), p = l & 15;
  const int pid = blockIdx.x;
  constexpr int SV = RL * KQ / 4;  // 16-byte pieces of this lane's state
  f32x4* scw = reinterpret_cast<f32x4*>(sc + (int64_t)pid * NGS * RL * KQ * THREADS);
  const unsigned sc_off = (unsigned)tid * SV;
  auto put_state = [&](int g, const float (&X)[RL][KQ]) {
#pragma unroll
    for (int m = 0; m < SV; ++m) {
      const int i = 4 * m / KQ, j = 4 * m % KQ;
      scw[(unsigned)(g * THREADS * SV) + (sc_off + m)] = f32x4{X[i][j], X[i][j + 1], X[i][j + 2], X[i][j + 3]};
    }
  };
  auto get_state = [&](int g, float (&X)[RL][KQ]) {
#pragma unroll
    for (int m = 0; m < SV; ++m) {
      const int i = 4 * m / KQ, j = 4 * m % KQ;
      const f32x4 t = scw[(unsigned)(g * THREADS * SV) + (sc_off + m)];
#pragma unroll
      for (int e = 0; e < 4; ++e) X[i][j + e] = t[e];
    }
  };
  f32x4 xr[NL];  // this thread's pieces of the next group's vectors (piece e: token e / PER), loaded a group ahead
  // The group's row scalars, one token per lane: lane p holds r of token p & 3 and row p >> 2 for p < 4 RL, dy likewise
  // for the next 4 RL lanes; and la of token l & 3
  const int ti = p & 3, si = p >> 2, srow_off = RL == 2 ? si & 1 : 0;
  const float* sp = (RL == 2 ? si >= 2 : (si & 1)) ? gy : r;
  float xn, ln, xc, ac, dn = 0.f, dc = 0.f;  // dn, dc (SPLIT): dv of token p & 3, row p >> 2, for p < 4 RL
  int v0 = 0, srow = 0;
  auto load_grp = [&](auto&& tok_at) {  // tok_at(i): token i of the group (< 0: an identity token)
#pragma unroll
    for (int m = 0; m < NL; ++m) {
      const int e = tid + m * THREADS, pi = e / TS::PER;
      xr[m] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (e < TS_GS * TS::PER) {
        const int64_t tk = tok_at(pi);
        if (tk >= 0) xr[m] = TS::load(k, u, q, tk, e - pi * TS::PER);
      }
    }
    const int64_t tk = tok_at(ti);
    xn = tk >= 0 && srow < V ? sp[tk * V + srow] : 0.f;
    ln = tk >= 0 ? la[tk] : 0.f;
    if constexpr (SPLIT) dn = tk >= 0 && p < 4 * RL && srow < V ? gv[tk * V + srow] : 0.f;
  };
  auto stage_grp = [&](int buf) {
#pragma unroll
    for (int m = 0; m < NL; ++m) {
      const int e = tid + m * THREADS, pi = e / TS::PER;
      if (e < TS_GS * TS::PER) TS::stage(sv[buf][pi], e - pi * TS::PER, xr[m]);
    }
    xc = xn;
    ac = expf(ln);
    dc = dn;
  };
  int par = 0;  // parity of the group: sv[par & 1] holds its vectors, sums[par & 1] takes its row sums
  float G[RL][KQ], S[RL][KQ];
  if constexpr (!SPLIT) {
    const int bh = pid / NB;
    v0 = (pid - bh * NB) * SH::ROWS + wave_id() * SH::WROWS + (l >> 4) * RL;  // this lane's rows, as in the forward
    srow = v0 + srow_off;
    const int64_t cb = (int64_t)bh * K * V + (int64_t)p * KQ * V + v0;  // [B, H, K, V] states, as in the forward
#pragma unroll
    for (int i = 0; i < RL; ++i)
#pragma unroll
      for (int j = 0; j < KQ; ++j) G[i][j] = dhT && v0 + i < V ? dhT[cb + (int64_t)j * V + i] : 0.f;
  }
  for (int it = SPLIT ? pid : NCH - 1; SPLIT ? it < nitems : it >= 0; it += SPLIT ? (int)gridDim.x : -1) {
    // uniform, and said so: the divisions leave their results in vector registers
    const int bc = SPLIT ? __builtin_amdgcn_readfirstlane(it / NB) : 0;  // (bh, chunk)
    const int bh = SPLIT ? __builtin_amdgcn_readfirstlane(bc / NCH) : pid / NB, c = SPLIT ? bc - bh * NCH : it;
    const int vb = SPLIT ? it - bc * NB : pid - bh * NB;
    const int b = bh / H, h = bh - b * H;
    if constexpr (SPLIT) {
      v0 = vb * SH::ROWS + wave_id() * SH::WROWS + (l >> 4) * RL;
      srow = v0 + srow_off;
    }
    // uniform bases and 32-bit lane offsets: per-lane 64-bit addresses of the unrolled accesses would fill the registers
    const float* stb = st + (int64_t)bh * NCH * K * V;
    const int64_t st_off = (int64_t)p * KQ * V + v0;
    float* const gout[3] = {gqp + (int64_t)vb * ntok * K, gup + (int64_t)vb * ntok * K, gkp + (int64_t)vb * ntok * K};
    float* gl_b = glap + (int64_t)vb * ntok;
    if constexpr (SPLIT) {
      const float* g0 = gst + ((int64_t)bh * NCH + c) * K * V;
#pragma unroll
      for (int i = 0; i < RL; ++i)
#pragma unroll
        for (int j = 0; j < KQ; ++j) G[i][j] = v0 + i < V ? g0[(int64_t)j * V + (st_off + i)] : 0.f;
    }
    const int n = min(TS_CT, T_ - c * TS_CT), ng = (n + TS_GS - 1) / TS_GS;
    const int64_t tok0 = ((int64_t)b * T_ + (int64_t)c * TS_CT) * H + h;
    auto tok_in = [&](int g, int i) -> int64_t {
      const int t = g * TS_GS + i;
      return t < n ? tok0 + (int64_t)t * H : -1;
    };
    auto load_state = [&](float (&X)[RL][KQ]) {  // the chunk's checkpoint
#pragma unroll
      for (int i = 0; i < RL; ++i)
#pragma unroll
        for (int j = 0; j < KQ; ++j)
          X[i][j] = v0 + i < V ? stb[(int64_t)c * K * V + (int64_t)j * V + (st_off + i)] : 0.f;
    };
    load_state(S);
    // forward from the checkpoint to the last group's start, storing the start states of groups 1 .. ng - 2: the chunk's
    // u staged whole (over the row sums, which are free between chunks), so no barrier stands between its groups
    if (ng > 1) {
      constexpr int NU = (TS_CT * TS::K4 + THREADS - 1) / THREADS;
      f32x4 xu[NU];
      float rc[RL][2], a32;
#pragma unroll
      for (int m = 0; m < NU; ++m) {
        const int e = tid + m * THREADS, t = e / TS::K4;
        xu[m] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (t < n) xu[m] = *reinterpret_cast<const f32x4*>(u + (tok0 + (int64_t)t * H) * K + 4 * (e - t * TS::K4));
      }
#pragma unroll
      for (int i = 0; i < RL; ++i)
#pragma unroll
        for (int m = 0; m < 2; ++m)
          rc[i][m] = p + 16 * m < n && v0 + i < V ? r[(tok0 + (int64_t)(p + 16 * m) * H) * V + v0 + i] : 0.f;
      a32 = (l & 31) < n ? la[tok0 + (int64_t)(l & 31) * H] : 0.f;
      ts_barrier();  // the previous chunk's last row sums read
      float* su = &sums.col[0][0][0][0][0];
      static_assert(sizeof(sums.col) >= TS_CT * TS::VEC * 4, "the chunk's u fits over the row sums");
#pragma unroll
      for (int m = 0; m < NU; ++m) {
        const int e = tid + m * THREADS, t = e / TS::K4, cc = 4 * (e - t * TS::K4), qd = cc / KQ;
        if (t < TS_CT) *reinterpret_cast<f32x4*>(su + t * TS::VEC + qd * TS::LD + cc - qd * KQ) = xu[m];
      }
      a32 = expf(a32);
      ts_barrier();
      ts_for<NGS - 1>([&](auto GI) {
        constexpr int g = decltype(GI)::value;
        __builtin_amdgcn_sched_barrier(0);  // one group's reads at a time (registers)
        if (g < ng - 1) {
          if (g > 0) put_state(g, S);
          float uu[TS_GS][KQ];
#pragma unroll
          for (int i = 0; i < TS_GS; ++i) TS::read(su + (g * TS_GS + i) * TS::VEC, 0, p, uu[i]);
          ts_for<TS_GS>([&](auto I) {
            constexpr int i = decltype(I)::value, t = g * TS_GS + i;
            const float a = ts_lane<t>(a32);
            ts_for<RL>([&](auto RI) {
              constexpr int rr = decltype(RI)::value;
              const float rt = ts_row_bcast<(t & 15)>(rc[rr][t >> 4]);
#pragma unroll
              for (int j = 0; j < KQ; ++j) S[rr][j] = fmaf(rt, uu[i][j], S[rr][j] * a);
            });
          });
        }
      });
    }
    auto flush = [&](int g, int pb) {  // the group's row sums, from LDS slots of parity pb, four columns at a time
      constexpr int KV = K / 4, NF = 3 * TS_GS * KV;
#pragma unroll
      for (int m = 0; m < (NF + THREADS - 1) / THREADS; ++m) {
        const int o = tid + m * THREADS;
        if (o < NF) {
          const int vec = o / (TS_GS * KV), rem = o - vec * TS_GS * KV, i = rem / KV, cc = 4 * (rem - i * KV);
          const int64_t tk = tok_in(g, i);
          if (tk >= 0) {
            float* dst = vec == 0 ? gout[0] : vec == 1 ? gout[1] : gout[2];
            *reinterpret_cast<f32x4*>(dst + tk * K + cc) = sums.col_sum4(pb, vec, i, cc);
          }
        }
      }
      if (tid < TS_GS) {
        const int64_t tk = tok_in(g, tid);
        if (tk >= 0) gl_b[tk] = sums.sca_sum(pb, tid);
      }
    };
    // groups last to first: TS_GS forward steps (tokens 0 .. TS_GS - 1 of the group), then TS_GS backward steps
    load_grp([&](int i) { return tok_in(ng - 1, i); });
    stage_grp(par & 1);
    if (ng > 1) load_grp([&](int i) { return tok_in(ng - 2, i); });
    ts_barrier();
    for (int g = ng - 1; g >= 0; --g, ++par) {
      const int pb = par & 1;
      // the state entering the group before this one, loaded while this one computes (split: while it walks backward,
      // S itself being free then)
      float Sn[RL][KQ];
      auto load_next = [&](float (&X)[RL][KQ]) {
        if (g > 1) get_state(g - 1, X);
        else if (!SPLIT || g == 1) load_state(X);  // the checkpoint (after the chunk's first group it is not used)
      };
      if constexpr (!SPLIT) load_next(Sn);
      if (g < ng - 1) flush(g + 1, pb ^ 1);
      float Sd[TS_GS][RL][KQ];  // e^{la} S_{t-1} of the group's tokens
      ts_for<TS_GS>([&](auto I) {
        constexpr int i = decltype(I)::value;
        __builtin_amdgcn_sched_barrier(0);
        const float a = ts_lane<i>(ac);
        float uu[KQ], t[KQ];
        TS::read(sv[pb][i], 1, p, uu);
        ts_for<RL>([&](auto RI) {
          constexpr int rr = decltype(RI)::value;
          const float rc = ts_row_bcast<4 * rr + i>(xc), gyc = ts_row_bcast<4 * RL + 4 * rr + i>(xc);
#pragma unroll
          for (int j = 0; j < KQ; ++j) {
            Sd[i][rr][j] = S[rr][j] * a;
            S[rr][j] = fmaf(rc, uu[j], Sd[i][rr][j]);
            t[j] = rr == 0 ? S[rr][j] * gyc : fmaf(S[rr][j], gyc, t[j]);
          }
        });
        ts_rows_rs(t);
        sums.put(pb, 0, i, t, l);
      });
      if constexpr (SPLIT) load_next(S);
      float out = 0.f, e4[TS_GS];  // lane p < 4 RL: dv of token p & 3, row p >> 2; the tokens' dla partials
      ts_for<TS_GS>([&](auto I) {
        constexpr int i = TS_GS - 1 - decltype(I)::value;
        if constexpr (SPLIT) __builtin_amdgcn_sched_barrier(0);  // one token's reads at a time (registers)
        const float a = ts_lane<i>(ac);
        float uu[KQ], kk[KQ], qq[KQ], t[KQ], t2[KQ];
        TS::read(sv[pb][i], 2, p, qq);
        if constexpr (!SPLIT) TS::read(sv[pb][i], 1, p, uu);
        TS::read(sv[pb][i], 0, p, kk);
        float d[RL], rc[RL];
        ts_for<RL>([&](auto RI) {
          constexpr int rr = decltype(RI)::value;
          rc[rr] = ts_row_bcast<4 * rr + i>(xc);
          const float gyc = ts_row_bcast<4 * RL + 4 * rr + i>(xc);
#pragma unroll
          for (int j = 0; j < KQ; ++j) G[rr][j] = fmaf(gyc, qq[j], G[rr][j]);
          if constexpr (SPLIT) d[rr] = ts_row_bcast<4 * rr + i>(dc);
          else d[rr] = ts_dot(G[rr], uu);
        });
        auto du_part = [&](int j) {
          t[j] = G[0][j] * rc[0];
          if constexpr (RL == 2) t[j] = fmaf(G[RL - 1][j], rc[RL - 1], t[j]);
        };
        if constexpr (SPLIT) {
#pragma unroll
          for (int j = 0; j < KQ; ++j) du_part(j);
        } else {
          ts_row_sums<RL, KQ>(d, du_part);
        }
        e4[i] = 0.f;
#pragma unroll
        for (int rr = 0; rr < RL; ++rr) {
          const float gr = d[rr];
          out = p == 4 * rr + i ? gr : out;
#pragma unroll
          for (int j = 0; j < KQ; ++j) {
            G[rr][j] = fmaf(-gr, kk[j], G[rr][j]);
            t2[j] = rr == 0 ? -Sd[i][rr][j] * gr : fmaf(-Sd[i][rr][j], gr, t2[j]);
          }
          e4[i] += ts_dot(G[rr], Sd[i][rr]);
#pragma unroll
          for (int j = 0; j < KQ; ++j) G[rr][j] *= a;
        }
        ts_rows_rs(t);
        sums.put(pb, 1, i, t, l);
        ts_rows_rs(t2);
        sums.put(pb, 2, i, t2, l);
      });
      ts_rows_rs(e4);  // lane group l >> 4: token l >> 4's partials
      e4[0] = sum16(e4[0]);
      if (p == 0) sums.sca[pb][wave_id()][l >> 4] = e4[0];
      if (g > 0) stage_grp((par + 1) & 1);  // the group before, loaded a group ago; ahead of the store, as in the forward
      if constexpr (!SPLIT) {
        const int64_t tk = tok_in(g, ti);
        if (p < 4 * RL && tk >= 0 && srow < V) gv[tk * V + srow] = out;
      }
      if (g > 1) load_grp([&](int i) { return tok_in(g - 2, i); });
      if constexpr (!SPLIT)
#pragma unroll
        for (int i = 0; i < RL; ++i)
#pragma unroll
          for (int j = 0; j < KQ; ++j) S[i][j] = Sn[i][j];
      ts_barrier();  // the group's vectors read and sums written; the group before staged
    }
    flush(0, (par - 1) & 1);
  }
  if constexpr (!SPLIT)
    if (dh0) {  // G is now the gradient of the state before the first token: the initial state's
      const int64_t cb = (int64_t)(pid / NB) * K * V + (int64_t)p * KQ * V + v0;
#pragma unroll
      for (int i = 0; i < RL; ++i)
        if (v0 + i < V) {
#pragma unroll
          for (int j = 0; j < KQ; ++j) dh0[cb + (int64_t)j * V + i] = G[i][j];
        }
    }
}

// The state gradient's own recurrence, in reverse time: dv, dh0 and G before each chunk's last token (gst).  The
// forward's mapping, blocks and staging with the token order reversed; per token
//     G = e^{la'} W + dy q^T (la' of the token after);  dv = G u;  W = G - dv k^T,
// dy q^T formed in the gaps of the row sum before.
template <int K, typename SH>
__global__ __launch_bounds__(SH::THREADS) void token_scan_gstate_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ u, const float* __restrict__ la,
    const float* __restrict__ gy, const float* __restrict__ dhT, float* __restrict__ gv, float* __restrict__ gst,
    float* __restrict__ dh0, int T_, int H, int V, int NCH, int NB) {
  using TS = TokStage<K>;
  static_assert(SH::RL == 1, "one row per lane");
  constexpr int KQ = TS::KQ, NL = (TS_TB * TS::PER + SH::THREADS - 1) / SH::THREADS;
  __shared__ __attribute__((aligned(16))) float sv[2][TS_TB][TS::SIZE];
  const int tid = threadIdx.x, l = lane_id(), p = l & 15;
  const int pid = blockIdx.x, bh = pid / NB, vb = pid - bh * NB;
  const int b = bh / H, h = bh - b * H;
  const int v0 = vb * SH::ROWS + wave_id() * SH::WROWS + (l >> 4);
  const bool row = v0 < V;
  const int64_t off = (int64_t)p * KQ * V + v0;  // this lane's entries of a [K][V] state: off + j V
  float* gb = gst + (int64_t)bh * NCH * K * V;
  const int64_t tok_first = (int64_t)b * T_ * H + h;
  const int ti = p >> 1;
  f32x4 xr[NL];
  float gn = 0.f, ln = 0.f;
  auto load_block = [&](int t0) {  // as in the forward, with dy in v's place
#pragma unroll
    for (int m = 0; m < NL; ++m) {
      const int e = tid + m * SH::THREADS, i = e / TS::PER;
      xr[m] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (e < TS_TB * TS::PER && t0 + i < T_)
        xr[m] = TS::load(k, u, q, tok_first + (int64_t)(t0 + i) * H, e - i * TS::PER);
    }
    const bool in = t0 + ti < T_;
    const int64_t tk = tok_first + (int64_t)(t0 + ti) * H;
    gn = in && row ? gy[tk * V + v0] : 0.f;
    ln = in ? la[tk] : 0.f;
  };
  auto stage_block = [&](float (*dst)[TS::SIZE]) {
#pragma unroll
    for (int m = 0; m < NL; ++m) {
      const int e = tid + m * SH::THREADS, i = e / TS::PER;
      if (e < TS_TB * TS::PER) TS::stage(dst[i], e - i * TS::PER, xr[m]);
    }
  };
  float G[KQ];
#pragma unroll
  for (int j = 0; j < KQ; ++j) G[j] = dhT && row ? dhT[(int64_t)bh * K * V + (int64_t)j * V + off] : 0.f;
  const int last = (T_ - 1) / TS_TB;  // T_ >= 1 here
  load_block(last * TS_TB);
  stage_block(sv[0]);
  float gc = gn, ac = expf(ln);
  if (last > 0) load_block((last - 1) * TS_TB);
  ts_barrier();
  for (int blk = last, buf = 0; blk >= 0; --blk, buf ^= 1) {
    const int t0 = blk * TS_TB;
    if (blk == last || (t0 + TS_TB) % TS_CT == 0) {  // the block ends its chunk
      const int64_t c = t0 / TS_CT;
      if (row) {
#pragma unroll
        for (int j = 0; j < KQ; ++j) gb[c * K * V + (int64_t)j * V + off] = G[j];
      }
    }
    const float(*sb)[TS::SIZE] = sv[buf];
    float vec[2][3][KQ], gq[KQ], dv = 0.f;  // lane 2 i: dv of token i
    auto read3 = [&](int i, float (&d)[3][KQ]) {
      TS::read(sb[i], 0, p, d[0]);
      TS::read(sb[i], 1, p, d[1]);
      TS::read(sb[i], 2, p, d[2]);
    };
    read3(TS_TB - 1, vec[(TS_TB - 1) & 1]);
    const float gy_last = ts_row_bcast<2 * (TS_TB - 1)>(gc);
#pragma unroll
    for (int j = 0; j < KQ; ++j) gq[j] = gy_last * vec[(TS_TB - 1) & 1][2][j];
    ts_for<TS_TB>([&](auto I) {
      constexpr int i = TS_TB - 1 - decltype(I)::value;
      if constexpr (i > 0) read3(i - 1, vec[(i - 1) & 1]);
      const auto& kk = vec[i & 1][0];
      const auto& uu = vec[i & 1][1];
      const float a = i + 1 < TS_TB ? ts_lane<(2 * i + 2) & 15>(ac) : 1.f;  // the block's last token: G is already decayed
#pragma unroll
      for (int j = 0; j < KQ; ++j) G[j] = i + 1 < TS_TB ? fmaf(a, G[j], gq[j]) : G[j] + gq[j];
      float d[1] = {ts_dot(G, uu)};
      const float gy_prev = i > 0 ? ts_row_bcast<(2 * i - 2) & 15>(gc) : 0.f;
      ts_row_sums<1, KQ>(d, [&](int j) {
        if constexpr (i > 0) gq[j] = gy_prev * vec[(i - 1) & 1][2][j];
      });
      dv = p == 2 * i ? d[0] : dv;
#pragma unroll
      for (int j = 0; j < KQ; ++j) G[j] = fmaf(-d[0], kk[j], G[j]);
    });
    const float a0 = ts_lane<0>(ac);
#pragma unroll
    for (int j = 0; j < KQ; ++j) G[j] *= a0;
    if (blk > 0) {  // stage the block before (loaded a block ago), ahead of the store, as in the forward
      stage_block(sv[buf ^ 1]);
      gc = gn;
      ac = expf(ln);
    }
    if (!(p & 1) && t0 + ti < T_ && row) gv[(tok_first + (int64_t)(t0 + ti) * H) * V + v0] = dv;
    if (blk > 1) load_block(t0 - 2 * TS_TB);
    ts_barrier();
  }
  if (dh0 && row) {
#pragma unroll
    for (int j = 0; j < KQ; ++j) dh0[(int64_t)bh * K * V + (int64_t)j * V + off] = G[j];
  }
}

// ---------------------------------------------------------------------------------------------------------
bool token_scan_supported(int K) { return K == 64 || K == 128; }
int token_scan_ct() { return TS_CT; }

// Rows per workgroup: 16 (one row per lane, four waves), 32 (eight waves) or, in the backward, 64 (two rows per lane).
// A lone workgroup's pace is set by its chain from token to token: with at most one workgroup per CU 16 rows are the
// fastest, and 32 cost less than two rounds of 16 (the token vectors staged once for twice the rows, half the
// backward's partial rows); two rows per lane share the row sums' reduce-scatter, so once there is more than one round
// of 32 the backward is bound by its arithmetic and 64 rows cost about three rounds of 16.  Hence the fewest rounds over
// the CUs in these weights (16: 1, 32: 2, 64: 3, ties to the larger of 16 and 32 and the smaller of 32 and 64).
// Measured, H4 K128 V256, forward + backward us at 16, 32 and 64 rows (forward: 32): T1024 B4 241 + 908, 311 + 1040,
// 313 + 1591; T512 B8 166 + 600, 163 + 553, 167 + 829; T512 B12 211 + 1035, 242 + 1086, 240 + 879; T512 B16 259 + 1182,
// 246 + 1116, 245 + 912; K64 V256 T256 B16 85 + 318, 83 + 333, 81 + 252; B36 T65 V96 42 + 147, 41 + 151, 40 + 234.
// (Before, with eight lanes per row and 64 rows per workgroup throughout: B4 507 + 1916, B8 257 + 987, B16 266 + 1029.)
// Fewer rows also mean more partial rows (12 bytes per row block, token and k): the blocks grow while those would take
// more than TS_PART_BYTES, which 64-row blocks may exceed.
constexpr int64_t TS_PART_BYTES = (int64_t)4 << 30;
static int ts_rows(int B, int T, int H, int K, int V, bool backward) {
  const int64_t cus = device_cu_count(), BH = (int64_t)B * H;
  auto rounds = [&](int rows) { return (BH * ((V + rows - 1) / rows) + cus - 1) / cus; };
  if (backward && 3 * rounds(64) < 2 * rounds(32)) return 64;
  int rows = rounds(16) < 2 * rounds(32) ? 16 : 32;
  if (backward)
    while (rows < 64 && BH * T * K * ((V + rows - 1) / rows) * 12 > TS_PART_BYTES) rows *= 2;
  return rows;
}

// The backward's plan.  split: the state gradient's recurrence in a launch of its own (G at every chunk's end into gst),
// the rest chunk by chunk in parallel, which pays while the whole chain's workgroups leave the chip waiting for it.
struct TsBwdPlan {
  bool split;
  int rows;                           // per workgroup (of the chunk kernel when split)
  int64_t items, wgs;                 // the chunk kernel's items when split; workgroups
  size_t gst_floats, scratch_floats;  // gst first, then the workgroups' group-start states
};
// Costs in hundredths of a token of a lone 16-row workgroup (0.87 us at K = 128), as measured at H4 K128 V256: the whole
// chain per token and round over the CUs 100 (16 rows; 135 for each pair of rounds), 125 (32) and 200 (64); split, the
// state gradient per token 25 (one round of 16 rows) or 35 a round of 32, and the chunk kernel per 32-token chunk and
// round 150 (16 rows, two workgroups a CU) or 205 (64 rows) times 32, and the second launch 1000.  The call, us, whole
// chain and split: B4 T1024 1229 and 939; B1 T4096 4381 and 2264; H1 V64 B1 T1500 1495 and 681; B8 T512 767 and 797; B16
// T512 1202 and 1408; H1 B120 T34 216 and 322 -- the rule takes the faster one in each.  gst is kept under TS_PART_BYTES.
static TsBwdPlan ts_bwd_plan(int B, int T, int H, int K, int V) {
  const int64_t cus = device_cu_count(), BH = (int64_t)B * H, NCH = (T + TS_CT - 1) / TS_CT;
  auto blocks = [&](int rows) { return (int64_t)((V + rows - 1) / rows); };
  auto rounds = [&](int64_t wgs, int64_t per_cu) { return (wgs + per_cu * cus - 1) / (per_cu * cus); };
  TsBwdPlan p{};
  p.rows = ts_rows(B, T, H, K, V, true);
  const int64_t r = rounds(BH * blocks(p.rows), 1);
  const int64_t whole = p.rows == 64 ? 200 * r : p.rows == 32 ? 125 * r : r == 1 ? 100 : 135 * ((r + 1) / 2);
  const int64_t c16 = 150 * rounds(BH * NCH * blocks(16), 2), c64 = 205 * rounds(BH * NCH * blocks(64), 1);
  const int64_t state = rounds(BH * blocks(16), 1) <= 1 ? 25 : 35 * rounds(BH * blocks(32), 1);
  const int64_t gst = BH * NCH * K * V;
  p.split = T * state + TS_CT * std::min(c16, c64) + 1000 < T * whole && gst * 4 <= TS_PART_BYTES;
  if (p.split) p.rows = c16 < c64 && BH * T * K * blocks(16) * 12 <= TS_PART_BYTES ? 16 : 64;
  p.items = BH * blocks(p.rows) * (p.split ? NCH : 1);
  // resident workgroups per CU: two of 16 rows (249 registers, 68 KB of LDS at K = 128), one of 64 (117 KB)
  p.wgs = p.split ? std::min<int64_t>(p.items, cus * (p.rows == 16 ? 2 : 1)) : p.items;
  p.gst_floats = p.split ? (size_t)((gst + 3) / 4 * 4) : 0;
  p.scratch_floats = p.gst_floats + (size_t)p.wgs * (TS_CT / TS_GS) * K * p.rows;
  return p;
}

int token_scan_row_blocks(int B, int T, int H, int K, int V) {
  const int rows = ts_bwd_plan(B, T, H, K, V).rows;
  return (V + rows - 1) / rows;
}
size_t token_scan_scratch_floats(int B, int T, int H, int K, int V) {
  return ts_bwd_plan(B, T, H, K, V).scratch_floats;
}

template <int K, typename SH>
static hipError_t token_scan_fwd_sh(const TokenScanArgs& a) {
  const int NB = (a.V + SH::ROWS - 1) / SH::ROWS, NCH = (a.T + TS_CT - 1) / TS_CT;
  auto go = [&](auto kern) {
    kern<<<dim3((unsigned)(a.B * a.H * NB)), SH::THREADS, 0, a.stream>>>(a.q, a.k, a.u, a.v, a.la, a.h0, a.y, a.r, a.st,
                                                                        a.hT, a.T, a.H, a.V, NCH, NB);
    return hipGetLastError();
  };
  return a.hT ? go(token_scan_fwd_kernel<K, SH, true>) : go(token_scan_fwd_kernel<K, SH, false>);
}

template <int K, typename SH>
static hipError_t token_scan_gstate_sh(const TokenScanArgs& a) {
  const int NB = (a.V + SH::ROWS - 1) / SH::ROWS, NCH = (a.T + TS_CT - 1) / TS_CT;
  token_scan_gstate_kernel<K, SH><<<dim3((unsigned)(a.B * a.H * NB)), SH::THREADS, 0, a.stream>>>(
      a.q, a.k, a.u, a.la, a.dy, a.dhT, a.dv, a.scratch, a.dh0, a.T, a.H, a.V, NCH, NB);
  return hipGetLastError();
}

template <int K, typename SH, bool SPLIT>
static hipError_t token_scan_bwd_sh(const TokenScanArgs& a, const TsBwdPlan& p) {
  const int NB = (a.V + SH::ROWS - 1) / SH::ROWS, NCH = (a.T + TS_CT - 1) / TS_CT;
  token_scan_bwd_kernel<K, SH, SPLIT><<<dim3((unsigned)p.wgs), SH::THREADS, 0, a.stream>>>(
      a.q, a.k, a.u, a.la, a.r, a.st, a.dy, a.dhT, a.dv, a.dq_part, a.du_part, a.dk_part, a.dla_part, a.dh0,
      a.scratch + p.gst_floats, a.scratch, (int)p.items, a.T, a.H, a.V, NCH, NB, (int64_t)a.B * a.T * a.H);
  return hipGetLastError();
}

template <int K>
static hipError_t token_scan_bwd_k(const TokenScanArgs& a, const TsBwdPlan& p) {
  if (p.split)
    return p.rows == 16 ? token_scan_bwd_sh<K, TsShape<1, 4>, true>(a, p) : token_scan_bwd_sh<K, TsShape<2, 8>, true>(a, p);
  switch (p.rows) {
    case 16: return token_scan_bwd_sh<K, TsShape<1, 4>, false>(a, p);
    case 32: return token_scan_bwd_sh<K, TsShape<1, 8>, false>(a, p);
    default: return token_scan_bwd_sh<K, TsShape<2, 8>, false>(a, p);
  }
}

template <int K>
static hipError_t token_scan_k(const TokenScanArgs& a, bool backward) {
  const bool narrow = ts_rows(a.B, a.T, a.H, K, a.V, false) == 16;  // one row per lane in 4 or 8 waves
  if (!backward)
    return narrow ? token_scan_fwd_sh<K, TsShape<1, 4>>(a) : token_scan_fwd_sh<K, TsShape<1, 8>>(a);
  const TsBwdPlan p = ts_bwd_plan(a.B, a.T, a.H, K, a.V);
  if (p.split) {
    const hipError_t e = narrow ? token_scan_gstate_sh<K, TsShape<1, 4>>(a) : token_scan_gstate_sh<K, TsShape<1, 8>>(a);
    if (e != hipSuccess) return e;
  }
  return token_scan_bwd_k<K>(a, p);
}

hipError_t launch_token_scan(const TokenScanArgs& a, bool backward) {
  switch (a.K) {
    case 64: return token_scan_k<64>(a, backward);
    case 128: return token_scan_k<128>(a, backward);
  }
  return hipErrorInvalidValue;
}

}  // namespace gdn
