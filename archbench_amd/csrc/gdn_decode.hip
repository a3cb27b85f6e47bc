// The input projections of one decoded token per sequence (fla's GatedDeltaNet q, k, v, gate, a and b linears at T = 1,
// archbench/layers/fla.py:36-38): y_i [M, rows_i] = x [M, d] W_i^T for up to six weights read where they lie, M <= 128
// tokens, bf16 activations, bf16 or fp32 weights (rounded to bf16 as the layer's cast does), fp32 sums.
// Bound: the weights' bytes (M is far below the 280 tokens at which they would take the matrix cores longer than HBM).
// Concatenating the weights for one GEMM reads them, writes them and reads them again.  d 1024 with 8 heads: 8 tokens
// 7.2 us, 64 tokens 14.2 us, 128 tokens 22.6 us; the concatenation and three GEMMs 28.9 us at 8 and 36.7 us at 128 tokens (past which
// they take over: two passes over the weights are then three).
// One workgroup per 16 weight rows, its four waves taking every fourth 32-wide step of d, so that all of a row block's
// loads are in flight at once (386 row blocks at d 1024 with 8 heads: one or two workgroups per CU, 8 KB in flight per
// wave); the four partial sums are added through LDS.  W rows are the A operand, tokens the B operand, so a lane ends
// with four consecutive outputs of one token.
#include <hip/hip_runtime.h>

#include "gdn_common.h"
#include "gdn_launch.h"

namespace gdn {

constexpr int DP_WAVES = 4, DP_UNROLL = 8;  // steps of a wave in flight

struct DecodeProjTable {
  const void* w[DECODE_MAX_WEIGHTS];
  bf16* y[DECODE_MAX_WEIGHTS];
  int rows[DECODE_MAX_WEIGHTS], ld[DECODE_MAX_WEIGHTS], tile0[DECODE_MAX_WEIGHTS];  // tile0: first row block
};

template <typename WT>
__device__ __forceinline__ bf16x8 dp_load(const WT* p) {
  if constexpr (sizeof(WT) == 2) {
    return *reinterpret_cast<const bf16x8*>(p);
  } else {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
    bf16x8 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = static_cast<bf16>(a[i]), r[4 + i] = static_cast<bf16>(b[i]);
    return r;
  }
}

// grid: row blocks x token blocks of 16 MT.  Tokens past M and rows past the weight's last repeat the last one and are not stored.
template <typename WT, int MT>
__global__ __launch_bounds__(64 * DP_WAVES) void decode_proj_kernel(const bf16* __restrict__ x, DecodeProjTable t,
                                                                    int nw, int M, int d) {
  __shared__ f32x4 red[DP_WAVES][MT][64];
  const int l = lane_id(), wv = __builtin_amdgcn_readfirstlane(wave_id()), tile = blockIdx.x;
  const int m0 = 16 * MT * blockIdx.y;
  int gi = 0;
  for (int i = 1; i < nw; ++i) gi = tile >= t.tile0[i] ? i : gi;
  const int rows = t.rows[gi], ld = t.ld[gi], n0 = 16 * (tile - t.tile0[gi]), kp = 8 * (l >> 4);
  const WT* wp = static_cast<const WT*>(t.w[gi]) + (int64_t)min(n0 + (l & 15), rows - 1) * d + kp;
  const bf16* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) xp[m] = x + (int64_t)min(m0 + 16 * m + (l & 15), M - 1) * d + kp;
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = d / 32;
  for (int s0 = wv; s0 < steps; s0 += DP_WAVES * DP_UNROLL) {
    bf16x8 a[DP_UNROLL];
#pragma unroll
    for (int u = 0; u < DP_UNROLL; ++u) {
      const int s = s0 + DP_WAVES * u;
      if (s < steps) a[u] = dp_load(wp + 32 * s);
    }
#pragma unroll
    for (int u = 0; u < DP_UNROLL; ++u) {
      const int s = s0 + DP_WAVES * u;
      if (s < steps) {
#pragma unroll
        for (int m = 0; m < MT; ++m) mma(acc[m], a[u], *reinterpret_cast<const bf16x8*>(xp[m] + 32 * s));
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) red[wv][m][l] = acc[m];
  __syncthreads();
  for (int e = threadIdx.x; e < MT * 64; e += 64 * DP_WAVES) {
    const int m = e >> 6, le = e & 63, tok = m0 + 16 * m + (le & 15), r = n0 + 4 * (le >> 4);
    const f32x4 s = (red[0][m][le] + red[1][m][le]) + (red[2][m][le] + red[3][m][le]);
    if (tok < M) {
      bf16* o = t.y[gi] + (int64_t)tok * ld + r;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (r + i < rows) o[i] = static_cast<bf16>(s[i]);
    }
  }
}

bool decode_proj_supported(int M, int d) { return M >= 1 && M <= DECODE_MAX_TOKENS && d >= 32 && d % 32 == 0; }

template <typename WT>
static hipError_t decode_proj_t(const DecodeProjArgs& a) {
  DecodeProjTable t{};
  int tiles = 0;
  for (int i = 0; i < a.n; ++i) {
    t.w[i] = a.w[i], t.y[i] = static_cast<bf16*>(a.y[i]), t.rows[i] = a.rows[i], t.ld[i] = a.ld[i], t.tile0[i] = tiles;
    tiles += (a.rows[i] + 15) / 16;
  }
  const bf16* x = static_cast<const bf16*>(a.x);
  if (a.M <= 16) decode_proj_kernel<WT, 1><<<tiles, 64 * DP_WAVES, 0, a.stream>>>(x, t, a.n, a.M, a.d);
  else if (a.M <= 32) decode_proj_kernel<WT, 2><<<tiles, 64 * DP_WAVES, 0, a.stream>>>(x, t, a.n, a.M, a.d);
  else decode_proj_kernel<WT, 4><<<dim3(tiles, (a.M + 63) / 64), 64 * DP_WAVES, 0, a.stream>>>(x, t, a.n, a.M, a.d);
  return hipGetLastError();
}

hipError_t launch_decode_proj(const DecodeProjArgs& a) {
  return a.w_dtype == DT_BF16 ? decode_proj_t<bf16>(a) : decode_proj_t<float>(a);
}

}  // namespace gdn
