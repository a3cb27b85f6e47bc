// The passes around the projections' gradient GEMMs that no GEMM makes by itself.
//   sum_parts_t: out [N, K] = sum over p of part_p [K, N], transposed -- a weight gradient whose products were taken
//     as x^T dy, split over the tokens, summed straight into its rows of the layer's gradient.
//   narrow_dx: out [M, C] = dx [M, C] + a [M, J] W [J, C] for a few columns J (the a and b projections' 2 H), dx and a
//     and W bf16, fp32 sums, out fp32 or bf16.  As a GEMM accumulating into dx this moves dx twice for J = 8 columns of
//     products, and the cast of dx to the layer's fp32 input follows in a pass of its own.
// Both are bound by HBM: a wave has 8 (narrow_dx) or 32 (sum_parts_t) 16- or 8-byte reads per lane in flight.
// Measured at B64 T1024 d512 H4 (M 65536, J 8): narrow_dx 37.5 us, 5.4 TB/s (the GEMM and the cast 40.5 + 30.8 us);
// sum_parts_t of 8 parts, N 2048, K 512, 12.1 us (the sum and the transposing copy 14.8 + 10.9 us).
#include <hip/hip_runtime.h>

#include "gdn_common.h"
#include "gdn_launch.h"

namespace gdn {

// grid: 64 x 64 tiles (n fastest); the tile's 16-byte pieces are summed over the parts in order, then turned in LDS
constexpr int ST_TILE = 64, ST_PARTS = 8;  // parts in flight
template <typename T>
__global__ __launch_bounds__(256) void sum_parts_t_kernel(const float* __restrict__ part, int nparts,
                                                          T* __restrict__ out, int N, int K) {
  __shared__ float tile[ST_TILE][ST_TILE + 1];
  const int nb = (N + ST_TILE - 1) / ST_TILE, n0 = (int)(blockIdx.x % nb) * ST_TILE, k0 = (int)(blockIdx.x / nb) * ST_TILE;
  const int r = threadIdx.x >> 4, c = 4 * (threadIdx.x & 15);
  const int64_t NK = (int64_t)N * K;
#pragma unroll
  for (int i = 0; i < ST_TILE / 16; ++i) {
    const int k = k0 + r + 16 * i;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    if (k < K && n0 + c < N) {
      const float* p = part + (int64_t)k * N + n0 + c;
      int j = 0;
      for (; j + ST_PARTS <= nparts; j += ST_PARTS) {
        f32x4 v[ST_PARTS];
#pragma unroll
        for (int u = 0; u < ST_PARTS; ++u) v[u] = *reinterpret_cast<const f32x4*>(p + (j + u) * NK);
#pragma unroll
        for (int u = 0; u < ST_PARTS; ++u) s += v[u];
      }
      for (; j < nparts; ++j) s += *reinterpret_cast<const f32x4*>(p + j * NK);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) tile[r + 16 * i][c + e] = s[e];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ST_TILE / 16; ++i) {
    const int n = n0 + r + 16 * i;
    if (n < N && k0 + c < K) {
      T* o = out + (int64_t)n * K + k0 + c;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = from_f<T>(tile[c + e][r + 16 * i]);
    }
  }
}

// A wave: 256 columns (4 per lane, W's rows for them in registers) of ND_ROWS rows.  A row's J values of a are uniform
// over the wave.
constexpr int ND_ROWS = 32, ND_UNROLL = 8;
template <typename OT, int JMAX>
__global__ __launch_bounds__(256) void narrow_dx_kernel(const bf16* __restrict__ dx, const bf16* __restrict__ a,
                                                        const bf16* __restrict__ w, OT* __restrict__ out, int64_t M,
                                                        int C, int J, int cblocks) {
  const int64_t item = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(wave_id());
  const int64_t m0 = item / cblocks * ND_ROWS;
  const int c = (int)(item % cblocks) * 256 + 4 * lane_id();
  if (m0 >= M) return;
  const bool on = c < C;
  const int cc = on ? c : 0;  // lanes past the columns compute on the first ones and store nothing
  float wk[JMAX][4];
#pragma unroll
  for (int j = 0; j < JMAX; ++j) {
    const bf16x4 t = *reinterpret_cast<const bf16x4*>(w + (int64_t)min(j, J - 1) * C + cc);
#pragma unroll
    for (int e = 0; e < 4; ++e) wk[j][e] = j < J ? static_cast<float>(t[e]) : 0.f;
  }
  const int rows = (int)min((int64_t)ND_ROWS, M - m0);
  for (int r0 = 0; r0 < rows; r0 += ND_UNROLL) {
    bf16x4 x[ND_UNROLL];
#pragma unroll
    for (int u = 0; u < ND_UNROLL; ++u)
      x[u] = *reinterpret_cast<const bf16x4*>(dx + (m0 + min(r0 + u, rows - 1)) * C + cc);
#pragma unroll
    for (int u = 0; u < ND_UNROLL; ++u) {
      const int64_t m = m0 + min(r0 + u, rows - 1);
      const uint32_t* ap = reinterpret_cast<const uint32_t*>(a + m * J);  // J even: pairs of bf16
      float s[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = static_cast<float>(x[u][e]);
#pragma unroll
      for (int j = 0; j < JMAX; j += 2)
        if (j < J) {
          const uint32_t p = ap[j / 2];
          const float a0 = __uint_as_float(p << 16), a1 = __uint_as_float(p & 0xffff0000u);
#pragma unroll
          for (int e = 0; e < 4; ++e) s[e] = fmaf(a1, wk[j + 1][e], fmaf(a0, wk[j][e], s[e]));
        }
      if (on && r0 + u < rows) {
        OT* o = out + m * C + c;
        if constexpr (sizeof(OT) == 4) *reinterpret_cast<f32x4*>(o) = f32x4{s[0], s[1], s[2], s[3]};
        else *reinterpret_cast<bf16x4*>(o) = bf16x4{static_cast<bf16>(s[0]), static_cast<bf16>(s[1]),
                                                    static_cast<bf16>(s[2]), static_cast<bf16>(s[3])};
      }
    }
  }
}

hipError_t launch_sum_parts_t(const float* part, int nparts, void* out, int N, int K, int dtype, hipStream_t st) {
  const dim3 grid((unsigned)(((N + ST_TILE - 1) / ST_TILE) * ((K + ST_TILE - 1) / ST_TILE)));
  if (dtype == DT_BF16) sum_parts_t_kernel<bf16><<<grid, 256, 0, st>>>(part, nparts, static_cast<bf16*>(out), N, K);
  else sum_parts_t_kernel<float><<<grid, 256, 0, st>>>(part, nparts, static_cast<float*>(out), N, K);
  return hipGetLastError();
}

template <typename OT>
static hipError_t narrow_dx_t(const bf16* dx, const bf16* a, const bf16* w, OT* out, int64_t M, int C, int J,
                              hipStream_t st) {
  const int cblocks = (C + 255) / 256;
  const dim3 grid((unsigned)(((M + ND_ROWS - 1) / ND_ROWS * cblocks + 3) / 4));
  if (J <= 8) narrow_dx_kernel<OT, 8><<<grid, 256, 0, st>>>(dx, a, w, out, M, C, J, cblocks);
  else if (J <= 16) narrow_dx_kernel<OT, 16><<<grid, 256, 0, st>>>(dx, a, w, out, M, C, J, cblocks);
  else narrow_dx_kernel<OT, 32><<<grid, 256, 0, st>>>(dx, a, w, out, M, C, J, cblocks);
  return hipGetLastError();
}

hipError_t launch_narrow_dx(const void* dx, const void* a, const void* w, void* out, int64_t M, int C, int J,
                            int out_dtype, hipStream_t st) {
  const bf16 *x = static_cast<const bf16*>(dx), *ab = static_cast<const bf16*>(a), *wb = static_cast<const bf16*>(w);
  return out_dtype == DT_BF16 ? narrow_dx_t(x, ab, wb, static_cast<bf16*>(out), M, C, J, st)
                              : narrow_dx_t(x, ab, wb, static_cast<float*>(out), M, C, J, st);
}

}  // namespace gdn
