// Scan across the segments of a segmented chunk sweep (sequence parallelism inside one GPU).
//
// The chunks of a sequence are cut into NS segments that are swept in parallel: a prefix pass gives, per segment s
// and head, the state the segment leaves from a zero entering state (loc_s, [K][V]; for the first segment from h0, so
// loc_0 = Phi_0 h0 + its local state) and the segment's transition Phi_s ([K][K], so that leaving = Phi_s entering +
// loc_s).  This kernel then carries the state across the segments in order, one small product per segment:
//     forward:  out_0 = h0,     S_1 = loc_0,            S_{s+1} = Phi_s S_s + loc_s (s >= 1),    out_s = S_s
// and the state gradient backwards, with the transposed transitions (dloc_{NS-1} likewise already carrying dhT):
//     reverse:  out_{NS-1} = dhT,  G_{NS-1} = dloc_{NS-1},  G_s = Phi_s^T G_{s+1} + dloc_s,      out_s = G_{s+1}
// (out_s: the state entering segment s, or the gradient w.r.t. the state leaving it).  All in fp32.  Phi of the first
// (forward) or last (reverse) segment is never read, and neither is the other end's: the main sweeps produce hT (from
// the last segment) and dh0 (from the first) themselves.
//
// One workgroup of K/16 waves per (b*h, 16-column block of V): wave w carries rows 16w .. 16w + 15 of the block as one
// fp32 MFMA accumulator.  What bounds it is the chain of NS products, so each step is short: the accumulator layout
// (lane (c, g) holds rows 4g + i of column c) is also the B operand of v_mfma_f32_16x16x4_f32 for the k slots
// 16j + 4g + i, so the waves pass their tiles through LDS as one 16-byte vector per lane (one LDS-only barrier a step,
// double-buffered), and Phi goes straight from global memory to the A operand in the same slot order (forward: 16-byte
// loads of its rows; reverse: its columns, 64-byte runs), loaded during the step before.  A step takes 2.4 us at
// K = 128 (its 64 products per SIMD; loads two steps ahead, or every head's blocks on one XCD, change nothing) and
// 0.8 us at K = 64.  At B1 T16384 H16 K128 V256 (256 workgroups, 4 segments): 13 us, against 20 us for fp32 FMAs on
// Phi staged in LDS.
#include <hip/hip_runtime.h>

#include "gdn_launch.h"

namespace gdn {

constexpr int SCAN_COLS = 16;
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int K, bool REVERSE>
__global__ __launch_bounds__(4 * K) void seg_scan_kernel(const float* __restrict__ phi, const float* __restrict__ loc,
                                                         const float* __restrict__ init, float* __restrict__ outs,
                                                         int NS, int H, int V) {
  constexpr int NW = K / 16;  // waves = row tiles
  __shared__ f32x4 sS[2][NW][64];
  const int ncb = V / SCAN_COLS;
  const int bh = blockIdx.x / ncb, cb = blockIdx.x - bh * ncb;
  const int b = bh / H, h = bh - b * H;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, m = l & 15, g = l >> 4;
  const int c = cb * SCAN_COLS + m;  // this lane's column of V; its rows of the carried block are row0 + i
  const int row0 = 16 * w + 4 * g;
  auto seg_of = [&](int step) { return (int64_t)(b * NS + (REVERSE ? NS - 1 - step : step)) * H + h; };
  // segment seg's Phi (or Phi^T) rows 16w + m, k slots 16j + 4g + e
  auto fetch_phi = [&](int64_t seg, f32x4 (&A)[NW]) {
    const float* p = phi + seg * K * K;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      if constexpr (!REVERSE) {
        A[j] = *reinterpret_cast<const f32x4*>(p + (16 * w + m) * K + 16 * j + 4 * g);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) A[j][e] = p[(16 * j + 4 * g + e) * K + 16 * w + m];
      }
    }
  };
  auto fetch_loc = [&](int64_t seg, f32x4& x) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = loc[(seg * K + row0 + i) * V + c];
  };
  f32x4 acc;
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = init ? init[((int64_t)bh * K + row0 + i) * V + c] : 0.f;
  f32x4 A[NW], lv;
  fetch_loc(seg_of(0), lv);
  for (int step = 0; step < NS - 1; ++step) {
    // the next product's operands, in flight during this step's (the last product reloads its own)
    f32x4 An[NW], ln;
    const int64_t sn = seg_of(step + 2 < NS ? step + 1 : NS - 2);
    if (NS > 2) fetch_phi(sn, An);
    fetch_loc(sn, ln);
    const int64_t seg = seg_of(step);
#pragma unroll
    for (int i = 0; i < 4; ++i) outs[(seg * K + row0 + i) * V + c] = acc[i];
    f32x4 nxt = lv;
    if (step > 0) {  // the first local state already carries init (uniform over the workgroup)
      sS[step & 1][w][l] = acc;
      // LDS-only barrier: __syncthreads() would also wait for the loads and stores in flight
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
      f32x4 s[NW], hi = {0.f, 0.f, 0.f, 0.f};  // two chains
#pragma unroll
      for (int j = 0; j < NW; ++j) s[j] = sS[step & 1][j][l];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < NW; j += 2) {
          nxt = __builtin_amdgcn_mfma_f32_16x16x4f32(A[j][e], s[j][e], nxt, 0, 0, 0);
          hi = __builtin_amdgcn_mfma_f32_16x16x4f32(A[j + 1][e], s[j + 1][e], hi, 0, 0, 0);
        }
      nxt += hi;
    }
#pragma unroll
    for (int j = 0; j < NW; ++j) A[j] = An[j];
    lv = ln;
    acc = nxt;
  }
  const int64_t seg = seg_of(NS - 1);  // nothing reads the state past the last segment
#pragma unroll
  for (int i = 0; i < 4; ++i) outs[(seg * K + row0 + i) * V + c] = acc[i];
}

hipError_t launch_seg_scan(const float* phi, const float* loc, const float* init, float* outs, int B, int NS, int H,
                           int K, int V, bool reverse, hipStream_t stream) {
  if (V % SCAN_COLS != 0) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((int64_t)B * H * (V / SCAN_COLS)));
  auto go = [&](auto kern) {
    kern<<<grid, 4 * K, 0, stream>>>(phi, loc, init, outs, NS, H, V);
    return hipGetLastError();
  };
  if (K == 64) return reverse ? go(seg_scan_kernel<64, true>) : go(seg_scan_kernel<64, false>);
  if (K == 128) return reverse ? go(seg_scan_kernel<128, true>) : go(seg_scan_kernel<128, false>);
  return hipErrorInvalidValue;
}

}  // namespace gdn
