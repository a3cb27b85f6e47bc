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
// loads of its rows; reverse: its columns, 64-byte runs), loaded during the step before into the other parity's registers (a
// copy between them, or a branch around the loads, made each step wait for its own loads).  A step takes about 1.6 us at
// K = 128 (its 64 products per SIMD) and 0.55 at K = 64; B1 T4096 H1 K128 V128 (11 segments) 29.1 -> 23.7 us, B1 T6007
// H8 K128 V256 (6) 17.6 -> 15.0.  At B1 T16384 H16 K128 V256 (256 workgroups, 4 segments): 13 us, against 20 us for fp32
// FMAs on Phi staged in LDS.
//   TREE: the order of a step's sum, for the calls in fp32.  Two chains of K / 8 products, the first begun from loc, round
// 64 terms at the size of the result: segments of four chunks (B1 T2048 and T4096, K 64) put o 0.8% and dg 2.6%
// further from 64 bits than sweeping the sequence whole.  Chains of two products, added pairwise and to loc last, put no
// output further (o 2.539e-7 both, 24 seeds) in the same time.  The calls in bf16 round their operands 10^4 times coarser and keep the chains.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gdn_launch.h"

namespace gdn {

constexpr int SCAN_COLS = 16;
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int K, bool REVERSE, bool TREE>
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
  auto put = [&](int64_t seg, const f32x4& x) {
#pragma unroll
    for (int i = 0; i < 4; ++i) outs[(seg * K + row0 + i) * V + c] = x[i];
  };
  f32x4 acc;
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = init ? init[((int64_t)bh * K + row0 + i) * V + c] : 0.f;
  f32x4 A[2][NW], lv[2];  // a step's operands and the next step's, by the parity of the step
  fetch_loc(seg_of(0), lv[0]);
  auto one = [&](auto P, int step) {
    constexpr int cur = decltype(P)::value;
    // the next product's operands, in flight during this step's (the last product reloads its own; with two segments
    // there is none, and what is loaded is not used): no branch and no copies, which every wait would include
    const int64_t sn = seg_of(step + 2 < NS ? step + 1 : NS - 2);
    fetch_phi(sn, A[cur ^ 1]);
    fetch_loc(sn, lv[cur ^ 1]);
    put(seg_of(step), acc);
    f32x4 nxt = lv[cur];
    if (step > 0) {  // the first local state already carries init (uniform over the workgroup)
      sS[cur][w][l] = acc;
      // LDS-only barrier: __syncthreads() would also wait for the loads and stores in flight
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
      f32x4 s[NW], zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NW; ++j) s[j] = sS[cur][j][l];
      auto mul = [&](int j, int e, const f32x4& c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(A[cur][j][e], s[j][e], c, 0, 0, 0);
      };
      if constexpr (TREE) {
        f32x4 t[2 * NW];
#pragma unroll
        for (int e = 0; e < 4; e += 2)
#pragma unroll
          for (int j = 0; j < NW; ++j) t[2 * j + e / 2] = mul(j, e, zero);
#pragma unroll
        for (int e = 0; e < 4; e += 2)
#pragma unroll
          for (int j = 0; j < NW; ++j) t[2 * j + e / 2] = mul(j, e + 1, t[2 * j + e / 2]);
#pragma unroll
        for (int n = NW; n >= 1; n /= 2)
#pragma unroll
          for (int j = 0; j < n; ++j) t[j] = t[2 * j] + t[2 * j + 1];
        nxt += t[0];
      } else {
        f32x4 hi = zero;  // two chains
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < NW; j += 2) {
            nxt = mul(j, e, nxt);
            hi = mul(j + 1, e, hi);
          }
        nxt += hi;
      }
    }
    acc = nxt;
  };
  for (int step = 0;;) {  // NS >= 2
    one(std::integral_constant<int, 0>{}, step);
    if (++step == NS - 1) break;
    one(std::integral_constant<int, 1>{}, step);
    if (++step == NS - 1) break;
  }
  put(seg_of(NS - 1), acc);  // nothing reads the state past the last segment
}

hipError_t launch_seg_scan(const float* phi, const float* loc, const float* init, float* outs, int B, int NS, int H,
                           int K, int V, int dtype, bool reverse, hipStream_t stream) {
  if (V % SCAN_COLS != 0 || NS < 2) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((int64_t)B * H * (V / SCAN_COLS)));
  auto go = [&](auto kern) {
    kern<<<grid, 4 * K, 0, stream>>>(phi, loc, init, outs, NS, H, V);
    return hipGetLastError();
  };
  if (dtype == DT_F32 && K == 64)  // the chunk ops in fp32 have no other K
    return reverse ? go(seg_scan_kernel<64, true, true>) : go(seg_scan_kernel<64, false, true>);
  if (K == 64) return reverse ? go(seg_scan_kernel<64, true, false>) : go(seg_scan_kernel<64, false, false>);
  if (K == 128) return reverse ? go(seg_scan_kernel<128, true, false>) : go(seg_scan_kernel<128, false, false>);
  return hipErrorInvalidValue;
}

}  // namespace gdn
