// MXFP4 MoE kernels for gfx950 (the reference's _mxfp4_moe_gemm_kernel,
// src/xkernels/ops/moe/triton/moe_mxfp4_kernel.py:87-352; math of the oracle
// mxfp4_reference.py:28-112 with the dequant of ops/gather/mxfp4.py:39-68).
//
//   stage 0 : gu = bf16(A[m]) @ w13[e]^T (+ b13[e]),  act[t, j] =
//             bf16(silu(min(g, L)) * clamp(u, -L, L)),  g = gu[j], u = gu[ispp + j]
//   stage 1 : row[t, n] = bf16(bf16(act[t] @ w2[e]^T) (+ b2[e, n]))
// followed by the weighted top-k combine (reduce.hip). The bf16 roundings sit
// where the reference's bf16 torch ops round (matmul output, bias add, act).
//
// Decode batches (bf16 activations, hidden and ispp multiples of 64, E <= 512,
// few routed rows per expert): both projections run mxfp4_stream_rs
// (int4_stream.hip) into fp32 partial planes; mxfp4_swiglu_planes below finishes
// stage 0 and the combine applies stage 1's roundings and bias. Every other
// batch runs the tile kernels (tile_gemm.hip), which finish both stages in
// their epilogues; fp32 activations are rounded to bf16 first.
#include <algorithm>
#include <type_traits>

#include "int4_common.h"

namespace xk {
namespace {

// Gate/up epilogue for the stream path: the projection's S fp32 partial planes
// [S, numel, 2 ispp] are summed and finished: gu = bf16(sum) (+ b13 -> bf16), g clamped from above, u on
// both sides, act = bf16(silu(g) * u). Four columns per thread; slots whose
// expert is not local (never computed) are skipped.
__global__ void __launch_bounds__(256)
mxfp4_swiglu_planes(const float* __restrict__ planes, int S, int64_t numel, int ispp,
                    const uint16_t* __restrict__ b13, const int32_t* __restrict__ topk_ids,
                    const int32_t* __restrict__ emap, int num_global, int num_local, float limit,
                    uint16_t* __restrict__ act) {
  const int64_t per_row = ispp / 4;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= numel * per_row) return;
  const int64_t t = idx / per_row;
  const int j0 = static_cast<int>(idx - t * per_row) * 4;
  const int e = map_expert(topk_ids[t], emap, num_global, num_local);
  if (e < 0) return;
  const int64_t pstride = numel * 2 * ispp;
  const float* row = planes + t * 2 * ispp;
  // the planes in groups of four loads in flight (a decode batch of one token
  // has 16 K slices: 9.5 -> 6.8 us; groups of eight measured 12.2 us)
  f32x4 g = *reinterpret_cast<const f32x4*>(row + j0);
  f32x4 u = *reinterpret_cast<const f32x4*>(row + ispp + j0);
  int sl = 1;
  for (; sl + 3 < S; sl += 4) {
    f32x4 gs[4], us[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      gs[i] = *reinterpret_cast<const f32x4*>(row + (sl + i) * pstride + j0);
      us[i] = *reinterpret_cast<const f32x4*>(row + (sl + i) * pstride + ispp + j0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      g += gs[i];
      u += us[i];
    }
  }
  for (; sl < S; ++sl) {
    g += *reinterpret_cast<const f32x4*>(row + sl * pstride + j0);
    u += *reinterpret_cast<const f32x4*>(row + sl * pstride + ispp + j0);
  }
  uint16_t r[4];
  const uint16_t* b = b13 ? b13 + static_cast<int64_t>(e) * 2 * ispp : nullptr;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = mxfp4_swiglu(g[i], u[i], b, j0 + i, ispp, limit);
  uint2 o;
  o.x = r[0] | (static_cast<uint32_t>(r[1]) << 16);
  o.y = r[2] | (static_cast<uint32_t>(r[3]) << 16);
  *reinterpret_cast<uint2*>(act + t * ispp + j0) = o;
}

// fp32 activations -> bf16 (the reference's bf16(A)), 8 per thread; n % 8 == 0.
__global__ void __launch_bounds__(256)
activations_to_bf16(const float* __restrict__ a, int64_t n, uint16_t* __restrict__ out) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
  if (i >= n) return;
  const f32x4 x = *reinterpret_cast<const f32x4*>(a + i), y = *reinterpret_cast<const f32x4*>(a + i + 4);
  u32x4 r;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    r[k] = f32_to_bf16(x[2 * k]) | (static_cast<uint32_t>(f32_to_bf16(x[2 * k + 1])) << 16);
    r[2 + k] = f32_to_bf16(y[2 * k]) | (static_cast<uint32_t>(f32_to_bf16(y[2 * k + 1])) << 16);
  }
  *reinterpret_cast<u32x4*>(out + i) = r;
}

}  // namespace

int mxfp4_block_size() { return 16; }

int launch_activations_to_bf16(const float* a, int64_t n, uint16_t* out, hipStream_t stream) {
  XK_REQUIRE(reinterpret_cast<uintptr_t>(a) % 16 == 0, "mxfp4: activations must be 16-byte aligned");
  hipLaunchKernelGGL(activations_to_bf16, dim3(static_cast<unsigned>(cdiv(n, 2048))), dim3(256), 0, stream, a,
                     n, out);
  XK_CHECK_LAUNCH("activations_to_bf16");
  return XK_OK;
}

int launch_mxfp4_swiglu(const float* planes, int S, int64_t numel, int64_t ispp, const uint16_t* b13,
                        const int32_t* topk_ids, const int32_t* emap, int num_global, int num_local,
                        float limit, uint16_t* act, hipStream_t stream) {
  XK_REQUIRE(ispp % 4 == 0, "mxfp4 swiglu: ispp %lld not a multiple of 4", (long long)ispp);
  const int64_t n = numel * (ispp / 4);
  if (n == 0) return XK_OK;
  hipLaunchKernelGGL(mxfp4_swiglu_planes, dim3(static_cast<unsigned>(cdiv(n, 256))), dim3(256), 0,
                     stream, planes, S, numel, int(ispp), b13, topk_ids, emap, num_global, num_local,
                     limit, act);
  XK_CHECK_LAUNCH("mxfp4_swiglu_planes");
  return XK_OK;
}

}  // namespace xk
