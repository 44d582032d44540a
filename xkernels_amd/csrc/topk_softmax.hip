// The MoE router step: softmax over the expert axis in fp32, top-k selection in
// descending probability with ties broken by ascending expert id, optional
// renormalisation of the selected weights (contract of the reference's
// src/xkernels/ops/moe/topk_softmax.py:33-95 and its Op Spec).
//
// Rows of up to 512 experts with k up to 16 take 16 lanes each in larger batches
// (topk_softmax_rows16 below). Otherwise one wave64 owns one row at a time. Lane
// l holds experts l, l+64, l+128, ...
// (every load instruction of the wave reads one contiguous run of logits), so a
// row of E experts sits in VPT = ceil(E/64) (rounded to a power of two)
// registers per lane. Max and sum are wave reductions; each of the k rounds
// takes the wave-wide largest (probability, -id) key below the previous
// round's winner with one xor-shuffle butterfly.
// Selections are staged in LDS so the renormalisation and the [M, k] output
// writes are contiguous across lanes.
//
// HBM bound: M*E logits in, M*k (weight, id) pairs out; no scratch. Rows of
// more than 2048 experts take a streaming variant (below).
#include <stdint.h>

#include "common.h"

namespace xk {
namespace {

constexpr int kTsWaves = 4;
constexpr int kTsThreads = kTsWaves * 64;

template <typename T>
__device__ __forceinline__ float logit_at(const T* p);
template <>
__device__ __forceinline__ float logit_at<uint16_t>(const uint16_t* p) {  // bf16 bits
  return __uint_as_float(uint32_t(*p) << 16);
}
template <>
__device__ __forceinline__ float logit_at<_Float16>(const _Float16* p) {
  return float(*p);
}
template <>
__device__ __forceinline__ float logit_at<float>(const float* p) {
  return *p;
}

// The reference's stable descending sort (torch.sort, topk_softmax.py:88)
// orders experts by probability, NaN above every number, and equal keys (NaN
// and NaN included) by lower id. One 64-bit key per expert encodes that order
// as an unsigned integer order: the high word is 0xFFFFFFFE for NaN and the
// probability's bit pattern + 1 otherwise (probabilities are +0 .. 1, whose
// bit patterns are ordered like the values; 0 is left for padding), the low
// word ~id (a lower id gives the larger key). Keys are unique and below ~0,
// the bound of the first selection, so selection t takes the largest key
// below selection t-1's. A row with a NaN or +inf logit, or only -inf
// logits, softmaxes to all NaN (as torch's does: the NaN or the inf - inf
// reaches the sum), so it selects experts 0 .. k-1 with NaN weights.
__device__ __forceinline__ uint64_t rank_key(float p, int e) {
  const uint32_t hi = __builtin_isnan(p) ? 0xFFFFFFFEu : __float_as_uint(p) + 1u;
  return (uint64_t(hi) << 32) | uint32_t(~e);
}
__device__ __forceinline__ float key_prob(uint64_t key) {
  const uint32_t hi = uint32_t(key >> 32);
  return hi == 0xFFFFFFFEu ? __builtin_nanf("") : __uint_as_float(hi - 1u);
}
__device__ __forceinline__ int key_id(uint64_t key) { return int(~uint32_t(key)); }

// Largest key of the wave.
__device__ __forceinline__ uint64_t wave_max_key(uint64_t b) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const uint32_t lo = __shfl_xor(uint32_t(b), off), hi = __shfl_xor(uint32_t(b >> 32), off);
    const uint64_t o = (uint64_t(hi) << 32) | lo;
    b = o > b ? o : b;
  }
  return b;
}

template <typename T, int VPT>
__global__ void __launch_bounds__(kTsThreads)
topk_softmax_rows(const T* __restrict__ logits, int64_t M, int E, int k, int renorm,
                  float* __restrict__ w_out, int32_t* __restrict__ id_out) {
  extern __shared__ __attribute__((aligned(16))) unsigned char ts_lds[];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  float* sel_w = reinterpret_cast<float*>(ts_lds) + wave * 2 * k;
  int32_t* sel_id = reinterpret_cast<int32_t*>(sel_w + k);

  for (int64_t row = int64_t(blockIdx.x) * kTsWaves + wave; row < M;
       row += int64_t(gridDim.x) * kTsWaves) {
    const T* g = logits + row * E;
    float p[VPT];
    float mx = -__builtin_inff();
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int e = j * 64 + lane;
      p[j] = e < E ? logit_at<T>(g + e) : -__builtin_inff();
      mx = fmaxf(mx, p[j]);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int e = j * 64 + lane;
      p[j] = e < E ? expf(p[j] - mx) : 0.f;
      sum += p[j];
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off);
    uint64_t key[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int e = j * 64 + lane;
      key[j] = e < E ? rank_key(p[j] / sum, e) : 0;  // padding ranks below every expert
    }

    float picked_sum = 0.f;
    uint64_t prev = ~uint64_t(0);
    for (int t = 0; t < k; ++t) {
      uint64_t best = 0;
#pragma unroll
      for (int j = 0; j < VPT; ++j) best = key[j] < prev && key[j] > best ? key[j] : best;
      // every lane now holds the same winner (k <= E: a real expert)
      prev = wave_max_key(best);
      const float bv = key_prob(prev);
      const int bid = key_id(prev);
      if (lane == 0) {
        sel_w[t] = bv;
        sel_id[t] = bid;
      }
      picked_sum += bv;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int t = lane; t < k; t += 64) {
      const float v = sel_w[t];
      w_out[row * k + t] = renorm ? v / picked_sum : v;
      id_out[row * k + t] = sel_id[t];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// Rows of up to 512 experts, k up to 16 (rows16_from): 16 lanes a row, four rows a wave. The
// selection rounds are VALU work (six instructions per key and round, the
// cross-lane steps beside), and a row's 16 lanes reduce with four DPP moves in
// place of six LDS permutes: the four rows of a wave cost about what one row
// over 64 lanes does. Lane i holds the 8-expert pieces i, i + 16, ...; lane t
// keeps selection t. 4,096 rows, E = 256, k = 8, bf16: 10.3 -> 7.2 us; 16,384 rows 24 -> 12 us per call.
template <int CTRL> __device__ __forceinline__ uint32_t dpp(uint32_t x) {
  return __builtin_amdgcn_update_dpp(x, x, CTRL, 0xF, 0xF, false);
}
// f over the partners of an all-reduce of 16 lanes: neighbours, pairs, the
// mirrored half row, the mirrored row.
template <typename F> __device__ __forceinline__ void row_steps(F&& f) {
  f([](uint32_t x) { return dpp<0xB1>(x); });
  f([](uint32_t x) { return dpp<0x4E>(x); });
  f([](uint32_t x) { return dpp<0x141>(x); });
  f([](uint32_t x) { return dpp<0x140>(x); });
}

template <typename T> struct piece8 {};  // 8 logits in 16-byte loads
template <> struct piece8<uint16_t> {
  __device__ __forceinline__ static void load(const uint16_t* g, float* v) {
    const u32x4 r = *reinterpret_cast<const u32x4*>(g);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(r[i] << 16);
      v[2 * i + 1] = __uint_as_float(r[i] & 0xFFFF0000u);
    }
  }
};
template <> struct piece8<_Float16> {
  __device__ __forceinline__ static void load(const _Float16* g, float* v) {
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    const h8 r = *reinterpret_cast<const h8*>(g);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = static_cast<float>(r[i]);
  }
};
template <> struct piece8<float> {
  __device__ __forceinline__ static void load(const float* g, float* v) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 r = reinterpret_cast<const f32x4*>(g)[h];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[4 * h + i] = r[i];
    }
  }
};

// WIDE: E a multiple of 8 and every row 16-byte aligned.
template <typename T, int PIECES, bool WIDE>
__global__ void __launch_bounds__(kTsThreads)
topk_softmax_rows16(const T* __restrict__ logits, int64_t M, int E, int k, int renorm,
                    float* __restrict__ w_out, int32_t* __restrict__ id_out) {
  constexpr int N = PIECES * 8;
  const int i16 = threadIdx.x & 15;
  const int64_t row = int64_t(blockIdx.x) * (kTsThreads / 16) + (threadIdx.x >> 4);
  if (row >= M) return;  // whole 16-lane rows
  const T* g = logits + row * E;
  float p[N];
  float mx = -__builtin_inff();
#pragma unroll
  for (int c = 0; c < PIECES; ++c) {
    const int e0 = (c * 16 + i16) * 8;
    if (WIDE) {
      if (e0 < E) {
        piece8<T>::load(g + e0, p + 8 * c);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) p[8 * c + i] = -__builtin_inff();
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) p[8 * c + i] = e0 + i < E ? logit_at<T>(g + e0 + i) : -__builtin_inff();
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) mx = fmaxf(mx, p[8 * c + i]);
  }
  row_steps([&](auto from) { mx = fmaxf(mx, __uint_as_float(from(__float_as_uint(mx)))); });
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int e = ((j >> 3) * 16 + i16) * 8 + (j & 7);
    p[j] = e < E ? expf(p[j] - mx) : 0.f;
    sum += p[j];
  }
  row_steps([&](auto from) { sum += __uint_as_float(from(__float_as_uint(sum))); });
  uint64_t key[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int e = ((j >> 3) * 16 + i16) * 8 + (j & 7);
    key[j] = e < E ? rank_key(p[j] / sum, e) : 0;  // padding ranks below every expert
  }
  float picked_sum = 0.f, my_w = 0.f;
  int my_id = 0;
  uint64_t prev = ~uint64_t(0);
  for (int t = 0; t < k; ++t) {
    uint64_t best = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) best = key[j] < prev && key[j] > best ? key[j] : best;
    row_steps([&](auto from) {
      const uint64_t o = (uint64_t(from(uint32_t(best >> 32))) << 32) | from(uint32_t(best));
      best = o > best ? o : best;
    });
    prev = best;
    const float bv = key_prob(prev);
    if (i16 == t) {
      my_w = bv;
      my_id = key_id(prev);
    }
    picked_sum += bv;
  }
  if (i16 < k) {
    w_out[row * k + i16] = renorm ? my_w / picked_sum : my_w;
    id_out[row * k + i16] = my_id;
  }
}

// Rows of more than 32 * 64 experts: the same selection without holding the
// row in registers. Round t re-reads the row (from L2) and takes the largest
// key below round t-1's winner (the same keys as above): k * E reads and
// exponentials per row. The lane t % 64 writes the t-th selection; the
// renormalisation then rescales each lane's own writes.
template <typename T>
__global__ void __launch_bounds__(kTsThreads)
topk_softmax_rows_stream(const T* __restrict__ logits, int64_t M, int E, int k, int renorm,
                         float* __restrict__ w_out, int32_t* __restrict__ id_out) {
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  for (int64_t row = int64_t(blockIdx.x) * kTsWaves + wave; row < M;
       row += int64_t(gridDim.x) * kTsWaves) {
    const T* g = logits + row * E;
    float mx = -__builtin_inff();
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, logit_at<T>(g + e));
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    float sum = 0.f;
    for (int e = lane; e < E; e += 64) sum += expf(logit_at<T>(g + e) - mx);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off);
    float picked_sum = 0.f;
    uint64_t prev = ~uint64_t(0);
    for (int t = 0; t < k; ++t) {
      uint64_t best = 0;
      for (int e = lane; e < E; e += 64) {
        const uint64_t v = rank_key(expf(logit_at<T>(g + e) - mx) / sum, e);
        best = v < prev && v > best ? v : best;
      }
      prev = wave_max_key(best);
      const float bv = key_prob(prev);
      const int bid = key_id(prev);
      if (lane == (t & 63)) {
        w_out[row * k + t] = bv;
        id_out[row * k + t] = bid;
      }
      picked_sum += bv;
    }
    if (renorm)
      for (int t = lane; t < k; t += 64) w_out[row * k + t] = w_out[row * k + t] / picked_sum;
  }
}

template <typename T, int VPT>
hipError_t launch_vpt(const void* logits, int64_t M, int E, int k, int renorm, float* w,
                      int32_t* ids, hipStream_t stream) {
  const int64_t blocks = (M + kTsWaves - 1) / kTsWaves;
  const int grid = int(blocks < 65536 ? blocks : 65536);
  const size_t lds = size_t(kTsWaves) * 2 * k * sizeof(float);
  hipLaunchKernelGGL((topk_softmax_rows<T, VPT>), dim3(grid), dim3(kTsThreads), lds, stream,
                     static_cast<const T*>(logits), M, E, k, renorm, w, ids);
  return hipGetLastError();
}

template <typename T, int PIECES>
hipError_t launch_rows16(const void* logits, int64_t M, int E, int k, int renorm, float* w, int32_t* ids,
                         hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(cdiv(M, kTsThreads / 16)));
  const T* g = static_cast<const T*>(logits);
  if (E % 8 == 0 && reinterpret_cast<uintptr_t>(g) % 16 == 0)
    hipLaunchKernelGGL((topk_softmax_rows16<T, PIECES, true>), grid, dim3(kTsThreads), 0, stream, g, M, E, k, renorm,
                       w, ids);
  else
    hipLaunchKernelGGL((topk_softmax_rows16<T, PIECES, false>), grid, dim3(kTsThreads), 0, stream, g, M, E, k, renorm,
                       w, ids);
  return hipGetLastError();
}

// Rows from which 16 lanes a row are faster than 64. A row's selection is four
// times as long on 16 lanes, which only batches that fill the chip hide, and
// beyond 128 experts it no longer pays for itself in cheaper cross-lane steps.
// Kernel times in us, 64 vs 16 lanes, bf16 (fp32 lies within 0.5 us):
//   E = 128: k = 1: 3.1 vs 3.0 at 1,024 rows; k = 8: 4.6 vs 4.2 at 1, 5.5 vs 4.5
//     at 1,024; E = 16, k = 1: 3.0 vs 3.1 at 1,024, 3.1 vs 3.1 at 1,500;
//   E = 256: k = 1: 3.7 vs 3.8 at 2,048, 4.0 vs 3.9 at 3,000; k = 2: 3.9 vs 4.1 at
//     1,024, 4.2 vs 4.2 at 2,048; k = 8: 5.3 vs 6.0 at 1, 6.3 vs 6.1 at 1,024, 9.4
//     vs 6.3 at 4,096; k = 16: 8.0 vs 9.1 at 1, 9.2 vs 8.7 at 64;
//   E = 384: k = 1: 5.2 vs 5.3 at 4,096, 12.3 vs 10.5 at 16,384; k = 8: 7.5 vs 9.3
//     at 1,024, 9.4 vs 9.3 at 3,000, 10.8 vs 9.5 at 4,096; k = 16: 9.6 vs 14.8 at
//     1, 12.7 vs 14.0 at 2,048, 14.9 vs 14.1 at 3,000.
}  // namespace
int64_t rows16_from(int E, int k) {
  if (E <= 128) return k < 4 ? 1500 : 0;
  if (E <= 256) return k < 2 ? 3000 : k < 4 ? 2048 : k < 8 ? 1300 : k == 8 ? 1024 : 16;
  return k < 4 ? 6000 : k < 8 ? 4096 : 3200;
}
namespace {

template <typename T>
hipError_t launch_typed(const void* logits, int64_t M, int E, int k, int renorm, float* w,
                        int32_t* ids, hipStream_t stream) {
  // a launch takes fewer than 2^32 threads (16 a row here; the kernels below
  // loop over the rows)
  if (k <= 16 && E <= 512 && M >= rows16_from(E, k) &&
      cdiv(M, kTsThreads / 16) * kTsThreads < (int64_t(1) << 32)) {
    if (E <= 128) return launch_rows16<T, 1>(logits, M, E, k, renorm, w, ids, stream);
    if (E <= 256) return launch_rows16<T, 2>(logits, M, E, k, renorm, w, ids, stream);
    return launch_rows16<T, 4>(logits, M, E, k, renorm, w, ids, stream);
  }
  const int per_lane = (E + 63) / 64;
  if (per_lane <= 1) return launch_vpt<T, 1>(logits, M, E, k, renorm, w, ids, stream);
  if (per_lane <= 2) return launch_vpt<T, 2>(logits, M, E, k, renorm, w, ids, stream);
  if (per_lane <= 4) return launch_vpt<T, 4>(logits, M, E, k, renorm, w, ids, stream);
  if (per_lane <= 8) return launch_vpt<T, 8>(logits, M, E, k, renorm, w, ids, stream);
  if (per_lane <= 16) return launch_vpt<T, 16>(logits, M, E, k, renorm, w, ids, stream);
  if (per_lane <= 32) return launch_vpt<T, 32>(logits, M, E, k, renorm, w, ids, stream);
  const int64_t blocks = (M + kTsWaves - 1) / kTsWaves;
  hipLaunchKernelGGL((topk_softmax_rows_stream<T>), dim3(int(blocks < 65536 ? blocks : 65536)),
                     dim3(kTsThreads), 0, stream, static_cast<const T*>(logits), M, E, k, renorm,
                     w, ids);
  return hipGetLastError();
}

}  // namespace

// Rows beyond 32 * 64 experts take the streaming kernel; ids and indices stay
// 32-bit.
int topk_softmax_max_experts() { return 1 << 30; }

int launch_topk_softmax(const void* logits, int dtype, int64_t M, int64_t E, int64_t k,
                        int renorm, float* w, int32_t* ids, hipStream_t stream) {
  hipError_t e;
  switch (dtype) {
    case XK_DT_BF16:
      e = launch_typed<uint16_t>(logits, M, int(E), int(k), renorm, w, ids, stream);
      break;
    case XK_DT_FP32:
      e = launch_typed<float>(logits, M, int(E), int(k), renorm, w, ids, stream);
      break;
    default:
      e = launch_typed<_Float16>(logits, M, int(E), int(k), renorm, w, ids, stream);
      break;
  }
  if (e != hipSuccess) return set_error(XK_ERR_LAUNCH, "topk_softmax launch: %s", hipGetErrorString(e));
  return XK_OK;
}

}  // namespace xk
