// Grouped INT4 W4A16 MoE GEMM for gfx950: kernel choice and launch (the
// reference's _fused_moe_int4_kernel launch, src/xkernels/ops/moe/triton/
// moe_int4_kernel.py:291-415; math of the oracle reference.py:22-70 with the
// dequant of w4a16.py:21-50).
//
// For every routed slot t (token m = t / top_k, local expert e) the kernels
// write the un-weighted fp32 row   slot_out[t, n] = sum_k A[m, k] * W[e, n, k]
// with W[e, n, k] = bf16((nibble(e, n, k) - 8) * scale[e, n, k / 32]) for bf16
// activations (the reference rounds the dequantised weight to A's dtype). The
// weighted top-k combine runs afterwards (reduce.hip). Kernels:
//   * int4_stream_rne (int4_stream.hip): decode regime, bf16 A, group 32 —
//     weight streaming with the exact bf16 dequant, K-slice partial planes;
//   * moe_tile (tile_gemm.hip) and int4_prefill_gemm (int4_prefill.hip): prefill
//     regime (>= 17 routed rows per expert on average), MFMA tiles of 128 and
//     256 rows, the same exact dequant;
//   * int4_simple_gemm (below): any dtype, group size or shape the MFMA
//     kernels do not take — one thread per (slot, column), exact dequant
//     rounded to A's dtype like the reference.
#include <algorithm>
#include <type_traits>

#include "int4_common.h"
#include "int4_flags.h"

namespace xk {
namespace {

// One thread per (slot, column); exact dequant rounded to A's dtype.
template <typename TA>
__global__ void __launch_bounds__(256)
int4_simple_gemm(const TA* __restrict__ A, int K, const uint32_t* __restrict__ packed,
                 const uint16_t* __restrict__ scale, int N, int group_size,
                 const int32_t* __restrict__ ids, const int32_t* __restrict__ emap,
                 int num_global, int num_local, int numel, int top_k,
                 float* __restrict__ out) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= static_cast<int64_t>(numel) * N) return;
  const int t = static_cast<int>(idx / N), n = static_cast<int>(idx - static_cast<int64_t>(t) * N);
  const int e = map_expert(ids[t], emap, num_global, num_local);
  if (e < 0) return;
  const int m = t / top_k;
  const int G = K / group_size;
  const uint32_t* wr = packed + (static_cast<int64_t>(e) * N + n) * (K >> 3);
  const uint16_t* sr = scale + (static_cast<int64_t>(e) * N + n) * G;
  const TA* ar = A + static_cast<int64_t>(m) * K;
  float acc = 0.f;
  for (int kw = 0; kw < (K >> 3); ++kw) {
    const uint32_t w = wr[kw];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = kw * 8 + j;
      const float s = bf16_to_f32(sr[k / group_size]);
      float v = static_cast<float>(static_cast<int>((w >> (4 * j)) & 0xFu) - 8) * s;
      if (sizeof(TA) == 2) v = round_bf16(v);
      acc = fmaf(io<TA>::load(ar + k), v, acc);
    }
  }
  out[static_cast<int64_t>(t) * N + n] = acc;
}

}  // namespace

// Number of compute units of the current device (cached per device).
int device_cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

// Token-slot block size the MFMA kernels consume (one MFMA row tile).
int int4_block_size() { return 16; }

bool int4_rs_group_ok(int64_t K, int group_size);

// The MFMA kernels take quantisation groups of 32, 64 or 128 and K a multiple
// of 32; bf16 or fp32 activations (fp32: the weight-streaming kernel only).
bool int4_use_stream(int a_dtype, int group_size, int64_t K) {
  return (a_dtype == XK_DT_BF16 || a_dtype == XK_DT_FP32) && K % 32 == 0 &&
         int4_rs_group_ok(K, group_size);
}

bool int4_prefill_ok(int a_dtype, int group_size, int64_t M, int64_t K, int64_t N, int64_t E);
bool int4_rs_ok(int64_t M, int64_t top_k, int64_t K, int64_t N, int64_t E, bool f32a,
                int group_size);
int int4_rs_slices(int64_t K, int64_t N, int64_t numel, int64_t E, bool f32a);
bool int4_rs_self_route_ok(int64_t numel);
int launch_int4_rs(const void* A, bool f32a, int64_t M, int64_t K, const int32_t* packed,
                   const uint16_t* scale, int64_t E, int64_t N, int64_t numel, int64_t top_k,
                   int group_size, const int32_t* sorted_ids, const int32_t* offsets,
                   const int32_t* topk_ids, const int32_t* emap, int num_global, float* slot_out,
                   hipStream_t stream);
bool int4_tile_ok(int a_dtype, int group_size, int64_t M, int64_t K, int64_t N, int64_t E);
int launch_int4_tile(const void* A, int64_t K, const int32_t* packed, const uint16_t* scale,
                     int64_t E, int64_t N, int64_t numel, int64_t top_k, int group_size,
                     const int32_t* sorted_ids, const int32_t* offsets, float* slot_out,
                     int* queue, int queue_stride, bool queue_cleared, hipStream_t stream);
int launch_int4_prefill(const void* A, int64_t K, const int32_t* packed, const uint16_t* scale,
                        int64_t E, int64_t N, int64_t numel, int64_t top_k, int group_size,
                        const int32_t* sorted_ids, const int32_t* offsets, float* slot_out,
                        int* queue, int queue_stride, bool queue_cleared, hipStream_t stream);

// Routed rows per expert (on average) from which the tile kernels replace the
// weight-streaming kernel, which streams every expert's weights once per
// 16-row pass. Measured per fused call, stream vs tile (moe_tile), uniform
// routing: E = 48, N = 4096, K = 7168, top_k = 8: 170 vs 201 us at 12 rows per
// expert, 248 vs 205 at 17, 321 vs 215 at 24, 559 vs 249 at 48. One line for all
// shapes, drawn at this one: N = 7168, K = 2048 crosses at 20 rows (124 vs 136 at
// 17, 162 vs 144 at 24), and few experts later (E = 16, N = K = 4096: 53 vs 54 at
// 17; N = 2048, K = 4096: 42 vs 49 at 24, 49 vs 50 at 32).
constexpr int64_t kPrefillRowsPerExpert = 17;
// K or N not a multiple of 256: the tile pads both, the stream kernel little. It
// runs from 40 rows per expert on where the stream kernel's work (local slots x N
// x K at about 100 million products a us) takes longer than a few rounds of tiles:
// about 15 us and K / 80 us a round of the 512 places. Per fused call, stream vs
// tile: E = 48, N = K = 2880: 146 vs 159 us at 40 rows; E = 64, N = K = 1440: 87
// vs 62 at 50; E = 16, N = 720, K = 544: 134 vs 56 at 1,200; E = 8, N = K = 2880:
// 50 vs 53 at 70; E = 1, N = 1440, K = 2880: 54 vs 64 at 1,200.
constexpr int64_t kPaddedTileRowsPerExpert = 40;
bool int4_padded_tile(int64_t rows, int64_t E, int64_t N, int64_t K) {
  const int64_t tiles = E * cdiv(N, 256) * cdiv(cdiv(rows, E), 128);
  return rows >= kPaddedTileRowsPerExpert * E && double(rows) * N * K >= 100e6 * (15.0 + K * cdiv(tiles, 512) / 80.0);
}

// The 256-row tile kernel (int4_prefill_gemm, one 8-wave workgroup a CU) in place
// of the 128-row one (moe_tile, two 4-wave workgroups). It runs, with tiles enough
// for all CUs, where most experts fill one 256-row tile but need two of 128 rows,
// and in the largest batches, where both draw the card's power limit and its one
// dequant per 256 rows saves up to 1 %; and at a short K with a round of 256-row
// tiles or more, where a tile is mostly its start and end and half as many are
// better. Per fused call, 256- vs 128-row, by rows per expert: N = 4096, K = 7168,
// E = 48: 399 vs 330 us at 100, 455 vs 448 at 128, 559 vs 595 at 180, 709 vs 672 at
// 240, 1,222 vs 1,228 at 400, Zipf 1,191 vs 1,167; N = 7168, K = 2048: 292 vs 277
// at 128, 367 vs 391 at 180, 455 vs 435 at 240; from 680 rows on 0.5 % more to 1.3 %
// less at four shapes (calls back to back; E = 48, 4,096 tokens, Zipf 1,848 vs
// 1,875); too few tiles: N = 2048, K = 4096, E = 16: 119 vs 80 at 180; K = 512, N =
// 2048, E = 48: 53 vs 43 at 100, 57 vs 65 at 128, 93 vs 104 at 320, 130 vs 136 at
// 500; K = 512, N = 4096, E = 8 (256 tiles): 63 vs 71 at 500.
bool int4_tall_tiles(int64_t rows, int64_t E, int64_t N, int64_t K) {
  if (rows < 120 * E) return false;
  const int64_t tiles = E * cdiv(N, 256) * cdiv(cdiv(rows, E), 256);
  if (K <= 1024 && tiles >= 256) return true;
  if (rows >= 600 * E) return E * cdiv(N, 256) >= 128;  // not by rows: parts of a batch take one kernel
  return rows >= 140 * E && rows < 224 * E && tiles >= 384;
}

int64_t tile_queue_bytes();
int tile_queue_stride(int64_t bytes);

// The GEMM stage's workspace: the tile kernels' queue (without one their tiles
// are dealt statically); the other kernels need none.
int64_t int4_gemm_workspace_bytes(int64_t M, int64_t K) {
  (void)M;
  (void)K;
  return tile_queue_bytes();
}

// The grouped-GEMM kernel a call runs, from its shapes and flags only (not
// from pointers), so that the number of partial planes is known before the
// call. Pointer alignment the chosen kernel needs is checked at launch.
enum class Int4Kernel { kSimple, kRs, kTile };

// ep_global > E: the call runs E local experts of ep_global under an expert
// map; the routed rows per local expert are then estimated as those of the
// dense call (numel * E / ep_global slots expected on the local experts), so
// that an expert-parallel rank picks the kernel the dense call picks for the
// same rows per expert. 0: every slot counts against the E experts.
int64_t int4_local_slots(int64_t numel, int64_t E, int64_t ep_global) {
  return ep_global > E ? (numel * E + ep_global - 1) / ep_global : numel;
}
Int4Kernel int4_choose(int64_t M, int64_t top_k, int64_t E, int64_t N, int64_t K, int a_dtype,
                       int group_size, int flags, int64_t ep_global) {
  if (!int4_use_stream(a_dtype, group_size, K)) return Int4Kernel::kSimple;
  const int64_t local = int4_local_slots(M * top_k, E, ep_global);
  const bool f32a = a_dtype == XK_DT_FP32;
  const bool padded = K % 256 != 0 || N % 256 != 0;
  const bool tile_ok = !f32a && int4_tile_ok(a_dtype, group_size, M, K, N, E) &&
                       (!padded || (flags & (XK_INT4_FUSED | XK_INT4_TEST_FORCE_TILE)));
  const bool rs_ok = int4_rs_ok(M, top_k, K, N, E, f32a, group_size);
  bool tile = tile_ok && (padded ? int4_padded_tile(local, E, N, K) : local >= kPrefillRowsPerExpert * E);
  if (flags & XK_INT4_TEST_FORCE_TILE) tile = tile_ok;
  if (flags & XK_INT4_TEST_FORCE_STREAM) tile = tile && !rs_ok;
  if (tile) return Int4Kernel::kTile;
  if (rs_ok) return Int4Kernel::kRs;
  return tile_ok ? Int4Kernel::kTile : Int4Kernel::kSimple;
}

// The kernel a call runs, for the C ABI's query: 0 the scalar kernel, 1 the
// decode stream kernel, 2 the prefill tile kernel.
int int4_kernel_code(int64_t M, int64_t top_k, int64_t E, int64_t N, int64_t K, int a_dtype,
                     int group_size, int flags, int64_t ep_global) {
  switch (int4_choose(M, top_k, E, N, K, a_dtype, group_size, flags, ep_global)) {
    case Int4Kernel::kRs: return 1;
    case Int4Kernel::kTile: return 2;
    default: return 0;
  }
}

// Number of fp32 partial planes [parts, M * top_k, N] the grouped GEMM
// writes: the K slices of the decode stream kernel, else one.
int int4_gemm_parts(int64_t M, int64_t top_k, int64_t E, int64_t N, int64_t K, int a_dtype,
                    int group_size, int flags, int64_t ep_global) {
  return int4_choose(M, top_k, E, N, K, a_dtype, group_size, flags, ep_global) == Int4Kernel::kRs
             ? int4_rs_slices(K, N, M * top_k, E, a_dtype == XK_DT_FP32)
             : 1;
}

// True when launch_int4_gemm may be called without align outputs (the decode
// kernel then routes the slots itself).
bool int4_gemm_self_routes(int64_t M, int64_t top_k, int64_t E, int64_t N, int64_t K, int a_dtype,
                           int group_size, int flags, int64_t ep_global) {
  return int4_choose(M, top_k, E, N, K, a_dtype, group_size, flags, ep_global) == Int4Kernel::kRs &&
         int4_rs_self_route_ok(M * top_k);
}

int launch_int4_gemm(const void* A, int a_dtype, int64_t M, int64_t K, const int32_t* packed,
                     const uint16_t* scale, int64_t E, int64_t N, int group_size,
                     const int32_t* topk_ids, int64_t top_k, const int32_t* emap,
                     int num_global, const int32_t* sorted_ids, const int32_t* offsets,
                     float* slot_out, int flags, int64_t ep_global, void* workspace,
                     int64_t workspace_bytes, bool queue_cleared, hipStream_t stream) {
  XK_REQUIRE(a_dtype == XK_DT_BF16 || a_dtype == XK_DT_FP32, "int4: bad A dtype %d", a_dtype);
  XK_REQUIRE(M >= 0 && top_k >= 1 && E >= 1 && N >= 1 && K >= 8, "int4: bad sizes");
  XK_REQUIRE(K % 8 == 0, "int4: K=%lld not a multiple of 8", (long long)K);
  XK_REQUIRE(group_size > 0 && K % group_size == 0, "int4: group_size=%d does not divide K",
             group_size);
  XK_REQUIRE(E <= 65535 && N < (int64_t(1) << 30) && K < (int64_t(1) << 30), "int4: size limit");
  const int64_t numel = M * top_k;
  XK_REQUIRE(numel < (int64_t(1) << 30), "int4: M*top_k too large");
  if (numel == 0) return XK_OK;
  Int4Kernel kern = int4_choose(M, top_k, E, N, K, a_dtype, group_size, flags, ep_global);
  // the decode kernel routes for itself when no align outputs are given
  const bool self_route = kern == Int4Kernel::kRs && sorted_ids == nullptr && offsets == nullptr &&
                          int4_rs_self_route_ok(numel);
  const bool aligned = reinterpret_cast<uintptr_t>(A) % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(packed) % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(scale) % 16 == 0;
  // pointers of any alignment run the scalar kernel at sizes that only the tile
  // kernel of all MFMA kernels takes and that are not multiples of 256 (more
  // than 512 experts, or a batch past the stream kernel's buffer reach)
  if (kern == Int4Kernel::kTile && !aligned && !(K % 256 == 0 && N % 256 == 0) &&
      !int4_rs_ok(M, top_k, K, N, E, false, group_size))
    kern = Int4Kernel::kSimple;
  if (kern != Int4Kernel::kSimple) {
    XK_REQUIRE(self_route || (sorted_ids && offsets),
               "int4: the MFMA kernels need the align outputs");
    XK_REQUIRE(aligned, "int4: A, packed weights and scales must be 16-byte aligned");
  }
  switch (kern) {
    case Int4Kernel::kTile: {
      // groups of 64 and 128 stay on the 256-row kernel (one scale load per
      // group and chunk in moe_tile: 120 tokens 264 vs 274 us, 1,400 Zipf 735 vs 790)
      const bool tall = ((flags & XK_INT4_TEST_TALL) || group_size != 32 ||
                         int4_tall_tiles(int4_local_slots(numel, E, ep_global), E, N, K)) &&
                        int4_prefill_ok(a_dtype, group_size, M, K, N, E);
      // the tile queue lives in the workspace; without one the tiles are
      // dealt statically
      return (tall ? launch_int4_prefill : launch_int4_tile)(
          A, K, packed, scale, E, N, numel, top_k, group_size, sorted_ids, offsets, slot_out,
          workspace != nullptr && workspace_bytes >= tile_queue_bytes() &&
                  reinterpret_cast<uintptr_t>(workspace) % 4 == 0
              ? static_cast<int*>(workspace)
              : nullptr,
          tile_queue_stride(workspace_bytes), queue_cleared, stream);
    }
    case Int4Kernel::kRs:
      return launch_int4_rs(A, a_dtype == XK_DT_FP32, M, K, packed, scale, E, N, numel, top_k,
                            group_size, sorted_ids, offsets, topk_ids, emap, num_global, slot_out,
                            stream);
    case Int4Kernel::kSimple:
      break;
  }
  const int64_t total = numel * N;
  const dim3 grid(static_cast<unsigned>(cdiv(total, 256)));
  if (a_dtype == XK_DT_BF16)
    hipLaunchKernelGGL((int4_simple_gemm<uint16_t>), grid, dim3(256), 0, stream,
                       static_cast<const uint16_t*>(A), int(K),
                       reinterpret_cast<const uint32_t*>(packed), scale, int(N), group_size,
                       topk_ids, emap, num_global, int(E), int(numel), int(top_k), slot_out);
  else
    hipLaunchKernelGGL((int4_simple_gemm<float>), grid, dim3(256), 0, stream,
                       static_cast<const float*>(A), int(K),
                       reinterpret_cast<const uint32_t*>(packed), scale, int(N), group_size,
                       topk_ids, emap, num_global, int(E), int(numel), int(top_k), slot_out);
  XK_CHECK_LAUNCH("int4_simple_gemm");
  return XK_OK;
}

}  // namespace xk
