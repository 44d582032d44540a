// Kernels for the smallest decode batches: at most 6 tokens and 64 routed
// slots (one user's decode step is 1 token). The INT4 call is one launch, the
// MXFP4 MLP two; both finish in the kernel, with no partial planes, no SwiGLU
// kernel and no combine (the same results as the stream path: reference.py:22-70,
// mxfp4_reference.py:28-112).
//
// At such sizes the stream kernel (int4_stream.hip) is bound by latency: its
// waves hold one 4 KiB line in flight, its launch, routing, first segment,
// planes and combine are most of the call (INT4, 1 token, N = 4096, K = 7168,
// 8 experts, 132 MB: 39.5 + 7.3 us; MXFP4, hidden 4096, ispp 512, 6 experts:
// 10.7 + 3.4 + 10.7 + 5.9). Here
//   * the MFMA's 16 rows are the batch's tokens, the same for every expert, so
//     the activations are loaded once and no rows are gathered; a token not
//     routed to an expert has its row of that expert's product left out;
//   * a workgroup owns 16 output columns for all experts (INT4, MXFP4 down) or
//     for one (MXFP4 gate/up), so the sum over a token's experts happens in
//     registers and LDS, in a fixed order;
//   * its waves split (expert, 512-k unit) pairs evenly, each with the next
//     unit's 16-byte loads in flight while one is contracted.
// Per call, stream path -> here: INT4 at N = 4096, K = 7168, 1 / 2 / 4 / 8 tokens
// 46 -> 31, 67 -> 57, 93 -> 86, 124 -> 123 us (other sizes: small_int4_faster); N =
// 7168, K = 2048, 1 / 4 / 8 tokens 25.5 -> 19, 51 -> 48, 67 -> 68 us; MXFP4, 1 / 4 /
// 8 tokens 28.8 -> 19.1, 39 -> 28, 53.5 -> 53 us. From 8 tokens on the experts'
// weights hide the latencies either way.
#include <algorithm>
#include <cmath>

#include "int4_common.h"

namespace xk {

int device_cu_count();

namespace {

constexpr int kTokens = 8;       // tokens the kernels hold
constexpr int kMaxTokens = 6;    // tokens they take: with 8 the stream path is as fast
constexpr int kSlots = 64;       // most routed slots: one lane each
constexpr int kUnitK = 512;      // k per unit: two 256-k lines
constexpr int kRowPad = 8;       // bf16 past each LDS row: rows 16 bytes apart modulo the banks

// The batch's routing, found by every workgroup from the ids (one lane per
// slot): the distinct local experts and, per expert and token, the summed
// routing weight of the token's slots there.
struct Routing {
  int n;                          // distinct experts
  int expert[kSlots];
  uint64_t slots[kSlots];         // slots of the expert
  float weight[kSlots][kTokens];
  uint8_t tokens[kSlots];         // bit m: token m is routed there
};

// Wave 0 lists the experts; the caller synchronises, then calls route_weights.
__device__ __forceinline__ void route_experts(Routing& r, int e, int lane) {
  uint64_t left = __ballot(e >= 0);
  int n = 0;
  while (left) {
    const int first = __builtin_ctzll(left);
    const int x = __builtin_amdgcn_readlane(e, first);
    const uint64_t same = __ballot(e == x);
    if (lane == 0) {
      r.expert[n] = x;
      r.slots[n] = same;
    }
    left &= ~same;
    ++n;
  }
  if (lane == 0) r.n = n;
}
__device__ __forceinline__ void route_weights(Routing& r, const float* w, int top_k, int tid, int threads) {
  for (int i = tid; i < r.n * kTokens; i += threads) {
    const int x = i / kTokens, m = i % kTokens;
    const uint64_t of_token = ((top_k == 64 ? ~0ull : (1ull << top_k) - 1) << min(m * top_k, 63)) &
                              (m * top_k < kSlots ? r.slots[x] : 0ull);
    float sum = 0.f;
    for (uint64_t s = of_token; s; s &= s - 1) sum += w != nullptr ? w[__builtin_ctzll(s)] : 1.0f;
    r.weight[x][m] = sum;
  }
  for (int x = tid; x < r.n; x += threads) {
    int bits = 0;
    for (uint64_t s = r.slots[x]; s; s &= s - 1) bits |= 1 << (__builtin_ctzll(s) / top_k);
    r.tokens[x] = static_cast<uint8_t>(bits);
  }
}

// `rows` rows of K bf16 (K a multiple of 8) into LDS, kRowPad apart.
__device__ __forceinline__ void stage_rows(uint16_t* lds, const uint16_t* A, int rows, int K, int tid,
                                           int threads) {
  const int per = K >> 3;
  for (int i = tid; i < rows * per; i += threads) {
    const int r = i / per, c = i - r * per;
    *reinterpret_cast<u32x4*>(lds + r * (K + kRowPad) + c * 8) =
        *reinterpret_cast<const u32x4*>(A + static_cast<int64_t>(r) * K + c * 8);
  }
}

enum class Fmt { kInt4, kFp4 };

// A 512-k unit of 16 columns in a wave's registers: lane (c, q) holds groups
// 4 h + q of both 256-k lines of column c, and 16 (8) bytes of the column's 16
// group scales.
template <Fmt FMT> struct Unit {
  u32x4 w[2][2];                                   // [line][h]
  uint32_t s[FMT == Fmt::kInt4 ? 4 : 2];           // INT4: line q & 1's 8 scales; MXFP4: line q & 1's 8 bytes
};

// Loads unit `ku` of the column whose packed row and scales start at w, s.
template <Fmt FMT>
__device__ __forceinline__ void load_unit(Unit<FMT>& u, const uint8_t* w, const uint8_t* s, int ku, int q) {
#pragma unroll
  for (int l = 0; l < 2; ++l)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      u.w[l][h] = *reinterpret_cast<const u32x4*>(w + ku * (kUnitK / 2) + l * 128 + h * 64 + q * 16);
  if constexpr (FMT == Fmt::kInt4) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(s + ku * 32 + (q & 1) * 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) u.s[i] = v[i];
  } else {
    const uint2 v = *reinterpret_cast<const uint2*>(s + ku * 16 + (q & 1) * 8);
    u.s[0] = v.x;
    u.s[1] = v.y;
  }
}

// acc += activation rows (row base `a` of this lane's token, at the unit's k)
// times the unit's 16 columns. Line l's scales sit in lanes q = l, l + 2: one
// cross-lane read per word (ds_bpermute) brings them to all four.
template <Fmt FMT>
__device__ __forceinline__ void contract_unit(f32x4& acc, const Unit<FMT>& u, const uint16_t* a, int q, int c16,
                                              uint32_t mlo, uint32_t mhi) {
#pragma unroll
  for (int l = 0; l < 2; ++l) {
    const int src = (l * 16 + c16) * 4;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // the scale of group 4 h + q
      RneScale ks;
      float fs = 0.f;
      uint32_t keep = ~0u;
      if constexpr (FMT == Fmt::kInt4) {
        const uint32_t lo = __builtin_amdgcn_ds_bpermute(src, u.s[2 * h]);
        const uint32_t hi = __builtin_amdgcn_ds_bpermute(src, u.s[2 * h + 1]);
        const uint32_t word = q & 2 ? hi : lo;
        ks = rne_scale(__uint_as_float(q & 1 ? word & 0xFFFF0000u : word << 16));
      } else {
        const uint32_t b = (__builtin_amdgcn_ds_bpermute(src, u.s[h]) >> (8 * q)) & 0xFFu;
        fs = e8m0_scale(b);
        keep = b == 0xFFu ? 0u : ~0u;  // read as 0
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        bf16x8 b;
        if constexpr (FMT == Fmt::kInt4) b = dequant_rne_nat(u.w[l][h][j], ks, mlo, mhi);
        else b = fp4x8_to_bf16(u.w[l][h][j] & keep, fs);
        const bf16x8 af = *reinterpret_cast<const bf16x8*>(a + l * 256 + (4 * h + q) * 32 + 8 * j);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, b, acc, 0, 0, 0);
      }
    }
  }
}

struct SmallArgs {
  const uint16_t* A;       // [M, K] bf16 (MXFP4 down: act [numel, K])
  const uint8_t* w;        // [E, N, K/2]
  const uint8_t* scale;    // [E, N, K/32] bf16 or e8m0
  const uint16_t* bias;    // MXFP4: [E, N] or null
  const int32_t* ids;      // [numel]
  const int32_t* emap;
  const float* weights;    // [numel] or null
  uint16_t* out;           // [M, N] bf16 (MXFP4 gate/up: act [numel, N / 2])
  int M, K, N, E, numel, top_k, num_global;
  float limit;
};

// INT4: out[m, n] = sum over the token's slots of weight * A[m] @ W[e, n].
template <int WAVES>
__global__ void __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(4, 4)))
small_int4(SmallArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint16_t rows[];  // [M][K + kRowPad]
  __shared__ Routing r;
  __shared__ float red[WAVES][kTokens][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int c16 = lane & 15, q = lane >> 4;
  const int K = p.K, N = p.N, n0 = blockIdx.x * 16;
  const uint32_t mlo = in_vgpr(0x000F000Fu), mhi = in_vgpr(0x00F000F0u);

  if (wave == 0)
    route_experts(r, lane < p.numel ? map_expert(p.ids[lane], p.emap, p.num_global, p.E) : -1, lane);
  stage_rows(rows, p.A, p.M, K, tid, WAVES * 64);
  __syncthreads();
  const int nu = K / kUnitK, total = r.n * nu;
  int u = total * wave / WAVES;
  const int end = total * (wave + 1) / WAVES;
  auto load = [&](int i, Unit<Fmt::kInt4>& d) __attribute__((always_inline)) {
    const int x = uniform(i / nu);
    const int64_t row = static_cast<int64_t>(r.expert[x]) * N + n0 + c16;
    load_unit<Fmt::kInt4>(d, p.w + row * (K >> 1), p.scale + row * (K >> 4), i - x * nu, q);
  };
  Unit<Fmt::kInt4> buf[2];
  if (u < end) load(u, buf[0]);
  route_weights(r, p.weights, p.top_k, tid, WAVES * 64);
  __syncthreads();

  f32x4 acc{0.f, 0.f, 0.f, 0.f};  // rows 4 q + v, column c16 of the current expert's product
  f32x4 sum{0.f, 0.f, 0.f, 0.f};  // weighted over experts
  const uint16_t* a = rows + (c16 < p.M ? c16 : 0) * (K + kRowPad);  // rows past M are not used
  auto unit = [&](int i, Unit<Fmt::kInt4>& cur, Unit<Fmt::kInt4>& nxt) __attribute__((always_inline)) {
    if (i + 1 < end) load(i + 1, nxt);
    const int x = uniform(i / nu), ku = i - x * nu;
    contract_unit<Fmt::kInt4>(acc, cur, a + ku * kUnitK, q, c16, mlo, mhi);
    if (ku == nu - 1 || i == end - 1) {  // this wave's part of expert x is done
      const int bits = r.tokens[x];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = 4 * q + v;
        if (q < 2 && (bits >> m & 1)) sum[v] += r.weight[x][m] * acc[v];
      }
      acc = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  for (; u < end; u += 2) {
    unit(u, buf[0], buf[1]);
    if (u + 1 < end) unit(u + 1, buf[1], buf[0]);
  }
  if (q < 2)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][4 * q + v][c16] = sum[v];
  __syncthreads();
  if (tid < p.M * 16) {
    const int m = tid >> 4, c = tid & 15;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) s += red[i][m][c];
    p.out[static_cast<int64_t>(m) * N + n0 + c] = f32_to_bf16(s);
  }
}

// MXFP4 gate/up of one expert and 16 activation columns: waves 0-3 the gate
// rows, 4-7 the up rows, a quarter of K each.
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4)))
small_mxfp4_gateup(SmallArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint16_t rows[];  // [M][K + kRowPad]
  __shared__ float red[8][kTokens][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int c16 = lane & 15, q = lane >> 4;
  const int K = p.K, ispp = p.N >> 1, j0 = blockIdx.x * 16;
  // the blockIdx.y-th distinct expert and its slots (every wave for itself)
  const int e = lane < p.numel ? map_expert(p.ids[lane], p.emap, p.num_global, p.E) : -1;
  uint64_t left = __ballot(e >= 0), slots = 0;
  int x = -1;
  for (int n = 0; left != 0 && n <= static_cast<int>(blockIdx.y); ++n) {
    x = __builtin_amdgcn_readlane(e, __builtin_ctzll(left));
    slots = __ballot(e == x);
    left &= ~slots;
    if (left == 0 && n < static_cast<int>(blockIdx.y)) x = -1;
  }
  if (x < 0) return;  // fewer experts than workgroup rows (the whole workgroup returns)
  const int64_t row = static_cast<int64_t>(x) * p.N + (wave >= 4 ? ispp : 0) + j0 + c16;
  const uint8_t* w = p.w + row * (K >> 1);
  const uint8_t* s = p.scale + row * (K >> 5);
  const int nu = K / kUnitK, part = wave & 3;
  int u = nu * part / 4;
  const int end = nu * (part + 1) / 4;
  Unit<Fmt::kFp4> buf[2];
  if (u < end) load_unit<Fmt::kFp4>(buf[0], w, s, u, q);
  if (u + 1 < end) load_unit<Fmt::kFp4>(buf[1], w, s, u + 1, q);
  stage_rows(rows, p.A, p.M, K, tid, 512);
  __syncthreads();
  f32x4 acc{0.f, 0.f, 0.f, 0.f};
  const uint16_t* a = rows + (c16 < p.M ? c16 : 0) * (K + kRowPad);
  for (; u < end; u += 2) {
    contract_unit<Fmt::kFp4>(acc, buf[0], a + u * kUnitK, q, c16, 0, 0);
    if (u + 2 < end) load_unit<Fmt::kFp4>(buf[0], w, s, u + 2, q);
    if (u + 1 < end) {
      contract_unit<Fmt::kFp4>(acc, buf[1], a + (u + 1) * kUnitK, q, c16, 0, 0);
      if (u + 3 < end) load_unit<Fmt::kFp4>(buf[1], w, s, u + 3, q);
    }
  }
  if (q < 2)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][4 * q + v][c16] = acc[v];
  __syncthreads();
  if (tid < p.M * 16) {
    const int m = tid >> 4, c = tid & 15;
    const uint64_t of_token = slots & ((p.top_k == 64 ? ~0ull : (1ull << p.top_k) - 1) << (m * p.top_k));
    if (of_token != 0) {
      float g = 0.f, up = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        g += red[i][m][c];
        up += red[4 + i][m][c];
      }
      const uint16_t* b = p.bias ? p.bias + static_cast<int64_t>(x) * p.N : nullptr;
      const uint16_t act = mxfp4_swiglu(g, up, b, j0 + c, ispp, p.limit);
      for (uint64_t t = of_token; t; t &= t - 1) p.out[static_cast<int64_t>(__builtin_ctzll(t)) * ispp + j0 + c] = act;
    }
  }
}

// MXFP4 down projection and combine of 16 output columns: a wave takes whole
// experts (the row is rounded to bf16 before the weight).
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4)))
small_mxfp4_down(SmallArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint16_t rows[];  // [numel][K + kRowPad]
  __shared__ Routing r;
  __shared__ float red[8][kTokens][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int c16 = lane & 15, q = lane >> 4;
  const int K = p.K, N = p.N, n0 = blockIdx.x * 16;
  if (wave == 0)
    route_experts(r, lane < p.numel ? map_expert(p.ids[lane], p.emap, p.num_global, p.E) : -1, lane);
  stage_rows(rows, p.A, p.numel, K, tid, 512);  // rows of dropped slots are never read
  __syncthreads();
  const int nu = K / kUnitK, total = ((r.n - wave + 7) / 8) * nu;  // experts wave, wave + 8, ...
  auto load = [&](int i, Unit<Fmt::kFp4>& d) __attribute__((always_inline)) {
    const int64_t row = static_cast<int64_t>(r.expert[wave + 8 * uniform(i / nu)]) * N + n0 + c16;
    load_unit<Fmt::kFp4>(d, p.w + row * (K >> 1), p.scale + row * (K >> 5), i % nu, q);
  };
  Unit<Fmt::kFp4> buf[2];
  if (total > 0) load(0, buf[0]);
  route_weights(r, p.weights, p.top_k, tid, 512);
  __syncthreads();
  f32x4 acc{0.f, 0.f, 0.f, 0.f}, sum{0.f, 0.f, 0.f, 0.f};
  auto unit = [&](int i, Unit<Fmt::kFp4>& cur, Unit<Fmt::kFp4>& nxt) __attribute__((always_inline)) {
    if (i + 1 < total) load(i + 1, nxt);
    const int x = wave + 8 * uniform(i / nu), ku = i % nu;
    // token c16's first slot at this expert; any slot's row where it has none
    const uint64_t of_token =
        c16 * p.top_k < kSlots
            ? r.slots[x] & ((p.top_k == 64 ? ~0ull : (1ull << p.top_k) - 1) << min(c16 * p.top_k, 63))
            : 0ull;
    const int slot = __builtin_ctzll(of_token != 0 ? of_token : r.slots[x]);
    contract_unit<Fmt::kFp4>(acc, cur, rows + slot * (K + kRowPad) + ku * kUnitK, q, c16, 0, 0);
    if (ku == nu - 1) {
      const int bits = r.tokens[x];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = 4 * q + v;
        if (q < 2 && (bits >> m & 1)) {
          float d = round_bf16(acc[v]);
          if (p.bias != nullptr)
            d = round_bf16(d + bf16_to_f32(p.bias[static_cast<int64_t>(r.expert[x]) * N + n0 + c16]));
          sum[v] += r.weight[x][m] * d;
        }
      }
      acc = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  for (int i = 0; i < total; i += 2) {
    unit(i, buf[0], buf[1]);
    if (i + 1 < total) unit(i + 1, buf[1], buf[0]);
  }
  if (q < 2)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][4 * q + v][c16] = sum[v];
  __syncthreads();
  if (tid < p.M * 16) {
    const int m = tid >> 4, c = tid & 15;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) s += red[i][m][c];
    p.out[static_cast<int64_t>(m) * N + n0 + c] = f32_to_bf16(s);
  }
}

constexpr int64_t kSmallLds = 140 * 1024;  // beside the static arrays
constexpr int64_t kStaticLds = 12 * 1024, kTwoWorkgroupLds = 80 * 1024;
int64_t row_lds(int64_t rows, int64_t K) { return rows * (K + kRowPad) * 2; }

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

// Whether small_int4 is expected to be faster than the stream kernel, from fits to
// both kernels' times with cold weights (2,130 sizes: X = 1 to 48 experts, N = 256
// to 14336, K = 512 to 14336; mean error 8 %; where the choice is wrong it costs 4
// us or less but for a few sizes). A workgroup walks the weights of 16 columns for
// every expert X of the batch, so beyond the bytes its time grows with X K per
// workgroup of a CU, more where the rows in the LDS leave a CU one workgroup of
// eight waves; the stream kernel splits experts x columns over all CUs. Stream vs
// here: N = 4096, K = 7168, E = 48, top_k 8: 1 token 44 vs 33 us, 3 tokens 69 vs
// 64, 6 tokens 114 vs 115; N = 7168, K = 2048: 3 tokens 41 vs 37, 6 tokens 61 vs
// 64; N = 5120, K = 7168: 3 tokens 81 vs 108, 6 tokens 142 vs 229; E = 8, top_k 2,
// N = 256, K = 14336, 4 tokens 24 vs 42; E = 256, top_k 8, N = 4096, K = 2048, 2
// tokens 30 vs 21.
bool small_int4_faster(int64_t M, int64_t top_k, int64_t E, int64_t routed, int64_t N, int64_t K) {
  // local experts that `M` tokens' slots are expected to reach
  const double miss = 1.0 - double(std::min(top_k, routed)) / double(routed);
  const double experts = double(E) * (1.0 - std::pow(miss, double(M)));
  const double k1 = double(K) / 1e3, all = experts * double(N) * double(K) / 1e7;
  const int64_t cus = device_cu_count(), per_cu = cdiv(N / 16, cus);
  const bool alone = per_cu > 1 && row_lds(M, K) + kStaticLds > kTwoWorkgroupLds;
  const double walk = experts * double(per_cu) * (alone ? 0.46 : 0.3) + 0.085 * double(M);
  const double here = 5.0 + 0.09 * experts + k1 * walk + 0.3 * all;
  const double stream = 10.5 + 0.1 * experts + k1 + 0.89 * all + 1.5e-6 * double(M * top_k) * double(N);
  return here < stream;
}

// Batches the one-launch INT4 kernel takes: bf16 activations, groups of 32, at
// most 6 tokens and 64 slots, K a multiple of 512, N of 16, 16-byte aligned
// pointers, the tokens' activations in the LDS. `routed`: the experts that the
// ids range over (under an expert map more than the E local ones).
bool small_int4_ok(int a_dtype, int64_t M, int64_t top_k, int64_t E, int64_t routed, int64_t N, int64_t K,
                   int group_size, const void* A, const void* packed, const void* scale) {
  return a_dtype == XK_DT_BF16 && group_size == 32 && M >= 1 && M <= kMaxTokens && M * top_k <= kSlots &&
         K % kUnitK == 0 && N % 16 == 0 && N / 16 < (1 << 30) && K < (1 << 24) && E <= 65535 &&
         row_lds(M, K) <= kSmallLds && aligned16(A) && aligned16(packed) && aligned16(scale) &&
         small_int4_faster(M, top_k, E, routed, N, K);
}

int launch_small_int4(const uint16_t* A, int64_t M, int64_t K, const int32_t* packed, const uint16_t* scale,
                      int64_t E, int64_t N, const int32_t* topk_ids, const float* weights, int64_t top_k,
                      const int32_t* emap, int num_global, uint16_t* out, hipStream_t stream) {
  const SmallArgs a{A, reinterpret_cast<const uint8_t*>(packed), reinterpret_cast<const uint8_t*>(scale), nullptr,
                    topk_ids, emap, weights, out, int(M), int(K), int(N), int(E), int(M * top_k), int(top_k),
                    num_global, 0.f};
  const dim3 grid(static_cast<unsigned>(N / 16));
  const size_t lds = row_lds(M, K);
  // 16 waves fill a CU; with more workgroups than CUs, two of 8 waves share one
  if (N / 16 > device_cu_count())
    hipLaunchKernelGGL(small_int4<8>, grid, dim3(512), lds, stream, a);
  else
    hipLaunchKernelGGL(small_int4<16>, grid, dim3(1024), lds, stream, a);
  XK_CHECK_LAUNCH("small_int4");
  return XK_OK;
}

// MXFP4: the same, for hidden and ispp multiples of 512, with rows in the LDS that
// leave room for two workgroups a CU where there are so many, and a down projection
// that its waves can share: a wave takes whole experts, so few experts of a long
// ispp leave most waves idle (sooner where few columns leave the CUs idle too), and
// every workgroup loads a row per slot, which costs it more from 3 tokens on.
// Stream vs here, cold weights: E = 256, hidden 7168, ispp 512, top_k 8, 5 tokens
// (70 KiB) 64 vs 62 us, 6 tokens (84 KiB) 73 vs 95, but E = 8, top_k 1 (up to 256
// workgroups) 27 vs 16; E = 64, hidden 4096, ispp 1024, top_k 8, 3 tokens (down 48
// KiB) 43 vs 42, 4 tokens (64.5 KiB) 50 vs 53; E = 8, hidden 1024, top_k 2: ispp
// 8192, 2 tokens 29 vs 35, ispp 14336, 1 token 33 vs 46; hidden 7168, ispp 8192, 1
// token 59 vs 51; E = 256, hidden 1024, ispp 512, top_k 8, 6 tokens 32 vs 34.
constexpr int64_t kSmallGateUpLds = 72 * 1024, kSmallDownLds = 64 * 1024, kSmallLoneLds = 128 * 1024;
bool small_mxfp4_ok(int a_dtype, int64_t M, int64_t top_k, int64_t E, int64_t hidden, int64_t ispp, const void* A,
                    const void* w13, const void* w13_scale, const void* w2, const void* w2_scale) {
  if (a_dtype != XK_DT_BF16 || M < 1 || M > kMaxTokens || M * top_k > kSlots || hidden % kUnitK != 0 ||
      ispp % kUnitK != 0 || hidden >= (1 << 24) || ispp >= (1 << 24) || E > 1024)
    return false;
  const int64_t numel = M * top_k, gate_up = row_lds(M, hidden), down = row_lds(numel, ispp);
  const bool few = ispp / 16 * std::min(E, numel) <= 2 * device_cu_count();
  return gate_up <= (few ? kSmallLoneLds : kSmallGateUpLds) && down <= (M <= 2 ? kSmallGateUpLds : kSmallDownLds) &&
         ispp * cdiv(numel, 8) <= (hidden >= 4096 ? 8192 : 7168) &&
         (hidden > 1024 || numel <= 8 || numel * ispp < 24576) && aligned16(A) && aligned16(w13) &&
         aligned16(w13_scale) && aligned16(w2) && aligned16(w2_scale);
}

int launch_small_mxfp4(const uint16_t* A, int64_t M, int64_t hidden, const uint8_t* w13, const uint8_t* s13,
                       const uint8_t* w2, const uint8_t* s2, int64_t E, int64_t ispp, const uint16_t* b13,
                       const uint16_t* b2, float limit, const int32_t* topk_ids, const float* weights,
                       int64_t top_k, const int32_t* emap, int num_global, uint16_t* act, uint16_t* out,
                       hipStream_t stream) {
  const int numel = int(M * top_k);
  const SmallArgs g{A, w13, s13, b13, topk_ids, emap, nullptr, act, int(M), int(hidden), int(2 * ispp), int(E),
                    numel, int(top_k), num_global, limit};
  hipLaunchKernelGGL(small_mxfp4_gateup, dim3(static_cast<unsigned>(ispp / 16), static_cast<unsigned>(numel)),
                     dim3(512), row_lds(M, hidden), stream, g);
  XK_CHECK_LAUNCH("small_mxfp4_gateup");
  const SmallArgs d{act, w2, s2, b2, topk_ids, emap, weights, out, int(M), int(ispp), int(hidden), int(E),
                    numel, int(top_k), num_global, 0.f};
  hipLaunchKernelGGL(small_mxfp4_down, dim3(static_cast<unsigned>(hidden / 16)), dim3(512), row_lds(numel, ispp),
                     stream, d);
  XK_CHECK_LAUNCH("small_mxfp4_down");
  return XK_OK;
}

}  // namespace xk
