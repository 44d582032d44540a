// Grouped GEMM of 4-bit weights for batches with many routed rows per expert
// (prefill and large decode batches): the INT4 W4A16 projection (the
// reference's _fused_moe_int4_kernel at large M, src/xkernels/ops/moe/triton/
// moe_int4_kernel.py:78-272; math of reference.py:22-70, dequant of
// w4a16.py:21-50) and both projections of the MXFP4 MoE (_mxfp4_moe_gemm_kernel,
// triton/moe_mxfp4_kernel.py:87-352; math of mxfp4_reference.py:28-112).
//
// For routed slot t of local expert e, W = the expert's bf16 weights:
//   kRows    INT4: slot row fp32[N] = A[t / div] @ W^T
//   kGateUp  MXFP4: act bf16[N / 2] = swiglu of bf16(A[t / div] @ W13^T) (+ b13)
//   kDown    MXFP4: slot row bf16[N] = bf16(act[t] @ W2^T) (+ b2 -> bf16)
// and the weighted top-k combine runs afterwards.
//
//   * a tile is (expert, up to 32 MAXRT consecutive rows of its padded slot
//     range, 256 weight rows), one 4-wave workgroup; wave w owns all the
//     tile's rows x 64 weight rows as MAXRT x 2 tiles of
//     v_mfma_f32_32x32x16_bf16, so each weight is dequantised once per tile;
//   * v_mfma_f32_32x32x16_bf16 and not the 16x16x32: one of the first hides 4 to
//     6 VALU instructions of the SIMD's other wave behind its 32 cycles, two of
//     the second about 4, and an LDS operand read feeds 32 rows instead of 16;
//   * lane (c, h) of a wave reads 16 bytes of column c: quantisation group
//     2 t + h of a 128-k chunk. Word j of it feeds MFMA j, which contracts k =
//     8 j .. 8 j + 7 of both groups. A chunk's weights and scales are loaded
//     into registers a chunk ahead;
//   * activations: 128-k chunks, double-buffered in LDS, filled a chunk ahead by
//     direct-to-LDS loads (8 rows x 128 contiguous bytes each). The 16-byte
//     pieces of a row are permuted by the row's low bits, so that the 32 lanes
//     of an operand read (32 rows, one piece each) spread over all banks;
//   * two workgroups share a CU, so one's barriers, first loads and row stores
//     run under the other's MFMAs (one 8-wave workgroup with 256-row tiles took
//     1,947 us where these take 1,867 at INT4, 4,096 tokens, K = 7168; 64-row
//     tiles with three workgroups a CU 240 where these take 220 at 80 tokens);
//   * a persistent grid takes the tiles from a queue. Row blocks are ordered by
//     height (the costliest first) and expert, a block's column tiles outside,
//     so consecutive tiles share a column tile's weights; runs of kRun
//     consecutive tiles are dealt to the 8 XCDs in turn, each with an L2 of its
//     own, and an XCD whose runs are used up takes other XCDs' tiles (runs of 4
//     to 128 tiles measured the same). The XCDs' counters sit a cache line apart
//     where the caller's buffer allows: atomics on one line wait for each other
//     over all XCDs, which cost a launch about 25 us (gate/up of E = 64, hidden
//     256, ispp 2048, 30 rows per expert, 1,024 tiles, per call: 105 -> 80 us).
//     Tiles that all fit the places at once are dealt without the queue (E = 64,
//     hidden = ispp = 256, 448 tokens, top_k 4, per call: 72 -> 36 us).
//
// Measured per fused call against the kernels it replaces (MXFP4: 32-row passes
// of a 4-wave workgroup per column block; INT4: the 256-row tile kernel): MXFP4
// E = 256, hidden 4096, ispp 512, top_k 6, 4,096 tokens 1,197 -> 468 us; INT4
// E = 48, N = 4096, K = 7168, top_k 8, 250 tokens 297 -> 246 us. At INT4, 4,096
// tokens it draws the card's power limit (1.73 GHz at 59 % MFMA busy; builds
// without the activation loads, the dequant and the weight loads run 265, 190 and
// 110 us faster).
#include <algorithm>
#include <type_traits>

#include "int4_common.h"

namespace xk {

int device_cu_count();

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kTileCols = kWaves * 64;  // weight rows per tile
constexpr int kStageK = 64;             // k per LDS stage (128 bytes a row)
constexpr int kChunkK = 128;            // k per step: two stages
constexpr int kMaxE = 1024;
constexpr int kXcds = 8;  // workgroup b runs on XCD b % 8
constexpr int kRun = 16;  // consecutive tiles dealt to one XCD

enum class Epi { kRows, kGateUp, kDown };
enum class Fmt { kInt4, kFp4 };

struct TileArgs {
  const uint16_t* A;      // [a_rows, K] bf16
  const uint8_t* w;       // [E, N, K/2]
  const uint8_t* scale;   // [E, N, K/32 >> glog]: bf16 (INT4) or e8m0 bytes (MXFP4)
  const uint16_t* bias;   // kGateUp, kDown: [E, N] bf16 or null
  const int32_t* sorted_ids;
  const int32_t* offsets;  // [E+1] padded slot prefix
  void* out;
  int* queue;              // tiles taken of each XCD's runs (zero at launch), or null
  int queue_stride;        // ints from one XCD's counter to the next
  int K, N, numel, num_experts;
  int a_row_div;           // A row of slot t: t / a_row_div
  int glog;                // INT4: log2(group size / 32)
  uint32_t a_bytes;
  float limit;             // kGateUp: swiglu clamp, <= 0 disables
};

// 16-byte piece `x` of row `row` sits at piece x ^ piece_swizzle(row) of the
// row's 128 LDS bytes: rows r .. r + 7 reach 8 different pieces, rows r and
// r + 8 (which share the parity of their 128-byte half) different ones too.
__device__ __forceinline__ int piece_swizzle(int row) { return (row & 7) ^ ((row >> 3) & 1); }

// A buffer resource in scalar registers. Its parts are forced wave-uniform: the
// compiler wraps a load whose resource it holds in vector registers in a loop
// over lane values.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t uniform_rsrc(const uint8_t* base, int bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  const uint64_t u = static_cast<uint64_t>(uniform(static_cast<uint32_t>(a))) |
                     static_cast<uint64_t>(uniform(static_cast<uint32_t>(a >> 32))) << 32;
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<uint8_t*>(u), 0, uniform(bytes), 0x00020000);
}

// The tile table of a workgroup: row blocks by height class, prefixes over the
// experts. Class c holds blocks of MAXRT - c row tiles (class 0: full blocks
// and the highest tails).
template <int MAXRT> struct TileTable {
  int full[kMaxE + 1];
  uint16_t tail[MAXRT - 1][kMaxE + 1];
};

// SCL false: K a multiple of 512 and groups of 32; scales load in blocks of 512
// k. True: any multiple of 32 and group of 32, 64, 128; one load per group, and
// the activations past K are zero in LDS (out-of-range loads land zeros), as
// are the scales there.
template <Fmt FMT, bool SCL, Epi EPI, int RT>
__device__ __forceinline__ void run_tile(const TileArgs& p, int e, int col_tile, u32x4* a_lds,
                                         const int* tok_lds, const int* slot_lds) {
  constexpr int SB = FMT == Fmt::kInt4 ? 2 : 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int c32 = lane & 31, h = lane >> 5;
  const int K = p.K, KB = K >> 1, G = K >> (5 + (SCL && FMT == Fmt::kInt4 ? p.glog : 0));
  const int glog = SCL && FMT == Fmt::kInt4 ? p.glog : 0;
  const int ncols = EPI == Epi::kGateUp ? p.N >> 1 : p.N;  // output columns
  const int nch = (K + kChunkK - 1) / kChunkK;
  // chunk buffers: four where the LDS of two 128-row chunks and the registers
  // allow (up to 64 rows, whose steps are too short to cover a load's latency)
  constexpr int kDepth = RT <= 2 ? 4 : 2;
  const uint32_t kNibMask = in_vgpr(0x000F000Fu), kNibMaskHi = in_vgpr(0x00F000F0u);

  // this wave's two column tiles: gate and up of the same columns, or neighbours
  const int col0 = EPI == Epi::kGateUp ? col_tile * (kTileCols / 2) + wave * 32
                                       : col_tile * kTileCols + wave * 64;
  __amdgpu_buffer_rsrc_t rw[2], rs[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int col = EPI == Epi::kGateUp ? col0 : col0 + 32 * t;
    const int valid = max(0, min(32, ncols - col));
    const int64_t row = static_cast<int64_t>(e) * p.N + min(col, ncols - 1) + (EPI == Epi::kGateUp ? t * ncols : 0);
    // a tile past the last column keeps one row (of it the last one; never
    // stored): an empty buffer would be smaller than the scalar offsets
    rw[t] = uniform_rsrc(p.w + row * KB, max(valid, 1) * KB);
    rs[t] = uniform_rsrc(p.scale + row * G * SB, max(valid, 1) * G * SB);
  }
  const i32x4 ra = make_rsrc(p.A, p.a_bytes);
  constexpr int kOut = static_cast<int>(0x80000000u);  // past every buffer

  // activation loads: load i of a stage covers rows 32 i + 8 wave .. + 7
  int a_off[RT];
  const int a_row = 8 * wave + (lane >> 3);  // + 32 i
  const int a_piece = (lane & 7) ^ piece_swizzle(a_row);
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int tok = tok_lds[32 * i + a_row];
    a_off[i] = tok >= 0 ? tok * K * 2 + a_piece * 16 : kOut;
  }
  auto load_a = [&](int ch, auto bufc) __attribute__((always_inline)) {
    constexpr int buf = decltype(bufc)::value;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int k0 = ch * kChunkK + g * kStageK;
      const bool past = SCL && k0 + a_piece * 8 >= K;
      const int soff = !SCL || k0 < K ? k0 * 2 : 0;
#pragma unroll
      for (int i = 0; i < RT; ++i)
        dma_16(ra, a_lds + ((buf * 2 + g) * RT + i) * 256 + wave * 64, past ? kOut : a_off[i], soff);
    }
  };

  // Weights of a 128-k chunk: two 16-byte groups of each column tile's column.
  const int w_off = c32 * KB + h * 16;
  struct Chunk {
    u32x4 w[2][2];     // [group pair][column tile]
    uint32_t s[2][2];  // SCL: the scale of the lane's group of each pair, [column tile][pair]
  };
  auto load_w = [&](int ch, Chunk& k) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const bool past = SCL && 4 * ch + 2 * g + h >= (K >> 5);
        k.w[g][t] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw[t], past ? kOut : w_off + 32 * g, ch * 64, 0));
      }
      if constexpr (SCL) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          const int blk = 4 * ch + 2 * g + h;
          const int off = blk < (K >> 5) ? (c32 * G + (blk >> glog)) * SB : kOut;
          if constexpr (FMT == Fmt::kInt4) k.s[t][g] = __builtin_amdgcn_raw_buffer_load_b16(rs[t], off, 0, 0);
          else k.s[t][g] = __builtin_amdgcn_raw_buffer_load_b8(rs[t], off, 0, 0);
        }
      }
    }
  };
  // Scales without SCL come in blocks of four chunks (512 k, 16 groups a
  // column): lane (c, h) loads groups 8 h .. 8 h + 7 of column c (a load per
  // chunk fetched a 128-byte line per column for 8 bytes of it, a third of the
  // kernel's L2 requests). It needs groups 4 q + 2 g + h of chunk q: the even
  // ones of both halves for h = 0, the odd ones for h = 1, which packing the
  // even and the odd ones and one half-wave swap per register pair gives.
  constexpr int kRaw = FMT == Fmt::kInt4 ? 4 : 2;
  struct ScaleBlock {
    uint32_t r[2][kRaw];  // [column tile]
  };
  auto load_s = [&](int blk, ScaleBlock& b) __attribute__((always_inline)) {
    const int off = c32 * G * SB + h * (8 * SB);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if constexpr (FMT == Fmt::kInt4) {
        const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs[t], off, blk * 32, 0));
#pragma unroll
        for (int i = 0; i < kRaw; ++i) b.r[t][i] = v[i];
      } else {
        const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs[t], off, blk * 16, 0));
#pragma unroll
        for (int i = 0; i < kRaw; ++i) b.r[t][i] = v[i];
      }
    }
  };
  // afterwards INT4 register q holds chunk q's two scales; MXFP4 register q / 2
  // chunk q's two in its byte pair q % 2
  auto arrange = [&](ScaleBlock& b) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      uint32_t ev[kRaw / 2], od[kRaw / 2];
#pragma unroll
      for (int i = 0; i < kRaw / 2; ++i) {
        constexpr uint32_t se = FMT == Fmt::kInt4 ? 0x05040100u : 0x06040200u;
        constexpr uint32_t so = FMT == Fmt::kInt4 ? 0x07060302u : 0x07050301u;
        ev[i] = __builtin_amdgcn_perm(b.r[t][2 * i + 1], b.r[t][2 * i], se);
        od[i] = __builtin_amdgcn_perm(b.r[t][2 * i + 1], b.r[t][2 * i], so);
      }
#pragma unroll
      for (int i = 0; i < kRaw / 2; ++i) {
        const auto x = __builtin_amdgcn_permlane32_swap(ev[i], od[i], false, false);
        b.r[t][i] = x[0];
        b.r[t][kRaw / 2 + i] = x[1];
      }
    }
  };

  f32x16 acc[RT][2];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][t][v] = 0.f;

  // operand read j of a row tile: piece 4 h + j of row c32 (+ 32 i)
  int a_rd[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) a_rd[j] = c32 * 8 + ((4 * h + j) ^ piece_swizzle(c32));

  // One chunk's contraction in 8 sub-steps (group pair g, word j): the next
  // sub-step's operands are read and dequantised between this one's MFMAs.
  // Dequant and MFMAs in separate runs leave the two waves of a SIMD in phase,
  // both in VALU or both in MFMA (INT4, 4,096 tokens, K = 7168: MFMA busy 51 %,
  // VALU 47 %, 62 cycles per MFMA; interleaved 53 cycles).
  auto compute = [&](const Chunk& k, const ScaleBlock& sb, auto qc) __attribute__((always_inline)) {
    constexpr int q = decltype(qc)::value;  // ch % 4: chunk of the scale block
    RneScale ks[2];    // of the group pair being dequantised
    float fs[2];
    uint32_t keep[2];  // MXFP4: 0 where the scale byte is 0xFF (read as 0)
    auto set_scale = [&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if constexpr (FMT == Fmt::kInt4) {
          const uint32_t r = SCL ? k.s[t][g] : sb.r[t][q];
          ks[t] = rne_scale(__uint_as_float(SCL || g == 0 ? r << 16 : r & 0xFFFF0000u));
        } else {
          const uint32_t b = SCL ? k.s[t][g] : (sb.r[t][q / 2] >> (16 * (q & 1) + 8 * g)) & 0xFFu;
          fs[t] = e8m0_scale(b);
          keep[t] = b == 0xFFu ? 0u : ~0u;
        }
      }
    };
    const u32x4* a = a_lds + (q % kDepth) * 2 * RT * 256;
    auto read = [&](auto ic, bf16x8 (&f)[RT]) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
#pragma unroll
      for (int r = 0; r < RT; ++r) f[r] = __builtin_bit_cast(bf16x8, a[((i >> 2) * RT + r) * 256 + a_rd[i & 3]]);
    };
    auto dequant = [&](auto ic, bf16x8 (&b)[2]) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value, g = i >> 2, j = i & 3;
      if constexpr (j == 0) set_scale(std::integral_constant<int, g>{});
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if constexpr (FMT == Fmt::kInt4) b[t] = dequant_rne_nat(k.w[g][t][j], ks[t], kNibMask, kNibMaskHi);
        else b[t] = fp4x8_to_bf16(k.w[g][t][j] & keep[t], fs[t]);
      }
    };
    bf16x8 af[2][RT], b[2][2];
    read(std::integral_constant<int, 0>{}, af[0]);
    dequant(std::integral_constant<int, 0>{}, b[0]);
    __builtin_amdgcn_sched_barrier(0);
    static_for<8>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value, cur = i & 1;
      if constexpr (i < 7) {
        read(std::integral_constant<int, i + 1>{}, af[cur ^ 1]);
        dequant(std::integral_constant<int, i + 1>{}, b[cur ^ 1]);
      }
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[r][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[cur][r], b[cur][t], acc[r][t], 0, 0, 0);
      if constexpr (i < 7) {
        constexpr int kValu = FMT == Fmt::kInt4 ? 34 : 10;
        static_for<2 * RT>([&](auto mc) __attribute__((always_inline)) {
          constexpr int m = decltype(mc)::value;
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // an MFMA
          if constexpr (m < RT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // an LDS read
          __builtin_amdgcn_sched_group_barrier(0x2, (kValu + 2 * RT - 1) / (2 * RT), 0);
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // Chunk ch: once its loads (issued kDepth - 1 chunks ago) have landed in every
  // wave, those of chunk ch + kDepth - 1 are issued into the buffers and
  // registers that chunk ch - 1 freed, and chunk ch is contracted. Until the
  // last chunks, only the loads of the kDepth - 2 chunks after ch may still be
  // in flight: 2 RT direct-to-LDS loads, 4 weight loads and the scale loads
  // each, in that order. (The compiler does not count the direct-to-LDS loads:
  // its own wait for the chunk's registers is placed, by passing them through
  // an empty asm, before the new loads are issued, so that it cannot wait for
  // those.)
  constexpr int kLoads = 2 * RT + 4 + (SCL ? 4 : 0);
  ScaleBlock sc, sn;
  Chunk ring[kDepth];
  auto chunk = [&](int ch, auto qc) __attribute__((always_inline)) {
    constexpr int q = decltype(qc)::value, cur = q % kDepth, nxt = (q + kDepth - 1) % kDepth;
    if (kDepth > 2 && ch + kDepth - 2 < nch) XK_WAIT_VMCNT((kDepth - 2) * kLoads);
    else XK_WAIT_VMCNT(0);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      asm volatile("" : "+v"(ring[cur].w[0][t]), "+v"(ring[cur].w[1][t]));
      if constexpr (SCL) {
        asm volatile("" : "+v"(ring[cur].s[t][0]), "+v"(ring[cur].s[t][1]));
      } else if constexpr (q == 0) {
#pragma unroll
        for (int i = 0; i < kRaw; ++i) {
          asm volatile("" : "+v"(sn.r[t][i]));
          sc.r[t][i] = sn.r[t][i];
        }
      }
    }
    lds_sync();  // and this wave's operand reads of the previous chunk are done
    // the next block's scales: before the chunk loads they are older than, so
    // the waits above need not count them
    if constexpr (!SCL && q == 3 - (kDepth - 2)) {
      if (ch + kDepth - 1 < nch) load_s((ch >> 2) + 1, sn);
    }
    if (ch + kDepth - 1 < nch) {
      load_a(ch + kDepth - 1, std::integral_constant<int, nxt>{});
      load_w(ch + kDepth - 1, ring[nxt]);
    }
    if constexpr (!SCL && q == 0) arrange(sc);
    compute(ring[cur], sc, qc);
  };
  if constexpr (!SCL) load_s(0, sn);
  static_for<kDepth - 1>([&](auto d) __attribute__((always_inline)) {
    if (decltype(d)::value < nch) {
      load_a(decltype(d)::value, d);
      load_w(decltype(d)::value, ring[d]);
    }
  });
  for (int ch = 0; ch < nch; ch += 4)
    static_for<4>([&](auto q) __attribute__((always_inline)) {
      if (!SCL || ch + decltype(q)::value < nch) chunk(ch + decltype(q)::value, q);  // SCL false: nch % 4 == 0
    });

  // C layout: register v of a lane is row 8 (v / 4) + 4 h + v % 4, column c32.
  auto slot_of = [&](int i, int v) { return slot_lds[32 * i + 8 * (v >> 2) + 4 * h + (v & 3)]; };
  if constexpr (EPI == Epi::kRows) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int slot = slot_of(i, v);
        float* orow = static_cast<float*>(p.out) + static_cast<int64_t>(slot) * ncols;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int col = col0 + 32 * t + c32;
          if (slot >= 0 && col < ncols) orow[col] = acc[i][t][v];
        }
      }
    return;
  }
  // bf16 outputs leave two columns at a time: a lane pair (c, c + 1) holds two
  // bf16 each in a register, of column tiles 0 and 1 (kDown) or of rows v and
  // v + 1 (kGateUp); the even lane takes both low halves, the odd lane both
  // high ones. The columns are multiples of 32 wide, so a tile is in or out.
  const bool odd = (lane & 1) != 0;
  const uint32_t pair_sel = odd ? 0x03020706u : 0x05040100u;
  auto pair_up = [&](uint32_t x) __attribute__((always_inline)) {
    const uint32_t y = __builtin_amdgcn_update_dpp(x, x, 0xB1, 0xF, 0xF, false);  // the neighbour's
    return __builtin_amdgcn_perm(y, x, pair_sel);
  };
  uint16_t* const out16 = static_cast<uint16_t*>(p.out);
  if constexpr (EPI == Epi::kGateUp) {
    const int col = col0 + (c32 & ~1);
    if (col0 >= ncols) return;
    const uint16_t* b = p.bias ? p.bias + static_cast<int64_t>(e) * p.N : nullptr;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int v = 0; v < 16; v += 2) {
        uint32_t x = mxfp4_swiglu(acc[i][0][v], acc[i][1][v], b, col0 + c32, ncols, p.limit);
        x |= static_cast<uint32_t>(mxfp4_swiglu(acc[i][0][v + 1], acc[i][1][v + 1], b, col0 + c32, ncols, p.limit)) << 16;
        const uint32_t o = pair_up(x);
        const int slot = slot_of(i, v + (odd ? 1 : 0));
        if (slot >= 0) *reinterpret_cast<uint32_t*>(out16 + static_cast<int64_t>(slot) * ncols + col) = o;
      }
  } else {
    const int col = col0 + (odd ? 32 : 0) + (c32 & ~1);
    float b[2] = {0.f, 0.f};
    if (p.bias != nullptr)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        b[t] = bf16_to_f32(p.bias[static_cast<int64_t>(e) * ncols + min(col0 + 32 * t + c32, ncols - 1)]);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        float d[2] = {acc[i][0][v], acc[i][1][v]};
        if (p.bias != nullptr)
#pragma unroll
          for (int t = 0; t < 2; ++t) d[t] = round_bf16(d[t]) + b[t];
        const uint32_t o = pair_up(f32_to_bf16(d[0]) | static_cast<uint32_t>(f32_to_bf16(d[1])) << 16);
        const int slot = slot_of(i, v);
        if (slot >= 0 && col < ncols)
          *reinterpret_cast<uint32_t*>(out16 + static_cast<int64_t>(slot) * ncols + col) = o;
      }
  }
}

template <Fmt FMT, bool SCL, Epi EPI, int MAXRT>
__device__ __forceinline__ void tile_body(const TileArgs& p) {
  constexpr int kRowsMax = 32 * MAXRT;
  __shared__ __attribute__((aligned(16))) u32x4 a_lds[4 * MAXRT * 256];
  __shared__ int tok_lds[kRowsMax];
  __shared__ int slot_lds[kRowsMax];
  __shared__ TileTable<MAXRT> tab;
  __shared__ int tile_lds;

  const int tid = threadIdx.x, lane = tid & 63;
  const int E = p.num_experts;
  const int ncols = EPI == Epi::kGateUp ? p.N >> 1 : p.N;
  const int per = EPI == Epi::kGateUp ? kTileCols / 2 : kTileCols;
  const int NB = (ncols + per - 1) / per;

  if (tid < 64) {
    int run[MAXRT] = {};
    for (int base = 0; base < E; base += 64) {
      const int e = base + lane;
      const int rows = e < E ? p.offsets[e + 1] - p.offsets[e] : 0;
      const int full = rows / kRowsMax, left = (rows - full * kRowsMax + 31) >> 5;
#pragma unroll
      for (int c = 0; c < MAXRT; ++c) {
        int x = c == 0 ? full + (left == MAXRT) : left == MAXRT - c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const int y = __shfl_up(x, d);
          if (lane >= d) x += y;
        }
        if (e < E) {
          if (c == 0) tab.full[e + 1] = run[0] + x;
          else tab.tail[c - 1][e + 1] = static_cast<uint16_t>(run[c] + x);
        }
        run[c] += __shfl(x, 63);
      }
    }
    if (lane == 0) {
      tab.full[0] = 0;
      for (int c = 1; c < MAXRT; ++c) tab.tail[c - 1][0] = 0;
    }
  }
  __syncthreads();
  int total = tab.full[E];
  for (int c = 1; c < MAXRT; ++c) total += tab.tail[c - 1][E];
  total *= NB;
  // XCD x takes runs x, x + 8, ... of kRun tiles
  auto xcd_tiles = [&](int x) {
    const int q = total / (kXcds * kRun), rem = total - q * kXcds * kRun;
    return q * kRun + min(kRun, max(0, rem - x * kRun));
  };
  auto xcd_tile = [&](int x, int n) { return ((n / kRun) * kXcds + x) * kRun + n % kRun; };
  const int xcd = blockIdx.x % kXcds;
  int n_next = blockIdx.x / kXcds;

  for (;;) {
    __syncthreads();  // every wave is done with the previous tile's LDS
    if (tid < 64) {
      int tt = -1;
      if (p.queue == nullptr || total <= static_cast<int>(gridDim.x)) {
        if (n_next < xcd_tiles(xcd)) tt = xcd_tile(xcd, n_next);
        n_next += gridDim.x / kXcds;
      } else {
        // the own XCD's queue first; then the next one that is not used up by one
        // read of them all (the counters only grow), each at most once
        auto take = [&](int x) {
          int n = 0;
          if (lane == 0) n = atomicAdd(&p.queue[x * p.queue_stride], 1);
          n = uniform(n);
          return n < xcd_tiles(x) ? xcd_tile(x, n) : -1;
        };
        tt = take(xcd);
        for (uint32_t left = 0xFFu & ~(1u << xcd); tt < 0 && left != 0;) {
          const bool open = lane < kXcds && (left >> lane & 1u) &&
                            __hip_atomic_load(&p.queue[lane * p.queue_stride], __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT) < xcd_tiles(lane);
          left = static_cast<uint32_t>(__ballot(open));
          if (left == 0) break;
          const uint32_t after = left & ~((2u << xcd) - 1);
          const int x = __builtin_ctz(after != 0 ? after : left);
          tt = take(x);
          left &= ~(1u << x);
        }
      }
      if (lane == 0) tile_lds = tt;
    }
    __syncthreads();
    int t = uniform(tile_lds);
    if (t < 0) break;
    // class, then (expert, column tile, row block): the expert whose tiles hold
    // position t of the class is counted by one ballot per 64 experts
    int cls = 0, e = 0, blk = 0, ct = 0;
    auto decode = [&](auto pre) __attribute__((always_inline)) {
      for (int base = 1; base < E; base += 64)
        e += __popcll(__ballot(base + lane < E && static_cast<int>(pre(base + lane)) * NB <= t));
      const int beg = pre(e), n = pre(e + 1) - beg;  // n row blocks
      const int at = t - beg * NB;
      ct = at / n;
      blk = at - ct * n;
    };
    if (t < tab.full[E] * NB) {
      decode([&](int i) { return tab.full[i]; });
    } else {
      t -= tab.full[E] * NB;
      for (cls = 1; cls < MAXRT - 1 && t >= tab.tail[cls - 1][E] * NB; ++cls) t -= tab.tail[cls - 1][E] * NB;
      decode([&](int i) { return static_cast<int>(tab.tail[cls - 1][i]); });
    }
    e = uniform(e);
    ct = uniform(ct);
    const int beg = p.offsets[e], rows_e = p.offsets[e + 1] - beg;
    // a class's block of an expert: its blk-th full block, or its tail
    const int row0 = beg + (cls == 0 ? blk : rows_e / kRowsMax) * kRowsMax;
    const int rows = uniform(min(kRowsMax, beg + rows_e - row0));
    if (tid < kRowsMax) {
      int slot = -1, tok = -1;
      if (tid < rows) {
        const int s = p.sorted_ids[row0 + tid];
        if (s < p.numel) { slot = s; tok = s / p.a_row_div; }
      }
      slot_lds[tid] = slot;
      tok_lds[tid] = tok;
    }
    __syncthreads();
    if constexpr (MAXRT >= 4) {
      if (rows > 96) { run_tile<FMT, SCL, EPI, 4>(p, e, ct, a_lds, tok_lds, slot_lds); continue; }
      if (rows > 64) { run_tile<FMT, SCL, EPI, 3>(p, e, ct, a_lds, tok_lds, slot_lds); continue; }
    }
    if (rows > 32) run_tile<FMT, SCL, EPI, 2>(p, e, ct, a_lds, tok_lds, slot_lds);
    else run_tile<FMT, SCL, EPI, 1>(p, e, ct, a_lds, tok_lds, slot_lds);
  }
}

// Zeroes the tile queues before a tile kernel (a kernel, not a memset, so that
// a captured graph holds no memset node).
__global__ void clear_queue(int* q, int n, int stride) {
  if (static_cast<int>(threadIdx.x) < n) q[threadIdx.x * stride] = 0;
}

// Two workgroups a CU: 256 registers a lane (128 of them sums at 128 rows).
template <Fmt FMT, bool SCL, Epi EPI>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
moe_tile(TileArgs p) {
  tile_body<FMT, SCL, EPI, 4>(p);
}

template <Fmt FMT, bool SCL, Epi EPI>
int launch_tile(const TileArgs& a, hipStream_t stream) {
  const int cus = std::max(kXcds, device_cu_count() / kXcds * kXcds);
  hipLaunchKernelGGL((moe_tile<FMT, SCL, EPI>), dim3(2 * cus), dim3(kThreads), 0, stream, a);
  XK_CHECK_LAUNCH("moe_tile");
  return XK_OK;
}

}  // namespace

// The least bytes of one tile kernel launch's queue, and the ints between its
// counters in a buffer of `bytes`: up to a cache line.
int64_t tile_queue_bytes() { return kXcds * sizeof(int); }
int64_t tile_queue_best_bytes() { return kXcds * 128; }
int tile_queue_stride(int64_t bytes) {
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(32, bytes / tile_queue_bytes())));
}

int launch_clear_queue(int* q, int n, int stride, hipStream_t stream) {
  hipLaunchKernelGGL(clear_queue, dim3(1), dim3(64), 0, stream, q, n, stride);
  XK_CHECK_LAUNCH("clear_queue");
  return XK_OK;
}

// Shapes the INT4 tile kernel takes: bf16 activations, groups of 32, 64 or
// 128, K a multiple of 32, N of 16, at most kMaxE local experts, A and one
// expert's packed weights each below 2^31 bytes (the reach of a buffer
// resource's 32-bit offsets).
bool int4_tile_ok(int a_dtype, int group_size, int64_t M, int64_t K, int64_t N, int64_t E) {
  return a_dtype == XK_DT_BF16 && (group_size == 32 || group_size == 64 || group_size == 128) &&
         K % 32 == 0 && K % group_size == 0 && N % 16 == 0 && E <= kMaxE && M * K * 2 < (int64_t(1) << 31) &&
         N * K / 2 < (int64_t(1) << 31);
}

int launch_int4_tile(const void* A, int64_t K, const int32_t* packed, const uint16_t* scale,
                        int64_t E, int64_t N, int64_t numel, int64_t top_k, int group_size,
                        const int32_t* sorted_ids, const int32_t* offsets, float* slot_out,
                        int* queue, int queue_stride, bool queue_cleared, hipStream_t stream) {
  XK_REQUIRE(reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(packed) % 16 == 0,
             "int4 tile: A and packed must be 16-byte aligned");
  const int64_t a_bytes = numel / std::max<int64_t>(top_k, 1) * K * 2;
  XK_REQUIRE(a_bytes < (int64_t(1) << 31), "int4 tile: A must be below 2^31 bytes");
  if (queue != nullptr && !queue_cleared)
    if (int rc = launch_clear_queue(queue, kXcds, queue_stride, stream)) return rc;
  TileArgs a{static_cast<const uint16_t*>(A), reinterpret_cast<const uint8_t*>(packed),
             reinterpret_cast<const uint8_t*>(scale), nullptr, sorted_ids, offsets, slot_out, queue, queue_stride,
             int(K), int(N), int(numel), int(E), int(top_k),
             group_size == 128 ? 2 : group_size == 64 ? 1 : 0, uint32_t(a_bytes), 0.f};
  if (K % 512 == 0 && a.glog == 0) return launch_tile<Fmt::kInt4, false, Epi::kRows>(a, stream);
  return launch_tile<Fmt::kInt4, true, Epi::kRows>(a, stream);
}

// One MXFP4 projection: stage 0 (gate/up, `rows` = 2 ispp weight rows, act
// bf16 [numel, ispp]) or stage 1 (down, rows = hidden, slot rows bf16
// [numel, hidden]). The queue is zero at launch.
int launch_mxfp4_tile(int stage, const uint16_t* A, int64_t a_rows, int64_t K, const uint8_t* w,
                      const uint8_t* ws, const uint16_t* bias, int64_t E, int64_t rows,
                      const int32_t* sorted_ids, const int32_t* offsets, int64_t numel,
                      int64_t a_row_div, float limit, uint16_t* out, int* queue, int queue_stride, hipStream_t stream) {
  XK_REQUIRE(K % 32 == 0 && K >= 32, "mxfp4: contraction %lld not a multiple of 32", (long long)K);
  XK_REQUIRE(reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0,
             "mxfp4: activations and weights must be 16-byte aligned");
  if (numel == 0) return XK_OK;
  TileArgs a{A, w, ws, bias, sorted_ids, offsets, out, queue, queue_stride, int(K), int(rows), int(numel), int(E),
             int(a_row_div), 0, uint32_t(a_rows * K * 2), limit};
  // block-wise scale loads need 4-byte aligned scale rows
  if (K % 512 == 0 && reinterpret_cast<uintptr_t>(ws) % 4 == 0)
    return stage == 0 ? launch_tile<Fmt::kFp4, false, Epi::kGateUp>(a, stream)
                      : launch_tile<Fmt::kFp4, false, Epi::kDown>(a, stream);
  return stage == 0 ? launch_tile<Fmt::kFp4, true, Epi::kGateUp>(a, stream)
                    : launch_tile<Fmt::kFp4, true, Epi::kDown>(a, stream);
}

}  // namespace xk
