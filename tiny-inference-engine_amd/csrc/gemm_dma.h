// One tile of a bfloat16 product whose operand slices go global memory -> LDS directly (buffer loads with the
// lds flag: no registers, no LDS write instructions), for K % 32 == 0.
//
// A workgroup of four waves (one per SIMD, 512 registers each), 2 x 2, owns a BM x BN tile; for 256 x BN a wave owns
// 128 x BN/2 of it, so that every byte read from LDS feeds twice the flops it does with the 64-wide
// wave tiles above. k advances in groups of G slices of 32 through a ring of LDS stages: while group t is
// multiplied, the groups behind it are landing or landed and the loads of t + STAGES - 1 (its w rows) and t + STAGES
// (its x rows) are issued, a few between the matrix instructions so that neither the texture
// path nor the in-order instruction stream of the one wave backs up. One barrier a group: it sits before the last 16 k's
// matrix instructions, when their fragments are in
// registers already, so that the stage is free and the next group's first fragments can be read
// while they multiply.
//
// A group is two slices wherever three stages of that size fit the LDS: half the barriers, and x's rows come as whole
// 128-byte lines. With one slice a row is half a line, for which the vector cache takes as long: the product then stood
// at 11 TB/s from the L2, which gives loads of whole lines 33, however many stages were in flight. Measured, four stages
// of one slice against three of two: 512 rows over 4096 x 12288 on 256 x 128 66.1 -> 58.6 us, 2048 rows over
// 4096 x 4096 on 128 x 256 74.7 -> 64.1, 128 rows over 24576 x 4096 on 128 x 128 58.0 -> 47.4, 2048 rows over
// 4096 x 12288 on 256 x 128 231 -> 185; experts of 768 x 2048, 256 rows each, on 128 x 256 86.5 -> 78.7 and 63.4 -> 59.8.
// Tiles of 256 x 256 and 256 x 192 have no room for that (two stages of two slices lose 10 to 15 %); tiles of 64 x 128
// are better off with three workgroups a compute unit (10 to 20 %).
//
// A staged row of x is G x 64 bytes, unpadded; its 16-byte chunks are exchanged by the row's number (gd_swizzle), which
// spreads the 32 rows a fragment read touches over the banks. Rows beyond M or N are clamped to the
// last row (their products land in output rows or columns that are never stored). With PW the weight
// comes in packed blocks of 16 rows x 32 k (1 KB in the matrix cores' operand order, as the decode
// product reads it): one load instruction stages one block, and the 16 lanes that LDS serves in a
// cycle read 256 consecutive bytes of it.
//
// The matrix instructions take w's fragment as their first operand: the tile comes out transposed,
// a lane holding 4 consecutive columns of one output row, which it stores as one 8- or 16-byte piece.
#pragma once
#include "common.h"
#include <type_traits>

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
typedef __attribute__((ext_vector_type(4))) float floatx4_t;
typedef __attribute__((address_space(3))) void lds_void_t;

#define GD_BK 32
// Stages of the ring and slices of a group, by the tile (above).
template <int BM, int BN>
struct GdShape {
  static constexpr bool PAIRS = BM * BN >= 128 * 128 && (BM + BN) * 3 * 2 * GD_BK * 2 <= 150 * 1024;
  static constexpr int GROUP = PAIRS ? 2 : 1;
  static constexpr int STAGES = PAIRS ? 3 : 4;
  static constexpr int LDS_BYTES = STAGES * GROUP * (BM + BN) * GD_BK * 2;
};
// Fourth word of a raw buffer descriptor on gfx9-family GPUs: 32-bit float data format, destination
// selects x, y, z, w; no swizzle, no stride (the compiler's own default for raw buffers on this target).
#define GD_RSRC_FLAGS 0x27000


#if defined(__HIP_DEVICE_COMPILE__)
template <int G>
__device__ __forceinline__ int gd_swizzle(int row) { return G == 1 ? (row >> 1) & 3 : row & 7; }
template <int G>
__device__ __forceinline__ int gd_stage_row(int lane, int wave) { return wave * (16 / G) + lane / (4 * G); }
template <int G>
__device__ __forceinline__ int gd_stage_chunk(int lane, int row) { return (lane & (4 * G - 1)) ^ gd_swizzle<G>(row); }

// acc = x w^T over `k_tiles` slices of 32, for a workgroup of four waves (2 x 2; a wave BM / 2 rows and BN / 2 columns).
// BM: 256, 128 or 64 rows of x. x's rows: byte offsets `a_off` into a_rsrc of the 16-byte chunk that this lane stages
// in wave instruction p (row 64 p / G + gd_stage_row, chunk gd_stage_chunk of it); w's rows: `b_off` likewise or, with
// PW, lane * 16 with `b_tile_off` the byte offset of block row 4 p + wave. A lane ends with, in acc[i][j], row
// wm BM / 2 + 32 i + lane % 32 and in word 4 g + v column wn BN / 2 + 32 j + 8 g + 4 (lane / 32) + v, wm = wave / 2 and
// wn = wave % 2.
template <int BM, int BN, bool PW>
__device__ __forceinline__ void gemm_dma_tile(bf16_t* lds, const __amdgpu_buffer_rsrc_t a_rsrc,
                                              const unsigned (&a_off)[BM * GdShape<BM, BN>::GROUP / 64], const __amdgpu_buffer_rsrc_t b_rsrc,
                                              const unsigned (&b_off)[BN / 64], const unsigned (&b_tile_off)[BN / 64],
                                              int k_tiles, floatx16 (&acc)[BM / 64][BN / 64]) {
  constexpr int G = GdShape<BM, BN>::GROUP, STAGES = GdShape<BM, BN>::STAGES;
  constexpr int BK = GD_BK;
  constexpr int TN = BN / 64;                   // 32-column MFMA tiles of a wave
  constexpr int TM = BM / 64;                   // 32-row MFMA tiles of a wave
  constexpr int PA = BM / 64;                   // wave instructions that stage x's rows (16 rows each, 4 waves)
  constexpr int PB = BN / 64;                   // wave instructions that stage w's rows likewise
  static_assert(BM == 256 || BM == 128 || BM == 64, "rows of a tile");
  static_assert(G == 1 || G == 2, "slices of a group");
  constexpr int BUF = G * (BM + BN) * BK;       // elements of one stage: x's rows over G slices, then w slice by slice
  constexpr int LOADS = G * (PA + PB);          // loads a wave issues a stage
  static_assert(STAGES >= 3 && (STAGES - 2) * LOADS < 64, "vmcnt has six bits");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane & 31;
  const int fk = lane >> 5;

  const int steps = (k_tiles + G - 1) / G;      // groups of G slices; a last one may lack some
  auto stage = [&](int s) { return lds + s * BUF; };          // group t lies in stage t % STAGES
  auto issue_x = [&](int t, int s) {           // of a group that lacks slices: what follows in memory, unused
    bf16_t* buf = stage(s);
#pragma unroll
    for (int p = 0; p < PA * G; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_void_t*)(buf + (p * 64 + wave * 16) * BK), 16, a_off[p],
                                               t * G * BK * 2, 0, 0);
  };
  auto issue_w = [&](int t, int s) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      bf16_t* buf = stage(s) + G * BM * BK + g * BN * BK;
      const int kt = G == 1 ? t : min(t * G + g, k_tiles - 1);      // a slice that is not there: the last one again, unused
#pragma unroll
      for (int p = 0; p < PB; ++p)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (lds_void_t*)(buf + (p * 64 + wave * 16) * BK), 16,
                                                 b_off[p], PW ? b_tile_off[p] + kt * 1024 : kt * BK * 2, 0, 0);
    }
  };

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // Fragment addresses. x's stage rows are swizzled (above); w's are too unless packed, where the
  // 16-byte piece of (row r of block t, k-chunk c) sits at t * 1 KB + (16 c + r) * 16 bytes: the 16 lanes
  // that one LDS cycle serves read 256 consecutive bytes.
  const int sw = gd_swizzle<1>(fr);
  const int a_row = (wm * (BM / 2) + fr) * G * BK;
  const int b_row = PW ? (wn * (BN / 32) + (fr >> 4)) * 512 + (fr & 15) * 8 : (wn * (BN / 2) + fr) * BK;

  bf16x8_t fa[2][TM], fb[2][TN];
  auto load_frags = [&](const bf16_t* buf, int ks, int set) {      // ks: a step of 16 k in the stage
    const int koff = ((ks * 2 + fk) ^ gd_swizzle<G>(fr)) * 8;
    const int koff_w = PW ? (ks % 2 * 2 + fk) * 128 : ((ks % 2 * 2 + fk) ^ sw) * 8;
    const bf16_t* bw = buf + G * BM * BK + ks / 2 * BN * BK;
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[set][i] = *reinterpret_cast<const bf16x8_t*>(buf + a_row + i * 32 * G * BK + koff);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[set][j] = *reinterpret_cast<const bf16x8_t*>(bw + b_row + j * 32 * BK + koff_w);
  };
  auto mfma_step = [&](int set) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[set][j], fa[set][i], acc[i][j], 0, 0, 0);
  };

  // A stage is free once every wave has passed the barrier of the slice that read it, which stands in the
  // middle of that slice (its last fragments are in registers by then). Slice j's x rows are asked for right
  // after the barrier of slice j - STAGES, into the stage that slice has just left, and its w rows before the barrier
  // of slice j - STAGES + 1: the loads of STAGES - 2 to STAGES - 1 slices are in flight at any time, which is what
  // the latency of L2 asks for at a slice every 0.4 us. (With four stages of 256 x 256, 64 to 96 KB; one slice less ahead,
  // the matrix cores waited a third of the time.) The first slices here.
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t) {
    if ((G > 1 || t > 2) && t >= steps) break;          // the host gives every range of K at least three slices
    issue_x(t, t);
    issue_w(t, t);
  }
  // s_waitcnt vmcnt(n) [lgkmcnt(0)], then the barrier (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt 6:4,
  // lgkmcnt 11:8; a counter at its maximum is not waited for).
  auto wait_barrier = [&](auto loads, auto lds_too) {
    constexpr int n = decltype(loads)::value;
    static_assert(n >= 0 && n < 64, "vmcnt has six bits");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | ((decltype(lds_too)::value ? 0 : 15) << 8));
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // The same with the loads of at most `slices` slices outstanding, for a number that is not known before.
  auto wait_slices = [&](int slices, auto lds_too) {
    auto at = [&](auto self, auto count) -> void {
      constexpr int c = decltype(count)::value;
      if constexpr (c == 0) wait_barrier(count, lds_too);
      else if (slices >= c) wait_barrier(std::integral_constant<int, c * LOADS>{}, lds_too);
      else self(self, std::integral_constant<int, c - 1>{});
    };
    at(at, std::integral_constant<int, STAGES - 2>{});
  };
  using Steady = std::integral_constant<int, (STAGES - 2) * LOADS>;
  // Slice 0 has landed when at most the loads of the slices behind it are outstanding.
  if constexpr (G == 1 && STAGES == 4) wait_barrier(Steady{}, std::false_type{});
  else wait_slices(min(STAGES - 1, steps) - 1, std::false_type{});
  load_frags(stage(0), 0, 0);
  if (STAGES - 1 < steps) issue_x(STAGES - 1, STAGES - 1);

  // Group t in stage s; its first fragments are in set 0 already. STEADY: groups up to t + STAGES exist, so the loads
  // sit in straight-line code and exactly those of STAGES - 2 groups may still be in flight at the barrier.
  auto group = [&](int t, int s, auto steady_tag) {
    constexpr bool STEADY = decltype(steady_tag)::value;
    const int have = STEADY || G == 1 ? 2 * G : min(2 * G, (k_tiles - t * G) * 2);     // steps of 16 k that are there
#pragma unroll
    for (int ks = 0; ks < 2 * G - 1; ++ks) {
      load_frags(stage(s), ks + 1, (ks + 1) & 1);
      if (ks == 0 && (STEADY || t + STAGES - 1 < steps)) issue_w(t + STAGES - 1, s == 0 ? STAGES - 1 : s - 1);
      if (STEADY || G == 1 || ks < have) mfma_step(ks & 1);
    }
    if (STEADY && BM == 256 && G == 1) {
#pragma unroll
      for (int q = 0; q < (4 + TN) / 2; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, TN / 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
#pragma unroll
      for (int q = 0; q < PB; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
    }
    // My share of group t + 1 has landed and my reads of this stage are in registers; after the
    // barrier that holds for every wave.
    if (STEADY) wait_barrier(Steady{}, std::true_type{});
    else wait_slices(max(0, min(STAGES - 2, steps - 2 - t)), std::true_type{});
    if (STEADY || t + 1 < steps) load_frags(stage(s == STAGES - 1 ? 0 : s + 1), 0, 0);
    if (STEADY || t + STAGES < steps) issue_x(t + STAGES, s);
    if (STEADY || G == 1 || 2 * G - 1 < have) mfma_step(1);
    if (STEADY && BM == 256 && G == 1) {
#pragma unroll
      for (int q = 0; q < (4 + TN) / 2; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, TN / 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  int t = 0;
  for (; t + 2 * STAGES - 1 < steps - (G > 1); t += STAGES) {
#pragma unroll
    for (int s = 0; s < STAGES; ++s) group(t + s, s, std::true_type{});
  }
  for (int s = 0; t < steps; ++t, s = s == STAGES - 1 ? 0 : s + 1) group(t, s, std::false_type{});
}
#endif
