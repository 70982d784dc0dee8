// One tile of a bfloat16 product whose operand slices go global memory -> LDS directly (buffer loads with the
// lds flag: no registers, no LDS write instructions), for K % 32 == 0.
//
// A workgroup of four waves (one per SIMD, 512 registers each), 2 x 2, owns a BM x BN tile; for 256 x BN a wave owns
// 128 x BN/2 of it, so that every byte read from LDS feeds twice the flops it does with the 64-wide
// wave tiles above. k advances in groups of G slices of 32 through a ring of LDS stages: while group t is
// multiplied, the groups behind it are landing or landed and the loads of t + STAGES - 1 (its w rows) and t + STAGES
// (its x rows) are issued, a few between the matrix instructions so that neither the texture
// path nor the in-order instruction stream of the one wave backs up. One barrier a group: it sits before the matrix
// instructions of the last steps of 16 k (GdShape::AHEAD: two in groups of two slices, else one), when their fragments are
// in registers already, so that the stage is free and the next group's first fragments can be read while they multiply.
//
// A group is two slices wherever three stages of that size fit the LDS: half the barriers, and x's rows come as whole
// 128-byte lines. With one slice a row is half a line, for which the vector cache takes as long: the product then stood
// at 11 TB/s from the L2, which gives loads of whole lines 33, however many stages were in flight. Measured, four stages
// of one slice against three of two: 512 rows over 4096 x 12288 on 256 x 128 66.1 -> 58.6 us, 2048 rows over
// 4096 x 4096 on 128 x 256 74.7 -> 64.1, 128 rows over 24576 x 4096 on 128 x 128 58.0 -> 47.4, 2048 rows over
// 4096 x 12288 on 256 x 128 231 -> 185; experts of 768 x 2048, 256 rows each, on 128 x 256 86.5 -> 78.7 and 63.4 -> 59.8.
// Tiles of 256 x 256 and 256 x 192 have no room for that (two stages of two slices lose 10 to 15 %): x alone comes in pairs
// of slices there, through a ring of three pairs, and w, whose blocks are whole lines anyway, slice by slice through one of
// four: 2048 rows over 24576 x 4096 on 256 x 256 366 -> 320 us, over 6144 x 4096 on 256 x 192 95 -> 86. Tiles of 64 x 128
// are better off with three workgroups a compute unit (10 to 20 %) and stage single slices of both.
//
// Fragments are read from LDS one step of 16 k ahead of their use, in tiles whose groups are pairs two steps, and the order
// of reads, loads and matrix instructions is stated to the compiler, which otherwise moves every read down to its use: a
// lone 256 x 128 tile took 0.335 us a slice, 0.261 now, where its matrix instructions take 0.213; 2048 rows over
// 4096 x 12288 on it 193 -> 175 us. The last groups of a range are straight-line code as well (512 rows over 2048 x 2048 in
// four ranges 12.7 -> 12.0 us). The large tiles are then at the clock that the card keeps with all matrix cores at work.
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
  static constexpr bool X_PAIRS = !PAIRS && BM == 256;
  static constexpr int GROUP = PAIRS ? 2 : 1;
  static constexpr int STAGES = PAIRS ? 3 : 4;
  static constexpr int AHEAD = PAIRS ? 2 : 1;            // steps that fragments are read ahead of their use
  static constexpr int X_GROUP = PAIRS || X_PAIRS ? 2 : 1;        // slices that x's rows are staged by
  static constexpr int LDS_BYTES = (X_PAIRS ? 3 * 2 * BM + 4 * BN : STAGES * GROUP * (BM + BN)) * GD_BK * 2;
};
// Fourth word of a raw buffer descriptor on gfx9-family GPUs: 32-bit float data format, destination
// selects x, y, z, w; no swizzle, no stride (the compiler's own default for raw buffers on this target).
#define GD_RSRC_FLAGS 0x27000
// The non-temporal bit of a buffer load's cache policy on gfx942 and gfx950.
#define GD_NT 2


#if defined(__HIP_DEVICE_COMPILE__)
template <int G>
__device__ __forceinline__ int gd_swizzle(int row) { return G == 1 ? (row >> 1) & 3 : row & 7; }
template <int G>
__device__ __forceinline__ int gd_stage_row(int lane, int wave) { return wave * (16 / G) + lane / (4 * G); }
template <int G>
__device__ __forceinline__ int gd_stage_chunk(int lane, int row) { return (lane & (4 * G - 1)) ^ gd_swizzle<G>(row); }

// How the instructions of one step of 16 k follow each other: a matrix instruction first, then two LDS reads behind each
// until all READS are out, then the LOADS spread over the rest.
template <int MFMAS, int READS, int LOADS>
__device__ __forceinline__ void gd_interleave() {
  if constexpr (MFMAS > 0) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    constexpr int reads = READS < 2 ? READS : MFMAS == 1 ? READS : 2;
    constexpr int loads = reads > 0 && MFMAS > 1 ? 0 : (LOADS + MFMAS - 1) / MFMAS;
    if constexpr (reads > 0) __builtin_amdgcn_sched_group_barrier(0x100, reads, 0);
    if constexpr (loads > 0) __builtin_amdgcn_sched_group_barrier(0x020, loads, 0);
    gd_interleave<MFMAS - 1, READS - reads, LOADS - loads>();
  }
}

// The same for steps of twelve matrix instructions and more: PER_READS of them before every two reads, then PER_LOAD before
// every load.
template <int PER_READS, int PER_LOAD, int READS, int LOADS>
__device__ __forceinline__ void gd_interleave_wide() {
#pragma unroll
  for (int q = 0; q < (READS + 1) / 2; ++q) {
    __builtin_amdgcn_sched_group_barrier(0x008, PER_READS, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
  }
#pragma unroll
  for (int q = 0; q < LOADS; ++q) {
    __builtin_amdgcn_sched_group_barrier(0x008, PER_LOAD, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
  }
}

// The same for tiles whose x comes in pairs of slices and whose w comes slice by slice (GdShape::X_PAIRS): x through a ring
// of three pairs, w through one of four slices.
template <int BM, int BN, bool PW>
__device__ __forceinline__ void gemm_dma_tile_x_pairs(bf16_t* lds, const __amdgpu_buffer_rsrc_t a_rsrc,
                                                      const unsigned (&a_off)[BM / 32], const __amdgpu_buffer_rsrc_t b_rsrc,
                                                      const unsigned (&b_off)[BN / 64], const unsigned (&b_tile_off)[BN / 64],
                                                      int k_tiles, floatx16 (&acc)[BM / 64][BN / 64]) {
  constexpr int BK = GD_BK;
  constexpr int TM = BM / 64, TN = BN / 64, PA = BM / 64, PB = BN / 64;
  constexpr int X_STAGE = 2 * BM * BK, W_STAGE = BN * BK;     // elements
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane & 31;
  const int fk = lane >> 5;
  bf16_t* const lds_w = lds + 3 * X_STAGE;

  auto issue_x = [&](int pair, int s, int half) {             // half the rows of a pair of slices: 32 p + 8 wave + lane / 8
#pragma unroll
    for (int p = half * PA; p < half * PA + PA; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_void_t*)(lds + s * X_STAGE + (p * 64 + wave * 16) * BK), 16,
                                               a_off[p], pair * 2 * BK * 2, 0, 0);
  };
  auto issue_w = [&](int t, int s) {
#pragma unroll
    for (int p = 0; p < PB; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (lds_void_t*)(lds_w + s * W_STAGE + (p * 64 + wave * 16) * BK), 16,
                                               b_off[p], PW ? b_tile_off[p] + t * 1024 : t * BK * 2, 0, 0);
  };

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const int sw = gd_swizzle<1>(fr);
  const int a_row = (wm * (BM / 2) + fr) * 2 * BK;
  const int b_row = PW ? (wn * (BN / 32) + (fr >> 4)) * 512 + (fr & 15) * 8 : (wn * (BN / 2) + fr) * BK;
  bf16x8_t fa[2][TM], fb[2][TN];
  auto load_frags = [&](int xs, int ws, int odd, int ks) {    // step ks of 16 k of the even or the odd slice of a pair
    const bf16_t* x = lds + xs * X_STAGE + a_row + ((odd * 4 + ks * 2 + fk) ^ gd_swizzle<2>(fr)) * 8;
    const bf16_t* w = lds_w + ws * W_STAGE + b_row + (PW ? (ks * 2 + fk) * 128 : ((ks * 2 + fk) ^ sw) * 8);
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[ks][i] = *reinterpret_cast<const bf16x8_t*>(x + i * 32 * 2 * BK);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[ks][j] = *reinterpret_cast<const bf16x8_t*>(w + j * 32 * BK);
  };
  auto mfma_step = [&](int set) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[set][j], fa[set][i], acc[i][j], 0, 0, 0);
  };
  auto wait_barrier = [&](auto loads, auto lds_too) {         // as above
    constexpr int n = decltype(loads)::value;
    static_assert(n >= 0 && n < 64, "vmcnt has six bits");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | ((decltype(lds_too)::value ? 0 : 15) << 8));
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  using All = std::integral_constant<int, 2 * PA + 2 * PB>;

  // Asked for in this order throughout, each request into a place that the barrier before it has freed: behind the barrier
  // of slice t half a pair of x (t even: the second half of pair t / 2 + 2, t odd: the first of pair (t - 1) / 2 + 3),
  // then before the barrier of slice t + 1 the w rows of slice t + 4. What slice t + 1 needs has landed when at most the
  // requests behind w's slice t + 1 (t even) or behind w's slice t + 1 and the pair before it (t odd) are outstanding:
  // two halves of x and two slices of w either way. The host gives every range of K at least three slices, so pairs 0
  // and 1 exist.
  issue_x(0, 0, 0);
  issue_x(0, 0, 1);
  issue_w(0, 0);
  issue_x(1, 1, 0);
  issue_w(1, 1);
  issue_x(1, 1, 1);
  issue_w(2, 2);
  wait_barrier(All{}, std::false_type{});
  load_frags(0, 0, 0, 0);
  if (4 < k_tiles) issue_x(2, 2, 0);

  int xs = 0, ws = 0;                                          // where slice t lies
  // STEADY: everything that slices t to t + 6 ask for exists, so the requests sit in straight-line code. (The last slices
  // in straight-line code as well, one by one, cost the compiler its accumulators' places: 2400 spills.)
  auto slice = [&](int t, auto odd_tag, auto steady_tag) {
    constexpr bool STEADY = decltype(steady_tag)::value;
    constexpr int ODD = decltype(odd_tag)::value;
    const int xs_next = ODD ? (xs == 2 ? 0 : xs + 1) : xs, ws_next = (ws + 1) & 3;
    load_frags(xs, ws, ODD, 1);
    if (STEADY || t + 3 < k_tiles) issue_w(t + 3, (ws + 3) & 3);
    mfma_step(0);
    if (STEADY) gd_interleave_wide<TN / 2, 2, TM + TN, PB>();
    if (STEADY || t + 4 < k_tiles) wait_barrier(All{}, std::true_type{});
    else if (t + 3 < k_tiles) wait_barrier(std::integral_constant<int, PA + 2 * PB>{}, std::true_type{});
    else if (t + 2 < k_tiles) wait_barrier(std::integral_constant<int, PB>{}, std::true_type{});
    else wait_barrier(std::integral_constant<int, 0>{}, std::true_type{});
    if (STEADY || t + 1 < k_tiles) load_frags(xs_next, ws_next, 1 - ODD, 0);
    const int pair = ODD ? t / 2 + 3 : t / 2 + 2;
    if (STEADY || 2 * pair < k_tiles) issue_x(pair, ODD ? xs : (xs == 0 ? 2 : xs - 1), 1 - ODD);
    mfma_step(1);
    if (STEADY) gd_interleave_wide<1, TN / 2, TM + TN, PA>();
    __builtin_amdgcn_sched_barrier(0);
    xs = xs_next;
    ws = ws_next;
  };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  int t = 0;
  for (; t + 6 < k_tiles; t += 2) {
    slice(t, even, std::true_type{});
    slice(t + 1, odd, std::true_type{});
  }
  for (; t < k_tiles; t += 2) {
    slice(t, even, std::false_type{});
    if (t + 1 < k_tiles) slice(t + 1, odd, std::false_type{});
  }
}

// acc = x w^T over `k_tiles` slices of 32, for a workgroup of four waves (2 x 2; a wave BM / 2 rows and BN / 2 columns).
// BM: 256, 128 or 64 rows of x. x's rows: byte offsets `a_off` into a_rsrc of the 16-byte chunk that this lane stages
// in wave instruction p (row 64 p / G + gd_stage_row, chunk gd_stage_chunk of it); w's rows: `b_off` likewise or, with
// PW, lane * 16 with `b_tile_off` the byte offset of block row 4 p + wave. A lane ends with, in acc[i][j], row
// wm BM / 2 + 32 i + lane % 32 and in word 4 g + v column wn BN / 2 + 32 j + 8 g + 4 (lane / 32) + v, wm = wave / 2 and
// wn = wave % 2.
template <int BM, int BN, bool PW, bool W_ONCE>
__device__ __forceinline__ void gemm_dma_tile_groups(bf16_t* lds, const __amdgpu_buffer_rsrc_t a_rsrc,
                                                     const unsigned (&a_off)[BM * GdShape<BM, BN>::X_GROUP / 64],
                                                     const __amdgpu_buffer_rsrc_t b_rsrc, const unsigned (&b_off)[BN / 64],
                                                     const unsigned (&b_tile_off)[BN / 64], int k_tiles,
                                                     floatx16 (&acc)[BM / 64][BN / 64]) {
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
                                                 b_off[p], PW ? b_tile_off[p] + kt * 1024 : kt * BK * 2, 0, W_ONCE ? GD_NT : 0);
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

  constexpr int STEPS = 2 * G;                  // steps of 16 k in a group
  constexpr int AHEAD = GdShape<BM, BN>::AHEAD, SETS = 2 * AHEAD;
  static_assert(STEPS % SETS == 0 && AHEAD < STEPS, "sets of fragments by the step's number");
  bf16x8_t fa[SETS][TM], fb[SETS][TN];
  auto load_frags = [&](const bf16_t* buf, int ks) {               // ks: a step of 16 k in the stage
    const int set = ks & (SETS - 1);
    const int koff = ((ks * 2 + fk) ^ gd_swizzle<G>(fr)) * 8;
    const int koff_w = PW ? (ks % 2 * 2 + fk) * 128 : ((ks % 2 * 2 + fk) ^ sw) * 8;
    const bf16_t* bw = buf + G * BM * BK + ks / 2 * BN * BK;
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[set][i] = *reinterpret_cast<const bf16x8_t*>(buf + a_row + i * 32 * G * BK + koff);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[set][j] = *reinterpret_cast<const bf16x8_t*>(bw + b_row + j * 32 * BK + koff_w);
  };
  auto mfma_step = [&](int ks) {
    const int set = ks & (SETS - 1);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[set][j], fa[set][i], acc[i][j], 0, 0, 0);
  };

  // A stage is free once every wave has passed the barrier of the group that read it, which stands in the
  // middle of that group (its last fragments are in registers by then). Group j's x rows are asked for right
  // after the barrier of group j - STAGES, into the stage that group has just left, and its w rows before the barrier
  // of group j - STAGES + 1: the loads of STAGES - 2 to STAGES - 1 groups are in flight at any time, which is what
  // the latency of L2 asks for. The first groups here.
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
  // Slice 0 has landed when at most the loads of the slices behind it are outstanding.
  wait_slices(min(STAGES - 1, steps) - 1, std::false_type{});
#pragma unroll
  for (int ks = 0; ks < AHEAD; ++ks) load_frags(stage(0), ks);
  if (STAGES - 1 < steps) issue_x(STAGES - 1, STAGES - 1);

  // Group t in stage s; the fragments of its first AHEAD steps are in registers already. LEFT groups follow it, or more
  // where LEFT is STAGES: which loads there are, and how many may still be in flight at the barrier, is then known here, and
  // the loads sit in straight-line code. LEFT = -1: not known.
  auto group = [&](int t, int s, auto left) {
    constexpr int LEFT = decltype(left)::value;
    constexpr bool KNOWN = LEFT >= 0;
    const int s_next = s == STAGES - 1 ? 0 : s + 1;
    const int have = G == 1 ? STEPS : min(STEPS, (k_tiles - t * G) * 2);     // steps of 16 k that are there
    const bool more = KNOWN ? LEFT > 0 : t + 1 < steps;
    const bool asks_w = KNOWN ? LEFT >= STAGES - 1 : t + STAGES - 1 < steps;
    const bool asks_x = KNOWN ? LEFT >= STAGES : t + STAGES < steps;
    __builtin_amdgcn_sched_barrier(0);
    auto step = [&](auto step_tag) {
      constexpr int ks = decltype(step_tag)::value;
      // My share of group t + 1 has landed and my reads of this stage are in registers; after the
      // barrier that holds for every wave.
      if (ks == STEPS - AHEAD) {
        if constexpr (KNOWN)
          wait_barrier(std::integral_constant<int, (LEFT - 1 < 0 ? 0 : LEFT - 1 < STAGES - 2 ? LEFT - 1 : STAGES - 2) * LOADS>{},
                       std::true_type{});
        else wait_slices(max(0, min(STAGES - 2, steps - 2 - t)), std::true_type{});
      }
      if (ks + AHEAD < STEPS) load_frags(stage(s), ks + AHEAD);
      else if (more) load_frags(stage(s_next), ks + AHEAD - STEPS);
      if (ks == 0 && asks_w) issue_w(t + STAGES - 1, s == 0 ? STAGES - 1 : s - 1);
      if (ks == STEPS - AHEAD && asks_x) issue_x(t + STAGES, s);
      if (LEFT > 0 || G == 1 || ks < 2 || ks < have) mfma_step(ks);
      if (G > 1 && LEFT > 0)
        gd_interleave<TM * TN, TM + TN,
                      (ks == 0 && LEFT >= STAGES - 1 ? G * PB : 0) + (ks == STEPS - AHEAD && LEFT >= STAGES ? G * PA : 0)>();
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    if constexpr (STEPS > 2) {
      step(std::integral_constant<int, 2>{});
      step(std::integral_constant<int, 3>{});
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  int t = 0, s = 0;
  constexpr std::integral_constant<int, STAGES> steady{};
  for (; t + 2 * STAGES - 1 < steps; t += STAGES) {              // whole rounds through the ring: no stage numbers to form
#pragma unroll
    for (int s0 = 0; s0 < STAGES; ++s0) group(t + s0, s0, steady);
  }
  if constexpr (G == 1) {
    // (Groups of one slice are too short for it: with each of the last ones known the compiler copies the accumulators
    // between the register files at every join, 64 rows over 512 x 128 4.0 -> 4.3 us.)
    for (; t < steps; ++t, s = s == STAGES - 1 ? 0 : s + 1) group(t, s, std::integral_constant<int, -1>{});
  } else {
    for (; t + STAGES < steps; ++t, s = s == STAGES - 1 ? 0 : s + 1) group(t, s, steady);
    auto last = [&](auto self, auto left) -> void {
      constexpr int LEFT = decltype(left)::value;
      if (t + LEFT < steps) {
        group(t, s, left);
        ++t;
        s = s == STAGES - 1 ? 0 : s + 1;
      }
      if constexpr (LEFT > 0) self(self, std::integral_constant<int, LEFT - 1>{});
    };
    last(last, std::integral_constant<int, STAGES - 1>{});
  }
}

template <int BM, int BN, bool PW, bool W_ONCE = false>
__device__ __forceinline__ void gemm_dma_tile(bf16_t* lds, const __amdgpu_buffer_rsrc_t a_rsrc,
                                              const unsigned (&a_off)[BM * GdShape<BM, BN>::X_GROUP / 64],
                                              const __amdgpu_buffer_rsrc_t b_rsrc, const unsigned (&b_off)[BN / 64],
                                              const unsigned (&b_tile_off)[BN / 64], int k_tiles,
                                              floatx16 (&acc)[BM / 64][BN / 64]) {
  if constexpr (GdShape<BM, BN>::X_PAIRS)
    gemm_dma_tile_x_pairs<BM, BN, PW>(lds, a_rsrc, a_off, b_rsrc, b_off, b_tile_off, k_tiles, acc);
  else
    gemm_dma_tile_groups<BM, BN, PW, W_ONCE>(lds, a_rsrc, a_off, b_rsrc, b_off, b_tile_off, k_tiles, acc);
}
#endif
