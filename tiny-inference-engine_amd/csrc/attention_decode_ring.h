// What the decode attention kernels share, and one wave of the kernel that walks pages of 16 positions or more
// (included after DH, the head size, is defined).
#pragma once
#include "qk_prepare.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

constexpr int KSTEPS = (DH + 31) / 32;  // k blocks of the first product
constexpr int DTILES = DH / 16;         // row tiles of the second product

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));   // native vectors: fragments stay in registers
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ bf16x8_t frag(u32x4_t v) { return *reinterpret_cast<const bf16x8_t*>(&v); }

// One tile of 32 keys for the 16 columns of a wave: scores, online softmax in float32, values. kf: the keys'
// fragments of the two 16-key sub-tiles, vf: the values' fragments, qf: the queries. Shared by the kernels
// below, so that a position's result does not depend on which of them ran.
template <bool CAPPED>
__device__ __forceinline__ void attend_tile(const u32x4_t (&kf)[2][KSTEPS], const u32x4_t (&vf)[DTILES],
                                            const u32x4_t (&qf)[KSTEPS], floatx4 (&acc)[DTILES], float& m, float& l,
                                            int base, int start, int pos, int quad, float scale_log2e, float cap) {
  // ---- first product: two 16-key sub-tiles
  floatx4 sc[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    sc[u] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int st = 0; st < KSTEPS; ++st)
      sc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(kf[u][st]), frag(qf[st]), sc[u], 0, 0, 0);
  }
  if constexpr (CAPPED) {     // capped scores: cap * tanh(s / cap), still in the units of the unscaled product
    const float inv_cap = 1.f / cap;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) sc[u][v] = cap * tanh_fast(sc[u][v] * inv_cap);
  }
  // ---- softmax of this lane's column over its 8 keys (quad * 8 + u * 4 + v), then across the four quads.
  // Scores stay unscaled; scale * log2(e) > 0 enters in the exponent: p = 2^(s c - m c).
  float sv[8];
  float tile_max = -INFINITY;
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int kp = base + quad * 8 + u * 4 + v;
      const float x = (kp <= pos && kp >= start) ? sc[u][v] : -INFINITY;
      sv[u * 4 + v] = x;
      tile_max = fmaxf(tile_max, x);
    }
  tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 16, TIE_WAVE));
  tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32, TIE_WAVE));
  const float m_new = fmaxf(m, tile_max);
  const float neg_mc = (m_new == -INFINITY) ? 0.f : -m_new * scale_log2e;
  const float corr = __builtin_amdgcn_exp2f(fmaf(m, scale_log2e, neg_mc));   // m = -inf: 0
  u32x4_t pf;
  float psum = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const float p0 = __builtin_amdgcn_exp2f(fmaf(sv[i], scale_log2e, neg_mc));       // masked: 0
    const float p1 = __builtin_amdgcn_exp2f(fmaf(sv[i + 1], scale_log2e, neg_mc));
    psum += p0;
    psum += p1;
    pf[i / 2] = pack_bf16x2(p0, p1);
  }
  l = l * corr + psum;
  m = m_new;
  // ---- second product
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt) {
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[dt][v] *= corr;
    acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(vf[dt]), frag(pf), acc[dt], 0, 0, 0);
  }
}

// What a wave leaves when its keys are done: the output row itself with one share, else its (maximum, sum,
// accumulator) for the merge. h: the query head of this lane's column, z: the sequence's place in the launch.
__device__ __forceinline__ void store_share(const floatx4 (&acc)[DTILES], float m, float l, bf16_t* __restrict__ out,
                                            float* __restrict__ part_o, float* __restrict__ part_ml, int t, int z,
                                            int h, int H, int quad, int nsplit, int split, float scale_log2e,
                                            const float* __restrict__ sinks) {
  if (nsplit == 1) {  // no merge needed: normalise and store
    bf16_t* o = out + (static_cast<size_t>(t) * H + h) * DH;
    const float inv = sinks != nullptr ? sink_normaliser(m * scale_log2e, l, sinks[h] * TIE_LOG2E) : 1.0f / l;
#pragma unroll
    for (int dt = 0; dt < DTILES; ++dt)
      *reinterpret_cast<u32x2_t*>(o + dt * 16 + quad * 4) =
          u32x2_t{pack_bf16x2(acc[dt][0] * inv, acc[dt][1] * inv), pack_bf16x2(acc[dt][2] * inv, acc[dt][3] * inv)};
    return;
  }
  const size_t slot = (static_cast<size_t>(z) * H + h) * nsplit + split;
  float* po = part_o + slot * DH;
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt)
    *reinterpret_cast<float4*>(po + dt * 16 + quad * 4) = make_float4(acc[dt][0], acc[dt][1], acc[dt][2], acc[dt][3]);
  if (quad == 0) {
    part_ml[slot * 2] = m * scale_log2e;     // the merge works in the exponent's units (base 2)
    part_ml[slot * 2 + 1] = l;
  }
}

// Pages of 16 positions or more, with DEPTH - 1 tiles in flight behind the one that is computed.
// The kernel for smaller pages asks for a tile's data after it has waited for the lookup of its pages, and the counter of
// outstanding vector loads runs in order: waiting for a lookup waits for every data load issued before it, so
// a wave never has more than one tile (16 KB at head size 128) on its way and its time is one memory latency
// a tile. Here a half tile of 16 positions lies in one page, so the two page numbers of a tile are the same
// for all lanes and are read from the wave's own copy of the page table in LDS, which has a counter of its own; the
// tiles live in a ring of DEPTH register sets that is walked with constant indices, so no set is copied (a copy would
// wait for its loads). The arithmetic of a tile and the order of the tiles are that kernel's: the same bits.
//
// A short step's time is trips to memory that wait for each other, 0.5 to 1.5 us each, so there are few: the lengths and
// the first TABLE_AHEAD entries of the sequence's page table (asked for whole, before it is known which of them the
// share needs) in one; everything the queries are made of, and behind it the share's first DEPTH tiles, in another.
// What is asked for ahead is asked for without a condition (a tile beyond the share's end is its last again): behind a
// condition the compiler does not know how many loads are younger than the one it waits for, and waits for them all.
//
// PREPARE: the kernel makes its queries itself from the projection's planes of partial sums (sum, per-head RMS
// norm, rotation by the step's table of angles: the q/k kernel's own functions, so the same bits), every wave
// those of its KV head's group, through LDS into the operand layout; and one wave of each (sequence, KV head) makes the
// newest token's key and value, sends them to the cache for later steps and attends to them from LDS, so nothing that
// counts is read from the cache in the launch that writes it. One kernel less a layer; head sizes 32 to 256 in powers
// of two (head_dim / 8 lanes a head). PREPARE_SHARES: the keys are cut into shares and the newest token is the last
// share, alone (attention_decode_newest; made by the wave of the last tiles, behind them, it kept that wave 2 us longer
// than the others). PREPARE_WHOLE: a wave walks a whole sequence and takes the newest token behind its tiles.
enum DecodePrepare { PREPARE_NOTHING, PREPARE_SHARES, PREPARE_WHOLE };

// Entries of a page table that a wave keeps: 4096 keys in pages of 16. A share that begins behind them asks again, a trip
// more than the others, and still no step over 8 k to 32 k keys is slower than with a scalar load a tile (1.7B, one sequence
// 1395 -> 1259 us over 8 k and 1722 -> 1608 over 32 k, four 1751 -> 1658 and 3251 -> 3181; 12 layers of the 8B shape, one
// 1396 -> 1350 over 32 k, eight 1693 -> 1678 over 8 k and 2998 -> 2985 over 32 k).
constexpr int TABLE_AHEAD = 256;

struct QkSource {
  const float* qkv;        // [planes][rows][in_row] float32: q heads, k heads, v heads of a row
  size_t plane_stride;
  int planes;
  int in_row;
  const float* q_weight;   // per-head norm weights, or null for no norm
  const float* k_weight;
  float eps;
  const float* angles;     // [rows][DH]: cos of the DH / 2 angles, then sin
  int write_kv;            // 0: the cache holds the newest token already (another layer's cache)
};

// A wave's lanes over heads of the projection: head_dim / 8 lanes a head, 4 elements of either half a lane.
constexpr int PREPARE_LPH = DH / 8, PREPARE_HALF = DH / 2, PREPARE_HEADS = PREPARE_LPH > 0 ? TIE_WAVE / PREPARE_LPH : 1;

// 4 + 4 elements of a head as the projection's planes hold them: up to four planes asked for at once, whatever their
// number (a plane beyond the last is the last again, and not added), further ones when the sum is formed.
struct HeadPieces {
  qk_f4_t a[4], b[4];
  const float* at;
  __device__ __forceinline__ void ask(const float* head, const QkSource& src, int p0) {
    at = head + p0;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float* plane = at + static_cast<size_t>(min(s, src.planes - 1)) * src.plane_stride;
      a[s] = load4(plane);
      b[s] = load4(plane + PREPARE_HALF);
    }
  }
  __device__ __forceinline__ void sum(const QkSource& src, qk_f4_t& va, qk_f4_t& vb) const {
    va = a[0];
    vb = b[0];
#pragma unroll
    for (int s = 1; s < 4; ++s) {
      const bool there = s < src.planes;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        va[e] = there ? va[e] + a[s][e] : va[e];
        vb[e] = there ? vb[e] + b[s][e] : vb[e];
      }
    }
    for (int s = 4; s < src.planes; ++s) {
      va += load4(at + static_cast<size_t>(s) * src.plane_stride);
      vb += load4(at + static_cast<size_t>(s) * src.plane_stride + PREPARE_HALF);
    }
  }
};

// What a head meets: the norm's weights (ones where there is no norm, which then is left out) and the token's angles.
struct HeadFactors {
  qk_f4_t wa, wb;
  bool normed;
  __device__ __forceinline__ void ask(const float* weight, const float* any, int p0) {
    normed = weight != nullptr;
    const float* w = normed ? weight : any;     // something to read without a condition
    wa = load4(w + p0);
    wb = load4(w + PREPARE_HALF + p0);
  }
};

__device__ __forceinline__ void head_norm_rotate(qk_f4_t a, qk_f4_t b, const HeadFactors& f, float eps, qk_f4_t cs, qk_f4_t sn,
                                                 qk_f4_t& o1, qk_f4_t& o2) {
  if (f.normed) qk_head_norm_by<PREPARE_LPH>(a, b, f.wa, f.wb, eps);
  qk_rotate_by(a, b, cs, sn, o1, o2);
}

// The rest of a group's queries (more than PREPARE_HEADS heads), then all of them from LDS into operand layout.
__device__ __forceinline__ void rest_of_queries(const float* row, int head0, int G, int lane, const QkSource& src,
                                                const HeadFactors& f, qk_f4_t cs, qk_f4_t sn, bf16_t* q_lds,
                                                u32x4_t (&qf)[KSTEPS]) {
  const int p0 = (lane % PREPARE_LPH) * 4;
  for (int g0 = PREPARE_HEADS; g0 < G; g0 += PREPARE_HEADS) {
    const int g = g0 + lane / PREPARE_LPH;
    HeadPieces q;
    q.ask(row + (static_cast<size_t>(head0) + min(g, G - 1)) * DH, src, p0);
    qk_f4_t a, b, o1, o2;
    q.sum(src, a, b);
    head_norm_rotate(a, b, f, src.eps, cs, sn, o1, o2);
    if (g < G) {
      store4(q_lds + g * DH + p0, o1);
      store4(q_lds + g * DH + PREPARE_HALF + p0, o2);
    }
  }
  __syncthreads();   // one wave: the writes above are done before the reads below
  const int col = lane & 15, quad = lane >> 4;
#pragma unroll
  for (int st = 0; st < KSTEPS; ++st) {
    const int d = st * 32 + quad * 8;
    qf[st] = (col < G && d < DH) ? *reinterpret_cast<const u32x4_t*>(q_lds + col * DH + d) : u32x4_t{0, 0, 0, 0};
  }
}

// The newest token of a (sequence, KV head): lanes 0 .. LPH - 1 hold its key's elements, the next LPH lanes its value's.
// To the cache (position `off` of its page) and, as the cache will hold them, in bfloat16, to LDS.
__device__ __forceinline__ void store_newest(int lane, qk_f4_t a, qk_f4_t b, const HeadFactors& f, float eps, qk_f4_t cs,
                                             qk_f4_t sn, bf16_t* k_page, bf16_t* v_page, int off, int block_size,
                                             bf16_t* newest_lds) {
  const int p0 = (lane % PREPARE_LPH) * 4;
  qk_f4_t o1, o2;
  head_norm_rotate(a, b, f, eps, cs, sn, o1, o2);     // (shuffles stay within a head's lanes)
  if (lane < PREPARE_LPH) {
    bf16_t* dst = k_page + static_cast<size_t>(off) * DH;
    store4(newest_lds + p0, o1);
    store4(newest_lds + PREPARE_HALF + p0, o2);
    store4(dst + p0, o1);
    store4(dst + PREPARE_HALF + p0, o2);
  } else if (lane < 2 * PREPARE_LPH) {
    store4(newest_lds + DH + p0, a);
    store4(newest_lds + DH + PREPARE_HALF + p0, b);
    // In a page the dimensions of a value lie block_size apart.
    bf16_t* dst = v_page + off;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      store_from_float(dst + static_cast<size_t>(p0 + j) * block_size, a[j]);
      store_from_float(dst + static_cast<size_t>(PREPARE_HALF + p0 + j) * block_size, b[j]);
    }
  }
}

// The newest key by itself: its score for this lane's column from the 32 dimensions the lane holds of the
// query, summed over the four quads; then one step of the online softmax with a single key, the
// probability rounded to bfloat16 as the tiles' are.
template <bool CAPPED>
__device__ __forceinline__ void attend_newest(const bf16_t* newest_lds, const u32x4_t (&qf)[KSTEPS], floatx4 (&acc)[DTILES],
                                              float& m, float& l, int quad, float scale_log2e, float cap) {
  float dot = 0.f;
#pragma unroll
  for (int st = 0; st < KSTEPS; ++st) {
    const int d = st * 32 + quad * 8;
    if (DH % 32 == 0 || d < DH) {
      const u32x4_t kq = *reinterpret_cast<const u32x4_t*>(newest_lds + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        dot = fmaf(__uint_as_float(qf[st][e] << 16), __uint_as_float(kq[e] << 16), dot);
        dot = fmaf(__uint_as_float(qf[st][e] & 0xffff0000u), __uint_as_float(kq[e] & 0xffff0000u), dot);
      }
    }
  }
  dot += __shfl_xor(dot, 16, TIE_WAVE);
  dot += __shfl_xor(dot, 32, TIE_WAVE);
  if constexpr (CAPPED) dot = cap * tanh_fast(dot / cap);
  const float m_new = fmaxf(m, dot);
  const float neg_mc = -m_new * scale_log2e;
  const float corr = __builtin_amdgcn_exp2f(fmaf(m, scale_log2e, neg_mc));   // m = -inf: 0
  const float p = __builtin_amdgcn_exp2f(fmaf(dot, scale_log2e, neg_mc));
  const float p_rounded = __uint_as_float(pack_bf16x2(p, 0.f) << 16);
  l = l * corr + (quad == 0 ? p : 0.f);
  m = m_new;
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt) {
    const u32x2_t vv = *reinterpret_cast<const u32x2_t*>(newest_lds + DH + dt * 16 + quad * 4);
    acc[dt][0] = fmaf(p_rounded, __uint_as_float(vv.x << 16), acc[dt][0] * corr);
    acc[dt][1] = fmaf(p_rounded, __uint_as_float(vv.x & 0xffff0000u), acc[dt][1] * corr);
    acc[dt][2] = fmaf(p_rounded, __uint_as_float(vv.y << 16), acc[dt][2] * corr);
    acc[dt][3] = fmaf(p_rounded, __uint_as_float(vv.y & 0xffff0000u), acc[dt][3] * corr);
  }
}

// One wave: the newest token of sequence `place` and unit `unit` as a share of its own, the last of nsplit.
template <bool CAPPED>
__device__ __forceinline__ void attention_decode_newest(
    int lane, int unit, int place, bf16_t* k_cache, bf16_t* v_cache, float* __restrict__ part_o, float* __restrict__ part_ml,
    const int* __restrict__ query_start, const int* __restrict__ context_lens, const int* __restrict__ block_tables,
    const int* __restrict__ seq_ids, int H, int KVH, int block_size, int block_shift, int max_blocks, float scale_log2e,
    float cap, int nsplit, QkSource src, bf16_t* q_lds, bf16_t* newest_lds) {
  const int col = lane & 15, quad = lane >> 4;
  const int heads_per_kv = H / KVH;             // at most 16: a unit is a KV head
  const int kvh = unit, head0 = kvh * heads_per_kv, G = heads_per_kv;
  const int s = seq_ids ? seq_ids[place] : place;
  const int t = __builtin_amdgcn_readfirstlane(query_start[s]);
  const int pos = __builtin_amdgcn_readfirstlane(context_lens[s]) - 1;
  asm volatile("" ::"s"(t), "s"(pos));
  const int p0 = (lane % PREPARE_LPH) * 4, g_first = lane / PREPARE_LPH;
  const float* row = src.qkv + static_cast<size_t>(t) * src.in_row;
  const float* angles = src.angles + static_cast<size_t>(t) * DH;
  HeadPieces q, n;
  HeadFactors fq, fk;
  n.ask(row + static_cast<size_t>(H + kvh + ((g_first & 1) != 0 ? KVH : 0)) * DH, src, p0);
  q.ask(row + (static_cast<size_t>(head0) + min(g_first, G - 1)) * DH, src, p0);
  fq.ask(src.q_weight, angles, p0);
  fk.ask(src.k_weight, angles, p0);
  const qk_f4_t cs = load4(angles + p0), sn = load4(angles + PREPARE_HALF + p0);
  const int page = block_tables[static_cast<size_t>(s) * max_blocks + (pos >> block_shift)];
  qk_f4_t a, b, o1, o2;
  q.sum(src, a, b);
  head_norm_rotate(a, b, fq, src.eps, cs, sn, o1, o2);
  if (g_first < G) {
    store4(q_lds + g_first * DH + p0, o1);
    store4(q_lds + g_first * DH + PREPARE_HALF + p0, o2);
  }
  n.sum(src, a, b);
  const size_t at = (static_cast<size_t>(page) * KVH + kvh) * block_size * DH;
  store_newest(lane, a, b, fk, src.eps, cs, sn, k_cache + at, v_cache + at, pos & (block_size - 1), block_size, newest_lds);
  u32x4_t qf[KSTEPS];
  rest_of_queries(row, head0, G, lane, src, fq, cs, sn, q_lds, qf);
  floatx4 acc[DTILES];
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt) acc[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  attend_newest<CAPPED>(newest_lds, qf, acc, m, l, quad, scale_log2e, cap);
  l += __shfl_xor(l, 16, TIE_WAVE);
  l += __shfl_xor(l, 32, TIE_WAVE);
  if (col < G)
    store_share(acc, m, l, nullptr, part_o, part_ml, t, place, head0 + col, H, quad, nsplit, nsplit - 1, scale_log2e, nullptr);
}

// What the wave's lanes have read from and written to LDS so far comes before what follows, for the compiler as well.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

// One wave: share `share` of `shares` of the keys, (KV head, group of 16 heads) `unit`, sequence `place` of the launch.
// nsplit: the shares the merge takes, one more than `shares` where the newest token is one of its own. table_lds:
// TABLE_AHEAD ints of LDS, the wave's own; q_lds (16 DH) and newest_lds (2 DH) only where it prepares.
template <int DEPTH, DecodePrepare PREPARE, bool CAPPED, bool KEEPS = false>
__device__ __forceinline__ void attention_decode_ring_wave(
    int lane, int share, int shares, int unit, int place,
    const bf16_t* __restrict__ q, bf16_t* k_cache, bf16_t* v_cache,
    bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
    const int* __restrict__ query_start, const int* __restrict__ context_lens,
    const int* __restrict__ block_tables, const int* __restrict__ seq_ids, int H, int KVH, int block_size,
    int block_shift, int max_blocks, float scale_log2e, float cap, int window, int nsplit,
    const float* __restrict__ sinks, const int* __restrict__ share_tiles,
    QkSource src, int keep, int* table_lds, bf16_t* q_lds = nullptr, bf16_t* newest_lds = nullptr) {
  const int col = lane & 15;
  const int quad = lane >> 4;
  // Workgroups go to the eight XCDs in turn by their number, of which the share is the fastest part: with shares
  // of one length, where the later shares of most sequences are empty, share j is therefore given to another
  // workgroup of the sequence's eight from pair to pair, or a few XCDs would carry all the work.
  const int split = share_tiles != nullptr ? (share + unit + place) % shares : share;
  // More than 16 query heads a KV head run as several waves of up to 16 columns each: unit counts
  // (KV head, group of 16 heads).
  const int heads_per_kv = H / KVH;
  const int column_groups = (heads_per_kv + 15) / 16;
  const int kvh = unit / column_groups;
  const int head0 = kvh * heads_per_kv + (unit % column_groups) * 16;   // column 0's query head
  const int s = seq_ids ? seq_ids[place] : place;
  const int G = min(16, kvh * heads_per_kv + heads_per_kv - head0);                          // this wave's columns
  const int* table = block_tables + static_cast<size_t>(s) * max_blocks;
  // The wave's copy of the page table: entries table_first .. + TABLE_AHEAD - 1, moved on where a share goes further.
  int table_first = 0, table_ahead[TABLE_AHEAD / TIE_WAVE];
  // (lanes read what other lanes wrote: the hardware keeps the order of a wave's LDS accesses, the fences have the compiler
  // keep it too, here and where the copy moves on; they wait for nothing)
  auto keep_table = [&] {
#pragma unroll
    for (int j = 0; j < TABLE_AHEAD / TIE_WAVE; ++j) table_lds[j * TIE_WAVE + lane] = table_ahead[j];
    wave_lds_order();
  };
#pragma unroll
  for (int j = 0; j < TABLE_AHEAD / TIE_WAVE; ++j) table_ahead[j] = table[min(j * TIE_WAVE + lane, max_blocks - 1)];
  const int t = __builtin_amdgcn_readfirstlane(query_start[s]);
  const int context = __builtin_amdgcn_readfirstlane(context_lens[s]);
  const int named = __builtin_amdgcn_readfirstlane(*(share_tiles != nullptr ? share_tiles : query_start));
  asm volatile("" ::"s"(t), "s"(context), "s"(named));      // here, together, not each where it is first used
  keep_table();
  const int pos = context - 1;
  const int start = first_visible_key(pos, window);   // window < 0: chunks of -window
  const int named_tiles = share_tiles != nullptr ? named : 0;

  const int first_tile = start / 32;
  const int num_tiles = pos / 32 + 1;
  // A share is the shares-th part of this sequence's tiles, or, where the step names a length for all shares
  // (share_tiles, in tiles; sequences of very different lengths), that many tiles if it is more: a short sequence
  // then fills fewer shares, the others are empty (the merge gives them no weight), and every wave that works
  // walks about as many keys. Whatever the step names, the shares cover the sequence.
  const int per_split = max((num_tiles - first_tile + shares - 1) / shares, named_tiles);
  const int tile_begin = first_tile + split * per_split;
  const int tile_end = min(num_tiles, tile_begin + per_split);
  if (nsplit > 1 && tile_begin >= tile_end) {
    // An empty share leaves at once: a maximum of -inf gives it no weight, and the merge does not read the rest.
    if (quad == 0 && col < G) {
      const size_t slot = (static_cast<size_t>(place) * H + head0 + col) * nsplit + split;
      part_ml[slot * 2] = -INFINITY;
      part_ml[slot * 2 + 1] = 0.f;
    }
    return;
  }

  const size_t page_stride = static_cast<size_t>(KVH) * block_size * DH;
  const size_t head_off = static_cast<size_t>(kvh) * block_size * DH;
  // Where the step's newest token comes from the projection, the newest position is left out of the tiles.
  const bool own_token = PREPARE != PREPARE_NOTHING && src.write_kv;
  const int last_cached = own_token ? pos - 1 : pos;     // the newest position the tiles may show
  u32x4_t qf[KSTEPS];
  floatx4 acc[DTILES];
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt) acc[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  const int krow0 = (col >> 2) * 8 + (col & 3);
  const bool keys_in_upper_half = krow0 >= 16;      // both sub-tiles' rows (krow0, krow0 + 4) lie in one half
  const bool values_in_upper_half = quad >= 2;      // positions quad * 8 .. + 7
  const int in_page = block_size - 1;
  const size_t dim_off = static_cast<size_t>(col) * block_size;

  struct Tile { u32x4_t k[2][KSTEPS]; u32x4_t v[DTILES]; };
  auto reach = [&](int first, int last) {     // the copy holds entries first to last (two or three) from here on
    if (first >= table_first && last < table_first + TABLE_AHEAD) return;
    table_first = first;
#pragma unroll
    for (int j = 0; j < TABLE_AHEAD / TIE_WAVE; ++j)
      table_ahead[j] = table[min(table_first + j * TIE_WAVE + lane, max_blocks - 1)];
    wave_lds_order();
    keep_table();
  };
  auto page_of = [&](int entry) { return __builtin_amdgcn_readfirstlane(table_lds[entry - table_first]); };
  // Positions are clamped into [start, pos] for addresses only; a clamped position stays in its half of 16.
  auto issue_in = [&](int tile, Tile& tl, int lo, int hi) {
    const int base = tile * 32;
    const int entry_lo = min(max(base, lo), hi) >> block_shift, entry_hi = min(max(base + 16, lo), hi) >> block_shift;
    reach(entry_lo, entry_hi);
    const int page_lo = page_of(entry_lo), page_hi = page_of(entry_hi);
    const bf16_t* kpage = k_cache + static_cast<size_t>(keys_in_upper_half ? page_hi : page_lo) * page_stride + head_off;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int kp = min(max(base + krow0 + u * 4, lo), hi);
      const bf16_t* kr = kpage + static_cast<size_t>(kp & in_page) * DH;
#pragma unroll
      for (int st = 0; st < KSTEPS; ++st) {
        // Every load is issued whatever the lane (a load under a lane's condition makes the count of loads
        // in flight unknown to the compiler, which then waits for all of them): a head size that is no
        // multiple of 32 reads its last step's upper pieces from the row's start and drops them.
        const int d = st * 32 + quad * 8;
        const bool inside = DH % 32 == 0 || d < DH;
        const u32x4_t piece = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(kr + (inside ? d : 0)));
        tl.k[u][st] = inside ? piece : u32x4_t{0, 0, 0, 0};
      }
    }
    const int vp = min(max(base + quad * 8, lo / 8 * 8), hi / 8 * 8);
    const bf16_t* vr = v_cache + static_cast<size_t>(values_in_upper_half ? page_hi : page_lo) * page_stride + head_off +
                       (vp & in_page) + dim_off;
#pragma unroll
    for (int dt = 0; dt < DTILES; ++dt)
      tl.v[dt] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(vr + static_cast<size_t>(dt) * 16 * block_size));
  };
  auto issue = [&](int tile, Tile& tl) { issue_in(tile, tl, start, pos); };

  Tile ring[DEPTH];
  constexpr int FIRST = KEEPS ? DEPTH - 1 : DEPTH;     // the kept keys go through the last set first
  auto issue_first = [&] {
#pragma unroll
    for (int j = 0; j < FIRST; ++j) issue(min(tile_begin + j, tile_end - 1), ring[j]);
  };
  if constexpr (PREPARE == PREPARE_NOTHING) {
    const bool valid = col < G;
    const bf16_t* qr = q + (static_cast<size_t>(t) * H + head0 + (valid ? col : 0)) * DH;
#pragma unroll
    for (int st = 0; st < KSTEPS; ++st) {
      const int d = st * 32 + quad * 8;
      const bool inside = DH % 32 == 0 || d < DH;
      const u32x4_t piece = *reinterpret_cast<const u32x4_t*>(qr + (inside ? d : 0));
      qf[st] = (valid && inside) ? piece : u32x4_t{0, 0, 0, 0};
    }
    issue_first();
  } else {
    // The group's queries, PREPARE_HEADS heads at a time with a head's lanes together (lanes beyond the group read its
    // last head again), and in a wave that walks a whole sequence the newest key (the first head's lanes) and value.
    const float* row = src.qkv + static_cast<size_t>(t) * src.in_row;
    const float* angles = src.angles + static_cast<size_t>(t) * DH;
    const int p0 = (lane % PREPARE_LPH) * 4, g_first = lane / PREPARE_LPH;
    HeadPieces qp, np;
    HeadFactors fq, fk;
    qp.ask(row + (static_cast<size_t>(head0) + min(g_first, G - 1)) * DH, src, p0);
    fq.ask(src.q_weight, angles, p0);
    if constexpr (PREPARE == PREPARE_WHOLE) {
      // (also where the cache holds the token already, and its columns of the projection with it: read, not used)
      np.ask(row + static_cast<size_t>(H + kvh + ((g_first & 1) != 0 ? KVH : 0)) * DH, src, p0);
      fk.ask(src.k_weight, angles, p0);
    }
    const qk_f4_t cs = load4(angles + p0), sn = load4(angles + PREPARE_HALF + p0);
    issue_first();
    qk_f4_t a, b, o1, o2;
    qp.sum(src, a, b);
    head_norm_rotate(a, b, fq, src.eps, cs, sn, o1, o2);
    if (g_first < G) {
      store4(q_lds + g_first * DH + p0, o1);
      store4(q_lds + g_first * DH + PREPARE_HALF + p0, o2);
    }
    if constexpr (PREPARE == PREPARE_WHOLE) {
      if (own_token) {
        np.sum(src, a, b);
        reach(pos >> block_shift, pos >> block_shift);
        const size_t at = static_cast<size_t>(page_of(pos >> block_shift)) * page_stride + head_off;
        store_newest(lane, a, b, fk, src.eps, cs, sn, k_cache + at, v_cache + at, pos & in_page, block_size, newest_lds);
      }
    }
    rest_of_queries(row, head0, G, lane, src, fq, cs, sn, q_lds, qf);
  }
  if constexpr (KEEPS) {
    // The kept keys the window has left behind, by the first share's wave, through the ring's last set (the
    // first tiles' loads are on their way in the others).
    const int kept_last = min(keep, start) - 1;
    if (split == 0) {
      for (int kt = 0; kt * 32 <= kept_last; ++kt) {
        issue_in(kt, ring[DEPTH - 1], 0, kept_last);
        attend_tile<CAPPED>(ring[DEPTH - 1].k, ring[DEPTH - 1].v, qf, acc, m, l, kt * 32, 0, kept_last, quad,
                            scale_log2e, cap);
      }
    }
    issue(min(tile_begin + DEPTH - 1, tile_end - 1), ring[DEPTH - 1]);
  }
  // Tile i of the wave lives in set i % DEPTH, and the tile DEPTH further on is asked for as soon as its set is read.
  // The groups of DEPTH tiles in the middle compute and issue without a condition, so the compiler knows how many
  // loads are in flight and waits for the oldest tile only; the last 2 DEPTH - 1 at most after them are under
  // conditions, where it waits for more than it must.
  int tile = tile_begin;
  for (; tile + 2 * DEPTH - 1 < tile_end; tile += DEPTH) {
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      attend_tile<CAPPED>(ring[j].k, ring[j].v, qf, acc, m, l, (tile + j) * 32, start, last_cached, quad, scale_log2e, cap);
      issue(tile + j + DEPTH, ring[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < 2 * DEPTH - 1; ++j) {
    if (tile + j < tile_end) {
      attend_tile<CAPPED>(ring[j % DEPTH].k, ring[j % DEPTH].v, qf, acc, m, l, (tile + j) * 32, start, last_cached, quad,
                          scale_log2e, cap);
      if (j < DEPTH - 1 && tile + j + DEPTH < tile_end) issue(tile + j + DEPTH, ring[j]);
    }
  }
  if constexpr (PREPARE == PREPARE_WHOLE) {
    if (own_token) attend_newest<CAPPED>(newest_lds, qf, acc, m, l, quad, scale_log2e, cap);
  }
  l += __shfl_xor(l, 16, TIE_WAVE);
  l += __shfl_xor(l, 32, TIE_WAVE);
  if (col >= G) return;
  store_share(acc, m, l, out, part_o, part_ml, t, place, head0 + col, H, quad, nsplit, split, scale_log2e,
              sinks);
}
