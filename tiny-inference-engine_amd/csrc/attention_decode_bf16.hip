// Paged attention for decoded tokens (one new row per sequence) on the gfx950 matrix cores,
// bfloat16 queries and cache, float32 softmax. Compiled per head size: -DHEAD_DIM=<multiple of 16>.
//
// One wave handles one (sequence, KV head, split of the keys). The G = H / KVH query heads that
// share the KV head are the 16 columns of the MFMA tiles (columns >= G are zeros), so keys and
// values are read once for the whole group; more than 16 heads a KV head are several waves of up to
// 16 columns each. Per 32 keys:
//
//   S^T[key, g] = K[key, :] . Q[g, :]      A = K rows (16 bytes a lane, straight from the cache),
//                                          B = Q (held in registers)          2 x HEAD_DIM/32 MFMAs
//   online softmax per column g in float32: running maximum, sum, rescale of the accumulator
//   O^T[d, g]  += V^T[d, key] . P^T[key, g]   A = V^T rows (the cache keeps values transposed inside a
//                                          page, so 8 positions of one dimension are 16 bytes),
//                                          B = P, which is exactly what the lane already holds
//                                          from the first product              HEAD_DIM/16 MFMAs
//
// Nothing passes through LDS and no lane ever needs another lane's scores. Splits of the keys
// run as separate waves; a second kernel merges their (maximum, sum, accumulator) triples in a
// fixed order. Keys are always cut at multiples of 32 positions, so what is computed for a
// position does not depend on the batch around it. Block-table lookups run two tiles ahead of the
// arithmetic and the data loads one tile ahead, so neither waits for the other.
//
// Formula: src/backend/cpu/cpu_backend.cpp:261-319 (score = scale * q.k, causal by position,
// online softmax, query head h reads KV head h / (H / KVH)).
#include "common.h"

#include <math.h>

#ifndef HEAD_DIM
#error "compile with -DHEAD_DIM=<head size>"
#endif
static_assert(HEAD_DIM % 16 == 0 && HEAD_DIM >= 16 && HEAD_DIM <= 256, "head size must be a multiple of 16 up to 256");

constexpr int DH = HEAD_DIM;
#include "attention_decode_ring.h"

// Keys of a 32-key tile are taken in runs of 8: row r of 16-key sub-tile u is key (r / 4) * 8 + u * 4 + r % 4
// of the tile. The scores a lane then holds (rows quad * 4 + v of both sub-tiles) are those of the 8
// consecutive keys quad * 8 .. + 7, which is also how the values of one dimension lie in a page: with
// WIDE (block sizes in steps of 8) a lane reads them in one 16-byte piece.
// KEEPS: beside a window the keys of positions below `keep` are read as well, at their true positions. The wave
// of the first share walks those the window has left behind, [0, min(keep, start)), tile by tile before its own
// tiles, with addresses clamped into that range (the pages between it and the window may be gone).
template <bool WIDE, bool CAPPED, bool KEEPS = false>
__global__ __launch_bounds__(TIE_WAVE) void attention_decode_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
    const int* __restrict__ query_start, const int* __restrict__ context_lens,
    const int* __restrict__ block_tables, const int* __restrict__ seq_ids, int H, int KVH, int block_size,
    int block_shift, int max_blocks, float scale_log2e, float cap, int window, int nsplit,
    const float* __restrict__ sinks, int keep) {
  const int lane = threadIdx.x;
  const int col = lane & 15;   // query head within the group (column of every tile)
  const int quad = lane >> 4;  // 0..3
  const int split = blockIdx.x;
  // More than 16 query heads a KV head run as several waves of up to 16 columns each: blockIdx.y counts
  // (KV head, group of 16 heads).
  const int heads_per_kv = H / KVH;
  const int column_groups = (heads_per_kv + 15) / 16;
  const int kvh = static_cast<int>(blockIdx.y) / column_groups;
  const int head0 = kvh * heads_per_kv + (static_cast<int>(blockIdx.y) % column_groups) * 16;   // column 0's query head
  const int s = seq_ids ? seq_ids[blockIdx.z] : blockIdx.z;
  const int G = min(16, kvh * heads_per_kv + heads_per_kv - head0);                          // this wave's columns
  const int t = query_start[s];            // the sequence's single new row
  const int pos = context_lens[s] - 1;     // its position; keys start..pos are read
  const int start = first_visible_key(pos, window);   // window < 0: chunks of -window
  const int* table = block_tables + static_cast<size_t>(s) * max_blocks;

  // Tiles of 32 keys at absolute positions; this split's share of them.
  const int first_tile = start / 32;
  const int num_tiles = pos / 32 + 1;
  const int per_split = (num_tiles - first_tile + nsplit - 1) / nsplit;
  const int tile_begin = first_tile + split * per_split;
  const int tile_end = min(num_tiles, tile_begin + per_split);

  // Q as the B operand: lane (col = g, quad) holds Q[g][step*32 + quad*8 .. +8].
  u32x4_t qf[KSTEPS];
  {
    const bool valid = col < G;
    const bf16_t* qr = q + (static_cast<size_t>(t) * H + head0 + (valid ? col : 0)) * DH;
#pragma unroll
    for (int st = 0; st < KSTEPS; ++st) {
      const int d = st * 32 + quad * 8;
      qf[st] = (valid && d < DH) ? *reinterpret_cast<const u32x4_t*>(qr + d) : u32x4_t{0, 0, 0, 0};
    }
  }

  floatx4 acc[DTILES];
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt) acc[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  const size_t page_stride = static_cast<size_t>(KVH) * block_size * DH;   // elements of one page, K or V
  const size_t head_off = static_cast<size_t>(kvh) * block_size * DH;
  // Positions are clamped into [start, pos] for addresses only (pages outside that range may be gone or
  // never have been there); what lies outside is masked in the softmax.
  auto page_of = [&](int kp) { return kp >> block_shift; };          // block sizes are powers of two here
  auto offset_of = [&](int kp) { return kp & (block_size - 1); };
  // This lane's keys of a tile: rows of the two sub-tiles, and the runs of values it reads.
  const int krow0 = (col >> 2) * 8 + (col & 3);        // sub-tile 1: + 4
  constexpr int VG = WIDE ? 8 : 4;

  // Pages first, one tile further ahead than the data, so that no data load waits for a lookup.
  struct Pages { int k[2]; int v[WIDE ? 1 : 2]; };
  auto lookup_in = [&](int base, Pages& pg, int lo, int hi) {
#pragma unroll
    for (int u = 0; u < 2; ++u) pg.k[u] = table[page_of(min(max(base + krow0 + u * 4, lo), hi))];
#pragma unroll
    for (int j = 0; j < (WIDE ? 1 : 2); ++j)
      pg.v[j] = table[page_of(min(max(base + quad * 8 + j * 4, lo / VG * VG), hi / VG * VG))];
  };
  auto lookup = [&](int base, Pages& pg) { lookup_in(base, pg, start, pos); };
  auto load_keys_in = [&](int base, const Pages& pg, u32x4_t (&kf)[2][KSTEPS], int lo, int hi) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int kp = min(max(base + krow0 + u * 4, lo), hi);
      const bf16_t* kr = k_cache + static_cast<size_t>(pg.k[u]) * page_stride + head_off +
                         static_cast<size_t>(offset_of(kp)) * DH;
#pragma unroll
      for (int st = 0; st < KSTEPS; ++st) {
        const int d = st * 32 + quad * 8;
        kf[u][st] = d < DH ? __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(kr + d)) : u32x4_t{0, 0, 0, 0};
      }
    }
  };
  auto load_keys = [&](int base, const Pages& pg, u32x4_t (&kf)[2][KSTEPS]) { load_keys_in(base, pg, kf, start, pos); };
  auto load_values_in = [&](int base, const Pages& pg, u32x4_t (&vf)[DTILES], int lo, int hi) {
    const bf16_t* vp[WIDE ? 1 : 2];
#pragma unroll
    for (int j = 0; j < (WIDE ? 1 : 2); ++j) {
      const int kp = min(max(base + quad * 8 + j * 4, lo / VG * VG), hi / VG * VG);
      vp[j] = v_cache + static_cast<size_t>(pg.v[j]) * page_stride + head_off + offset_of(kp);
    }
#pragma unroll
    for (int dt = 0; dt < DTILES; ++dt) {
      const size_t d_off = static_cast<size_t>(dt * 16 + col) * block_size;
      if (WIDE) {
        vf[dt] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(vp[0] + d_off));
      } else {
        const u32x2_t h0 = *reinterpret_cast<const u32x2_t*>(vp[0] + d_off);
        const u32x2_t h1 = *reinterpret_cast<const u32x2_t*>(vp[WIDE ? 0 : 1] + d_off);
        vf[dt] = u32x4_t{h0.x, h0.y, h1.x, h1.y};
      }
    }
  };
  auto load_values = [&](int base, const Pages& pg, u32x4_t (&vf)[DTILES]) { load_values_in(base, pg, vf, start, pos); };

  // The loads of tile t + 1 are issued before the arithmetic of tile t, so memory latency and the
  // matrix cores overlap; the pages of tile t + 2 are looked up at the same time.
  u32x4_t kf[2][KSTEPS], vf[DTILES], kf_next[2][KSTEPS], vf_next[DTILES];
  Pages pages;
  if constexpr (KEEPS) {
    const int kept_last = min(keep, start) - 1;     // the kept keys before the window: 0 .. kept_last
    if (split == 0) {
      for (int base = 0; base <= kept_last; base += 32) {
        lookup_in(base, pages, 0, kept_last);
        load_keys_in(base, pages, kf, 0, kept_last);
        load_values_in(base, pages, vf, 0, kept_last);
        attend_tile<CAPPED>(kf, vf, qf, acc, m, l, base, 0, kept_last, quad, scale_log2e, cap);
      }
    }
  }
  if (tile_begin < tile_end) {
    lookup(tile_begin * 32, pages);
    load_keys(tile_begin * 32, pages, kf_next);
    load_values(tile_begin * 32, pages, vf_next);
    if (tile_begin + 1 < tile_end) lookup(tile_begin * 32 + 32, pages);
  }
  for (int tile = tile_begin; tile < tile_end; ++tile) {
    const int base = tile * 32;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int st = 0; st < KSTEPS; ++st) kf[u][st] = kf_next[u][st];
#pragma unroll
    for (int dt = 0; dt < DTILES; ++dt) vf[dt] = vf_next[dt];
    if (tile + 1 < tile_end) {
      load_keys(base + 32, pages, kf_next);
      load_values(base + 32, pages, vf_next);
      if (tile + 2 < tile_end) lookup(base + 64, pages);
    }
    attend_tile<CAPPED>(kf, vf, qf, acc, m, l, base, start, pos, quad, scale_log2e, cap);
  }

  // The column's sum over all keys of this split.
  l += __shfl_xor(l, 16, TIE_WAVE);
  l += __shfl_xor(l, 32, TIE_WAVE);
  if (col >= G) return;
  store_share(acc, m, l, out, part_o, part_ml, t, blockIdx.z, head0 + col, H, quad, nsplit, split, scale_log2e,
              sinks);
}

// The most register sets of the ring: a set holds a tile's 32 keys and values, DH / 2 registers, and beside them stand the
// accumulators (DH / 4), the queries (DH / 8) and some 60 more, 512 in all. Sets that do not fit go through scratch memory
// on every tile (heads of 256, 64 sequences of 94 to 1500 keys: whole sequences in four sets 375 us a layer and in two 87,
// shares of 17 tiles in three sets 106 and in two 92), and the compiler has been seen to lose the fourth register of a
// piece of 16 bytes that it had put away in two parts: wrong results.
constexpr int RING_DEPTH = DH <= 160 ? 4 : (DH <= 224 ? 3 : 2);

// One wave a workgroup; shares are the fastest part of its number. Newest tokens that are shares of their own come
// behind all others (places from num_seqs on), as they are short: between the others they would shift which compute
// units carry one wave more (8 sequences of 8 KV heads and 4090 keys, 512 long waves and 64 short ones: 4 % of a step).
template <int DEPTH, DecodePrepare PREPARE, bool CAPPED, bool KEEPS = false>
__global__ __launch_bounds__(TIE_WAVE) void attention_decode_ring_kernel(
    const int* __restrict__ query_start, const int* __restrict__ context_lens,
    const int* __restrict__ block_tables, const int* __restrict__ seq_ids, int max_blocks, int num_seqs, int window, int nsplit,
    int H, int KVH,
    const bf16_t* __restrict__ q, bf16_t* k_cache, bf16_t* v_cache,
    bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml, int block_size,
    int block_shift, float scale_log2e, float cap,
    const float* __restrict__ sinks, const int* __restrict__ share_tiles, QkSource src, int keep) {
  constexpr bool PREPARES = PREPARE != PREPARE_NOTHING;
  __shared__ int table_lds[TABLE_AHEAD];
  __shared__ __attribute__((aligned(16))) bf16_t q_lds[PREPARES ? 16 * DH : 8], newest_lds[PREPARES ? 2 * DH : 8];
  const int lane = threadIdx.x;
  if constexpr (PREPARE == PREPARE_SHARES) {
    if (static_cast<int>(blockIdx.z) >= num_seqs) {
      const int units = gridDim.y;
      const int at = ((static_cast<int>(blockIdx.z) - num_seqs) * units + static_cast<int>(blockIdx.y)) *
                         static_cast<int>(gridDim.x) + static_cast<int>(blockIdx.x);
      if (at < units * num_seqs)
        attention_decode_newest<CAPPED>(lane, at % units, at / units, k_cache, v_cache, part_o, part_ml, query_start,
                                        context_lens, block_tables, seq_ids, H, KVH, block_size, block_shift, max_blocks,
                                        scale_log2e, cap, nsplit, src, q_lds, newest_lds);
      return;
    }
  }
  attention_decode_ring_wave<DEPTH, PREPARE, CAPPED, KEEPS>(
      lane, static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x), static_cast<int>(blockIdx.y),
      static_cast<int>(blockIdx.z), q, k_cache, v_cache, out, part_o, part_ml, query_start, context_lens, block_tables, seq_ids,
      H, KVH, block_size, block_shift, max_blocks, scale_log2e, cap, window, nsplit, sinks, share_tiles, src, keep, table_lds,
      q_lds, newest_lds);
}

#include "attention_merge.h"

extern "C" int tie_attention_decode_head_dim() { return DH; }
extern "C" int tie_attention_max_splits() { return MERGE_MAX_SPLITS; }

constexpr bool PREPARE_HEAD_DIM = DH == 32 || DH == 64 || DH == 128 || DH == 256;

static int launch_decode(const bf16_t* q, const QkSource* src, bf16_t* k_cache, bf16_t* v_cache, bf16_t* out,
                         float* part_o, float* part_ml, const int* query_start, const int* context_lens,
                         const int* block_tables, const int* seq_ids, int num_seqs, int H, int KVH, int block_size,
                         int max_blocks, float scale, float softcap, int window, int nsplit, const int* share_tiles,
                         int depth, const float* sinks, hipStream_t stream, int keep = 0) {
  // kept first positions go beside a window, with uncapped scores and queries that come ready
  if (keep < 0 || (keep > 0 && (window <= 0 || softcap > 0.f || src != nullptr))) return TIE_BAD_ARGUMENT;
  const int column_groups = KVH > 0 ? (H / KVH + 15) / 16 : 1;    // waves of up to 16 query heads a KV head
  if (num_seqs <= 0 || num_seqs > 65535 || H <= 0 || KVH <= 0 || KVH * column_groups > 65535 || H % KVH != 0 ||
      (src != nullptr && H / KVH > 16) ||
      block_size < 4 || (block_size & (block_size - 1)) != 0 || max_blocks <= 0 || nsplit <= 0 ||
      nsplit > MERGE_MAX_SPLITS || depth < 0 || depth > 4 || (depth > 1 && block_size < 16) ||
      !(scale > 0.f))   // the running maximum is kept on unscaled scores
    return TIE_BAD_ARGUMENT;
  if (nsplit > 1 && (part_o == nullptr || part_ml == nullptr)) return TIE_BAD_ARGUMENT;
  // Measured: the ring of three register sets where the keys are cut into shares, of four where a wave walks
  // a whole sequence.
  if (depth == 0) depth = block_size < 16 ? 1 : (nsplit == 1 ? 4 : 3);
  if (depth > RING_DEPTH) depth = RING_DEPTH;
  if (src != nullptr && (depth < 2 || !PREPARE_HEAD_DIM)) return TIE_BAD_ARGUMENT;
  if (share_tiles != nullptr && (depth < 2 || nsplit == 1)) return TIE_BAD_ARGUMENT;   // the ring kernel's, with a merge
  const dim3 grid(nsplit, KVH * column_groups, num_seqs);
  // A prepared step whose newest tokens are shares of their own: the grid holds the other shares, then those, of as many
  // sequences as fit its third dimension (two places a sequence at most).
  const bool newest_alone = src != nullptr && src->write_kv && nsplit > 1;
  const int tile_shares = newest_alone ? nsplit - 1 : nsplit;      // the ring kernel's `shares`
  constexpr int SEQS_AT_ONCE = 32767;
  const int block_shift = __builtin_ctz(block_size);
  const float scale_log2e = scale * 1.44269504088896340736f;
  const float cap = softcap > 0.f ? softcap / scale : 0.f;   // softcap * tanh(scale s / softcap) = scale * cap tanh(s / cap)
#define RING_ARGS query_start, context_lens, block_tables, seq_ids, max_blocks, num_seqs, window, nsplit, H, KVH, q, k_cache, \
                  v_cache, out, part_o, part_ml, block_size, block_shift, scale_log2e, cap, sinks, share_tiles
  // Capped scores are an instantiation of their own: the uncapped kernels carry none of it.
#define LAUNCH_RING(DEPTH)                                                                                               \
  {                                                                                                                      \
    if (keep > 0) {                                                                                                      \
      attention_decode_ring_kernel<DEPTH, PREPARE_NOTHING, false, true><<<grid, TIE_WAVE, 0, stream>>>(RING_ARGS, QkSource{}, keep); \
    } else if (src == nullptr && cap > 0.f) {                                                                            \
      attention_decode_ring_kernel<DEPTH, PREPARE_NOTHING, true><<<grid, TIE_WAVE, 0, stream>>>(RING_ARGS, QkSource{}, 0); \
    } else if (src == nullptr) {                                                                                         \
      attention_decode_ring_kernel<DEPTH, PREPARE_NOTHING, false><<<grid, TIE_WAVE, 0, stream>>>(RING_ARGS, QkSource{}, 0); \
    } else if constexpr (PREPARE_HEAD_DIM) {                                                                             \
      if (nsplit > 1)                                                                                                    \
        for (int first = 0; first < num_seqs; first += SEQS_AT_ONCE) {                                                   \
          const int count = num_seqs - first < SEQS_AT_ONCE ? num_seqs - first : SEQS_AT_ONCE, at = seq_ids ? 0 : first; \
          const size_t slot = static_cast<size_t>(first) * H * nsplit;                                                   \
          attention_decode_ring_kernel<DEPTH, PREPARE_SHARES, false>                                                     \
              <<<dim3(tile_shares, KVH, count + (newest_alone ? (count + tile_shares - 1) / tile_shares : 0)), TIE_WAVE, 0, stream>>>( \
                  query_start + at, context_lens + at, block_tables + static_cast<size_t>(at) * max_blocks,              \
                  seq_ids ? seq_ids + first : nullptr, max_blocks, count, window, nsplit, H, KVH, q, k_cache, v_cache,   \
                  out, part_o + slot * DH, part_ml + slot * 2, block_size, block_shift, scale_log2e, cap, sinks,         \
                  share_tiles, *src, 0);                                                                                 \
        }                                                                                                                \
      else                                                                                                               \
        attention_decode_ring_kernel<DEPTH, PREPARE_WHOLE, false><<<grid, TIE_WAVE, 0, stream>>>(RING_ARGS, *src, 0);    \
    }                                                                                                                    \
  }
#define ARGS out, part_o, part_ml, query_start, context_lens, block_tables, seq_ids, H, KVH, block_size, block_shift, \
             max_blocks, scale_log2e, cap, window, nsplit, sinks
#define LAUNCH_PLAIN(WIDE)                                                                                   \
  {                                                                                                          \
    if (keep > 0)                                                                                            \
      attention_decode_kernel<WIDE, false, true><<<grid, TIE_WAVE, 0, stream>>>(q, k_cache, v_cache, ARGS, keep); \
    else if (cap > 0.f) attention_decode_kernel<WIDE, true><<<grid, TIE_WAVE, 0, stream>>>(q, k_cache, v_cache, ARGS, 0); \
    else attention_decode_kernel<WIDE, false><<<grid, TIE_WAVE, 0, stream>>>(q, k_cache, v_cache, ARGS, 0);  \
  }
  if (src != nullptr && cap > 0.f) return TIE_BAD_ARGUMENT;   // the kernel that makes its own queries caps nothing
  if (depth == 4) LAUNCH_RING((RING_DEPTH < 4 ? RING_DEPTH : 4))
  else if (depth == 3) LAUNCH_RING((RING_DEPTH < 3 ? RING_DEPTH : 3))
  else if (depth == 2) LAUNCH_RING(2)
  else if (block_size % 8 == 0) LAUNCH_PLAIN(true)
  else LAUNCH_PLAIN(false)
#undef LAUNCH_PLAIN
#undef LAUNCH_RING
#undef RING_ARGS
#undef ARGS
  int status = tie_launch_status();
  if (status != TIE_OK || nsplit == 1) return status;
  launch_attention_merge(part_o, part_ml, out, nullptr, query_start, seq_ids, H, nsplit, num_seqs, sinks, stream);
  return tie_launch_status();
}

// depth: 0 = by the rule, 1 = the kernel that looks its pages up per lane (any page size), 2 to 4 = the ring
// kernel with that many register sets, or as many as fit (RING_DEPTH; pages of 16 positions or more); for tests and sweeps.
// share_tiles (or null): one int on the device, the tiles of 32 keys of a share where the sequences' lengths differ
// much (the ring kernel and more than one share only; 0 there means shares by each sequence's own length).
// chunk > 0 (then window must be 0): a query reads the keys of its own chunk of that many positions, counted from
// position 0. sinks (or null): one float a query head whose exponential joins the head's softmax denominator.
// keep > 0 (beside a window, with uncapped scores): the keys of positions below keep are read as well.
extern "C" int tie_attention_decode_bf16_keeping(const void* q, const void* k_cache, const void* v_cache, void* out,
                                                 float* part_o, float* part_ml, const int* query_start,
                                                 const int* context_lens, const int* block_tables, const int* seq_ids,
                                                 int num_seqs, int H, int KVH, int block_size, int max_blocks,
                                                 float scale, float softcap, int window, int nsplit,
                                                 const int* share_tiles, int depth, int chunk, const float* sinks,
                                                 int keep, hipStream_t stream) {
  if (window < 0 || chunk < 0 || (window > 0 && chunk > 0)) return TIE_BAD_ARGUMENT;
  if (chunk > 0) window = -chunk;
  return launch_decode(static_cast<const bf16_t*>(q), nullptr, static_cast<bf16_t*>(const_cast<void*>(k_cache)),
                       static_cast<bf16_t*>(const_cast<void*>(v_cache)), static_cast<bf16_t*>(out), part_o, part_ml,
                       query_start, context_lens, block_tables, seq_ids, num_seqs, H, KVH, block_size, max_blocks,
                       scale, softcap, window, nsplit, share_tiles, depth, sinks, stream, keep);
}

extern "C" int tie_attention_decode_bf16_with(const void* q, const void* k_cache, const void* v_cache, void* out,
                                              float* part_o, float* part_ml, const int* query_start,
                                              const int* context_lens, const int* block_tables, const int* seq_ids,
                                              int num_seqs, int H, int KVH, int block_size, int max_blocks,
                                              float scale, float softcap, int window, int nsplit,
                                              const int* share_tiles, int depth, int chunk, const float* sinks,
                                              hipStream_t stream) {
  return tie_attention_decode_bf16_keeping(q, k_cache, v_cache, out, part_o, part_ml, query_start, context_lens,
                                           block_tables, seq_ids, num_seqs, H, KVH, block_size, max_blocks, scale,
                                           softcap, window, nsplit, share_tiles, depth, chunk, sinks, 0, stream);
}

// The same for a step of single decoded tokens whose queries, newest keys and values still lie in the QKV
// projection's output: qkv is float32 [planes][rows][in_row] (plane p at qkv + p * plane_stride; a row holds H
// query heads, KVH key heads, KVH value heads), summed over the planes by the kernel; q_weight / k_weight (or
// null) the per-head RMS norm weights with eps; angles [rows][head_dim] the step's table of cos and sin.
// write_kv = 0 where the cache is another layer's and holds the token already. Where it is written and nsplit > 1, the
// newest token is a share of its own, the last: the cached keys are cut into nsplit - 1. Pages of 16 positions or more
// and head sizes 32, 64, 128, 256; refused otherwise (tie_attention_decode_prepares tells).
extern "C" int tie_attention_decode_prepares(int block_size) { return PREPARE_HEAD_DIM && block_size >= 16 ? 1 : 0; }

extern "C" int tie_attention_decode_prepared_bf16(const float* qkv, long plane_stride, int planes, int in_row,
                                                  const float* q_weight, const float* k_weight, float eps,
                                                  const float* angles, int write_kv, void* k_cache, void* v_cache,
                                                  void* out, float* part_o, float* part_ml, const int* query_start,
                                                  const int* context_lens, const int* block_tables,
                                                  const int* seq_ids, int num_seqs, int H, int KVH, int block_size,
                                                  int max_blocks, float scale, int window, int nsplit,
                                                  const int* share_tiles, int depth, hipStream_t stream) {
  if (qkv == nullptr || angles == nullptr || planes < 1 || planes > 8 || plane_stride < 0 || block_size < 16 ||
      depth == 1 || H <= 0 || KVH <= 0 || in_row < (H + 2 * KVH) * DH || in_row % 4 != 0 || plane_stride % 4 != 0 ||
      reinterpret_cast<uintptr_t>(qkv) % 16 != 0 || reinterpret_cast<uintptr_t>(angles) % 16 != 0 ||
      reinterpret_cast<uintptr_t>(q_weight) % 16 != 0 || reinterpret_cast<uintptr_t>(k_weight) % 16 != 0 ||
      reinterpret_cast<uintptr_t>(k_cache) % 16 != 0)
    return TIE_BAD_ARGUMENT;
  const QkSource src = {qkv, static_cast<size_t>(plane_stride), planes, in_row, q_weight, k_weight, eps, angles, write_kv};
  return launch_decode(nullptr, &src, static_cast<bf16_t*>(k_cache), static_cast<bf16_t*>(v_cache),
                       static_cast<bf16_t*>(out), part_o, part_ml, query_start, context_lens, block_tables, seq_ids,
                       num_seqs, H, KVH, block_size, max_blocks, scale, 0.f, window, nsplit, share_tiles, depth, nullptr, stream);
}

extern "C" int tie_attention_decode_bf16(const void* q, const void* k_cache, const void* v_cache, void* out,
                                         float* part_o, float* part_ml, const int* query_start,
                                         const int* context_lens, const int* block_tables, const int* seq_ids,
                                         int num_seqs, int H, int KVH, int block_size, int max_blocks, float scale,
                                         float softcap, int window, int nsplit, hipStream_t stream) {
  return tie_attention_decode_bf16_with(q, k_cache, v_cache, out, part_o, part_ml, query_start, context_lens,
                                        block_tables, seq_ids, num_seqs, H, KVH, block_size, max_blocks, scale, softcap,
                                        window, nsplit, nullptr, 0, 0, nullptr, stream);
}

// What a launch list may hold (common.h).
TIE_LIST_ENTRY(tie_attention_decode_bf16)
TIE_LIST_ENTRY(tie_attention_decode_prepared_bf16)
TIE_LIST_ENTRY(tie_attention_decode_bf16_with)
TIE_LIST_ENTRY(tie_attention_decode_bf16_keeping)
