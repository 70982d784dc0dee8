// Paged causal attention in float32 on the matrix cores (v_mfma_f32_16x16x4_f32: float32 products and sums), for
// prompt portions and decoded tokens alike, over float32, bfloat16 or float16 pages. Head sizes in steps of 16 up to
// 256, pages in steps of 16 positions; other sizes, and kept first positions, go to attention_generic, whose rules of
// masks, chunks, caps and sinks these are.
//
// A workgroup owns 16 columns (query rows of one sequence times the query heads that share a KV head) and one KV head;
// its W waves take the tiles of 16 keys in turn, each with a running maximum, sum and accumulator of its own, and meet
// in LDS at the end, pairs first, in a fixed order. Everything a tile needs goes from memory to the operand registers:
//   S^T = K Q^T   lane (r, c) = (lane % 16, lane / 16) holds key r's dimensions 16 j + 4 c .. + 3 and column r's; its
//                 sums are column r's scores for keys 4 c .. 4 c + 3
//   O^T = V^T P^T the weights are those sums in place: instruction i takes keys 4 c + i, for which a page, whose values
//                 lie transposed, holds 16 consecutive bytes a dimension
// so a tile of 16 keys and a head size of 128 is 16 loads and 64 instructions of 32 cycles, without LDS or barriers.
// Bound by latency at the sizes the 32-bit path sees: four sequences of 600 keys, 16 heads over 8, take 11.1 us with the
// merge (in two shares of the keys 16.5; one workgroup a row and head, key by key, took 150), a prompt of 301 tokens 17.7
// (463). A workgroup of eight waves of 211 registers fills a compute unit.
// Keys are cut into shares over workgroups where the columns alone leave the chip idle; a second kernel merges them.
// Key tiles are cut at multiples of 16 positions: what is computed for a position does not depend on pages, on other
// sequences or on the cutting into steps, beyond rounding (shares and waves follow from the step's sizes).
#include "common.h"

#include <math.h>

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t af_load4(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }
__device__ __forceinline__ f32x4_t af_load4(const bf16_t* p) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  return f32x4_t{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                 __uint_as_float(v.y & 0xffff0000u)};
}
__device__ __forceinline__ f32x4_t af_load4(const f16_t* p) {
  typedef f16_t f16x4_t __attribute__((ext_vector_type(4)));
  const f16x4_t v = *reinterpret_cast<const f16x4_t*>(p);
  return f32x4_t{static_cast<float>(v[0]), static_cast<float>(v[1]), static_cast<float>(v[2]), static_cast<float>(v[3])};
}

__device__ __forceinline__ bool af_finite(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }

// e^(a - b) with e^(-inf - -inf) = 0: a share without a key weighs nothing.
__device__ __forceinline__ float af_weight(float a, float b) { return a == -INFINITY ? 0.f : expf(a - b); }

// Column tiles of a sequence with n new rows, `rows` of them a tile.
__device__ __forceinline__ int af_tiles(int n, int rows) { return (n + rows - 1) / rows; }

template <int DT, int W, typename TC>
__global__ __launch_bounds__(W* TIE_WAVE) void attention_f32_kernel(
    const float* __restrict__ q, const TC* __restrict__ k_cache, const TC* __restrict__ v_cache,
    float* __restrict__ out, const int* __restrict__ query_start, const int* __restrict__ context_lens,
    const int* __restrict__ block_tables, int T, int S, int H, int KVH, int block_size, int max_blocks, float scale,
    float softcap, int window, int chunk, const float* __restrict__ sinks, int nsplit, float* __restrict__ part_o,
    float* __restrict__ part_ml) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int DH = DT * 16;
  __shared__ f32x4_t acc_s[W / 2][DT][TIE_WAVE];
  __shared__ float ml_s[W / 2][2][16];
  const int lane = threadIdx.x & (TIE_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TIE_WAVE);
  const int r = lane % 16, c = lane / 16;
  const int group = H / KVH;
  const int kvh = blockIdx.x % KVH;
  const int head_tile = blockIdx.x / KVH;                    // more than one only where group > 16
  const int heads = min(16, group - 16 * head_tile);         // query heads of a row in this tile
  const int rows = group <= 16 ? 16 / group : 1;             // query rows of a tile

  // The sequence of this column tile: tiles are counted sequence by sequence. The last ones start first: a portion's late
  // rows see the most keys, and what a second round of workgroups gets should be short (a prompt of 301 tokens, 304
  // workgroups of which 256 run at once, 23.3 -> 17.7 us; 400 tokens 29.9 -> 24.4).
  const int column_tile = static_cast<int>(gridDim.y - 1 - blockIdx.y);
  int s = column_tile, first_row = 0;
  if (T != S) {
    int before = 0;
    s = -1;
    for (int base = 0; base < S && s < 0; base += TIE_WAVE) {
      const int mine = base + lane < S ? af_tiles(query_start[base + lane + 1] - query_start[base + lane], rows) : 0;
      int upto = mine;
#pragma unroll
      for (int off = 1; off < TIE_WAVE; off <<= 1) {
        const int v = __shfl_up(upto, off, TIE_WAVE);
        if (lane >= off) upto += v;
      }
      const unsigned long long past = __ballot(before + upto > column_tile);
      if (past != 0) {
        const int at = __ffsll(static_cast<long long>(past)) - 1;
        s = base + at;
        first_row = (column_tile - before - (__shfl(upto, at, TIE_WAVE) - __shfl(mine, at, TIE_WAVE))) * rows;
      }
      before += __shfl(upto, TIE_WAVE - 1, TIE_WAVE);
    }
    if (s < 0) return;          // a grid larger than the tiles there are
  }
  s = __builtin_amdgcn_readfirstlane(s);
  first_row = __builtin_amdgcn_readfirstlane(first_row);
  const int* table = block_tables + static_cast<size_t>(s) * max_blocks;
  // The table's first entries come with the lengths, so that the first tile of a short context is not asked for a trip
  // to memory later.
  const int table_ahead = table[min(lane, max_blocks - 1)];
  const int start_row = query_start[s];
  const int n_new = query_start[s + 1] - start_row;
  const int cached = context_lens[s] - n_new;                // row i sits at position cached + i
  const int last_row = min(first_row + rows, n_new) - 1;
  const int row = first_row + r / heads;
  const bool valid = r < rows * heads && row <= last_row;
  const int my_row = valid ? row : first_row;
  const int my_head = kvh * group + 16 * head_tile + (valid ? r % heads : 0);
  const int pos = cached + my_row;
  const int start = first_visible_key(pos, window, chunk);

  // Key tiles of 16 this workgroup's share holds, wave by wave in turn.
  const int tile_lo = first_visible_key(cached + first_row, window, chunk) / 16;
  const int tile_hi = (cached + last_row) / 16 + 1;
  const int full_from = first_visible_key(cached + last_row, window, chunk);   // keys from here to ...
  const int full_to = cached + first_row;                                      // ... here: every column sees them
  const int share = (tile_hi - tile_lo + nsplit - 1) / nsplit;
  const int lo = tile_lo + static_cast<int>(blockIdx.z) * share;
  const int hi = min(tile_hi, lo + share);

  f32x4_t qf[DT];
  const float* qr = q + (static_cast<size_t>(start_row + my_row) * H + my_head) * DH + 4 * c;
#pragma unroll
  for (int j = 0; j < DT; ++j) qf[j] = af_load4(qr + 16 * j);

  f32x4_t acc[DT];
#pragma unroll
  for (int j = 0; j < DT; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;       // l: the sum over this lane's keys

  f32x4_t kf[DT], vf[DT];
  const unsigned key_at = r * DH + 4 * c, value_at = r * block_size + 4 * c;      // this lane's place in a tile
  auto page_of = [&](int tile) { return table[tile * 16 / block_size]; };
  auto ask_keys = [&](int tile, int page) {
    const TC* p = k_cache + ((static_cast<size_t>(page) * KVH + kvh) * block_size + tile * 16 % block_size) * DH;
#pragma unroll
    for (int j = 0; j < DT; ++j) kf[j] = af_load4(p + (key_at + 16 * j));
  };
  // A tile of page `page`. With NEXT the keys of this wave's tile behind it, of page `next_page`, are asked for as soon as
  // this one's are read. Two instantiations and not a condition: behind one the compiler does not know how many loads
  // are younger than the values it waits for, and waits for the next keys too.
  auto step = [&](int tile, int page, int next_page, auto has_next) {
    constexpr bool NEXT = decltype(has_next)::value;
    const TC* vp = v_cache + (static_cast<size_t>(page) * KVH + kvh) * DH * block_size + tile * 16 % block_size;
#pragma unroll
    for (int j = 0; j < DT; ++j) vf[j] = af_load4(vp + 16 * j * block_size + value_at);
    f32x4_t sc = {0.f, 0.f, 0.f, 0.f};
    f32x4_t sc2 = {0.f, 0.f, 0.f, 0.f};       // two chains: an instruction need not wait for the one before it
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i % 2 == 0) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][i], qf[j][i], sc, 0, 0, 0);
        else sc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][i], qf[j][i], sc2, 0, 0, 0);
      }
    if constexpr (NEXT) ask_keys(tile + W, next_page);
    const int key0 = tile * 16 + 4 * c;
    const bool partly = tile * 16 < full_from || tile * 16 + 15 > full_to;      // some column does not see some key
    float p[4];
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = scale * (sc[i] + sc2[i]);
      if (softcap > 0.f) v = softcap * tanhf(v / softcap);
      if (partly && (key0 + i < start || key0 + i > pos)) v = -INFINITY;
      p[i] = v;
      top = fmaxf(top, v);
    }
    top = fmaxf(top, __shfl_xor(top, 16, TIE_WAVE));
    top = fmaxf(top, __shfl_xor(top, 32, TIE_WAVE));
    const float m_new = fmaxf(m, top);
    if (__any(m_new > m)) {
      const float corr = af_weight(m, m_new);
      l *= corr;
#pragma unroll
      for (int j = 0; j < DT; ++j) acc[j] *= corr;
    }
    m = m_new;
    float own = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = p[i] == -INFINITY ? 0.f : expf(p[i] - m);      // hidden, or a score of -inf: no weight, also where m is -inf
      own += p[i];
    }
    l += own;
    bool plain = true;
    if (partly) {
      // A weight of zero does not silence an infinity or a NaN: values of keys behind the last column's position are
      // not there yet, and where a key that only some columns see holds one, the tile goes key by key.
      bool odd = false;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < DT; ++j) {
          if (key0 + i > cached + last_row) vf[j][i] = 0.f;
          odd = odd || !af_finite(vf[j][i]);
        }
      plain = !__any(odd);
    }
    if (plain) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < DT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[j][i], p[i], acc[j], 0, 0, 0);
    } else {
#pragma unroll
      for (int j = 0; j < DT; ++j) {
#pragma unroll 1
        for (int key = 0; key < 16; ++key) {
          const float own_p = key % 4 == 0 ? p[0] : key % 4 == 1 ? p[1] : key % 4 == 2 ? p[2] : p[3];
          const float pk = __shfl(own_p, r + 16 * (key / 4), TIE_WAVE);
          const int at = tile * 16 + key;
          if (at < start || at > pos) continue;
          unsigned one = 4 * c * block_size;
          asm volatile("" : "+v"(one));      // worked out here, not kept in registers through the whole walk
#pragma unroll
          for (int i = 0; i < 4; ++i)
            acc[j][i] = fmaf(pk, load_as_float(vp + (16 * j + i) * block_size + key + one), acc[j][i]);
        }
      }
    }
  };
  int tile = lo + wave;
  if (tile < hi) {
    const int entry = tile * 16 / block_size;
    int page = entry < TIE_WAVE ? __builtin_amdgcn_readlane(table_ahead, entry) : table[entry];
    ask_keys(tile, page);
    while (tile + W < hi) {
      const int next_page = page_of(tile + W);
      step(tile, page, next_page, std::true_type{});
      page = next_page;
      tile += W;
    }
    step(tile, page, 0, std::false_type{});
  }
  l += __shfl_xor(l, 16, TIE_WAVE);
  l += __shfl_xor(l, 32, TIE_WAVE);

  // The waves' shares meet: the upper half hands over to the lower, until one is left.
#pragma unroll
  for (int half = W / 2; half >= 1; half /= 2) {
    if (wave >= half && wave < 2 * half) {
#pragma unroll
      for (int j = 0; j < DT; ++j) acc_s[wave - half][j][lane] = acc[j];
      if (c == 0) {
        ml_s[wave - half][0][r] = m;
        ml_s[wave - half][1][r] = l;
      }
    }
    __syncthreads();
    if (wave < half) {
      const float m2 = ml_s[wave][0][r], l2 = ml_s[wave][1][r];
      const float m_new = fmaxf(m, m2);
      const float f1 = af_weight(m, m_new), f2 = af_weight(m2, m_new);
      l = l * f1 + l2 * f2;
#pragma unroll
      for (int j = 0; j < DT; ++j) acc[j] = acc[j] * f1 + acc_s[wave][j][lane] * f2;
      m = m_new;
    }
    __syncthreads();
  }
  if (wave != 0 || !valid) return;
  const size_t where = static_cast<size_t>(start_row + my_row) * H + my_head;
  if (nsplit > 1) {
    const size_t slot = where * nsplit + blockIdx.z;
    if (c == 0) {
      part_ml[slot * 2] = m;
      part_ml[slot * 2 + 1] = l;
    }
#pragma unroll
    for (int j = 0; j < DT; ++j) *reinterpret_cast<f32x4_t*>(part_o + slot * DH + 16 * j + 4 * c) = acc[j];
    return;
  }
  if (sinks != nullptr) {              // one more term of the denominator, under the same maximum
    const float sink = sinks[my_head];
    const float m_new = fmaxf(m, sink);
    const float f = af_weight(m, m_new);
    l = l * f + expf(sink - m_new);
#pragma unroll
    for (int j = 0; j < DT; ++j) acc[j] *= f;
  }
#pragma unroll
  for (int j = 0; j < DT; ++j) *reinterpret_cast<f32x4_t*>(out + where * DH + 16 * j + 4 * c) = acc[j] / l;
#endif
}

// One wave a (row, head): its shares' maxima and sums, four dimensions a lane, in the order of the shares. The first
// AHEAD shares' accumulators are asked for together with the maxima and sums: one trip to memory (four rows of 16 heads
// in 5 shares: 3.9 us with a trip a share).
template <int AHEAD>
__global__ __launch_bounds__(TIE_WAVE) void attention_f32_merge_kernel(const float* __restrict__ part_o,
                                                                       const float* __restrict__ part_ml,
                                                                       float* __restrict__ out, int H, int Dh, int nsplit,
                                                                       const float* __restrict__ sinks) {
  const size_t where = static_cast<size_t>(blockIdx.y) * H + blockIdx.x;
  const int lane = threadIdx.x;
  const float* ml = part_ml + where * nsplit * 2;
  const float mine = lane < nsplit ? ml[2 * lane] : -INFINITY;
  const float sum = lane < nsplit ? ml[2 * lane + 1] : 0.f;
  const int d = 4 * lane;                       // head sizes up to 256
  const float* po = part_o + where * nsplit * Dh + (d < Dh ? d : 0);
  f32x4_t ahead[AHEAD];
#pragma unroll
  for (int k = 0; k < AHEAD; ++k) ahead[k] = af_load4(po + min(k, nsplit - 1) * Dh);
  const float sink = sinks != nullptr ? sinks[blockIdx.x] : -INFINITY;
  const float m = fmaxf(wave_max(mine), sink);
  const float weight = af_weight(mine, m);
  float l = af_weight(sink, m);
  for (int k = 0; k < nsplit; ++k) l += __shfl(weight, k, TIE_WAVE) * __shfl(sum, k, TIE_WAVE);
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < AHEAD; ++k)
    if (k < nsplit) o += ahead[k] * __shfl(weight, k, TIE_WAVE);
#pragma unroll 8
  for (int k = AHEAD; k < nsplit; ++k) o += af_load4(po + k * Dh) * __shfl(weight, k, TIE_WAVE);
  if (d < Dh) *reinterpret_cast<f32x4_t*>(out + where * Dh + d) = o / l;
}

// Column tiles: one a sequence in steps of single tokens, otherwise counted by the caller, who knows the sequences'
// rows (a count too large is harmless). nsplit > 1: part_o [T * H * nsplit * Dh], part_ml [T * H * nsplit * 2].
extern "C" int tie_attention_f32(const float* q, const void* k_cache, const void* v_cache, int cache_dtype, float* out,
                                 const int* query_start, const int* context_lens, const int* block_tables, int tiles, int T,
                                 int S, int H, int KVH, int Dh, int block_size, int max_blocks, float scale, float softcap,
                                 int window, int chunk, const float* sinks, int nsplit, float* part_o, float* part_ml,
                                 hipStream_t stream) {
  if (T <= 0 || T > 65535 || S <= 0 || S > T || tiles <= 0 || tiles > 65535 || H <= 0 || KVH <= 0 || H % KVH != 0 ||
      Dh < 16 || Dh > 256 || Dh % 16 != 0 || block_size <= 0 || block_size % 16 != 0 || max_blocks <= 0 ||
      (window > 0 && chunk > 0) || nsplit < 1 || nsplit > TIE_WAVE || (nsplit > 1 && (part_o == nullptr || part_ml == nullptr)))
    return TIE_BAD_ARGUMENT;
  if (T == S && tiles != S) return TIE_BAD_ARGUMENT;
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(k_cache) |
       reinterpret_cast<uintptr_t>(v_cache) | reinterpret_cast<uintptr_t>(part_o)) % 16 != 0)
    return TIE_BAD_ARGUMENT;
  const int head_tiles = (H / KVH + 15) / 16;
  const dim3 grid(KVH * head_tiles, tiles, nsplit);
#define LAUNCH(DT, W, TC)                                                                                              \
  attention_f32_kernel<DT, W, TC><<<grid, W * TIE_WAVE, 0, stream>>>(                                                   \
      q, static_cast<const TC*>(k_cache), static_cast<const TC*>(v_cache), out, query_start, context_lens, block_tables, \
      T, S, H, KVH, block_size, max_blocks, scale, softcap, window, chunk, sinks, nsplit, part_o, part_ml)
#define BY_TYPE(DT, W)                                              \
  do {                                                              \
    if (cache_dtype == TIE_F32) LAUNCH(DT, W, float);               \
    else if (cache_dtype == TIE_BF16) LAUNCH(DT, W, bf16_t);        \
    else if (cache_dtype == TIE_F16) LAUNCH(DT, W, f16_t);          \
    else return TIE_BAD_ARGUMENT;                                   \
  } while (0)
  switch (Dh / 16) {
    case 1: BY_TYPE(1, 8); break;
    case 2: BY_TYPE(2, 8); break;
    case 3: BY_TYPE(3, 8); break;
    case 4: BY_TYPE(4, 8); break;
    case 5: BY_TYPE(5, 8); break;
    case 6: BY_TYPE(6, 8); break;
    case 7: BY_TYPE(7, 8); break;
    case 8: BY_TYPE(8, 8); break;
    case 9: BY_TYPE(9, 4); break;
    case 10: BY_TYPE(10, 4); break;
    case 11: BY_TYPE(11, 4); break;
    case 12: BY_TYPE(12, 4); break;
    case 13: BY_TYPE(13, 4); break;
    case 14: BY_TYPE(14, 4); break;
    case 15: BY_TYPE(15, 4); break;
    default: BY_TYPE(16, 4); break;
  }
#undef BY_TYPE
#undef LAUNCH
  int status = tie_launch_status();
  if (status != TIE_OK || nsplit == 1) return status;
  const dim3 pairs(H, T);
  if (nsplit <= 4) attention_f32_merge_kernel<4><<<pairs, TIE_WAVE, 0, stream>>>(part_o, part_ml, out, H, Dh, nsplit, sinks);
  else if (nsplit <= 8) attention_f32_merge_kernel<8><<<pairs, TIE_WAVE, 0, stream>>>(part_o, part_ml, out, H, Dh, nsplit, sinks);
  else attention_f32_merge_kernel<24><<<pairs, TIE_WAVE, 0, stream>>>(part_o, part_ml, out, H, Dh, nsplit, sinks);
  return tie_launch_status();
}

// What a launch list may hold (common.h).
TIE_LIST_ENTRY(tie_attention_f32)
