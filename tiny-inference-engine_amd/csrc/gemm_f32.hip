// The float32 matrix product for gfx950: out[M, N] (+)= x[M, K] . w[N, K]^T on v_mfma_f32_16x16x4_f32, whose
// products and sums are float32 (the same precision as multiply-adds on the vector units, at four times the rate a
// plain tile reached there). It carries the projections of the 32-bit path over few rows, gemm_f32_pieces those over many,
// gemm_f32_rows those of one to four (gemm_f32_plan.h chooses); operands of mixed types and rows that are no multiple of
// four floats go to gemm_generic, routed experts to moe_gemm_generic. Shape and ranges follow from the step's sizes: a
// row's sums in steps of other sizes agree to rounding, not bit for bit as the plain tile's do.
//
// A wave owns MT tiles of 16 rows of x and NT tiles of 16 rows of w over one range of K and walks it in blocks of 32 k,
// 2 KB of a tile: two 16-byte loads a lane, eight lanes on the 128 bytes of a row, one whole line. The matrix instruction
// wants rows side by side in lanes instead; loaded so, a load costs the vector cache about 65 cycles and not 16, which
// held 64 x 64 tiles to half of what the matrix cores give, and blocks of 16 k, half a line a row, held the stream of w
// to 3 to 4 TB/s (16 rows over a gated 12288 x 2048: 30.2 us, 22.0 in whole lines; 2560 x 9728 in eight ranges 32.2 and
// 21.3; 4096 x 2048 in two 10.5 and 8.6; 64 rows and more within 2 to 7 %). So a block passes through LDS, in a place of
// the wave's own: written as loaded, read by lane l at row l % 16 and floats 4 (l / 16) .. + 3 of either half, the places
// of a row's eight pieces exchanged by row % 8 so that neither way meets a bank twice. Four instructions take one of the
// four floats each - which k an instruction sums is a permutation that both operands share.
// The WK waves of a workgroup share one tile and cut its range of K between them, without a barrier on the way; their
// sums meet in LDS and are added in the order of the waves. Where tiles are too few for the chip, K is cut over
// workgroups as well and planes of partial sums are left for the consumer, who adds them in order. No atomics: every
// sum's order follows from the sizes.
//
// Few rows are bound by the stream of w (4 bytes a weight): U blocks a wave are asked for while it works on U others;
// many rows are bound by the matrix cores (157 TFLOP/s). Measured over 12288 x 2048: 8 rows 19.7 us (5.1 TB/s), 90 rows
// 55 us (82 TFLOP/s; 58.7 in blocks of 16 k). Straight from memory into the operand registers, without LDS, a prompt's
// products took a third longer. Against 64 bits a sum over 16 to 48 chains is off by half of what one chain is.
#include "common.h"
#include "gemm_f32_plan.h"

#include <math.h>

typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <bool STREAM>
__device__ __forceinline__ f32x4_t gf_load(const float* p) {
  if (STREAM) return __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(p));
  return *reinterpret_cast<const f32x4_t*>(p);
}

template <int MT, int NT, int WK, int U, bool STREAM>
__global__ __launch_bounds__(WK* TIE_WAVE) void gemm_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                float* __restrict__ out, int M, int N, int K,
                                                                int accumulate, int gated, int splits, int row_tiles) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int STAGED = 2 * U * (MT + NT), SUMS = MT * NT;  // pieces of 1 KB a wave holds in LDS on the way, at the end
  __shared__ f32x4_t lds[WK][STAGED > SUMS ? STAGED : SUMS][TIE_WAVE];
  // Workgroups go to the eight dies in turn. The row tiles of one piece of w follow each other on one die, so that w
  // comes from memory once and from that die's cache afterwards.
  const int turn = blockIdx.x / 8;
  const int unit = turn / row_tiles * 8 + blockIdx.x % 8;
  const int col_tiles = (N + 16 * NT - 1) / (16 * NT);
  if (unit >= col_tiles * splits) return;
  const int t0 = turn % row_tiles * (16 * MT);
  const int n0 = unit / splits * (16 * NT);
  const int split = unit % splits;

  const int lane = threadIdx.x & (TIE_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TIE_WAVE);
  const int row_in = lane / 8, piece_in = (lane % 8) ^ row_in;                   // what this lane loads of 8 rows of a block
  // Whose loaded piece it multiplies, in the block's first half of k and in its second.
  const int from = lane % 16 * 8, first = (lane / 16) ^ (lane % 8), second = first ^ 4;
  // A wave's range of K in whole blocks, or in halves of one where K is so short that waves would be left without any.
  const int halves = (K + 15) / 16;
  int per = (halves + splits * WK - 1) / (splits * WK);
  if (per > 1) per += per % 2;
  const int k0 = 16 * min(halves, (split * WK + wave) * per);
  const int k1 = min(K, k0 + 16 * per);
  const int blocks = (k1 - k0 + 31) / 32;

  // Rows beyond the operands' last are that row again: their sums are not stored.
  const float* wb = w + static_cast<size_t>(n0) * K;
  const float* xb = x + static_cast<size_t>(t0) * K;
  unsigned wo[NT][2], xo[MT][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int j = 0; j < NT; ++j) wo[j][h] = static_cast<unsigned>(min(16 * j + 8 * h + row_in, N - 1 - n0)) * static_cast<unsigned>(K);
#pragma unroll
    for (int m = 0; m < MT; ++m) xo[m][h] = static_cast<unsigned>(min(16 * m + 8 * h + row_in, M - 1 - t0)) * static_cast<unsigned>(K);
  }

  f32x4_t acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[m][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  f32x4_t aw[U][NT][2], ax[U][MT][2];    // what has been asked for
  auto ask = [&](int at) {               // blocks behind the range's end: its last one again
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned k = min(k0 + 32 * min(at + u, blocks - 1) + 4 * piece_in, K - 4);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < NT; ++j) aw[u][j][h] = gf_load<STREAM>(wb + (wo[j][h] + k));
#pragma unroll
        for (int m = 0; m < MT; ++m) ax[u][m][h] = gf_load<false>(xb + (xo[m][h] + k));
      }
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < NT; ++j) lds[wave][2 * (u * (MT + NT) + j) + h][lane] = aw[u][j][h];
#pragma unroll
        for (int m = 0; m < MT; ++m) lds[wave][2 * (u * (MT + NT) + NT + m) + h][lane] = ax[u][m][h];
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");     // the wave's own lanes only: nothing to wait for
  };
  auto multiply = [&](int u) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int at = from + (half == 0 ? first : second);
      f32x4_t bw[NT], bx[MT];
#pragma unroll
      for (int j = 0; j < NT; ++j) bw[j] = (&lds[wave][2 * (u * (MT + NT) + j)][0])[at];
#pragma unroll
      for (int m = 0; m < MT; ++m) bx[m] = (&lds[wave][2 * (u * (MT + NT) + NT + m)][0])[at];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bw[j][i], bx[m][i], acc[m][j], 0, 0, 0);
    }
  };

  // Whole batches of U whole blocks; the next batch's loads are in flight behind this one's instructions.
  const int whole = max(0, k1 - k0) / 32 / U;
  const int rest = whole * U;
  if (blocks > 0) ask(0);
  for (int b = 1; b <= whole; ++b) {
    stage();
    if (b * U < blocks) ask(b * U);
#pragma unroll
    for (int u = 0; u < U; ++u) multiply(u);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  if (rest < blocks) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k0 + 32 * (rest + u) + 4 * piece_in >= k1) {  // a range that ends inside a block: nothing from behind its end
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int j = 0; j < NT; ++j) aw[u][j][h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int m = 0; m < MT; ++m) ax[u][m][h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      }
    stage();
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (rest + u < blocks) multiply(u);
  }

  // Lane l of a tile's sums: row l % 16 of x, rows 4 (l / 16) .. + 3 of w.
  float* plane = out + static_cast<size_t>(split) * M * N;
  auto store = [&](int m, int j, int at, f32x4_t v) {
    const int t = t0 + 16 * m + at % 16;
    const int n = n0 + 16 * j + at / 16 * 4;
    if (t >= M || n >= N) return;
    float* o = plane + static_cast<size_t>(t) * N + n;
    if (N % 4 == 0) {
      f32x4_t* o4 = reinterpret_cast<f32x4_t*>(o);
      *o4 = accumulate ? *o4 + v : v;
    } else {
      for (int i = 0; i < 4 && n + i < N; ++i) o[i] = accumulate ? o[i] + v[i] : v[i];
    }
  };
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < NT; ++j) lds[wave][m * NT + j][lane] = acc[m][j];      // over the wave's own blocks
  __syncthreads();
  for (int tile = wave; tile < MT * NT; tile += WK) {
    f32x4_t v = lds[0][tile][lane];
#pragma unroll
    for (int k = 1; k < WK; ++k) v += lds[k][tile][lane];
    if (!gated) {
      store(tile / NT, tile % NT, lane, v);
      continue;
    }
    // A tile of w is 8 rows of gates and the 8 rows of ups that go with them: lane l holds gates 4 (l / 16) .. + 3 up to
    // lane 31, the ups of lane l - 32 from there on.
    f32x4_t up;
#pragma unroll
    for (int i = 0; i < 4; ++i) up[i] = __shfl_down(v[i], 32, TIE_WAVE);
    const int t = t0 + 16 * (tile / NT) + lane % 16;
    const int n = n0 + 16 * (tile % NT);
    if (lane >= 32 || t >= M || n >= N) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (gated == 1 ? v[i] / (1.0f + expf(-v[i])) : gelu_tanh_exact(v[i])) * up[i];
    *reinterpret_cast<f32x4_t*>(out + static_cast<size_t>(t) * (N / 2) + n / 2 + lane / 16 * 4) = v;
  }
#endif
}

// Ranges of K the product is best cut into when its caller adds planes of partial sums.
extern "C" int tie_gemm_f32_splits(int M, int N, int K) { return M > 0 && N > 0 && K > 0 ? gf_plan(M, N, K, 0).splits : 1; }

// The shape a product with so many ranges of K takes: 1 to 8 for tie_gemm_f32, 8 + 1 to 8 + 4 for tie_gemm_f32_pieces,
// -1 to -3 for tie_gemm_f32_rows.
extern "C" int tie_gemm_f32_shape(int M, int N, int K, int splits) {
  if (M <= 0 || N <= 0 || K <= 0 || splits <= 0) return 1;
  const GfPlan plan = gf_plan(M, N, K, 0);
  return (plan.splits == splits ? plan : gf_plan(M, N, K, splits)).shape + 1;
}

// splits > 1: out is [splits][M][N] planes of partial sums. gated 1 or 2: w's rows are 8 gates and 8 ups in turn, out is
// [M][N / 2] and receives silu(gate) * up or gelu_tanh(gate) * up. shape: entry shape - 1 of GF_SHAPES.
extern "C" int tie_gemm_f32(const float* x, const float* w, float* out, int accumulate, int gated, int M, int N, int K,
                            int splits, int shape, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K < 4 || K % 4 != 0 || K > (1 << 24) || splits < 1 || splits > GF_MAX_SPLITS ||
      (splits > 1 && accumulate) || shape < 1 || shape > GF_COUNT || gated < 0 || gated > 2 ||
      (gated && (accumulate || splits > 1 || N % 16 != 0)))
    return TIE_BAD_ARGUMENT;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) % 16 != 0)
    return TIE_BAD_ARGUMENT;
  const int chosen = shape - 1;
  const GfShape s = GF_SHAPES[chosen];
  const int row_tiles = (M + 16 * s.mt - 1) / (16 * s.mt);
  const long units = static_cast<long>((N + 16 * s.nt - 1) / (16 * s.nt)) * splits;
  const long grid = (units + 7) / 8 * 8 * row_tiles;
  if (grid > 0x7fffffffL) return TIE_BAD_ARGUMENT;
#define LAUNCH(MT, NT, WK, U, STREAM)                                                                            \
  gemm_f32_kernel<MT, NT, WK, U, STREAM><<<static_cast<unsigned>(grid), WK * TIE_WAVE, 0, stream>>>(             \
      x, w, out, M, N, K, accumulate, gated, splits, row_tiles)
  // One row tile: w is read once, past the caches. Several: from the die's cache behind the first (48 rows over 2048 x 6144
  // in eight ranges, tiles of 16 x 16: 41.6 us past the caches, 31.4 through them).
  const bool once = row_tiles == 1;
  switch (chosen) {
    case 0:
      if (once) LAUNCH(1, 1, 8, 2, true);
      else LAUNCH(1, 1, 8, 2, false);
      break;
    case 1:
      if (once) LAUNCH(1, 2, 8, 1, true);
      else LAUNCH(1, 2, 8, 1, false);
      break;
    case 2: LAUNCH(2, 1, 8, 1, false); break;
    case 3: LAUNCH(2, 2, 8, 1, false); break;
    case 4: LAUNCH(3, 2, 4, 1, false); break;
    case 5: LAUNCH(2, 4, 4, 1, false); break;
    case 6: LAUNCH(3, 4, 4, 1, false); break;
    case 7: LAUNCH(4, 4, 4, 1, false); break;
    default: return TIE_BAD_ARGUMENT;
  }
#undef LAUNCH
  return tie_launch_status();
}

// What a launch list may hold (common.h).
TIE_LIST_ENTRY(tie_gemm_f32)
