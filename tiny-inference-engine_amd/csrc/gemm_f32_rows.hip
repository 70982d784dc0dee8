// The float32 product for one to four rows, gfx950: out[M, N] (+)= x[M, K] . w[N, K]^T on ordinary multiply-adds. So few rows are bound by the stream of w, 4 bytes a weight, and here nothing stands in its way: a load is
// 1 KB of one row of w, w goes from memory to the registers that multiply it, without LDS, and x is read for the rows there
// are, where the matrix instructions (gemm_f32.hip) take 16.
//
// A wave owns ROWS rows of w (four; eight where there are three and four rows of x, which halves what x costs) over one
// range of K and walks it in chunks of 256 k, lane l the floats 4 l .. + 3 of each, of w as of x; DEPTH chunks are in flight
// behind the one that is multiplied. So a sum of K products is 64 sums of every 64th four, added over the lanes at the end
// (half of the values change hands at each step), then over the waves that cut K between them, in LDS, in their order. No
// planes: a product is whole in one launch, and every sum's order follows from the sizes. Against 64 bits a sum is off by
// half to two thirds of what the matrix instructions' longer chains are.
//
// Measured, one row and four, with the best of the float32 matrix instructions beside it: a gated 12288 x 2048 18.6 us and
// 19.1 (20.3 and 18.9), 151936 x 2048 175 (7.1 TB/s) and 186 (183 and 180), 4096 x 4096 13.5 and 13.9 (13.7 and 12.9).
// Three and four chunks a batch gained nothing over a wave's 2 to 10
// (registers, and waves, against it); at eight rows x outweighs w (23.5 us, 19.7). Built and slower: the RMS norms' work in
// this kernel's ends, as the bfloat16 decode product does it (four rows, a step of 28 layers: 2189 -> 2317 us, though
// 55 norm kernels of 3.3 us go: the stream read behind the sums and the sums of squares ahead of them cost more).
#include "common.h"
#include "gemm_f32_plan.h"

#include <math.h>

typedef float f32x4_t __attribute__((ext_vector_type(4)));

static_assert(GR_CHUNK == 4 * TIE_WAVE, "a load of a wave");

template <int MT, int ROWS, int DEPTH>
__global__ __launch_bounds__(4 * TIE_WAVE) void gemm_f32_rows_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                     float* __restrict__ out, int M, int N, int K,
                                                                     int accumulate, int gated, int wk) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int HALF = ROWS / 2;
  constexpr int SUMS = ROWS * MT, LANES = TIE_WAVE / SUMS;       // lanes that end with the same sum
  __shared__ float lds[4][SUMS];
  const int lane = threadIdx.x & (TIE_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TIE_WAVE);
  const int part = wave % wk;
  const int groups = (N + ROWS - 1) / ROWS;
  const int asked = blockIdx.x * (static_cast<int>(blockDim.x / TIE_WAVE) / wk) + wave / wk;
  const int group = min(asked, groups - 1);            // beyond the last one: its sums again, not stored
  // Gated: half of them gates, half the ups that go with them, eight rows further on.
  const float* wr[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int row = gated ? group / (16 / ROWS) * 16 + group % (16 / ROWS) * HALF + r % HALF + r / HALF * 8 : min(group * ROWS + r, N - 1);
    wr[r] = w + static_cast<size_t>(row) * K;
  }
  const float* xr[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) xr[m] = x + static_cast<size_t>(min(m, M - 1)) * K;

  const int chunks = (K + GR_CHUNK - 1) / GR_CHUNK;
  const int per = (chunks + wk - 1) / wk;
  const int begin = min(chunks, part * per);
  const int end = min(chunks, begin + per);

  float acc[SUMS];
#pragma unroll
  for (int i = 0; i < SUMS; ++i) acc[i] = 0.f;
  f32x4_t rw[DEPTH][ROWS], rx[DEPTH][MT];
  auto ask = [&](int j, int chunk) {     // behind the range's end: its last chunk again; behind a row's end: its last piece
    const unsigned k = min(min(chunk, end - 1) * GR_CHUNK + 4 * lane, K - 4);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) rw[j][r] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(wr[r] + k));
#pragma unroll
    for (int m = 0; m < MT; ++m) rx[j][m] = *reinterpret_cast<const f32x4_t*>(xr[m] + k);
  };
  auto multiply = [&](int j) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < ROWS; ++r) acc[m * ROWS + r] = fmaf(rw[j][r][i], rx[j][m][i], acc[m * ROWS + r]);
  };
  if (begin < end) {
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) ask(j, begin + j);
    int chunk = begin;
    for (; chunk + DEPTH < end; chunk += DEPTH) {
#pragma unroll
      for (int j = 0; j < DEPTH; ++j) {
        multiply(j);
        ask(j, chunk + DEPTH + j);
      }
    }
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      if ((chunk + j) * GR_CHUNK + 4 * lane >= K) {      // nothing from behind a row's end
#pragma unroll
        for (int r = 0; r < ROWS; ++r) rw[j][r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < MT; ++m) rx[j][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
      if (chunk + j < end) multiply(j);
    }
  }

  // The lanes' sums: half of the values change hands at each step, until lane l has value l / LANES.
#pragma unroll
  for (int n = SUMS / 2, across = TIE_WAVE / 2; across > 0; n /= 2, across /= 2) {
    const bool upper = (lane & across) != 0;
    if (n > 0) {
#pragma unroll
      for (int i = 0; i < n; ++i) {
        const float keep = upper ? acc[i + n] : acc[i], give = upper ? acc[i] : acc[i + n];
        acc[i] = keep + __shfl_xor(give, across, TIE_WAVE);
      }
    } else {
      acc[0] += __shfl_xor(acc[0], across, TIE_WAVE);
    }
  }
  if (lane % LANES == 0) lds[wave][lane / LANES] = acc[0];
  __syncthreads();
  if (part != 0 || lane >= SUMS || asked >= groups) return;
  float v = lds[wave][lane];
  for (int k = 1; k < wk; ++k) v += lds[wave + k][lane];
  const int m = lane / ROWS, r = lane % ROWS;
  if (gated) {
    const float up = __shfl_down(v, HALF, TIE_WAVE);
    if (m >= M || r >= HALF) return;
    v = (gated == 1 ? v / (1.0f + expf(-v)) : gelu_tanh_exact(v)) * up;
    out[static_cast<size_t>(m) * (N / 2) + group * HALF + r] = v;
    return;
  }
  const int n = group * ROWS + r;
  if (m >= M || n >= N) return;
  float* o = out + static_cast<size_t>(m) * N + n;
  *o = accumulate ? *o + v : v;
#endif
}

// gated 1 or 2: w's rows are 8 gates and 8 ups in turn, out is [M][N / 2] and receives silu(gate) * up or gelu_tanh(gate) * up.
// shape: entry shape - 1 of GR_SHAPES.
extern "C" int tie_gemm_f32_rows(const float* x, const float* w, float* out, int accumulate, int gated, int M, int N, int K,
                                 int shape, hipStream_t stream) {
  if (M <= 0 || M > GR_MAX_ROWS || N <= 0 || K < 4 || K % 4 != 0 || K > (1 << 24) || shape < 1 || shape > GR_COUNT ||
      gated < 0 || gated > 2 || (gated && (accumulate || N % 16 != 0)))
    return TIE_BAD_ARGUMENT;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) % 16 != 0)
    return TIE_BAD_ARGUMENT;
  const int wk = GR_SHAPES[shape - 1];
  const int side = wk == 2 ? 2 : 1;                        // groups of rows a workgroup takes
  const int rows = M <= 2 ? 4 : 8;
  const int groups = (N + rows - 1) / rows;
  const unsigned grid = static_cast<unsigned>((groups + side - 1) / side);
#define LAUNCH(MT, ROWS) \
  gemm_f32_rows_kernel<MT, ROWS, GR_DEPTH><<<grid, side * wk * TIE_WAVE, 0, stream>>>(x, w, out, M, N, K, accumulate, gated, wk)
  if (M == 1) LAUNCH(1, 4);
  else if (M == 2) LAUNCH(2, 4);
  else LAUNCH(4, 8);
#undef LAUNCH
  return tie_launch_status();
}

// What a launch list may hold (common.h).
TIE_LIST_ENTRY(tie_gemm_f32_rows)
