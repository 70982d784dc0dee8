// Shared device helpers for the gfx950 kernels: element types, conversions,
// wave and block reductions. Every kernel file includes only this header.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

// Element type codes of the C interface.
#define TIE_F32 0
#define TIE_BF16 1
#define TIE_F16 2   // a cache of keys and values only (beside float32 arithmetic)

// Error codes of the C interface (besides hipError_t values, which are > 0).
#define TIE_OK 0
#define TIE_BAD_ARGUMENT (-1)

#define TIE_WAVE 64

typedef uint16_t bf16_t;  // raw bfloat16 bits
typedef _Float16 f16_t;   // IEEE half precision, converted by the hardware (round to nearest even)

__device__ __forceinline__ float bf16_to_float(bf16_t v) {
  return __uint_as_float(static_cast<uint32_t>(v) << 16);
}

// Round to nearest even; NaN stays NaN (quieted).
// Round to nearest even, NaN stays NaN: gfx950 converts in hardware (v_cvt_pk_bf16_f32).
typedef __bf16 tie_bf16x2_t __attribute__((ext_vector_type(2)));
typedef float tie_floatx2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  const tie_floatx2_t f = {lo, hi};
  const tie_bf16x2_t b = __builtin_convertvector(f, tie_bf16x2_t);
  return *reinterpret_cast<const uint32_t*>(&b);
}

__device__ __forceinline__ bf16_t float_to_bf16(float f) { return static_cast<bf16_t>(pack_bf16x2(f, 0.f) & 0xffffu); }

template <typename T>
__device__ __forceinline__ float load_as_float(const T* p);
template <>
__device__ __forceinline__ float load_as_float<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float load_as_float<bf16_t>(const bf16_t* p) { return bf16_to_float(*p); }

template <>
__device__ __forceinline__ float load_as_float<f16_t>(const f16_t* p) { return static_cast<float>(*p); }

template <typename T>
__device__ __forceinline__ void store_from_float(T* p, float v);
template <>
__device__ __forceinline__ void store_from_float<f16_t>(f16_t* p, float v) { *p = static_cast<f16_t>(v); }
template <>
__device__ __forceinline__ void store_from_float<float>(float* p, float v) { *p = v; }
template <>
__device__ __forceinline__ void store_from_float<bf16_t>(bf16_t* p, float v) { *p = float_to_bf16(v); }

// tanh(x) = 1 - 2 / (e^(2x) + 1) on the hardware's 2^x and reciprocal: absolute error of a few 1e-7, saturating
// at +-1 for large |x|. For the bfloat16 attention kernels' capped scores; float32 paths call tanhf.
__device__ __forceinline__ float tanh_fast(float x) {
  const float e = __builtin_amdgcn_exp2f(x * 2.88539008177792681472f);
  return 1.f - 2.f * __builtin_amdgcn_rcpf(e + 1.f);
}

// The tanh form of gelu, 0.5 z (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3))), with the library's tanhf (float32 paths)
// and with tanh_fast (epilogues of the bfloat16 products, whose results are rounded to 8 bits of mantissa anyway).
__device__ __forceinline__ float gelu_tanh_exact(float z) {
  return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}
__device__ __forceinline__ float gelu_tanh_fast(float z) {
  return 0.5f * z * (1.0f + tanh_fast(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// The first key a query at position pos reads: every key (0), the last `window` ones, or those of its own
// chunk of `chunk` positions counted from position 0 of the sequence. At most one of the two is positive.
__device__ __forceinline__ int first_visible_key(int pos, int window, int chunk) {
  if (window > 0) return max(0, pos - window + 1);
  if (chunk > 0) return pos - pos % chunk;
  return 0;
}

// The same with both in one number, as the matrix-core attention kernels carry it: span > 0 a window of span
// positions, span < 0 chunks of -span positions, 0 every key.
__device__ __forceinline__ int first_visible_key(int pos, int span) {
  if (span > 0) return max(0, pos - span + 1);
  if (span < 0) return pos - pos % (-span);
  return 0;
}

// A softmax with a sink: exp(sink) is one more term of the denominator, with no key and no value. Given the
// running maximum m_e of the keys' scores and the sink, both in the exponent's units (base 2), and the keys' sum l
// under that maximum, returns the factor that turns the unnormalised accumulator into the output.
__device__ __forceinline__ float sink_normaliser(float m_e, float l, float sink_e) {
  const float top = fmaxf(m_e, sink_e);
  const float f = exp2f(m_e - top);
  return f / (l * f + exp2f(sink_e - top));
}
#define TIE_LOG2E 1.44269504088896340736f

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = TIE_WAVE / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, TIE_WAVE);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = TIE_WAVE / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, TIE_WAVE));
  return v;
}

// Sum over a block of up to 1024 threads; `scratch` holds >= 16 floats of LDS.
// Every thread receives the total. The order of additions is fixed by the
// thread layout alone, so a row's sum does not depend on what else runs.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (TIE_WAVE - 1);
  const int wave = threadIdx.x / TIE_WAVE;
  const int waves = (blockDim.x + TIE_WAVE - 1) / TIE_WAVE;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < waves; ++w) total += scratch[w];
  return total;
}

__device__ __forceinline__ float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & (TIE_WAVE - 1);
  const int wave = threadIdx.x / TIE_WAVE;
  const int waves = (blockDim.x + TIE_WAVE - 1) / TIE_WAVE;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = scratch[0];
  for (int w = 1; w < waves; ++w) total = fmaxf(total, scratch[w]);
  return total;
}

// A launch as data: TIE_LIST_ENTRY(f) defines f_list, which calls the C function f with its arguments from an array of
// 64-bit words (pointers and whole numbers as they are, a float's bits in the lower half), so that launch_list.hip runs
// a layer's launches one after the other without a call from Python for each.
template <typename A>
static inline A tie_argument(uint64_t word) {
  if constexpr (std::is_pointer<A>::value) {
    return reinterpret_cast<A>(word);
  } else if constexpr (std::is_same<A, float>::value) {
    const uint32_t bits = static_cast<uint32_t>(word);
    float value;
    __builtin_memcpy(&value, &bits, sizeof(value));
    return value;
  } else {
    static_assert(std::is_integral<A>::value, "pointers, floats and whole numbers");
    return static_cast<A>(word);
  }
}

template <typename... A, size_t... I>
static inline int tie_call_words(int (*f)(A...), const uint64_t* words, std::index_sequence<I...>) {
  return f(tie_argument<A>(words[I])...);
}

template <typename... A>
static inline int tie_call_words(int (*f)(A...), const uint64_t* words) {
  return tie_call_words(f, words, std::index_sequence_for<A...>{});
}

#define TIE_LIST_ENTRY(f) \
  extern "C" int f##_list(const uint64_t* words) { return tie_call_words(&f, words); }

static inline int tie_launch_status() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? TIE_OK : static_cast<int>(e);
}

// Dispatch helpers: call `fn.template operator()<T>()` style lambdas are avoided;
// instead each launcher switches on the dtype codes explicitly.
