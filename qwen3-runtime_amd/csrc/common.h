// Shared declarations of the HIP library (gfx950, wave64).
//
// Every entry point is extern "C", takes raw device pointers plus sizes and a
// stream, validates what it can on the host, launches on that stream and
// returns 0, or a negative code after recording a message that
// qrt_last_error() returns. Nothing here allocates device memory.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16_t;
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

#define QRT_WAVE 64

// dtype codes shared with the Python side
#define QRT_F32 0
#define QRT_BF16 1

extern "C" const char* qrt_last_error();
int qrt_fail(const char* fmt, ...);

#define QRT_CHECK(cond, ...)                 \
  do {                                       \
    if (!(cond)) return qrt_fail(__VA_ARGS__); \
  } while (0)

#define QRT_LAUNCH_CHECK(name)                                                     \
  do {                                                                             \
    hipError_t e_ = hipGetLastError();                                             \
    if (e_ != hipSuccess) return qrt_fail("%s: launch failed: %s", name, hipGetErrorString(e_)); \
  } while (0)

// The wave's number within its block, in a scalar register: what follows from it (the wave's rows,
// its share of a loop) is then the same for the whole wave to the compiler too, and branches on it
// become scalar branches. For kernels with MFMA instructions this is needed, not only faster:
// MFMA does not look at the EXEC mask, so one inside a branch that the compiler lowered to an
// EXEC mask of zeros, without a jump over it, runs all the same, on registers never loaded.
__device__ __forceinline__ int uniform_wave_number() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// Eight bfloat16 of a matrix that a step reads exactly once (weights streamed past few rows of
// activations): a non-temporal load, which leaves the caches to data that is read again. A plain
// read of 4 GiB runs at 6.1 TB/s on this device, a non-temporal one at 6.9; the few-row products
// of a decode step gain 2 to 5 % by it (the products with 17 to 64 rows lose 2 %, and keep
// plain loads).
__device__ __forceinline__ bf16x8_t load_once8(const bf16_t* p) {
  return __builtin_bit_cast(bf16x8_t, __builtin_nontemporal_load((const u32x4_t*)p));
}

template <typename T> __device__ __forceinline__ float to_f32(T x);
template <> __device__ __forceinline__ float to_f32<float>(float x) { return x; }
template <> __device__ __forceinline__ float to_f32<bf16_t>(bf16_t x) { return (float)x; }

template <typename T> __device__ __forceinline__ T from_f32(float x);
template <> __device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float x) { return (bf16_t)x; }

// Sine and cosine of a rotation angle held in float32 (position times frequency: up to
// millions of radians). The library routine reduces such arguments with a table it loads from
// memory; here the angle is reduced to [-pi, pi] in float64 (exact to 1e-10 rad) first, so the
// routine stays on its short path and the kernel has no loads in its middle. The result is the
// sine and cosine of the float32 angle to within one unit in the last place.
__device__ __forceinline__ void sincos_angle(float angle, float* sn, float* cs) {
  const double turns = (double)angle * 0.15915494309189535;  // 1 / (2 pi)
  const float reduced = (float)((turns - rint(turns)) * 6.283185307179586);
  sincosf(reduced, sn, cs);
}

// Gated activations of feed-forwards, float32. SWIGLU: silu(g) u. CLAMPED: g and u are held to
// `limit` first (g from above only, u from both sides), then g sigmoid(1.702 g) (u + 1).
#define QRT_ACT_SWIGLU 0
#define QRT_ACT_CLAMPED 1
__device__ __forceinline__ float gated_act(float g, float u, int kind, float limit) {
  if (kind == QRT_ACT_CLAMPED) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
  }
  return g / (1.0f + expf(-g)) * u;
}

// What lanes 32, 16, 8, 4, 2 and 1 apart hold, joined step by step: by swaps and rotations of registers, where a shuffle through
// LDS takes some 60 cycles a step (after each step lanes that far apart hold the same, so a rotation within 16 lanes brings the
// partner's). Every lane of the wave takes part. A norm's block sums and the serial loop they ended with took 1 of 5.8 us.
template <class Join>
__device__ __forceinline__ float wave_join(float x, Join join) {
  typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
  const unsigned int u = __float_as_uint(x);
  const u32x2_t a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  x = join(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const unsigned int v = __float_as_uint(x);
  const u32x2_t b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  x = join(__uint_as_float(b[0]), __uint_as_float(b[1]));
  x = join(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x128, 0xF, 0xF, true)));  // row_ror:8
  x = join(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x124, 0xF, 0xF, true)));  // row_ror:4
  x = join(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x122, 0xF, 0xF, true)));  // row_ror:2
  x = join(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x121, 0xF, 0xF, true)));  // row_ror:1
  return x;
}
__device__ __forceinline__ float wave_sum(float x) {
  return wave_join(x, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float x) {
  return wave_join(x, [](float a, float b) { return fmaxf(a, b); });
}

// Sum over a block of up to 1024 threads, in whole waves; every thread gets the result, from
// parts that all of them add in the order of the waves. `red` is shared memory of at least 16 floats.
template <class Join>
__device__ __forceinline__ float block_join(float x, float* red, float none, Join join) {
  x = wave_join(x, join);
  const int wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = x;
  __syncthreads();
  float s = none;
  if (nw <= 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) s = i < nw ? join(s, red[i]) : s;
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) s = i < nw ? join(s, red[i]) : s;
  }
  return s;
}
__device__ __forceinline__ float block_sum(float x, float* red) {
  return block_join(x, red, 0.f, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float block_max(float x, float* red) {
  return block_join(x, red, -INFINITY, [](float a, float b) { return fmaxf(a, b); });
}
