// Shared device helpers for the gfx950 (CDNA4) DSpark kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dspark {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int WAVE = 64;
constexpr int PAGE = 32;  // tokens per KV page (the reference's BlockTokens)

// D = A(16x32) * B(32x16) + C on the matrix cores. Lane l holds A row l%16 / B column l%16, k = 8*(l/16)+0..7;
// C/D: column l%16, rows 4*(l/16)+0..3.
__device__ __forceinline__ f32x4 mfma16x16x32(half8 a, half8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ half8 as_half8(u32x4 u) {
  half8 h;
  __builtin_memcpy(&h, &u, 16);
  return h;
}

// Eight biased int8 weights (two words) as halves, exactly: byte b (= q + 128) under 0x64 is the half 1024 + b.
__device__ __forceinline__ half8 i8x8_to_half8(uint32_t w0, uint32_t w1) {
  const uint32_t k64 = 0x64646464u;
  const uint32_t a0 = __builtin_amdgcn_perm(k64, w0, 0x04010400u);
  const uint32_t a1 = __builtin_amdgcn_perm(k64, w0, 0x04030402u);
  const uint32_t a2 = __builtin_amdgcn_perm(k64, w1, 0x04010400u);
  const uint32_t a3 = __builtin_amdgcn_perm(k64, w1, 0x04030402u);
  u32x4 u = {a0, a1, a2, a3};
  half8 h = as_half8(u);
  const half8 bias = {1152, 1152, 1152, 1152, 1152, 1152, 1152, 1152};
  return h - bias;
}

// x / d by one multiplication: div_magic(d) = ceil(2^32 / d), exact for x d < 2^32 (0 stands for d = 1). A division by a
// run-time value is some 20 dependent instructions, most of them before a kernel's first load.
inline uint32_t div_magic(uint32_t d) { return d > 1 ? (uint32_t)((0x100000000ull + d - 1) / d) : 0u; }
__device__ __forceinline__ int div_by(int x, uint32_t magic) { return magic ? (int)(((uint64_t)(uint32_t)x * magic) >> 32) : x; }

// A wave-uniform word that nothing writes while the kernel runs, by a scalar load (a plain load becomes a vector load in
// kernels where the compiler sees a store that might reach it).
template <typename T>
__device__ __forceinline__ T ldc(const T* p) {
  typedef __attribute__((address_space(4))) const T CT;
  return *(CT*)(uintptr_t)p;
}

template <typename T>
__device__ __forceinline__ T ldg(const T* p) {
  typedef __attribute__((address_space(1))) const T GT;
  return *(const GT*)p;
}

template <typename T>
__device__ __forceinline__ T ldg_nt(const T* p) {
  typedef __attribute__((address_space(1))) const T GT;
  return __builtin_nontemporal_load((const GT*)p);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// s_waitcnt immediate (gfx9 encoding): vmcnt(n) with expcnt and lgkmcnt left at their maxima.
__device__ __forceinline__ constexpr int vmcnt_imm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }

// A ring step's hand-over: this wave's direct-to-LDS loads but the N youngest done, and its reads of the step before (whose
// slot the loads issued next overwrite), then every wave's. The wait and barrier builtins do not order memory operations
// for the compiler, which sees no other writer of the slot read next: the empty asm holds every access on its side, and the
// LDS count is waited for because the uses of the last step's reads may sink below.
template <int N>
__device__ __forceinline__ void ring_barrier() {
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(N) & ~0x0F00);  // lgkmcnt(0) too
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Every wave's LDS accesses done, none moved across (loads from memory stay in flight). The barrier of every hand-over of
// LDS between waves that is not a ring step's or a __syncthreads() (which would drain the loads).
__device__ __forceinline__ void lds_barrier() { ring_barrier<63>(); }

// Butterfly over a whole wave without the LDS unit (a shuffle there costs about 100 cycles a level): level by level each
// lane's value is combined with lane ^ 32's and lane ^ 16's by the half-wave swaps, then with lane ^ 8's, ^ 4's, ^ 2's
// and ^ 1's by row rotations -- after a level the values repeat with half the period, so that a rotation by 4 in a row of
// 16 brings lane ^ 4's value, and so on. The same pairs in the same order as an xor-shuffle butterfly, hence the same bits
// (the operations commute). Every lane of the wave must be active.
template <int N>
__device__ __forceinline__ uint32_t row_ror(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x120 + N, 0xf, 0xf, false);
}
template <typename F>
__device__ __forceinline__ uint32_t wave_butterfly(uint32_t v, F op) {
  const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  v = op(a[0], a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = op(b[0], b[1]);
  v = op(v, row_ror<8>(v));
  v = op(v, row_ror<4>(v));
  v = op(v, row_ror<2>(v));
  return op(v, row_ror<1>(v));
}
__device__ __forceinline__ float wave_max(float v) {
  return __uint_as_float(wave_butterfly(__float_as_uint(v), [](uint32_t a, uint32_t b) {
    return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
  }));
}
__device__ __forceinline__ float wave_sum(float v) {
  return __uint_as_float(wave_butterfly(__float_as_uint(v), [](uint32_t a, uint32_t b) {
    return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
  }));
}
// The sum of each half of a wave, in every lane of the half (the bits of wave_sum with zeros in the other half).
__device__ __forceinline__ float half_wave_sum(float v) {
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  v += __uint_as_float(row_ror<8>(__float_as_uint(v)));
  v += __uint_as_float(row_ror<4>(__float_as_uint(v)));
  v += __uint_as_float(row_ror<2>(__float_as_uint(v)));
  return v + __uint_as_float(row_ror<1>(__float_as_uint(v)));
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  return wave_butterfly(v, [](uint32_t a, uint32_t b) { return max(a, b); });
}

// quantize_pair (kernels/ops.hip:212-224) of a record's 128 values, one IEEE fp32 operation per step: the scale from
// the values' absolute maximum, and the int8 code of x with inv = 1 / scale.
__device__ __forceinline__ float rec_scale(float amax) { return fmaxf(__fdiv_rn(amax, 127.f), 1e-6f); }
__device__ __forceinline__ int rec_code(float x, float inv) {
  float a = __fmul_rn(x, inv);
  a = a >= 0.f ? __fadd_rn(a, 0.5f) : __fsub_rn(a, 0.5f);
  return (int)truncf(fminf(fmaxf(a, -128.f), 127.f));
}

// Argmax key (reference dspark.hip:967-971): ordered float bits above, 0xFFFFFFFF - index below. The maximum key is the
// largest value and, among equal values, the smallest index.
__device__ __forceinline__ uint32_t argmax_ord(float v) {  // float bits in the order of the values
  const uint32_t u = __float_as_uint(v);
  return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}
__device__ __forceinline__ uint64_t argmax_key(float v, uint32_t idx) {
  return ((uint64_t)argmax_ord(v) << 32) | (uint64_t)(0xffffffffu - idx);
}

// K/V page formats (one block of PAGE keys x D dims per (page, KV head)). K is stored in the operand order of
// v_mfma_f32_16x16x32_f16: key `slot` is row n = 4 (slot / 8) + slot % 4 of key block b = (slot / 4) % 2, and dim d sits
// in k-step d / 32 of lane n + 16 ((d % 32) / 8), element d % 8. V is stored transposed: [d][slot].
__device__ __forceinline__ int k_page_elem(int slot, int d, int D) {
  const int b = (slot >> 2) & 1, n = 4 * (slot >> 3) + (slot & 3);
  return ((b * (D / 32) + d / 32) * 64 + n + 16 * ((d % 32) / 8)) * 8 + d % 8;
}
__device__ __forceinline__ int v_page_elem(int slot, int d) { return d * PAGE + slot; }

// Activations a verify GEMM reads as X ([M][K] fp16, M <= 16 tbs) in the B-operand order of v_mfma_f32_16x16x32_f16:
// 1 KB blocks [K / 64 chunks][tbs token blocks][2 halves] of 64 lanes x 8 halves, lane 16 g + n holding token
// 16 tb + n, columns 64 c + 16 g + 8 h .. + 7. A wave's X operand load is then one contiguous 1 KB (row-major X
// gathers 64 bytes from each of 16 token rows). Four consecutive columns from a multiple of 4 stay contiguous.
__device__ __forceinline__ size_t xop_elem(int t, int k, int tbs) {
  return ((((size_t)(k >> 6) * tbs + (t >> 4)) * 2 + ((k >> 3) & 1)) * 64 + ((k >> 4) & 3) * 16 + (t & 15)) * 8 +
         (k & 7);
}

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int m) {
  const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, m);
  const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), m);
  return ((uint64_t)hi << 32) | lo;
}

// (every lane of the wave active) The largest high word, then the largest low word under it.
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) {
  const uint32_t hi = wave_max_u32((uint32_t)(v >> 32));
  const uint32_t lo = wave_max_u32((uint32_t)(v >> 32) == hi ? (uint32_t)v : 0u);
  return ((uint64_t)hi << 32) | lo;
}

}  // namespace dspark
