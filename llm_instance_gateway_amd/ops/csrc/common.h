// Common device helpers for the gfx950 (MI355X / CDNA4) kernels.
//
// Written for CDNA4 only: wave64, MFMA, 160 KiB LDS per CU, HBM3E.
// No CUDA-compat shims, no multi-arch dispatch.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <cstdint>

#define WAVE_SIZE 64

#define LIG_DEVICE __device__ __forceinline__

// ---- bf16 <-> f32 -----------------------------------------------------------

LIG_DEVICE float bf16_to_f32(uint16_t h) {
  union {
    uint32_t u;
    float f;
  } v;
  v.u = static_cast<uint32_t>(h) << 16;
  return v.f;
}

// round-to-nearest-even, one hardware conversion
LIG_DEVICE uint16_t f32_to_bf16(float f) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}

// 8 bf16 = 16 B: the unit of a fully-coalesced per-lane load (16 B/lane x
// 64 lanes = 1 KiB per instruction).
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

LIG_DEVICE f32x8 bf16x8_to_f32x8(u16x8 h) {
  f32x8 out;
#pragma unroll
  for (int i = 0; i < 8; ++i) out[i] = bf16_to_f32(h[i]);
  return out;
}

// As vectors: one conversion makes two numbers, element by element each takes a
// conversion and the packing another.
LIG_DEVICE u16x8 f32x8_to_bf16x8(f32x8 f) {
  typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
  return __builtin_bit_cast(u16x8, __builtin_convertvector(f, bf16x8));
}

LIG_DEVICE uint32_t pack_bf16(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}

// ---- wave reductions --------------------------------------------------------
// Butterfly over the full 64-lane wave; result replicated in every lane.

LIG_DEVICE float wave_reduce_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE_SIZE);
  return v;
}

LIG_DEVICE float wave_reduce_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, WAVE_SIZE));
  return v;
}

// Partial butterfly: reduce within groups of `width` lanes (width = power of 2).
template <int WIDTH>
LIG_DEVICE float group_reduce_sum(float v) {
#pragma unroll
  for (int off = WIDTH / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE_SIZE);
  return v;
}

// Reduce ACROSS groups: lanes i, i+STRIDE, i+2*STRIDE ... combined.
template <int STRIDE, int N>
LIG_DEVICE float stride_reduce_sum(float v) {
#pragma unroll
  for (int off = STRIDE; off < STRIDE * N; off <<= 1) v += __shfl_xor(v, off, WAVE_SIZE);
  return v;
}

template <int STRIDE, int N>
LIG_DEVICE float stride_reduce_max(float v) {
#pragma unroll
  for (int off = STRIDE; off < STRIDE * N; off <<= 1)
    v = fmaxf(v, __shfl_xor(v, off, WAVE_SIZE));
  return v;
}

// Max over the four 16-lane groups, result in all of them; no LDS traffic.
LIG_DEVICE float max_over_groups(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const float y = fmaxf(__builtin_bit_cast(float, (uint32_t)a[0]), __builtin_bit_cast(float, (uint32_t)a[1]));
  const uint32_t v = __builtin_bit_cast(uint32_t, y);
  auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return fmaxf(__builtin_bit_cast(float, (uint32_t)b[0]), __builtin_bit_cast(float, (uint32_t)b[1]));
}

// ---- memory -> LDS ------------------------------------------------------------
// 16 bytes per lane to `lds` (uniform) + lane * 16, no registers in between.  As
// the builtin, every LDS read behind it would wait for it, whatever it reads: a
// tile could not be on its way while another is used.  So these are invisible to
// the compiler's counting, and the code that reads the bytes waits by itself:
// loads_landed<n> before the barrier behind which they are read.  (The compiler's
// own waits for loads count in order and can only be longer for it.)
// One wait state between a write to m0 and its use.
LIG_DEVICE uint32_t lds_address(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p);
}
LIG_DEVICE void load_to_lds(const void* base, uint32_t offset, uint32_t lds) {  // base: uniform
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %0" ::"s"(base), "v"(offset), "{m0}"(lds) : "memory");
}
// of bytes that nobody reads again: they do not displace others in the caches
LIG_DEVICE void stream_to_lds(const void* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %0 nt" ::"s"(base), "v"(offset), "{m0}"(lds) : "memory");
}
LIG_DEVICE void load_to_lds(const void* p, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(p), "{m0}"(lds) : "memory");
}
// Whether a weight [N, K] that one workgroup reads once is loaded as a stream, past
// the caches: from 32 MiB on, where a model's weights together no longer stay in the
// 256 MB of the last-level cache from one step to the next.  Streams of 32 MiB and
// more gain 4 to 13 % (row_product.hip), smaller ones nothing, and a model small
// enough to stay in that cache would lose up to 10 %.
__host__ __device__ constexpr bool streams(int N, int K) { return (long)N * K >= 1L << 24; }
// All but this wave's last N loads have landed and its LDS reads are done, and so
// are those of the other waves.
template <int N>
LIG_DEVICE void loads_landed() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

constexpr float LOG2E = 1.44269504088896340736f;

// log2 of a cache's block size, -1 if that is no power of two
static inline int shift_of(int block_size) {
  return block_size > 0 && (block_size & (block_size - 1)) == 0 ? __builtin_ctz((unsigned)block_size) : -1;
}

LIG_DEVICE int cdiv(int a, int b) { return (a + b - 1) / b; }
