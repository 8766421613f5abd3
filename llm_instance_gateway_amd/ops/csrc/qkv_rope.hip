// Everything between the fused q/k/v projection of the Llama path and its
// attention: rotation of q and k, k and v into the paged cache, q packed; bf16,
// head sizes a multiple of 64, gfx950.
//
// Launches and passes over memory bound it: as three strided copies, a
// rotation in place and a scatter it was five launches of 4.5 us in a decode
// layer (two for a single token) and 55 us for 4096 tokens, besides the copy
// of the attention's result; one pass is one launch. Engine steps over 8
// layers: 33 requests 3.13 -> 3.01 ms, a prompt of 202 3.13 -> 2.91 ms, 20 of
// 200 15.8 -> 15.3 ms.  A wave takes 16 tokens by 32
// rotation pairs of 4 heads: lane (li, lg) holds 8 neighbouring entries of
// token li and their partners half a head away, so the rotation stays in the
// lane, loads and stores are 16 bytes, and a token's cosines and sines are read
// once for the 4 heads.

#include "common.h"

#define QR_HEADS 4  // per wave

__global__ __launch_bounds__(256) void qkv_rope_cache_kernel(
    uint16_t* __restrict__ q_out,              // [T, Hq * D]
    const uint16_t* __restrict__ qkv,          // [T, (Hq + 2 Hkv) * D]
    const int64_t* __restrict__ positions,     // [T]
    const float* __restrict__ cos_sin,         // [P, D]: D/2 cosines | D/2 sines
    uint16_t* __restrict__ k_cache,            // [B, Hkv, BS, D]
    uint16_t* __restrict__ v_cache,
    const int64_t* __restrict__ slot_mapping,  // [T], negative: not cached
    const int num_tokens, const int num_q_heads, const int num_kv_heads, const int head_dim,
    const int block_size, const int block_shift) {
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int parts = head_dim / 64;  // of 32 pairs
  const int wid = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int heads = num_q_heads + 2 * num_kv_heads;
  const int h0 = (wid / parts) * QR_HEADS;
  const int row = blockIdx.x * 16 + li;
  if (h0 >= heads || row >= num_tokens) return;
  const int half = head_dim / 2;
  const int c = (wid % parts) * 32 + lg * 8;

  const float* cs = cos_sin + positions[row] * head_dim + c;
  float co[8], si[8];
#pragma unroll
  for (int i = 0; i < 8; i += 4) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(cs + i);
    const f32x4 b = *reinterpret_cast<const f32x4*>(cs + half + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      co[i + j] = a[j];
      si[i + j] = b[j];
    }
  }
  const int64_t slot = slot_mapping[row];
  // a division of 64 bits is some hundred instructions
  const size_t blk = slot < 0 ? 0 : block_shift >= 0 ? slot >> block_shift : slot / block_size;
  const size_t off = slot < 0 ? 0 : slot - (int64_t)blk * block_size;

  const uint16_t* src = qkv + ((size_t)row * heads + h0) * head_dim + c;
  u16x8 x[QR_HEADS][2];
#pragma unroll
  for (int i = 0; i < QR_HEADS; ++i) {
    const int h = min(h0 + i, heads - 1) - h0;
    x[i][0] = *reinterpret_cast<const u16x8*>(src + h * head_dim);
    x[i][1] = *reinterpret_cast<const u16x8*>(src + h * head_dim + half);
  }
#pragma unroll
  for (int i = 0; i < QR_HEADS; ++i) {
    const int h = h0 + i;
    if (h >= heads) break;
    if (h < num_q_heads + num_kv_heads) {
      const f32x8 a = bf16x8_to_f32x8(x[i][0]), b = bf16x8_to_f32x8(x[i][1]);
      f32x8 o1, o2;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        o1[j] = a[j] * co[j] - b[j] * si[j];
        o2[j] = b[j] * co[j] + a[j] * si[j];
      }
      x[i][0] = f32x8_to_bf16x8(o1);
      x[i][1] = f32x8_to_bf16x8(o2);
    }
    uint16_t* dst;
    if (h < num_q_heads) {
      dst = q_out + ((size_t)row * num_q_heads + h) * head_dim;
    } else {
      if (slot < 0) continue;
      const bool key = h < num_q_heads + num_kv_heads;
      const int g = h - num_q_heads - (key ? 0 : num_kv_heads);
      dst = (key ? k_cache : v_cache) + ((blk * num_kv_heads + g) * block_size + off) * head_dim;
    }
    *reinterpret_cast<u16x8*>(dst + c) = x[i][0];
    *reinterpret_cast<u16x8*>(dst + half + c) = x[i][1];
  }
}

extern "C" void lig_qkv_rope_cache_launch(uint16_t* q_out, const uint16_t* qkv, const int64_t* positions,
                                          const float* cos_sin, uint16_t* k_cache, uint16_t* v_cache,
                                          const int64_t* slot_mapping, int num_tokens, int num_q_heads,
                                          int num_kv_heads, int head_dim, int block_size, hipStream_t stream) {
  const int heads = num_q_heads + 2 * num_kv_heads;
  const int waves = (head_dim / 64) * ((heads + QR_HEADS - 1) / QR_HEADS);
  hipLaunchKernelGGL(qkv_rope_cache_kernel, dim3((num_tokens + 15) / 16, (waves + 3) / 4), dim3(256), 0, stream, q_out,
                     qkv, positions, cos_sin, k_cache, v_cache, slot_mapping, num_tokens, num_q_heads, num_kv_heads,
                     head_dim, block_size, shift_of(block_size));
}
