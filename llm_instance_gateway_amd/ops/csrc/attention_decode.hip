// Paged-attention DECODE of the Llama path (one query token per sequence),
// bf16, gfx950 / CDNA4.  Heads of 64 and 128 run flash_decode.h's kernel
// without any of the options of the hybrid families; heads of 16, which only
// the tiny test models have, a plain walk.
//
// Cache layout: [num_blocks, num_kv_heads, block_size, head_dim] bf16.
// Capability parity: the paged attention the reference delegates to vLLM.

#include "flash_decode.h"

// One wave per (sequence, query head): 8 lanes of 2 entries per key, 8 keys
// side by side, each with its own running maximum, merged at the end.
__global__ __launch_bounds__(WAVE_SIZE) void paged_attention_decode_16_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache,
    const uint16_t* __restrict__ v_cache, const int* __restrict__ block_tables,
    const int* __restrict__ context_lens, const float scale, const int num_q_heads, const int num_kv_heads,
    const int block_size, const int max_blocks) {
  constexpr int D = 16;
  const int seq = blockIdx.x, qh = blockIdx.y;
  const int kvh = qh / (num_q_heads / num_kv_heads);
  const int tok = threadIdx.x >> 3, d = (threadIdx.x & 7) * 2;
  const int ctx = context_lens[seq];
  const int* bt = block_tables + (size_t)seq * max_blocks;
  const size_t at = ((size_t)seq * num_q_heads + qh) * D + d;
  const float q0 = bf16_to_f32(q[at]), q1 = bf16_to_f32(q[at + 1]);

  float m = -INFINITY, l = 0.f, o0 = 0.f, o1 = 0.f;
  for (int t0 = 0; t0 < ctx; t0 += 8) {
    const int t = t0 + tok;
    const bool valid = t < ctx;
    float s = 0.f, v0 = 0.f, v1 = 0.f;
    if (valid) {
      const size_t base =
          (((size_t)bt[t / block_size] * num_kv_heads + kvh) * block_size + (t % block_size)) * D + d;
      s = q0 * bf16_to_f32(k_cache[base]) + q1 * bf16_to_f32(k_cache[base + 1]);
      v0 = bf16_to_f32(v_cache[base]);
      v1 = bf16_to_f32(v_cache[base + 1]);
    }
    s = group_reduce_sum<8>(s);
    s = valid ? s * scale : -INFINITY;
    const float mn = fmaxf(m, s);
    if (mn == -INFINITY) continue;
    const float alpha = m == -INFINITY ? 0.f : __expf(m - mn);
    const float p = s == -INFINITY ? 0.f : __expf(s - mn);
    m = mn;
    l = l * alpha + p;
    o0 = o0 * alpha + p * v0;
    o1 = o1 * alpha + p * v1;
  }
  const float gm = stride_reduce_max<8, 8>(m);
  const float w = m == -INFINITY ? 0.f : __expf(m - gm);
  l = stride_reduce_sum<8, 8>(l * w);
  o0 = stride_reduce_sum<8, 8>(o0 * w);
  o1 = stride_reduce_sum<8, 8>(o1 * w);
  if (tok == 0) {
    const float f = l > 0.f ? 1.f / l : 0.f;
    out[at] = f32_to_bf16(o0 * f);
    out[at + 1] = f32_to_bf16(o1 * f);
  }
}

// scratch: fp32 [N, Hq, nsplits, D + 2] where nsplits > 1, else unused
extern "C" void lig_paged_attention_decode_launch(
    uint16_t* out, const uint16_t* q, const uint16_t* k_cache,
    const uint16_t* v_cache, const int* block_tables,
    const int* context_lens, float* scratch, float scale, int num_seqs,
    int num_q_heads, int num_kv_heads, int head_dim, int block_size,
    int max_blocks, int nsplits, hipStream_t stream) {
  if (head_dim == 16) {
    hipLaunchKernelGGL(paged_attention_decode_16_kernel, dim3(num_seqs, num_q_heads), dim3(WAVE_SIZE), 0, stream, out,
                       q, k_cache, v_cache, block_tables, context_lens, scale, num_q_heads, num_kv_heads, block_size,
                       max_blocks);
    return;
  }
  flash_decode::Args a{};
  a.out = out;
  a.q = q;
  a.q_stride = (long)num_q_heads * head_dim;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.block_tables = block_tables;
  a.context_lens = context_lens;
  a.scratch = scratch;
  a.scale = scale;
  a.rows = num_seqs;
  a.num_q_heads = num_q_heads;
  a.num_kv_heads = num_kv_heads;
  a.v_row = head_dim;
  a.block_size = block_size;
  a.block_shift = flash_decode::shift_of(block_size);
  a.max_blocks = max_blocks;
  a.nsplits = nsplits;
  if (head_dim == 64)
    flash_decode::launch_mode<64, false, false, false>(a, stream);
  else  // the caller lets only 16, 64 and 128 through
    flash_decode::launch_mode<128, false, false, false>(a, stream);
}
