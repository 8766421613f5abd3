// Paged-attention DECODE of the Llama path (one query token per sequence),
// bf16, gfx950 / CDNA4.  Heads of 64 and 128 run flash_decode.h's kernel
// without any of the options of the hybrid families; heads of 16, which only
// the tiny test models have, a walk without matrix instructions.
//
// Cache layout: [num_blocks, num_kv_heads, block_size, head_dim] bf16.
// Capability parity: the paged attention the reference delegates to vLLM.

#include "flash_decode.h"

// One wave per (sequence, query head, part of the walk), four heads to a workgroup: 8 lanes of 2 entries
// per key, 32 keys a step of which a group of lanes takes 4, each group with its
// own running maximum, merged at the end.  Parts are flash_decode.h's and merged
// by its second kernel.  What bounds it is the chain of a step (table entry, key,
// reduction, exponential) and not bandwidth, hence 4 keys at once and the cut.
// 4 query and 2 key/value heads: one row of 16000 keys 26 us, 4 of 4000 19, 64
// of 3000 24; with 8 keys a step and uncut 775, 197 and 156.
__global__ __launch_bounds__(4 * WAVE_SIZE) void paged_attention_decode_16_kernel(const flash_decode::Args a) {
  constexpr int D = 16, U = flash_decode::KT / 8;
  const int seq = blockIdx.x, qh = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (qh >= a.num_q_heads) return;
  const flash_decode::Walk wk = flash_decode::walk_of<false>(a, seq);
  if ((int)blockIdx.z >= wk.parts) return;
  const int kvh = qh / (a.num_q_heads / a.num_kv_heads);
  const int tok = (threadIdx.x & 63) >> 3, d = (threadIdx.x & 7) * 2;
  const int* bt = a.block_tables + (size_t)seq * a.max_blocks;
  const size_t item = (size_t)seq * a.num_q_heads + qh, at = item * D + d;
  const float c = a.scale * LOG2E;
  const float q0 = bf16_to_f32(a.q[at]), q1 = bf16_to_f32(a.q[at + 1]);
  const int span = (wk.steps + wk.parts - 1) / wk.parts;
  const int s0 = blockIdx.z * span, s1 = min(wk.steps, s0 + span);

  float m = -INFINITY, l = 0.f, o0 = 0.f, o1 = 0.f;
  for (int st = s0; st < s1; ++st) {
    const int t0 = st * flash_decode::KT + tok;
    size_t base[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = min(t0 + u * 8, wk.pos);  // past the end: the last key again, unused
      base[u] = (((size_t)bt[t / a.block_size] * a.num_kv_heads + kvh) * a.block_size + (t % a.block_size)) * D + d;
    }
    float s[U], v0[U], v1[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s[u] = q0 * bf16_to_f32(a.k_cache[base[u]]) + q1 * bf16_to_f32(a.k_cache[base[u] + 1]);
      v0[u] = bf16_to_f32(a.v_cache[base[u]]);
      v1[u] = bf16_to_f32(a.v_cache[base[u] + 1]);
    }
    float mn = m;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s[u] = group_reduce_sum<8>(s[u]);
      s[u] = t0 + u * 8 <= wk.pos ? s[u] * c : -INFINITY;
      mn = fmaxf(mn, s[u]);
    }
    const float mm = mn == -INFINITY ? 0.f : mn;
    const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mm);
    m = mn;
    l *= alpha;
    o0 *= alpha;
    o1 *= alpha;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool valid = t0 + u * 8 <= wk.pos;
      const float p = valid ? __builtin_amdgcn_exp2f(s[u] - mm) : 0.f;
      l += p;
      o0 += valid ? p * v0[u] : 0.f;
      o1 += valid ? p * v1[u] : 0.f;
    }
  }
  const float gm = stride_reduce_max<8, 8>(m);
  const float w = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - gm);
  l = stride_reduce_sum<8, 8>(l * w);
  o0 = stride_reduce_sum<8, 8>(o0 * w);
  o1 = stride_reduce_sum<8, 8>(o1 * w);
  if (tok != 0) return;
  if (wk.parts > 1) {
    float* sp = a.scratch + (item * a.nsplits + blockIdx.z) * (D + 2);
    sp[d] = o0;
    sp[d + 1] = o1;
    if (d == 0) {
      sp[D] = gm;
      sp[D + 1] = l;
    }
  } else {
    const float f = l > 0.f ? 1.f / l : (l == 0.f ? 0.f : l);
    a.out[at] = f32_to_bf16(o0 * f);
    a.out[at + 1] = f32_to_bf16(o1 * f);
  }
}

// scratch: fp32 [N, Hq, nsplits, D + 2] where nsplits > 1, else unused.  Unmerged, rows
// that were cut are left there for their reader.
extern "C" void lig_paged_attention_decode_launch(
    uint16_t* out, const uint16_t* q, const uint16_t* k_cache,
    const uint16_t* v_cache, const int* block_tables,
    const int* context_lens, float* scratch, float scale, int num_seqs,
    int num_q_heads, int num_kv_heads, int head_dim, int block_size,
    int max_blocks, int nsplits, int unmerged, hipStream_t stream) {
  flash_decode::Args a{};
  a.out = out;
  a.q = q;
  a.q_stride = (long)num_q_heads * head_dim;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.block_tables = block_tables;
  a.tables = num_seqs;
  a.context_lens = context_lens;
  a.scratch = scratch;
  a.scale = scale;
  a.rows = num_seqs;
  a.num_q_heads = num_q_heads;
  a.num_kv_heads = num_kv_heads;
  a.v_row = head_dim;
  a.block_size = block_size;
  a.block_shift = shift_of(block_size);
  a.max_blocks = max_blocks;
  a.nsplits = nsplits;
  a.unmerged = unmerged;
  if (head_dim == 16) {
    hipLaunchKernelGGL(paged_attention_decode_16_kernel, dim3(num_seqs, (num_q_heads + 3) / 4, nsplits),
                       dim3(4 * WAVE_SIZE), 0, stream, a);
    flash_decode::launch_merge<16, false, false>(a, stream);
  } else if (head_dim == 64)
    flash_decode::launch_mode<64, false, false, false>(a, stream);
  else  // the caller lets only 16, 64 and 128 through
    flash_decode::launch_mode<128, false, false, false>(a, stream);
}
