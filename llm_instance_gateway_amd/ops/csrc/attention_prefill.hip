// Paged-attention PREFILL of the Llama path: causal softmax attention of the
// step's prompt portions over the paged KV cache, bf16, heads of 64 or 128,
// gfx950 / CDNA4.  The kernel is flash_prefill.h's, without any of the options
// of the hybrid families.
// Capability parity: flash prefill the reference delegates to vLLM.

#include "flash_prefill.h"

// Parts of the keys that a call of that size is cut into: above one it needs room for
// [rows, num_q_heads, parts, head_dim + 4] floats.
extern "C" int lig_paged_attention_prefill_parts(long ntiles, long rows, int num_q_heads, int head_dim, long keys) {
  return flash_prefill::parts(ntiles, rows, num_q_heads, head_dim, keys);
}

extern "C" void lig_paged_attention_prefill_launch(
    uint16_t* out, const uint16_t* q, const uint16_t* k_cache,
    const uint16_t* v_cache, const int* tile_seq, const int* tile_qstart,
    const int* query_start_locs, const int* context_lens,
    const int* block_tables, float scale, int ntiles, int num_q_heads,
    int num_kv_heads, int head_dim, int block_size, int max_blocks, int num_seqs,
    int nsplit, float* partial, hipStream_t stream) {
  flash_prefill::Args a{};
  a.out = out;
  a.q = q;
  a.q_stride = (long)num_q_heads * head_dim;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.tile_seq = tile_seq;
  a.tile_qstart = tile_qstart;
  a.query_start_locs = query_start_locs;
  a.context_lens = context_lens;
  a.block_tables = block_tables;
  a.scale = scale;
  a.num_q_heads = num_q_heads;
  a.num_kv_heads = num_kv_heads;
  a.v_row = head_dim;
  a.block_size = block_size;
  a.block_shift = shift_of(block_size);
  a.max_blocks = max_blocks;
  a.num_seqs = num_seqs;
  a.nsplit = nsplit;
  a.partial = partial;
  if (nsplit > 1) {
    if (head_dim == 64) flash_prefill::launch_parts<64>(a, ntiles, stream);
    else flash_prefill::launch_parts<128>(a, ntiles, stream);
  } else if (head_dim == 64)
    flash_prefill::launch_mode<64, false, false, false>(a, ntiles, stream);
  else  // the caller lets only 64 and 128 through
    flash_prefill::launch_mode<128, false, false, false>(a, ntiles, stream);
}
