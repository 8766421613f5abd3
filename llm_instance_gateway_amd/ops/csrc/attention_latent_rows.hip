// Multi-query attention over a paged latent cache on MFMA tiles, bf16, gfx950:
// every query head of a token reads the SAME cache rows, keys being the whole
// row (D entries) and values its leading Dv entries.
//
// Because all heads share the keys, the query rows of a tile are (token,
// head) pairs: row rho = token * H + head inside a sequence's segment of the
// step, 64 consecutive rho per workgroup (4 waves x 16 rows).  A key/value
// tile is read from HBM/L2 once per workgroup and serves every head in it,
// so a decode step (one token, H heads) is one pass over the sequence's cache
// and a prompt portion moves H times fewer key bytes than a per-head grid.
// Prompt portions and single tokens go through the same kernel: a segment is
// (first row, token count, context length after the step), and a row's
// causal bound is its token's position.
//
// What bounds it: a decode step reads every cache row once (HBM), a prompt
// portion does 2 * (D + Dv) flops per (row, key) on matrix cores.  Per tile:
//   * cache rows go from memory straight into LDS (16 bytes per lane, no
//     registers), once, XOR-swizzled by key through the choice of what a lane
//     fetches; the next tile is on its way while this one is used;
//   * S^T = K Q^T reads keys in the order in which a lane's scores are the
//     operand of O^T += V^T P^T, so weights stay in registers and a row's
//     statistics are one scalar per lane;
//   * V^T comes from the SAME rows through transposing LDS reads
//     (ds_read_b64_tr_b16).
// The kernel this replaces staged every row through registers, stored it a
// second time transposed in 2-byte pieces, sent the weights through LDS, and
// with one 83 KB workgroup per CU had 36 KB on the way.
// A wave owns 16 rows. Segments of more than 32 rows: 64 per workgroup, tiles of
// 32 keys, two workgroups per CU. Others (one token of up to 32 heads): 32 per
// workgroup, tiles of 64 keys of which waves 0-1 and 2-3 take a half each and
// merge at the end, one workgroup with 144 KB on the way or in use per CU.
// The fetches are load_to_lds: as the compiler's builtin, the first LDS read of a
// tile waited for the next tile's fetches too, and nothing was on its way meanwhile.
// Measured with rows of 576 and values of 512 (us; a kernel that staged through
// registers -> with the builtin -> now): 256 single tokens on 700-1024 keys, 32
// heads 148 -> 72 -> 63 (255 MB of rows, 4.1 TB/s); 4 prompts of 700-1000, 16 heads
// 322 -> 121 -> 97 (546 TFLOP/s; with the tiles dealt by length 83, weights ahead of others' products 79). Two row blocks per wave, which halve the LDS
// reads, lost more by leaving one wave per SIMD (keys of 320: 372 us before, 136
// now, 208 so; of 128: 149, 73, 135).
// Weights handed to all waves, so that each adds up a quarter of the columns of all rows and
// reads a quarter of the values from LDS, cost a second barrier and changed nothing (101 and 99 us).
// Scores, running max and sum are fp32; an optional per-head sink starts a
// row's running max at sink_h and its sum at one; an optional gate multiplies
// the (token, head) output row by one sigmoid (it commutes with whatever
// linear map per head follows).
//
// window > 0 restricts a row at position p to keys j with p - j < window; a
// tile's walk starts at the oldest key its first token sees.
//
// Grid = (ceil(max segment rows / 64 or 32), segments, splits), dealt anew by `deal`; workgroups
// without a tile exit at once.  With splits > 1 (few rows, long
// contexts) each z-slice walks an equal share of the tile's visible keys and
// leaves its unnormalised sum with its running max and sum in an fp32
// scratch; a second kernel merges the slices.  The sink is counted by slice
// zero only.

#include <type_traits>

#include "elem_types.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_of8 __attribute__((ext_vector_type(4), aligned(8)));  // outputs are not asked for more

constexpr int LR_PART_PAD = 4;  // a slice row is Dv values, running max (log2 units), running sum, 2 unused

// Workgroups begin in the order of x, then y, one to each XCD in turn, and one whose
// XCD is full holds up the others.  Segment for segment, a late one's longest walks
// began when the others were at their last, and empty workgroups between left XCDs
// unevenly full.  So the tiles that have rows are dealt by the lengths of their walks, the longest
// of all segments first: by their number in the segment, counted from the first token of the sequence,
// of which a window sees so many.  Of 4 prompts of 700-1000 with 16 heads 512 workgroups ran for
// 60 us and less and less of them for 38 more: 94 -> 83 us, with results in 16-byte pieces and
// one round of loads ahead of the block table less; 8 of them 197 -> 174, 16 of 70-100 23.1 -> 19.9.
// By the number in the segment alone the longest walks came last where tokens are cached: 6 of 512-1000 on
// 600-4000 keys 249 us in their order, 395 so, 232 now; 32 heads, 100 on 4000 keys beside 15 of 200 192, 490, 197.
// More than 16 segments, whose keys would no longer stay in the L2 (64 prompts of 210-300: 190 us
// in their order, 249 dealt), and single tiles stay as they are.  False: no tile is left.
struct Walk {
  int seg, tile, n, start, ctx;
};
template <typename F>
LIG_DEVICE int over_row(int v, const F& f) {  // of 16 lanes side by side, in each of them
  v = f(v, __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true));  // rotated by 8
  v = f(v, __builtin_amdgcn_mov_dpp(v, 0x124, 0xF, 0xF, true));
  v = f(v, __builtin_amdgcn_mov_dpp(v, 0x122, 0xF, 0xF, true));
  return f(v, __builtin_amdgcn_mov_dpp(v, 0x121, 0xF, 0xF, true));
}
LIG_DEVICE bool deal(const int* seg_start, const int* seg_len, const int* seg_ctx, int H, int rows, int window, Walk& w) {
  const unsigned segs = gridDim.y, most = gridDim.x;
  if (most == 1 || segs == 1 || segs > 16 || most > 65535) {
    w.seg = blockIdx.y;
    w.tile = most - 1 - blockIdx.x;
    w.n = seg_len[w.seg];
    w.start = seg_start[w.seg];
    w.ctx = seg_ctx[w.seg];
    return (long)w.tile * rows < (long)w.n * H;
  }
  // every 16 lanes hold all segments
  const int lane = threadIdx.x & 63, seg = lane & 15, at = min(seg, (int)segs - 1);
  const int n = seg_len[at], start = seg_start[at], ctx = seg_ctx[at];
  const int tiles = seg < (int)segs && n > 0 ? (int)min((long)most, ((long)n * H + rows - 1) / rows) : 0;
  auto sum = [](int v) { return over_row(v, [](int a, int b) { return a + b; }); };  // under 2^21
  const int i = blockIdx.y * most + blockIdx.x;
  if (i >= __builtin_amdgcn_readfirstlane(sum(tiles))) return false;
  // tiles of its tokens before these, or of those that the window's first row sees
  constexpr long MOST = 1 << 24;
  long before = min(MOST, (long)max(ctx - n, 0) * H / rows);
  if (window > 0) before = min(before, ((long)window * H + rows - 1) / rows);
  const int ahead = tiles > 0 ? (int)before : 0, end = ahead + tiles;
  auto from = [&](int t) { return sum(min(max(end - t, 0), tiles)); };  // tiles that end at t + 1 and behind
  // the last number from which on there are more than i tiles: four at a time, one for each 16 lanes
  int lo = 0;
  for (int width = __builtin_amdgcn_readfirstlane(over_row(end, [](int a, int b) { return max(a, b); })); width > 1;) {
    const int step = (width + 4) / 5;
    lo += __popcll(__ballot(from(lo + ((lane >> 4) + 1) * step) > i) & 0x0001000100010001) * step;
    width = step;
  }
  // the segments that have such a tile, in their order
  const int k = i - __builtin_amdgcn_readfirstlane(from(lo + 1)), tile = lo - ahead;
  const bool has = lane < 16 && tile >= 0 && tile < tiles;
  const uint32_t have = (uint32_t)__ballot(has);
  w.seg = __builtin_ctzll(__ballot(has && (int)__builtin_amdgcn_mbcnt_lo(have, 0) == k));
  w.tile = __builtin_amdgcn_readlane(tile, w.seg);
  w.n = __builtin_amdgcn_readlane(n, w.seg);
  w.start = __builtin_amdgcn_readlane(start, w.seg);
  w.ctx = __builtin_amdgcn_readlane(ctx, w.seg);
  return true;
}

// KG key groups of 32 keys per tile, 4 / KG waves of 16 rows for each.
// FULL: D == DKP, Dv == DVP and the block size is a power of two, at least 8
template <int DKP, int DVP, int KG, bool FULL>
__global__ __launch_bounds__(256, KG == 1 ? 2 : 1) void latent_attention_rows_kernel(
    uint16_t* __restrict__ out,          // [R, H * Dv]
    const uint16_t* __restrict__ q,      // [R, H * D] contiguous
    const uint16_t* __restrict__ cache,  // [blocks, 1, BS, D]
    const float* __restrict__ sink,      // nullable, [H]
    const uint16_t* __restrict__ gate, long gate_stride,  // nullable, [R, H] pre-sigmoid
    const int* __restrict__ seg_start, const int* __restrict__ seg_len,
    const int* __restrict__ seg_ctx,     // tokens of the sequence after this step
    const int* __restrict__ block_tables, int max_blocks, float scale, int H,
    int D_, int Dv_, int block_size, int block_shift, int window, int nsplit,
    float* __restrict__ partial) {  // [R * H, nsplit, Dv + 4] when nsplit > 1
  const int D = FULL ? DKP : D_, Dv = FULL ? DVP : Dv_;
  static_assert(DVP <= DKP && DKP % 64 == 0 && DVP % 16 == 0, "values are a prefix of the key row");
  constexpr int DB = DVP / 16;
  constexpr int KB = DKP / 32;
  constexpr int CHP = DKP / 8;              // 16-byte chunks of an LDS row, a multiple of 8
  constexpr int KT = 32 * KG;               // keys per tile
  constexpr int NI = KT * CHP / 256;        // fetches per wave and tile
  constexpr int ROWS = 64 / KG;
  constexpr int TILE = KT * DKP;
  constexpr int MERGE = KG > 1 ? 2 * 16 * (DVP + 4) * 2 : 0;  // fp32 rows of two waves, in 16-bit units
  constexpr int LDS = 2 * TILE > MERGE ? 2 * TILE : MERGE;
  __shared__ __align__(16) uint16_t sm[LDS];

  Walk walk;  // the longest first
  if (!deal(seg_start, seg_len, seg_ctx, H, ROWS, window, walk)) return;
  const int s = walk.seg, n = walk.n, ctx = walk.ctx;
  const long lo = walk.start;
  const long nrows = (long)n * H;
  const long rho0 = (long)walk.tile * ROWS;
  const int* bt = block_tables + (size_t)s * max_blocks;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int rblk = wave % (4 / KG);
  const int kg = wave / (4 / KG);

  // a wave whose rows all lie past the segment only helps fetching
  const bool wave_active = rho0 + rblk * 16 < nrows;
  const long rho = rho0 + rblk * 16 + li;
  const long rr = rho < nrows ? rho : rho0;
  const int tok = (int)(rr / H);
  const int head = (int)(rr - (long)tok * H);
  const int qpos = ctx - n + tok;

  const int z = blockIdx.z;
  const long last_rho = (rho0 + ROWS < nrows ? rho0 + ROWS : nrows) - 1;
  const int first_tok = (int)(rho0 / H);
  const int kv_end = ctx - n + (int)(last_rho / H) + 1;  // keys any row of the tile sees
  // oldest key any row of the tile sees, and the start of its piece of 8
  const int kv_seen = window > 0 ? max(0, ctx - n + first_tok - window + 1) : 0;
  const int kv_first = kv_seen & ~7;
  int kv_lo = kv_first, kv_hi = kv_end;
  if (nsplit > 1) {
    const int nt = (kv_end - kv_first + KT - 1) / KT;
    const int per = (nt + nsplit - 1) / nsplit;
    kv_lo = kv_first + z * per * KT;  // past the end: an empty slice
    kv_hi = min(kv_end, kv_lo + per * KT);
  }
  // bounds that hold for every row of the tile: no mask between them
  const int all_end = ctx - n + first_tok + 1;
  const int all_lo = window > 0 ? kv_end - window : 0;

  // ---- fetching: chunk c of key t of a tile goes to place (c % 8) ^ f(t) of the 8 that
  // columns c / 8 * 64 on have there.
  // Keys past the end repeat the last one, keys before the first that some row
  // sees that one: their weight is zero, but what they hold would still meet it in
  // a product, and the blocks before may be gone.
  // A fetch brings 64 columns (8 chunks) of 8 keys, 128 bytes a key side by side in
  // LDS, so that a lane's offset is the same for all fetches of 8 keys (as whole rows
  // the offsets took 27 slow multiplications a tile, as long as the products).
  // FULL: 8 keys, aligned, are one contiguous piece of a block; a wave takes
  // KT / 32 such pieces.  Lane j looks up the block of piece j of the tile after
  // next.  Else every lane looks for its own key's block.
  const uint32_t lds = lds_address(sm);
  const int CH = D / 8;
  constexpr int NP = CHP / 8;  // fetches per piece
  auto block_of = [&](int kv0) {
    const int t = min(FULL ? kv0 + (lane & 7) * 8 : max(kv0 + (lane & (KT - 1)), kv_seen), kv_end - 1);
    return bt[FULL ? t >> block_shift : t / block_size];
  };
  // Only a walk's first tile can hold keys before the first visible one (FIRST).
  auto fetch = [&](auto first_tile, int kv0, int blks, int buf) {
    constexpr bool FIRST = decltype(first_tile)::value;
    int here = lane;
    if (KG == 1) asm volatile("" : "+v"(here));  // worked out anew for each tile: held for the loop, it would spill
    const int row = here >> 3, place = here & 7;
    if constexpr (FULL) {
#pragma unroll
      for (int w = 0; w < KG; ++w) {
        const int piece = wave * KG + w;
        const int t0 = min(kv0 + piece * 8, (kv_end - 1) & ~7);
        const int blk = __builtin_amdgcn_readlane(blks, piece);
        const uint16_t* g = cache + ((size_t)blk * block_size + (t0 & (block_size - 1))) * D;
        const int last = kv_end - 1 - t0;
        const int from = min(FIRST ? max(row, kv_seen - t0) : row, last);
        const uint32_t off = __umul24(from, DKP * 2) + ((place ^ ((row & 3) | ((piece & 1) << 2))) << 4);
#pragma unroll
        for (int i = 0; i < NP; ++i) load_to_lds(g + i * 64, off, lds + (buf * TILE + (piece * NP + i) * 512) * 2);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int f = wave * NI + i, key = f / NP * 8 + row;
        const int c = f % NP * 8 + (place ^ ((key & 3) | ((key >> 1) & 4)));
        const int off = min(FIRST ? max(kv0 + key, kv_seen) : kv0 + key, kv_end - 1) % block_size;
        const int blk = __shfl(blks, key, 64);
        if (c < CH)
          load_to_lds(cache + ((size_t)blk * block_size + off) * D + c * 8, lds + (buf * TILE + f * 512) * 2);
      }
    }
  };

  if (!FULL && CH < CHP) {  // the chunks past a row's end are never fetched
    for (int i = tid; i < LDS / 8; i += 256) reinterpret_cast<u32x4*>(sm)[i] = u32x4{0, 0, 0, 0};
    __syncthreads();
  }
  int blks = kv_lo < kv_hi ? block_of(kv_lo) : 0;
  if (kv_lo < kv_hi) {
    fetch(std::true_type{}, kv_lo, blks, 0);
    blks = block_of(kv_lo + KT);
  }

  // a negative scale goes into the sign of the query
  const uint32_t flip = scale < 0.f ? 0x80008000u : 0u;
  const float c2 = fabsf(scale) * LOG2E;
  bf16x8_t q_frag[KB];
  {
    const uint16_t* qp = q + ((size_t)lo * H + rr) * D;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int d0 = kb * 32 + lg * 8;
      u32x4 raw = u32x4{0, 0, 0, 0};
      if (FULL || d0 < D) raw = *reinterpret_cast<const u32x4*>(qp + d0);
#pragma unroll
      for (int e = 0; e < 4; ++e) raw[e] ^= flip;
      q_frag[kb] = __builtin_bit_cast(bf16x8_t, raw);
    }
  }

  const bool with_sink = sink != nullptr && z == 0 && kg == 0;
  float m = with_sink ? sink[head] * LOG2E : -INFINITY;
  float l = with_sink && lg == 0 ? 1.0f : 0.0f;  // this lane's part of the sum
  f32x4_t acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  int buf = 0;
  for (int kv0 = kv_lo; kv0 < kv_hi; kv0 += KT, buf ^= 1) {
    loads_landed<0>();  // the tile is in LDS, and the other buffer is free
    if (kv0 + KT < kv_hi) {
      fetch(std::false_type{}, kv0 + KT, blks, buf ^ 1);
      blks = block_of(kv0 + 2 * KT);
    }
    const int k0 = kv0 + kg * 32;  // this wave's keys
    if (!wave_active || k0 >= kv_hi) continue;
    const uint16_t* tile = sm + buf * TILE + kg * 32 * DKP;
    // LDS addresses anew for each tile as well: a spilled one is loaded back
    // behind the next tile's fetches, and waits for them
    int here = lane;
    if (KG == 1) asm volatile("" : "+v"(here));
    const int li = here & 15, lg = here >> 4;

    // Operands are read from LDS in batches of 4, the next batch ahead of the
    // products of this one.
    // S^T = K Q^T: tile row li stands for key (li/4)*8 + li%4 (+4 in the second).
    // Two addresses and constants reach all of a row
    f32x4_t s4[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
    {
      const int key = ((li >> 2) << 3) | (li & 3);
      const int f = (key & 3) | ((key >> 1) & 4);  // the same for key + 4
      const uint16_t* row = tile + (key >> 3) * 8 * DKP + (key & 7) * 64;
      const uint16_t* kp[2] = {row + (lg ^ f) * 8, row + ((4 + lg) ^ f) * 8};
      bf16x8_t kf[2][4];
      auto load = [&](int b) {  // steps 2b and 2b+1 of both tiles
#pragma unroll
        for (int j = 0; j < 4; ++j)
          kf[b & 1][j] = __builtin_bit_cast(
              bf16x8_t, *reinterpret_cast<const u32x4*>(kp[j >> 1] + (j & 1) * 4 * 64 + b * 512));
      };
      load(0);
#pragma unroll
      for (int b = 0; b < KB / 2; ++b) {
        if (b + 1 < KB / 2) load(b + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          s4[j & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[b & 1][j], q_frag[b * 2 + (j >> 1)], s4[j & 1], 0, 0, 0);
      }
    }

    // V^T: lane li of a 16-lane group reads 4 entries of key li/4 and receives
    // entry li of keys 0..3
    const int vkey = lg * 8 + (li >> 2);
    const int vf_swz = (vkey & 3) | ((vkey >> 1) & 4);  // the same for key + 4
    const uint16_t* vp[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      vp[j] = tile + (vkey >> 3) * 8 * DKP + (vkey & 7) * 64 + ((j * 2 + ((li >> 1) & 1)) ^ vf_swz) * 8 + (li & 1) * 4;
    bf16x8_t vf[2][4];
    auto load_v = [&](int b) {  // entry blocks 4b .. 4b+3
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint16_t* v0 = vp[j] + b * 512;
        const u32x2 b0 = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)v0));
        const u32x2 b1 = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(v0 + 4 * 64)));
        vf[b & 1][j] = __builtin_bit_cast(bf16x8_t, (u32x4{b0[0], b0[1], b1[0], b1[1]}));
      }
    };
    load_v(0);

    // the other workgroup's products give way to these few instructions, behind which
    // this wave's own wait: 4 prompts of 700-1000 83 -> 79 us, one of 4000 298 -> 292
    if constexpr (KG == 1) __builtin_amdgcn_s_setprio(1);
    // ---- weights of keys k0 + lg*8 + e -----------------------------------------
    const bool masked = k0 + 32 > min(all_end, kv_hi) || k0 < all_lo;
    uint32_t dead = 0;
    if (masked) {
      const int key_lo = window > 0 ? qpos - window + 1 : 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int key = k0 + lg * 8 + e;
        if (key > qpos || key < key_lo || key >= kv_hi) {
          dead |= 1u << e;
          s4[e >> 2][e & 3] = -INFINITY;
        }
      }
    }
    float mx = s4[0][0];
#pragma unroll
    for (int e = 1; e < 8; ++e) mx = fmaxf(mx, s4[e >> 2][e & 3]);
    mx = max_over_groups(mx);
    mx = mx == -INFINITY ? mx : mx * c2;
    if (__any(mx > m)) {
      const float m_new = fmaxf(m, mx);
      const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[db][i] *= alpha;
    }
    const float mm = m == -INFINITY ? 0.f : m;
    float p[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s4[e >> 2][e & 3], c2, -mm));
    if (masked) {
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e] = (dead >> e) & 1 ? 0.f : p[e];
    }
    u32x4 pw;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      l += p[2 * e] + p[2 * e + 1];
      pw[e] = pack_bf16(p[2 * e], p[2 * e + 1]);
    }
    const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, pw);

    if constexpr (KG == 1) __builtin_amdgcn_s_setprio(0);
    // ---- O^T += V^T P^T -----------------------------------------------------------
#pragma unroll
    for (int b = 0; b < DB / 4; ++b) {
      if (b + 1 < DB / 4) load_v(b + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[b * 4 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[b & 1][j], pf, acc[b * 4 + j], 0, 0, 0);
    }
  }

  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  // ---- the second key group hands its sums to the first ---------------------------
  if constexpr (KG > 1) {
    __syncthreads();
    float* fs = reinterpret_cast<float*>(sm) + (rblk * 16 + li) * (DVP + 4);
    if (kg == 1) {
#pragma unroll
      for (int db = 0; db < DB; ++db) *reinterpret_cast<f32x4_t*>(fs + db * 16 + lg * 4) = acc[db];
      if (lg == 0) {
        fs[DVP] = m;
        fs[DVP + 1] = l;
      }
    }
    __syncthreads();
    if (kg == 1) return;
    const float m1 = fs[DVP], l1 = fs[DVP + 1];
    const float gm = fmaxf(m, m1);
    const float w0 = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - gm);
    const float w1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - gm);
    m = gm;
    l = l * w0 + l1 * w1;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const f32x4_t o1 = *reinterpret_cast<const f32x4_t*>(fs + db * 16 + lg * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[db][i] = acc[db][i] * w0 + o1[i] * w1;
    }
  }

  if (nsplit > 1) {
    if (rho >= nrows) return;
    // ---- partial result: unnormalised sums, running max and sum -------------------
    float* pp = partial + (((size_t)lo * H + rho) * nsplit + z) * ((size_t)Dv + LR_PART_PAD);
    if (lg == 0) {
      pp[Dv] = m;
      pp[Dv + 1] = l;
    }
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int d = db * 16 + lg * 4;
      if (FULL || d < Dv) *reinterpret_cast<f32x4_t*>(pp + d) = acc[db];
    }
    return;
  }

  // ---- normalise, gate, store --------------------------------------------------------
  float f = l > 0.f ? 1.0f / l : (l == 0.f ? 0.f : l);
  if (gate != nullptr) f *= sigmoid_fast(bf16_to_f32(gate[(lo + tok) * gate_stride + head]));
  // a lane has 4 entries of each of two blocks: neighbouring groups swap, for 8 of one
  const int col = (lg & 1) * 16 + (lg >> 1) * 8;
  uint16_t* op = out + ((size_t)lo * H + rho) * Dv + col;
#pragma unroll
  for (int db = 0; db < DB; db += 2) {
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const auto both = __builtin_amdgcn_permlane16_swap(pack_bf16(acc[db][2 * e] * f, acc[db][2 * e + 1] * f),
                                                         pack_bf16(acc[db + 1][2 * e] * f, acc[db + 1][2 * e + 1] * f), false, false);
      w[e] = both[0];
      w[2 + e] = both[1];
    }
    if ((FULL || db * 16 + col < Dv) && rho < nrows) *reinterpret_cast<u32x4_of8*>(op + db * 16) = w;
  }
}

// Merge the z-slices of every row: m* = max m_z, out = sum_z 2^(m_z - m*) acc_z
// / sum_z 2^(m_z - m*) l_z.  One wave per row.  Lane z holds slice z's weight
// (up to 64 slices); the lanes then own float4 columns of the value row and
// add up the slices with independent 16-byte loads (slice rows are padded
// to Dv + 4 floats so that they stay 16-byte aligned).
__global__ __launch_bounds__(256) void latent_attention_rows_combine_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ partial,
    const uint16_t* __restrict__ gate, long gate_stride, const int* __restrict__ seg_start, const int* __restrict__ seg_len, int H,
    int Dv, int nsplit) {
  const int s = blockIdx.y;
  const long nrows = (long)seg_len[s] * H;
  const long rho = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (rho >= nrows) return;  // whole waves leave; no workgroup barrier below
  const int lane = threadIdx.x & 63;
  const size_t g = (size_t)seg_start[s] * H + rho;
  const size_t stride = (size_t)Dv + LR_PART_PAD;
  const float* pp = partial + g * nsplit * stride;
  float mz = -INFINITY, lz = 0.f;
  if (lane < nsplit) {
    mz = pp[lane * stride + Dv];
    lz = pp[lane * stride + Dv + 1];
  }
  const float mstar = wave_reduce_max(mz);
  const float wz = (mz == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(mz - mstar);
  const float lsum = wave_reduce_sum(wz * lz);
  float inv = lsum > 0.f ? 1.0f / lsum : 0.f;
  if (gate != nullptr) {
    const long tok = rho / H;
    inv *= sigmoid_fast(bf16_to_f32(gate[(seg_start[s] + tok) * gate_stride + (rho - tok * H)]));
  }
  for (int d0 = 0; d0 < Dv; d0 += 256) {  // uniform trip count: every lane feeds the shuffles
    const int d = d0 + lane * 4;
    const bool act = d < Dv;
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    const float* col = pp + (act ? d : 0);
    int zz = 0;
    for (; zz + 4 <= nsplit; zz += 4) {  // four slices' loads in flight at a time
      f32x4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const f32x4*>(col + (zz + u) * stride);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float w = __shfl(wz, zz + u, 64);
        a0 += w * v[u][0];
        a1 += w * v[u][1];
        a2 += w * v[u][2];
        a3 += w * v[u][3];
      }
    }
    for (; zz < nsplit; ++zz) {
      const float w = __shfl(wz, zz, 64);
      const f32x4 v = *reinterpret_cast<const f32x4*>(col + zz * stride);
      a0 += w * v[0];
      a1 += w * v[1];
      a2 += w * v[2];
      a3 += w * v[3];
    }
    if (!act) continue;
    uint2 packed;
    packed.x = (uint32_t)f32_to_bf16(a0 * inv) | ((uint32_t)f32_to_bf16(a1 * inv) << 16);
    packed.y = (uint32_t)f32_to_bf16(a2 * inv) | ((uint32_t)f32_to_bf16(a3 * inv) << 16);
    *reinterpret_cast<uint2*>(out + g * Dv + d) = packed;
  }
}

}  // namespace

// Returns 0 when launched, 1 when the shape is not served (the caller then
// uses another kernel).
extern "C" int lig_latent_attention_rows(
    void* out, const void* q, const void* cache, const float* sink,
    const void* gate, long gate_stride,
    const int* seg_start, const int* seg_len, const int* seg_ctx,
    const int* block_tables, int max_blocks, float scale, int num_segs,
    int max_seg_len, int H, int D, int Dv, int block_size, int window, int nsplit,
    float* partial, hipStream_t stream) {
  if (D % 8 != 0 || Dv % 8 != 0 || D <= 0 || Dv <= 0 || Dv > D || D > 576 ||
      Dv > 512 || !aligned16(q) || !aligned16(cache) || H <= 0)
    return 1;
  if (num_segs <= 0 || max_seg_len <= 0) return 0;
  // one token of up to 32 heads: all four waves on 32 rows
  const bool few = (long)max_seg_len * H <= 32;
  const int rows = few ? 32 : 64;
  const long tiles = ((long)max_seg_len * H + rows - 1) / rows;
  const int shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz((unsigned)block_size) : -1;
  if (tiles > 2147483647L || num_segs > 65535) return 1;
  if (nsplit < 1 || nsplit > 64 || (nsplit > 1 && partial == nullptr)) return 1;
  dim3 grid((unsigned)tiles, num_segs, nsplit);
  dim3 block(256);
#define LAUNCH_LR_KG(DKP, DVP, KG, FULL)                                                      \
  hipLaunchKernelGGL((latent_attention_rows_kernel<DKP, DVP, KG, FULL>), grid, block, 0,      \
                     stream, (uint16_t*)out, (const uint16_t*)q, (const uint16_t*)cache, sink, \
                     (const uint16_t*)gate, gate_stride, seg_start, seg_len, seg_ctx,         \
                     block_tables, max_blocks, scale, H, D, Dv, block_size, shift, window,    \
                     nsplit, partial)
#define LAUNCH_LR(DKP, DVP)                                \
  do {                                                     \
    const bool full = D == DKP && Dv == DVP && shift >= 3; \
    if (few && full)                                       \
      LAUNCH_LR_KG(DKP, DVP, 2, true);                     \
    else if (few)                                          \
      LAUNCH_LR_KG(DKP, DVP, 2, false);                    \
    else if (full)                                         \
      LAUNCH_LR_KG(DKP, DVP, 1, true);                     \
    else                                                   \
      LAUNCH_LR_KG(DKP, DVP, 1, false);                    \
  } while (0)
  if (D <= 64 && Dv <= 64) LAUNCH_LR(64, 64);
  else if (D <= 128 && Dv <= 64) LAUNCH_LR(128, 64);
  else if (D <= 128) LAUNCH_LR(128, 128);
  else if (D <= 192 && Dv <= 128) LAUNCH_LR(192, 128);
  else if (D <= 320 && Dv <= 256) LAUNCH_LR(320, 256);
  else LAUNCH_LR(576, 512);
#undef LAUNCH_LR
#undef LAUNCH_LR_KG
  if (nsplit > 1) {
    const long rows4 = ((long)max_seg_len * H + 3) / 4;
    hipLaunchKernelGGL(latent_attention_rows_combine_kernel,
                       dim3((unsigned)rows4, num_segs), dim3(256), 0, stream,
                       (uint16_t*)out, partial, (const uint16_t*)gate, gate_stride, seg_start, seg_len, H, Dv, nsplit);
  }
  return 0;
}
