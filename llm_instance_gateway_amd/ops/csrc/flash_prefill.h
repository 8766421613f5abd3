// Paged flash attention over prompt portions on MFMA tiles: bf16, key and
// value heads of the same size 64 or 128, gfx950.  Shared by the Llama path
// (torch extension) and the hybrid families' path (light library).
//
// What bounds it: at a few thousand keys the two contractions, 4 * D flops per
// (row, key) pair and head.  The kernel this replaces gave a workgroup ONE
// query head and 16 rows per wave, so every 16 rows of every head read the K
// and V tile from LDS again, and its scores went through LDS between the two
// products.  Here
//   * a workgroup serves a tile of 64 query rows of GH heads of one key/value
//     head, a wave RB = GH blocks of 16 rows of one of them, so an operand
//     read from LDS feeds RB matrix instructions.  Two heads where that still
//     gives every CU two workgroups, else one (heads_of_workgroup);
//   * keys are dealt to the rows of the S^T = K Q^T tiles in the order in
//     which a lane's scores ARE the operand of O^T += V^T P^T (rows g*4+i of
//     two tiles hold keys g*8+i and g*8+4+i), so the weights never leave the
//     registers, and row statistics are one scalar per lane for both products;
//   * heads of 128: rows go from memory straight into LDS (load_to_lds), the next 64
//     keys while the current ones are used, V transposed by the reads; chunks are
//     XOR-swizzled by key through the choice of what a lane fetches, so that no read
//     meets a bank twice.  Heads of 64 and odd block sizes: through registers, V
//     transposed by byte permutes.  LDS is double-buffered: one barrier per 64 keys;
//   * the accumulators are only rescaled when a row's maximum grew, and masks
//     are only evaluated on tiles that cross a row's visible range.
// Measured so far, 32 query and 8 key/value heads of 128, with rows still through
// registers, against the kernel this replaces: 4096 rows on 4000 cached keys 3409 ->
// 495 us (820 TFLOP/s; 571 between the products of an engine step); 20 prompts of
// 200 130 -> 37 us; one of 202 20.6 -> 8.9 us; 8 of 1000 with a window of 512 571 ->
// 110 us, with a soft cap 578 -> 133, with sigmoid weights 566 -> 103.
// What then bound it were vector instructions (64 % of the cycles, and LDS 53 %, half
// of that conflicts).  Without selects for masked keys, with pairs rounded at once,
// rows by DMA and their block's row number worked out once per group of keys: 4000
// rows on 4000 keys 560 -> 441 us (between products), 20 prompts of 200 37 -> 33, one
// of 202 8.9 -> 7.9, 8 of 1000 with the window and a cap 120 -> 96.
// A cap's tanh goes into the weight's exponent as it comes: 8 of 1000 with the window and a cap,
// replayed without pauses, 95.8 -> 93.3 us, 3 of 1500 59.3 -> 58.0; results are rounded unlike, 1e-4
// apart.  Weights are summed in fp32, ahead of their rounding; summed as the matrix cores see them,
// two to an instruction, they took as long (8 of 1000 with the window and a cap 93.3 us, unrounded 92.5; 4000
// rows of one prompt 150.7, 152.4; 24 of 640 107.5, 107.4; steps level).
// Results in 16-byte pieces, a lane's four entries of a block swapped with its neighbour's for
// eight, instead of 8-byte ones: 20 prompts of 200 28.3 -> 24.4, 24 of 640 118 -> 107, 40 of 400 99.8 ->
// 87.5; 8 of 1000 with the window and a cap, their tiles in turn by length as well, 94 -> 85.
// Matrix and vector instructions hardly overlap (24 and 64 % of the cycles).  Products of the next
// tile between the weights of this one spilled registers (121 us); three workgroups per CU,
// values in one buffer, at 168 registers did too (107).
// Four heads per workgroup and 64 rows per wave (all 512 registers, one wave
// per SIMD) was slower everywhere: 781 us in the first of these.
#pragma once

#include <algorithm>

#include "common.h"

namespace flash_prefill {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_of8 __attribute__((ext_vector_type(4), aligned(8)));  // outputs are not asked for more

constexpr int KT = 64;      // keys per tile
constexpr int TQ = 64;      // query rows of a tile of the caller's tile list

struct Args {
  uint16_t* out;            // [R, Hq * D]
  const uint16_t* q;        // rows q_stride entries apart
  long q_stride;
  const uint16_t* k_cache;  // [blocks, Hkv, BS, D]
  const uint16_t* v_cache;  // rows v_row entries apart
  const uint16_t* gate;     // nullable
  long gate_stride;
  const float* sink;        // nullable, [Hq]
  const int* tile_seq;
  const int* tile_qstart;
  const int* query_start_locs;
  const int* context_lens;
  const int* block_tables;
  const float* score_bias;  // nullable, [Hq]
  float scale;
  float temp_coef, temp_every;
  int temp_every_int;
  int num_q_heads, num_kv_heads;
  int v_row;
  int block_size, block_shift;  // block_shift < 0: not a power of two
  int max_blocks;
  int num_seqs;             // portions that query_start_locs and context_lens hold
  int chunk, window;
  int gate_per_head;
  float softcap;
  int turns;                // tiles take their turns by length: the most 64-key steps one walks, 0: they don't
  int nsplit;               // SPLIT: parts of a tile's keys, and
  float* partial;           // [R, Hq, nsplit, D + 4]: sums of weighted values, then largest score (log2) and sum of weights
};

// Tiles of keys to a part where nt are cut into nsplit: the last parts may be empty, as
// are all where a context is shorter than its own rows and a tile sees no key (nt <= 0).
LIG_DEVICE int tiles_of_part(int nt, int nsplit) { return max(1, (nt + nsplit - 1) / nsplit); }

// Where the 16-byte chunks of key t's row, and (not DMA) of entry d's row of keys,
// lie: chunk c at c ^ swizzle.  The reads of 16 lanes (0-3, 12-15 and of the next 16
// 4-11, or the others) then meet all 64 banks, as do V's transposing reads of 8 keys,
// whose pairs of chunks are spread by 2 ((t & 3) | (t / 8 % 2) * 4).
template <int D>
LIG_DEVICE int key_swizzle(int t) {
  return D == 128 ? (t & 3) | ((t >> 1) & 12) : (t & 3) | ((t >> 1) & 4);
}
LIG_DEVICE int entry_swizzle(int d) { return (d ^ (d >> 3)) & 7; }

LIG_DEVICE u32x2 transposed(const uint16_t* p) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p));
}

// The oldest key that some row of a tile whose first row is at qpos0 sees.
template <bool EXTRA>
LIG_DEVICE int oldest_key(const Args& a, int qpos0) {
  int first = 0;
  if (EXTRA) {
    if (a.chunk > 0) first = (qpos0 / a.chunk) * a.chunk;
    if (a.window > 0) first = max(first, qpos0 - a.window + 1);
    first = max(first, 0);
  }
  return first;
}

// Which tile of the list is this workgroup's: the longest walks first, so that the last
// workgroups to begin are the shortest; of equal ones the last in the list first.  Lane i
// brings portion i's numbers in the round of loads that brings the list.
constexpr int TURN_TILES = 256, TURN_SEQS = 63;  // at most: a lane for each portion and the end of the last
template <bool EXTRA>
LIG_DEVICE void tile_in_turn(const Args& a, int& seq, int& qt) {
  constexpr int MOST = TURN_TILES / 64;
  const int lane = threadIdx.x & 63, nt = gridDim.y, longest = a.turns;
  const int first = a.query_start_locs[min(lane, a.num_seqs)], held = a.context_lens[min(lane, a.num_seqs - 1)];
  int s[MOST], q[MOST], key[MOST];
#pragma unroll
  for (int j = 0; j < MOST; ++j) {
    if (j * 64 >= nt) continue;
    const int at = max(nt - 1 - (j * 64 + lane), 0);
    s[j] = a.tile_seq[at];
    q[j] = a.tile_qstart[at];
  }
#pragma unroll
  for (int j = 0; j < MOST; ++j) {
    key[j] = -1;
    if (j * 64 >= nt) continue;
    const int n = __shfl(first, s[j] + 1, 64) - __shfl(first, s[j], 64), ctx = __shfl(held, s[j], 64);
    const int qpos0 = ctx - n + q[j];
    const int steps = (min(ctx, qpos0 + TQ) + KT - 1) / KT - oldest_key<EXTRA>(a, qpos0) / KT;
    if (j * 64 + lane < nt) key[j] = q[j] < n ? min(max(steps, 0), longest) : 0;
  }
  auto from = [&](int k) {  // tiles with that key or a higher one
    int c = 0;
#pragma unroll
    for (int j = 0; j < MOST; ++j)
      if (j * 64 < nt) c += __popcll(__ballot(key[j] >= k));
    return c;
  };
  const int turn = blockIdx.y;
  int k = 0;  // the highest key from which on there are more than `turn` tiles
  for (int bit = 1 << (31 - __builtin_clz(longest)); bit > 0; bit >>= 1)
    if (from(k + bit) > turn) k += bit;
  int before = turn - from(k + 1);
#pragma unroll
  for (int j = 0; j < MOST; ++j) {
    if (j * 64 >= nt) continue;
    const uint64_t have = __ballot(key[j] == k);
    const int at = __builtin_amdgcn_mbcnt_hi((uint32_t)(have >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)have, 0));
    const uint64_t mine = __ballot(key[j] == k && at == before);
    if (mine) {
      const int l = __builtin_ctzll(mine);
      seq = __builtin_amdgcn_readlane(s[j], l);
      qt = __builtin_amdgcn_readlane(q[j], l);
      return;
    }
    before -= __popcll(have);
  }
}

// PB: block size a power of two, at least 4.  CAP: scores bent by softcap * tanh(score / softcap).  SIG: unnormalised
// sigmoid(score + bias) weights.  EXTRA: temperature, gate, sink, chunk and
// window are looked at (the plain causal kernel leaves them out).  SPLIT: blockIdx.z
// walks its part of the keys only and leaves sums that flash_prefill_merge_kernel adds up.
template <int D, int GH, bool PB, bool CAP, bool SIG, bool EXTRA, bool SPLIT = false>
__global__ __launch_bounds__(256, 2) void flash_prefill_kernel(const Args a) {
  constexpr int RB = GH;       // blocks of 16 rows per wave

  constexpr int KS = D / 32;   // matrix steps over the head size
  constexpr int DB = D / 16;   // blocks of 16 output entries
  constexpr int CH = D / 8;    // 16-byte chunks of a row
  constexpr int TPT = KT * CH / 256;  // keys a thread stages: 4 (D = 128) or 2
  constexpr bool DMA = PB && D == 128;  // rows go straight into LDS, 4 to an instruction
  static_assert(!SPLIT || !(CAP || SIG || EXTRA), "parts of the plain causal kernel");
  static_assert(16 * RB * (4 / GH) == TQ, "a workgroup serves one query tile of each of its heads");

  struct Shared {
    uint16_t K[2][KT * D];
    uint16_t VT[2][D * KT];  // DMA: V as it lies in memory, [KT][D]
  };
  __shared__ Shared sm;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15;
  const int lg = lane >> 4;

  // grid.x runs over the head groups, so that with a multiple of 8 of them
  // every XCD keeps to some heads' keys in its own L2
  int s, qt;
  if (!SPLIT && a.turns > 0) {
    tile_in_turn<EXTRA>(a, s, qt);
  } else {  // backwards, so that of one prompt the rows with the most keys start first
    s = a.tile_seq[gridDim.y - 1 - blockIdx.y];
    qt = a.tile_qstart[gridDim.y - 1 - blockIdx.y];
  }
  const int lo = a.query_start_locs[s];
  const int n = a.query_start_locs[s + 1] - lo;
  if (qt >= n || n <= 0) return;
  const int ctx = a.context_lens[s];
  const int* bt = a.block_tables + (size_t)s * a.max_blocks;
  const int group = a.num_q_heads / a.num_kv_heads;
  const int per_kv = group / GH;
  const int kvh = blockIdx.x / per_kv;
  const int h = kvh * group + (blockIdx.x % per_kv) * GH + wave % GH;
  const int row0 = qt + (wave / GH) * (16 * RB);  // first row of this wave in the portion

  // ---- rows of this wave: row rb*16 + li belongs to this lane ---------------
  bf16x8_t q_frag[RB][KS];
  float c[RB];         // log2 units per unit of the raw score; CAP: twice those of the score over the cap
  int key_lo[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int r = row0 + rb * 16 + li;
    const int rr = r < n ? r : n - 1;
    const int qpos = ctx - n + rr;
    float sc = a.scale;
    key_lo[rb] = 0;
    if (EXTRA) {
      if (a.temp_coef != 0.f) {
        const float m = a.temp_every_int > 0 ? (float)((qpos + 1) / a.temp_every_int)
                                             : floorf((float)(qpos + 1) / a.temp_every);
        sc *= 1.f + a.temp_coef * logf(m + 1.f);
      }
      if (a.chunk > 0) key_lo[rb] = (qpos / a.chunk) * a.chunk;
      if (a.window > 0) key_lo[rb] = max(key_lo[rb], qpos - a.window + 1);
    }
    // a negative scale goes into the sign of the query, so that the largest
    // raw score is the largest scaled one
    const uint32_t flip = sc < 0.f ? 0x80008000u : 0u;
    sc = fabsf(sc);
    // not zero: a masked score is minus infinity, and stays so times c
    c[rb] = CAP ? sc / a.softcap * (2.f * LOG2E) : fmaxf(sc * LOG2E, 1e-30f);
    const uint16_t* qp = a.q + (size_t)(lo + rr) * a.q_stride + (size_t)h * D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      u32x4 raw = *reinterpret_cast<const u32x4*>(qp + ks * 32 + lg * 8);
#pragma unroll
      for (int e = 0; e < 4; ++e) raw[e] ^= flip;
      q_frag[rb][ks] = __builtin_bit_cast(bf16x8_t, raw);
    }
  }
  const float bias = SIG && a.score_bias ? a.score_bias[h] * LOG2E : 0.f;
  const float cap2 = CAP ? a.softcap * LOG2E : 0.f;

  float m[RB], l[RB];
  f32x4_t acc[RB][DB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    m[rb] = -INFINITY;
    l[rb] = 0.f;
    if (EXTRA && !SIG && a.sink) {
      // a key with that unscaled score and no value; each lane sums its own keys, so
      // only one of the four groups starts with it
      m[rb] = a.sink[h] * LOG2E;
      l[rb] = lg == 0 ? 1.f : 0.f;
    }
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[rb][db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  // ---- walk ------------------------------------------------------------------
  const int qpos0 = ctx - n + qt;
  const int kv_end = min(ctx, qpos0 + TQ);
  if (kv_end <= 0) {
    // a context shorter than its own rows, of which this tile's see no key: nothing to fetch ahead
    if constexpr (!SPLIT) {
      const int h0 = kvh * group + (blockIdx.x % per_kv) * GH;
      for (int i = tid; i < TQ * GH * (D / 4); i += 256) {
        const int r = qt + i / (GH * (D / 4));
        uint16_t* op = a.out + ((size_t)(lo + r) * a.num_q_heads + h0) * D + i % (GH * (D / 4)) * 4;
        if (r < n) *reinterpret_cast<u32x2*>(op) = u32x2{0, 0};
      }
    }
    return;
  }
  const int first_key = oldest_key<EXTRA>(a, qpos0);
  int kv_begin = first_key & ~(KT - 1), kv_stop = kv_end;
  if constexpr (SPLIT) {
    const int part = tiles_of_part((kv_end + KT - 1) / KT, a.nsplit) * KT;
    kv_begin = blockIdx.z * part;
    if (kv_begin >= kv_end) return;
    kv_stop = min(kv_end, kv_begin + part);
  }
  const int wave_first = ctx - n + row0;                                   // position of the wave's first row
  const int wave_last_lo = __builtin_amdgcn_readlane(key_lo[RB - 1], 15);  // largest lower bound

  // staging: this thread brings chunk `ch` of keys st*TPT .. +TPT
  const int ch = tid % CH;
  const int st = tid / CH;
  const size_t kv_head_rows = (size_t)kvh * a.block_size;
  const size_t block_rows = (size_t)a.num_kv_heads * a.block_size;
  u32x4 kreg[TPT], vreg[TPT];

  // Keys that no row of the tile sees are replaced by the nearest one that some
  // row does: their weight is zero, but what they hold would still meet it in a
  // product, and the blocks before may be gone.  PB: the TPT keys of a thread lie
  // in one block (tiles start at multiples of 64), whose number is read one tile
  // ahead; no branch may stand between the loads, or each would be waited for
  auto visible = [&](int t) { return min(EXTRA ? max(t, first_key) : t, kv_end - 1); };
  auto block_of = [&](int kv0) { return PB ? bt[visible(kv0 + st * TPT) >> a.block_shift] : 0; };
  auto fetch = [&](int kv0, int blk) {
    if constexpr (PB) {
      const size_t rows = (size_t)blk * block_rows + kv_head_rows;
      const uint16_t* kb = a.k_cache + rows * D + ch * 8;
      const uint16_t* vb = a.v_cache + rows * a.v_row + ch * 8;
      int row[TPT];
#pragma unroll
      for (int i = 0; i < TPT; ++i) row[i] = visible(kv0 + st * TPT + i) & (a.block_size - 1);
#pragma unroll
      for (int i = 0; i < TPT; ++i) {
        kreg[i] = *reinterpret_cast<const u32x4*>(kb + row[i] * D);
        vreg[i] = *reinterpret_cast<const u32x4*>(vb + (size_t)(uint32_t)row[i] * (uint32_t)a.v_row);
      }
    } else {
      size_t row[TPT];
#pragma unroll
      for (int i = 0; i < TPT; ++i) {
        const int t = visible(kv0 + st * TPT + i), b = t / a.block_size;
        row[i] = (size_t)bt[b] * block_rows + kv_head_rows + (t - b * a.block_size);
      }
#pragma unroll
      for (int i = 0; i < TPT; ++i) {
        kreg[i] = *reinterpret_cast<const u32x4*>(a.k_cache + row[i] * D + ch * 8);
        vreg[i] = *reinterpret_cast<const u32x4*>(a.v_cache + row[i] * a.v_row + ch * 8);
      }
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TPT; ++i) {
      const int t = st * TPT + i;
      const int f = key_swizzle<D>(t);
      *reinterpret_cast<u32x4*>(&sm.K[buf][t * D + ((ch ^ f) * 8)]) = kreg[i];
    }
    // entry e of key i -> row ch*8+e, key i; eight 16-byte units of 8 keys per row
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int d = ch * 8 + e;
      const int unit = ((st * TPT) >> 3) ^ entry_swizzle(d);
      uint16_t* p = &sm.VT[buf][d * KT + unit * 8 + ((st * TPT) & 7)];
      const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
      if constexpr (TPT == 4) {
        u32x2 w;
        w[0] = __builtin_amdgcn_perm(vreg[1][e / 2], vreg[0][e / 2], sel);
        w[1] = __builtin_amdgcn_perm(vreg[3][e / 2], vreg[2][e / 2], sel);
        *reinterpret_cast<u32x2*>(p) = w;
      } else {
        *reinterpret_cast<uint32_t*>(p) = __builtin_amdgcn_perm(vreg[1][e / 2], vreg[0][e / 2], sel);
      }
    }
  };

  // ---- DMA: a wave brings keys wave * 16 .. +16, four to an instruction (a block holds
  // at least 4), whose 16 lanes a row choose the chunk that belongs to their place.
  // Lane j knows the block of the tile's keys 4 j .. +4, read one tile ahead.  Tiles
  // with all 64 keys visible take one offset per pair of fetches, the others clamp.
  const uint32_t lds_k = lds_address(sm.K), lds_v = lds_address(sm.VT);
  const int place = lane & 15, quarter = lane >> 4;  // chunk's place; row of the four
  uint32_t k_off[2], v_off[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    k_off[j] = ((place ^ (quarter | ((wave * 2 + j) & 3) << 2)) << 4) + quarter * (D * 2);
    v_off[j] = ((place ^ ((quarter | j << 2) << 1)) << 4) + quarter * (uint32_t)a.v_row * 2;
  }
  auto blocks_of = [&](int kv0) { return bt[visible(kv0 + (lane & 15) * 4) >> a.block_shift]; };
  auto fetch_dma = [&](int kv0, int blks, int buf) {
    // offsets have no sign: where keys are clamped they count from the block's first row
    const bool whole = kv0 + KT <= kv_end && (!EXTRA || kv0 >= first_key);
    // cache rows of 256 bytes and more: their number has 32 bits
    const uint32_t first = (uint32_t)blks * (uint32_t)block_rows + (uint32_t)kv_head_rows +
                           (whole ? (kv0 + (lane & 15) * 4) & (a.block_size - 1) : 0);
    auto bring = [&](int j, uint32_t ko, uint32_t vo) __attribute__((always_inline)) {
      const uint32_t row = __builtin_amdgcn_readlane(first, wave * 4 + j);
      const uint32_t to = (buf * KT + wave * 16 + j * 4) * D * 2;
      load_to_lds(a.k_cache + (size_t)row * D, ko, lds_k + to);
      load_to_lds(a.v_cache + (size_t)row * (uint32_t)a.v_row, vo, lds_v + to);
    };
    if (whole) {
#pragma unroll
      for (int j = 0; j < 4; ++j) bring(j, k_off[j >> 1], v_off[j >> 1]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = visible(kv0 + wave * 16 + j * 4 + quarter) & (a.block_size - 1), d = row - quarter;
        bring(j, k_off[j >> 1] + d * (D * 2), v_off[j >> 1] + d * a.v_row * 2);
      }
    }
  };

  int blk_next = DMA ? blocks_of(kv_begin) : block_of(kv_begin);
  if constexpr (DMA) {
    fetch_dma(kv_begin, blk_next, 0);
    blk_next = blocks_of(kv_begin + KT);
  } else {
    fetch(kv_begin, blk_next);
    blk_next = block_of(kv_begin + KT);
    stage(0);
    __syncthreads();
  }

  // A wave behind the portion's last row only stages, tile for tile with the
  // others, in a loop of its own: a branch in the one below costs full tiles 2 to
  // 5 %.  300 portions of 3 rows on 60 keys 34.5 -> 30.8 us (32 query and 8 key/value
  // heads of 64), 21.5 -> 16.4 (16 and 16), 53 -> 49.5 (32 and 8 of 128), 200 of 20
  // 29.5 -> 26.8, 16.5 -> 15.9, 43.8 -> 42.4.  The kernel before took 27.9, 15.9,
  // 70.8 and 24.6, 14.4, 56.7: with heads of 64 it fits more workgroups on a CU.
  if (row0 >= n) {
    for (int kv0 = kv_begin, buf = 1; kv0 < kv_stop; kv0 += KT, buf ^= 1) {
      if constexpr (DMA) loads_landed<0>();
      if (kv0 + KT < kv_stop) {
        if constexpr (DMA) {
          fetch_dma(kv0 + KT, blk_next, buf);
          blk_next = blocks_of(kv0 + 2 * KT);
        } else {
          fetch(kv0 + KT, blk_next);
          blk_next = block_of(kv0 + 2 * KT);
          stage(buf);
        }
      }
      if constexpr (!DMA) __syncthreads();
    }
    return;
  }

  int buf = 0;
  for (int kv0 = kv_begin; kv0 < kv_stop; kv0 += KT, buf ^= 1) {
    const bool more = kv0 + KT < kv_stop;
    if constexpr (DMA) loads_landed<0>();  // this tile is in LDS, and the other buffer is free
    if (more) {
      if constexpr (DMA) {
        fetch_dma(kv0 + KT, blk_next, buf ^ 1);
        blk_next = blocks_of(kv0 + 2 * KT);
      } else {
        fetch(kv0 + KT, blk_next);
        blk_next = block_of(kv0 + 2 * KT);
      }
    }

    // ---- S^T = K Q^T --------------------------------------------------------------
    // s[rb][t2][x][i]: key kv0 + t2*32 + lg*8 + x*4 + i of row rb*16 + li
    f32x4_t s4[RB][2][2];
    {
      // tile row li stands for key (li/4)*8 + li%4 (+4 in the second tile)
      const int key_row = ((li >> 2) << 3) | (li & 3);
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const int t = t2 * 32 + key_row + x * 4;
          const int f = key_swizzle<D>(t);
          bf16x8_t kf[KS];
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
            kf[ks] = __builtin_bit_cast(
                bf16x8_t, *reinterpret_cast<const u32x4*>(&sm.K[buf][t * D + (((ks * 4 + lg) ^ f) * 8)]));
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) {
            s4[rb][t2][x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
              s4[rb][t2][x] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks], q_frag[rb][ks], s4[rb][t2][x], 0, 0, 0);
          }
        }
      }
    }

    // ---- weights -------------------------------------------------------------------
    const bool masked = kv0 + KT - 1 > wave_first || kv0 < wave_last_lo;
    bf16x8_t p_frag[RB][2];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float(&v)[16] = reinterpret_cast<float(&)[16]>(s4[rb]);  // key kv0 + (e / 8) * 32 + lg * 8 + e % 8
      // softcap * tanh(score * scale / softcap) is cap2 + 2 cap2 v in log2 units, which the
      // weight's exponent takes as it is
      if constexpr (CAP) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = __builtin_amdgcn_rcpf(-1.f - __builtin_amdgcn_exp2f(v[e] * c[rb]));
      }
      // a masked score's weight is 2^-inf or 1 / (1 + 2^inf): no further select
      if (masked) {
        const int first = kv0 + lg * 8;
        const int last = min(ctx - n + row0 + rb * 16 + li, ctx - 1) - first, low = key_lo[rb] - first;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int k = (e >> 3) * 32 + (e & 7);
          if (k > last || (EXTRA && k < low)) v[e] = -INFINITY;
        }
      }
      if constexpr (!SIG) {
        float mx = v[0];
#pragma unroll
        for (int e = 1; e < 16; ++e) mx = fmaxf(mx, v[e]);
        mx = max_over_groups(mx);
        mx = CAP ? __builtin_fmaf(mx, 2.f * cap2, cap2) : mx * c[rb];
        if (__any(mx > m[rb])) {
          const float m_new = fmaxf(m[rb], mx);
          const float alpha = m[rb] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[rb] - m_new);
          m[rb] = m_new;
          l[rb] *= alpha;
#pragma unroll
          for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[rb][db][i] *= alpha;
        }
      }
      const float mm = m[rb] == -INFINITY ? 0.f : m[rb];
      float p[16];
      const float slope = CAP ? 2.f * cap2 : c[rb];
      const float level = SIG ? (CAP ? -cap2 - bias : -bias) : (CAP ? cap2 - mm : -mm);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        if constexpr (SIG) p[e] = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(__builtin_fmaf(v[e], -slope, level)));
        else p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(v[e], slope, level));
      }
      if constexpr (!SIG) {
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) sum += p[e];
        l[rb] += sum;
      }
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        u32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = pack_bf16(p[t2 * 8 + 2 * e], p[t2 * 8 + 2 * e + 1]);
        p_frag[rb][t2] = __builtin_bit_cast(bf16x8_t, w);
      }
    }

    // ---- O^T += V^T P^T --------------------------------------------------------------
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        bf16x8_t vf;
        if constexpr (DMA) {
          // lane li of 16 reads 4 entries of key li / 4 and receives entry li of keys 0..3
          const int key = t2 * 32 + lg * 8 + (li >> 2), w = (li >> 2) | (lg & 1) << 2;
          const uint16_t* v0 = &sm.VT[buf][key * D + (db ^ w) * 16 + (li & 3) * 4];
          const u32x2 b0 = transposed(v0), b1 = transposed(v0 + 4 * D);
          vf = __builtin_bit_cast(bf16x8_t, (u32x4{b0[0], b0[1], b1[0], b1[1]}));
        } else {
          const int d = db * 16 + li;
          const int unit = (t2 * 4 + lg) ^ entry_swizzle(d);
          vf = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(&sm.VT[buf][d * KT + unit * 8]));
        }
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          acc[rb][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, p_frag[rb][t2], acc[rb][db], 0, 0, 0);
      }
    }

    if constexpr (!DMA) {
      if (more) stage(buf ^ 1);
      __syncthreads();
    }
  }

  // ---- normalise, gate, store: this lane holds entries db*16 + lg*4 + i of its row ----
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int r = row0 + rb * 16 + li;
    float f = 1.f;
    if constexpr (!SIG) {
      float t = l[rb];
      t += __shfl_xor(t, 16, 64);
      t += __shfl_xor(t, 32, 64);
      f = t > 0.f ? 1.f / t : (t == 0.f ? 0.f : t);
      if constexpr (SPLIT) {
        if (r >= n) continue;
        float* sp = a.partial + (((size_t)(lo + r) * a.num_q_heads + h) * a.nsplit + blockIdx.z) * (D + 4);
#pragma unroll
        for (int db = 0; db < DB; ++db) *reinterpret_cast<f32x4_t*>(sp + db * 16 + lg * 4) = acc[rb][db];
        if (lg == 0) {
          sp[D] = m[rb];
          sp[D + 1] = t;
        }
        continue;
      }
    }
    const bool stored = r < n;
    const int rr = stored ? r : n - 1;
    const uint16_t* gp = nullptr;
    if (EXTRA && a.gate) {
      gp = a.gate + (size_t)(lo + rr) * a.gate_stride;
      if (a.gate_per_head) {
        f *= __builtin_amdgcn_rcpf(1.f + __expf(-bf16_to_f32(gp[h])));
        gp = nullptr;
      } else {
        gp += (size_t)h * D;
      }
    }
    // a lane has 4 entries of each of two blocks: neighbouring groups swap, for 8 of one
    uint16_t* op = a.out + ((size_t)(lo + rr) * a.num_q_heads + h) * D + (lg & 1) * 16 + (lg >> 1) * 8;
#pragma unroll
    for (int db = 0; db < DB; db += 2) {
      uint32_t pair[2][2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          o[i] = acc[rb][db + x][i] * f;
          if (EXTRA && gp) o[i] *= __builtin_amdgcn_rcpf(1.f + __expf(-bf16_to_f32(gp[(db + x) * 16 + lg * 4 + i])));
        }
        pair[x][0] = pack_bf16(o[0], o[1]);
        pair[x][1] = pack_bf16(o[2], o[3]);
      }
      u32x4 w;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const auto both = __builtin_amdgcn_permlane16_swap(pair[0][e], pair[1][e], false, false);
        w[e] = both[0];
        w[2 + e] = both[1];
      }
      if (stored) *reinterpret_cast<u32x4_of8*>(op + db * 16) = w;
    }
  }
}

// Adds up the parts of every (row, head) of a tile, 4 entries per lane.
template <int D>
__global__ __launch_bounds__(256) void flash_prefill_merge_kernel(const Args a) {
  constexpr int LP = D / 4;
  const int s = a.tile_seq[blockIdx.y], qt = a.tile_qstart[blockIdx.y];
  const int lo = a.query_start_locs[s], n = a.query_start_locs[s + 1] - lo;
  const int item = blockIdx.x * (256 / LP) + threadIdx.x / LP;
  const int r = qt + item / a.num_q_heads, h = item % a.num_q_heads;
  if (item >= TQ * a.num_q_heads || r >= n) return;
  const int ctx = a.context_lens[s];
  const int nt = (min(ctx, ctx - n + qt + TQ) + KT - 1) / KT, per = tiles_of_part(nt, a.nsplit);
  const int parts = (nt + per - 1) / per;
  const int d = (threadIdx.x % LP) * 4;
  const float* base = a.partial + ((size_t)(lo + r) * a.num_q_heads + h) * a.nsplit * (D + 4);
  float m = -INFINITY, l = 0.f;
  for (int z = 0; z < parts; ++z) m = fmaxf(m, base[(size_t)z * (D + 4) + D]);
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int z = 0; z < parts; ++z) {
    const float* sp = base + (size_t)z * (D + 4);
    const float f = sp[D] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sp[D] - m);
    l += sp[D + 1] * f;
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(sp + d);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] += v[i] * f;
  }
  const float f = l > 0.f ? 1.f / l : (l == 0.f ? 0.f : l);
  u32x2 w;
  w[0] = pack_bf16(o[0] * f, o[1] * f);
  w[1] = pack_bf16(o[2] * f, o[3] * f);
  *reinterpret_cast<u32x2*>(a.out + ((size_t)(lo + r) * a.num_q_heads + h) * D + d) = w;
}

// What the kernel takes.  The Llama path has no other kernel and does not ask: its
// binding admits contiguous bf16 tensors with heads of 64 or 128 only, and relies
// on the allocator's alignment and on head counts that divide.
static inline bool serves(const Args& a, int D, int Dv) {
  auto al = [](const void* p, unsigned to) { return (reinterpret_cast<uintptr_t>(p) & (to - 1)) == 0; };
  return D == Dv && (D == 64 || D == 128) && a.q_stride % 8 == 0 && a.v_row % 8 == 0 && a.v_row >= D &&
         al(a.q, 16) && al(a.k_cache, 16) && al(a.v_cache, 16) && al(a.out, 8);
}

// Two heads per workgroup halve the reads of K and V; the line is where
// that leaves two workgroups for every CU (heads of 128, 32 over 8; two heads
// against one): 1280 workgroups 37.5 us against 44.0, 512 of 200 keys 17.0
// against 21.8, of 2048 71.4 against 72.6, 4096 rows on 4000 keys 498 against
// 683, but 256 workgroups of 4000 keys 126 us against 109, 96 of 1000 37.9
// against 28.3, 64 11.5 against 8.9
static inline int heads_of_workgroup(const Args& a, long ntiles) {
  return a.num_q_heads / a.num_kv_heads % 2 == 0 && ntiles * (a.num_q_heads / 2) >= 512 ? 2 : 1;
}

// Whether a launch's tiles take their turns by length: Args::turns.  It pays where walks
// are long against the look at the list, unlike each other, and the chip is full few times over, so
// that the last ones count.  The host knows no lengths but the mean portion's rows and the most
// that a row can see.  In the list's order, in turn (us; 32 query and 8 key/value heads of 128): 8
// prompts of 1000 113.6, 100.2; with a window of 512 and a cap 99.1, 93.2; 14 of 512 61.2, 58.5; 4 of
// 500 24.6, 21.6; 6 of 512 to 1000 rows on contexts of 600 to 4000 132.9, 109.1; 2 of 128 on 4000
// listed ahead of 2 of 1500 130.8, 99.0.  As listed stay 20 of 202 (29.4, 30.7; with one of 600 33.4, 34.1),
// 16 of 448 (54.4, 57.5), 24 of 640 (134.0, 141.7: 3840 workgroups) and one alone, which is in order (4000 rows
// 145.5, 146.6).  With a cap, whose scores take longer, 20 of 202 beside one of 600 gain: 42.1, 40.5.
static inline int turns(const Args& a, long ntiles) {
  const long wgs = ntiles * (a.num_q_heads / heads_of_workgroup(a, ntiles));
  long seen = (long)a.max_blocks * a.block_size;  // by a tile
  if (a.window > 0) seen = std::min(seen, (long)a.window + TQ);
  if (a.chunk > 0) seen = std::min(seen, (long)a.chunk + TQ);
  const bool pays = a.num_seqs > 1 && a.num_seqs <= TURN_SEQS && ntiles >= (a.softcap > 0.f ? 4L : 8L) * a.num_seqs &&
                    ntiles <= TURN_TILES && wgs > 256 && wgs <= 2048 && seen >= 512;
  return pays ? (int)(seen < 65472 ? seen / KT + 1 : 1023) : 0;
}

template <int D, int GH, bool CAP, bool SIG, bool EXTRA>
static void launch_heads(const Args& args, int ntiles, hipStream_t stream) {
  const dim3 grid(args.num_q_heads / GH, ntiles), block(256);
  Args a = args;
  a.turns = turns(a, ntiles);
  if (a.block_shift >= 2)
    hipLaunchKernelGGL((flash_prefill_kernel<D, GH, true, CAP, SIG, EXTRA>), grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL((flash_prefill_kernel<D, GH, false, CAP, SIG, EXTRA>), grid, block, 0, stream, a);
}

template <int D, bool CAP, bool SIG, bool EXTRA>
static void launch_mode(const Args& a, int ntiles, hipStream_t stream) {
  if (heads_of_workgroup(a, ntiles) == 2)
    launch_heads<D, 2, CAP, SIG, EXTRA>(a, ntiles, stream);
  else
    launch_heads<D, 1, CAP, SIG, EXTRA>(a, ntiles, stream);
}

// Parts to cut the keys of ntiles tiles into, by the least estimated time in us: a
// workgroup takes 0.0145 a key alone on its CU and 0.02 beside a second one, the merge
// and what begins and ends a part 8, their sums, written and read, at 6 TB/s.  A tile of
// few rows on many keys is a chain of 64-key steps on an idle chip: steps of 8 layers of
// 32 and 8 heads of 128, uncut and in parts, 20 rows on 4000 cached keys 1505 us, 1200;
// 100 on 4000 1832, 1510; on 1200 1470, 1417; 300 on 3000 2268, 2147; 2 of 60 on 2000
// 1604, 1488.  With 4 for the 8, 4 portions of 20 on 1000 lose 1 %.
static inline int parts(long ntiles, long rows, int num_q_heads, int D, long keys) {
  const long wgs = ntiles * num_q_heads;
  if (rows > ntiles * TQ) return 1;  // room for rows of no tile would have no bound
  int best = 1;
  double least = keys * 0.0145;
  for (int n = 2; n <= 16 && wgs * n <= 512 && keys / n >= 256; ++n) {
    const double us = keys / (double)n * (wgs * n <= 256 ? 0.0145 : 0.02) + 8 + rows * num_q_heads * n * (D + 4) * 8e-6 / 6;
    if (us < least) least = us, best = n;
  }
  return best;
}

template <int D>
static void launch_parts(const Args& a, int ntiles, hipStream_t stream) {
  const dim3 grid(a.num_q_heads, ntiles, a.nsplit), block(256);
  if (a.block_shift >= 2)
    hipLaunchKernelGGL((flash_prefill_kernel<D, 1, true, false, false, false, true>), grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL((flash_prefill_kernel<D, 1, false, false, false, false, true>), grid, block, 0, stream, a);
  hipLaunchKernelGGL(flash_prefill_merge_kernel<D>, dim3((TQ * a.num_q_heads * (D / 4) + 255) / 256, ntiles), block, 0, stream,
                     a);
}

}  // namespace flash_prefill
