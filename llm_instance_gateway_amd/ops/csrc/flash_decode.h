// Paged attention of single query rows on MFMA tiles: bf16, key and value
// heads of the same size 64 or 128, up to 16 query heads per key/value head,
// gfx950.  Shared by the Llama decode path (torch extension) and the hybrid
// families' row kernel (light library).
//
// What bounds it: every cached key and value is read once, so HBM.  The kernel
// this replaces gave every query head a wave of its own: each cache line came
// through the vector L1 once per head of the group, every product was a VALU
// instruction, and 8 keys per step with a serial softmax left too little in
// flight (1.5 TB/s on long ragged contexts, 2.7 at 384 requests).  Here one
// wave serves all heads of the group and takes 32 keys per step:
//   * S^T = K Q^T and O^T += V^T P^T are matrix instructions whose spare
//     columns carry the group's heads; operands come straight from global
//     memory in 16-byte loads of whole rows, no LDS;
//   * keys are dealt to the rows of the two S^T tiles so that a lane's scores
//     are its part of the second product's operand; V is transposed by byte
//     permutes in registers; a lane keeps one head's statistics;
//   * weights enter the second product as the sum of three bf16 numbers, which
//     is all of their 24 bits.  With up to 8 heads the middle parts ride in
//     columns 8..15, which would be idle, and are added at the end.  Share of
//     results that differ from the rounded 64-bit ones, over 1 to 300 keys: with
//     fp32 products (the kernel before) 0.7 to 3.2e-5 with softmax or sigmoid
//     weights, with two parts 0.3 to 3.5e-4, now 0.7 to 2.4e-5, at no cost in
//     time.  Sigmoid weights and gates by rcp and exp2 are inside these figures;
//   * the next step's K is requested once S^T is formed, its V once O^T is, so
//     a wave always has 8 to 16 KB on the way;
//   * the waves of a workgroup take steps in turn and merge through LDS; long
//     contexts are also cut over workgroups (nsplits) and merged by a second
//     kernel.
// Measured, 32 query and 8 key/value heads of 128, before -> after: 384
// requests of 190-381 tokens 173 -> 84 us (5.3 TB/s; a large copy reaches 4.9);
// 33 of 3000-6000 370 -> 119 us (5.0 TB/s); 16 of 190-381 30 -> 8.2 us; 64 rows
// with a window of 512 and sigmoid weights 54 -> 25.2 us (27.1 before values were
// loaded as streams; on rows just read 23.5 either way).  Eight waves per workgroup
// were slower from 64 requests on (101 us at 384), two on few (9.2 us at 16).
#pragma once

#include <type_traits>

#include "common.h"

namespace flash_decode {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int KT = 32;  // keys per step

struct Args {
  uint16_t* out;            // [R, Hq * D]
  const uint16_t* q;        // rows q_stride entries apart
  long q_stride;
  const uint16_t* k_cache;  // [blocks, Hkv, BS, D]
  const uint16_t* v_cache;  // rows v_row entries apart
  const uint16_t* gate;     // nullable
  long gate_stride;
  const float* sink;        // nullable, [Hq]
  const float* score_bias;  // nullable, [Hq]
  const int* block_tables;  // [tables, max_blocks]
  int tables;
  // row r belongs to table row tok_seq[r] (negative: none) and sees keys up to
  // positions[r]; without them it is table row r, up to context_lens[r] - 1
  const int* tok_seq;
  const int64_t* positions;
  const int* context_lens;
  float* scratch;           // [R, Hq, nsplits, D + 2] with nsplits > 1
  float scale;
  float temp_coef, temp_every;
  int temp_every_int;
  int rows, num_q_heads, num_kv_heads;
  int v_row;
  int block_size, block_shift;  // block_shift < 0: not a power of two
  int max_blocks;
  int chunk, window;
  int gate_per_head;
  float softcap;
  int nsplits;
  int unmerged;             // whoever reads the result merges the parts
};

// The steps of a row: its position and lower bound, and into how many parts
// its walk is cut: the caller's number, but no part under 16 steps (512 keys),
// which one workgroup takes in the time of the merge.
struct Walk {
  int seq, pos, key_lo, first, steps, parts;
};
LIG_DEVICE int parts_of(int steps, int nsplits) { return max(1, min(nsplits, steps / 16)); }
template <bool EXTRA>
LIG_DEVICE Walk walk_of(const Args& a, int row) {
  Walk w;
  w.seq = a.tok_seq ? a.tok_seq[row] : row;
  w.pos = w.seq < 0 ? -1 : a.positions ? (int)a.positions[row] : a.context_lens[row] - 1;
  w.key_lo = 0;
  if (EXTRA && w.pos >= 0) {
    if (a.chunk > 0) w.key_lo = (w.pos / a.chunk) * a.chunk;
    if (a.window > 0) w.key_lo = max(w.key_lo, w.pos - a.window + 1);
  }
  w.first = w.key_lo / KT;
  w.steps = w.pos < 0 ? 0 : w.pos / KT + 1 - w.first;
  w.parts = parts_of(w.steps, a.nsplits);
  return w;
}

// final scaling of 4 entries of a (row, head), common to both kernels
template <int D, bool EXTRA>
LIG_DEVICE void store_entries(const Args& a, int row, int h, int d, const float (&o)[4], float f) {
  const uint16_t* gp = nullptr;
  if (EXTRA && a.gate) {
    gp = a.gate + (size_t)row * a.gate_stride;
    if (a.gate_per_head) {
      f *= __builtin_amdgcn_rcpf(1.f + __expf(-bf16_to_f32(gp[h])));
      gp = nullptr;
    } else {
      gp += (size_t)h * D + d;
    }
  }
  u32x2 w;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    float x = o[2 * i] * f, y = o[2 * i + 1] * f;
    if (EXTRA && gp) {
      x *= __builtin_amdgcn_rcpf(1.f + __expf(-bf16_to_f32(gp[2 * i])));
      y *= __builtin_amdgcn_rcpf(1.f + __expf(-bf16_to_f32(gp[2 * i + 1])));
    }
    w[i] = (uint32_t)f32_to_bf16(x) | ((uint32_t)f32_to_bf16(y) << 16);
  }
  *reinterpret_cast<u32x2*>(a.out + ((size_t)row * a.num_q_heads + h) * D + d) = w;
}

// W waves per workgroup; LOWCOL: at most 8 heads per group, the weights' middle
// parts in columns 8..15; PB: block size a power of two, at least 8.  CAP, SIG, EXTRA as in the prompt kernel.
template <int D, int W, bool LOWCOL, bool PB, bool STREAM, bool CAP, bool SIG, bool EXTRA>
__global__ __launch_bounds__(64 * W, 2) void flash_decode_kernel(const Args a) {
  constexpr int KS = D / 32;
  constexpr int DV = D / 16;          // entries of a value row per lane
  constexpr int GM = LOWCOL ? 8 : 16;  // heads a wave can hold
  using vload = typename std::conditional<DV == 8, u32x4, u32x2>::type;

  // [W][group][D] sums, [W][GM] maxima, [W][GM] weight sums
  extern __shared__ float smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int kvh = blockIdx.x % a.num_kv_heads;
  const int row = blockIdx.x / a.num_kv_heads;
  const int group = a.num_q_heads / a.num_kv_heads;
  float* const m_s = smem + W * group * D;
  float* const l_s = m_s + W * GM;

  const Walk wk = walk_of<EXTRA>(a, row);
  if ((int)blockIdx.y >= wk.parts) return;
  if (wk.seq < 0) {  // a row of no sequence
    for (int d = tid; d < group * D; d += 64 * W) a.out[((size_t)row * a.num_q_heads + kvh * group) * D + d] = 0;
    return;
  }
  // Waves without a step would hold their registers against the workgroups that
  // wait, and a walk of one step has nothing to merge.  384 rows of 10-20 keys 10.7
  // us (20.4 with all four waves at the barrier, 15.9 in the kernel before), of
  // 30-60 19.1 (23.2, 28.4), with 64 heads 25.6 (32.6, 52); walks of 3 to 5 steps
  // up to 5 % slower.  Where every head has keys of its own, short rows remain
  // slower than before, with a matrix for one head: 32 heads, 384 rows of 10-20
  // keys 29 (51, 20), of 30-60 56 (65, 48), of 50-100 87 (92, 96).  One wave per
  // key/value head and four of these to a workgroup was slower: 22 for the first.
  const bool one_step = wk.steps <= 1;
  const int nw = min(W, max(1, wk.steps));
  if (wave >= nw) return;  // a barrier waits only for waves that have not ended
  const int pos = wk.pos, key_lo = wk.key_lo;
  const int* bt = a.block_tables + (size_t)wk.seq * a.max_blocks;
  float sc = a.scale;
  if (EXTRA && a.temp_coef != 0.f) {
    const float t = a.temp_every_int > 0 ? (float)((pos + 1) / a.temp_every_int)
                                         : floorf((float)(pos + 1) / a.temp_every);
    sc *= 1.f + a.temp_coef * logf(t + 1.f);
  }
  const int span = (wk.steps + wk.parts - 1) / wk.parts;
  const int c0 = wk.first + blockIdx.y * span;
  const int c1 = min(wk.first + wk.steps, c0 + span);

  // a negative scale goes into the sign of the query, so that the largest raw
  // score is the largest scaled one
  const uint32_t flip = sc < 0.f ? 0x80008000u : 0u;
  sc = fabsf(sc);
  const float c = CAP ? sc / a.softcap : sc * LOG2E;
  const float cap2 = CAP ? a.softcap * LOG2E : 0.f;
  const int hl = LOWCOL ? li & 7 : li;       // head of this lane in the group
  const int h = kvh * group + min(hl, group - 1);
  const float bias = SIG && a.score_bias ? a.score_bias[h] : 0.f;
  bf16x8_t q_frag[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    u32x4 raw = *reinterpret_cast<const u32x4*>(a.q + (size_t)row * a.q_stride + (size_t)h * D + ks * 32 + lg * 8);
#pragma unroll
    for (int e = 0; e < 4; ++e) raw[e] ^= flip;
    q_frag[ks] = __builtin_bit_cast(bf16x8_t, raw);
  }

  // rows of a step: S^T tile row li stands for key (li/4)*8 + li%4 (+4 in the
  // second tile), this lane's values are keys lg*8 .. +8.  Keys past the end
  // repeat the last one, keys before the first visible one that one: their
  // weight is zero, but what they hold would still meet it in a product, and
  // their blocks may be gone.  PB: a lane's 8 keys lie in one block, whose number
  // is read one step ahead; no branch may stand between the loads, or each
  // would be waited for by itself
  const size_t block_rows = (size_t)a.num_kv_heads * a.block_size;
  const size_t head_rows = (size_t)kvh * a.block_size;
  const int kt0 = (li >> 2) * 8, vt0 = lg * 8;
  const int shift = a.block_shift;
  auto visible = [&](int t) { return min(EXTRA ? max(t, key_lo) : t, pos); };
  auto block_at = [&](int st, int t0) { return PB ? bt[visible(st * KT + t0) >> shift] : 0; };
  u32x4 kreg[2][KS];
  vload vreg[8];
  // cache rows of N keys of the 8 from t0 on
  auto rows_of = [&](int t0, int first_t, int by, int blk, auto& r) {
    constexpr int N = sizeof(r) / sizeof(r[0]);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int t = visible(t0 + first_t + i * by);
      if constexpr (PB) {
        r[i] = (size_t)blk * block_rows + head_rows + (t & (a.block_size - 1));
      } else {
        const int b = t / a.block_size;
        r[i] = (size_t)bt[b] * block_rows + head_rows + (t - b * a.block_size);
      }
    }
  };
  auto fetch_k = [&](int st, int blk) {
    size_t r[2];
    rows_of(st * KT + kt0, li & 3, 4, blk, r);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kreg[x][ks] = *reinterpret_cast<const u32x4*>(a.k_cache + r[x] * D + lg * 8 + ks * 32);
  };
  auto fetch_v = [&](int st, int blk) {
    size_t r[8];
    rows_of(st * KT + vt0, 0, 1, blk, r);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const vload* src = reinterpret_cast<const vload*>(a.v_cache + r[t] * a.v_row + li * DV);
      vreg[t] = STREAM ? __builtin_nontemporal_load(src) : *src;
    }
  };

  float m = -INFINITY, l = 0.f;
  f32x4_t acc[DV];  // O^T: head column li, entries (lg*4 + i) * DV + j
#pragma unroll
  for (int j = 0; j < DV; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  int st = c0 + wave;
  if (st < c1) {
    int kb = block_at(st, kt0), vb = block_at(st, vt0);
    fetch_k(st, kb);
    fetch_v(st, vb);
    kb = block_at(st + W, kt0);
    vb = block_at(st + W, vt0);
    for (; st < c1; st += W) {
      const bool more = st + W < c1;
      f32x4_t s4[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        s4[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          s4[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kreg[x][ks]), q_frag[ks], s4[x],
                                                          0, 0, 0);
      }
      // the block numbers of the step after next are asked for first: loads
      // return in order, so waiting for them must not mean waiting for V
      const int kb2 = block_at(st + 2 * W, kt0), vb2 = block_at(st + 2 * W, vt0);
      if (more) fetch_k(st + W, kb);

      // weights of keys st*32 + lg*8 + e
      const bool masked = st * KT + KT - 1 > pos || st * KT < key_lo;
      float p[8];
      uint32_t dead = 0;
      if (masked) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int key = st * KT + lg * 8 + e;
          if (key > pos || key < key_lo) {
            dead |= 1u << e;
            s4[e >> 2][e & 3] = -INFINITY;
          }
        }
      }
      float mm = 0.f;
      if constexpr (!SIG) {
        float mx = s4[0][0];
#pragma unroll
        for (int e = 1; e < 8; ++e) mx = fmaxf(mx, s4[e >> 2][e & 3]);
        mx = max_over_groups(mx);
        mx = mx == -INFINITY ? mx : CAP ? cap2 * tanhf(mx * c) : mx * c;
        if (__any(mx > m)) {
          const float m_new = fmaxf(m, mx);
          const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
          m = m_new;
          l *= alpha;
#pragma unroll
          for (int j = 0; j < DV; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[j][i] *= alpha;
        }
        mm = m == -INFINITY ? 0.f : m;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = s4[e >> 2][e & 3];
        float w;
        if constexpr (CAP) {
          // tanhf: forms by the exponential alone are off by 1e-7 of the cap, however small the score
          const float b = cap2 * tanhf(v * c);
          if constexpr (SIG)
            w = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-(b + bias * LOG2E)));
          else
            w = __builtin_amdgcn_exp2f(b - mm);
        } else if constexpr (SIG) {
          w = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-(v * c + bias * LOG2E)));
        } else {
          w = __builtin_amdgcn_exp2f(__builtin_fmaf(v, c, -mm));
        }
        p[e] = w;
      }
      if (masked) {
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] = (dead >> e) & 1 ? 0.f : p[e];
      }
      // p = hi + mid + low, exactly
      u32x4 hi, mid, low;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint16_t w[2][3];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          float r = p[2 * e + i];
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            w[i][k] = f32_to_bf16(r);
            r -= bf16_to_f32(w[i][k]);
          }
        }
        hi[e] = (uint32_t)w[0][0] | ((uint32_t)w[1][0] << 16);
        mid[e] = (uint32_t)w[0][1] | ((uint32_t)w[1][1] << 16);
        low[e] = (uint32_t)w[0][2] | ((uint32_t)w[1][2] << 16);
        if constexpr (!SIG) l += p[2 * e] + p[2 * e + 1];
      }
      bf16x8_t pf = __builtin_bit_cast(bf16x8_t, hi), pm = __builtin_bit_cast(bf16x8_t, mid),
               pl = __builtin_bit_cast(bf16x8_t, low);
      if constexpr (LOWCOL) {
        pf = li < 8 ? pf : pm;
        pl = li < 8 ? pl : bf16x8_t{};
      }

#pragma unroll
      for (int j = 0; j < DV; ++j) {
        const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
        u32x4 vt;
#pragma unroll
        for (int w = 0; w < 4; ++w) vt[w] = __builtin_amdgcn_perm(vreg[2 * w + 1][j / 2], vreg[2 * w][j / 2], sel);
        const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, vt);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf, acc[j], 0, 0, 0);
        if constexpr (!LOWCOL) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pm, acc[j], 0, 0, 0);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pl, acc[j], 0, 0, 0);
      }
      if (more) fetch_v(st + W, vb);
      kb = kb2;
      vb = vb2;
    }
  }

  // ---- merge the waves: low columns onto their heads, then over the waves ------
  if constexpr (LOWCOL) {
#pragma unroll
    for (int j = 0; j < DV; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][i] += __shfl_xor(acc[j][i], 8, 64);
  }
  if constexpr (!SIG) {
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
  }
  if (one_step) {
    if (li < group && li < GM) {
      const bool sink = EXTRA && !SIG && a.sink;
      const float sm = sink ? a.sink[h] * LOG2E : -INFINITY, gm = fmaxf(m, sm);
      const float w = SIG ? 1.f : m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - gm);
      const float gl = l * w + (sink ? __builtin_amdgcn_exp2f(sm - gm) : 0.f);
      const float f = SIG ? 1.f : (gl > 0.f ? 1.f / gl : (gl == 0.f ? 0.f : gl));
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < DV; j += 4) {
          const float o[4] = {acc[j][i] * w, acc[j + 1][i] * w, acc[j + 2][i] * w, acc[j + 3][i] * w};
          store_entries<D, EXTRA>(a, row, h, (lg * 4 + i) * DV + j, o, f);
        }
    }
    return;
  }
  if (li < group && li < GM) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < DV; j += 4)
        *reinterpret_cast<f32x4_t*>(&smem[(wave * group + li) * D + (lg * 4 + i) * DV + j]) =
            f32x4_t{acc[j][i], acc[j + 1][i], acc[j + 2][i], acc[j + 3][i]};
    if (lg == 0) {
      m_s[wave * GM + li] = m;
      l_s[wave * GM + li] = l;
    }
  }
  __syncthreads();
  for (int it = tid; it < group * (D / 4); it += 64 * nw) {
    const int hh = it / (D / 4), d = (it % (D / 4)) * 4;
    const int head = kvh * group + hh;
    const bool sink = EXTRA && !SIG && a.sink && wk.parts == 1;
    float gm = sink ? a.sink[head] * LOG2E : -INFINITY;
    float gl = 0.f;
    float o[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (!SIG) {
      const float sm = gm;
#pragma unroll
      for (int w = 0; w < W; ++w)
        if (w < nw) gm = fmaxf(gm, m_s[w * GM + hh]);
      if (sink) gl = __builtin_amdgcn_exp2f(sm - gm);
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
      if (w >= nw) break;
      float f = 1.f;
      if constexpr (!SIG) {
        f = m_s[w * GM + hh] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_s[w * GM + hh] - gm);
        gl += l_s[w * GM + hh] * f;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] += smem[(w * group + hh) * D + d + i] * f;
    }
    if (wk.parts > 1) {
      float* sp = a.scratch + (((size_t)row * a.num_q_heads + head) * a.nsplits + blockIdx.y) * (D + 2);
#pragma unroll
      for (int i = 0; i < 4; ++i) sp[d + i] = o[i];
      if (d == 0) {
        sp[D] = gm;
        sp[D + 1] = gl;
      }
    } else {
      const float f = SIG ? 1.f : (gl > 0.f ? 1.f / gl : (gl == 0.f ? 0.f : gl));
      store_entries<D, EXTRA>(a, row, head, d, o, f);
    }
  }
}

// merges the parts of a (row, head), 4 entries per lane
template <int D, bool SIG, bool EXTRA>
__global__ __launch_bounds__(64) void flash_decode_merge_kernel(const Args a) {
  constexpr int LP = D / 4;  // lanes per (row, head)
  const int item = blockIdx.x * (64 / LP) + threadIdx.x / LP;
  if (item >= a.rows * a.num_q_heads) return;
  const int row = item / a.num_q_heads, head = item % a.num_q_heads;
  const int parts = walk_of<EXTRA>(a, row).parts;
  if (parts == 1) return;  // stored by the first kernel
  const int d = (threadIdx.x % LP) * 4;
  const float* base = a.scratch + (size_t)item * a.nsplits * (D + 2);
  const bool sink = EXTRA && !SIG && a.sink;
  float gm = sink ? a.sink[head] * LOG2E : -INFINITY, gl = 0.f;
  if constexpr (!SIG) {
    const float sm = gm;
    for (int z = 0; z < parts; ++z) gm = fmaxf(gm, base[(size_t)z * (D + 2) + D]);
    if (sink) gl = __builtin_amdgcn_exp2f(sm - gm);
  }
  float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int z = 0; z < parts; ++z) {
    const float* sp = base + (size_t)z * (D + 2);
    float f = 1.f;
    if constexpr (!SIG) {
      f = sp[D] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sp[D] - gm);
      gl += sp[D + 1] * f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] += sp[d + i] * f;
  }
  const float f = SIG ? 1.f : (gl > 0.f ? 1.f / gl : (gl == 0.f ? 0.f : gl));
  store_entries<D, EXTRA>(a, row, head, d, o, f);
}

// What the kernel takes.
static inline bool serves(const Args& a, int D, int Dv) {
  auto al = [](const void* p, unsigned to) { return (reinterpret_cast<uintptr_t>(p) & (to - 1)) == 0; };
  return D == Dv && (D == 64 || D == 128) && a.num_q_heads % a.num_kv_heads == 0 &&
         a.num_q_heads / a.num_kv_heads <= 16 && a.q_stride % 8 == 0 && a.v_row % 8 == 0 && a.v_row >= D &&
         al(a.q, 16) && al(a.k_cache, 16) && al(a.v_cache, 16) && al(a.out, 8);
}

template <int D, bool SIG, bool EXTRA>
static void launch_merge(const Args& a, hipStream_t stream) {
  if (a.nsplits <= 1 || a.unmerged) return;
  const long lanes = (long)a.rows * a.num_q_heads * (D / 4);
  hipLaunchKernelGGL((flash_decode_merge_kernel<D, SIG, EXTRA>), dim3((unsigned)((lanes + 63) / 64)), dim3(64), 0,
                     stream, a);
}

template <int D, bool CAP, bool SIG, bool EXTRA>
static void launch_rows(const Args& a, hipStream_t stream) {
  constexpr int W = 4;
  const int group = a.num_q_heads / a.num_kv_heads;
  const dim3 grid(a.rows * a.num_kv_heads, a.nsplits), block(64 * W);
  const bool low = group <= 8, pb = a.block_shift >= 3;
  const size_t lds = (size_t)W * (group * D + 2 * (low ? 8 : 16)) * sizeof(float);
  // Values as a stream past the caches (non-temporal) where no other row reads them,
  // as far as the host can tell, and where rows are many: their caches don't stay in
  // the last-level cache from one step to the next.  One row of a few hundred keys has
  // them there, and a step of it is 1 % slower with streams; 8 rows on each of 32 tables
  // of 1000 keys 83 -> 91 us.  Streamed, over 1 GB of caches in turn: 64 rows of 1000
  // keys 47.9 -> 43.7 us, 384 of 286 84.0 -> 75.8, 32 of 4000 98.4 -> 89.8, 40 of 300
  // 15.1 -> 14.6, 64 x 100 9.6 -> 9.3; with a window of 512 64 rows 27.1 -> 25.2, 32 rows
  // 16.0 -> 15.0.  The same rows again (64 with the window, 134 MB): 23.1 -> 23.5.
  // Keys too, whose lines take two loads, gives half of that back.
  const bool many = (long)a.rows * a.num_kv_heads >= 256 && a.rows <= a.tables;
#define LIG_FD(LOWCOL, PB, STREAM)                                                                             \
  hipLaunchKernelGGL((flash_decode_kernel<D, W, LOWCOL, PB, STREAM, CAP, SIG, EXTRA>), grid, block, lds, stream, a)
  if (low && pb && many) LIG_FD(true, true, true);
  else if (low && pb) LIG_FD(true, true, false);
  else if (low) LIG_FD(true, false, false);
  else if (pb && many) LIG_FD(false, true, true);
  else if (pb) LIG_FD(false, true, false);
  else LIG_FD(false, false, false);
#undef LIG_FD
  launch_merge<D, SIG, EXTRA>(a, stream);
}

template <int D, bool CAP, bool SIG, bool EXTRA>
static void launch_mode(Args a, hipStream_t stream) {
  // a grid holds less than 2^32 threads a dimension, and drops the rest without an
  // error: 256 per (row, key/value head) here, D / 4 per (row, head) in the merge
  const long per_row = (long)a.num_kv_heads * 256 > (long)a.num_q_heads * (D / 4) ? (long)a.num_kv_heads * 256
                                                                                 : (long)a.num_q_heads * (D / 4);
  const long most = ((1L << 32) - 256) / per_row;
  for (long left = a.rows; left > 0; left -= most) {
    a.rows = (int)(left < most ? left : most);
    launch_rows<D, CAP, SIG, EXTRA>(a, stream);
    const long r = a.rows, heads = r * a.num_q_heads;
    a.out += heads * D;
    a.q += r * a.q_stride;
    if (a.gate) a.gate += r * a.gate_stride;
    if (a.tok_seq) {
      a.tok_seq += r;
    } else {
      a.block_tables += r * a.max_blocks;
    }
    if (a.positions) a.positions += r;
    if (a.context_lens) a.context_lens += r;
    if (a.scratch) a.scratch += heads * a.nsplits * (D + 2);
  }
}

}  // namespace flash_decode
