// The gated delta rule in chunks of 64 tokens on MFMA tiles, gfx950 (bf16 q,
// k, v; fp32 state): the delta form of matrix_state_scan.hip, same arguments
// and state rows; these kernels take the long portions.
//
// Inside a chunk, with G_t the sum of the log decays up to token t, unit
// vectors k, q and S the state the chunk starts from, the corrections u solve
// a unit lower triangular system:
//     u_t + b_t sum_{s<t} e^(G_t-G_s) (k_t . k_s) u_s = b_t (v_t - e^(G_t) S^T k_t)
//     o_t = e^(G_t) S^T q_t + sum_{s<=t} e^(G_t-G_s) (q_t . k_s) u_s
//     S  <- e^(G_end) S + sum_s e^(G_end-G_s) k_s u_s^T
// (the WY form of the chunked delta rule).  The system's matrix does not
// depend on S, so its inverse is computed for all chunks of the step at once:
//
// delta_chunk_prepare_kernel, one workgroup (4 waves) per (chunk, segment,
// head): k . k and q . k by MFMA on bf16 rows (exact products), fp32 from there
// on.  The four 16 x 16 diagonal blocks of the system are inverted by
// substitution, a column per lane; the blocks below them follow level by level,
//     T_ij = -T_ii sum_{j<=m<i} A_im T_mj,
// with fp32 MFMA (16x16x4).  The inverse times diag(b) and the weighted scores
// e^(G_t-G_s) (q_t . k_s) leave as two bf16 halves each, with the token factors
// the second kernel needs.  The log decays are summed in double: a token that
// decays nearly everything must not cost the differences after it their
// precision.  Bound by its chain of short steps (loads, norms, exponentials,
// substitution, three levels), so a wave loads its own 16 rows only, all at
// once, and takes the others' from LDS: 47 us for 8 prompts of 1000 tokens and
// 32 heads, 65 with a load per tile in turn.  With the chunks of a portion side by side in
// the grid the last of the longer ones fell to the same XCDs: heads side by side, both calls
// 141.6 -> 138.8 us; 16 of 500, 64 heads 314 -> 291.
//
// delta_chunk_scan_kernel, one workgroup per (segment, head, one or two
// blocks of 64 value columns), walks the chunks; wave w owns 16 columns of
// the state, [D, 16] fp32 in MFMA accumulators for the whole segment.  The
// state, the right-hand sides and the corrections go from accumulators
// straight into the next product as an operand: a contraction may visit its
// inner index in any order as long as both operands agree, so the other
// operand is read from LDS in the order the accumulators hold it; k transposed
// and the values come through transposing reads.  The next chunk's rows are
// fetched into registers during the arithmetic.
//
// The walk is the serial part and the whole chip has one workgroup per CU at
// 8 prompts of 32 heads, so what can be done for all chunks at once (inverse,
// scores, norms) is done by the first kernel.  8 prompts of 1000 tokens, 32
// heads of 128 x 128: 154 us with the scores inside, a transposed copy of k and
// 2-byte loads of values, 125 without the last two, 95 with the first of the two walks
// below: some 11 000 cycles a chunk, 7800 of them of LDS traffic.  8-byte reads run at
// half the rate of 16-byte ones (128 bytes a cycle), and the transposing reads of k met
// banks twice to four times.  delta_chunk_walk_kernel, for the heads that models have, reads
// 16 bytes a lane everywhere, from places without conflicts, and brings its rows by DMA:
// 84 us, 8300 cycles a chunk, of which 2700 are the loads of the next one (70 KB) and the
// barrier, 5600 the arithmetic (4200 of matrix cores; at 1.65 GHz).  The DMA alone, with
// 8-byte reads, was slower than rows through registers (106 us).
// Four waves per workgroup and two workgroups per CU: slower by 30 us, as q, k and the first
// kernel's blocks come and go twice; but where that still leaves every workgroup a CU of its
// own, a chunk takes less time.  Two waves each, on up to four times the CUs, are no
// faster than four.
//
// Precision: products of bf16 numbers are exact in fp32, sums are fp32, fp32
// operands are split into two bf16 halves (lo * lo left out).  The unit norms
// stay fp32 scalars outside the bf16 vectors.

#include "matrix_state.h"
#include "matrix_state_mfma.h"

#define DC_BLOCKS 10  // 16 x 16 blocks of a chunk's square on and below the diagonal

// Factors of a chunk's tokens.
struct DeltaFactors {
  float ek[MC_T];     // e^G / |k|
  float eg[MC_T];     // e^G
  float wk[MC_T];     // e^(G_end - G) / |k|, 0 past the portion's end
  float c[MC_T];      // e^G * q_scale / |q|
};

// What the first kernel leaves for one (chunk, head): inverse * diag(b) and the
// weighted scores, each as high and low halves of the blocks (i, j), j <= i, at
// i (i + 1) / 2 + j.
struct DeltaChunk {
  uint16_t w[2][2][DC_BLOCKS][16][16];
  DeltaFactors f;
};

// The same for delta_chunk_walk_kernel: the inverse as its lanes hold it as an operand, rows of
// 16 tokens (`walk_row`) by pairs of blocks up to the diagonal, zeros included, so that
// a lane reads its 16 bytes at its own place.
#define DC_PAIRS 6
struct DeltaWalkChunk {
  uint16_t inverse[2][DC_PAIRS][WAVE_SIZE][8];
  uint16_t scores[2][DC_BLOCKS][16][16];
  DeltaFactors f;
};
LIG_DEVICE constexpr int walk_pair(int tt, int u) { return (tt < 2 ? tt : 2 * tt - 2) + u; }

// Entry i of rows 0 to 3 in lane i of a group of 16, from 8 bytes of row L / 4
// and columns 4 (L % 4) on at lane L.
LIG_DEVICE u16x4 mc_ld_tr(const uint16_t* p) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                       (__attribute__((address_space(3))) s16x4*)p));
}

// Chunk c of segment seg (first row r0): segments lie in row order, so these
// places are distinct and below R / 64 + S + 1.
LIG_DEVICE long delta_chunk_slot(long r0, int c, int seg) { return r0 / MC_T + c + seg; }

extern "C" long lig_gated_delta_scratch(int R, int S, int H) {
  static_assert(sizeof(DeltaWalkChunk) >= sizeof(DeltaChunk), "room for either");
  return ((long)R / MC_T + S + 1) * H * (long)sizeof(DeltaWalkChunk);
}

#define DI_THREADS 256
#define DI_ROW 68  // padded fp32 LDS row
// Waves to a SIMD, of which a workgroup brings one to each.  For five the compiler keeps to 96
// registers and does without copies in accumulation registers (heads of 192, 8 prompts of 1000, four waves and
// five, both kernels 215 -> 209 us); at 80, for six, heads of 128 spill and gain nothing.  Heads of 256 take 116
// for four; asked for five it gave them 130, for three (16 heads with values of 128 128.2 -> 125.4 us, 16 prompts of
// 500 with values of 64 174 -> 170).
#define DI_WAVES(DP) ((DP) <= 192 ? 5 : 4)

template <int DP, typename Chunk>
__global__ __launch_bounds__(DI_THREADS, DI_WAVES(DP)) void delta_chunk_prepare_kernel(
    const MsArgs A, Chunk* __restrict__ scratch) {
  constexpr bool WALK = __is_same(Chunk, DeltaWalkChunk);
  constexpr int KB = DP / 32;
  // One square holds both triangles in 16 x 16 blocks: the system's block (i,
  // j) at its own place, the inverse's block (i, j) at place (j, i), each in
  // row order; a diagonal block of the inverse replaces the system's.
  // Before that its room holds k, for the waves whose tokens come later.
  constexpr int KROW = DP + 8;
  union Square {
    float a[MC_T][DI_ROW];
    uint16_t k[MC_T][KROW];
  };
  __shared__ __align__(16) Square sq;
  float(*a_s)[DI_ROW] = sq.a;
  __shared__ __align__(16) double g_s[MC_T];
  __shared__ __align__(16) float b_s[MC_T], ik_s[MC_T];
  __shared__ float iq_s[MC_T];

  // XCDs take workgroups in turn: each gets an eighth of the heads, whose neighbours share
  // keys, and as many chunks as the others
  const int seg = blockIdx.y, chunk = blockIdx.x / A.H, x = blockIdx.x - chunk * A.H;
  const int h = A.H % 8 == 0 ? (x & 7) * (A.H >> 3) + (x >> 3) : x;
  const int n = A.seg_len[seg];
  const long r0 = A.seg_start[seg];
  const int c0 = chunk * MC_T;
  if (c0 >= n || n < A.len_min) return;
  const int cnt = min(MC_T, n - c0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const uint16_t* k = (const uint16_t*)A.k + (h / A.rep) * A.D + (r0 + c0) * A.k_stride;
  const uint16_t* q = (const uint16_t*)A.q + (h / A.rep) * A.D + (r0 + c0) * A.q_stride;
  Chunk* out = scratch + delta_chunk_slot(r0, chunk, seg) * A.H + h;
  uint16_t(*scores)[DC_BLOCKS][16][16];  // high and low halves
  if constexpr (WALK) scores = out->scores;
  else scores = out->w[1];

  // ---- k . k and q . k: wave's 16 tokens (columns) against the tokens up to them ----------
  // rows past the portion's end read its last token: their write strength is zero
  const u16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  auto row = [&](const uint16_t* x, long stride, int t, int kb) __attribute__((always_inline)) {
    const int d = kb * 32 + lg * 8;
    const u16x8 v = mc_ld16(x + min(t, cnt - 1) * stride + (d < A.D ? d : 0));
    return d < A.D ? v : zero8;
  };
  u16x8 kf[KB], qf[KB];
  f32x4 kk[4], qk[4], qq = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    kf[kb] = row(k, A.k_stride, wave * 16 + li, kb);
    qf[kb] = row(q, A.q_stride, wave * 16 + li, kb);
  }
  if (wave == 0) {
    float b = 0.f, lgd = 0.f;
    if (lane < cnt) {
      const long r = (r0 + c0 + lane) * A.gate_stride + h;
      b = sigmoid_f32(A.gate_i[r]);
      lgd = ms_log_decay(A.gate_f[r], A.bias_i[h], A.bias_f[h]);
    }
    double G = (double)lgd;
#pragma unroll
    for (int d = 1; d < MC_T; d <<= 1) {
      const double u = __shfl_up(G, d, WAVE_SIZE);
      if (lane >= d) G += u;
    }
    g_s[lane] = G;
    b_s[lane] = b;
  }

#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    *reinterpret_cast<u16x8*>(&sq.k[wave * 16 + li][kb * 32 + lg * 8]) = kf[kb];
    qq = mc_mfma(qf[kb], qf[kb], qq);
  }
  __syncthreads();
#pragma unroll
  for (int st = 0; st < 4; ++st) {
    kk[st] = qk[st] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (st <= wave) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const u16x8 ks = *reinterpret_cast<const u16x8*>(&sq.k[st * 16 + li][kb * 32 + lg * 8]);
        kk[st] = mc_mfma(ks, kf[kb], kk[st]);
        qk[st] = mc_mfma(ks, qf[kb], qk[st]);
      }
    }
  }
  // token li's squares are entry li % 4 of lane group li / 4, column li
  if (lg == li >> 2) {
    const f32x4 d = wave == 0 ? kk[0] : wave == 1 ? kk[1] : wave == 2 ? kk[2] : kk[3];
    auto own = [&](f32x4 x) __attribute__((always_inline)) {
      return (li & 2) ? ((li & 1) ? x[3] : x[2]) : ((li & 1) ? x[1] : x[0]);
    };
    ik_s[wave * 16 + li] = 1.0f / sqrtf(own(d) + A.unit_eps);
    iq_s[wave * 16 + li] = A.q_scale / sqrtf(own(qq) + A.unit_eps);
  }
  __syncthreads();
  // ---- the system's strictly lower part; the weighted scores --------------------------------
  {
    const int t = wave * 16 + li;
    const double Gt = g_s[t];
    const float bt = b_s[t] * ik_s[t], iq = iq_s[t];
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      if (st <= wave) {
        const int s0 = st * 16 + lg * 4;
        const f32x4 ik = *reinterpret_cast<const f32x4*>(&ik_s[s0]);
        f32x4 a, p;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float e = ik[r] * __expf((float)(Gt - g_s[s0 + r]));
          a[r] = s0 + r < t ? bt * e * kk[st][r] : 0.f;
          p[r] = s0 + r <= t ? iq * e * qk[st][r] : 0.f;
        }
        *reinterpret_cast<f32x4*>(&a_s[t][s0]) = a;
        uint32_t h0, h1, l0, l1;
        mc_split2(p[0], p[1], h0, l0);
        mc_split2(p[2], p[3], h1, l1);
        const int blk = wave * (wave + 1) / 2 + st;
        *reinterpret_cast<u32x2*>(&scores[0][blk][li][lg * 4]) = u32x2{h0, h1};
        *reinterpret_cast<u32x2*>(&scores[1][blk][li][lg * 4]) = u32x2{l0, l1};
      }
    }
  }
  __syncthreads();
  // ---- diagonal blocks: lane li solves for column li of the inverse ------------------------
  {
    const int b = wave * 16;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float v = i == li ? 1.f : 0.f;
#pragma unroll
      for (int m = 0; m < i; ++m) v -= a_s[b + i][b + m] * x[m];
      x[i] = v;
    }
    if (lg == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) a_s[b + i][b + li] = x[i];
    }
  }
  __syncthreads();
  // ---- blocks below the diagonal, one level of distance at a time --------------------------
#pragma unroll
  for (int lvl = 1; lvl < 4; ++lvl) {
    if (wave + lvl < 4) {
      const int bi = (wave + lvl) * 16, bj = wave * 16;
      f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
      for (int m = bj; m < bi; m += 16) {
#pragma unroll
        for (int e = 0; e < 16; e += 4)
          x = __builtin_amdgcn_mfma_f32_16x16x4f32(a_s[bi + li][m + e + lg], a_s[bj + e + lg][m + li],
                                                   x, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)  // x's rows lg * 4 + r are this lane's share of the contraction
        y = __builtin_amdgcn_mfma_f32_16x16x4f32(a_s[bi + li][bi + lg * 4 + r], x[r], y, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) a_s[bj + lg * 4 + r][bi + li] = -y[r];
    }
    __syncthreads();
  }
  // ---- write out ------------------------------------------------------------------------------
  {
    const int t = tid >> 2, s0 = (tid & 3) * 16, ti = t >> 4;
    if (s0 <= (WALK ? t | 31 : t)) {
      const int blk = ti * (ti + 1) / 2 + (tid & 3);
      const float* src = &a_s[s0 + (t & 15)][t & ~15];  // row t of block (t / 16, s0 / 16)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        u32x4 hi, lo;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int s = half * 8 + e * 4;
          mc_split4(*reinterpret_cast<const f32x4*>(src + s) *
                        *reinterpret_cast<const f32x4*>(&b_s[s0 + s]), e, hi, lo);
        }
        if constexpr (WALK) {
          // row t of its pair of blocks: the place that walk_row gives a lane
          const int pair = walk_pair(t / 32 * 2 + (t >> 2 & 1), s0 >> 5);
          const int at = ((s0 >> 3 & 3) + half) * 16 + (t >> 3 & 3) * 4 + (t & 3);
          if (s0 > t) hi = lo = u32x4{0, 0, 0, 0};
          *reinterpret_cast<u32x4*>(&out->inverse[0][pair][at][0]) = hi;
          *reinterpret_cast<u32x4*>(&out->inverse[1][pair][at][0]) = lo;
        } else {
          *reinterpret_cast<u32x4*>(&out->w[0][0][blk][t & 15][half * 8]) = hi;
          *reinterpret_cast<u32x4*>(&out->w[0][1][blk][t & 15][half * 8]) = lo;
        }
      }
    }
  }
  if (tid < MC_T) {
    const double G = g_s[tid], G_end = g_s[MC_T - 1];  // tokens past the end decay nothing
    const float ik = ik_s[tid], eg = expf((float)G);
    out->f.c[tid] = eg * iq_s[tid];
    out->f.eg[tid] = eg;
    out->f.ek[tid] = eg * ik;
    out->f.wk[tid] = tid < cnt ? expf((float)(G_end - G)) * ik : 0.f;
  }
}

// NW waves: 4 walk one block of 64 value columns, 8 walk two that share q, k,
// the inverse and the weighted scores.
template <int DP, int NW, bool VEC>
__global__ __launch_bounds__(NW * WAVE_SIZE) void delta_chunk_scan_kernel(
    const MsArgs A, const DeltaChunk* __restrict__ scratch) {
  // LDS rows advance by 2 banks (mod 32), so that the 8-byte operand reads of
  // 16 rows spread over all of them
  constexpr int KB = DP / 32, DT = DP / 16, DROW = DP + 4, TROW = MC_T + 4;
  constexpr int NTHR = NW * WAVE_SIZE, VC = NW * 2, VROW = NW * 16 + 4;
  constexpr int CC = DP / 8;                        // 16-byte chunks of a q or k row
  constexpr int NCH = (MC_T * CC + NTHR - 1) / NTHR;  // of them per thread
  constexpr int WCH = 4 * DC_BLOCKS * 32;           // 16-byte pieces of the inverse and the scores
  constexpr int NT = (WCH + NTHR - 1) / NTHR;       // of them per thread
  constexpr int NV = MC_T * VC / NTHR;              // chunks of values per thread
  constexpr int NF = sizeof(DeltaFactors) / 8;      // 8-byte pieces of the token factors
  static_assert(NF <= NTHR, "threads");
  struct Shared {
    uint16_t q[MC_T][DROW];
    uint16_t k[MC_T][DROW];
    uint16_t v[MC_T][VROW];
    uint16_t w[2][2][MC_T][TROW];  // the inverse, the scores: high and low halves
    DeltaFactors f;
  };
  __shared__ __align__(16) Shared sm;

  const int seg = blockIdx.x, h = blockIdx.y;
  const int n = A.seg_len[seg];
  if (n <= 0 || n < A.len_min) return;
  const int H = A.H, D = A.D, Dv = A.Dv, CB = A.CB;
  const long r0 = A.seg_start[seg];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int blk = blockIdx.z * (NW / 4) + (wave >> 2);
  const bool active = blk < A.NB;  // others compute on zeros and store nothing
  const int c0 = blk * CB, ncol = active ? min(CB, Dv - c0) : 0;
  const int col = (wave & 3) * 16 + li;  // the state column this lane holds
  const uint16_t* q = (const uint16_t*)A.q + (h / A.rep) * D;
  const uint16_t* k = (const uint16_t*)A.k + (h / A.rep) * D;
  const uint16_t* v = (const uint16_t*)A.v + h * Dv;
  const DeltaChunk* ch = scratch + delta_chunk_slot(r0, 0, seg) * H + h;

  const int out_row = H * Dv * 4;
  // chunk c of a staged row of values: the column it comes from, and whether there is one
  auto v_in = [&](int c) __attribute__((always_inline)) {
    const int b = blockIdx.z * (NW / 4) + c / 8;
    return b < A.NB && c % 8 * 8 < min(CB, Dv - b * CB);
  };
  auto v_at = [&](int c) __attribute__((always_inline)) {
    return v_in(c) ? (blockIdx.z * (NW / 4) + c / 8) * CB + c % 8 * 8 : 0;
  };

  // ---- state row: [head][block][entry][column * split + key lane] ----------------------
  const int nthr = CB * A.split, Dst = A.split * A.kpt;
  float* srow = A.state + (long)A.seg_slot[seg] * A.state_stride + (long)(h * A.NB + blk) * A.kpt * nthr;
  const bool resume = A.seg_fresh[seg] == 0;
  // entry i0 of a state column; kpt is a multiple of 4, so the next three follow nthr apart
  auto at = [&](int i0) __attribute__((always_inline)) {
    const int j = i0 / A.kpt;
    return srow + (long)(i0 - j * A.kpt) * nthr + col * A.split + j;
  };
  f32x4 S[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    S[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int i0 = dt * 16 + lg * 4;
    if (active && resume && i0 < Dst && col < CB) {
      const float* src = at(i0);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[dt][r] = src[(long)r * nthr];
    }
  }
  // the blocks above the diagonal are never written: zero for the whole walk
  for (int e = tid; e < 4 * MC_T * TROW / 8; e += NTHR)
    reinterpret_cast<u16x8*>(&sm.w[0][0][0][0])[e] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};

  // 16-byte chunks of neighbouring threads lie side by side in a row.  Rows past
  // the portion's end read its last token instead: their write strength and
  // their weight in the state are zero and their outputs are not stored.  No
  // load stands in a branch: a branch would make the next chunk's first use
  // wait for everything still on its way.
  u16x8 qr[NCH], kr[NCH], tr[NT], vr[NV];
  u32x2 fr;
  const u16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const int q_stride = (int)A.q_stride, k_stride = (int)A.k_stride, v_stride = (int)A.v_stride;
  auto fetch = [&](int t0) __attribute__((always_inline)) {
    const uint16_t* qb = q + (r0 + t0) * A.q_stride;
    const uint16_t* kb = k + (r0 + t0) * A.k_stride;
    const uint16_t* vb = v + (r0 + t0) * A.v_stride;
    const int last = min(n - 1 - t0, MC_T - 1);
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      const int e = tid + j * NTHR, row = min(e / CC, last), d = e % CC * 8 < D ? e % CC * 8 : 0;
      qr[j] = mc_ld16(qb + row * q_stride + d);
      kr[j] = mc_ld16(kb + row * k_stride + d);
    }
    const DeltaChunk* c = ch + (long)(t0 / MC_T) * H;
#pragma unroll
    for (int j = 0; j < NT; ++j) tr[j] = mc_ld16(&c->w[0][0][0][0][0] + min(tid + j * NTHR, WCH - 1) * 8);
    fr = reinterpret_cast<const u32x2*>(&c->f)[min(tid, NF - 1)];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int e = tid + j * NTHR, row = min(e / VC, last);
      const uint16_t* src = vb + row * v_stride + v_at(e % VC);
      if (VEC) {
        vr[j] = mc_ld16(src);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) vr[j][i] = src[i];
      }
    }
  };
  fetch(0);
  // The walk waits for its loads but not for the stores behind them, which it
  // can do only if it is entered with as many stores: four into an empty buffer.
  {
    const auto none = __builtin_amdgcn_make_buffer_rsrc(A.out, 0, 0, 0x00027000);
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{0, 0, 0, 0}, none, tt * 16, 0, 0);
  }

#pragma nounroll
  for (int t0 = 0; t0 < n; t0 += MC_T) {
    const int cnt = min(MC_T, n - t0);
    __syncthreads();  // the previous chunk's readers are done
    // ---- staging -------------------------------------------------------------------------
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      const int e = tid + j * NTHR, row = e / CC, d = e % CC * 8;
      if (MC_T * CC % NTHR && row >= MC_T) continue;
      mc_st8x2(&sm.q[row][d], d < D ? qr[j] : zero8);
      mc_st8x2(&sm.k[row][d], d < D ? kr[j] : zero8);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int e = tid + j * NTHR, blk = e / 32 % DC_BLOCKS, part = e / 32 / DC_BLOCKS;
      const int bi = (blk >= 1) + (blk >= 3) + (blk >= 6), bj = blk - bi * (bi + 1) / 2;
      if (e < WCH) mc_st8x2(&sm.w[part >> 1][part & 1][bi * 16 + e / 2 % 16][bj * 16 + e % 2 * 8], tr[j]);
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int e = tid + j * NTHR;
      mc_st8x2(&sm.v[e / VC][e % VC * 8], v_in(e % VC) ? vr[j] : zero8);
    }
    if (tid < NF) reinterpret_cast<u32x2*>(&sm.f)[tid] = fr;
    __syncthreads();
    fetch(min(t0 + MC_T, (n - 1) / MC_T * MC_T));

    f32x4 o[4];
    u32x4 uh[2], ul[2], wh[2], wl[2];
    {
      // ---- the chunk's starting state with all keys and all queries ---------------------------
      f32x4 x[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) x[tt] = o[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < KB; ++u) {
        u32x4 sh, sl;
        mc_split4(S[2 * u], 0, sh, sl);
        mc_split4(S[2 * u + 1], 1, sh, sl);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          const uint16_t* kp = &sm.k[tt * 16 + li][u * 32 + lg * 4];
          const uint16_t* qp = &sm.q[tt * 16 + li][u * 32 + lg * 4];
          const u16x8 a = mc_ld8x2(kp, kp + 16), b = mc_ld8x2(qp, qp + 16);
          x[tt] = mc_mfma(a, sh, x[tt]);
          o[tt] = mc_mfma(sh, b, o[tt]);
          x[tt] = mc_mfma(a, sl, x[tt]);
          o[tt] = mc_mfma(sl, b, o[tt]);
        }
      }
      // ---- right-hand sides: v - e^G S^T k ---------------------------------------------------
      u32x4 rh[2], rl[2];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const f32x4 ek = *reinterpret_cast<const f32x4*>(&sm.f.ek[tt * 16 + lg * 4]);
        const u16x4 vv = mc_ld_tr(&sm.v[tt * 16 + lg * 4 + (li >> 2)][wave * 16 + (li & 3) * 4]);
        f32x4 val;
#pragma unroll
        for (int i = 0; i < 4; ++i) val[i] = bf16_to_f32(vv[i]);
        mc_split4(val - ek * x[tt], tt & 1, rh[tt / 2], rl[tt / 2]);
      }
      // ---- corrections u = inverse * right-hand sides ----------------------------------------
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u <= tt / 2; ++u) {
          const uint16_t* th = &sm.w[0][0][tt * 16 + li][u * 32 + lg * 4];
          const uint16_t* tl = &sm.w[0][1][tt * 16 + li][u * 32 + lg * 4];
          const u16x8 a = mc_ld8x2(th, th + 16);
          c = mc_mfma(a, rh[u], c);
          c = mc_mfma(a, rl[u], c);
          c = mc_mfma(mc_ld8x2(tl, tl + 16), rh[u], c);
        }
        const f32x4 wk = *reinterpret_cast<const f32x4*>(&sm.f.wk[tt * 16 + lg * 4]);
        mc_split4(c, tt & 1, uh[tt / 2], ul[tt / 2]);
        mc_split4(c * wk, tt & 1, wh[tt / 2], wl[tt / 2]);
      }
    }
    {
      // ---- weighted scores with the corrections; outputs -----------------------------------------
      const auto dst = __builtin_amdgcn_make_buffer_rsrc(A.out + (r0 + t0) * (long)(H * Dv) + h * Dv + (active ? c0 : 0), 0,
                                                         active ? (cnt - 1) * out_row + ncol * 4 : 0, 0x00027000);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const int t = tt * 16 + li;
        o[tt] *= sm.f.c[t];
#pragma unroll
        for (int u = 0; u <= tt / 2; ++u) {
          const uint16_t* ph = &sm.w[1][0][t][u * 32 + lg * 4];
          const uint16_t* pl = &sm.w[1][1][t][u * 32 + lg * 4];
          const u16x8 b = mc_ld8x2(ph, ph + 16);
          o[tt] = mc_mfma(uh[u], b, o[tt]);
          o[tt] = mc_mfma(ul[u], b, o[tt]);
          o[tt] = mc_mfma(uh[u], mc_ld8x2(pl, pl + 16), o[tt]);
        }
        const int vc = (wave & 3) * 16 + lg * 4;
        // past the rows or the columns: past the buffer's end, dropped
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o[tt]), dst,
                                               vc < ncol ? t * out_row + vc * 4 : 0x7fffffff, 0, 0);
      }
      // ---- the keys' products join the state --------------------------------------------------------
      const float g_end = sm.f.eg[MC_T - 1];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        S[dt] *= g_end;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const u16x4 k0 = mc_ld_tr(&sm.k[u * 32 + lg * 4 + (li >> 2)][dt * 16 + (li & 3) * 4]);
          const u16x4 k1 = mc_ld_tr(&sm.k[u * 32 + 16 + lg * 4 + (li >> 2)][dt * 16 + (li & 3) * 4]);
          const u16x8 a = {k0[0], k0[1], k0[2], k0[3], k1[0], k1[1], k1[2], k1[3]};
          S[dt] = mc_mfma(a, wh[u], S[dt]);
          S[dt] = mc_mfma(a, wl[u], S[dt]);
        }
      }
    }
  }

  if (active && col < CB) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int i0 = dt * 16 + lg * 4;
      if (i0 < Dst) {
        float* dst = at(i0);
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[(long)r * nthr] = S[dt][r];
      }
    }
  }
}

// The same walk for heads of 128 key entries and value blocks of 64 columns, rows straight
// from memory into LDS (load_to_lds), a chunk ahead: one barrier a chunk, and no registers
// or LDS writes between.
// Every operand is 16 bytes a lane: accumulators hold the rows of a pair of blocks in the order
// of walk_row, so that a lane has eight neighbours of a contraction.  Rows of q and k are 16
// pieces of 16 bytes, piece c of row r at c ^ r or c ^ k_swizzle(r): the 16 lanes of a pass
// (0-3, 12-15 and of the next group 4-11, or the others) meet all banks, k's transposing
// reads of 32 lanes two pieces a bank.  Rows of v keep pairs of pieces together.
// 8 prompts of 1000 tokens, 32 heads, both kernels and the first tokens behind (us; start ->
// now) 151 -> 142; 1 of 4844 284 -> 237; 2 of 1838, 64 heads 157 -> 135; 14 of 283 114 -> 102;
// 13 of 20 74 -> 70.

// Row i of block tt: blocks come in pairs whose rows are dealt so that a lane's four rows of both
// are eight neighbours, an operand of the next product that the other side reads as 16 bytes.
LIG_DEVICE constexpr int walk_row(int tt, int i) { return tt / 2 * 32 + i / 4 * 8 + i % 4 + tt % 2 * 4; }
LIG_DEVICE int k_swizzle(int r) {
  const int x = r >> 3 & 3;
  return (r & 3) << 2 | ((x ^ x >> 1) & 1) << 1 | x >> 1;
}
LIG_DEVICE int v_swizzle(int r) { return (r & 3) | (r >> 3 & 1) << 2; }

// VEC: values lie where 16-byte loads may read them, else they come through registers.
template <int NW, bool VEC>
__global__ __launch_bounds__(NW * WAVE_SIZE, 1) void delta_chunk_walk_kernel(const MsArgs A, const DeltaWalkChunk* __restrict__ scratch) {
  constexpr int D = 128, KB = D / 32, DT = D / 16;
  constexpr int QK = MC_T * D, V = MC_T * NW * 16;  // 16-bit units
  constexpr int CHUNK = sizeof(DeltaWalkChunk) / 2, BUF = 2 * QK + V + CHUNK;
  static_assert(sizeof(DeltaWalkChunk) % 1024 == 0 && 2 * BUF <= 80 * 1024, "LDS of a CU");
  __shared__ __align__(16) uint16_t sm[2 * BUF];

  const int seg = blockIdx.x, h = blockIdx.y;
  const int n = A.seg_len[seg];
  if (n <= 0 || n < A.len_min) return;
  const int H = A.H, Dv = A.Dv, CB = MS_COLS;
  const long r0 = A.seg_start[seg];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int blk = blockIdx.z * (NW / 4) + (wave >> 2);
  const bool active = blk < A.NB;  // others compute on another block's values and store nothing
  const int c0 = blk * CB;
  const int col = (wave & 3) * 16 + li;  // the state column this lane holds
  const uint16_t* q = (const uint16_t*)A.q + (h / A.rep) * D;
  const uint16_t* k = (const uint16_t*)A.k + (h / A.rep) * D;
  const uint16_t* v = (const uint16_t*)A.v + h * Dv;
  const DeltaWalkChunk* ch = scratch + delta_chunk_slot(r0, 0, seg) * H + h;
  const int out_row = H * Dv * 4;

  const uint32_t lds = lds_address(sm);
  u16x8 vr[2];
  auto fetch = [&](int t0, int buf) __attribute__((always_inline)) {
    // rows past the portion's end read its last token: their write strength and their
    // weight in the state are zero and their outputs are not stored
    const int last = min(n - 1 - t0, MC_T - 1);
    const uint32_t to = lds + buf * BUF * 2;
    const uint16_t* qb = q + (r0 + t0) * A.q_stride;
    const uint16_t* kb = k + (r0 + t0) * A.k_stride;
    const uint16_t* vb = v + (r0 + t0) * A.v_stride;
#pragma unroll
    for (int j = 0; j < 16 / NW; ++j) {
      const int i = wave + j * NW, row = i * 4 + (lane >> 4), at = min(row, last);
      load_to_lds(qb, (uint32_t)at * (uint32_t)A.q_stride * 2 + (((lane & 15) ^ (row & 15)) << 4), to + i * 1024);
      load_to_lds(kb, (uint32_t)at * (uint32_t)A.k_stride * 2 + (((lane & 15) ^ k_swizzle(row)) << 4), to + QK * 2 + i * 1024);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = wave + j * NW;
      const int row = NW == 8 ? i * 4 + (lane >> 4) : i * 8 + (lane >> 3), at = min(row, last);
      const int c = NW == 8 ? (lane & 15) ^ v_swizzle(row) << 1 : (lane & 7) ^ v_swizzle(row) >> 1 << 1;
      const int b = blockIdx.z * (NW / 4) + (c >> 3);
      const uint32_t off = (uint32_t)at * (uint32_t)A.v_stride + (b < A.NB ? b * CB + (c & 7) * 8 : 0);
      if constexpr (VEC) {
        load_to_lds(vb, off * 2, to + QK * 4 + i * 1024);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) vr[j][e] = vb[off + e];
      }
    }
    const char* cb = reinterpret_cast<const char*>(ch + (long)(t0 / MC_T) * H);
#pragma unroll
    for (int j = 0; j < (CHUNK / 512 + NW - 1) / NW; ++j) {
      const int i = wave + j * NW;
      if (i < CHUNK / 512) load_to_lds(cb + i * 1024, lane * 16, to + (QK * 2 + V) * 2 + i * 1024);
    }
  };
  auto keep = [&](int buf) __attribute__((always_inline)) {  // values from registers
    if constexpr (!VEC) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        *reinterpret_cast<u16x8*>(sm + buf * BUF + 2 * QK + (wave + j * NW) * 512 + lane * 8) = vr[j];
    }
  };
  fetch(0, 0);
  keep(0);

  // ---- state row: [head][block][entry][column * split + key lane] ----------------------
  const int nthr = CB * A.split, Dst = A.split * A.kpt;
  float* srow = A.state + (long)A.seg_slot[seg] * A.state_stride + (long)(h * A.NB + blk) * A.kpt * nthr;
  const bool resume = A.seg_fresh[seg] == 0;
  // entry i0 of a state column; kpt is a multiple of 4, so the next three follow nthr apart
  auto at = [&](int i0) __attribute__((always_inline)) {
    const int j = i0 / A.kpt;
    return srow + (long)(i0 - j * A.kpt) * nthr + col * A.split + j;
  };
  f32x4 S[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    S[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int i0 = walk_row(dt, 0) + lg * 8;
    if (active && resume && i0 < Dst) {
      const float* src = at(i0);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[dt][r] = src[(long)r * nthr];
    }
  }
  // The walk waits for its loads but not for the four stores of outputs behind them; the
  // first chunk has four into an empty buffer.
  {
    const auto none = __builtin_amdgcn_make_buffer_rsrc(A.out, 0, 0, 0x00027000);
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{0, 0, 0, 0}, none, tt * 16, 0, 0);
  }

  // rows of q, and of k in the order of walk_row
  const int q_at = li * D, k_row = walk_row(0, li), k_at = k_row * D;
  const int q_own = lg ^ li, k_own = lg ^ k_swizzle(k_row);
  // the row that a lane brings a transposing read
  const int tr_row = lg * 8 + (li >> 2), tr_own = (li & 3) ^ k_swizzle(tr_row);
  const int v_at = tr_row * NW * 16 + (((wave & (NW - 1)) ^ (NW == 8 ? v_swizzle(tr_row) : v_swizzle(tr_row) >> 1)) << 4) + (li & 3) * 4;
  const int s_at = (lg >> 1) * 256 + li * 16 + (lg & 1) * 8;

  int buf = 0;
#pragma nounroll
  for (int t0 = 0; t0 < n; t0 += MC_T, buf ^= 1) {
    const int cnt = min(MC_T, n - t0);
    loads_landed<4>();  // the chunk is in LDS, and the other buffer is free
    if (t0 + MC_T < n) fetch(t0 + MC_T, buf ^ 1);
    const uint16_t* qs = sm + buf * BUF;
    const uint16_t* ks = qs + QK;
    const uint16_t* vs = ks + QK;
    const uint16_t* ws = vs + V;
    const DeltaFactors& f = *reinterpret_cast<const DeltaFactors*>(ws + (2 * DC_PAIRS * 2 + 2 * DC_BLOCKS) * 256);
    auto inverse = [&](int half, int tt, int u) __attribute__((always_inline)) {
      return mc_ld16(ws + (half * DC_PAIRS + walk_pair(tt, u)) * 512 + lane * 8);
    };
    // blocks (tt, 2 u) and (tt, 2 u + 1), zeros above the diagonal
    auto scores = [&](int half, int tt, int u) __attribute__((always_inline)) {
      const u16x8 b = mc_ld16(ws + 2 * DC_PAIRS * 512 + (half * DC_BLOCKS + tt * (tt + 1) / 2 + 2 * u) * 256 + s_at);
      return 2 * u + 1 <= tt || lg < 2 ? b : u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    };

    // Batches of products, their operands read one batch ahead; the scalar work of the
    // chain (state -> right-hand sides -> corrections -> state) stands beside products that
    // are not on it.
    const auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
    u16x8 a[2][4];  // rows of k, then of q: 32 entries of all 4 blocks of tokens
    auto read_q = [&](int u) __attribute__((always_inline)) {
      const uint16_t* p = qs + q_at + ((u * 4 ^ q_own) << 3);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) a[u & 1][tt] = mc_ld16(p + tt * 16 * D);
    };
    auto read_k = [&](int u) __attribute__((always_inline)) {
      const uint16_t* p = ks + k_at + ((u * 4 ^ k_own) << 3);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) a[u & 1][tt] = mc_ld16(p + walk_row(tt, 0) * D);
    };
    f32x4 x[4], o[4], c[4];
    u32x4 sh[KB], sl[KB], rh[2], rl[2], uh[2], ul[2], wh[2], wl[2];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) x[tt] = o[tt] = c[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto halves = [&](int u) __attribute__((always_inline)) {
      mc_split4(S[2 * u], 0, sh[u], sl[u]);
      mc_split4(S[2 * u + 1], 1, sh[u], sl[u]);
    };
    // right-hand sides: v - e^G S^T k
    u16x4 vv[4];
    f32x4 ek[4];
    auto right = [&](int tt) __attribute__((always_inline)) {
      f32x4 val;
#pragma unroll
      for (int i = 0; i < 4; ++i) val[i] = bf16_to_f32(vv[tt][i]);
      mc_split4(val - ek[tt] * x[tt], tt & 1, rh[tt / 2], rl[tt / 2]);
    };
    auto correct = [&](int tt, f32x4 wk) __attribute__((always_inline)) {
      mc_split4(c[tt], tt & 1, uh[tt / 2], ul[tt / 2]);
      mc_split4(c[tt] * wk, tt & 1, wh[tt / 2], wl[tt / 2]);
    };
    // ---- the chunk's starting state with all keys, then with all queries --------------------
    read_k(0);
    halves(0);
#pragma unroll
    for (int u = 0; u < KB; ++u) {
      fence();
      if (u + 1 < KB) {
        read_k(u + 1);
        halves(u + 1);
      } else {
        read_q(0);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          vv[tt] = mc_ld_tr(vs + v_at + walk_row(tt, 0) * NW * 16);
          ek[tt] = *reinterpret_cast<const f32x4*>(&f.ek[walk_row(tt, 0) + lg * 8]);
        }
      }
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) x[tt] = mc_mfma(a[u & 1][tt], sh[u], x[tt]);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) x[tt] = mc_mfma(a[u & 1][tt], sl[u], x[tt]);
    }
    auto with_q = [&](int u) __attribute__((always_inline)) {
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) o[tt] = mc_mfma(sh[u], a[u & 1][tt], o[tt]);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) o[tt] = mc_mfma(sl[u], a[u & 1][tt], o[tt]);
    };
    u16x8 th[4][2], tl[4][2];  // the inverse, then the scores: blocks tt, pairs u
    auto read_inverse = [&](int t_lo) __attribute__((always_inline)) {
#pragma unroll
      for (int tt = t_lo; tt < t_lo + 2; ++tt)
#pragma unroll
        for (int u = 0; u <= tt / 2; ++u) {
          th[tt][u] = inverse(0, tt, u);
          tl[tt][u] = inverse(1, tt, u);
        }
    };
    auto read_scores = [&](int t_lo) __attribute__((always_inline)) {
#pragma unroll
      for (int tt = t_lo; tt < t_lo + 2; ++tt)
#pragma unroll
        for (int u = 0; u <= tt / 2; ++u) {
          th[tt][u] = scores(0, tt, u);
          tl[tt][u] = scores(1, tt, u);
        }
    };
    fence();
    read_q(1);
    with_q(0);
    right(0);
    right(1);
    fence();
    read_q(2);
    read_inverse(0);
    with_q(1);
    right(2);
    right(3);
    fence();
    read_q(3);
    read_inverse(2);
    f32x4 wk[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) wk[tt] = *reinterpret_cast<const f32x4*>(&f.wk[walk_row(tt, 0) + lg * 8]);
    with_q(2);
    // ---- corrections u = inverse * right-hand sides ----------------------------------------
    auto solve = [&](int t_lo, int u) __attribute__((always_inline)) {
#pragma unroll
      for (int tt = t_lo; tt < t_lo + 2; ++tt) c[tt] = mc_mfma(th[tt][u], rh[u], c[tt]);
#pragma unroll
      for (int tt = t_lo; tt < t_lo + 2; ++tt) c[tt] = mc_mfma(th[tt][u], rl[u], c[tt]);
#pragma unroll
      for (int tt = t_lo; tt < t_lo + 2; ++tt) c[tt] = mc_mfma(tl[tt][u], rh[u], c[tt]);
    };
    solve(0, 0);
    fence();
    solve(2, 0);
    solve(2, 1);
    correct(0, wk[0]);
    correct(1, wk[1]);
    fence();
    read_scores(0);
    with_q(3);
    correct(2, wk[2]);
    correct(3, wk[3]);
    // ---- weighted scores with the corrections; outputs; the keys' products join the state -------
    const auto dst = __builtin_amdgcn_make_buffer_rsrc(A.out + (r0 + t0) * (long)(H * Dv) + h * Dv + (active ? c0 : 0), 0,
                                                       active ? (cnt - 1) * out_row + CB * 4 : 0, 0x00027000);
    const float g_end = f.eg[MC_T - 1];
    float oc[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) oc[tt] = f.c[tt * 16 + li];
    u16x8 kt[2][4];
    auto read_kt = [&](int g) __attribute__((always_inline)) {  // tokens 32 (g & 1) .. of entries 64 (g >> 1) ..
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int dt = (g >> 1) * 4 + j;
        const uint16_t* p = ks + ((g & 1) * 32 + tr_row) * D + (((dt >> 1) * 4 ^ tr_own) << 3) + (dt & 1) * 4;
        const u16x4 k0 = mc_ld_tr(p), k1 = mc_ld_tr(p + 4 * D);
        kt[g & 1][j] = u16x8{k0[0], k0[1], k0[2], k0[3], k1[0], k1[1], k1[2], k1[3]};
      }
    };
    auto join = [&](int g) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 4; ++j) S[(g >> 1) * 4 + j] = mc_mfma(kt[g & 1][j], wh[g & 1], S[(g >> 1) * 4 + j]);
#pragma unroll
      for (int j = 0; j < 4; ++j) S[(g >> 1) * 4 + j] = mc_mfma(kt[g & 1][j], wl[g & 1], S[(g >> 1) * 4 + j]);
    };
    auto emit = [&](int t_lo, int u) __attribute__((always_inline)) {
#pragma unroll
      for (int tt = t_lo; tt < t_lo + 2; ++tt) o[tt] = mc_mfma(uh[u], th[tt][u], o[tt]);
#pragma unroll
      for (int tt = t_lo; tt < t_lo + 2; ++tt) o[tt] = mc_mfma(ul[u], th[tt][u], o[tt]);
#pragma unroll
      for (int tt = t_lo; tt < t_lo + 2; ++tt) o[tt] = mc_mfma(uh[u], tl[tt][u], o[tt]);
    };
    auto store = [&](int tt) __attribute__((always_inline)) {
      // past the rows: past the buffer's end, dropped
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o[tt]), dst,
                                             (tt * 16 + li) * out_row + ((wave & 3) * 16 + lg * 4) * 4, 0, 0);
    };
    read_kt(0);
    fence();
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) o[tt] *= oc[tt];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) S[dt] *= g_end;
    read_scores(2);
    emit(0, 0);
    read_kt(1);
    join(0);
    fence();
    store(0);
    store(1);
    emit(2, 0);
    read_kt(2);
    join(1);
    fence();
    emit(2, 1);
    read_kt(3);
    join(2);
    fence();
    store(2);
    store(3);
    join(3);
    if (!VEC && t0 + MC_T < n) keep(buf ^ 1);
  }

  if (active) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int i0 = walk_row(dt, 0) + lg * 8;
      if (i0 < Dst) {
        float* dst = at(i0);
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[(long)r * nthr] = S[dt][r];
      }
    }
  }
}

// Workgroups of the first kernel that a CU holds, of heads of that many key entries; 0: unknown.
extern "C" int lig_gated_delta_prepare_workgroups(int D) {
  int n = 0;
  const void* f = D <= 32    ? (const void*)delta_chunk_prepare_kernel<32, DeltaChunk>
                  : D <= 64  ? (const void*)delta_chunk_prepare_kernel<64, DeltaChunk>
                  : D == 128 ? (const void*)delta_chunk_prepare_kernel<128, DeltaWalkChunk>
                  : D < 128  ? (const void*)delta_chunk_prepare_kernel<128, DeltaChunk>
                  : D <= 192 ? (const void*)delta_chunk_prepare_kernel<192, DeltaChunk>
                             : (const void*)delta_chunk_prepare_kernel<256, DeltaChunk>;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, DI_THREADS, 0) == hipSuccess ? n : 0;
}

bool ms_delta_chunks_served(const MsArgs& a) {
  // offsets inside a chunk are 32-bit
  const long lim = 2147483647L / MC_T;
  return a.q_stride <= lim && a.k_stride <= lim && a.v_stride <= lim && a.D % 8 == 0 &&
         a.Dv % 8 == 0 && a.D <= 256 && (long)a.H * a.Dv * 4 <= lim && a.q_stride % 8 == 0 &&
         a.k_stride % 8 == 0 && aligned16(a.q) && aligned16(a.k) && aligned16(a.out);
}

void ms_delta_chunks_launch(const MsArgs& a, int S, int max_seg_len, void* scratch,
                            hipStream_t st) {
  DeltaChunk* sc = (DeltaChunk*)scratch;
  const dim3 gi((max_seg_len + MC_T - 1) / MC_T * a.H, S);
  // Two value blocks per workgroup share the staged operands where the
  // registers of eight waves hold the state, and a workgroup each would not
  // find a CU each.  One call, 32 heads of 128 x 128, one block here and two: 1 prompt
  // of 4000 tokens 192 us, 243; of 1000 62, 77; 2 of these 68, 82; 4 (256 workgroups) 79, 92;
  // 5 124, 97; 8 156, 131; 64 heads, 2 of 1000 79, 91, 3 134, 107; 16 of 500 354, 283.  The other
  // walk: values of 96, 4 of 1000 88, 101, 5 145, 106; heads of 64 x 128 66, 80 and 89, 84, but 8
  // 120, 123; past 128 entries it has no pairs.  That is prompts alone: S counts
  // every segment of a call, also those too short for these kernels, whose workgroups are
  // over at once, so that a prompt beside a few single tokens gets pairs.
  const bool pair = a.NB > 1 && (long)S * a.H * a.NB > 256;
  const bool vec = a.v_stride % 8 == 0 && aligned16(a.v);
  if (a.D == 128 && a.Dv % MS_COLS == 0) {
    DeltaWalkChunk* wc = (DeltaWalkChunk*)scratch;
    hipLaunchKernelGGL((delta_chunk_prepare_kernel<128, DeltaWalkChunk>), gi, dim3(DI_THREADS), 0, st, a, wc);
#define LIG_DW(NW, VEC)                                                                                           \
  hipLaunchKernelGGL((delta_chunk_walk_kernel<NW, VEC>), dim3(S, a.H, (a.NB + NW / 4 - 1) / (NW / 4)), dim3(NW * WAVE_SIZE), \
                     0, st, a, wc)
    if (pair && vec) LIG_DW(8, true);
    else if (pair) LIG_DW(8, false);
    else if (vec) LIG_DW(4, true);
    else LIG_DW(4, false);
#undef LIG_DW
    return;
  }
#define LIG_DS(DP, NW, VEC)                                                                   \
  hipLaunchKernelGGL((delta_chunk_scan_kernel<DP, NW, VEC>),                                  \
                     dim3(S, a.H, (a.NB + NW / 4 - 1) / (NW / 4)), dim3(NW * WAVE_SIZE), 0, st, a, sc)
#define LIG_DC(DP)                                                                            \
  do {                                                                                        \
    hipLaunchKernelGGL((delta_chunk_prepare_kernel<DP, DeltaChunk>), gi, dim3(DI_THREADS), 0, st, a, sc);   \
    constexpr int NW = DP <= 128 ? 8 : 4;                                                     \
    if (pair && vec) LIG_DS(DP, NW, true);                                                    \
    else if (pair) LIG_DS(DP, NW, false);                                                     \
    else if (vec) LIG_DS(DP, 4, true);                                                        \
    else LIG_DS(DP, 4, false);                                                                \
  } while (0)
  if (a.D <= 32) LIG_DC(32);
  else if (a.D <= 64) LIG_DC(64);
  else if (a.D <= 128) LIG_DC(128);
  else if (a.D <= 192) LIG_DC(192);
  else LIG_DC(256);
#undef LIG_DS
#undef LIG_DC
}
