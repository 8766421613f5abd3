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
// 32 heads, 65 with a load per tile in turn.
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
// 2-byte loads of values, 125 without the last two, 95 now: some 11 000 cycles
// a chunk, of which the operand reads of q and k by all waves take 2600 (LDS
// bandwidth) and the two barriers 1200.  Four waves per workgroup and two
// workgroups per CU: slower by 30 us, as q, k and the first kernel's blocks
// come and go twice; but where that still leaves every workgroup a CU of its
// own, a chunk takes 8700 cycles instead of 11000.  Two waves each, on up to
// four times the CUs, are no faster than four.  A second set of staged rows,
// one barrier a chunk: slower by 4 to 10 %.
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
  return ((long)R / MC_T + S + 1) * H * (long)sizeof(DeltaChunk);
}

#define DI_THREADS 256
#define DI_ROW 68  // padded fp32 LDS row

template <int DP>
__global__ __launch_bounds__(DI_THREADS) void delta_chunk_prepare_kernel(
    const MsArgs A, DeltaChunk* __restrict__ scratch) {
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

  const int seg = blockIdx.y, h = blockIdx.z;
  const int n = A.seg_len[seg];
  const int c0 = blockIdx.x * MC_T;
  if (c0 >= n || n < A.len_min) return;
  const int cnt = min(MC_T, n - c0);
  const long r0 = A.seg_start[seg];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const uint16_t* k = (const uint16_t*)A.k + (h / A.rep) * A.D + (r0 + c0) * A.k_stride;
  const uint16_t* q = (const uint16_t*)A.q + (h / A.rep) * A.D + (r0 + c0) * A.q_stride;
  DeltaChunk* out = scratch + delta_chunk_slot(r0, blockIdx.x, seg) * A.H + h;

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
        *reinterpret_cast<u32x2*>(&out->w[1][0][blk][li][lg * 4]) = u32x2{h0, h1};
        *reinterpret_cast<u32x2*>(&out->w[1][1][blk][li][lg * 4]) = u32x2{l0, l1};
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
    if (s0 <= t) {
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
        *reinterpret_cast<u32x4*>(&out->w[0][0][blk][t & 15][half * 8]) = hi;
        *reinterpret_cast<u32x4*>(&out->w[0][1][blk][t & 15][half * 8]) = lo;
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
  const dim3 gi((max_seg_len + MC_T - 1) / MC_T, S, a.H);
  // Two value blocks per workgroup share the staged operands where the
  // registers of eight waves hold the state, and a workgroup each would not
  // find a CU each.  Both calls, 32 heads of 128 x 128, one block here and two:
  // 1 prompt of 4000 tokens 244 us, 298; of 1000 78, 95; 2 of these 85, 100;
  // 4 (256 workgroups) 100, 114; 5 153, 123; 8 183, 151.  That is prompts alone: S counts
  // every segment of a call, also those too short for these kernels, whose workgroups are
  // over at once, so that a prompt beside a few single tokens gets pairs.
  const bool pair = a.NB > 1 && (long)S * a.H * a.NB > 256;
  const bool vec = a.v_stride % 8 == 0 && aligned16(a.v);
#define LIG_DS(DP, NW, VEC)                                                                   \
  hipLaunchKernelGGL((delta_chunk_scan_kernel<DP, NW, VEC>),                                  \
                     dim3(S, a.H, (a.NB + NW / 4 - 1) / (NW / 4)), dim3(NW * WAVE_SIZE), 0, st, a, sc)
#define LIG_DC(DP)                                                                            \
  do {                                                                                        \
    hipLaunchKernelGGL(delta_chunk_prepare_kernel<DP>, gi, dim3(DI_THREADS), 0, st, a, sc);   \
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
