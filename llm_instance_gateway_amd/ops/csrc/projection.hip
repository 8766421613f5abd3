// Projections of up to 1024 rows, long weights' of up to 1792, gfx950, bf16: y = x W^T with x [M, K], W [N, K].
//
// Bound by how fast a CU gets its tiles, W once from HBM, x again for every tile of W's
// rows from the L2, and with some hundred rows by the matrix products.  The launch picks
// tile and cut of K by a sum of what these take (`plan`).
//   * Rows go from memory straight into LDS, stages of 64 or 128 columns in a ring,
//     XOR-swizzled through the choice of what a lane fetches (no bank conflicts, by the
//     counter);
//   * weights under 2^24 entries, where the estimate says so (few rows, or many on so few
//     outputs that larger tiles would be fewer than CUs), and up to 8 rows of a vocabulary:
//     small tiles with the columns of a stage dealt to the waves, whose sums meet in LDS;
//     else projection_wide_kernel;
//   * XCDs start at different quarters of K: in step, all 256 CUs would ask for the same
//     columns of rows 8 KB apart, that is for few memory channels.  Inside an XCD the CUs
//     stay in step and find x in its L2; the tiles of an XCD lie side by side;
//   * where N has too few tiles for the chip, K is cut into parts whose fp32 sums their
//     reader, or a second kernel, adds up in order;
//   * where one tile holds all rows, loads of a large W are non-temporal (`streams`).
#include <type_traits>

#include "common.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// waits for all but the last `behind` stages of NI loads, at most MAX of them
template <int NI, int MAX>
LIG_DEVICE void stages_landed(int behind) {
  if constexpr (MAX == 0) {
    loads_landed<0>();
  } else {
    if (behind >= MAX) loads_landed<MAX * NI>();
    else stages_landed<NI, MAX - 1>(behind);
  }
}

constexpr int XCD_PHASES = 4;  // starting points in K

// acc[i][j]: 16 columns i of W's tile by 16 rows j of x's, as the products leave them.
// A lane holds row li of a tile's 16, 4 columns of it, 8 of a pair: stored so, neighbouring
// lanes are in 16 rows and every one of them is an access of its own, 64 to a kilobyte.  So
// 16 rows at a time go through LDS (`room`, this wave's own) and leave in the order in which
// they lie in memory: parts of 4096 x 14336 at 202 rows 35.0 -> 33.0 us, 384 46 -> 44.4; of 4096 x
// 4096 at 786 32.8 -> 31.1; 28672 x 4096 rounded, 786 rows 151 -> 148; in the mean of 10 weights 202 rows
// 2.5 % faster, 100 and 64 1 %, 48 level, 2 to 33 up to 1.7 % slower (a tenth of a us), which blocks of rows past
// M left out do not mend (1 % at 2 rows, and a branch that costs 0.5 % at 64).
template <int TN, bool PARTIAL>
constexpr int ROOM_ROW = TN * 16 * (PARTIAL ? 4 : 2) + 16;  // bytes of a row, for rows to start 4 banks apart
template <int TM, int TN, bool PARTIAL>
LIG_DEVICE void store_tile(const f32x4_t (&acc)[TN][TM], uint16_t* __restrict__ y, float* __restrict__ part, const int m_at,
                           const int n_at, const int z, const int M, const int N, char* room) {
  constexpr bool PAIRS = TN % 2 == 0;
  constexpr int ROW = ROOM_ROW<TN, PARTIAL>, ES = PARTIAL ? 4 : 2, PIECES = TN * ES;  // 16-byte pieces of a row
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    char* own = room + li * ROW + lg * (PAIRS ? 8 : 4) * ES;
#pragma unroll
    for (int i = 0; i < TN; i += PAIRS ? 2 : 1) {
      char* to = own + i * 16 * ES;
      if constexpr (PARTIAL) {
        *reinterpret_cast<f32x4_t*>(to) = acc[i][j];
        if constexpr (PAIRS) *reinterpret_cast<f32x4_t*>(to + 16) = acc[i + 1][j];
      } else if constexpr (PAIRS) {
        f32x8 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[i][j][e];
          v[4 + e] = acc[i + 1][j][e];
        }
        *reinterpret_cast<u16x8*>(to) = f32x8_to_bf16x8(v);
      } else {
        u32x2 v;
        v[0] = (uint32_t)f32_to_bf16(acc[i][j][0]) | ((uint32_t)f32_to_bf16(acc[i][j][1]) << 16);
        v[1] = (uint32_t)f32_to_bf16(acc[i][j][2]) | ((uint32_t)f32_to_bf16(acc[i][j][3]) << 16);
        *reinterpret_cast<u32x2*>(to) = v;
      }
    }
#pragma unroll
    for (int k = 0; k < (16 * PIECES + 63) / 64; ++k) {
      const int piece = k * 64 + lane, r = piece / PIECES, c = piece % PIECES;
      const int m = m_at + j * 16 + r, n = n_at + c * (16 / ES);
      if (16 * PIECES % 64 && piece >= 16 * PIECES) continue;
      const u32x4 v = *reinterpret_cast<const u32x4*>(room + r * ROW + c * 16);
      if (m >= M || n >= N) continue;
      if constexpr (PARTIAL) *reinterpret_cast<u32x4*>(part + ((size_t)z * M + m) * N + n) = v;
      else *reinterpret_cast<u32x4*>(y + (size_t)m * N + n) = v;
    }
  }
}

// Small weights: tiles of BM x BN, each wave a quarter of a stage's 128 columns.
// PARTIAL: fp32 sums of a part of K to part[z][M][N].
template <int BM, int BN, int ST, bool PARTIAL>
__global__ __launch_bounds__(256, 1) void projection_kernel(
    uint16_t* __restrict__ y, float* __restrict__ part, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
    const int M, const int N, const int K, const int mtiles, const int ntiles) {
  constexpr int NW = 4, PK = 2;
  constexpr int ROWS = BN + BM;              // of a panel of 64 columns: W's, then x's
  constexpr int TM = BM / 16, TN = BN / 16;
  constexpr int NF = PK * ROWS / 8;          // fetches of 8 rows per stage
  constexpr int NI = (NF + NW - 1) / NW;     // of a wave; some of the last wave's may be done twice
  constexpr int STAGE = PK * ROWS * 64;
  static_assert(BM % 16 == 0 && BN % 16 == 0 && (ST - 2) * NI < 64, "");
  constexpr int RING = ST * STAGE, SUMS = (NW - 1) * BM * BN * 2;  // in 16-bit units
  static_assert(RING <= 80 * 1024 && SUMS <= 80 * 1024, "LDS of a CU");
  __shared__ __align__(16) uint16_t sm[RING > SUMS ? RING : SUMS];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // blocks are dealt to the XCDs in turn; the tiles of one lie together
  const int total = gridDim.x, xcd = blockIdx.x & 7;
  const int t = xcd * (total >> 3) + min(xcd, total & 7) + (blockIdx.x >> 3);
  const int mt = t % mtiles, nt = t / mtiles % ntiles, z = t / (mtiles * ntiles);
  const int splits = total / (mtiles * ntiles);
  const int m0 = mt * BM, n0 = nt * BN;
  const int all = K / (64 * PK);
  const int first = (int)((long)all * z / splits);
  const int steps = (int)((long)all * (z + 1) / splits) - first;
  const int shift = (xcd % XCD_PHASES) * steps / XCD_PHASES;

  // 16-byte chunk c of row r goes to c ^ f(r).  Rows past the end repeat the last.
  // With an even number of tiles a wave's W rows are dealt to pairs of them so
  // that a lane ends up with 8 neighbouring columns of y; f is the one for which
  // the 16 rows of an operand read meet all banks.
  constexpr bool PAIRS = TN % 2 == 0;
  auto f_w = [](int r) { return PAIRS ? (r & 3) | ((r >> 1) & 4) : r & 7; };
  const uint32_t lds = lds_address(sm);
  const bool stream_w = mtiles == 1 && streams(N, K);  // no second workgroup reads these rows
  uint32_t off[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int idx = min(wave * NI + i, NF - 1);
    const int panel = idx / (ROWS / 8), r = idx % (ROWS / 8) * 8 + (lane >> 3);
    const bool of_w = r < BN;
    const int row = of_w ? min(r, N - 1 - n0) : min(r - BN, M - 1 - m0);
    off[i] = (uint32_t)row * (uint32_t)K * 2 + panel * 128 + (((lane & 7) ^ (of_w ? f_w(r) : r & 7)) << 4);
  }
  const uint16_t* wp = w + (size_t)n0 * K + (size_t)first * 64 * PK;
  const uint16_t* xp = x + (size_t)m0 * K + (size_t)first * 64 * PK;
  auto fetch = [&](int step) __attribute__((always_inline)) {
    int at = step + shift;
    if (at >= steps) at -= steps;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int idx = min(wave * NI + i, NF - 1);
      const bool of_w = idx % (ROWS / 8) * 8 < BN;
      const uint16_t* base = (of_w ? wp : xp) + (size_t)at * 64 * PK;
      const uint32_t to = lds + (step % ST * STAGE + idx * 512) * 2;
      if (of_w && stream_w) stream_to_lds(base, off[i], to);
      else load_to_lds(base, off[i], to);
    }
  };

  f32x4_t acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int s = 0; s < ST - 1; ++s)
    if (s < steps) fetch(s);

  const int w_row = PAIRS ? (li >> 2) * 8 + (li & 3) : li;
  const int w_f = f_w(w_row);
  const int x_row = BN + li;
  const int c = (wave & 1) * 4 + lg;
  for (int s = 0; s < steps; ++s) {
    stages_landed<NI, ST - 2>(steps - 1 - s);  // and the stage before this one is free
    if (s + ST - 1 < steps) fetch(s + ST - 1);
    const uint16_t* panel = sm + s % ST * STAGE + (wave >> 1) * ROWS * 64;
    bf16x8_t a[TN], b[TM];
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int r = w_row + (PAIRS ? (i >> 1) * 32 + (i & 1) * 4 : i * 16);
      a[i] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(panel + r * 64 + ((c ^ w_f) << 3)));
    }
#pragma unroll
    for (int j = 0; j < TM; ++j)
      b[j] = __builtin_bit_cast(
          bf16x8_t, *reinterpret_cast<const u32x4*>(panel + (x_row + j * 16) * 64 + ((c ^ (li & 7)) << 3)));
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
  }

  float* sums = reinterpret_cast<float*>(sm) + lane * 4;
  constexpr int WAVE = TM * TN * 256;
  __syncthreads();
  if (wave > 0) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
        *reinterpret_cast<f32x4_t*>(sums + (wave - 1) * WAVE + (i * TM + j) * 256) = acc[i][j];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int k = 0; k < NW - 1; ++k)
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] += *reinterpret_cast<const f32x4_t*>(sums + k * WAVE + (i * TM + j) * 256);
  static_assert(16 * ROOM_ROW<TN, PARTIAL> <= sizeof(sm), "");
  store_tile<TM, TN, PARTIAL>(acc, y, part, m0, n0, z, M, N, reinterpret_cast<char*>(sm));
}

// c += a b with c in accumulation registers.  The compiler's own choice between them
// and the others changed from one half of a step to the next, with copies of all of c.
LIG_DEVICE void mfma_acc(f32x4_t& c, bf16x8_t a, bf16x8_t b) {
  asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
// It does not count the cycles to keep between other uses of c and these either.
template <int TN, int TM>
LIG_DEVICE void mfma_apart(f32x4_t (&c)[TN][TM]) {
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) asm volatile("" : "+a"(c[i][j]));
  asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) asm volatile("" : "+a"(c[i][j]));
}

// Waits until no more of this wave's loads are on their way than those of the last
// `left` stages, of which CX of x and CW of W can have been issued.
template <int NX, int NWL, int CX, int CW>
LIG_DEVICE void later_stages(int left) {
  static_assert(CX * NX + CW * NWL < 64, "vmcnt has 6 bits");
  if constexpr (CW == 0) {
    loads_landed<0>();
  } else {
    if (left >= CW) loads_landed<CX * NX + CW * NWL>();
    else later_stages<NX, NWL, (CX < CW - 1 ? CX : CW - 1), CW - 1>(left);
  }
}

// Tiles of 64 rows and more: 2 x 2 waves, one per SIMD, each with a quarter of the
// tile.  Eight waves of an eighth each, which this replaces, read every row of x and W 2 to 4
// times from LDS and waited for each other twice a step; four read two thirds of that, and
// what other waves covered is laid out here by hand:
//   * a step's products come in halves of 32 columns, and between them stand the reads
//     of the next half's operands and the loads of later stages, evenly: neither the
//     matrix cores nor the loads pause.  One barrier per step, at half time;
//   * x has SX slots of 64 columns, W one more: its rows come from memory, x's from the
//     L2.  With the whole LDS so used, two to three stages of W and one to five of x are
//     on their way (a ring of two for both waited 0.5 us per step for its loads);
//   * columns come 64 at a time, a full line of 128 bytes a row: 32 at a time, in a ring
//     of finer grain, they arrived at little more than half the rate.
// Llama-3-8B widths, weights not in any cache (us; eight waves -> this, the library; without the
// other tiles below and with results stored as lanes hold them):
//   rows      gate_up               down                o                 qkv
//    202   71 -> 55 ( 66)     36 -> 35 ( 57)     17 -> 15 (21)     22 -> 20 (25)
//    384  110 -> 77 ( 79)     54 -> 49 ( 75)     23 -> 20 (24)     33 -> 29 (35)
//    832  223 -> 172 (170)   103 -> 81 (128)     40 -> 33 (39)     56 -> 44 (47)
// A head of 128256 x 4096: 202 rows 252 -> 197 (297), 384 rows 409 -> 333 (436).
template <int BM, int BN, int SX, bool PARTIAL, bool STREAM>
__global__ __launch_bounds__(256, 1) void projection_wide_kernel(
    uint16_t* __restrict__ y, float* __restrict__ part, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
    const int M, const int N, const int K, const int mtiles, const int ntiles) {
  constexpr int SW = SX + 1;
  constexpr int TM = BM / 32, TN = BN / 32;  // 16 x 16 tiles of a wave, and its loads of 8 rows per stage
  static_assert(BM % 32 == 0 && BN % 32 == 0 && TM * TN >= 4 && SX >= 2, "");
  constexpr int XS = BM * 64, WS = BN * 64, X0 = SW * WS;
  static_assert(X0 + SX * XS <= 80 * 1024, "LDS of a CU");
  __shared__ __align__(16) uint16_t sm[X0 + SX * XS];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;

  // as above: the tiles of an XCD lie together, XCDs start at different quarters of K
  const int total = gridDim.x, xcd = blockIdx.x & 7;
  const int t = xcd * (total >> 3) + min(xcd, total & 7) + (blockIdx.x >> 3);
  const int mt = t % mtiles, nt = t / mtiles % ntiles, z = t / (mtiles * ntiles);
  const int splits = total / (mtiles * ntiles);
  const int m0 = mt * BM, n0 = nt * BN;
  const int all = K / 64;
  const int first = (int)((long)all * z / splits);
  const int steps = (int)((long)all * (z + 1) / splits) - first;
  const int shift = (xcd % XCD_PHASES) * steps / XCD_PHASES;

  constexpr bool PAIRS = TN % 2 == 0;
  auto f_w = [](int r) { return PAIRS ? (r & 3) | ((r >> 1) & 4) : r & 7; };
  const uint32_t lds = lds_address(sm);
  uint32_t xoff[TM], woff[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = (wave + i * 4) * 8 + (lane >> 3);
    xoff[i] = (uint32_t)min(r, M - 1 - m0) * (uint32_t)K * 2 + (((lane & 7) ^ (r & 7)) << 4);
  }
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int r = (wave + i * 4) * 8 + (lane >> 3);
    woff[i] = (uint32_t)min(r, N - 1 - n0) * (uint32_t)K * 2 + (((lane & 7) ^ f_w(r)) << 4);
  }
  const uint16_t* wp = w + (size_t)n0 * K + (size_t)first * 64;
  const uint16_t* xp = x + (size_t)m0 * K + (size_t)first * 64;
  auto at = [&](int step) {
    const int a = step + shift;
    return (size_t)(a >= steps ? a - steps : a) * 64;
  };
  auto fetch_x = [&](int step, int i) __attribute__((always_inline)) {
    load_to_lds(xp + at(step), xoff[i], lds + (X0 + step % SX * XS + wave * 512) * 2 + i * 4096);
  };
  auto fetch_w = [&](int step, int i) __attribute__((always_inline)) {
    const uint32_t to = lds + (step % SW * WS + wave * 512) * 2 + i * 4096;
    if (STREAM) stream_to_lds(wp + at(step), woff[i], to);
    else load_to_lds(wp + at(step), woff[i], to);
  };

  f32x4_t acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  mfma_apart(acc);

  // loads go out in one order throughout: W(0), x(0), W(1), x(1), ...
#pragma unroll
  for (int s = 0; s < SX; ++s) {
    if (s < steps) {
#pragma unroll
      for (int i = 0; i < TN; ++i) fetch_w(s, i);
#pragma unroll
      for (int i = 0; i < TM; ++i) fetch_x(s, i);
    }
  }

  const int w_row = wn * TN * 16 + (PAIRS ? (li >> 2) * 8 + (li & 3) : li);
  const int w_f = f_w(w_row);
  const int x_row = wm * TM * 16 + li;
  const uint16_t* wl[2] = {sm + w_row * 64 + ((lg ^ w_f) << 3), sm + w_row * 64 + (((4 + lg) ^ w_f) << 3)};
  const uint16_t* xl[2] = {sm + X0 + x_row * 64 + ((lg ^ (li & 7)) << 3), sm + X0 + x_row * 64 + (((4 + lg) ^ (li & 7)) << 3)};
  bf16x8_t a[2][TN], b[2][TM];
  // operand r of half kk of a stage: x's rows, then W's
  auto read = [&](int kk, int ws, int xs, int r) __attribute__((always_inline)) {
    if (r < TM) {
      b[kk][r] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(xl[kk] + xs * XS + r * 16 * 64));
    } else {
      const int i = r - TM;
      a[kk][i] = __builtin_bit_cast(
          bf16x8_t, *reinterpret_cast<const u32x4*>(wl[kk] + ws * WS + (PAIRS ? (i >> 1) * 32 + (i & 1) * 4 : i * 16) * 64));
    }
  };
  // The products of half kk of stage s.  READ: between them the operands of the half
  // behind it, from slots ws and xs, over three quarters of the time; FETCH: the loads
  // of stage s + SX, W's in the first half, into the slot of the stage before, x's in
  // the second, into this one's, read by all at the barrier between.
  constexpr int OPS = TM + TN, MM = TM * TN, BUSY = MM * 3 / 4;
  auto half = [&](auto kk_, auto fetch_, auto read_, int s, int ws, int xs) __attribute__((always_inline)) {
    constexpr int kk = decltype(kk_)::value;
    constexpr bool FETCH = decltype(fetch_)::value, READ = decltype(read_)::value;
    constexpr int LOADS = kk == 0 ? TN : TM;
#pragma unroll
    for (int m = 0; m < MM; ++m) {
      const int i = m / TM, j = m % TM;
      mfma_acc(acc[i][j], a[kk][i], b[kk][j]);
      if (READ) {
#pragma unroll
        for (int r = (m * OPS + BUSY - 1) / BUSY; r < ((m + 1) * OPS + BUSY - 1) / BUSY && r < OPS; ++r) read(kk ^ 1, ws, xs, r);
      }
      if (FETCH) {
#pragma unroll
        for (int r = (m * LOADS + MM - 1) / MM; r < ((m + 1) * LOADS + MM - 1) / MM && r < LOADS; ++r) {
          if (kk == 0) fetch_w(s + SX, r);
          else fetch_x(s + SX, r);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr std::integral_constant<int, 0> k0{};
  constexpr std::integral_constant<int, 1> k1{};
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  later_stages<TM, TN, SX - 1, SX - 1>(steps - 1);
#pragma unroll
  for (int r = 0; r < OPS; ++r) read(0, 0, 0, r);
  int s = 0;
  for (; s + SX < steps; ++s) {
    half(k0, yes, yes, s, s % SW, s % SX);
    later_stages<TM, TN, SX - 2, SX - 1>(SX);  // the next stage is there; this one's operands have been read
    half(k1, yes, yes, s, (s + 1) % SW, (s + 1) % SX);
  }
  for (; s + 1 < steps; ++s) {
    half(k0, no, yes, s, s % SW, s % SX);
    later_stages<TM, TN, SX - 2, SX - 2>(steps - 2 - s);
    half(k1, no, yes, s, (s + 1) % SW, (s + 1) % SX);
  }
  half(k0, no, yes, s, s % SW, s % SX);
  half(k1, no, no, 0, 0, 0);
  mfma_apart(acc);
  // the last stage has been read by all
  __syncthreads();
  constexpr int ROOM = 16 * ROOM_ROW<TN, PARTIAL>;
  static_assert(4 * ROOM <= sizeof(sm), "");
  store_tile<TM, TN, PARTIAL>(acc, y, part, m0 + wm * TM * 16, n0 + wn * TN * 16, z, M, N, reinterpret_cast<char*>(sm) + wave * ROOM);
}

__global__ __launch_bounds__(256) void projection_sum_kernel(uint16_t* __restrict__ y, const float* __restrict__ part,
                                                             const long n, const int splits) {
  const long e = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
  if (e >= n) return;
  f32x8 s = *reinterpret_cast<const f32x8*>(part + e);
  for (int k = 1; k < splits; ++k) s += *reinterpret_cast<const f32x8*>(part + k * n + e);
  *reinterpret_cast<u16x8*>(y + e) = f32x8_to_bf16x8(s);
}

// Small weights: BM, BN, ST of projection_kernel (4 waves over the columns, steps of 128).
#define LIG_TILES(X) \
  X(16, 16, 8)       \
  X(16, 32, 6)       \
  X(32, 32, 8)
// Else BM, BN, SX of projection_wide_kernel.  What is left of 34 shapes when those go
// that no size of 17 projections and 23 row counts misses by more than a few per cent:
// the one picked is 2 % slower than the best of all in the mean, 17 % at the worst.
#define LIG_WIDE_TILES(X) \
  X(64, 64, 5)            \
  X(64, 96, 5)            \
  X(64, 128, 4)           \
  X(96, 128, 4)           \
  X(128, 128, 3)          \
  X(128, 192, 2)          \
  X(128, 256, 2)          \
  X(160, 128, 3)          \
  X(160, 256, 2)          \
  X(192, 256, 2)          \
  X(224, 96, 3)           \
  X(224, 128, 3)          \
  X(224, 256, 2)          \
  X(256, 256, 2)

// And tiles that run in the place of one of these, with the same parts of K, where the
// estimate is 3 % lower: of 224 and 288 columns where 28672 outputs are 112 tiles of 256
// each row of tiles and leave the chip's last turn half empty, and other products likewise.
// Llama-3-8B's gate_up (us, before -> after; launch behind launch, and between copies): 384
// rows 79.6 -> 74.6, 83.7 -> 82.3; 512 97 -> 95, 93.5 -> 92.5; 786 166 -> 151, 163 -> 152; 1000 184 -> 180,
// 180 -> 172.  They run 91 of 527 sizes of 19 projections at 48 to 1024 rows, 7 % faster in the
// mean launch behind launch, one of them 1 % slower.  Stages of x and W by loaders of their own,
// W's up to eight ahead, changed nothing (gate_up at 202 rows 54.5 us and 57): under that
// load the chip runs at 1.7 to 1.9 GHz, and at 2.0 without any loads.
#define LIG_OTHER_TILES(X) \
  X(160, 224, 2)           \
  X(160, 288, 2)           \
  X(192, 128, 3)           \
  X(192, 224, 2)           \
  X(224, 192, 2)           \
  X(224, 224, 2)           \
  X(256, 192, 2)           \
  X(256, 224, 2)           \
  X(288, 224, 2)

struct TileShape {
  int bm, bn, k_step;
};
constexpr TileShape TILES[] = {
#define X(BM, BN, ST) {BM, BN, 128},
    LIG_TILES(X)
#undef X
#define X(BM, BN, SX) {BM, BN, 64},
    LIG_WIDE_TILES(X)
#undef X
};
constexpr TileShape OTHER_TILES[] = {
#define X(BM, BN, SX) {BM, BN, 64},
    LIG_OTHER_TILES(X)
#undef X
};
constexpr int FEW = 3;  // tiles of the first kind
constexpr int TILE_COUNT = sizeof(TILES) / sizeof(TILES[0]), OTHER_COUNT = sizeof(OTHER_TILES) / sizeof(OTHER_TILES[0]);
constexpr int MAX_SPLITS = 8;
constexpr int CUS = 256;

struct Plan {
  int tile, splits;
};

// A kernel's time in us, as a regression on: per step of 64 columns of a tile its products,
// its rows of W, its rows of x; launch, tile; W from memory at `hbm` TB/s; a cut of K
// and, in millionths, every sum of it.  Fitted to 17000 measured times, 6 % off them: 1 to
// 2048 rows (FEW_COST 1 to 128), 1536 to 128256 outputs, 2048 to 28672 columns.  Outside of
// these it picks a tile that is right but was not measured, and its terms are no prices: with
// few rows those of W and x come out negative.
struct Cost {
  double area, w_row, x_row, step, launch, tile, hbm, cut, sum;
};
constexpr Cost FEW_COST = {0.0005405, -0.005728, -0.0135, 0.2466, 3.263, 0.1869, 8.987, -0.6106, 3.765};
constexpr Cost WIDE_COST = {9.45e-06, 0.001368, 0.001277, 0.004109, 0.9942, 2.333, 7.596, -0.2958, 1.212};

double estimate(const TileShape& s, const Cost& c, int splits, int M, int N, int K) {
  const long tiles = (long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn);
  const double step = s.bm * s.bn * c.area + s.bn * c.w_row + s.bm * c.x_row + c.step;
  const double stream = N * (double)K * 2e-6 / c.hbm;
  const double work = (tiles * splits + CUS - 1) / CUS * (K / 64.0 / splits * step + c.tile);
  const double t = c.launch + sqrt(work * work + stream * stream);
  return splits > 1 ? t + c.cut + c.sum * 1e-6 * splits * M * N : t;
}

// Tall tiles that would be mostly padding were not measured.
bool padding(const TileShape& s, int M) { return s.bm > 64 && 5 * M < 3 * s.bm; }

// The first tiles are for small weights: 16 rows of 28672 x 4096 take 41 us on them, 36
// on tiles of 64 x 128; of 4096 x 4096 both 7.7; of 2048 x 2048 4.1 and 4.7.
Plan plan(int M, int N, int K) {
  // one wave of workgroups after the other, each over in a few us: 1 row of 128256 x 4096
  // 149 us, 153 to 156 on the next best tiles; 8 rows of 57344 x 8192 140, 149; 16 rows level
  if (M <= 8 && N > 32768 && K % TILES[0].k_step == 0) return {0, 1};
  Plan best = {-1, 0};
  double least = 0;
  for (int i = 0; i < TILE_COUNT; ++i) {
    const TileShape& s = TILES[i];
    if (K % s.k_step || (i < FEW ? (long)N * K >= 1L << 24 : padding(s, M))) continue;
    const long tiles = (long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn);
    for (int splits = 1; splits <= MAX_SPLITS; ++splits) {
      if (splits > 1 && (tiles * splits > 2 * CUS + 88 || K / s.k_step / splits < 6)) break;
      const double t = estimate(s, i < FEW ? FEW_COST : WIDE_COST, splits, M, N, K);
      if (best.tile < 0 || t < least) {
        least = t;
        best = {i, splits};
      }
    }
  }
  return best;
}

// The tile that runs a plan: its own, or TILE_COUNT and more for one of the others.  Its tiles begin at
// other places in K, so that sums are of the same terms in another order: of 786 x 28672 x 4096 one
// rounded result in 80000 differs, and the fp32 error against 64 bits stays 3.95e-7.
int tile_of(const Plan& p, int M, int N, int K) {
  if (p.tile < FEW || M > 1024) return p.tile;  // not measured
  int tile = p.tile;
  double least = 0.97 * estimate(TILES[tile], WIDE_COST, p.splits, M, N, K);
  for (int i = 0; i < OTHER_COUNT; ++i) {
    if (padding(OTHER_TILES[i], M)) continue;
    const double t = estimate(OTHER_TILES[i], WIDE_COST, p.splits, M, N, K);
    if (t < least) {
      least = t;
      tile = TILE_COUNT + i;
    }
  }
  return tile;
}

struct Product {
  uint16_t* y;
  float* part;
  const uint16_t *x, *w;
  int M, N, K;
  hipStream_t stream;
};

template <int BM, int BN, int ST>
void launch_few(const Product& p, int splits) {
  const int mtiles = (p.M + BM - 1) / BM, ntiles = (p.N + BN - 1) / BN;
  const dim3 grid(mtiles * ntiles * (p.part ? splits : 1)), block(256);
#define LAUNCH(PARTIAL)                                                                                                \
  hipLaunchKernelGGL((projection_kernel<BM, BN, ST, PARTIAL>), grid, block, 0, p.stream, p.y, p.part, p.x, p.w, p.M, p.N, \
                     p.K, mtiles, ntiles)
  if (p.part) LAUNCH(true);
  else LAUNCH(false);
#undef LAUNCH
}

template <int BM, int BN, int SX>
void launch_wide(const Product& p, int splits) {
  const int mtiles = (p.M + BM - 1) / BM, ntiles = (p.N + BN - 1) / BN;
  const dim3 grid(mtiles * ntiles * (p.part ? splits : 1)), block(256);
#define LAUNCH(PARTIAL, STREAM)                                                                                          \
  hipLaunchKernelGGL((projection_wide_kernel<BM, BN, SX, PARTIAL, STREAM>), grid, block, 0, p.stream, p.y, p.part, p.x, p.w, \
                     p.M, p.N, p.K, mtiles, ntiles)
  const bool stream = mtiles == 1 && streams(p.N, p.K);  // no second workgroup reads these rows
  if (p.part && stream) LAUNCH(true, true);
  else if (p.part) LAUNCH(true, false);
  else if (stream) LAUNCH(false, true);
  else LAUNCH(false, false);
#undef LAUNCH
}

}  // namespace

extern "C" {

// Sizes that these kernels are for where their reader adds up the parts of K.  Above 256
// rows, from 3072 columns on, they take 0.6 to 1 of the library's time, of the largest
// matrices 0.9 to 1 (384 rows: 6144 x 4096 27 us here, 37 there; 4096 x 14336 45, 79;
// 28672 x 4096 75, 82; 786: 150, 172; 960: 177, 183).  With many tiles of fewer columns neither
// was ahead, on the planned tiles and with results as lanes hold them (16384 x 2048: 288 rows 24, 27; 384 29, 27).
// Above 1024 rows it is large weights with long rows, to 1792, where all of K in one part
// fills the chip (here, the library's; 8192 x 28672: 1152 rows 440, 440; 1408 500, 512; 1792
// 572, 779; 8192 x 16384: 1280 250, 262; 12288 x 28672: 1536 842, 1422; 5120 x 13824: 1792 207,
// 216).  From 1793 on, measured like 16384 x 2048, they lost as often as they won (1920: 644, 647; 373, 363;
// 16384 x 53248 2438, 2299).  In parts 4096 x 14336 would win too (1216 rows 115, 149), but where a step's
// other products are the library's nothing adds them up, and the sum takes what the cut gains.
bool lig_projection_serves(long M, long N, long K) {
  if (M < 1 || M > 1792 || N < 1 || N > (1 << 24) || K < 64 || K > (1 << 20) || N % 8 || K % 64) return false;
  if (M > 1024) return K >= 8192 && K >= 2 * N && N * K >= 1L << 26 && plan((int)M, (int)N, (int)K).splits == 1;
  return M <= 256 || ((M + 255) / 256) * ((N + 255) / 256) <= 64 || K >= 3072 || (M <= 384 && N >= 65536);
}

// Whether a served product that has to come rounded, its parts added up by a launch
// of its own, runs here too (us here, the library's):
//   * to 128 rows it does (100 x 28672 x 4096: 43, 56), but for a vocabulary's worth of short
//     rows of W, which gain little (24 x 57344 x 1024: 22, 24);
//   * to 256 rows where K is cut (202 x 4096 x 14336: 41, 57; 202 x 4096 x 4096: 19, 22, but
//     256 of these 20, 23 with a launch more) or the weight large (202 x 28672 x 4096: 56, 66;
//     202 x 57344 x 8192: 189, 200);
//   * above, large weights do at any row count (384 x 4096 x 14336: 53, 79; 384 x 28672 x
//     4096: 75, 82) and others where K is cut into many parts.  What is left gains a few us
//     at most (1000 x 4096 x 4096: 38, 42; 786 x 6144 x 4096: 43, 47; 448: 34, 33).
// Of smaller weights the library's call takes longer on the host than is gained, which steps
// of narrow models wait for: 300 rows, 16 layers of 2048 columns 2106 us, 2488 with its
// products.
bool lig_projection_pays(long M, long N, long K) {
  if (M > 16 && N > 32768 && K < 2048) return false;
  if (M <= 128 || N >= 65536 || N * K < 1L << 24) return true;
  if (M > 1024) return true;
  const int splits = plan((int)M, (int)N, (int)K).splits;
  if (M > 256) return splits >= 4 || N * K >= 1L << 25;
  if (splits > 1) return (K > N || M <= 224 || N >= 6144) && (splits > 2 || (N >= 4096 && N <= 16384));
  return (K <= 4096 && N >= 8192 && N <= 32768) || N * K >= 1L << 28;
}

// Tile and parts of K, as one number.  To launch it, on that tile or one in its place: y alone where K is in one part,
// y and room for the fp32 sums [parts, M, N], or that room alone, which then holds the
// parts for the caller to add up.
int lig_projection_plan(int M, int N, int K) {
  const Plan p = plan(M, N, K);
  return p.tile * (MAX_SPLITS + 1) + p.splits;
}
int lig_projection_splits(int p) { return p % (MAX_SPLITS + 1); }
int lig_projection_tile(int p) { return TILES[p / (MAX_SPLITS + 1)].bm * 1000 + TILES[p / (MAX_SPLITS + 1)].bn; }
int lig_projection_runs(int p, int M, int N, int K) {
  const int tile = tile_of({p / (MAX_SPLITS + 1), p % (MAX_SPLITS + 1)}, M, N, K);
  const TileShape& s = tile < TILE_COUNT ? TILES[tile] : OTHER_TILES[tile - TILE_COUNT];
  return s.bm * 1000 + s.bn;
}

void lig_projection_launch(int p, uint16_t* y, float* part, const uint16_t* x, const uint16_t* w, int M, int N, int K,
                           hipStream_t stream) {
  const int splits = p % (MAX_SPLITS + 1), tile = tile_of({p / (MAX_SPLITS + 1), splits}, M, N, K);
  int i = 0;
  const Product a = {y, part, x, w, M, N, K, stream};
#define X(BM, BN, ST) \
  if (tile == i++) launch_few<BM, BN, ST>(a, splits);
  LIG_TILES(X)
#undef X
#define X(BM, BN, SX) \
  if (tile == i++) launch_wide<BM, BN, SX>(a, splits);
  LIG_WIDE_TILES(X)
  LIG_OTHER_TILES(X)
#undef X
  if (part && y) {
    const long n = (long)M * N;
    hipLaunchKernelGGL(projection_sum_kernel, dim3((n / 8 + 255) / 256), dim3(256), 0, stream, y, part, n, splits);
  }
}

}  // extern "C"
