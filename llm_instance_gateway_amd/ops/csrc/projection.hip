// Projections of up to 1024 rows, gfx950, bf16: y = x W^T with x [M, K], W [N, K].
//
// Bound by how fast a CU gets its tiles: W once from HBM, x again for every tile
// of W's rows from the L2.  A CU keeps about 32 KB of memory loads on their way,
// whatever room it has for them, and they return in order, so the time of a step
// of 64 columns is BN rows of W at the HBM's latency plus BM rows of x at the L2's
// (2.9 and 2.0 ns a row), or the matrix products where those take longer (the tile
// at 1.5 PFLOP/s over 256 CUs).  The launch picks tile and cut of K by that sum
// (`plan`).  Therefore
//   * rows go from memory straight into LDS, a ring of ST stages of PK * 64
//     columns, XOR-swizzled through the choice of what a lane fetches (no bank
//     conflicts, by the counter);
//   * few rows get small tiles with the columns of a stage dealt to the waves
//     (WK), whose sums meet in LDS;
//   * XCDs start at different quarters of K: in step, all 256 CUs would ask for
//     the same columns of rows 8 KB apart, that is for few memory channels
//     (28672 x 4096, 48 rows: 41 us, 52 without).  Inside an XCD the CUs stay in
//     step and find x in its L2; the tiles of an XCD lie side by side.
//   * where N has too few tiles for the chip, K is cut into parts whose fp32 sums
//     a second kernel adds up in order.
// A deeper ring, one of 32-column stages, and operands read a product ahead into
// registers brought nothing.
// Llama-3-8B widths, weights not in any cache, against the library's products (us):
//   rows            gate_up          down           o          qkv
//     48         41 ( 60)       26 ( 37)    11 ( 15)    15 ( 17)
//    202         59 ( 72)       42 ( 62)    19 ( 25)    25 ( 27)  (library at 256)
//    384             (77)       56 ( 77)    26 ( 24)    33 ( 36)
//    832                       103 (115 with tiles of 256 rows)
//   1024                       115 (127)    41 ( 41)
// A head of 128256 x 4096: 256 rows 261 (295), 384 rows 409 (433).
// gate_up at 48 rows reads W at 5.7 TB/s.  Where one tile holds all rows, loads of a
// large W are non-temporal (`streams`): a step of 33 decodes with all its products
// 2326 -> 2267 us, of a prompt of 202 rows 1793 -> 1753.
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

// Tiles of BM x BN, WM x WN waves on them, times WK over the columns.
// PARTIAL: fp32 sums of a part of K to part[z][M][N].
template <int BM, int BN, int WM, int WN, int WK, int PK, int ST, bool PARTIAL>
__global__ __launch_bounds__(64 * WM * WN * WK, WM * WN * WK / 4) void projection_kernel(
    uint16_t* __restrict__ y, float* __restrict__ part, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
    const int M, const int N, const int K, const int mtiles, const int ntiles) {
  constexpr int NW = WM * WN * WK;
  constexpr int ROWS = BN + BM;              // of a panel of 64 columns: W's, then x's
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int NF = PK * ROWS / 8;          // fetches of 8 rows per stage
  constexpr int NI = (NF + NW - 1) / NW;     // of a wave; some of the last wave's may be done twice
  constexpr int STAGE = PK * ROWS * 64;
  static_assert(BM % (16 * WM) == 0 && BN % (16 * WN) == 0 && PK * 2 % WK == 0 && (ST - 2) * NI < 64, "");
  constexpr int RING = ST * STAGE, SUMS = (WK - 1) * BM * BN * 2;  // in 16-bit units
  static_assert(RING <= 80 * 1024 && SUMS <= 80 * 1024, "LDS of a CU");
  __shared__ __align__(16) uint16_t sm[RING > SUMS ? RING : SUMS];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM % WN, wk = wave / (WM * WN);

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

  const int w_row = wn * TN * 16 + (PAIRS ? (li >> 2) * 8 + (li & 3) : li);
  const int w_f = f_w(w_row);
  const int x_row = BN + wm * TM * 16 + li;
  for (int s = 0; s < steps; ++s) {
    stages_landed<NI, ST - 2>(steps - 1 - s);  // and the stage before this one is free
    if (s + ST - 1 < steps) fetch(s + ST - 1);
    const uint16_t* stage = sm + s % ST * STAGE;
#pragma unroll
    for (int kk = 0; kk < PK * 2 / WK; ++kk) {
      const int k32 = wk + kk * WK;
      const uint16_t* panel = stage + (k32 >> 1) * ROWS * 64;
      const int c = (k32 & 1) * 4 + lg;
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
  }

  if constexpr (WK > 1) {
    float* sums = reinterpret_cast<float*>(sm) + lane * 4;
    constexpr int WAVE = TM * TN * 256;
    __syncthreads();
    if (wk > 0) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
          *reinterpret_cast<f32x4_t*>(sums + (wave - WM * WN) * WAVE + (i * TM + j) * 256) = acc[i][j];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int k = 0; k < WK - 1; ++k)
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
          acc[i][j] += *reinterpret_cast<const f32x4_t*>(sums + (k * WM * WN + wave) * WAVE + (i * TM + j) * 256);
  }

  // ---- lane: row li of a tile's 16, 4 columns of it, 8 of a pair -----------------------
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int m = m0 + (wm * TM + j) * 16 + li;
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < TN; i += PAIRS ? 2 : 1) {
      const int n = n0 + (wn * TN + i) * 16 + lg * (PAIRS ? 8 : 4);
      if (n >= N) continue;
      if constexpr (PARTIAL) {
        float* o = part + ((size_t)z * M + m) * N + n;
        *reinterpret_cast<f32x4_t*>(o) = acc[i][j];
        if constexpr (PAIRS) *reinterpret_cast<f32x4_t*>(o + 4) = acc[i + 1][j];
      } else if constexpr (PAIRS) {
        f32x8 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[i][j][e];
          v[4 + e] = acc[i + 1][j][e];
        }
        *reinterpret_cast<u16x8*>(y + (size_t)m * N + n) = f32x8_to_bf16x8(v);
      } else {
        u32x2 v;
        v[0] = (uint32_t)f32_to_bf16(acc[i][j][0]) | ((uint32_t)f32_to_bf16(acc[i][j][1]) << 16);
        v[1] = (uint32_t)f32_to_bf16(acc[i][j][2]) | ((uint32_t)f32_to_bf16(acc[i][j][3]) << 16);
        *reinterpret_cast<u32x2*>(y + (size_t)m * N + n) = v;
      }
    }
  }
}

__global__ __launch_bounds__(256) void projection_sum_kernel(uint16_t* __restrict__ y, const float* __restrict__ part,
                                                             const long n, const int splits) {
  const long e = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
  if (e >= n) return;
  f32x8 s = *reinterpret_cast<const f32x8*>(part + e);
  for (int k = 1; k < splits; ++k) s += *reinterpret_cast<const f32x8*>(part + k * n + e);
  *reinterpret_cast<u16x8*>(y + e) = f32x8_to_bf16x8(s);
}

// BM, BN, WM, WN, WK, PK, ST: what is left of 40 shapes when those go that no size
// of 12 projections and 21 row counts misses by more than a few per cent
#define LIG_TILES(X)          \
  X(16, 16, 1, 1, 4, 2, 8)    \
  X(16, 32, 1, 1, 4, 2, 6)    \
  X(32, 32, 1, 1, 4, 2, 8)    \
  X(32, 64, 1, 4, 1, 1, 8)    \
  X(64, 64, 2, 2, 1, 1, 6)    \
  X(64, 128, 2, 4, 1, 1, 5)   \
  X(96, 64, 2, 2, 1, 1, 5)    \
  X(96, 96, 2, 2, 1, 1, 5)    \
  X(128, 128, 2, 4, 1, 1, 4)  \
  X(192, 64, 4, 2, 1, 1, 4)   \
  X(192, 128, 4, 2, 1, 1, 3)  \
  X(224, 128, 2, 4, 1, 1, 3)  \
  X(128, 256, 2, 4, 1, 1, 3)  \
  X(256, 96, 4, 2, 1, 1, 3)   \
  X(208, 256, 1, 8, 1, 1, 2)  \
  X(192, 256, 2, 4, 1, 1, 2)  \
  X(256, 256, 2, 4, 1, 1, 2)

struct TileShape {
  int bm, bn, k_step;
};
constexpr TileShape TILES[] = {
#define X(BM, BN, WM, WN, WK, PK, ST) {BM, BN, PK * 64},
    LIG_TILES(X)
#undef X
};
constexpr int MAX_SPLITS = 8;
constexpr int CUS = 256;

struct Plan {
  int tile, splits;
};

// Least estimated time, in us: launch; per round of workgroups, its steps of 64
// columns, each the longer of fetching and multiplying; not below W from HBM; the
// sums of a cut K.  The constants are a fit to 5500 measured times, within 8 % of
// them; the tile picked was 1 % slower than the best one in the mean, 17 % at most.
Plan plan(int M, int N, int K) {
  Plan best = {-1, 0};
  double least = 0;
  for (int i = 0; i < (int)(sizeof(TILES) / sizeof(TILES[0])); ++i) {
    const TileShape& s = TILES[i];
    if (K % s.k_step) continue;
    const long tiles = (long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn);
    const double step = fmax(s.bm * s.bn * 2.08e-5, s.bn * 2.9e-3 + s.bm * 2.04e-3);
    for (int splits = 1; splits <= MAX_SPLITS; ++splits) {
      if (splits > 1 && (tiles * splits > 2 * CUS + 88 || K / s.k_step / splits < 6)) break;
      const long rounds = (tiles * splits + CUS - 1) / CUS;
      double t = 3.3 + fmax(rounds * (K / 64.0 / splits * step + 0.2), N * (double)K * 2 / 5.9e6);
      if (splits > 1) t += 2.4 + 2.1e-6 * splits * M * N;
      if (best.tile < 0 || t < least) {
        least = t;
        best = {i, splits};
      }
    }
  }
  return best;
}

}  // namespace

extern "C" {

// Sizes that these kernels are for where their reader adds up the parts of K: the
// library's large tiles are ahead where they are enough for the chip (384 x 28672 x
// 4096: 101 us here, 80 there; 786 x 6144 x 4096: 51 and 47), and behind where N needs
// a cut of K (786 x 4096 x 14336: 100 and 118; 384: 57 and 77) or rows are few.  On a
// vocabulary of 128256 x 4096 it falls behind up to 384 rows: 256 rows 261 us here, 295
// there; 320 399, 401; 384 409, 433; 448 491, 490; 640 709, 620.
bool lig_projection_serves(long M, long N, long K) {
  if (M < 1 || M > 1024 || N < 1 || N > (1 << 24) || K < 64 || K > (1 << 20) || N % 8 || K % 64) return false;
  return M <= 256 || ((M + 255) / 256) * ((N + 255) / 256) <= 64 || (M <= 384 && N >= 65536);
}

// Whether a served product that has to come rounded, its parts added up by a launch
// of its own, is the faster one here.  Drawn from 1912 products, N of 1024 to 128256,
// K of 1024 to 28672, 22 row counts, weights from memory (us here, the library's):
//   * to 128 rows it is, 1.3 times in the mean (100 x 28672 x 4096: 46, 56);
//   * a vocabulary's worth of short rows of W is not (24 x 57344 x 1024: 35, 24);
//   * to 256 rows it is where K is cut (160 x 4096 x 7168: 28, 46), by 1.3 in the mean.
//     In one part it is where N makes about one full round of the chip (202 x 28672 x
//     4096: 64, 67; 256: 75, 69, but the same in a step), not for fewer or longer tiles
//     (256 x 4096 x 4096: 25.9, 22.8; 256 x 57344 x 8192: 263, 220);
//   * above, only a cut into many parts gains more than its sum costs (384 x 4096 x
//     14336: 64, 78; in two 448 x 6144 x 4096: 40, 33; in one 300 x 6144 x 4096: 37, 29).
// Of smaller weights that is a few us, less than what the library's call takes longer
// on the host, which steps of narrow models wait for: 300 rows, 16 layers of 2048
// columns 2106 us, 2488 with the library's.
bool lig_projection_pays(long M, long N, long K) {
  if (M > 16 && N > 32768 && K < 2048) return false;
  if (M <= 128 || N >= 65536 || N * K < 1L << 24) return true;
  const int splits = plan((int)M, (int)N, (int)K).splits;
  if (M > 256) return splits >= 4;
  if (splits > 1) return splits > 2 || (N >= 4096 && N <= 16384);
  return K <= 4096 && N >= 8192 && N <= 32768;
}

// Tile and parts of K, as one number.  To launch it: y alone where K is in one part,
// y and room for the fp32 sums [parts, M, N], or that room alone, which then holds the
// parts for the caller to add up.
int lig_projection_plan(int M, int N, int K) {
  const Plan p = plan(M, N, K);
  return p.tile * (MAX_SPLITS + 1) + p.splits;
}
int lig_projection_splits(int p) { return p % (MAX_SPLITS + 1); }
int lig_projection_tile(int p) { return TILES[p / (MAX_SPLITS + 1)].bm * 1000 + TILES[p / (MAX_SPLITS + 1)].bn; }

void lig_projection_launch(int p, uint16_t* y, float* part, const uint16_t* x, const uint16_t* w, int M, int N, int K,
                           hipStream_t stream) {
  const int tile = p / (MAX_SPLITS + 1), splits = p % (MAX_SPLITS + 1);
  int i = 0;
#define X(BM, BN, WM, WN, WK, PK, ST)                                                                             \
  if (tile == i++) {                                                                                              \
    const int mtiles = (M + BM - 1) / BM, ntiles = (N + BN - 1) / BN;                                             \
    if (part)                                                                                                     \
      hipLaunchKernelGGL((projection_kernel<BM, BN, WM, WN, WK, PK, ST, true>), dim3(mtiles * ntiles * splits),   \
                         dim3(64 * WM * WN * WK), 0, stream, y, part, x, w, M, N, K, mtiles, ntiles);             \
    else                                                                                                          \
      hipLaunchKernelGGL((projection_kernel<BM, BN, WM, WN, WK, PK, ST, false>), dim3(mtiles * ntiles),           \
                         dim3(64 * WM * WN * WK), 0, stream, y, part, x, w, M, N, K, mtiles, ntiles);             \
  }
  LIG_TILES(X)
#undef X
  if (part && y) {
    const long n = (long)M * N;
    hipLaunchKernelGGL(projection_sum_kernel, dim3((n / 8 + 255) / 256), dim3(256), 0, stream, y, part, n, splits);
  }
}

}  // extern "C"
