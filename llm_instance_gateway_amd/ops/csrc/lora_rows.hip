// Multi-LoRA of a Llama layer inside the kernels that stand between its GEMMs;
// bf16, rank 16, gfx950.
//
// y = W x + B (A x) with an adapter per token.  As kernels of their own, the
// products with A read every GEMM input once more and those with B read and
// wrote every GEMM output once more: 3.5 of 15.3 ms of a step with 4000 prompt
// tokens over 8 layers, and two launches of 5-12 us per GEMM in decode steps.
// (That step takes 11.5 ms now; norm with both products of 33 tokens of 8 adapters
// 11.6 us for 15 before, of 384 of 32 16.8 for 26, of 4000 38 for 133.)
// Here
//   * B u is added where the GEMM's output is read anyway: the rotation and
//     cache write (qkv), the residual add and norm (o, down), the gated silu
//     (gate_up);
//   * A x is formed where the GEMM's input is written anyway (norm -> qkv and
//     gate_up, silu -> down); only the attention's output needs a pass (o);
//   * u stays fp32 between the two, where a bf16 workspace held it before.
// Both are matrix instructions.  The rows of a launch are tiles of up to 16
// tokens of one adapter (or of none), listed by the host 16 places a tile, so
// that a lane finds its row in one load; steps without adapters give no list.  In all kernels lane
// (li, lg) holds 8 neighbouring columns lg*8 .. of token li in a group of 32:
//   * u^T = A x^T: those 8 values are the second operand as they are;
//   * y^T += B u^T: with B's rows dealt to two tiles (rows lg*4+i hold columns
//     lg*8+i and lg*8+4+i) the result lands on them.  K is 32 and the rank 16:
//     the upper half of K carries the low parts of u = hi + lo against the same
//     B, so u enters with 16 significant bits at no further instruction.
//
// u: fp32 [parts][tiles][16 tokens][16], summed over the parts by the reader.

#include "common.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int R = 16;  // rank

struct Tile {
  int n, slot;  // tokens, adapter (negative: none)
  int row;      // token of this lane (some token of the tile for lanes past n)
  bool valid;
};

// Workgroups are dealt to the 8 XCDs in turn.  (tile, strip) of this one such that an
// XCD has neighbouring tiles of one strip: tiles of an adapter lie together, and its
// weights come into one L2 instead of all.
struct Place {
  int tile, strip;
};
LIG_DEVICE Place place_of() {
  const unsigned at = blockIdx.x + gridDim.x * blockIdx.y, total = gridDim.x * gridDim.y, xcd = at & 7;
  const unsigned p = xcd * (total >> 3) + min(xcd, total & 7) + (at >> 3);
  return {(int)(p % gridDim.x), (int)(p / gridDim.x)};
}

// without a list: rows in their order, none with an adapter
LIG_DEVICE Tile tile_of(const int* toks, const int* len, const int* slot, int tile, int li, int rows = 0) {
  Tile t;
  if (toks == nullptr) {
    t.n = min(16, rows - tile * 16);
    t.slot = -1;
    t.row = tile * 16 + min(li, t.n - 1);
    t.valid = li < t.n;
    return t;
  }
  t.row = toks[tile * 16 + li];
  t.n = len[tile];
  t.slot = slot[tile];
  t.valid = li < t.n;
  return t;
}

// this lane's operand of B u^T: ranks (lg & 1) * 8 .. of token li, high parts in
// lanes lg < 2 and low parts in the others; u: [16 tokens][16]
LIG_DEVICE bf16x8_t u_operand(const float* u, int li, int lg, bool valid) {
  const f32x4_t a = *reinterpret_cast<const f32x4_t*>(u + li * R + (lg & 1) * 8);
  const f32x4_t b = *reinterpret_cast<const f32x4_t*>(u + li * R + (lg & 1) * 8 + 4);
  u16x8 o;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float v = valid ? (i < 4 ? a[i & 3] : b[i & 3]) : 0.f;
    const uint16_t hi = f32_to_bf16(v);
    o[i] = lg < 2 ? hi : f32_to_bf16(v - bf16_to_f32(hi));
  }
  return __builtin_bit_cast(bf16x8_t, o);
}

// the same from a u in several parts, added up through LDS (256 floats);
// called by all threads of the workgroup
LIG_DEVICE bf16x8_t u_of(const float* u, int parts, int tiles, float* smem, int li, int lg, bool valid) {
  if (parts == 1) return u_operand(u, li, lg, valid);
  for (int e = threadIdx.x; e < 16 * R; e += blockDim.x) {
    float v = 0.f;
#pragma unroll 8
    for (int k = 0; k < parts; ++k) v += u[(size_t)k * tiles * 16 * R + e];
    smem[e] = v;
  }
  __syncthreads();
  const bf16x8_t o = u_operand(smem, li, lg, valid);
  __syncthreads();  // smem is used again
  return o;
}

// In the kernels below the loads of several groups come first and no branch
// stands between them: as `if (lora)` around each group's products, every load
// was waited for by itself (36 us for the norm of 33 rows, 19 so).

// the operands of columns c0 + lg*8 .. +8 of (B u); b: [columns][16] of the adapter
struct BOperand {
  u16x8 lo, hi;
};
LIG_DEVICE BOperand load_b(const uint16_t* b, int c0, int li, int lg) {
  const uint16_t* p = b + (size_t)(c0 + ((li >> 2) << 3) + (li & 3)) * R + (lg & 1) * 8;
  return {*reinterpret_cast<const u16x8*>(p), *reinterpret_cast<const u16x8*>(p + 4 * R)};
}
LIG_DEVICE f32x8 expand(const BOperand& b, bf16x8_t u) {
  const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
  const f32x4_t x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b.lo), u, z, 0, 0, 0);
  const f32x4_t y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b.hi), u, z, 0, 0, 0);
  f32x8 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[i] = x[i];
    o[4 + i] = y[i];
  }
  return o;
}

// columns c0 + lg*8 .. of rank li; a: [16][width] of the adapter
LIG_DEVICE u16x8 load_a(const uint16_t* a, size_t width, int c0, int li, int lg) {
  return *reinterpret_cast<const u16x8*>(a + li * width + c0 + lg * 8);
}
LIG_DEVICE f32x4_t shrink(u16x8 a, u16x8 x, f32x4_t acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, x), acc,
                                                 0, 0, 0);
}
LIG_DEVICE u16x8 load8(const uint16_t* p) { return *reinterpret_cast<const u16x8*>(p); }

// the W waves' sums of u to u_out[tile] (tokens past the tile's end: whatever)
template <int W>
LIG_DEVICE void store_u(float* u_out, f32x4_t acc, float (*red)[16][R], int wave, int li, int lg) {
  *reinterpret_cast<f32x4_t*>(&red[wave][li][lg * 4]) = acc;
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * R; i += 64 * W) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) s += red[w][i / R][i % R];
    u_out[i] = s;
  }
}

// residual += x + B u (ADD), h = rms_norm(residual) * weight, u_out = A h.  One
// workgroup per tile holds its rows in registers in between: 8 waves, each every
// eighth group of 32 columns, NG of them.
template <bool ADD, int NG, bool DELTA, bool TO_U>
LIG_DEVICE void norm_rows(const Tile& t, uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
                          uint16_t* __restrict__ residual, const uint16_t* __restrict__ weight, const float eps,
                          const bf16x8_t u, const uint16_t* __restrict__ b, const uint16_t* __restrict__ a,
                          float* u_out, float (*ss_s)[16], float (*red)[16][R], int wave, int li, int lg) {
  constexpr int hidden = NG * 256;
  constexpr int NB = NG % 8 == 0 ? 8 : NG % 4 == 0 ? 4 : NG;  // groups whose loads are issued together
  constexpr int NB2 = NG % 4 == 0 ? 4 : NG;
  const size_t base = (size_t)t.row * hidden + lg * 8;
  f32x8 v[NG];
  float ss = 0.f;
#pragma unroll
  for (int i0 = 0; i0 < NG; i0 += NB) {
    u16x8 xr[NB], rr[NB];
    BOperand br[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int c0 = ((i0 + i) * 8 + wave) * 32;
      xr[i] = load8(x + base + c0);
      if constexpr (ADD) rr[i] = load8(residual + base + c0);
      if constexpr (DELTA) br[i] = load_b(b, c0, li, lg);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      f32x8& w = v[i0 + i];
      w = bf16x8_to_f32x8(xr[i]);
      if constexpr (ADD) w += bf16x8_to_f32x8(rr[i]);
      if constexpr (DELTA) w += expand(br[i], u);
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += w[j] * w[j];
    }
  }
  if (ADD && t.valid) {
#pragma unroll
    for (int i = 0; i < NG; ++i)
      *reinterpret_cast<u16x8*>(residual + base + (i * 8 + wave) * 32) = f32x8_to_bf16x8(v[i]);
  }
  u16x8 wr[NB2], ar[NB2];
  auto load_second = [&](int i0) {
#pragma unroll
    for (int i = 0; i < NB2; ++i) {
      const int c0 = ((i0 + i) * 8 + wave) * 32;
      wr[i] = load8(weight + c0 + lg * 8);
      if constexpr (TO_U) ar[i] = load_a(a, hidden, c0, li, lg);
    }
  };
  load_second(0);  // on their way while the sums meet
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  if (lg == 0) ss_s[wave][li] = ss;
  __syncthreads();
  ss = 0.f;
#pragma unroll
  for (int w = 0; w < 8; ++w) ss += ss_s[w][li];
  const float inv = rsqrtf(ss / hidden + eps);

  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  u16x8 h[NG];
#pragma unroll
  for (int i0 = 0; i0 < NG; i0 += NB2) {
    if (i0 > 0) load_second(i0);
#pragma unroll
    for (int i = 0; i < NB2; ++i) {
      const f32x8 w = bf16x8_to_f32x8(wr[i]);
      f32x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = v[i0 + i][j] * inv * w[j];
      h[i0 + i] = f32x8_to_bf16x8(o);
      if constexpr (TO_U) acc = shrink(ar[i], h[i0 + i], acc);
    }
  }
  if (t.valid) {
#pragma unroll
    for (int i = 0; i < NG; ++i) *reinterpret_cast<u16x8*>(out + base + (i * 8 + wave) * 32) = h[i];
  }
  if constexpr (TO_U) store_u<8>(u_out, acc, red, wave, li, lg);
}

template <bool ADD, int NG>
__global__ __launch_bounds__(512) void lora_rms_norm_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x, uint16_t* __restrict__ residual,
    const uint16_t* __restrict__ weight, const float eps, const int* __restrict__ toks,
    const int* __restrict__ len, const int* __restrict__ slot,
    const float* u_in, const int parts, const int tiles, const uint16_t* __restrict__ b_stack,
    const uint16_t* __restrict__ a_stack, float* u_out) {
  constexpr int hidden = NG * 256;
  __shared__ float ss_s[8][16];
  __shared__ __align__(16) float red[8][16][R];
  const int tile = place_of().tile;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Tile t = tile_of(toks, len, slot, tile, li);
  if (t.n == 0) return;
  const bool delta = u_in != nullptr && t.slot >= 0, to_u = u_out != nullptr && t.slot >= 0;
  const bf16x8_t u = delta ? u_of(u_in + (size_t)tile * 16 * R, parts, tiles, &red[0][0][0], li, lg, t.valid) : bf16x8_t{};
  const uint16_t* b = delta ? b_stack + (size_t)t.slot * hidden * R : nullptr;
  const uint16_t* a = to_u ? a_stack + (size_t)t.slot * R * hidden : nullptr;
  float* uo = to_u ? u_out + (size_t)tile * 16 * R : nullptr;
#define ROWS(DELTA, TO_U) \
  norm_rows<ADD, NG, DELTA, TO_U>(t, out, x, residual, weight, eps, u, b, a, uo, ss_s, red, wave, li, lg)
  if (ADD && delta && to_u) ROWS(ADD, true);
  else if (ADD && delta) ROWS(ADD, false);
  else if (to_u) ROWS(false, true);
  else ROWS(false, false);
#undef ROWS
}

// The same in two launches for steps of few tiles: one workgroup per tile pulls
// the adapter's 2 x 128 KB and the rows at a single CU's rate (18 us for 9 tiles
// of 4096 columns).  Workgroups here take 256 columns of a tile; the first kernel
// leaves the sums of squares of its columns, the second forms the same values
// again and has the whole row's sum at hand.  u_out gets a part per 256 columns.
constexpr int NORM_STRIP = 256;

template <bool ADD, bool DELTA, bool TO_U, bool SUM>
LIG_DEVICE void norm_strip(const Tile& t, uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
                           uint16_t* __restrict__ residual, const uint16_t* __restrict__ weight, const float eps,
                           const int hidden, const float* u_in, const int parts, const int tiles,
                           const uint16_t* __restrict__ b, const uint16_t* __restrict__ a, float* u_out,
                           const int tiles_out, float* sums,
                           float* smem, int wave, int li, int lg) {
  constexpr int NB = NORM_STRIP / 128;
  const int c_first = place_of().strip * NORM_STRIP + wave * 32;
  const size_t base = (size_t)t.row * hidden + lg * 8;
  u16x8 xr[NB], rr[NB], wr[NB], ar[NB];
  BOperand br[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int c0 = c_first + i * 128;
    xr[i] = load8(x + base + c0);
    if constexpr (ADD) rr[i] = load8(residual + base + c0);
    if constexpr (DELTA) br[i] = load_b(b, c0, li, lg);
    if constexpr (!SUM) wr[i] = load8(weight + c0 + lg * 8);
    if constexpr (!SUM && TO_U) ar[i] = load_a(a, hidden, c0, li, lg);
  }
  const int strips = hidden / NORM_STRIP;
  float total = 0.f;
  if constexpr (!SUM) {
#pragma unroll 8
    for (int k = 0; k < strips; ++k) total += sums[k * 16 + li];
  }
  bf16x8_t u = {};
  if constexpr (DELTA) u = u_of(u_in, parts, tiles, smem, li, lg, t.valid);
  f32x8 v[NB];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    v[i] = bf16x8_to_f32x8(xr[i]);
    if constexpr (ADD) v[i] += bf16x8_to_f32x8(rr[i]);
    if constexpr (DELTA) v[i] += expand(br[i], u);
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += v[i][j] * v[i][j];
  }
  if constexpr (SUM) {
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    if (lg == 0) smem[wave * 16 + li] = ss;
    __syncthreads();
    if (threadIdx.x < 16)
      sums[place_of().strip * 16 + threadIdx.x] =
          smem[threadIdx.x] + smem[16 + threadIdx.x] + smem[32 + threadIdx.x] + smem[48 + threadIdx.x];
  } else {
    const float inv = rsqrtf(total / hidden + eps);
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    u16x8 h[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const f32x8 w = bf16x8_to_f32x8(wr[i]);
      f32x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = v[i][j] * inv * w[j];
      h[i] = f32x8_to_bf16x8(o);
      if constexpr (TO_U) acc = shrink(ar[i], h[i], acc);
    }
    if (t.valid) {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int c0 = c_first + i * 128;
        *reinterpret_cast<u16x8*>(out + base + c0) = h[i];
        if constexpr (ADD) *reinterpret_cast<u16x8*>(residual + base + c0) = f32x8_to_bf16x8(v[i]);
      }
    }
    if constexpr (TO_U) {
      float(*red)[16][R] = reinterpret_cast<float(*)[16][R]>(smem);
      store_u<4>(u_out + (size_t)place_of().strip * tiles_out * 16 * R, acc, red, wave, li, lg);
    }
  }
}

template <bool ADD, bool SUM>
__global__ __launch_bounds__(256) void lora_norm_strip_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x, uint16_t* __restrict__ residual,
    const uint16_t* __restrict__ weight, const float eps, const int hidden, const int* __restrict__ toks,
    const int* __restrict__ len, const int* __restrict__ slot, const float* u_in, const int parts, const int tiles,
    const uint16_t* __restrict__ b_stack, const uint16_t* __restrict__ a_stack, float* u_out, const int tiles_out,
    float* sums) {
  __shared__ __align__(16) float smem[4 * 16 * R];
  const int tile = place_of().tile;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Tile t = tile_of(toks, len, slot, tile, li);
  if (t.n == 0) return;
  const bool delta = u_in != nullptr && t.slot >= 0, to_u = u_out != nullptr && t.slot >= 0;
  const float* ui = delta ? u_in + (size_t)tile * 16 * R : nullptr;
  const uint16_t* b = delta ? b_stack + (size_t)t.slot * hidden * R : nullptr;
  const uint16_t* a = to_u ? a_stack + (size_t)t.slot * R * hidden : nullptr;
  float* uo = to_u ? u_out + (size_t)tile * 16 * R : nullptr;
  float* sm = sums + (size_t)tile * (hidden / NORM_STRIP) * 16;
#define STRIP(DELTA, TO_U)                                                                                          \
  norm_strip<ADD, DELTA, TO_U, SUM>(t, out, x, residual, weight, eps, hidden, ui, parts, tiles, b, a, uo, tiles_out, sm, \
                                    smem, wave, li, lg)
  if (ADD && delta && to_u) STRIP(ADD, true);
  else if (ADD && delta) STRIP(ADD, false);
  else if (to_u) STRIP(false, true);
  else STRIP(false, false);
#undef STRIP
}

// G groups of 8 columns of a product in fp32 parts, in order; N parts are asked for at a
// time.
template <int G, int N, bool FIRST>
LIG_DEVICE void add_some(f32x8 (&v)[G], const float* __restrict__ p, const size_t stride, const int (&at)[G]) {
  f32x8 r[N][G];
#pragma unroll
  for (int j = 0; j < N; ++j)
#pragma unroll
    for (int i = 0; i < G; ++i) r[j][i] = *reinterpret_cast<const f32x8*>(p + j * stride + at[i]);
#pragma unroll
  for (int j = 0; j < N; ++j)
#pragma unroll
    for (int i = 0; i < G; ++i) v[i] = FIRST && j == 0 ? r[0][i] : v[i] + r[j][i];
}
// As many loads as there are parts: four at a time whatever their number, the last one
// again, took 22.5 and 13.6 us in the rotation of 786 rows in one part and 384 in two, 16.7
// and 11.5 now, and 22.4 and 13.7 in the norms (two and four, two and eight), 19.3 and 12.3.
template <int G>
LIG_DEVICE void add_parts(f32x8 (&v)[G], const float* __restrict__ p, const int parts, const size_t stride, const int (&at)[G]) {
  if (parts == 1) return add_some<G, 1, true>(v, p, stride, at);
  if (parts == 2) return add_some<G, 2, true>(v, p, stride, at);
  if (parts == 3) return add_some<G, 3, true>(v, p, stride, at);
  add_some<G, 4, true>(v, p, stride, at);
  int k = 4;
  for (; k + 4 <= parts; k += 4) add_some<G, 4, false>(v, p + k * stride, stride, at);
  for (; k < parts; ++k) add_some<G, 1, false>(v, p + k * stride, stride, at);
}

// The same strips in one launch, for readers that can wait for the norm's factor:
// out = residual' * weight, u_out = A out, and the sums of squares of each strip.
// A product's rows carry the factor through, so it is left to the kernel that reads
// the product (factor_of).  x may come as the parts that projection.hip cuts K into.
// As sum of the parts, sums of squares and norm these were three launches.  With both
// adapter products, 4096 columns, in a step: 48 rows, 4 parts 16.6 -> 7.1 us; 202 rows,
// 4 and 8 parts 17.4 -> 9.3; 384 rows 22.7 -> 13.4.  With strips of 512 columns 8.9, 13.5
// and 14.2.
template <bool ADD, bool DELTA, bool TO_U, bool PARTS>
LIG_DEVICE void open_strip(const Tile& t, uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
                           const float* __restrict__ xp, const int xparts, const size_t xstride,
                           uint16_t* __restrict__ residual, const uint16_t* __restrict__ weight, const int hidden,
                           const float* u_in, const int parts, const int tiles, const uint16_t* __restrict__ b,
                           const uint16_t* __restrict__ a, float* u_out, const int tiles_out, float* sums, float* smem,
                           int wave, int li, int lg) {
  constexpr int NB = NORM_STRIP / 128;
  const int c_first = place_of().strip * NORM_STRIP + wave * 32;
  const size_t base = (size_t)t.row * hidden + lg * 8;
  u16x8 xr[NB], rr[NB], wr[NB], ar[NB];
  BOperand br[NB];
  f32x8 v[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int c0 = c_first + i * 128;
    if constexpr (!PARTS) xr[i] = load8(x + base + c0);
    if constexpr (ADD) rr[i] = load8(residual + base + c0);
    if constexpr (DELTA) br[i] = load_b(b, c0, li, lg);
    wr[i] = load8(weight + c0 + lg * 8);
    if constexpr (TO_U) ar[i] = load_a(a, hidden, c0, li, lg);
  }
  if constexpr (PARTS) {
    int at[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) at[i] = c_first + i * 128;
    add_parts(v, xp + base, xparts, xstride, at);
  }
  bf16x8_t u = {};
  if constexpr (DELTA) u = u_of(u_in, parts, tiles, smem, li, lg, t.valid);
  float ss = 0.f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  u16x8 h[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if constexpr (!PARTS) v[i] = bf16x8_to_f32x8(xr[i]);
    if constexpr (ADD) v[i] += bf16x8_to_f32x8(rr[i]);
    if constexpr (DELTA) v[i] += expand(br[i], u);
    const f32x8 w = bf16x8_to_f32x8(wr[i]);
    f32x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      ss += v[i][j] * v[i][j];
      o[j] = v[i][j] * w[j];
    }
    h[i] = f32x8_to_bf16x8(o);
    if constexpr (TO_U) acc = shrink(ar[i], h[i], acc);
  }
  if (t.valid) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int c0 = c_first + i * 128;
      *reinterpret_cast<u16x8*>(out + base + c0) = h[i];
      if constexpr (ADD) *reinterpret_cast<u16x8*>(residual + base + c0) = f32x8_to_bf16x8(v[i]);
    }
  }
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  if (lg == 0) smem[wave * 16 + li] = ss;
  __syncthreads();
  if (threadIdx.x < 16)
    sums[place_of().strip * 16 + threadIdx.x] =
        smem[threadIdx.x] + smem[16 + threadIdx.x] + smem[32 + threadIdx.x] + smem[48 + threadIdx.x];
  if constexpr (TO_U) {
    __syncthreads();
    store_u<4>(u_out + (size_t)place_of().strip * tiles_out * 16 * R, acc, reinterpret_cast<float(*)[16][R]>(smem), wave, li, lg);
  }
}

template <bool ADD, bool PARTS>
__global__ __launch_bounds__(256) void lora_norm_open_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x, const float* __restrict__ xp, const int xparts,
    const size_t xstride, uint16_t* __restrict__ residual, const uint16_t* __restrict__ weight, const int hidden,
    const int* __restrict__ toks, const int* __restrict__ len, const int* __restrict__ slot, const float* u_in,
    const int parts, const int tiles, const uint16_t* __restrict__ b_stack, const uint16_t* __restrict__ a_stack,
    float* u_out, const int tiles_out, float* sums, const int rows) {
  __shared__ __align__(16) float smem[4 * 16 * R];
  const int tile = place_of().tile;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Tile t = tile_of(toks, len, slot, tile, li, rows);
  if (t.n == 0) return;
  const bool delta = u_in != nullptr && t.slot >= 0, to_u = t.slot >= 0;
  const float* ui = delta ? u_in + (size_t)tile * 16 * R : nullptr;
  const uint16_t* b = delta ? b_stack + (size_t)t.slot * hidden * R : nullptr;
  const uint16_t* a = to_u ? a_stack + (size_t)t.slot * R * hidden : nullptr;
  float* uo = to_u ? u_out + (size_t)tile * 16 * R : nullptr;
  float* sm = sums + (size_t)tile * (hidden / NORM_STRIP) * 16;
#define STRIP(DELTA, TO_U)                                                                                          \
  open_strip<ADD, DELTA, TO_U, PARTS>(t, out, x, xp, xparts, xstride, residual, weight, hidden, ui, parts, tiles, b, a, \
                                      uo, tiles_out, sm, smem, wave, li, lg)
  if (ADD && delta) STRIP(ADD, true);
  else if (to_u) STRIP(false, true);
  else STRIP(false, false);
#undef STRIP
}

// The factor that lora_norm_open left out, of token li of a tile; without sums none was.
struct Factor {
  const float* sums;  // [tiles][width / strip][16]
  int width;
  float eps;
};
LIG_DEVICE float factor_of(const Factor& f, int tile, int li) {
  if (f.sums == nullptr) return 1.f;
  const int strips = f.width / NORM_STRIP;
  const float* s = f.sums + (size_t)tile * strips * 16 + li;
  float total = 0.f;
#pragma unroll 8
  for (int k = 0; k < strips; ++k) total += s[k * 16];
  return rsqrtf(total / f.width + f.eps);
}

// g / (1 + e^-g) of n = g / 4, the quotient as a division rounds it: corrected once by
// its remainder (Markstein 1990), which v_rcp_f32's 1 ulp allows, both sides over 4 so
// that no reciprocal is subnormal; v_div_fixup_f32 sees to infinities and NaN.  The
// compiler's division takes twice the instructions.
LIG_DEVICE float silu_of_quarter(float n) {
  const float d = __builtin_fmaf(__builtin_amdgcn_exp2f(n * (-4.f * LOG2E)), 0.25f, 0.25f);
  const float r = __builtin_amdgcn_rcpf(d), q = n * r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, n), r, q), d, n);
}

// load_b's two operands by one load: lanes lg < 2 bring the first, the others the second.
LIG_DEVICE u16x8 load_b_once(const uint16_t* b, int c0, int li, int lg) {
  return *reinterpret_cast<const u16x8*>(b + (size_t)(c0 + ((li >> 2) << 3) + (li & 3) + (lg >> 1) * 4) * R + (lg & 1) * 8);
}
LIG_DEVICE BOperand both_halves(u16x8 x) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 v = __builtin_bit_cast(u32x4, x);
  u32x4 lo, hi;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto s = __builtin_amdgcn_permlane32_swap(v[i], v[i], false, false);
    lo[i] = s[0];
    hi[i] = s[1];
  }
  return {__builtin_bit_cast(u16x8, lo), __builtin_bit_cast(u16x8, hi)};
}

// out = silu(gate + B u) * (up + B u), u_out[strip] = A_down out.  Workgroups of
// a tile take strips of 1024 of the d columns.
// In the products' layout 16 lanes side by side hold 16 rows, and a load costs an access
// of the L1 per lane instead of one per four: 331 accesses for 32 columns of a tile, which
// took 62 % of the time at 4000 rows.  So rows come as they lie, 256 bytes of 4 rows to a
// load, straight into LDS, and leave through it; 16-byte piece c of row r at c ^ r, for
// reads and writes without conflicts.  A wave uses its own part of LDS only.
// A wave's columns lie side by side, so that A's sums, in fp32 as ever, add up in another order
// than with every eighth group of 32: u differs by 1.3e-7 of its size, its error against 64 bits (14336 columns)
// is 9.1e-8 at 33 rows and 1.1e-7 at 384, where it was 9.5e-8 and 1.1e-7.
constexpr int SILU_STRIP = 1024;
constexpr int SILU_BATCH = 128;  // columns of a wave at a time
constexpr int SILU_ROOM = 3 * 16 * SILU_BATCH;  // gate, up and A's rows of a batch, 16-bit units

// A batch of columns on its way: rows and A's into LDS, B's operands.
struct SiluBatch {
  static constexpr int NB = SILU_BATCH / 32;
  u16x8 gate[NB], up[NB];
  int row[4];  // of tokens 4 j + lg, whose pieces this lane moves

  LIG_DEVICE void issue(const uint16_t* x, const int d, const int c0, const uint16_t* b, const uint16_t* a, const uint16_t* room,
                        int li, int lg) {
    const uint32_t lds = lds_address(room);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = min(c0 + (li ^ (4 * j + lg)) * 8, d - 8);  // pieces past the end: the last one again, unused
      load_to_lds(x + (size_t)row[j] * 2 * d + c, lds + j * 1024);
      load_to_lds(x + (size_t)row[j] * 2 * d + d + c, lds + (4 + j) * 1024);
      load_to_lds(a + (size_t)(4 * j + lg) * d + c, lds + (8 + j) * 1024);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int c = min(c0 + i * 32, d - 32);
      gate[i] = load_b_once(b, c, li, lg);
      up[i] = load_b_once(b, d + c, li, lg);
    }
  }

  // acc + A out of the batch
  LIG_DEVICE f32x4_t finish(const Tile& t, uint16_t* out, const int d, const int c0, const bf16x8_t u, const float factor,
                            uint16_t* room, f32x4_t acc, int li, int lg) const {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (c0 + i * 32 >= d) break;
      uint16_t* at = room + li * SILU_BATCH + ((i * 4 + lg) ^ li) * 8;
      f32x8 gv = bf16x8_to_f32x8(load8(at)) + expand(both_halves(gate[i]), u), r;
      f32x8 uv = bf16x8_to_f32x8(load8(at + 16 * SILU_BATCH)) + expand(both_halves(up[i]), u);
      gv *= 0.25f * factor;
      uv *= factor;
#pragma unroll
      for (int e = 0; e < 8; ++e) r[e] = silu_of_quarter(gv[e]) * uv[e];
      const u16x8 rb = f32x8_to_bf16x8(r);
      acc = shrink(load8(at + 32 * SILU_BATCH), rb, acc);
      *reinterpret_cast<u16x8*>(at) = rb;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = c0 + (li ^ (4 * j + lg)) * 8;
      const u16x8 rb = load8(room + (j * 64 + lg * 16 + li) * 8);
      if (4 * j + lg < t.n && c < d) *reinterpret_cast<u16x8*>(out + (size_t)row[j] * d + c) = rb;
    }
    return acc;
  }
};

// The columns c_first .. c_end of rows without an adapter, as they lie.
LIG_DEVICE void silu_plain(const Tile& t, uint16_t* out, const uint16_t* x, const int d, const int c_first, const int c_end,
                           const float factor, const int (&row)[4], int li, int lg) {
  float own[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) own[j] = __shfl(factor, 4 * j + lg, 64);
  for (int c0 = c_first; c0 < min(c_end, d); c0 += SILU_BATCH) {
    const int c = min(c0 + li * 8, d - 8);  // pieces past the end: the last one again, unused
    u16x8 gr[4], ur[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      gr[j] = load8(x + (size_t)row[j] * 2 * d + c);
      ur[j] = load8(x + (size_t)row[j] * 2 * d + d + c);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x8 gv = bf16x8_to_f32x8(gr[j]), uv = bf16x8_to_f32x8(ur[j]), r;
      gv *= 0.25f * own[j];
      uv *= own[j];
#pragma unroll
      for (int e = 0; e < 8; ++e) r[e] = silu_of_quarter(gv[e]) * uv[e];
      if (4 * j + lg < t.n && c0 + li * 8 < d) *reinterpret_cast<u16x8*>(out + (size_t)row[j] * d + c) = f32x8_to_bf16x8(r);
    }
  }
}

// 8 waves take a strip in one pass each, 4 in two: faster where the workgroups find a
// CU each, slower from there on.  14 strips, weights of 8 or 32 adapters in no cache (us with
// 8 and 4 waves): 96 rows 8.5, 10.2; 256 (16 tiles) 10.3, 12.2; 288 (24) 15.2, 13.6; 384
// of 32 adapters 20.8, 18.7; 740 26.3, 21.4; 1851 56.1, 43.3.  As rows came in the products'
// layout (and their fewer waves per CU notwithstanding): 384 rows of 32 adapters 20.4 -> 18.7,
// 786 34.4 -> 28.8, 1500 of 5 48.0 -> 37.3, 4040 of 32 115.8 -> 91.5 (4.3 TB/s with the
// adapters' weights once); without adapters 384 11.3 -> 10.1, 1000 18.5 -> 16.6, but 256, whose
// 224 workgroups of 8 waves just find a CU each, 7.0 -> 7.4.
// Without LISTED no row has an adapter.
template <int W, bool LISTED>
__global__ __launch_bounds__(64 * W) void lora_silu_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x, const int d, const int* __restrict__ toks,
    const int* __restrict__ len, const int* __restrict__ slot,
    const float* __restrict__ u_in, const int parts, const int tiles, const uint16_t* __restrict__ b_stack,
    const uint16_t* __restrict__ a_stack, float* __restrict__ u_out, const int tiles_out, const Factor norm,
    const int rows) {
  const int tile = place_of().tile, strip = place_of().strip;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Tile t = tile_of(LISTED ? toks : nullptr, len, slot, tile, li, rows);
  if (t.n == 0) return;
  const int c_first = strip * SILU_STRIP + wave * (SILU_STRIP / W), c_end = c_first + SILU_STRIP / W;
  SiluBatch batch;
#pragma unroll
  for (int j = 0; j < 4; ++j) batch.row[j] = LISTED ? __shfl(t.row, 4 * j + lg, 64) : tile * 16 + min(4 * j + lg, t.n - 1);
  if (!LISTED || t.slot < 0) {
    silu_plain(t, out, x, d, c_first, c_end, factor_of(norm, tile, li), batch.row, li, lg);
    return;
  }
  if constexpr (LISTED) {
    __shared__ __align__(16) float red[W][16][R];
    __shared__ __align__(16) uint16_t rooms[W * SILU_ROOM];
    uint16_t* room = rooms + wave * SILU_ROOM;
    const uint16_t* b = b_stack + (size_t)t.slot * 2 * d * R;
    const uint16_t* a = a_stack + (size_t)t.slot * R * d;
    if (c_first < d) batch.issue(x, d, c_first, b, a, room, li, lg);
    const float factor = factor_of(norm, tile, li);
    const bf16x8_t u = u_of(u_in + (size_t)tile * 16 * R, parts, tiles, &red[0][0][0], li, lg, t.valid);
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int c0 = c_first; c0 < min(c_end, d); c0 += SILU_BATCH) {
      if (c0 > c_first) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the batch before has been read
        batch.issue(x, d, c0, b, a, room, li, lg);
      }
      acc = batch.finish(t, out, d, c0, u, factor, room, acc, li, lg);
    }
    store_u<W>(u_out + ((size_t)strip * tiles_out + tile) * 16 * R, acc, red, wave, li, lg);
  }
}

// u_out = A x, a part per strip of 512 columns
constexpr int SHRINK_STRIP = 512;

__global__ __launch_bounds__(256) void lora_shrink_kernel(
    const uint16_t* __restrict__ x, const int width, const int* __restrict__ toks, const int* __restrict__ len,
    const int* __restrict__ slot, const uint16_t* __restrict__ a_stack, float* __restrict__ u_out,
    const int tiles_out) {
  constexpr int NB = SHRINK_STRIP / 128;
  __shared__ __align__(16) float red[4][16][R];
  const int tile = place_of().tile;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Tile t = tile_of(toks, len, slot, tile, li);
  if (t.n == 0 || t.slot < 0) return;
  const uint16_t* a = a_stack + (size_t)t.slot * R * width;
  const uint16_t* row = x + (size_t)t.row * width + lg * 8;
  const int c_first = place_of().strip * SHRINK_STRIP + wave * 32;
  u16x8 xr[NB], ar[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int c0 = min(c_first + i * 128, width - 32);  // groups past the end: the last one again, unused
    xr[i] = load8(row + c0);
    ar[i] = load_a(a, width, c0, li, lg);
  }
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NB; ++i)
    if (c_first + i * 128 < width) acc = shrink(ar[i], xr[i], acc);
  store_u<4>(u_out + ((size_t)place_of().strip * tiles_out + tile) * 16 * R, acc, red, wave, li, lg);
}

// qkv_rope.hip's pass with B u added to the projection on the way in.  PARTS: the
// projection as fp32 parts of K.
// Waves take 4 heads, of parts one: 2 to 8 times the bytes (48 rows in 4 parts 8.3 us,
// 12.7 with 4 heads; sum and rotation as two launches 11.1).
template <bool PARTS>
__global__ __launch_bounds__(256) void lora_qkv_rope_cache_kernel(
    uint16_t* __restrict__ q_out, const uint16_t* __restrict__ qkv, const float* __restrict__ qkv_parts, const int nparts,
    const size_t part_stride, const Factor norm, const int64_t* __restrict__ positions,
    const float* __restrict__ cos_sin, uint16_t* __restrict__ k_cache, uint16_t* __restrict__ v_cache,
    const int64_t* __restrict__ slot_mapping, const int num_q_heads, const int num_kv_heads, const int head_dim,
    const int block_size, const int block_shift, const int* __restrict__ toks, const int* __restrict__ len,
    const int* __restrict__ slot, const float* __restrict__ u_in, const int u_parts, const int tiles,
    const uint16_t* __restrict__ b_stack, const int rows) {
  constexpr int QR_HEADS = PARTS ? 1 : 4;
  __shared__ __align__(16) float smem[16 * R];
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int parts = head_dim / 64;  // of 32 rotation pairs
  const int tile = place_of().tile;
  const int wid = place_of().strip * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int heads = num_q_heads + 2 * num_kv_heads;
  const int h0 = (wid / parts) * QR_HEADS;
  const Tile t = tile_of(toks, len, slot, tile, li, rows);
  if (t.n == 0) return;
  bf16x8_t u = {};
  if (t.slot >= 0) u = u_of(u_in + (size_t)tile * 16 * R, u_parts, tiles, smem, li, lg, t.valid);
  if (h0 >= heads) return;  // whole waves: no lane may miss the matrix instructions
  const int half = head_dim / 2;
  const int p0 = (wid % parts) * 32, c = p0 + lg * 8;

  const float* cs = cos_sin + positions[t.row] * head_dim + c;
  float co[8], si[8];
#pragma unroll
  for (int i = 0; i < 8; i += 4) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(cs + i);
    const f32x4 b = *reinterpret_cast<const f32x4*>(cs + half + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      co[i + j] = a[j];
      si[i + j] = b[j];
    }
  }
  const int64_t at = slot_mapping[t.row];
  // a division of 64 bits is some hundred instructions
  const size_t blk = at < 0 ? 0 : block_shift >= 0 ? at >> block_shift : at / block_size;
  const size_t off = at < 0 ? 0 : at - (int64_t)blk * block_size;
  const size_t src = ((size_t)t.row * heads + h0) * head_dim + c;
  f32x8 v[QR_HEADS][2];
  if constexpr (PARTS) {
    f32x8 y[2];
    const int at[2] = {0, half};
    add_parts(y, qkv_parts + src, nparts, part_stride, at);
    v[0][0] = y[0];
    v[0][1] = y[1];
  } else {
    u16x8 x[QR_HEADS][2];
#pragma unroll
    for (int i = 0; i < QR_HEADS; ++i) {
      const int h = min(h0 + i, heads - 1) - h0;
      x[i][0] = load8(qkv + src + h * head_dim);
      x[i][1] = load8(qkv + src + h * head_dim + half);
    }
#pragma unroll
    for (int i = 0; i < QR_HEADS; ++i) {
      v[i][0] = bf16x8_to_f32x8(x[i][0]);
      v[i][1] = bf16x8_to_f32x8(x[i][1]);
    }
  }
  if (t.slot >= 0) {
    const uint16_t* b = b_stack + (size_t)t.slot * heads * head_dim * R;
    BOperand br[QR_HEADS][2];
#pragma unroll
    for (int i = 0; i < QR_HEADS; ++i) {
      const int h = min(h0 + i, heads - 1);
      br[i][0] = load_b(b, h * head_dim + p0, li, lg);
      br[i][1] = load_b(b, h * head_dim + half + p0, li, lg);
    }
#pragma unroll
    for (int i = 0; i < QR_HEADS; ++i) {
      v[i][0] += expand(br[i][0], u);
      v[i][1] += expand(br[i][1], u);
    }
  }
  const float factor = factor_of(norm, tile, li);
#pragma unroll
  for (int i = 0; i < QR_HEADS; ++i) {
    v[i][0] *= factor;
    v[i][1] *= factor;
  }
#pragma unroll
  for (int i = 0; i < QR_HEADS; ++i) {
    const int h = h0 + i;
    if (h >= heads) break;
    const bool turned = h < num_q_heads + num_kv_heads;
    if (turned) {
      f32x8 o1, o2;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        o1[j] = v[i][0][j] * co[j] - v[i][1][j] * si[j];
        o2[j] = v[i][1][j] * co[j] + v[i][0][j] * si[j];
      }
      v[i][0] = o1;
      v[i][1] = o2;
    }
    uint16_t* dst;
    if (h < num_q_heads) {
      dst = q_out + ((size_t)t.row * num_q_heads + h) * head_dim;
    } else {
      const int g = h - num_q_heads - (turned ? 0 : num_kv_heads);
      dst = (turned ? k_cache : v_cache) + ((blk * num_kv_heads + g) * block_size + off) * head_dim;
    }
    if (t.valid && (h < num_q_heads || at >= 0)) {
      *reinterpret_cast<u16x8*>(dst + c) = f32x8_to_bf16x8(v[i][0]);
      *reinterpret_cast<u16x8*>(dst + half + c) = f32x8_to_bf16x8(v[i][1]);
    }
  }
}

}  // namespace

extern "C" {

// Returns 1 for a row width that is not served.
int lig_lora_rms_norm_launch(uint16_t* out, const uint16_t* x, uint16_t* residual, const uint16_t* weight, float eps,
                             int hidden, const int* toks, const int* len, const int* slot, int ntiles,
                             const float* u_in, int parts, int tiles, const uint16_t* b_stack,
                             const uint16_t* a_stack, float* u_out, hipStream_t stream) {
#define LAUNCH_N(NG)                                                                                                 \
  case NG * 256:                                                                                                     \
    if (residual)                                                                                                    \
      hipLaunchKernelGGL((lora_rms_norm_kernel<true, NG>), dim3(ntiles), dim3(512), 0, stream, out, x, residual,     \
                         weight, eps, toks, len, slot, u_in, parts, tiles, b_stack, a_stack, u_out);            \
    else                                                                                                             \
      hipLaunchKernelGGL((lora_rms_norm_kernel<false, NG>), dim3(ntiles), dim3(512), 0, stream, out, x, residual,    \
                         weight, eps, toks, len, slot, u_in, parts, tiles, b_stack, a_stack, u_out);            \
    return 0
  switch (hidden) {
    LAUNCH_N(1);
    LAUNCH_N(2);
    LAUNCH_N(4);
    LAUNCH_N(8);
    LAUNCH_N(12);
    LAUNCH_N(16);
  }
#undef LAUNCH_N
  return 1;
}

int lig_lora_silu_strip() { return SILU_STRIP; }
int lig_lora_norm_strip() { return NORM_STRIP; }

// sums: fp32 [tiles, hidden / strip, 16]; hidden a multiple of the strip
void lig_lora_rms_norm_strips_launch(uint16_t* out, const uint16_t* x, uint16_t* residual, const uint16_t* weight,
                                     float eps, int hidden, const int* toks, const int* len, const int* slot, int ntiles,
                                     const float* u_in, int parts, int tiles, const uint16_t* b_stack,
                                     const uint16_t* a_stack, float* u_out, int tiles_out, float* sums,
                                     hipStream_t stream) {
#define LAUNCH_S(ADD, SUM)                                                                                      \
  hipLaunchKernelGGL((lora_norm_strip_kernel<ADD, SUM>), dim3(ntiles, hidden / NORM_STRIP), dim3(256), 0, stream, out, \
                     x, residual, weight, eps, hidden, toks, len, slot, u_in, parts, tiles, b_stack, a_stack, u_out,  \
                     tiles_out, sums)
  if (residual) {
    LAUNCH_S(true, true);
    LAUNCH_S(true, false);
  } else {
    LAUNCH_S(false, true);
    LAUNCH_S(false, false);
  }
#undef LAUNCH_S
}

// sums as above; x bf16, or xparts fp32 parts of rows * hidden each in xp.  Without
// a residual x itself, in bf16, is what is normed
void lig_lora_norm_open_launch(uint16_t* out, const uint16_t* x, const float* xp, int xparts, long xstride,
                               uint16_t* residual, const uint16_t* weight, int hidden, const int* toks, const int* len,
                               const int* slot, int ntiles, const float* u_in, int parts, int tiles,
                               const uint16_t* b_stack, const uint16_t* a_stack, float* u_out, int tiles_out,
                               float* sums, int rows, hipStream_t stream) {
#define LAUNCH_O(ADD, PARTS)                                                                                        \
  hipLaunchKernelGGL((lora_norm_open_kernel<ADD, PARTS>), dim3(ntiles, hidden / NORM_STRIP), dim3(256), 0, stream, out, \
                     x, xp, xparts, (size_t)xstride, residual, weight, hidden, toks, len, slot, u_in, parts, tiles,  \
                     b_stack, a_stack, u_out, tiles_out, sums, rows)
  if (!residual) LAUNCH_O(false, false);
  else if (xp) LAUNCH_O(true, true);
  else LAUNCH_O(true, false);
#undef LAUNCH_O
}

void lig_lora_silu_launch(uint16_t* out, const uint16_t* x, int d, const int* toks, const int* len,
                          const int* slot, int ntiles, const float* u_in, int parts, int tiles,
                          const uint16_t* b_stack, const uint16_t* a_stack, float* u_out, int tiles_out,
                          const float* sums, int width, float eps, int rows, hipStream_t stream) {
#define LAUNCH_A1(W, LISTED)                                                                                         \
  hipLaunchKernelGGL((lora_silu_kernel<W, LISTED>), dim3(ntiles, (d + SILU_STRIP - 1) / SILU_STRIP), dim3(64 * W), 0, stream, \
                     out, x, d, toks, len, slot, u_in, parts, tiles, b_stack, a_stack, u_out, tiles_out,             \
                     Factor{sums, width, eps}, rows)
#define LAUNCH_A(W)               \
  do {                            \
    if (toks) LAUNCH_A1(W, true); \
    else LAUNCH_A1(W, false);     \
  } while (0)
  // A decode graph's list has room for one tile per adapter more than full ones, and of
  // those few are in use where adapters have about as many requests each
  const int likely = (ntiles + 3 * ((rows + 15) / 16)) / 4;
  if (likely * ((d + SILU_STRIP - 1) / SILU_STRIP) <= 256) LAUNCH_A(8);
  else LAUNCH_A(4);
#undef LAUNCH_A
#undef LAUNCH_A1
}

int lig_lora_shrink_strip() { return SHRINK_STRIP; }

void lig_lora_shrink_launch(const uint16_t* x, int width, const int* toks, const int* len, const int* slot, int ntiles,
                            const uint16_t* a_stack, float* u_out, int tiles_out, hipStream_t stream) {
  hipLaunchKernelGGL(lora_shrink_kernel, dim3(ntiles, (width + SHRINK_STRIP - 1) / SHRINK_STRIP), dim3(256), 0, stream, x,
                     width, toks, len, slot, a_stack, u_out, tiles_out);
}

void lig_lora_qkv_rope_cache_launch(uint16_t* q_out, const uint16_t* qkv, const float* qkv_parts, int nparts,
                                    long part_stride, const float* sums, int width, float eps, const int64_t* positions,
                                    const float* cos_sin, uint16_t* k_cache, uint16_t* v_cache,
                                    const int64_t* slot_mapping, int num_q_heads, int num_kv_heads, int head_dim,
                                    int block_size, const int* toks, const int* len, const int* slot,
                                    int ntiles, const float* u_in, int u_parts, int tiles, const uint16_t* b_stack,
                                    int rows, hipStream_t stream) {
  const int heads = num_q_heads + 2 * num_kv_heads;
  const int waves = (head_dim / 64) * (qkv_parts ? heads : (heads + 3) / 4);
#define LAUNCH_R(PARTS)                                                                                             \
  hipLaunchKernelGGL((lora_qkv_rope_cache_kernel<PARTS>), dim3(ntiles, (waves + 3) / 4), dim3(256), 0, stream, q_out, qkv, \
                     qkv_parts, nparts, (size_t)part_stride, Factor{sums, width, eps}, positions, cos_sin, k_cache,   \
                     v_cache, slot_mapping, num_q_heads, num_kv_heads, head_dim, block_size, shift_of(block_size), toks, len, slot, u_in, \
                     u_parts, tiles, b_stack, rows)
  if (qkv_parts) LAUNCH_R(true);
  else LAUNCH_R(false);
#undef LAUNCH_R
}

}  // extern "C"
