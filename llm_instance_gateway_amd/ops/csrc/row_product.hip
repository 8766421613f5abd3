// Projections of a single token, gfx950, bf16: y = W h for one row h, with the
// norm before it and the activation behind it in the same kernel.
//
// Bound by streaming W once.  A wave takes two rows of W and keeps eight to
// sixteen 16-byte loads a lane on their way, the first of them issued before h
// is ready; h is formed by every workgroup for itself in LDS (24 KB from the
// L2 against 64 KB and more of W) and shared by its waves.
//   norm: residual' = x + residual, h = rms_norm(residual') * weight, as
//         fused_add_rms_norm (the norm over the unrounded sum); the first
//         workgroup writes residual' to a place of its own, since the others
//         may still read the old one.
//   silu: the two rows are a gate and its up row, y = silu(gate) * up of both
//         rounded to bf16, as silu_and_mul after the projection.
// Widths of Llama-3-8B, weights not in any cache, against the library's product
// with the norm and activation as kernels of their own: norm + qkv 12.7 us (18.5),
// o 8.4 (13.0), norm + gate_up + silu 40.9 (69.2, now 5.7 TB/s), down 21.7 (26.5).
// Loads of a large W are non-temporal (`streams`): without that gate_up 43.9, down
// 24.7, qkv 13.5, o 8.8, a gate_up of 24576 x 8192 63.9 instead of 69.6.  Starting the
// waves at different columns changed nothing.
//   rotation: the two rows of a wave are a rotation pair of a query or key head (of a
//         value head just half a head apart), and lane 0 rotates them and writes them
//         where they belong: q, or the paged caches.  As a launch of its own 5.1 us a layer.
//   parts: h is the attention's result, which where its walk was cut is still in parts;
//         every workgroup merges them for itself, as flash_decode_merge_kernel does, which
//         has nothing to do for walks under 1024 keys.
// A step of one token on 381 cached, 8 layers of 8B widths: 991 us, 947 with both.
#include "flash_decode.h"

namespace {

// Where a lone token's query, key and value heads go.
struct Heads {
  const int64_t* position;
  const float* cos_sin;      // [P, D]: D/2 cosines | D/2 sines
  const int64_t* slot;       // negative: not cached
  uint16_t *k_cache, *v_cache;  // [B, num_kv, block_size, D]
  int num_q, num_kv, D, block_size;
};

// An attention's result in parts: scratch [heads, nsplits, D + 2] of a walk of that many keys.
struct Parts {
  const float* scratch;  // null: none
  const int* context_len;
  int nsplits, D;
};

// 8 entries of head h from d on
LIG_DEVICE u16x8 merged(const Parts& p, int parts, int h, int d) {
  const float* base = p.scratch + (size_t)h * p.nsplits * (p.D + 2);
  float gm = -INFINITY, gl = 0.f;
  for (int z = 0; z < parts; ++z) gm = fmaxf(gm, base[(size_t)z * (p.D + 2) + p.D]);
  f32x8 o = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int z = 0; z < parts; ++z) {
    const float* sp = base + (size_t)z * (p.D + 2);
    const float f = sp[p.D] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sp[p.D] - gm);
    gl += sp[p.D + 1] * f;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] += sp[d + i] * f;
  }
  const float f = gl > 0.f ? 1.f / gl : (gl == 0.f ? 0.f : gl);
  return f32x8_to_bf16x8(o * f);
}

constexpr int NORM_MAX = 8192;  // columns of a row with a norm
constexpr int PLAIN_MAX = 16384;
constexpr int U = 4;  // loads of a row per batch, 512 columns each

template <int NTHR, bool NORM, bool SILU, bool STREAM, bool ROTATE>
__global__ __launch_bounds__(NTHR) void row_product_kernel(
    uint16_t* __restrict__ y, const uint16_t* __restrict__ w, const int N, const int K, const uint16_t* __restrict__ x,
    const uint16_t* __restrict__ residual, uint16_t* __restrict__ residual_out, const uint16_t* __restrict__ weight,
    const float eps, const Heads heads, const Parts parts) {
  constexpr int NW = NTHR / WAVE_SIZE, MAXC = NORM_MAX / 8 / NTHR;
  extern __shared__ __align__(16) uint16_t h[];  // [K]
  __shared__ float part[NW];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // outputs, of which a wave makes two (one from two rows with SILU)
  const int outs = SILU ? N / 2 : N;
  const int n0 = (blockIdx.x * NW + wave) * (SILU ? 1 : 2);
  const int half = ROTATE ? heads.D / 2 : 1;
  const int head = ROTATE ? n0 / 2 / half : 0, entry = ROTATE ? n0 / 2 % half : 0;
  const int ra = ROTATE ? min(head * heads.D + entry, outs - 1 - half) : min(n0, outs - 1);
  const int rb = SILU ? ra + outs : ROTATE ? ra + half : min(n0 + 1, outs - 1);
  float co = 0.f, si = 0.f;
  int64_t slot = -1;
  if (ROTATE) {
    const float* cs = heads.cos_sin + *heads.position * heads.D + entry;
    co = cs[0];
    si = cs[half];
    slot = *heads.slot;
  }
  const uint16_t* wr[2] = {w + (size_t)ra * K + lane * 8, w + (size_t)rb * K + lane * 8};
  const int batches = (K / 512 + U - 1) / U;

  u16x8 buf[2][U][2];
  auto load = [&](int b, int batch) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int c = min((batch * U + i) * 512, K - 512);  // past the end: the last columns again, unused
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const u16x8* src = reinterpret_cast<const u16x8*>(wr[r] + c);
        buf[b][i][r] = STREAM ? __builtin_nontemporal_load(src) : *src;
      }
    }
  };
  load(0, 0);
  load(1, 1);

  // ---- h ------------------------------------------------------------------------
  const int chunks = K / 8;
  if (NORM) {
    f32x8 v[MAXC];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < MAXC; ++j) {
      const int c = tid + j * NTHR;
      if (j * NTHR >= chunks) break;
      if (c < chunks) {
        v[j] = bf16x8_to_f32x8(*reinterpret_cast<const u16x8*>(x + c * 8));
        if (residual) {
          const f32x8 r = bf16x8_to_f32x8(*reinterpret_cast<const u16x8*>(residual + c * 8));
#pragma unroll
          for (int i = 0; i < 8; ++i) v[j][i] += r[i];
          if (blockIdx.x == 0) *reinterpret_cast<u16x8*>(residual_out + c * 8) = f32x8_to_bf16x8(v[j]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += v[j][i] * v[j][i];
      }
    }
    ss = wave_reduce_sum(ss);
    if (lane == 0) part[wave] = ss;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) total += part[i];
    const float inv = rsqrtf(total / K + eps);
#pragma unroll
    for (int j = 0; j < MAXC; ++j) {
      const int c = tid + j * NTHR;
      if (j * NTHR >= chunks) break;
      if (c < chunks) {
        const f32x8 g = bf16x8_to_f32x8(*reinterpret_cast<const u16x8*>(weight + c * 8));
        f32x8 o;
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = v[j][i] * inv * g[i];
        *reinterpret_cast<u16x8*>(h + c * 8) = f32x8_to_bf16x8(o);
      }
    }
  } else {
    int cut = 1;
    if (parts.scratch) {
      const int pos = *parts.context_len - 1;
      cut = flash_decode::parts_of(pos < 0 ? 0 : pos / flash_decode::KT + 1, parts.nsplits);
    }
    for (int c = tid; c < chunks; c += NTHR)
      *reinterpret_cast<u16x8*>(h + c * 8) =
          cut > 1 ? merged(parts, cut, c * 8 / parts.D, c * 8 % parts.D) : *reinterpret_cast<const u16x8*>(x + c * 8);
  }
  __syncthreads();

  // ---- products --------------------------------------------------------------------
  float acc[2] = {0.f, 0.f};
  auto compute = [&](int b, int batch) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int c = (batch * U + i) * 512;
      if (c < K) {
        const f32x8 hv = bf16x8_to_f32x8(*reinterpret_cast<const u16x8*>(h + c + lane * 8));
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const f32x8 wv = bf16x8_to_f32x8(buf[b][i][r]);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[r] = fmaf(wv[e], hv[e], acc[r]);
        }
      }
    }
  };
  for (int batch = 0;; batch += 2) {
    compute(0, batch);
    if (batch + 2 >= batches) {
      compute(1, batch + 1);
      break;
    }
    load(0, batch + 2);
    compute(1, batch + 1);
    load(1, batch + 3);
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) acc[r] = wave_reduce_sum(acc[r]);
  if (lane == 0 && n0 < outs) {
    if (SILU) {
      const float g = bf16_to_f32(f32_to_bf16(acc[0])), u = bf16_to_f32(f32_to_bf16(acc[1]));
      y[n0] = f32_to_bf16(g / (1.0f + __expf(-g)) * u);
    } else if (ROTATE) {
      // the product rounded first, as it is to its reader elsewhere
      float a = bf16_to_f32(f32_to_bf16(acc[0])), b = bf16_to_f32(f32_to_bf16(acc[1]));
      const bool query = head < heads.num_q, turned = head < heads.num_q + heads.num_kv;
      if (turned) {
        const float t = a * co - b * si;
        b = b * co + a * si;
        a = t;
      }
      uint16_t* dst = y + head * heads.D;
      if (!query) {
        const int64_t blk = slot / heads.block_size, off = slot - blk * heads.block_size;
        const int g = head - heads.num_q - (turned ? 0 : heads.num_kv);
        dst = (turned ? heads.k_cache : heads.v_cache) + ((blk * heads.num_kv + g) * heads.block_size + off) * heads.D;
      }
      if (query || slot >= 0) {
        dst[entry] = f32_to_bf16(a);
        dst[entry + half] = f32_to_bf16(b);
      }
    } else {
      y[n0] = f32_to_bf16(acc[0]);
      if (n0 + 1 < outs) y[n0 + 1] = f32_to_bf16(acc[1]);
    }
  }
}

}  // namespace

extern "C" int lig_row_product_max(bool norm) { return norm ? NORM_MAX : PLAIN_MAX; }

namespace {
template <int NTHR, bool NORM, bool SILU, bool ROTATE>
void launch(uint16_t* y, const uint16_t* w, int N, int K, const uint16_t* x, const uint16_t* residual,
            uint16_t* residual_out, const uint16_t* weight, float eps, const Heads& heads, const Parts& parts,
            hipStream_t stream) {
  constexpr int ROWS = NTHR / WAVE_SIZE * 2;
  const dim3 grid((N + ROWS - 1) / ROWS), block(NTHR);
  if (streams(N, K))
    hipLaunchKernelGGL((row_product_kernel<NTHR, NORM, SILU, true, ROTATE>), grid, block, (size_t)K * 2, stream, y, w, N, K, x,
                       residual, residual_out, weight, eps, heads, parts);
  else
    hipLaunchKernelGGL((row_product_kernel<NTHR, NORM, SILU, false, ROTATE>), grid, block, (size_t)K * 2, stream, y, w, N, K, x,
                       residual, residual_out, weight, eps, heads, parts);
}
}  // namespace

// scratch, context_len, nsplits, D: of an x that may be in parts (no norm), else null
extern "C" void lig_row_product_launch(uint16_t* y, const uint16_t* w, int N, int K, const uint16_t* x,
                                       const uint16_t* residual, uint16_t* residual_out, const uint16_t* weight,
                                       float eps, bool silu, const float* scratch, const int* context_len, int nsplits,
                                       int D, hipStream_t stream) {
  // with a norm 8 waves share the h they form.  Measured with cached loads of W: 6144 x
  // 4096 12.7 us (14.8 with 4 waves), 12288 x 4096 20.5 (25.2), 24576 x 8192 72 (76),
  // 3072 x 2048 8.1 (8.5)
  const Parts p = {scratch, context_len, nsplits, D};
  if (silu) launch<512, true, true, false>(y, w, N, K, x, residual, residual_out, weight, eps, {}, p, stream);
  else if (weight) launch<512, true, false, false>(y, w, N, K, x, residual, residual_out, weight, eps, {}, p, stream);
  else launch<256, false, false, false>(y, w, N, K, x, residual, residual_out, weight, eps, {}, p, stream);
}

// N = (num_q + 2 num_kv) * D rows; the queries to q_out, keys and values to the caches
extern "C" void lig_row_product_heads_launch(uint16_t* q_out, const uint16_t* w, int N, int K, const uint16_t* x,
                                             const uint16_t* residual, uint16_t* residual_out, const uint16_t* weight,
                                             float eps, const int64_t* position, const float* cos_sin, uint16_t* k_cache,
                                             uint16_t* v_cache, const int64_t* slot, int num_q, int num_kv, int D,
                                             int block_size, hipStream_t stream) {
  const Heads heads = {position, cos_sin, slot, k_cache, v_cache, num_q, num_kv, D, block_size};
  launch<512, true, false, true>(q_out, w, N, K, x, residual, residual_out, weight, eps, heads, {}, stream);
}
