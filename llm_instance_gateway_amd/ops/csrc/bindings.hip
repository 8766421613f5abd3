// Python bindings for the gfx950 kernels (torch extension, compiled by hipcc).
//
// Convention: every op takes the current HIP stream as an int64 handle
// (Python side passes torch.cuda.current_stream().cuda_stream) so the kernels
// serialize correctly with the library GEMMs on torch's stream without
// depending on the HIP/CUDA stream-masquerading ATen headers.

#include <algorithm>
#include <map>
#include <optional>
#include <vector>

#include <torch/extension.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <pybind11/numpy.h>
#if PY_VERSION_HEX < 0x030B0000
#include <longintrepr.h>
#endif

#include "common.h"

// LIG_DEBUG (make build-debug): host-side validation of device index tensors
// BEFORE a kernel dereferences them — a D2H copy per check, so debug-only.
#ifdef LIG_DEBUG
static void lig_check_range(const torch::Tensor& idx, long lo, long hi,
                            const char* what) {
  if (idx.numel() == 0) return;
  auto c = idx.to(torch::kCPU);
  const long mn = c.min().item<long>();
  const long mx = c.max().item<long>();
  TORCH_CHECK(mn >= lo && mx < hi, "LIG_DEBUG: ", what, " out of range [",
              lo, ", ", hi, "): min=", mn, " max=", mx);
}
#define LIG_CHECK_RANGE(t, lo, hi, what) lig_check_range(t, lo, hi, what)
#else
#define LIG_CHECK_RANGE(t, lo, hi, what) \
  do {                                   \
  } while (0)
#endif

extern "C" {
void lig_rms_norm_launch(uint16_t*, const uint16_t*, const uint16_t*, float,
                         int, int, hipStream_t);
void lig_fused_add_rms_norm_launch(uint16_t*, const uint16_t*, uint16_t*,
                                   const uint16_t*, float, int, int,
                                   hipStream_t);
void lig_rope_launch(const int64_t*, uint16_t*, uint16_t*, const float*, int,
                     int, int, int, hipStream_t);
void lig_reshape_and_cache_launch(const uint16_t*, const uint16_t*, uint16_t*,
                                  uint16_t*, const int64_t*, int, int, int,
                                  int, hipStream_t);
void lig_qkv_rope_cache_launch(uint16_t*, const uint16_t*, const int64_t*,
                               const float*, uint16_t*, uint16_t*,
                               const int64_t*, int, int, int, int, int,
                               hipStream_t);
bool lig_projection_serves(long, long, long);
bool lig_projection_pays(long, long, long);
int lig_projection_plan(int, int, int);
int lig_projection_splits(int);
int lig_projection_tile(int);
int lig_projection_runs(int, int, int, int);
void lig_projection_launch(int, uint16_t*, float*, const uint16_t*, const uint16_t*, int, int, int, hipStream_t);
int lig_row_product_max(bool);
void lig_row_product_launch(uint16_t*, const uint16_t*, int, int, const uint16_t*, const uint16_t*, uint16_t*,
                            const uint16_t*, float, bool, const float*, const int*, int, int, hipStream_t);
void lig_row_product_heads_launch(uint16_t*, const uint16_t*, int, int, const uint16_t*, const uint16_t*, uint16_t*,
                                  const uint16_t*, float, const int64_t*, const float*, uint16_t*, uint16_t*,
                                  const int64_t*, int, int, int, int, hipStream_t);
void lig_argmax_rows_launch(const void*, bool, long, int, int, int64_t*, hipStream_t);
void lig_silu_and_mul_launch(uint16_t*, const uint16_t*, int, int,
                             hipStream_t);
void lig_paged_attention_decode_launch(
    uint16_t*, const uint16_t*, const uint16_t*, const uint16_t*,
    const int*, const int*, float*, float, int, int, int, int, int, int,
    int, int, hipStream_t);
void lig_mfma_probe_launch(float*, const uint16_t*, const uint16_t*,
                           hipStream_t);
void lig_sgmv_shrink_launch(uint16_t*, const uint16_t*, const uint16_t*,
                            const int*, int, int, int, int, hipStream_t);
void lig_sgmv_expand_launch(uint16_t*, const uint16_t*, const uint16_t*,
                            const int*, float, int, int, int, int,
                            hipStream_t);
void lig_quant_fp8_rowwise_launch(uint8_t*, float*, const uint16_t*, int,
                                  int, hipStream_t);
void lig_sgmv_shrink_units_launch(uint16_t*, const uint16_t*, const uint16_t*,
                                  const int*, const int*, const int*,
                                  const int*, int, int, int, hipStream_t);
void lig_sgmv_expand_lds_launch(uint16_t*, const uint16_t*, const uint16_t*,
                                const int*, const int*, const int*,
                                const int*, float, int, int, int, int,
                                hipStream_t);
void lig_sgmv_expand_units_launch(uint16_t*, const uint16_t*, const uint16_t*,
                                  const int*, const int*, const int*,
                                  const int*, float, int, int, int,
                                  hipStream_t);
void lig_sgmv_shrink_tiled_launch(uint16_t*, const uint16_t*, const uint16_t*,
                                  const int*, const int*, const int*, int,
                                  int, int, int, hipStream_t);
void lig_sgmv_expand_tiled_launch(uint16_t*, const uint16_t*, const uint16_t*,
                                  const int*, const int*, const int*, int,
                                  float, int, int, int, hipStream_t);
int lig_lora_rms_norm_launch(uint16_t*, const uint16_t*, uint16_t*,
                             const uint16_t*, float, int, const int*,
                             const int*, const int*, int,
                             const float*, int, int, const uint16_t*,
                             const uint16_t*, float*, hipStream_t);
int lig_lora_silu_strip();
int lig_lora_norm_strip();
void lig_lora_rms_norm_strips_launch(
    uint16_t*, const uint16_t*, uint16_t*, const uint16_t*, float, int,
    const int*, const int*, const int*, int, const float*, int, int,
    const uint16_t*, const uint16_t*, float*, int, float*, hipStream_t);
void lig_lora_norm_open_launch(uint16_t*, const uint16_t*, const float*, int, long, uint16_t*, const uint16_t*, int,
                               const int*, const int*, const int*, int, const float*, int, int, const uint16_t*,
                               const uint16_t*, float*, int, float*, int, hipStream_t);
void lig_lora_silu_launch(uint16_t*, const uint16_t*, int, const int*,
                          const int*, const int*, int, const float*, int, int,
                          const uint16_t*, const uint16_t*, float*, int,
                          const float*, int, float, int, hipStream_t);
void lig_lora_shrink_launch(const uint16_t*, int, const int*, const int*,
                            const int*, int, const uint16_t*, float*, int,
                            hipStream_t);
int lig_lora_shrink_strip();
void lig_lora_qkv_rope_cache_launch(
    uint16_t*, const uint16_t*, const float*, int, long, const float*, int, float, const int64_t*, const float*, uint16_t*,
    uint16_t*, const int64_t*, int, int, int, int, const int*, const int*,
    const int*, int, const float*, int, int, const uint16_t*, int, hipStream_t);
int lig_paged_attention_prefill_parts(long, long, int, int, long);
void lig_paged_attention_prefill_launch(
    uint16_t*, const uint16_t*, const uint16_t*, const uint16_t*, const int*,
    const int*, const int*, const int*, const int*, float, int, int, int,
    int, int, int, int, int, float*, hipStream_t);
}

namespace {

inline uint16_t* bf16_ptr(torch::Tensor& t) {
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16, "expected bf16 tensor");
  TORCH_CHECK(t.is_contiguous(), "expected contiguous tensor");
  TORCH_CHECK(t.is_cuda(), "expected device tensor");
  return reinterpret_cast<uint16_t*>(t.data_ptr());
}

inline const uint16_t* bf16_cptr(const torch::Tensor& t) {
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16, "expected bf16 tensor");
  TORCH_CHECK(t.is_contiguous(), "expected contiguous tensor");
  TORCH_CHECK(t.is_cuda(), "expected device tensor");
  return reinterpret_cast<const uint16_t*>(t.data_ptr());
}

inline hipStream_t as_stream(int64_t s) {
  return reinterpret_cast<hipStream_t>(s);
}

void rms_norm(torch::Tensor out, torch::Tensor input, torch::Tensor weight,
              double eps, int64_t stream) {
  const int T = input.size(0);
  const int H = input.size(1);
  TORCH_CHECK(H % 8 == 0, "hidden must be a multiple of 8");
  lig_rms_norm_launch(bf16_ptr(out), bf16_cptr(input), bf16_cptr(weight),
                      (float)eps, T, H, as_stream(stream));
}

void fused_add_rms_norm(torch::Tensor out, torch::Tensor input,
                        torch::Tensor residual, torch::Tensor weight,
                        double eps, int64_t stream) {
  const int T = input.size(0);
  const int H = input.size(1);
  TORCH_CHECK(H % 8 == 0, "hidden must be a multiple of 8");
  lig_fused_add_rms_norm_launch(bf16_ptr(out), bf16_cptr(input),
                                bf16_ptr(residual), bf16_cptr(weight),
                                (float)eps, T, H, as_stream(stream));
}

void rotary_embedding(torch::Tensor positions, torch::Tensor q,
                      torch::Tensor k, torch::Tensor cos_sin,
                      int64_t head_dim, int64_t stream) {
  TORCH_CHECK(positions.scalar_type() == torch::kInt64);
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32);
  TORCH_CHECK(head_dim % 4 == 0, "head_dim must be a multiple of 4");
  const int T = q.size(0);
  const int hq = q.size(1) / head_dim;
  const int hk = k.size(1) / head_dim;
  lig_rope_launch(positions.data_ptr<int64_t>(), bf16_ptr(q), bf16_ptr(k),
                  cos_sin.data_ptr<float>(), T, hq, hk, (int)head_dim,
                  as_stream(stream));
}

void reshape_and_cache(torch::Tensor k, torch::Tensor v,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor slot_mapping, int64_t stream) {
  TORCH_CHECK(slot_mapping.scalar_type() == torch::kInt64);
  const int T = k.size(0);
  const int Hkv = k_cache.size(1);
  const int BS = k_cache.size(2);
  const int D = k_cache.size(3);
  TORCH_CHECK(D % 8 == 0, "head_dim must be a multiple of 8");
  lig_reshape_and_cache_launch(bf16_cptr(k), bf16_cptr(v), bf16_ptr(k_cache),
                               bf16_ptr(v_cache),
                               slot_mapping.data_ptr<int64_t>(), T, Hkv, D, BS,
                               as_stream(stream));
}

void qkv_rope_cache(torch::Tensor q_out, torch::Tensor qkv,
                    torch::Tensor positions, torch::Tensor cos_sin,
                    torch::Tensor k_cache, torch::Tensor v_cache,
                    torch::Tensor slot_mapping, int64_t stream) {
  TORCH_CHECK(positions.scalar_type() == torch::kInt64);
  TORCH_CHECK(slot_mapping.scalar_type() == torch::kInt64);
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32 && cos_sin.is_contiguous());
  const int T = qkv.size(0);
  const int Hkv = k_cache.size(1);
  const int BS = k_cache.size(2);
  const int D = k_cache.size(3);
  const int Hq = q_out.size(1) / D;
  TORCH_CHECK(D % 64 == 0, "head_dim must be a multiple of 64");
  TORCH_CHECK(cos_sin.size(1) == D && v_cache.sizes() == k_cache.sizes());
  TORCH_CHECK(qkv.size(1) == (int64_t)(Hq + 2 * Hkv) * D && q_out.size(0) == T &&
                  q_out.size(1) == (int64_t)Hq * D,
              "qkv rows must hold the query, key and value heads");
  TORCH_CHECK(positions.numel() >= T && slot_mapping.numel() >= T);
  if (T == 0) return;
  lig_qkv_rope_cache_launch(bf16_ptr(q_out), bf16_cptr(qkv),
                            positions.data_ptr<int64_t>(),
                            cos_sin.data_ptr<float>(), bf16_ptr(k_cache),
                            bf16_ptr(v_cache), slot_mapping.data_ptr<int64_t>(),
                            T, Hq, Hkv, D, BS, as_stream(stream));
}

// y = W h of one row: h = x, or the norm of x (+ residual, whose sum goes to
// residual_out) with `weight`; silu: W = [gate | up], y = silu(gate h) * (up h).
void row_product(torch::Tensor y, torch::Tensor w, torch::Tensor x, c10::optional<torch::Tensor> residual,
                 c10::optional<torch::Tensor> residual_out, c10::optional<torch::Tensor> weight, double eps, bool silu,
                 c10::optional<torch::Tensor> scratch, c10::optional<torch::Tensor> context_lens, int64_t nsplits,
                 int64_t head_dim, int64_t stream) {
  TORCH_CHECK(w.dim() == 2 && w.is_contiguous() && w.size(0) < (1 << 30));
  const int N = (int)w.size(0), K = (int)w.size(1);
  TORCH_CHECK(K > 0 && K % 512 == 0 && K <= lig_row_product_max(weight.has_value()), "width ", K);
  TORCH_CHECK(N > 0 && (!silu || (N % 2 == 0 && weight.has_value())));
  auto row = [&](torch::Tensor t, int n) {
    TORCH_CHECK(t.is_contiguous() && t.numel() == n && ((uintptr_t)t.data_ptr() & 15) == 0, "a contiguous row of ", n);
    return bf16_ptr(t);
  };
  TORCH_CHECK(residual.has_value() == residual_out.has_value() && (weight.has_value() || !residual.has_value()));
  TORCH_CHECK(((uintptr_t)w.data_ptr() & 15) == 0);
  TORCH_CHECK(y.is_contiguous() && y.numel() == (silu ? N / 2 : N));
  if (scratch) {
    TORCH_CHECK(!weight && context_lens && context_lens->scalar_type() == torch::kInt32 && context_lens->numel() >= 1);
    TORCH_CHECK(head_dim > 0 && head_dim % 8 == 0 && K % head_dim == 0 && nsplits >= 1 &&
                scratch->scalar_type() == torch::kFloat32 && scratch->numel() >= K / head_dim * nsplits * (head_dim + 2));
  }
  lig_row_product_launch(bf16_ptr(y), bf16_cptr(w), N, K, row(x, K), residual ? row(*residual, K) : nullptr,
                         residual_out ? row(*residual_out, K) : nullptr, weight ? row(*weight, K) : nullptr, (float)eps,
                         silu, scratch ? scratch->data_ptr<float>() : nullptr,
                         scratch ? context_lens->data_ptr<int>() : nullptr, (int)nsplits, (int)head_dim, as_stream(stream));
}

// The same product of a norm with a fused q, k and v projection, whose heads go where
// qkv_rope_cache puts them.
void row_product_heads(torch::Tensor q_out, torch::Tensor w, torch::Tensor x, c10::optional<torch::Tensor> residual,
                       c10::optional<torch::Tensor> residual_out, torch::Tensor weight, double eps, torch::Tensor positions,
                       torch::Tensor cos_sin, torch::Tensor k_cache, torch::Tensor v_cache, torch::Tensor slot_mapping,
                       int64_t stream) {
  TORCH_CHECK(w.dim() == 2 && w.is_contiguous() && w.size(0) < (1 << 30) && ((uintptr_t)w.data_ptr() & 15) == 0);
  const int N = (int)w.size(0), K = (int)w.size(1);
  TORCH_CHECK(K > 0 && K % 512 == 0 && K <= lig_row_product_max(true), "width ", K);
  auto row = [&](torch::Tensor t, int n) {
    TORCH_CHECK(t.is_contiguous() && t.numel() == n && ((uintptr_t)t.data_ptr() & 15) == 0, "a contiguous row of ", n);
    return bf16_ptr(t);
  };
  TORCH_CHECK(residual.has_value() == residual_out.has_value());
  TORCH_CHECK(positions.scalar_type() == torch::kInt64 && slot_mapping.scalar_type() == torch::kInt64);
  TORCH_CHECK(positions.numel() >= 1 && slot_mapping.numel() >= 1);
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32 && cos_sin.is_contiguous());
  TORCH_CHECK(k_cache.dim() == 4 && v_cache.sizes() == k_cache.sizes() && k_cache.is_contiguous() && v_cache.is_contiguous());
  const int Hkv = (int)k_cache.size(1), D = (int)k_cache.size(3);
  TORCH_CHECK(D % 64 == 0 && cos_sin.size(1) == D && q_out.is_contiguous() && q_out.numel() % D == 0);
  const int Hq = (int)(q_out.numel() / D);
  TORCH_CHECK(N == (Hq + 2 * Hkv) * D, "w must hold the query, key and value heads");
  lig_row_product_heads_launch(bf16_ptr(q_out), bf16_cptr(w), N, K, row(x, K), residual ? row(*residual, K) : nullptr,
                               residual_out ? row(*residual_out, K) : nullptr, row(weight, K), (float)eps,
                               positions.data_ptr<int64_t>(), cos_sin.data_ptr<float>(), bf16_ptr(k_cache),
                               bf16_ptr(v_cache), slot_mapping.data_ptr<int64_t>(), Hq, Hkv, D, (int)k_cache.size(2),
                               as_stream(stream));
}

// Whether a dispatch mode, a trace or a transform follows what is called
bool watched() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || torch::jit::tracer::isTracing() ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// Whether the kernels of projection.hip take that many rows against w, in parts: what
// Python would ask in a dozen attributes, ten times a layer (3 us each time)
bool projection_takes(const torch::Tensor& w, int64_t rows) {
  return w.is_cuda() && w.scalar_type() == torch::kBFloat16 && w.dim() == 2 && w.is_contiguous() &&
         ((uintptr_t)w.data_ptr() & 15) == 0 && !(w.requires_grad() && at::GradMode::is_enabled()) &&
         !watched() && lig_projection_serves(rows, w.size(0), w.size(1));
}

// and of the rows x
bool projection_takes_rows(const torch::Tensor& x, const torch::Tensor& w) {
  return x.is_cuda() && x.scalar_type() == torch::kBFloat16 && x.dim() == 2 && w.dim() == 2 &&
         x.size(1) == w.size(1) && x.device() == w.device() && x.is_contiguous() &&
         ((uintptr_t)x.data_ptr() & 15) == 0 && !(x.requires_grad() && at::GradMode::is_enabled()) &&
         projection_takes(w, x.size(0));
}

// y = x W^T of up to 1792 rows (projection.hip); sizes that it does not serve are refused
void projection(torch::Tensor y, torch::Tensor x, torch::Tensor w, int64_t stream) {
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && y.dim() == 2);
  const long M = x.size(0), N = w.size(0), K = w.size(1);
  TORCH_CHECK(x.size(1) == K && y.size(0) == M && y.size(1) == N && lig_projection_serves(M, N, K), "shape");
  for (const torch::Tensor* t : {&x, &w, &y})
    TORCH_CHECK(t->is_cuda() && t->is_contiguous() && ((uintptr_t)t->data_ptr() & 15) == 0, "contiguous, aligned");
  const int plan = lig_projection_plan((int)M, (int)N, (int)K), splits = lig_projection_splits(plan);
  torch::Tensor part;
  if (splits > 1) part = torch::empty({splits, M, N}, x.options().dtype(torch::kFloat32));
  lig_projection_launch(plan, bf16_ptr(y), splits > 1 ? part.data_ptr<float>() : nullptr, bf16_cptr(x), bf16_cptr(w),
                        (int)M, (int)N, (int)K, as_stream(stream));
}

// The same as fp32 [parts, M, N] that add up to it
torch::Tensor projection_parts(torch::Tensor x, torch::Tensor w, int64_t stream) {
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2);
  const long M = x.size(0), N = w.size(0), K = w.size(1);
  TORCH_CHECK(x.size(1) == K && lig_projection_serves(M, N, K), "shape");
  for (const torch::Tensor* t : {&x, &w})
    TORCH_CHECK(t->is_cuda() && t->is_contiguous() && ((uintptr_t)t->data_ptr() & 15) == 0, "contiguous, aligned");
  const int plan = lig_projection_plan((int)M, (int)N, (int)K);
  torch::Tensor part = torch::empty({lig_projection_splits(plan), M, N}, x.options().dtype(torch::kFloat32));
  lig_projection_launch(plan, nullptr, part.data_ptr<float>(), bf16_cptr(x), bf16_cptr(w), (int)M, (int)N, (int)K,
                        as_stream(stream));
  return part;
}

// (rows of y, columns of y) of the tile that a served size is planned for, and the parts of K
std::tuple<int, int, int> projection_plan(int M, int N, int K) {
  TORCH_CHECK(lig_projection_serves(M, N, K), "shape");
  const int plan = lig_projection_plan(M, N, K), tile = lig_projection_tile(plan);
  return {tile / 1000, tile % 1000, lig_projection_splits(plan)};
}

// and of the tile that runs in its place, or its own
std::tuple<int, int> projection_runs(int M, int N, int K) {
  TORCH_CHECK(lig_projection_serves(M, N, K), "shape");
  const int tile = lig_projection_runs(lig_projection_plan(M, N, K), M, N, K);
  return {tile / 1000, tile % 1000};
}

void argmax_rows(torch::Tensor out, torch::Tensor x, int64_t stream) {
  const bool bf16 = x.scalar_type() == torch::kBFloat16;
  TORCH_CHECK(x.is_cuda() && (bf16 || x.scalar_type() == torch::kFloat32), "bf16 or fp32 rows on the device");
  TORCH_CHECK(x.dim() == 2 && x.stride(1) == 1 && x.size(1) > 0 && x.size(1) < (1L << 31) - 1024 &&
                  x.size(0) < (1L << 22),
              "[N, V] rows");
  TORCH_CHECK(out.is_cuda() && out.scalar_type() == torch::kInt64 && out.is_contiguous() && out.dim() == 1 &&
              out.size(0) == x.size(0));
  lig_argmax_rows_launch(x.data_ptr(), bf16, x.stride(0), (int)x.size(0), (int)x.size(1), out.data_ptr<int64_t>(),
                         as_stream(stream));
}

void silu_and_mul(torch::Tensor out, torch::Tensor x, int64_t stream) {
  const int T = x.size(0);
  const int d = x.size(1) / 2;
  TORCH_CHECK(d % 8 == 0, "intermediate must be a multiple of 8");
  lig_silu_and_mul_launch(bf16_ptr(out), bf16_cptr(x), T, d,
                          as_stream(stream));
}

void paged_attention_decode(torch::Tensor out, torch::Tensor q,
                            torch::Tensor k_cache, torch::Tensor v_cache,
                            torch::Tensor block_tables,
                            torch::Tensor context_lens, double scale,
                            int64_t stream) {
  TORCH_CHECK(block_tables.scalar_type() == torch::kInt32);
  TORCH_CHECK(context_lens.scalar_type() == torch::kInt32);
  const int N = q.size(0);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hkv = k_cache.size(1);
  const int BS = k_cache.size(2);
  const int max_blocks = block_tables.size(1);
  TORCH_CHECK(D == 16 || D == 64 || D == 128, "head_dim must be 16/64/128");
  TORCH_CHECK(Hq % Hkv == 0 && Hq / Hkv <= 16, "bad GQA group size");
  if (N == 0) return;
  LIG_CHECK_RANGE(block_tables, 0, k_cache.size(0), "decode block_tables");
  LIG_CHECK_RANGE(context_lens, 0, (long)block_tables.size(1) * BS + 1,
                  "decode context_lens");
  lig_paged_attention_decode_launch(
      bf16_ptr(out), bf16_cptr(q), bf16_cptr(k_cache), bf16_cptr(v_cache),
      block_tables.data_ptr<int>(), context_lens.data_ptr<int>(), nullptr,
      (float)scale, N, Hq, Hkv, D, BS, max_blocks, 1, 0, as_stream(stream));
}

// Flash-decoding variant: every context cut over up to nsplits workgroups with
// an fp32 partial scratch [N, Hq, nsplits, D+2] and a merging pass, or without
// that for a reader that merges by itself.
template <bool MERGE>
void paged_attention_decode_split(torch::Tensor out, torch::Tensor q,
                                  torch::Tensor k_cache,
                                  torch::Tensor v_cache,
                                  torch::Tensor block_tables,
                                  torch::Tensor context_lens,
                                  torch::Tensor scratch, double scale,
                                  int64_t nsplits, int64_t stream) {
  TORCH_CHECK(block_tables.scalar_type() == torch::kInt32);
  TORCH_CHECK(context_lens.scalar_type() == torch::kInt32);
  TORCH_CHECK(scratch.scalar_type() == torch::kFloat32);
  const int N = q.size(0);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hkv = k_cache.size(1);
  const int BS = k_cache.size(2);
  const int max_blocks = block_tables.size(1);
  TORCH_CHECK(D == 16 || D == 64 || D == 128, "head_dim must be 16/64/128");
  TORCH_CHECK(Hq % Hkv == 0 && Hq / Hkv <= 16, "bad GQA group size");
  TORCH_CHECK(nsplits >= 1, "nsplits must be positive");
  TORCH_CHECK(scratch.numel() >= (int64_t)N * Hq * nsplits * (D + 2),
              "scratch too small");
  if (N == 0) return;
  lig_paged_attention_decode_launch(
      bf16_ptr(out), bf16_cptr(q), bf16_cptr(k_cache), bf16_cptr(v_cache),
      block_tables.data_ptr<int>(), context_lens.data_ptr<int>(),
      scratch.data_ptr<float>(), (float)scale, N, Hq, Hkv, D, BS,
      max_blocks, (int)nsplits, !MERGE, as_stream(stream));
}

void paged_attention_prefill(torch::Tensor out, torch::Tensor q,
                             torch::Tensor k_cache, torch::Tensor v_cache,
                             torch::Tensor tile_seq, torch::Tensor tile_qstart,
                             torch::Tensor query_start_locs,
                             torch::Tensor context_lens,
                             torch::Tensor block_tables, double scale,
                             int64_t stream) {
  TORCH_CHECK(tile_seq.scalar_type() == torch::kInt32);
  TORCH_CHECK(tile_qstart.scalar_type() == torch::kInt32);
  TORCH_CHECK(query_start_locs.scalar_type() == torch::kInt32);
  TORCH_CHECK(context_lens.scalar_type() == torch::kInt32);
  TORCH_CHECK(block_tables.scalar_type() == torch::kInt32);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hkv = k_cache.size(1);
  const int BS = k_cache.size(2);
  const int ntiles = tile_seq.size(0);
  const int max_blocks = block_tables.size(1);
  TORCH_CHECK(D == 64 || D == 128, "prefill MFMA kernel needs head_dim 64/128");
  if (ntiles == 0) return;
  const int parts = lig_paged_attention_prefill_parts(ntiles, q.size(0), Hq, D, (long)max_blocks * BS);
  torch::Tensor partial;
  if (parts > 1) partial = torch::empty({q.size(0), Hq, parts, D + 4}, q.options().dtype(torch::kFloat32));
  lig_paged_attention_prefill_launch(
      bf16_ptr(out), bf16_cptr(q), bf16_cptr(k_cache), bf16_cptr(v_cache),
      tile_seq.data_ptr<int>(), tile_qstart.data_ptr<int>(),
      query_start_locs.data_ptr<int>(), context_lens.data_ptr<int>(),
      block_tables.data_ptr<int>(), (float)scale, ntiles, Hq, Hkv, D, BS,
      max_blocks, (int)std::min(query_start_locs.size(0) - 1, context_lens.size(0)), parts, parts > 1 ? partial.data_ptr<float>() : nullptr, as_stream(stream));
}

void sgmv_shrink(torch::Tensor u, torch::Tensor x, torch::Tensor a_stack,
                 torch::Tensor slots, int64_t stream) {
  TORCH_CHECK(slots.scalar_type() == torch::kInt32);
  const int T = x.size(0);
  const int H = x.size(1);
  const int R = a_stack.size(1);
  TORCH_CHECK(a_stack.size(2) == H, "A stack in-features mismatch");
  TORCH_CHECK(H % 8 == 0 && R <= 64);
  if (T == 0) return;
  lig_sgmv_shrink_launch(bf16_ptr(u), bf16_cptr(x), bf16_cptr(a_stack),
                         slots.data_ptr<int>(), T, R, H, T >= 256,
                         as_stream(stream));
}

// one call = shrink + expand (halves Python dispatch; u is a caller-owned
// workspace so no per-call allocation)
void sgmv_apply(torch::Tensor y, torch::Tensor x, torch::Tensor a_stack,
                torch::Tensor b_stack, torch::Tensor u_ws,
                torch::Tensor slots, double scaling, bool use_wide,
                int64_t stream) {
  TORCH_CHECK(slots.scalar_type() == torch::kInt32);
  const int T = x.size(0);
  const int H = x.size(1);
  const int R = a_stack.size(1);
  const int O = y.size(1);
  TORCH_CHECK(u_ws.size(0) >= T && u_ws.size(1) == R, "u workspace too small");
  TORCH_CHECK(R % 8 == 0 && R <= 64, "rank must be 8/16/32/64");
  if (T == 0) return;
  LIG_CHECK_RANGE(slots, -1, a_stack.size(0), "sgmv slots");
  hipStream_t st = as_stream(stream);
  lig_sgmv_shrink_launch(bf16_ptr(u_ws), bf16_cptr(x), bf16_cptr(a_stack),
                         slots.data_ptr<int>(), T, R, H, use_wide, st);
  lig_sgmv_expand_launch(bf16_ptr(y), bf16_cptr(u_ws), bf16_cptr(b_stack),
                         slots.data_ptr<int>(), (float)scaling, T, R, O,
                         use_wide, st);
}

// Slot-grouped units: shrink via the proven v2 kernels (occupancy-
// first), expand via the LDS-staged unit kernel — full per-token thread
// parallelism with B read once per <=32-token unit instead of per token
// (profiles/r02_kernel_stats.md: the per-token kernels were 27% of all
// kernel time).  Static shapes (padded empty units) so the hipGraph decode
// path can bake it.  Requires O % 256 == 0 (every serving module dim);
// caller falls back to sgmv_apply otherwise.
void sgmv_apply_units(torch::Tensor y, torch::Tensor x, torch::Tensor a_stack,
                      torch::Tensor b_stack, torch::Tensor u_ws,
                      torch::Tensor slots, torch::Tensor order,
                      torch::Tensor unit_t0, torch::Tensor unit_len,
                      torch::Tensor unit_slot, double scaling, bool use_wide,
                      int64_t stream) {
  TORCH_CHECK(slots.scalar_type() == torch::kInt32);
  TORCH_CHECK(order.scalar_type() == torch::kInt32);
  TORCH_CHECK(unit_t0.scalar_type() == torch::kInt32);
  TORCH_CHECK(unit_len.scalar_type() == torch::kInt32);
  TORCH_CHECK(unit_slot.scalar_type() == torch::kInt32);
  const int T = x.size(0);
  const int H = x.size(1);
  const int R = a_stack.size(1);
  const int O = y.size(1);
  const int U = unit_t0.size(0);
  TORCH_CHECK(u_ws.size(0) >= T && u_ws.size(1) == R, "u workspace too small");
  TORCH_CHECK(R % 8 == 0 && R <= 64, "rank must be 8/16/32/64");
  TORCH_CHECK(H % 8 == 0 && O % 256 == 0, "units expand needs O%256==0");
  if (T == 0 || U == 0) return;
  LIG_CHECK_RANGE(slots, -1, a_stack.size(0), "sgmv slots");
  LIG_CHECK_RANGE(order, 0, T, "sgmv unit order");
  LIG_CHECK_RANGE(unit_t0, 0, T, "sgmv unit_t0");
  LIG_CHECK_RANGE(unit_len, 0, T + 1, "sgmv unit_len");
  LIG_CHECK_RANGE(unit_slot, -1, b_stack.size(0), "sgmv unit_slot");
  hipStream_t st = as_stream(stream);
  lig_sgmv_shrink_launch(bf16_ptr(u_ws), bf16_cptr(x), bf16_cptr(a_stack),
                         slots.data_ptr<int>(), T, R, H, use_wide, st);
  lig_sgmv_expand_lds_launch(
      bf16_ptr(y), bf16_cptr(u_ws), bf16_cptr(b_stack),
      order.data_ptr<int>(), unit_t0.data_ptr<int>(),
      unit_len.data_ptr<int>(), unit_slot.data_ptr<int>(), (float)scaling, U,
      T, R, O, st);
}

// Prefill LoRA: one shrink+expand over host-built 64-token segment tiles
// (MFMA path; engine/model_runner.py builds the tiles).
void sgmv_apply_tiled(torch::Tensor y, torch::Tensor x, torch::Tensor a_stack,
                      torch::Tensor b_stack, torch::Tensor u_ws,
                      torch::Tensor tile_t0, torch::Tensor tile_len,
                      torch::Tensor tile_slot, double scaling,
                      int64_t stream) {
  const int T = x.size(0);
  const int H = x.size(1);
  const int R = a_stack.size(1);
  const int O = y.size(1);
  const int ntiles = tile_t0.size(0);
  TORCH_CHECK(tile_t0.scalar_type() == torch::kInt32);
  TORCH_CHECK(u_ws.size(0) >= T && u_ws.size(1) == R, "u workspace too small");
  TORCH_CHECK(R % 8 == 0 && R <= 64, "rank must be 8/16/32/64");
  TORCH_CHECK(H % 32 == 0 && O % 64 == 0, "tiled sgmv needs H%32==0, O%64==0");
  if (T == 0 || ntiles == 0) return;
  hipStream_t st = as_stream(stream);
  lig_sgmv_shrink_tiled_launch(bf16_ptr(u_ws), bf16_cptr(x),
                               bf16_cptr(a_stack), tile_t0.data_ptr<int>(),
                               tile_len.data_ptr<int>(),
                               tile_slot.data_ptr<int>(), ntiles, T, R, H, st);
  lig_sgmv_expand_tiled_launch(bf16_ptr(y), bf16_cptr(u_ws),
                               bf16_cptr(b_stack), tile_t0.data_ptr<int>(),
                               tile_len.data_ptr<int>(),
                               tile_slot.data_ptr<int>(), ntiles,
                               (float)scaling, T, R, O, st);
}

void sgmv_expand(torch::Tensor y, torch::Tensor u, torch::Tensor b_stack,
                 torch::Tensor slots, double scaling, int64_t stream) {
  TORCH_CHECK(slots.scalar_type() == torch::kInt32);
  const int T = u.size(0);
  const int R = u.size(1);
  const int O = y.size(1);
  TORCH_CHECK(b_stack.size(1) == O && b_stack.size(2) == R, "B stack mismatch");
  TORCH_CHECK(O % 8 == 0 && R % 8 == 0 && R <= 64, "rank must be 8/16/32/64");
  if (T == 0) return;
  lig_sgmv_expand_launch(bf16_ptr(y), bf16_cptr(u), bf16_cptr(b_stack),
                         slots.data_ptr<int>(), (float)scaling, T, R, O,
                         T >= 256, as_stream(stream));
}

void quant_fp8_rowwise(torch::Tensor xq, torch::Tensor xs, torch::Tensor x,
                       int64_t stream) {
  TORCH_CHECK(x.scalar_type() == torch::kBFloat16, "x must be bf16");
  TORCH_CHECK(xq.element_size() == 1, "xq must be an 8-bit (fp8) tensor");
  TORCH_CHECK(xs.scalar_type() == torch::kFloat32, "xs must be fp32");
  TORCH_CHECK(x.dim() == 2 && xq.sizes() == x.sizes(), "shape mismatch");
  const int T = x.size(0);
  const int K = x.size(1);
  TORCH_CHECK(K % 8 == 0, "K must be a multiple of 8");
  TORCH_CHECK(xs.numel() == T, "xs must have one scale per row");
  TORCH_CHECK(x.is_contiguous() && xq.is_contiguous() && xs.is_contiguous());
  TORCH_CHECK(xq.is_cuda() && xs.is_cuda());
  lig_quant_fp8_rowwise_launch(reinterpret_cast<uint8_t*>(xq.data_ptr()),
                               xs.data_ptr<float>(), bf16_cptr(x), T, K,
                               as_stream(stream));
}

// ---- LoRA inside the layer's kernels (lora_rows.hip) ------------------------
// toks [tiles, 16], len, slot: tiles of up to 16 tokens of one adapter that
// together list every row; u: fp32 [parts, tiles, 16, 16]; A [slots, 16, in], B [slots,
// out, 16].

inline const int* i32_cptr(const torch::Tensor& t) {
  TORCH_CHECK(t.scalar_type() == torch::kInt32 && t.is_contiguous() && t.is_cuda());
  return t.data_ptr<int>();
}

inline float* u_ptr(const torch::Tensor& u, int64_t parts, int64_t ntiles) {
  TORCH_CHECK(u.scalar_type() == torch::kFloat32 && u.is_contiguous() && u.is_cuda());
  TORCH_CHECK(u.dim() == 4 && u.size(0) >= parts && u.size(1) >= ntiles &&
                  u.size(2) == 16 && u.size(3) == 16,
              "u is [parts, tiles, 16, 16]");
  return u.data_ptr<float>();
}

inline const uint16_t* a_ptr(const torch::Tensor& a, int64_t width) {
  TORCH_CHECK(a.dim() == 3 && a.size(1) == 16 && a.size(2) == width, "A stack mismatch");
  return bf16_cptr(a);
}

inline const uint16_t* b_ptr(const torch::Tensor& b, int64_t width) {
  TORCH_CHECK(b.dim() == 3 && b.size(1) == width && b.size(2) == 16, "B stack mismatch");
  return bf16_cptr(b);
}

inline int check_tiles(const torch::Tensor& toks, const torch::Tensor& len,
                       const torch::Tensor& slot, int64_t T, int64_t slots) {
  TORCH_CHECK(toks.numel() == 16 * len.numel() && slot.numel() == len.numel());
  LIG_CHECK_RANGE(toks, 0, T, "lora rows toks");
  LIG_CHECK_RANGE(len, 0, 17, "lora rows len");
  LIG_CHECK_RANGE(slot, -1, slots, "lora rows slot");
  return len.numel();
}

void lora_rms_norm(torch::Tensor out, torch::Tensor x,
                   std::optional<torch::Tensor> residual, torch::Tensor weight,
                   double eps, torch::Tensor toks,
                   torch::Tensor len, torch::Tensor slot,
                   std::optional<torch::Tensor> u_in,
                   std::optional<torch::Tensor> b_stack,
                   std::optional<torch::Tensor> a_stack,
                   std::optional<torch::Tensor> u_out,
                   std::optional<torch::Tensor> sums, int64_t stream) {
  const int T = x.size(0), H = x.size(1);
  TORCH_CHECK(out.sizes() == x.sizes() && weight.numel() == H);
  TORCH_CHECK(!residual || residual->sizes() == x.sizes());
  TORCH_CHECK(u_in.has_value() == b_stack.has_value() && u_out.has_value() == a_stack.has_value());
  const int64_t slots = b_stack ? b_stack->size(0) : a_stack ? a_stack->size(0) : 1 << 30;
  const int n = check_tiles(toks, len, slot, T, slots);
  if (n == 0 || T == 0) return;
  if (sums) {  // strips of columns in two launches; u_out has a part for each
    const int strip = lig_lora_norm_strip();
    TORCH_CHECK(H % strip == 0 && sums->scalar_type() == torch::kFloat32 &&
                sums->is_cuda() && sums->numel() >= (int64_t)n * (H / strip) * 16);
    lig_lora_rms_norm_strips_launch(
        bf16_ptr(out), bf16_cptr(x), residual ? bf16_ptr(*residual) : nullptr,
        bf16_cptr(weight), (float)eps, H, i32_cptr(toks), i32_cptr(len),
        i32_cptr(slot), n, u_in ? u_ptr(*u_in, 1, n) : nullptr,
        u_in ? (int)u_in->size(0) : 0, u_in ? (int)u_in->size(1) : 0,
        b_stack ? b_ptr(*b_stack, H) : nullptr,
        a_stack ? a_ptr(*a_stack, H) : nullptr,
        u_out ? u_ptr(*u_out, H / strip, n) : nullptr,
        u_out ? (int)u_out->size(1) : 0, sums->data_ptr<float>(), as_stream(stream));
    return;
  }
  const int rc = lig_lora_rms_norm_launch(
      bf16_ptr(out), bf16_cptr(x), residual ? bf16_ptr(*residual) : nullptr,
      bf16_cptr(weight), (float)eps, H, i32_cptr(toks),
      i32_cptr(len), i32_cptr(slot), n,
      u_in ? u_ptr(*u_in, 1, n) : nullptr, u_in ? (int)u_in->size(0) : 0,
      u_in ? (int)u_in->size(1) : 0, b_stack ? b_ptr(*b_stack, H) : nullptr,
      a_stack ? a_ptr(*a_stack, H) : nullptr,
      u_out ? u_ptr(*u_out, 1, n) : nullptr, as_stream(stream));
  TORCH_CHECK(rc == 0, "lora_rms_norm: rows of ", H, " entries not served");
}

using OptTensor = std::optional<torch::Tensor>;

// sums of squares per tile and strip of rows of `width` columns
inline float* sums_ptr(const std::optional<torch::Tensor>& sums, int64_t width, int64_t n) {
  if (!sums) return nullptr;
  const int strip = lig_lora_norm_strip();
  TORCH_CHECK(width > 0 && width % strip == 0 && sums->scalar_type() == torch::kFloat32 && sums->is_cuda() &&
              sums->is_contiguous() && sums->numel() >= n * (width / strip) * 16);
  return sums->data_ptr<float>();
}

// tiles of a step: listed, or the rows in their order without adapters
struct RowTiles {
  const int *toks = nullptr, *len = nullptr, *slot = nullptr;
  int n;
};
inline RowTiles tiles_of(const OptTensor& toks, const OptTensor& len, const OptTensor& slot, int64_t T, int64_t slots) {
  RowTiles t;
  TORCH_CHECK(toks.has_value() == len.has_value() && toks.has_value() == slot.has_value());
  if (!toks) {
    t.n = (int)((T + 15) / 16);
    return t;
  }
  t.n = check_tiles(*toks, *len, *slot, T, slots);
  t.toks = i32_cptr(*toks);
  t.len = i32_cptr(*len);
  t.slot = i32_cptr(*slot);
  return t;
}

// out = (residual + x + B u_in) * weight, which residual becomes without the weight, u_out = A out and
// `sums` for the norm's factor; x bf16 [T, H] or the fp32 parts [S, T, H] of a product
void lora_norm_open(torch::Tensor out, torch::Tensor x, OptTensor residual, torch::Tensor weight, OptTensor toks,
                    OptTensor len, OptTensor slot, OptTensor u_in, OptTensor b_stack, OptTensor a_stack,
                    OptTensor u_out, torch::Tensor sums, int64_t stream) {
  const bool parts = x.dim() == 3;
  const int T = out.size(0), H = out.size(1);
  TORCH_CHECK(x.size(-1) == H && x.size(-2) == T && x.is_contiguous() && x.is_cuda() && weight.numel() == H);
  TORCH_CHECK(!parts || (x.scalar_type() == torch::kFloat32 && x.size(0) > 0 && residual));
  TORCH_CHECK(!residual || residual->sizes() == out.sizes());
  TORCH_CHECK(u_in.has_value() == b_stack.has_value() && (!u_in || residual));
  TORCH_CHECK(u_out.has_value() == a_stack.has_value() && u_out.has_value() == toks.has_value());
  const RowTiles t = tiles_of(toks, len, slot, T, a_stack ? a_stack->size(0) : 0);
  if (t.n == 0 || T == 0) return;
  lig_lora_norm_open_launch(
      bf16_ptr(out), parts ? nullptr : bf16_cptr(x), parts ? x.data_ptr<float>() : nullptr, parts ? (int)x.size(0) : 0,
      (long)T * H, residual ? bf16_ptr(*residual) : nullptr, bf16_cptr(weight), H, t.toks, t.len, t.slot, t.n,
      u_in ? u_ptr(*u_in, 1, t.n) : nullptr, u_in ? (int)u_in->size(0) : 0, u_in ? (int)u_in->size(1) : 0,
      b_stack ? b_ptr(*b_stack, H) : nullptr, a_stack ? a_ptr(*a_stack, H) : nullptr,
      u_out ? u_ptr(*u_out, H / lig_lora_norm_strip(), t.n) : nullptr, u_out ? (int)u_out->size(1) : 0,
      sums_ptr(sums, H, t.n), T, as_stream(stream));
}

void lora_silu(torch::Tensor out, torch::Tensor x, OptTensor toks, OptTensor len, OptTensor slot, OptTensor u_in,
               OptTensor b_stack, OptTensor a_stack, OptTensor u_out, OptTensor sums, int64_t width, double eps,
               int64_t stream) {
  const int T = x.size(0), d = out.size(1);
  TORCH_CHECK(out.size(0) == T && x.size(1) == 2 * (int64_t)d && d % 32 == 0);
  for (const OptTensor* o : {&u_in, &b_stack, &a_stack, &u_out}) TORCH_CHECK(o->has_value() == toks.has_value());
  const RowTiles t = tiles_of(toks, len, slot, T, b_stack ? b_stack->size(0) : 0);
  if (t.n == 0 || T == 0) return;
  const int strip = lig_lora_silu_strip();
  TORCH_CHECK(!toks || a_stack->size(0) == b_stack->size(0));
  lig_lora_silu_launch(bf16_ptr(out), bf16_cptr(x), d, t.toks, t.len, t.slot, t.n,
                       toks ? u_ptr(*u_in, 1, t.n) : nullptr, toks ? (int)u_in->size(0) : 0,
                       toks ? (int)u_in->size(1) : 0, toks ? b_ptr(*b_stack, 2 * (int64_t)d) : nullptr,
                       toks ? a_ptr(*a_stack, d) : nullptr, toks ? u_ptr(*u_out, (d + strip - 1) / strip, t.n) : nullptr,
                       toks ? (int)u_out->size(1) : 0, sums_ptr(sums, width, t.n), (int)width, (float)eps, T,
                       as_stream(stream));
}

void lora_shrink(torch::Tensor x, torch::Tensor toks,
                 torch::Tensor len, torch::Tensor slot, torch::Tensor a_stack,
                 torch::Tensor u_out, int64_t stream) {
  const int T = x.size(0), W = x.size(1);
  TORCH_CHECK(W % 32 == 0, "row width must be a multiple of 32");
  const int n = check_tiles(toks, len, slot, T, a_stack.size(0));
  if (n == 0 || T == 0) return;
  lig_lora_shrink_launch(bf16_cptr(x), W, i32_cptr(toks),
                         i32_cptr(len), i32_cptr(slot), n, a_ptr(a_stack, W),
                         u_ptr(u_out, (W + lig_lora_shrink_strip() - 1) / lig_lora_shrink_strip(), n),
                         (int)u_out.size(1), as_stream(stream));
}

void lora_qkv_rope_cache(torch::Tensor q_out, torch::Tensor qkv,
                         torch::Tensor positions, torch::Tensor cos_sin,
                         torch::Tensor k_cache, torch::Tensor v_cache,
                         torch::Tensor slot_mapping, OptTensor toks, OptTensor len, OptTensor slot,
                         OptTensor u_in, OptTensor b_stack, OptTensor sums, int64_t width, double eps,
                         int64_t stream) {
  TORCH_CHECK(positions.scalar_type() == torch::kInt64);
  TORCH_CHECK(slot_mapping.scalar_type() == torch::kInt64);
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32 && cos_sin.is_contiguous());
  const bool parts = qkv.dim() == 3;  // fp32 parts of the product
  TORCH_CHECK(!parts || (qkv.scalar_type() == torch::kFloat32 && qkv.is_contiguous() && qkv.is_cuda() && qkv.size(0) > 0));
  const int T = qkv.size(-2), Hkv = k_cache.size(1), BS = k_cache.size(2), D = k_cache.size(3);
  const int Hq = q_out.size(1) / D;
  TORCH_CHECK(D % 64 == 0 && cos_sin.size(1) == D && v_cache.sizes() == k_cache.sizes());
  TORCH_CHECK(qkv.size(-1) == (int64_t)(Hq + 2 * Hkv) * D && q_out.size(0) == T &&
              q_out.size(1) == (int64_t)Hq * D);
  TORCH_CHECK(positions.numel() >= T && slot_mapping.numel() >= T);
  TORCH_CHECK(u_in.has_value() == toks.has_value() && b_stack.has_value() == toks.has_value());
  const RowTiles t = tiles_of(toks, len, slot, T, b_stack ? b_stack->size(0) : 0);
  if (t.n == 0 || T == 0) return;
  lig_lora_qkv_rope_cache_launch(
      bf16_ptr(q_out), parts ? nullptr : bf16_cptr(qkv), parts ? qkv.data_ptr<float>() : nullptr,
      parts ? (int)qkv.size(0) : 0, (long)T * qkv.size(-1), sums_ptr(sums, width, t.n), (int)width, (float)eps,
      positions.data_ptr<int64_t>(), cos_sin.data_ptr<float>(), bf16_ptr(k_cache), bf16_ptr(v_cache),
      slot_mapping.data_ptr<int64_t>(), Hq, Hkv, D, BS, t.toks, t.len, t.slot, t.n,
      toks ? u_ptr(*u_in, 1, t.n) : nullptr, toks ? (int)u_in->size(0) : 0, toks ? (int)u_in->size(1) : 0,
      toks ? b_ptr(*b_stack, qkv.size(-1)) : nullptr, T, as_stream(stream));
}

}  // namespace

// Row i of `rows` (whole numbers) to out[i, :len], or one after another into a
// one-dimensional `out` (int32 or int64).
namespace py = pybind11;

template <typename I>
static void pack_rows_as(const py::sequence& rows, py::array& out) {
  const bool flat = out.ndim() == 1;
  const ssize_t n = py::len(rows), width = flat ? out.shape(0) : out.shape(1);
  TORCH_CHECK(flat || n <= out.shape(0), "more rows than room");
  I* dst = (I*)out.mutable_data();
  ssize_t at = 0;
  for (ssize_t i = 0; i < n; ++i) {
    const py::object row =
        py::reinterpret_steal<py::object>(PySequence_Fast(py::object(rows[i]).ptr(), "a row is a list"));
    if (!row) throw py::error_already_set();
    const ssize_t len = PySequence_Fast_GET_SIZE(row.ptr());
    I* to = flat ? dst + at : dst + i * width;
    TORCH_CHECK(len <= width - (flat ? at : 0), "a row of ", len, " numbers is longer than its room");
    for (ssize_t j = 0; j < len; ++j) {
      PyObject* e = PySequence_Fast_GET_ITEM(row.ptr(), j);
      const long long v = PyLong_Check(e) ? PyLong_AsLongLong(e)
                                          : py::reinterpret_borrow<py::object>(e).cast<long long>();
      if (v == -1 && PyErr_Occurred()) throw py::error_already_set();
      TORCH_CHECK(v == (long long)(I)v, v, " does not fit");
      to[j] = (I)v;
    }
    at += len;
  }
  TORCH_CHECK(!flat || at == width, at, " numbers for ", width, " places");
}

static void pack_rows(py::sequence rows, py::array out) {
  TORCH_CHECK((out.ndim() == 1 || out.ndim() == 2) && (out.flags() & py::array::c_style), "1-d or 2-d in row order");
  if (py::isinstance<py::array_t<int32_t>>(out)) pack_rows_as<int32_t>(rows, out);
  else if (py::isinstance<py::array_t<int64_t>>(out)) pack_rows_as<int64_t>(rows, out);
  else TORCH_CHECK(false, "int32 or int64");
}

// What sequences that each process their token at num_computed_tokens bring: that
// token, its position, and their cache blocks in a row of `tables` (int32, zeros).
// Arrays of other types are refused (noconvert): a converted one would be filled and
// dropped.
static void pack_decodes(py::list seqs, int64_t block_size, py::array_t<int64_t> ids, py::array_t<int64_t> positions,
                         py::array_t<int32_t> tables) {
  const ssize_t n = py::len(seqs);
  TORCH_CHECK(block_size > 0 && ids.ndim() == 1 && positions.ndim() == 1 && tables.ndim() == 2 && ids.shape(0) == n &&
              positions.shape(0) == n && tables.shape(0) == n);
  for (const py::array* a : {(py::array*)&ids, (py::array*)&positions, (py::array*)&tables})
    TORCH_CHECK(a->flags() & py::array::c_style, "in row order");
  static PyObject* names[4] = {PyUnicode_InternFromString("num_computed_tokens"), PyUnicode_InternFromString("block_table"),
                               PyUnicode_InternFromString("prompt_token_ids"),
                               PyUnicode_InternFromString("output_token_ids")};
  auto get = [](PyObject* o, PyObject* name) {
    PyObject* v = PyObject_GetAttr(o, name);
    if (!v) throw py::error_already_set();
    return py::reinterpret_steal<py::object>(v);
  };
  auto number = [](PyObject* e) {
#if PY_VERSION_HEX < 0x030B0000
    // one digit, as cache blocks and tokens are: read in place, a fifth of the call's time
    if (PyLong_CheckExact(e) && (size_t)Py_SIZE(e) <= 1) return (long long)(Py_SIZE(e) ? ((PyLongObject*)e)->ob_digit[0] : 0);
#endif
    const long long v = PyLong_Check(e) ? PyLong_AsLongLong(e) : py::reinterpret_borrow<py::object>(e).cast<long long>();
    if (v == -1 && PyErr_Occurred()) throw py::error_already_set();
    return v;
  };
  auto fast = [](const py::object& o) {
    PyObject* f = PySequence_Fast(o.ptr(), "a list of numbers");
    if (!f) throw py::error_already_set();
    return py::reinterpret_steal<py::object>(f);
  };
  int64_t *id = ids.mutable_data(), *at = positions.mutable_data();
  int32_t* row = tables.mutable_data();
  const ssize_t width = tables.shape(1);
  for (ssize_t i = 0; i < n; ++i, row += width) {
    PyObject* q = PyList_GET_ITEM(seqs.ptr(), i);
    const long long p = number(get(q, names[0]).ptr());
    const py::object blocks = fast(get(q, names[1])), prompt = fast(get(q, names[2]));
    const ssize_t len = PySequence_Fast_GET_SIZE(blocks.ptr()), known = PySequence_Fast_GET_SIZE(prompt.ptr());
    if (p < 0 || p / block_size >= len) throw py::index_error("a sequence has fewer cache blocks than tokens");
    TORCH_CHECK(len <= width, "a row of ", len, " numbers is longer than its room");
    for (ssize_t j = 0; j < len; ++j) {
      const long long v = number(PySequence_Fast_GET_ITEM(blocks.ptr(), j));
      TORCH_CHECK(v == (long long)(int32_t)v, v, " does not fit");
      row[j] = (int32_t)v;
    }
    at[i] = p;
    if (p < known) {
      id[i] = number(PySequence_Fast_GET_ITEM(prompt.ptr(), p));
    } else {
      const py::object more = fast(get(q, names[3]));
      if (p - known >= PySequence_Fast_GET_SIZE(more.ptr())) throw py::index_error("a sequence has no such token");
      id[i] = number(PySequence_Fast_GET_ITEM(more.ptr(), p - known));
    }
  }
}

// Cache slot and context length of a decode bucket's rows, from their positions and tables.
static void decode_slots(py::array_t<int64_t> positions, py::array_t<int32_t> tables, int64_t block_size,
                         py::array_t<int64_t> slots, py::array_t<int32_t> context) {
  const ssize_t n = positions.size();
  TORCH_CHECK(block_size > 0 && positions.ndim() == 1 && tables.ndim() == 2 && tables.shape(0) == n && slots.ndim() == 1 &&
              slots.shape(0) == n && context.ndim() == 1 && context.shape(0) == n);
  for (const py::array* a : {(py::array*)&positions, (py::array*)&tables, (py::array*)&slots, (py::array*)&context})
    TORCH_CHECK(a->flags() & py::array::c_style, "in row order");
  const int64_t* at = positions.data();
  const int32_t* row = tables.data();
  int64_t* slot = slots.mutable_data();
  int32_t* ctx = context.mutable_data();
  const ssize_t width = tables.shape(1);
  for (ssize_t i = 0; i < n; ++i, row += width) {
    const int64_t b = at[i] / block_size;
    if (at[i] < 0 || b >= width) throw py::index_error("a position past its row of blocks");
    slot[i] = row[b] * block_size + (at[i] - b * block_size);
    ctx[i] = (int32_t)(at[i] + 1);
  }
}

// lora/manager.py's tiles of a decode bucket: its rows by adapter slot (slot_of(name), -1
// for rows past the sequences), up to 16 a tile; the tiles past the last one empty.
// Returns their number.
static int64_t decode_lora_rows(py::list seqs, py::object slot_of, int64_t rows, py::array_t<int32_t> toks,
                                py::array_t<int32_t> len, py::array_t<int32_t> slot) {
  const ssize_t n = py::len(seqs), room = len.size();
  TORCH_CHECK(rows >= n && toks.ndim() == 2 && toks.shape(0) == room && toks.shape(1) == 16 && len.ndim() == 1 &&
              slot.ndim() == 1 && slot.shape(0) == room);
  for (const py::array* a : {(py::array*)&toks, (py::array*)&len, (py::array*)&slot})
    TORCH_CHECK(a->flags() & py::array::c_style, "in row order");
  static PyObject* name_attr = PyUnicode_InternFromString("lora_name");
  std::map<int, std::vector<int32_t>> by_slot;
  py::dict known;  // name -> slot, asked once per name
  for (ssize_t i = 0; i < n; ++i) {
    PyObject* v = PyObject_GetAttr(PyList_GET_ITEM(seqs.ptr(), i), name_attr);
    if (!v) throw py::error_already_set();
    const py::object name = py::reinterpret_steal<py::object>(v);
    PyObject* found = PyDict_GetItemWithError(known.ptr(), v);
    if (!found && PyErr_Occurred()) throw py::error_already_set();
    int at;
    if (found) {
      at = (int)PyLong_AsLong(found);
    } else {
      const int truth = PyObject_IsTrue(v);
      if (truth < 0) throw py::error_already_set();
      at = truth && !slot_of.is_none() ? slot_of(name).cast<int>() : -1;
      known[name] = at;
    }
    by_slot[at].push_back((int32_t)i);
  }
  for (ssize_t i = n; i < rows; ++i) by_slot[-1].push_back((int32_t)i);
  int32_t *tok = toks.mutable_data(), *l = len.mutable_data(), *s = slot.mutable_data();
  ssize_t t = 0;
  for (const auto& [at, of] : by_slot) {
    for (size_t first = 0; first < of.size(); first += 16, ++t) {
      TORCH_CHECK(t < room, "more tiles than room");
      const int m = (int)std::min<size_t>(16, of.size() - first);
      for (int j = 0; j < 16; ++j) tok[t * 16 + j] = of[first + std::min(j, m - 1)];
      l[t] = m;
      s[t] = at;
    }
  }
  const ssize_t used = t;
  for (; t < room; ++t) {
    std::fill(tok + t * 16, tok + t * 16 + 16, 0);
    l[t] = 0;
    s[t] = -1;
  }
  return used;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "MI355X (gfx950) native kernels for llm_instance_gateway_amd";
  m.def("rms_norm", &rms_norm);
  m.def("fused_add_rms_norm", &fused_add_rms_norm);
  m.def("rotary_embedding", &rotary_embedding);
  m.def("reshape_and_cache", &reshape_and_cache);
  m.def("qkv_rope_cache", &qkv_rope_cache);
  m.def("silu_and_mul", &silu_and_mul);
  m.def("argmax_rows", &argmax_rows);
  m.def("pack_decodes", &pack_decodes, py::arg("seqs"), py::arg("block_size"), py::arg("ids").noconvert(),
        py::arg("positions").noconvert(), py::arg("tables").noconvert());
  m.def("decode_slots", &decode_slots, py::arg("positions").noconvert(), py::arg("tables").noconvert(), py::arg("block_size"),
        py::arg("slots").noconvert(), py::arg("context").noconvert());
  m.def("decode_lora_rows", &decode_lora_rows, py::arg("seqs"), py::arg("slot_of"), py::arg("rows"), py::arg("toks").noconvert(),
        py::arg("len").noconvert(), py::arg("slot").noconvert());
  m.def("projection", &projection);
  m.def("projection_parts", &projection_parts);
  m.def("projection_plan", &projection_plan);
  m.def("projection_runs", &projection_runs);
  m.def("projection_serves", &lig_projection_serves);
  m.def("projection_pays", &lig_projection_pays);
  m.def("projection_takes", &projection_takes);
  m.def("projection_takes_rows", &projection_takes_rows);
  m.def("row_product", &row_product);
  m.def("row_product_heads", &row_product_heads);
  m.def("row_product_max", &lig_row_product_max);
  m.def("paged_attention_decode", &paged_attention_decode);
  m.def("paged_attention_decode_split", &paged_attention_decode_split<true>);
  m.def("paged_attention_decode_open", &paged_attention_decode_split<false>);
  m.def("paged_attention_prefill", &paged_attention_prefill);
  m.def("paged_attention_prefill_parts", &lig_paged_attention_prefill_parts);
  m.def("sgmv_shrink", &sgmv_shrink);
  m.def("sgmv_apply", &sgmv_apply);
  m.def("sgmv_apply_units", &sgmv_apply_units);
  m.def("sgmv_apply_tiled", &sgmv_apply_tiled);
  m.def("sgmv_expand", &sgmv_expand);
  m.def("quant_fp8_rowwise", &quant_fp8_rowwise);
  m.def("lora_rms_norm", &lora_rms_norm);
  m.def("lora_norm_open", &lora_norm_open);
  m.def("lora_silu", &lora_silu);
  m.def("lora_silu_strip", &lig_lora_silu_strip);
  m.def("lora_norm_strip", &lig_lora_norm_strip);
  m.def("lora_shrink_strip", &lig_lora_shrink_strip);
  m.def("lora_shrink", &lora_shrink);
  m.def("lora_qkv_rope_cache", &lora_qkv_rope_cache);
  m.def("pack_rows", &pack_rows);
  m.def("mfma_probe", [](torch::Tensor out, torch::Tensor a, torch::Tensor b,
                         int64_t stream) {
    TORCH_CHECK(out.scalar_type() == torch::kFloat32);
    lig_mfma_probe_launch(out.data_ptr<float>(), bf16_cptr(a), bf16_cptr(b),
                          as_stream(stream));
  });
}
