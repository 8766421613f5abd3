// Greedy sampling, gfx950: the place of a row's largest value, rows of bf16 or
// fp32 logits [N, V] -> int64 [N].  The first of equals; a NaN counts as the
// largest (torch.argmax's order).
//
// Bound by one pass over the logits: 384 rows of 128256 bf16 are 98 MB.  A
// workgroup of 16 waves takes a row, 16 bytes a lane and load.  Per 16 bytes
// only the largest value is formed and compared with the best so far (3 ops a
// value); the place inside the winning 16 bytes is looked up at the end.
// 384 rows 23 us (4.3 TB/s; 25 in an engine step), one row 8.7 (11); torch's
// reduction after a conversion to fp32 took 104 and 39, without it 59 and 31.
#include "common.h"

namespace {

constexpr int NT = 1024;

template <typename E>
struct Vec;
template <>
struct Vec<uint16_t> {
  static constexpr int N = 8;
  static LIG_DEVICE float value(uint16_t x) { return bf16_to_f32(x); }
};
template <>
struct Vec<float> {
  static constexpr int N = 4;
  static LIG_DEVICE float value(float x) { return x; }
};

template <typename E>
__global__ __launch_bounds__(NT) void argmax_rows_kernel(const E* __restrict__ x, const long stride, const int V,
                                                         int64_t* __restrict__ out) {
  constexpr int N = Vec<E>::N;
  typedef E vec __attribute__((ext_vector_type(N)));
  __shared__ float best_s[NT / WAVE_SIZE];
  __shared__ int at_s[NT / WAVE_SIZE], nan_s[NT / WAVE_SIZE];
  const E* row = x + blockIdx.x * stride;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // whole vectors from the first aligned place on, single values around them
  const int head = min(V, (int)((16 - ((uintptr_t)row & 15)) & 15) / (int)sizeof(E));
  const int nvec = (V - head) / N;
  const vec* body = reinterpret_cast<const vec*>(row + head);

  float best = -INFINITY;
  int at = -1;   // place of `best`; -1: nothing above -inf seen
  bool nan = false;
  auto one = [&](int i) __attribute__((always_inline)) {
    const float v = Vec<E>::value(row[i]);
    nan |= v != v;
    if (v > best || (v == best && i < at)) best = v, at = i;
  };
  if (tid < head) one(tid);
  int group = -1;
#pragma unroll 4
  for (int g = tid; g < nvec; g += NT) {
    const vec u = body[g];
    float m = Vec<E>::value(u[0]);
    bool bad = m != m;
#pragma unroll
    for (int e = 1; e < N; ++e) {
      const float v = Vec<E>::value(u[e]);
      bad |= v != v;
      m = fmaxf(m, v);
    }
    nan |= bad;
    if (m > best) best = m, group = g;
  }
  if (group >= 0) {
    const vec u = body[group];
    for (int e = N - 1; e >= 0; --e)
      if (Vec<E>::value(u[e]) == best) at = head + group * N + e;
  }
  const int tail = head + nvec * N + tid;
  if (tail < V) one(tail);

  // a value that was found beats none; then the larger; then the earlier
  auto take = [&](float b, int a) __attribute__((always_inline)) {
    if (a >= 0 && (at < 0 || b > best || (b == best && a < at))) best = b, at = a;
  };
#pragma unroll
  for (int d = 32; d; d >>= 1) take(__shfl_xor(best, d, WAVE_SIZE), __shfl_xor(at, d, WAVE_SIZE));
  const int any_nan = __any(nan);
  if (lane == 0) best_s[wave] = best, at_s[wave] = at, nan_s[wave] = any_nan;
  __syncthreads();
  int found = 0;
  for (int w = 0; w < NT / WAVE_SIZE; ++w) found |= nan_s[w];
  if (found) {  // rare: the first NaN of the row
    __syncthreads();
    int first = V;
    for (int i = tid; i < V; i += NT) {
      const float v = Vec<E>::value(row[i]);
      if (v != v && i < first) first = i;
    }
#pragma unroll
    for (int d = 32; d; d >>= 1) first = min(first, __shfl_xor(first, d, WAVE_SIZE));
    if (lane == 0) at_s[wave] = first;
    __syncthreads();
    if (tid == 0) {
      for (int w = 0; w < NT / WAVE_SIZE; ++w) first = min(first, at_s[w]);
      out[blockIdx.x] = first;
    }
    return;
  }
  if (tid == 0) {
    for (int w = 1; w < NT / WAVE_SIZE; ++w) take(best_s[w], at_s[w]);
    out[blockIdx.x] = max(at, 0);  // a row of nothing but -inf: its first place
  }
}

}  // namespace

extern "C" void lig_argmax_rows_launch(const void* x, bool bf16, long stride, int rows, int V, int64_t* out, hipStream_t stream) {
  if (rows == 0) return;
  if (bf16)
    hipLaunchKernelGGL(argmax_rows_kernel<uint16_t>, dim3(rows), dim3(NT), 0, stream, (const uint16_t*)x, stride, V, out);
  else
    hipLaunchKernelGGL(argmax_rows_kernel<float>, dim3(rows), dim3(NT), 0, stream, (const float*)x, stride, V, out);
}
