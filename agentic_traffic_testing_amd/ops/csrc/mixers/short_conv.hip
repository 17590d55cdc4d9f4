// Short causal convolution over time, per channel, followed by SiLU, on ragged batches of
// portions with the last taps - 1 inputs of every sequence carried in its state slot.
//
//   y[t, c] = silu(b[c] + sum_j w[c, j] * x[t - (taps - 1) + j, c]),  x = 0 before position 0
// (the bias b is optional).
//
// Inputs before the portion's first row come from conv_state[slot, taps - 1, C] - but only where their position is
// >= 0, so a slot's stale contents never reach a sequence that starts at position 0.  Channels in multiples of 8 at
// aligned addresses: one kernel for the convolution and the new tails (below).  Others: an element-wise kernel, grid
// (rows, channel blocks), and a second one after it on the same stream that reads old tail and portion, then writes.
#include "mix_common.h"
#include "mixers.h"

namespace mixk {

constexpr int kMaxTaps = 8;

template <typename T>
__global__ void short_conv_silu_kernel(T* __restrict__ out, const T* __restrict__ x,
                                       int64_t x_stride, const T* __restrict__ w,
                                       const T* __restrict__ bias,
                                       const T* __restrict__ conv_state,
                                       const int* __restrict__ positions,
                                       const int* __restrict__ seq_qstart,
                                       const int* __restrict__ seq_slot, int S, int C, int taps) {
  __shared__ int sh[2];
  const int r = blockIdx.x;
  if (threadIdx.x == 0) {
    const int s = seq_of_row(seq_qstart, S, r);
    sh[0] = s < 0 ? -1 : seq_slot[s];
    sh[1] = s < 0 ? 0 : seq_qstart[s];
  }
  __syncthreads();
  const int slot = sh[0], first = sh[1];
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  T* o = out + static_cast<int64_t>(r) * C + c;
  if (slot < 0) {
    stf(o, 0.f);
    return;
  }
  const int pos = positions[r];
  const int j = r - first;  // row index inside the portion
  float acc = bias != nullptr ? ldf(bias + c) : 0.f;
  for (int t = 0; t < taps; ++t) {
    const int back = taps - 1 - t;        // how many tokens before this row
    if (pos - back < 0) continue;
    float xv;
    if (j - back >= 0) {
      xv = ldf(x + (r - back) * x_stride + c);
    } else {
      // tail entry u holds the input (taps - 1 - u) tokens before the portion's first row
      const int u = (taps - 1) + (j - back);
      xv = ldf(conv_state + (static_cast<int64_t>(slot) * (taps - 1) + u) * C + c);
    }
    acc += ldf(w + static_cast<int64_t>(c) * taps + t) * xv;
  }
  stf(o, siluf_(acc));
}

// Sixteen bytes at a time, the state's update included: a workgroup takes up to ROWS rows of one portion, a
// thread 8 channels of them, with the last TAPS - 1 inputs in registers as it walks down the rows, up to 8 rows of loads
// ahead.  Only a portion's first workgroup reads its state slot (ROWS >= TAPS - 1), so the same threads write
// the new tail: no second launch, no order between workgroups.
//
// Workgroup -> portion without a host plan: with `at(k)` the first row of portion k, portion k owns the workgroups
// from at(k) / ROWS + k on; there are at least ceil(n / ROWS) of them.  Portion 0 stands for the rows
// before the first sequence and portion S + 1 for those after the last one (zeros, as for padding sequences).
//
// Bound: one read and one write of the rows; the SiLU's arithmetic (library functions: 35 of 45 instructions per result,
// 52 us in the first line).  Measured, before (8 rows per workgroup, every tap loaded again, a second launch for the
// tails) -> now: 7580 rows of 6144 channels in bf16 125 -> 43 us (copy: 38); 1023 rows of 8448 in fp32 87 -> 20 (14);
// 16 decode rows 13 -> 5.
//
// A thread takes its rows one after the other, about 0.5 us each, so batches that do not fill the chip have workgroups of
// 4 rows (8 where a tail is longer).  16 rows / 4 rows, us, 6144 channels in bf16: 64 rows 9.4 / 7.1, 1024 10.9 / 9.0, 2048
// 17.2 / 14.0, 4096 (768 workgroups of 16) 23.1 / 24.0, 8000 40.0 / 42.0; 8448 in fp32: 64 13.0 / 7.3, 2048 35.6 / 33.7,
// 4096 61.6 / 60.8, 6000 92 / 104.
// In 32 bits, from 480 workgroups on (two per CU) now one and now the other is faster, and 16 rows are kept: 2048 channels,
// 4 x 2000 rows 28.1 / 30.9, 8192 29.8 / 31.4, 12000 38.9 / 43.4; 4096 channels, 4096 rows 29.7 / 32.7, 16 x 256 35.5 / 32.4.
constexpr int kConvRows = 16;
constexpr int conv_few(size_t item) { return item == 4 ? 480 : 768; }   // workgroups

template <typename T, int TAPS, int ROWS>
__global__ void __launch_bounds__(256)
short_conv_rows_kernel(T* __restrict__ out, const T* __restrict__ x, int64_t x_stride, const T* __restrict__ w,
                       const T* __restrict__ bias, T* __restrict__ conv_state, const int* __restrict__ positions,
                       const int* __restrict__ seq_qstart, const int* __restrict__ seq_slot, int T_, int S, int C) {
  constexpr int KEEP = TAPS - 1, NH = KEEP > 0 ? KEEP : 1, AHEAD = ROWS < 8 ? ROWS : 8;
  static_assert(KEEP <= AHEAD, "only a portion's first workgroup reads the state");
  const int b = blockIdx.x, lane = threadIdx.x & 63;
  // the last portion whose first workgroup is not after b (every wave looks, 64 portions at a time)
  int k = -1, first = 0;
  for (int k0 = 0; k0 <= S + 1; k0 += kWave) {
    const int i = k0 + lane, at = i == 0 || i > S + 1 ? 0 : seq_qstart[i - 1];
    const uint64_t m = __ballot(i <= S + 1 && at / ROWS + i <= b);
    if (m == 0) break;
    const int top = 63 - __builtin_clzll(m);
    k = k0 + top;
    first = __builtin_amdgcn_readlane(at, top);
    if (m != ~0ull) break;
  }
  const int end = k <= S ? seq_qstart[k] : T_;
  const int n = end - first, j0 = (b - (first / ROWS + k)) * ROWS;   // row of the portion
  if (j0 >= n) return;
  const int c = (blockIdx.y * 256 + threadIdx.x) * 8;
  if (c >= C) return;
  const int slot = k >= 1 && k <= S ? seq_slot[k - 1] : -1;
  const int rows = min(ROWS, n - j0), r0 = first + j0;
  T* o = out + static_cast<int64_t>(r0) * C + c;
  if (slot < 0) {
    const float zero[8] = {};
    for (int j = 0; j < rows; ++j) st8(o + static_cast<int64_t>(j) * C, zero);
    return;
  }
  const T* xr = x + r0 * x_stride + c;
  const int pos = positions[r0];
  T* tail = conv_state + static_cast<int64_t>(slot) * KEEP * C + c;
  float xv[AHEAD][8], hist[NH][8], wv[TAPS * 8], bv[8];   // hist[u]: the input KEEP - u tokens before the row
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) ld8(xr + min(j, rows - 1) * x_stride, xv[j]);
#pragma unroll
  for (int u = 0; u < KEEP; ++u) ld8(j0 == 0 ? tail + static_cast<int64_t>(u) * C : xr + (u - KEEP) * x_stride, hist[u]);
#pragma unroll
  for (int t = 0; t < TAPS; ++t) ld8(w + static_cast<int64_t>(c) * TAPS + 8 * t, wv + 8 * t);   // [channel][tap]
#pragma unroll
  for (int e = 0; e < 8; ++e) bv[e] = 0.f;
  if (bias != nullptr) ld8(bias + c, bv);
#pragma unroll
  for (int u = 0; u < KEEP; ++u)   // before position 0: nothing, whatever the slot holds
    if (pos - KEEP + u < 0)
#pragma unroll
      for (int e = 0; e < 8; ++e) hist[u][e] = 0.f;
  if (KEEP > 0 && j0 == 0) {
    // new tail entry u = element n + u of [old tail (KEEP entries), portion (n rows)]
    float nv[NH][8];
#pragma unroll
    for (int u = 0; u < KEEP; ++u) ld8(x + (first + max(n + u - KEEP, 0)) * x_stride + c, nv[u]);
#pragma unroll
    for (int u = 0; u < KEEP; ++u) {
#pragma unroll
      for (int i = u + 1; i < KEEP; ++i)
        if (n + u == i)
#pragma unroll
          for (int e = 0; e < 8; ++e) nv[u][e] = hist[i][e];
      st8(tail + static_cast<int64_t>(u) * C, nv[u]);
    }
  }
  for (int j = 0; j < rows; j += AHEAD) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      if (j + i >= rows) break;
      float acc[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = bv[e];
#pragma unroll
      for (int t = 0; t < TAPS; ++t) {
        if (pos < KEEP && pos + j + i - (KEEP - t) < 0) continue;   // no product with an input that does not exist
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += wv[e * TAPS + t] * (t + i < KEEP ? hist[(t + i) % NH][e] : xv[t + i - KEEP < 0 ? 0 : t + i - KEEP][e]);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = gate_silu<T>(acc[e]);
      st8(o + static_cast<int64_t>(j + i) * C, acc);
    }
    if (ROWS <= AHEAD || j + AHEAD >= rows) break;
#pragma unroll
    for (int u = 0; u < KEEP; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) hist[u][e] = xv[AHEAD - KEEP + u][e];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) ld8(xr + min(j + AHEAD + i, rows - 1) * x_stride, xv[i]);
  }
}

template <typename T>
int launch_conv_rows(T* out, const T* x, int64_t x_stride, const T* w, const T* bias, T* conv_state,
                     const int* positions, const int* seq_qstart, const int* seq_slot, int T_, int S, int C, int taps,
                     hipStream_t st) {
  const unsigned cols = (C / 8 + 255) / 256;
  const bool few = (static_cast<int64_t>(T_) / kConvRows + S) * cols < conv_few(sizeof(T));
  const dim3 grid(T_ / (few ? (taps <= 5 ? 4 : 8) : kConvRows) + S + 2, cols);
#define MIXK_TAPS(N)                                                                                                \
  case N:                                                                                                           \
    if (few)                                                                                                        \
      hipLaunchKernelGGL((short_conv_rows_kernel<T, N, (N <= 5 ? 4 : 8)>), grid, dim3(256), 0, st, out, x, x_stride, \
                         w, bias, conv_state, positions, seq_qstart, seq_slot, T_, S, C);                           \
    else                                                                                                            \
      hipLaunchKernelGGL((short_conv_rows_kernel<T, N, kConvRows>), grid, dim3(256), 0, st, out, x, x_stride, w,    \
                         bias, conv_state, positions, seq_qstart, seq_slot, T_, S, C);                              \
    break;
  switch (taps) {
    MIXK_TAPS(1) MIXK_TAPS(2) MIXK_TAPS(3) MIXK_TAPS(4) MIXK_TAPS(5) MIXK_TAPS(6) MIXK_TAPS(7) MIXK_TAPS(8)
  }
#undef MIXK_TAPS
  return static_cast<int>(hipGetLastError());
}

template <typename T>
__global__ void conv_state_update_kernel(const T* __restrict__ x, int64_t x_stride,
                                         T* __restrict__ conv_state,
                                         const int* __restrict__ positions,
                                         const int* __restrict__ seq_qstart,
                                         const int* __restrict__ seq_slot, int C, int taps) {
  const int s = blockIdx.x;
  const int slot = seq_slot[s];
  const int first = seq_qstart[s], n = seq_qstart[s + 1] - first;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (slot < 0 || n <= 0 || c >= C) return;
  const int start = positions[first];
  const int keep = taps - 1;
  T* tail = conv_state + static_cast<int64_t>(slot) * keep * C + c;
  float nv[kMaxTaps];
  for (int u = 0; u < keep; ++u) {
    // new tail entry u = element n + u of [old tail (keep entries), portion (n rows)]
    const int i = n + u;
    if (i >= keep) {
      nv[u] = ldf(x + (first + i - keep) * x_stride + c);
    } else {
      // old tail entry i is the input at position start - keep + i
      nv[u] = start - keep + i >= 0 ? ldf(tail + static_cast<int64_t>(i) * C) : 0.f;
    }
  }
  for (int u = 0; u < keep; ++u) stf(tail + static_cast<int64_t>(u) * C, nv[u]);
}

}  // namespace mixk

using namespace mixk;

extern "C" int mixk_short_conv_silu(void* out, const void* x, int64_t x_stride, const void* w,
                                    const void* bias, void* conv_state, const int* positions, const int* seq_qstart,
                                    const int* seq_slot, int T_, int S, int C, int taps, int dtype,
                                    hipStream_t st) {
  if (T_ <= 0 || S <= 0) return 0;
  if (taps < 1 || taps > kMaxTaps) return -1;
  const int cb = (C + 255) / 256;
  const uintptr_t at = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out) |
                       reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(bias) |
                       reinterpret_cast<uintptr_t>(conv_state);
  const bool vec = C % 8 == 0 && x_stride % 8 == 0 && at % 16 == 0;
  MIXK_DISPATCH(dtype, {
    if (vec)
      return launch_conv_rows<T>(static_cast<T*>(out), static_cast<const T*>(x), x_stride, static_cast<const T*>(w),
                                 static_cast<const T*>(bias), static_cast<T*>(conv_state), positions, seq_qstart,
                                 seq_slot, T_, S, C, taps, st);
    hipLaunchKernelGGL(short_conv_silu_kernel<T>, dim3(T_, cb), dim3(256), 0, st,
                       static_cast<T*>(out), static_cast<const T*>(x), x_stride, static_cast<const T*>(w),
                       static_cast<const T*>(bias), static_cast<const T*>(conv_state), positions, seq_qstart,
                       seq_slot, S, C, taps);
    if (taps > 1)
      hipLaunchKernelGGL(conv_state_update_kernel<T>, dim3(S, cb), dim3(256), 0, st,
                         static_cast<const T*>(x), x_stride, static_cast<T*>(conv_state),
                         positions, seq_qstart, seq_slot, C, taps);
  });
  return static_cast<int>(hipGetLastError());
}
