// Fused rotary embedding + paged KV-cache write (SURVEY §2.4 K4 + K5).
//
// One workgroup per token (decode-sized batches) or per 16-token tile (prefill, V staged
// through LDS for coalesced transposed stores).  Reads the packed QKV projection row once, applies
// neox-style (rotate-half) RoPE to q and k using a host-precomputed fp32 cos|sin table
// (llama3 frequency scaling is folded into that table on the host), writes rotated q to
// `q_out` and writes rotated k / raw v straight into the paged cache.
//
// Cache layouts (chosen for the MFMA attention kernels in attention.hip):
//   k_cache [num_blocks, n_kv_heads, block_size, head_dim]   (token rows contiguous)
//   v_cache [num_blocks, n_kv_heads, head_dim, block_size]   (transposed: a 16x16 V^T tile
//                                                             is the A operand of the PV MFMA)
// slot_mapping[t] (int32) = page * block_size + offset, or -1 to skip the cache write (padding).
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace atta {

template <typename T>
__global__ __launch_bounds__(256) void rope_cache_kernel(
    uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_cache, uint16_t* __restrict__ v_cache,
    const uint16_t* __restrict__ qkv, const int* __restrict__ positions,
    const int* __restrict__ slot_mapping, const float* __restrict__ cos_sin, int n_q_heads,
    int n_kv_heads, int head_dim, int block_size, int64_t qkv_stride, int64_t q_out_stride) {
  const int64_t t = blockIdx.x;
  const int64_t pos = positions[t];
  const int64_t slot = slot_mapping[t];
  const int half = head_dim >> 1;
  const int hv = half >> 3;      // 8-wide vectors per half head
  const int dv = head_dim >> 3;  // 8-wide vectors per full head
  const float* cs = cos_sin + pos * head_dim;
  const uint16_t* row = qkv + t * qkv_stride;
  const int nq = n_q_heads * hv;
  const int nk = n_kv_heads * hv;
  const int nv = n_kv_heads * dv;
  const int64_t page = slot >= 0 ? slot / block_size : 0;
  const int off = slot >= 0 ? static_cast<int>(slot % block_size) : 0;

  for (int task = threadIdx.x; task < nq + nk + nv; task += blockDim.x) {
    if (task < nq + nk) {
      const bool is_q = task < nq;
      const int local = is_q ? task : task - nq;
      const int h = local / hv;
      const int i0 = (local % hv) * 8;
      const uint16_t* src = row + (is_q ? h * head_dim : (n_q_heads + h) * head_dim);
      Pack8 a = *reinterpret_cast<const Pack8*>(src + i0);
      Pack8 b = *reinterpret_cast<const Pack8*>(src + i0 + half);
      Pack8 ra, rb;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float c = cs[i0 + j];
        const float s = cs[half + i0 + j];
        const float x1 = to_f32<T>(a.v[j]);
        const float x2 = to_f32<T>(b.v[j]);
        ra.v[j] = from_f32<T>(x1 * c - x2 * s);
        rb.v[j] = from_f32<T>(x2 * c + x1 * s);
      }
      if (is_q) {
        uint16_t* dst = q_out + t * q_out_stride + h * head_dim;
        *reinterpret_cast<Pack8*>(dst + i0) = ra;
        *reinterpret_cast<Pack8*>(dst + i0 + half) = rb;
      } else if (slot >= 0) {
        uint16_t* dst =
            k_cache + ((page * n_kv_heads + h) * static_cast<int64_t>(block_size) + off) * head_dim;
        *reinterpret_cast<Pack8*>(dst + i0) = ra;
        *reinterpret_cast<Pack8*>(dst + i0 + half) = rb;
      }
    } else if (slot >= 0) {
      const int local = task - nq - nk;
      const int h = local / dv;
      const int d0 = (local % dv) * 8;
      Pack8 a = *reinterpret_cast<const Pack8*>(row + (n_q_heads + n_kv_heads + h) * head_dim + d0);
      uint16_t* dst = v_cache + ((page * n_kv_heads + h) * static_cast<int64_t>(head_dim) + d0) *
                                    block_size + off;
#pragma unroll
      for (int j = 0; j < 8; ++j) dst[j * block_size] = a.v[j];
    }
  }
}

// 16-token tiles (prefill): one workgroup per (16 tokens, KV head) - the GQA group's q heads
// and the k head rotated as above, the head's V staged through LDS so the transposed V-cache
// stores are coalesced: lanes 16j..16j+15 write one dim's 16 consecutive token offsets (one
// 32-byte run when the tile's tokens fill one page) instead of the per-token kernel's 8
// single-element stores 32 B apart per lane.
constexpr int kRopeTile = 16;
template <typename T>
__global__ __launch_bounds__(256) void rope_cache_tile_kernel(
    uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_cache, uint16_t* __restrict__ v_cache,
    const uint16_t* __restrict__ qkv, const int* __restrict__ positions,
    const int* __restrict__ slot_mapping, const float* __restrict__ cos_sin, int num_tokens,
    int n_q_heads, int n_kv_heads, int head_dim, int block_size, int64_t qkv_stride,
    int64_t q_out_stride) {
  extern __shared__ uint16_t vtile[];  // [kRopeTile][head_dim + 2]
  __shared__ int s_slot[kRopeTile];
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kRopeTile;
  const int hk = blockIdx.y;
  const int nt = min(kRopeTile, static_cast<int>(num_tokens - t0));
  const int G = n_q_heads / n_kv_heads;
  const int half = head_dim >> 1;
  const int hv = half >> 3;              // 8-wide vectors per half head
  const int per_tok = (G + 1) * hv;      // q heads of the group + the k head
  const int ldw = head_dim + 2;          // padded LDS row (16 rows on distinct banks)
  const int dv = head_dim >> 3;
  if (threadIdx.x < kRopeTile) s_slot[threadIdx.x] = threadIdx.x < nt ? slot_mapping[t0 + threadIdx.x] : -1;
  const int64_t vcol = static_cast<int64_t>(n_q_heads + n_kv_heads + hk) * head_dim;
  for (int e = threadIdx.x; e < nt * dv; e += blockDim.x) {
    const int i = e / dv, c = e - i * dv;
    const Pack8 a = *reinterpret_cast<const Pack8*>(qkv + (t0 + i) * qkv_stride + vcol + c * 8);
    uint16_t* d = vtile + i * ldw + c * 8;
#pragma unroll
    for (int j = 0; j < 8; j += 2)  // 4-byte LDS stores (the padded row is 4-byte aligned)
      *reinterpret_cast<uint32_t*>(d + j) = static_cast<uint32_t>(a.v[j]) |
                                            (static_cast<uint32_t>(a.v[j + 1]) << 16);
  }
  for (int task = threadIdx.x; task < nt * per_tok; task += blockDim.x) {
    const int i = task / per_tok, local = task - i * per_tok;
    const int64_t t = t0 + i;
    const int hh = local / hv;
    const int i0 = (local - hh * hv) * 8;
    const bool is_q = hh < G;
    const int slot = slot_mapping[t];
    if (!is_q && slot < 0) continue;
    const int head = is_q ? hk * G + hh : n_q_heads + hk;  // column block in the qkv row
    const float* cs = cos_sin + static_cast<int64_t>(positions[t]) * head_dim;
    const uint16_t* src = qkv + t * qkv_stride + static_cast<int64_t>(head) * head_dim;
    const Pack8 a = *reinterpret_cast<const Pack8*>(src + i0);
    const Pack8 b = *reinterpret_cast<const Pack8*>(src + i0 + half);
    Pack8 ra, rb;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float c = cs[i0 + j];
      const float sn = cs[half + i0 + j];
      const float x1 = to_f32<T>(a.v[j]);
      const float x2 = to_f32<T>(b.v[j]);
      ra.v[j] = from_f32<T>(x1 * c - x2 * sn);
      rb.v[j] = from_f32<T>(x2 * c + x1 * sn);
    }
    uint16_t* dst = is_q ? q_out + t * q_out_stride + static_cast<int64_t>(head) * head_dim
                         : k_cache + ((static_cast<int64_t>(slot / block_size) * n_kv_heads + hk) *
                                          block_size + slot % block_size) * head_dim;
    *reinterpret_cast<Pack8*>(dst + i0) = ra;
    *reinterpret_cast<Pack8*>(dst + i0 + half) = rb;
  }
  __syncthreads();
  // transposed V writes: element f -> token f & 15, dim f >> 4
  for (int f = threadIdx.x; f < kRopeTile * head_dim; f += blockDim.x) {
    const int i = f & (kRopeTile - 1);
    const int d = f >> 4;
    const int slot = s_slot[i];
    if (slot < 0) continue;  // also tokens past the end (s_slot = -1)
    v_cache[((static_cast<int64_t>(slot / block_size) * n_kv_heads + hk) * head_dim + d) *
                block_size + slot % block_size] = vtile[i * ldw + d];
  }
}

// The same for heads of 128 and a group of G query heads known here: a thread has one token and 8 + 8 of a head's channels
// throughout, so all of its rows, its V and its 16 numbers of the table are loaded before any is used (above, every task's
// loads wait for its token's position), and the pages' addresses are worked out once per token.
// Workgroups of a tile's KV heads are neighbours, so that a token's row is read at one time.
// Bound: memory traffic.  Llama layer of 7580 tokens, 32 + 8 + 8 heads (186 MB in 33 us; a copy of as many bytes takes 26 us
// between buffers that stay in the 256 MB cache, 36 from and to memory): tiles 169.9 us, here 165.7, KV heads side by side
// 164.2.
template <typename T, int G>
__global__ __launch_bounds__(256) void rope_cache_group_kernel(
    uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_cache, uint16_t* __restrict__ v_cache,
    const uint16_t* __restrict__ qkv, const int* __restrict__ positions,
    const int* __restrict__ slot_mapping, const float* __restrict__ cos_sin, int num_tokens,
    int n_kv_heads, int block_size, int64_t qkv_stride, int64_t q_out_stride) {
  constexpr int kDim = 128, kHalf = kDim / 2, N = (G + 2) / 2;   // N: heads of a thread, the k head after the query heads
  typedef __attribute__((ext_vector_type(4))) float f32x4_t;
  __shared__ uint32_t vtile[kRopeTile][kDim / 2 + 1];   // 16-bit numbers, rows on distinct banks
  __shared__ int64_t v_at[kRopeTile];
  const int64_t t0 = static_cast<int64_t>(blockIdx.x / n_kv_heads) * kRopeTile;
  const int hk = blockIdx.x % n_kv_heads, i = threadIdx.x >> 4, c = threadIdx.x & 15, n_q_heads = G * n_kv_heads;
  const bool live = t0 + i < num_tokens;
  const int64_t t = live ? t0 + i : num_tokens - 1;
  const int pos = positions[t], slot = live ? slot_mapping[t] : -1;
  const int i0 = (c & 7) * 8, first = c >> 3;   // heads first, first + 2 ...
  const uint16_t* row = qkv + t * qkv_stride;
  auto column = [&](int n) {
    const int h = min(2 * n + first, G);
    return static_cast<int64_t>(h < G ? hk * G + h : n_q_heads + hk) * kDim + i0;
  };
  Pack8 a[N], b[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    a[n] = *reinterpret_cast<const Pack8*>(row + column(n));
    b[n] = *reinterpret_cast<const Pack8*>(row + column(n) + kHalf);
  }
  const Pack8 v = *reinterpret_cast<const Pack8*>(row + static_cast<int64_t>(n_q_heads + n_kv_heads + hk) * kDim + c * 8);
  float cs[8], sn[8];
  const float* table = cos_sin + static_cast<int64_t>(pos) * kDim + i0;
#pragma unroll
  for (int j = 0; j < 8; j += 4) {
    const f32x4_t x = *reinterpret_cast<const f32x4_t*>(table + j), y = *reinterpret_cast<const f32x4_t*>(table + kHalf + j);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      cs[j + e] = x[e];
      sn[j + e] = y[e];
    }
  }
  const int64_t page = slot >= 0 ? static_cast<int64_t>(slot / block_size) * n_kv_heads + hk : 0;
  const int off = slot >= 0 ? slot % block_size : 0;
  if (c == 0) v_at[i] = slot >= 0 ? page * kDim * block_size + off : -1;
#pragma unroll
  for (int j = 0; j < 8; j += 2)
    vtile[i][c * 4 + j / 2] = static_cast<uint32_t>(v.v[j]) | (static_cast<uint32_t>(v.v[j + 1]) << 16);
#pragma unroll
  for (int n = 0; n < N; ++n) {
    Pack8 ra, rb;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float x1 = to_f32<T>(a[n].v[j]), x2 = to_f32<T>(b[n].v[j]);
      ra.v[j] = from_f32<T>(x1 * cs[j] - x2 * sn[j]);
      rb.v[j] = from_f32<T>(x2 * cs[j] + x1 * sn[j]);
    }
    const int h = 2 * n + first;
    uint16_t* dst = nullptr;
    if (h < G && live) dst = q_out + t * q_out_stride + static_cast<int64_t>(hk * G + h) * kDim;
    else if (h == G && slot >= 0) dst = k_cache + (page * block_size + off) * kDim;
    if (dst != nullptr) {
      *reinterpret_cast<Pack8*>(dst + i0) = ra;
      *reinterpret_cast<Pack8*>(dst + i0 + kHalf) = rb;
    }
  }
  __syncthreads();
  // V: 16 lanes write one channel's 16 tokens
  const int64_t at = v_at[c];
  if (at < 0) return;
  const uint16_t* from = reinterpret_cast<const uint16_t*>(vtile[c]);
#pragma unroll
  for (int d = 0; d < kDim; d += 16)
    v_cache[at + static_cast<int64_t>(d + i) * block_size] = from[d + i];
}

}  // namespace atta

using namespace atta;

int atta_rope_cache(void* q_out, void* k_cache, void* v_cache, const void* qkv,
                    const int* positions, const int* slot_mapping, const float* cos_sin,
                    int num_tokens, int n_q_heads, int n_kv_heads, int head_dim, int block_size,
                    int64_t qkv_stride, int64_t q_out_stride, int dtype, hipStream_t stream) {
  if (head_dim % 16 != 0) return -1;
  if (num_tokens == 0) return 0;
  auto qo = static_cast<uint16_t*>(q_out);
  auto kc = static_cast<uint16_t*>(k_cache);
  auto vc = static_cast<uint16_t*>(v_cache);
  auto in = static_cast<const uint16_t*>(qkv);
  const size_t lds = static_cast<size_t>(kRopeTile) * (head_dim + 2) * 2;
  if (num_tokens >= kRopeTile && n_q_heads % n_kv_heads == 0 && qkv_stride % 8 == 0) {
    dim3 g((num_tokens + kRopeTile - 1) / kRopeTile, n_kv_heads), b(256);
    const uintptr_t at = reinterpret_cast<uintptr_t>(q_out) | reinterpret_cast<uintptr_t>(k_cache) |
                         reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(cos_sin);
    if (head_dim == 128 && at % 16 == 0 && q_out_stride % 8 == 0) {
      auto launch = [&](auto group) {
        constexpr int G = decltype(group)::value;
        auto go = [&](auto kernel) {
          hipLaunchKernelGGL(kernel, dim3(g.x * n_kv_heads), b, 0, stream, qo, kc, vc, in, positions, slot_mapping, cos_sin, num_tokens,
                             n_kv_heads, block_size, qkv_stride, q_out_stride);
        };
        if (dtype == 0) go(rope_cache_group_kernel<__bf16, G>);
        else go(rope_cache_group_kernel<_Float16, G>);
        return static_cast<int>(hipGetLastError());
      };
      switch (n_q_heads / n_kv_heads) {   // (other groups: the kernel for any)
        case 1: return launch(std::integral_constant<int, 1>{});
        case 2: return launch(std::integral_constant<int, 2>{});
        case 3: return launch(std::integral_constant<int, 3>{});
        case 4: return launch(std::integral_constant<int, 4>{});
        case 8: return launch(std::integral_constant<int, 8>{});
      }
    }
    if (dtype == 0)
      rope_cache_tile_kernel<__bf16><<<g, b, lds, stream>>>(
          qo, kc, vc, in, positions, slot_mapping, cos_sin, num_tokens, n_q_heads, n_kv_heads,
          head_dim, block_size, qkv_stride, q_out_stride);
    else
      rope_cache_tile_kernel<_Float16><<<g, b, lds, stream>>>(
          qo, kc, vc, in, positions, slot_mapping, cos_sin, num_tokens, n_q_heads, n_kv_heads,
          head_dim, block_size, qkv_stride, q_out_stride);
    return static_cast<int>(hipGetLastError());
  }
  dim3 grid(num_tokens), block(256);
  if (dtype == 0)
    rope_cache_kernel<__bf16><<<grid, block, 0, stream>>>(qo, kc, vc, in, positions, slot_mapping,
                                                          cos_sin, n_q_heads, n_kv_heads, head_dim,
                                                          block_size, qkv_stride, q_out_stride);
  else
    rope_cache_kernel<_Float16><<<grid, block, 0, stream>>>(
        qo, kc, vc, in, positions, slot_mapping, cos_sin, n_q_heads, n_kv_heads, head_dim,
        block_size, qkv_stride, q_out_stride);
  return static_cast<int>(hipGetLastError());
}
