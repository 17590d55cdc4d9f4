// Sigmoid attention in 32 bits on the fp32 matrix cores: the rows kernel's arithmetic (sigmoid_attention.hip: fp32 scores, the
// library's functions, weights mixed in the order of the heads) for head widths in multiples of 16 up to 128, up to 32 heads
// and pages of a multiple of 16 tokens, all 16 bytes aligned.  Other shapes keep the rows kernel.
//
// A workgroup of eight waves has 16 query tokens of all heads (decode: a sequence's one row in every column, over a partition
// of 64 keys, for the rows kernel's combine); wave w has heads HW w ... HW w + HW - 1.  Per block of 16 keys
//     S^T[16 keys x 16 tokens] = K . Q^T, weights in fp32 -> LDS (lane (m, r): keys 4 r ... + 3 of token m, one 16-byte entry)
//     mixed[keys x tokens] of the wave's heads: the same entry of every head from LDS, on the vector units
//     O^T[16 channels x 16 tokens] += V^T . mixed^T   (V pages are channel-major; the mixed weights are where it wants them)
// The mix needs entries of the own lane only, so a block costs one barrier (two LDS buffers) and mixed weights stay in registers.
// Queries of more than one head of 128 channels per wave (two of 64) do not fit beside the sums: read again in every block.
//
// Bound: the fp32 matrix cores, 64 products of 32 cycles per head, block and 128 + 128 channels, and loads in front of them.
// A call in 32 bits, heads of 128, us, rows kernel / here: 8 + 2 heads, prompts of 4 x 512 tokens 4082 / 163, of 100 761 / 38,
// four rows over 512 keys 86 / 26; 24 + 8 heads, prompts of 2 x 700 8990 / 863, eight rows over 1500 keys 233 / 74; 32 + 8
// heads, 4 x 512 11743 / 941.  Error against 64 bits: 0.68 to 0.86 of the rows kernel's.
#include "mix_common.h"
#include "sigmoid_attention.h"

namespace mixk {
namespace sgf {

typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// dim <= 16 ND, vdim <= 16 ND, H <= 8 HW
template <int HW, int ND, bool DECODE>
__global__ void __launch_bounds__(512)
sigmoid_float_kernel(float* __restrict__ out, const float* __restrict__ q, const float* __restrict__ k_cache,
                     const float* __restrict__ v_cache, SigArgs a) {
  __shared__ f32x4 weights[2][8 * HW][kWave];
  const int lane = threadIdx.x & 63, m = lane & 15, r = lane >> 4, rep = a.H / a.G;
  const int h0 = HW * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nd = a.dim >> 4, nv = a.vdim >> 4, bs = a.block_size;
  int s, row, columns, qfirst, kbeg = 0, kend;
  if (DECODE) {
    s = blockIdx.x;
    row = a.seq_qstart[s];
    columns = 1;
    const int kvlen = a.seq_kvlen[s];
    qfirst = kvlen - 1;
    kbeg = blockIdx.y * kSgPart;
    kend = min(kvlen, kbeg + kSgPart);
    if (kbeg >= kend) return;
  } else {
    const int tile = blockIdx.x >> 2, qo = a.tile_qoff[tile] + 16 * (blockIdx.x & 3);
    s = a.tile_seq[tile];
    const int row0 = a.seq_qstart[s], n = a.seq_qstart[s + 1] - row0, kvlen = a.seq_kvlen[s];
    if (n <= 0 || kvlen <= 0 || qo >= n) return;
    columns = min(16, n - qo);
    row = row0 + qo;
    qfirst = kvlen - n + qo;
    kend = qfirst + columns;
  }
  const int col = min(m, columns - 1), qpos = qfirst + col;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  constexpr bool kHold = HW * ND <= 8;   // queries stay in registers, values are asked for ahead of the mix

  const float* qr = q + static_cast<int64_t>(row + col) * a.H * a.dim + 4 * r;
  f32x4 Q[kHold ? HW : 1][ND], O[HW][ND];
#pragma unroll
  for (int i = 0; i < HW; ++i)
#pragma unroll
    for (int t = 0; t < ND; ++t) {
      if (kHold) Q[i][t] = h0 + i < a.H && t < nd ? *reinterpret_cast<const f32x4*>(qr + (h0 + i) * a.dim + 16 * t) : zero;
      O[i][t] = zero;
    }
  const int* bt = a.block_tables + static_cast<int64_t>(s) * a.bt_width;
  int buf = 0;
#pragma unroll 1
  for (int k0 = kbeg; k0 < kend; k0 += 16, buf ^= 1) {
    const int64_t page = bt[k0 / bs];
    const int off = k0 % bs;
#pragma unroll
    for (int i = 0; i < HW; ++i) {
      const int h = h0 + i;
      if (h >= a.H) break;
      const float* kp = k_cache + ((page * a.G + h / rep) * bs + off + m) * a.dim + 4 * r;   // (a page's rows are all there)
      f32x4 K[ND], S[2] = {zero, zero};   // (two sums: a product waits for the one before the last)
#pragma unroll
      for (int t = 0; t < ND; ++t)
        if (t < nd) {
          K[t] = *reinterpret_cast<const f32x4*>(kp + 16 * t);
          if (!kHold) Q[0][t] = *reinterpret_cast<const f32x4*>(qr + h * a.dim + 16 * t);
        }
#pragma unroll
      for (int t = 0; t < ND; ++t)
        if (t < nd)
#pragma unroll
          for (int e = 0; e < 4; ++e) S[e & 1] = mma(K[t][e], Q[kHold ? i : 0][t][e], S[e & 1]);
      const float bias = a.bias[h];
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float z = (S[0][e] + S[1][e]) * a.scale;
        if (a.cap > 0.f) z = a.cap * tanhf(z / a.cap);
        x[e] = k0 + 4 * r + e <= qpos ? sigmoidf_(z + bias) : 0.f;   // (no position of a column is past kend)
      }
      weights[buf][h][lane] = x;
      if (!kHold) __builtin_amdgcn_sched_barrier(0);   // (loads of all heads at once do not fit)
    }
    f32x4 V[ND];
    auto values = [&](int h) {
      const float* vp = v_cache + ((page * a.G + h / rep) * a.vdim + m) * static_cast<int64_t>(bs) + off + 4 * r;
#pragma unroll
      for (int t = 0; t < ND; ++t)
        if (t < nv) V[t] = *reinterpret_cast<const f32x4*>(vp + static_cast<int64_t>(16 * t) * bs);
    };
    if (kHold && h0 < a.H) values(h0);
    lds_barrier();
    f32x4 p[HW];
#pragma unroll
    for (int i = 0; i < HW; ++i) p[i] = zero;
    if (h0 < a.H)
      for (int g = 0; g < a.H; ++g) {
        const f32x4 x = weights[buf][g][lane];
#pragma unroll
        for (int i = 0; i < HW; ++i) {
          const float f = a.talk[min(h0 + i, a.H - 1) * a.H + g];
#pragma unroll
          for (int e = 0; e < 4; ++e) p[i][e] = fmaf(f, x[e], p[i][e]);
        }
      }
#pragma unroll
    for (int i = 0; i < HW; ++i) {
      const int h = h0 + i;
      if (h >= a.H) break;
      if (!kHold) __builtin_amdgcn_sched_barrier(0);
      if (!kHold || i > 0) values(h);
      bool odd = false;
      if (k0 + 15 > qfirst) {   // the block of the last keys (uniform)
#pragma unroll
        for (int t = 0; t < ND; ++t)
          if (t < nv)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if (k0 + 4 * r + e >= kend) V[t][e] = 0.f;   // behind the last key: whatever is there
              odd |= !(fabsf(V[t][e]) < INFINITY);
            }
        odd = !DECODE && __ballot(odd) != 0;
      }
      if (!odd) {
#pragma unroll
        for (int t = 0; t < ND; ++t)
          if (t < nv)
#pragma unroll
            for (int e = 0; e < 4; ++e) O[i][t] = mma(V[t][e], p[i][e], O[i][t]);
        continue;
      }
      // infinities and NaN among the tokens' own keys: key by key, so that no earlier token gets 0 times one of them
#pragma unroll 1
      for (int key = 0; key < 16 && k0 + key < kend; ++key)
#pragma unroll
        for (int t = 0; t < ND; ++t)
          if (t < nv) {
            f32x4 x = zero;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const bool own = 4 * r + e == key;
              x = mma(own ? V[t][e] : 0.f, own ? p[i][e] : 0.f, x);
            }
            if (k0 + key <= qpos) O[i][t] += x;
          }
    }
  }
  if (m >= columns) return;
#pragma unroll
  for (int i = 0; i < HW; ++i) {
    const int h = h0 + i;
    if (h >= a.H) return;
    float* o = (DECODE ? a.part + ((static_cast<int64_t>(s) * a.H + h) * a.max_parts + blockIdx.y) * a.vdim
                       : out + (static_cast<int64_t>(row + m) * a.H + h) * a.vdim) + 4 * r;
#pragma unroll
    for (int t = 0; t < ND; ++t)
      if (t < nv) *reinterpret_cast<f32x4*>(o + 16 * t) = O[i][t];
  }
}

}  // namespace sgf

bool launch_sigmoid_float(void* out, const void* q, const void* k_cache, const void* v_cache, const SigArgs& a,
                          int num_tiles, int num_decode, int parts, hipStream_t st) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(a.part) |
                       reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache);
  if (a.dim % 16 != 0 || a.vdim % 16 != 0 || a.dim > 128 || a.vdim > 128 || a.block_size % 16 != 0 || a.H > 32 || at % 16 != 0)
    return false;
  auto go = [&](auto prompts, auto decode) {
    auto launch = [&](auto kernel, dim3 grid) {
      hipLaunchKernelGGL(kernel, grid, dim3(512), 0, st, static_cast<float*>(out), static_cast<const float*>(q),
                         static_cast<const float*>(k_cache), static_cast<const float*>(v_cache), a);
    };
    if (num_tiles > 0) launch(prompts, dim3(num_tiles * (kSgTile / 16)));
    if (num_decode > 0) launch(decode, dim3(num_decode, parts));
  };
#define MIXK_SG(HW, ND) go(sgf::sigmoid_float_kernel<HW, ND, false>, sgf::sigmoid_float_kernel<HW, ND, true>)
#define MIXK_SG_HEADS(ND)            \
  switch ((a.H + 7) / 8) {           \
    case 1: MIXK_SG(1, ND); break;   \
    case 2: MIXK_SG(2, ND); break;   \
    case 3: MIXK_SG(3, ND); break;   \
    default: MIXK_SG(4, ND); break;  \
  }
  if (a.dim <= 64 && a.vdim <= 64) {
    MIXK_SG_HEADS(4)
  } else {
    MIXK_SG_HEADS(8)
  }
#undef MIXK_SG_HEADS
#undef MIXK_SG
  return true;
}

}  // namespace mixk
