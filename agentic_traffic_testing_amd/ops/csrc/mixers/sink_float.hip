// Softmax attention in 32 bits on the fp32 matrix cores: the rows kernel's arithmetic (sink_attention.hip: fp32 scores, weights
// and sums, the library's exponential) for head widths in multiples of 16 up to 256 and pages of a multiple of 16 tokens, all
// 16 bytes aligned.  Other shapes keep the rows kernel.
//
// A workgroup has 16 columns: query tokens of one head, or, decode, the query heads of a KV head for a sequence's one row and
// a partition of its keys (the rows kernel's, for the same join).  Its four waves take every fourth block of 16 keys each,
// straight from the pages (a block lies in one page), and put their sums together at the end.  Per block
//     S^T[16 keys x 16 columns] = K . Q^T    (16x16x4 products; Q in registers; lane (m, r) holds channels 16 t + 4 r ... + 3
//                                             of key or column m, four products per 16-byte load)
//     O^T[16 channels x 16 columns] += V^T . P^T   (V pages are channel-major: lane (m, r) loads keys 4 r ... + 3 of channel m,
//                                             and the weights are already where the second operand wants them)
// so weights never leave registers, a column's statistics are one lane's and three others', and nothing goes through LDS.
//
// Bound: the fp32 matrix cores (64 products of 32 cycles per block of 128 + 128 channels) and one block's loads per wave in
// flight.  A layer's call in 32 bits, us, rows kernel / here (prompts of 4 x 512 tokens; a prompt of 100; 4 rows over 512 keys):
//     sinks 816 / 83, 128 / 27, 120 / 27;  windows 804 / 82, 133 / 29, 117 / 26;
//     latent (256 and 192 channels) 1392 / 189, 210 / 29, 188 / 31;  two maps 907 / 108, 99 / 26, 91 / 25.
// (25 us of each are the host's: a call's time and not its kernel's.)  Error against 64 bits: 0.6 to 0.97 of the rows kernel's.
#include "mix_common.h"
#include "sink_attention.h"

namespace mixk {
namespace sfl {

typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// dim <= 16 ND, vdim <= 16 NV
template <int ND, int NV, bool DECODE>
__global__ void __launch_bounds__(256)
sink_float_kernel(float* __restrict__ out, const float* __restrict__ q, const float* __restrict__ k_cache,
                  const float* __restrict__ v_cache, AttnArgs a) {
  __shared__ f32x4 sums[3][NV][kWave];
  __shared__ float stats[4][2][16];
  const int lane = threadIdx.x & 63, m = lane & 15, r = lane >> 4, rep = a.H / a.G;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // column c: row0 + step c of q and, decode, head h0 + c; keys [klo, kkeep) and [kbeg, kend) are seen by somebody
  int s, g, h0, row, columns, qpos, klo = 0, kbeg, kend;
  if (DECODE) {
    const int hb = (rep + 15) / 16;
    s = blockIdx.x;
    g = blockIdx.y / hb;
    h0 = g * rep + (blockIdx.y % hb) * 16;
    columns = min(16, (g + 1) * rep - h0);
    row = a.seq_qstart[s];
    const int kvlen = a.seq_kvlen[s], z = blockIdx.z;
    if (kvlen <= 0) return;
    qpos = kvlen - 1;
    const int wstart = window_start(qpos, a.window), kp = keep_parts(a.keep, wstart);
    klo = z < kp ? z * kPartTokens : (wstart / kPartTokens + z - kp) * kPartTokens;
    kend = min(z < kp ? a.keep : kvlen, klo + kPartTokens);
    kbeg = z < kp ? klo : max(klo, wstart);
    if (kbeg >= kend) return;
  } else {
    const int tile = blockIdx.x >> 2, qo = a.tile_qoff[tile] + 16 * (blockIdx.x & 3);
    s = a.tile_seq[tile];
    h0 = blockIdx.y;
    g = h0 / rep;
    const int row0 = a.seq_qstart[s], n = a.seq_qstart[s + 1] - row0, kvlen = a.seq_kvlen[s];
    if (n <= 0 || kvlen <= 0 || qo >= n) return;
    columns = min(16, n - qo);
    row = row0 + qo;
    qpos = kvlen - n + qo;
    kbeg = window_start(qpos, a.window);
    kend = qpos + columns;
    qpos += min(m, columns - 1);
  }
  const int qlow = window_start(qpos, a.window), kkeep = min(a.keep, kbeg), col = min(m, columns - 1);
  const int head = DECODE ? h0 + col : h0, nd = a.dim >> 4, nv = a.vdim >> 4, bs = a.block_size;
  const int gv = g / a.v_share, GV = a.G / a.v_share;
  if (!DECODE) row += col;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

  f32x4 Q[ND], O[NV];
  const float* qr = q + row * a.q_stride + static_cast<int64_t>(head) * a.dim + 4 * r;
#pragma unroll
  for (int t = 0; t < ND; ++t) Q[t] = t < nd ? *reinterpret_cast<const f32x4*>(qr + 16 * t) : zero;
#pragma unroll
  for (int t = 0; t < NV; ++t) O[t] = zero;
  float mx = kNegBig, l = 0.f;   // of column m
  if (!DECODE && a.sink && w == 0) {   // (decode: the join adds the sink once)
    mx = a.sink_val != nullptr ? a.sink_val[head] : 0.f;
    l = 1.f;
  }
  const int* bt = a.block_tables + static_cast<int64_t>(s) * a.bt_width;
  // blocks of 16 keys: those with kept ones in front of the window, then those from the window's first key on
  const int b0 = klo >> 4, kept = max(0, ((kkeep + 15) >> 4) - b0), first = max(kbeg >> 4, b0 + kept);
  const int blocks = kept + max(0, ((kend + 15) >> 4) - first);
  for (int i = w; i < blocks; i += 4) {
    const int k0 = 16 * (i < kept ? b0 + i : first + i - kept);
    const int64_t page = bt[k0 / bs];
    const int off = k0 % bs;
    const float* kp = k_cache + ((page * a.G + g) * bs + off + m) * a.dim + 4 * r;   // (a page's rows are all there)
    const float* vp = v_cache + ((page * GV + gv) * a.vdim + m) * static_cast<int64_t>(bs) + off + 4 * r;
    f32x4 K[ND], V[NV];
#pragma unroll
    for (int t = 0; t < ND; ++t)
      if (t < nd) K[t] = *reinterpret_cast<const f32x4*>(kp + 16 * t);
#pragma unroll
    for (int t = 0; t < NV; ++t)
      if (t < nv) V[t] = *reinterpret_cast<const f32x4*>(vp + static_cast<int64_t>(16 * t) * bs);
    f32x4 S[2] = {zero, zero};   // (two sums: a product waits for the one before the last)
#pragma unroll
    for (int t = 0; t < ND; ++t)
      if (t < nd)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[e & 1] = mma(K[t][e], Q[t][e], S[e & 1]);
    float p[4], top = kNegBig, sum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int key = k0 + 4 * r + e;
      p[e] = key <= qpos && key < kend && (key >= qlow || key < a.keep) ? (S[0][e] + S[1][e]) * a.scale : kNegBig;
      top = fmaxf(top, p[e]);
    }
    top = fmaxf(top, __shfl_xor(top, 16, kWave));
    top = fmaxf(top, __shfl_xor(top, 32, kWave));
    const float next = fmaxf(mx, top), alpha = expf(mx - next);
    mx = next;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p[e] = p[e] <= kNegBig ? 0.f : expf(p[e] - next);
      sum += p[e];
    }
    sum += __shfl_xor(sum, 16, kWave);
    sum += __shfl_xor(sum, 32, kWave);
    l = l * alpha + sum;
    if (k0 + 16 > kend || (k0 < kbeg && k0 + 16 > kkeep)) {   // values that nobody sees: whatever is there (uniform)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = k0 + 4 * r + e;
        if (key >= kend || (key < kbeg && key >= kkeep))
#pragma unroll
          for (int t = 0; t < NV; ++t) V[t][e] = 0.f;
      }
    }
#pragma unroll
    for (int t = 0; t < NV; ++t)
      if (t < nv) {
        O[t] *= alpha;
#pragma unroll
        for (int e = 0; e < 4; ++e) O[t] = mma(V[t][e], p[e], O[t]);
      }
  }
  // the waves' sums
  if (r == 0) {
    stats[w][0][m] = mx;
    stats[w][1][m] = l;
  }
  __syncthreads();
  float all = stats[0][0][m], total = 0.f, own = 0.f;
#pragma unroll
  for (int i = 1; i < 4; ++i) all = fmaxf(all, stats[i][0][m]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float f = expf(stats[i][0][m] - all);
    total += stats[i][1][m] * f;
    own = i == w ? f : own;
  }
#pragma unroll
  for (int t = 0; t < NV; ++t) {
    O[t] *= own;
    if (w > 0 && t < nv) sums[w - 1][t][lane] = O[t];
  }
  __syncthreads();
  if (w != 0 || m >= columns) return;
  auto sum_of = [&](int t) { return (O[t] + sums[0][t][lane]) + (sums[1][t][lane] + sums[2][t][lane]); };
  if (DECODE) {
    float* o = a.part + ((static_cast<int64_t>(s) * a.H + head) * a.max_parts + blockIdx.z) * (a.vdim + 2);
#pragma unroll
    for (int t = 0; t < NV; ++t)
      if (t < nv) {
        const f32x4 x = sum_of(t);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[16 * t + 4 * r + e] = x[e];   // (partials' rows are not aligned)
      }
    if (r == 0) {
      o[a.vdim] = all;
      o[a.vdim + 1] = total;
    }
    return;
  }
  const float inv = (total > 0.f ? 1.0f / total : 0.f) * head_gate_of<float>(a, row, head);
  float* o = out + (static_cast<int64_t>(row) * a.H + head) * a.vdim + 4 * r;
#pragma unroll
  for (int t = 0; t < NV; ++t)
    if (t < nv) *reinterpret_cast<f32x4*>(o + 16 * t) = sum_of(t) * inv;
}

}  // namespace sfl

bool launch_sink_float(void* out, const void* q, const void* k_cache, const void* v_cache, const AttnArgs& a, int num_tiles,
                       int num_decode, int parts, hipStream_t st) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(q) |
                       reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache);
  if (a.dim % 16 != 0 || a.vdim % 16 != 0 || a.dim > 256 || a.vdim > 256 || a.block_size % 16 != 0 || a.q_stride % 4 != 0 ||
      at % 16 != 0)
    return false;
  auto go = [&](auto prompts, auto decode) {
    auto launch = [&](auto kernel, dim3 grid) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, static_cast<float*>(out), static_cast<const float*>(q),
                         static_cast<const float*>(k_cache), static_cast<const float*>(v_cache), a);
    };
    if (num_tiles > 0) launch(prompts, dim3(num_tiles * 4, a.H));
    if (num_decode > 0) launch(decode, dim3(num_decode, a.G * ((a.H / a.G + 15) / 16), parts));
  };
#define MIXK_WIDTHS(ND, NV) go(sfl::sink_float_kernel<ND, NV, false>, sfl::sink_float_kernel<ND, NV, true>)
  if (a.dim <= 64 && a.vdim <= 64) MIXK_WIDTHS(4, 4);
  else if (a.dim <= 64 && a.vdim <= 128) MIXK_WIDTHS(4, 8);
  else if (a.dim <= 128 && a.vdim <= 128) MIXK_WIDTHS(8, 8);
  else if (a.vdim <= 192) MIXK_WIDTHS(16, 12);
  else MIXK_WIDTHS(16, 16);
#undef MIXK_WIDTHS
  return true;
}

}  // namespace mixk
