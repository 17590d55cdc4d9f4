// Decode rows of the softmax attention on the matrix cores (bf16), and the join of a row's partitions.
//
// Partition kernel: one workgroup of four waves per (sequence, KV head, 128 keys, 32 query heads of its group).
// Nothing is staged: a wave takes the scores of 32 keys, its K rows straight from the pages into the fragments
// (A = K, B = Q, a query head per column), and then the output channels of every fourth block of 32 over all 128
// keys, whose V fragments it also reads straight from the channel-major pages.  All of a workgroup's loads - K, V
// and Q - are in flight at once, behind a single look at the block table; between the two products only the
// column maxima, sums and the weights go through LDS.  O needs no sum over waves.  The weights are rounded against the
// maximum of their own 32 keys, so the largest of every tile is exactly 1, and the tiles' values are put together in
// fp32; the sums are those of the rounded weights.  Error against 64 bits, 16 rows of 2000, with one maximum per
// partition / here (1e-3): 32 + 8 heads of 128 2.73 / 2.63 (the kernel before, a running maximum of 32 keys: 2.69),
// latent 1.86 / 1.82 (1.85), two maps 2.33 / 2.17 (2.27); 0 - 0.3 us.
//
// Bound: latency of one chain (row, context length -> block table -> keys -> weights -> store) for short contexts,
// the pages' bytes for long ones.  Measured, tiles staged in LDS one after the other -> now: 8 rows,
// contexts of 1500, 32 + 8 heads of 128: 15.4 -> 10.8 us (32 rows of 2000: 38 us, 6.9 TB/s with the last-level cache's
// help); latent, 16 rows of 2000: 26 -> 12.1; two maps 21 -> 10.
//
// Join: four waves per (row, head) take every fourth partition, with the first four of them loaded before their
// weights are known: 6.2 -> 3.7 us, latent 10.7 -> 4.4, two maps 7.1 -> 5.7.  One look at the partitions' maxima and sums,
// of both maps at once, in place of two or four in turn: layers, 16 rows of 2000, two maps 31.4 -> 30.9 us, small, 6 rows of
// 1300, 19.2 -> 18.5, latent as before within 1 %.  (The partition kernel with the pages fetched beside the context's
// length, one trip less, is slower: latent 28.7 -> 29.5, 32 + 8 heads 39.3 -> 39.7.)
#include "sink_attention.h"

namespace mixk {
namespace sd {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kWaves = 4, kTile = 32;
constexpr int kPStride = kPartTokens + 8;
static_assert(kPartTokens == kWaves * kTile, "a wave per tile");
constexpr float kLog2e = 1.44269504088896341f;

// dim = 16 ND, vdim = 32 NV
template <int ND, int NV>
__global__ void __launch_bounds__(256, ND > 8 ? 1 : 2)
sink_decode_kernel(const __bf16* __restrict__ q, const __bf16* __restrict__ k_cache,
                   const __bf16* __restrict__ v_cache, AttnArgs a) {
  constexpr int D = 16 * ND, VD = 32 * NV, VT = (NV + kWaves - 1) / kWaves, VS = kPartTokens / 16;
  __shared__ __attribute__((aligned(16))) __bf16 lds_p[32 * kPStride];
  __shared__ float lds_m[kWaves][32], lds_l[kWaves][32];
  const int rep = a.H / a.G, cb = (rep + 31) / 32;
  const int s = blockIdx.x, g = blockIdx.y / cb, c0 = (blockIdx.y % cb) * 32, z = blockIdx.z;
  const int kvlen = a.seq_kvlen[s];
  if (kvlen <= 0) return;
  const int wstart = window_start(kvlen - 1, a.window), kp = keep_parts(a.keep, wstart);
  const bool keep_part = z < kp;   // kept keys only
  const int part0 = keep_part ? z * kPartTokens : (wstart / kPartTokens + z - kp) * kPartTokens;
  const int kbeg = keep_part ? part0 : max(part0, wstart & ~(kTile - 1));
  const int kend = min(keep_part ? a.keep : kvlen, part0 + kPartTokens);
  if (kbeg >= kend) return;
  const int kkeep = min(a.keep, kbeg);   // kept keys [part0, kkeep) in front of the window
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int shift = a.bs_shift, mask = a.block_size - 1;
  const int* bt = a.block_tables + static_cast<int64_t>(s) * a.bt_width;
  // tiles of 32 keys that hold a key of this partition; loads of the others go to kbeg's and are not used
  auto live = [&](int k0) { return (k0 < kkeep || k0 >= kbeg) && k0 < kend; };

  bf16x8 kf[ND], qf[ND], vf[VT][VS];
  const int k0 = part0 + kTile * w;
  const bool on = live(k0);
  // lane i: where the 16 keys of V step i (mod VS) are, so that one load brings all pages
  const int t_lane = part0 + 16 * (lane & (VS - 1));
  const int step_at = live(t_lane & ~(kTile - 1)) && t_lane < kend ? t_lane : kbeg;
  const int step_page = bt[step_at >> shift];
  {
    const int key = min((on ? k0 : kbeg) + r, kend - 1);
    const __bf16* p = k_cache + ((static_cast<int64_t>(bt[key >> shift]) * a.G + g) * a.block_size + (key & mask)) * D +
                      8 * h;
#pragma unroll
    for (int st = 0; st < ND; ++st) kf[st] = *reinterpret_cast<const bf16x8*>(p + 16 * st);
  }
  const int col = c0 + r, head = g * rep + min(col, rep - 1);   // columns past the group repeat its last head
  {
    const __bf16* p = q + static_cast<int64_t>(a.seq_qstart[s]) * a.q_stride + static_cast<int64_t>(head) * D + 8 * h;
#pragma unroll
    for (int st = 0; st < ND; ++st) qf[st] = *reinterpret_cast<const bf16x8*>(p + 16 * st);
  }
  const int GV = a.G / a.v_share, gv = g / a.v_share;
  const __bf16* vbase = v_cache + (static_cast<int64_t>(gv) * VD + w * 32 + r) * a.block_size + 8 * h;
#pragma unroll
  for (int vt = 0; vt < VT; ++vt) {
    if (kWaves * vt + kWaves > NV && w + kWaves * vt >= NV) continue;   // uniform over the wave
#pragma unroll
    for (int st = 0; st < VS; ++st) {   // 16 keys of one page
      const int64_t page = __builtin_amdgcn_readlane(step_page, st);
      const int in_page = __builtin_amdgcn_readlane(step_at, st) & mask;
      vf[vt][st] = *reinterpret_cast<const bf16x8*>(vbase + page * GV * VD * a.block_size + in_page +
                                                    vt * kWaves * 32 * a.block_size);
    }
  }
  __builtin_amdgcn_sched_barrier(0);   // no load waits for a product to free its registers

  f32x16 S;
#pragma unroll
  for (int i = 0; i < 16; ++i) S[i] = 0.f;
#pragma unroll
  for (int st = 0; st < ND; ++st) S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[st], qf[st], S, 0, 0, 0);
  // scores in log2 units; the maximum starts at the finite kNegBig, so a tile of masked keys has weights of 0
  const int qlow = wstart;
  const float scale2 = a.scale * kLog2e;
  float m = kNegBig;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int key = k0 + 8 * (i >> 2) + 4 * h + (i & 3);
    S[i] = on && key < kend && (key >= qlow || key < a.keep) ? S[i] * scale2 : -INFINITY;
    m = fmaxf(m, S[i]);
  }
  m = fmaxf(m, __shfl_xor(m, 32, kWave));
  float l = 0.f;   // of the weights as the value products take them, rounded
#pragma unroll
  for (int i4 = 0; i4 < 4; ++i4) {
    bf16x4 e;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      e[j] = static_cast<__bf16>(__builtin_amdgcn_exp2f(S[4 * i4 + j] - m));
      l += static_cast<float>(e[j]);
    }
    *reinterpret_cast<bf16x4*>(lds_p + r * kPStride + kTile * w + 8 * i4 + 4 * h) = e;
  }
  l += __shfl_xor(l, 32, kWave);
  if (h == 0) {
    lds_m[w][r] = m;
    lds_l[w][r] = l;
  }
  lds_barrier();
  float alpha[kWaves];   // of the tiles' weights against the partition's maximum
  m = fmaxf(fmaxf(lds_m[0][r], lds_m[1][r]), fmaxf(lds_m[2][r], lds_m[3][r]));
#pragma unroll
  for (int t = 0; t < kWaves; ++t) alpha[t] = __builtin_amdgcn_exp2f(lds_m[t][r] - m);
  const int np = min(kPartTokens, kend - part0);
  f32x16 O[VT];
#pragma unroll
  for (int vt = 0; vt < VT; ++vt)
#pragma unroll
    for (int i = 0; i < 16; ++i) O[vt][i] = 0.f;
#pragma unroll
  for (int t = 0; t < kWaves; ++t) {
    if (!live(part0 + kTile * t)) continue;   // uniform over the workgroup
    f32x16 P[VT];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int i = 0; i < 16; ++i) P[vt][i] = 0.f;
#pragma unroll
    for (int st = 2 * t; st < 2 * t + 2; ++st) {
      if (16 * st >= np) continue;
      const bf16x8 pf = *reinterpret_cast<const bf16x8*>(lds_p + r * kPStride + 16 * st + 8 * h);
      const bool last = 16 * st + 16 > np;   // V of the keys past the end must be exactly zero
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        if (kWaves * vt + kWaves > NV && w + kWaves * vt >= NV) continue;
        bf16x8 x = vf[vt][st];
        if (last)
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (16 * st + 8 * h + j >= np) x[j] = static_cast<__bf16>(0.f);
        P[vt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, pf, P[vt], 0, 0, 0);
      }
    }
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int i = 0; i < 16; ++i) O[vt][i] += alpha[t] * P[vt][i];
  }
  if (col >= rep) return;
  float* po = a.part + ((static_cast<int64_t>(s) * a.H + head) * a.max_parts + z) * (VD + 2);
#pragma unroll
  for (int vt = 0; vt < VT; ++vt)
    if (w + kWaves * vt < NV)
#pragma unroll
      for (int i = 0; i < 16; ++i) po[(w + kWaves * vt) * 32 + 8 * (i >> 2) + 4 * h + (i & 3)] = O[vt][i];
  if (w == 0 && h == 0) {
    po[VD] = m / kLog2e;   // the join works in natural-log units
    po[VD + 1] = (lds_l[0][r] * alpha[0] + lds_l[1][r] * alpha[1]) + (lds_l[2][r] * alpha[2] + lds_l[3][r] * alpha[3]);
  }
}

// partitions of a decode row
__device__ __forceinline__ int live_parts(const AttnArgs& a, int kvlen) {
  const int wstart = window_start(kvlen - 1, a.window);
  return (kvlen + kPartTokens - 1) / kPartTokens - wstart / kPartTokens + keep_parts(a.keep, wstart);
}

// vdim <= 64 NJ.  NMAP 1: out[row, h] = the merged partitions (and the sink) of head h, times the head's gate.
// NMAP 2: o = a1 - lam a2 of the two maps' heads, / its root mean square, * post * sigmoid(gate per channel), into
// out [T, H / 2, vdim].
template <typename T, int NMAP, int NJ>
__global__ void __launch_bounds__(256)
sink_join_kernel(void* __restrict__ out, AttnArgs a) {
  constexpr int kAhead = 4;
  __shared__ float sums[NMAP][4][NJ * kWave];
  const int s = blockIdx.x, ho = blockIdx.y, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int kvlen = a.seq_kvlen[s];
  if (kvlen <= 0) return;
  const int np = live_parts(a, kvlen), vdim = a.vdim, ps = vdim + 2, rep = a.H / a.G;
  auto head_of = [&](int mp) { return NMAP == 2 ? (2 * (ho / rep) + mp) * rep + ho % rep : ho; };   // G counts a K head per map
  auto base_of = [&](int mp) { return a.part + (static_cast<int64_t>(s) * a.H + head_of(mp)) * a.max_parts * ps; };
  // a lane's partition among the first 64: its maximum and sum; with the values of the first four per wave all of a chain's
  // loads, of both maps, in one trip
  float inv[NMAP], ahead[NMAP][kAhead][NJ], top[NMAP], sum[NMAP];
#pragma unroll
  for (int mp = 0; mp < NMAP; ++mp) {
    const float* base = base_of(mp);
    const float* e = base + static_cast<int64_t>(min(lane, np - 1)) * ps + vdim;
    top[mp] = e[0];
    sum[mp] = e[1];
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        ahead[mp][i][j] = base[static_cast<int64_t>(min(w + 4 * i, np - 1)) * ps + min(lane + kWave * j, vdim - 1)];
  }
#pragma unroll
  for (int mp = 0; mp < NMAP; ++mp) {
    const int h = head_of(mp);
    const float* base = base_of(mp);
    float acc[NJ];
    const float sink_score = a.sink && a.sink_val != nullptr ? a.sink_val[h] : 0.f;
    float M = a.sink ? sink_score : kNegBig, L = 0.f;
    M = fmaxf(M, top[mp]);   // (lanes past the last partition hold it again)
    for (int p = lane + kWave; p < np; p += kWave) M = fmaxf(M, base[static_cast<int64_t>(p) * ps + vdim]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, kWave));
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[j] = 0.f;
    for (int p0 = 0; p0 < np; p0 += kWave) {
      float e0 = top[mp], e1 = sum[mp];
      if (p0 > 0) {
        const float* e = base + static_cast<int64_t>(min(p0 + lane, np - 1)) * ps + vdim;
        e0 = e[0];
        e1 = e[1];
      }
      const float wp = p0 + lane < np ? expf(e0 - M) : 0.f;
      L += p0 + lane < np ? e1 * wp : 0.f;   // (a partition past the end may hold anything)
      auto weight = [&](int i) {
        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wp), i));
      };
      int i = w;
      if (p0 == 0)
#pragma unroll
        for (int k = 0; k < kAhead; ++k, i += 4)
          if (i < np)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[j] += ahead[mp][k][j] * weight(i);
#pragma unroll 4
      for (; i < min(kWave, np - p0); i += 4)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[j] += base[static_cast<int64_t>(p0 + i) * ps + min(lane + kWave * j, vdim - 1)] * weight(i);
    }
    L = wave_sum(L) + (a.sink ? expf(sink_score - M) : 0.f);
    inv[mp] = L > 0.f ? 1.0f / L : 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) sums[mp][w][lane + kWave * j] = acc[j];
  }
  __syncthreads();
  if (w != 0) return;
  const int64_t row = a.seq_qstart[s];
  float o[NJ], ss = 0.f;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int d = lane + kWave * j;
    auto total = [&](int mp) { return (sums[mp][0][d] + sums[mp][1][d]) + (sums[mp][2][d] + sums[mp][3][d]); };
    o[j] = total(0) * inv[0];
    if (NMAP == 2) o[j] -= a.lam * (total(NMAP - 1) * inv[NMAP - 1]);
    ss += d < vdim ? o[j] * o[j] : 0.f;
  }
  float f = 1.f;
  const T* gt = nullptr;
  if (NMAP == 2) {
    f = a.post / sqrtf(wave_sum(ss) / static_cast<float>(vdim) + a.eps);
    if (a.gate != nullptr)
      gt = static_cast<const T*>(a.gate) + row * a.gate_stride + static_cast<int64_t>(ho) * vdim;
  } else {
    f = head_gate_of<T>(a, row, ho);
  }
  const int64_t at = (row * (a.H / NMAP) + ho) * vdim;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int d = lane + kWave * j;
    if (d >= vdim) continue;
    const float y = o[j] * f * (gt != nullptr ? sigmoidf_(ldf(gt + d)) : 1.0f);
    if (NMAP == 1 && a.out_f32)
      static_cast<float*>(out)[at + d] = y;
    else
      stf(static_cast<T*>(out) + at + d, y);
  }
}

template <int ND, int NV>
bool launch(const void* q, const void* k_cache, const void* v_cache, const AttnArgs& a, int num_decode, int parts,
            hipStream_t st) {
  const int64_t gy = static_cast<int64_t>(a.G) * ((a.H / a.G + 31) / 32);
  if (gy > 65535 || parts > 65535) return false;
  hipLaunchKernelGGL((sink_decode_kernel<ND, NV>), dim3(num_decode, static_cast<unsigned>(gy), parts), dim3(256), 0, st,
                     static_cast<const __bf16*>(q), static_cast<const __bf16*>(k_cache),
                     static_cast<const __bf16*>(v_cache), a);
  return true;
}

template <typename T, int NMAP>
void join(void* out, const AttnArgs& a, int num_decode, hipStream_t st) {
  const dim3 grid(num_decode, a.H / NMAP);
  if (a.vdim <= 64)
    hipLaunchKernelGGL((sink_join_kernel<T, NMAP, 1>), grid, dim3(256), 0, st, out, a);
  else if (a.vdim <= 128)
    hipLaunchKernelGGL((sink_join_kernel<T, NMAP, 2>), grid, dim3(256), 0, st, out, a);
  else if (a.vdim <= 256)
    hipLaunchKernelGGL((sink_join_kernel<T, NMAP, 4>), grid, dim3(256), 0, st, out, a);
  else
    hipLaunchKernelGGL((sink_join_kernel<T, NMAP, 8>), grid, dim3(256), 0, st, out, a);
}

}  // namespace sd

// The served head widths, pages of 16 keys or more (a step of 16 keys lies in one page).
bool launch_sink_decode(const void* q, const void* k_cache, const void* v_cache, const AttnArgs& a, int num_decode,
                        int parts, hipStream_t st) {
  if (a.block_size < 16) return false;
#define SD(D, V) \
  if (a.dim == D && a.vdim == V) return sd::launch<D / 16, V / 32>(q, k_cache, v_cache, a, num_decode, parts, st);
  SD(64, 64)
  SD(64, 128)
  SD(128, 128)
  SD(256, 192)
#undef SD
  return false;
}

void launch_sink_join(void* out, const AttnArgs& a, int num_decode, int dtype, hipStream_t st) {
  MIXK_DISPATCH(dtype, {
    if (a.pair)
      sd::join<T, 2>(out, a, num_decode, st);
    else
      sd::join<T, 1>(out, a, num_decode, st);
  });
}

}  // namespace mixk
