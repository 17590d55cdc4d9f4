// Prefill of the paged softmax attention on the matrix cores (bf16, gfx950): flash form of the kernel in
// sink_attention.hip, same masks, sink, gates and pair epilogue (see there for what they mean).
//
// A workgroup = NW waves x 32 columns, a column = (query token, query head of the KV head's group); it walks
// 64-key blocks:
//   S^T[32 keys x 32 cols] = K . Q^T    (mfma 32x32x16, A = K rows from LDS, B = Q in registers)
//   O^T[vdim x 32 cols]   += V^T . P^T  (A = V^T rows from LDS, B = P^T from the S^T registers)
// A lane holds one column of S^T, so the softmax statistics are lane-local plus one exchange with
// lane ^ 32.  K rows are read in the order that swaps bits 2 and 3 of the row: the eight probabilities a
// lane half then holds per 16-key step belong to eight neighbouring keys, so a V^T fragment is one plain
// 16-byte read.
//
// The next block's K / V are fetched into registers behind the score products and stored to the other LDS
// buffer after the value products: one barrier per block.  A wave fetches keys of ONE 16-key group, which
// lie in one page (pages of 16 tokens or more), so its page and the group's place in the page are scalars and
// every lane offset a loop constant; the sequence's page list sits in LDS.  O and l are rescaled on blocks that raise some column's
// maximum.  (Letting the maximum lag by up to 2^8 saves ~3 % but then the largest weight is not exactly 1
// and its rounding counts: error against 64 bits 3.2e-3 instead of 3.0e-3.)
//
// Pair form: a workgroup's first four waves carry the first map, the other four the second one, over the
// same columns and one V block; the second map's result goes to the first's waves through LDS at the end.
//
// Bound (128 wide): per block and wave 1024 cycles of matrix products and ~1000 of softmax on the vector
// units; two waves per SIMD overlap them only in part (matrix cores 37 % busy, vector units 45 %, LDS port
// 34 %, at 1.8 GHz).  Wave priority from the score products to the end of the value products lets the other
// wave fall behind and fill gaps instead of running the same phase in step: 7580 rows of 32 + 8 heads of 128
// 5 %, latent 2 %, two maps 1 %.  (Taking block b + 1's scores beside block b's weights in the same wave: 128 wide 6 %
// less, latent 2.1 times, two maps 1.1 times the time - registers.)
#include "sink_attention.h"

namespace mixk {
namespace sf {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

constexpr int kBlock = 64;               // keys per block (two 32-key score tiles)
constexpr int kVS = kBlock + 8;          // V^T row in LDS: 144 B, 16-byte reads free of bank conflicts
constexpr int kPages = 2048;             // page-table entries in LDS
// Pair form: in the first blocks each of the two tiles has its own maximum.  Largest weights are rounded to exactly 1;
// with a maximum per 64 keys there are fewer of them than per 32, half of the difference from the first block, 90 %
// from four.  Error against 64 bits, prompts of 600 (1e-3): one per block 2.345, the first four split 2.328 (the kernel
// before, 32 keys: 2.332); 5 x 1165 tokens, window 1024: 82.2 -> 83.3 us, with all blocks split 85.3.  (One map: sums of
// the rounded weights make up for more than that: 2.928 against 2.935.)
constexpr int kSplitBlocks = 4;
constexpr float kLog2e = 1.44269504088896341f;

__device__ __forceinline__ float xor32(float v, int idx4) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(idx4, __builtin_bit_cast(int, v)));
}

// DK = 16 ND (q / k width), DV = 32 NV (value width).
template <int ND, int NV, int NMAP, int NW, int WPS, bool WIN>
__global__ void __launch_bounds__(NW * 64, WPS)
sink_flash_kernel(void* __restrict__ out, const __bf16* __restrict__ q,
                  const __bf16* __restrict__ k_cache, const __bf16* __restrict__ v_cache, AttnArgs a,
                  int num_tiles, int chunks) {
  constexpr int DK = 16 * ND, DV = 32 * NV, CW = NW / NMAP, COLS = CW * 32;
  constexpr int KS = DK + 8;
  constexpr int WPG = NW / 4;                       // waves per 16-key group
  constexpr int KU = 16 * (DK / 8) / (64 * WPG);    // 16-byte chunks of K per lane, map and block
  constexpr int VU = 2 * DV / (64 * WPG);           // ... of V
  static_assert(NMAP == 1 || NW == 8, "pair form: four waves per map");
  static_assert(KU * 64 * WPG == 2 * DK && VU * 64 * WPG == 2 * DV, "staging covers a block");
  typedef __bf16 KBuf[2][NMAP][kBlock * KS];
  typedef __bf16 VBuf[2][DV * kVS];
  __shared__ __attribute__((aligned(16))) char lds[sizeof(KBuf) + sizeof(VBuf)];
  KBuf& lds_k = *reinterpret_cast<KBuf*>(lds);
  VBuf& lds_v = *reinterpret_cast<VBuf*>(lds + sizeof(KBuf));
  __shared__ int lds_bt[kPages];
  const int H = a.H, G = a.G, bs = a.block_size;
  const int rep = H / G, GO = G / NMAP, GV = G / a.v_share;
  // KV head fastest: workgroups are dealt round-robin to the eight XCDs, so with eight KV heads a head's
  // K / V stay in one L2.  Tiles are listed in token order: the longest go first.
  const int bid = static_cast<int>(blockIdx.x);
  const int g = bid % GO;                           // K head (pair form: V head, K heads 2 g and 2 g + 1)
  const int rest = bid / GO;
  const int chunk = chunks - 1 - rest % chunks;
  const int tile = num_tiles - 1 - rest / chunks;
  const int gv = NMAP == 2 ? g : g / a.v_share;
  const int s = a.tile_seq[tile], qo = a.tile_qoff[tile];
  const int row0 = a.seq_qstart[s], n = a.seq_qstart[s + 1] - row0, kvlen = a.seq_kvlen[s];
  if (n <= 0 || kvlen <= 0 || qo >= n) return;
  const int cols_total = min(kTileTokens, n - qo) * rep;
  const int col0 = chunk * COLS;
  if (col0 >= cols_total) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5, x32 = (lane ^ 32) << 2;
  const int ctx = kvlen - n + qo;                   // position of the tile's first token
  const int mp = NMAP == 2 ? w / CW : 0;            // the wave's map
  const int wcol = col0 + (w % CW) * 32;       // the wave's first column
  const bool wave_on = wcol < cols_total;
  const int w_last = min(cols_total, wcol + 32) - 1;
  const int pos_first = ctx + wcol / rep, pos_last = ctx + max(w_last, 0) / rep;
  const int kend = min(kvlen, ctx + (min(cols_total, col0 + COLS) - 1) / rep + 1);
  // key blocks: the kept keys in front of the window, then from the window's start (block-aligned)
  const int klow = window_start(ctx + col0 / rep, a.window);   // no column sees keys in [keep, klow)
  const int kbeg = klow & ~(kBlock - 1);
  const int kkeep = min(a.keep, kbeg);
  const int nk = (kkeep + kBlock - 1) / kBlock;
  const int nb = nk + (kend - kbeg + kBlock - 1) / kBlock;
  auto block_key = [&](int b) { return b < nk ? b * kBlock : kbeg + (b - nk) * kBlock; };

  const int* btg = a.block_tables + static_cast<int64_t>(s) * a.bt_width;
  const int npages = min((kend + bs - 1) >> a.bs_shift, kPages);   // (the launcher bounds the table)
  for (int i = tid; i < npages; i += NW * 64) lds_bt[i] = btg[i];

  const int col = wcol + r;
  const bool valid = col < cols_total;
  const int tok = valid ? col / rep : 0, head = (NMAP * g + mp) * rep + (valid ? col % rep : 0);
  const int64_t row = row0 + qo + tok;
  const int qpos = valid ? ctx + tok : -1;          // no key is visible to a column that is not there
  const int qlow = window_start(qpos, a.window);
  bf16x8 qf[ND];
  const __bf16* qp = q + row * a.q_stride + static_cast<int64_t>(head) * DK + 8 * h;
#pragma unroll
  for (int st = 0; st < ND; ++st) qf[st] = *reinterpret_cast<const bf16x8*>(qp + 16 * st);
  float m = kNegBig, l = 0.f;   // l: of the lane's keys
  if (a.sink) {   // the sink is the state the online softmax starts from (log2 units)
    m = a.sink_val != nullptr ? a.sink_val[head] * kLog2e : 0.f;
    l = h == 0 ? 1.f : 0.f;
  }
  f32x16 O[NV];
#pragma unroll
  for (int vt = 0; vt < NV; ++vt)
#pragma unroll
    for (int i = 0; i < 16; ++i) O[vt][i] = 0.f;
  __syncthreads();

  // staging: wave w moves keys of group sg = w / WPG; its part of the group's chunks starts at `sub`
  const int sg = w / WPG, sub = (w % WPG) * 64 + lane;
  int k_src[KU], k_dst[KU], v_src[VU], v_dst[VU];
#pragma unroll
  for (int u = 0; u < KU; ++u) {
    const int i = sub + u * 64 * WPG, key = i / (DK / 8), c8 = i % (DK / 8);
    k_src[u] = key * DK + c8 * 8;
    k_dst[u] = (16 * sg + key) * KS + c8 * 8;
  }
#pragma unroll
  for (int u = 0; u < VU; ++u) {
    const int i = sub + u * 64 * WPG, ch = i >> 1;
    v_src[u] = ch * bs + 8 * (i & 1);
    v_dst[u] = ch * kVS + 16 * sg + 8 * (i & 1);
  }
  const int last_page = npages - 1;
  u32x4 kr[NMAP][KU], vr[VU];
  auto load_block = [&](int k0) {
    // keys at or past kend read a clamped page or stale slots, keys in front of the window whatever is there: their
    // scores are masked and their V zeroed (0 x NaN)
    const int key = k0 + 16 * sg, at = key & (bs - 1);   // (a page may hold several blocks)
    const int pg = __builtin_amdgcn_readfirstlane(lds_bt[min(key >> a.bs_shift, last_page)]);
    const __bf16* kb = k_cache + ((static_cast<int64_t>(pg) * G + NMAP * g) * bs + at) * DK;
    const __bf16* vb = v_cache + (static_cast<int64_t>(pg) * GV + gv) * DV * bs + at;
#pragma unroll
    for (int e = 0; e < NMAP; ++e)
#pragma unroll
      for (int u = 0; u < KU; ++u)
        kr[e][u] = *reinterpret_cast<const u32x4*>(kb + e * bs * DK + k_src[u]);
#pragma unroll
    for (int u = 0; u < VU; ++u) vr[u] = *reinterpret_cast<const u32x4*>(vb + v_src[u]);
  };
  auto store_block = [&](int buf, int k0) {
#pragma unroll
    for (int e = 0; e < NMAP; ++e)
#pragma unroll
      for (int u = 0; u < KU; ++u)
        *reinterpret_cast<u32x4*>(&lds_k[buf][e][k_dst[u]]) = kr[e][u];
    const int key = k0 + 16 * sg + 8 * (lane & 1);
    if (key + 8 > kend || (WIN && key < klow && key + 8 > a.keep)) {
      auto seen = [&](int t) { return t < kend && (!WIN || t >= klow || t < a.keep); };
#pragma unroll
      for (int u = 0; u < VU; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          vr[u][j] &= (seen(key + 2 * j) ? 0x0000ffffu : 0u) | (seen(key + 2 * j + 1) ? 0xffff0000u : 0u);
    }
#pragma unroll
    for (int u = 0; u < VU; ++u) *reinterpret_cast<u32x4*>(&lds_v[buf][v_dst[u]]) = vr[u];
  };

  const float scale2 = a.scale * kLog2e;
  // A row of the score products: key with bits 2 and 3 swapped
  const int krow = (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1);
  // keys at or below the window start of the wave's latest column are outside somebody's window
  const int edge_lo = a.window > 0 ? pos_last - a.window : -1;
  const int low_first = window_start(pos_first, a.window);   // no column of the wave sees keys below

  load_block(block_key(0));
  store_block(0, block_key(0));
  __syncthreads();
  for (int b = 0; b < nb; ++b) {
    const int buf = b & 1, k0 = block_key(b);
    const bool more = b + 1 < nb;
    bool issued = false;
    if (wave_on && k0 <= pos_last && (k0 + kBlock > low_first || k0 < a.keep)) {
      f32x16 S[2];
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int i = 0; i < 16; ++i) S[t][i] = 0.f;
#pragma unroll
        for (int st = 0; st < ND; ++st) {
          const bf16x8 kf =
              *reinterpret_cast<const bf16x8*>(&lds_k[buf][mp][(32 * t + krow) * KS + 16 * st + 8 * h]);
          S[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[st], S[t], 0, 0, 0);
        }
      }
      if (more) load_block(block_key(b + 1));   // in flight behind the softmax and the value products
      issued = true;
      // register i of tile t holds key k0 + 8 h + 32 t + 16 (i >> 3) + (i & 7)
      if (k0 + kBlock - 1 > pos_first || (WIN && k0 <= edge_lo)) {
        const int hi = qpos + 1 - k0 - 8 * h, lo = qlow - k0 - 8 * h, kp = a.keep - k0 - 8 * h;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int o = 32 * t + 16 * (i >> 3) + (i & 7);
            if (o >= hi || (WIN && o < lo && o >= kp)) S[t][i] = -INFINITY;
          }
      }
      // maxima of the block: one, or in the pair form's first blocks one per tile (kSplitBlocks)
      constexpr int MT = NMAP, TPM = 2 / MT;
      float tmax[MT], mt[MT], psum[MT];
#pragma unroll
      for (int e = 0; e < MT; ++e) {
        tmax[e] = S[e * TPM][0];
#pragma unroll
        for (int t = e * TPM; t < (e + 1) * TPM; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) tmax[e] = fmaxf(tmax[e], S[t][i]);
      }
#pragma unroll
      for (int e = 0; e < MT; ++e) tmax[e] = fmaxf(tmax[e], xor32(tmax[e], x32)) * scale2;
      if (MT > 1 && b >= kSplitBlocks) tmax[0] = fmaxf(tmax[0], tmax[MT - 1]);
      auto rescale = [&](float alpha) {
        l *= alpha;
#pragma unroll
        for (int vt = 0; vt < NV; ++vt)
#pragma unroll
          for (int i = 0; i < 16; ++i) O[vt][i] *= alpha;
      };
      bool grow = tmax[0] > m;   // (scale > 0; all keys masked: -inf, never)
      mt[0] = grow ? tmax[0] : m;
      if (__any(grow)) rescale(__builtin_amdgcn_exp2f(m - mt[0]));
      grow = MT > 1 && tmax[MT - 1] > mt[0];
      mt[MT - 1] = grow ? tmax[MT - 1] : mt[0];
      m = mt[MT - 1];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          S[t][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[t][i], scale2, -mt[t / TPM]));
      bf16x8 pf[4];
#pragma unroll
      for (int e = 0; e < MT; ++e) psum[e] = 0.f;   // of the weights as the value products take them, rounded
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        u32x4 wv;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          wv[j] = __builtin_bit_cast(unsigned int, __builtin_convertvector(
                      (f32x2{S[ks >> 1][8 * (ks & 1) + 2 * j], S[ks >> 1][8 * (ks & 1) + 2 * j + 1]}),
                      bf16x2));
        pf[ks] = __builtin_bit_cast(bf16x8, wv);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          psum[(ks >> 1) / TPM] += __builtin_bit_cast(float, wv[j] << 16) + __builtin_bit_cast(float, wv[j] & 0xffff0000u);
      }
#pragma unroll
      for (int e = 0; e < MT; ++e) {
        if (e > 0 && __any(grow)) rescale(__builtin_amdgcn_exp2f(mt[0] - m));
        l += psum[e];
#pragma unroll
        for (int vt = 0; vt < NV; ++vt)
#pragma unroll
          for (int ks = 2 * e * TPM; ks < 2 * (e + 1) * TPM; ++ks) {
            const bf16x8 vf = *reinterpret_cast<const bf16x8*>(&lds_v[buf][(32 * vt + r) * kVS + 16 * ks + 8 * h]);
            O[vt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[ks], O[vt], 0, 0, 0);
          }
      }
      __builtin_amdgcn_s_setprio(0);
    }
    if (more) {
      if (!issued) load_block(block_key(b + 1));
      store_block(buf ^ 1, block_key(b + 1));
    }
    __syncthreads();
  }

  l += xor32(l, x32);
  if constexpr (NMAP == 2) {
    // the second map's waves hand lam / l * O to the first map's through LDS (the K / V buffers are free)
    static_assert(sizeof(lds_k) + sizeof(lds_v) >= CW * 64 * 16 * NV * sizeof(float), "room for the second map");
    f32x4* xch = reinterpret_cast<f32x4*>(lds) + (w % CW) * 4 * NV * 64 + lane;
    const float il = l > 0.f ? (mp == 0 ? 1.0f : a.lam) / l : 0.f;
    if (mp == 1) {
#pragma unroll
      for (int vt = 0; vt < NV; ++vt)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          xch[(vt * 4 + i4) * 64] = f32x4{O[vt][4 * i4] * il, O[vt][4 * i4 + 1] * il,
                                          O[vt][4 * i4 + 2] * il, O[vt][4 * i4 + 3] * il};
    }
    __syncthreads();
    if (mp == 1 || !valid) return;   // both halves of a column are valid together
    const int ho = g * rep + col % rep;
    float ss = 0.f;
#pragma unroll
    for (int vt = 0; vt < NV; ++vt)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const f32x4 o2 = xch[(vt * 4 + i4) * 64];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float o = O[vt][4 * i4 + j] * il - o2[j];
          O[vt][4 * i4 + j] = o;
          ss += o * o;
        }
      }
    ss += __shfl_xor(ss, 32, kWave);
    const float f = a.post / sqrtf(ss / static_cast<float>(DV) + a.eps);
    const __bf16* gt = a.gate != nullptr ? static_cast<const __bf16*>(a.gate) + row * a.gate_stride +
                                               static_cast<int64_t>(ho) * DV : nullptr;
    __bf16* o = static_cast<__bf16*>(out) + (row * (H / 2) + ho) * DV;
#pragma unroll
    for (int vt = 0; vt < NV; ++vt)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int ch = vt * 32 + 8 * i4 + 4 * h;
        bf16x4 gv4, ev;
        if (gt != nullptr) gv4 = *reinterpret_cast<const bf16x4*>(gt + ch);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          ev[j] = static_cast<__bf16>(O[vt][4 * i4 + j] * f *
                                      (gt != nullptr ? sigmoidf_(static_cast<float>(gv4[j])) : 1.0f));
        *reinterpret_cast<bf16x4*>(o + ch) = ev;
      }
    return;
  }
  if (!valid) return;
  const float inv = (l > 0.f ? 1.0f / l : 0.f) * head_gate_of<__bf16>(a, row, head);
  const int64_t o = (row * H + head) * DV;
#pragma unroll
  for (int vt = 0; vt < NV; ++vt)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int64_t at = o + vt * 32 + 8 * i4 + 4 * h;
      if (a.out_f32) {
        f32x4 ev;
#pragma unroll
        for (int j = 0; j < 4; ++j) ev[j] = O[vt][4 * i4 + j] * inv;
        *reinterpret_cast<f32x4*>(static_cast<float*>(out) + at) = ev;
      } else {
        bf16x4 ev;
#pragma unroll
        for (int j = 0; j < 4; ++j) ev[j] = static_cast<__bf16>(O[vt][4 * i4 + j] * inv);
        *reinterpret_cast<bf16x4*>(static_cast<__bf16*>(out) + at) = ev;
      }
    }
}

template <int ND, int NV, int NMAP, int NW, int WPS>
bool launch(void* out, const void* q, const void* k_cache, const void* v_cache, const AttnArgs& a,
            int num_tiles, hipStream_t st) {
  constexpr int COLS = NW / NMAP * 32;
  const int chunks = (kTileTokens * (a.H / a.G) + COLS - 1) / COLS;
  const unsigned grid = static_cast<unsigned>(num_tiles) * (a.G / NMAP) * chunks;
  auto* kernel = a.window > 0 ? sink_flash_kernel<ND, NV, NMAP, NW, WPS, true>
                              : sink_flash_kernel<ND, NV, NMAP, NW, WPS, false>;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(NW * 64), 0, st, out, static_cast<const __bf16*>(q),
                     static_cast<const __bf16*>(k_cache), static_cast<const __bf16*>(v_cache), a,
                     num_tiles, chunks);
  return true;
}

}  // namespace sf

// The shapes of the served families (head width 128, the latent cache of 192 + 64 channels, narrow heads,
// two maps of 64 over values of 128); other shapes, pages below 16 tokens (a 16-key group would span two)
// and contexts past the LDS page list run sink_attention.hip's kernel.  Measured at 4 prompts of ~1850
// tokens (us, old kernel -> this one; variants at the same shapes):
//   128 / 128, 32 heads over 8:  463 -> 159 (8 waves per workgroup: +1 %; 64 columns per wave: +30 %)
//   256 / 192, 32 heads over 1: 1052 -> 261 (4 waves +50 %: one wave per SIMD hides no latency)
//   two maps 64 / 128, 8 over 2, 5 x 1165 tokens, window 1024: 126 -> 72 (both maps in each of 4 waves
//     +45 %: few workgroups there, so a wave's own chain counts; 2 waves per SIMD +10 %, 4 spill)
// The workgroups of the 256 / 192 form hold 8 tokens (the old kernel's 4): so far ahead a NaN value reaches back (a weight
// of 0 times NaN), as it did there.
bool launch_sink_flash(void* out, const void* q, const void* k_cache, const void* v_cache,
                       const AttnArgs& a, int num_tiles, hipStream_t st) {
  if (a.block_size < 16 || a.bt_width > sf::kPages || !(a.scale > 0.f)) return false;
#define SF(D, V, MAPS, NW, WPS)                              \
  if (a.dim == D && a.vdim == V && (a.pair ? 2 : 1) == MAPS) \
    return sf::launch<D / 16, V / 32, MAPS, NW, WPS>(out, q, k_cache, v_cache, a, num_tiles, st);
  SF(64, 64, 1, 4, 2)
  SF(128, 128, 1, 4, 2)
  SF(256, 192, 1, 8, 2)
  SF(64, 128, 2, 8, 3)
#undef SF
  return false;
}

}  // namespace mixk
