// Prefill flash attention over the paged KV cache, LDS-staged K/V tiles on 32x32x16 MFMA
// (the attention that vLLM runs under engine.generate(), reference llm/serve_llm.py:527-531).  Varlen batches, causal with a context offset (chunked prefill
// and prefix-cache hits: query token i of a sequence sits at position kvlen - qlen + i),
// GQA G = Hq / Hkv in {1, 2, 3, 4, 8}, head_dim 128, bf16 / fp16 (G = 3: Llama-3.2-3B, 24 q /
// 8 kv heads; a wave's last 32 mod 3 = 2 columns idle).
//
// Work decomposition: grid tiles x Hkv (1-D, KV head fastest).  A workgroup = 4 waves owns 128 "columns" = the G
// query heads of one KV head x 128 / G consecutive query tokens of one sequence; wave w owns
// columns 32w..32w+31 (column c: token c / G, head c % G).  Every K/V tile is staged ONCE in
// LDS per workgroup and read by all 128 columns (G x the reuse of a per-head kernel).
//
// Per 64-key block (two 32-key sub-tiles), per wave ("swapped QK^T"):
//   S^T[32 keys x 32 cols] = K[32 x 128] . Q^T[128 x 32]       8 x mfma_f32_32x32x16
//     A = K rows from LDS, B = Q (registers); the accumulator has the column on the lane, so the online-softmax row
//     statistics are lane-local over 16 registers plus one xor-32 exchange;
//   O^T[128 x 32] += V^T[128 x 32 keys] . P^T[32 keys x 32]    8 x mfma_f32_32x32x16
//     B = P^T straight from the S^T accumulator registers (pairs packed to 16 bit), A = V^T rows from LDS.
// O^T is rescaled only when a running max grew by more than 2^8 (defer-max).
// Pipelining: step i takes the scores of block i, the weights of block i - 1 and the value products of block i - 2, which
// do not depend on each other, and deals them out by hand (`quick`): a product (32 cycles of the matrix core), then the
// vector instructions that fit behind it.  Left to the compiler, products and softmax ran one after the other in every
// wave.  Blocks on the diagonal and both ends go part by part.  K and V of the next blocks go straight from memory to LDS in
// the meantime: no registers, one wait and one workgroup barrier per block.  The sequence's block-table slice is staged in
// LDS once so K/V addresses need no dependent global load inside the loop.
// Short prompts and chunks behind a cached prefix: with its start and its masked blocks a workgroup of few blocks is latency
// from end to end, so the first V comes with the first K, the queries are asked for behind the page list and not waited for
// with it (1000 of 12500 cycles at 17 tokens), the parts' products have their operands on the way and go on different sums
// in turn, and up to three blocks go without steps, their code in a row (another 1200 of them: fetches of instructions).
// Kernel, us, 32 + 8 heads, one part after the other / pipeline without this / now; bound by the chain of loads and parts: 17
// tokens 6.3 / 7.3 / 6.0, 85 8.1 / 9.0 / 7.3, 188 10.3 / 11.2 / 8.9, 475 17.6 / 15.5 / 14.4; behind cached ones: 5 x 17 on 600
// 17.9 / 16.2 / 15.0, 5 x 85 on 500 19.6 / 19.0 / 17.2, 188 on 512 21.2 / 18.0 / 17.1, 475 on 2000 43.3 / 37.2 / 35.3, 17 on 4096
// (split) 29.0 / 29.6 / 27.4; bound by matrix and vector units together, at a clock that gives way: 16 x 100 14.5 / 13.7 / 12.7,
// 1 x 2000 61 / 49 / 48, 4 x 2k 157 / 144 / 136.  24 + 8 heads: 17 tokens 6.1 / 7.1 / 6.1, 85 8.9 / 9.6 / 7.7, 188 10.3 / 11.4 /
// 9.1, 4 x 2k 130 / 124 / 115.
#include <type_traits>
#include <utility>

#include "common.h"
#include "kernels.h"

namespace atta {
namespace fp {

constexpr int kD = 128;
constexpr int kNS = 2;                   // 32-key sub-tiles per block
constexpr int kKB = 32 * kNS;            // keys per block
// LDS images: K rows as they are (256 B), V as [16-key group][channel][16 keys]; the 16-byte chunks of a K row and the
// halves of a V row change places (row & 15, channel bit 3) so that the fragments' ds_read_b128 have no bank conflicts.
constexpr int kKTile = kKB * kD;         // elements
constexpr int kVTile = kD * kKB;
constexpr int kBtLds = 2048;             // block-table entries staged in LDS
constexpr float kNegInf = -__builtin_huge_valf();
// Workgroups of so many blocks take them one after the other.  Cycles of one of 3 / 4 / 6 blocks, alone on its CU: in steps
// 17700 / 20400 / 24700, one after the other 15400 / 20100 / 25700.
constexpr int kBrief = 3;
constexpr float kRescale = 8.f;  // defer-max threshold (log2 units)

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef u32x4 __attribute__((aligned(2))) u32x4_any;   // in memory, wherever it begins
typedef __attribute__((address_space(3))) void* lds_ptr;
#define FP_INLINE __attribute__((always_inline))

template <typename T>
struct Mf32;
template <>
struct Mf32<__bf16> {
  typedef bf16x8 frag;
  __device__ static __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mf32<_Float16> {
  typedef f16x8 frag;
  __device__ static __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

struct FlashParams {
  uint16_t* out;            // [n_q_tokens, Hq, D] rows of out_stride
  const uint16_t* q;        // [n_q_tokens, Hq, D] rows of q_stride
  const uint16_t* k_cache;  // [nb, Hkv, BS, D]
  const uint16_t* v_cache;  // [nb, Hkv, D, BS]
  const int* block_tables;  // [S, bt_stride]
  const int* seq_kvlen;
  const int* seq_qstart;
  const int* tile_seq;
  const int* tile_qoff;
  int num_tiles;
  int64_t q_stride, out_stride;
  int bt_stride, n_kv_heads, bs_shift;
  float scale_log2;
  // split-KV (few tiles over long cached prefixes: the cached burst / planning steps): up to
  // nsplit workgroups per (tile, KV head) each walk a contiguous range of key blocks and
  // publish (O, m, l) partials; the last to arrive merges them (device-scope hand-over)
  int nsplit;
  int split_blocks;  // key blocks per split at least (atta_set_flash_split_blocks)
  float* part;    // [tile, Hkv, nsplit] slots of kPartBytes
  int* counters;  // [tile * Hkv], zero between launches (the last arriver re-arms)
  int wide_out;   // rows of out start on 16-byte borders
  int wide_in;    // the caches do: otherwise they go through registers, block by block
};
// one split's partial: 128 columns x 128 fp32 O values, then 128 (m, l) pairs
constexpr uint32_t kPartOBytes = 128 * kD * 4;
constexpr uint32_t kPartBytes = kPartOBytes + 128 * 8;
constexpr int kMaxSplit = 8;
constexpr int kSplitBlocks = 8;  // 512 keys: the default of split_blocks

// two floats -> one packed 16-bit pair.  bf16: a single v_cvt_pk_bf16_f32 (RNE); element-wise
// conversion compiled to 2 converts + shift + or per pair, 64 VALU per block per wave.
template <typename T>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return static_cast<uint32_t>(from_f32<T>(a)) | (static_cast<uint32_t>(from_f32<T>(b)) << 16);
}
template <>
__device__ __forceinline__ uint32_t pack2<__bf16>(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{a, b}), bf16x2_t));
}

// lane l <-> lane l ^ 32 exchange: one ds_bpermute with the byte index hoisted out of the loop
// (__shfl_xor recomputed it per call: 7 VALU).
__device__ __forceinline__ float xor32(float v, int idx4) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(idx4, __builtin_bit_cast(int, v)));
}
// larger value of the lane's and lane ^ 32's, without a trip through LDS.  (As an instruction: with both operands the same
// value the compiler folded the builtin's two results into one.)
__device__ __forceinline__ float both_max(float v) {
  float a = v, b = v;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
#endif
  return fmaxf(a, b);
}
// 16 bytes per lane from base + offset to 1 KB of LDS from address `to` on, without registers; there after wait_sent().
// (After the builtin the compiler makes every read of LDS wait for all transfers.)  The base goes through a scalar move:
// five wait states belong between a vector instruction that writes a scalar register, such as the reload of a spilled one,
// and a memory instruction that reads it, and the compiler does not put them in front of assembly.  (The same in
// mixers/sink_flash.hip, a library of its own.)
__device__ __forceinline__ void send16(const void* base, uint32_t offset, uint32_t to) {
#if defined(__HIP_DEVICE_COMPILE__)
  uint64_t from;
  asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 %0, %2\n\tglobal_load_lds_dwordx4 %1, %0"
               : "=&s"(from) : "v"(offset), "s"(base), "s"(to) : "m0", "memory");
#endif
}
// the same by way of registers: from memory off 16-byte borders
__device__ __forceinline__ void copy16(const void* base, uint32_t offset, uint32_t to, int lane) {
  typedef __attribute__((address_space(3))) u32x4* lds_u32x4;
  *(lds_u32x4)(to + 16u * lane) = *reinterpret_cast<const u32x4_any*>(static_cast<const char*>(base) + offset);
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr)(const_cast<void*>(p))));
}
__device__ __forceinline__ void wait_sent() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
}
// the value is there at this point of the program
template <typename X>
__device__ __forceinline__ void hold(const X& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" ::"v"(x));
#endif
}

// the value, computed anew from here on (not kept in a register until then)
__device__ __forceinline__ int fresh(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(v));
#endif
  return v;
}
// f(0), f(1), ... as constants
template <int... N, typename F>
__device__ __forceinline__ void each(std::integer_sequence<int, N...>, const F& f) {
  (f(std::integral_constant<int, N>()), ...);
}

// NW = 8 (two workgroup halves): each staged K/V block serves 256 columns and a wave sends half as much.
template <typename T, int G, int NW>
__global__ __launch_bounds__(NW * 64, 2) void flash_prefill_kernel(FlashParams p) {
  using MF = Mf32<T>;
  using frag = typename MF::frag;
  constexpr int kTokPerWave = 32 / G;
  constexpr int kTokPerWg = NW * kTokPerWave;
  __shared__ __attribute__((aligned(1024))) uint16_t lds_k[2 * kKTile], lds_v[2 * kVTile];
  __shared__ int lds_bt[kBtLds];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform -> SGPR
  const int r = lane & 31;   // column within the wave / row within a 32-row operand
  const int h = lane >> 5;   // lane half
  const int x32 = (lane ^ 32) << 2;  // ds_bpermute byte index of the partner lane
  // 1-D grid, KV head fastest: blocks are dealt round-robin over the 8 XCDs, so with 8 KV
  // heads every tile of head hk runs on one XCD and the head's K/V (re-read by all its
  // tiles) stays in that XCD's L2 instead of being pulled into all eight (placement is a
  // speed choice only, never correctness).  Heaviest (latest-token) tiles first: tiles are
  // emitted in token order per sequence.
  const int bid = static_cast<int>(blockIdx.x);
  const int hk = bid % p.n_kv_heads;
  const int rest = bid / p.n_kv_heads;
  const int sp = rest % p.nsplit;  // key-range split of this workgroup
  const int tile = p.num_tiles - 1 - rest / p.nsplit;
  const int s = p.tile_seq[tile];
  const int qoff = p.tile_qoff[tile];
  const int kvlen = p.seq_kvlen[s];  // >= wg_end: every key this workgroup reads is below it
  const int qstart = p.seq_qstart[s];
  const int qlen = p.seq_qstart[s + 1] - qstart;
  const int ctx0 = kvlen - qlen;
  const int BS = 1 << p.bs_shift;
  const int* bt = p.block_tables + static_cast<int64_t>(s) * p.bt_stride;

  // this lane's column
  const int c_tok = qoff + wid * kTokPerWave + r / G;
  const int c_head = hk * G + r % G;
  // (G = 3: columns 30, 31 of a wave would spill into the next wave's tokens)
  const bool c_valid = r < kTokPerWave * G && c_tok < qlen;
  const int c_end = c_valid ? ctx0 + c_tok + 1 : 0;  // keys [0, c_end) are visible
  // workgroup key range: up to the last valid token's causal limit
  const int wg_last_tok = min(qoff + kTokPerWg, qlen) - 1;
  const int wg_end = ctx0 + wg_last_tok + 1;
  const int nblocks = (wg_end + kKB - 1) / kKB;
  // wave key range (wave-uniform): blocks at or past it only need the wave at the barrier
  const int w_last_tok = min(qoff + (wid + 1) * kTokPerWave, qlen) - 1;
  const int w_end = w_last_tok >= qoff + wid * kTokPerWave ? ctx0 + w_last_tok + 1 : 0;
  const int w_first = qoff + wid * kTokPerWave;  // first token: fully visible below ctx0+w_first+1
  // this tile's splits: >= kSplitBlocks key blocks each (a split pays a publish + merge chain
  // of ~2 us: at the cached burst's ~10 blocks per tile it measured a wash), workgroups past
  // them exit before any barrier
  const int ns = max(1, min(p.nsplit, nblocks / p.split_blocks));
  if (sp >= ns) return;
  const int kb0 = sp * nblocks / ns, kb1 = (sp + 1) * nblocks / ns;

  // ---- block table slice -> LDS -------------------------------------------------------
  const int npages = min((wg_end + BS - 1) >> p.bs_shift, kBtLds);
  for (int i = tid; i < npages; i += NW * 64) lds_bt[i] = bt[i];

  // ---- Q (B operand): Q[col r][16 st + 8 h .. +8], 8 k-steps over D ----------------------
  // (behind the page list, which would wait with them: loads under a condition)
  frag qf[8];
  {
    const uint16_t* qp = p.q + static_cast<int64_t>(qstart + (c_valid ? c_tok : 0)) * p.q_stride +
                         static_cast<int64_t>(c_head) * kD + 8 * h;
#pragma unroll
    for (int st = 0; st < 8; ++st)
      qf[st] = c_valid ? *reinterpret_cast<const frag*>(qp + 16 * st) : frag{};
  }
  __syncthreads();  // lds_bt ready

  // ---- staging of one K/V block: memory -> LDS, past the registers ----------------------
  // A wave sends keys of ONE 16-key group for both tensors: with BS >= 16 they sit in one page, so the page lookup and
  // the keys' place in the page are wave-uniform (one LDS read + readfirstlane, a scalar base) and every lane offset is a
  // constant.  A transfer is 1 KiB of contiguous memory: 4 K rows, or 32 channels x 16 keys (at BS = 16).
  // Keys past the workgroup's range (>= wg_end) read a clamped page or the unused tail slots of the last page - stale
  // bytes of whatever sequence held that page before.  Their scores are masked (P = 0), and their V^T columns are zeroed once
  // they are there, by the wave that sent them, so that a non-finite stale value cannot turn 0 * V into NaN.
  constexpr int WPG = NW / 4, U = 4 / WPG;   // waves per group, transfers per wave and tensor
  const int sg = wid & 3, part = wid >> 2;
  const int last_page = npages - 1;
  uint32_t k_src[U], v_src[U];   // bytes
  const int v_half = 8 * ((lane ^ (lane >> 4)) & 1);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int row = 4 * (u * WPG + part) + (lane >> 4);
    k_src[u] = 2u * (row * kD + ((lane & 15) ^ row) * 8);
    v_src[u] = 2u * ((32 * (u * WPG + part) + (lane >> 1)) * BS + v_half);
  }
  const int k_lds = 16 * sg * kD + part * 512, v_lds = sg * kD * 16 + part * 512;
  const uint16_t* k_base = p.k_cache + (static_cast<uint64_t>(hk) << (p.bs_shift + 7));
  const uint16_t* v_base = p.v_cache + (static_cast<uint64_t>(hk) << (p.bs_shift + 7));
  const uint32_t page = static_cast<uint32_t>(p.n_kv_heads) << (p.bs_shift + 7);   // elements of a page, all heads
  auto page_at = [&](int k0) FP_INLINE { return lds_bt[min((k0 + 16 * sg) >> p.bs_shift, last_page)]; };
  auto k_at = [&](int pg, int k0) FP_INLINE {
    return k_base + static_cast<uint64_t>(static_cast<uint32_t>(pg)) * page + ((k0 + 16 * sg) & (BS - 1)) * kD;
  };
  auto v_at = [&](int pg, int k0) FP_INLINE {
    return v_base + static_cast<uint64_t>(static_cast<uint32_t>(pg)) * page + ((k0 + 16 * sg) & (BS - 1));
  };
  // (`b`: which of the two buffers, its lowest bit)
  const uint32_t k_to = lds_address(lds_k) + 2 * k_lds, v_to = lds_address(lds_v) + 2 * v_lds;
  auto move16 = [&](const uint16_t* base, uint32_t offset, uint32_t to, bool direct) FP_INLINE {
    if (direct) send16(base, offset, to);
    else copy16(base, offset, to, fresh(lane));
  };
  auto send_k = [&](const uint16_t* kb, int b, int u, bool direct) FP_INLINE {
    move16(kb, k_src[u], k_to + (b & 1) * 2 * kKTile + u * WPG * 1024, direct);
  };
  auto send_v = [&](const uint16_t* vb, int b, int u, bool direct) FP_INLINE {
    move16(vb, v_src[u], v_to + (b & 1) * 2 * kVTile + u * WPG * 1024, direct);
  };
  auto send_block_k = [&](int k0, int b) FP_INLINE {
    const uint16_t* kb = k_at(__builtin_amdgcn_readfirstlane(page_at(k0)), k0);
    if (__builtin_expect(p.wide_in, 1)) {
#pragma unroll
      for (int u = 0; u < U; ++u) send_k(kb, b, u, true);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) send_k(kb, b, u, false);
    }
  };
  auto send_block_v = [&](int k0, int b) FP_INLINE {
    const uint16_t* vb = v_at(__builtin_amdgcn_readfirstlane(page_at(k0)), k0);
    if (__builtin_expect(p.wide_in, 1)) {
#pragma unroll
      for (int u = 0; u < U; ++u) send_v(vb, b, u, true);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) send_v(vb, b, u, false);
    }
  };
  auto clear_block_v = [&](int k0, int b) FP_INLINE {
    if (k0 + kKB <= wg_end) return;
    const int ln = fresh(lane), key = k0 + 16 * sg + 8 * ((ln ^ (ln >> 4)) & 1);
    u32x4 mask;
#pragma unroll
    for (int j = 0; j < 4; ++j) mask[j] = (key + 2 * j < wg_end ? 0x0000ffffu : 0u) | (key + 2 * j + 1 < wg_end ? 0xffff0000u : 0u);
    uint16_t* to = lds_v + (b & 1) * kVTile + v_lds + ln * 8;
#pragma unroll
    for (int u = 0; u < U; ++u) *reinterpret_cast<u32x4*>(to + u * WPG * 512) &= mask;
  };
  // ---- fragments.  A row of the score products: key with bits 2 and 3 swapped, so that register i of a tile holds key
  // 16 (i >> 3) + 8 h + (i & 7) and a V^T fragment is one plain 16-byte read
  const int krow = (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1);
  int kofs[8];
#pragma unroll
  for (int st = 0; st < 8; ++st) kofs[st] = krow * kD + ((2 * st + h) ^ (krow & 15)) * 8;
  const int vofs = r * 16 + 8 * (h ^ ((r >> 3) & 1));
  auto kf = [&](const uint16_t* b, int t, int st) FP_INLINE { return *reinterpret_cast<const frag*>(b + 32 * t * kD + kofs[st]); };
  auto vf = [&](const uint16_t* b, int dt, int ks) FP_INLINE {
    return *reinterpret_cast<const frag*>(b + vofs + ks * kD * 16 + dt * 512);
  };

  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  float m_run = kNegInf, l_run = 0.f;   // l_run: of the lane's keys

  // defer-max: the running max m_run moves only when some column's max grew by more than kRescale (log2 units), so
  // P = 2^(s - m_run) stays <= 2^kRescale; O and l are rescaled only then - with the max nearly settled after the first
  // block, the multiplies of the rescale were paid on most blocks.  O, l and P of a block always use the same m_run, so
  // the result is exact up to rounding.  Answers the factor of the columns that moved.
  auto raise = [&](const f32x16 (&S)[kNS], float& alpha) FP_INLINE {
    float tm[4];   // running max on the raw scores (scale > 0)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      tm[c] = kNegInf;
#pragma unroll
      for (int i = 0; i < 8; ++i) tm[c] = fmaxf(tm[c], S[c >> 1][8 * (c & 1) + i]);
    }
    const float m_cand = fmaxf(m_run, both_max(fmaxf(fmaxf(tm[0], tm[1]), fmaxf(tm[2], tm[3]))) * p.scale_log2);
    const bool grow = m_cand > m_run + kRescale;  // m_run == -inf: any finite m_cand
    const float m_new = grow ? m_cand : m_run;
    alpha = __builtin_amdgcn_exp2f(m_run - ((m_new == kNegInf) ? 0.f : m_new));
    if (!grow) alpha = 1.f;
    m_run = m_new;
    return grow;
  };
  auto rescale = [&](float alpha) FP_INLINE {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
  };
  // softmax in the log2 domain with the scale folded into one fma per element: p = 2^(s * scale_log2 - m); weights 2 u
  // and 2 u + 1 of the block, and their place in the row sum's two chains
  auto weight2 = [&](const f32x16 (&S)[kNS], int u, float neg_m, float& s0, float& s1) FP_INLINE {
    const int t = u / 8, i = 2 * (u % 8);
    const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(S[t][i], p.scale_log2, neg_m));
    const float y = __builtin_amdgcn_exp2f(__builtin_fmaf(S[t][i + 1], p.scale_log2, neg_m));
    s0 += x;
    s1 += y;
    return pack2<T>(x, y);
  };
  // (products with their operands on the way, on different sums in turn: left to the compiler each waited for its own)
  auto scores = [&](const uint16_t* kl, f32x16 (&S)[kNS]) FP_INLINE {
    constexpr int N = 8 * kNS, LA = 4;
    frag fr[N];
    auto read = [&](int n) FP_INLINE { fr[n] = kf(kl, n % kNS, n / kNS); };
#pragma unroll
    for (int n = 0; n < LA; ++n) read(n);
    each(std::make_integer_sequence<int, N>(), [&](auto slot) FP_INLINE {
      constexpr int n = slot;
      __builtin_amdgcn_sched_barrier(0);
      if (n + LA < N) read(n + LA);
      S[n % kNS] = MF::mma(fr[n], qf[n / kNS], n < kNS ? f32x16{} : S[n % kNS]);
    });
    __builtin_amdgcn_sched_barrier(0);
  };
  auto values = [&](const uint16_t* vl, const u32x4 (&P)[4]) FP_INLINE {
    constexpr int N = 16, LA = 4;
    frag fr[N];
    auto read = [&](int n) FP_INLINE { fr[n] = vf(vl, n % 4, n / 4); };
#pragma unroll
    for (int n = 0; n < LA; ++n) read(n);
    each(std::make_integer_sequence<int, N>(), [&](auto slot) FP_INLINE {
      constexpr int n = slot;
      __builtin_amdgcn_sched_barrier(0);
      if (n + LA < N) read(n + LA);
      o[n % 4] = MF::mma(fr[n], __builtin_bit_cast(frag, P[n / 4]), o[n % 4]);
    });
    __builtin_amdgcn_sched_barrier(0);
  };
  auto weights = [&](int k0, f32x16 (&S)[kNS], u32x4 (&P)[4]) FP_INLINE {
    // mask: only blocks crossing the diagonal of the wave's first token (wave-uniform branch).  Register i of a tile holds
    // its key 16 (i >> 3) + 8 h + (i & 7): a bit of a word per tile.  (A comparison per key, whose result waits in a scalar
    // register: 800 cycles per block.)
    if (k0 + kKB > ctx0 + w_first + 1) {
#pragma unroll
      for (int t = 0; t < kNS; ++t) {
        const int n = c_end - k0 - 8 * h - 32 * t;
        const unsigned int out = n <= 0 ? ~0u : n >= 32 ? 0u : ~0u << n;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float v = S[t][i];
          const unsigned int x = __builtin_amdgcn_sbfe(out, 16 * (i >> 3) + (i & 7), 1);
          S[t][i] = __builtin_bit_cast(float, (x & 0xff800000u) | (~x & __builtin_bit_cast(unsigned int, v)));
        }
      }
    }
    float alpha, s0 = 0.f, s1 = 0.f;
    if (__any(raise(S, alpha))) {
      l_run *= alpha;
      rescale(alpha);
    }
    const float neg_m = m_run == kNegInf ? 0.f : -m_run;
#pragma unroll
    for (int u = 0; u < 16; ++u) P[u / 4][u % 4] = weight2(S, u, neg_m, s0, s1);
    l_run += s0 + s1;
  };
  // One block's scores, the weights of the one before and the value products of the one before that: a product (32 cycles of
  // the matrix core), then the vector instructions that fit behind it.  The same sums in the same order as the parts above.
  auto quick = [&](const uint16_t* kl, const uint16_t* vl, int b, int bk, int bv, const f32x16 (&Si)[kNS],
                   f32x16 (&So)[kNS], const u32x4 (&Pi)[4], u32x4 (&Po)[4]) FP_INLINE {
    constexpr int NP = 16, NF = 32, LA = 3, NB = 30;   // NB: slots of the exponentials
    frag fr[NF];
    auto read = [&](int n) FP_INLINE { fr[n] = n < NP ? vf(vl, n / 8 * 2 + n % 2, n % 8 / 2) : kf(kl, n % 2, (n - NP) / 2); };
    const int kpg = page_at(bk), vpg = page_at(bv);
#pragma unroll
    for (int n = 0; n < LA; ++n) read(n);
    __builtin_amdgcn_sched_barrier(0);
    float alpha, s0 = 0.f, s1 = 0.f;
    const bool grow = raise(Si, alpha);
    const float neg_m = m_run == kNegInf ? 0.f : -m_run;
    const uint16_t *kb = nullptr, *vb = nullptr;
#pragma unroll
    for (int t = 0; t < kNS; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) So[t][i] = 0.f;
#pragma unroll
    for (int n = 0; n < NF; ++n) {
      __builtin_amdgcn_sched_barrier(0);
      if (n + LA < NF) read(n + LA);
      if (n < NP) {
        const int dt = n / 8 * 2 + n % 2;
        o[dt] = MF::mma(fr[n], __builtin_bit_cast(frag, Pi[n % 8 / 2]), o[dt]);
        hold(o[dt]);
      } else {
        So[n % 2] = MF::mma(fr[n], qf[(n - NP) / 2], So[n % 2]);
        hold(So[n % 2]);
      }
      if (n == 1) {
        kb = k_at(__builtin_amdgcn_readfirstlane(kpg), bk);
        vb = v_at(__builtin_amdgcn_readfirstlane(vpg), bv);
      }
      if (n >= 2 && n < 2 + U) send_k(kb, b, n - 2, true);
      if (n >= 2 + U && n < 2 + 2 * U) send_v(vb, b, n - 2 - U, true);
#pragma unroll
      for (int u = 16 * n / NB; n < NB && u < 16 * (n + 1) / NB; ++u) {
        const uint32_t x = weight2(Si, u, neg_m, s0, s1);
        hold(x);
        Po[u / 4][u % 4] = x;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (__any(grow)) {
      l_run *= alpha;
      rescale(alpha);
    }
    l_run += s0 + s1;
  };

  // ---- step i: scores of block kb0 + i, weights of the block before, value products of the one before that; the next K
  // and this V on their way to the other buffers
  const int nb = kb1 - kb0, kfirst = kb0 * kKB;
  auto kbuf = [&](int i) FP_INLINE { return lds_k + (i & 1) * kKTile; };
  auto vbuf = [&](int i) FP_INLINE { return lds_v + (i & 1) * kVTile; };
  auto needed = [&](int i) FP_INLINE { return i >= 0 && i < nb && kfirst + i * kKB < w_end; };   // wave-uniform
  f32x16 sacc[kNS];
  u32x4 pw[4];
  const bool brief = nb <= kBrief;
  if (nb > 0) {   // (the first V with the first K: a workgroup of few blocks waits once for both, and for the second ones)
    send_block_k(kfirst, 0);
    send_block_v(kfirst, 0);
    if (__builtin_expect(brief && nb > 1, 0)) {
      send_block_k(kfirst + kKB, 1);
      send_block_v(kfirst + kKB, 1);
    }
  }
#pragma unroll
  for (int st = 0; st < 8; ++st) hold(qf[st]);   // (there before the loop, which would wait for its transfers with them)
  wait_sent();
  if (nb > 0) clear_block_v(kfirst, 0);
  if (__builtin_expect(brief && nb > 1, 0)) clear_block_v(kfirst + kKB, 1);
  __syncthreads();
  // steps [2, quick1): the block before has no masked key, this one is needed
  const int quick1 = w_end > 0 && p.wide_in ? min(min(nb, (ctx0 + w_first + 1 - kfirst) / kKB + 1), (w_end - 1 - kfirst) / kKB + 1) : 0;
  auto quick_step = [&](int i, const f32x16 (&Si)[kNS], f32x16 (&So)[kNS], const u32x4 (&Pi)[4], u32x4 (&Po)[4]) FP_INLINE {
    quick(kbuf(i), vbuf(i), i + 1, kfirst + (i + 1) * kKB, kfirst + (i - 1) * kKB, Si, So, Pi, Po);
    wait_sent();
    __syncthreads();
  };
  // (Few blocks: one after the other, code in a row, the third's keys and values on their way behind the second.  Steps lie on
  // both sides of the dealt-out ones, and each place that is come to for the first time costs a fetch of instructions.)
  if (brief) {
    for (int i = 0; i < nb; ++i) {
      if (needed(i)) {
        scores(kbuf(i), sacc);
        weights(kfirst + i * kKB, sacc, pw);
        values(vbuf(i), pw);
      }
      if (__builtin_expect(nb > 2, 0)) {
        if (i == 1) {
          wait_sent();
          clear_block_v(kfirst + 2 * kKB, 0);
        }
        __syncthreads();
        if (i == 0) {
          send_block_k(kfirst + 2 * kKB, 0);
          send_block_v(kfirst + 2 * kKB, 0);
        }
      }
    }
    __syncthreads();   // (the results' way out is K's buffers)
  }
  for (int i = 0; !brief && i <= nb; ++i) {
    for (; i >= 2 && i + 1 < quick1; i += 2) {
      f32x16 s2[kNS];
      u32x4 p2[4];
      quick_step(i, sacc, s2, pw, p2);
      quick_step(i + 1, s2, sacc, p2, pw);
    }
    const int k0 = kfirst + (i - 1) * kKB;
    if (i + 1 < nb) send_block_k(k0 + 2 * kKB, i + 1);
    if (i >= 2) send_block_v(k0, i + 1);
    if (needed(i - 2)) values(vbuf(i), pw);
    if (needed(i - 1)) weights(k0, sacc, pw);
    if (needed(i)) scores(kbuf(i), sacc);
    wait_sent();
    if (i >= 2) clear_block_v(k0, i + 1);
    __syncthreads();
  }
  if (!brief && needed(nb - 1)) values(vbuf(nb + 1), pw);
  l_run += xor32(l_run, x32);

  if (__builtin_expect(ns > 1, 0)) {
    // ---- split-KV hand-over: publish (O, m, l) with device-scope stores, count arrivals; the
    // last workgroup of the tile merges every split's partial into its own registers
    __shared__ int fl_last;
    const auto rw = dev_rsrc(p.part);
    const int pair = tile * p.n_kv_heads + hk;
    const uint32_t base = static_cast<uint32_t>(pair * p.nsplit) * kPartBytes;
    const int col = wid * 32 + r;
    // lane (col r, half h): O^T element (dt, i) is d = 32 dt + 8 (i >> 2) + 4 h + (i & 3)
    if (c_valid) {
      const uint32_t mine = base + static_cast<uint32_t>(sp) * kPartBytes;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          dev_store16(rw, mine + (col * kD + 32 * dt + 8 * g + 4 * h) * 4,
                      u32x4{__float_as_uint(o[dt][4 * g]), __float_as_uint(o[dt][4 * g + 1]),
                            __float_as_uint(o[dt][4 * g + 2]), __float_as_uint(o[dt][4 * g + 3])});
      if (h == 0) {
        dev_store4(rw, mine + kPartOBytes + col * 8, m_run);
        dev_store4(rw, mine + kPartOBytes + col * 8 + 4, l_run);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores acknowledged
    __syncthreads();
    if (tid == 0) {
      const int old = __hip_atomic_fetch_add(p.counters + pair, 1, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
      fl_last = old == ns - 1;
    }
    __syncthreads();
    if (!fl_last) return;  // block-uniform
    if (tid == 0)
      __hip_atomic_store(p.counters + pair, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (c_valid) {
      float mq[kMaxSplit], lq[kMaxSplit];  // fully unrolled: registers, not scratch
      float M = m_run;
#pragma unroll
      for (int q = 0; q < kMaxSplit; ++q) {
        mq[q] = kNegInf;
        lq[q] = 0.f;
        if (q >= ns || q == sp) continue;
        const uint32_t at = base + static_cast<uint32_t>(q) * kPartBytes + kPartOBytes + col * 8;
        mq[q] = dev_load4(rw, at);
        lq[q] = dev_load4(rw, at + 4);
        M = fmaxf(M, mq[q]);
      }
      // every split's O and l are relative to its own running max (log2 units)
      const float Mu = M == kNegInf ? 0.f : M;
      const float wself = __builtin_amdgcn_exp2f(m_run - Mu);
      l_run *= wself;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= wself;
#pragma unroll
      for (int q = 0; q < kMaxSplit; ++q) {
        if (q >= ns || q == sp) continue;
        const float wq = __builtin_amdgcn_exp2f(mq[q] - Mu);
        l_run += wq * lq[q];
        const uint32_t at = base + static_cast<uint32_t>(q) * kPartBytes;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const u32x4 v = dev_load16(rw, at + (col * kD + 32 * dt + 8 * g + 4 * h) * 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) o[dt][4 * g + j] += wq * __uint_as_float(v[j]);
          }
      }
    }
  }

  // ---- epilogue: O = O^T / l, lane (col r, half h) holds d = 32 dt + (i & 3) + 8 (i >> 2) + 4 h; 64 channels at a time
  // through LDS (the wave's own 4 KB; K is read no more), so that a store has whole rows: 8-byte pieces of 32 rows keep the
  // memory pipe busy
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  auto two = [&](int dt, int i) FP_INLINE {
    return u32x2{pack2<T>(o[dt][i] * inv, o[dt][i + 1] * inv), pack2<T>(o[dt][i + 2] * inv, o[dt][i + 3] * inv)};
  };
  uint16_t* const op = p.out + static_cast<int64_t>(qstart + qoff + wid * kTokPerWave) * p.out_stride + static_cast<int64_t>(hk) * G * kD;
  if (__builtin_expect(p.wide_out, 1)) {
    char* x = reinterpret_cast<char*>(lds_k) + wid * 4096;
#pragma unroll
    for (int d2 = 0; d2 < 2; ++d2) {
#pragma unroll
      for (int c = 0; c < 8; ++c)
        *reinterpret_cast<u32x2*>(x + r * 128 + ((c ^ ((r >> 1) & 7)) * 16) + 8 * h) = two(2 * d2 + c / 4, c % 4 * 4);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int rr = 8 * j + (lane >> 3), tok = rr / G;
        const u32x4 e = *reinterpret_cast<const u32x4*>(x + rr * 128 + (((lane & 7) ^ ((rr >> 1) & 7)) * 16));
        if (rr < kTokPerWave * G && w_first + tok < qlen)
          *reinterpret_cast<u32x4*>(op + tok * p.out_stride + (rr - tok * G) * kD + 64 * d2 + 8 * (lane & 7)) = e;
      }
      __builtin_amdgcn_wave_barrier();
    }
  } else if (c_valid) {
    uint16_t* oc = op + (r / G) * p.out_stride + (r % G) * kD + 4 * h;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) *reinterpret_cast<u32x2*>(oc + 32 * dt + 8 * g) = two(dt, 4 * g);
  }
}

template <typename T, int NW>
static int launch_nw(int G, dim3 grid, hipStream_t st, const FlashParams& p) {
  switch (G) {
    case 1: flash_prefill_kernel<T, 1, NW><<<grid, NW * 64, 0, st>>>(p); return 0;
    case 2: flash_prefill_kernel<T, 2, NW><<<grid, NW * 64, 0, st>>>(p); return 0;
    case 3: flash_prefill_kernel<T, 3, NW><<<grid, NW * 64, 0, st>>>(p); return 0;
    case 4: flash_prefill_kernel<T, 4, NW><<<grid, NW * 64, 0, st>>>(p); return 0;
    case 8: flash_prefill_kernel<T, 8, NW><<<grid, NW * 64, 0, st>>>(p); return 0;
    default: return -1;
  }
}

// waves per workgroup (4 or 8); the host's tiles must hold NW * (32 / G) tokens
// (ops.prefill_tile_tokens reads the same setting)
static int g_flash_waves = 4;

template <typename T>
static int launch(int G, dim3 grid, hipStream_t st, const FlashParams& p) {
  return g_flash_waves == 8 ? launch_nw<T, 8>(G, grid, st, p) : launch_nw<T, 4>(G, grid, st, p);
}

}  // namespace fp
}  // namespace atta

using namespace atta;

void atta_set_flash_waves(int nw) { fp::g_flash_waves = nw == 8 ? 8 : 4; }
static int g_split_blocks = fp::kSplitBlocks;
void atta_set_flash_split_blocks(int nb) { g_split_blocks = nb < 1 ? 1 : nb; }

int atta_flash_prefill(void* out, const void* q, const void* k_cache, const void* v_cache,
                       const int* block_tables, const int* seq_kvlen, const int* seq_qstart,
                       const int* tile_seq, const int* tile_qoff, int num_tiles, int n_q_heads,
                       int n_kv_heads, int head_dim, int block_size, int bt_stride,
                       int64_t q_stride, int64_t out_stride, float scale, int nsplit,
                       float* part, int* counters, int dtype, hipStream_t stream) {
  const int G = n_q_heads / n_kv_heads;
  int shift = 0;
  while ((1 << shift) < block_size) ++shift;
  if (head_dim != fp::kD || (1 << shift) != block_size || block_size < 16) return -1;
  if (n_q_heads % n_kv_heads || G > 8 || ((G & (G - 1)) && G != 3)) return -1;
  // 16-byte row loads of q / stores of out need 8-element aligned row strides
  if (q_stride % 8 || out_stride % 4) return -1;
  if (bt_stride > fp::kBtLds) return -1;  // the block-table row is staged whole in LDS
  if (num_tiles == 0) return 0;
  fp::FlashParams prm{};
  prm.out = static_cast<uint16_t*>(out);
  prm.q = static_cast<const uint16_t*>(q);
  prm.k_cache = static_cast<const uint16_t*>(k_cache);
  prm.v_cache = static_cast<const uint16_t*>(v_cache);
  prm.block_tables = block_tables;
  prm.seq_kvlen = seq_kvlen;
  prm.seq_qstart = seq_qstart;
  prm.tile_seq = tile_seq;
  prm.tile_qoff = tile_qoff;
  prm.num_tiles = num_tiles;
  prm.q_stride = q_stride;
  prm.out_stride = out_stride;
  prm.bt_stride = bt_stride;
  prm.n_kv_heads = n_kv_heads;
  prm.bs_shift = shift;
  prm.scale_log2 = scale * 1.4426950408889634f;
  if (nsplit < 1 || nsplit > fp::kMaxSplit) return -1;
  if (nsplit > 1 && (part == nullptr || counters == nullptr)) return -2;
  // 32-bit byte offsets of the device-scope partial stores
  if (static_cast<int64_t>(num_tiles) * n_kv_heads * nsplit * fp::kPartBytes > 0x7FFFFFFF) return -1;
  prm.nsplit = nsplit;
  prm.split_blocks = g_split_blocks;
  prm.part = part;
  prm.counters = counters;
  prm.wide_in = (reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) % 16 == 0;
  prm.wide_out = out_stride % 8 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
  dim3 grid(num_tiles * n_kv_heads * nsplit);
  const int rc = dtype == 0 ? fp::launch<__bf16>(G, grid, stream, prm)
                            : fp::launch<_Float16>(G, grid, stream, prm);
  if (rc) return rc;
  return static_cast<int>(hipGetLastError());
}
