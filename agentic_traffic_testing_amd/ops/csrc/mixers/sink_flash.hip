// Prefill of the paged softmax attention on the matrix cores (bf16, gfx950): flash form of the kernel in
// sink_attention.hip, same masks, sink, gates and pair epilogue (see there for what they mean).
//
// A piece of work = up to NW x 32 columns of one 64-token tile, a column = (query token, query head of the KV head's
// group); its workgroup walks blocks of 64 keys:
//   S^T[32 keys x 32 cols] = K . Q^T    (mfma 32x32x16, A = K rows from LDS, B = Q in registers)
//   O^T[vdim x 32 cols]   += V^T . P^T  (A = V^T rows from LDS, B = P^T from the S^T registers)
// A lane holds one column of S^T, so the softmax statistics are lane-local plus one exchange with
// lane ^ 32.  K rows are read in the order that swaps bits 2 and 3 of the row: the eight probabilities a
// lane half then holds per 16-key step belong to eight neighbouring keys, so a V^T fragment is one plain
// 16-byte read.  O and l are rescaled by every block's maximum.  (Letting the maximum lag by up to 2^8 saves time but then
// the largest weight is not exactly 1 and its rounding counts: error against 64 bits 3.2e-3 instead of 3.0e-3.)
//
// Pipeline: step i takes the scores of block i, the weights of block i - 1 and the value products of block i - 2, so that
// matrix and vector work of one step do not depend on each other, and `quick` deals them out by hand: a product (32 cycles
// of the matrix core), then as many vector instructions as fit behind it.  Left to the compiler the two ran one after the
// other, also across the two waves of a SIMD.  Steps with masks, at the window's edges and at both ends go part by part.  K
// of block i + 1 and V of block i - 1 travel straight from memory to LDS in the meantime: no registers, one wait and one
// barrier per step.  A wave moves keys of ONE 16-key group, which lie in one page (pages of 16 tokens or more), so its page
// and the group's place in it are scalars.
//
// Work: the hardware hands workgroups to the shader engines strictly in turn, a free place in one waits for its turn, and a
// workgroup's start (page list, queries, first keys: a chain of loads) costs 3 - 4 us; both together left CUs idle a fifth
// of the time.  So the latent form and the one of two maps, whose registers let a CU hold eight waves, run one workgroup of
// eight waves per CU that takes several pieces: sorted by length and dealt back and forth (their sums come out equal
// within 3 %), the next piece's page list, queries and first keys on their way behind the present one's last steps.  The
// others run one piece per workgroup of four waves, two workgroups per CU (figures at launch_sink_flash).
//
// Short prompts: with its start and its masked blocks a piece of few blocks is latency from end to end, so its first values
// come with its first keys, its queries behind its first pages, the parts' products have their operands on the way and go
// on different sums in turn, and a piece of up to three blocks goes without steps, its code in a row.  Kernel, us, one part
// after the other / pipeline without this / now: one prompt of 17 tokens, 32 + 8 heads 6.7 / 7.3 / 6.2, latent 15.3 / 15.0 / 12.0,
// 16 + 4 heads of 64 5.6 / 6.0 / 5.3, two maps of 8 9.4 / 11.4 / 9.0; of 85 tokens 8.6 / 9.2 / 7.6, 18.6 / 19.1 / 14.5, 6.8 / 7.3 /
// 6.3, 11.4 / 14.0 / 11.0; of 188 11.2 / 11.2 / 9.1, 22.0 / 22.2 / 17.5, 8.3 / 8.8 / 7.4, 14.0 / 16.7 / 13.3; two maps, several
// pieces per workgroup, 32 heads 14 x 220 59.4 / 64.5 / 60.1, 16 x 85 30.1 / 32.2 / 30.1; 475 tokens on 2000 cached ones 72 / 47 / 46,
// 139 / 116 / 97, 50 / 34 / 33, 50 / 45 / 39.
//
// Pair form: a workgroup's first four waves carry the first map, the other four the second one, over the
// same columns and one V block; at the end each wave finishes half of the channels.
//
// Bound: matrix cores and vector units together, over the whole kernel 44 and 48 % busy (128 wide; latent 47 and 45, two maps 18
// and 42, with few pieces per CU), at a clock that gives way.  4 prompts of ~1.9k tokens, us, one part after the other /
// pipeline with 32 keys per block of the latent form / now: 32 + 8 heads of 128 159 / 137 / 139, latent 257 / 227 / 208, two maps
// (8 heads, 5 x 1165, window 1024) 72 / 49 / 48, the last ones on a card that is 3 % slower (128 wide the last two are alike).
#include <algorithm>
#include <type_traits>
#include <utility>

#include "sink_attention.h"

namespace mixk {
namespace sf {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef u32x4 __attribute__((aligned(2))) u32x4_any;   // in memory, wherever it begins
typedef f32x4 __attribute__((aligned(4))) f32x4_any;
typedef __attribute__((address_space(3))) void* lds_ptr;

constexpr int KT = 2;                    // tiles of 32 keys per block
constexpr int kPages = 2048;             // page-table entries in LDS
constexpr int kSortTiles = 1024;         // tiles that a workgroup puts in order
constexpr int kBrief = 3;                // pieces of so many blocks take them one after the other (the line as measured in flash_prefill.hip)
constexpr int kPieces = 64;              // pieces of work per workgroup in LDS
// Pair form: in the first blocks each of the two tiles has its own maximum.  Largest weights are rounded to exactly 1;
// with a maximum per 64 keys there are fewer of them than per 32, half of the difference from the first block, 90 %
// from four.  Error against 64 bits, prompts of 600 (1e-3): one per block 2.345, the first four split 2.328.  (One map:
// sums of the rounded weights make up for more than that.)
constexpr int kSplitBlocks = 4;
constexpr float kLog2e = 1.44269504088896341f;
#define SF_INLINE __attribute__((always_inline))

// larger value, or the sum, of the lane's and lane ^ 32's (the builtin's two results are taken for one where both operands
// are the same value)
__device__ __forceinline__ f32x2 halves(float v) {
  float a = v, b = v;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
#endif
  return f32x2{a, b};
}
__device__ __forceinline__ float both(float v) {
  const f32x2 x = halves(v);
  return fmaxf(x[0], x[1]);
}
__device__ __forceinline__ float both_sum(float v) {
  const f32x2 x = halves(v);
  return x[0] + x[1];
}
// 16 (send4: 4) bytes per lane from base + offset to 64 lanes' LDS from address `to` on, without registers; there after
// wait_sent().  (After the builtin the compiler makes every read of LDS wait for all transfers.)  The base goes through a
// scalar move: five wait states belong between a vector instruction that writes a scalar register, such as the reload of
// a spilled one, and a memory instruction that reads it, and the compiler does not put them in front of assembly.  (The
// same in flash_prefill.hip, a library of its own.)
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
__device__ __forceinline__ void send4(const void* base, uint32_t offset, uint32_t to) {
#if defined(__HIP_DEVICE_COMPILE__)
  uint64_t from;
  asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 %0, %2\n\tglobal_load_lds_dword %1, %0"
               : "=&s"(from) : "v"(offset), "s"(base), "s"(to) : "m0", "memory");
#endif
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr)(const_cast<void*>(p))));
}
__device__ __forceinline__ void wait_sent() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
}
// the value, computed anew from here on (what follows from it is not kept in registers from one piece of work to the next)
__device__ __forceinline__ int fresh(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(v));
#endif
  return v;
}
// the value is there at this point of the program
template <typename X>
__device__ __forceinline__ void hold(const X& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" ::"v"(x));
#endif
}

// f(0), f(1), ... as constants (a loop of so much in a turn is not unrolled)
template <int... N, typename F>
__device__ __forceinline__ void each(std::integer_sequence<int, N...>, const F& f) {
  (f(std::integral_constant<int, N>()), ...);
}

// DK = 16 ND (q / k width), DV = 32 NV (value width).  BORDERS: the caches begin on 16-byte borders, as transfers past the
// registers need them; otherwise blocks go through registers, part by part.
template <int ND, int NV, int NMAP, int NW, bool WIN, bool BORDERS>
__global__ void __launch_bounds__(NW * 64, 2)
sink_flash_kernel(void* __restrict__ out, const __bf16* __restrict__ q, const __bf16* __restrict__ k_cache,
                  const __bf16* __restrict__ v_cache, AttnArgs a, int num_tiles, int chunks, int workers) {
  constexpr int DK = 16 * ND, DV = 32 * NV, CW = NW / NMAP, COLS = CW * 32, BLK = 32 * KT;
  constexpr bool MANY = NW == 8;                    // a workgroup takes several pieces of work in turn
  constexpr int GR = 2 * KT, WPG = NW / GR;         // 16-key groups of a block, waves per group
  constexpr int CK = DK / 8;                        // 16-byte chunks of a K row
  constexpr int KN = CK / 4, KU = (KN + WPG - 1) / WPG;   // transfers (64 chunks) of K per group and map; per wave
  constexpr int VN = NV, VU = (VN + WPG - 1) / WPG;
  constexpr int RB = CK < 16 ? 16 / CK : 1;         // K rows per 256 bytes
  constexpr int KB = NMAP * BLK * DK, VB = DV * BLK;   // elements of a buffer
  constexpr int MT = NMAP, TPM = KT / MT;           // maxima per block, tiles per maximum
  // Queries of 256 and values of 192 channels take 160 registers, and two tiles' scores beside the ones before them all of the
  // others: the tiles take turns, a tile's scores in the registers of the same tile of the block before.
  constexpr bool TURNS = ND > 8;
  static_assert(NMAP == 1 || NW == 8, "pair form: four waves per map");
  __shared__ __attribute__((aligned(1024))) __bf16 lds_k[2 * KB], lds_v[2 * VB];
  __shared__ __attribute__((aligned(1024))) char lds_x[NMAP == 2 ? 65536 : 16];
  __shared__ float lds_ss[NMAP == 2 ? NW : 1][32];
  __shared__ int lds_bt[MANY ? 2 : 1][kPages];
  __shared__ int lds_piece[MANY ? kPieces : 1][8];
  const int H = a.H, G = a.G, bs = a.block_size;
  const int rep = H / G, GO = G / NMAP, GV = G / a.v_share;
  // KV head fastest: workgroups are dealt round-robin to the eight XCDs, so with eight KV heads a head's
  // K / V stay in one L2.
  const int bid = static_cast<int>(blockIdx.x);
  const int g = bid % GO;                           // K head (pair form: V head, K heads 2 g and 2 g + 1)
  const int worker = bid / GO;
  const int gv = NMAP == 2 ? g : g / a.v_share;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int mp = NMAP == 2 ? w / CW : 0;            // the wave's map
  const float scale2 = a.scale * kLog2e;
  const uint32_t per = 0xffffffffu / rep + 1;       // (columns x rep < 2^32; rep 1: 0)
  auto token_of = [&](int c) SF_INLINE { return rep == 1 ? c : static_cast<int>(__umulhi(static_cast<uint32_t>(c), per)); };

  // ---- transfers: wave w moves keys of group w % GR, all in one page.  K rows lie in LDS as they are, V as
  // [group][channel][16 keys]; the 16-byte chunks of a K row and the halves of a V row change places so that the
  // fragments' reads have no bank conflicts
  const int sg = w % GR, part = w / GR;
  uint32_t k_src[TURNS ? 1 : KU];   // bytes (TURNS: the others are worked out where they are used)
#pragma unroll
  for (int u = 0; u < (TURNS ? 1 : KU); ++u) {
    const int row = (u * WPG + part) * (64 / CK) + lane / CK;   // of the group
    k_src[u] = 2u * (row * DK + ((lane % CK) ^ ((row / RB) & (CK - 1) & 15)) * 8);
  }
  const int v_half = 8 * ((lane ^ (lane >> 4)) & 1);
  uint32_t v_src[TURNS ? 1 : VU];
#pragma unroll
  for (int u = 0; u < (TURNS ? 1 : VU); ++u) v_src[u] = 2u * ((32 * (u * WPG + part) + (lane >> 1)) * bs + v_half);
  const int k_lds = 16 * sg * DK + part * 512, v_lds = sg * DV * 16 + part * 512;
  const __bf16* k_base = k_cache + static_cast<int64_t>(NMAP * g) * bs * DK;
  const __bf16* v_base = v_cache + static_cast<int64_t>(gv) * DV * bs;
  const uint32_t k_page = G * bs * DK, v_page = GV * DV * bs;
  auto k_at = [&](int pg, int k0) SF_INLINE {
    return k_base + static_cast<uint64_t>(static_cast<uint32_t>(pg)) * k_page + ((k0 + 16 * sg) & (bs - 1)) * DK;
  };
  auto v_at = [&](int pg, int k0) SF_INLINE {
    return v_base + static_cast<uint64_t>(static_cast<uint32_t>(pg)) * v_page + ((k0 + 16 * sg) & (bs - 1));
  };
  // (`b`: which of the two buffers, its lowest bit)
  const uint32_t k_to = lds_address(lds_k) + 2 * k_lds, v_to = lds_address(lds_v) + 2 * v_lds;
  auto move16 = [&](const __bf16* base, uint32_t offset, uint32_t to) SF_INLINE {
    if constexpr (BORDERS) send16(base, offset, to);
    else copy16(base, offset, to, fresh(lane));
  };
  auto send_k = [&](const __bf16* kb, int b, int u) SF_INLINE {
    const uint32_t to = k_to + (b & 1) * 2 * KB + u % KU * WPG * 1024 + u / KU * 2 * BLK * DK;
    if constexpr (TURNS) {   // rows 4 further on: bits 2 and 3 of the chunk's place
      static_assert(!TURNS || (NMAP == 1 && CK == 32 && WPG == 2), "four rows per transfer of the group's waves");
      move16(kb + 4 * u * DK, fresh(k_src[0]) ^ (64u * u), to);
    } else if (KU * WPG == KN || (u % KU) * WPG + part < KN) {
      move16(kb + (u / KU) * bs * DK, k_src[u % KU], to);
    }
  };
  auto send_v = [&](const __bf16* vb, int b, int u) SF_INLINE {
    const uint32_t to = v_to + (b & 1) * 2 * VB + u * WPG * 1024;
    if (VU * WPG == VN || u * WPG + part < VN) move16(TURNS ? vb + 32 * u * WPG * bs : vb, v_src[TURNS ? 0 : u], to);
  };
  // ---- fragments.  A row of the score products: key with bits 2 and 3 swapped
  const int vfrag = r * 16 + 8 * (h ^ ((r >> 3) & 1));
  constexpr int KO = ND < 8 ? ND : 8;
  typedef int Places[KO];   // of the first steps of a row
  auto places_of = [&](int ln, Places& to) SF_INLINE {
    const int row = (ln & 19) | ((ln & 4) << 1) | ((ln & 8) >> 1);
    const int at = mp * BLK * DK + row * DK + ((ln >> 5) ^ ((row / RB) & (CK - 1) & 15)) * 8;
#pragma unroll
    for (int st = 0; st < KO; ++st) to[st] = at ^ (16 * st);
  };
  Places kept;
  if (!TURNS) places_of(lane, kept);
  auto places = [&](Places& to) SF_INLINE {   // (TURNS: no registers to keep them)
    if (TURNS) return places_of(fresh(lane), to);
#pragma unroll
    for (int st = 0; st < KO; ++st) to[st] = kept[st];
  };
  auto kf = [&](const __bf16* b, const Places& at, int t, int st) SF_INLINE {
    return *reinterpret_cast<const bf16x8*>(b + 32 * t * DK + at[st % 8] + st / 8 * 128);
  };
  auto vf = [&](const __bf16* b, int vt, int ks) SF_INLINE {
    return *reinterpret_cast<const bf16x8*>(b + vfrag + ks * DV * 16 + vt * 512);
  };

  // ---- the workgroup's pieces of work, `mine` of them
  const int pieces = num_tiles * chunks;
  // every other round the other way about: long pieces come together with short ones
  auto rank_of = [&](int k) { return k * workers + ((k & 1) ? workers - 1 - worker : worker); };
  int mine = pieces / workers;
  if (rank_of(mine) < pieces) ++mine;
  struct Piece {
    int s, qo, col0, row0, n, kvlen;
  };
  auto cols_of = [&](const Piece& p) SF_INLINE { return min(kTileTokens, p.n - p.qo) * rep; };
  auto kend_of = [&](const Piece& p) SF_INLINE {
    return p.kvlen - p.n + p.qo + token_of(min(cols_of(p), p.col0 + COLS) - 1) + 1;
  };
  auto fetch = [&](int item) SF_INLINE {
    Piece p;
    const int tile = item / chunks;
    p.s = a.tile_seq[tile], p.qo = a.tile_qoff[tile], p.col0 = item % chunks * COLS;
    p.row0 = a.seq_qstart[p.s], p.n = a.seq_qstart[p.s + 1] - p.row0, p.kvlen = a.seq_kvlen[p.s];
    // nothing to do: an empty sequence, a chunk past a short tile's columns
    if (p.n <= 0 || p.kvlen <= 0 || p.qo >= p.n || p.col0 >= min(kTileTokens, p.n - p.qo) * rep) p.n = 0;
    return p;
  };
  // (one piece each: no trip through LDS)
  const bool many = MANY && pieces > workers;
  const Piece only = fetch(pieces - 1 - worker);
  if (many) {
    // Long ones first: a piece's rank among the tiles' numbers of blocks, found by bisection of the keys (blocks, then
    // place in the list: no two are alike), which every wave holds for itself
    constexpr int KR = kSortTiles / 64;
    if (num_tiles <= kSortTiles) {
      unsigned int key[KR];
      Piece own[KR];
      const int most = (a.bt_width << a.bs_shift) / BLK + 2;
#pragma unroll
      for (int i = 0; i < KR; ++i) {
        key[i] = 0;
        own[i] = Piece{};
        if (64 * i >= num_tiles) continue;
        const int t = min(lane + 64 * i, num_tiles - 1);
        own[i] = fetch(t * chunks);
        const int first = window_start(own[i].kvlen - own[i].n + own[i].qo, a.window);
        if (lane + 64 * i < num_tiles)
          key[i] = static_cast<unsigned int>(min(max((own[i].kvlen - own[i].n + min(own[i].n, own[i].qo + kTileTokens) - first) / BLK, 0) + 1, most)) << 10 | (kSortTiles - 1 - t);
      }
      for (int k = w; k < mine; k += NW) {
        const int rk = rank_of(k), want = rk / chunks, col0 = (chunks - 1 - rk % chunks) * COLS;
        unsigned int v = 0;   // the largest value that more than `want` keys reach: that rank's key
        for (int bit = 31 - __builtin_clz(most << 10 | (kSortTiles - 1)); bit >= 0; --bit) {
          const unsigned int c = v | 1u << bit;
          int n = 0;
#pragma unroll
          for (int i = 0; i < KR; ++i) {
            if (64 * i >= num_tiles) break;
            n += __builtin_popcountll(__ballot(key[i] >= c));
          }
          if (n > want) v = c;
        }
#pragma unroll
        for (int i = 0; i < KR; ++i)
          if (key[i] == v) {
            const Piece& p = own[i];
            int* e = lds_piece[k];
            e[0] = p.s, e[1] = p.qo, e[2] = col0, e[3] = p.row0, e[4] = col0 < cols_of(p) ? p.n : 0, e[5] = p.kvlen;
          }
      }
    } else {
      for (int k = w; k < mine; k += NW) {
        const Piece p = fetch(pieces - 1 - rank_of(k));
        int* e = lds_piece[k];
        if (lane == 0) e[0] = p.s, e[1] = p.qo, e[2] = p.col0, e[3] = p.row0, e[4] = p.n, e[5] = p.kvlen;
      }
    }
    __syncthreads();
  }
  // the next piece with work, from number k on
  auto next_piece = [&](int& k, Piece& p) SF_INLINE {
    if (!many) {
      p = only;
      return k == 0 && p.n > 0;
    }
    // (each workgroup begins at another of its pieces: queries and results of all of them do not come at once)
    for (; k < mine; ++k) {
      const int* e = lds_piece[MANY ? (k + worker) % mine : 0];
      p.n = __builtin_amdgcn_readfirstlane(e[4]);
      if (p.n == 0) continue;
      p.s = __builtin_amdgcn_readfirstlane(e[0]), p.qo = __builtin_amdgcn_readfirstlane(e[1]);
      p.col0 = __builtin_amdgcn_readfirstlane(e[2]), p.row0 = __builtin_amdgcn_readfirstlane(e[3]);
      p.kvlen = __builtin_amdgcn_readfirstlane(e[5]);
      return true;
    }
    return false;
  };
  // ---- what a piece needs before its first step
  auto pages_of = [&](const Piece& p) SF_INLINE { return min((kend_of(p) + bs - 1) >> a.bs_shift, kPages); };   // (the launcher bounds the table)
  // key blocks: the kept keys in front of the window, then from the window's start (block-aligned)
  auto klow_of = [&](const Piece& p) SF_INLINE { return window_start(p.kvlen - p.n + p.qo + token_of(p.col0), a.window); };
  auto first_key = [&](const Piece& p) SF_INLINE { return min(a.keep, klow_of(p) & ~(BLK - 1)) > 0 ? 0 : klow_of(p) & ~(BLK - 1); };
  auto send_pages = [&](const Piece& p, int from, int list) SF_INLINE {   // of the page list from entry `from` on, into list 0 or 1
    const int* btg = a.block_tables + static_cast<int64_t>(p.s) * a.bt_width;
    const int npages = pages_of(p), ln = fresh(lane);
    for (int i = from + w * 64; i < npages; i += NW * 64)
      if (i + ln < npages) send4(btg, 4u * (i + ln), lds_address(lds_bt) + 4 * (list * kPages + i));
  };
  auto send_block_k = [&](const int* bt, int last_page, int k0, int b) SF_INLINE {
    const __bf16* kb = k_at(__builtin_amdgcn_readfirstlane(bt[min((k0 + 16 * sg) >> a.bs_shift, last_page)]), k0);
#pragma unroll
    for (int u = 0; u < NMAP * KU; ++u) send_k(kb, b, u);
  };
  bf16x8 qf[ND];
  auto load_q = [&](const Piece& p, bool real) SF_INLINE {
    const int ln = fresh(lane), col = p.col0 + (w % CW) * 32 + (ln & 31);
    const bool valid = col < cols_of(p);
    const int tok = valid ? token_of(col) : 0, head = (NMAP * g + mp) * rep + (valid ? col - tok * rep : 0);
    // (`real` false: nobody reads them; one row, whose lines are one)
    const __bf16* qp = q + (real ? (p.row0 + p.qo + tok) * a.q_stride + static_cast<int64_t>(head) * DK + 8 * (ln >> 5) : 0);
#pragma unroll
    for (int st = 0; st < ND; ++st) qf[st] = *reinterpret_cast<const bf16x8*>(qp + 16 * st);
  };

  int pn = 0;
  Piece now, nxt;
  if (!next_piece(pn, now)) return;
  // (queries are there before a loop, which would wait for its transfers with them)
  auto hold_q = [&]() SF_INLINE {
#pragma unroll
    for (int st = 0; st < ND; ++st) hold(qf[st]);
  };
  {   // queries on their way behind the first pages, which do not wait for them
    const int* btg = a.block_tables + static_cast<int64_t>(now.s) * a.bt_width;
    const int npages = pages_of(now), page = btg[max(min(tid, npages - 1), 0)];
    load_q(now, true);
    if (tid < npages) lds_bt[0][tid] = page;
    if (npages > NW * 64) {
      send_pages(now, NW * 64, 0);
      wait_sent();
    }
  }
  __syncthreads();
  send_block_k(lds_bt[0], pages_of(now) - 1, first_key(now), 0);

  bool was_brief = false;   // the piece before: the present one's first keys and queries are still on their way
  for (int turn = 0;; ++turn) {
    ++pn;
    nxt = now;
    const bool more = next_piece(pn, nxt);
    const int* const bt = lds_bt[MANY ? turn & 1 : 0];
    const int qo = now.qo, row0 = now.row0, kvlen = now.kvlen, col0 = now.col0;
    const int cols_total = cols_of(now);
    const int ctx = kvlen - now.n + qo;               // position of the tile's first token
    const int wcol = col0 + (w % CW) * 32;            // the wave's first column
    const bool wave_on = wcol < cols_total;
    const int w_last = min(cols_total, wcol + 32) - 1;
    const int pos_first = ctx + token_of(wcol), pos_last = ctx + token_of(max(w_last, 0));
    const int kend = kend_of(now), last_page = pages_of(now) - 1;
    const int klow = klow_of(now), kbeg = klow & ~(BLK - 1);   // no column sees keys in [keep, klow)
    const int nk = (min(a.keep, kbeg) + BLK - 1) / BLK;
    const int nb = nk + (kend - kbeg + BLK - 1) / BLK;
    auto block_key = [&](int b) SF_INLINE { return b < nk ? b * BLK : kbeg + (b - nk) * BLK; };
    // the lane's column (worked out anew where it is used)
    struct Column {
      bool valid;
      int tok, member;   // member: of the KV head's group
    };
    auto column = [&](int ln) SF_INLINE {
      Column c;
      const int col = wcol + (ln & 31);
      c.valid = col < cols_total;
      c.tok = c.valid ? token_of(col) : 0;
      c.member = c.valid ? col - c.tok * rep : 0;
      return c;
    };
    const Column c0 = column(fresh(lane));
    const int head = (NMAP * g + mp) * rep + c0.member;
    float m = kNegBig, l = 0.f;   // l: of the lane's keys
    if (a.sink) {   // the sink is the state the online softmax starts from (log2 units)
      m = a.sink_val != nullptr ? a.sink_val[head] * kLog2e : 0.f;
      l = fresh(lane) < 32 ? 1.f : 0.f;
    }
    f32x16 O[NV];
#pragma unroll
    for (int vt = 0; vt < NV; ++vt)
#pragma unroll
      for (int i = 0; i < 16; ++i) O[vt][i] = 0.f;

    // keys at or past kend read a clamped page or stale slots, keys in front of the window whatever is there: their
    // scores are masked and their V zeroed (0 x NaN) once it is there, by the wave that fetched it
    auto seen = [&](int t) SF_INLINE { return t < kend && (!WIN || t >= klow || t < a.keep); };
    auto send_block_v = [&](int k0, int b) SF_INLINE {
      const __bf16* vb = v_at(__builtin_amdgcn_readfirstlane(bt[min((k0 + 16 * sg) >> a.bs_shift, last_page)]), k0);
#pragma unroll
      for (int u = 0; u < VU; ++u) send_v(vb, b, u);
    };
    auto clear_block_v = [&](int k0, __bf16* to) SF_INLINE {
      if (k0 + BLK <= kend && !(WIN && k0 < klow && k0 + BLK > a.keep)) return;
      const int ln = fresh(lane), key = k0 + 16 * sg + 8 * ((ln ^ (ln >> 4)) & 1);
      u32x4 seen2;
#pragma unroll
      for (int j = 0; j < 4; ++j) seen2[j] = (seen(key + 2 * j) ? 0x0000ffffu : 0u) | (seen(key + 2 * j + 1) ? 0xffff0000u : 0u);
#pragma unroll
      for (int u = 0; u < VU; ++u)
        if (VU * WPG == VN || u * WPG + part < VN) *reinterpret_cast<u32x4*>(to + v_lds + u * WPG * 512 + ln * 8) &= seen2;
    };

    // keys at or below the window start of the wave's latest column are outside somebody's window
    const int edge_lo = a.window > 0 ? pos_last - a.window : -1;
    const int low_first = window_start(pos_first, a.window);   // no column of the wave sees keys below
    float carry = 1.f;   // pair form: of the second tile's maximum over the first one's, until the value products
    auto needed = [&](int b) SF_INLINE {
      const int k0 = block_key(b);
      return b >= 0 && b < nb && wave_on && k0 <= pos_last && (k0 + BLK > low_first || k0 < a.keep);
    };
    // (products with their operands on the way, on different sums in turn: left to the compiler each waited for its own)
    auto scores = [&](const __bf16* from, f32x16 (&S)[KT]) SF_INLINE {
      Places at;
      places(at);
      constexpr int N = KT * ND, LA = TURNS ? 3 : 4;
      bf16x8 fr[N];
      auto read = [&](int n) SF_INLINE { fr[n] = kf(from, at, n % KT, n / KT); };
#pragma unroll
      for (int n = 0; n < LA; ++n) read(n);
      each(std::make_integer_sequence<int, N>(), [&](auto slot) SF_INLINE {
        constexpr int n = slot;
        __builtin_amdgcn_sched_barrier(0);
        if (n + LA < N) read(n + LA);
        S[n % KT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[n], qf[n / KT], n < KT ? f32x16{} : S[n % KT], 0, 0, 0);
      });
      __builtin_amdgcn_sched_barrier(0);
    };
    auto rescale = [&](float alpha) SF_INLINE {
#pragma unroll
      for (int vt = 0; vt < NV; ++vt)
#pragma unroll
        for (int i = 0; i < 16; ++i) O[vt][i] *= alpha;
    };
    auto values = [&](const __bf16* from, const bf16x8 (&P)[2 * KT], bool split) SF_INLINE {
      constexpr int N = 2 * TPM * NV, LA = TURNS ? 3 : 4;
      each(std::make_integer_sequence<int, MT>(), [&](auto half) SF_INLINE {
        constexpr int e = half;
        if (e > 0 && split && __any(carry != 1.f)) rescale(carry);
        bf16x8 fr[N];
        auto read = [&](int n) SF_INLINE { fr[n] = vf(from, n % NV, 2 * e * TPM + n / NV); };
#pragma unroll
        for (int n = 0; n < LA; ++n) read(n);
        each(std::make_integer_sequence<int, N>(), [&](auto slot) SF_INLINE {
          constexpr int n = slot;
          __builtin_amdgcn_sched_barrier(0);
          if (n + LA < N) read(n + LA);
          O[n % NV] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[n], P[2 * e * TPM + n / NV], O[n % NV], 0, 0, 0);
        });
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    // a maximum and what it makes of the sums so far (a sink may be infinite or NaN: an infinity stays the maximum, and its
    // own factor is 1; a NaN stays)
    auto higher = [](float t, float m) SF_INLINE { return t > m ? t : m; };
    auto factor = [](float t, float m) SF_INLINE { return t > m ? __builtin_amdgcn_exp2f(m - t) : 1.f; };
    auto weights = [&](int b, f32x16 (&S)[KT], bf16x8 (&P)[2 * KT]) SF_INLINE {
      const int k0 = block_key(b);
      if (k0 + BLK - 1 > pos_first || (WIN && k0 <= edge_lo)) {
        const int ln = fresh(lane);
        const Column c = column(ln);
        const int qpos = c.valid ? ctx + c.tok : -1;   // no key is visible to a column that is not there
        // Register i of tile t holds key k0 + 8 h + 32 t + 16 (i >> 3) + (i & 7): bit 16 (i >> 3) + (i & 7) of a tile's
        // word.  (A comparison per key, whose result waits in a scalar register: 800 cycles per block.)
        auto below = [](int n) SF_INLINE { return n <= 0 ? 0u : n >= 32 ? ~0u : (1u << n) - 1; };
#pragma unroll
        for (int t = 0; t < KT; ++t) {
          const int k8 = k0 + 8 * (ln >> 5) + 32 * t;
          unsigned int out = ~below(qpos + 1 - k8);
          if (WIN) out |= below(window_start(qpos, a.window) - k8) & ~below(a.keep - k8);
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const float v = S[t][i];
            const unsigned int x = __builtin_amdgcn_sbfe(out, 16 * (i >> 3) + (i & 7), 1);
            S[t][i] = __builtin_bit_cast(float, (x & 0xff800000u) | (~x & __builtin_bit_cast(unsigned int, v)));
          }
        }
      }
      float tmax[MT], mt[MT], psum[MT];
#pragma unroll
      for (int e = 0; e < MT; ++e) {
        tmax[e] = -INFINITY;
#pragma unroll
        for (int t = e * TPM; t < (e + 1) * TPM; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) tmax[e] = fmaxf(tmax[e], S[t][i]);
      }
#pragma unroll
      for (int e = 0; e < MT; ++e) tmax[e] = fmaxf(both(tmax[e]) * scale2, kNegBig);   // (all keys masked: never above a maximum)
      if (MT > 1 && b >= kSplitBlocks) tmax[0] = fmaxf(tmax[0], tmax[MT - 1]);
      mt[0] = higher(tmax[0], m);
      if (__any(tmax[0] > m)) {
        const float alpha = factor(tmax[0], m);
        l *= alpha;
        rescale(alpha);
      }
      mt[MT - 1] = MT > 1 ? higher(tmax[MT - 1], mt[0]) : mt[0];
      m = mt[MT - 1];
#pragma unroll
      for (int e = 0; e < MT; ++e) psum[e] = 0.f;   // of the weights as the value products take them, rounded
#pragma unroll
      for (int ks = 0; ks < 2 * KT; ++ks) {
        u32x4 wv;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int t = ks >> 1, i = 8 * (ks & 1) + 2 * j;
          const f32x2 x{__builtin_amdgcn_exp2f(__builtin_fmaf(S[t][i], scale2, -mt[t / TPM])),
                        __builtin_amdgcn_exp2f(__builtin_fmaf(S[t][i + 1], scale2, -mt[t / TPM]))};
          wv[j] = __builtin_bit_cast(unsigned int, __builtin_convertvector(x, bf16x2));
          psum[t / TPM] += __builtin_bit_cast(float, wv[j] << 16) + __builtin_bit_cast(float, wv[j] & 0xffff0000u);
        }
        P[ks] = __builtin_bit_cast(bf16x8, wv);
      }
      l += psum[0];
      if (MT > 1) {
        carry = factor(tmax[MT - 1], mt[0]);
        l = l * carry + psum[MT - 1];
      }
    };
    // One block's scores, the weights of the one before and the value products of the one before that: a product and a
    // few vector instructions in turn
    auto quick = [&](auto parted, const Places& at, bool one_max, const __bf16* kr, const __bf16* vr, int b, int bk, int bv, const f32x16 (&Si)[KT],
                     f32x16 (&So)[KT], const bf16x8 (&Pi)[2 * KT], bf16x8 (&Po)[2 * KT]) SF_INLINE {
      constexpr int NP = 2 * KT * NV, NF = NP + KT * ND, LA = TURNS ? 2 : 3;
      constexpr bool MSUM = !TURNS;   // the weights' sums by products with a half
      constexpr int NS = NF + (MSUM ? 2 * KT : 0);
      constexpr int WE = (MSUM ? 56 : 88) * KT, WR = 16 * NV;
      constexpr int NB = std::min(std::max(NP, NS * WE / (WE + WR)), NS - 4 * KT - 1);   // slots of the exponentials; then O's factors
      constexpr int SUM0 = NB + 1;                            // the weights' sums: products with a half, every other slot
      static_assert(!MSUM || SUM0 + 4 * KT <= NS, "room for the sums");
      // two maxima: the first tile's value products of all channels, a factor, the second tile's
      constexpr bool PARTED = decltype(parted)::value;
      constexpr int KP = PARTED ? 2 : 2 * KT;   // value products of a channel tile in a row
      auto vt_of = [](int n) { return n % (KP * NV) / (2 * KP) * 2 + n % 2; };
      auto ks_of = [](int n) { return n / (KP * NV) * KP + n % (2 * KP) / 2; };
      bf16x8 fr[NF];
      auto tile_of = [](int n) { return TURNS ? (n - NP) / ND : (n - NP) % KT; };
      auto step_of = [](int n) { return TURNS ? (n - NP) % ND : (n - NP) / KT; };
      // (TURNS: a tile's weights are done before the products that take its scores' registers)
      static_assert(!TURNS || (NB <= KT * NP && NB <= NP + ND), "scores and weights of a tile in the same registers");
      auto frag = [&](int n) SF_INLINE { fr[n] = n < NP ? vf(vr, vt_of(n), ks_of(n)) : kf(kr, at, tile_of(n), step_of(n)); };
      const int kpg = bt[min((bk + 16 * sg) >> a.bs_shift, last_page)], vpg = bt[min((bv + 16 * sg) >> a.bs_shift, last_page)];
#pragma unroll
      for (int n = 0; n < LA; ++n) frag(n);
      __builtin_amdgcn_sched_barrier(0);
      float tm[2 * KT];
#pragma unroll
      for (int c = 0; c < 2 * KT; ++c) {
        tm[c] = kNegBig;
#pragma unroll
        for (int i = 0; i < 8; ++i) tm[c] = fmaxf(tm[c], Si[c >> 1][8 * (c & 1) + i]);
      }
      float top[2] = {fmaxf(tm[0], tm[1]), fmaxf(tm[2 * KT - 2], tm[2 * KT - 1])};
      if (!PARTED || one_max) top[0] = fmaxf(top[0], top[1]);
      const float t0 = both(top[0]) * scale2, m0 = higher(t0, m), alpha = factor(t0, m);
      const float before = carry;
      m = m0;
      if constexpr (PARTED) {
        const float t1 = both(top[1]) * scale2;
        m = higher(t1, m0);
        carry = factor(t1, m0);
      }
      const float mt[2] = {m0, m};
      l *= alpha;
      const __bf16 *kb = nullptr, *vb = nullptr;
      unsigned int wv[8 * KT];
      f32x16 sums;
      float ps[2] = {0.f, 0.f};
      bf16x8 half;
#pragma unroll
      for (int j = 0; j < 8; ++j) half[j] = static_cast<__bf16>(0.5f);   // (the lane's and lane ^ 32's l are added at the end)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        sums[i] = 0.f;
#pragma unroll
        for (int t = 0; t < KT && !TURNS; ++t) So[t][i] = 0.f;
      }
      each(std::make_integer_sequence<int, NS>(), [&](auto slot) SF_INLINE {
        constexpr int n = slot;
        __builtin_amdgcn_sched_barrier(0);
        const bool summing = MSUM && n >= SUM0 && n < SUM0 + 4 * KT && (n - SUM0) % 2 == 0;
        const int f = !MSUM || n < SUM0 ? n : n < SUM0 + 4 * KT ? SUM0 + (n - SUM0) / 2 : n - 2 * KT;   // fragment of this slot
        if (!summing && f + LA < NF) frag(f + LA);
        if (summing) {
          const int ks = (n - SUM0) / 2;
          if (PARTED && ks == 2) sums[0] *= carry;
          sums = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              half, __builtin_bit_cast(bf16x8, (u32x4{wv[4 * ks], wv[4 * ks + 1], wv[4 * ks + 2], wv[4 * ks + 3]})), sums, 0, 0, 0);
          hold(sums);
        } else if (f < NP) {
          const int vt = vt_of(f);
          O[vt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[f], Pi[ks_of(f)], O[vt], 0, 0, 0);
          hold(O[vt]);
        } else {
          const int t = tile_of(f), st = step_of(f);
          So[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[f], qf[st], TURNS && st == 0 ? f32x16{} : So[t], 0, 0, 0);
          hold(So[t]);
        }
        if (n == 1) {
          kb = k_at(__builtin_amdgcn_readfirstlane(kpg), bk);
          vb = v_at(__builtin_amdgcn_readfirstlane(vpg), bv);
        }
        // the next blocks on their way
        if (n >= 2 && n < 2 + NMAP * KU) send_k(kb, b, n - 2);
        if (n >= 2 + NMAP * KU && n < 2 + NMAP * KU + VU) send_v(vb, b, n - 2 - NMAP * KU);
        if constexpr (PARTED) {   // O of two channel tiles between their products of the first and of the second tile
          constexpr int G2 = 2 * KP;
          if (n >= G2 && n < G2 + KP * NV) {
            const int pair2 = (n - G2) / G2 * 2, at = (n - G2) % G2;
#pragma unroll
            for (int c = 32 * at / G2; c < 32 * (at + 1) / G2; ++c) O[pair2 + c / 16][c % 16] *= before;
            hold(O[pair2]);
            hold(O[pair2 + 1]);
          }
        }
        if (n < NB) {
#pragma unroll
          for (int u = 8 * KT * n / NB; u < 8 * KT * (n + 1) / NB; ++u) {
            const int t = u / 8, i = 2 * (u % 8);
            const float mx = PARTED ? mt[t] : m;
            const f32x2 x{__builtin_amdgcn_exp2f(__builtin_fmaf(Si[t][i], scale2, -mx)),
                          __builtin_amdgcn_exp2f(__builtin_fmaf(Si[t][i + 1], scale2, -mx))};
            wv[u] = __builtin_bit_cast(unsigned int, __builtin_convertvector(x, bf16x2));
            if constexpr (!MSUM)
              ps[u % 2] += __builtin_bit_cast(float, wv[u] << 16) + __builtin_bit_cast(float, wv[u] & 0xffff0000u);
            hold(wv[u]);
          }
        } else {
#pragma unroll
          for (int c = WR * (n - NB) / (NS - NB); c < WR * (n - NB + 1) / (NS - NB); ++c) {
            O[c / 16][c % 16] *= alpha;
            hold(static_cast<float>(O[c / 16][c % 16]));
          }
        }
      });
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < 2 * KT; ++ks)
        Po[ks] = __builtin_bit_cast(bf16x8, (u32x4{wv[4 * ks], wv[4 * ks + 1], wv[4 * ks + 2], wv[4 * ks + 3]}));
      l = !MSUM ? l + (ps[0] + ps[1]) : PARTED ? l * carry + sums[0] : l + sums[0];
    };

    // ---- step i: scores of block i, weights of block i - 1, value products of block i - 2; K of block i + 1 and V of
    // block i - 1 on their way to the other buffers
    f32x16 S[KT];
    bf16x8 P[2 * KT];
    auto kbuf = [&](int i) SF_INLINE { return lds_k + (i & 1) * KB; };
    auto vbuf = [&](int i) SF_INLINE { return lds_v + (i & 1) * VB; };
    // steps [quick0, quick1): block i - 1 has no masked key, block i is needed
    const int above = WIN ? max(edge_lo, low_first) : -1;   // (block i - 2 has a key that the wave sees)
    const int quick0 = max(nk + 2, nk + ((above + BLK - kbeg) / BLK) + 1);
    const int quick1 = BORDERS && wave_on ? nk + min(min(nb - nk, (pos_first + 1 - kbeg + BLK) / BLK), (pos_last - kbeg) / BLK + 1) : 0;
    auto quick_step = [&](auto parted, const Places& at, int i, const f32x16 (&Si)[KT], f32x16 (&So)[KT], const bf16x8 (&Pi)[2 * KT],
                          bf16x8 (&Po)[2 * KT]) SF_INLINE {
      quick(parted, at, i - 1 >= kSplitBlocks, kbuf(i), vbuf(i), i + 1, kbeg + (i + 1 - nk) * BLK,
            kbeg + (i - 1 - nk) * BLK, Si, So, Pi, Po);
      wait_sent();
      __syncthreads();
    };
    auto quick_two = [&](auto parted, const Places& at, int i) SF_INLINE {
      f32x16 other[KT];
      f32x16 (&S2)[KT] = TURNS ? S : other;
      bf16x8 P2[2 * KT];
      quick_step(parted, at, i, S, S2, P, P2);
      quick_step(parted, at, i + 1, S2, S, P2, P);
    };
    bf16x4 gates[8];   // pair form: of the wave's half of the channels
    auto load_gates = [&]() SF_INLINE {
      if (NMAP == 1 || a.gate == nullptr) return;
      const int ln = fresh(lane);
      const Column c = column(ln);
      const __bf16* gt = static_cast<const __bf16*>(a.gate) + static_cast<int64_t>(row0 + qo + c.tok) * a.gate_stride +
                         static_cast<int64_t>(g * rep + c.member) * DV + mp * (DV / 2) + 4 * (ln >> 5);
#pragma unroll
      for (int j = 0; j < 8; ++j) gates[j] = *reinterpret_cast<const bf16x4*>(gt + 8 * j);
    };
    // A piece of few blocks takes them one after the other, code in a row, the first two after one wait, the third's keys and
    // values on their way behind the second: the pipeline would be filled and emptied for them, its steps' parts lie on both
    // sides of the dealt-out ones, and each place that is come to for the first time costs a fetch of instructions.
    const bool brief = nb <= kBrief, v_first = turn == 0 || brief;
    if (v_first || was_brief) {
      if (MANY && NMAP == 1 && turn > 0) __syncthreads();   // (V's buffers were the results' way out)
      if (v_first) send_block_v(block_key(0), 0);
      if (__builtin_expect(brief && nb > 1, 0)) {
        send_block_k(bt, last_page, block_key(1), 1);
        send_block_v(block_key(1), 1);
      }
      if (MANY && brief && more) send_pages(nxt, 0, (turn & 1) ^ 1);
      wait_sent();
      hold_q();
      if (v_first) clear_block_v(block_key(0), vbuf(0));
      if (__builtin_expect(brief && nb > 1, 0)) clear_block_v(block_key(1), vbuf(1));
      __syncthreads();
    }
    was_brief = brief;
    if (__builtin_expect(brief, 0)) {
      load_gates();
      for (int i = 0; i < nb; ++i) {
        if (needed(i)) {
          scores(kbuf(i), S);
          weights(i, S, P);
          values(vbuf(i), P, i < kSplitBlocks);
        }
        if (__builtin_expect(nb > 2, 0)) {
          if (i == 1) {
            wait_sent();
            clear_block_v(block_key(2), vbuf(0));
          }
          __syncthreads();
          if (i == 0) {
            send_block_k(bt, last_page, block_key(2), 0);
            send_block_v(block_key(2), 0);
          }
        }
      }
      if (!MANY || more) __syncthreads();   // (the results' way out is K's buffers)
      if (MANY && more) {   // on their way behind the results
        send_block_k(lds_bt[(turn & 1) ^ 1], pages_of(nxt) - 1, first_key(nxt), 0);
        load_q(nxt, true);
      }
    }
    for (int i = 0; !brief && i < nb; ++i) {
      if (BORDERS && i >= quick0 && i + 1 < quick1) {
        Places at;
        places(at);
        if constexpr (MT > 1)
          for (; i + 1 < quick1 && i - 2 < kSplitBlocks; i += 2) quick_two(std::true_type(), at, i);
        for (; i + 1 < quick1; i += 2) quick_two(std::false_type(), at, i);
      }
      if (i == nb) break;
      if (i + 1 < nb) send_block_k(bt, last_page, block_key(i + 1), i + 1);
      const bool v_now = i > (v_first ? 1 : 0);
      if (v_now) send_block_v(block_key(i - 1), i + 1);
      if (MANY && i == 0 && more) send_pages(nxt, 0, (turn & 1) ^ 1);
      if (needed(i - 2)) values(vbuf(i), P, i - 2 < kSplitBlocks);
      if (needed(i - 1)) weights(i - 1, S, P);
      if (needed(i)) scores(kbuf(i), S);
      wait_sent();
      if (v_now) clear_block_v(block_key(i - 1), vbuf(i + 1));
      __syncthreads();
    }
    // steps nb and nb + 1 have no scores; the next piece's queries and first keys are on their way
    if (__builtin_expect(!brief, 1)) {
      const bool v_now = nb > (v_first ? 1 : 0);
      if (v_now) send_block_v(block_key(nb - 1), nb + 1);
      if (MANY && more) send_block_k(lds_bt[(turn & 1) ^ 1], pages_of(nxt) - 1, first_key(nxt), 0);
      if (needed(nb - 2)) values(vbuf(nb), P, nb - 2 < kSplitBlocks);
      if (needed(nb - 1)) weights(nb - 1, S, P);
      if (MANY) load_q(nxt, more);
      if (MANY) hold_q();
      wait_sent();
      if (v_now) clear_block_v(block_key(nb - 1), vbuf(nb + 1));
      __syncthreads();
      load_gates();
      if (needed(nb - 1)) values(vbuf(nb + 1), P, nb - 1 < kSplitBlocks);
    }

    l = both_sum(l);
    if constexpr (NMAP == 2) {
      // The two waves of a column set finish half of its channels each: they hand each other lam / l * O of the second
      // and O / l of the first map through LDS, add up their squares, and exchange the sums.
      constexpr int HV = NV / 2;
      static_assert(NMAP == 1 || sizeof(lds_x) >= NW * 64 * 16 * HV * sizeof(float), "room for both halves");
      const float il = l > 0.f ? (mp == 0 ? 1.0f : a.lam) / l : 0.f;
      f32x16 own[HV], theirs[HV];
#pragma unroll
      for (int hv = 0; hv < HV; ++hv)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          own[hv][i] = mp == 0 ? O[hv][i] : O[HV + hv][i];
          theirs[hv][i] = mp == 0 ? O[HV + hv][i] : O[hv][i];
        }
      f32x4* const give = reinterpret_cast<f32x4*>(lds_x) + w * HV * 4 * 64 + lane;
      const f32x4* const take = reinterpret_cast<const f32x4*>(lds_x) + (w ^ CW) * HV * 4 * 64 + lane;
#pragma unroll
      for (int hv = 0; hv < HV; ++hv)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          give[(hv * 4 + i4) * 64] = f32x4{theirs[hv][4 * i4] * il, theirs[hv][4 * i4 + 1] * il, theirs[hv][4 * i4 + 2] * il,
                                           theirs[hv][4 * i4 + 3] * il};
      __syncthreads();
      float ss = 0.f;
#pragma unroll
      for (int hv = 0; hv < HV; ++hv)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const f32x4 o2 = take[(hv * 4 + i4) * 64];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float mine = own[hv][4 * i4 + j] * il, o = mp == 0 ? mine - o2[j] : o2[j] - mine;
            own[hv][4 * i4 + j] = o;
            ss += o * o;
          }
        }
      ss = both_sum(ss);
      if (h == 0) lds_ss[w][r] = ss;
      __syncthreads();
      ss += lds_ss[w ^ CW][r];
      const float f = a.post / sqrtf(ss / static_cast<float>(DV) + a.eps);
      const int ln = fresh(lane), er = ln & 31, eh = ln >> 5, el = ln >> 3, ec = ln & 7;
      char* x = lds_x + w * 4096;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const f32x16& o = own[c / 4];
        const int i = c % 4 * 4;
        f32x4 e{o[i] * f, o[i + 1] * f, o[i + 2] * f, o[i + 3] * f};
        if (a.gate != nullptr) {
#pragma unroll
          for (int j = 0; j < 4; ++j) e[j] *= sigmoidf_(static_cast<float>(gates[c][j]));
        }
        const u32x2 b{__builtin_bit_cast(unsigned int, __builtin_convertvector((f32x2{e[0], e[1]}), bf16x2)),
                      __builtin_bit_cast(unsigned int, __builtin_convertvector((f32x2{e[2], e[3]}), bf16x2))};
        *reinterpret_cast<u32x2*>(x + er * 128 + ((c ^ ((er >> 1) & 7)) * 16) + 8 * eh) = b;
      }
      __builtin_amdgcn_wave_barrier();
      __bf16* ob = static_cast<__bf16*>(out) + (static_cast<int64_t>(row0 + qo) * (H / 2) + g * rep) * DV + 64 * mp + 8 * ec;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int rr = 8 * j + el, cc = wcol + rr;
        const u32x4 e = *reinterpret_cast<const u32x4*>(x + rr * 128 + ((ec ^ ((rr >> 1) & 7)) * 16));
        if (cc < cols_total)
          *reinterpret_cast<u32x4_any*>(ob + (static_cast<int64_t>(token_of(cc)) * (H / 2 - rep) + cc) * DV) = e;
      }
    } else {
      const int ln = fresh(lane), er = ln & 31, eh = ln >> 5, el = ln >> 3, ec = ln & 7;
      const Column c = column(ln);
      const int64_t row = row0 + qo + c.tok;
      const int head = g * rep + c.member;
      const float inv = c.valid && l > 0.f ? head_gate_of<__bf16>(a, row, head) / l : 0.f;
      if (MANY) __syncthreads();
      if (a.out_f32) {
        if (c.valid) {
          float* o = static_cast<float*>(out) + (row * H + head) * DV + 4 * eh;
#pragma unroll
          for (int vt = 0; vt < NV; ++vt)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4)
              *reinterpret_cast<f32x4_any*>(o + vt * 32 + 8 * i4) =
                  f32x4{O[vt][4 * i4] * inv, O[vt][4 * i4 + 1] * inv, O[vt][4 * i4 + 2] * inv, O[vt][4 * i4 + 3] * inv};
        }
      } else {
        // 64 channels at a time through LDS, the wave's own 4 KB (32 rows of 128 bytes, chunks changing places), so that
        // a store has whole rows: 8-byte pieces of 32 rows kept the memory pipe busy for 2 us per piece of work.  (What
        // depends on the lane is worked out here: kept over a piece it was spilled, and its reload waited for the stores.)
        static_assert(NMAP == 2 || 4 * (MANY ? VB : KB) >= 4096 * NW, "room for the rows");
        char* x = reinterpret_cast<char*>(MANY ? lds_v : lds_k) + w * 4096;
        __bf16* ob = static_cast<__bf16*>(out) + (static_cast<int64_t>(row0 + qo) * H + g * rep) * DV + 8 * ec;
#pragma unroll
        for (int v2 = 0; v2 < NV / 2; ++v2) {
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            const int vt = 2 * v2 + c / 4, i = c % 4 * 4;
            const u32x2 e{__builtin_bit_cast(unsigned int, __builtin_convertvector((f32x2{O[vt][i] * inv, O[vt][i + 1] * inv}), bf16x2)),
                          __builtin_bit_cast(unsigned int, __builtin_convertvector((f32x2{O[vt][i + 2] * inv, O[vt][i + 3] * inv}), bf16x2))};
            *reinterpret_cast<u32x2*>(x + er * 128 + ((c ^ ((er >> 1) & 7)) * 16) + 8 * eh) = e;
          }
          __builtin_amdgcn_wave_barrier();
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int rr = 8 * j + el, cc = wcol + rr;
            const u32x4 e = *reinterpret_cast<const u32x4*>(x + rr * 128 + ((ec ^ ((rr >> 1) & 7)) * 16));
            const int t = token_of(cc);
            if (cc < cols_total)
              *reinterpret_cast<u32x4_any*>(ob + (static_cast<int64_t>(t) * (H - rep) + cc) * DV + 64 * v2) = e;
          }
          __builtin_amdgcn_wave_barrier();
        }
      }
    }
    if (!MANY || !more) return;
    now = nxt;
  }
}

template <int ND, int NV, int NMAP, int NW>
bool launch(void* out, const void* q, const void* k_cache, const void* v_cache, const AttnArgs& a,
            int num_tiles, int cus, hipStream_t st) {
  constexpr int COLS = NW / NMAP * 32;
  const int chunks = (kTileTokens * (a.H / a.G) + COLS - 1) / COLS, heads = a.G / NMAP;
  const int pieces = num_tiles * chunks;
  const int workers = NW == 8 ? std::min(pieces, std::max({1, cus / heads, (pieces + kPieces - 1) / kPieces})) : pieces;
  const bool borders = (reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) % 16 == 0;
  auto* kernel = !borders       ? sink_flash_kernel<ND, NV, NMAP, NW, true, false>
                 : a.window > 0 ? sink_flash_kernel<ND, NV, NMAP, NW, true, true>
                                : sink_flash_kernel<ND, NV, NMAP, NW, false, true>;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(workers) * heads), dim3(NW * 64), 0, st, out,
                     static_cast<const __bf16*>(q), static_cast<const __bf16*>(k_cache),
                     static_cast<const __bf16*>(v_cache), a, num_tiles, chunks, workers);
  return true;
}

}  // namespace sf

// The shapes of the served families (head width 128, the latent cache of 192 + 64 channels, narrow heads,
// two maps of 64 over values of 128); other shapes, pages below 16 tokens (a 16-key group would span two) and contexts past the
// LDS page list run sink_attention.hip's kernel.
//
// One map of 64 or 128 goes by four waves, one piece each, two workgroups per CU.  Eight, with several pieces per workgroup in
// turn, were better by 2 % at best, and a NaN value of a later token (a weight of 0 times NaN) reached back twice as far once
// a batch was large.  us, four / eight waves: 32 + 8 heads, 4 x 2k 136 / 136, 3 x 2500 172 / 168, 2 x 4000 246 / 245, 8 x 1000 86 / 89,
// 16 x 500 56 / 61, 60 x 100 39 / 44; in a window of 1024 4 x 2k 115 / 122, 2 x 4000 132 / 145; 64 wide 4 x 2k 55.9 / 54.9.
// A value reaches back 128 columns, 32 tokens at four heads per group (latent: 8).
bool launch_sink_flash(void* out, const void* q, const void* k_cache, const void* v_cache,
                       const AttnArgs& a, int num_tiles, hipStream_t st) {
  if (a.block_size < 16 || a.bt_width > sf::kPages || !(a.scale > 0.f)) return false;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return false;
#define SF(D, V, MAPS, NW)                                   \
  if (a.dim == D && a.vdim == V && (a.pair ? 2 : 1) == MAPS) \
    return sf::launch<D / 16, V / 32, MAPS, NW>(out, q, k_cache, v_cache, a, num_tiles, cus, st);
  SF(64, 64, 1, 4)
  SF(128, 128, 1, 4)
  SF(256, 192, 1, 8)
  SF(64, 128, 2, 8)
#undef SF
  return false;
}

}  // namespace mixk
