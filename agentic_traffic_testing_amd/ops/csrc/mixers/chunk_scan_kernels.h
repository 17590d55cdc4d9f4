// Recurrences with a matrix state over ragged batches of portions, in chunks of 16 tokens on the matrix cores.  Per head, S [dk, dv] the state, per token
//     S = diag(a) S;   u = v   or, delta rule,   u = beta (v - S^T k);   S = S + k u^T;   o = S^T q
// with a one number per head (fixed: retention; from the data: state-space form, delta rule) or per head and
// key channel (forget-gate form, delta rule).  Inside a chunk, with P_i the product of a up to token i and
// D_ij the product over the tokens j + 1 ... i, the recurrence is
//     W = (P_i k_i) . S0;   U = T (V - W)  (delta; T = (I + L)^-1 diag(beta), L_ij = beta_i k_i . (D_ij k_j),
//     j < i)  or  U = V;    O = (P_i q_i) . S0 + A U,  A_ij = q_i . (D_ij k_j), j <= i;
//     S1 = P_end S0 + sum_j (D_end,j k_j) u_j^T.
//
// Every decay factor is a product of decays, never a quotient or a difference of summed logarithms: a
// factor is at most 1, underflows to 0 where the true one does, and is exact to a few roundings whatever the
// decays are (also 0).  For A and L with per-channel decays that takes levels of halving: in a block of
// 2 h tokens the pairs (later half, earlier half) factor as (product from the middle to i) x (product from j
// to the middle); h = 8, 4, 2, 1 covers all pairs j < i.  (16-bit inputs: h = 8 and 4, and the pairs inside four tokens as
// sums on the vector units.)
//
// * scores kernel: a wave or two (score_pairs) per (chunk, head) prepare what does not need the state - A, T and the
//   per-token scales - into a record in scratch.  All chunks at once, off the serial chain.
// * walk kernel: a workgroup walks the chunks of one (sequence, head), or of two heads with the same keys, for 64 or 128
//   value columns (walk_shape).  Four waves hold 16 or 32 columns of S each, in accumulators: the accumulator tiles of
//   16 x 16 are, split, at once the operands of the products with S, so S, W and U never leave registers, and a wave does
//   not wait for another one's products.  The others prepare the chunks' operands in LDS, one step ahead (one barrier per
//   chunk), with their loads one or two steps ahead of that.
//
// Bound of the walk: the chain of a chunk's products, parts and LDS reads in a wave that has a SIMD's matrix unit to itself,
// and the operands' vector work beside it (vector and matrix units busy, of the kernel's time: delta rule per channel 50 and
// 42 %, forget gate 55 and 33, second pass of state space in 32 bits 32 and 28, of retention 39 and 21; scores of the first
// two vector 79 and 67, matrix 14 and 8).  fp32 matrix products run on the vector units (the walk with 16x16x4 products:
// matrix busy 36 - 42 %, vector busy 50 %, and twelve waves per CU bring no more than eight), bf16 ones beside them.
// So the products with the state are made of bf16 parts: three parts hold the 24 bits of a number, six products of parts leave
// errors below fp32 products' (they add eight terms between roundings, those four), and a sum over 128 rows takes 24
// instructions of 16 cycles instead of 32 of 32 cycles.  What a part leaves of its number is a matrix product too (Identity):
// the parts of 128 rows take 48 vector instructions in place of 176.
// The products' waves go through chunks in an order of their own (`ours` below), 32 columns per wave where the operands
// serve 128, so that every operand read from LDS is used twice.  Walk, us, before / with parts by products / in order:
// delta rule per channel, 4 x 1.9k tokens 257 / 241 / 222, forget gate, 16 x 460 158 / 148 / 129; without the operands'
// waves' work 207 / 196 and 125 / 119, without the products' 165 / 135 and 114 / 104.
// Per-channel decays are worked out once, by the scores kernel, and kept in the records (8 KB per 16 tokens and head
// written and read twice, against 26 instructions per decay in two more places): forget gate 280 -> 262 us, delta rule
// 377 -> 373.
// Measured: the token-by-token kernels, fp32 products with 64 columns per workgroup, bf16 parts, and with the scores' halves of
// channels, pairs inside four tokens and values in one part where they are exact (us, scores + walk; 32 heads of 128, bf16
// unless noted):
//   delta rule, per-channel decay, 4 x ~1850 tokens: 1798, 130 + 343, 132 + 262, 99 + 256, today 84 + 232
//   forget gate, 16 x ~460 tokens:                    777, 111 + 308, 98 + 168, 83 + 158, today 70 + 136 + 5 (both passes)
//   state space, 96 heads of 128 x 64, 1023 tokens, fp32: 250, 21 + 94, 22 + 64, 18 + 64 in five segments of head pairs
//   retention, one portion of 1500 tokens (+ 11 rows): 260, 21 + 88, 22 + 69, 21 + 61 in eight segments, the rows inside the
//   scores launch
// What did not work: 16x16x4 products with a second wave per SIMD for the read-out (delta rule: no gain, see above);
// waves of a SIMD half a step apart without that; a higher priority for the operands' waves (delta rule + 15 %); four tiles
// of S at a time in the update (no change).
#pragma once

#include <algorithm>
#include <type_traits>

#include "step_scan.h"

namespace mixk {
namespace cs {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) double f64x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {   // bf16, 32 terms
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                 0, 0, 0);
}

// x0 and x1 as three bf16 numbers each, exact (8 + 8 + 8 bits and the signs; the parts of one number side by side with
// the other's): part 0 rounded to nearest, part 1 what that leaves, rounded, part 2 what is left.
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  return __builtin_bit_cast(unsigned, bf16x2{static_cast<__bf16>(a), static_cast<__bf16>(b)});
}
// the two numbers of a pair (of a shift in place of the permutation the compiler makes another conversion)
__device__ __forceinline__ float bf16_low(unsigned p) {
  return __builtin_bit_cast(float, __builtin_amdgcn_perm(0u, p, 0x01000c0cu));
}
__device__ __forceinline__ float bf16_high(unsigned p) { return __builtin_bit_cast(float, p & 0xffff0000u); }
__device__ __forceinline__ void split(float x0, float x1, unsigned& p0, unsigned& p1, unsigned& p2) {
  p0 = pack_bf16(x0, x1);
  const float r0 = x0 - bf16_low(p0), r1 = x1 - bf16_high(p0);
  p1 = pack_bf16(r0, r1);
  p2 = pack_bf16(r0 - bf16_low(p1), r1 - bf16_high(p1));
}
// Infinities, and finite numbers above all of bf16's (kSplitMax), have no parts: part 2 is NaN.  What products with them, or
// with rows whose scales come later, leave not finite is taken again in fp32 (join): an infinity of the inputs or the state
// is one of the results, as in the token-by-token form, and no other entry changes a bit.  The walk checks a chunk with sums
// of absolute values and one branch, the steps behind it twice in the code: 1 - 4 % (us without / with checks, 32 heads: one
// prompt of 2048 delta rule 228 / 233, per channel 275 / 285, state space 80 / 82, forget gate 16 x 512 284 / 288).
constexpr float kSplitMax = 0x1.fep127f;
__device__ __forceinline__ float join(unsigned p0, unsigned p1, unsigned p2, bool high) {
  const float a = high ? bf16_high(p0) : bf16_low(p0), b = high ? bf16_high(p1) : bf16_low(p1);
  const float c = high ? bf16_high(p2) : bf16_low(p2);
  if (fabsf(a) <= kSplitMax || a != a) return a + (b + c);
  return b != b ? a : copysignf(__FLT_MAX__, a);   // (a finite number that part 0 rounds to infinity: the largest)
}
__device__ __forceinline__ float abs_sum(const f32x4 x) { return (fabsf(x[0]) + fabsf(x[1])) + (fabsf(x[2]) + fabsf(x[3])); }
// The same for four numbers per lane, what a part leaves by the matrix cores: minus the identity times the part, added to
// the numbers.  Their layout as 16 x 16 numbers is that of the part as an operand of 16 rows, and one product (16 cycles
// beside the vector units) takes the place of four instructions that unpack the part and four that subtract it; the
// difference has at most 24 bits, and it is exact.  Between a product of 16 terms, as this one is, and one of 32 that adds to
// its result a vector instruction has to use that result (the compiler leaves too few cycles: first_parts()); what is left of
// a number is packed into the next part, so it always does.  A number without parts leaves NaN in the lane's and the column's
// other three lanes' parts 1 and 2, so it is for numbers whose products are looked at by column, or that have parts.
struct Identity {
  u32x2 minus;   // row m, columns 4 gr ... + 3
  __device__ __forceinline__ explicit Identity(int lane) {
    const int i = (lane & 15) - 4 * (lane >> 4);
    minus = u32x2{i == 0 ? 0xbf80u : i == 1 ? 0xbf800000u : 0u, i == 2 ? 0xbf80u : i == 3 ? 0xbf800000u : 0u};
  }
  __device__ __forceinline__ f32x4 rest(const f32x4 x, unsigned p0, unsigned p1) const {
    typedef __attribute__((ext_vector_type(4))) short s16x4;
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, minus), __builtin_bit_cast(s16x4, u32x2{p0, p1}),
                                                     x, 0, 0, 0);
  }
  template <int FIRST = 0>
  __device__ __forceinline__ void split(f32x4 x, unsigned (&p)[3][2]) const {
#pragma unroll
    for (int i = FIRST; i < 3; ++i) {
      p[i][0] = pack_bf16(x[0], x[1]);
      p[i][1] = pack_bf16(x[2], x[3]);
      if (i < 2) x = rest(x, p[i][0], p[i][1]);
    }
  }
};
// Part 0 of products a b, and what it leaves of them unrounded, which the other parts then hold (as a product rounded first,
// per-channel delta rule in 32 bits, results 8 % further from 64 bits).
__device__ __forceinline__ f32x4 split_product(const f32x4 a, const f32x4 b, unsigned (&p0)[2]) {
  p0[0] = pack_bf16(a[0] * b[0], a[1] * b[1]);
  p0[1] = pack_bf16(a[2] * b[2], a[3] * b[3]);
  return f32x4{__builtin_fmaf(a[0], b[0], -bf16_low(p0[0])), __builtin_fmaf(a[1], b[1], -bf16_high(p0[0])),
               __builtin_fmaf(a[2], b[2], -bf16_low(p0[1])), __builtin_fmaf(a[3], b[3], -bf16_high(p0[1]))};
}
// ... of eight numbers, in eleven steps to go between matrix products
struct SplitSteps {
  f32x4 r[2];
  __device__ __forceinline__ void step(int i, u32x4 (&p)[3], const Identity& id) {   // (i known when compiled)
    const int part = i / 5, j = i % 5;
    if (j == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) p[part][e] = pack_bf16(r[e >> 1][2 * (e & 1)], r[e >> 1][2 * (e & 1) + 1]);
    } else if (j < 3) {
      r[j - 1] = id.rest(r[j - 1], p[part][2 * (j - 1)], p[part][2 * (j - 1) + 1]);
    }
  }
};

// value of the lane 8 away in the row of 16
__device__ __forceinline__ float row_other_half(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xF, 0xF,
                                                               true));   // row_ror:8
}

// The values of a lane and of the one 16 (32) lanes away: that of the lower of the two, and the other's.
struct Pair {
  float lower, upper;
};
template <int N>
__device__ __forceinline__ Pair swap_rows(float v) {
  float u = v;   // (the compiler takes the builtin's two results for one; the instruction wants two idle cycles before it)
  if (N == 16) asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(v), "+v"(u));
  else asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(v), "+v"(u));
  return {v, u};
}

template <int MODE>
constexpr bool per_channel() { return MODE == kModeForget || MODE == kModeDeltaChannel; }

// ---- a chunk as a wave holds it -----------------------------------------------------------------------
// Lane (tg, c) = (lane / 16, lane % 16) holds CPL = DK / 16 adjacent channels CPL c ... of the tokens 4 tg ... + 3:
// a row is one 16-byte load per lane and 4 rows are one instruction.
template <typename T, int MODE, int CPL>
struct Raw {
  T q[4][CPL], k[4][CPL];
  T d[per_channel<MODE>() ? 4 : 1][CPL];
  // the channels that the rotation pairs with these (few channels per lane: no exchange between lanes)
  T pq[MODE == kModeRetention && CPL <= 2 ? 4 : 1][CPL], pk[MODE == kModeRetention && CPL <= 2 ? 4 : 1][CPL];
  float cs[MODE == kModeRetention ? 4 : 1][CPL], sn[MODE == kModeRetention ? 4 : 1][CPL];
};

// (1 + e^x)^-b with the error of expf(-b * log1pf(expf(x))), which takes four times the instructions (scores and walk of
// the per-channel delta rule, 4 x 1.9k tokens: twice the time).  In powers of two:
// log2(1 + e^x) = max(x, 0) log2 e + log2(1 + t) with t = e^-|x|, the hardware exponential of a reduced argument, and
// log2(1 + t) = t (log2 e + t p(t)), p of degree 8 with a relative error of 2^-27.5 on [0, 1] (least squares at
// Chebyshev nodes, weighted towards the largest error).
// Measured, rms in 2^-24 for rates 1 / 16: x in -10 ... -4 0.305 / 0.317 (library 0.305 / 0.319), -4 ... -1 0.34 / 1.36
// (0.35 / 1.37), -1 ... 5 1.18 / 17.6 (1.34 / 20.2).  (The hardware logarithm of 1 + e^x: 0.64 / 9.2 in the first range,
// no decay at all below x = -17, and 5 % less time.)
__device__ __forceinline__ float softplus_decay(float x, float b) {
  constexpr float kHi = 1.44269502162933350f, kLo = 1.92596299e-8f;   // log2 e in two parts
  constexpr float kInt = 12582912.f;   // 1.5 x 2^23: a sum with it is rounded to an integer, which its low bits hold
  const float z = __builtin_elementwise_maximum(-fabsf(x), -80.f);
  const float k = __builtin_fmaf(z, kHi, kInt), n = k - kInt;
  const float f = __builtin_amdgcn_exp2f(__builtin_fmaf(z, kLo, __builtin_fmaf(z, kHi, -n)));
  const float t = __builtin_bit_cast(float, (__builtin_bit_cast(unsigned, k) << 23) + __builtin_bit_cast(unsigned, f));
  float p = -0.00479013659f;
  p = __builtin_fmaf(p, t, 0.0291612372f);
  p = __builtin_fmaf(p, t, -0.0832162574f);
  p = __builtin_fmaf(p, t, 0.154113725f);
  p = __builtin_fmaf(p, t, -0.221548006f);
  p = __builtin_fmaf(p, t, 0.284150839f);
  p = __builtin_fmaf(p, t, -0.360077679f);
  p = __builtin_fmaf(p, t, 0.48085779f);
  p = __builtin_fmaf(p, t, -0.721346557f);
  const float m = __builtin_elementwise_maximum(x, 0.f);   // (lets NaN through)
  const float l = __builtin_fmaf(m, kHi, __builtin_fmaf(m, kLo, __builtin_fmaf(t, kHi, t * __builtin_fmaf(t, p, kLo))));
  return __builtin_amdgcn_exp2f(-b * l);
}

// A uniform base and a lane's offset of 32 bits in bytes, an addressing mode of its own (16 rows stay below 2^32 bytes,
// launch_scan_batch checks): of indices the compiler makes 64-bit sums.
template <typename P>
__device__ __forceinline__ P& at_bytes(void* base, unsigned bytes) {
  return *reinterpret_cast<P*>(static_cast<char*>(base) + bytes);
}
template <typename P>
__device__ __forceinline__ const P& at_bytes(const void* base, unsigned bytes) {
  return *reinterpret_cast<const P*>(static_cast<const char*>(base) + bytes);
}

// VEC: aligned rows, dk a multiple of CPL.  (A template argument: behind a branch the number of loads in flight
// is unknown, and every wait for one of them becomes a wait for all.)
template <bool VEC, typename T, int CPL>
__device__ __forceinline__ void load_cpl(T (&o)[CPL], const T* row, int c0, int dk) {
  if constexpr (VEC && CPL > 1) {
    const T* p = row + min(c0, dk - CPL);
    constexpr int B = CPL * sizeof(T) < 16 ? CPL * sizeof(T) : 16, N = CPL * sizeof(T) / B;
    typedef __attribute__((ext_vector_type(B / 4))) unsigned int word;
#pragma unroll
    for (int i = 0; i < N; ++i)
      reinterpret_cast<word*>(o)[i] = reinterpret_cast<const word*>(p)[i];
  } else {
#pragma unroll
    for (int j = 0; j < CPL; ++j) o[j] = row[min(c0 + j, dk - 1)];
  }
}

// addresses are clamped, and what is not there is dropped where the values are used: a branch or a select
// per load would wait for it
// (uniform 64-bit bases and 32-bit lane offsets: 16 rows stay below 2^31 elements, launch_scan_batch checks)
template <bool VEC, typename T, int MODE, int CPL>
__device__ __forceinline__ void load_raw(Raw<T, MODE, CPL>& r, const ChunkArgs& a, int h, int g, int64_t row0,
                                         int nt, int lane, int c0) {
  const int t0 = (lane >> 4) * 4;
  const T* qb = static_cast<const T*>(a.q) + row0 * a.q_stride + static_cast<int64_t>(g) * a.dk;
  const T* kb = static_cast<const T*>(a.k) + row0 * a.k_stride + static_cast<int64_t>(g) * a.dk;
  const T* db = MODE == kModeDeltaChannel ? static_cast<const T*>(a.dec) + row0 * a.dec_stride +
                                                static_cast<int64_t>(h) * a.dk : nullptr;
  const int qs = static_cast<int>(a.q_stride), ks = static_cast<int>(a.k_stride), ds = static_cast<int>(a.dec_stride);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = min(t0 + i, nt - 1);
    load_cpl<VEC, T, CPL>(r.q[i], qb + t * qs, c0, a.dk);
    if (MODE == kModeForget)
      load_cpl<VEC, T, CPL>(r.d[per_channel<MODE>() ? i : 0], kb + t * ks, c0, a.dk);
    else
      load_cpl<VEC, T, CPL>(r.k[i], kb + t * ks, c0, a.dk);
    if (MODE == kModeDeltaChannel)
      load_cpl<VEC, T, CPL>(r.d[per_channel<MODE>() ? i : 0], db + t * ds, c0, a.dk);
    if (MODE == kModeRetention && a.n_freq > 0) {   // uniform
      const int n = a.n_freq;
      const float* tab = a.cos_sin + row0 * 2 * n + t * 2 * n;
      float (&cs)[CPL] = r.cs[MODE == kModeRetention ? i : 0], (&sn)[CPL] = r.sn[MODE == kModeRetention ? i : 0];
      if constexpr (VEC && CPL <= 2) {
        const int f = c0 < n ? c0 : c0 < 2 * n ? c0 - n : 0, pc = c0 < n ? c0 + n : f;
        load_cpl<VEC, float, CPL>(cs, tab, f, n);
        load_cpl<VEC, float, CPL>(sn, tab + n, f, n);
        load_cpl<VEC, T, CPL>(r.pq[MODE == kModeRetention && CPL <= 2 ? i : 0], qb + t * qs, pc, a.dk);
        load_cpl<VEC, T, CPL>(r.pk[MODE == kModeRetention && CPL <= 2 ? i : 0], kb + t * ks, pc, a.dk);
      } else if constexpr (VEC) {
        const int f = c0 < n ? c0 : c0 < 2 * n ? c0 - n : 0;
#pragma unroll
        for (int j = 0; j < CPL; j += 4) {
          *reinterpret_cast<f32x4*>(cs + j) = *reinterpret_cast<const f32x4*>(tab + f + j);
          *reinterpret_cast<f32x4*>(sn + j) = *reinterpret_cast<const f32x4*>(tab + n + f + j);
        }
      } else {
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
          const int c = c0 + j, f = c < n ? c : c < 2 * n ? c - n : 0;
          cs[j] = tab[f];
          sn[j] = tab[n + f];
          if constexpr (CPL <= 2) {
            const int pc = min(c < n ? c + n : f, a.dk - 1);
            r.pq[MODE == kModeRetention && CPL <= 2 ? i : 0][j] = qb[t * qs + pc];
            r.pk[MODE == kModeRetention && CPL <= 2 ? i : 0][j] = kb[t * ks + pc];
          }
        }
      }
    }
  }
}

// Per-channel decays, 1 for a token or channel that is not there (FULL: all are).  Parameters per channel: (f_bias, lower
// bound) or (dt_bias, exp(A_log)).
template <int MODE, int CPL>
__device__ __forceinline__ void decay_params(const ChunkArgs& a, int h, int c0, float (&b0)[CPL], float (&b1)[CPL]) {
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    const int c = min(c0 + j, a.dk - 1);
    b0[j] = a.p0[h * a.dk + c];
    b1[j] = MODE == kModeForget ? a.p1[h * a.dk + c] : expf(a.p1[h]);
  }
}
template <bool FULL, typename T, int MODE, int CPL>
__device__ __forceinline__ void decays(const Raw<T, MODE, CPL>& r, const ChunkArgs& a, int nt, int lane, int c0,
                                       const float (&b0)[CPL], const float (&b1)[CPL], float (&d)[4][CPL]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const float raw = static_cast<float>(r.d[per_channel<MODE>() ? i : 0][j]);
      float x;
      if (MODE == kModeForget) {
        x = b1[j] + (1.0f - b1[j]) * gate_sigmoid<T>(raw + b0[j]);
      } else if (sizeof(T) == 4) {
        x = expf(-b1[j] * softplusf_(raw + b0[j]));
      } else {
        x = softplus_decay(raw + b0[j], b1[j]);
      }
      d[i][j] = FULL || ((lane >> 4) * 4 + i < nt && c0 + j < a.dk) ? x : 1.f;
    }
}

// q and k in fp32, 0 for a token or channel that is not there.  Forget-gate form: k = 1 - decay.  Retention
// rotates channel c with c +- n_freq, which another lane of the row holds (all lanes take part).
template <bool FULL, bool VEC, typename T, int MODE, int CPL>
__device__ __forceinline__ void queries_keys(const Raw<T, MODE, CPL>& r, const ChunkArgs& a, int g, int64_t row0,
                                             int nt, int lane, int c0, const float (&d)[4][CPL], float (&q)[4][CPL],
                                             float (&k)[4][CPL]) {
  const int t0 = (lane >> 4) * 4;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      q[i][j] = static_cast<float>(r.q[i][j]);
      if (MODE == kModeForget) q[i][j] = gate_silu<T>(q[i][j]);
      k[i][j] = MODE == kModeForget ? 1.0f - d[i][j] : static_cast<float>(r.k[i][j]);
    }
  if (MODE == kModeRetention) {
    const int n = a.n_freq;
    if (n > 0) {   // uniform
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float (&cs)[CPL] = r.cs[MODE == kModeRetention ? i : 0];
        const float (&sn)[CPL] = r.sn[MODE == kModeRetention ? i : 0];
        float pq[CPL], pk[CPL];
        if constexpr (CPL <= 2) {
#pragma unroll
          for (int j = 0; j < CPL; ++j) {
            pq[j] = static_cast<float>(r.pq[MODE == kModeRetention && CPL <= 2 ? i : 0][j]);
            pk[j] = static_cast<float>(r.pk[MODE == kModeRetention && CPL <= 2 ? i : 0][j]);
          }
        } else if (n == 8 * CPL) {   // the whole row turns: the partner is channel j of the lane 8 further
#pragma unroll
          for (int j = 0; j < CPL; ++j) {
            pq[j] = row_other_half(q[i][j]);
            pk[j] = row_other_half(k[i][j]);
          }
        } else if (VEC || n % CPL == 0) {   // ... of another lane
          const int src = (lane & 48) + ((c0 < n ? c0 + n : c0 - n) / CPL & 15);
#pragma unroll
          for (int j = 0; j < CPL; ++j) {
            pq[j] = __shfl(q[i][j], src, kWave);
            pk[j] = __shfl(k[i][j], src, kWave);
          }
        } else {
          const int64_t row = row0 + min(t0 + i, nt - 1);
          const T* qr = static_cast<const T*>(a.q) + row * a.q_stride + static_cast<int64_t>(g) * a.dk;
          const T* kr = static_cast<const T*>(a.k) + row * a.k_stride + static_cast<int64_t>(g) * a.dk;
#pragma unroll
          for (int j = 0; j < CPL; ++j) {
            const int c = c0 + j, pc = c < n ? c + n : c < 2 * n ? c - n : 0;
            pq[j] = static_cast<float>(qr[pc]);
            pk[j] = static_cast<float>(kr[pc]);
          }
        }
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
          const int c = c0 + j;
          const float s = c < n ? -sn[j] : sn[j];
          q[i][j] = c < 2 * n ? q[i][j] * cs[j] + pq[j] * s : q[i][j];
          k[i][j] = c < 2 * n ? k[i][j] * cs[j] + pk[j] * s : k[i][j];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < CPL; ++j) k[i][j] *= a.kscale;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const bool in = FULL || (t0 + i < nt && c0 + j < a.dk);
      q[i][j] = in ? q[i][j] : 0.f;
      k[i][j] = in ? k[i][j] : 0.f;
    }
}

// y += a[j] of lane LANE of each 16, times x[j], for N of them.  (The broadcast operand wants two idle cycles behind its last
// write, which the compiler does not see here; from the builtin it makes a move and a multiply-add.)
#define MIXK_TERM(A, X) "v_fmac_f32_dpp %0, " A ", " X " row_newbcast:%1 row_mask:0xf bank_mask:0xf\n\t"
template <int LANE, int N>
__device__ __forceinline__ void add_broadcast(float& y, const float* a, const float* x) {
  if constexpr (N == 1)
    asm("s_nop 1\n\t" MIXK_TERM("%2", "%3") : "+&v"(y) : "n"(LANE), "v"(a[0]), "v"(x[0]));
  if constexpr (N == 2)
    asm("s_nop 1\n\t" MIXK_TERM("%2", "%3") MIXK_TERM("%4", "%5")
        : "+&v"(y) : "n"(LANE), "v"(a[0]), "v"(x[0]), "v"(a[1]), "v"(x[1]));
  if constexpr (N == 3)
    asm("s_nop 1\n\t" MIXK_TERM("%2", "%3") MIXK_TERM("%4", "%5") MIXK_TERM("%6", "%7")
        : "+&v"(y) : "n"(LANE), "v"(a[0]), "v"(x[0]), "v"(a[1]), "v"(x[1]), "v"(a[2]), "v"(x[2]));
  if constexpr (N == 4)
    asm("s_nop 1\n\t" MIXK_TERM("%2", "%3") MIXK_TERM("%4", "%5") MIXK_TERM("%6", "%7") MIXK_TERM("%8", "%9")
        : "+&v"(y) : "n"(LANE), "v"(a[0]), "v"(x[0]), "v"(a[1]), "v"(x[1]), "v"(a[2]), "v"(x[2]), "v"(a[3]), "v"(x[3]));
}
#undef MIXK_TERM

// ---- scores -------------------------------------------------------------------------------------------
constexpr int kScoreWaves = 4;
// Per-channel decays of 16-bit inputs: two waves per chunk, half of its channels each; the sums come together at the end.  (A
// lane with eight channels of q, k and the decays takes 195 - 209 registers, two waves per SIMD; with four, three and four.
// Scores, us, one wave / two / two and T from broadcast operands: delta rule, 4 x 1.9k tokens 99 / 97 / 83 - vector units
// busy 54 / - / 80 % -, forget gate, 16 x 460 84 / 71; with no more than 128 registers for the delta rule 111, spilled.)
template <typename T, int MODE, int DK>
constexpr bool score_pairs() { return per_channel<MODE>() && sizeof(T) == 2 && DK == 128; }

template <typename T, int MODE, int DK, bool VEC>
__global__ void __launch_bounds__(64 * kScoreWaves, (score_pairs<T, MODE, DK>() ? (MODE == kModeForget ? 4 : 3) : 2))
scan_scores_kernel(ChunkArgs a, int step_blocks, int step_cols, int v4) {
  constexpr bool PAIRS = score_pairs<T, MODE, DK>();
  constexpr int CPL = DK / 16 / (PAIRS ? 2 : 1), kDecay = scan_rec_decay(MODE);
  // (the kernels for any alignment take keys of all widths)
  const int REC = scan_record_floats(MODE, VEC ? DK : a.dk), DS = scan_decay_width(VEC ? DK : a.dk);
  constexpr bool DELTA = MODE >= kModeDelta, CH = per_channel<MODE>();
  // bf16 q and k as they are (one number as the decay): their products are those of the matrix cores, and the operands
  // plain loads.  Layers, us, through fp32 rows in LDS / here: state space 4 x 1000, 128 heads 292 / 265, 1000, 96 heads
  // 98 / 93, delta rule 4 x 2048, 32 heads 358 / 349.
  constexpr bool EXACT = VEC && DK == 128 && sizeof(T) == 2 && (MODE == kModeStateSpace || MODE == kModeDelta);
  constexpr int ROWS = EXACT ? 1 : MODE == kModeDeltaChannel ? 24 : 32;
  // Operand rows hold half of the channels at a time, in half the LDS, and what is worked out for them is not kept: more waves
  // per CU (rows of 128 channels, 62 and 79 KB per workgroup, let eight onto it).  us: delta rule per channel, 4 x 1.9k
  // tokens, 111 -> 101; forget gate, 16 x 460, 94 -> 85; state space in 32 bits, 1023, 21.1 -> 18.7; retention 21.1 -> 20.9.
  constexpr int HALVES = DK == 128 && !EXACT && !PAIRS ? 2 : 1, WIDE = DK / HALVES / (PAIRS ? 2 : 1), CH_HALF = CPL / HALVES;
  struct Lds {
    float row[ROWS][WIDE + 4];      // operand rows of the products
    float sq[16][20], sk[DELTA ? 16 : 1][20];   // A; L
    float sc[4][16];                // scale of q, of k, beta, scalar decay
    float sum[PAIRS ? 3 : 1][16];   // of half of the channels: q . q, k . k, q . k
  };
  constexpr size_t LDS_BYTES = sizeof(Lds) * kScoreWaves > sizeof(ss::StepLds<MODE, DK / 16>)
                                   ? sizeof(Lds) * kScoreWaves : sizeof(ss::StepLds<MODE, DK / 16>);
  __shared__ __attribute__((aligned(16))) char lds_raw[LDS_BYTES];
  if (static_cast<int>(blockIdx.x) < step_blocks) {   // short portions, token by token
    auto& l = *reinterpret_cast<ss::StepLds<MODE, DK / 16>*>(lds_raw);
    const int s = blockIdx.x / step_cols, bx = blockIdx.x - s * step_cols;
    if (v4)
      ss::scan_step<T, MODE, DK / 16, true>(a, a.min_rows - 1, bx, s, l);
    else
      ss::scan_step<T, MODE, DK / 16, false>(a, a.min_rows - 1, bx, s, l);
    return;
  }
  Lds* lds_all = reinterpret_cast<Lds*>(lds_raw);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  Lds& s = lds_all[w];
  // the wave's chunk and head, and with two waves its first channel; waves without a chunk stay for nothing but the pairs'
  // barrier
  const int64_t item = (static_cast<int64_t>(blockIdx.x - step_blocks) * kScoreWaves + w) / (PAIRS ? 2 : 1);
  const int ch0 = PAIRS ? DK / 2 * (w & 1) : 0;
  const int slot = static_cast<int>(item / a.H), h = static_cast<int>(item % a.H);
  int lo = 0, hi = a.S - 1;   // last sequence whose first slot is at or below `slot`
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.seq_qstart[mid] / kScanChunk + mid <= slot) lo = mid; else hi = mid - 1;
  }
  const int first = a.seq_qstart[lo], n = a.seq_qstart[lo + 1] - first;
  const int t0 = (slot - first / kScanChunk - lo) * kScanChunk;
  const bool none = slot >= a.n_slots || n < a.min_rows || t0 >= n || a.seq_slot[lo] < 0;
  if (none) {
    if (PAIRS) lds_barrier();
    return;
  }
  const int nt = min(kScanChunk, n - t0);
  const int g = MODE == kModeForget ? h : h / (a.H / a.G);
  const int64_t row0 = first + t0;
  float* rec = a.rec + (static_cast<int64_t>(slot) * a.H + h) * REC;
  const int m = lane & 15, gr = lane >> 4;   // as (c, tg) of the layout above, and as MFMA (column, group)

  float q[4][CPL], k[4][CPL], d[4][CPL];
  float no_parts = 0.f;   // keys that split() cannot take (not where the walk's are scaled to at most 1)
  f32x4 xq = {0.f, 0.f, 0.f, 0.f}, xk = xq, xqq = xq;   // EXACT: q . k, k . k, q . q; row 4 gr + i, column m
  if constexpr (EXACT) {
    // rows of tokens that are not there repeat the last one: what comes of them is multiplied by 0 or not used
    const int64_t row = row0 + min(m, nt - 1);
    const T* qr = static_cast<const T*>(a.q) + row * a.q_stride + static_cast<int64_t>(g) * a.dk;
    const T* kr = static_cast<const T*>(a.k) + row * a.k_stride + static_cast<int64_t>(g) * a.dk;
    u32x4 qf[DK / 32], kf[DK / 32];
#pragma unroll
    for (int t = 0; t < DK / 32; ++t) {
      const int c = 32 * t + 8 * gr, at = min(c, a.dk - 8);
      qf[t] = *reinterpret_cast<const u32x4*>(qr + at);
      kf[t] = *reinterpret_cast<const u32x4*>(kr + at);
      if (c >= a.dk) qf[t] = kf[t] = u32x4{0, 0, 0, 0};
    }
    f32x4 yq = xq, yk = xq, yqq = xq;   // (two sums of half the length each)
#pragma unroll
    for (int t = 0; t < DK / 32; t += 2) {
      xq = mma(qf[t], kf[t], xq);
      yq = mma(qf[t + 1], kf[t + 1], yq);
      if (DELTA) {
        xk = mma(kf[t], kf[t], xk);
        yk = mma(kf[t + 1], kf[t + 1], yk);
        xqq = mma(qf[t], qf[t], xqq);
        yqq = mma(qf[t + 1], qf[t + 1], yqq);
      }
    }
    xq += yq;
    xk += yk;
    xqq += yqq;
    if constexpr (!DELTA) {   // (a product with zeros: 0 but for keys that are not finite)
      f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < DK / 32; ++t) z = mma(kf[t], u32x4{0, 0, 0, 0}, z);
      no_parts = __any(abs_sum(z) != 0.f) ? kSplitMax : 0.f;
    }
  } else {
    Raw<T, MODE, CPL> r;
    load_raw<VEC, T, MODE, CPL>(r, a, h, g, row0, nt, lane, ch0 + m * CPL);
    float b0[CPL], b1[CPL];
    if constexpr (CH) decay_params<MODE, CPL>(a, h, ch0 + m * CPL, b0, b1);
    if (VEC && CH && nt == kScanChunk && a.dk == DK) {   // (uniform)
      if constexpr (CH) decays<true, T, MODE, CPL>(r, a, nt, lane, ch0 + m * CPL, b0, b1, d);
      queries_keys<true, VEC, T, MODE, CPL>(r, a, g, row0, nt, lane, ch0 + m * CPL, d, q, k);
    } else {
      if constexpr (CH) decays<false, T, MODE, CPL>(r, a, nt, lane, ch0 + m * CPL, b0, b1, d);
      queries_keys<false, VEC, T, MODE, CPL>(r, a, g, row0, nt, lane, ch0 + m * CPL, d, q, k);
    }
    if constexpr (!CH) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < CPL; j += 4) sum += abs_sum(f32x4{k[i][j], k[i][j + 1], k[i][j + 2], k[i][j + 3]});
      no_parts = __any(!(sum <= kSplitMax)) ? kSplitMax : 0.f;
    }
    if constexpr (scan_keeps_decays(MODE))
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < CPL; j += 4)
          if (VEC || ch0 + m * CPL < DS)
            *reinterpret_cast<f32x4*>(rec + kDecay + (4 * gr + i) * DS + ch0 + m * CPL + j) =
                f32x4{d[i][j], d[i][j + 1], d[i][j + 2], d[i][j + 3]};
  }
  // per-token numbers of token m: beta, scalar decay and its products, dt, inverse norms
  float beta = 0.f, dec = 1.f, dt = 1.f, qi = 1.f, ki = 1.f;
  const bool live = m < nt;
  const int64_t rl = row0 + (live ? m : 0);
  if (DELTA)
    beta = live ? sigmoidf_(ldf(static_cast<const T*>(a.beta) + rl * a.beta_stride + h)) : 0.f;
  if (MODE == kModeStateSpace || MODE == kModeDelta) {
    const float sp = softplusf_(ldf(static_cast<const T*>(a.dec) + rl * a.dec_stride + h) + a.p0[h]);
    dec = live ? expf(-expf(a.p1[h]) * sp) : 1.f;
    if (MODE == kModeStateSpace) dt = live ? sp : 0.f;
  }
  auto wave_sync = [] {   // LDS hand-over inside the wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  if constexpr (EXACT && DELTA) {   // the squares are on the diagonals
    if (m >> 2 == gr) {
      auto at = [&](const f32x4 x) { return m & 2 ? (m & 1 ? x[3] : x[2]) : m & 1 ? x[1] : x[0]; };
      s.sc[0][m] = at(xqq);
      s.sc[1][m] = at(xk);
    }
    wave_sync();
    qi = 1.0f / (sqrtf(static_cast<float>(a.dk)) * sqrtf(s.sc[0][m] + 1e-6f));
    ki = 1.0f / sqrtf(s.sc[1][m] + 1e-6f);
  } else if constexpr (DELTA || CH) {
    // row sums |q|^2, |k|^2 and q . k of the lane's four tokens over the 16 lanes that share them
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float qq = 0.f, kk = 0.f, qk = 0.f;
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        qq += q[i][j] * q[i][j];
        kk += k[i][j] * k[i][j];
        qk += q[i][j] * k[i][j];
      }
      if (DELTA) {
        qq = group_sum<16>(qq);
        kk = group_sum<16>(kk);
      }
      if (CH) qk = group_sum<16>(qk);
      if (PAIRS && m == 0) {
        s.sum[0][4 * gr + i] = qq;
        s.sum[PAIRS ? 1 : 0][4 * gr + i] = kk;
        s.sum[PAIRS ? 2 : 0][4 * gr + i] = qk;
      } else if (m == 0) {
        s.sc[0][4 * gr + i] = qq;
        s.sc[1][4 * gr + i] = kk;
        s.sc[3][4 * gr + i] = qk;
      }
    }
    wave_sync();
    if (DELTA && !PAIRS) {
      qi = 1.0f / (sqrtf(static_cast<float>(a.dk)) * sqrtf(s.sc[0][m] + 1e-6f));
      ki = 1.0f / sqrtf(s.sc[1][m] + 1e-6f);
    }
  }
  const float diag = CH && !PAIRS ? s.sc[3][m] : 0.f;
  // prefix and suffix products of the scalar decay, by every lane of the token (a fixed decay's powers come
  // from the table, rounded once: a slow head remembers thousands of tokens)
  const float* pw = MODE == kModeRetention ? a.p0 + h * kPowers : nullptr;
  float pre = 1.f, suf = 1.f, end = 1.f;
  if (MODE == kModeRetention) {
    pre = pw[m + 1];
    suf = pw[max(nt - 1 - m, 0)];
    end = pw[nt];
  } else if (!CH) {
    // scans over the 16 lanes of a group, rounded once at the end
    double up = dec, down = dec;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const double u = __shfl(up, lane - o, kWave), d = __shfl(down, lane + o, kWave);
      up *= m >= o ? u : 1.0;
      down *= m + o < 16 ? d : 1.0;
    }
    const double behind = __shfl(down, lane + 1, kWave);
    pre = static_cast<float>(up);
    suf = m < 15 ? static_cast<float>(behind) : 1.f;
    end = __shfl(pre, lane | 15, kWave);
  }
  wave_sync();
  if (!PAIRS && lane < 16) {
    rec[kRecQ + lane] = qi * pre;
    rec[kRecK + lane] = ki * pre;
    rec[kRecKt + lane] = ki * dt * suf;
    rec[kRecEnd + lane] = lane == kRecNoParts - kRecEnd ? no_parts : end;
    s.sc[0][lane] = qi;
    s.sc[1][lane] = ki * dt;
    s.sc[2][lane] = beta;
    s.sc[3][lane] = dec;
  }

  // channels of half `hf` of a row: x(j) of the lane's
  auto put = [&](int row, auto hf, auto x) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < CH_HALF; j += 4) {
      const int c = hf * CH_HALF + j;
      // (the channels of a row in any order, the same for both operands: neighbours' stores side by side)
      *reinterpret_cast<f32x4*>(&s.row[row][16 * j + 4 * m]) = f32x4{x(c), x(c + 1), x(c + 2), x(c + 3)};
    }
  };
  // Rows ra .. ra + 15 times rows rb .. rb + nb - 1: entry i of lane (column m, group gr) is row 4 gr + i.  Of fp32
  // results the rounding of these sums of 128 terms is most of the error: eight sums of 16 terms, and with 32-bit inputs
  // the fp64 matrix cores.  Results of 32-bit prompts of 500 tokens, errors against 64 bits token by token / with sums in
  // fp32 / here (1e-7): delta rule 1.26 / 1.30 / 1.19, per channel 1.30 / 1.32 / 1.26, state space 1.14 / 1.20 / 1.10.
  // (`rows` puts down a half's rows; with `self` also rows rb .. times themselves, into `own`)
  typedef std::conditional_t<sizeof(T) == 4, f64x4, f32x4> sums;
  auto product = [&](auto rows, int ra, int rb, int nb, auto self, sums& own) __attribute__((always_inline)) {
    constexpr int N = sizeof(T) == 4 ? 2 : PAIRS ? 4 : 8;
    sums x[N], y[N];
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = y[i] = sums{0, 0, 0, 0};
    const float* pb = s.row[rb + (m & (nb - 1))] + 4 * gr;
    // (fp64: its entry i is row 4 i + gr)
    const int am = sizeof(T) == 4 ? 4 * (m & 3) + (m >> 2) : m;
    const float *pa = s.row[ra + am] + 4 * gr, *ps = s.row[rb + am] + 4 * gr;
    auto half = [&](auto hf) __attribute__((always_inline)) {
      rows(hf);
      wave_sync();
#pragma unroll
      for (int t = 0; t < WIDE / 16; ++t) {
        const f32x4 av = *reinterpret_cast<const f32x4*>(pa + 16 * t);
        const f32x4 bv = *reinterpret_cast<const f32x4*>(pb + 16 * t);
        f32x4 sv = av;
        if constexpr (self) sv = *reinterpret_cast<const f32x4*>(ps + 16 * t);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (sizeof(T) == 4) {
            x[i & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i], bv[i], x[i & 1], 0, 0, 0);
            if constexpr (self) y[i & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(sv[i], bv[i], y[i & 1], 0, 0, 0);
          } else {
            const int e = (4 * t + i) % N;
            x[e] = mma(av[i], bv[i], x[e]);
            if constexpr (self) y[e] = mma(sv[i], bv[i], y[e]);
          }
        }
      }
    };
    half(std::integral_constant<int, 0>{});
    if constexpr (HALVES == 2) {
      wave_sync();
      half(std::integral_constant<int, 1>{});
    }
    auto total = [](const sums* z) {
      if constexpr (sizeof(T) == 4) return z[0] + z[1];
      else if constexpr (N == 4) return (z[0] + z[1]) + (z[2] + z[3]);
      else return ((z[0] + z[1]) + (z[2] + z[3])) + ((z[4] + z[5]) + (z[6] + z[7]));
    };
    own = total(y);
    return total(x);
  };
  if constexpr (!CH) {
    wave_sync();
    f64x4 zq, zk;   // (32-bit inputs: of 64 bits)
    auto score = [&](int i) {
      if constexpr (sizeof(T) == 4) return zq[i];
      else return xq[i];
    };
    auto key_score = [&](int i) {
      if constexpr (sizeof(T) == 4) return zk[i];
      else return xk[i];
    };
    if constexpr (!EXACT) {
      auto rows = [&](auto hf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          put(4 * gr + i, hf, [&](int j) { return q[i][j]; });
          put(16 + 4 * gr + i, hf, [&](int j) { return k[i][j]; });
        }
      };
      if constexpr (sizeof(T) == 4) zq = product(rows, 0, 16, 16, std::bool_constant<DELTA>{}, zk);
      else xq = product(rows, 0, 16, 16, std::bool_constant<DELTA>{}, xk);
    }
    // D_ij for this lane's column j = m and rows i = 4 gr .. + 3
    float D[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) D[i] = MODE == kModeRetention ? pw[max(4 * gr + i - m, 0)] : 1.f;
    if (MODE != kModeRetention) {
      // tokens in fours: what is left of j's four, whole fours between, i's four up to i
      auto four = [&](int b) { return *reinterpret_cast<const f32x4*>(&s.sc[3][4 * b]); };
      const int bj = m >> 2, mm = m & 3;
      const f32x4 dj = four(bj), di = four(gr), d1 = four(1), d2 = four(2);
      const float x1 = mm < 1 ? dj[1] : 1.f, x2 = mm < 2 ? dj[2] : 1.f, x3 = mm < 3 ? dj[3] : 1.f;
      const float left[4] = {1.f, x1, x1 * x2, x1 * x2 * x3};
      const float up[4] = {di[0], di[0] * di[1], di[0] * di[1] * di[2], (di[0] * di[1]) * (di[2] * di[3])};
      const float between = (bj < 1 && gr > 1 ? (d1[0] * d1[1]) * (d1[2] * d1[3]) : 1.f) *
                            (bj < 2 && gr > 2 ? (d2[0] * d2[1]) * (d2[2] * d2[3]) : 1.f);
#pragma unroll
      for (int i = 0; i < 4; ++i) D[i] = bj == gr ? left[i] : left[3] * between * up[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ti = 4 * gr + i;
      s.sq[ti][m] = m <= ti ? score(i) * D[i] * s.sc[0][ti] * s.sc[1][m] : 0.f;
      if (DELTA) s.sk[ti][m] = m < ti ? key_score(i) * D[i] * s.sc[1][ti] * s.sc[1][m] * s.sc[2][ti] : 0.f;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ti = 4 * gr + i;
      s.sq[ti][m] = 0.f;
      if (DELTA) s.sk[ti][m] = 0.f;
    }
    wave_sync();
    if (!PAIRS && lane < 16) s.sq[lane][lane] = diag * s.sc[0][lane] * s.sc[1][lane];
    // local products of the lane's four tokens, for the channels of a half: from the first on, and behind a token to the last
    struct Local {
      float pf[4][CH_HALF], sf[4][CH_HALF];
    };
    auto local = [&](auto hf) __attribute__((always_inline)) {
      Local l;
#pragma unroll
      for (int j = 0; j < CH_HALF; ++j) {
        const int c = hf * CH_HALF + j;
        l.pf[0][j] = d[0][c];
        l.sf[3][j] = 1.f;
#pragma unroll
        for (int i = 1; i < 4; ++i) {
          l.pf[i][j] = l.pf[i - 1][j] * d[i][c];
          l.sf[3 - i][j] = l.sf[4 - i][j] * d[4 - i][c];
        }
      }
      return l;
    };
    // A level, delta rule: rows 0 - 7 q of the later halves, 8 - 15 their k, 16 - 23 k of the earlier halves; u counts
    // the tokens of a kind.  Forget gate: only q, so two levels share a product: 8 - 15 and 24 - 31 are q and k of the
    // second one, and the blocks of two levels are not used.
    constexpr int LK = DELTA ? 0 : 8;   // the second level's rows behind the first's
    auto level = [&](auto half_a, auto half_b, auto rows) __attribute__((always_inline)) {   // (delta rule: half_a only)
      constexpr int HA = decltype(half_a)::value, HB = decltype(half_b)::value;
      sums none;
      const auto x = product(rows, 0, 16, DELTA ? 8 : 16, std::false_type{}, none);
      if (DELTA ? m < 8 : m >> 3 == gr >> 1)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int u = 4 * (gr & 1) + i, v = m & 7;
          auto pair = [&](auto half) {
            constexpr int HS = decltype(half)::value;
            if (u / HS == v / HS) {
              const int ti = (u / HS) * 2 * HS + HS + u % HS, tj = (v / HS) * 2 * HS + v % HS;
              if (!DELTA || gr < 2) s.sq[ti][tj] = DELTA && !PAIRS ? x[i] * s.sc[0][ti] * s.sc[1][tj] : x[i];
              else s.sk[ti][tj] = PAIRS ? x[i] : x[i] * s.sc[1][ti] * s.sc[1][tj] * s.sc[2][ti];
            }
          };
          if (DELTA || gr < 2) pair(std::integral_constant<int, HA>{});
          else pair(std::integral_constant<int, HB>{});
        }
      wave_sync();
    };
    using std::integral_constant;
    const bool far = gr == 3 || gr == 0;
    auto rows8 = [&](auto hf, const Local& l) __attribute__((always_inline)) {   // halves of 8: later groups 2, 3, earlier groups 0, 1
      float other[CH_HALF];
#pragma unroll
      for (int j = 0; j < CH_HALF; ++j) other[j] = __shfl_xor(l.pf[3][j], 16, kWave);   // the neighbour group's four tokens
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        auto f = [&](int c) {
          const int j = c - hf * CH_HALF;
          return (gr >= 2 ? l.pf[i][j] : l.sf[i][j]) * (far ? other[j] : 1.f);
        };
        if (gr >= 2) {
          put(4 * (gr - 2) + i, hf, [&](int c) { return q[i][c] * f(c); });
          if (DELTA) put(8 + 4 * (gr - 2) + i, hf, [&](int c) { return k[i][c] * f(c); });
        } else {
          put(16 + 4 * gr + i, hf, [&](int c) { return k[i][c] * f(c); });
          asm volatile("");   // (two branches, not one with a choice of q's and k's addresses, which would put them into memory)
        }
      }
    };
    auto rows4 = [&](auto hf, const Local& l) __attribute__((always_inline)) {   // halves of 4: later groups 1, 3, earlier groups 0, 2
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (gr & 1) {
          put(LK + 4 * (gr >> 1) + i, hf, [&](int c) { return q[i][c] * l.pf[i][c - hf * CH_HALF]; });
          if (DELTA) put(8 + 4 * (gr >> 1) + i, hf, [&](int c) { return k[i][c] * l.pf[i][c - hf * CH_HALF]; });
        } else {
          put(16 + LK + 4 * (gr >> 1) + i, hf, [&](int c) { return k[i][c] * l.sf[i][c - hf * CH_HALF]; });
          asm volatile("");
        }
      }
    };
    if constexpr (DELTA) {
      level(integral_constant<int, 8>{}, integral_constant<int, 8>{}, [&](auto hf) __attribute__((always_inline)) { rows8(hf, local(hf)); });
      level(integral_constant<int, 4>{}, integral_constant<int, 4>{}, [&](auto hf) __attribute__((always_inline)) { rows4(hf, local(hf)); });
    } else {
      level(integral_constant<int, 8>{}, integral_constant<int, 4>{}, [&](auto hf) __attribute__((always_inline)) {
        const Local l = local(hf);
        rows8(hf, l);
        rows4(hf, l);
      });
    }
    // Pairs inside a lane's four tokens: with 16-bit inputs sums on the vector units, eight channels per lane and a tree over
    // the 16 lanes.  Products of matrices would have 8 (32) of their 256 (512) results used, and in fp32 they take the
    // vector units as long as four times these instructions (us: delta rule per channel, 4 x 1.9k tokens, 132 -> 111;
    // forget gate, 16 x 460, 101 -> 94).  (32-bit inputs: sums of 64 bits, on the matrix cores.)
    constexpr bool FOURS = sizeof(T) == 2;
    if constexpr (FOURS) {
      constexpr int N = DELTA ? 12 : 6;
      float x[N];   // q_i k_j of (1, 0), (2, 0), (3, 0), (2, 1), (3, 1), (3, 2); delta rule: then k_i k_j
#pragma unroll
      for (int e = 0; e < N; ++e) x[e] = 0.f;
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        int e = 0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          float f = k[j][c];
#pragma unroll
          for (int i = j + 1; i < 4; ++i, ++e) {
            f *= d[i][c];
            x[e] = __builtin_fmaf(q[i][c], f, x[e]);
            if constexpr (DELTA) x[6 + e] = __builtin_fmaf(k[i][c], f, x[6 + e]);
          }
        }
      }
#pragma unroll
      for (int e = 0; e < N; ++e) x[e] = group_sum<16>(x[e]);
      float y = x[0];   // lane e puts down sum e
#pragma unroll
      for (int e = 1; e < N; ++e) y = m == e ? x[e] : y;
      const int e = m < 6 ? m : m - 6, j = e < 3 ? 0 : e < 5 ? 1 : 2, i = e < 3 ? e + 1 : e < 5 ? e - 1 : 3;
      const int ti = 4 * gr + i, tj = 4 * gr + j;
      if (DELTA && !PAIRS) y *= s.sc[m < 6 ? 0 : 1][ti] * s.sc[1][tj] * (m < 6 ? 1.f : s.sc[2][ti]);
      if (m < N) (m < 6 ? s.sq : s.sk)[ti][tj] = y;
    }
    if constexpr (!FOURS) {
      auto rows2 = [&](auto hf) __attribute__((always_inline)) {   // halves of 2: tokens 2, 3 and 0, 1 of every group
        put(2 * gr, hf, [&](int j) { return q[2][j] * d[2][j]; });
        put(2 * gr + 1, hf, [&](int j) { return q[3][j] * (d[2][j] * d[3][j]); });
        if (DELTA) {
          put(8 + 2 * gr, hf, [&](int j) { return k[2][j] * d[2][j]; });
          put(8 + 2 * gr + 1, hf, [&](int j) { return k[3][j] * (d[2][j] * d[3][j]); });
        }
        put(16 + 2 * gr, hf, [&](int j) { return k[0][j] * d[1][j]; });
        put(16 + 2 * gr + 1, hf, [&](int j) { return k[1][j]; });
      };
      auto rows1 = [&](auto hf) __attribute__((always_inline)) {   // neighbours
        put(LK + 2 * gr, hf, [&](int j) { return q[1][j] * d[1][j]; });
        put(LK + 2 * gr + 1, hf, [&](int j) { return q[3][j] * d[3][j]; });
        if (DELTA) {
          put(8 + 2 * gr, hf, [&](int j) { return k[1][j] * d[1][j]; });
          put(8 + 2 * gr + 1, hf, [&](int j) { return k[3][j] * d[3][j]; });
        }
        put(16 + LK + 2 * gr, hf, [&](int j) { return k[0][j]; });
        put(16 + LK + 2 * gr + 1, hf, [&](int j) { return k[2][j]; });
      };
      if constexpr (DELTA) {
        level(integral_constant<int, 2>{}, integral_constant<int, 2>{}, rows2);
        level(integral_constant<int, 1>{}, integral_constant<int, 1>{}, rows1);
      } else {
        level(integral_constant<int, 2>{}, integral_constant<int, 1>{}, [&](auto hf) __attribute__((always_inline)) {
          rows2(hf);
          rows1(hf);
        });
      }
    }
  }
  if constexpr (PAIRS) {
    lds_barrier();
    const Lds &s0 = lds_all[w & ~1], &s1 = lds_all[w | 1];
    auto sum = [&](int e) { return s0.sum[PAIRS ? e : 0][m] + s1.sum[PAIRS ? e : 0][m]; };
    const float qk = sum(2);
    if (DELTA) {
      qi = 1.0f / (sqrtf(static_cast<float>(a.dk)) * sqrtf(sum(0) + 1e-6f));
      ki = 1.0f / sqrtf(sum(1) + 1e-6f);
    }
    if (lane < 16) s.sc[1][lane] = ki;
    wave_sync();
    const f32x4 kj = *reinterpret_cast<const f32x4*>(&s.sc[1][4 * gr]);   // of the columns 4 gr ...
    auto both = [&](const float (&x)[20], const float (&y)[20]) {
      return *reinterpret_cast<const f32x4*>(&x[4 * gr]) + *reinterpret_cast<const f32x4*>(&y[4 * gr]);
    };
    if ((w & 1) == 0) {   // A and the scales
      f32x4 x = both(s0.sq[m], s1.sq[m]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {   // (zeros above the diagonal: a later token's scale may be NaN)
        const int j = 4 * gr + i;
        x[i] = j <= m ? (j == m ? qk : x[i]) * qi * kj[i] : 0.f;
      }
      *reinterpret_cast<f32x4*>(rec + m * 16 + 4 * gr) = x;
      if (lane < 16) {
        rec[kRecQ + lane] = qi;
        rec[kRecK + lane] = ki;
        rec[kRecKt + lane] = ki;
        rec[kRecEnd + lane] = lane == kRecNoParts - kRecEnd ? 0.f : 1.f;
      }
      return;
    }
    if constexpr (DELTA) {   // L
      f32x4 x = both(s0.sk[m], s1.sk[m]);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = 4 * gr + i < m ? x[i] * ki * kj[i] * beta : 0.f;
      *reinterpret_cast<f32x4*>(&s.sk[m][4 * gr]) = x;
      wave_sync();
    } else {
      return;
    }
  } else {
    wave_sync();
    *reinterpret_cast<f32x4*>(rec + m * 16 + 4 * gr) = *reinterpret_cast<const f32x4*>(&s.sq[m][4 * gr]);
  }
  if constexpr (DELTA) {
    // (I + L) T = diag(beta), one column per lane (lanes 16 - 63 repeat the columns).  Lane m of each 16 has row m of L, and
    // L_ij comes from there as the multiply-add's own broadcast operand (read from LDS it is waited for, row by row).
    float L[16], x[16];
#pragma unroll
    for (int j = 0; j < 16; j += 4) {
      const f32x4 l = *reinterpret_cast<const f32x4*>(&s.sk[m][j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) L[j + e] = -l[e];
    }
    const float bc = PAIRS ? beta : s.sc[2][m];
    auto row_of = [&](auto self, auto i_) __attribute__((always_inline)) -> void {
      constexpr int i = decltype(i_)::value, last = i & ~3;
      x[i] = i == m ? bc : 0.f;
#pragma unroll
      for (int j = 0; j < last; j += 4) add_broadcast<i, 4>(x[i], L + j, x + j);
      add_broadcast<i, i - last>(x[i], L + last, x + last);
      if constexpr (i < 15) self(self, std::integral_constant<int, i + 1>{});
    };
    row_of(row_of, std::integral_constant<int, 0>{});
#pragma unroll
    for (int i = 0; i < 4; ++i) {   // lane group gr stores rows 4 gr .. of its column
      float v = x[i];
#pragma unroll
      for (int b = 1; b < 4; ++b) v = gr == b ? x[4 * b + i] : v;
      rec[kRecT + (4 * gr + i) * 16 + m] = v;
    }
  }
}

// A token's infinity or NaN must not reach earlier tokens of its chunk (0 x inf in a triangular product): x
// loses its non-finite entries, and the result is 0, or NaN from a column's first such token on.  Lane (column,
// group gr) holds token 4 gr + i in entry i.
__device__ __forceinline__ f32x4 take_nonfinite(f32x4& x, int lane) {
  f32x4 p = x * 0.f;
  const float sum = (p[0] + p[1]) + (p[2] + p[3]);
  float before = 0.f;
#pragma unroll
  for (int g = 0; g < 3; ++g) {
    const float t = __shfl(sum, (lane & 15) + 16 * g, kWave);
    before += g < lane >> 4 ? t : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[i] = p[i] == 0.f ? x[i] : 0.f;
    before += p[i];
    p[i] = before;
  }
  return p;
}

// ---- walk ---------------------------------------------------------------------------------------------

// Portion y of those that run in chunks, -1: there are fewer.  Every wave looks through the lengths, 64 at a time.
// Of S portions with T rows at most T / min_rows have min_rows, and the grid has so many where that is less than S: a
// workgroup of 12 waves and 120 KB that finds nothing to do takes its CU as long as its launch takes (state space, 32
// heads, us with a workgroup per portion / here: 200 decode rows beside 900 362 / 312, 127 beside 256 172 / 123; delta
// rule 291 / 275, 136 / 125).
__device__ __forceinline__ int find_portion(const ChunkArgs& a, int y) {
  if (a.walk_portions >= a.S) return y < a.S ? y : -1;   // (a workgroup per portion, also without chunks)
  const int lane = threadIdx.x & 63;
  for (int s0 = 0; s0 < a.S; s0 += kWave) {
    const int s = min(s0 + lane, a.S - 1);
    const bool on = s0 + lane < a.S && a.seq_slot[s] >= 0 && a.seq_qstart[s + 1] - a.seq_qstart[s] >= a.min_rows;
    const uint64_t m = __ballot(on);
    const int n = __popcll(m);
    if (y < n) {
      const int rank = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(m >> 32),
                                                 __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(m), 0));
      return s0 + __builtin_ctzll(__ballot(on && rank == y));
    }
    y -= n;
  }
  return -1;
}

// Segment y of the batch: segment j of the P of portion s, whose first segment's state is number `state` (cut
// portions only).  Every wave works it out from the portions' lengths, 64 at a time.
//
// Portions that are not cut run beside the first pass, so a cut pays only if the longest portion takes longer than the
// longest uncut one and the two passes over the longest segment together: in units of 0.05 us per chunk 39 with outputs,
// 24 without, and 120 for the second pass's start.  The recurrences differ from that by a common factor (forget gate
// 1.7 us per chunk with outputs, retention and state space 1.5), and where the cut begins to pay is the same for all: one
// portion in 8 heads, whole / in two segments: 300 rows forget gate 51 / 51, 350 rows forget gate 56 / 55, retention
// 46 / 49, state space 43 / 42; 400 rows 61 / 58, 50 / 52, 47 / 45.  A batch that could be cut and is not pays for the
// second launch, 4 - 5 us.
struct Segment {
  int s, j, P, state, len;   // len: chunks per segment
};
template <bool CUT>   // count the segments of cut portions only
__device__ __forceinline__ Segment find_segment(const ChunkArgs& a, int y) {
  const int lane = threadIdx.x & 63;
  auto chunks_of = [&](int s) {
    const int n = s < a.S && a.seq_slot[min(s, a.S - 1)] >= 0 ? a.seq_qstart[s + 1] - a.seq_qstart[s] : 0;
    return n >= a.min_rows ? (n + kScanChunk - 1) / kScanChunk : 0;
  };
  int longest = 0, uncut = 0, part = 0;
  for (int s0 = 0; s0 < a.S; s0 += kWave) {
    const int nc = chunks_of(s0 + lane), len = scan_segment_chunks(nc, a.seg_chunks);
    longest = max(longest, nc);
    if (len >= nc) uncut = max(uncut, nc);
    else part = max(part, len);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    longest = max(longest, __shfl_xor(longest, o, kWave));
    uncut = max(uncut, __shfl_xor(uncut, o, kWave));
    part = max(part, __shfl_xor(part, o, kWave));
  }
  if (39 * longest <= 39 * uncut + (24 + 39) * part + 120)   // units of 0.05 us
    return {CUT ? -1 : find_portion(a, y), 0, 1, 0, 0};      // every portion whole
  int pairs = 0, states = 0;
  for (int s0 = 0; s0 < a.S; s0 += kWave) {
    const int nc = chunks_of(s0 + lane), len = scan_segment_chunks(nc, a.seg_chunks);
    const int P = (nc + len - 1) / len, Q = P > 1 ? P : 0, N = CUT ? Q : P;
    int ip = N, iq = Q;   // inclusive sums over the lanes
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int up = __shfl_up(ip, o, kWave), uq = __shfl_up(iq, o, kWave);
      ip += lane >= o ? up : 0;
      iq += lane >= o ? uq : 0;
    }
    const uint64_t hit = __ballot(pairs + ip > y);
    if (hit != 0) {
      const int l = __builtin_ctzll(hit);
      auto of = [&](int v) { return __builtin_amdgcn_readlane(v, l); };
      return {s0 + l, y - (pairs + of(ip) - of(N)), of(P), states + of(iq) - of(Q), of(len)};
    }
    pairs += __builtin_amdgcn_readlane(ip, 63);
    states += __builtin_amdgcn_readlane(iq, 63);
  }
  return {-1, 0, 0, 0, 0};
}

// Retention: a slow head remembers hundreds of chunks, and the decay over a chunk, rounded, would be off by the same
// rounding in each (error of a state of 8000 tokens at a decay of 0.9999: 5.6e-6, 1.8e-6 with the chunks of 64 tokens
// before, 1.4e-6 here).  What it leaves is taken from the power of 64, and the chunks' factors are the two nearest
// numbers in turn, so that their product stays within a rounding of the true power.
struct ChunkDecay {
  float e = 1.f, rest = 0.f;      // the rounded decay, and what it leaves
  float up = 0.f, down = 0.f;     // to its neighbours
  float err = 0.f;                // what the factors so far leave
  __device__ void set(const float* pw) {
    e = pw[kScanChunk];
    const float x = pw[64];
    if (!(e > 0.25f)) return;     // (forgotten before it counts)
    const double e2 = static_cast<double>(e) * e;
    rest = static_cast<float>(x - e2 * e2) / (4.f * e * e * e);   // x = (e + rest)^4
    up = __builtin_bit_cast(float, __builtin_bit_cast(int, e) + 1) - e;
    down = e - __builtin_bit_cast(float, __builtin_bit_cast(int, e) - 1);
  }
  __device__ float next() {
    err += rest;
    const float s = err > 0.5f * up ? up : err < -0.5f * down ? -down : 0.f;
    err -= s;
    return e + s;
  }
};

// V is exact in one part where it goes into the state and the outputs as it came, in 16 bits: its scale is in the keys.
// (State space: two heads with scales of their own share the keys.)  Two products per tile of S in place of four, and two
// of bf16 in place of four in fp32 for A V: walk of the forget gate, 16 x ~460 tokens, 166 -> 157 us, of retention, 1500
// tokens, 27 + 43 -> 25 + 41; results in 1e-7 from 64 bits (forget gate, 2500 tokens) 1.12 -> 1.08.  (With 8-byte reads of
// the first part and products of 16 terms, which come without the zeros, 151 us, but a product of 32 terms followed by one
// of 16 that adds to it loses two of four rows: the compiler leaves too few cycles between the two.)
template <typename T, int MODE>
constexpr bool exact_values() { return sizeof(T) == 2 && (MODE == kModeForget || MODE == kModeRetention); }

// Queries and keys are exact in one part where they go into the products as they came, in 16 bits: their scales and the one
// number of the decay come afterwards.  A sum over S's rows then takes three products in place of six, and kt U, as kt is the
// keys, two per tile; no part is worked out, and a third of the operands goes through LDS.  Walk, us, three parts / one:
// delta rule, 32 heads of 128, 4 x 1.9k tokens 206 / 156, state space, 128 heads of 128 x 64 43.5 + 82 / 32.5 + 67 (states
// 7 % closer to 64 bits).
template <typename T, int MODE>
constexpr bool exact_rows() { return sizeof(T) == 2 && (MODE == kModeStateSpace || MODE == kModeDelta); }

// A chunk's operands.
template <int MODE, int DK, bool EXACT, bool ONE>
struct WalkBuf {
  static constexpr bool DELTA = MODE >= kModeDelta, CH = per_channel<MODE>();
  static constexpr int COLS = DELTA ? kWalkCols : 2 * kWalkCols, HEADS = MODE == kModeStateSpace ? 2 : 1;
  // rows in three parts, per four tokens and channel as the lane that prepares them holds them; the reads transpose
  static constexpr int ROW = DK + (DK == 64 ? 8 : 16);
  typedef u32x2 Rows[ONE ? 1 : 3][4][ROW];
  Rows qe;                              // P_i q_i; one number as the decay: q_i
  u32x2 ke[DELTA && !ONE ? 3 : 1][DELTA ? 4 : 1][DELTA ? ROW : 1];   // P_i k_i; k_i
  // D_end,j k_j; not EXACT and one number as the decay: k_j.  Per four tokens and channel two parts of each
  // parts 0 and 1; EXACT: 0; ONE: the number, which a delta rule has in ke
  std::conditional_t<EXACT || ONE, u32x2, u32x4> kt01[DELTA && ONE ? 1 : 4][DK];
  u32x4 kt20[ONE ? 1 : 4][DK];          // ... 2 and 0; EXACT: 2 and 1
  __bf16 amat[EXACT ? 2 : 1][16][4][8]; // EXACT: A per row and four tokens: part 0, and zeros; parts 2 and 1
  f32x4 v[4][COLS];                     // per four tokens and column
  float mat[HEADS][DELTA ? 512 : 256];  // of the record: A, and T
  float scale[HEADS][64];               // ... kRecQ, kRecK, kRecKt, kRecEnd
  float end[CH ? DK : 4];               // P_end
};
template <int MODE, int DK, bool EXACT, bool ONE>
struct WalkLds {
  static constexpr bool DELTA = MODE >= kModeDelta;
  static constexpr int BUFS = DELTA ? 2 : 3;
  union {
    WalkBuf<MODE, DK, EXACT, ONE> buf[BUFS];
    float start[DELTA ? 1 : DK][2 * kWalkCols + 4];   // the state at a segment's start
  };
};
// The walk's workgroup: four waves with products, and those with operands.
constexpr int kWalkWaves = 4;
template <int MODE, int DK>
constexpr int walk_threads() { return kWave * (kWalkWaves + operand_waves(MODE, DK)); }
// Waves per SIMD that its registers are for: one workgroup's; with keys of up to 64 channels and one tile of columns per wave
// those of two workgroups of eight waves, whose buffers fit on a CU too (us, one / two of them, 32 portions of 20 in 32 bits,
// 32 heads of 64: state space 46 / 36, delta rule 35 / 30).
template <int MODE, int DK, int CT>
constexpr int walk_simd_waves() { return walk_threads<MODE, DK>() > 512 ? 3 : CT == 1 && DK == 64 ? 4 : 2; }
constexpr size_t kLdsBytes = 160 * 1024;

// VEC 2: aligned rows of q, k and v; 1: but for v (an odd width or row, which only the loads of two columns at once mind: with
// the rows of q and k element by element as well, a retention of 16 x 512 tokens, 32 heads of 64 with rows of v one element
// apart from alignment, took 386 us, here 129, aligned 125); 0: loads element by element.
// PASS 0: whole portions.  1 and 2: cut portions.  Pass 1 has no outputs: the first segment goes from the sequence's
// state (of which it leaves a copy, since pass 2 overwrites it) to the state at its end; the others but the last from
// zero to what they add to the state, with the decay over them.  Pass 2 puts the state at a segment's start together
// from these and walks it; the last segment writes the sequence's state.
template <typename T, int MODE, int DK, int VEC, int PASS, int CT>
__device__ __forceinline__ void walk(const ChunkArgs& a, const Segment sg, WalkLds<MODE, DK, exact_values<T, MODE>(), exact_rows<T, MODE>()>& lds) {
  constexpr int NT = DK / 16, kDecay = scan_rec_decay(MODE);
  const int REC = scan_record_floats(MODE, VEC ? DK : a.dk), DS = scan_decay_width(VEC ? DK : a.dk);   // (scan_scores_kernel)
  constexpr bool DELTA = MODE >= kModeDelta, CH = per_channel<MODE>();
  // A . U of 32-bit inputs on the fp64 matrix cores, as A itself (scan_scores_kernel): with A alone the forget gate's
  // results, which have fewer roundings in front of the recurrence than the others', are at 0.83 x 1e-7 from 64 bits
  // (token by token 0.78), with both at 0.74.  The others do not need it (state space: 6 us of 67).
  constexpr bool F64 = sizeof(T) == 4 && MODE == kModeForget;
  constexpr bool EXACT = exact_values<T, MODE>();
  constexpr bool ONE = exact_rows<T, MODE>();
  constexpr int RP = ONE ? 1 : 3;   // parts of the rows
  using Buf = WalkBuf<MODE, DK, EXACT, ONE>;
  constexpr int BUFS = WalkLds<MODE, DK, EXACT, ONE>::BUFS, OW = operand_waves(MODE, DK);
  static_assert(DK != 64 || 2 * sizeof(lds) <= kLdsBytes, "two workgroups per CU (walk_simd_waves)");
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Identity id(lane);
  constexpr int waves = kWalkWaves, tiles = CT * waves;   // of the products; columns in 16s
  const int hb = a.H / a.walk_heads, cb = blockIdx.x / hb, h0 = blockIdx.x % hb * a.walk_heads;
  // wave w: 16 CT columns of a head
  const bool two = a.walk_heads == 2;
  const int h = two && w < waves ? h0 + (CT * w >> 2) : h0;
  const int col0 = DELTA || two ? cb * kWalkCols + 16 * (CT * w & 3) : 16 * (cb * tiles + CT * w);
  const int s = sg.s, slot = a.seq_slot[s];
  int first = a.seq_qstart[s], n = a.seq_qstart[s + 1] - first;
  if (slot < 0 || n < a.min_rows) return;
  const float* rec0 = a.rec + (static_cast<int64_t>(first / kScanChunk + s) * a.H + h) * REC;
  const int64_t rec_step = static_cast<int64_t>(a.H) * REC;
  if (PASS != 0) {   // the segment's rows
    const int c0 = sg.j * sg.len;
    rec0 += c0 * rec_step;
    first += c0 * kScanChunk;
    n = min(n - c0 * kScanChunk, sg.len * kScanChunk);
  }
  const int nc = (n + kScanChunk - 1) / kScanChunk;
  // scratch of a cut portion's segment j: the decay over it, by row of S; a state [dk, dv] (the last segment's: the
  // copy of the sequence's)
  auto seg_decay = [&](int j, int h) { return a.seg + (static_cast<int64_t>(sg.state + j) * a.H + h) * 128; };
  auto seg_state = [&](int j, int h) {
    return a.seg + static_cast<int64_t>(a.seg_states) * a.H * 128 +
           (static_cast<int64_t>(sg.state + j) * a.H + h) * a.dk * a.dv;
  };
  if constexpr (PASS == 2 && !DELTA) {
    if (sg.j > 0) {   // by all 512 threads, 64 columns four at a time, up to four segments' loads ahead
      static_assert(PASS != 2 || DELTA || walk_threads<MODE, DK>() == 512);
      auto put_together = [&](auto blocks) {
        constexpr int B = decltype(blocks)::value, U = DK * (kWalkCols / 4) / 512, AHEAD = 4 / B;
        f32x4 acc[B][U];
        const bool v4 = a.dv % 4 == 0;
        auto head = [&](int b) { return two ? h0 + b : h0; };
        auto at = [&](int j, int b, int u) {
          const int f = tid + 512 * u, d = min(f >> 4, a.dk - 1);
          const int col = (two ? cb : B * cb + b) * kWalkCols + 4 * (f & 15);
          const float* r = seg_state(j, head(b)) + static_cast<int64_t>(d) * a.dv;
          if (v4) return *reinterpret_cast<const f32x4*>(r + min(col, a.dv - 4));
          f32x4 x;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = r[min(col + e, a.dv - 1)];
          return x;
        };
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
          for (int u = 0; u < U; ++u) acc[b][u] = at(0, b, u);
        for (int j = 1; j < sg.j; j += AHEAD) {
          f32x4 x[AHEAD][B][U];
          float D[AHEAD][B][U];
#pragma unroll
          for (int e = 0; e < AHEAD; ++e)
#pragma unroll
            for (int b = 0; b < B; ++b)
#pragma unroll
              for (int u = 0; u < U; ++u) {
                const int i = min(j + e, sg.j - 1), d = min((tid + 512 * u) >> 4, a.dk - 1);
                x[e][b][u] = at(i, b, u);
                D[e][b][u] = seg_decay(i, head(b))[CH ? d : 0];
              }
#pragma unroll
          for (int e = 0; e < AHEAD; ++e)
            if (j + e < sg.j)
#pragma unroll
              for (int b = 0; b < B; ++b)
#pragma unroll
                for (int u = 0; u < U; ++u) acc[b][u] = acc[b][u] * D[e][b][u] + x[e][b][u];
        }
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int f = tid + 512 * u;
            *reinterpret_cast<f32x4*>(&lds.start[f >> 4][kWalkCols * b + 4 * (f & 15)]) = acc[b][u];
          }
      };
      put_together(std::integral_constant<int, CT>{});
      lds_barrier();
    }
  }

  if (w < waves) {
    // ---- products
    __builtin_amdgcn_s_setprio(1);   // (their chain is the longer one: walk of the per-channel delta rule 224 -> 222 us)
    const int m = lane & 15, gr = lane >> 4;
    float* st = a.state + (static_cast<int64_t>(slot) * a.H + h) * a.dk * a.dv;
    f32x4 S[CT][NT];
    // (the last segment of a cut portion holds the copy of the sequence's state)
    const float* from = PASS == 2 ? seg_state(sg.P - 1, h) : st;
    const bool blank = PASS == 1 && sg.j > 0, fresh = (PASS == 0 || sg.j == 0) && a.positions[first] == 0;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int t = 0; t < NT; ++t) S[ct][t] = zero;
    if (!fresh && !blank)   // (uniform)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const int col = col0 + 16 * ct + m;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int d = 16 * t + 4 * gr + i;
            const bool in = col < a.dv && d < a.dk;
            const float x = PASS == 2 && sg.j > 0 ? lds.start[DELTA ? 0 : d][16 * (CT * w + ct) + m]
                                                  : from[static_cast<int64_t>(min(d, a.dk - 1)) * a.dv + min(col, a.dv - 1)];
            S[ct][t][i] = in ? x : 0.f;
          }
      }
    if (PASS == 2 && sg.j > 0) lds_barrier();   // (the operands' buffers are the same memory)
    auto store_state = [&](float* p) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        int c = col0 + 16 * ct + m, r = 4 * gr;   // (new values: the addresses of the loads would be kept over the chunks)
        asm volatile("" : "+v"(c), "+v"(r));
        if (c < a.dv)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int d = 16 * t + r + i;
              if (d < a.dk) p[static_cast<int64_t>(d) * a.dv + c] = S[ct][t][i];
            }
      }
    };
    if (PASS == 1 && sg.j == 0 && !fresh) store_state(seg_state(sg.P - 1, h));
    float* op = a.out + (static_cast<int64_t>(first) * a.H + h) * a.dv;
    const int o_stride = a.H * a.dv;
    const float skip = MODE == kModeStateSpace ? a.p2[h] : 0.f;
    ChunkDecay fixed;
    if (MODE == kModeRetention) fixed.set(a.p0 + h * kPowers);
    float over = 1.f;   // one number as the decay: over the chunks so far
    const int head = Buf::HEADS == 2 && two ? CT * w >> 2 : 0;
    // of the record: A or T (row m; the fp64 product's results want the rows in another order), and the scales of the
    // tokens 4 gr ...
    auto matrix = [&](const Buf& b, int at) {
      return *reinterpret_cast<const f32x4*>(&b.mat[head][at + 16 * (F64 ? 4 * (m & 3) + (m >> 2) : m) + 4 * gr]);
    };
    auto scale = [&](const Buf& b, int at) {
      return MODE == kModeForget ? zero : *reinterpret_cast<const f32x4*>(&b.scale[head][at - kRecQ + 4 * gr]);
    };
    auto decay_of = [&](const Buf& b) { return CH ? 1.f : b.scale[head][kRecEnd - kRecQ]; };
    // A sum over the rows of S: the products of the first parts, and the smaller ones by themselves (products of parts 1
    // and 2 are below a 32-bit rounding of the result).
    struct Sum {
      f32x4 big, small[2];
    };
    // The rows of the 16 tokens, 32 channels in the order that a product over 32 rows of S takes them (of two tiles of S the
    // rows 4 gr + i).  The read transposes pieces of four tokens in groups of 16 lanes, four channels of all tokens; a lane's
    // own piece is at (token group m % 4, channel m / 4).
    auto row = [&](const u32x2 (&x)[4][Buf::ROW], int s) {
      typedef __attribute__((ext_vector_type(4))) short s16x4;
      auto get = [&](int t) {
        const u32x2* at = &x[m & 3][32 * s + 16 * t + 4 * gr + (m >> 2)];
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                             (__attribute__((address_space(3))) s16x4*)(void*)const_cast<u32x2*>(at)));
      };
      const u32x2 lo = get(0), hi = get(1);
      return u32x4{lo[0], lo[1], hi[0], hi[1]};
    };
    // product i of six of rows r and a state's parts q (ONE: of three)
    auto product = [&](Sum& x, const u32x4 (&r)[3], const u32x4 (&q)[3], int i) {
      constexpr int kRow[] = {0, 2, 0, 1, 1, 0}, kState[] = {2, 0, 0, 1, 0, 1}, kSum[] = {0, 1, 2, 0, 1, 0};
      if (kRow[i] >= RP) return;
      f32x4& to = kSum[i] == 2 ? x.big : x.small[kSum[i] % 2];
      to = mma(r[kRow[i]], q[kState[i]], to);
    };
    auto add = [&](Sum& x, const typename Buf::Rows& rows, const u32x4 (&p)[3], int s) {
      u32x4 r[3];
#pragma unroll
      for (int e = 0; e < RP; ++e) r[e] = row(rows[e], s);
#pragma unroll
      for (int i = 0; i < 6; ++i) product(x, r, p, i);
    };
    auto total = [](const Sum& x) {
      f32x4 y = x.big + (x.small[0] + x.small[1]);
      asm volatile("" : "+v"(y));   // (here, not where it is used: the sums would be kept until then)
      return y;
    };
    // The same in fp32, where parts are missing or the sum of rows that are not scaled is not finite; here they are (`scales`:
    // the scales in the record).
    auto sum_fp32 = [&](const Buf& b, const typename Buf::Rows& rows, int scales, const f32x4 (&S)[NT]) {
      const float sc = MODE == kModeForget ? 1.f : b.scale[head][scales - kRecQ + m];
      f32x4 x = zero;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          __builtin_amdgcn_sched_barrier(0);
          unsigned r[3];
#pragma unroll
          for (int e = 0; e < RP; ++e)
            r[e] = reinterpret_cast<const unsigned short*>(&rows[e][m >> 2][16 * t + 4 * gr + i])[m & 3];
          x = mma((ONE ? bf16_low(r[0]) : join(r[0], r[ONE ? 0 : 1], r[ONE ? 0 : 2], false)) * sc, S[t][i], x);
        }
      return x;
    };
    // the rows 32 s ... of S in parts
    auto state_parts = [&](u32x4 (&p)[3], int s, const f32x4 (&S)[NT]) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        unsigned x[3][2];
        id.split(S[2 * s + t], x);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          p[i][2 * t] = x[i][0];
          p[i][2 * t + 1] = x[i][1];
        }
      }
    };
    // U in parts, as the other operand of 16 tokens: half of a product's 32 terms, the other half takes other parts
    // (beside the parts 0 and 1, or 2 and 0, of the first operand)
    struct Parts {
      u32x4 p0, p10, p1, p02;
    };
    // EXACT: the number itself, beside part 0, or the parts 2 and 1, of the keys and of A.
    // ONE: parts 2 and 1, of products with the keys twice.
    auto as_parts = [](const unsigned (&u)[3][2]) {
      if constexpr (ONE) return Parts{u32x4{u[0][0], u[0][1], 0, 0}, u32x4{}, u32x4{}, u32x4{u[2][0], u[2][1], u[1][0], u[1][1]}};
      return Parts{u32x4{u[0][0], u[0][1], 0, 0}, u32x4{u[1][0], u[1][1], u[0][0], u[0][1]},
                   u32x4{0, 0, u[1][0], u[1][1]}, u32x4{u[0][0], u[0][1], u[2][0], u[2][1]}};
    };
    // of V, scaled as the state gets it
    auto parts = [&](const f32x4 V, const f32x4 by) {
      if constexpr (EXACT) {
        const unsigned u = pack_bf16(V[0], V[1]), v = pack_bf16(V[2], V[3]);
        return Parts{u32x4{u, v, 0, 0}, u32x4{}, u32x4{}, u32x4{u, v, u, v}};
      } else {
        unsigned u[3][2];
        if constexpr (CH) id.split(V, u);
        else id.template split<1>(split_product(V, by, u[0]), u);
        return as_parts(u);
      }
    };
    auto abs = [](const f32x4 x) { return f32x4{fabsf(x[0]), fabsf(x[1]), fabsf(x[2]), fabsf(x[3])}; };
    // numbers that split() takes, and sums that were not of others; `U`: as the state gets them
    auto ordinary = [&](const Buf& b, const f32x4 U, const f32x4 R) {
      const float keys = CH ? 0.f : b.scale[head][kRecNoParts - kRecQ];
      return !__any(!(abs_sum(U) + abs_sum(R) + keys <= 0.5f * kSplitMax));
    };
    auto finite = [](float x) { return fabsf(x) < HUGE_VALF; };
    // The product of the first parts.  EXACT and ONE: of 16 terms and, but for retention, as many zeros (a product adds the sum
    // so far to four terms and zeros at a time and rounds, one of 16 terms to more of them: states are 0.2 - 2 % further from
    // 64 bits with it, retention's are not, and the walk 2 - 4 % faster).
    // Where a product of 32 terms adds to one of 16, a vector instruction has to be in between: the compiler leaves too few
    // cycles.
    constexpr bool SHORT = MODE == kModeRetention;
    typedef std::conditional_t<EXACT || ONE, u32x2, u32x4> Kt;
    auto key_at = [&](const Buf& b, int t) -> Kt {
      if constexpr (DELTA && ONE) return b.ke[0][DELTA ? gr : 0][16 * t + m];
      else return b.kt01[gr][16 * t + m];
    };
    auto key_rest = [&](const Buf& b, int t) {
      if constexpr (ONE) return u32x4{};
      else return b.kt20[gr][16 * t + m];
    };
    auto first_parts = [](const Kt& x, const Parts& u, const f32x4 D) {
      if constexpr (EXACT || ONE) {
        typedef __attribute__((ext_vector_type(4))) short s16x4;
        if constexpr (SHORT)
          return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, x),
                                                           __builtin_bit_cast(s16x4, u32x2{u.p0[0], u.p0[1]}), D, 0, 0, 0);
        else
          return mma(u32x4{x[0], x[1], 0, 0}, u.p0, D);
      } else {
        return mma(x, u.p0, D);
      }
    };
    auto decay_rows = [&](const Buf& b, float end, int t) {
      if (CH) return *reinterpret_cast<const f32x4*>(&b.end[CH ? 16 * t + 4 * gr : 0]);
      return f32x4{end, end, end, end};
    };
    // A tile of S where U or the keys are not ordinary: as advance(), and what comes out not finite in fp32, with kt scaled
    // and not U.
    auto advance_odd = [&](const Buf& b, const f32x4 V, const Parts& u, float end, int t, const Kt x, const u32x4 y, f32x4 D,
                           f32x4 (&S)[NT]) {
      const f32x4 sc = CH || EXACT ? f32x4{1.f, 1.f, 1.f, 1.f} : scale(b, kRecKt);
      const f32x4 f = decay_rows(b, end, t);
      f32x4 other = S[t] * f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const unsigned p1 = EXACT ? y[2 + (i >> 1)] : x[(2 + (i >> 1)) % (sizeof(Kt) / 4)];
        const float k = ONE ? (i & 1 ? bf16_high(x[i >> 1]) : bf16_low(x[i >> 1])) : join(x[i >> 1], p1, y[i >> 1], i & 1);
        other = mma(k * sc[i], V[i], other);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) D[i] = __builtin_fmaf(S[t][i], f[i], D[i]);
      D = first_parts(x, u, D);
#pragma unroll
      for (int i = 0; i < 4; ++i) S[t][i] = finite(D[i]) ? D[i] : other[i];
    };
    // the smaller parts' products
    auto small_parts = [&](const Kt& x, const u32x4& y, const Parts& u) {
      if constexpr (ONE) return mma(u32x4{x[0], x[1], x[0], x[1]}, u.p02, zero);
      f32x4 D = mma(y, u.p02, zero);
      if constexpr (!EXACT && !ONE) {
        D = mma(x, u.p1, D);
        D = mma(x, u.p10, D);
      }
      return D;
    };
    // S = P_end S + kt U.  A product adds eight terms and the sum so far at a time, less exactly the wider their range; so
    // the first parts' come by themselves and last, on top of what the state's decay leaves, in the tokens' order: what
    // decays have made small is rounded while it is alone.  (Error of 16 tokens whose decay is 1 / 0.5 each, 1e-8, fp32
    // products / with parts 0 x 0 and 1 x 0 in one product / here: 8.5 / 5.1 / 3.8 and 2.9 / 4.2 / 3.3.)
    // `V`: not scaled; `is_odd`: U or the keys are not ordinary
    auto advance = [&](const Buf& b, const f32x4 V, float end, auto is_odd, f32x4 (&S)[NT]) {
      const Parts u = parts(V, CH || EXACT ? zero : scale(b, kRecKt));
      bool odd = false;
      // Two tiles at a time, whose products do not wait for each other, and the next two's operands on their way (left to
      // itself the compiler loads all of them first, and spills).
      Kt hm[2][2];
      u32x4 lh[2][2];
      auto ahead = [&](int t) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          hm[t >> 1 & 1][e] = key_at(b, t + e);
          lh[t >> 1 & 1][e] = key_rest(b, t + e);
        }
      };
      ahead(0);
#pragma unroll
      for (int t = 0; t < NT; t += 2) {
        const int p = t >> 1 & 1;
        f32x4 D[2];
        if (t + 2 < NT) ahead(t + 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 2; ++e) D[e] = small_parts(hm[p][e], lh[p][e], u);
        if (t == 0) odd = is_odd();   // (here the latency of a check is hidden)
        if (__builtin_expect(odd, 0)) {
#pragma unroll
          for (int e = 0; e < 2; ++e) advance_odd(b, V, u, end, t + e, hm[p][e], lh[p][e], D[e], S);
          continue;
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const f32x4 f = decay_rows(b, end, t + e);
#pragma unroll
          for (int i = 0; i < 4; ++i) S[t + e][i] = __builtin_fmaf(S[t + e][i], f[i], D[e][i]);
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) S[t + e] = first_parts(hm[p][e], u, S[t + e]);
      }
    };
    auto replace = [&](f32x4& x, f32x4& scale, const f32x4 with) {   // what is not finite
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        scale[i] = finite(x[i]) ? scale[i] : 1.f;
        x[i] = finite(x[i]) ? x[i] : with[i];
      }
    };
    auto read_out = [&](const f32x4 A, const f32x4 U) {   // A U
      std::conditional_t<F64, f64x4, f32x4> X = {0, 0, 0, 0}, Y = X;
      if constexpr (F64) {   // (A's rows are read in the order that puts the result's in the order of the others)
#pragma unroll
        for (int i = 0; i < 4; ++i) X = __builtin_amdgcn_mfma_f64_16x16x4f64(A[i], U[i], X, 0, 0, 0);
        return X;
      } else {
        X = mma(A[0], U[0], X);
        Y = mma(A[1], U[1], Y);
        X = mma(A[2], U[2], X);
        Y = mma(A[3], U[3], Y);
        return X + Y;
      }
    };
    // A V, the smaller parts of A first
    auto read_out_exact = [&](const Buf& b, const f32x4 V) {
      const Parts u = parts(V, zero);
      u32x4 x[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) x[e] = *reinterpret_cast<const u32x4*>(&b.amat[EXACT ? e : 0][m][gr][0]);
      return mma(x[0], u.p0, mma(x[1], u.p02, zero));
    };
    // AV: EXACT, and ordinary: the sum A U
    auto write = [&](const Buf& b, const f32x4 U, const f32x4 R, const f32x4 sq, const f32x4 V, int c, auto odd, const f32x4 AV, int col0) {
      const int col = col0 + m;
      float* oc = op + static_cast<int64_t>(c) * kScanChunk * o_stride;
      f32x4 x = U, bad;
      if constexpr (odd) bad = take_nonfinite(x, lane);
      auto X = [&] {
        if constexpr (EXACT && !odd) return AV;
        else return read_out(matrix(b, 0), x);
      }();
      if constexpr (EXACT && odd) {   // (what is finite has the bits of an ordinary chunk)
        const f32x4 Y = read_out_exact(b, x);
#pragma unroll
        for (int i = 0; i < 4; ++i) X[i] = finite(Y[i]) ? Y[i] : X[i];
      }
      if constexpr (odd)
#pragma unroll
        for (int i = 0; i < 4; ++i) X[i] += bad[i];
      f32x4 O;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        O[i] = MODE == kModeForget ? static_cast<float>(X[i] + R[i]) : __builtin_fmaf(R[i], sq[i], static_cast<float>(X[i]));
      if (MODE == kModeStateSpace) O += skip * V;
      const unsigned at = (4 * gr * o_stride + col) * sizeof(float);
      if (n - c * kScanChunk >= kScanChunk && col0 + 16 <= a.dv) {   // (uniform)
#pragma unroll
        for (int i = 0; i < 4; ++i) at_bytes<float>(oc + i * o_stride, at) = O[i];
      } else {
        const int rows = col < a.dv ? n - c * kScanChunk - 4 * gr : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (i < rows) at_bytes<float>(oc + i * o_stride, at) = O[i];
      }
    };
    auto order = [] { __builtin_amdgcn_sched_barrier(0); };
    // beside product i of six: a part of the next rows, and what it leaves
    auto part_beside = [&](SplitSteps& next, int i, u32x4 (&q)[3]) {
      if (i % 2 == 0) {
        next.step(5 * (i / 2), q, id);
        if (i < 4) {
          next.step(5 * (i / 2) + 1, q, id);
          next.step(5 * (i / 2) + 2, q, id);
        }
      }
    };
    // A wave without columns only keeps the barriers: the first, a chunk's, and the last of an odd number of them.  (With a
    // delta rule, whose waves have one tile, the exit spills two registers more of waves that have their columns: + 0.4 %.)
    if (!DELTA && col0 >= a.dv) {
      for (int c = 0; c <= nc + (nc & 1); ++c) lds_barrier();
      return;
    }
    // Chunks of ordinary numbers (delta rule: full ones of full columns) are walked in loops of their own.  A wave issues in
    // order, and left to itself the compiler puts every load, part and product right in front of what waits for it; here all
    // have been on their way for a few products.  A chunk that is not ordinary is left, untouched, to the loop behind (two ways
    // in one loop cost a move per number of the state and chunk), which takes a wave's two tiles one after the other, and
    // everybody waits for it at the barrier.  Columns past the last one go along, on copies of the last one's values, and tokens
    // past it, on zeros; neither is stored.  us, such waves and chunks in the loop behind / here: 32 heads, 16 x 512, 96 columns,
    // forget gate 267 / 233, state space 190 / 150; 96 heads of 40, one prompt of 1023 in 32 bits 97 / 86; state space, 32 heads,
    // 64 x 12 tokens 90 / 85, keys of 66 channels in 32 bits 100 / 96.
    const int ours = !DELTA ? nc : col0 + 16 <= a.dv ? n / kScanChunk : 0;
    int c = 0;
    lds_barrier();
    if constexpr (DELTA) {
      SplitSteps next;
      auto take = [&](int s) {
#pragma unroll
        for (int e = 0; e < 2; ++e) next.r[e] = S[0][(2 * s + e) % NT];
      };
      if constexpr (NT == 8) {
        u32x4 p[3][3];   // of S's rows 0 - 31 and 96 - 127, 32 - 63, 64 - 95
        state_parts(p[0], 0, S[0]);
        for (; c < ours; ++c) {
          const Buf& b = lds.buf[c % BUFS];
          const auto& key_rows = *reinterpret_cast<const typename Buf::Rows*>(&b.ke);
          Sum Ws = {zero, {zero, zero}}, Rs = Ws;
          u32x4 ra[3], rb[3], rc[3];
          auto load = [&](u32x4 (&r)[3], const typename Buf::Rows& rows, int s, int e) { r[e] = row(rows[e], s); };
          // six products of rows r and the parts q; beside them what `more` does in step i
          auto products = [&](Sum& x, const u32x4 (&r)[3], const u32x4 (&q)[3], auto more) {
#pragma unroll
            for (int i = 0; i < 6; ++i) {
              product(x, r, q, i);
              order();
              more(i);
              order();
            }
          };
#pragma unroll
          for (int e = 0; e < RP; ++e) load(ra, key_rows, 0, e);
#pragma unroll
          for (int e = 0; e < RP; ++e) load(rc, b.qe, 0, e);
#pragma unroll
          for (int e = 0; e < RP; ++e) load(rb, key_rows, 1, e);
          order();
          take(1);   // (while the rows come)
#pragma unroll
          for (int i = 0; i < 11; ++i) {
            next.step(i, p[1], id);
            order();
          }
          take(2);
          products(Ws, ra, p[0], [&](int i) { part_beside(next, i, p[2]); });
          products(Rs, rc, p[0], [&](int i) { if (i < RP) load(ra, key_rows, 2, i); });
          take(3);
          products(Ws, rb, p[1], [&](int i) {
            if (i < RP) load(rc, b.qe, 1, i);
            part_beside(next, i, p[0]);
          });
          products(Ws, ra, p[2], [&](int i) { if (i < RP) load(rb, key_rows, 3, i); });
          f32x4 M, v, sk, skt;
          products(Ws, rb, p[0], [&](int i) {
            if (i == 0) M = matrix(b, DELTA ? 256 : 0);
            if (i == 1) v = b.v[gr][16 * w + m];
            if (i == 2) sk = scale(b, kRecK);
            if (i == 2) skt = CH ? zero : scale(b, kRecKt);
            if (i >= 3 && i - 3 < RP) load(ra, b.qe, 2, i - 3);
          });
          // From here on W's sum, U and its parts one after the other, and between them the sum for the outputs.
          f32x4 X, U, U2, rest;
          float sum = 0.f;
          unsigned u[3][2];
          products(Rs, rc, p[1], [&](int i) {
            if (i < RP) load(rb, b.qe, 3, i);
            if (i == 1) X = Ws.big + (Ws.small[0] + Ws.small[1]);
            if (i == 2) X = v - sk * X;
            if (i == 3) U = mma(M[0], X[0], zero);
            if (i == 3) U2 = mma(M[1], X[1], zero);
            if (i == 5) U = mma(M[2], X[2], U);
            if (i == 5) U2 = mma(M[3], X[3], U2);
          });
          products(Rs, ra, p[2], [&](int i) {
            if (i == 0) sum = abs_sum(X) + (abs_sum(M) + (CH ? 0.f : b.scale[head][kRecNoParts - kRecQ]));
            if (i == 2) {
              U += U2;
              if constexpr (CH) {
                u[0][0] = pack_bf16(U[0], U[1]);
                u[0][1] = pack_bf16(U[2], U[3]);
                rest = id.rest(U, u[0][0], u[0][1]);
              } else {
                rest = split_product(U, skt, u[0]);
              }
            }
            if (i == 5) {
              u[1][0] = pack_bf16(rest[0], rest[1]);
              u[1][1] = pack_bf16(rest[2], rest[3]);
              rest = id.rest(rest, u[1][0], u[1][1]);
            }
          });
          Kt hm[2][2];
          u32x4 lh[2][2];
          f32x4 f[2][2];
          auto keys = [&](int t) {
            const int q = t / 2 % 2;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              lh[q][e] = key_rest(b, t + e);
              hm[q][e] = key_at(b, t + e);
              if (CH) f[q][e] = decay_rows(b, 0.f, t + e);
            }
          };
          f32x4 A, sq;
          products(Rs, rb, p[0], [&](int i) {
            if (i == 0) keys(0);
            if (i == 2) keys(2);
            if (i == 3) {
              u[2][0] = pack_bf16(rest[0], rest[1]);
              u[2][1] = pack_bf16(rest[2], rest[3]);
            }
            if (i == 4) A = matrix(b, 0);
            if (i == 5) sq = scale(b, kRecQ);
          });
          const Parts parts_u = as_parts(u);
          const float end = decay_of(b);
          f32x4 D[2][2];
          auto small = [&](int t) {   // small_parts(), the two tiles in turn
            const int q = t / 2 % 2, r = q;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              if constexpr (ONE) D[r][e] = small_parts(hm[q][e], lh[q][e], parts_u);
              else D[r][e] = mma(lh[q][e], parts_u.p02, zero);
              order();
            }
            if constexpr (!EXACT && !ONE) {
#pragma unroll
              for (int e = 0; e < 2; ++e) {
                D[r][e] = mma(hm[q][e], parts_u.p1, D[r][e]);
                order();
              }
#pragma unroll
              for (int e = 0; e < 2; ++e) {
                D[r][e] = mma(hm[q][e], parts_u.p10, D[r][e]);
                order();
              }
            }
          };
          small(0);
          const f32x4 R = total(Rs);
          sum += abs_sum(R);
          // (sums of 16 of these products and of 128 rows, scaled, are far from the ends of the range)
          if (__builtin_expect(__any(!(sum <= 0x1p50f)), 0)) break;
          f32x4 Y[2];
#pragma unroll
          for (int t = 0; t < NT; t += 2) {
            const int q = t / 2 % 2, r = q;
            order();
            if (t + 2 < NT) small(t + 2);
            order();
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
              for (int i = 0; i < 4; ++i) S[0][t + e][i] = __builtin_fmaf(S[0][t + e][i], CH ? f[q][e][i] : end, D[r][e][i]);
            order();
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              S[0][t + e] = first_parts(hm[q][e], parts_u, S[0][t + e]);
              order();
            }
            if (t + 4 < NT) keys(t + 4);
            if (t < 4) {   // A U
#pragma unroll
              for (int e = 0; e < 2; ++e) {
                Y[e] = mma(A[t + e], U[t + e], t == 0 ? zero : Y[e]);
                order();
              }
            }
            if (t == 2) {
              take(0);
              next.step(0, p[0], id);
              next.step(1, p[0], id);
              order();
              next.step(2, p[0], id);
            }
            if (t == 4) {
              next.step(5, p[0], id);
              next.step(6, p[0], id);
              order();
              next.step(7, p[0], id);
              Y[0] += Y[1];
              float* oc = op + static_cast<int64_t>(c) * kScanChunk * o_stride;
              const unsigned at = (4 * gr * o_stride + col0 + m) * sizeof(float);
#pragma unroll
              for (int i = 0; i < 4; ++i) at_bytes<float>(oc + i * o_stride, at) = __builtin_fmaf(R[i], sq[i], Y[0][i]);
            }
          }
          order();
          next.step(10, p[0], id);
          lds_barrier();
        }
      }
      u32x4 p[2][3];
      state_parts(p[0], 0, S[0]);
      for (; c < nc; ++c) {
        const Buf& b = lds.buf[c % BUFS];
        Sum Ws = {zero, {zero, zero}}, Rs = Ws;
        u32x4 rows[2][2][3];   // of ke and qe
        const auto& key_rows = *reinterpret_cast<const typename Buf::Rows*>(&b.ke);
        auto ahead = [&](int s, int i) {
          if (i % 3 < RP) rows[s & 1][i / 3][i % 3] = row(i < 3 ? key_rows[i % 3 % RP] : b.qe[i % 3 % RP], s);
        };
#pragma unroll
        for (int i = 0; i < 6; ++i) ahead(0, i);
        // A wave issues in order: the next rows' parts go between the products, in whose shadow they run, in an order that
        // the compiler would not keep.
#pragma unroll
        for (int s = 0; s < NT / 2; ++s) {
          const bool more = s + 1 < NT / 2;
          SplitSteps next;
          if (more)
#pragma unroll
            for (int e = 0; e < 2; ++e) next.r[e] = S[0][(2 * s + 2 + e) % NT];
#pragma unroll
          for (int i = 0; i < 12; ++i) {   // products of ke and qe in turn
            product(i & 1 ? Rs : Ws, rows[s & 1][i & 1], p[s & 1], i >> 1);
            if (more && i < 6) ahead(s + 1, i);
            if (more && i < 11) next.step(i, p[s + 1 & 1], id);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        const f32x4 M = matrix(b, DELTA ? 256 : 0);
        f32x4 R = total(Rs), sq = scale(b, kRecQ);
        const f32x4 v = b.v[gr][16 * w + m];
        f32x4 X = v - scale(b, kRecK) * total(Ws), bad = zero;
        auto finish = [&](auto odd) {
          f32x4 U2 = bad, U = zero;
          U = mma(M[0], X[0], U);
          U2 = mma(M[1], X[1], U2);
          U = mma(M[2], X[2], U);
          U2 = mma(M[3], X[3], U2);
          U += U2;
          advance(b, U, decay_of(b), [] { return decltype(odd)::value; }, S[0]);
          write(b, U, R, sq, zero, c, odd, zero, col0);
          state_parts(p[0], 0, S[0]);
        };
        // (sums of 16 of these products and of 128 rows, scaled, are far from the ends of the range)
        const float keys = CH ? 0.f : b.scale[head][kRecNoParts - kRecQ];
        if (__builtin_expect(!__any(!(abs_sum(X) + abs_sum(R) + (abs_sum(M) + keys) <= 0x1p50f)), 1)) {
          finish(std::false_type{});
        } else {
          f32x4 one = {1.f, 1.f, 1.f, 1.f};
          replace(R, sq, sum_fp32(b, b.qe, kRecQ, S[0]));
          replace(X, one, v - sum_fp32(b, key_rows, kRecK, S[0]));
          bad = take_nonfinite(X, lane);
          finish(std::true_type{});
        }
        lds_barrier();
      }
      if (nc & 1) lds_barrier();
      store_state(st);
    } else {
      // The chunk's decay where it is one number, and over the chunks so far.
      auto end_of = [&](const Buf& b, int c) {
        float end = decay_of(b);
        if (MODE == kModeRetention) {
          const float e = fixed.next();
          end = n - c * kScanChunk >= kScanChunk ? e : end;
        }
        if (PASS == 1 && !CH) over *= end;
        return end;
      };
      auto worst = [&](const Buf& b) { return CH ? 0.f : b.scale[head][kRecNoParts - kRecQ]; };
      for (; c < ours; ++c) {
        const Buf& b = lds.buf[c % BUFS];
        f32x4 U[CT], f[2][2];
        Kt hm[2][2];
        u32x4 lh[2][2];
        Parts u[CT];
        auto keys = [&](int t) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            lh[t >> 1 & 1][e] = key_rest(b, t + e);
            hm[t >> 1 & 1][e] = key_at(b, t + e);
            if (CH) f[t >> 1 & 1][e] = decay_rows(b, 0.f, t + e);
          }
        };
        float sum = worst(b);
        if constexpr (PASS != 1) {
          u32x4 rows[2][3], p[2][CT][3], A[2];
          Sum Rs[CT];
          f32x4 AV[CT];
          auto ahead = [&](int s, int e) { rows[s & 1][e] = row(b.qe[e], s); };
#pragma unroll
          for (int e = 0; e < RP; ++e) ahead(0, e);
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            U[ct] = b.v[gr][16 * (CT * w + ct) + m];
            Rs[ct] = {zero, {zero, zero}};
          }
          const f32x4 sq = scale(b, kRecQ), sk = CH || EXACT ? zero : scale(b, kRecKt);
          f32x4 M = zero;
          if constexpr (EXACT) {
#pragma unroll
            for (int e = 0; e < 2; ++e) A[e] = *reinterpret_cast<const u32x4*>(&b.amat[EXACT ? e : 0][m][gr][0]);
          } else {
            M = matrix(b, 0);
          }
          order();
          SplitSteps next[CT];
          auto take = [&](int s) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
              for (int e = 0; e < 2; ++e) next[ct].r[e] = S[ct][2 * s + e];
          };
          take(0);
#pragma unroll
          for (int i = 0; i < 11; ++i) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) next[ct].step(i, p[0][ct], id);
            order();
          }
#pragma unroll
          for (int s = 0; s < NT / 2; ++s) {
            const bool more = s + 1 < NT / 2;
            if (more) take(s + 1);
#pragma unroll
            for (int i = 0; i < 6; ++i) {
#pragma unroll
              for (int ct = 0; ct < CT; ++ct) {
                product(Rs[ct], rows[s & 1], p[s & 1][ct], i);
                if (more) {
                  if (ct == 0 && i < RP) ahead(s + 1, i);
                  part_beside(next[ct], i, p[s + 1 & 1][ct]);
                } else if (i == 0) {
                  u[ct] = parts(U[ct], sk);
                  sum += abs_sum(CH || EXACT ? U[ct] : U[ct] * sk);
                  if (ct == 0) keys(0);
                } else if (EXACT && i == 2) {
                  AV[ct] = mma(A[1], u[ct].p02, zero);
                } else if (EXACT && i == 4) {
                  AV[ct] = mma(A[0], u[ct].p0, AV[ct]);
                }
                order();
              }
            }
          }
          f32x4 R[CT];
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            if constexpr (!EXACT && !F64) AV[ct] = read_out(M, U[ct]);
            R[ct] = total(Rs[ct]);
            sum += abs_sum(R[ct]);
            if (EXACT) sum += abs_sum(AV[ct]);
          }
          if (__builtin_expect(__any(!(sum <= 0.5f * kSplitMax)), 0)) break;
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            f32x4 O;
            if constexpr (F64) {
              const auto X = read_out(M, U[ct]);
#pragma unroll
              for (int i = 0; i < 4; ++i) O[i] = static_cast<float>(X[i] + R[ct][i]);
            } else {
#pragma unroll
              for (int i = 0; i < 4; ++i)
                O[i] = MODE == kModeForget ? AV[ct][i] + R[ct][i] : __builtin_fmaf(R[ct][i], sq[i], AV[ct][i]);
            }
            if (MODE == kModeStateSpace) O += skip * U[ct];
            float* oc = op + static_cast<int64_t>(c) * kScanChunk * o_stride;
            const unsigned at = (4 * gr * o_stride + col0 + 16 * ct + m) * sizeof(float);
            if (n - c * kScanChunk >= kScanChunk) {   // (uniform)
              if (col0 + 16 * ct + m < a.dv)
#pragma unroll
                for (int i = 0; i < 4; ++i) at_bytes<float>(oc + i * o_stride, at) = O[i];
            } else {
              const int rows = col0 + 16 * ct + m < a.dv ? n - c * kScanChunk - 4 * gr : 0;
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (i < rows) at_bytes<float>(oc + i * o_stride, at) = O[i];
            }
          }
        } else {
          keys(0);
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            U[ct] = b.v[gr][16 * (CT * w + ct) + m];
            const f32x4 sk = CH || EXACT ? zero : scale(b, kRecKt);
            sum += abs_sum(CH || EXACT ? U[ct] : U[ct] * sk);
            u[ct] = parts(U[ct], sk);
          }
          if (__builtin_expect(__any(!(sum <= 0.5f * kSplitMax)), 0)) break;
        }
        const float end = end_of(b, c);
        f32x4 D[2][2][CT];
        auto small = [&](int t) {
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) D[t >> 1 & 1][e][ct] = small_parts(hm[t >> 1 & 1][e], lh[t >> 1 & 1][e], u[ct]);
        };
        small(0);
#pragma unroll
        for (int t = 0; t < NT; t += 2) {
          const int q = t >> 1 & 1;
          if (t + 2 < NT) keys(t + 2);
          order();
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                S[ct][t + e][i] = __builtin_fmaf(S[ct][t + e][i], CH ? f[q][e][i] : end, D[q][e][ct][i]);
          order();
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) S[ct][t + e] = first_parts(hm[q][e], u[ct], S[ct][t + e]);
          if (t + 2 < NT) small(t + 2);
          order();
        }
        lds_barrier();
      }
      for (; c < nc; ++c) {
        const Buf& b = lds.buf[c % BUFS];
        const float end = end_of(b, c);
        auto chunk = [&](f32x4 (&S)[NT], int ct) __attribute__((always_inline)) {
          const f32x4 U = b.v[gr][16 * (CT * w + ct) + m], Us = CH || EXACT ? U : U * scale(b, kRecKt);
          f32x4 R = zero, AV = zero;
          if (PASS != 1) {
            if constexpr (EXACT) AV = read_out_exact(b, U);
            Sum Rs = {zero, {zero, zero}};
#pragma unroll
            for (int s = 0; s < NT / 2; ++s) {
              u32x4 p[3];
              state_parts(p, s, S);
              add(Rs, b.qe, p, s);
            }
            R = total(Rs);
          }
          if constexpr (PASS == 1) {
            advance(b, U, end, [&] { return !ordinary(b, Us, zero); }, S);
          } else if (__builtin_expect(ordinary(b, Us, EXACT ? abs(R) + abs(AV) : R), 1)) {
            write(b, U, R, scale(b, kRecQ), U, c, std::false_type{}, AV, col0 + 16 * ct);
            advance(b, U, end, [] { return false; }, S);
          } else {
            f32x4 sq = scale(b, kRecQ);
            replace(R, sq, sum_fp32(b, b.qe, kRecQ, S));
            write(b, U, R, sq, U, c, std::true_type{}, AV, col0 + 16 * ct);
            advance(b, U, end, [] { return true; }, S);
          }
        };
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) chunk(S[ct], ct);
        lds_barrier();
      }
      if (nc & 1) lds_barrier();
      if (PASS == 1) {
        store_state(seg_state(sg.j, h));
        if (!CH && lane == 0 && col0 == 0) {
          if (MODE == kModeRetention) {   // (all its chunks are full)
            double p = 1., f = static_cast<double>(fixed.e) + fixed.rest;
            for (int i = nc; i > 0; i >>= 1, f *= f)
              if (i & 1) p *= f;
            over = static_cast<float>(p);
          }
          seg_decay(sg.j, h)[0] = over;
        }
      } else if (sg.j == sg.P - 1) {
        store_state(st);
      }
    }
    return;
  }

  // ---- operands: lane (token group tg, c) with CPW adjacent channels of four tokens
  constexpr int CPW = DK / 16 / OW, VC = Buf::COLS / (16 * OW) > 0 ? Buf::COLS / (16 * OW) : 1;
  const int tg = lane >> 4, c0 = CPW * (16 * (w - waves) + (lane & 15));
  const int g = MODE == kModeForget ? h0 : h0 / (a.H / a.G);
  constexpr bool KEPT = scan_keeps_decays(MODE);
  float b0[CPW], b1[CPW], over[CPW];   // over: the decay over the chunks so far (lanes of the last token group)
  if constexpr (CH && !KEPT) decay_params<MODE, CPW>(a, h0, c0, b0, b1);
#pragma unroll
  for (int j = 0; j < CPW; ++j) over[j] = 1.f;
  constexpr int HEADS = Buf::HEADS;
  struct In {
    Raw<T, MODE, CPW> r;
    T v[4][VC];            // VC columns of the four tokens
    float mat[HEADS][DELTA ? 2 : 1], scale[HEADS];
    f32x4 kt;              // the scale of k into the state, where it is not in U
    float d[KEPT ? 4 : 1][CPW];   // decays
  };
  // Retention's rows come with their partners and tables: two chunks of them ahead are 172 bytes of spilled registers per
  // lane in 32 bits (us with two / one, 32 heads of 128: 16 x 512 463 / 279, 1023 109 / 77, 300 61 / 45; bf16, where few
  // are spilled, 245 / 242, 69.5 / 69.5, 42 / 41; 32 heads of 64, bf16, where two workgroups fit on a CU with one, 121 / 113,
  // values at odd addresses 194 / 125).
  constexpr int AHEAD = MODE == kModeRetention ? 1 : 2;
  In raw[AHEAD];
  // A lane's offsets into the chunk's rows; only the last chunk's differ.  Channels that are not there: the last ones.
  constexpr bool KEYS = MODE != kModeForget, DEC = MODE == kModeDeltaChannel, SCALED = DEC || (EXACT && !CH), TURN = MODE == kModeRetention;
  unsigned oq[4], ok[4], od[DEC ? 4 : 1], ot[TURN ? 4 : 1], ov[4];
  const int ow = w - waves, vc = VC * ((16 * ow + (lane & 15)) % (Buf::COLS / VC));   // (of fewer columns some twice)
  const int vhead = two ? vc >> 6 : 0, vcol = DELTA || two ? cb * kWalkCols + (vc & 63) : 16 * tiles * cb + vc;
  const int at_mat = 256 / OW * ow + lane % (256 / OW), at_scale = 64 / OW * ow + lane % (64 / OW);
  const unsigned mat_off = at_mat * sizeof(float), scale_off = (kRecQ + at_scale) * sizeof(float);
  const int cl = min(c0, a.dk - CPW), nf = TURN ? a.n_freq : 0;
  const int fq = c0 < nf ? c0 : c0 < 2 * nf ? c0 - nf : 0, partner = (c0 < nf ? c0 + nf : fq) - cl;
  auto offsets = [&](int nt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = min(4 * tg + i, nt - 1);
      oq[i] = (t * static_cast<int>(a.q_stride) + cl) * sizeof(T);
      ok[i] = (t * static_cast<int>(a.k_stride) + cl) * sizeof(T);
      if (DEC) od[DEC ? i : 0] = (t * static_cast<int>(a.dec_stride) + cl) * sizeof(T);
      if (TURN) ot[TURN ? i : 0] = (t * 2 * nf + fq) * sizeof(float);
      ov[i] = (t * static_cast<int>(a.v_stride) + vhead * a.dv + min(vcol, a.dv - (VEC == 2 ? VC : 1))) * sizeof(T);
    }
  };
  // (loads of chunks past the last one are repeats of it: conditional ones would be waited for where the paths join)
  auto load = [&](In& in, int c) {
    Raw<T, MODE, CPW>& r = in.r;
    c = min(c, nc - 1);
    const int nt = min(kScanChunk, n - c * kScanChunk);
    const int64_t row0 = first + c * kScanChunk;
    if (nt < kScanChunk) offsets(nt);
    const T* vb = static_cast<const T*>(a.v) + row0 * a.v_stride + static_cast<int64_t>(h0) * a.dv;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (VEC == 2) {
        struct __attribute__((aligned(VC * sizeof(T)))) Some { T x[VC]; };
        const Some v = at_bytes<Some>(vb, ov[i]);
#pragma unroll
        for (int j = 0; j < VC; ++j) in.v[i][j] = v.x[j];
      } else {
#pragma unroll
        for (int j = 0; j < VC; ++j) in.v[i][j] = at_bytes<T>(vb, ov[i] + (vcol + j < a.dv ? j * sizeof(T) : 0));
      }
    }
    const float* rec = rec0 + c * rec_step;
    if (SCALED) in.kt = at_bytes<f32x4>(rec + kRecKt, 4 * tg * sizeof(float));
    if constexpr (KEPT) {
      struct __attribute__((aligned(CPW * sizeof(float)))) Some { float x[CPW]; };
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const Some v = at_bytes<Some>(rec + kDecay + i * DS, (4 * tg * DS + (VEC ? c0 : min(c0, DS - CPW))) * sizeof(float));
#pragma unroll
        for (int j = 0; j < CPW; ++j) in.d[KEPT ? i : 0][j] = VEC || c0 < DS ? v.x[j] : 1.f;
      }
    }
#pragma unroll
    for (int e = 0; e < HEADS; ++e) {
      const float* p = two ? rec + e * REC : rec;
      if (PASS != 1) in.mat[e][0] = at_bytes<float>(p, mat_off);
      if (DELTA) in.mat[e][DELTA ? 1 : 0] = at_bytes<float>(p + kRecT, mat_off);
      if (MODE != kModeForget) in.scale[e] = at_bytes<float>(p, scale_off);
    }
    if constexpr (!VEC) {
      load_raw<false, T, MODE, CPW>(r, a, h0, g, row0, nt, lane, c0);
    } else {
      const T* qb = static_cast<const T*>(a.q) + row0 * a.q_stride + static_cast<int64_t>(g) * a.dk;
      const T* kb = static_cast<const T*>(a.k) + row0 * a.k_stride + static_cast<int64_t>(g) * a.dk;
      const T* db = DEC ? static_cast<const T*>(a.dec) + row0 * a.dec_stride + static_cast<int64_t>(h0) * a.dk : nullptr;
      const float* tab = TURN ? a.cos_sin + row0 * 2 * nf : nullptr;
      struct __attribute__((aligned(CPW * sizeof(T)))) Some { T x[CPW]; };
      struct __attribute__((aligned(CPW * sizeof(float)))) Turn { float x[CPW]; };
      auto get = [](T (&o)[CPW], const T* base, unsigned off) {
        const Some v = at_bytes<Some>(base, off);
#pragma unroll
        for (int j = 0; j < CPW; ++j) o[j] = v.x[j];
      };
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (PASS != 1) get(r.q[i], qb, oq[i]);
        if (KEYS) get(r.k[i], kb, ok[i]);
        else if (!KEPT) get(r.d[per_channel<MODE>() ? i : 0], kb, ok[i]);
        if (DEC && !KEPT) get(r.d[per_channel<MODE>() ? i : 0], db, od[DEC ? i : 0]);
        if (TURN && nf > 0) {   // (uniform)
          constexpr int P = TURN ? 4 : 1;
          const Turn cs = at_bytes<Turn>(tab, ot[i % P]), sn = at_bytes<Turn>(tab + nf, ot[i % P]);
#pragma unroll
          for (int j = 0; j < CPW; ++j) {
            r.cs[i % P][j] = cs.x[j];
            r.sn[i % P][j] = sn.x[j];
          }
          if (PASS != 1) get(r.pq[i % P], qb, oq[i] + partner * static_cast<int>(sizeof(T)));
          get(r.pk[i % P], kb, ok[i] + partner * static_cast<int>(sizeof(T)));
        }
      }
    }
  };
  auto prepare = [&](In& in, int c) {
    const Raw<T, MODE, CPW>& r = in.r;
    Buf& b = lds.buf[c % BUFS];
    const int t0 = c * kScanChunk, nt = min(kScanChunk, n - t0);
    float q[4][CPW], k[4][CPW], d[4][CPW];
    if constexpr (KEPT)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < CPW; ++j) d[i][j] = in.d[KEPT ? i : 0][j];
    if (VEC && nt == kScanChunk && a.dk == DK) {
      if constexpr (CH && !KEPT) decays<true, T, MODE, CPW>(r, a, nt, lane, c0, b0, b1, d);
      queries_keys<true, (VEC > 0), T, MODE, CPW>(r, a, g, first + t0, nt, lane, c0, d, q, k);
    } else {
      if constexpr (CH && !KEPT) decays<false, T, MODE, CPW>(r, a, nt, lane, c0, b0, b1, d);
      queries_keys<false, (VEC > 0), T, MODE, CPW>(r, a, g, first + t0, nt, lane, c0, d, q, k);
    }
#pragma unroll
    for (int j = 0; j < VC; ++j) {
      f32x4 x;
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = 4 * tg + i < nt ? static_cast<float>(in.v[i][j]) : 0.f;
      b.v[tg][vc + j] = x;
    }
#pragma unroll
    for (int e = 0; e < HEADS; ++e) {
      if (PASS != 1)
        b.mat[e][at_mat] = in.mat[e][0];
      if (DELTA) b.mat[e][(DELTA ? 256 : 0) + at_mat] = in.mat[e][DELTA ? 1 : 0];
      if (MODE != kModeForget) b.scale[e][at_scale] = in.scale[e];
    }
    if constexpr (EXACT && PASS != 1) {
      unsigned p[3];
      split(in.mat[0][0], 0.f, p[0], p[1], p[2]);
      auto part = [&](int e, int half) -> unsigned short& {
        return *reinterpret_cast<unsigned short*>(&b.amat[EXACT ? e : 0][at_mat >> 4][at_mat >> 2 & 3][4 * half + (at_mat & 3)]);
      };
      part(0, 0) = static_cast<unsigned short>(p[0]);
      part(0, 1) = 0;
      part(1, 0) = static_cast<unsigned short>(p[2]);
      part(1, 1) = static_cast<unsigned short>(p[1]);
    }
    const f32x4 kts = in.kt;
    load(in, c + AHEAD);
    // numbers that have no parts, or may get beyond (decays are at most 1, the keys' scales make them so)
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < CPW; ++j) {
        if (PASS != 1) sum += fabsf(q[i][j]);
        sum += fabsf(k[i][j]);
        if (CH && MODE != kModeForget) sum += d[i][j];   // (the forget gate's key holds it)
      }
    // (Keys of up to 64 channels: a lane has one, and would wait for the products.  On the vector units, a layer's call, us, 32
    // heads of 64, bf16, products / here: retention 16 x 512 124 / 121, 64 x 12 69 / 65, 16 x 100 49 / 46.)
    constexpr bool VECTOR = DK == 64 && !ONE;
    const bool odd = VECTOR || (!ONE && __any(!(sum <= 0.5f * kSplitMax)));
    float f[CPW], behind[CPW];   // products of the decays of the lane groups before / behind this one
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
      f[j] = behind[j] = 1.f;
      if (CH) {
        const float own = (d[0][j] * d[1][j]) * (d[2][j] * d[3][j]);
        const Pair near = swap_rows<16>(own), far = swap_rows<32>(near.lower * near.upper);
        f[j] = (tg & 1 ? near.lower : 1.f) * (tg & 2 ? far.lower : 1.f);
        behind[j] = (tg & 1 ? 1.f : near.upper) * (tg & 2 ? 1.f : far.upper);
      }
    }
    // per channel of the lane: P_i q_i, P_i k_i and D_end,j k_j of its four tokens
    constexpr int KE = PASS != 1 ? CPW : 0, KT = KE + (DELTA ? CPW : 0), N = KT + CPW;
    f32x4 x[N];   // (with a product, first the one factor, then what part 0 leaves)
    unsigned p[N][3][2];
    auto factor = [&](int j) {   // of the rows
      f32x4 y;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f[j] *= d[i][j];
        y[i] = f[j];
      }
      return y;
    };
    auto tokens = [](const float (&z)[4][CPW], int j) { return f32x4{z[0][j], z[1][j], z[2][j], z[3][j]}; };
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
      if constexpr (CH) {
        const f32x4 by = factor(j);
        if (PASS != 1) x[j % N] = split_product(tokens(q, j), by, p[j % N][0]);
        if (DELTA) x[(KE + j) % N] = split_product(tokens(k, j), by, p[(KE + j) % N][0]);
        if (tg == 3) b.end[CH ? c0 + j : 0] = f[j];   // the whole chunk
      } else {
        if (PASS != 1) x[j % N] = tokens(q, j);
        if (DELTA) x[(KE + j) % N] = tokens(k, j);
      }
      if (PASS == 1) over[j] *= c < nc ? f[j] : 1.f;   // (a chunk for nobody has the last one's)
      if constexpr (CH || SCALED) {
        f32x4 by = kts;
        float e = behind[j];
        if (CH)
#pragma unroll
          for (int i = 3; i >= 0; --i) {
            by[i] = DELTA ? e * kts[i] : e;
            e *= d[i][j];
          }
        x[KT + j] = split_product(tokens(k, j), by, p[KT + j][0]);
      } else {
        x[KT + j] = tokens(k, j);
      }
    }
    const auto from = [](int g) { return CH || (SCALED && g >= KT) ? 1 : 0; };   // the first part that is not there
    if (__builtin_expect(odd, 0)) {
#pragma unroll
      for (int g = 0; g < N; ++g)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          float lo = x[g][2 * e], hi = x[g][2 * e + 1];
#pragma unroll
          for (int i = from(g); i < 3; ++i) {
            p[g][i][e] = pack_bf16(lo, hi);
            lo -= bf16_low(p[g][i][e]);
            hi -= bf16_high(p[g][i][e]);
          }
        }
    } else {   // all side by side: a product's result is there after the others' instructions
#pragma unroll
      for (int i = 0; i < 3; ++i) {
#pragma unroll
        for (int g = 0; g < N; ++g)
          if (i >= from(g) && i < RP) {
            p[g][i][0] = pack_bf16(x[g][0], x[g][1]);
            p[g][i][1] = pack_bf16(x[g][2], x[g][3]);
            if (i + 1 < RP) x[g] = id.rest(x[g], p[g][i][0], p[g][i][1]);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    auto put = [&](u32x2 (&rows)[RP][4][Buf::ROW], int g) {
#pragma unroll
      for (int e = 0; e < RP; ++e) {
        if constexpr (CPW == 2)
          *reinterpret_cast<u32x4*>(&rows[e][tg][c0]) = u32x4{p[g][e][0], p[g][e][1], p[(g + 1) % N][e][0], p[(g + 1) % N][e][1]};
        else
          rows[e][tg][c0] = u32x2{p[g][e][0], p[g][e][1]};
      }
    };
    if constexpr (PASS != 1) put(b.qe, 0);
    if constexpr (DELTA) put(b.ke, KE % N);
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
      const unsigned (&y)[3][2] = p[KT + j];
      if constexpr (ONE) {
        if constexpr (!DELTA) b.kt01[tg][c0 + j] = u32x2{y[0][0], y[0][1]};
      } else if constexpr (EXACT) {
        b.kt01[tg][c0 + j] = u32x2{y[0][0], y[0][1]};
        b.kt20[tg][c0 + j] = u32x4{y[2][0], y[2][1], y[1][0], y[1][1]};
      } else {
        b.kt01[tg][c0 + j] = u32x4{y[0][0], y[0][1], y[1][0], y[1][1]};
        b.kt20[tg][c0 + j] = u32x4{y[2][0], y[2][1], y[0][0], y[0][1]};
      }
    }
    lds_barrier();
  };
  offsets(min(kScanChunk, n));
  load(raw[0], 0);
  __builtin_amdgcn_sched_barrier(0);   // (in this order, as in the loop: the waits count the loads behind)
  if constexpr (AHEAD == 2) load(raw[AHEAD - 1], 1);
  if (PASS == 2 && sg.j > 0) lds_barrier();
  // in the step before the products'; a chunk behind an odd number of them is prepared for nobody, for the same reason
  for (int c = 0; c < nc; c += 2) {
    prepare(raw[0], c);
    prepare(raw[AHEAD - 1], c + 1);
  }
  lds_barrier();
  if (PASS == 1 && CH && tg == 3 && cb == 0)
#pragma unroll
    for (int j = 0; j < CPW; ++j) seg_decay(sg.j, h0)[c0 + j] = over[j];
}

template <typename T, int MODE, int DK, int VEC, int CT>
__global__ void __launch_bounds__((walk_threads<MODE, DK>()), (walk_simd_waves<MODE, DK, CT>()))
scan_walk_kernel(ChunkArgs a, int portion0) {
  __shared__ __attribute__((aligned(16))) WalkLds<MODE, DK, exact_values<T, MODE>(), exact_rows<T, MODE>()> lds;
  const Segment sg{find_portion(a, portion0 + static_cast<int>(blockIdx.y)), 0, 1, 0, 0};
  if (sg.s >= 0) walk<T, MODE, DK, VEC, 0, CT>(a, sg, lds);
}

// segment0 + blockIdx.y = segment of the batch.  First kernel: pass 1, and the portions that are not cut.
template <typename T, int MODE, int DK, int VEC, int CT>
__global__ void __launch_bounds__((walk_threads<MODE, DK>()), (walk_simd_waves<MODE, DK, CT>()))
scan_segments_kernel(ChunkArgs a, int segment0) {
  __shared__ __attribute__((aligned(16))) WalkLds<MODE, DK, exact_values<T, MODE>(), exact_rows<T, MODE>()> lds;
  const Segment sg = find_segment<false>(a, segment0 + blockIdx.y);
  if (sg.s < 0) return;
  if (sg.P == 1)
    walk<T, MODE, DK, VEC, 0, CT>(a, sg, lds);
  else if (sg.j < sg.P - 1 && sg.state + sg.P <= a.seg_states)   // (the bound holds: scan_segments)
    walk<T, MODE, DK, VEC, 1, CT>(a, sg, lds);
}
template <typename T, int MODE, int DK, int VEC, int CT>
__global__ void __launch_bounds__((walk_threads<MODE, DK>()), (walk_simd_waves<MODE, DK, CT>()))
scan_segments_end_kernel(ChunkArgs a, int segment0) {
  __shared__ __attribute__((aligned(16))) WalkLds<MODE, DK, exact_values<T, MODE>(), exact_rows<T, MODE>()> lds;
  const Segment sg = find_segment<true>(a, segment0 + blockIdx.y);
  if (sg.s >= 0 && sg.state + sg.P <= a.seg_states) walk<T, MODE, DK, VEC, 2, CT>(a, sg, lds);
}

template <typename T, int MODE, int DK, int VEC>
int launch(const ChunkArgs& a, hipStream_t st) {
  const int64_t items = static_cast<int64_t>(a.n_slots) * a.H, cols = (a.dv + ss::kCols - 1) / ss::kCols;
  // Short portions go along with the scores (a launch less) unless their workgroups, here two per CU by the scores' LDS,
  // are what takes the time: 15 rows beside 32 of the delta rule 29 us, in a launch of their own 31; 31 rows 45 and 43;
  // 127 rows beside 128 149 and 123.
  const bool apart = cols * a.H * a.S >= 2048;
  if (apart)
    if (const int rc = launch_step_scan(a, MODE, a.min_rows - 1, sizeof(T) == 4 ? 2 : 0, st)) return rc;
  const int64_t score_waves = items * (score_pairs<T, MODE, DK>() ? 2 : 1);
  const int64_t steps = apart ? 0 : cols * a.H * a.S, blocks = steps + (score_waves + kScoreWaves - 1) / kScoreWaves;
  if (blocks > 0x7fffffff) return -1;
  hipLaunchKernelGGL((scan_scores_kernel<T, MODE, DK, (VEC > 0)>), dim3(static_cast<unsigned>(blocks)),
                     dim3(64 * kScoreWaves), 0, st, a, static_cast<int>(steps), static_cast<int>(cols * a.H),
                     static_cast<int>(ss::scan_step_v4(a)));
  ChunkArgs b = a;
  const WalkShape shape = walk_shape(a.T, a.S, a.H, a.G, a.dv, MODE);
  b.walk_heads = shape.heads;
  b.walk_portions = static_cast<int>(std::min<int64_t>(a.S, a.T / a.min_rows));
  const unsigned gx = a.H / shape.heads * ((a.dv + shape.cols - 1) / shape.cols);
  auto walk = [&](auto tiles) {
    constexpr int CT = decltype(tiles)::value;
    const dim3 block(walk_threads<MODE, DK>());
    if constexpr (MODE < kModeDelta) {
      if (a.seg_states > 0) {
        // at most a segment per portion, and those of the cut ones
        scan_grids(gx, static_cast<int64_t>(b.walk_portions) + a.seg_states, [&](dim3 grid, int first) {
          hipLaunchKernelGGL((scan_segments_kernel<T, MODE, DK, VEC, CT>), grid, block, 0, st, b, first);
        });
        scan_grids(gx, a.seg_states, [&](dim3 grid, int first) {
          hipLaunchKernelGGL((scan_segments_end_kernel<T, MODE, DK, VEC, CT>), grid, block, 0, st, b, first);
        });
        return;
      }
    }
    scan_grids(gx, b.walk_portions, [&](dim3 grid, int first) {
      hipLaunchKernelGGL((scan_walk_kernel<T, MODE, DK, VEC, CT>), grid, block, 0, st, b, first);
    });
  };
  constexpr bool WIDE = MODE < kModeDelta;
  if (WIDE && shape.tiles == 8) walk(std::integral_constant<int, WIDE ? 2 : 1>{});
  else walk(std::integral_constant<int, 1>{});
  return static_cast<int>(hipGetLastError());
}

template <typename T, int MODE>
int launch_dk(const ChunkArgs& a, hipStream_t st) {
  // row loads of a lane's channels at once need aligned rows and a width that splits into them
  const int cpl = a.dk <= 64 ? 4 : 8, bytes = min(16, cpl * static_cast<int>(sizeof(T)));
  const bool dec = MODE == kModeDeltaChannel, table = MODE == kModeRetention;
  const uintptr_t at = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) |
                       (dec ? reinterpret_cast<uintptr_t>(a.dec) : 0);
  const bool rows = a.dk % cpl == 0 && a.q_stride % cpl == 0 && a.k_stride % cpl == 0 &&
                    (!dec || a.dec_stride % cpl == 0) && at % bytes == 0 &&
                    (!table || (a.n_freq % cpl == 0 && reinterpret_cast<uintptr_t>(a.cos_sin) % 16 == 0));
  if (!rows) return launch<T, MODE, 128, 0>(a, st);
  if constexpr (MODE < kModeDelta)   // (with a delta rule a lane loads one column)
    if (a.dv % 2 != 0 || a.v_stride % 2 != 0 || reinterpret_cast<uintptr_t>(a.v) % (2 * sizeof(T)) != 0)
      return a.dk <= 64 ? launch<T, MODE, 64, 1>(a, st) : launch<T, MODE, 128, 1>(a, st);
  return a.dk <= 64 ? launch<T, MODE, 64, 2>(a, st) : launch<T, MODE, 128, 2>(a, st);
}

// (every form in a translation unit of its own, chunk_scan_*.hip: together they take minutes to compile)
template <int MODE>
int launch_mode(const ChunkArgs& a, int dtype, hipStream_t st) {
  int rc = -1;
  MIXK_DISPATCH(dtype, rc = (launch_dk<T, MODE>(a, st)));
  return rc;
}

}  // namespace cs
}  // namespace mixk
