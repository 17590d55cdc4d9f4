// Decode rows and short portions of the matrix-state recurrences (chunk_scan.h: the same forms and
// arguments), token by token.
//
// A workgroup owns 64 value columns of one (sequence, head): thread (row group rg, lane c) holds rows rg + 16 j
// of the columns 4 c ... 4 c + 3 in registers, so the state moves in coalesced 16-byte accesses.  q, k and the
// decays of a token go through LDS once; the column sums over the rows are two lane exchanges in a wave and one
// trip through LDS.  The delta rule needs S^T k before u and S^T q after it, but
//     S1^T q = (a S0)^T q + (k . q) u,   so both sums are taken of the decayed state in one pass.
//
// Bound: the state is read and written once, 128 KB per (sequence, head) of 128 x 128.  Its loads are issued first
// and nothing waits for them until the token's operands are in LDS (an LDS-only barrier; __syncthreads() would
// wait).  Measured at 16 sequences, 32 heads, delta rule: 46 -> 12.3 us (half of the 134 MB from the last-level cache);
// 8 sequences: forget gate 13.5 -> 6.9, state space (128 heads of 128 x 64) 23 -> 10.8.
#pragma once

#include "chunk_scan.h"

namespace mixk {
namespace ss {

typedef __attribute__((ext_vector_type(4))) float f32x4;
constexpr int kCols = 64;

// R: rows per thread (dk <= 16 R <= 256); V4: 16-byte state accesses (dv % 4 == 0, aligned state)
template <int MODE, int R>
struct StepLds {
  static constexpr bool DELTA = MODE >= kModeDelta, CH = MODE == kModeForget || MODE == kModeDeltaChannel;
  __attribute__((aligned(16))) float part[2][DELTA ? 2 : 1][4][kCols];
  float sq[2][16 * R], sk[2][16 * R], sa[2][CH ? 16 * R : 1];
  float sums[2][4][3];
};

// Workgroup bx of sequence s: 256 threads.
template <typename T, int MODE, int R, bool V4>
__device__ __forceinline__ void scan_step(const ChunkArgs& a, int max_rows, int bx, int s, StepLds<MODE, R>& lds) {
  constexpr bool DELTA = MODE >= kModeDelta;
  constexpr bool CH = MODE == kModeForget || MODE == kModeDeltaChannel;
  auto& sq = lds.sq;
  auto& sk = lds.sk;
  auto& sa = lds.sa;
  auto& sums = lds.sums;
  auto& part = lds.part;
  const int cb = bx / a.H, h = bx % a.H, tid = threadIdx.x;
  const int slot = a.seq_slot[s];
  const int first = a.seq_qstart[s], n = a.seq_qstart[s + 1] - first;
  if (slot < 0 || n <= 0 || n > max_rows) return;
  const int dk = a.dk, dv = a.dv, w = tid >> 6;
  const int rg = tid >> 4, cl = (tid & 15) * 4, col = cb * kCols + cl;
  const int g = MODE == kModeForget ? h : h / (a.H / a.G);
  float* st = a.state + (static_cast<int64_t>(slot) * a.H + h) * dk * dv;
  const bool fresh = a.positions[first] == 0;
  f32x4 S[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {   // clamped addresses: every load is in bounds and issued without a branch
    const float* p = st + static_cast<int64_t>(min(rg + 16 * j, dk - 1)) * dv;
    if (V4)
      S[j] = *reinterpret_cast<const f32x4*>(p + min(col, dv - 4));
    else
#pragma unroll
      for (int e = 0; e < 4; ++e) S[j][e] = p[min(col + e, dv - 1)];
  }
  // this thread's channel of q, k and the decays
  const int ch = min(tid, dk - 1);
  const bool ch_on = tid < dk;
  float b0 = 0.f, b1 = 0.f, skip = 0.f;
  if (MODE == kModeForget) {
    b0 = a.p0[h * dk + ch];
    b1 = a.p1[h * dk + ch];
  } else if (MODE != kModeRetention) {
    b0 = a.p0[CH ? h * dk + ch : h];
    b1 = expf(a.p1[h]);
    if (MODE == kModeStateSpace) skip = a.p2[h];
  }
  const float fixed = MODE == kModeRetention ? a.p0[h * kPowers + 1] : 1.f;
  for (int t = 0; t < n; ++t) {
    const int64_t row = first + t;
    const int b = t & 1;
    const T* qr = static_cast<const T*>(a.q) + row * a.q_stride + static_cast<int64_t>(g) * dk;
    const T* kr = static_cast<const T*>(a.k) + row * a.k_stride + static_cast<int64_t>(g) * dk;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = ldf(static_cast<const T*>(a.v) + row * a.v_stride + static_cast<int64_t>(h) * dv + min(col + e, dv - 1));
    float q = ldf(qr + ch), k = ldf(kr + ch), dec = 1.f, dt = 1.f, beta = 0.f;
    if (MODE == kModeRetention && a.n_freq > 0) {   // rotate-half pairs (c, c + n)
      const int nf = a.n_freq, p = ch < nf ? ch + nf : ch < 2 * nf ? ch - nf : ch, f = ch < nf ? ch : p;
      const float* tab = a.cos_sin + row * 2 * nf;
      const float qp = ldf(qr + p), kp = ldf(kr + p);
      if (ch < 2 * nf) {
        const float cs = tab[f], sn = ch < nf ? -tab[nf + f] : tab[nf + f];
        q = q * cs + qp * sn;
        k = k * cs + kp * sn;
      }
    }
    if (MODE == kModeRetention) {
      k *= a.kscale;
      dec = fixed;
    } else if (MODE == kModeForget) {
      dec = b1 + (1.0f - b1) * sigmoidf_(k + b0);
      k = 1.0f - dec;
      q = siluf_(q);
    } else {
      const float raw = ldf(static_cast<const T*>(a.dec) + row * a.dec_stride + (CH ? h * dk + ch : h));
      const float sp = softplusf_(raw + b0);
      dec = expf(-b1 * sp);
      if (MODE == kModeStateSpace) {
        dt = sp;
        k *= dt;
      } else {
        beta = sigmoidf_(ldf(static_cast<const T*>(a.beta) + row * a.beta_stride + h));
      }
    }
    q = ch_on ? q : 0.f;   // channels past dk: nothing
    k = ch_on ? k : 0.f;
    if (tid < 16 * R) {
      sq[b][tid] = q;
      sk[b][tid] = k;
      if (CH) sa[b][CH ? tid : 0] = ch_on ? dec : 1.f;
    }
    if (DELTA) {
      const float qq = wave_sum(q * q), kk = wave_sum(k * k), qk = wave_sum(q * k);
      if ((tid & 63) == 0) {
        sums[b][w][0] = qq;
        sums[b][w][1] = kk;
        sums[b][w][2] = qk;
      }
    }
    lds_barrier();
    if (t == 0) {
#pragma unroll
      for (int j = 0; j < R; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[j][e] = !fresh && rg + 16 * j < dk && col + e < dv ? S[j][e] : 0.f;
    }
    float qi = 1.f, ki = 1.f, kq = 0.f;
    if (DELTA) {
      float x[3];
#pragma unroll
      for (int e = 0; e < 3; ++e) x[e] = (sums[b][0][e] + sums[b][1][e]) + (sums[b][2][e] + sums[b][3][e]);
      qi = 1.0f / (sqrtf(static_cast<float>(dk)) * sqrtf(x[0] + 1e-6f));
      ki = 1.0f / sqrtf(x[1] + 1e-6f);
      kq = x[2] * qi * ki;
    }
    f32x4 os[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, rs[2] = {os[0], os[0]};   // (short sums round less)
    const f32x4 vv = {v[0], v[1], v[2], v[3]};
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float kd = sk[b][rg + 16 * j] * ki, qd = sq[b][rg + 16 * j] * qi;
      const float ad = CH ? sa[b][CH ? rg + 16 * j : 0] : dec;
      if (DELTA) {
        S[j] *= ad;
        rs[j & 1] += S[j] * kd;
      } else {
        S[j] = S[j] * ad + vv * kd;
      }
      os[j & 1] += S[j] * qd;
    }
    f32x4 o = os[0] + os[1], r = rs[0] + rs[1];
    // over the four row groups of the wave, then over the waves
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] += __shfl_xor(o[e], 16, kWave);
      o[e] += __shfl_xor(o[e], 32, kWave);
      if (DELTA) {
        r[e] += __shfl_xor(r[e], 16, kWave);
        r[e] += __shfl_xor(r[e], 32, kWave);
      }
    }
    if ((tid & 63) < 16) {
      *reinterpret_cast<f32x4*>(&part[b][0][w][cl]) = o;
      if (DELTA) *reinterpret_cast<f32x4*>(&part[b][DELTA ? 1 : 0][w][cl]) = r;
    }
    lds_barrier();
    auto total = [&](int which) {
      f32x4 x[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = *reinterpret_cast<const f32x4*>(&part[b][which][e][cl]);
      return (x[0] + x[1]) + (x[2] + x[3]);
    };
    f32x4 u = vv;
    if (DELTA) {
      u = (vv - total(DELTA ? 1 : 0)) * beta;
#pragma unroll
      for (int j = 0; j < R; ++j) S[j] += u * (sk[b][rg + 16 * j] * ki);
    }
    if (rg == 0) {
      f32x4 y = total(0);
      if (DELTA) y += u * kq;
      if (MODE == kModeStateSpace) y += vv * skip;
      float* op = a.out + (row * a.H + h) * dv + col;
      if (V4) {
        if (col < dv) *reinterpret_cast<f32x4*>(op) = y;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < dv) op[e] = y[e];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int d = rg + 16 * j;
    if (d < dk) {
      float* p = st + static_cast<int64_t>(d) * dv + col;
      if (V4) {
        if (col < dv) *reinterpret_cast<f32x4*>(p) = S[j];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < dv) p[e] = S[j][e];
      }
    }
  }
}

inline bool scan_step_v4(const ChunkArgs& a) {
  return a.dv % 4 == 0 && ((reinterpret_cast<uintptr_t>(a.state) | reinterpret_cast<uintptr_t>(a.out)) & 15) == 0;
}

}  // namespace ss
}  // namespace mixk
