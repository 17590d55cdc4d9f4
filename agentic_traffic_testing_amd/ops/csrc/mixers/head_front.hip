// Front ends of the attention mixers in 16-byte accesses, one launch each: q / k norm, rotary positions, K pages
// and V pages (or the plain K / V write); absorbed latent queries, normed latent, K and V pages.  The arithmetic
// is that of the element-wise kernels in rope_cache.hip, which keep the shapes that do not fit here.
//
// q and k: a group of L lanes (a power of two) holds one head of one row, 8 channels per lane; sums and the
// partners of rotate-half pairs are exchanged inside the group.  A thread takes the same head of ROWS consecutive
// rows, all loaded first.  WHOLE (norm over the whole projection): the workgroup holds all heads of the row, so
// the projection is read once and there is no second kernel.
//
// V pages are channel-major, so 8 consecutive slots of a channel are one 16-byte store: a group of lanes takes
// the aligned run of 8 slots that starts in its 8 rows (the rows may reach into the next 8), transposes 8 x 8 in
// registers, and stores the rows that belong to no whole run element by element.  Runs are found by slot, not by
// row, so portions that start anywhere in the batch are stored 16 bytes at a time.
//
// Bound: memory traffic.  Measured, before (element-wise, two or three launches) -> now, with the time of a copy of
// the same bytes: 7580 rows, 32 + 8 + 8 heads of 128: 119 -> 38.5 us (38); latent, 7580 rows x 32 heads of 192 + 64:
// 137 -> 57.6 (51), 1300 rows x 8 heads 9.7; norm over the projection, 1908 rows of 24 + 8 + 8 heads: 33 -> 13.9.
// V workgroups come first in the grid: their chain (slots, rows, norm, transposed stores: 11 us) is the longest (the last
// lines 63.7, 13.5 and 13.9 us; at the grid's end 68.7, 16.8 and 16.4).  Sums over a group's lanes are taken of all rows
// of a thread at once (one after the other: 41.2, 63.7, 13.5 us in the first three).
#include <initializer_list>
#include <type_traits>

#include "head_front.h"

namespace mixk {
namespace hf {

// y of 8 channels [8 c, 8 c + 8) of a head rotated with the row's table (all lanes of the group take part)
struct Table {
  float cs[8], sn[8];
};
__device__ __forceinline__ Table load_table(const float* tab, int c, int n_freq, int half) {
  Table r;
  if (half) {   // chunks outside the rotated ones read a valid one and do not use it
    const int nc = n_freq >> 3, f = (c < nc ? c : c < 2 * nc ? c - nc : 0) * 8;
    ld8(tab + f, r.cs);
    ld8(tab + n_freq + f, r.sn);
  } else {
    const int f = 8 * c < 2 * n_freq ? 4 * c : 0;
    const f32x4v a = *reinterpret_cast<const f32x4v*>(tab + f);
    const f32x4v b = *reinterpret_cast<const f32x4v*>(tab + n_freq + f);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      r.cs[e] = a[e];
      r.sn[e] = b[e];
    }
  }
  return r;
}
// lane0: the lane that holds channel chunk 0
__device__ __forceinline__ void rotate(float* y, const Table& t, int lane0, int c, int n_freq, int half) {
  if (half) {
    const int nc = n_freq >> 3;
    const bool on = c >= 0 && c < 2 * nc, low = c < nc;
    const int from = on ? lane0 + (low ? c + nc : c - nc) : lane0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float p = __shfl(y[e], from, kWave);
      if (on) y[e] = low ? y[e] * t.cs[e] - p * t.sn[e] : y[e] * t.cs[e] + p * t.sn[e];
    }
  } else if (c >= 0 && 8 * c < 2 * n_freq) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = y[2 * e], b = y[2 * e + 1];
      y[2 * e] = a * t.cs[e] - b * t.sn[e];
      y[2 * e + 1] = b * t.cs[e] + a * t.sn[e];
    }
  }
}

// sums over the lanes of a group, of several rows at once: an exchange's latency is paid once per step
template <int N>
__device__ __forceinline__ void lane_group_sums(float (&v)[N], int L) {
  for (int o = L >> 1; o > 0; o >>= 1)
#pragma unroll
    for (int r = 0; r < N; ++r) v[r] += __shfl_xor(v[r], o, kWave);
}

// Workgroup (rb, y) of the V part: rows [2 HR rb, 2 HR (rb + 1)) in two halves; item = (head, half), L lanes each.
// NORM: every row's head divided by its root mean square over vdim, times v_weight.
template <typename T, int HR, bool NORM>
__device__ __forceinline__ void v_part(const FrontArgs& a, int rb, int y, int lsh) {
  constexpr int kVRows = 2 * HR;
  __shared__ int slot_lds[kVRows + 14], mask_lds[2];
  __shared__ int64_t at_lds[kVRows];   // page * channels + slot in the page: where a row goes, without its head
  const int tid = threadIdx.x, r0 = rb * kVRows, L = 1 << lsh, bs = a.block_size;
  const int item = y * (static_cast<int>(blockDim.x) >> lsh) + (tid >> lsh), c = tid & (L - 1);
  const int half = item & 1, g = min(item >> 1, a.GV - 1);
  const bool on = c * 8 < a.vdim && (item >> 1) < a.GV;
  const int ch = c * 8 < a.vdim ? c * 8 : 0;
  const T* src = static_cast<const T*>(a.vx) + g * a.vdim + ch;
  float v[8][8], w[8];
  auto load = [&](int first, int rows) {
#pragma unroll
    for (int j = 0; j < rows; ++j) ld8(src + min(first + j, a.T - 1) * a.v_stride, v[j]);
  };
  load(r0 + HR * half, HR);   // in flight while the slots are looked at
#pragma unroll
  for (int e = 0; e < 8; ++e) w[e] = 1.f;
  if (a.v_weight != nullptr) ld8(static_cast<const T*>(a.v_weight) + ch, w);
  if (tid < kVRows + 14) {   // rows r0 - 7 ... r0 + 2 HR + 6
    const int r = r0 - 7 + tid, s = r >= 0 && r < a.T ? a.slots[r] : -1;
    slot_lds[tid] = s;
    if (tid >= 7 && tid < kVRows + 7) at_lds[tid - 7] = static_cast<int64_t>(s / bs) * a.GV * a.vdim * bs + s % bs;
  }
  lds_barrier();
  if (tid < kWave) {
    const int r = min(tid, kVRows - 1), s = slot_lds[r + 7];
    bool run = tid < kVRows && s >= 0 && (bs & 7) == 0;
    if (run)
#pragma unroll
      for (int i = 0; i < 8; ++i) run = run && slot_lds[r + 7 - (s & 7) + i] == s - (s & 7) + i;
    const uint64_t runs = __ballot(run), heads = __ballot(run && (s & 7) == 0);
    const uint64_t live = __ballot(tid < kVRows && s >= 0);
    if (tid == 0) {
      mask_lds[0] = static_cast<int>(heads);
      mask_lds[1] = static_cast<int>(live & ~runs);
    }
  }
  lds_barrier();
  const int heads = (mask_lds[0] >> (HR * half)) & ((1 << HR) - 1);
  const int single = (mask_lds[1] >> (HR * half)) & ((1 << HR) - 1);
  T* cache = static_cast<T*>(a.v_cache) + (static_cast<int64_t>(g) * a.vdim + ch) * bs;
  auto norm = [&](auto rows) {
    constexpr int R = decltype(rows)::value;
    float ss[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      ss[j] = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) ss[j] += v[j][e] * v[j][e];
      ss[j] = on ? ss[j] : 0.f;
    }
    lane_group_sums(ss, L);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float inv = 1.0f / sqrtf(ss[j] / static_cast<float>(a.vdim) + a.eps);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[j][e] = v[j][e] * inv * w[e];
    }
  };
  if (NORM) norm(std::integral_constant<int, HR>{});
#pragma unroll
  for (int j = 0; j < HR; ++j) {
    if (!on || !(single >> j & 1)) continue;
    T* dst = cache + at_lds[HR * half + j];
#pragma unroll
    for (int e = 0; e < 8; ++e) stf(dst + static_cast<int64_t>(e) * bs, v[j][e]);
  }
  if (heads == 0) return;
  const int j0 = __builtin_ctz(heads);
  if (HR < 8 || j0 != 0) {
    load(r0 + HR * half + j0, 8);
    if (NORM) norm(std::integral_constant<int, 8>{});
  }
  if (!on) return;
  T* dst = cache + at_lds[HR * half + j0];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = v[j][e];
    st8(dst + static_cast<int64_t>(e) * bs, o);
  }
}

template <typename T, int ROWS, int VH, bool WHOLE>
__global__ void __launch_bounds__(WHOLE ? 1024 : 256)
head_front_kernel(FrontArgs a, int v_blocks, int uy, int lsh, int vy, int vlsh) {
  __shared__ float sums[WHOLE ? ROWS : 1][2][16];
  const int vb = blockIdx.x, bid = vb - v_blocks;
  if (bid < 0) {   // uniform over the workgroup
    if (a.v_norm)
      v_part<T, VH, true>(a, vb / vy, vb % vy, vlsh);
    else
      v_part<T, VH, false>(a, vb / vy, vb % vy, vlsh);
    return;
  }
  const int rb = bid / uy, y = bid - rb * uy, t0 = rb * ROWS, tid = threadIdx.x, L = 1 << lsh;
  const int item = y * (static_cast<int>(blockDim.x) >> lsh) + (tid >> lsh), c = tid & (L - 1);
  const bool on = item < a.H + a.G && c * 8 < a.dim, is_q = item < a.H;
  const int head = min(item, a.H + a.G - 1) - (is_q ? 0 : a.H), ch = c * 8 < a.dim ? c * 8 : 0;
  const T* src = is_q ? static_cast<const T*>(a.qx) : static_cast<const T*>(a.kx);
  const int64_t stride = is_q ? a.q_stride : a.k_stride;
  src += static_cast<int64_t>(head) * a.dim + ch;
  float x[ROWS][8], w[8];
  Table tab[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) ld8(src + min(t0 + r, a.T - 1) * stride, x[r]);
  const T* wp = is_q ? static_cast<const T*>(a.q_norm) : static_cast<const T*>(a.k_norm);
  const bool whole = WHOLE || a.row_inv != nullptr;
#pragma unroll
  for (int e = 0; e < 8; ++e) w[e] = 1.f;
  if (wp != nullptr) ld8(wp + (whole ? static_cast<int64_t>(head) * a.dim : 0) + ch, w);
  if (a.n_freq > 0)
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      tab[r] = load_table(a.cos_sin + static_cast<int64_t>(min(t0 + r, a.T - 1)) * 2 * a.n_freq, c, a.n_freq, a.half);
  int slot[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) slot[r] = a.slots[min(t0 + r, a.T - 1)];
  const int lane0 = (tid & 63) & ~(L - 1);
  float ss[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    if (a.n_freq > 0 && a.norm_last) rotate(x[r], tab[r], lane0, c, a.n_freq, a.half);
    ss[r] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss[r] += x[r][e] * x[r][e];
    ss[r] = on ? ss[r] : 0.f;
  }
  if (WHOLE) {
    float both[2 * ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      both[2 * r] = is_q ? ss[r] : 0.f;
      both[2 * r + 1] = is_q ? 0.f : ss[r];
    }
    lane_group_sums(both, kWave);
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      if ((tid & 63) == 0) {
        sums[WHOLE ? r : 0][0][tid >> 6] = both[2 * r];
        sums[WHOLE ? r : 0][1][tid >> 6] = both[2 * r + 1];
      }
    lds_barrier();
  } else if (!a.plain && !whole) {
    lane_group_sums(ss, L);
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int t = t0 + r;
    if (t >= a.T) break;
    float inv;
    if (a.plain) {
      inv = 1.0f;
    } else if (WHOLE) {
      float s = 0.f;
      for (int i = 0; i < static_cast<int>(blockDim.x) >> 6; ++i) s += sums[WHOLE ? r : 0][is_q ? 0 : 1][i];
      inv = 1.0f / sqrtf(s / static_cast<float>((is_q ? a.H : a.G) * a.dim) + a.eps);
    } else if (whole) {
      inv = a.row_inv[2 * static_cast<int64_t>(t) + (is_q ? 0 : 1)];
    } else {
      inv = 1.0f / sqrtf(ss[r] / static_cast<float>(a.dim) + a.eps);
    }
    // (the temperature is a common factor of the head, so it commutes with the rotation)
    if (is_q && a.temp_coef != 0.f)
      inv *= 1.0f + a.temp_coef * logf(floorf(static_cast<float>(a.positions[t] + 1) / a.temp_every) + 1.0f);
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = x[r][e] * inv * w[e];
    if (a.n_freq > 0 && !a.norm_last) rotate(o, tab[r], lane0, c, a.n_freq, a.half);
    if (!on || (!is_q && slot[r] < 0)) continue;
    T* dst = is_q ? static_cast<T*>(a.q_out) + (static_cast<int64_t>(t) * a.H + head) * a.dim
                  : static_cast<T*>(a.k_cache) + ((static_cast<int64_t>(slot[r] / a.block_size) * a.G + head) *
                                                      a.block_size + slot[r] % a.block_size) * a.dim;
    st8(dst + ch, o);
  }
}

// Latent form: item = query head (copy of q_lat | rotated channels of qx) or, last, the row's key.
template <typename T, int ROWS, int VH>
__global__ void __launch_bounds__(256)
latent_front_kernel(FrontArgs a, int v_blocks, int uy, int lsh, int vy, int vlsh) {
  const int vb = blockIdx.x, bid = vb - v_blocks;
  if (bid < 0) {
    v_part<T, VH, true>(a, vb / vy, vb % vy, vlsh);
    return;
  }
  const int rb = bid / uy, y = bid - rb * uy, t0 = rb * ROWS, tid = threadIdx.x, L = 1 << lsh;
  const int item = y * (256 >> lsh) + (tid >> lsh), c = tid & (L - 1);
  const int rank = a.rank, kd = a.dim, rc = rank >> 3;
  const bool is_q = item < a.H, on = item < a.H + (a.kx != nullptr ? 1 : 0) && c * 8 < kd;
  const int head = min(item, a.H - 1), cr = c - rc;   // cr >= 0: chunk of the rotated part
  const int ch = on ? c * 8 : 0;
  // one address per row: all loads are issued before any is used
  const T* src;
  int64_t stride;
  if (is_q || a.kx == nullptr) {
    if (ch < rank) {
      src = static_cast<const T*>(a.q_lat) + static_cast<int64_t>(head) * a.T * rank + ch;
      stride = rank;
    } else {
      src = static_cast<const T*>(a.qx) + static_cast<int64_t>(head) * (a.qdim + a.rot) + a.qdim + (ch - rank);
      stride = a.q_stride;
    }
  } else {
    src = static_cast<const T*>(a.kx) + ch;
    stride = a.k_stride;
  }
  float x[ROWS][8], w[8];
  Table tab[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) ld8(src + min(t0 + r, a.T - 1) * stride, x[r]);
#pragma unroll
  for (int e = 0; e < 8; ++e) w[e] = 1.f;
  if (!is_q && a.kx != nullptr && ch < rank) ld8(static_cast<const T*>(a.k_norm) + ch, w);
  if (a.n_freq > 0 && cr >= 0)   // (the lanes that copy would load twice what they copy)
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      tab[r] = load_table(a.cos_sin + static_cast<int64_t>(min(t0 + r, a.T - 1)) * 2 * a.n_freq, cr, a.n_freq, a.half);
  int slot[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) slot[r] = a.slots[min(t0 + r, a.T - 1)];
  const int lane0 = ((tid & 63) & ~(L - 1)) + rc;
  if (__any(on && !is_q)) {   // (most waves hold queries only)
    float ss[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      ss[r] = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) ss[r] += x[r][e] * x[r][e];
      ss[r] = on && ch < rank ? ss[r] : 0.f;
    }
    lane_group_sums(ss, L);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const float inv = 1.0f / sqrtf(ss[r] / static_cast<float>(rank) + a.eps);
      if (!is_q && cr < 0)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[r][e] = x[r][e] * inv * w[e];
    }
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int t = t0 + r;
    if (t >= a.T) break;
    if (a.n_freq > 0) rotate(x[r], tab[r], lane0, cr, a.n_freq, a.half);
    if (!on || (!is_q && slot[r] < 0)) continue;
    T* dst = is_q ? static_cast<T*>(a.q_out) + (static_cast<int64_t>(t) * a.H + item) * kd
                  : static_cast<T*>(a.k_cache) + static_cast<int64_t>(slot[r]) * kd;
    st8(dst + ch, x[r]);
  }
}

int lanes_log2(int width) {   // lanes of 8 channels, rounded up to a power of two
  int l = 0;
  while ((8 << l) < width) ++l;
  return l;
}

constexpr int kManyRows = 4;

// Rows per half of a V workgroup.  A row on its own costs a store of 2 bytes per channel, each to a line of its own:
// up to kFewRows rows (decode steps) every row gets a workgroup's half.  32 decode rows of 8 heads: 11 -> 5 us;
// at 480 rows of one prompt, where runs of 8 leave most halves idle, the two are level (8.7, 8.4).
constexpr int kFewRows = 512;
int v_half_rows(int T) { return T <= kFewRows ? 1 : 8; }

bool aligned(std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if (reinterpret_cast<uintptr_t>(p) & 15) return false;
  return true;
}

// frequencies whose chunks of 8 channels are rotated whole
bool rotary_ok(int n_freq, int half) { return n_freq % (half ? 8 : 4) == 0; }

int ceil_div(int64_t a, int64_t b) { return static_cast<int>((a + b - 1) / b); }

}  // namespace hf

bool launch_head_front(const FrontArgs& args, bool whole, int dtype, hipStream_t st) {
  FrontArgs a = args;
  if (a.dim % 8 || a.vdim % 8 || a.dim > 512 || a.vdim > 512 || !hf::rotary_ok(a.n_freq, a.half) ||
      (a.H > 0 && a.q_stride % 8) || a.k_stride % 8 || a.v_stride % 8 ||
      !hf::aligned({a.q_out, a.qx, a.kx, a.vx, a.q_norm, a.k_norm, a.k_cache, a.v_cache, a.cos_sin}))
    return false;
  const int vh = hf::v_half_rows(a.T), lsh = hf::lanes_log2(a.dim), vlsh = hf::lanes_log2(a.vdim);
  const int64_t lanes = static_cast<int64_t>(a.H + a.G) << lsh;
  // A workgroup that holds a row's heads, up to 1024 lanes; wider rows read the inverse RMS of the projections
  const bool wide = whole && lanes <= 1024;
  if (whole && !wide) return false;
  const int threads = wide ? max(256, hf::ceil_div(lanes, 64) * 64) : 256;
  // Four rows per thread once a quarter of the threads fills the chip (256 CUs x 2048 lanes): 7580 rows of 40 heads of
  // 128 take 30 % more time with one row per thread, 9 % with two; latent 30 % and 12 %.
  const int rows = static_cast<int64_t>(a.T) * lanes >= hf::kManyRows * 256 * 2048 && vh == 8 ? hf::kManyRows : 1;
  const int uy = wide ? 1 : hf::ceil_div(lanes, threads);
  const int64_t qk = static_cast<int64_t>(hf::ceil_div(a.T, rows)) * uy;
  const int vy = hf::ceil_div(static_cast<int64_t>(2 * a.GV) << vlsh, threads);
  const int64_t grid = qk + static_cast<int64_t>(hf::ceil_div(a.T, 2 * vh)) * vy;
  if (grid > 0x7fffffff) return false;
  if (wide) a.row_inv = nullptr;
#define MIXK_FRONT(R, V, W)                                                                                      \
  MIXK_DISPATCH(dtype, hipLaunchKernelGGL((hf::head_front_kernel<T, R, V, W>), dim3(static_cast<unsigned>(grid)), \
                                          dim3(threads), 0, st, a, static_cast<int>(grid - qk), uy, lsh, vy, vlsh))
  if (wide) {
    if (rows == hf::kManyRows) MIXK_FRONT(hf::kManyRows, 8, true);
    else if (vh == 8) MIXK_FRONT(1, 8, true);
    else MIXK_FRONT(1, 1, true);
  } else {
    if (rows == hf::kManyRows) MIXK_FRONT(hf::kManyRows, 8, false);
    else if (vh == 8) MIXK_FRONT(1, 8, false);
    else MIXK_FRONT(1, 1, false);
  }
#undef MIXK_FRONT
  return true;
}

bool launch_latent_front(const FrontArgs& a, int dtype, hipStream_t st) {
  if (a.rank % 8 || a.rot % 8 || a.qdim % 8 || a.dim > 512 || !hf::rotary_ok(a.n_freq, a.half) || a.q_stride % 8 ||
      a.k_stride % 8 ||
      !hf::aligned({a.q_out, a.qx, a.kx, a.q_lat, a.k_norm, a.k_cache, a.v_cache, a.cos_sin}))
    return false;
  const int vh = hf::v_half_rows(a.T), lsh = hf::lanes_log2(a.dim), vlsh = hf::lanes_log2(a.rank);
  const int64_t lanes = static_cast<int64_t>(a.H + 1) << lsh;
  const int rows = static_cast<int64_t>(a.T) * lanes >= hf::kManyRows * 256 * 2048 && vh == 8 ? hf::kManyRows : 1;   // as above
  const int uy = hf::ceil_div(lanes, 256);
  const int64_t qk = static_cast<int64_t>(hf::ceil_div(a.T, rows)) * uy;
  const int vy = hf::ceil_div(2ll << vlsh, 256);
  const int64_t grid = qk + (a.kx != nullptr ? static_cast<int64_t>(hf::ceil_div(a.T, 2 * vh)) * vy : 0);
  if (grid > 0x7fffffff) return false;
#define MIXK_FRONT(R, V)                                                                                        \
  MIXK_DISPATCH(dtype, hipLaunchKernelGGL((hf::latent_front_kernel<T, R, V>), dim3(static_cast<unsigned>(grid)), \
                                          dim3(256), 0, st, a, static_cast<int>(grid - qk), uy, lsh, vy, vlsh))
  if (rows == hf::kManyRows) MIXK_FRONT(hf::kManyRows, 8);
  else if (vh == 8) MIXK_FRONT(1, 8);
  else MIXK_FRONT(1, 1);
#undef MIXK_FRONT
  return true;
}

}  // namespace mixk
