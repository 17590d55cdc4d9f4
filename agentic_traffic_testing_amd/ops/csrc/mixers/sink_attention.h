// What the softmax-attention kernels share: the launch arguments and the window arithmetic.
#pragma once

#include "mix_common.h"

namespace mixk {

constexpr int kTileTokens = 64;   // query tokens per prefill tile (host tiling)
constexpr int kPartTokens = 128;  // keys per decode partition
constexpr float kNegBig = -1.0e30f;

struct AttnArgs {
  const int* block_tables;
  const int* seq_kvlen;
  const int* seq_qstart;
  const int* tile_seq;
  const int* tile_qoff;
  float* part;          // decode partials [S, H, max_parts, vdim + 2]
  const float* sink_val;  // [H] score of the sink per query head (nullptr: 0)
  int bt_width, H, G, dim, vdim, block_size, sink, KT, max_parts, bs_shift;
  float scale;
  int window;   // 0: every earlier key
  int keep;     // with a window: the first keys stay visible
  int v_share;  // K heads per V head
  int64_t q_stride;   // elements between two rows of q
  int out_f32;  // results are stored as fp32 whatever T
  int pair;     // pair form: a1 - lam a2, then / rms (eps) * post, gate [T, H / 2 * vdim]
  float lam, post, eps;
  const void* gate;       // row-strided [T, H] of the activation dtype, or nullptr: head h's output
  int64_t gate_stride;    // of row t is multiplied by sigmoid(gate[t, h])
};

template <typename T>
__device__ __forceinline__ float head_gate_of(const AttnArgs& a, int64_t row, int head) {
  if (a.gate == nullptr) return 1.0f;
  return sigmoidf_(ldf(static_cast<const T*>(a.gate) + row * a.gate_stride + head));
}

// first key a query at position qpos sees
__device__ __forceinline__ int window_start(int qpos, int window) {
  return window > 0 ? max(0, qpos - window + 1) : 0;
}

// decode partitions that hold only kept keys, all in front of the window's first partition
__device__ __forceinline__ int keep_parts(int keep, int wstart) {
  return min((keep + kPartTokens - 1) / kPartTokens, wstart / kPartTokens);
}

// Flash form of the matrix-core prefill (sink_flash.hip); false: no instance for these shapes.
bool launch_sink_flash(void* out, const void* q, const void* k_cache, const void* v_cache,
                       const AttnArgs& a, int num_tiles, hipStream_t st);

// Prompts and decode partitions in 32 bits on the matrix cores (sink_float.hip); false: not these shapes.
bool launch_sink_float(void* out, const void* q, const void* k_cache, const void* v_cache, const AttnArgs& a,
                       int num_tiles, int num_decode, int parts, hipStream_t st);

// Partition kernel of the decode rows (sink_decode.hip); false: no instance for these shapes.
bool launch_sink_decode(const void* q, const void* k_cache, const void* v_cache, const AttnArgs& a, int num_decode,
                        int parts, hipStream_t st);
// Join of the decode rows' partitions (both maps of a pair), whichever kernel wrote them.
void launch_sink_join(void* out, const AttnArgs& a, int num_decode, int dtype, hipStream_t st);

}  // namespace mixk
