// Retention: linear attention with one fixed decay g per head over ragged batches of portions, state
// carried per sequence in fp32.
//
// Per head, with S [dk, dv] the state, per token:   S = g S + k v^T,   o = S^T q
// q and k are rotated here (rotate-half pairs (i, i + n_freq) over the first 2 n_freq channels,
// cos / sin from the step's table) and k times dk^-1/2, so everything after the projections is fp32.
// A portion whose first position is 0 starts from the zero state whatever its slot holds.
// Kernels: chunk_scan_kernels.h (portions), step_scan.hip (decode rows, short portions, keys wider than 128).
#include "chunk_scan.h"
#include "mixers.h"

using namespace mixk;

// `rec`: scratch for the chunked form (nullptr: every portion token by token); T rows in all.
extern "C" int mixk_retention(float* out, float* state, const void* q, int64_t q_stride,
                              const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                              const float* powers, int n_powers, const float* cos_sin, int n_freq,
                              const int* positions, const int* seq_qstart, const int* seq_slot,
                              int T, int S, int H, int dk, int dv, float* rec, int dtype,
                              hipStream_t st) {
  if (S <= 0) return 0;
  if (dk <= 0 || dk > 256 || dv <= 0 || H <= 0 || n_powers != kPowers || 2 * n_freq > dk) return -1;
  ChunkArgs c{};
  c.out = out; c.state = state; c.q = q; c.k = k; c.v = v; c.p0 = powers; c.cos_sin = cos_sin; c.rec = rec;
  c.positions = positions; c.seq_qstart = seq_qstart; c.seq_slot = seq_slot;
  c.q_stride = q_stride; c.k_stride = k_stride; c.v_stride = v_stride;
  c.S = S; c.H = c.G = H; c.dk = dk; c.dv = dv; c.n_freq = n_freq;
  c.kscale = 1.0f / sqrtf(static_cast<float>(dk));
  return launch_scan_batch(c, kModeRetention, T, dtype, st);
}
