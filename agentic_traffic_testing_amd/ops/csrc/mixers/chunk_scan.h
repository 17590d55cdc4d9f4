// Chunked form of the recurrences S = diag(a) S + k u^T, o = S^T q (chunk_scan_kernels.h).
#pragma once

#include "mix_common.h"

namespace mixk {

constexpr int kScanChunk = 16;         // tokens per chunk
constexpr int kPowers = 65;            // retention: powers 0 ... 64 of a head's decay
enum ScanMode { kModeRetention = 0, kModeForget = 1, kModeStateSpace = 2, kModeDelta = 3,
                kModeDeltaChannel = 4 };
constexpr int kWalkCols = 64;          // value columns of the walk's four waves with one tile of 16 each
// the walk's waves that prepare operands for keys of up to dk channels
constexpr int operand_waves(int mode, int dk) { return mode >= kModeDelta ? dk / 16 : 4; }

struct ChunkArgs {
  float* out;             // [T, H, dv]
  float* state;           // [slots, H, dk, dv]
  const void* q;          // [T, G dk]; head h reads the columns of h / (H / G)
  const void* k;          // like q; forget-gate form: the gate logits
  const void* v;          // [T, H dv]
  const void* dec;        // delta: decay logits [T, H] or [T, H dk]; state-space: dt [T, H]
  const void* beta;       // delta: [T, H]
  const float* p0;        // delta, state-space: dt_bias; forget-gate: f_bias; retention: powers [H, kPowers]
  const float* p1;        // delta, state-space: A_log; forget-gate: lower bound
  const float* p2;        // state-space: skip
  const float* cos_sin;   // retention: [T, 2 n_freq]
  float* rec;             // scratch: a record of scan_record_floats() per (chunk, head)
  const int* positions;
  const int* seq_qstart;
  const int* seq_slot;
  int64_t q_stride, k_stride, v_stride, dec_stride, beta_stride;
  int S, H, G, dk, dv, n_freq, n_slots;   // n_slots: chunk slots (scan_chunk_slots)
  int min_rows;           // shorter portions of a chunked batch run token by token (kScanMinRows)
  float* seg;             // scratch: states at the ends of segments and the decays over them (scan_segments)
  int seg_chunks, seg_states;
  float kscale;
  int64_t T;              // rows in all
  int walk_heads;         // heads per workgroup of the walk (walk_shape)
  int walk_portions;      // portions of the walk's grid: at most so many of the S have min_rows rows
};

// Chunk c of sequence s has the slot seq_qstart[s] / 16 + s + c: disjoint runs, known on the device only.
inline int64_t scan_chunk_slots(int64_t T, int64_t S) { return T / kScanChunk + S; }
// record: A [16][16], then the 16-entry scales of q, of k against the state and of k into the state, the
// decay over the chunk (x 16, but for the mark of keys without bf16 parts), then with a delta rule T [16][16], then with a
// decay per channel the decays [16][64 or 128] of the chunk, 1 for a token or channel that is not there: 5.4 or 9.5 KB per
// chunk and head (8192 tokens, 32 heads of 128: forget gate 155 MB, per-channel delta rule 172, the others 21 and 38)
constexpr int kRecQ = 256, kRecK = 272, kRecKt = 288, kRecEnd = 304, kRecNoParts = 305, kRecT = 320;
constexpr int scan_rec_decay(int mode) { return mode >= kModeDelta ? 576 : 320; }
constexpr int scan_decay_width(int dk) { return dk <= 64 ? 64 : 128; }
constexpr bool scan_keeps_decays(int mode) { return mode == kModeForget || mode == kModeDeltaChannel; }
constexpr int scan_record_floats(int mode, int dk) {
  return scan_rec_decay(mode) + (scan_keeps_decays(mode) ? kScanChunk * scan_decay_width(dk) : 0);
}
// A long portion in few heads leaves most of the chip idle: with one number or one per channel as the decay it is cut
// into segments that run side by side, in two passes (chunk_scan_kernels.h).  `chunks`: a segment's length with which the
// batch makes about 256 workgroups (one per CU: the registers allow no second one), at least 7 and a 16th of the batch
// (a segment's start is put together from all segments before it; us with at least 10 / 7, 8 heads: 350 rows forget gate
// 55 / 46, state space 42 / 35, retention 49 / 40, 600 rows 53 / 48, 40 / 36, 46 / 41).  A batch of less than 20 chunks is
// not cut.
// A workgroup of the walk: four waves beside four that prepare the operands, with two tiles of 16 columns of S each (wide:
// the operands serve 128 columns, or two heads of 64 whose keys are the same) or with one, 64 columns; so the delta rule,
// whose portions are not cut, with up to eight waves for its operands.  256 workgroups run at once.  In `units` of a head's
// 64 columns, S portions make S x units of them:
// - From 512 on wide, if there are 6 chunks per CU: few rows in many portions are decode rows and one prompt, which is
//   done sooner in more workgroups (state space, 32 heads, us, narrow / wide: 63 rows + 128 64 / 69, 127 + 256
//   125 / 128, 31 + 300 68 / 75, but 64 x 12 92 / 86, 127 + 600 184 / 162, 8 x 512 103 / 88 and, on the wrong side of the
//   line, 20 + 8 x 40 47 / 42); from 257 on if there are as many as for long portions.
// - 192 - 256 fill the chip with narrow ones, and uncut: a portion in half the workgroups would have to be cut to fill it
//   (32 heads, narrow uncut / wide cut: retention 4 x 350 60 / 68, 4 x 1000 134 / 138, 4 x 2000 260 / 269, forget gate
//   4 x 700 107 / 112, state space 4 x 1000 98 / 114, 8 heads 16 x 512 59 / 77).
// - Fewer: long portions are cut, and wide where a 16th of the batch per segment is enough to fill the chip (32
//   heads, one prompt of 2048, narrow / wide: retention 112 / 89, state space 82 / 76; 8 heads, 4 x 2000: retention
//   114 / 127, one of 8192 121 / 141).
struct WalkShape {
  int tiles, heads, cols;   // of 16 columns, one or two per wave; heads per workgroup; columns per workgroup and head
};
inline int64_t walk_units(int64_t H, int64_t dv) { return H * ((dv + kWalkCols - 1) / kWalkCols); }
inline WalkShape walk_shape(int64_t T, int64_t S, int64_t H, int64_t G, int64_t dv, int mode) {
  const int64_t units = walk_units(H, dv), chunks = T / kScanChunk * units, busy = S * units;
  const bool wide = busy >= 512 && chunks >= 1536 ? true : chunks >= 5120 && (busy > 256 || (busy < 192 && units >= 32));
  if (mode < kModeDelta && wide) {
    if (dv > kWalkCols) return {8, 1, 2 * kWalkCols};
    if (mode == kModeStateSpace && H / G % 2 == 0) return {8, 2, kWalkCols};
  }
  return {4, 1, kWalkCols};
}
struct ScanSegments {
  int64_t chunks, states;   // states: an upper bound of the cut portions' segments, 0: no portion can be cut
};
// Chunks per segment of a portion of n chunks.  The number of segments is rounded down (from 3 / 4 on up), so that
// they do not fill the chip one time and a bit.
__host__ __device__ inline int scan_segment_chunks(int n, int chunks) {
  const int P = (4 * n + chunks) / (4 * chunks);
  return P < 2 ? (n > 0 ? n : 1) : (n + P - 1) / P;
}
inline ScanSegments scan_segments(int64_t T, int64_t S, int64_t H, int64_t G, int64_t dk, int64_t dv, int mode) {
  const int64_t n = T / kScanChunk, units = walk_units(H, dv);
  // As many units as run at once, or twice as many for a long prompt in workgroups of 64 columns where these fill the chip
  // better so (units that do not divide 256: 96 heads of 64, one prompt of 2048, twice / once: retention 196 / 217, forget
  // gate 240 / 264, state space 157 / 180 us) or fit on a CU twice (the forget gate's with keys of up to 64: 64 heads of
  // 64, one prompt of 2048 86 / 95, 2 x 1000 84 / 93; retention, that do not, 107 / 95).
  const int64_t busy = S * units;
  const bool wide = walk_shape(T, S, H, G, dv, mode).tiles == 8;
  const bool fits = 512 / units * 10 > 256 / units * 24 || (mode == kModeForget && dk <= 64);
  const int64_t all = wide || (fits && n * units >= 5120 && (busy < 192 || busy > 256)) ? 512 : 256;
  int64_t chunks = (n * units + all - 1) / all;
  if (chunks < 7) chunks = 7;
  if (chunks < (n + 15) / 16) chunks = (n + 15) / 16;
  // (one prompt of 300 rows or less gains nothing: 8 heads, forget gate 51 / 51; find_segment cuts by the lengths)
  if (mode >= kModeDelta || n + 1 < 20 || 4 * (n + 1) < 7 * chunks) return {0, 0};
  // Cut portions have m >= 1.75 `chunks` of them, so at least 13, and at most m / chunks + 1 / 4 <= 8 / 7 m / chunks
  // segments; m is the rows' 16ths rounded up, at most 13 / 12.06 of them: 8 / 7 x 13 / 12.06 < 5 / 4.
  return {chunks, 5 * (n + 1) / (4 * chunks) + 2};
}
constexpr int64_t scan_segment_floats(int64_t H, int64_t dk, int64_t dv) { return H * (dk * dv + 128); }
// floats of scratch: the records, then the segments
inline int64_t scan_scratch_floats(int64_t T, int64_t S, int64_t H, int64_t G, int64_t dk, int64_t dv, int mode) {
  return scan_chunk_slots(T, S) * H * scan_record_floats(mode, static_cast<int>(dk)) +
         scan_segments(T, S, H, G, dk, dv, mode).states * scan_segment_floats(H, dk, dv);
}

// Which kernels take a batch.  The host knows its T rows and S portions; if every portion has a row, the longest has at
// most T - S + 1.  All at 32 heads of 128, bf16, us; "R + N" R decode rows beside a portion of N, "S x N" S portions.
// - Rows (step_scan.h) cost the state's traffic and then 1 us per token of the longest portion, 2 us with a delta rule.
// - Chunks cost 15 us (25 with per-channel decays) besides the state's traffic, then 1.7 us per 16 tokens: they pay from
//   7 - 28 rows on, a sixth of a row later per portion (decode rows share the scores' launch).  Rows / chunks: delta rule
//   15 + 8 25 / 27, 15 + 32 75 / 26, 63 + 32 106 / 60; per channel 15 + 16 42 / 33, 63 + 32 105 / 68; forget gate
//   15 + 24 33 / 37, 15 + 32 45 / 31; state space 7 + 16 26 / 14; retention 15 + 16 28 / 22, 127 + 256 437 / 129.
// - Tokens (delta_rule.hip, linear_scan.hip) load a round of tokens ahead, 0.3 - 0.7 us per token, but with slower state
//   accesses: for short portions whose workgroups find room at once.  Rows / chunks / tokens: forget gate 1 x 33
//   36 / 33 / 21, 4 x 16 22 / 30 / 20; per channel 1 x 12 27 / 28 / 18, 2 x 16 35 / 28 / 20; state space 1 x 9
//   14 / 12 / 9, 2 x 16 22 / 13 / 11.  A long portion among decode rows must not be taken for many short ones, hence
//   the bounds on T - S.  Keys wider than a chunk's: for anything but a few rows per portion.
// In a chunked batch, portions below kScanMinRows run token by token: a chunk that is not full costs as much as one that
// is, and with portions in many heads the row kernel's tokens overlap: 16 x 8, rows / chunks: forget gate 24 / 67, per
// channel 36 / 67, retention 21 / 46.
enum ScanRoute { kScanRows, kScanChunks, kScanTokens };
constexpr int kScanMinRows[] = {12, 28, 9, 7, 12};   // by ScanMode
inline ScanRoute scan_route(int64_t T, int64_t S, int64_t H, int64_t dk, int64_t dv, int mode) {
  const int64_t longest = T - S + 1;
  if (dk > 128) return mode != kModeRetention && T > 3 * S ? kScanTokens : kScanRows;
  if (S * H * ((dv + 31) / 32) <= 512) {
    if (mode == kModeForget && (T > 3 * S || longest >= 12) && T < 96 * S && T - S < 256) return kScanTokens;
    if (mode == kModeStateSpace && longest >= 5 && T < 24 * S && T - S < 31) return kScanTokens;
    if (mode == kModeDeltaChannel && longest >= 6 && T < 32 * S && T - S < 48) return kScanTokens;
  }
  return longest >= kScanMinRows[mode] + S / 6 ? kScanChunks : kScanRows;
}
// gx workgroups for each of n portions: launch(grid, first portion).  A grid's y ends at 65535, portions do not.
template <typename F>
inline void scan_grids(unsigned gx, int64_t n, F launch) {
  for (int64_t y = 0; y < n; y += 65535)
    launch(dim3(gx, static_cast<unsigned>(n - y < 65535 ? n - y : 65535)), static_cast<int>(y));
}

// A batch with scratch (a.rec, a.n_slots, a.seg): portions of kScanMinRows rows or more in chunks, the others token by
// token (dk <= 128).
int launch_chunk_scan(const ChunkArgs& a, int mode, int dtype, hipStream_t st);
// Portions of up to max_rows rows, token by token (dk <= 256).
int launch_step_scan(const ChunkArgs& a, int mode, int max_rows, int dtype, hipStream_t st);
// A batch on the route kScanChunks (with scratch for it) or kScanRows.
inline int launch_scan_batch(ChunkArgs a, int mode, int64_t T, int dtype, hipStream_t st) {
  // (the chunk kernels address the 16 rows of a chunk with 32 bits)
  const int64_t strides[] = {a.q_stride, a.k_stride, a.v_stride, a.dec_stride, static_cast<int64_t>(a.H) * a.dv};
  for (const int64_t x : strides)
    if (x >= 1ll << 26) a.rec = nullptr;
  if (a.rec == nullptr) return launch_step_scan(a, mode, 1 << 30, dtype, st);
  a.T = T;
  a.n_slots = static_cast<int>(scan_chunk_slots(T, a.S));
  a.min_rows = kScanMinRows[mode];
  const ScanSegments g = scan_segments(T, a.S, a.H, a.G, a.dk, a.dv, mode);
  a.seg = a.rec + static_cast<int64_t>(a.n_slots) * a.H * scan_record_floats(mode, a.dk);
  a.seg_chunks = static_cast<int>(g.chunks);
  a.seg_states = static_cast<int>(g.states);
  return launch_chunk_scan(a, mode, dtype, st);
}

}  // namespace mixk
