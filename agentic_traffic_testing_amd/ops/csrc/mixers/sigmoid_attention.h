// Arguments of the sigmoid attention's kernels.
#pragma once
#include "mix_common.h"

namespace mixk {

constexpr int kSgTile = 64;     // query tokens per entry of the host's tile list
constexpr int kSgPart = 64;     // keys per decode partition

struct SigArgs {
  const int* block_tables;
  const int* seq_kvlen;
  const int* seq_qstart;
  const int* tile_seq;
  const int* tile_qoff;
  float* part;          // decode partials [S, H, max_parts, vdim]
  const float* bias;    // [H]
  const float* talk;    // [H, H]
  int bt_width, H, G, dim, vdim, block_size, bs_shift, max_parts, rows;
  float scale, cap;
  float* split_out;     // prefill split over the keys: fp32 partial rows [split, T, H, vdim]
  int split, total_rows;   // split: most shares
  int room;                // query tiles that take as long together as one alone
};

// Prompts and decode partitions in 32 bits on the matrix cores (sigmoid_float.hip); false: not these shapes.
bool launch_sigmoid_float(void* out, const void* q, const void* k_cache, const void* v_cache, const SigArgs& a,
                          int num_tiles, int num_decode, int parts, hipStream_t st);

}  // namespace mixk
