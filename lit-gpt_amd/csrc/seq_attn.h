// The operands of the layered models' softmax attentions, and their matrix-core form for prompts (seq_attn_tiles.hip).
#pragma once

#include "seq_common.h"

namespace lgs {

struct AttnArgs {
  const float* q;  // prepared queries at q + row * ld + h * MAPS d
  long ld;
  const void* cache_k;
  const void* cache_v;
  const int *seq_start, *seq_slot, *seq_pos0;
  float* out;       // [T][H * dv]
  uint16_t* out16;  // optional bf16 copy
  float* part;      // splits > 1: [T][H][splits][MAPS (2 + dv)]
  int H, G, d, dv, S, chunk, tiles;
  float scale, cap, lambda, eps, post;
  const float* sink;  // one map: exp(sink[h]) joins the softmax normaliser (NULL: no sink)
  const float* gate;  // one map: the head's output is multiplied by sigmoid(gate[row * ldg + h]) (NULL: not)
  long ldg;
  int gate_cols;      // 1: a gate per head (above); else one per output column, gate[row * ldg + h * dv + c]
  int window;         // one map: a query sees the last `window` positions (0: all before it)
  const float *pool_k, *pool_v;  // one map: pooled blocks [slots][pool_rows][G][d], [..][dv] before the window
  int pool, pool_rows;           // (pool 0: none)
  const float* v_freq;  // one map, [dv / 2]: the finished output is turned back by the query's position (values are
  int interleaved;      // cached rotated), pairs (2m, 2m + 1) or (m, m + dv / 2)
  const float* score_bias;  // [H]: sigmoid weights, each sigmoid(score + score_bias[h]) (null: softmax)
};

// Keys and values of the matrix-core form: bf16 rows of `parts` summands each ([parts][MAPS d] and [parts][dv]; a value is
// the sum of its summands), a position's rows `krow` and `vrow` elements apart, a key head's part of them MAPS d parts
// (dv parts) elements. `packed`: position 0 of sequence b is row seq_start[b]; else row seq_slot[b] * S of a cache.
struct AttnTileArgs {
  AttnArgs a;
  const uint16_t *k, *v;
  long krow, vrow;
  int packed, heads;  // heads: query heads of one key head that a workgroup takes (1, 2 or 4)
};
// whether a prompt step (max_len tokens in its longest sequence) of these sizes takes it; launches it, 0 or an error
bool attn_tiles_fit(const AttnArgs& a, int maps, int parts, int max_len);
int attn_tiles_launch(const AttnTileArgs& p, int maps, int parts, int B, int max_len, hipStream_t stream);

}  // namespace lgs
