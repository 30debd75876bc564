// The matrix cores' attention with changed scores for steps of single tokens (attention_singles.hip), for the entry point
// that chooses between it and the vector units.
#pragma once
#include "common.h"

struct SinglesArgs {
  const bf16_t* q; int64_t q_stride;
  const bf16_t *k_pages, *v_pages;             // [pages][kv_heads][page_size][D], [pages][v_heads][V][page_size]
  bf16_t* out; float* out32; int64_t out_stride;
  const int *kv_len, *block_tables; int table_stride;
  int q_heads, kv_heads, v_heads, D, V, page_size;
  float scale; int window, chunk, keep_first, sink;
  const float *r1, *r2, *sinks, *gate; int64_t gate_stride;
  float* parts; int splits;                    // splits > 1: [entries][q_heads][splits][V + 2], to be merged
  int group, head_tiles; PageOf page_of;       // q_heads / kv_heads, its tiles of 16, the page of a tile of 16 keys
};

bool attention_singles_takes(const void* q, int64_t q_stride, const void* k_pages, const void* v_pages, int head_dim, int value_dim,
                             int page_size);
// Over how many workgroups an entry's keys are cut, of which at most `most_keys` are seen.
int attention_singles_splits(int q_heads, int kv_heads, int entries, int64_t most_keys);
int attention_singles(const SinglesArgs& a, int entries, hipStream_t stream);
