// The matrix cores' attention of the 32-bit path (attention_f32.hip), for the entry point that chooses between it and
// the vector units.
#pragma once
#include "common.h"

// Whether it takes these heads, pages and rows (16-byte loads and stores).
bool attention_f32_takes(const void* q, int64_t q_stride, const void* k_pages, const void* v_pages, const void* out,
                         int64_t out_stride, int head_dim, int page_size);
// `tile_rows`: the height of the list's tiles.
int attention_f32(const float* q, int64_t q_stride, const float* k_pages, const float* v_pages, float* out, int64_t out_stride,
                  const int* q_start, const int* kv_len, const int* block_tables, int table_stride, const int* tile_entry,
                  const int* tile_q0, int tiles, int tile_rows, int q_heads, int kv_heads, int head_dim, int page_size,
                  float scale, int window, hipStream_t stream);
