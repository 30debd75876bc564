// The product kernel for results of about one tile a compute unit (tile_gemm.hip), for gemm_lt.hip.
#pragma once
#include "common.h"

bool tile_gemm_takes(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* out, int64_t ldo, int64_t rows, int64_t feats,
                     int64_t k, bool out_f32);
int tile_gemm(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, void* out, int64_t ldo, int64_t rows,
              int64_t feats, int64_t k, bool out_f32, hipStream_t stream);
