// Paged causal attention of the true 32-bit path on the matrix cores' 32-bit form (v_mfma_f32_16x16x4_f32: IEEE
// single-precision products and sums): heads of 64 or 128, pages of whole blocks of 16 keys, portions of prompts
// and single tokens alike. Everything else takes the vector units (attention_generic.hip).
//
// A workgroup takes 16 consecutive queries of one request and one query head. Its eight waves take the request's blocks
// of 16 keys in turn (block b is wave b % 8's, so a row's result does not depend on the tile that it falls in) and
// keep an online softmax each; the eight are merged through LDS at the end. In a block a wave makes K Q^T, so that
// lane (i, g) holds the scores of query i with keys 4 g .. + 3, its own queries' maximum is two exchanges away, and these
// four registers are at once the operand of V^T P^T (step s of four takes key 4 g + s): no weight passes through LDS,
// and every load brings 16 bytes a lane straight from a page.
//
// What bounds it: the loads of K and V by 16 rows a wave (four neighbouring lanes lie in four rows, a quarter of the
// caches' rate), ahead of the matrix cores; at few queries the chain of load, scores, exponentials and sums per block.
// Measured at SmolLM2-135M's sizes (9 heads of 64 on 3), mean of one step with prompts of 333 and 178 tokens and four steps
// of two single tokens over them: 12.2 us a layer, against 183 on the vector units (a workgroup of 32 queries and one
// head walks all keys alone, and single tokens leave 31 of 32 queries idle). Over the range it takes, us on the vector units
// and here: prompts of 17, 128, 512, 2,048 and 8,192 tokens, 9 heads of 64 on 3, 18 and 15, 53 and 21, 187 and 23, 821
// and 112, 5,996 and 1,075; 24 heads of 128 on 8, 4,096 tokens 9,413 and 1,607; one token on 64, 4,096 and 16,384 keys 38 and
// 9, 1,667 and 77, 7,227 and 281; 64 tokens on 2,048 keys each, 32 heads of 64 on 8, 2,488 and 479; a window of 256
// over 2,048 tokens 130 and 37.
#include "attention_f32.h"

typedef float af4 __attribute__((ext_vector_type(4)));
#define AF_WAVES 8

template <int DT>   // head size in 16s
__global__ __launch_bounds__(64 * AF_WAVES) void attention_f32_kernel(
    const float* __restrict__ q, int64_t q_stride, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
    float* __restrict__ out, int64_t out_stride, const int* __restrict__ q_start, const int* __restrict__ kv_len,
    const int* __restrict__ block_tables, int table_stride, const int* __restrict__ tile_entry, const int* __restrict__ tile_q0,
    int per_tile, int group, int kv_heads, int page_size, PageOf page_of_tile, float scale, int window) {
  constexpr int D = 16 * DT;
  __shared__ af4 accs[AF_WAVES][DT][64];
  __shared__ float ms[AF_WAVES][16], ls[AF_WAVES][16];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), i = lane % 16, g = lane / 16;
  const int tile = blockIdx.x / per_tile, entry = tile_entry[tile], head = blockIdx.y, kvh = head / group;
  const int q0 = tile_q0[tile] + blockIdx.x % per_tile * 16;
  const int tok0 = q_start[entry], q_len = q_start[entry + 1] - tok0;
  if (q0 >= q_len) return;   // (the list's tiles are 16 * per_tile queries high)
  const int rows = min(16, q_len - q0), first_pos = kv_len[entry] - q_len + q0;
  const int pos = first_pos + min(i, rows - 1);   // rows past the end repeat the last one and are not stored
  const int* table = block_tables + (int64_t)entry * table_stride;

  af4 fq[DT], acc[DT];
  const float* qr = q + (int64_t)(tok0 + q0 + min(i, rows - 1)) * q_stride + (int64_t)head * D + 4 * g;
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    fq[t] = *reinterpret_cast<const af4*>(qr + 16 * t) * scale;
    acc[t] = af4{0.f, 0.f, 0.f, 0.f};
  }
  float m = -INFINITY, l = 0.f;   // (the sum: of this lane's keys alone until the end)
  const int b_end = (first_pos + rows + 15) / 16;   // blocks that some query sees
  int b = window > 0 ? max(0, first_pos - window + 1) / 16 : 0;
  b += (wave - b % AF_WAVES + AF_WAVES) % AF_WAVES;
  // Block b's page is looked up two turns ahead and its keys are asked for one turn ahead, on the scalar unit where they are
  // the same for all lanes: a turn then waits for no table entry. (A block past the last reads the last one's page.)
  const int b_last = max(b_end - 1, 0);
  struct Where {
    int64_t page;   // (a page that a window has passed: any page, its keys are not seen)
    int off;        // the block's first key in it
  };
  const auto look_up = [&](int block) {
    const unsigned t = (unsigned)min(block, b_last), page = page_of_tile.page(t);
    return Where{(int64_t)max(table[page], 0) * kv_heads + kvh, (int)(t - page * page_of_tile.tiles) * 16};
  };
  af4 fk[DT];
  const auto load_keys = [&](const Where& at) {
    const float* kr = k_pages + (at.page * page_size + at.off) * D;
#pragma unroll
    for (int t = 0; t < DT; ++t) fk[t] = *reinterpret_cast<const af4*>(kr + i * D + 4 * g + 16 * t);
  };
  Where here{0, 0}, next{0, 0};
  if (b < b_end) {
    here = look_up(b);
    next = look_up(b + AF_WAVES);
    load_keys(here);
  }
  for (; b < b_end; b += AF_WAVES) {
    const int j0 = b * 16 + 4 * g;
    af4 fv[DT];
    const float* vr = v_pages + here.page * D * page_size + here.off;
#pragma unroll
    for (int t = 0; t < DT; ++t) fv[t] = *reinterpret_cast<const af4*>(vr + (i + 16 * t) * page_size + 4 * g);
    const Where after = look_up(b + 2 * AF_WAVES);
    // two sums side by side: a chain of products waits for itself
    af4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < DT; t += 2)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(fk[t][e], fq[t][e], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(fk[t + 1][e], fq[t + 1][e], s1, 0, 0, 0);
      }
    if (b + AF_WAVES < b_end) load_keys(next);
    here = next;
    next = after;
    af4 s = s0 + s1;
    float top = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool seen = j0 + e <= pos && (window <= 0 || j0 + e > pos - window);
      s[e] = seen ? s[e] : -INFINITY;
      top = fmaxf(top, s[e]);
    }
    top = max_across32(max_across16(top));
    const float m_new = fmaxf(m, top);
    float alpha = 1.f;
    af4 p = {0.f, 0.f, 0.f, 0.f};
    if (m_new > -INFINITY) {
      alpha = expf(m - m_new);
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = expf(s[e] - m_new);
    }
    if (b * 16 + 16 > first_pos + rows) {   // the last block: past its keys lies what no request may have written
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) fv[t][e] = j0 + e < first_pos + rows ? fv[t][e] : 0.f;
    }
    l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
    m = m_new;
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] *= alpha;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < DT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(fv[t][e], p[e], acc[t], 0, 0, 0);
  }
  l = add_across32(add_across16(l));
  if (g == 0) {
    ms[wave][i] = m;
    ls[wave][i] = l;
  }
#pragma unroll
  for (int t = 0; t < DT; ++t) accs[wave][t][lane] = acc[t];
  __syncthreads();
  if (wave >= DT) return;
  float top = -INFINITY, total = 0.f, w[AF_WAVES], m_c[AF_WAVES], l_c[AF_WAVES];
#pragma unroll
  for (int c = 0; c < AF_WAVES; ++c) {   // (all read before the first is used)
    m_c[c] = ms[c][i];
    l_c[c] = ls[c][i];
  }
#pragma unroll
  for (int c = 0; c < AF_WAVES; ++c) top = fmaxf(top, m_c[c]);
#pragma unroll
  for (int c = 0; c < AF_WAVES; ++c) {
    w[c] = m_c[c] > -INFINITY ? expf(m_c[c] - top) : 0.f;
    total += l_c[c] * w[c];
  }
  const float inv = total > 0.f ? 1.f / total : 0.f;
  for (int t = wave; t < DT; t += AF_WAVES) {
    af4 sum = {0.f, 0.f, 0.f, 0.f}, part[AF_WAVES];
#pragma unroll
    for (int c = 0; c < AF_WAVES; ++c) part[c] = accs[c][t][lane];
#pragma unroll
    for (int c = 0; c < AF_WAVES; ++c) sum += part[c] * w[c];
    if (i < rows)
      *reinterpret_cast<af4*>(out + (int64_t)(tok0 + q0 + i) * out_stride + (int64_t)head * D + 16 * t + 4 * g) = sum * inv;
  }
}

extern "C" int dli_attention_f32_supports(int head_dim, int page_size) {
  return (head_dim == 64 || head_dim == 128) && page_size > 0 && page_size % 16 == 0;
}

bool attention_f32_takes(const void* q, int64_t q_stride, const void* k_pages, const void* v_pages, const void* out,
                         int64_t out_stride, int head_dim, int page_size) {
  return dli_attention_f32_supports(head_dim, page_size) && q_stride % 4 == 0 && out_stride % 4 == 0 &&
         (((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages | (uintptr_t)out) % 16) == 0;
}

int attention_f32(const float* q, int64_t q_stride, const float* k_pages, const float* v_pages, float* out, int64_t out_stride,
                  const int* q_start, const int* kv_len, const int* block_tables, int table_stride, const int* tile_entry,
                  const int* tile_q0, int tiles, int tile_rows, int q_heads, int kv_heads, int head_dim, int page_size,
                  float scale, int window, hipStream_t stream) {
  const int per_tile = (tile_rows + 15) / 16;
  const dim3 grid(tiles * per_tile, q_heads);
#define AF_LAUNCH(DT)                                                                                               \
  attention_f32_kernel<DT><<<grid, 64 * AF_WAVES, 0, stream>>>(q, q_stride, k_pages, v_pages, out, out_stride, q_start, kv_len, \
      block_tables, table_stride, tile_entry, tile_q0, per_tile, q_heads / kv_heads, kv_heads, page_size, page_of_tile(page_size), scale, window)
  if (head_dim == 64) AF_LAUNCH(4);
  else AF_LAUNCH(8);
#undef AF_LAUNCH
  return dli_launch_status();
}
