// Attention with changed scores for steps of single tokens, bfloat16 pages, on the matrix cores, weights and sums in 32-bit:
// the same changes and results as the vector units' kernel (attention_generic.hip lists them), sizes of up to 128 in steps of
// 16, pages of 1 to 16 tiles of 16 keys.
//
// A workgroup takes one (entry, kv head, 16 of its query heads, split); its four waves take the visible tiles of 16 keys in
// turn, each with an online softmax of its own, merged through LDS. S = K Q^T and O^T = V^T P^T (v_mfma_f32_16x16x16_bf16): lane
// (col, grp) holds the scores of head `col` with keys 4 grp .. + 3, which are the operand of the second product as they stand.
// A weight is not rounded: it goes into the second product as the three bfloat16 values that add up to its 24 bits, three
// products for one (there is little else for the matrix cores to do here). Its bits are cut into three, none of them negative and,
// where the rest is none, 2^-32 of the weight instead: an infinite value then stays infinite and makes no NaN of its own.
//
// What bounds it: the chain of trips to memory (table entry, keys and values) of a wave's pairs of tiles, of which two are on
// their way at a time, and fetching its own instructions: every launch finds the instruction cache cold, so the code is
// kept short (one multiplication finds a tile's page, the penalty is a kernel of its own, results leave by way of LDS: together
// 7.8 -> 6.7 us a call). On the vector units a lane reads a key's whole row alone and every weight passes through LDS. Us a call,
// merges with them, before -> now: 4 requests of 32 heads of 64 on 8, 256 keys 15.0 -> 6.7, 1,024 keys 21.8 -> 9.3, 16,384 keys
// 44.1 -> 29.6 (4.5 TB/s); 64 such requests of 1,024 keys 41.5 -> 26.4, of 16,384 keys 581 -> 360 (6.0 TB/s); 8 requests of 16
// heads of 128 on 2, 1,024 keys 29.6 -> 12.8.
#include "attention_singles.h"

typedef short as_s4 __attribute__((ext_vector_type(4)));
typedef float as_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float as_column_max(float v) {   // over the four lanes that share a column
  return max_across32(max_across16(v));
}

template <int DCH, int VCH, bool PEN>   // keys of up to 16 DCH components, values of up to 16 VCH; with r1 and r2
__global__ __launch_bounds__(256) void attention_singles_kernel(SinglesArgs a) {
  constexpr float LOG2E = 1.4426950408889634f, LN2 = 0.6931471805599453f;
  __shared__ __attribute__((aligned(16))) float sm_o[4][16][16 * VCH + 4];
  __shared__ float sm_m[4][16], sm_l[4][16];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), col = lane % 16, grp = lane / 16;
  // (quotients by numbers that the compiler does not know cost some twenty instructions each before the first key is asked for:
  // the host makes them, and what is one in most calls is not divided by)
  const int entry = a.splits == 1 ? blockIdx.x : blockIdx.x / a.splits, split = blockIdx.x - entry * a.splits;
  const int group = a.group, head_tiles = a.head_tiles;
  const int kvh = head_tiles == 1 ? blockIdx.y : blockIdx.y / head_tiles, head_tile = blockIdx.y - kvh * head_tiles;
  const int vh = a.v_heads == a.kv_heads ? kvh : kvh % a.v_heads, in_group = head_tile * 16 + col;
  const bool valid = in_group < group;
  const int head = kvh * group + min(in_group, group - 1), nd = a.D / 16, nv = a.V / 16, ps = a.page_size;
  const int pos = a.kv_len[entry] - 1;
  const int* table = a.block_tables + (int64_t)entry * a.table_stride;

  as_s4 fq[DCH];
  const bf16_t* qr = a.q + (int64_t)entry * a.q_stride + (int64_t)head * a.D + 4 * grp;
#pragma unroll
  for (int c = 0; c < DCH; ++c) {   // (components past the last: zero, so that whatever stands in for a key's there counts nothing)
    const as_s4 x = *reinterpret_cast<const as_s4*>(qr + 16 * min(c, nd - 1));
    fq[c] = c < nd && valid ? x : as_s4{0, 0, 0, 0};
  }
  // scores, reference points and sinks in units of log 2
  const float scale = a.scale * LOG2E;
  const float r1 = PEN ? a.r1[head] * LOG2E : 0.f, r2 = PEN ? a.r2[head] : 0.f;
  const bool sink = (a.sinks != nullptr || a.sink) && split == 0 && wave == 0;   // counted once
  float m = sink ? (a.sinks != nullptr ? a.sinks[head] * LOG2E : 0.f) : -INFINITY;
  float l = sink && grp == 0 ? 1.f : 0.f;                                        // (lane by lane until the end)
  as_f4 acc[VCH];
#pragma unroll
  for (int c = 0; c < VCH; ++c) acc[c] = as_f4{0.f, 0.f, 0.f, 0.f};

  const int j_lo = a.chunk > 0 && pos >= a.chunk ? pos / a.chunk * a.chunk : 0;   // nothing before it is seen
  const int j_begin = a.window > 0 ? max(j_lo, pos - a.window + 1) : j_lo;
  const int keep = a.window > 0 ? a.keep_first : 0;                              // keys below it are seen from any distance
  // the tiles that hold something visible: those of the kept keys that lie before the window's, then the window's
  const int t_win = j_begin / 16, n_keep = keep > j_lo ? max(min((keep + 15) / 16, t_win) - j_lo / 16, 0) : 0;
  const int n_all = pos >= 0 ? n_keep + pos / 16 - t_win + 1 : 0;
  const int stride = 8 * a.splits;
  const auto seen = [&](int j) { return j <= pos && j >= j_lo && (j >= j_begin || j < keep); };
  const auto first_key = [&](int b) { return (b < n_keep ? j_lo / 16 + b : t_win + b - n_keep) * 16; };
  struct Pair { as_s4 k[2][DCH], v[2][VCH]; };
  struct Place { int page[2], off[2]; };
  const unsigned lane_k = col * a.D + 4 * grp, lane_v = col * ps + 4 * grp;
  const auto look = [&](int b) {   // (a page that a window has passed: any page, its keys are not seen)
    Place at;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int tile = first_key(min(b + u, n_all - 1)) / 16, nth = (int)a.page_of.page((unsigned)tile);
      at.page[u] = __builtin_amdgcn_readfirstlane(max(table[min(nth, a.table_stride - 1)], 0));
      at.off[u] = (tile - nth * (int)a.page_of.tiles) * 16;
    }
    return at;
  };
  const auto fetch = [&](Pair& t, const Place& at) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bf16_t* kr = a.k_pages + (((int64_t)at.page[u] * a.kv_heads + kvh) * ps + at.off[u]) * a.D;
      const bf16_t* vr = a.v_pages + ((int64_t)at.page[u] * a.v_heads + vh) * a.V * ps + at.off[u];
#pragma unroll
      for (int c = 0; c < DCH; ++c) t.k[u][c] = *reinterpret_cast<const as_s4*>(kr + 16 * min(c, nd - 1) + lane_k);
#pragma unroll
      for (int c = 0; c < VCH; ++c) t.v[u][c] = *reinterpret_cast<const as_s4*>(vr + 16 * min(c, nv - 1) * ps + lane_v);
    }
  };
  const auto attend = [&](Pair& t, int b) {
    if (b >= n_all) return;
    as_f4 s[2];
    float top = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s[u] = as_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < DCH; ++c) s[u] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(t.k[u][c], fq[c], s[u], 0, 0, 0);
      s[u] *= scale;
      const int first = first_key(min(b + u, n_all - 1)), j0 = first + 4 * grp;
      if constexpr (PEN)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[u][i] -= r1 * log1pf(r2 * (float)(pos - j0 - i));
      if (b + u >= n_all || first < j_begin || first + 15 > pos) {   // not every key is seen; what no one may have written
#pragma unroll                                                       // weighs nothing as it stands
        for (int i = 0; i < 4; ++i) {
          const bool counts = b + u < n_all && seen(j0 + i);
          s[u][i] = counts ? s[u][i] : -INFINITY;
#pragma unroll
          for (int c = 0; c < VCH; ++c) t.v[u][c][i] = counts ? t.v[u][c][i] : (short)0;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) top = fmaxf(top, s[u][i]);
    }
    const float m_new = fmaxf(m, as_column_max(top)), m_safe = m_new > -INFINITY ? m_new : 0.f;
    const float alpha = __builtin_amdgcn_exp2f(m - m_safe);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int c = 0; c < VCH; ++c) acc[c] *= alpha;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      as_s4 part[3];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = __builtin_amdgcn_exp2f(s[u][i] - m_safe);
        const float least = p * 0x1p-32f;
        float part_of = p;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const unsigned bits = __builtin_bit_cast(unsigned, part_of) & 0xffff0000u;
          part[k][i] = (short)(bits >> 16);
          part_of = fmaxf(part_of - __builtin_bit_cast(float, bits), least);
        }
        l += p;
      }
#pragma unroll
      for (int k = 2; k >= 0; --k)   // the smallest first
#pragma unroll
        for (int c = 0; c < VCH; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(t.v[u][c], part[k], acc[c], 0, 0, 0);
    }
  };
  int b = 2 * (split * 4 + wave);
  if (b < n_all) {   // two sets of registers take turns; the pages of the pairs behind them have been asked for
    Pair t0, t1;
    Place p0 = look(b), p1 = look(b + stride);
    fetch(t0, p0);
    fetch(t1, p1);
    p0 = look(b + 2 * stride);
    p1 = look(b + 3 * stride);
    for (; b < n_all; b += 2 * stride) {
      attend(t0, b);
      fetch(t0, p0);
      p0 = look(b + 4 * stride);
      attend(t1, b + stride);
      fetch(t1, p1);
      p1 = look(b + 5 * stride);
    }
  }
  l = add_across32(add_across16(l));
  if (grp == 0) {
    sm_m[wave][col] = m;
    sm_l[wave][col] = l;
  }
#pragma unroll
  for (int c = 0; c < VCH; ++c) *reinterpret_cast<as_f4*>(&sm_o[wave][col][16 * c + 4 * grp]) = acc[c];
  __syncthreads();
  // four neighbouring values of a head a thread
  const int quads = a.V / 4, heads = min(16, group - head_tile * 16);
  for (int idx = threadIdx.x; idx < heads * quads; idx += 256) {
    const int h = idx / quads, v0 = idx % quads * 4, out_head = kvh * group + head_tile * 16 + h;
    float top = sm_m[0][h], sum = 0.f;
#pragma unroll
    for (int w = 1; w < 4; ++w) top = fmaxf(top, sm_m[w][h]);
    const float safe = top > -INFINITY ? top : 0.f;
    as_f4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = __builtin_amdgcn_exp2f(sm_m[w][h] - safe);
      sum += sm_l[w][h] * f;
      o += *reinterpret_cast<const as_f4*>(&sm_o[w][h][v0]) * f;
    }
    if (a.splits > 1) {   // this workgroup's share: the sum as it is, its reference point and denominator behind it
      float* part = a.parts + (((int64_t)entry * a.q_heads + out_head) * a.splits + split) * (a.V + 2);
#pragma unroll
      for (int i = 0; i < 4; ++i) part[v0 + i] = o[i];
      if (v0 == 0) {
        part[a.V] = top * LN2;
        part[a.V + 1] = sum;
      }
      continue;
    }
    o *= sum > 0.f ? 1.f / sum : 0.f;
    const int64_t at = (int64_t)out_head * a.V + v0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (a.gate != nullptr) o[i] *= 1.f / (1.f + expf(-a.gate[(int64_t)entry * a.gate_stride + at + i]));
      if (a.out32 != nullptr) a.out32[(int64_t)entry * a.out_stride + at + i] = o[i];
      else a.out[(int64_t)entry * a.out_stride + at + i] = (bf16_t)o[i];
    }
  }
}

bool attention_singles_takes(const void* q, int64_t q_stride, const void* k_pages, const void* v_pages, int head_dim, int value_dim,
                             int page_size) {
  return head_dim % 16 == 0 && head_dim <= 128 && value_dim % 16 == 0 && value_dim <= 128 && page_size % 16 == 0 && page_size <= 256 && q_stride % 4 == 0 &&
         (((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) % 8) == 0;
}

// Few workgroups and many keys: the keys are cut, one run for each 128 up to a workgroup a compute unit, one for each 512 up to
// two. (us a call with 1, 4, 8 and 16 runs, the merge of the shares with them: 4 requests, 32 heads of 64 on 8, 256 keys 6.7, 8.9,
// 8.9, 12.5; 1,024 keys 13.7, 9.6, 9.3, 12.7; 4,096 keys 40.1, 17.3, 13.4, 14.3. 16 heads of 32 on 16, 4,096 keys 30.2, 14.5,
// 12.3, 13.0.) Below 512 keys one workgroup is as fast as the merge.
int attention_singles_splits(int q_heads, int kv_heads, int entries, int64_t most_keys) {
  const int64_t workgroups = (int64_t)entries * kv_heads * ((q_heads / kv_heads + 15) / 16);
  if (most_keys < 512) return 1;
  const auto least = [](int64_t x, int64_t y) { return x < y ? x : y; };
  const int64_t one = least(most_keys / 128, 256 / workgroups), two = least(most_keys / 512, 512 / workgroups);
  const int64_t splits = least(one > two ? one : two, 16);
  return splits < 1 ? 1 : (int)splits;
}

template <int DCH, int VCH>
static void launch_singles(const SinglesArgs& a, const dim3& grid, hipStream_t stream) {
  if (a.r1 != nullptr) attention_singles_kernel<DCH, VCH, true><<<grid, 256, 0, stream>>>(a);
  else attention_singles_kernel<DCH, VCH, false><<<grid, 256, 0, stream>>>(a);
}

template <int DCH>
static void launch_singles(const SinglesArgs& a, const dim3& grid, hipStream_t stream) {
  if (a.V <= 32) launch_singles<DCH, 2>(a, grid, stream);
  else if (a.V <= 64) launch_singles<DCH, 4>(a, grid, stream);
  else launch_singles<DCH, 8>(a, grid, stream);
}

int attention_singles(const SinglesArgs& a, int entries, hipStream_t stream) {
  const dim3 grid(entries * a.splits, a.kv_heads * a.head_tiles);
  if (grid.y > 65535) return DLI_ERR_ARGUMENT;
  if (a.D <= 32) launch_singles<2>(a, grid, stream);
  else if (a.D <= 64) launch_singles<4>(a, grid, stream);
  else launch_singles<8>(a, grid, stream);
  return dli_launch_status();
}
