// Matrix product for a few rows of activations (decode): y[m][n] = sum_k xhat[m][k] * w[n][k],
// m < 64, with the work that surrounds it in a decoder layer fused in, so that a layer needs few
// launches and the weights stream from HBM exactly once.
//
// One workgroup owns 16 output features (rows n of w) for all activation rows; its waves split k
// among themselves and add up through LDS in a fixed order. Products run on the matrix cores as
//   acc[16 n x 16 m] += W[16 n x 32 k] * xhat^T[32 k x 16 m]      (v_mfma_f32_16x16x32_bf16)
// where lane l supplies row/column l%16 and eight k values. Inside a block of 128 k the lane
// group g = l/16 takes the contiguous run [32g, 32g+32) and the four products of the block use its
// four runs of eight: the same permutation of k for both operands, so the sum is unchanged and a
// lane reads 64 contiguous bytes of its weight row.
//
// TILED: the weights are stored tile by tile instead of row by row, as
//   t[tile][block][q][g][c][8] = w[16*tile + c][128*block + 32*g + 8*q + (0..7)],
// so that the 16 features x 128 k of one tile and block are 4 KB of consecutive memory in the
// order in which the lanes take them (lane = 16*g + c) and every load of a wave is 1 KB of
// consecutive bytes. Needs K % 128 == 0 and whole tiles (N % 16 == 0, gate and up parts included); EPI_QKV behind a
// norm also takes K % 32 == 0, the last block filled up with zeros.
//
// Fused in (template switches):
//   NORM     xhat = cast(norm_w[k] * cast(x[m][k] * rs[m])), rs[m] = rsqrt(sum_k x^2 / K + eps),
//            the row sums of squares being handed over in parts by the kernel that wrote x
//            (RMSNorm: src/dli/model/llama.py:40-44); otherwise xhat = x.
//   EPI_STORE     y (+ bias) stored as bf16
//   EPI_SWIGLU    two products per workgroup, rows n (gate) and n + up_offset (up) of w:
//                 stores cast(silu(gate)) * up (src/dli/model/llama.py:190), or another form (GluForm)
//   EPI_RESIDUAL  stream[m][n] = cast(stream[m][n] + cast(y + bias)) in place (the residual sum, in
//                 32-bit), and this tile's part of sum_n stream[m][n]^2 for the norm that follows
//   EPI_F32       y stored as float32 (logits)
//   EPI_QKV       the fused q/k/v projection of a decode step with what follows it: rotary
//                 rotation of the q and k heads (src/dli/model/rope.py:50-70) and the write of the
//                 rotated keys and the values into the cache pages, so that no rotation kernel
//                 runs. TILED only, and the tile order of the q and k heads is a special one: tile
//                 t of a head holds its dimensions 8t..8t+7 and half+8t..half+8t+7, i.e. eight
//                 rotary pairs, whose partners sit 32 lanes apart in the product's result. q is
//                 stored to out in the usual order; k and v go to the pages only.
//   MERGED   the activations are not read from x but made in the kernel from the split-key partial
//            results of the decode attention (o_s, m_s, l_s per request, head and run of keys):
//            x[m][head*D + d] = cast(sum_s o_s[d] 2^(m_s - M) / sum_s l_s 2^(m_s - M)), the same
//            arithmetic in the same order as attention_merge_kernel, so that the o projection of a
//            step of one to four rows needs no merge kernel before it. Each wave merges the run of
//            k that it multiplies (all loads of a lane in flight at once) and hands it to its
//            lanes through LDS. EPI_RESIDUAL, at most 16 runs. TILED, or, where K is no whole blocks of 128, in chunks:
//              t[tile][chunk][c][8] = w[16*tile + c][8*chunk + (0..7)],
//            of which a wave can take any steps of 32 k in whole lines. k is then split and summed as the product of several rows,
//            which reads such weights row by row, does it: a row alone in its step has the same bits as among others. (Row by
//            row here too, whose loads touch a line a lane: 135M sizes 5.05 ms a pass of eight steps, 360M sizes 6.46.)
#include "common.h"
#include "merge_splits.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));

enum { EPI_STORE = 0, EPI_SWIGLU = 1, EPI_RESIDUAL = 2, EPI_F32 = 3, EPI_QKV = 4 };

// What EPI_QKV needs beside the product: cos/sin of the rows' positions ([rows][2][head_dim/2]
// float32, rounded to bfloat16 values), the rows' cache slots (negative: not cached), the pages
// (K page [kv_heads][page_size][head_dim], V page [kv_heads][head_dim][page_size]) and the heads.
struct QkvRope {
  const float* angles;
  const int* slots;
  bf16_t* k_pages;
  bf16_t* v_pages;
  int q_heads, kv_heads, head_dim, page_size;
};

// What MERGED reads instead of x: part_o [rows][heads][splits][head_dim] and part_ml
// [rows][heads][splits][2] (running maximum in units of log2, sum) float32.
struct MergedIn {
  const float* part_o;
  const float* part_ml;
  int splits, heads, head_dim;
};
#define MERGE_ROWS 4     // rows of a step whose o projection merges by itself
#define MERGE_RANGE 512  // the longest run of k of one wave

__device__ __forceinline__ float4v mfma32(bf16x8 a, bf16x8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Activation fragment of eight k values: the raw loads, and the norm applied afterwards (so the
// loads can be issued a block ahead of their use).
template <bool NORM>
struct XFrag {
  bf16x8 v;
  float4v w0, w1;
};
template <>
struct XFrag<false> {
  bf16x8 v;
};

template <bool NORM>
__device__ __forceinline__ XFrag<NORM> fetch_x(const bf16_t* __restrict__ xrow,
                                               const float* __restrict__ norm_w, int k) {
  XFrag<NORM> f;
  f.v = *reinterpret_cast<const bf16x8*>(xrow + k);
  if constexpr (NORM) {
    f.w0 = *reinterpret_cast<const float4v*>(norm_w + k);
    f.w1 = *reinterpret_cast<const float4v*>(norm_w + k + 4);
  }
  return f;
}

template <bool NORM>
__device__ __forceinline__ bf16x8 finish_x(const XFrag<NORM>& f, float rs) {
  if constexpr (!NORM) {
    return f.v;
  } else {
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float normed = (float)(bf16_t)((float)f.v[i] * rs);
      v[i] = (bf16_t)((i < 4 ? f.w0[i] : f.w1[i - 4]) * normed);
    }
    return v;
  }
}

// KS waves split k, NS groups of waves split the workgroup's tiles, each wave owns NT tiles:
// a workgroup computes NS*NT tiles of 16 features with KS*NS waves. The activation fragments are
// loaded once per block of k and reused for the wave's NT tiles.
// AHEAD: up to four rows, no wave has a single block of k (two_blocks_or_none), and the second sets out with the first.
// RUNS: 0, or (MERGED) 2, 4, 8 or 16, no fewer than the runs of keys that are merged.
template <int KS, int NS, int NT, int MT, int EPI, bool NORM, bool TILED, bool AHEAD, int RUNS = 0>
__global__ __launch_bounds__(KS * NS * 64) void skinny_gemm_kernel(
    const bf16_t* __restrict__ x, int64_t ldx, const float* __restrict__ ssq_in, int ssq_parts,
    const float* __restrict__ norm_w, float eps, const bf16_t* __restrict__ w,
    const bf16_t* __restrict__ bias, void* __restrict__ out, int64_t ldo,
    bf16_t* __restrict__ stream, int64_t lds_, float* __restrict__ ssq_out, int M, int N, int K,
    int up_offset, QkvRope qr, MergedIn mi, GluForm glu) {
  constexpr bool MERGED = RUNS != 0;
  static_assert(EPI != EPI_QKV || (TILED && MT == 1), "the q/k/v epilogue reads tiled weights, at most 16 rows");
  static_assert(!MERGED || (MT == 1 && NS == 1 && NT == 1 && !NORM), "merged activations: one tile of rows and of features");
  static_assert(!AHEAD || (MT == 1 && !NORM && !MERGED), "one row tile, no sums of squares to wait for");
  static_assert(KS * NS * 64 >= 256, "a thread for each output of a tile");
  // MERGED: each wave's run of k for up to MERGE_ROWS rows
  __shared__ __align__(16) bf16_t xs[MERGED ? KS : 1][MERGED ? MERGE_ROWS : 1][MERGED ? MERGE_RANGE : 8];
  constexpr int NA = EPI == EPI_SWIGLU ? 2 : 1;  // weight row sets per tile (gate and up)
  constexpr bool PADDED = EPI == EPI_QKV;        // the weights' last block of 128 k may be filled up with zeros
  constexpr bool CHUNKS = MERGED && !TILED;      // weights in chunks of eight k, sixteen rows' chunks one behind the other
  // What follows the last product is a chain that nothing hides, so it is kept short. With one row
  // tile and one group of waves (SHORT) all waves leave their parts in LDS and thread t makes
  // output t of each tile: element t % 4 of lane t / 4 of the product's result, that is row
  // t / 4 % 16 and feature 4 (t / 64) + t % 4. Otherwise k-split waves 1.. hand their parts to wave 0. So do q, k and v,
  // which wave 0 stores four values at a time (a value a thread, 2 and 8 rows: 6.9 us for 6.4 and 6.8 for 6.7 at the 1B sizes,
  // 10.4 for 9.0 and 9.9 for 9.0 at the 1.7B sizes, 13.3 for 11.9 and 12.6 for 11.7 at the 3B sizes).
  constexpr bool SHORT = MT == 1 && NS == 1 && EPI != EPI_QKV;
  constexpr int KR = SHORT ? KS : (KS > 1 ? KS - 1 : 1);
  __shared__ float4v red[KR][NS][NT][NA][MT][64];

  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int ks = wave % KS, ns = wave / KS;
  const int col = lane % 16, grp = lane / 16;
  const int tile0 = (blockIdx.x * NS + ns) * NT;  // first of this wave's tiles

  // weight rows of this lane (clamped at the matrix's end: such rows are computed and dropped)
  const bf16_t* wrow[NT][NA];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      if constexpr (TILED) {
        // the tile's first block, at this lane's 16 bytes of a 1 KB load
        const int tile = min(tile0 + j, (N - 1) / 16) + a * (up_offset / 16);
        wrow[j][a] = w + (int64_t)tile * 16 * (PADDED ? (K + 127) / 128 * 128 : K) + lane * 8;
      } else if constexpr (CHUNKS) {
        wrow[j][a] = w + (int64_t)min(tile0 + j, (N - 1) / 16) * 16 * K + col * 8;
      } else {
        const int n = min((tile0 + j) * 16 + col, N - 1) + a * up_offset;
        wrow[j][a] = w + (int64_t)n * K + grp * 32;
      }
    }
  // (row by row a line's parts are asked for by several loads, which a line that leaves the caches first would not outlive: steps of
  // the 360M sizes with 10 requests 5% longer)
  auto load_weights = [](const bf16x8* at) __attribute__((always_inline)) {
    if constexpr (TILED || CHUNKS) return load_streamed(at);
    else return *at;
  };
  // where a lane finds its eight k values of product q in the block that starts at step s
  auto w_at = [&](const bf16_t* base, int s, int q) __attribute__((always_inline)) {
    if (CHUNKS) return reinterpret_cast<const bf16x8*>(base + (4 * (s + grp) + q) * 128);
    return reinterpret_cast<const bf16x8*>(TILED ? base + (s / 4) * 2048 + q * 512 : base + s * 32 + q * 8);
  };

  // What the end adds to the product (the stream's values, the bias) is asked for now, so that the end does not wait for a
  // trip to memory of its own. In every wave and for every element (an element past the edge reads the edge's and is not
  // stored; a missing bias is a resource without bytes, which reads zeros): a load under a
  // condition is waited for on the spot, one trip to memory after the other, and leaves the count
  // of loads on their way unknown to everything behind it.
  constexpr int EL = SHORT ? 1 : 4;  // a thread's (SHORT) or lane's elements of a tile
  const int e_row = SHORT ? threadIdx.x / 4 % 16 : col;
  const int e_grp = SHORT ? threadIdx.x / 64 % 4 : grp, e_i = SHORT ? threadIdx.x % 4 : 0;
  const int e_n = 4 * e_grp + e_i;   // first of them within the tile
  bf16_t old_s[EPI == EPI_RESIDUAL ? NT : 1][EPI == EPI_RESIDUAL ? MT : 1][EL];
  if constexpr (EPI == EPI_RESIDUAL) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < EL; ++i) {
          const int n = (tile0 + j) * 16 + e_n + i, m = t * 16 + e_row;
          old_s[j][t][i] = stream[(int64_t)min(m, M - 1) * lds_ + min(n, N - 1)];
        }
  }
  const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)bias, 0, bias != nullptr ? (unsigned)(N + (NA - 1) * up_offset) * 2u : 0u, 0x00020000);
  auto bias_at = [&](int n) __attribute__((always_inline)) {
    union {
      unsigned short raw;
      bf16_t v;
    } b;
    b.raw = __builtin_amdgcn_raw_buffer_load_b16(bres, n * 2, 0, 0);
    return b.v;
  };
  bf16_t b_at[NT][NA][EL];
  auto load_bias = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int i = 0; i < EL; ++i) b_at[j][a][i] = bias_at(min((tile0 + j) * 16 + e_n + i, N - 1) + a * up_offset);
  };
  // (several row tiles: at the end, the registers are taken; q/k/v: there as well, with what the rotation needs)
  constexpr bool EARLY = MT == 1 && EPI != EPI_QKV;
  if constexpr (EARLY) load_bias();

  const bf16_t* xrow[MT];
  float rs[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = t * 16 + col;
    xrow[t] = x + (int64_t)min(m, M - 1) * ldx;
    rs[t] = 1.f;
  }
  float4v acc[NT][NA][MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[j][a][t] = float4v{0.f, 0.f, 0.f, 0.f};

  // this wave's share of the k steps of 32
  const int steps = K / 32;
  const int whole = PADDED ? (steps + 3) / 4 : steps / 4;
  const int s_begin = TILED ? 4 * (int)((int64_t)whole * ks / KS) : (int)((int64_t)steps * ks / KS);
  const int s_end = TILED ? 4 * (int)((int64_t)whole * (ks + 1) / KS) : (int)((int64_t)steps * (ks + 1) / KS);
  int s = s_begin;
  // Blocks of 128: lane group g reads k in [32g, 32g + 32). The weights and activations of the
  // next block are asked for before the products of the current one. The two sets of registers
  // take turns in a loop that is written out for both, with the last block's products apart, so
  // that at every product the number of younger loads is known and the wait is for the block's
  // own loads alone (with one body for every turn, the turn without younger loads decides the
  // wait of all: each block was then waited for right after it had been asked for). Rows past
  // the last read the last row again (their results are dropped), so no load is conditional.
  struct Block {
    bf16x8 a[NT][NA][4];
    XFrag<NORM> x[MT][4];
  };
  auto fetch_weights = [&](Block& b, int at) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int q = 0; q < 4; ++q) b.a[j][a][q] = load_weights(w_at(wrow[j][a], at, q));
  };
  auto fetch_rows = [&](Block& b, int at) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = at * 32 + grp * 32 + q * 8;   // (past K, where the weights are zeros: the last values again)
        b.x[t][q] = fetch_x<NORM>(xrow[t], norm_w, EPI == EPI_QKV ? min(k, K - 8) : k);
      }
  };
  auto multiply = [&](const Block& b) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bf16x8 bf = finish_x<NORM>(b.x[t][q], rs[t]);
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int a = 0; a < NA; ++a) acc[j][a][t] = mfma32(b.a[j][a][q], bf, acc[j][a][t]);
      }
    }
  };
  int blocks = (s_end - s) / 4;
  Block b0, b1;
  // single steps behind the last block (not TILED): lane group g reads k in [8g, 8g + 8)
  auto w_single_at = [&](const bf16_t* base, int s) __attribute__((always_inline)) {
    return reinterpret_cast<const bf16x8*>(CHUNKS ? base + (4 * s + grp) * 128 : base - grp * 32 + s * 32 + grp * 8);
  };
  bf16x8 w_single[MERGED && !TILED ? 3 : 1];   // MERGED: asked for ahead of the merge, like the blocks
  if constexpr (NORM) {
    // rs[m] from the parts of sum x^2 that the producer of x left. The parts are dealt out to
    // all lane groups of all waves (group q of W*4 takes the parts q, q + 4W, ...), eight loads
    // at a time so that they share one trip to memory; a wave adds its four groups, the waves'
    // sums meet in LDS and are added in wave order. The first block of weights and rows is asked
    // for right behind the first eight parts and before anything waits for them, so that it is
    // on its way while the sums are made.
    constexpr int W = KS * NS;
    __shared__ float rsum[W][MT][16];
    float first[MT][8];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = min(t * 16 + col, M - 1);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        // no load is conditional (a part past the last reads the last and counts as zero), so
        // that the number of loads on their way is known where the first is waited for
        const int p = wave * 4 + grp + u * 4 * W;
        const float part = ssq_in[(int64_t)min(p, ssq_parts - 1) * M + m];
        first[t][u] = p < ssq_parts ? part : 0.f;
      }
    }
    // (a wave without a block of its own, k being short, reads the matrix's first block)
    if (TILED || blocks > 0) {
      fetch_rows(b0, blocks > 0 ? s : 0);
      fetch_weights(b0, blocks > 0 ? s : 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = min(t * 16 + col, M - 1);
      float sum = 0.f;
#pragma unroll
      for (int u = 0; u < 8; ++u) sum += first[t][u];
      for (int p0 = wave * 4 + grp + 32 * W; p0 < ssq_parts; p0 += 32 * W) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int p = p0 + u * 4 * W;
          v[u] = p < ssq_parts ? ssq_in[(int64_t)p * M + m] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += v[u];
      }
      sum = add_across32(add_across16(sum));
      if (grp == 0) rsum[wave][t][col] = sum;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      float sum = 0.f;
#pragma unroll
      for (int wv = 0; wv < W; ++wv) sum += rsum[wv][t][col];
      rs[t] = rsqrtf(sum / (float)K + eps);
    }
  } else if constexpr (!MERGED) {
    if (blocks > 0) fetch_weights(b0, s);
  }
  if constexpr (MERGED) {
    // The wave's run of k, four values a lane and turn, merged as attention_merge_kernel does. The
    // first turn's partial results are asked for before the first two blocks of weights (loads
    // come back in their order), which are on their way while the merge is made.
    const int kb0 = s_begin * 32, quads = (s_end - s_begin) * 8, items = M * quads;
    const int D = mi.head_dim, S = mi.splits;
    MergeQuad<MERGED ? RUNS : 2> parts;
    auto ask = [&](int item) __attribute__((always_inline)) {
      const int row = item / quads, k = kb0 + (item - row * quads) * 4, head = k / D;
      parts.ask(mi.part_o, mi.part_ml, ((int64_t)row * mi.heads + head) * S, S, D, k - head * D);
    };
    if (items > 0) ask(min(lane, items - 1));
    __builtin_amdgcn_sched_barrier(0);
    if (blocks > 0) fetch_weights(b0, s);
    if (blocks > 1) fetch_weights(b1, s + 4);
    if constexpr (!TILED) {
#pragma unroll
      for (int u = 0; u < 3; ++u) w_single[u] = load_weights(w_single_at(wrow[0][0], min(s + 4 * blocks + u, steps - 1)));
    }
    __builtin_amdgcn_sched_barrier(0);
    for (int item0 = 0; item0 < items; item0 += 64) {
      const int item = item0 + lane;
      if (item0 > 0) ask(min(item, items - 1));
      const float4v merged = parts.merged(S);
      if (item < items) {
        const int row = item / quads;
        bf16_t* dst = &xs[ks][row][(item - row * quads) * 4];
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[i] = (bf16_t)merged[i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) xrow[t] = &xs[ks][min(t * 16 + col, M - 1)][0] - kb0;
  }
  if constexpr (!NORM) {
    if (blocks > 0) fetch_rows(b0, s);
    if (MERGED ? blocks > 1 : AHEAD && blocks > 0) {
      fetch_rows(b1, s + 4);
      if constexpr (!MERGED) fetch_weights(b1, s + 4);
    }
  }
  if constexpr (MT > 1) {
    // several row tiles: one body for every turn (the registers do not hold two whole blocks)
    for (; s + 4 <= s_end; s += 4) {
      const bool more = s + 8 <= s_end;
      if (more) {
        fetch_weights(b1, s + 4);
        fetch_rows(b1, s + 4);
      }
      multiply(b0);
      if (more) b0 = b1;
    }
  } else if (NORM && blocks == 1) {
    multiply(b0);
    s += 4;
  } else if (blocks > 0) {
    // Where the second block is asked for, us with the first, and after what is waited for before the first product:
    //  - A wave of one block would read it twice: o, 8 rows, 3.8 and 3.2 at the 135M sizes, 1 row 4.2 and 3.7 at the 360M sizes.
    //  - With two and more and few rows it pays: o, 1 row, 4.4 and 4.6 at the 1B sizes, 5.6 and 6.0 at the 3B sizes.
    //  - With more rows not, and there a block is best asked for right before the other's products, not after them: down, 16
    //    rows, 17.5 and 16.6 at the 3B sizes; 32-bit sums of 8,192 features of 2,048, 16 rows, 12.2 and 11.4.
    //  - In front of sums of squares it stands, with rows and norm weights, in the vector cache's way: gate and up, 8 and 16
    //    rows, 6.6 and 5.2, 6.8 and 5.3 at the 135M sizes. Right after the other's products is best there: 16 rows, 15.9 at
    //    the 1B sizes, 16.9 before them.
    if constexpr (NORM || AHEAD || MERGED) {
      if constexpr (NORM) {
        fetch_rows(b1, s + 4);
        fetch_weights(b1, s + 4);
        __builtin_amdgcn_sched_barrier(0);
      }
      while (blocks >= 4) {
        multiply(b0);
        fetch_rows(b0, s + 8);
        fetch_weights(b0, s + 8);
        __builtin_amdgcn_sched_barrier(0);  // all of a block's loads leave before the other's products
        multiply(b1);
        fetch_rows(b1, s + 12);
        fetch_weights(b1, s + 12);
        __builtin_amdgcn_sched_barrier(0);
        s += 8;
        blocks -= 2;
      }
      if (blocks == 3) {
        multiply(b0);
        fetch_rows(b0, s + 8);
        fetch_weights(b0, s + 8);
        __builtin_amdgcn_sched_barrier(0);
        multiply(b1);
        multiply(b0);
      } else {
        multiply(b0);
        if (!MERGED || blocks == 2) multiply(b1);
      }
    } else {
      while (blocks >= 3) {
        fetch_rows(b1, s + 4);
        fetch_weights(b1, s + 4);
        __builtin_amdgcn_sched_barrier(0);
        multiply(b0);
        fetch_rows(b0, s + 8);
        fetch_weights(b0, s + 8);
        __builtin_amdgcn_sched_barrier(0);
        multiply(b1);
        s += 8;
        blocks -= 2;
      }
      if (blocks == 2) {
        fetch_rows(b1, s + 4);
        fetch_weights(b1, s + 4);
        __builtin_amdgcn_sched_barrier(0);
        multiply(b0);
        multiply(b1);
      } else {
        multiply(b0);
      }
    }
    s = s_begin + (s_end - s_begin) / 4 * 4;
  }
  if constexpr (MERGED && !TILED) {
#pragma unroll
    for (int u = 0; u < 3; ++u)
      if (s + u < s_end) acc[0][0][0] = mfma32(w_single[u], fetch_x<false>(xrow[0], nullptr, (s + u) * 32 + grp * 8).v, acc[0][0][0]);
    s = s_end;
  }
  for (; !TILED && s < s_end; ++s) {  // single steps
    const int kb = s * 32 + grp * 8;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const bf16x8 bf = finish_x<NORM>(fetch_x<NORM>(xrow[t], norm_w, kb), rs[t]);
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int a = 0; a < NA; ++a)
          acc[j][a][t] = mfma32(load_weights(w_single_at(wrow[j][a], s)), bf, acc[j][a][t]);
    }
  }

  if constexpr (SHORT) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int a = 0; a < NA; ++a) red[ks][0][j][a][0][lane] = acc[j][a][0];
    __syncthreads();
    // this thread's elements: the waves' parts, all read before the first is added, in wave order
    const int m = e_row;
    const bool here = (int)threadIdx.x < 256 && m < M;
    float y[NT][NA];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      float part[NA][KS];
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        const float* src = reinterpret_cast<const float*>(&red[0][0][j][a][0][0]) + threadIdx.x % 256;
#pragma unroll
        for (int wv = 0; wv < KS; ++wv) part[a][wv] = src[wv * (NT * NA * 256)];
      }
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        float sum = part[a][0];
#pragma unroll
        for (int wv = 1; wv < KS; ++wv) sum += part[a][wv];
        if (bias != nullptr) sum += (float)b_at[j][a][0];  // (past the last feature: dropped)
        y[j][a] = sum;
      }
    }
    __shared__ float sqs[EPI == EPI_RESIDUAL ? NT : 1][4][16];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int tile = tile0 + j, n = tile * 16 + e_n;
      if (EPI == EPI_RESIDUAL) {
        const bf16_t summed = (bf16_t)((float)old_s[EPI == EPI_RESIDUAL ? j : 0][0][0] + (float)(bf16_t)y[j][0]);
        const bool in = here && n < N;
        if (in) stream[(int64_t)m * lds_ + n] = summed;
        const float sq = quad_sum(in ? (float)summed * (float)summed : 0.f);
        if ((int)threadIdx.x < 256 && e_i == 0) sqs[j][e_grp][m] = sq;
      } else if (here && n < N) {
        const int64_t place = (int64_t)m * ldo + n;
        if (EPI == EPI_STORE) reinterpret_cast<bf16_t*>(out)[place] = (bf16_t)y[j][0];
        else if (EPI == EPI_F32) reinterpret_cast<float*>(out)[place] = y[j][0];
        else reinterpret_cast<bf16_t*>(out)[place] = glu_bf16((float)(bf16_t)y[j][0], (float)(bf16_t)y[j][NA - 1], glu);
      }
    }
    if (EPI == EPI_RESIDUAL) {
      __syncthreads();
#pragma unroll
      for (int j = 0; j < NT; ++j)
        if ((int)threadIdx.x < M && (tile0 + j) * 16 < N)
          ssq_out[(int64_t)(tile0 + j) * M + threadIdx.x] =
              (sqs[j][0][threadIdx.x] + sqs[j][1][threadIdx.x]) + (sqs[j][2][threadIdx.x] + sqs[j][3][threadIdx.x]);
    }
    return;
  }

  // k-split wave 0 of each group adds the other waves' partial tiles to its own, in wave order
  if constexpr (!SHORT && KS > 1) {
    if (ks != 0) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
          for (int t = 0; t < MT; ++t) red[ks - 1][ns][j][a][t][lane] = acc[j][a][t];
    }
    __syncthreads();
    if (ks == 0) {  // all of a tile's parts are read before the first is added
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          float4v part[NA][KR];
#pragma unroll
          for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int wv = 0; wv < KS - 1; ++wv) part[a][wv] = red[wv][ns][j][a][t][lane];
#pragma unroll
          for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int wv = 0; wv < KS - 1; ++wv) acc[j][a][t] += part[a][wv];
        }
    }
  }

  // lane holds y[m = 16t + col][n = 16*tile + 4*grp + i]
  if constexpr (!SHORT) {
  if (ks == 0) {
  if constexpr (!EARLY) load_bias();
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int tile = tile0 + j;
    const int nb = tile * 16 + 4 * grp;
    if (tile * 16 >= N) continue;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = t * 16 + col;
      float y[NA][4];
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          y[a][i] = acc[j][a][t][i];
          if (bias != nullptr) y[a][i] += (float)b_at[j][a][i];  // (past the last feature: dropped)
        }
      if constexpr (EPI == EPI_QKV) {
        // all lanes take part in the exchange of partners; rows beyond M hold zeros
        const int d = qr.head_dim, half = d / 2;
        const int head = tile * 16 / d, t_in = (tile * 16 - head * d) / 16;
        const bool rotary = head < qr.q_heads + qr.kv_heads;
        const int mm = min(m, M - 1), slot = qr.slots[mm];
        float v[4], partner[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = (float)(bf16_t)y[0][i];
          partner[i] = __shfl_xor(v[i], 32, 64);
        }
        if (rotary) {
          const int j = 8 * t_in + 4 * (grp & 1);  // first of this lane's four rotary pairs
          const float4v cs = *reinterpret_cast<const float4v*>(qr.angles + ((int64_t)mm * 2 + 0) * half + j);
          const float4v sn = *reinterpret_cast<const float4v*>(qr.angles + ((int64_t)mm * 2 + 1) * half + j);
          bf16_t r[4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            r[i] = grp < 2 ? (bf16_t)(v[i] * cs[i] - partner[i] * sn[i]) : (bf16_t)(v[i] * cs[i] + partner[i] * sn[i]);
          const int dim = (grp < 2 ? 0 : half) + j;
          bf16_t* dst = nullptr;
          if (head < qr.q_heads) {
            dst = reinterpret_cast<bf16_t*>(out) + (int64_t)m * ldo + head * d + dim;
          } else if (slot >= 0) {
            const int64_t page = slot / qr.page_size;
            const int off = slot - (int)page * qr.page_size;
            dst = qr.k_pages + ((page * qr.kv_heads + (head - qr.q_heads)) * qr.page_size + off) * d + dim;
          }
          if (m < M && dst != nullptr) {
            typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));
            *reinterpret_cast<bf16x4*>(dst) = bf16x4{r[0], r[1], r[2], r[3]};
          }
        } else if (m < M && slot >= 0) {
          const int64_t page = slot / qr.page_size;
          const int off = slot - (int)page * qr.page_size;
          const int hv = head - qr.q_heads - qr.kv_heads;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            qr.v_pages[((page * qr.kv_heads + hv) * d + 16 * t_in + 4 * grp + i) * qr.page_size + off] = (bf16_t)v[i];
        }
        continue;
      }
      float sq = 0.f;
      if (m < M) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int n = nb + i;
          if (n >= N) continue;
          if (EPI == EPI_STORE) {
            reinterpret_cast<bf16_t*>(out)[(int64_t)m * ldo + n] = (bf16_t)y[0][i];
          } else if (EPI == EPI_F32) {
            reinterpret_cast<float*>(out)[(int64_t)m * ldo + n] = y[0][i];
          } else if (EPI == EPI_SWIGLU) {
            const float g = (float)(bf16_t)y[0][i], u = (float)(bf16_t)y[NA - 1][i];
            reinterpret_cast<bf16_t*>(out)[(int64_t)m * ldo + n] = glu_bf16(g, u, glu);
          } else {  // EPI_RESIDUAL
            bf16_t* sp = stream + (int64_t)m * lds_ + n;
            const bf16_t summed = (bf16_t)((float)old_s[EPI == EPI_RESIDUAL ? j : 0][EPI == EPI_RESIDUAL ? t : 0][i] + (float)(bf16_t)y[0][i]);
            *sp = summed;
            sq += (float)summed * (float)summed;
          }
        }
      }
      if (EPI == EPI_RESIDUAL) {
        sq = add_across32(add_across16(sq));
        if (grp == 0 && m < M) ssq_out[(int64_t)tile * M + m] = sq;
      }
    }
  }
  }
  }
}

// Embedding rows with the sum of squares of each (one part), for the first layer's norm.
__global__ void embedding_ssq_kernel(const bf16_t* __restrict__ table, const int* __restrict__ ids,
                                     bf16_t* __restrict__ out, float* __restrict__ ssq, int width) {
  __shared__ float scratch[16];
  const int64_t row = blockIdx.x;
  const bf16_t* src = table + (int64_t)ids[row] * width;
  float s = 0.f;
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    const bf16_t v = src[i];
    out[row * width + i] = v;
    s += (float)v * (float)v;
  }
  const float total = block_sum(s, scratch);
  if (threadIdx.x == 0) ssq[row] = total;
}

#define SK_PARAMS                                                                                 \
  const void *x, int64_t ldx, const float *ssq_in, int ssq_parts, const float *norm_w, float eps,   \
      const void *w, const void *bias, void *out, int64_t ldo, void *stream_buf, int64_t lds_,      \
      float *ssq_out, int M, int N, int K, int up_offset, QkvRope qr, GluForm glu, hipStream_t stream
#define SK_ARGS \
  x, ldx, ssq_in, ssq_parts, norm_w, eps, w, bias, out, ldo, stream_buf, lds_, ssq_out, M, N, K, up_offset, qr, glu, stream

// The products that open the two halves of a decode layer (q/k/v with rotation and cache write, gate and up), with the
// row norm inside: at most four rows, weights in tile order, k split over the KS waves of a workgroup,
// which owns NT tiles. What bounds such a launch beside its weights is the time until they are asked
// for and the vector cache, which accepts 64 bytes a cycle and compute unit:
//  - The workgroup normalises the rows once, into LDS, and its waves read their fragments from there.
//    (Read from memory by every wave, a block's fragments are 12 KB, 16 bytes of x and 32 of norm
//    weights a lane and product, beside 4 KB of weights a tile.)
//  - Sums of squares, rows, norm weights and the first SETS blocks of weights are asked for in this order before
//    anything is waited for (loads come back in their order), with few instructions on the way:
//    through buffer resources, which count what lies past their end as zeros, so that no load needs a condition
//    or a bound of its own. What only the end needs is asked for last.
// MR: one row, or up to four.
// (Its times beside the general kernel's: dli_normed_tiles_ahead, launches one after the other in a replayed graph; traced in a decode
// step of one row q/k/v takes 4.1 us at the 135M sizes and 5.4 at the 1B sizes.)
struct NormedArgs {
  const bf16_t* x;
  const float* ssq_in;
  const float* norm_w;
  const bf16_t* w;
  const bf16_t* bias;
  bf16_t* out;
  int64_t ldo;
  int ldx, ssq_parts, M, N, K, up_offset;
  float eps;
  QkvRope qr;
  GluForm glu;
};

// Values per row of the normalised rows in LDS: whole blocks, and 16 bytes more, so that the sixteen
// rows that a fragment reads lie in different banks.
__host__ __device__ constexpr int normed_row(int K) { return (K + 127) / 128 * 128 + 8; }

template <int KS, int NT, int EPI, int SETS, int MR, bool IN_TURN>
__global__ __launch_bounds__(KS * 64) void normed_tiles_kernel(NormedArgs p) {
  static_assert(EPI == EPI_SWIGLU || EPI == EPI_QKV, "the products behind a norm");
  constexpr int NA = EPI == EPI_SWIGLU ? 2 : 1;  // weight row sets per tile (gate and up)
  constexpr int BA = 2;                          // sums a thread makes per tile: gate and up, or a feature and its rotary partner
  constexpr int PARTS = IN_TURN ? 1 : MR == 1 ? 2 : MR;  // loads of 64 parts of the sums of squares a wave asks for at the start
  constexpr int PRE = KS == 4 ? 3 : 2;           // pieces of 256 values of the rows likewise
  constexpr unsigned OUTSIDE = 0x80000000u;      // an offset past the end of every resource here
  typedef short short4v __attribute__((ext_vector_type(4)));
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  __shared__ float red[KS][NT][NA][256];
  __shared__ float rsum[KS][16];
  extern __shared__ __attribute__((aligned(16))) bf16_t xs[];  // rows of normed_row(K) values

  const int lane = threadIdx.x % 64, ks = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int col = lane % 16, grp = lane / 16;
  const int tile0 = blockIdx.x * NT, tiles = p.N / 16;
  const int M = p.M, K = p.K, row = normed_row(K);

  // The parts of sum x^2 that the producer of x left, [part][row]. Where the rows are a power of two
  // (decode graphs) a wave takes 64 of them in a row, lane l for row l % M; else the lane group grp takes
  // part 4 ks + grp, and every 4 KS-th behind it, for row l % 16.
  // IN_TURN (one row): the lane group's parts likewise, one a lane, added in their order as the general kernel adds them. More rows
  // of such a product take that kernel, and a row then has the same bits whether others share the product or not.
  const __amdgpu_buffer_rsrc_t sres = __builtin_amdgcn_make_buffer_rsrc((void*)p.ssq_in, 0, (unsigned)(p.ssq_parts * M * 4), 0x00020000);
  const bool even = (M & (M - 1)) == 0;
  const int s_at = IN_TURN ? (4 * ks + grp + col * 4 * KS) * 4 : even ? threadIdx.x * 4 : ((4 * ks + grp) * M + min(col, M - 1)) * 4;
  const int s_step = even ? 256 * KS : 16 * KS * M, s_end = p.ssq_parts * M * 4;
  float first[PARTS];
#pragma unroll
  for (int u = 0; u < PARTS; ++u) first[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(sres, s_at + u * s_step, 0, 0));
  // rows: wave ks takes the pieces ks, ks + KS, ... of 256 values, four a lane
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, (unsigned)(((M - 1) * p.ldx + K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t gres = __builtin_amdgcn_make_buffer_rsrc((void*)p.norm_w, 0, (unsigned)(K * 4), 0x00020000);
  union Four {
    u32x2 raw;
    bf16_t e[4];
  };
  union Gain {
    u32x4 raw;
    float e[4];
  };
  Four piece[PRE][MR];
  Gain gain[PRE];
  auto ask_gain = [&](Gain& g, int j) __attribute__((always_inline)) {
    g.raw = __builtin_amdgcn_raw_buffer_load_b128(gres, ((ks + j * KS) * 256 + lane * 4) * 4, 0, 0);
  };
  auto ask_rows = [&](Four (&v)[MR], int j) __attribute__((always_inline)) {   // (a row past the last lies past the resource's end)
    const int k = (ks + j * KS) * 256 + lane * 4;
    const unsigned at = k < K ? (unsigned)(k * 2) : OUTSIDE;
#pragma unroll
    for (int u = 0; u < MR; ++u) v[u].raw = __builtin_amdgcn_raw_buffer_load_b64(xres, at + (unsigned)(u * p.ldx * 2), 0, 0);
  };
#pragma unroll
  for (int j = 0; j < PRE; ++j) {
    ask_gain(gain[j], j);
    ask_rows(piece[j], j);
  }
  // weights: this wave's share of the blocks of 128 k
  const int whole = (K + 127) / 128, c0 = whole * ks / KS, blocks = whole * (ks + 1) / KS - c0;
  const bf16_t* wrow[NT][NA];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int a = 0; a < NA; ++a)
      wrow[j][a] = p.w + ((int64_t)min(tile0 + j, tiles - 1) + a * (p.up_offset / 16)) * 16 * (whole * 128) + c0 * 2048;
  struct Set {
    bf16x8 a[NT][NA][4];
  } sets[SETS];
  auto fetch = [&](Set& b, int c) __attribute__((always_inline)) {
    const int at = max(min(c, blocks - 1), 0) * 2048;  // (a wave without a block: one that is there, for nothing)
    const int from = blocks > 0 ? at : -c0 * 2048;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int q = 0; q < 4; ++q) b.a[j][a][q] = load_streamed(reinterpret_cast<const bf16x8*>(wrow[j][a] + from + q * 512 + lane * 8));
  };
#pragma unroll
  for (int d = 0; d < SETS; ++d) fetch(sets[d], d);
  __builtin_amdgcn_sched_barrier(0);
  // What the end adds. Thread t makes output t of each tile: element t % 4 of lane t / 4 of the
  // product's result, that is row t / 4 % 16 and feature 4 (t / 64) + t % 4.
  const int o_m = threadIdx.x / 4 % 16, o_grp = threadIdx.x / 64 % 4, o_n = 4 * o_grp + threadIdx.x % 4;
  const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)p.bias, 0, p.bias != nullptr ? (unsigned)(p.N + (NA - 1) * p.up_offset) * 2u : 0u, 0x00020000);
  union Half {
    unsigned short raw;
    bf16_t v;
  } b_at[NT][BA];
  float cs_at[NT], sn_at[NT];
  int slot = -1;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = (tile0 + j) * 16;
    b_at[j][0].raw = __builtin_amdgcn_raw_buffer_load_b16(bres, (n + o_n) * 2, 0, 0);
    b_at[j][1].raw = __builtin_amdgcn_raw_buffer_load_b16(bres, (EPI == EPI_SWIGLU ? n + o_n + p.up_offset : n + (o_n ^ 8)) * 2, 0, 0);
  }
  if constexpr (EPI == EPI_QKV) {
    const int half = p.qr.head_dim / 2, m = min(o_m, M - 1);
    slot = p.qr.slots[m];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int t_in = min(tile0 + j, tiles - 1) % (p.qr.head_dim / 16);
      const float* at = p.qr.angles + (int64_t)m * 2 * half + 8 * t_in + (o_n & 7);  // the rotary pair
      cs_at[j] = at[0];
      sn_at[j] = at[half];
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  // 1 / rms of row `col`: the lane's parts, the wave's lanes of a row, the waves in order
  float sum = 0.f;
  auto add_parts = [&](float v) __attribute__((always_inline)) {
    sum += v;
    if constexpr (IN_TURN) {   // (zeros behind the last part; no branch, which would wait for the weights as well)
      sum += row_shl<1>(v); sum += row_shl<2>(v); sum += row_shl<3>(v); sum += row_shl<4>(v); sum += row_shl<5>(v);
      sum += row_shl<6>(v); sum += row_shl<7>(v); sum += row_shl<8>(v); sum += row_shl<9>(v); sum += row_shl<10>(v);
      sum += row_shl<11>(v); sum += row_shl<12>(v); sum += row_shl<13>(v); sum += row_shl<14>(v); sum += row_shl<15>(v);
    }
  };
#pragma unroll
  for (int u = 0; u < PARTS; ++u) add_parts(first[u]);
  for (int at = PARTS * s_step; at < s_end; at += s_step) add_parts(__uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(sres, s_at + at, 0, 0)));
  if constexpr (IN_TURN) {
    sum = add_across32(add_across16(sum));
  } else {
    sum = add_halves(sum, sum);
    sum = add_rows(sum, sum);
    if (even) {
      sum += row_ror<8>(sum);
      sum += row_ror<4>(sum);
      if (M == 1) sum = quad_sum(sum);
      else if (M == 2) sum = quad_pairs(sum);
    }
  }
  if (lane < M) rsum[ks][lane] = sum;
  __syncthreads();
  float part[KS], total = 0.f;
#pragma unroll
  for (int wv = 0; wv < KS; ++wv) part[wv] = rsum[wv][min(col, M - 1)];
#pragma unroll
  for (int wv = 0; wv < KS; ++wv) total += part[wv];
  const float rs = rsqrtf(total / (float)K + p.eps);
  auto put_rows = [&](const Four (&v)[MR], const Gain& g, int j) __attribute__((always_inline)) {
    const int k = (ks + j * KS) * 256 + lane * 4;
#pragma unroll
    for (int u = 0; u < MR; ++u)
      if (u < M) {
        const float rsm = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rs), u));
        Four h;
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // (past K values and weights are zeros)
          const float normed = (float)(bf16_t)((float)v[u].e[i] * rsm);
          h.e[i] = (bf16_t)(g.e[i] * normed);
        }
        if (k < whole * 128) *reinterpret_cast<u32x2*>(xs + u * row + k) = h.raw;
      }
  };
#pragma unroll
  for (int j = 0; j < PRE; ++j)
    if ((ks + j * KS) * 256 < whole * 128) put_rows(piece[j], gain[j], j);
  for (int j = PRE; (ks + j * KS) * 256 < whole * 128; ++j) {   // further pieces of long rows
    Four v[MR];
    Gain g;
    ask_gain(g, j);
    ask_rows(v, j);
    put_rows(v, g, j);
  }
  __syncthreads();

  float4v acc[NT][NA];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[j][a] = float4v{0.f, 0.f, 0.f, 0.f};
  const bf16_t* frag = xs + min(col, M - 1) * row + c0 * 128 + grp * 32;
  auto multiply = [&](const Set& b, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bf16x8 bf = *reinterpret_cast<const bf16x8*>(frag + c * 128 + q * 8);
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int a = 0; a < NA; ++a) acc[j][a] = mfma32(b.a[j][a][q], bf, acc[j][a]);
    }
  };
  int c = 0;
  for (; c + 2 * SETS <= blocks; c += SETS) {
#pragma unroll
    for (int d = 0; d < SETS; ++d) {
      multiply(sets[d], c + d);
      fetch(sets[d], c + d + SETS);
      __builtin_amdgcn_sched_barrier(0);  // the loads leave before the next block's products
    }
  }
#pragma unroll
  for (int d = 0; d < SETS; ++d) {
    if (c + d < blocks) multiply(sets[d], c + d);
    if (c + d + SETS < blocks) fetch(sets[d], c + d + SETS);
  }
#pragma unroll
  for (int d = 0; d < SETS; ++d)
    if (c + d + SETS < blocks) multiply(sets[d], c + d + SETS);

#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int a = 0; a < NA; ++a) *reinterpret_cast<float4v*>(&red[ks][j][a][lane * 4]) = acc[j][a];
  __syncthreads();
  if (KS > 4 && ks >= 4) return;  // 256 outputs a tile
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    float part_y[BA][KS], y[BA];
#pragma unroll
    for (int wv = 0; wv < KS; ++wv) {
      part_y[0][wv] = red[wv][j][0][threadIdx.x];
      part_y[1][wv] = EPI == EPI_SWIGLU ? red[wv][j][NA - 1][threadIdx.x] : red[wv][j][0][threadIdx.x ^ 128];
    }
#pragma unroll
    for (int a = 0; a < BA; ++a) {
      y[a] = part_y[a][0];
#pragma unroll
      for (int wv = 1; wv < KS; ++wv) y[a] += part_y[a][wv];
      if (p.bias != nullptr) y[a] += (float)b_at[j][a].v;
    }
    const int tile = tile0 + j;
    if (o_m >= M || tile >= tiles) continue;
    if constexpr (EPI == EPI_SWIGLU) {
      p.out[(int64_t)o_m * p.ldo + tile * 16 + o_n] = glu_bf16((float)(bf16_t)y[0], (float)(bf16_t)y[1], p.glu);
    } else {
      const int d = p.qr.head_dim, half = d / 2;
      const int head = tile * 16 / d, t_in = (tile * 16 - head * d) / 16;
      const float v = (float)(bf16_t)y[0], partner = (float)(bf16_t)y[1];
      const int64_t page = slot / p.qr.page_size;
      const int off = slot - (int)page * p.qr.page_size;
      if (head < p.qr.q_heads + p.qr.kv_heads) {  // rotary
        const bf16_t r = o_grp < 2 ? (bf16_t)(v * cs_at[j] - partner * sn_at[j]) : (bf16_t)(v * cs_at[j] + partner * sn_at[j]);
        const int dim = (o_grp < 2 ? 0 : half) + 8 * t_in + (o_n & 7);
        if (head < p.qr.q_heads) p.out[(int64_t)o_m * p.ldo + head * d + dim] = r;
        else if (slot >= 0) p.qr.k_pages[((page * p.qr.kv_heads + (head - p.qr.q_heads)) * p.qr.page_size + off) * d + dim] = r;
      } else if (slot >= 0) {
        const int hv = head - p.qr.q_heads - p.qr.kv_heads;
        p.qr.v_pages[((page * p.qr.kv_heads + hv) * d + 16 * t_in + o_n) * p.qr.page_size + off] = (bf16_t)v;
      }
    }
  }
}

// More than 40 KB of LDS beside the kernel's own has to be allowed; whether the runtime refused (it
// then holds an error, which the launch's status reports).
static bool lds_refused(const void* kernel, size_t lds) {
  return lds > 40 * 1024 &&
         hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024) != hipSuccess;
}

// Whether normed_tiles_kernel takes the product. Its workgroups each normalise all rows before their first product, which with
// more rows costs more than the shared reads save, and the lanes' sums of squares go by rows that are a power of two. Cold, us with
// skinny_gemm_kernel and with this one at 1, 2, 3, 4, 8 and 16 rows:
//   q/k/v    135M sizes  4.1 3.9  4.2 4.5  4.2 4.3  4.2 4.4  4.3 5.1  4.4 6.2      1B    6.4 5.3  6.4 5.8  6.5 5.8  6.5 5.8  6.7 6.8  7.2 8.1
//            1.7B        8.9 8.7  9.0 9.1  9.0 9.7  9.1 9.2  9.0 9.8  9.9 12.1     3B    11.8 9.8  11.9 10.4  12.0 11.8  11.3 10.3  11.7 11.6
//            width 1,536, 24 heads on 24     6.9 7.1  6.9 7.6  6.9 7.6  7.0 7.5  7.3 8.5  8.0 10.6
//   gate/up  1B          -  15.4 14.8  15.3 16.0  15.3 15.0  15.8 16.4  16.9 19.0  3B    -  22.1 21.0  21.4 22.5  21.5 20.4  21.7 21.5
//            width 1,024, 4,096 wide         -  6.5 6.7  6.0 6.6  6.1 6.8  6.2 6.5  6.4 7.6
// So: one row, but not a short one whose tiles are more than the compute units; two and four rows of 2,048 values and more; three
// such where the tiles are no more than the units (a gated product's half are as many: never).
extern "C" int dli_normed_tiles_ahead(int M, int N, int K, int gated, int units) {
  const bool few = (N + 15) / 16 <= units, deep = K >= 2048;
  if (M == 1) return few || deep;
  return deep && (M == 2 || M == 4 || (M == 3 && few && !gated));
}

// Besides, its rows have to leave room in LDS for two workgroups on a compute unit, and to lie within what its 31-bit offsets
// reach. Four blocks of weights on their way where every wave has three or more, else two; a gated pair of two tiles takes the
// registers of two.
template <int KS, int NT, int EPI>
static bool launch_normed_tiles(SK_PARAMS) {
  constexpr int PER = NT * (EPI == EPI_SWIGLU ? 2 : 1);
  const size_t lds = (size_t)M * normed_row(K) * 2;
  if (!dli_normed_tiles_ahead(M, N, K, EPI == EPI_SWIGLU, dli_compute_units()) || lds + (size_t)KS * PER * 1024 + 1024 > 80 * 1024 || N % 16 != 0 ||
      ldx > INT32_MAX / 64 || ssq_parts > INT32_MAX / 256 || (int64_t)N + up_offset > INT32_MAX / 4)
    return false;
  const NormedArgs args{(const bf16_t*)x, ssq_in, norm_w, (const bf16_t*)w, (const bf16_t*)bias, (bf16_t*)out, ldo, (int)ldx,
                        ssq_parts, M, N, K, up_offset, eps, qr, glu};
  const int groups = (N / 16 + NT - 1) / NT;
  // A single row where more rows take the general kernel: its sums in that kernel's order (a step of the 135M sizes 0.2% longer, of
  // the 1B sizes, where two and four rows take this one as well, 0.6% without need).
  const bool alone = M == 1 && !dli_normed_tiles_ahead(2, N, K, EPI == EPI_SWIGLU, dli_compute_units());
#define NORMED_LAUNCH(SETS_, MR_, IN_TURN_)                                              \
  {                                                                                      \
    const auto kernel = normed_tiles_kernel<KS, NT, EPI, SETS_, MR_, IN_TURN_>;           \
    if (!lds_refused((const void*)kernel, lds)) kernel<<<groups, KS * 64, lds, stream>>>(args); \
  }
  if constexpr (PER <= 2) {
    if ((K + 127) / 128 / KS >= 3) {
      if (alone) NORMED_LAUNCH(4, 1, true)
      else if (M == 1) NORMED_LAUNCH(4, 1, false)
      else NORMED_LAUNCH(4, 4, false)
      return true;
    }
  }
  if (alone) NORMED_LAUNCH(2, 1, true)
  else if (M == 1) NORMED_LAUNCH(2, 1, false)
  else NORMED_LAUNCH(2, 4, false)
#undef NORMED_LAUNCH
  return true;
}

// Whether each of KS waves that share K has at least two blocks of 128, or none has any (whole blocks are dealt out in tile
// order, else steps of 32).
static bool two_blocks_or_none(int K, int KS, bool tiled) {
  const int least = tiled ? K / 128 / KS : K / 32 / KS / 4;
  const int most = tiled ? (K / 128 + KS - 1) / KS : (K / 32 + KS - 1) / KS / 4;
  return least >= 2 || most == 0;
}

template <int KS, int NS, int NT, int MT, int EPI, bool NORM, bool TILED>
static void launch_skinny(SK_PARAMS) {
  const int tiles = (N + 15) / 16;
  const int groups = (tiles + NS * NT - 1) / (NS * NT);
  if constexpr (NORM && TILED && MT == 1 && NS == 1 && (EPI == EPI_SWIGLU || EPI == EPI_QKV)) {
    if (launch_normed_tiles<KS, NT, EPI>(SK_ARGS)) return;
  }
#define SK_LAUNCH(AHEAD_)                                                                                          \
  skinny_gemm_kernel<KS, NS, NT, MT, EPI, NORM, TILED, AHEAD_><<<groups, KS * NS * 64, 0, stream>>>(                \
      (const bf16_t*)x, ldx, ssq_in, ssq_parts, norm_w, eps, (const bf16_t*)w, (const bf16_t*)bias,               \
      out, ldo, (bf16_t*)stream_buf, lds_, ssq_out, M, N, K, up_offset, qr, MergedIn{}, glu)
  if constexpr (MT == 1 && !NORM && EPI != EPI_QKV) {
    if (M <= 4 && two_blocks_or_none(K, KS, TILED)) {
      SK_LAUNCH(true);
      return;
    }
  }
  SK_LAUNCH(false);
#undef SK_LAUNCH
}

// shapes of the workgroup: 0: 4 k-waves x 1 tile (few tiles, short k); 1: 8 k-waves x 1 tile (few
// tiles, long k); 2: 4 n-waves x 2 tiles, no k split (many tiles: the activations are read once
// per 8 tiles); 3: 2 k-waves x 2 n-waves x 2 tiles; 4: 4 k-waves x 2 tiles (many tiles in tile order)
template <int MT, int EPI, bool NORM, bool TILED>
static void dispatch_shape(int shape, SK_PARAMS) {
  switch (shape) {
    case 0: launch_skinny<4, 1, 1, MT, EPI, NORM, TILED>(SK_ARGS); break;
    case 1: launch_skinny<8, 1, 1, MT, EPI, NORM, TILED>(SK_ARGS); break;
    case 2: launch_skinny<1, 4, 2, MT, EPI, NORM, TILED>(SK_ARGS); break;
    case 4: launch_skinny<4, 1, 2, MT, EPI, NORM, TILED>(SK_ARGS); break;
    default: launch_skinny<2, 2, 2, MT, EPI, NORM, TILED>(SK_ARGS); break;
  }
}

// tiled weights serve the decode steps of few rows: one row tile only
template <int EPI, bool NORM>
static int dispatch_skinny(int shape, int mt, bool tiled, SK_PARAMS) {
  if (tiled) dispatch_shape<1, EPI, NORM, true>(shape, SK_ARGS);
  else if (mt == 1) dispatch_shape<1, EPI, NORM, false>(shape, SK_ARGS);
  else if (mt == 2) dispatch_shape<2, EPI, NORM, false>(shape, SK_ARGS);
  else dispatch_shape<4, EPI, NORM, false>(shape, SK_ARGS);
  return dli_launch_status();
}

extern "C" int dli_skinny_gemm_max_rows() { return 64; }

// epilogue: 0 store bf16, 1 swiglu (N = features of one half, up rows at +up_offset), 2 residual,
// 3 store float32. norm_w == nullptr: no norm. shape: the workgroup shape, see dispatch_shape.
// tiled: w is in the tile order described at the top (at most 16 rows, K % 128 == 0, whole tiles).
extern "C" int dli_skinny_gemm(const void* x, int64_t ldx, const float* ssq_in, int ssq_parts,
                               const float* norm_w, float eps, const void* w, const void* bias,
                               void* out, int64_t ldo, void* stream_buf, int64_t lds_,
                               float* ssq_out, int M, int N, int K, int up_offset, int epilogue,
                               int shape, int tiled, int glu_form, float limit, float alpha, float up_shift,
                               hipStream_t stream) {
  const QkvRope qr{};
  const GluForm glu{glu_form, limit, alpha, up_shift};
  if (M <= 0 || N <= 0) return DLI_OK;
  if (tiled && (M > 16 || K % 128 != 0 || N % 16 != 0 || up_offset % 16 != 0)) return DLI_ERR_ARGUMENT;
  if (M > 64 || K <= 0 || K % 32 != 0 || ldx % 8 != 0 || shape < 0 || shape > 4 || epilogue < 0 ||
      epilogue > 3 || (norm_w != nullptr && (ssq_in == nullptr || ssq_parts <= 0)) ||
      (epilogue == EPI_RESIDUAL && (stream_buf == nullptr || ssq_out == nullptr || norm_w != nullptr)) ||
      (epilogue != EPI_RESIDUAL && out == nullptr))
    return DLI_ERR_ARGUMENT;
  const int mt = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
  const bool norm = norm_w != nullptr;
  switch (epilogue) {
    case EPI_STORE:
      return norm ? dispatch_skinny<EPI_STORE, true>(shape, mt, tiled != 0, SK_ARGS) : dispatch_skinny<EPI_STORE, false>(shape, mt, tiled != 0, SK_ARGS);
    case EPI_SWIGLU:
      return norm ? dispatch_skinny<EPI_SWIGLU, true>(shape, mt, tiled != 0, SK_ARGS) : dispatch_skinny<EPI_SWIGLU, false>(shape, mt, tiled != 0, SK_ARGS);
    case EPI_RESIDUAL:
      return dispatch_skinny<EPI_RESIDUAL, false>(shape, mt, tiled != 0, SK_ARGS);
    default:
      return norm ? dispatch_skinny<EPI_F32, true>(shape, mt, tiled != 0, SK_ARGS) : dispatch_skinny<EPI_F32, false>(shape, mt, tiled != 0, SK_ARGS);
  }
}

// The fused q/k/v projection of a decode step with rotation and cache write inside (EPI_QKV):
// w_tiled is the [(q_heads + 2*kv_heads) * head_dim, K] matrix in tile order (K filled up with zeros to whole blocks of 128;
// the norm's K is a multiple of 32) with the q and k
// heads' tiles made of rotary pairs (see the top), bias (optional) in the same feature order.
// q goes to out[row][head*head_dim + dim] (row stride ldo), rotated; rotated k and v go to the
// pages at slots[row]. angles: [M][2][head_dim/2] float32 cos/sin of the rows' positions.
extern "C" int dli_skinny_gemm_qkv_rope(const void* x, int64_t ldx, const float* ssq_in, int ssq_parts,
                                        const float* norm_w, float eps, const void* w_tiled,
                                        const void* bias, void* out, int64_t ldo, const float* angles,
                                        const int* slots, void* k_pages, void* v_pages, int M, int K,
                                        int q_heads, int kv_heads, int head_dim, int page_size,
                                        int shape, hipStream_t stream) {
  if (M <= 0) return DLI_OK;
  // (without the norm a last block of zeros could make a NaN of an infinite activation)
  if (M > 16 || K <= 0 || K % (norm_w != nullptr ? 32 : 128) != 0 || ldx % 8 != 0 || ldo % 8 != 0 || shape < 0 || shape > 4 ||
      q_heads <= 0 || kv_heads <= 0 || head_dim <= 0 || head_dim % 16 != 0 || page_size <= 0 ||
      out == nullptr || angles == nullptr || slots == nullptr || k_pages == nullptr ||
      v_pages == nullptr || (norm_w != nullptr && (ssq_in == nullptr || ssq_parts <= 0)))
    return DLI_ERR_ARGUMENT;
  const QkvRope qr{angles, slots, (bf16_t*)k_pages, (bf16_t*)v_pages, q_heads, kv_heads, head_dim, page_size};
  const int N = (q_heads + 2 * kv_heads) * head_dim, up_offset = 0;
  void* stream_buf = nullptr;
  float* ssq_out = nullptr;
  const int64_t lds_ = 0;
  const void* w = w_tiled;
  const GluForm glu{};
  if (norm_w != nullptr) dispatch_shape<1, EPI_QKV, true, true>(shape, SK_ARGS);
  else dispatch_shape<1, EPI_QKV, false, true>(shape, SK_ARGS);
  return dli_launch_status();
}

// The o projection of a decode step of at most MERGE_ROWS rows, fed with the split-key partial
// results of the attention instead of its merged output (MERGED above): stream += merge(...) @ w^T
// (+ bias), and the parts of the rows' sums of squares. w [N, K], K = heads * head_dim, in tile order where K is whole blocks of
// 128, else in chunks; splits 2..MERGE_SPLITS; shape 0 or 1 (4 or 8 waves split k).
extern "C" int dli_skinny_gemm_merged(const float* part_o, const float* part_ml, int splits, int heads,
                                      int head_dim, const void* w, const void* bias, void* stream_buf,
                                      int64_t lds_, float* ssq_out, int M, int N, int shape, hipStream_t stream) {
  if (M <= 0 || N <= 0) return DLI_OK;
  const int64_t K64 = (int64_t)heads * head_dim;
  if (M > MERGE_ROWS || splits < 2 || splits > MERGE_SPLITS || heads <= 0 || head_dim <= 0 || head_dim % 4 != 0 ||
      K64 % 32 != 0 || K64 > (1 << 20) || N % 16 != 0 || (shape != 0 && shape != 1) || part_o == nullptr ||
      part_ml == nullptr || w == nullptr || stream_buf == nullptr || ssq_out == nullptr)
    return DLI_ERR_ARGUMENT;
  const int K = (int)K64, ks = shape == 0 ? 4 : 8;
  const bool tiled = K % 128 == 0;
  if ((tiled ? ((K / 128 + ks - 1) / ks) * 128 : ((K / 32 + ks - 1) / ks) * 32) > MERGE_RANGE) return DLI_ERR_ARGUMENT;
  const MergedIn mi{part_o, part_ml, splits, heads, head_dim};
  const int groups = N / 16;
#define MERGED_LAUNCH(KS, TILED, RUNS)                                                             \
  skinny_gemm_kernel<KS, 1, 1, 1, EPI_RESIDUAL, false, TILED, false, RUNS><<<groups, KS * 64, 0, stream>>>( \
      nullptr, 0, nullptr, 0, nullptr, 0.f, (const bf16_t*)w, (const bf16_t*)bias, nullptr, 0,     \
      (bf16_t*)stream_buf, lds_, ssq_out, M, N, K, 0, QkvRope{}, mi, GluForm{})
#define MERGED_RUNS(KS, TILED)                       \
  if (splits <= 2) MERGED_LAUNCH(KS, TILED, 2);      \
  else if (splits <= 4) MERGED_LAUNCH(KS, TILED, 4); \
  else if (splits <= 8) MERGED_LAUNCH(KS, TILED, 8); \
  else MERGED_LAUNCH(KS, TILED, 16)
  if (tiled) {
    if (shape == 0) {
      MERGED_RUNS(4, true);
    } else {
      MERGED_RUNS(8, true);
    }
  } else if (shape == 0) {
    MERGED_RUNS(4, false);
  } else {
    MERGED_RUNS(8, false);
  }
#undef MERGED_RUNS
#undef MERGED_LAUNCH
  return dli_launch_status();
}

extern "C" int dli_skinny_gemm_merged_limits(int* rows, int* splits) {
  *rows = MERGE_ROWS;
  *splits = MERGE_SPLITS;
  return DLI_OK;
}

extern "C" int dli_embedding_ssq(const void* table, const int* ids, void* out, float* ssq, int rows,
                                 int width, hipStream_t stream) {
  if (rows <= 0) return DLI_OK;
  if (width <= 0) return DLI_ERR_ARGUMENT;
  embedding_ssq_kernel<<<rows, 256, 0, stream>>>((const bf16_t*)table, ids, (bf16_t*)out, ssq, width);
  return dli_launch_status();
}
