// 32-bit matrix product for the true 32-bit path: out[m][n] = sum_k a[m][k] * w[n][k]
// (+ bias[n]) (+ residual[m][n]), on the matrix cores' 32-bit form (v_mfma_f32_16x16x4_f32: IEEE
// single-precision products and sums, no narrower operand anywhere).
//
// Every output element sums its k in one order that depends on k alone, whatever the tile it falls
// in and however many waves share the work, so a row's result does not depend on how many other rows
// are in the batch: 128 consecutive k make a run, whose sum grows four k at a time; the sums of
// consecutive runs add up to at most GF_SEGMENTS segments, and the segments' sums are added in
// ascending order (the rounding error of a long sum then grows with the length of a run plus the
// number of runs, not with k).
//
// What bounds it: for few rows the stream of w, for many the matrix cores (157 TFLOP/s dense in 32-bit; a library product of
// 8,192^3 reaches 152), in between the launch and the few tiles there are. Measured, us a product m x n x k, before (64 x 64
// tiles of vector FMAs through LDS) and now:
//   2 x 3072 x 576      37.6 ->   5.6     498 x 960 x 576     39.2 -> 12.5     512 x 3072 x 2048      152 ->   79
//   2 x 576 x 1536      95.6 ->   5.7     498 x 3072 x 576    47.2 -> 28.5     512 x 16384 x 2048     491 ->  290
//   2 x 49152 x 576     60.9 ->  21.6     498 x 576 x 1536     109 -> 22.6     2048 x 16384 x 2048   1827 -> 1128 (122 TFLOP/s)
//   4 x 128256 x 2048    445 ->   177 (5.9 TB/s)                               2048 x 2048 x 8192     985 ->  606 (113 TFLOP/s)
// (Reading both operands straight from memory also with many rows, a wave a tile: 44 us at 498 x 3072 x 576, 1,980 at 2048 x
// 16384 x 2048: neighbouring lanes of a load lie in different rows. Choosing between a loaded value and zero beside the load
// makes a wave wait for it at once: whole steps load without the choice, or choose when the value goes to LDS.)
#include "common.h"

#define GF_RUN 128
#define GF_SEGMENTS 16

typedef float gf4 __attribute__((ext_vector_type(4)));

struct GfArgs {
  const float* a;
  const float* w;
  const float* bias;
  const float* residual;
  float* out;
  int64_t lda, ldw, ldr, ldo;
  int m, n, k;
  int segments, seg_runs;   // the sum's order: `segments` of `seg_runs` runs each (the last may be shorter)
};

// What a few-row product of the recorded decode steps takes in besides: the norm before it, and what follows it.
#define GF_PLAIN 0
#define GF_GLU 1    // silu(gate) * up: the first half of w's rows are gates, the second ups
#define GF_ROPE 2   // q, k and v heads: q and k rotated (the pairs i, i + head_dim / 2), k and v written at their slots
// How it reads w: word by word, 16 bytes a lane, or 16 bytes a lane by way of LDS (whole halves of runs).
#define GF_WORDS 0
#define GF_WIDE 1
#define GF_STAGED 2
struct GfAround {
  const float* norm_w;
  float eps;
  int norm_waves;   // waves of the norm's own kernel, whose order of sums this one keeps
  const int* positions;
  const float* inv_freq;
  const int* slots;
  float* k_pages;
  float* v_pages;
  int q_heads, kv_heads, head_dim, page_size;
};

struct Zero { static constexpr int value = 0; };
struct One { static constexpr int value = 1; };

// The four values of `row` from k = kk on. What lies past the row's end is zero.
template <bool VEC>
__device__ __forceinline__ gf4 gf_load(const float* row, int kk, int k) {
  if constexpr (VEC) {
    const gf4 v = *reinterpret_cast<const gf4*>(row + min(kk, k - 4));   // (k is a multiple of four: never across the end)
    return kk < k ? v : gf4{0.f, 0.f, 0.f, 0.f};
  } else {
    gf4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = row[min(kk + e, k - 1)];
      v[e] = kk + e < k ? x : 0.f;
    }
    return v;
  }
}

// 16 bytes a lane from its own address into LDS, the wave's lanes one behind the other, without passing registers.
// (the host's pass over the source does not know this builtin, and would drop every kernel that names it)
__device__ __forceinline__ void gf_to_lds(const float* from, gf4* to) {
#ifdef __HIP_DEVICE_COMPILE__
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from, (__attribute__((address_space(3))) void*)to, 16, 0, 0);
#endif
}
// Waits until at most N of the wave's loads are outstanding.
template <int N>
__device__ __forceinline__ void gf_wait() {
  static_assert(N >= 0 && N < 64, "6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
  asm volatile("" ::: "memory");
}

// Waits for the wave's reads of LDS.
__device__ __forceinline__ void gf_wait_lds() {
  __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
  asm volatile("" ::: "memory");
}

// Lane (i, g) holds rows 4 g .. + 3 of a tile of 16 x 16, column i.
__device__ __forceinline__ void gf_store(const GfArgs& p, gf4 sum, int m0, int n0, int i, int g) {
  const int col = n0 + i;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = m0 + 4 * g + e;
    if (row >= p.m || col >= p.n) continue;
    float v = sum[e];
    if (p.bias != nullptr) v += p.bias[col];
    if (p.residual != nullptr) v += p.residual[(int64_t)row * p.ldr + col];
    p.out[(int64_t)row * p.ldo + col] = v;
  }
}

// Up to 16 rows: KW waves share a tile of 16 x 16 NT and take its segments in turn, each straight from memory: half a run's
// operands are on their way while the other half is multiplied. The lanes that multiply lie in 16 rows, four neighbours in four
// of them: a load so laid out passes the compute unit's loads at a quarter of their rate, and few tiles mean few units.
// READ == GF_STAGED (k of whole half runs, a tile of sixteen columns) therefore brings w into LDS, four neighbours in 64 bytes of
// one row, and reads it from there; both halves of a wave's first run are asked for at once. us, weights from memory, two rows,
// before and now: 576 x 576 4.5 3.3, 576 x 1,536 6.7 5.7, 2,048 x 8,192 24.2 20.6, 49,152 x 576 26.8 21.6, 100,000 x 1,024 77.6 75.1;
// 16 rows: 576 x 576 5.4 4.0, 2,048 x 8,192 34.0 28.0.
//
// FORM GF_GLU and GF_ROPE: the rows are normalised on their way to the matrix cores and the sums go on where they are, so that a
// decode step's norms, activations and rotations are no kernels of their own (each 2.8 to 3.9 us of a step of two rows, which
// this one's 5 to 6 outlasts by less than one; two prompts of 333 and 178 tokens and four steps at the 135M sizes:
// 9.00 -> 8.06 ms a pass, and 7.38 with w through LDS and what the norm and the rotation read asked for ahead of it: q, k and v
// of two rows at these sizes 6.8 -> 5.0 us, gate and up 6.9 -> 5.5). A tile's sixteen columns are then eight of one half and the
// eight that they are paired with, a rotation by eight lanes away. The norm's sum of squares and its products are those of
// its own kernel, bit for bit: a wave takes a row, while the first weights are on their way.
template <int NT, int KW, int READ, int FORM = GF_PLAIN>
__global__ __launch_bounds__(64 * KW) void gemm_f32_few_kernel(GfArgs p, GfAround x) {
  constexpr bool VEC = READ != GF_WORDS, STAGED = READ == GF_STAGED;
  static_assert((FORM == GF_PLAIN || VEC) && (NT == 1 || (FORM == GF_PLAIN && !STAGED)), "one tile of whole vectors");
  constexpr int LOADS = FORM == GF_PLAIN ? 8 : 12;   // a wave's loads for half a run
  extern __shared__ gf4 gf_sums[];   // [segments][NT][64], then, STAGED, [KW][2][4][64]
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), i = lane % 16, g = lane / 16;
  __shared__ float rstd[16];
  int n0 = blockIdx.x * 16 * NT;
  const float* ra = p.a + (int64_t)min(i, p.m - 1) * p.lda;   // (rows past the end: not stored)
  int head = 0;
  bool rotates = false;
  if constexpr (FORM == GF_GLU) n0 = blockIdx.x * 8;
  if constexpr (FORM == GF_ROPE) {
    head = blockIdx.x / (x.head_dim / 16);
    rotates = head < x.q_heads + x.kv_heads;
  }
  const auto row_of_w = [&](int at) {   // of the tile's row `at`
    if constexpr (FORM == GF_GLU) return (at < 8 ? 0 : p.n / 2) + min(n0 + at % 8, p.n / 2 - 1);
    if constexpr (FORM == GF_ROPE) {
      const int t = blockIdx.x % (x.head_dim / 16);
      return head * x.head_dim + (rotates ? 8 * t + at % 8 + (at < 8 ? 0 : x.head_dim / 2) : 16 * t + at);
    }
    return min(n0 + at, p.n - 1);
  };
  const int feature = row_of_w(i);   // this lane's row of w (the first of NT)
  const float* rw[NT];
#pragma unroll
  for (int y = 0; y < NT; ++y) rw[y] = p.w + (int64_t)row_of_w(16 * y + i) * p.ldw;
  // STAGED: what the lane brings, chunk lane % 4 ^ row / 4 of row lane / 4, and where its own chunk g of row i then lies: a load's
  // four neighbours in one line, a read's sixteen lanes in banks of their own
  gf4* const stage = gf_sums + p.segments * NT * 64 + wave * 512;
  const float* const brings = p.w + (int64_t)row_of_w(lane / 4) * p.ldw + (lane % 4 ^ lane / 16) * 4;
  const int own = 4 * i + (g ^ i / 4);
  gf4 seg[NT], acc[NT], fa[2][4], fw[2][4][NT], fn[2][FORM != GF_PLAIN ? 4 : 1];
#pragma unroll
  for (int y = 0; y < NT; ++y) seg[y] = gf4{0.f, 0.f, 0.f, 0.f};

  const auto load = [&](auto half, int k0) {   // 64 k from k0 on
    constexpr int b = decltype(half)::value;
    if (STAGED || (VEC && k0 + GF_RUN / 2 <= p.k)) {   // (no choice between the value and zero: it would wait for the load at once)
      if constexpr (STAGED) {
        k0 = min(k0, p.k - GF_RUN / 2);   // (behind the last half run: not used)
#pragma unroll
        for (int t = 0; t < 4; ++t) gf_to_lds(brings + k0 + 16 * t, stage + (4 * b + t) * 64);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        fa[b][t] = *reinterpret_cast<const gf4*>(ra + k0 + 4 * g + 16 * t);
        if constexpr (FORM != GF_PLAIN) fn[b][t] = *reinterpret_cast<const gf4*>(x.norm_w + k0 + 4 * g + 16 * t);
        if constexpr (!STAGED)
#pragma unroll
          for (int y = 0; y < NT; ++y) fw[b][t][y] = *reinterpret_cast<const gf4*>(rw[y] + k0 + 4 * g + 16 * t);
      }
      if constexpr (STAGED) asm volatile("" ::: "memory");   // (loads are counted: none moves into another half's)
      return;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      fa[b][t] = gf_load<VEC>(ra, k0 + 16 * t + 4 * g, p.k);
      if constexpr (FORM != GF_PLAIN) fn[b][t] = gf_load<VEC>(x.norm_w, k0 + 16 * t + 4 * g, p.k);
#pragma unroll
      for (int y = 0; y < NT; ++y) fw[b][t][y] = gf_load<VEC>(rw[y], k0 + 16 * t + 4 * g, p.k);
    }
  };
  float r = 1.f;
  // `behind`: the other half's loads were asked for behind this one's
  const auto multiply = [&](auto half, auto behind) {
    constexpr int b = decltype(half)::value;
    if constexpr (STAGED) {
      gf_wait<decltype(behind)::value ? LOADS : 0>();
#pragma unroll
      for (int t = 0; t < 4; ++t) fw[b][t][0] = stage[(4 * b + t) * 64 + own];
    }
    if constexpr (FORM != GF_PLAIN)
#pragma unroll
      for (int t = 0; t < 4; ++t) fa[b][t] = fn[b][t] * (fa[b][t] * r);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int y = 0; y < NT; ++y) acc[y] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[b][t][s], fw[b][t][y][s], acc[y], 0, 0, 0);
  };

  // What the norm and the rotation read is asked for before the weights, and so is there long before them: loads come back in
  // their order. (Of the wave's first row, up to 1,024 values.)
  gf4 row_in[4];
  float freq = 0.f;
  int at_position[4], at_slot[4];
  if constexpr (FORM != GF_PLAIN) {
    if (wave < p.m) {
      const float* xr = p.a + (int64_t)wave * p.lda;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int at = min(512 * q + 8 * lane, p.k - 8);
        row_in[2 * q] = *reinterpret_cast<const gf4*>(xr + at);
        row_in[2 * q + 1] = *reinterpret_cast<const gf4*>(xr + at + 4);
      }
    }
    if constexpr (FORM == GF_ROPE) {
      if (wave == 0) {   // the wave that ends the tile
        freq = x.inv_freq[feature % x.head_dim % (x.head_dim / 2)];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          at_position[e] = x.positions[min(4 * g + e, p.m - 1)];
          at_slot[e] = x.slots[min(4 * g + e, p.m - 1)];
        }
      }
    }
    asm volatile("" ::: "memory");
  }
  const int runs = (p.k + GF_RUN - 1) / GF_RUN;
  int s = wave, left = 0;
  gf4 c = {1.f, 1.f, 1.f, 1.f}, sn = {0.f, 0.f, 0.f, 0.f};
  int slot[4] = {-1, -1, -1, -1};
  const auto prepare = [&](auto behind) {   // the rows' factors to LDS, this lane's rotations
    if constexpr (STAGED) gf_wait<decltype(behind)::value ? 2 * LOADS : 0>();
    const auto squares = [](gf4 lo, gf4 hi, float part) {
#pragma unroll
      for (int e = 0; e < 4; ++e) part = fmaf(lo[e], lo[e], part);
#pragma unroll
      for (int e = 0; e < 4; ++e) part = fmaf(hi[e], hi[e], part);
      return part;
    };
    const auto factor = [&](int row, float ss) {
      if (lane == 0) rstd[row] = rsqrtf(ss / (float)p.k + x.eps);
    };
    int row = wave;
    if (row < p.m && p.k <= 1024) {
#pragma unroll
      for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(row_in[q]));   // (not used before the weights are asked for)
      float ss = 0.f, part = 8 * lane < p.k ? squares(row_in[0], row_in[1], 0.f) : 0.f;
      if (x.norm_waves == 2) {
        ss = wave_sum(part);
        part = 0.f;
      }
      if (512 + 8 * lane < p.k) part = squares(row_in[2], row_in[3], part);
      factor(row, ss + wave_sum(part));
      row += KW;
    }
    for (; row < p.m; row += KW) {
      const float* xr = p.a + (int64_t)row * p.lda;
      float ss = 0.f;
      for (int j = 0; j < x.norm_waves; ++j) {
        float part = 0.f;
        for (int at = (64 * j + lane) * 8; at < p.k; at += 512 * x.norm_waves)
          part = squares(*reinterpret_cast<const gf4*>(xr + at), *reinterpret_cast<const gf4*>(xr + at + 4), part);
        ss += wave_sum(part);
      }
      factor(row, ss);
    }
    if constexpr (FORM == GF_ROPE) {
      if (wave == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          asm volatile("" : "+v"(at_position[e]), "+v"(at_slot[e]));
          if (4 * g + e >= p.m) continue;
          slot[e] = at_slot[e];
          if (rotates) {
            float sine, cosine;
            sincosf((float)at_position[e] * freq, &sine, &cosine);
            c[e] = cosine;
            sn[e] = i < 8 ? -sine : sine;
          }
        }
      }
    }
  };
  if (s < p.segments) {
    load(Zero{}, s * p.seg_runs * GF_RUN);
    if constexpr (STAGED) load(One{}, s * p.seg_runs * GF_RUN + GF_RUN / 2);
    left = min(p.seg_runs, runs - s * p.seg_runs);
    if constexpr (FORM != GF_PLAIN) prepare(One{});   // (written out for both sides: how many loads are behind the row's is known then)
  } else if constexpr (FORM != GF_PLAIN) {
    prepare(Zero{});
  }
  if constexpr (FORM != GF_PLAIN) {
    __syncthreads();
    r = rstd[min(i, p.m - 1)];
  }
  const auto begin = [&] {
#pragma unroll
    for (int y = 0; y < NT; ++y) acc[y] = gf4{0.f, 0.f, 0.f, 0.f};
  };
  const auto end = [&](bool last) {   // of a run, the last of its segment
#pragma unroll
    for (int y = 0; y < NT; ++y) {
      seg[y] += acc[y];
      if (last) {
        gf_sums[(s * NT + y) * 64 + lane] = seg[y];
        seg[y] = gf4{0.f, 0.f, 0.f, 0.f};
      }
    }
  };
  if (s < p.segments) {
    for (int u = s * p.seg_runs;;) {   // run u of segment s, `left` runs of it to go; its first half is on its way (STAGED: both)
      const bool last = --left == 0;
      const int s_next = last ? s + KW : s, r_next = last ? s_next * p.seg_runs : u + 1;
      begin();
      if constexpr (!STAGED) load(One{}, u * GF_RUN + GF_RUN / 2);
      multiply(Zero{}, One{});
      if (s_next >= p.segments) {
        if (u * GF_RUN + GF_RUN / 2 < p.k) multiply(One{}, Zero{});   // (the sum's last run may have one half)
        end(last);
        break;
      }
      if constexpr (STAGED) gf_wait_lds();   // what is read here has been read
      load(Zero{}, r_next * GF_RUN);
      multiply(One{}, One{});
      if constexpr (STAGED) {
        gf_wait_lds();
        load(One{}, r_next * GF_RUN + GF_RUN / 2);
      }
      end(last);
      if (last) left = min(p.seg_runs, runs - r_next);
      s = s_next;
      u = r_next;
    }
  }
  __syncthreads();
#pragma unroll
  for (int y = 0; y < NT; ++y) {
    if (y % KW != wave) continue;
    gf4 sum = gf4{0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < p.segments; ++c) sum += gf_sums[(c * NT + y) * 64 + lane];
    if constexpr (FORM == GF_PLAIN) {
      gf_store(p, sum, 0, n0 + 16 * y, i, g);
      continue;
    }
    if (p.bias != nullptr) sum += p.bias[feature];
    gf4 other;   // the tile's other half (all lanes take part)
#pragma unroll
    for (int e = 0; e < 4; ++e) other[e] = row_ror<8>(sum[e]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 4 * g + e;
      if (row >= p.m) continue;
      if constexpr (FORM == GF_GLU) {
        if (i < 8 && n0 + i < p.n / 2) p.out[(int64_t)row * p.ldo + n0 + i] = silu<float>(sum[e]) * other[e];
      } else {
        const float v = rotates ? rotated(sum[e], other[e], c[e], sn[e]) : sum[e];
        const int d = feature - head * x.head_dim;
        if (head < x.q_heads) {
          p.out[(int64_t)row * p.ldo + feature] = v;
        } else if (slot[e] >= 0) {
          const int64_t page = slot[e] / x.page_size;
          const int off = slot[e] % x.page_size;
          if (rotates) x.k_pages[((page * x.kv_heads + head - x.q_heads) * x.page_size + off) * x.head_dim + d] = v;
          else x.v_pages[((page * x.kv_heads + head - x.q_heads - x.kv_heads) * x.head_dim + d) * x.page_size + off] = v;
        }
      }
    }
  }
}

// More rows: a wave makes a tile of 32 x 32 out of LDS, into which 32 k of its rows come in whole cache lines (rows of 36
// floats there: the 16 rows of a read lie in banks of their own), the next 32 k in flight meanwhile. KG == 1: WM x WN
// waves lie side by side and share what they stage. KG > 1 (few tiles, long sums): KG waves share one tile and take
// its segments in turn, each in a part of LDS of its own: its lanes hand each other what they stage behind a fence of
// the wave, without a wait for other waves.
#define GF_BK 32
#define GF_LD 36

template <int WM, int WN, int KG, bool VEC>
__global__ __launch_bounds__(64 * WM * WN * KG) void gemm_f32_tile_kernel(GfArgs p) {
  static_assert(KG == 1 || WM * WN == 1, "waves that take segments in turn stage for themselves");
  constexpr int BM = 32 * WM, BN = 32 * WN, THREADS = 64 * WM * WN, PER = (BM + BN) * (GF_BK / 4) / THREADS;
  extern __shared__ gf4 gf_sums[];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, i = lane % 16, g = lane / 16;
  const int part = KG > 1 ? wave : 0, tid = KG > 1 ? lane : threadIdx.x;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int wm = KG > 1 ? 0 : wave / WN * 32, wn = KG > 1 ? 0 : wave % WN * 32;
  float* stage = reinterpret_cast<float*>(gf_sums) + part * 2 * (BM + BN) * GF_LD;   // two of them in turn

  const float* src[PER];   // this thread's share of the tile's rows: 16 bytes of each 32 k
  int dst[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int c = u * THREADS + tid, row = c / (GF_BK / 4), at = c % (GF_BK / 4) * 4;
    src[u] = (row < BM ? p.a + (int64_t)min(m0 + row, p.m - 1) * p.lda : p.w + (int64_t)min(n0 + row - BM, p.n - 1) * p.ldw) ;
    dst[u] = row * GF_LD + at;
  }
  const int at = tid % (GF_BK / 4) * 4;   // (THREADS is a multiple of eight: the same place in every row)
  gf4 flight[PER];
  const auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      if constexpr (VEC) flight[u] = *reinterpret_cast<const gf4*>(src[u] + min(k0 + at, p.k - 4));
      else flight[u] = gf_load<false>(src[u], k0 + at, p.k);
    }
  };
  const auto put = [&](float* to, int k0) {   // (what lies past the row's end is zero; chosen here, long after the load)
#pragma unroll
    for (int u = 0; u < PER; ++u)
      *reinterpret_cast<gf4*>(to + dst[u]) = !VEC || k0 + at < p.k ? flight[u] : gf4{0.f, 0.f, 0.f, 0.f};
  };

  // What has been put there is seen by the lanes that read it, and nothing put later overtakes what they read.
  const auto staged = [&] {
    if constexpr (KG == 1) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  };

  gf4 total[2][2], seg[2][2], acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) total[x][y] = seg[x][y] = acc[x][y] = gf4{0.f, 0.f, 0.f, 0.f};

  gf4 kept[KG > 1 ? GF_SEGMENTS / KG : 1][2][2];   // KG > 1: the sums of this wave's segments (others' lie between them)
  int seen = 0;
  const int seg_k = p.seg_runs * GF_RUN;
  int s = part, k0 = part * seg_k, buf = 0;
  if (s < p.segments) {
    fetch(k0);
    put(stage, k0);
  }
  staged();
  while (s < p.segments) {
    int k_next = k0 + GF_BK, s_next = s;
    const bool seg_ends = k_next >= p.k || k_next % seg_k == 0;
    if (seg_ends) {
      s_next = s + KG;
      k_next = s_next * seg_k;
    }
    if (s_next < p.segments) fetch(k_next);
    const float* cur = stage + buf * (BM + BN) * GF_LD;
    const float *ca = cur + (wm + i) * GF_LD + 4 * g, *cw = cur + (BM + wn + i) * GF_LD + 4 * g;
#pragma unroll
    for (int t = 0; t < GF_BK / 16; ++t) {
      gf4 fa[2], fw[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        fa[x] = *reinterpret_cast<const gf4*>(ca + 16 * x * GF_LD + 16 * t);
        fw[x] = *reinterpret_cast<const gf4*>(cw + 16 * x * GF_LD + 16 * t);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[x][e], fw[y][e], acc[x][y], 0, 0, 0);
    }
    if (seg_ends || k_next % GF_RUN == 0) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          seg[x][y] += acc[x][y];
          acc[x][y] = gf4{0.f, 0.f, 0.f, 0.f};
          if (seg_ends) {
            if constexpr (KG > 1) {
#pragma unroll
              for (int c = 0; c < GF_SEGMENTS / KG; ++c)
                if (c == seen) kept[c][x][y] = seg[x][y];
            } else {
              total[x][y] += seg[x][y];
            }
            seg[x][y] = gf4{0.f, 0.f, 0.f, 0.f};
          }
        }
      if (seg_ends) ++seen;
    }
    buf ^= 1;
    if (s_next < p.segments) put(stage + buf * (BM + BN) * GF_LD, k_next);
    staged();
    k0 = k_next;
    s = s_next;
  }
  if constexpr (KG > 1) {   // the segments' sums go where the staging was: [segments][4][64]
    __syncthreads();
#pragma unroll
    for (int c = 0; c < GF_SEGMENTS / KG; ++c)
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          if (wave + c * KG < p.segments) gf_sums[((wave + c * KG) * 4 + 2 * x + y) * 64 + lane] = kept[c][x][y];
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      if (KG > 1 && (2 * x + y) % KG != wave) continue;
      gf4 sum = total[x][y];
      if constexpr (KG > 1)
        for (int c = 0; c < p.segments; ++c) sum += gf_sums[(c * 4 + 2 * x + y) * 64 + lane];
      gf_store(p, sum, m0 + wm + 16 * x, n0 + wn + 16 * y, i, g);
    }
}

// The same with k in whole GF_BK: loads write LDS without passing registers, STAGES - 1 blocks of k ahead, and a block has one
// barrier. The kernel above waits for each block's loads; here most of the time is the matrix cores'.
// us before and now: 1,500 x 3,072 x 576 73.5 61.7, 511 x 16,384 x 2,048 331 290, 2,048 x 16,384 x 2,048 1,290 1,128, 2,048 x 2,048 x
// 8,192 662 606, and for tiles of 32 x 32 with four waves each 511 x 3,072 x 576 36.6 28.5, 1,000 x 960 x 2,560 77.5 59.7. (Three
// stages are ahead of four where units have several tiles, 1,500 x 3,072 x 576 67.0 with four; four where they have one.)
// The eight chunks of a row lie at chunk ^ gf_turn(row): a load's lanes in whole lines, a read's sixteen lanes in banks of their own.
__device__ __forceinline__ int gf_turn(int row) { return (row ^ (row >> 3 & 1)) & 7; }

template <int WM, int WN, int STAGES>
__global__ __launch_bounds__(64 * WM * WN) void gemm_f32_ahead_kernel(GfArgs p) {
  constexpr int BM = 32 * WM, BN = 32 * WN, WAVES = WM * WN, STAGE = (BM + BN) * 8, LOADS = (BM + BN) / 8 / WAVES;
  static_assert(LOADS * 8 * WAVES == BM + BN, "whole loads");
  extern __shared__ gf4 gf_sums[];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), i = lane % 16, g = lane / 16;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN, wm = wave / WN * 32, wn = wave % WN * 32;
  const float* src[LOADS];   // this lane's share of a block: 16 bytes of eight rows
#pragma unroll
  for (int u = 0; u < LOADS; ++u) {
    const int row = 8 * (u * WAVES + wave) + lane / 8;
    src[u] = (row < BM ? p.a + (int64_t)min(m0 + row, p.m - 1) * p.lda : p.w + (int64_t)min(n0 + row - BM, p.n - 1) * p.ldw) +
             4 * (lane % 8 ^ gf_turn(row));
  }
  const auto load = [&](int block) {
#pragma unroll
    for (int u = 0; u < LOADS; ++u) gf_to_lds(src[u] + block * GF_BK, gf_sums + block % STAGES * STAGE + (u * WAVES + wave) * 64);
  };
  const int blocks = p.k / GF_BK, seg_blocks = p.seg_runs * (GF_RUN / GF_BK);
#pragma unroll
  for (int b = 0; b < STAGES - 1; ++b)
    if (b < blocks) load(b);
  gf4 total[2][2], seg[2][2], acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) total[x][y] = seg[x][y] = acc[x][y] = gf4{0.f, 0.f, 0.f, 0.f};
  const int turn = gf_turn(i);
  for (int b = 0; b < blocks; ++b) {
    gf_wait_lds();   // what was read of the stage that is loaded next
    if (b + STAGES - 2 < blocks) gf_wait<(STAGES - 2) * LOADS>();
    else gf_wait<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (b + STAGES - 1 < blocks) load(b + STAGES - 1);
    const gf4 *ca = gf_sums + b % STAGES * STAGE + (wm + i) * 8, *cw = gf_sums + b % STAGES * STAGE + (BM + wn + i) * 8;
    gf4 fa[GF_BK / 16][2], fw[GF_BK / 16][2];
#pragma unroll
    for (int t = 0; t < GF_BK / 16; ++t)
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        fa[t][x] = ca[16 * x * 8 + (4 * t + g ^ turn)];
        fw[t][x] = cw[16 * x * 8 + (4 * t + g ^ turn)];
      }
#pragma unroll
    for (int t = 0; t < GF_BK / 16; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[t][x][e], fw[t][y][e], acc[x][y], 0, 0, 0);
    const bool last = b + 1 == blocks;
    if (!last && (b + 1) % (GF_RUN / GF_BK) != 0) continue;
    const bool seg_ends = last || (b + 1) % seg_blocks == 0;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        seg[x][y] += acc[x][y];
        acc[x][y] = gf4{0.f, 0.f, 0.f, 0.f};
        if (seg_ends) {
          total[x][y] += seg[x][y];
          seg[x][y] = gf4{0.f, 0.f, 0.f, 0.f};
        }
      }
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) gf_store(p, total[x][y], m0 + wm + 16 * x, n0 + wn + 16 * y, i, g);
}

template <int NT, int KW, int READ, int FORM>
static int gf_few_launch(const GfArgs& p, const GfAround& x, int grid, hipStream_t stream) {
  // (sums: at most 16 KiB a tile; what a wave stages: 8)
  const size_t lds = (size_t)p.segments * NT * 64 * sizeof(gf4) + (READ == GF_STAGED ? KW * 8192 : 0);
  const auto kernel = gemm_f32_few_kernel<NT, KW, READ, FORM>;
  if (lds > 65536 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, KW * 8192 + 16 * 1024) != hipSuccess)
    return DLI_ERR_LAUNCH;
  kernel<<<grid, 64 * KW, lds, stream>>>(p, x);
  return dli_launch_status();
}

template <int NT, int KW>
static int gf_few(const GfArgs& p, bool vec, hipStream_t stream) {
  const int grid = (p.n + 16 * NT - 1) / (16 * NT);
  if constexpr (NT == 1)
    if (vec && p.k % (GF_RUN / 2) == 0) return gf_few_launch<1, KW, GF_STAGED, GF_PLAIN>(p, GfAround{}, grid, stream);
  return vec ? gf_few_launch<NT, KW, GF_WIDE, GF_PLAIN>(p, GfAround{}, grid, stream) : gf_few_launch<NT, KW, GF_WORDS, GF_PLAIN>(p, GfAround{}, grid, stream);
}

template <int KW, int FORM>
static int gf_few_form(const GfArgs& p, const GfAround& x, int grid, hipStream_t stream) {
  return p.k % (GF_RUN / 2) == 0 ? gf_few_launch<1, KW, GF_STAGED, FORM>(p, x, grid, stream) : gf_few_launch<1, KW, GF_WIDE, FORM>(p, x, grid, stream);
}

template <int FORM>
static int gf_few_around(const GfArgs& p, const GfAround& x, int rule, int grid, hipStream_t stream) {
  switch (rule) {
    case 0: return gf_few_form<16, FORM>(p, x, grid, stream);
    case 1: return gf_few_form<8, FORM>(p, x, grid, stream);
    default: return gf_few_form<4, FORM>(p, x, grid, stream);
  }
}

template <int WM, int WN, int KG>
static int gf_tiles(const GfArgs& p, bool vec, hipStream_t stream) {
  const dim3 grid((p.n + 32 * WN - 1) / (32 * WN), (p.m + 32 * WM - 1) / (32 * WM));
  if (grid.y > 65535) return DLI_ERR_ARGUMENT;
  // (KG of 4 and 8: 72 and 144 KiB, where up to 64 KiB of segments' sums find room afterwards)
  constexpr size_t lds = (size_t)KG * 2 * 32 * (WM + WN) * GF_LD * sizeof(float);
  static_assert(KG == 1 || (KG >= 4 && lds >= (size_t)GF_SEGMENTS * 4 * 64 * sizeof(gf4)), "room for the segments' sums");
  const auto kernel = vec ? gemm_f32_tile_kernel<WM, WN, KG, true> : gemm_f32_tile_kernel<WM, WN, KG, false>;
  if (lds > 65536 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
    return DLI_ERR_LAUNCH;
  kernel<<<grid, 64 * WM * WN * KG, lds, stream>>>(p);
  return dli_launch_status();
}

template <int WM, int WN, int STAGES>
static int gf_ahead(const GfArgs& p, hipStream_t stream) {
  const dim3 grid((p.n + 32 * WN - 1) / (32 * WN), (p.m + 32 * WM - 1) / (32 * WM));
  if (grid.y > 65535) return DLI_ERR_ARGUMENT;
  constexpr size_t lds = (size_t)STAGES * 32 * (WM + WN) * GF_BK * sizeof(float);
  const auto kernel = gemm_f32_ahead_kernel<WM, WN, STAGES>;
  if (lds > 65536 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return DLI_ERR_LAUNCH;
  kernel<<<grid, 64 * WM * WN, lds, stream>>>(p);
  return dli_launch_status();
}

// Which kernel takes m rows, n columns and `segments` segments: 0 to 3 the few-row kernel, from sixteen waves a tile down to two for
// two tiles, 4 to 7 the tile kernel, from eight waves a tile of 32 x 32 up to tiles of 128 x 64.
// As many waves as the device has SIMDs, where the sum has segments enough: 498 x 3072 x 576 (1,536 tiles) takes 32.6 us
// with four waves a tile and 44 with tiles of 64 x 64 for four waves (28.5 where those have loads ahead); 2048 x 16384 x 2048
// 1,280 us in tiles of 128 x 64 (1,128).
static int gf_rule(int m, int n, int segments) {
  const int64_t simds = 4 * dli_compute_units();
  if (m <= 16) {
    const int64_t tiles = (n + 15) / 16;
    if (segments > 8 && tiles * 8 < 2 * simds) return 0;
    if (segments > 4 && tiles * 4 < 2 * simds) return 1;
    return segments >= 2 && tiles < 8 * simds ? 2 : 3;
  }
  const int64_t tiles = (int64_t)((n + 31) / 32) * ((m + 31) / 32);
  if (tiles * 4 <= simds && segments > 4) return 4;
  if (tiles <= 2 * simds && segments >= 2) return 5;
  return tiles < 8 * simds ? 6 : 7;
}

// Where the rule names four waves a tile of 32 x 32: whether tiles of 64 x 64 with loads ahead take less, by how many of either a
// compute unit gets. (Rows that half fill their last tile of 64, and tiles just past a round, make many of them.) us with four
// waves a tile and with loads ahead, m x n, tiles of either on the busiest unit:
//   k 576    24 x 12,198  2 1  13.8 16.8   192 x 2,800  3 1  21.0 17.6   556 x 1,826  5 2  29.2 25.7   1,004 x 1,378  6 2  34.0 26.5
//   k 960    1,265 x 302  2 1  17.8 25.3   192 x 2,800  3 1  26.7 25.8   556 x 1,826  5 2  39.0 39.8   1,004 x 1,378  6 2  45.9 40.6
//   k 2,048  28 x 14,961  2 1  33.4 48.3   192 x 2,800  3 1  48.0 48.6   700 x 1,280  4 1  57.1 48.6   556 x 1,826    5 2  74.6 79.8
//            1,004 x 1,378  6 2  84.4 78.7   93 x 10,291  4 2  63.0 80.4   757 x 2,716  8 3  118 122
extern "C" int dli_gemm_f32_few_waves_ahead(int m, int n, int k, int units) {
  const auto on_a_unit = [&](int side) {
    const int64_t tiles = (int64_t)((n + side - 1) / side) * ((m + side - 1) / side);
    return (tiles + units - 1) / units;
  };
  const int64_t small = on_a_unit(32), large = on_a_unit(64);
  if (k < 960 || (k <= 1024 && large == 1)) return small > 2 * large;
  return small >= (large == 1 ? 4 : 3 * large);
}

// The order of a sum over k: `segments` of `seg_runs` runs each.
static void gf_order(int k, int& segments, int& seg_runs) {
  const int runs = (k + GF_RUN - 1) / GF_RUN;
  seg_runs = (runs + GF_SEGMENTS - 1) / GF_SEGMENTS;
  segments = (runs + seg_runs - 1) / seg_runs;
}

extern "C" int dli_gemm_f32_rule(int m, int n, int k) {
  if (m <= 0 || n <= 0 || k <= 0) return -1;
  int segments, seg_runs;
  gf_order(k, segments, seg_runs);
  return gf_rule(m, n, segments);
}

extern "C" int dli_gemm_f32_nt(const float* a, int64_t lda, const float* w, int64_t ldw,
                               const float* bias, const float* residual, int64_t ldr, float* out,
                               int64_t ldo, int m, int n, int k, hipStream_t stream) {
  if (m <= 0 || n <= 0) return DLI_OK;
  if (k <= 0 || lda < k || ldw < k || ldo < n || (residual != nullptr && ldr < n)) return DLI_ERR_ARGUMENT;
  int segments, seg_runs;
  gf_order(k, segments, seg_runs);
  const GfArgs p = {a, w, bias, residual, out, lda, ldw, ldr, ldo, m, n, k, segments, seg_runs};
  const bool vec = k % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && (((uintptr_t)a | (uintptr_t)w) % 16) == 0;
  const bool ahead = vec && k % GF_BK == 0;
  switch (gf_rule(m, n, segments)) {
    case 0: return gf_few<1, 16>(p, vec, stream);
    case 1: return gf_few<1, 8>(p, vec, stream);
    case 2: return gf_few<1, 4>(p, vec, stream);
    case 3: return gf_few<2, 2>(p, vec, stream);
    case 4: return gf_tiles<1, 1, 8>(p, vec, stream);
    case 5: return ahead && dli_gemm_f32_few_waves_ahead(m, n, k, dli_compute_units()) ? gf_ahead<2, 2, 4>(p, stream) : gf_tiles<1, 1, 4>(p, vec, stream);
    case 6: return ahead ? gf_ahead<2, 2, 3>(p, stream) : gf_tiles<2, 2, 1>(p, vec, stream);
    default: return ahead ? gf_ahead<4, 2, 3>(p, stream) : gf_tiles<4, 2, 1>(p, vec, stream);
  }
}

// The few-row products of a decode step behind a norm: act = silu(gate) * up of rms_norm(x) (positions null; w: the gates' rows,
// then the ups'), or q, k and v of it, rotated and written (q to `out`). Up to 16 rows, k a multiple of eight, heads of
// whole tiles, x, w and norm_w of whole vectors: what else there is takes the kernels one by one.
extern "C" int dli_gemm_f32_normed(const float* x, int64_t ldx, const float* w, const float* bias, const float* norm_w, float eps,
                                   float* out, int64_t ldo, int m, int n, int k, const int* positions, const float* inv_freq,
                                   const int* slots, float* k_pages, float* v_pages, int q_heads, int kv_heads, int head_dim,
                                   int page_size, hipStream_t stream) {
  if (m <= 0) return DLI_OK;
  if (m > 16 || n <= 0 || k <= 0 || k % 8 != 0 || ldx < k || ldx % 4 != 0 ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)norm_w) % 16) != 0)
    return DLI_ERR_ARGUMENT;
  int segments, seg_runs;
  gf_order(k, segments, seg_runs);
  const GfArgs p = {x, w, bias, nullptr, out, ldx, k, 0, ldo, m, n, k, segments, seg_runs};
  const int threads = k / 8 >= 256 ? 256 : (k / 8 >= 128 ? 128 : 64);   // (as dli_rms_norm's)
  const GfAround around = {norm_w, eps, threads / 64, positions, inv_freq, slots, k_pages, v_pages, q_heads, kv_heads, head_dim, page_size};
  const int rule = gf_rule(m, n, segments);
  if (positions == nullptr) {
    if (n % 2 != 0 || ldo < n / 2) return DLI_ERR_ARGUMENT;
    return gf_few_around<GF_GLU>(p, around, rule, (n / 2 + 7) / 8, stream);
  }
  if (inv_freq == nullptr || slots == nullptr || k_pages == nullptr || v_pages == nullptr || q_heads <= 0 || kv_heads <= 0 ||
      head_dim <= 0 || head_dim % 16 != 0 || page_size <= 0 || n != (q_heads + 2 * kv_heads) * head_dim || ldo < q_heads * head_dim)
    return DLI_ERR_ARGUMENT;
  return gf_few_around<GF_ROPE>(p, around, rule, n / 16, stream);
}
