// Feed-forward layers beyond the gated product: a polynomial activation with norms, and a mixture of
// small experts with a router. T is the type of what the matrix products read and write (float on the
// 32-bit path, bf16 when serving); statistics, the router and every sum are 32-bit.
//
//   poly_norm        out(T) = a N(z) + b N(z^2) + c N(z^3) + e, powers element by element, N(x) = x / sqrt(mean(x^2) + eps)
//                    over the row; z is the 32-bit result of the product before it
//   clamped_glu      y = g sigmoid(alpha g) (u + shift), g = min(gate, limit), u = clamp(up, -limit, limit); an infinite
//                    limit, alpha 1 and shift 0 give the plain silu(gate) * up
//   gelu_glu         y = gelu(gate) * up, tanh form (the same kernels)
//   router_choose    softmax over all router outputs, or the sigmoid of each; choice = score + correction; only the
//                    `keep` groups of neighbours with the largest best choice stay; the `top` largest choices; weights =
//                    the chosen scores (without correction) / (their sum + 1e-20) * scale, or scores * scale alone
//   expert_sort      the (token, choice) slots of real experts in runs by expert, and the list of row tiles
//   expert_up/down   the experts' products over those tiles (on the matrix cores for bfloat16 and sizes that are
//                    multiples of 32, else on the vector units, any size), the clamped activation between
//                    them; the down product leaves each slot's 32-bit result in the slot's own row. Where a slot's
//                    weight belongs on the expert's input, the up kernels multiply their 32-bit sums by it
//   expert_combine   out = sum_j w_j (expert j's result, or the input itself for an identity expert)
//                    + sigmoid(shared gate) * shared expert's result
//
// A row's result never depends on its place in a tile or on the other rows: every output sums its k in
// ascending order.
#include <type_traits>

#include "common.h"

// A workgroup a row. Bound by the trips to memory of a thread's values, which are asked for together and held for the second
// pass (the first POLY_HELD of a thread; longer rows read the rest twice): us a call, 4 and 3,000 rows
// of 8,192, one value after the other 7.4 and 47.3, now 4.0 and 29.0.
#define POLY_HELD 16
template <int HELD>   // (short rows hold what they have: 3,000 rows of 192 values 5.5 us, with sixteen rounds of loads 8.8)
__global__ __launch_bounds__(512) void poly_norm_kernel_f32in(const float* __restrict__ z, int64_t z_stride, const float* __restrict__ coef,
                                                              void* __restrict__ out_, int64_t out_stride, int ff, float eps, int out_is_bf16) {
  __shared__ float scratch[3][16];
  const int64_t row = blockIdx.x;
  const float* zr = z + row * z_stride;
  const int lane = threadIdx.x % DLI_WAVE, wave = threadIdx.x / DLI_WAVE, waves = blockDim.x / DLI_WAVE;
  const float a = coef[0], b = coef[1], c = coef[2], e = coef[3];
  float held[HELD];
#pragma unroll
  for (int k = 0; k < HELD; ++k) held[k] = zr[min((int)(threadIdx.x + k * blockDim.x), ff - 1)];
  float s2 = 0.f, s4 = 0.f, s6 = 0.f;
  auto add = [&](float x) {
    const float x2 = x * x, x3 = x2 * x;
    s2 += x2;
    s4 += x2 * x2;
    s6 += x3 * x3;
  };
#pragma unroll
  for (int k = 0; k < HELD; ++k)
    if ((int)(threadIdx.x + k * blockDim.x) < ff) add(held[k]);
  for (int i = threadIdx.x + HELD * blockDim.x; i < ff; i += blockDim.x) add(zr[i]);
  // the three sums meet in one exchange through LDS
  s2 = wave_sum(s2); s4 = wave_sum(s4); s6 = wave_sum(s6);
  if (lane == 0) { scratch[0][wave] = s2; scratch[1][wave] = s4; scratch[2][wave] = s6; }
  __syncthreads();
  float t2 = 0.f, t4 = 0.f, t6 = 0.f;
  for (int w = 0; w < waves; ++w) { t2 += scratch[0][w]; t4 += scratch[1][w]; t6 += scratch[2][w]; }   // same order in every thread
  const float r1 = 1.f / sqrtf(t2 / (float)ff + eps), r2 = 1.f / sqrtf(t4 / (float)ff + eps), r3 = 1.f / sqrtf(t6 / (float)ff + eps);
  auto put = [&](int i, float x) {
    const float x2 = x * x;
    const float y = a * (x * r1) + b * (x2 * r2) + c * ((x2 * x) * r3) + e;
    if (out_is_bf16) ((bf16_t*)out_)[row * out_stride + i] = (bf16_t)y;
    else ((float*)out_)[row * out_stride + i] = y;
  };
#pragma unroll
  for (int k = 0; k < HELD; ++k) {
    const int i = threadIdx.x + k * blockDim.x;
    if (i < ff) put(i, held[k]);
  }
  for (int i = threadIdx.x + HELD * blockDim.x; i < ff; i += blockDim.x) put(i, zr[i]);
}

template <typename T>
__global__ void clamped_glu_kernel(const T* __restrict__ gate_up, int64_t stride, T* __restrict__ out, int ff, GluForm f) {
  const int64_t row = blockIdx.x;
  const int i = blockIdx.y * blockDim.x + threadIdx.x;
  if (i >= ff) return;
  const float g = to_f32(gate_up[row * stride + i]), u = to_f32(gate_up[row * stride + ff + i]);
  out[row * ff + i] = from_f32<T>(f.form == GLU_GELU ? gelu_glu(g, u) : clamped_glu(g, u, f.limit, f.alpha, f.up_shift));
}

// Eight neighbours a thread (rows and sizes of whole 16 bytes).
template <bool GELU>
__global__ __launch_bounds__(256) void clamped_glu_bf16x8_kernel(const bf16_t* __restrict__ gate_up, int64_t stride,
                                                                 bf16_t* __restrict__ out, int ff, GluForm f) {
  typedef __bf16 b8 __attribute__((ext_vector_type(8)));
  const int64_t row = blockIdx.x;
  const int i = 8 * (blockIdx.y * 256 + threadIdx.x);
  if (i >= ff) return;
  const b8 g = *reinterpret_cast<const b8*>(gate_up + row * stride + i);
  const b8 u = *reinterpret_cast<const b8*>(gate_up + row * stride + ff + i);
  b8 y;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (GELU) {
      const float z = (float)g[e];
      y[e] = (bf16_t)(z * __builtin_amdgcn_rcpf(1.f + __expf(-1.5957691216057308f * (z + 0.044715f * z * z * z))) * (float)u[e]);
    } else {
      const float a = fminf((float)g[e], f.limit), b = fminf(fmaxf((float)u[e], -f.limit), f.limit);
      y[e] = (bf16_t)(a * __builtin_amdgcn_rcpf(1.f + __expf(-f.alpha * a)) * (b + f.up_shift));
    }
  }
  *reinterpret_cast<b8*>(out + row * ff + i) = y;
}

// The better of two (value, index) pairs: the larger value, the lower index on a tie.
__device__ __forceinline__ void wave_argmax(float& v, int& i) {
#pragma unroll
  for (int m = DLI_WAVE / 2; m > 0; m >>= 1) {
    const float v2 = __shfl_xor(v, m, DLI_WAVE);
    const int i2 = __shfl_xor(i, m, DLI_WAVE);
    if (v2 > v || (v2 == v && i2 < i)) { v = v2; i = i2; }
  }
}

// A wave a token. logits [rows][stride]: the first `total` columns are the router's outputs.
__global__ __launch_bounds__(64) void router_choose_kernel(const float* __restrict__ logits, int64_t stride,
                                                           const float* __restrict__ bias,
                                                           const float* __restrict__ correction, int total, int count,
                                                           int keep, int top, float scale, int sigmoid, int normalize,
                                                           int* __restrict__ ids, float* __restrict__ weights) {
  extern __shared__ float sh[];
  float *s = sh, *choice = sh + total, *gbest = sh + 2 * total;
  const int64_t row = blockIdx.x;
  const int lane = threadIdx.x;
  const float* z = logits + row * stride;
  float m = -INFINITY, sum = 0.f;
  if (sigmoid) {
    for (int i = lane; i < total; i += DLI_WAVE) s[i] = 1.f / (1.f + expf(-(z[i] + (bias != nullptr ? bias[i] : 0.f))));
    sum = 1.f;
  } else {
    for (int i = lane; i < total; i += DLI_WAVE) m = fmaxf(m, z[i] + (bias != nullptr ? bias[i] : 0.f));
    m = wave_max(m);
    for (int i = lane; i < total; i += DLI_WAVE) {
      const float e = expf(z[i] + (bias != nullptr ? bias[i] : 0.f) - m);
      s[i] = e;
      sum += e;
    }
    sum = wave_sum(sum);
  }
  for (int i = lane; i < total; i += DLI_WAVE) {
    const float p = s[i] / sum;
    s[i] = p;
    choice[i] = p + (correction != nullptr ? correction[i] : 0.f);
  }
  __syncthreads();
  if (count > 1) {
    const int per = total / count;
    for (int g = lane; g < count; g += DLI_WAVE) {
      float b = -INFINITY;
      for (int i = g * per; i < (g + 1) * per; ++i) b = fmaxf(b, choice[i]);
      gbest[g] = b;
    }
    __syncthreads();
    for (int round = 0; round < keep; ++round) {
      float bv = -INFINITY;
      int bi = 0x7fffffff;
      for (int g = lane; g < count; g += DLI_WAVE) {
        const float v = gbest[g];
        if (v == v && (v > bv || (v == bv && g < bi))) { bv = v; bi = g; }   // (NaN marks a group already kept)
      }
      wave_argmax(bv, bi);
      __syncthreads();
      if (lane == 0 && bi < count) gbest[bi] = __builtin_nanf("");
      __syncthreads();
    }
    for (int i = lane; i < total; i += DLI_WAVE) {
      const float g = gbest[i / per];
      if (g == g) choice[i] = -INFINITY;        // its group was not kept
    }
    __syncthreads();
  }
  float chosen_sum = 0.f, mine = 0.f;            // lane j keeps the j-th choice (top <= 64)
  int my_id = 0;
  for (int j = 0; j < top; ++j) {
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for (int i = lane; i < total; i += DLI_WAVE) {
      const float v = choice[i];
      if (v == v && (v > bv || (v == bv && i < bi))) { bv = v; bi = i; }      // (NaN marks an expert already chosen)
    }
    wave_argmax(bv, bi);
    bi = min(bi, total - 1);
    __syncthreads();
    const float p = s[bi];
    chosen_sum += p;
    if (lane == j) { mine = p; my_id = bi; }
    if (lane == 0) choice[bi] = __builtin_nanf("");
    __syncthreads();
  }
  if (lane < top) {
    ids[row * top + lane] = my_id;
    weights[row * top + lane] = (normalize ? mine / (chosen_sum + 1e-20f) : mine) * scale;
  }
}

#define EX_BM 32
#define EX_BN 64
#define EX_BK 16

// One workgroup. ids [slots]: the chosen expert of every (token, choice) slot; ids at or above `experts`
// (identity experts) have no rows. Leaves offsets [experts + 1], order [rows of real experts] (the slot of
// every sorted row; inside an expert's run the rows come in whatever order the counter hands out, which
// no value depends on), the tiles (expert, first sorted row) of at most tile_rows rows, and their number.
//
// The runs' and tiles' first places are sums over the experts before: in-wave sums, the waves' totals through LDS, 1024 experts at
// a time. (One thread that walked the experts took 1.3 us longer at 32 experts and 7.4 at 128, 8 slots; 35 at 256, 4,096 slots.)
__device__ __forceinline__ int sum_before(int v) {   // over the lanes before this one
  const int lane = threadIdx.x % DLI_WAVE;
  int s = v;
#pragma unroll
  for (int d = 1; d < DLI_WAVE; d <<= 1) {
    const int up = __shfl_up(s, d, DLI_WAVE);
    s += lane >= d ? up : 0;
  }
  return s - v;
}
// With a table (TableChoice) the kernel looks the choices up itself and writes them and their weights: a kernel of its own for that took
// 4.3 us a layer of a step of two rows, this one takes 4.7 without it and 4.6 with it (9,216 slots, nine a thread: about as much longer as it saves, so not there).
struct TableChoice { const int* table; const int* token_ids; int vocab, top; float* weights; };
__device__ __forceinline__ int table_choice(const int* table, const int* token_ids, int vocab, int top, int i) {
  const int t = i / top, tok = min(max(token_ids[t], 0), vocab - 1);
  return table[(int64_t)tok * top + i - t * top];
}
__global__ __launch_bounds__(1024) void expert_sort_kernel(int* ids, TableChoice choice, int slots, int experts,
                                                           int* __restrict__ offsets, int* __restrict__ order,
                                                           int* __restrict__ tile_expert, int* __restrict__ tile_row0,
                                                           int* __restrict__ tile_count, int max_tiles, int tile_rows) {
  extern __shared__ int shi[];
  __shared__ int rows_of[16], tiles_of[16];
  int *counts = shi, *cursor = shi + experts;
  const int lane = threadIdx.x % DLI_WAVE, wave = threadIdx.x / DLI_WAVE;
  for (int e = threadIdx.x; e < experts; e += 1024) counts[e] = 0;
  __syncthreads();
  int own = -1;   // the first slot's choice (the others are read once more)
  for (int i = threadIdx.x; i < slots; i += 1024) {
    int e;
    if (choice.table != nullptr) {
      e = table_choice(choice.table, choice.token_ids, choice.vocab, choice.top, i);
      ids[i] = e;
      choice.weights[i] = 1.f / (float)choice.top;
    } else {
      e = ids[i];
    }
    if (i == (int)threadIdx.x) own = e;
    if (e >= 0 && e < experts) atomicAdd(&counts[e], 1);
  }
  __syncthreads();
  int at = 0, tiles = 0;                                        // of the experts before these 1024
  for (int e0 = 0; e0 < experts; e0 += 1024) {
    const int e = e0 + threadIdx.x, rows = e < experts ? counts[e] : 0, parts = (rows + tile_rows - 1) / tile_rows;
    int row = sum_before(rows), tile = sum_before(parts);
    if (lane == DLI_WAVE - 1) { rows_of[wave] = row + rows; tiles_of[wave] = tile + parts; }
    __syncthreads();
    row += at;
    tile += tiles;
    for (int w = 0; w < 16; ++w) {
      const int r = rows_of[w], t = tiles_of[w];
      if (w < wave) { row += r; tile += t; }
      at += r;
      tiles += t;
    }
    if (e < experts) {
      offsets[e] = row;
      cursor[e] = row;
      for (int k = 0; k < parts && tile + k < max_tiles; ++k) {
        tile_expert[tile + k] = e;
        tile_row0[tile + k] = row + k * tile_rows;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    offsets[experts] = at;
    tile_count[0] = min(tiles, max_tiles);
  }
  for (int i = threadIdx.x; i < slots; i += 1024) {
    const int e = i == (int)threadIdx.x ? own : ids[i];
    if (e >= 0 && e < experts) order[atomicAdd(&cursor[e], 1)] = i;
  }
}

struct ExpertArgs {
  const int* tile_expert; const int* tile_row0; const int* tile_count; const int* offsets; const int* order;
  int top, width, ff;
  const float* in_weight;   // [slots], what multiplies an expert's input (nullptr: nothing)
};

// y[sorted row][ff] = clamped_glu(h[token] . w_gate[e], h[token] . w_up[e]); w_gate, w_up [experts][ff][width].
template <typename T>
__global__ __launch_bounds__(256) void expert_up_kernel(ExpertArgs p, const T* __restrict__ h, int64_t h_stride,
                                                        const T* __restrict__ w_gate, const T* __restrict__ w_up,
                                                        T* __restrict__ y, float limit, float alpha, float up_shift) {
  const int tile = blockIdx.x;
  if (tile >= p.tile_count[0]) return;
  __shared__ float as[EX_BK][EX_BM + 1], gs[EX_BK][EX_BN + 4], us[EX_BK][EX_BN + 4];
  __shared__ int tok[EX_BM];
  const int e = p.tile_expert[tile], r0 = p.tile_row0[tile], rend = p.offsets[e + 1];
  const int n0 = blockIdx.y * EX_BN;
  const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
  if (tid < EX_BM) tok[tid] = r0 + tid < rend ? p.order[r0 + tid] / p.top : -1;
  __syncthreads();
  const T* wg = w_gate + (int64_t)e * p.ff * p.width;
  const T* wu = w_up + (int64_t)e * p.ff * p.width;
  float accg[2][4] = {}, accu[2][4] = {};
  for (int k0 = 0; k0 < p.width; k0 += EX_BK) {
    for (int i = tid; i < EX_BM * EX_BK; i += 256) {
      const int r = i / EX_BK, k = i % EX_BK;
      as[k][r] = tok[r] >= 0 && k0 + k < p.width ? to_f32(h[(int64_t)tok[r] * h_stride + k0 + k]) : 0.f;
    }
    for (int i = tid; i < EX_BN * EX_BK; i += 256) {
      const int c = i / EX_BK, k = i % EX_BK;
      const bool ok = n0 + c < p.ff && k0 + k < p.width;
      gs[k][c] = ok ? to_f32(wg[(int64_t)(n0 + c) * p.width + k0 + k]) : 0.f;
      us[k][c] = ok ? to_f32(wu[(int64_t)(n0 + c) * p.width + k0 + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EX_BK; ++k) {
      const float a0 = as[k][ty * 2], a1 = as[k][ty * 2 + 1];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float g = gs[k][tx * 4 + j], u = us[k][tx * 4 + j];
        accg[0][j] = fmaf(a0, g, accg[0][j]);
        accg[1][j] = fmaf(a1, g, accg[1][j]);
        accu[0][j] = fmaf(a0, u, accu[0][j]);
        accu[1][j] = fmaf(a1, u, accu[1][j]);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = r0 + ty * 2 + i;
    if (r >= rend) continue;
    const float iw = p.in_weight != nullptr ? p.in_weight[p.order[r]] : 1.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = n0 + tx * 4 + j;
      if (c < p.ff) y[(int64_t)r * p.ff + c] = from_f32<T>(clamped_glu(iw * accg[i][j], iw * accu[i][j], limit, alpha, up_shift));
    }
  }
}

// z[slot][width] = y[sorted row] . w_down[e]; w_down [experts][width][ff].
template <typename T>
__global__ __launch_bounds__(256) void expert_down_kernel(ExpertArgs p, const T* __restrict__ y, const T* __restrict__ w_down,
                                                          float* __restrict__ z) {
  const int tile = blockIdx.x;
  if (tile >= p.tile_count[0]) return;
  __shared__ float as[EX_BK][EX_BM + 1], ws[EX_BK][EX_BN + 4];
  const int e = p.tile_expert[tile], r0 = p.tile_row0[tile], rend = p.offsets[e + 1];
  const int n0 = blockIdx.y * EX_BN;
  const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
  const T* wd = w_down + (int64_t)e * p.width * p.ff;
  float acc[2][4] = {};
  for (int k0 = 0; k0 < p.ff; k0 += EX_BK) {
    for (int i = tid; i < EX_BM * EX_BK; i += 256) {
      const int r = i / EX_BK, k = i % EX_BK;
      as[k][r] = r0 + r < rend && k0 + k < p.ff ? to_f32(y[(int64_t)(r0 + r) * p.ff + k0 + k]) : 0.f;
    }
    for (int i = tid; i < EX_BN * EX_BK; i += 256) {
      const int c = i / EX_BK, k = i % EX_BK;
      ws[k][c] = n0 + c < p.width && k0 + k < p.ff ? to_f32(wd[(int64_t)(n0 + c) * p.ff + k0 + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EX_BK; ++k) {
      const float a0 = as[k][ty * 2], a1 = as[k][ty * 2 + 1];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float w = ws[k][tx * 4 + j];
        acc[0][j] = fmaf(a0, w, acc[0][j]);
        acc[1][j] = fmaf(a1, w, acc[1][j]);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = r0 + ty * 2 + i;
    if (r >= rend) continue;
    const int64_t slot = p.order[r];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = n0 + tx * 4 + j;
      if (c < p.width) z[slot * p.width + c] = acc[i][j];
    }
  }
}

// The same two products on the matrix cores (bfloat16; width and ff multiples of 32): tiles of 16 MB sorted rows, a
// workgroup of four waves takes 64 NB features, each wave 16 NB of them for all rows of the tile.
// v_mfma_f32_16x16x32_bf16 with the weights as the first operand: lane l supplies feature l % 16 of a block and row
// l % 16 of each block of 16 rows, and the eight k values 8 (l / 16) .. + 7 of a step of 32, read straight from memory (16
// bytes a lane and operand; the rows of a tile are re-read by the four waves from the cache); the operands of the next
// step are on their way while a step's products are issued. A lane's results are four neighbouring features of one row.
// Every output sums its k in ascending steps of 32 whatever its tile, so a row's result depends on
// nothing beside the row.
#define EXM_BM 64
#define EXM_FEW 16
typedef __bf16 exm_bf16x8 __attribute__((ext_vector_type(8)));
typedef float exm_float4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ exm_bf16x8 exm_load(const bf16_t* p) { return *reinterpret_cast<const exm_bf16x8*>(p); }

// Few rows an expert: the products wait for the weights alone. Lanes that read 16 rows at once, as the operands ask for them, get
// a quarter of the cache's rate and 16 pages a load, so the weights pass through LDS: a workgroup takes 32 rows of weights (16
// gate rows and their 16 up rows, or 32 of the down product) and up to 16 rows of the input, in chunks of 256 k, a half wave a row
// (512 neighbouring bytes), EXF_AHEAD chunks on their way in registers and two in LDS; two of the four waves issue the products.
// Piece p (16 bytes) of row r lies at place p ^ (r % 16), so that the 16 rows of an operand lie in different banks. Sums run over
// k in ascending steps of 32, as in the other kernels, and have the same bits.
// Us of the up and down product with a wave a block of 16 features, eight steps ahead -> now: 32 experts of 1,024 on 2,048, 2 rows
// (8 experts, 67 and 34 MB) 38.7 -> 15.1 and 9.1 -> 8.4, 32 rows (260 MB) 68 -> 51; 64 experts of 1,408, 32 rows (704 MB) 157 ->
// 117 (6.0 TB/s); 8 of 2,048 on 4,096, 1 row (67 MB) 72.5 -> 17.3. Four chunks ahead: the same.
#define EXF_K 256
#define EXF_AHEAD 3
// A few choices: every workgroup sorts them for itself, a choice a lane, and no kernel does it before. That kernel takes 4.5 us; sorting
// here takes the longer the more choices there are, in every workgroup of both products. All of it, us, by the kernel and here, at 4, 8,
// 16, 32 and 64 choices: 4 of 32 experts, 1,024 of 2,048 wide 20.4 17.6, 26.9 24.8, 48 48, 68 78, 80 101; 512 of 1,024 14.2 11.6, 16.6
// 13.7, 20.4 21.0, 31.7 38, 36.6 46; 8 of 64, 256 of 1,024 (8 on) 14.1 11.7, 17.2 16.5, 21.4 25.3, 33.3 51.8; one of 128, 128 of 512 11.6
// 9.0, 12.1 9.9, 12.7 11.5, 14.3 15.7, 18.9 30.
#define EXF_SLOTS 16
static_assert(EXF_SLOTS <= DLI_WAVE, "a choice a lane");
struct FewChoices {
  int* ids; TableChoice choice;   // choice.table: looked up, and written to ids with the weights by the first workgroup of the up product
  int slots, experts;
};
// Tile `tile`: its expert, first sorted row and the last's end; -1 where there are not so many. order[sorted row]: the slot (every wave
// leaves all of it). Inside an expert's run the rows come in the order of their slots.
__device__ __forceinline__ int few_tile(const FewChoices& f, bool writes, int tile, int* order, int& r0, int& rend) {
  const int lane = threadIdx.x % DLI_WAVE, slot = min(lane, f.slots - 1);
  const int chosen = f.choice.table != nullptr ? table_choice(f.choice.table, f.choice.token_ids, f.choice.vocab, f.choice.top, slot) : f.ids[slot];
  if (writes && (int)threadIdx.x < f.slots) {
    f.ids[slot] = chosen;
    f.choice.weights[slot] = 1.f / (float)f.choice.top;
  }
  const int e = lane < f.slots && chosen >= 0 && chosen < f.experts ? chosen : f.experts;   // (those without rows behind all others)
  int before = 0, among = 0;                                    // sorted rows before this one, and of its own expert
  for (int j = 0; j < f.slots; ++j) {
    const int other = __builtin_amdgcn_readlane(e, j);
    before += other < e || (other == e && j < lane) ? 1 : 0;
    among += other == e && j < lane ? 1 : 0;
  }
  const bool live = e < f.experts, first = live && among % EXM_FEW == 0;
  int tiles = 0;                                                // before this row's
  for (unsigned long long left = __ballot(first); left != 0; left &= left - 1)
    tiles += __builtin_amdgcn_readlane(before, __builtin_ctzll(left)) < before ? 1 : 0;
  if (live) order[before] = lane;
  const unsigned long long mine = __ballot(first && tiles == tile);
  if (mine == 0) return -1;
  const int at = __builtin_ctzll(mine), expert = __builtin_amdgcn_readlane(e, at);
  r0 = __builtin_amdgcn_readlane(before, at);
  rend = min(r0 + EXM_FEW, r0 - __builtin_amdgcn_readlane(among, at) + (int)__popcll(__ballot(e == expert)));
  return expert;
}

template <bool UP, bool SORTS>
__global__ __launch_bounds__(256) void expert_few_kernel(ExpertArgs p, FewChoices choices, const bf16_t* __restrict__ x, int64_t x_stride,
                                                         const bf16_t* __restrict__ w0, const bf16_t* __restrict__ w1,
                                                         bf16_t* __restrict__ y, float* __restrict__ z, float limit, float alpha,
                                                         float up_shift) {
  const int tile = blockIdx.x;
  __shared__ __attribute__((aligned(16))) bf16_t sm[2][48][EXF_K];
  __shared__ __attribute__((aligned(16))) float up_sums[64][4];
  __shared__ int sorted[SORTS ? EXF_SLOTS : 1];
  int e, r0, rend;
  if constexpr (SORTS) {
    e = few_tile(choices, UP && choices.choice.table != nullptr && blockIdx.x == 0 && blockIdx.y == 0, tile, sorted, r0, rend);
    if (e < 0) return;
  } else {
    if (tile >= p.tile_count[0]) return;
    e = p.tile_expert[tile];
    r0 = p.tile_row0[tile];
    rend = min(p.offsets[e + 1], r0 + 16);
  }
  const auto slot_of = [&](int r) { return SORTS ? sorted[r] : p.order[r]; };
  const int depth = UP ? p.width : p.ff, features = UP ? p.ff : p.width, n0 = blockIdx.y * (UP ? 16 : 32);
  const int at_row = threadIdx.x / 32, at = threadIdx.x % 32;
  const bf16_t* src[6];
#pragma unroll
  for (int i = 0; i < 4; ++i) {                                                  // (a feature past the end repeats the last)
    const int f = at_row + 8 * i, n = min(n0 + (UP ? f % 16 : f), features - 1);
    src[i] = (UP && f >= 16 ? w1 : w0) + ((int64_t)e * features + n) * depth;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {                                                  // (a row past the end repeats the last)
    const int r = min(r0 + at_row + 8 * i, rend - 1);
    src[4 + i] = x + (int64_t)(UP ? slot_of(r) / p.top : r) * x_stride;
  }
  const int lane = threadIdx.x % DLI_WAVE, wave = threadIdx.x / DLI_WAVE, c = lane % 16, g = lane / 16;
  const int chunks = (depth + EXF_K - 1) / EXF_K;
  exm_bf16x8 held[EXF_AHEAD][6];
  auto fetch = [&](int j, int chunk) {                                           // (past the end: pieces that no product takes)
    const int k0 = min(chunk, chunks - 1) * EXF_K;
    const auto from = [&](int i) {
      return reinterpret_cast<const exm_bf16x8*>(src[i] + min(k0 + 8 * (at ^ ((at_row + 8 * i) % 16)), depth - 8));
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) held[j][i] = load_streamed(from(i));   // (a choice between this load and the other would become the other)
#pragma unroll
    for (int i = 4; i < 6; ++i) held[j][i] = *from(i);
  };
#pragma unroll
  for (int j = 0; j < EXF_AHEAD; ++j) fetch(j, j);
  exm_float4 acc = {0.f, 0.f, 0.f, 0.f};
  int buffer = 0;
  for (int chunk0 = 0; chunk0 < chunks; chunk0 += EXF_AHEAD) {
#pragma unroll
    for (int j = 0; j < EXF_AHEAD; ++j) {
      const int chunk = chunk0 + j;
      if (chunk < chunks) {                                                      // (the same in all threads)
#pragma unroll
        for (int i = 0; i < 6; ++i) *reinterpret_cast<exm_bf16x8*>(&sm[buffer][at_row + 8 * i][8 * at]) = held[j][i];
        fetch(j, chunk + EXF_AHEAD);
        __syncthreads();
        if (wave < 2) {
          const int steps = min(EXF_K, depth - chunk * EXF_K) / 32;
#pragma unroll
          for (int s = 0; s < EXF_K / 32; ++s) {
            if (s < steps) {
              const int place = 8 * ((4 * s + g) ^ c);
              acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(exm_load(&sm[buffer][16 * wave + c][place]), exm_load(&sm[buffer][32 + c][place]),
                                                            acc, 0, 0, 0);
            }
          }
        }
        buffer ^= 1;
      }
    }
  }
  // a lane's results are four neighbouring features of row c
  if (UP) {
    if (wave == 1) *reinterpret_cast<exm_float4*>(up_sums[lane]) = acc;
    __syncthreads();
  }
  const int r = r0 + c, n = n0 + (UP ? 0 : 16 * wave) + 4 * g;
  if (wave >= (UP ? 1 : 2) || r >= rend || n >= features) return;               // (features come in fours)
  if (UP) {
    // (a table's weights are known: the first workgroup may still be on its way to writing them)
    const bool table_weight = SORTS && choices.choice.table != nullptr;
    const float iw = p.in_weight == nullptr ? 1.f : table_weight ? 1.f / (float)choices.choice.top : p.in_weight[slot_of(r)];
    const exm_float4 up = *reinterpret_cast<const exm_float4*>(up_sums[lane]);
    for (int i = 0; i < 4; ++i) y[(int64_t)r * p.ff + n + i] = (bf16_t)clamped_glu(iw * acc[i], iw * up[i], limit, alpha, up_shift);
  } else {
    const int64_t slot = slot_of(r);
    for (int i = 0; i < 4; ++i) z[slot * p.width + n + i] = acc[i];
  }
}

template <int MB, int NB>
__global__ __launch_bounds__(256) void expert_up_mfma_kernel(ExpertArgs p, const bf16_t* __restrict__ h, int64_t h_stride,
                                                             const bf16_t* __restrict__ w_gate,
                                                             const bf16_t* __restrict__ w_up, bf16_t* __restrict__ y,
                                                             float limit, float alpha, float up_shift) {
  const int tile = blockIdx.x;
  if (tile >= p.tile_count[0]) return;
  const int e = p.tile_expert[tile], r0 = p.tile_row0[tile], rend = min(p.offsets[e + 1], r0 + 16 * MB);
  const int lane = threadIdx.x % DLI_WAVE, wave = threadIdx.x / DLI_WAVE;
  const int c = lane % 16, kq = (lane / 16) * 8;
  const int nw = (blockIdx.y * 4 + wave) * 16 * NB;
  const bf16_t *wg[NB], *wu[NB], *xr[MB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int n = min(nw + nb * 16 + c, p.ff - 1);                              // (a feature past the end repeats the last)
    wg[nb] = w_gate + ((int64_t)e * p.ff + n) * p.width + kq;
    wu[nb] = w_up + ((int64_t)e * p.ff + n) * p.width + kq;
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int r = min(r0 + mb * 16 + c, rend - 1);                              // (a row past the end repeats the last)
    xr[mb] = h + (int64_t)(p.order[r] / p.top) * h_stride + kq;
  }
  exm_float4 accg[NB][MB], accu[NB][MB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) accg[nb][mb] = accu[nb][mb] = exm_float4{0.f, 0.f, 0.f, 0.f};
  const int blocks = (rend - r0 + 15) / 16;                                     // blocks of 16 rows that hold a row
  exm_bf16x8 a[NB], b[NB], x[MB];
  auto fetch = [&](int k) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) { a[nb] = exm_load(wg[nb] + k); b[nb] = exm_load(wu[nb] + k); }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) x[mb] = exm_load(xr[mb] + k);                // (unconditional: clamped rows are valid memory)
  };
  fetch(0);
  for (int k = 0; k < p.width; k += 32) {
    exm_bf16x8 a0[NB], b0[NB], x0[MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) { a0[nb] = a[nb]; b0[nb] = b[nb]; }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) x0[mb] = x[mb];
    fetch(min(k + 32, p.width - 32));                                           // the last turn asks for its own step again
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      if (mb < blocks) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          accg[nb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[nb], x0[mb], accg[nb][mb], 0, 0, 0);
          accu[nb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0[nb], x0[mb], accu[nb][mb], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int r = r0 + mb * 16 + c;
    if (r >= rend) continue;
    const float iw = p.in_weight != nullptr ? p.in_weight[p.order[r]] : 1.f;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int n0 = nw + nb * 16 + (lane / 16) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n0 + i < p.ff)
          y[(int64_t)r * p.ff + n0 + i] = (bf16_t)clamped_glu(iw * accg[nb][mb][i], iw * accu[nb][mb][i], limit, alpha, up_shift);
    }
  }
}

template <int MB, int NB>
__global__ __launch_bounds__(256) void expert_down_mfma_kernel(ExpertArgs p, const bf16_t* __restrict__ y,
                                                               const bf16_t* __restrict__ w_down, float* __restrict__ z) {
  const int tile = blockIdx.x;
  if (tile >= p.tile_count[0]) return;
  const int e = p.tile_expert[tile], r0 = p.tile_row0[tile], rend = min(p.offsets[e + 1], r0 + 16 * MB);
  const int lane = threadIdx.x % DLI_WAVE, wave = threadIdx.x / DLI_WAVE;
  const int c = lane % 16, kq = (lane / 16) * 8;
  const int nw = (blockIdx.y * 4 + wave) * 16 * NB;
  const bf16_t *wd[NB], *yr[MB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) wd[nb] = w_down + ((int64_t)e * p.width + min(nw + nb * 16 + c, p.width - 1)) * p.ff + kq;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) yr[mb] = y + (int64_t)min(r0 + mb * 16 + c, rend - 1) * p.ff + kq;
  exm_float4 acc[NB][MB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = exm_float4{0.f, 0.f, 0.f, 0.f};
  const int blocks = (rend - r0 + 15) / 16;
  exm_bf16x8 a[NB], x[MB];
  auto fetch = [&](int k) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) a[nb] = exm_load(wd[nb] + k);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) x[mb] = exm_load(yr[mb] + k);
  };
  fetch(0);
  for (int k = 0; k < p.ff; k += 32) {
    exm_bf16x8 a0[NB], x0[MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) a0[nb] = a[nb];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) x0[mb] = x[mb];
    fetch(min(k + 32, p.ff - 32));
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      if (mb < blocks)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[nb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[nb], x0[mb], acc[nb][mb], 0, 0, 0);
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int r = r0 + mb * 16 + c;
    if (r >= rend) continue;
    const int64_t slot = p.order[r];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int n0 = nw + nb * 16 + (lane / 16) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n0 + i < p.width) z[slot * p.width + n0 + i] = acc[nb][mb][i];
    }
  }
}

// The same two products for many rows an expert (bfloat16, sizes that are multiples of 64 and 128 as the host checks): tiles of
// EXL_BM sorted rows, a workgroup of four waves takes 128 rows of weights (the up product: 64 of each half), both
// operands through LDS 64 k at a time, the next 64 in flight in registers meanwhile. A wave takes half of the
// tile's rows and half of the weights' rows, sixteen 16 x 16 blocks. Rows in LDS are padded by 16 bytes. Every output sums its k in
// ascending steps of 32, as in the kernels above. The workgroups of one XCD take neighbouring tiles with all their
// features, so that an expert's weights are read into one L2 (or two).
#define EXL_BM 128
#define EXL_BK 64
#define EXL_LD (EXL_BK + 8)
template <bool UP>
__global__ __launch_bounds__(256, 2) void expert_tiled_kernel(ExpertArgs p, const bf16_t* __restrict__ x, int64_t x_stride,
                                                              const bf16_t* __restrict__ w0, const bf16_t* __restrict__ w1,
                                                              bf16_t* __restrict__ y, float* __restrict__ z, int blocks_n,
                                                              float limit, float alpha, float up_shift) {
  __shared__ __align__(16) bf16_t xs[2][EXL_BM * EXL_LD], ws[2][128 * EXL_LD];
  const int count = p.tile_count[0], per = (count + 7) / 8, local = blockIdx.x / 8;
  const int tile = (blockIdx.x % 8) * per + local / blocks_n, block = local % blocks_n;
  if (local / blocks_n >= per || tile >= count) return;
  const int e = p.tile_expert[tile], r0 = p.tile_row0[tile], rend = min(p.offsets[e + 1], r0 + EXL_BM);
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), c = lane % 16, g = lane / 16;
  const int wm = wave & 1, wn = wave >> 1;
  const int K = UP ? p.width : p.ff;
  // this thread's 16-byte pieces: piece tid % 8 of the rows tid / 8 + 32 m
  const bf16_t *xr[4], *wr[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int row = tid / 8 + 32 * m, r = min(r0 + row, rend - 1);              // (a row past the end repeats the last)
    xr[m] = x + (int64_t)(UP ? p.order[r] / p.top : r) * x_stride + 8 * (tid % 8);
    if (UP) wr[m] = (row < 64 ? w0 : w1) + ((int64_t)e * p.ff + 64 * block + row % 64) * K + 8 * (tid % 8);
    else wr[m] = w0 + ((int64_t)e * p.width + 128 * block + row) * K + 8 * (tid % 8);
  }
  exm_bf16x8 rx[4], rw[4];
  auto fetch = [&](int k) {
#pragma unroll
    for (int m = 0; m < 4; ++m) { rx[m] = exm_load(xr[m] + k); rw[m] = exm_load(wr[m] + k); }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int at = (tid / 8 + 32 * m) * EXL_LD + 8 * (tid % 8);
      *reinterpret_cast<exm_bf16x8*>(&xs[buf][at]) = rx[m];
      *reinterpret_cast<exm_bf16x8*>(&ws[buf][at]) = rw[m];
    }
  };
  exm_float4 acc[4][4];                                                          // [weights' block][rows' block]
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[n][m] = exm_float4{0.f, 0.f, 0.f, 0.f};
  // the weights' blocks: gate 32 wn and 32 wn + 16, then the same of up; or 64 wn on
  int wrow[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) wrow[n] = UP ? 64 * (n / 2) + 32 * wn + 16 * (n % 2) : 64 * wn + 16 * n;
  // (An expert's last tile is part empty: a wave leaves out the products of rows that are not there, and their reads of LDS. 2,304 tokens,
  // 4 of 32 experts each, 288 rows an expert: up 153 -> 149 us, down 86 -> 83.)
  const int row_blocks = (rend - r0 - 64 * wm + 15) / 16;
  fetch(0);
  put(0);
  __syncthreads();
  int buf = 0;
  for (int k = 0; k < K; k += EXL_BK, buf ^= 1) {
    const bool more = k + EXL_BK < K;
    if (more) fetch(k + EXL_BK);
    const auto multiply = [&](auto blocks_of_16) __attribute__((always_inline)) {
      constexpr int M = decltype(blocks_of_16)::value;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        exm_bf16x8 a[4], b[M];
#pragma unroll
        for (int n = 0; n < 4; ++n) a[n] = exm_load(&ws[buf][(wrow[n] + c) * EXL_LD + 32 * s + 8 * g]);
#pragma unroll
        for (int m = 0; m < M; ++m) b[m] = exm_load(&xs[buf][(64 * wm + 16 * m + c) * EXL_LD + 32 * s + 8 * g]);
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int m = 0; m < M; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[n], b[m], acc[n][m], 0, 0, 0);
      }
    };
    if (row_blocks > 2) multiply(std::integral_constant<int, 4>());
    else if (row_blocks > 0) multiply(std::integral_constant<int, 2>());
    if (more) put(buf ^ 1);
    __syncthreads();
  }
  typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int r = r0 + 64 * wm + 16 * m + c;
    if (r >= rend) continue;
    if (UP) {
      const float iw = p.in_weight != nullptr ? p.in_weight[p.order[r]] : 1.f;
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        bf4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = (bf16_t)clamped_glu(iw * acc[n][m][i], iw * acc[n + 2][m][i], limit, alpha, up_shift);
        *reinterpret_cast<bf4*>(y + (int64_t)r * p.ff + 64 * block + 32 * wn + 16 * n + 4 * g) = o;
      }
    } else {
      const int64_t slot = p.order[r];
#pragma unroll
      for (int n = 0; n < 4; ++n)
        *reinterpret_cast<exm_float4*>(z + slot * p.width + 128 * block + wrow[n] + 4 * g) = acc[n][m];
    }
  }
}

// (weights nullptr: ones)
// out[token] = sum_j weights[token][j] * (ids[token][j] < experts ? z[token * top + j] : h[token])
//            + sigmoid(shared_gate[token]) * shared[token]       (the shared expert, if there is one)
template <typename T>
__global__ void expert_combine_kernel(const int* __restrict__ ids, const float* __restrict__ weights,
                                      const float* __restrict__ z, const T* __restrict__ h, int64_t h_stride,
                                      const float* __restrict__ shared_gate, int64_t gate_stride,
                                      const float* __restrict__ shared, int64_t shared_stride, float* __restrict__ out,
                                      int top, int experts, int width) {
  const int64_t row = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= width) return;
  float sum = 0.f;
  for (int j = 0; j < top; ++j) {
    const int e = ids[row * top + j];
    const float v = e < experts ? z[(row * top + j) * width + c] : to_f32(h[row * h_stride + c]);
    sum = fmaf(weights != nullptr ? weights[row * top + j] : 1.f, v, sum);
  }
  if (shared != nullptr) {
    const float g = shared_gate != nullptr ? 1.f / (1.f + expf(-shared_gate[row * gate_stride])) : 1.f;
    sum = fmaf(g, shared[row * shared_stride + c], sum);
  }
  out[row * width + c] = sum;
}

// The same with four columns a thread: widths, strides and addresses of whole 16-byte pieces.
template <typename T>
__global__ __launch_bounds__(256) void expert_combine4_kernel(const int* __restrict__ ids, const float* __restrict__ weights,
                                                              const float* __restrict__ z, const T* __restrict__ h, int64_t h_stride,
                                                              const float* __restrict__ shared_gate, int64_t gate_stride,
                                                              const float* __restrict__ shared, int64_t shared_stride,
                                                              float* __restrict__ out, int top, int experts, int width) {
  const int64_t row = blockIdx.x;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= width) return;
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j < top; ++j) {
    const float wt = weights != nullptr ? weights[row * top + j] : 1.f;
    float v[4];
    if (ids[row * top + j] < experts) {
      const float4 f = *reinterpret_cast<const float4*>(z + (row * top + j) * width + c);
      v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = to_f32(h[row * h_stride + c + i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] = fmaf(wt, v[i], sum[i]);
  }
  if (shared != nullptr) {
    const float g = shared_gate != nullptr ? 1.f / (1.f + expf(-shared_gate[row * gate_stride])) : 1.f;
    const float4 f = *reinterpret_cast<const float4*>(shared + row * shared_stride + c);
    sum[0] = fmaf(g, f.x, sum[0]); sum[1] = fmaf(g, f.y, sum[1]); sum[2] = fmaf(g, f.z, sum[2]); sum[3] = fmaf(g, f.w, sum[3]);
  }
  *reinterpret_cast<float4*>(out + row * width + c) = float4{sum[0], sum[1], sum[2], sum[3]};
}

// The combination, the residual sum of a block whose two sublayers stand side by side and the norms that the stream meets next, a
// workgroup a row: x += a + out (out as above), out1 and out2 = w1 and w2 times x / sqrt(mean(x^2) + eps) (w1 nullptr: no norms).
// What bounds it: with few rows one trip to memory after another, ids, then results, then the sum over the row, which are asked
// for four choices at a time, the norms' weights with them; three kernels (the combination, the sum, the norms) took
// 13.7 us of a decode step of two rows of 2,048 values, this one 4.4; with 2,304 rows 45 and 25.8.
struct CombineStream {
  const int* ids; const float* weights; const float* z;
  const float* shared_gate; int64_t gate_stride; const float* shared; int64_t shared_stride;
  float* x; const float* a;
  const float *w1, *w2; float eps;
  int top, experts, width;
};
template <typename T>
__global__ __launch_bounds__(512) void expert_combine_stream_kernel(CombineStream p, const T* __restrict__ h, int64_t h_stride,
                                                                    T* __restrict__ out1, T* __restrict__ out2) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef T t4 __attribute__((ext_vector_type(4)));
  constexpr int HELD = 2;   // pieces of four values a thread keeps; wider rows are read once more
  __shared__ float scratch[16];
  const int64_t row = blockIdx.x;
  const int step = 4 * blockDim.x, c0 = 4 * threadIdx.x;
  const int* ids = p.ids + row * p.top;
  float* x = p.x + row * p.width;
  const auto at4 = [](const float* at) { return *reinterpret_cast<const f4*>(at); };
  const auto summed = [&](int c) {
    const f4 old = at4(x + c), other = at4(p.a + row * p.width + c);
    f4 add = {0.f, 0.f, 0.f, 0.f}, sum = {0.f, 0.f, 0.f, 0.f};
    if (p.shared != nullptr) add = at4(p.shared + row * p.shared_stride + c);
    for (int j0 = 0; j0 < p.top; j0 += 4) {
      f4 v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = at4(p.z + (row * p.top + min(j0 + e, p.top - 1)) * p.width + c);   // (identity: not looked at)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (j0 + e >= p.top) break;
        if (ids[j0 + e] >= p.experts) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[e][i] = to_f32(h[row * h_stride + c + i]);
        }
        const float wt = p.weights != nullptr ? p.weights[row * p.top + j0 + e] : 1.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] = fmaf(wt, v[e][i], sum[i]);
      }
    }
    if (p.shared != nullptr) {
      const float g = p.shared_gate != nullptr ? 1.f / (1.f + expf(-p.shared_gate[row * p.gate_stride])) : 1.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[i] = fmaf(g, add[i], sum[i]);
    }
    const f4 now = old + (other + sum);
    *reinterpret_cast<f4*>(x + c) = now;
    return now;
  };
  f4 held[HELD], w1[HELD], w2[HELD];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < HELD; ++k) {
    const int c = c0 + k * step;
    if (c >= p.width) continue;
    if (p.w1 != nullptr) {
      w1[k] = at4(p.w1 + c);
      w2[k] = at4(p.w2 + c);
    }
    held[k] = summed(c);
#pragma unroll
    for (int i = 0; i < 4; ++i) ss = fmaf(held[k][i], held[k][i], ss);
  }
  for (int c = c0 + HELD * step; c < p.width; c += step) {
    const f4 now = summed(c);
#pragma unroll
    for (int i = 0; i < 4; ++i) ss = fmaf(now[i], now[i], ss);
  }
  if (p.w1 == nullptr) return;
  const float r = 1.f / sqrtf(block_sum(ss, scratch) / (float)p.width + p.eps);
  const auto store = [&](int c, const f4& v, const f4& a, const f4& b) {
    t4 one, two;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      one[i] = from_f32<T>(a[i] * (v[i] * r));
      two[i] = from_f32<T>(b[i] * (v[i] * r));
    }
    *reinterpret_cast<t4*>(out1 + row * p.width + c) = one;
    *reinterpret_cast<t4*>(out2 + row * p.width + c) = two;
  };
#pragma unroll
  for (int k = 0; k < HELD; ++k)
    if (c0 + k * step < p.width) store(c0 + k * step, held[k], w1[k], w2[k]);
  for (int c = c0 + HELD * step; c < p.width; c += step) store(c, at4(x + c), at4(p.w1 + c), at4(p.w2 + c));   // (this thread's own values)
}

// A router that is a table: the experts of a token are the row of `table` [vocabulary][top] at its token id,
// each with the weight 1 / top. A thread a (token, choice).
__global__ void table_choose_kernel(const int* __restrict__ table, const int* __restrict__ token_ids, int n, int top,
                                    int vocab, int* __restrict__ ids, float* __restrict__ weights) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n * top) return;
  ids[i] = table_choice(table, token_ids, vocab, top, i);
  weights[i] = 1.f / (float)top;
}

extern "C" {

int dli_poly_norm(const float* z, int64_t z_stride, const float* coef, void* out, int64_t out_stride, int rows, int ff,
                  float eps, int out_is_bf16, hipStream_t stream) {
  if (rows <= 0) return DLI_OK;
  if (ff <= 0 || z_stride < ff || out_stride < ff) return DLI_ERR_ARGUMENT;
  const int threads = ff >= 4096 ? 512 : 256;
  if (ff <= threads)
    poly_norm_kernel_f32in<1><<<rows, threads, 0, stream>>>(z, z_stride, coef, out, out_stride, ff, eps, out_is_bf16);
  else if (ff <= 4 * threads)
    poly_norm_kernel_f32in<4><<<rows, threads, 0, stream>>>(z, z_stride, coef, out, out_stride, ff, eps, out_is_bf16);
  else
    poly_norm_kernel_f32in<POLY_HELD><<<rows, threads, 0, stream>>>(z, z_stride, coef, out, out_stride, ff, eps, out_is_bf16);
  return dli_launch_status();
}

int dli_clamped_glu(const void* gate_up, int64_t stride, void* out, int rows, int ff, int form, float limit, float alpha, float up_shift,
                    int is_bf16, hipStream_t stream) {
  if (rows <= 0) return DLI_OK;
  if (ff <= 0 || stride < 2 * (int64_t)ff || (form != GLU_CLAMPED && form != GLU_GELU)) return DLI_ERR_ARGUMENT;
  const dim3 grid(rows, (ff + 255) / 256), grid8(rows, (ff / 8 + 255) / 256);
  const GluForm f{form, limit, alpha, up_shift};
  if (is_bf16 && ff % 8 == 0 && stride % 8 == 0 && ((uintptr_t)gate_up | (uintptr_t)out) % 16 == 0) {
    if (form == GLU_GELU) clamped_glu_bf16x8_kernel<true><<<grid8, 256, 0, stream>>>((const bf16_t*)gate_up, stride, (bf16_t*)out, ff, f);
    else clamped_glu_bf16x8_kernel<false><<<grid8, 256, 0, stream>>>((const bf16_t*)gate_up, stride, (bf16_t*)out, ff, f);
  } else if (is_bf16) clamped_glu_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)gate_up, stride, (bf16_t*)out, ff, f);
  else clamped_glu_kernel<float><<<grid, 256, 0, stream>>>((const float*)gate_up, stride, (float*)out, ff, f);
  return dli_launch_status();
}

int dli_router_choose(const float* logits, int64_t stride, const float* bias, const float* correction, int rows, int total, int count, int keep,
                      int top, float scale, int sigmoid, int normalize, int* ids, float* weights, hipStream_t stream) {
  if (rows <= 0) return DLI_OK;
  if (total <= 0 || total > 4096 || stride < total || top < 1 || top > 64 || top > total || count < 1 || total % count ||
      keep < 1 || keep > count || (int64_t)keep * (total / count) < top)
    return DLI_ERR_ARGUMENT;
  router_choose_kernel<<<rows, 64, (2 * total + count) * sizeof(float), stream>>>(logits, stride, bias, correction, total, count, keep,
                                                                                  top, scale, sigmoid, normalize, ids, weights);
  return dli_launch_status();
}

// Whether the matrix-core kernels take these sizes, and the rows of a tile of the kernels that will run.
static bool expert_mfma(int width, int ff, int is_bf16) { return is_bf16 && width % 32 == 0 && ff % 32 == 0; }
// Many rows an expert, and sizes that tile: the kernels that pass both operands through LDS.
static bool expert_tiled(int64_t slots, int experts, int width, int ff, int is_bf16) {
  return is_bf16 && width % 128 == 0 && ff % 64 == 0 && slots >= 48 * (int64_t)experts;
}
// Few rows an expert: the kernels that wait for the weights alone.
static bool expert_few(int64_t slots, int experts, int width, int ff) {
  return slots <= 16 * (int64_t)experts && ff <= 16 * 65535 && width <= 16 * 65535;
}
int dli_expert_tile_rows(int64_t slots, int experts, int width, int ff, int is_bf16) {
  if (expert_tiled(slots, experts, width, ff, is_bf16)) return EXL_BM;
  if (!expert_mfma(width, ff, is_bf16)) return EX_BM;
  return expert_few(slots, experts, width, ff) ? EXM_FEW : EXM_BM;
}

int dli_table_choose(const int* table, const int* token_ids, int n, int top, int vocab, int* ids, float* weights,
                     hipStream_t stream) {
  if (n <= 0) return DLI_OK;
  if (top <= 0 || vocab <= 0 || (int64_t)n * top > 0x7fffffff) return DLI_ERR_ARGUMENT;
  table_choose_kernel<<<(n * top + 255) / 256, 256, 0, stream>>>(table, token_ids, n, top, vocab, ids, weights);
  return dli_launch_status();
}

// The experts' part of a mixture for `rows` tokens: sort, up product with activation, down product.
// ids [rows][top]; scratch: offsets [experts + 1], order [rows * top], tile_expert and tile_row0 [max_tiles],
// tile_count [1] (int32), y [rows * top][ff] (T), z [rows * top][width] (float32). in_weight [rows][top] (may be nullptr):
// what each slot's expert input is multiplied by.
// table [vocab][top] (may be nullptr): ids and weights [rows][top] are written here, the row of each token's id with weights of 1 / top.
int dli_expert_products(int* ids, const int* table, const int* token_ids, int vocab, float* weights, const void* h, int64_t h_stride,
                        const void* w_gate, const void* w_up,
                        const void* w_down, int* offsets, int* order, int* tile_expert, int* tile_row0, int* tile_count,
                        int max_tiles, void* y, float* z, const float* in_weight, int rows, int top, int experts, int width,
                        int ff, float limit, float alpha, float up_shift, int is_bf16, hipStream_t stream) {
  if (rows <= 0) return DLI_OK;
  const int64_t slots = (int64_t)rows * top;
  if (top < 1 || experts < 1 || experts > 4096 || width <= 0 || ff <= 0 || h_stride < width || slots > (1 << 30) ||
      max_tiles < 1 || max_tiles > 65535 * 16 || (table != nullptr && (token_ids == nullptr || vocab < 1 || weights == nullptr)))
    return DLI_ERR_ARGUMENT;
  const bool mfma = expert_mfma(width, ff, is_bf16);
  if (mfma && ((h_stride % 8) || ((uintptr_t)h % 16) || ((uintptr_t)w_gate % 16) || ((uintptr_t)w_up % 16) ||
               ((uintptr_t)w_down % 16) || ((uintptr_t)y % 16)))
    return DLI_ERR_ARGUMENT;
  TableChoice choice = {table, token_ids, vocab, top, weights};
  if (table != nullptr && slots > 1024) {   // (several a thread: one workgroup's trips to memory, one after the other)
    if (dli_table_choose(table, token_ids, rows, top, vocab, ids, weights, stream) != DLI_OK) return DLI_ERR_LAUNCH;
    choice.table = nullptr;
  }
  ExpertArgs p;
  p.tile_expert = tile_expert; p.tile_row0 = tile_row0; p.tile_count = tile_count; p.offsets = offsets; p.order = order;
  p.top = top; p.width = width; p.ff = ff; p.in_weight = in_weight;
  // (with a table the products write its weights themselves, so of weights on the inputs they take none or those)
  const bool own_weights = choice.table == nullptr || in_weight == nullptr || in_weight == weights;
  if (mfma && own_weights && slots <= EXF_SLOTS && !expert_tiled(slots, experts, width, ff, is_bf16) && expert_few(slots, experts, width, ff)) {
    const FewChoices choices = {ids, choice, (int)slots, experts}, chosen = {ids, {nullptr, nullptr, 0, top, nullptr}, (int)slots, experts};
    expert_few_kernel<true, true><<<dim3(max_tiles, (ff + 15) / 16), 256, 0, stream>>>(p, choices, (const bf16_t*)h, h_stride, (const bf16_t*)w_gate,
                                                                                       (const bf16_t*)w_up, (bf16_t*)y, nullptr, limit, alpha, up_shift);
    expert_few_kernel<false, true><<<dim3(max_tiles, (width + 31) / 32), 256, 0, stream>>>(p, chosen, (const bf16_t*)y, ff, (const bf16_t*)w_down,
                                                                                           nullptr, nullptr, z, 0.f, 0.f, 0.f);
    return dli_launch_status();
  }
  expert_sort_kernel<<<1, 1024, 2 * experts * sizeof(int), stream>>>(ids, choice, (int)slots, experts, offsets, order, tile_expert,
                                                                     tile_row0, tile_count, max_tiles,
                                                                     dli_expert_tile_rows(slots, experts, width, ff, is_bf16));
  if (dli_launch_status() != DLI_OK) return DLI_ERR_LAUNCH;
  if (expert_tiled(slots, experts, width, ff, is_bf16)) {
    const unsigned tiles8 = 8 * ((max_tiles + 7) / 8);
    if ((int64_t)tiles8 * (ff / 64 + width / 128) > 0x7fffffff || ((uintptr_t)z % 16)) return DLI_ERR_ARGUMENT;
    expert_tiled_kernel<true><<<tiles8 * (ff / 64), 256, 0, stream>>>(p, (const bf16_t*)h, h_stride, (const bf16_t*)w_gate,
                                                                      (const bf16_t*)w_up, (bf16_t*)y, nullptr, ff / 64, limit, alpha, up_shift);
    expert_tiled_kernel<false><<<tiles8 * (width / 128), 256, 0, stream>>>(p, (const bf16_t*)y, ff, (const bf16_t*)w_down, nullptr,
                                                                           nullptr, z, width / 128, 0.f, 0.f, 0.f);
    return dli_launch_status();
  }
  if (mfma && expert_few(slots, experts, width, ff)) {
    expert_few_kernel<true, false><<<dim3(max_tiles, (ff + 15) / 16), 256, 0, stream>>>(p, FewChoices(), (const bf16_t*)h, h_stride, (const bf16_t*)w_gate,
                                                                                 (const bf16_t*)w_up, (bf16_t*)y, nullptr, limit, alpha, up_shift);
    expert_few_kernel<false, false><<<dim3(max_tiles, (width + 31) / 32), 256, 0, stream>>>(p, FewChoices(), (const bf16_t*)y, ff, (const bf16_t*)w_down, nullptr,
                                                                                     nullptr, z, 0.f, 0.f, 0.f);
    return dli_launch_status();
  }
  const int bn = mfma ? 128 : EX_BN;
  const dim3 up_grid(max_tiles, (ff + bn - 1) / bn), down_grid(max_tiles, (width + bn - 1) / bn);
  if (mfma) {
    expert_up_mfma_kernel<4, 2><<<up_grid, 256, 0, stream>>>(p, (const bf16_t*)h, h_stride, (const bf16_t*)w_gate, (const bf16_t*)w_up,
                                                             (bf16_t*)y, limit, alpha, up_shift);
    expert_down_mfma_kernel<4, 2><<<down_grid, 256, 0, stream>>>(p, (const bf16_t*)y, (const bf16_t*)w_down, z);
  } else if (is_bf16) {
    expert_up_kernel<bf16_t><<<up_grid, 256, 0, stream>>>(p, (const bf16_t*)h, h_stride, (const bf16_t*)w_gate,
                                                          (const bf16_t*)w_up, (bf16_t*)y, limit, alpha, up_shift);
    expert_down_kernel<bf16_t><<<down_grid, 256, 0, stream>>>(p, (const bf16_t*)y, (const bf16_t*)w_down, z);
  } else {
    expert_up_kernel<float><<<up_grid, 256, 0, stream>>>(p, (const float*)h, h_stride, (const float*)w_gate,
                                                         (const float*)w_up, (float*)y, limit, alpha, up_shift);
    expert_down_kernel<float><<<down_grid, 256, 0, stream>>>(p, (const float*)y, (const float*)w_down, z);
  }
  return dli_launch_status();
}

int dli_expert_combine_stream(const int* ids, const float* weights, const float* z, const void* h, int64_t h_stride,
                              const float* shared_gate, int64_t gate_stride, const float* shared, int64_t shared_stride, float* x,
                              const float* a, const float* w1, const float* w2, float eps, void* out1, void* out2, int rows, int top,
                              int experts, int width, int is_bf16, hipStream_t stream) {
  if (rows <= 0) return DLI_OK;
  if (top < 1 || width <= 0 || width % 4 != 0 || h_stride < width || z == nullptr ||
      (shared != nullptr && (shared_stride < width || shared_stride % 4 != 0)) ||
      (w1 != nullptr && (w2 == nullptr || out1 == nullptr || out2 == nullptr)) ||
      (((uintptr_t)z | (uintptr_t)shared | (uintptr_t)x | (uintptr_t)a | (uintptr_t)w1 | (uintptr_t)w2 | (uintptr_t)out1 | (uintptr_t)out2) % 16) != 0)
    return DLI_ERR_ARGUMENT;
  const CombineStream p = {ids, weights, z, shared_gate, gate_stride, shared, shared_stride, x, a, w1, w2, eps, top, experts, width};
  const int threads = width > 1024 ? 512 : 256;
  if (is_bf16) expert_combine_stream_kernel<bf16_t><<<rows, threads, 0, stream>>>(p, (const bf16_t*)h, h_stride, (bf16_t*)out1, (bf16_t*)out2);
  else expert_combine_stream_kernel<float><<<rows, threads, 0, stream>>>(p, (const float*)h, h_stride, (float*)out1, (float*)out2);
  return dli_launch_status();
}

int dli_expert_combine(const int* ids, const float* weights, const float* z, const void* h, int64_t h_stride,
                       const float* shared_gate, int64_t gate_stride, const float* shared, int64_t shared_stride, float* out,
                       int rows, int top, int experts, int width, int is_bf16, hipStream_t stream) {
  if (rows <= 0) return DLI_OK;
  if (top < 1 || width <= 0 || h_stride < width || (shared != nullptr && shared_stride < width)) return DLI_ERR_ARGUMENT;
  auto whole = [](const void* at) { return (uintptr_t)at % 16 == 0; };
  // (with few rows the extra workgroups of one column a thread hide more of the wait)
  const bool fours = rows >= 256 && width % 4 == 0 && whole(z) && whole(out) && (shared == nullptr || (whole(shared) && shared_stride % 4 == 0));
  const int cols = fours ? 1024 : 256;
  const dim3 grid(rows, (width + cols - 1) / cols);
#define COMBINE(KERNEL, T) KERNEL<T><<<grid, 256, 0, stream>>>(ids, weights, z, (const T*)h, h_stride, shared_gate, gate_stride, \
                                                               shared, shared_stride, out, top, experts, width)
  if (is_bf16) { if (fours) COMBINE(expert_combine4_kernel, bf16_t); else COMBINE(expert_combine_kernel, bf16_t); }
  else { if (fours) COMBINE(expert_combine4_kernel, float); else COMBINE(expert_combine_kernel, float); }
#undef COMBINE
  return dli_launch_status();
}


}  // extern "C"
