// All layers of a decode step of one row in one launch: pre-norm blocks of RMSNorm, rotary grouped-query attention over pages and a
// feed-forward with SwiGLU, bfloat16, of models so small that a layer's kernels are mostly their launches.
//
// A layer is five kinds of work (q/k/v with norm, rotation and cache write; attention; o with the merge of the attention's runs and the
// residual sum; gate and up with norm and SwiGLU; down with the residual sum), each cut into workgroups that do one piece of it: ask
// for their rows of weights (or their keys and values), wait for what the kind before leaves, multiply, and leave their own. Nothing but
// these values orders them, so a piece's weights are on their way while the pieces before it still run, two layers ahead and more.
//
// Handing over. A value goes out at the device's scope as one word with the launch's number beside it (16 bits of bfloat16 and 16 of
// the number; 32-bit sums as two words stored together), so that whoever needs it sees by the word itself that it is there: one
// store and one load, no counters, no fences. Every layer has words of its own, and every launch writes all that its readers wait for.
//
// Why every wait ends. A workgroup takes its piece by a ticket, in the order of layers and kinds, and a piece waits only for pieces of
// smaller tickets, whose workgroups have begun: whatever else the device runs, the smallest unfinished one has nothing to wait
// for. (A wait gives up after about a second all the same, and its value is then not a number.)
//
// What bounds it: a kind's chain of store, load (0.9 to 1.5 us from one workgroup's store to another's registers), sum over lanes,
// barrier, reads of LDS, products and their sum, 2.6 us a kind where a kernel of its own takes 3.8. 150 kinds without any work between
// them took 1.35 us each with 16 workgroups and 1.8 with 96, so pieces are few and large: eight rows a wave and eight waves, not four. One
// request, a step and seven more, ms, kernel by kernel -> now: 135M sizes, 48 keys 4.63 3.14, 512 4.77 3.43, 8,000 6.04 4.08; 360M sizes
// 5.98 3.92, 6.26 4.23, 7.18 4.85. (Wider models are refused: their weights do not wait in registers two layers ahead, and 4 KB of
// values for each of some hundred workgroups is traffic that the waiting itself makes.)
#include <type_traits>

#include "common.h"
#include "merge_splits.h"

namespace {

typedef __bf16 flow_bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned flow_u4 __attribute__((ext_vector_type(4)));
typedef float flow_f4 __attribute__((ext_vector_type(4)));

constexpr int FLOW_THREADS = 512, FLOW_WAVES = FLOW_THREADS / 64, FLOW_SPLITS = 16, FLOW_WAIT = 1 << 20;
// Blocks of 128 k that a lane holds of its rows of weights: of the stream's size (two quads a wave where rows are paired), of the inner size.
constexpr int FLOW_BLOCKS = 8, FLOW_INNER_BLOCKS = 24;

struct FlowLayer {
  const float *norm1, *norm2;
  const bf16_t *w_qkv, *w_o, *w_gate_up, *w_down;
  bf16_t *k_pages, *v_pages;
};

struct FlowArgs {
  const FlowLayer* layers; int num_layers;
  unsigned long long* tickets;   // this launch's number, and in the lower half the next ticket
  void* words; unsigned layer_bytes, at_part, at_x1, at_act, at_x2;   // a layer's words: q/k/v first, then what begins at these bytes
  bf16_t* x; float* ssq_out;
  const float* angles; const int *slots, *kv_len, *block_table; int table_width;
  int hidden, q_heads, kv_heads, inner, page_size; PageOf page_of;
  float eps, scale_log2e;
  int rows[4], wgs[4];        // q/k/v, o, gate/up, down: rows of weights a workgroup, workgroups a layer
  int splits, layer_wgs;   // splits: the most that a request's keys are cut into
};

// Waits until four words carry the tag in their lower half.
template <int N>
__device__ __forceinline__ void flow_wait(__amdgpu_buffer_rsrc_t r, const unsigned (&at)[N], unsigned tag, flow_u4 (&v)[N]) {
  for (int tries = 0;; ++tries) {
    asm volatile("" ::: "memory");   // (asked for anew every time)
    unsigned wrong = 0;
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = __builtin_amdgcn_raw_buffer_load_b128(r, (int)at[k], 0, DEVICE_SCOPE);
#pragma unroll
    for (int k = 0; k < N; ++k) wrong |= (v[k][0] ^ tag) | (v[k][1] ^ tag) | (v[k][2] ^ tag) | (v[k][3] ^ tag);
    if ((wrong & 0xffffu) == 0) return;
    if (tries == FLOW_WAIT) {
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = flow_u4{0x7fc00000u, 0x7fc00000u, 0x7fc00000u, 0x7fc00000u};
      return;
    }
  }
}
// The same for pairs of (32-bit value, tag).
template <int N>
__device__ __forceinline__ void flow_wait_pairs(__amdgpu_buffer_rsrc_t r, const unsigned (&at)[N], unsigned tag, flow_u4 (&v)[N]) {
  for (int tries = 0;; ++tries) {
    asm volatile("" ::: "memory");
    unsigned wrong = 0;
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = __builtin_amdgcn_raw_buffer_load_b128(r, (int)at[k], 0, DEVICE_SCOPE);
#pragma unroll
    for (int k = 0; k < N; ++k) wrong |= (v[k][1] ^ tag) | (v[k][3] ^ tag);
    if (wrong == 0) return;
    if (tries == FLOW_WAIT) {
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = flow_u4{0x7fc00000u, tag, 0x7fc00000u, tag};
      return;
    }
  }
}
__device__ __forceinline__ unsigned flow_wait_word(__amdgpu_buffer_rsrc_t r, unsigned at, unsigned tag) {
  for (int tries = 0;; ++tries) {
    asm volatile("" ::: "memory");
    const unsigned v = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, (int)at, 0, DEVICE_SCOPE);
    if (((v ^ tag) & 0xffffu) == 0) return v;
    if (tries == FLOW_WAIT) return 0x7fc00000u;
  }
}
__device__ __forceinline__ float flow_value(unsigned word) { return __uint_as_float(word & 0xffff0000u); }
__device__ __forceinline__ void flow_leave(__amdgpu_buffer_rsrc_t r, unsigned at, bf16_t v, unsigned tag) {
  const unsigned word = ((unsigned)__builtin_bit_cast(unsigned short, v) << 16) | tag;
  __builtin_amdgcn_raw_buffer_store_b32(word, r, (int)at, 0, DEVICE_SCOPE);
}

typedef short flow_s4 __attribute__((ext_vector_type(4)));
union FlowChunk {
  flow_u4 raw;
  flow_s4 h[2];
};

// Q quads of neighbouring rows (`rows[q]` the first of each), BLOCKS blocks of 128 k at most, in registers, and their products with a row
// in LDS on sixteen independent 4 x 4 x 4 blocks a matrix instruction, as the products of few rows do it (skinny4_gemm.hip): lane l takes
// row l % 4 of a quad and chunk l / 4 of each block, a load's sixteen neighbours whole lines. A lane is left with the sum of the quad's
// row flow_row(). (By way of LDS a kind took 0.7 us longer: 74 KB of weights a compute unit pass it in 600 cycles at best.)
template <int Q, int BLOCKS>
struct FlowWeights {
  FlowChunk w[BLOCKS][Q];
  __device__ __forceinline__ void ask(const bf16_t* weights, int k, const int (&rows)[Q]) {   // (past k: the last chunk again)
    const int lane = threadIdx.x % 64, r = lane % 4, blk = lane / 4, chunks = k / 8;
    const flow_u4* at[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) at[q] = reinterpret_cast<const flow_u4*>(weights + (int64_t)(rows[q] + r) * k);
#pragma unroll
    for (int u = 0; u < BLOCKS; ++u)
#pragma unroll
      for (int q = 0; q < Q; ++q) w[u][q].raw = load_streamed(at[q] + min(16 * u + blk, chunks - 1));
  }
  __device__ __forceinline__ void multiply(int k, const bf16_t* xs, float (&y)[Q]) {
    const int blk = threadIdx.x % 64 / 4, chunks = k / 8;
    flow_f4 acc[Q][2];
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[q][0] = acc[q][1] = flow_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u0 = 0; u0 < BLOCKS; u0 += 4) {   // four blocks' reads of LDS are on their way together
      if (16 * u0 >= chunks) break;
      FlowChunk x[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) x[v].raw = *reinterpret_cast<const flow_u4*>(xs + min(16 * (u0 + v) + blk, chunks - 1) * 8);
      if (16 * (u0 + 4) > chunks)   // (past k: zeros)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const bool there = 16 * (u0 + v) + blk < chunks;
          x[v].raw = there ? x[v].raw : flow_u4{0u, 0u, 0u, 0u};
#pragma unroll
          for (int q = 0; q < Q; ++q) w[u0 + v][q].raw = there ? w[u0 + v][q].raw : flow_u4{0u, 0u, 0u, 0u};
        }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (16 * (u0 + v) >= chunks) break;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < Q; ++q) acc[q][h] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(w[u0 + v][q].h[h], x[v].h[h], acc[q][h], 0, 0, 0);
      }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const flow_f4 both = acc[q][0] + acc[q][1];
      float v = add_rows(add_halves(both[0], both[1]), add_halves(both[2], both[3]));
      v += row_ror<8>(v);
      y[q] = v + row_ror<4>(v);
    }
  }
};
__device__ __forceinline__ int flow_row() {   // of the quad, whose sum this lane has (sixteen lanes a row)
  const int j = threadIdx.x % 64 / 16;
  return j / 2 + j % 2 * 2;
}

// Pairs of tiles of the keys that lie in the pages, and one more for the new token's; a pair a wave, more where the runs are as many
// as they may be.
__host__ __device__ constexpr int flow_pairs(int n_keys) { return (n_keys - 1 + 31) / 32; }
__host__ __device__ constexpr int flow_splits(int n_keys) {
  const int runs = (flow_pairs(n_keys) + FLOW_WAVES) / FLOW_WAVES;
  return runs < 1 ? 1 : runs > FLOW_SPLITS ? FLOW_SPLITS : runs;
}

__device__ __forceinline__ flow_f4 flow_mfma(flow_u4 a, flow_u4 b, flow_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(flow_bf16x8, a), __builtin_bit_cast(flow_bf16x8, b), c, 0, 0, 0);
}

// One (kv head, run of keys): the arithmetic of the decode attention (attention_mfma.hip). The new token's key and value come by way
// of their words, as a pair of tiles of which one key counts; after WAIT looks at them it gives up.
template <int D, int WAIT, typename Near>
__device__ __forceinline__ void flow_attention(const FlowArgs& p, const FlowLayer& L, __amdgpu_buffer_rsrc_t words, unsigned layer_at, unsigned tag,
                                               unsigned tag32, int kvh, int split, unsigned char* lds, const Near& near) {
  constexpr int KC = D / 32, DCH = D / 16;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), col = lane % 16, grp = lane / 16;
  const int n_keys = p.kv_len[0], old = n_keys - 1, splits = flow_splits(n_keys), group = p.q_heads / p.kv_heads;
  if (split >= splits) return;
  const int pairs = flow_pairs(n_keys), stride = FLOW_WAVES * splits, ps = p.page_size;
  struct Pair { flow_u4 k[2][KC], v[DCH]; };
  const int k_row = (col >> 2 & 1) * 8 + (col & 3);
  const auto fetch = [&](Pair& g, int pair) {   // (past the end: the last tile again, masked)
    const bf16_t *kp[2], *vp[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const unsigned tile = (unsigned)max(min(2 * pair + u, (old - 1) / 16), 0), nth = p.page_of.page(tile);
      const int64_t page = __builtin_amdgcn_readfirstlane(p.block_table[min((int)nth, p.table_width - 1)]);
      const int off = (int)(tile - nth * p.page_of.tiles) * 16;
      const int64_t at = (max(page, (int64_t)0) * p.kv_heads + kvh) * ps * D;
      kp[u] = L.k_pages + at + (int64_t)off * D;
      vp[u] = L.v_pages + at + off;
    }
    const bf16_t* k = (col >= 8 ? kp[1] : kp[0]) + k_row * D + grp * 8;
    const bf16_t* v = (grp >= 2 ? vp[1] : vp[0]) + col * ps + 8 * (grp & 1);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int c = 0; c < KC; ++c) g.k[u][c] = *reinterpret_cast<const flow_u4*>(k + 4 * u * D + c * 32);
#pragma unroll
    for (int c = 0; c < DCH; ++c) g.v[c] = *reinterpret_cast<const flow_u4*>(v + c * 16 * ps);
  };
  Pair sets[2];
  int pair = split * FLOW_WAVES + wave;
  fetch(sets[0], pair);
  fetch(sets[1], pair + stride);
  near();

  const int head = kvh * group + col;
  // The query, and for the wave that takes the new token its key and value, in one round of waiting. (Each lane asks for what it will use;
  // the rest goes past the end of the words, which costs no traffic: all lanes all the time are 1,500 cycles of the vector cache a round.)
  const bool takes_new = pairs % stride == split * FLOW_WAVES + wave;
  const bool asks_q = col < group, asks_k = takes_new && col == 0, asks_v = takes_new && grp == 0;
  constexpr unsigned NOWHERE = 0xffffff00u;
  flow_u4 q[KC], k_new[KC];
  unsigned v_new[DCH];
  {
    unsigned at[4 * KC], at_v[DCH];
    flow_u4 w[4 * KC];
#pragma unroll
    for (int c = 0; c < 2 * KC; ++c) {
      const int dim = c / 2 * 32 + grp * 8 + c % 2 * 4;
      at[c] = asks_q ? layer_at + (head * D + dim) * 4 : NOWHERE;
      at[2 * KC + c] = asks_k ? layer_at + ((p.q_heads + kvh) * D + dim) * 4 : NOWHERE;
    }
#pragma unroll
    for (int c = 0; c < DCH; ++c) at_v[c] = asks_v ? layer_at + ((p.q_heads + p.kv_heads + kvh) * D + c * 16 + col) * 4 : NOWHERE;
    for (int tries = 0;; ++tries) {
      asm volatile("" ::: "memory");
      unsigned wrong = 0;
#pragma unroll
      for (int c = 0; c < 4 * KC; ++c) w[c] = __builtin_amdgcn_raw_buffer_load_b128(words, (int)at[c], 0, DEVICE_SCOPE);
#pragma unroll
      for (int c = 0; c < DCH; ++c) v_new[c] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(words, (int)at_v[c], 0, DEVICE_SCOPE);
#pragma unroll
      for (int c = 0; c < 4 * KC; ++c) {
        const unsigned off = (w[c][0] ^ tag) | (w[c][1] ^ tag) | (w[c][2] ^ tag) | (w[c][3] ^ tag);
        wrong |= (c < 2 * KC ? asks_q : asks_k) ? off : 0u;
      }
#pragma unroll
      for (int c = 0; c < DCH; ++c) wrong |= asks_v ? v_new[c] ^ tag : 0u;
      if ((wrong & 0xffffu) == 0) break;
      if (tries == WAIT) {   // (of the value, what is not there is told by its word, below)
#pragma unroll
        for (int c = 0; c < 4 * KC; ++c) w[c] = flow_u4{0x7fc00000u, 0x7fc00000u, 0x7fc00000u, 0x7fc00000u};
        break;
      }
    }
    const auto packed = [&](int c, int i) { return w[c + i / 2][i % 2 * 2] >> 16 | (w[c + i / 2][i % 2 * 2 + 1] & 0xffff0000u); };
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        q[c][i] = packed(2 * c, i);
        k_new[c][i] = packed(2 * KC + 2 * c, i);
      }
  }
  float m = -INFINITY, l = 0.f;
  flow_f4 o[DCH];
#pragma unroll
  for (int c = 0; c < DCH; ++c) o[c] = flow_f4{0.f, 0.f, 0.f, 0.f};
  const auto attend = [&](const Pair& g, int t, int count) {   // keys t + 8 grp + i, those below `count` count
    float sv[8];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      flow_f4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < KC; ++c) s = flow_mfma(g.k[u][c], q[c], s);
#pragma unroll
      for (int i = 0; i < 4; ++i) sv[4 * u + i] = s[i] * p.scale_log2e;
    }
    const int here = t + 8 * grp;
    flow_u4 v[DCH];
#pragma unroll
    for (int c = 0; c < DCH; ++c) v[c] = g.v[c];
    if (t + 32 > count) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (here + i >= count) sv[i] = -INFINITY;
      // a zero probability must not multiply whatever a not yet written slot holds
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const unsigned keep = (here + 2 * j < count ? 0xffffu : 0u) | (here + 2 * j + 1 < count ? 0xffff0000u : 0u);
#pragma unroll
        for (int c = 0; c < DCH; ++c) v[c][j] &= keep;
      }
    }
    float top = m;
#pragma unroll
    for (int i = 0; i < 8; ++i) top = fmaxf(top, sv[i]);
    const float m_new = max_across32(max_across16(top)), m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m - m_safe);
    float sum = 0.f;
    flow_bf16x8 pb;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float e = __builtin_amdgcn_exp2f(sv[i] - m_safe);
      sum += e;
      pb[i] = (bf16_t)e;
    }
    l = l * alpha + sum;
    m = m_new;
#pragma unroll
    for (int c = 0; c < DCH; ++c) o[c] *= alpha;
#pragma unroll
    for (int c = 0; c < DCH; ++c) o[c] = flow_mfma(v[c], __builtin_bit_cast(flow_u4, pb), o[c]);
  };
  for (; pair < pairs; pair += 2 * stride) {
    attend(sets[0], pair * 32, old);
    if (pair + stride < pairs) attend(sets[1], (pair + stride) * 32, old);
    if (pair + 2 * stride < pairs) {
      fetch(sets[0], pair + 2 * stride);
      fetch(sets[1], pair + 3 * stride);
    }
  }
  if (takes_new) {   // the new token's key: the first of a pair of tiles
    Pair g;
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      g.k[0][c] = col == 0 ? k_new[c] : flow_u4{0u, 0u, 0u, 0u};
      g.k[1][c] = flow_u4{0u, 0u, 0u, 0u};
    }
    // A lane's query is its column's head's alone, its part of the value every head's: a word that never came is not a number here. (Made
    // so where the wait gives up, the loop's registers moved about: 1.7% of a step of the 135M sizes.)
#pragma unroll
    for (int c = 0; c < DCH; ++c) {
      const unsigned value = ((v_new[c] ^ tag) & 0xffffu) == 0 ? v_new[c] >> 16 : 0x7fc0u;
      g.v[c] = flow_u4{grp == 0 ? value : 0u, 0u, 0u, 0u};
    }
    attend(g, 0, 1);
  }
  l = add_across32(add_across16(l));

  // the waves' states meet in LDS: [wave][quad of dims][head] and their statistics
  flow_f4* sm_o = reinterpret_cast<flow_f4*>(lds);
  float* sm_ml = reinterpret_cast<float*>(lds + FLOW_WAVES * (D / 4) * 16 * 16);
  if (grp == 0) {
    sm_ml[wave * 32 + col] = m;
    sm_ml[wave * 32 + 16 + col] = l;
  }
#pragma unroll
  for (int c = 0; c < DCH; ++c) sm_o[(wave * (D / 4) + c * 4 + grp) * 16 + col] = o[c];
  __syncthreads();
  for (int item = threadIdx.x; item < 16 * (D / 4); item += FLOW_THREADS) {
    const int h = item % 16, quad = item / 16;
    if (h >= group) continue;
    float top = sm_ml[h];
#pragma unroll
    for (int w = 1; w < FLOW_WAVES; ++w) top = fmaxf(top, sm_ml[w * 32 + h]);
    const float safe = top == -INFINITY ? 0.f : top;
    float sum = 0.f;
    flow_f4 all = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < FLOW_WAVES; ++w) {
      const float f = __builtin_amdgcn_exp2f(sm_ml[w * 32 + h] - safe);
      sum += sm_ml[w * 32 + 16 + h] * f;
      all = all + sm_o[(w * (D / 4) + quad) * 16 + h] * f;
    }
    const unsigned at = layer_at + p.at_part + ((kvh * group + h) * FLOW_SPLITS + split) * (D + 2) * 8;
    const auto leave = [&](unsigned to, float a, float b) {
      __builtin_amdgcn_raw_buffer_store_b128(flow_u4{__float_as_uint(a), tag32, __float_as_uint(b), tag32}, words, (int)to, 0, DEVICE_SCOPE);
    };
    if (quad == 0) leave(at, top, sum);
    leave(at + 16 + quad * 32, all[0], all[1]);
    leave(at + 16 + quad * 32 + 16, all[2], all[3]);
  }
}

// grid: layers x layer_wgs. Dynamic LDS: the row, or the attention's states.
template <int D, int WAIT>
__global__ __launch_bounds__(FLOW_THREADS) void decode_flow_kernel(FlowArgs p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  __shared__ unsigned long long sh_ticket;
  __shared__ float scratch[FLOW_WAVES], sums[FLOW_WAVES];
  bf16_t* const xs = reinterpret_cast<bf16_t*>(lds);
  const int tid = threadIdx.x;
  if (tid == 0) sh_ticket = __hip_atomic_fetch_add(p.tickets, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const unsigned ticket = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)sh_ticket);
  const unsigned tag32 = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(sh_ticket >> 32)) + 1, tag = tag32 & 0xffffu;
  // (all tickets are out: the next launch's begin at zero)
  if (tid == 0 && ticket + 1 == (unsigned)(p.num_layers * p.layer_wgs)) 
    __hip_atomic_store(p.tickets, (unsigned long long)tag32 << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int layer = (int)(ticket / (unsigned)p.layer_wgs);
  int piece = (int)(ticket - (unsigned)(layer * p.layer_wgs));
  const FlowLayer L = p.layers[layer];
  const __amdgpu_buffer_rsrc_t words = __builtin_amdgcn_make_buffer_rsrc(p.words, 0, p.num_layers * p.layer_bytes, 0x00020000);
  const unsigned at_layer = (unsigned)layer * p.layer_bytes, at_before = at_layer - p.layer_bytes;
  // Only the two kinds that are next look at their values all the time; others look at one word of the kind before theirs now and then.
  const auto near = [&](unsigned at, unsigned mask, unsigned want) {
    if (tid < 64)
      for (int tries = 0; tries < FLOW_WAIT; ++tries) {
        asm volatile("" ::: "memory");
        if ((((unsigned)__builtin_amdgcn_raw_buffer_load_b32(words, (int)at, 0, DEVICE_SCOPE) ^ want) & mask) == 0) break;
        __builtin_amdgcn_s_sleep(8);
      }
    __syncthreads();
  };
  const int hidden = p.hidden, attn = p.q_heads * D;

  const int wave = __builtin_amdgcn_readfirstlane(tid / 64), mine = flow_row();
  const bool stores = tid % 16 == 0;   // one lane for each of a wave's four sums

  // A row of the stream (four values a thread) times the norm's weights into LDS. Its scale multiplies the products' sums instead, so
  // that only one barrier lies between the values and the products; they are rounded once.
  const auto weighted = [&](const float* weight, bool plain, unsigned at) {
    const int quad = min(tid, hidden / 4 - 1);
    const flow_f4 w = *reinterpret_cast<const flow_f4*>(weight + 4 * quad);
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (plain) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (float)p.x[4 * quad + i];
    } else if (64 * wave < hidden / 4) {   // (the waves that have values to wait for)
      const unsigned from[1] = {at + quad * 16};
      flow_u4 got[1];
      flow_wait(words, from, tag, got);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = flow_value(got[0][i]);
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) ss = fmaf(v[i], v[i], ss);
    ss = wave_sum(tid < hidden / 4 ? ss : 0.f);
    if (tid % 64 == 0) scratch[wave] = ss;
    typedef bf16_t four __attribute__((ext_vector_type(4)));
    if (tid < hidden / 4) *reinterpret_cast<four*>(xs + 4 * tid) = four{(bf16_t)(w[0] * v[0]), (bf16_t)(w[1] * v[1]), (bf16_t)(w[2] * v[2]), (bf16_t)(w[3] * v[3])};
  };
  const auto over_waves = [](const float (&of)[FLOW_WAVES]) {
    float sum = of[0];
#pragma unroll
    for (int w = 1; w < FLOW_WAVES; ++w) sum += of[w];
    return sum;
  };
  const auto scale = [&] { return rsqrtf(over_waves(scratch) / (float)hidden + p.eps); };
  // the products of `rows` rows, four a wave, added to the stream
  const auto stream_value = [&](int rows, int n0, bool plain, unsigned at) {   // of the row whose sum this lane gets
    const int n = n0 + min(4 * wave, rows - 4) + mine;
    return plain ? (float)p.x[n] : flow_value(flow_wait_word(words, at + n * 4, tag));
  };
  const auto add_to_stream = [&](auto& weights, float old, int rows, int k, int n0, unsigned at, bool last, int part) {
    __syncthreads();
    float square = 0.f;
    if (wave < rows / 4) {
      const int n = n0 + 4 * wave + mine;
      float y[1];
      weights.multiply(k, xs, y);
      const bf16_t sum = (bf16_t)(old + (float)(bf16_t)y[0]);
      if (stores) {
        if (last) p.x[n] = sum;
        else flow_leave(words, at + n * 4, sum, tag);
        square = (float)sum * (float)sum;
      }
    }
    if (last) {
      square = wave_sum(square);
      if (tid % 64 == 0) sums[wave] = square;
      __syncthreads();
      if (tid == 0) p.ssq_out[part] = over_waves(sums);
    }
  };

  if (piece < p.wgs[0]) {   // q, k and v: pairs that are rotated together
    const int rows = p.rows[0], half = rows / 2, pair0 = piece * half, head = pair0 / (D / 2), j0 = pair0 % (D / 2), row0 = head * D + j0;
    const int quad = min(4 * wave, half - 4), first[2] = {row0 + quad, row0 + D / 2 + quad};
    FlowWeights<2, FLOW_BLOCKS> weights;
    weights.ask(L.w_qkv, hidden, first);
    const bool rotates = head < p.q_heads + p.kv_heads;
    const int at = quad + mine, slot = p.slots[0];   // this lane's pair
    const float c = p.angles[j0 + at], s = p.angles[D / 2 + j0 + at];
    if (layer > 0) near(at_before + p.at_act, 0xffffu, tag);
    weighted(L.norm1, layer == 0, at_before + p.at_x2);
    __syncthreads();
    if (wave >= half / 4) return;
    const float rs = scale();
    float y[2];
    weights.multiply(hidden, xs, y);
    if (stores) {
      const float a = y[0] * rs, b = y[1] * rs;
      const bf16_t lo = (bf16_t)(rotates ? a * c - b * s : a), hi = (bf16_t)(rotates ? b * c + a * s : b);
      const int n = row0 + at;
      flow_leave(words, at_layer + n * 4, lo, tag);
      flow_leave(words, at_layer + (n + D / 2) * 4, hi, tag);
      if (head >= p.q_heads && slot >= 0) {
        const int64_t page = slot / p.page_size, off = slot % p.page_size;
        const int d = j0 + at;
        if (rotates) {
          bf16_t* k = L.k_pages + ((page * p.kv_heads + head - p.q_heads) * p.page_size + off) * D + d;
          k[0] = lo;
          k[D / 2] = hi;
        } else {
          bf16_t* v = L.v_pages + ((page * p.kv_heads + head - p.q_heads - p.kv_heads) * D + d) * p.page_size + off;
          v[0] = lo;
          v[(int64_t)D / 2 * p.page_size] = hi;
        }
      }
    }
    return;
  }
  piece -= p.wgs[0];
  if (piece < p.kv_heads * p.splits) {
    flow_attention<D, WAIT>(p, L, words, at_layer, tag, tag32, piece % p.kv_heads, piece / p.kv_heads, lds, [&] {
      if (layer > 0) near(at_before + p.at_x2, 0xffffu, tag);
    });
    return;
  }
  piece -= p.kv_heads * p.splits;
  if (piece < p.wgs[1]) {   // o, behind the merge of the runs
    const int rows = p.rows[1], n0 = piece * rows;
    const int first[1] = {n0 + min(4 * wave, rows - 4)};
    FlowWeights<1, FLOW_BLOCKS> weights;
    weights.ask(L.w_o, attn, first);
    const int splits = flow_splits(p.kv_len[0]);
    near(at_layer, 0xffffu, tag);
    const float old = stream_value(rows, n0, layer == 0, at_before + p.at_x2);
    {
      const int quad = min(tid, attn / 4 - 1), head = quad / (D / 4), dq = quad % (D / 4);
      const unsigned at = at_layer + p.at_part + head * FLOW_SPLITS * (D + 2) * 8;
      float top = -INFINITY, sum = 0.f;
      flow_f4 all = {0.f, 0.f, 0.f, 0.f};
      const auto merge = [&](auto at_once) {   // (a run past the last: the last again, which counts as nothing)
        constexpr int RUNS = decltype(at_once)::value;
        for (int s0 = 0; s0 < splits; s0 += RUNS) {
          unsigned from[3 * RUNS];
          flow_u4 got[3 * RUNS];
#pragma unroll
          for (int k = 0; k < RUNS; ++k) {
            const unsigned run = at + min(s0 + k, splits - 1) * (D + 2) * 8;
            from[3 * k] = run;
            from[3 * k + 1] = run + 16 + dq * 32;
            from[3 * k + 2] = run + 32 + dq * 32;
          }
          flow_wait_pairs(words, from, tag32, got);
          float new_top = top;
#pragma unroll
          for (int k = 0; k < RUNS; ++k)
            if (s0 + k < splits) new_top = fmaxf(new_top, __uint_as_float(got[3 * k][0]));
          const float safe = new_top == -INFINITY ? 0.f : new_top, keep = __builtin_amdgcn_exp2f(top - safe);
          sum *= keep;
          all *= keep;
          top = new_top;
#pragma unroll
          for (int k = 0; k < RUNS; ++k) {
            const float f = s0 + k < splits ? __builtin_amdgcn_exp2f(__uint_as_float(got[3 * k][0]) - safe) : 0.f;
            sum = fmaf(__uint_as_float(got[3 * k][2]), f, sum);
            all[0] = fmaf(__uint_as_float(got[3 * k + 1][0]), f, all[0]);
            all[1] = fmaf(__uint_as_float(got[3 * k + 1][2]), f, all[1]);
            all[2] = fmaf(__uint_as_float(got[3 * k + 2][0]), f, all[2]);
            all[3] = fmaf(__uint_as_float(got[3 * k + 2][2]), f, all[3]);
          }
        }
      };
      // (a round of waiting is a trip to memory: two to eight runs each)
      if (64 * wave < attn / 4) {
        if (splits <= 2) merge(std::integral_constant<int, 2>());
        else if (splits <= 4) merge(std::integral_constant<int, 4>());
        else merge(std::integral_constant<int, 8>());
      }
      const float inv = sum > 0.f ? 1.f / sum : 0.f;
      if (tid < attn / 4)
#pragma unroll
        for (int i = 0; i < 4; ++i) xs[4 * tid + i] = (bf16_t)(all[i] * inv);
    }
    add_to_stream(weights, old, rows, attn, n0, at_layer + p.at_x1, false, 0);
    return;
  }
  piece -= p.wgs[1];
  if (piece < p.wgs[2]) {   // gate and up
    const int rows = p.rows[2], half = rows / 2, n0 = piece * half;
    const int quad = min(4 * wave, half - 4), first[2] = {n0 + quad, p.inner + n0 + quad};
    FlowWeights<2, FLOW_BLOCKS> weights;
    weights.ask(L.w_gate_up, hidden, first);
    near(at_layer + p.at_part + 4, 0xffffffffu, tag32);
    weighted(L.norm2, false, at_layer + p.at_x1);
    __syncthreads();
    if (wave >= half / 4) return;
    const float rs = scale();
    float y[2];
    weights.multiply(hidden, xs, y);
    if (stores) {
      const GluForm silu_form = {GLU_SILU, 0.f, 0.f, 0.f};
      flow_leave(words, at_layer + p.at_act + (n0 + 4 * wave + mine) * 4, glu_bf16((float)(bf16_t)(y[0] * rs), (float)(bf16_t)(y[1] * rs), silu_form), tag);
    }
    return;
  }
  piece -= p.wgs[2];
  {   // down
    const int rows = p.rows[3], n0 = piece * rows;
    const int first[1] = {n0 + min(4 * wave, rows - 4)};
    FlowWeights<1, FLOW_INNER_BLOCKS> weights;
    weights.ask(L.w_down, p.inner, first);
    near(at_layer + p.at_x1, 0xffffu, tag);
    const float old = stream_value(rows, n0, false, at_layer + p.at_x1);
    constexpr int QUADS = (FLOW_INNER_BLOCKS * 32 + FLOW_THREADS - 1) / FLOW_THREADS;   // a thread's
    const int quads = p.inner / 4;
    const auto take = [&](auto each) {
      constexpr int N = decltype(each)::value;
      unsigned from[N];
      flow_u4 got[N];
#pragma unroll
      for (int k = 0; k < N; ++k) from[k] = at_layer + p.at_act + min(tid + k * FLOW_THREADS, quads - 1) * 16;
      flow_wait(words, from, tag, got);
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const int quad = tid + k * FLOW_THREADS;
        if (quad < quads)
          *reinterpret_cast<uint2*>(xs + 4 * quad) = uint2{got[k][0] >> 16 | (got[k][1] & 0xffff0000u), got[k][2] >> 16 | (got[k][3] & 0xffff0000u)};
      }
    };
    if (quads > FLOW_THREADS) take(std::integral_constant<int, QUADS>());
    else if (64 * wave < quads) take(std::integral_constant<int, 1>());
    add_to_stream(weights, old, rows, p.inner, n0, at_layer + p.at_x2, layer + 1 == p.num_layers, piece);
  }
}

// Rows of weights a workgroup, four or eight a wave: no more than divide the matrix. 0: none do.
int flow_rows(int n, bool paired) {
  for (int rows = (paired ? 8 : 4) * FLOW_WAVES; rows >= (paired ? 8 : 4); rows /= 2)
    if (n % rows == 0) return rows;
  return 0;
}

bool flow_plan(FlowArgs& a, int layers, int hidden, int q_heads, int kv_heads, int head_dim, int inner) {
  if (layers < 1 || hidden < 8 || q_heads < 1 || kv_heads < 1 || q_heads % kv_heads || q_heads / kv_heads > 16 || inner < 8) return false;
  if (head_dim != 64 && head_dim != 128) return false;
  const int64_t attn = (int64_t)q_heads * head_dim, qkv = attn + 2 * (int64_t)kv_heads * head_dim;
  if (hidden > 128 * FLOW_BLOCKS || attn > 128 * FLOW_BLOCKS || inner > 128 * FLOW_INNER_BLOCKS || hidden % 8 || inner % 8) return false;
  const int n[4] = {(int)qkv, hidden, 2 * inner, hidden};
  a.layer_wgs = 0;
  for (int i = 0; i < 4; ++i) {
    a.rows[i] = flow_rows(n[i], i % 2 == 0);
    if (a.rows[i] == 0) return false;
    a.wgs[i] = n[i] / a.rows[i];
    a.layer_wgs += a.wgs[i];
  }
  const auto whole = [](int64_t bytes) { return (bytes + 127) / 128 * 128; };
  const int64_t part = whole(qkv * 4), x1 = part + whole((int64_t)q_heads * FLOW_SPLITS * (head_dim + 2) * 8), act = x1 + whole((int64_t)hidden * 4),
                x2 = act + whole((int64_t)inner * 4), end = x2 + whole((int64_t)hidden * 4);
  if (end * layers >= (int64_t)1 << 31 || (int64_t)(a.layer_wgs + kv_heads * FLOW_SPLITS) * layers >= (int64_t)1 << 31) return false;
  a.at_part = (unsigned)part; a.at_x1 = (unsigned)x1; a.at_act = (unsigned)act; a.at_x2 = (unsigned)x2; a.layer_bytes = (unsigned)end;
  a.num_layers = layers; a.hidden = hidden; a.q_heads = q_heads; a.kv_heads = kv_heads; a.inner = inner;
  return true;
}

}  // namespace

extern "C" {

// Bytes of the words of such a model (which begin as zeros and are the launches' own), 0 where the kernel does not take its sizes.
int dli_decode_flow_bytes(int layers, int hidden, int q_heads, int kv_heads, int head_dim, int inner) {
  FlowArgs a;
  return flow_plan(a, layers, hidden, q_heads, kv_heads, head_dim, inner) ? (int)(a.layer_bytes * (unsigned)layers) : 0;
}

// Parts of the row's sum of squares that a launch leaves.
int dli_decode_flow_parts(int layers, int hidden, int q_heads, int kv_heads, int head_dim, int inner) {
  FlowArgs a;
  return flow_plan(a, layers, hidden, q_heads, kv_heads, head_dim, inner) ? a.wgs[3] : 0;
}

// x [hidden] bfloat16: the stream, in place; ssq_out float32 [dli_decode_flow_parts]. layers_at: per layer the addresses norm1, norm2, w_qkv,
// w_o, w_gate_up, w_down, k_pages, v_pages (on the device). tickets: one zero before the first launch, then the launches' own.
// At most table_width * page_size keys. impatient: the attention gives up on the new token's query, key and value at its first look, so
// that what it leaves then can be seen (a kernel of its own: the limit as an argument took 0.5% of a step of the 135M sizes).
int dli_decode_flow(const void* layers_at, int layers, void* words, void* tickets, void* x, float* ssq_out, const float* angles, const int* slots,
                    const int* kv_len, const int* block_table, int table_width, int hidden, int q_heads, int kv_heads, int head_dim, int inner,
                    int page_size, float eps, float scale, int impatient, hipStream_t stream) {
  FlowArgs a;
  if (!flow_plan(a, layers, hidden, q_heads, kv_heads, head_dim, inner) || page_size < 16 || page_size % 16 || table_width < 1 ||
      (int64_t)table_width * page_size > (int64_t)1 << 30) return DLI_ERR_ARGUMENT;
  a.layers = (const FlowLayer*)layers_at; a.words = words; a.tickets = (unsigned long long*)tickets;
  a.x = (bf16_t*)x; a.ssq_out = ssq_out; a.angles = angles; a.slots = slots; a.kv_len = kv_len; a.block_table = block_table; a.table_width = table_width;
  a.splits = flow_splits(table_width * page_size);
  a.layer_wgs += kv_heads * a.splits;
  a.page_size = page_size; a.page_of = page_of_tile(page_size); a.eps = eps; a.scale_log2e = scale * 1.4426950408889634f;
  const int rows = 2 * 128 * FLOW_INNER_BLOCKS, states = FLOW_WAVES * ((head_dim / 4) * 16 * 16 + 32 * 4), bytes = rows > states ? rows : states;
  const auto kernel = head_dim == 64 ? (impatient ? decode_flow_kernel<64, 0> : decode_flow_kernel<64, FLOW_WAIT>)
                                     : (impatient ? decode_flow_kernel<128, 0> : decode_flow_kernel<128, FLOW_WAIT>);
  if (bytes > 65536 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return DLI_ERR_LAUNCH;
  kernel<<<layers * a.layer_wgs, FLOW_THREADS, bytes, stream>>>(a);
  return dli_launch_status();
}

}  // extern "C"
