// The gated delta rule: a matrix state S [key][value] per head in 32-bit, carried from token to token
// of a request in its state slot, with one decay g and one write strength beta per head and token:
//
//   S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q      (in this order: o is made from the state that already holds the token)
//
// Keys and values may differ in size (D keys, V values a head), and several value heads may share
// the q and k of one of `kv_heads` heads. Around it, in the same 32-bit arithmetic:
//
//   conv_prepare       from the 32-bit projections of a step's rows: a short causal convolution over
//                      time per channel of q, k and v (the last taps-1 inputs of the step before come
//                      from the request's state; zeros before position 0), silu, q and k made unit
//                      vectors per head (q also times D^-1/2), beta = sigmoid(b),
//                      g = exp(-exp(A_log) softplus(a + dt_bias))
//   conv_keep          the step's last taps-1 inputs into the request's state
//   causal_conv        the short causal convolution alone, for any mixer: per channel, with an optional bias and
//                      silu, from the same kind of kept inputs; the result in 32-bit and, if wanted, once more
//                      in the type of the product that reads it next
//   gated_delta_scan   the recurrence; o in 32-bit
//   gated_delta_single all of it, with each head's norm and gate, for a step of single tokens
//
// With old state S, ks = S^T k and qs = S^T q (both from the old S, so their sums run side by side):
// u = beta (v - g ks), S_new = g S + k u^T, o = g qs + u (k . q).
//
// One wave takes one (entry, head, slice of 4 value columns) and walks the entry's tokens in order.
// Sixteen lanes (a DPP row) share a column: lane (col, part) keeps S[part's D/16 keys][col] in
// registers, and the two dot products of a token meet in four DPP swaps each. The vectors of 16
// tokens are staged in LDS while the next 16 are in flight, so the chain reads LDS and registers
// only. Heads whose D is no multiple of 16 (or above 256) take a thread-per-column kernel that keeps
// the state in memory: slow, there so that no size is refused.
//
// State slot: [heads][V][D] floats, then [taps-1][channels] floats of kept inputs (the last row is
// the newest). A request whose first row of the step has position 0 starts from zeros; nothing
// needs clearing when a slot changes hands.
#include <type_traits>

#include "common.h"
#include "scan_runs.h"

// The entry that holds `row`: the last e with q_start[e] <= row.
__device__ __forceinline__ int gd_entry_of_row(const int* __restrict__ q_start, int entries, int row) {
  int lo = 0, hi = entries - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (q_start[mid] <= row) lo = mid; else hi = mid - 1;
  }
  return lo;
}

struct PrepArgs {
  const float* proj; int64_t stride;       // [rows][stride]: q | k | v channels from column 0, then what follows
  int b_off, a_off;                        // columns of beta's and the decay's pre-activations (heads each)
  const float* conv_w;                     // [channels][taps], the last column the current token's
  const float* a_log; const float* dt_bias;  // [heads]
  const float* kept; int64_t state_stride; // the requests' kept inputs: state + offset, [taps-1][channels] a slot
  float* keep;                             // the same where every entry is one row: its wave also writes the new ones (else nullptr)
  const int* q_start; const int* positions; const int* state_slots;
  float* out; int64_t out_stride;          // [rows][channels + 2 heads]: q | k | v | beta | g
  int entries, heads, kv_heads, dim, vdim, taps;
};

// The convolution of channel c at `row`, which lies at position pos of its request, whose step starts at row `first`, and silu. An
// input lies among the step's rows or the kept inputs, or before the sequence (zero; another input is read in its place). The taps
// are asked for together (TAPS of them, or where that is 0 four at a time): no load hangs on a condition. Oldest input first.
// keep: an entry's only row also leaves the inputs that the next one needs, one place further back, so that a step of single tokens needs
// no kernel for that after this one (4.8 us of a step of four requests): tap t's input, from place t, goes to place t - 1, which
// has been read.
template <int TAPS>
__device__ __forceinline__ float conv_silu(const PrepArgs& p, const float* kept, float* keep, int channels, int row, int first, int pos, int c) {
  constexpr int AT_ONCE = TAPS > 0 ? TAPS : 4;
  const int taps = TAPS > 0 ? TAPS : p.taps;
  const float* w = p.conv_w + (int64_t)c * taps;
  float acc = 0.f;
  if (row - (taps - 1) >= first) {                              // (most rows of a portion)
    const float* x = p.proj + (int64_t)(row - (taps - 1)) * p.stride + c;
#pragma unroll 4
    for (int t = 0; t < taps; ++t) acc = fmaf(w[t], x[(int64_t)t * p.stride], acc);
  } else {
    for (int t0 = 0; t0 < taps; t0 += AT_ONCE) {                // tap t: the input taps - 1 - t places back
      float in[AT_ONCE], wt[AT_ONCE];
#pragma unroll
      for (int k = 0; k < AT_ONCE; ++k) {
        const int t = min(t0 + k, taps - 1), back = min(taps - 1 - t, pos), src = row - back;
        in[k] = *(src >= first ? p.proj + (int64_t)src * p.stride + c : kept + (int64_t)(taps - 1 - (first - src)) * channels + c);
        wt[k] = w[t];
      }
#pragma unroll
      for (int k = 0; k < AT_ONCE; ++k) {
        const float x = taps - 1 - (t0 + k) <= pos ? in[k] : 0.f;
        if (t0 + k < taps) acc = fmaf(wt[k], x, acc);
        if (keep != nullptr && t0 + k >= 1 && t0 + k < taps) keep[(int64_t)(t0 + k - 1) * channels + c] = x;
      }
    }
  }
  return acc / (1.f + expf(-acc));
}

// Units: the 2 kv_heads heads of q and k (convolution, silu, unit length), then the channels of v in runs of 64 (convolution,
// silu), then one for beta and g of all heads.
__device__ __forceinline__ void conv_prepare_gates(float b, float a_pre, float a_log, float dt_bias, float& beta, float& g) {
  const float a = a_pre + dt_bias;
  const float softplus = a > 20.f ? a : log1pf(expf(a));
  beta = 1.f / (1.f + expf(-b));
  g = expf(-expf(a_log) * softplus);
}
__device__ __forceinline__ void conv_prepare_gates(const PrepArgs& p, int row, int h, float* out) {
  const float* proj = p.proj + (int64_t)row * p.stride;
  conv_prepare_gates(proj[p.b_off + h], proj[p.a_off + h], p.a_log[h], p.dt_bias[h], out[0], out[p.heads]);
}
__device__ __forceinline__ float conv_unit_scale(const PrepArgs& p, int unit, float ss) {
  return (1.f / sqrtf(wave_sum(ss) + 1e-6f)) * (unit < p.kv_heads ? 1.f / sqrtf((float)p.dim) : 1.f);
}
// One row of a unit of q, k or v.
template <int TAPS>
__device__ __forceinline__ void conv_prepare_row(const PrepArgs& p, int row, int unit) {
  const int lane = threadIdx.x, qk = p.kv_heads * p.dim, channels = 2 * qk + p.heads * p.vdim;
  float* out = p.out + (int64_t)row * p.out_stride;
  const int e = gd_entry_of_row(p.q_start, p.entries, row);
  const int first = p.q_start[e], pos = p.positions[row];
  const float* kept = p.kept + (int64_t)p.state_slots[e] * p.state_stride;
  float* keep = p.keep != nullptr ? p.keep + (int64_t)p.state_slots[e] * p.state_stride : nullptr;
  if (unit >= 2 * p.kv_heads) {
    const int c = 2 * qk + (unit - 2 * p.kv_heads) * 64 + lane;
    if (c < channels) out[c] = conv_silu<TAPS>(p, kept, keep, channels, row, first, pos, c);
    return;
  }
  const int c0 = unit * p.dim;                                  // q heads, then k heads
  float ss = 0.f;
  for (int c = lane; c < p.dim; c += DLI_WAVE) {
    const float y = conv_silu<TAPS>(p, kept, keep, channels, row, first, pos, c0 + c);
    out[c0 + c] = y;
    ss += y * y;
  }
  const float r = conv_unit_scale(p, unit, ss);
  for (int c = lane; c < p.dim; c += DLI_WAVE) out[c0 + c] *= r;   // (each lane scales what it wrote itself)
}

// A wave a (row, unit): steps of few rows.
template <int TAPS>
__global__ __launch_bounds__(64) void conv_prepare_kernel(PrepArgs p) {
  const int row = blockIdx.x, unit = blockIdx.y;
  if (unit + 1 < (int)gridDim.y) { conv_prepare_row<TAPS>(p, row, unit); return; }
  const int channels = 2 * p.kv_heads * p.dim + p.heads * p.vdim;
  for (int h = threadIdx.x; h < p.heads; h += DLI_WAVE)
    conv_prepare_gates(p, row, h, p.out + (int64_t)row * p.out_stride + channels + h);
}

// A wave PREP_RUN neighbouring rows of a unit, up to PREP_TAPS taps: a channel's inputs are read once for all rows that they reach
// where the run lies in one entry with its inputs among the step's rows; other runs take the rows one by one, in the same order of
// sums. Us a call, 3,072 channels and 32 heads, a wave a row -> now: 2,990 rows of 4 requests 53 -> 26, 1,100 of one 23.5 -> 16. It
// takes enough waves to make up for a wave's eight rows one after the other, the more the fewer taps a row has: with heads of 64
// and four taps 3,328 waves 13.4 -> 12.4 us and 2,444 11.5 -> 12.6, with two taps and heads of 32 6,144 16.5 -> 16.0 and 4,500
// 13.3 -> 14.5; heads above 64, whose lanes store before they scale, three taps, heads of 128: 12,375 41.8 -> 34.5, 8,448 30.8 ->
// 33.7. Not below 1,024 rows (256 rows of 4 requests 8.5 and 13.6) nor with under 64 rows a request (1,030 of 32 25.1 and 25.9).
#define PREP_RUN 8
#define PREP_TAPS 4
#define PREP_FROM_ROWS 1024
static bool conv_prepare_in_runs(int rows, int entries, int units, int dim, int taps) {
  const int64_t waves = (int64_t)((rows + PREP_RUN - 1) / PREP_RUN) * units;
  return rows >= PREP_FROM_ROWS && rows / 64 >= entries && taps <= PREP_TAPS && waves * taps >= (dim <= DLI_WAVE ? 16000 : 29000);
}
__global__ __launch_bounds__(64) void conv_prepare_run_kernel(PrepArgs p, int rows) {
  // (of several entries the runs are turned by the unit: those that take their rows one by one lie where entries begin, often at
  // multiples of eight runs, and would all fall to one XCD: 16 requests of 128 rows, 32 heads, 40.6 us, so 24.3)
  const int unit = blockIdx.y, turn = p.entries > 1 ? (blockIdx.x + blockIdx.y) % gridDim.x : blockIdx.x;
  const int row0 = turn * PREP_RUN, lane = threadIdx.x;
  const int last = min(row0 + PREP_RUN, rows);
  const int qk = p.kv_heads * p.dim, channels = 2 * qk + p.heads * p.vdim;
  if (unit + 1 == (int)gridDim.y) {
    for (int i = lane; i < (last - row0) * p.heads; i += DLI_WAVE) {
      const int row = row0 + i / p.heads, h = i % p.heads;
      conv_prepare_gates(p, row, h, p.out + (int64_t)row * p.out_stride + channels + h);
    }
    return;
  }
  const int e = gd_entry_of_row(p.q_start, p.entries, row0);
  if (row0 - (PREP_TAPS - 1) < p.q_start[e] || row0 + PREP_RUN > p.q_start[e + 1]) {
    for (int row = row0; row < last; ++row) conv_prepare_row<0>(p, row, unit);
    return;
  }
  const auto convolve = [&](int c, float (&y)[PREP_RUN]) {
    float w[PREP_TAPS], in[PREP_RUN + PREP_TAPS - 1];           // w[j]: the input j places back
#pragma unroll
    for (int j = 0; j < PREP_TAPS; ++j) w[j] = p.conv_w[(int64_t)c * p.taps + max(p.taps - 1 - j, 0)];
#pragma unroll
    for (int k = 0; k < PREP_RUN + PREP_TAPS - 1; ++k) in[k] = p.proj[(int64_t)(row0 - (PREP_TAPS - 1) + k) * p.stride + c];
#pragma unroll
    for (int r = 0; r < PREP_RUN; ++r) {
      float acc = 0.f;
#pragma unroll
      for (int j = PREP_TAPS - 1; j >= 0; --j)
        if (j < p.taps) acc = fmaf(w[j], in[r + PREP_TAPS - 1 - j], acc);   // oldest input first
      y[r] = acc / (1.f + expf(-acc));
    }
  };
  float y[PREP_RUN];
  float* out = p.out + (int64_t)row0 * p.out_stride;
  if (unit >= 2 * p.kv_heads) {
    const int c = 2 * qk + (unit - 2 * p.kv_heads) * 64 + lane;
    if (c >= channels) return;
    convolve(c, y);
#pragma unroll
    for (int r = 0; r < PREP_RUN; ++r) out[r * p.out_stride + c] = y[r];
    return;
  }
  float ss[PREP_RUN];
#pragma unroll
  for (int r = 0; r < PREP_RUN; ++r) ss[r] = 0.f;
  for (int c = lane; c < p.dim; c += DLI_WAVE) {
    convolve(unit * p.dim + c, y);
#pragma unroll
    for (int r = 0; r < PREP_RUN; ++r) {
      ss[r] += y[r] * y[r];
      if (p.dim > DLI_WAVE) out[r * p.out_stride + unit * p.dim + c] = y[r];
    }
  }
#pragma unroll
  for (int r = 0; r < PREP_RUN; ++r) {
    const float f = conv_unit_scale(p, unit, ss[r]);
    float* o = out + r * p.out_stride + unit * p.dim;
    if (p.dim > DLI_WAVE) {
      for (int c = lane; c < p.dim; c += DLI_WAVE) o[c] *= f;   // (each lane scales what it wrote itself)
    } else if (lane < p.dim) {
      o[lane] = y[r] * f;
    }
  }
}

// A thread a channel: it reads what it needs of the old kept inputs before it writes the new ones,
// and no other thread touches its channel. (Runs after conv_prepare of the same step, which reads what this overwrites for all rows
// of an entry, unless every entry is one row.)
#define GD_MAX_TAPS 16
__global__ void conv_keep_kernel(const float* __restrict__ proj, int64_t stride, float* kept_base, int64_t state_stride,
                                 const int* __restrict__ q_start, const int* __restrict__ positions,
                                 const int* __restrict__ state_slots, int channels, int taps, const float* __restrict__ in_bias) {
  const int e = blockIdx.x;
  const int first = q_start[e], end = q_start[e + 1];
  if (end <= first) return;
  const int pos0 = positions[first];
  float* kept = kept_base + (int64_t)state_slots[e] * state_stride;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  float fresh[GD_MAX_TAPS];
  for (int i = 0; i < taps - 1; ++i) {            // new kept row i holds the input `taps-1-i` places before `end`
    const int src = end - (taps - 1 - i);
    float x;
    if (src >= first) x = proj[(int64_t)src * stride + c] + (in_bias != nullptr ? in_bias[c] : 0.f);
    else if (pos0 - (first - src) < 0) x = 0.f;
    else x = kept[(int64_t)(taps - 1 - (first - src)) * channels + c];
    fresh[i] = x;
  }
  for (int i = 0; i < taps - 1; ++i) kept[(int64_t)i * channels + c] = fresh[i];
}

// A thread a (row, channel). x [rows][stride] holds the inputs of `channels` channels from column 0.
template <typename T>
__global__ void causal_conv_kernel(const float* __restrict__ x, int64_t stride, const float* __restrict__ conv_w,
                                   const float* __restrict__ bias, const float* kept_base, int64_t state_stride,
                                   const int* __restrict__ q_start, int entries, const int* __restrict__ positions,
                                   const int* __restrict__ state_slots, float* __restrict__ out, int64_t out_stride,
                                   T* __restrict__ rounded, int64_t rounded_stride, int channels, int taps, int act,
                                   const float* __restrict__ in_bias) {
  const int row = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const int e = gd_entry_of_row(q_start, entries, row);
  const int first = q_start[e], pos = positions[row];
  const float* kept = kept_base + (int64_t)state_slots[e] * state_stride;
  float acc = bias != nullptr ? bias[c] : 0.f;
  const float ib = in_bias != nullptr ? in_bias[c] : 0.f;        // (part of every input that exists, not of the zeros before)
  for (int j = taps - 1; j >= 0; --j) {                          // oldest input first
    float in = 0.f;
    if (pos - j >= 0) {
      const int src = row - j;
      in = src >= first ? x[(int64_t)src * stride + c] + ib : kept[(int64_t)(taps - 1 - (first - src)) * channels + c];
    }
    acc = fmaf(conv_w[(int64_t)c * taps + (taps - 1 - j)], in, acc);
  }
  if (act == 1) acc = acc / (1.f + expf(-acc));
  if (out != nullptr) out[(int64_t)row * out_stride + c] = acc;
  if (rounded != nullptr) rounded[(int64_t)row * rounded_stride + c] = from_f32<T>(acc);
}

// Every entry one row (a step of single tokens): the thread that reads a channel's kept inputs also moves them on.
template <typename T>
__global__ void causal_conv_single_kernel(const float* __restrict__ x, int64_t stride, const float* __restrict__ conv_w,
                                          const float* __restrict__ bias, float* kept_base, int64_t state_stride,
                                          const int* __restrict__ positions, const int* __restrict__ state_slots,
                                          float* __restrict__ out, int64_t out_stride, T* __restrict__ rounded,
                                          int64_t rounded_stride, int channels, int taps, int act,
                                          const float* __restrict__ in_bias) {
  const int row = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  float* kept = kept_base + (int64_t)state_slots[row] * state_stride + c;
  const int pos = positions[row];
  const float now = x[(int64_t)row * stride + c] + (in_bias != nullptr ? in_bias[c] : 0.f);
  float acc = bias != nullptr ? bias[c] : 0.f, old[GD_MAX_TAPS];
  for (int i = 0; i < taps - 1; ++i)                             // kept row i: the input taps - 1 - i places back
    old[i] = pos - (taps - 1 - i) >= 0 ? kept[(int64_t)i * channels] : 0.f;
  for (int i = 0; i < taps - 1; ++i) acc = fmaf(conv_w[(int64_t)c * taps + i], old[i], acc);   // oldest input first
  acc = fmaf(conv_w[(int64_t)c * taps + taps - 1], now, acc);
  for (int i = 0; i + 1 < taps - 1; ++i) kept[(int64_t)i * channels] = old[i + 1];
  if (taps > 1) kept[(int64_t)(taps - 2) * channels] = now;
  if (act == 1) acc = acc / (1.f + expf(-acc));
  if (out != nullptr) out[(int64_t)row * out_stride + c] = acc;
  if (rounded != nullptr) rounded[(int64_t)row * rounded_stride + c] = from_f32<T>(acc);
}

// The same as causal_conv, a thread RUN neighbouring rows of a channel: an input is read once for all rows it reaches where the run
// lies in one entry with its inputs among the step's rows; other runs take the rows one by one. TAPS at least `taps`.
template <typename T, int TAPS, int RUN>
__global__ __launch_bounds__(256) void causal_conv_run_kernel(const float* __restrict__ x, int64_t stride,
                                                              const float* __restrict__ conv_w, const float* __restrict__ bias,
                                                              const float* kept_base, int64_t state_stride,
                                                              const int* __restrict__ q_start, int entries,
                                                              const int* __restrict__ positions,
                                                              const int* __restrict__ state_slots, float* __restrict__ out,
                                                              int64_t out_stride, T* __restrict__ rounded, int64_t rounded_stride,
                                                              int rows, int channels, int taps, int act,
                                                              const float* __restrict__ in_bias) {
  const int row0 = blockIdx.x * RUN, c = blockIdx.y * 256 + threadIdx.x;
  if (c >= channels) return;
  const float ib = in_bias != nullptr ? in_bias[c] : 0.f, b = bias != nullptr ? bias[c] : 0.f;
  float w[TAPS];                                                // w[j]: the input j places back
#pragma unroll
  for (int j = 0; j < TAPS; ++j) w[j] = j < taps ? conv_w[(int64_t)c * taps + (taps - 1 - j)] : 0.f;
  const int e0 = gd_entry_of_row(q_start, entries, row0);
  const bool inside = row0 - (TAPS - 1) >= q_start[e0] && row0 + RUN <= q_start[e0 + 1];
  float y[RUN];
  if (inside) {                                                 // (the same for the whole workgroup)
    float in[RUN + TAPS - 1];
#pragma unroll
    for (int k = 0; k < RUN + TAPS - 1; ++k) in[k] = x[(int64_t)(row0 - (TAPS - 1) + k) * stride + c] + ib;
#pragma unroll
    for (int r = 0; r < RUN; ++r) {
      y[r] = b;
#pragma unroll
      for (int j = TAPS - 1; j >= 0; --j) y[r] = fmaf(w[j], in[r + TAPS - 1 - j], y[r]);   // oldest input first
    }
  } else {
    for (int r = 0; r < RUN; ++r) {
      const int row = row0 + r;
      float acc = b;
      if (row < rows) {
        const int e = gd_entry_of_row(q_start, entries, row);
        const int first = q_start[e], pos = positions[row];
        const float* kept = kept_base + (int64_t)state_slots[e] * state_stride;
#pragma unroll
        for (int j = TAPS - 1; j >= 0; --j)
          if (j < taps && pos - j >= 0) {
            const int src = row - j;
            acc = fmaf(w[j], src >= first ? x[(int64_t)src * stride + c] + ib : kept[(int64_t)(taps - 1 - (first - src)) * channels + c], acc);
          }
      }
#pragma unroll
      for (int q = 0; q < RUN; ++q) y[q] = q == r ? acc : y[q];
    }
  }
#pragma unroll
  for (int r = 0; r < RUN; ++r) {
    const int row = row0 + r;
    if (row >= rows) break;
    float v = y[r];
    if (act == 1) v = v / (1.f + expf(-v));
    if (out != nullptr) out[(int64_t)row * out_stride + c] = v;
    if (rounded != nullptr) rounded[(int64_t)row * rounded_stride + c] = from_f32<T>(v);
  }
}

struct GdArgs {
  const float* prep; int64_t stride;   // [rows][stride]: q | k | v | beta | g as conv_prepare leaves them
  float* state; int64_t state_stride;
  const int* q_start; const int* positions; const int* state_slots;
  float* o; int64_t o_stride;          // [rows][heads * V]
  int heads, kv_heads, vdim;
};

__device__ __forceinline__ float gd_row_sum(float x) {
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0xB1, 0xF, 0xF, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x4E, 0xF, 0xF, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x141, 0xF, 0xF, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x140, 0xF, 0xF, false));
  return x;
}

// NK keys a lane, D = 16 NK; TB tokens staged at once (1 in a step of single tokens).
template <int NK, int TB>
__global__ __launch_bounds__(64) void gated_delta_scan_kernel(GdArgs p) {
  constexpr int D = NK * 16, COLS = 4, PER = (TB * D + 63) / 64;
  __shared__ float sk[PER * 64], sq[PER * 64], sv[TB * COLS], sbg[TB * 2], skq[TB];
  const int lane = threadIdx.x, vloc = lane / 16, part = lane % 16;
  const int entry = blockIdx.x, head = blockIdx.y;
  const int V = p.vdim;
  const int col = min((int)blockIdx.z * COLS + vloc, V - 1);   // lanes past the last column repeat it and store nothing
  const bool live = (int)blockIdx.z * COLS + vloc < V;
  const int row0 = p.q_start[entry], n_rows = p.q_start[entry + 1] - row0;
  if (n_rows <= 0) return;
  const int kvh = head / (p.heads / p.kv_heads);
  const int qk = p.kv_heads * D;
  const int64_t q_col = (int64_t)kvh * D, k_col = qk + (int64_t)kvh * D, v_col = 2 * (int64_t)qk + (int64_t)head * V;
  const int64_t b_col = 2 * (int64_t)qk + (int64_t)p.heads * V + head, g_col = b_col + p.heads;
  float* st = p.state + (int64_t)p.state_slots[entry] * p.state_stride + ((int64_t)head * V + col) * D + part * NK;
  float s[NK];
  const bool fresh = p.positions[row0] == 0;
#pragma unroll
  for (int i = 0; i < NK; ++i) s[i] = fresh ? 0.f : st[i];

  float pk[PER], pq[PER], pv = 0.f, pbg = 0.f;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int m = 0; m < PER; ++m) {
      const int e = min(lane + 64 * m, TB * D - 1), t = e / D, c = e - t * D;
      const int64_t row = row0 + min(t0 + t, n_rows - 1);
      pk[m] = p.prep[row * p.stride + k_col + c];
      pq[m] = p.prep[row * p.stride + q_col + c];
    }
    if (lane < TB * COLS) {
      const int64_t row = row0 + min(t0 + lane / COLS, n_rows - 1);
      pv = p.prep[row * p.stride + v_col + min((int)blockIdx.z * COLS + lane % COLS, V - 1)];
    }
    if (lane < TB * 2) {
      const int64_t row = row0 + min(t0 + lane / 2, n_rows - 1);
      pbg = p.prep[row * p.stride + ((lane & 1) ? g_col : b_col)];
    }
  };
  auto step = [&](int t, int64_t row) {
    const float* kt = sk + t * D + part * NK;
    const float* qt = sq + t * D + part * NK;
    const float v = sv[t * COLS + vloc], beta = sbg[2 * t], g = sbg[2 * t + 1], kq = skq[t];
    float ks0 = 0.f, ks1 = 0.f, qs0 = 0.f, qs1 = 0.f;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      if (i & 1) { ks1 = fmaf(kt[i], s[i], ks1); qs1 = fmaf(qt[i], s[i], qs1); }
      else { ks0 = fmaf(kt[i], s[i], ks0); qs0 = fmaf(qt[i], s[i], qs0); }
    }
    const float ks = gd_row_sum(ks0 + ks1), qs = gd_row_sum(qs0 + qs1);
    const float u = beta * (v - g * ks);
#pragma unroll
    for (int i = 0; i < NK; ++i) s[i] = fmaf(kt[i], u, g * s[i]);
    if (part == 0 && live) p.o[row * p.o_stride + (int64_t)head * V + col] = fmaf(u, kq, g * qs);
  };
  fetch(0);
  for (int t0 = 0; t0 < n_rows; t0 += TB) {
#pragma unroll
    for (int m = 0; m < PER; ++m) {
      sk[lane + 64 * m] = pk[m];
      sq[lane + 64 * m] = pq[m];
    }
    if (lane < TB * COLS) sv[lane] = pv;
    if (lane < TB * 2) sbg[lane] = pbg;
    if (TB > 1 && t0 + TB < n_rows) fetch(t0 + TB);  // on their way while the chain below runs
    __syncthreads();
    // each token's k . q: four lanes a token add up a quarter of the keys each
    for (int t = lane >> 2; t < TB; t += 16) {
      float kq = 0.f;
      for (int c = (lane & 3) * (D / 4); c < ((lane & 3) + 1) * (D / 4); ++c) kq = fmaf(sk[t * D + c], sq[t * D + c], kq);
      kq = quad_sum(kq);
      if ((lane & 3) == 0) skq[t] = kq;
    }
    __syncthreads();
    const int nb = min(TB, n_rows - t0);
    if (nb == TB) {
#pragma unroll
      for (int t = 0; t < TB; ++t) step(t, row0 + t0 + t);
    } else {
      for (int t = 0; t < nb; ++t) step(t, row0 + t0 + t);
    }
    __syncthreads();  // the chain has read this batch before the next one is written
  }
  if (live)
#pragma unroll
    for (int i = 0; i < NK; ++i) st[i] = s[i];
}

// A step of single tokens in one kernel: convolution, recurrence, and each head's norm and gate (as conv_prepare, gated_delta_scan and
// head_norm_gate make them, sums in their order: the same bits). Apart they are three launches whose waves each wait for two or three
// trips to memory and hand a few kilobytes on: 4.9 + 5.0 + 4.6 us of a step of four requests (32 heads of 64 on 8), 5.9 to 6.4 together (both traced in a step).
//
// A workgroup takes a (request, q/k head) with all the value heads that share it, since the q and k channels' kept inputs are moved
// on by whoever has read them. Its sixteen waves are units first (q, k, then runs of 64 channels of v, the last one the gates), then
// each holds four value columns a turn as gated_delta_scan_kernel does, IT turns; all of a wave's state is asked for together, behind
// the convolution's inputs. Last a wave a value head.
struct GdSingleArgs {
  PrepArgs p;
  float* state;
  int g_off;                            // columns of the gate's pre-activations in proj
  const float* norm_w; float eps;       // [heads * vdim]
  void* out; int64_t out_stride;
};
#define GD_SINGLE_WAVES 16
#define GD_SINGLE_TAPS 4

template <typename T, int NK, int IT>
__global__ __launch_bounds__(64 * GD_SINGLE_WAVES) void gated_delta_single_kernel(GdSingleArgs a) {
  constexpr int D = NK * 16, COLS = 4 * GD_SINGLE_WAVES, CH = (D + 63) / 64;   // COLS: value columns a turn
  __shared__ float sq[D], sk[D], sv[IT * COLS], so[IT * COLS], sbg[2 * GD_SINGLE_WAVES];
  const PrepArgs& p = a.p;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), vloc = lane / 16, part = lane % 16;
  const int row = blockIdx.x, kvh = blockIdx.y, group = p.heads / p.kv_heads, V = p.vdim, cols = group * V;
  const int qk = p.kv_heads * D, channels = 2 * qk + p.heads * V;
  const int slot = p.state_slots[row], pos = p.positions[row];
  const float* proj = p.proj + (int64_t)row * p.stride;
  float* kept = p.keep + (int64_t)slot * p.state_stride;

  // the convolution's inputs (channels past the unit's last: the last again), oldest tap first
  const bool is_qk = wave < 2, is_v = !is_qk && (wave - 2) * 64 < cols;
  const int c_first = wave == 0 ? kvh * D : wave == 1 ? qk + kvh * D : 2 * qk + kvh * cols + (wave - 2) * 64;
  const int c_count = is_qk ? D : min(cols - (wave - 2) * 64, 64);
  float in[CH][GD_SINGLE_TAPS], wt[CH][GD_SINGLE_TAPS];
  if (is_qk || is_v) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = c_first + min(lane + 64 * i, c_count - 1);
#pragma unroll
      for (int k = 0; k < GD_SINGLE_TAPS; ++k) {
        const int t = min(k, p.taps - 1), back = min(p.taps - 1 - t, pos);
        in[i][k] = *(back == 0 ? proj + c : kept + (int64_t)(p.taps - 1 - back) * channels + c);
        wt[i][k] = p.conv_w[(int64_t)c * p.taps + t];
      }
    }
  }
  // this wave's part of the state, and the gate and weight of its value head
  float s[IT][NK];
  float* st[IT];
#pragma unroll
  for (int it = 0; it < IT; ++it) {   // (columns past the last repeat it and store nothing)
    const int col = min(it * COLS + wave * 4 + vloc, cols - 1);
    st[it] = a.state + (int64_t)slot * p.state_stride + ((int64_t)kvh * cols + col) * D + part * NK;
#pragma unroll
    for (int i = 0; i < NK; ++i) s[it][i] = st[it][i];
  }
  const int64_t head_at = ((int64_t)kvh * group + min(wave, group - 1)) * V;
  float gate[2], weight[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = min(lane + 64 * i, V - 1);
    gate[i] = proj[a.g_off + head_at + c];
    weight[i] = a.norm_w[head_at + c];
  }
  __builtin_amdgcn_sched_barrier(0);
  if (is_qk || is_v) {
    float y[CH], ss = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = lane + 64 * i;
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < GD_SINGLE_TAPS; ++k) {
        const float x = p.taps - 1 - k <= pos ? in[i][k] : 0.f;
        if (k < p.taps) acc = fmaf(wt[i][k], x, acc);
        if (k >= 1 && k < p.taps && c < c_count) kept[(int64_t)(k - 1) * channels + c_first + c] = x;
      }
      y[i] = acc / (1.f + expf(-acc));
      if (c < c_count) ss += y[i] * y[i];
    }
    const float r = is_qk ? conv_unit_scale(p, wave == 0 ? 0 : p.kv_heads, ss) : 1.f;
    float* to = wave == 0 ? sq : wave == 1 ? sk : sv + (wave - 2) * 64;
#pragma unroll
    for (int i = 0; i < CH; ++i)
      if (lane + 64 * i < c_count) to[lane + 64 * i] = is_qk ? y[i] * r : y[i];
  } else if (wave == GD_SINGLE_WAVES - 1 && lane < group) {
    const int h = kvh * group + lane;
    conv_prepare_gates(proj[p.b_off + h], proj[p.a_off + h], p.a_log[h], p.dt_bias[h], sbg[2 * lane], sbg[2 * lane + 1]);
  }
  __syncthreads();
  float kq = 0.f;
  for (int c = (lane & 3) * (D / 4); c < ((lane & 3) + 1) * (D / 4); ++c) kq = fmaf(sk[c], sq[c], kq);
  kq = quad_sum(kq);
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int col = min(it * COLS + wave * 4 + vloc, cols - 1), h = col / V;
    const float *kt = sk + part * NK, *qt = sq + part * NK;
    const float v = sv[col], beta = sbg[2 * h], g = sbg[2 * h + 1];
    if (pos == 0)
#pragma unroll
      for (int i = 0; i < NK; ++i) s[it][i] = 0.f;
    float ks0 = 0.f, ks1 = 0.f, qs0 = 0.f, qs1 = 0.f;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      if (i & 1) { ks1 = fmaf(kt[i], s[it][i], ks1); qs1 = fmaf(qt[i], s[it][i], qs1); }
      else { ks0 = fmaf(kt[i], s[it][i], ks0); qs0 = fmaf(qt[i], s[it][i], qs0); }
    }
    const float ks = gd_row_sum(ks0 + ks1), qs = gd_row_sum(qs0 + qs1);
    const float u = beta * (v - g * ks);
    if (it * COLS + wave * 4 + vloc < cols) {
#pragma unroll
      for (int i = 0; i < NK; ++i) st[it][i] = fmaf(kt[i], u, g * s[it][i]);
      if (part == 0) so[col] = fmaf(u, kq, g * qs);
    }
  }
  __syncthreads();
  if (wave >= group) return;
  float v[2], ss = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    v[i] = so[wave * V + min(lane + 64 * i, V - 1)];
    if (lane + 64 * i < V) ss += v[i] * v[i];
  }
  const float r = 1.f / sqrtf(wave_sum(ss) / (float)V + a.eps);
  T* out = reinterpret_cast<T*>(a.out) + (int64_t)row * a.out_stride + head_at;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (lane + 64 * i < V) out[lane + 64 * i] = from_f32<T>(v[i] * r * weight[i] * (gate[i] / (1.f + expf(-gate[i]))));
}

// Sizes that a workgroup holds: heads of q and k of 16 to 128, a wave's state in 32 registers a lane, a wave for every unit.
static bool gated_delta_single_takes(int heads, int kv_heads, int dim, int vdim, int taps) {
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || vdim <= 0 || vdim > 128 || taps < 1 || taps > GD_SINGLE_TAPS) return false;
  if (dim != 16 && dim != 32 && dim != 64 && dim != 128) return false;
  const int64_t group = heads / kv_heads, cols = group * vdim;
  return kv_heads <= 65535 && group <= GD_SINGLE_WAVES && cols <= 64 * 8 && cols * dim <= 64 * 512;
}

// Any D and V: a thread a value column, the column's state in the request's slot.
__global__ void gated_delta_any_kernel(GdArgs p, int D) {
  extern __shared__ float sh[];
  float *sk = sh, *sq = sh + D;
  const int v = blockIdx.z * blockDim.x + threadIdx.x, V = p.vdim;
  const bool live = v < V;
  const int entry = blockIdx.x, head = blockIdx.y;
  const int row0 = p.q_start[entry], n_rows = p.q_start[entry + 1] - row0;
  if (n_rows <= 0) return;
  const int kvh = head / (p.heads / p.kv_heads);
  const int qk = p.kv_heads * D;
  const int64_t q_col = (int64_t)kvh * D, k_col = qk + (int64_t)kvh * D, v_col = 2 * (int64_t)qk + (int64_t)head * V;
  const int64_t b_col = 2 * (int64_t)qk + (int64_t)p.heads * V + head, g_col = b_col + p.heads;
  float* st = p.state + (int64_t)p.state_slots[entry] * p.state_stride + ((int64_t)head * V + (live ? v : 0)) * D;
  if (live && p.positions[row0] == 0)
    for (int c = 0; c < D; ++c) st[c] = 0.f;
  for (int t = 0; t < n_rows; ++t) {
    const int64_t row = row0 + t;
    __syncthreads();
    for (int c = threadIdx.x; c < D; c += blockDim.x) {
      sk[c] = p.prep[row * p.stride + k_col + c];
      sq[c] = p.prep[row * p.stride + q_col + c];
    }
    __syncthreads();
    if (!live) continue;
    const float beta = p.prep[row * p.stride + b_col], g = p.prep[row * p.stride + g_col];
    const float vv = p.prep[row * p.stride + v_col + v];
    float ks = 0.f, qs = 0.f, kq = 0.f;
    for (int c = 0; c < D; ++c) {
      ks = fmaf(sk[c], st[c], ks);
      qs = fmaf(sq[c], st[c], qs);
      kq = fmaf(sk[c], sq[c], kq);
    }
    const float u = beta * (vv - g * ks);
    for (int c = 0; c < D; ++c) st[c] = fmaf(sk[c], u, g * st[c]);
    p.o[row * p.o_stride + (int64_t)head * V + v] = fmaf(u, kq, g * qs);
  }
}

extern "C" {

int dli_gated_delta_max_taps() { return GD_MAX_TAPS; }

// Whether a step's rows are convolved PREP_RUN at a time.
int dli_conv_prepare_in_runs(int rows, int entries, int heads, int kv_heads, int dim, int vdim, int taps) {
  return rows > 0 && entries > 0 && conv_prepare_in_runs(rows, entries, 2 * kv_heads + (int)(((int64_t)heads * vdim + 63) / 64) + 1, dim, taps);
}

int dli_conv_prepare(const float* proj, int64_t stride, int b_off, int a_off, const float* conv_w, const float* a_log,
                     const float* dt_bias, float* state, int64_t state_stride, int64_t kept_offset, const int* q_start,
                     const int* positions, const int* state_slots, float* out, int64_t out_stride, int entries, int rows,
                     int heads, int kv_heads, int dim, int vdim, int taps, int singles, hipStream_t stream) {
  if (rows <= 0 || entries <= 0) return DLI_OK;
  if (singles && rows != entries) return DLI_ERR_ARGUMENT;
  const int64_t channels = 2 * (int64_t)kv_heads * dim + (int64_t)heads * vdim;
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || vdim <= 0 || taps < 1 || taps > GD_MAX_TAPS ||
      stride < channels || out_stride < channels + 2 * heads || b_off < channels || a_off < channels ||
      b_off + heads > stride || a_off + heads > stride || state_stride < kept_offset + (taps - 1) * channels)
    return DLI_ERR_ARGUMENT;
  PrepArgs p;
  p.proj = proj; p.stride = stride; p.b_off = b_off; p.a_off = a_off; p.conv_w = conv_w; p.a_log = a_log;
  p.dt_bias = dt_bias; p.kept = state + kept_offset; p.keep = singles ? state + kept_offset : nullptr; p.state_stride = state_stride; p.q_start = q_start;
  p.positions = positions; p.state_slots = state_slots; p.out = out; p.out_stride = out_stride; p.entries = entries;
  p.heads = heads; p.kv_heads = kv_heads; p.dim = dim; p.vdim = vdim; p.taps = taps;
  const int units = 2 * kv_heads + (int)(((int64_t)heads * vdim + 63) / 64) + 1;
  if (units > 65535) return DLI_ERR_ARGUMENT;
  if (conv_prepare_in_runs(rows, entries, units, dim, taps))
    conv_prepare_run_kernel<<<dim3((rows + PREP_RUN - 1) / PREP_RUN, units), 64, 0, stream>>>(p, rows);
  else if (taps == 3)   // (numbers that four does not divide: known ones are asked for together)
    conv_prepare_kernel<3><<<dim3(rows, units), 64, 0, stream>>>(p);
  else if (taps == 2)
    conv_prepare_kernel<2><<<dim3(rows, units), 64, 0, stream>>>(p);
  else
    conv_prepare_kernel<0><<<dim3(rows, units), 64, 0, stream>>>(p);
  if (dli_launch_status() != DLI_OK) return DLI_ERR_LAUNCH;
  if (taps > 1 && !singles) {
    const dim3 grid(entries, (unsigned)((channels + 255) / 256));
    conv_keep_kernel<<<grid, 256, 0, stream>>>(proj, stride, state + kept_offset, state_stride, q_start, positions,
                                               state_slots, (int)channels, taps, nullptr);
  }
  return dli_launch_status();
}

// act: 0 none, 1 silu. rounded (may be nullptr): the result once more, bf16 if rounded_is_bf16 else float; out may be nullptr
// where it is not.
int dli_causal_conv(const float* x, int64_t stride, const float* conv_w, const float* bias, const float* in_bias, float* state,
                    int64_t state_stride, int64_t kept_offset, const int* q_start, const int* positions,
                    const int* state_slots, float* out, int64_t out_stride, void* rounded, int64_t rounded_stride,
                    int rounded_is_bf16, int entries, int rows, int channels, int taps, int act, hipStream_t stream) {
  if (rows <= 0 || entries <= 0) return DLI_OK;
  if (channels <= 0 || taps < 1 || taps > GD_MAX_TAPS || stride < channels || (out != nullptr ? out_stride < channels : rounded == nullptr) ||
      (rounded != nullptr && rounded_stride < channels) || act < 0 || act > 1 ||
      state_stride < kept_offset + (int64_t)(taps - 1) * channels)
    return DLI_ERR_ARGUMENT;
  const dim3 grid(rows, (channels + 255) / 256);
  if (grid.y > 65535) return DLI_ERR_ARGUMENT;
  if (rows == entries) {
#define CONV_SINGLE(T)                                                                                                 \
  causal_conv_single_kernel<T><<<grid, 256, 0, stream>>>(x, stride, conv_w, bias, state + kept_offset, state_stride,   \
                                                         positions, state_slots, out, out_stride, (T*)rounded,         \
                                                         rounded_stride, channels, taps, act, in_bias)
    if (rounded_is_bf16) CONV_SINGLE(bf16_t);
    else CONV_SINGLE(float);
#undef CONV_SINGLE
    return dli_launch_status();
  }
#define CONV_RUN(T, TAPS)                                                                                              \
  causal_conv_run_kernel<T, TAPS, 8><<<dim3((rows + 7) / 8, grid.y), 256, 0, stream>>>(                                \
      x, stride, conv_w, bias, state + kept_offset, state_stride, q_start, entries, positions, state_slots, out,      \
      out_stride, (T*)rounded, rounded_stride, rows, channels, taps, act, in_bias)
  if (taps <= 4 && rows >= 8 * entries && rows >= 256) {       // portions: runs of rows
    if (rounded_is_bf16) CONV_RUN(bf16_t, 4);
    else CONV_RUN(float, 4);
  } else
#undef CONV_RUN
  if (rounded_is_bf16)
    causal_conv_kernel<bf16_t><<<grid, 256, 0, stream>>>(x, stride, conv_w, bias, state + kept_offset, state_stride, q_start,
                                                         entries, positions, state_slots, out, out_stride, (bf16_t*)rounded,
                                                         rounded_stride, channels, taps, act, in_bias);
  else
    causal_conv_kernel<float><<<grid, 256, 0, stream>>>(x, stride, conv_w, bias, state + kept_offset, state_stride, q_start,
                                                        entries, positions, state_slots, out, out_stride, (float*)rounded,
                                                        rounded_stride, channels, taps, act, in_bias);
  if (dli_launch_status() != DLI_OK) return DLI_ERR_LAUNCH;
  if (taps > 1) {
    const dim3 keep(entries, (channels + 255) / 256);
    conv_keep_kernel<<<keep, 256, 0, stream>>>(x, stride, state + kept_offset, state_stride, q_start, positions,
                                               state_slots, channels, taps, in_bias);
  }
  return dli_launch_status();
}

int dli_gated_delta_single_takes(int heads, int kv_heads, int dim, int vdim, int taps) {
  return gated_delta_single_takes(heads, kv_heads, dim, vdim, taps);
}

// A step of single tokens, a row a request: everything between the projections and the output product. g_off: the first
// column of the gate's pre-activations (heads * vdim of them).
int dli_gated_delta_single(const float* proj, int64_t stride, int b_off, int a_off, int g_off, const float* conv_w, const float* a_log,
                           const float* dt_bias, float* state, int64_t state_stride, int64_t kept_offset, const int* positions,
                           const int* state_slots, const float* norm_w, float eps, void* out, int64_t out_stride, int entries, int heads,
                           int kv_heads, int dim, int vdim, int taps, int is_bf16, hipStream_t stream) {
  if (entries <= 0) return DLI_OK;
  if (!gated_delta_single_takes(heads, kv_heads, dim, vdim, taps)) return DLI_ERR_ARGUMENT;
  const int64_t hv = (int64_t)heads * vdim, channels = 2 * (int64_t)kv_heads * dim + hv;
  if (b_off < channels || a_off < channels || g_off < channels || b_off + heads > stride || a_off + heads > stride || g_off + hv > stride ||
      out_stride < hv || kept_offset < hv * dim || state_stride < kept_offset + (taps - 1) * channels)
    return DLI_ERR_ARGUMENT;
  GdSingleArgs a = {};
  a.p.proj = proj; a.p.stride = stride; a.p.b_off = b_off; a.p.a_off = a_off; a.p.conv_w = conv_w; a.p.a_log = a_log; a.p.dt_bias = dt_bias;
  a.p.keep = state + kept_offset; a.p.state_stride = state_stride; a.p.positions = positions; a.p.state_slots = state_slots;
  a.p.entries = entries; a.p.heads = heads; a.p.kv_heads = kv_heads; a.p.dim = dim; a.p.vdim = vdim; a.p.taps = taps;
  a.state = state; a.g_off = g_off; a.norm_w = norm_w; a.eps = eps; a.out = out; a.out_stride = out_stride;
  const int64_t cols = (int64_t)heads / kv_heads * vdim;
  const dim3 grid(entries, kv_heads);
  const auto launch = [&](auto nk, auto it) {
    constexpr int NK = decltype(nk)::value, IT = decltype(it)::value;
    if (is_bf16) gated_delta_single_kernel<bf16_t, NK, IT><<<grid, 64 * GD_SINGLE_WAVES, 0, stream>>>(a);
    else gated_delta_single_kernel<float, NK, IT><<<grid, 64 * GD_SINGLE_WAVES, 0, stream>>>(a);
  };
  const auto turns = [&](auto nk) {
    constexpr int NK = decltype(nk)::value;
    if (cols <= 64) launch(nk, std::integral_constant<int, 1>());
    else if (cols <= 128) launch(nk, std::integral_constant<int, 2>());
    else if (cols <= 256) launch(nk, std::integral_constant<int, 4>());
    else if constexpr (NK <= 4) launch(nk, std::integral_constant<int, 8>());
  };
  switch (dim) {
    case 16: turns(std::integral_constant<int, 1>()); break;
    case 32: turns(std::integral_constant<int, 2>()); break;
    case 64: turns(std::integral_constant<int, 4>()); break;
    default: turns(std::integral_constant<int, 8>());
  }
  return dli_launch_status();
}

int dli_gated_delta_scan(const float* prep, int64_t stride, float* state, int64_t state_stride, const int* q_start,
                         const int* positions, const int* state_slots, float* o, int64_t o_stride, int entries, int rows,
                         int heads, int kv_heads, int dim, int vdim, int singles, int run_rows, int runs, float* y, float* ends,
                         float* moves, hipStream_t stream) {
  if (rows <= 0 || entries <= 0) return DLI_OK;
  if (rows < entries || heads <= 0 || heads > 65535 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || dim > 4096 ||
      vdim <= 0 || state_stride < (int64_t)heads * vdim * dim || o_stride < (int64_t)heads * vdim ||
      stride < 2 * (int64_t)kv_heads * dim + (int64_t)heads * vdim + 2 * heads)
    return DLI_ERR_ARGUMENT;
  GdArgs p;
  p.prep = prep; p.stride = stride; p.state = state; p.state_stride = state_stride; p.q_start = q_start;
  p.positions = positions; p.state_slots = state_slots; p.o = o; p.o_stride = o_stride; p.heads = heads;
  p.kv_heads = kv_heads; p.vdim = vdim;
  if (run_rows > 0) {
    // the rows of the entries behind the first `singles`, which bring one row each and keep the kernel of steps of single
    // tokens, in runs that are walked side by side (the caller's choice and scratch)
    if (dim != 64 || vdim != 64 || singles < 0 || singles >= entries) return DLI_ERR_ARGUMENT;
    const int64_t qk = (int64_t)kv_heads * dim;
    const RunsArgs q = {prep, prep + qk, prep + 2 * qk, prep + 2 * qk + (int64_t)heads * vdim, nullptr, nullptr, nullptr, nullptr,
                        stride, stride, stride, stride, 0, 0, 0.f, state, state_stride, q_start + singles, positions,
                        state_slots + singles, o, o_stride, nullptr, 0, y, ends, moves, heads, heads / kv_heads, run_rows, runs,
                        entries - singles, rows - singles, singles};
    if (!scan_runs_takes(q, RUNS_GATED, RUNS_FINISH_SUM, 0)) return DLI_ERR_ARGUMENT;
    if (singles > 0) gated_delta_scan_kernel<4, 1><<<dim3(singles, heads, vdim / 4), 64, 0, stream>>>(p);
    return scan_runs(q, RUNS_GATED, RUNS_FINISH_SUM, 0, stream);
  }
  const bool single = rows == entries;
  const dim3 grid(entries, heads, (vdim + 3) / 4);
#define GD_CASE(NK, TBM)                                                                     \
  case NK * 16:                                                                              \
    if (single) gated_delta_scan_kernel<NK, 1><<<grid, 64, 0, stream>>>(p);                  \
    else gated_delta_scan_kernel<NK, TBM><<<grid, 64, 0, stream>>>(p);                       \
    break;
  switch (dim) {
    GD_CASE(1, 16) GD_CASE(2, 16) GD_CASE(3, 16) GD_CASE(4, 16) GD_CASE(5, 8) GD_CASE(6, 8) GD_CASE(7, 8) GD_CASE(8, 8)
    GD_CASE(12, 4) GD_CASE(16, 4)
    default: {
      const int threads = vdim >= 256 ? 256 : (vdim + 63) / 64 * 64;
      gated_delta_any_kernel<<<dim3(entries, heads, (vdim + threads - 1) / threads), threads, 2 * dim * sizeof(float),
                               stream>>>(p, dim);
    }
  }
#undef GD_CASE
  return dli_launch_status();
}

}  // extern "C"
