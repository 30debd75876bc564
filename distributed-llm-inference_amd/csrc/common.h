// Shared device helpers for the gfx950 kernels: element types, conversions and reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16_t;

#define DLI_WAVE 64

// What a launch reads once and no other workgroup or launch soon again, the weights of a decode step's products above all: they leave
// the level-2 cache first, so that what the kernels behind them read again stays there (their code and arguments, a small request's
// keys and values, activations). Bits do not depend on it. A step of the requests and seven more, all weights so, ms before and after:
// 135M sizes, one request, 5.03 4.77; 1B sizes, one 5.82 5.55, eight 7.73 7.64, 64 18.67 18.01 (gate and up of 64 rows 25.6 -> 22.5 us).
// Only where a load's lanes take whole lines: a line whose parts several loads ask for does not outlive the first of them. Keys and
// values so: 8 requests 1.4% less, one 1.3 to 3.2% more, 64 0.5% more, so they are read as before; 32-bit weights: no difference.
// Experts' weights so, though an expert's further tiles of rows read them again: prompts of Betepel with eight decode steps 1 to 5% less
// (1 to 16 requests). Eight of 1B's requests are within what two runs differ by; a model whose weights are little more than the level-2
// caches hold loses: 8 layers 512 wide (50 MB), 2 requests 1.44 -> 1.47, 8 1.46 -> 1.52, 40 the same.
template <typename V>
__device__ __forceinline__ V load_streamed(const V* p) { return __builtin_nontemporal_load(p); }
constexpr int STREAMED = 1 << 1;   // the same as the cache policy of a buffer load

// Status codes returned by every extern "C" entry point.
#define DLI_OK 0
#define DLI_ERR_ARGUMENT -1   // sizes that the kernel does not take
#define DLI_ERR_LAUNCH -2     // the runtime refused the launch

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(bf16_t x) { return (float)x; }

template <typename T> __device__ __forceinline__ T from_f32(float x);
template <> __device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float x) { return (bf16_t)x; }

// Round through the storage type: what a value becomes when it is written as T and read back.
template <typename T> __device__ __forceinline__ float round_to(float x) { return to_f32(from_f32<T>(x)); }

// silu(g) = g * sigmoid(g) in 32-bit (reference: src/dli/model/llama.py:190). Faster forms of the
// exponential and the division were tried for bfloat16 and changed no timing: the kernels that
// use it wait for memory.
template <typename T> __device__ __forceinline__ float silu(float g) { return g / (1.f + expf(-g)); }

// The gated activation of a feed-forward's two halves: g sigmoid(alpha g) (u + shift) with g = min(gate, limit),
// u = clamp(up, -limit, limit). An infinite limit, alpha 1 and shift 0: silu(gate) * up.
__device__ __forceinline__ float clamped_glu(float gate, float up, float limit, float alpha, float up_shift) {
  const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
  return g / (1.f + expf(-alpha * g)) * (u + up_shift);
}

// gelu(gate) * up in its tanh form, 0.5 z (1 + tanh t) = z sigmoid(2 t), t = sqrt(2 / pi) (z + 0.044715 z^3).
__device__ __forceinline__ float gelu_glu(float z, float up) {
  const float t2 = 1.5957691216057308f * (z + 0.044715f * z * z * z);
  return z / (1.f + expf(-t2)) * up;
}

// The activation inside a few-row product: `form` 0 is cast(silu(gate)) * up, 1 the clamped form, 2 gelu(gate) * up.
#define GLU_SILU 0
#define GLU_CLAMPED 1
#define GLU_GELU 2
struct GluForm { int form; float limit, alpha, up_shift; };
__device__ __forceinline__ bf16_t glu_bf16(float gate, float up, const GluForm& f) {
  if (f.form == GLU_CLAMPED) return (bf16_t)clamped_glu(gate, up, f.limit, f.alpha, f.up_shift);
  if (f.form == GLU_GELU) return (bf16_t)gelu_glu(gate, up);
  return (bf16_t)((float)(bf16_t)silu<bf16_t>(gate) * up);
}

// Exchanges between lanes without a trip through LDS (all lanes of the wave take part).
template <int SHIFT>
__device__ __forceinline__ float row_ror(float v) {  // rotated by SHIFT within each row of sixteen lanes
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + SHIFT, 0xf, 0xf, true));
}
template <int SHIFT>
__device__ __forceinline__ float row_shl(float v) {  // the value SHIFT lanes further on in the row of sixteen, 0 past its end
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + SHIFT, 0xf, 0xf, true));
}
__device__ __forceinline__ float quad_sum(float v) {  // over the lanes l, l^1, l^2, l^3
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xb1, 0xf, 0xf, true));
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4e, 0xf, 0xf, true));
}
__device__ __forceinline__ float quad_pairs(float v) {  // over the lanes l, l^2
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4e, 0xf, 0xf, true));
}
// a[l] + a[l^32] in the lower half of the lanes, b[l] + b[l^32] in the upper
__device__ __forceinline__ float add_halves(float a, float b) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
// a[l] + a[l^16] in the rows of sixteen lanes 0 and 2, b[l] + b[l^16] in the rows 1 and 3
__device__ __forceinline__ float add_rows(float a, float b) {
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// v[l] + v[l^32] and v[l] + v[l^16] in every lane, and the larger of the two
__device__ __forceinline__ float add_across32(float v) { return add_halves(v, v); }
__device__ __forceinline__ float add_across16(float v) { return add_rows(v, v); }
__device__ __forceinline__ float max_across32(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ __forceinline__ float max_across16(float v) {
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
template <int MASK>
__device__ __forceinline__ float quad_xor(float v) {  // the value of lane l ^ MASK, MASK 1 or 2
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), MASK == 1 ? 0xb1 : 0x4e, 0xf, 0xf, true));
}

// Sum and maximum over the wave, the same in every lane, by exchanges with the lanes l ^ 32, 16, 8, 4, 2, 1 in this order (once the
// first three are done a value repeats every eight lanes, and a rotation by four is the exchange with l ^ 4). All in registers: six
// exchanges through LDS, one after the other, take 0.3 us.
__device__ __forceinline__ float wave_sum(float v) {
  v = add_across16(add_across32(v));
  v += row_ror<8>(v);
  v += row_ror<4>(v);
  v += quad_xor<2>(v);
  return v + quad_xor<1>(v);
}
__device__ __forceinline__ float wave_max(float v) {
  v = max_across16(max_across32(v));
  v = fmaxf(v, row_ror<8>(v));
  v = fmaxf(v, row_ror<4>(v));
  v = fmaxf(v, quad_xor<2>(v));
  return fmaxf(v, quad_xor<1>(v));
}

// Sum over a block of up to 1024 threads; every thread gets the result. `scratch` holds 16 floats.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x % DLI_WAVE, wave = threadIdx.x / DLI_WAVE;
  const int nwaves = (blockDim.x + DLI_WAVE - 1) / DLI_WAVE;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int i = 0; i < nwaves; ++i) total += scratch[i];  // same order in every thread
  return total;
}

// A component of a rotated pair: `own` turned by the angle's cosine and sine, the sine with the pair's sign (negative for the first
// component). The one product is rounded, the other goes into the sum unrounded, written out so that every kernel that
// rotates 32-bit values gives the same bits: a request's keys do not depend on which of them a step takes.
__device__ __forceinline__ float rotated(float own, float other, float cosine, float signed_sine) {
  return fmaf(own, cosine, other * signed_sine);
}

// Page of a tile of sixteen keys, page size in tiles. A quotient by a number that the compiler does not know costs some
// twenty instructions, eight cycles each where one waits for the other, and an attention kernel's waves need several of them
// before their first keys are asked for: so the host hands over 2^32 / tiles, rounded up, whose product's upper
// half is the quotient for every tile below 2^32 / tiles.
struct PageOf {
  unsigned tiles, reciprocal;
  // (pages of one tile: reciprocal 0 and the tile itself; no branch, which would part the loads that wait for their pages)
  __device__ __forceinline__ unsigned page(unsigned tile) const { return __umulhi(tile, reciprocal) + (tiles == 1 ? tile : 0u); }
};
static inline PageOf page_of_tile(int page_size) {
  const unsigned tiles = (unsigned)page_size / 16;
  return PageOf{tiles, tiles > 1 ? (unsigned)((0x100000000ull + tiles - 1) / tiles) : 0u};
}

static inline int dli_launch_status() {
  return hipGetLastError() == hipSuccess ? DLI_OK : DLI_ERR_LAUNCH;
}

// Compute units of the current device (256 if the runtime does not say), asked once per device.
static inline int dli_compute_units() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}
