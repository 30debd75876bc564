// bfloat16 products of many rows whose result is about one tile of 128 x 128 for every compute unit:
//   out[r][f] = sum_k x[r][k] * w[f][k] (+ bias[f]),  32-bit accumulation, bfloat16 result or the 32-bit sums themselves.
// Other products of many rows go to the vendor library (gemm_lt.hip), which is ahead where tiles of 256 x 256 fill the chip: they
// need half the bytes a product. Where there are too few of those, the library's smaller tiles leave matrix cores waiting for
// their loads, which it asks for in bunches: a compute unit takes a load of 1 KB into LDS in about 32 cycles, and a wave that
// has asked for eight in a row issues no product meanwhile.
//
// Four waves of 64 x 64, one on each SIMD, blocks of 64 k, four stages of 32 KB that loads write without passing registers. A
// wave's instructions are written in the order in which they are to leave: between two products a read of a fragment for the
// next half block or a load for the stage after the next two, never more. The barrier of a block stands in its middle, when
// the products of its second half have their fragments already. What is left of the time is the way into LDS, 30 bytes a cycle and
// unit, however many stages (five: 3% less); to start
// each column of tiles at a k of its own changes nothing.
//
// Bank conflicts: the sixteen-byte chunks of a row lie at chunk ^ (row & 7) (w: at chunk ^ the same function of the lane that
// reads the row), which the loads' own addresses arrange. Which features a product takes is free: rows 4 g + i of the products
// 2 j and 2 j + 1 are the features 32 j + 8 g + 4 (0, 1) + i, so that a lane ends with eight consecutive features of a row.
#include "common.h"
#include "tile_gemm.h"

#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int TILE = 128, WT = 64, STAGES = 4, STAGE = 2 * TILE * 128;   // a workgroup's and a wave's tile, bytes of a stage
constexpr int LOADS = 8, HALF = LOADS / 2;                                // a wave's loads of 1 KB for a stage
constexpr int FRAGS = WT / 16, READS = 2 * FRAGS, PRODUCTS = FRAGS * FRAGS;

__device__ __forceinline__ float4v mfma32(bf16x8 a, bf16x8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// (the host's pass over the source does not know this builtin, and would drop every kernel that names it)
__device__ __forceinline__ void load16_to_lds(__amdgpu_buffer_rsrc_t from, void* to, unsigned at, int base) {
#ifdef __HIP_DEVICE_COMPILE__
  __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (__attribute__((address_space(3))) void*)to, 16, at, base, 0, 0);
#endif
}
// waits until at most N of the wave's vector memory loads are outstanding (nothing else awaited)
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// without the fence of __syncthreads(), which would wait for the later stages' loads as well
__device__ __forceinline__ void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

struct TileArgs {
  const bf16_t* x;
  const bf16_t* w;
  const bf16_t* bias;
  void* out;
  int64_t ldo;
  int ldx, ldw, rows, feats, k, tiles_r, tiles_f;
};

template <bool OUT_F32>
__global__ __launch_bounds__(256, 1) void tile_gemm_kernel(TileArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int c = lane % 16, g = lane / 16, wr = wave / 2, wf = wave % 2;
  // The eight XCDs take workgroups in turn; each gets a run of neighbouring tiles, eight tiles of rows deep, which share rows
  // and weights in its level-2 cache.
  const int tiles = p.tiles_r * p.tiles_f, xcd = blockIdx.x % 8;
  const int at = xcd * (tiles / 8) + min(xcd, tiles % 8) + blockIdx.x / 8;
  const int band = at / (8 * p.tiles_f), in_band = at - band * 8 * p.tiles_f, deep = min(8, p.tiles_r - 8 * band);
  const int tf = in_band / deep, r0 = (8 * band + in_band - tf * deep) * TILE, f0 = tf * TILE;

  // Loads: load i of a wave brings eight rows of 128 bytes, rows past the end the last one's again (computed and dropped).
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, (unsigned)(((p.rows - 1) * (int64_t)p.ldx + p.k) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, 0, (unsigned)(((p.feats - 1) * (int64_t)p.ldw + p.k) * 2), 0x00020000);
  unsigned from[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = 8 * (i % HALF * 4 + wave) + lane / 8;
    if (i < HALF) from[i] = (unsigned)min(r0 + row, p.rows - 1) * (unsigned)(p.ldx * 2) + (lane % 8 ^ (row & 7)) * 16;
    else from[i] = (unsigned)min(f0 + row, p.feats - 1) * (unsigned)(p.ldw * 2) + (lane % 8 ^ ((row & 3) | (row >> 3 & 1) << 2)) * 16;
  }
  const int blocks = p.k / 64;   // at least STAGES
  auto load = [&](int block, int stage, int i) __attribute__((always_inline)) {
    load16_to_lds(i < HALF ? xres : wres, lds + stage * STAGE + (i / HALF) * (STAGE / 2) + 1024 * (i % HALF * 4 + wave), from[i], block * 128);
  };
  // Fragments of a half block `h` (32 k): the lane's row and chunk.
  struct Frags {
    bf16x8 w[FRAGS], x[FRAGS];
  };
  const int chunk = (g ^ (c & 7)) * 16;
  const int x_at = (wr * WT + c) * 128 + chunk, w_at = STAGE / 2 + (wf * WT + 8 * (c / 4) + c % 4) * 128 + chunk;
  auto read = [&](Frags& f, int stage, int h, int i) __attribute__((always_inline)) {
    const char* base = lds + stage * STAGE;
    if (i < FRAGS) f.w[i] = *reinterpret_cast<const bf16x8*>(base + (w_at ^ (h * 64)) + (32 * (i / 2) + 4 * (i % 2)) * 128);
    else f.x[i - FRAGS] = *reinterpret_cast<const bf16x8*>(base + (x_at ^ (h * 64)) + (i - FRAGS) * 16 * 128);
  };
  float4v acc[FRAGS][FRAGS];
#pragma unroll
  for (int u = 0; u < FRAGS; ++u)
#pragma unroll
    for (int t = 0; t < FRAGS; ++t) acc[u][t] = float4v{0.f, 0.f, 0.f, 0.f};

  // all loads of the first stages but the last half of the last, which the first block's first half asks for
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
#pragma unroll
    for (int i = 0; i < (s == STAGES - 2 ? HALF : LOADS); ++i) load(s, s, i);
  Frags f0_, f1_;
  wait_loads<(STAGES - 3) * LOADS + HALF>();
  stage_barrier();
#pragma unroll
  for (int i = 0; i < READS; ++i) read(f0_, 0, 0, i);
  int stage = 0;
  // The products of `cur`, and between them the reads of `nxt` (half `nh` of the block in stage `ns`) and N loads from number
  // `first` on for `block` into stage `to`; the order is kept as written.
  auto half = [&](const Frags& cur, Frags& nxt, int ns, int nh, int block, int to, int first, auto loads) __attribute__((always_inline)) {
    constexpr int N = decltype(loads)::value, SLOTS = READS + N;
#pragma unroll
    for (int j = 0; j < PRODUCTS; ++j) {
      acc[j / FRAGS][j % FRAGS] = mfma32(cur.w[j % FRAGS], cur.x[j / FRAGS], acc[j / FRAGS][j % FRAGS]);
#pragma unroll
      for (int q = j * SLOTS / PRODUCTS; q < (j + 1) * SLOTS / PRODUCTS; ++q) {
        const int l = q * N / SLOTS;
        if ((q + 1) * N / SLOTS > l) load(block, to, first + l);
        else read(nxt, ns, nh, q - l);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Block `b`, in stage b % STAGES. SECOND: its first half asks for the rest of block b + STAGES - 2, into the stage of block
  // b - 2; FIRST: its second half for the first part of block b + STAGES - 1, into the stage of block b - 1, which every wave
  // has read once it is past the barrier. What the barrier orders besides: block b + 1 is there.
  auto step = [&](int b, auto second, auto first) __attribute__((always_inline)) {
    constexpr bool SECOND = decltype(second)::value, FIRST = decltype(first)::value;
    const int next = (stage + 1) % STAGES, before = (stage + STAGES - 1) % STAGES, before2 = (stage + STAGES - 2) % STAGES;
    half(f0_, f1_, stage, 1, b + STAGES - 2, before2, HALF, std::integral_constant<int, SECOND ? HALF : 0>());
    if (FIRST) wait_loads<(STAGES - 3) * LOADS>();
    else wait_loads<0>();
    stage_barrier();
    half(f1_, f0_, next, 0, b + STAGES - 1, before, 0, std::integral_constant<int, FIRST ? HALF : 0>());   // (behind the last: nothing uses them)
    stage = next;
  };
  int b = 0;
  for (; b < blocks - STAGES + 1; ++b) step(b, std::true_type(), std::true_type());
  step(b++, std::true_type(), std::false_type());
#pragma unroll 1
  for (; b < blocks; ++b) step(b, std::false_type(), std::false_type());

  // a lane: row c of each sixteen, features 32 j + 8 g .. + 7
#pragma unroll
  for (int j = 0; j < FRAGS / 2; ++j) {
    const int f = f0 + wf * WT + 32 * j + 8 * g;
    if (f >= p.feats) continue;   // (a multiple of eight)
    float add[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) add[i] = p.bias != nullptr ? (float)p.bias[f + i] : 0.f;
#pragma unroll
    for (int u = 0; u < FRAGS; ++u) {
      const int r = r0 + wr * WT + 16 * u + c;
      if (r >= p.rows) continue;
      float4v y[2] = {acc[u][2 * j], acc[u][2 * j + 1]};
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i / 4][i % 4] += add[i];
      if constexpr (OUT_F32) {
        float4v* to = reinterpret_cast<float4v*>(static_cast<float*>(p.out) + r * p.ldo + f);
        to[0] = y[0];
        to[1] = y[1];
      } else {
        bf16x8 v;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (bf16_t)y[i / 4][i % 4];
        *reinterpret_cast<bf16x8*>(static_cast<bf16_t*>(p.out) + r * p.ldo + f) = v;
      }
    }
  }
}

}  // namespace

// Whether this kernel takes the product: no compute unit has two tiles and enough of them have one, the sizes are whole loads (64
// k, eight features) of at least as many blocks as stages. The library cuts k where there are few tiles, so that the line lies at
// half of the units for a short k and at four fifths for a long one. us, weights from memory, library and here, rows x features:
//   k 1,024: 984 x 2,304 (144 tiles) 14.9 12.2, 1,368 x 2,048 (176) 12.9 12.2, 2,008 x 2,048 (256) 14.3 12.1
//   k 2,048: 984 x 2,304 23.1 20.4, 2,008 x 1,152 (144) 21.0 19.8, 1,500 x 2,048 (192) 21.8 20.8, 2,048 x 2,048 24.2 21.6
//   k 3,072: 984 x 2,304 28.3 29.5, 984 x 3,072 (192) 30.7 29.9, 2,008 x 1,536 (192) 27.4 28.5, 1,100 x 3,072 (216) 32.3 30.2
//   k 8,192: 984 x 2,304 61.9 65.4, 1,464 x 2,048 (192) 58.3 64.8, 1,100 x 3,072 (216) 71.8 68.2, 2,048 x 2,048 74.3 67.2
// Where the last tile of rows is half empty or emptier, tiles of 64 rows may fill a single round as well, and the library has those.
// It is ahead with them from a k of 2,048 on:
//   k 1,024: 136 x 8,320 13.1 11.8, 260 x 6,144 13.0 11.8   k 1,984: 136 x 8,320 21.2 18.9, 288 x 6,400 21.3 19.1, 530 x 3,456 20.2 18.6
//   k 2,048: 136 x 8,320 16.9 19.8, 288 x 6,400 17.4 20.1, 530 x 3,456 16.5 19.3; 352 x 6,144 (288 tiles of 64 rows) 24.5 21.0,
//     129 x 16,384 (384) 28.4 25.5, 256 x 16,384 (512) 29.0 24.8   k 3,072: 129 x 16,384 31.6 31.1, 256 x 16,384 40.9 35.9
// and, where up to 64 rows leave half of every tile empty, from above 1,024 on:
//   k 1,024: 17 x 17,000 14.0 12.1, 64 x 25,000 15.6 14.0   k 1,280: 13.6 14.8, 17.5 17.6   k 1,792: 17.0 18.3, 21.5 21.2
//   k 2,560: 20 x 27,000 28.8 30.9, 64 x 32,000 34.3 35.9   k 4,096: 50.2 50.4, 62.9 63.8
extern "C" int dli_tile_gemm_takes(int64_t rows, int64_t feats, int64_t k, int units) {
  if (rows <= 0 || feats <= 0 || feats % 8 != 0 || k % 64 != 0 || k < 64 * STAGES) return 0;
  const int64_t across = (feats + TILE - 1) / TILE, tiles = (rows + TILE - 1) / TILE * across;
  if ((rows + 63) / 64 * across <= units && (rows <= 64 ? k > 1024 : k >= 2048)) return 0;
  return (k <= 2048 ? 2 * tiles > units : 5 * tiles > 4 * units) && tiles <= units;
}

bool tile_gemm_takes(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* out, int64_t ldo, int64_t rows, int64_t feats,
                     int64_t k, bool out_f32) {
  return dli_tile_gemm_takes(rows, feats, k, dli_compute_units()) && ldx % 8 == 0 && ldw % 8 == 0 && ldo % (out_f32 ? 4 : 8) == 0 &&
         (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16) == 0 && (rows * ldx + k) * 2 < (int64_t)1 << 31 &&
         (feats * ldw + k) * 2 < (int64_t)1 << 31;
}

int tile_gemm(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, void* out, int64_t ldo, int64_t rows,
              int64_t feats, int64_t k, bool out_f32, hipStream_t stream) {
  const TileArgs args{(const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, out, ldo, (int)ldx, (int)ldw, (int)rows, (int)feats, (int)k,
                      (int)((rows + TILE - 1) / TILE), (int)((feats + TILE - 1) / TILE)};
  const auto kernel = out_f32 ? tile_gemm_kernel<true> : tile_gemm_kernel<false>;
  if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, STAGES * STAGE) != hipSuccess) return DLI_ERR_LAUNCH;
  kernel<<<args.tiles_r * args.tiles_f, 256, STAGES * STAGE, stream>>>(args);
  return dli_launch_status();
}
