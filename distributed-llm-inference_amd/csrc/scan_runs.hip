// Matrix-state recurrences for steps with portions, heads of 64 keys and 64 values: a request's rows are cut into runs that
// are walked at the same time, all in 32-bit. Token by token a request is one chain of 50 instructions a token on
// 512 waves that have a SIMD each to themselves (2,048 tokens and 32 heads: 578 us the generalized delta rule, 378 the decayed
// sums with a bonus, at one instruction every four to five cycles); cut into runs the chip's waves are full. A run's effect
// on the state before it is linear, S_after = M S_before + E, o_t = o_t(from zero) + S_before^T y_t, so:
//
//   walk     every run token by token (RUNS_GATED: sixteen at a time, on the matrix cores), from a state of zeros (an entry's
//            first run from the request's own, which makes its results final): o and E. Where the rule mixes keys (RUNS_DELTA, RUNS_GATED) 64 more columns start from the unit
//            matrix and take no input: they end as M, and their outputs are y. Where it does not (RUNS_BONUS), M is the
//            product of the run's decays per key and y_t = r_t times their product before t.
//   carry    per request and head the states between the runs, one after the other: E_s <- M_s E_(s-1) + E_s on the matrix
//            cores (v_mfma_f32_16x16x4_f32); the last one is the request's new state.
//   finish   o_t += E_(s-1)^T y_t on the matrix cores, and in the same pass the per-head norm and gate where the rule has them.
//
// walk, token by token: a workgroup of four waves takes one (run, head) and 64 columns, values or unit matrix; sixteen lanes
// (a DPP row) share four columns and hold four keys of each, so that five 16-byte reads of LDS a token serve sixteen columns (with one column
// a lane, as token by token, LDS is what bounds it). The vectors of sixteen tokens are staged by the workgroup, the next
// sixteen are on their way meanwhile. What bounds it: vector instructions, some 75 to 110 a token and wave at four cycles each (110 to 130
// while a sum over the lanes took each column by itself: the walk of one prompt of 2,048 tokens 133 -> 108 us RUNS_DELTA, 54 -> 49
// RUNS_BONUS, and as far from 64 bits or less).
//
// Measured (one prompt of 2,048 tokens, 32 heads, walk + carry + finish, us): RUNS_DELTA 108 + 15 + 21 against 578 and 17 for
// the norm, RUNS_BONUS 49 + 8 + 17 against 378 and 17, RUNS_GATED 90 in all against 410. Where the cut lies: ops.scan_runs.
// Beside 255 single tokens, which keep the kernel of steps of single tokens: 245, 168 and (walked token by token then) 183 us a
// layer (5,150, 2,880 and 2,610 token by token; 1,048, 1,301 and 818 with every entry cut and the launch as large as the longest entry times the entries).
// Distance from the rules in 64 bits against token by token (2-norm; 300 to 4,096 tokens, 8 to 32 heads, every row of outputs and
// the state left): 0.99 to 1.00 times as far RUNS_DELTA, 1.01 to 1.03 RUNS_BONUS, 4e-8 to 2e-7 either way.
#include "scan_runs.h"

typedef float rf4 __attribute__((ext_vector_type(4)));
typedef double rd4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float runs_row_sum(float x) {   // over the sixteen lanes of a DPP row
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0xB1, 0xF, 0xF, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x4E, 0xF, 0xF, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x141, 0xF, 0xF, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x140, 0xF, 0xF, false));
  return x;
}

// Four sums over the sixteen lanes of a DPP row, each where it is wanted: the lanes of quad b hold column (b + j) % 4 in register j, so
// column b's other parts lie 4 j lanes back, and three rotated additions bring them together; two more sum the quad. Column
// by column it is four additions each, sixteen in all.
__device__ __forceinline__ float runs_own_sum(const rf4& x) {
  return quad_sum(((x[0] + row_ror<8>(x[2])) + (row_ror<4>(x[1]) + row_ror<12>(x[3]))));
}
// Every quad's own value to the registers of its column.
__device__ __forceinline__ rf4 runs_to_columns(float own) { return rf4{own, row_ror<12>(own), row_ror<8>(own), row_ror<4>(own)}; }

// Runs lie one behind the other in slots, by entry and place, and a launch has a workgroup a slot and head: as large as the rows
// are and not as the longest entry times the entries, what is left over at its end (empty workgroups between the others leave
// the compute units unevenly filled: 360 us instead of 221 for 16 prompts of 375 tokens). A wave looks its run up, 64 entries a trip.
struct RunsPlace { int entry, run, first, n, row0; };
__device__ __forceinline__ int runs_of(const RunsArgs& p, int entry) {
  return entry < p.entries ? (p.q_start[entry + 1] - p.q_start[entry] + p.run_rows - 1) / p.run_rows : 0;
}
__device__ __forceinline__ RunsPlace runs_place(const RunsArgs& p, int slot) {
  const int lane = threadIdx.x % 64;
  RunsPlace at = {0, slot, 0, 0, 0};
  if (p.entries > 1) {
    int before = 0, e0 = 0;
    for (;; e0 += 64) {
      if (e0 >= p.entries) return at;   // past the last run
      const int own = runs_of(p, e0 + lane);
      int upto = own;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(upto, d, DLI_WAVE);
        upto += lane >= d ? up : 0;
      }
      const uint64_t behind = __ballot(before + upto > slot);
      if (behind != 0) {
        const int l = __ffsll((unsigned long long)behind) - 1;
        at.entry = e0 + l;
        at.run = __builtin_amdgcn_readfirstlane(slot - before - __shfl(upto - own, l, DLI_WAVE));
        break;
      }
      before += __builtin_amdgcn_readfirstlane(__shfl(upto, 63, DLI_WAVE));
    }
  }
  at.first = p.q_start[at.entry];
  at.row0 = at.first + at.run * p.run_rows;
  at.n = min(p.run_rows, p.q_start[at.entry + 1] - at.row0);
  return at;
}
// The slot of an entry's first run.
__device__ __forceinline__ int runs_before(const RunsArgs& p, int entry) {
  int sum = 0;
  for (int e = threadIdx.x % 64; e < entry; e += 64) sum += runs_of(p, e);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d, DLI_WAVE);
  return __builtin_amdgcn_readfirstlane(sum);
}

template <int RULE>
__global__ __launch_bounds__(256) void scan_runs_walk_kernel(RunsArgs p) {
  constexpr int D = 64, TB = 16;
  __shared__ rf4 sk[TB * 16], sr[TB * 16], sv[TB * 16], sw[TB * 16], sc[RULE == RUNS_DELTA ? TB * 16 : 1];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, vloc = lane / 16, part = lane % 16;
  const RunsPlace place = runs_place(p, blockIdx.y);
  const int entry = place.entry, run = place.run, first = place.first, row0 = place.row0, n = place.n, head = blockIdx.x;
  const bool unit = blockIdx.z != 0;   // the columns of the unit matrix
  if (n <= 0 || (unit && run == 0)) return;
  const int col = wave * 16 + vloc * 4, quad = part / 4;   // the first of these sixteen lanes' four columns; the one whose sums are this lane's
  int column[4];   // of s's registers (runs_own_sum)
#pragma unroll
  for (int c = 0; c < 4; ++c) column[c] = col + (quad + c) % 4;
  const int64_t qk_col = (int64_t)(head / p.group) * D, v_col = (int64_t)head * D;

  float s[4][4];   // [key][column]
  rf4 bonus = {0.f, 0.f, 0.f, 0.f}, decay = {1.f, 1.f, 1.f, 1.f};
  const bool real = run == 0 && p.positions[first] != 0;
  const float* st = p.state + (int64_t)p.state_slots[entry] * p.state_stride + (int64_t)head * D * D;   // [value][key]
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    rf4 old = {0.f, 0.f, 0.f, 0.f};
    if (real) old = *reinterpret_cast<const rf4*>(st + column[c] * D + part * 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i][c] = unit ? (part * 4 + i == column[c] ? 1.f : 0.f) : old[i];
  }
  if (RULE == RUNS_BONUS) bonus = *reinterpret_cast<const rf4*>(p.bonus + v_col + part * 4);

  // staging: sixteen threads a token, four values each
  const int bt = tid / 16, bc = tid % 16 * 4;
  rf4 fk, fr, fv = {0.f, 0.f, 0.f, 0.f}, fw, fa;
  const auto fetch = [&](int t0) {
    const int64_t row = row0 + min(t0 + bt, n - 1);
    fk = *reinterpret_cast<const rf4*>(p.k + row * p.k_stride + qk_col + bc);
    fr = *reinterpret_cast<const rf4*>(p.r + row * p.r_stride + qk_col + bc);
    if (!unit) fv = *reinterpret_cast<const rf4*>(p.v + row * p.v_stride + v_col + bc);
    fw = *reinterpret_cast<const rf4*>(p.w + row * p.w_stride + v_col + bc);
    if constexpr (RULE == RUNS_DELTA) fa = *reinterpret_cast<const rf4*>(p.a + row * p.a_stride + v_col + bc);
  };
  const int64_t dst_stride = unit ? (int64_t)p.heads * D : p.o_stride;
  float* dst = unit ? p.y + (row0 - p.row0) * dst_stride : p.o + row0 * dst_stride;
  const auto step = [&](int t) {
    const rf4 k = sk[t * 16 + part], r = sr[t * 16 + part];
    const float v_own = reinterpret_cast<const float*>(sv)[t * 64 + col + quad];
    rf4 o;
    if constexpr (RULE == RUNS_BONUS) {
      const rf4 w = sw[t * 16 + part], v = runs_to_columns(v_own);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float kv = k[i] * v[c];
          float& sum = i & 1 ? o1 : o0;
          sum = fmaf(fmaf(bonus[i], kv, s[i][c]), r[i], sum);
          s[i][c] = fmaf(w[i], s[i][c], kv);
        }
        o[c] = o0 + o1;
      }
      if (wave == 0 && vloc == 0 && run > 0)
        *reinterpret_cast<rf4*>(p.y + (int64_t)(row0 - p.row0 + t) * p.heads * D + v_col + part * 4) = r * decay;
      decay *= w;
    } else {
      rf4 us;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        us[c] = fmaf(k[3], s[3][c], fmaf(k[2], s[2][c], fmaf(k[1], s[1][c], k[0] * s[0][c])));
      }
      const float us_own = runs_own_sum(us);
      const rf4 w = sw[t * 16 + part], a = sc[t * 16 + part], v = runs_to_columns(v_own);
      us = runs_to_columns(us_own);
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i][c] = fmaf(w[i], s[i][c], fmaf(k[i], v[c], -a[i] * us[c]));
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        o[c] = fmaf(r[3], s[3][c], fmaf(r[2], s[2][c], fmaf(r[1], s[1][c], r[0] * s[0][c])));
      }
    }
    return runs_own_sum(o);
  };

  fetch(0);
  for (int t0 = 0; t0 < n; t0 += TB) {
    __syncthreads();   // the batch before has been walked
    if constexpr (RULE == RUNS_DELTA) {
      const float kn = 1.f / sqrtf(runs_row_sum(fk[0] * fk[0] + fk[1] * fk[1] + (fk[2] * fk[2] + fk[3] * fk[3])) + 1e-6f);
      sc[tid] = fa * (fk * kn) * kn;   // a u (u^T S) = (a u kn) (k^T S)
    }
    sk[tid] = fk;
    sr[tid] = fr;
    sv[tid] = fv;
    sw[tid] = fw;
    if (t0 + TB < n) fetch(t0 + TB);   // on their way while this batch is walked
    __syncthreads();
    const int nb = min(TB, n - t0);
    float* od = dst + t0 * dst_stride + v_col + col + quad;
    if (nb == TB) {
#pragma unroll 4
      for (int t = 0; t < TB; ++t) {
        const float o = step(t);
        if (part % 4 == 0) od[t * dst_stride] = o;
      }
    } else {
      for (int t = 0; t < nb; ++t) {
        const float o = step(t);
        if (part % 4 == 0) od[t * dst_stride] = o;
      }
    }
    if constexpr (RULE == RUNS_BONUS) p.y += (int64_t)TB * p.heads * D;   // (the step counts its rows from the batch's first)
  }
  const int64_t at = ((int64_t)blockIdx.y * p.heads + head) * D;
  float* end = (unit ? p.moves : p.ends) + at * D;
#pragma unroll
  for (int c = 0; c < 4; ++c) *reinterpret_cast<rf4*>(end + column[c] * D + part * 4) = rf4{s[0][c], s[1][c], s[2][c], s[3][c]};
  if (RULE == RUNS_BONUS && wave == 0 && vloc == 0) *reinterpret_cast<rf4*>(p.moves + at + part * 4) = decay;
}

// The walk of RUNS_GATED, sixteen tokens at a time on the matrix cores (v_mfma_f32_16x16x4_f32, 32-bit products and sums). With S the
// state before the sixteen, G_t the product of their g up to t, D_ts that of g behind s up to t, b beta:
//
//   u_t = b_t (v_t - G_t S^T k_t - sum_(s<t) D_ts (k_t . k_s) u_s)      (forward substitution: four tokens at a time, the others' sums
//   o_t = G_t S^T r_t + sum_(s<=t) D_ts (r_t . k_s) u_s                  go on as a product)
//   S  <- G_T S + sum_s D_Ts k_s u_s^T
//
// The products of g are made as products, never as quotients, and a factor that is left out is left out by choice and not by a
// product with zero: what is infinite at a token stays out of the tokens before it. A workgroup of four waves takes one (run, head)
// and 64 columns, a wave sixteen of them: lane (c, g) holds keys 16 kb + 4 g .. + 3 of column c, which are operands and results of the
// products as they stand. The dot products of the tokens with each other are made a quarter a wave.
// What bounds it: 63 products of 32 cycles a wave and sixteen tokens, and four meetings of the workgroup. Token by token, as
// the other rules are walked (their decays are a value a key), the vector units spent some 80 instructions of four cycles a token
// and wave: walk, carry and sums of 32 heads, us, four prompts of 2,990 tokens 169 -> 120, one of 2,048 111 -> 90 and of 300 37 -> 30,
// sixteen of 375 148 -> 112, one of 8,192 368 -> 280. As far from 64 bits as token by token or less
// (2-norm; 300 to 2,048 tokens, 8 to 32 heads, g near 1, from 0.37 on, from 0.0025 on and with zeros among them, keys alike and not:
// outputs 0.62 to 1.04 times, before 0.86 to 1.21; the state left 0.82 to 1.08, before 0.97 to 1.18).
template <int SHIFT>
__device__ __forceinline__ float runs_before_by(float x) {   // the value SHIFT lanes before in the DPP row, 1 before its first
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0x3f800000, __builtin_bit_cast(int, x), 0x110 + SHIFT, 0xF, 0xF, false));
}
template <int SHIFT>
__device__ __forceinline__ float runs_behind_by(float x) {   // SHIFT lanes behind, 1 past its last
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0x3f800000, __builtin_bit_cast(int, x), 0x100 + SHIFT, 0xF, 0xF, false));
}
__device__ __forceinline__ float runs_product_behind(float x) {   // of the lanes behind this one in its DPP row
  x = runs_behind_by<1>(x);
  x *= runs_behind_by<1>(x);
  x *= runs_behind_by<2>(x);
  x *= runs_behind_by<4>(x);
  return x * runs_behind_by<8>(x);
}
__global__ __launch_bounds__(256, 4) void scan_gated_walk_kernel(RunsArgs p) {
  constexpr int D = 64, TB = 16, WIDE = 84, SQ = 20;   // (rows of LDS: no two of sixteen lanes' 16-byte reads on one bank)
  __shared__ __attribute__((aligned(16))) float sk[TB * WIDE], sr[TB * WIDE], keep[TB * SQ], give[TB * SQ];
  __shared__ __attribute__((aligned(16))) float dots[2][4][TB * SQ];
  __shared__ __attribute__((aligned(16))) float s_g[TB], s_b[TB], s_bg[TB], s_e[TB];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, c = lane % 16, g = lane / 16, bt = tid / 16;
  const RunsPlace place = runs_place(p, blockIdx.y);
  const int run = place.run, row0 = place.row0, n = place.n, head = blockIdx.x;
  const bool unit = blockIdx.z != 0;   // the columns of the unit matrix
  if (n <= 0 || (unit && run == 0)) return;
  const int col = wave * 16 + c;
  const int64_t qk_col = (int64_t)(head / p.group) * D, v_col = (int64_t)head * D;

  rf4 s[4];   // keys 16 kb + 4 g + i of the column
  const bool real = run == 0 && p.positions[place.first] != 0;
  const float* st = p.state + (int64_t)p.state_slots[place.entry] * p.state_stride + (int64_t)head * D * D;   // [value][key]
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    rf4 old = {0.f, 0.f, 0.f, 0.f};
    if (real) old = *reinterpret_cast<const rf4*>(st + col * D + 16 * kb + 4 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[kb][i] = unit ? (16 * kb + 4 * g + i == col ? 1.f : 0.f) : old[i];
  }
  rf4 fk, fr, fv = {0.f, 0.f, 0.f, 0.f};
  float fb = 0.f, fg = 1.f;
  const auto fetch = [&](int t0) {
    const int64_t row = row0 + min(t0 + bt, n - 1), token = row0 + min(t0 + c, n - 1);
    fk = *reinterpret_cast<const rf4*>(p.k + row * p.k_stride + qk_col + 4 * c);
    fr = *reinterpret_cast<const rf4*>(p.r + row * p.r_stride + qk_col + 4 * c);
    fb = p.w[token * p.w_stride + head];
    fg = p.w[token * p.w_stride + p.heads + head];
    if (!unit)
#pragma unroll
      for (int i = 0; i < 4; ++i) fv[i] = p.v[(int64_t)(row0 + min(t0 + 4 * g + i, n - 1)) * p.v_stride + v_col + col];
  };
  const int64_t dst_stride = unit ? (int64_t)p.heads * D : p.o_stride;
  float* dst = (unit ? p.y + (row0 - p.row0) * dst_stride : p.o + row0 * dst_stride) + v_col + col;

  fetch(0);
  for (int t0 = 0; t0 < n; t0 += TB) {
    const bool there = t0 + bt < n;   // rows past the last: keys and values of zero, g of one, beta of zero
    __syncthreads();   // the sixteen before have been walked
    *reinterpret_cast<rf4*>(&sk[bt * WIDE + 4 * c]) = there ? fk : rf4{0.f, 0.f, 0.f, 0.f};
    *reinterpret_cast<rf4*>(&sr[bt * WIDE + 4 * c]) = fr;
    const float decay = t0 + c < n ? fg : 1.f, beta = t0 + c < n ? fb : 0.f;   // token c's
    float upto = decay;
    upto *= runs_before_by<1>(upto);
    upto *= runs_before_by<2>(upto);
    upto *= runs_before_by<4>(upto);
    upto *= runs_before_by<8>(upto);
    const float behind = runs_product_behind(c <= bt ? decay : 1.f);   // D of token bt and token c
    if (tid < TB) {
      s_g[c] = upto;
      s_b[c] = beta;
      s_bg[c] = beta * upto;
      s_e[c % 4 * 4 + c / 4] = runs_product_behind(decay);
    }
    const float all = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, upto), 15));
    const rf4 v = fv;
    if (t0 + TB < n) fetch(t0 + TB);   // on their way while these are walked
    __syncthreads();
    {
      const rf4 kw = *reinterpret_cast<const rf4*>(&sk[c * WIDE + 16 * wave + 4 * g]);
      const rf4 rw = *reinterpret_cast<const rf4*>(&sr[c * WIDE + 16 * wave + 4 * g]);
      rd4 kk = {0., 0., 0., 0.}, rk = {0., 0., 0., 0.};   // (in 64-bit: each of them counts in as many sums as there are columns)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        kk = __builtin_amdgcn_mfma_f64_16x16x4f64((double)kw[i], (double)kw[i], kk, 0, 0, 0);
        rk = __builtin_amdgcn_mfma_f64_16x16x4f64((double)rw[i], (double)kw[i], rk, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {   // (these results lie in rows g, g + 4, ..)
        dots[0][wave][(4 * i + g) * SQ + c] = (float)kk[i];
        dots[1][wave][(4 * i + g) * SQ + c] = (float)rk[i];
      }
    }
    rf4 ks[4], rs[4];   // (sixteen keys a sum, and a tree of these: one sum over all 64 is half again as far from 64 bits)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const rf4 ka = *reinterpret_cast<const rf4*>(&sk[c * WIDE + 16 * kb + 4 * g]);
      const rf4 ra = *reinterpret_cast<const rf4*>(&sr[c * WIDE + 16 * kb + 4 * g]);
      ks[kb] = rs[kb] = rf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ks[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[i], s[kb][i], ks[kb], 0, 0, 0);
        rs[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[i], s[kb][i], rs[kb], 0, 0, 0);
      }
    }
    const rf4 from_s = (ks[0] + ks[1]) + (ks[2] + ks[3]);
    rf4 o = (rs[0] + rs[1]) + (rs[2] + rs[3]);
    __syncthreads();
    {
      const int at = bt * SQ + c;
      const float kk = (dots[0][0][at] + dots[0][1][at]) + (dots[0][2][at] + dots[0][3][at]);
      const float rk = (dots[1][0][at] + dots[1][1][at]) + (dots[1][2][at] + dots[1][3][at]);
      float within = -(s_b[bt] * behind) * kk;
      asm("" : "+v"(within));   // (made by every lane: behind a branch the reads of LDS would wait for each other)
      keep[bt * SQ + c] = there && c < bt ? within : 0.f;
      give[bt * SQ + c % 4 * 4 + c / 4] = c <= bt ? behind * rk : 0.f;   // (a lane's four tokens g, g + 4, .. side by side)
    }
    __syncthreads();
    // A lane's own four tokens to all lanes of its column by way of LDS (in registers it is fourteen instructions a value). What is
    // taken off v is summed first and u rounded once at its own size: taken off term by term it doubles the distance from 64 bits.
    float* turned = &dots[0][wave][c * SQ];   // (the wave's own, and v behind it)
    rf4 off;
    {
      const rf4 bg4 = *reinterpret_cast<const rf4*>(&s_bg[4 * g]);
      rf4 vz = v;
#pragma unroll
      for (int i = 0; i < 4; ++i) off[i] = -bg4[i] * from_s[i];
      if (t0 + TB > n)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          off[i] = t0 + 4 * g + i < n ? off[i] : 0.f;
          vz[i] = t0 + 4 * g + i < n ? vz[i] : 0.f;
        }
      *reinterpret_cast<rf4*>(turned + 4 * g) = off;
      *reinterpret_cast<rf4*>(turned + 4 * TB * SQ + 4 * g) = vz;
      o *= *reinterpret_cast<const rf4*>(&s_g[4 * g]);
    }
    rf4 mine;   // u of tokens g, g + 4, g + 8, g + 12
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      __builtin_amdgcn_wave_barrier();
      rf4 y = *reinterpret_cast<const rf4*>(turned + 4 * q), u;
      const rf4 vq = *reinterpret_cast<const rf4*>(turned + 4 * TB * SQ + 4 * q), bq = *reinterpret_cast<const rf4*>(&s_b[4 * q]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const rf4 l = *reinterpret_cast<const rf4*>(&keep[(4 * q + i) * SQ + 4 * q]);
#pragma unroll
        for (int j = 0; j < i; ++j) y[i] = fmaf(l[j], u[j], y[i]);
        u[i] = fmaf(bq[i], vq[i], y[i]);
      }
      asm("" : "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]));
      mine[q] = g < 2 ? (g == 0 ? u[0] : u[1]) : (g == 2 ? u[2] : u[3]);
      if (q < 3) {
        off = __builtin_amdgcn_mfma_f32_16x16x4f32(keep[c * SQ + 4 * q + g], mine[q], off, 0, 0, 0);
        __builtin_amdgcn_wave_barrier();
        *reinterpret_cast<rf4*>(turned + 4 * g) = off;
      }
    }
    const bool finite = __builtin_isfinite(mine[0]) && __builtin_isfinite(mine[1]) && __builtin_isfinite(mine[2]) && __builtin_isfinite(mine[3]);
    if (__ballot(!finite) == 0) {
      const rf4 part = *reinterpret_cast<const rf4*>(&give[c * SQ + 4 * g]);
#pragma unroll
      for (int q = 0; q < 4; ++q) o = __builtin_amdgcn_mfma_f32_16x16x4f32(part[q], mine[q], o, 0, 0, 0);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        for (int j = 0; j < 4; ++j) {   // token 4 q + j
          const float u = __shfl(mine[q], 16 * j + c, DLI_WAVE);
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = 4 * q + j <= 4 * g + i ? fmaf(give[(4 * g + i) * SQ + 4 * j + q], u, o[i]) : o[i];
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (t0 + 4 * g + i < n) dst[(t0 + 4 * g + i) * dst_stride] = o[i];
    mine *= *reinterpret_cast<const rf4*>(&s_e[4 * g]);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) s[kb] *= all;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(sk[(4 * q + g) * WIDE + 16 * kb + c], mine[q], s[kb], 0, 0, 0);
  }
  float* end = (unit ? p.moves : p.ends) + ((int64_t)blockIdx.y * p.heads + head) * D * D;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) *reinterpret_cast<rf4*>(end + col * D + 16 * kb + 4 * g) = s[kb];
}

// A workgroup takes sixteen values of one (entry, head) through all its runs. Lane (i, g) of wave w makes keys 16 w + i of
// values 4 g .. + 3: S^T M^T, S^T out of LDS, M^T and E (the next run's while this one is multiplied) from memory.
template <int RULE>
__global__ __launch_bounds__(256) void scan_runs_carry_kernel(RunsArgs p) {
  constexpr int D = 64, LD = 68;
  __shared__ __attribute__((aligned(16))) float ss[16 * LD];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, i = lane % 16, g = lane / 16;
  const int entry = blockIdx.x, head = blockIdx.y, v0 = blockIdx.z * 16;
  const int first = p.q_start[entry], len = p.q_start[entry + 1] - first;
  if (len <= 0) return;
  const int runs = (len + p.run_rows - 1) / p.run_rows;
  const int64_t slot = runs_before(p, entry), per_run = (int64_t)p.heads * D * D;
  float* ends = p.ends + (slot * p.heads + head) * D * D + v0 * D;
  float* st = p.state + (int64_t)p.state_slots[entry] * p.state_stride + ((int64_t)head * D + v0) * D;
  const int vr = tid / 16, kc = tid % 16 * 4;   // whole rows of the slice, 16 bytes a thread
  rf4 s = *reinterpret_cast<const rf4*>(ends + vr * D + kc);
  if constexpr (RULE == RUNS_BONUS) {
    const float* moves = p.moves + (slot * p.heads + head) * D + kc;
    for (int run = 1; run < runs; ++run) {
      const rf4 m = *reinterpret_cast<const rf4*>(moves + (int64_t)run * p.heads * D);
      float* e = ends + run * per_run + vr * D + kc;
      s = m * s + *reinterpret_cast<const rf4*>(e);
      *reinterpret_cast<rf4*>(e) = s;
    }
  } else {
    *reinterpret_cast<rf4*>(ss + vr * LD + kc) = s;
    const float* moves = p.moves + (slot * p.heads + head) * D * D + 16 * wave + i;
    float fm[16], fe[4];
    const auto fetch = [&](int run) {
#pragma unroll
      for (int x = 0; x < 16; ++x) fm[x] = moves[run * per_run + (x / 4 * 16 + 4 * g + x % 4) * D];
#pragma unroll
      for (int e = 0; e < 4; ++e) fe[e] = ends[run * per_run + (4 * g + e) * D + 16 * wave + i];
    };
    if (runs > 1) fetch(1);
    for (int run = 1; run < runs; ++run) {
      __syncthreads();
      rf4 acc[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const rf4 a = *reinterpret_cast<const rf4*>(ss + i * LD + 16 * t + 4 * g);
        acc[t] = rf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], fm[4 * t + e], acc[t], 0, 0, 0);
      }
      // (E last: what M leaves of the old state is mostly small beside it, and would round at E's size sixteen times)
      const rf4 sum = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + rf4{fe[0], fe[1], fe[2], fe[3]};
      if (run + 1 < runs) fetch(run + 1);
      __syncthreads();   // the old state has been read
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ss[(4 * g + e) * LD + 16 * wave + i] = sum[e];
        ends[run * per_run + (4 * g + e) * D + 16 * wave + i] = sum[e];
      }
    }
    __syncthreads();
    s = *reinterpret_cast<const rf4*>(ss + vr * LD + kc);
  }
  *reinterpret_cast<rf4*>(st + vr * D + kc) = s;
}

// A wave takes sixteen rows of one run and head: lane (i, g) holds values 16 c + 4 g .. + 3 of row i.
template <typename T, int FINISH>
__global__ __launch_bounds__(256) void scan_runs_finish_kernel(RunsArgs p) {
  constexpr int D = 64;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, i = lane % 16, g = lane / 16;
  const RunsPlace place = runs_place(p, blockIdx.y);
  const int run = place.run, row0 = place.row0, n = place.n, head = blockIdx.x, t0 = blockIdx.z * 64 + wave * 16;
  if (t0 >= n || (FINISH == RUNS_FINISH_SUM && run == 0)) return;
  const int64_t row = row0 + min(t0 + i, n - 1), c0 = (int64_t)head * D + 4 * g;
  rf4 o[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) o[c] = *reinterpret_cast<const rf4*>(p.o + row * p.o_stride + c0 + 16 * c);
  if (run > 0) {
    const float* s = p.ends + ((int64_t)(blockIdx.y - 1) * p.heads + head) * D * D + i * D + 4 * g;
    const float* y = p.y + (row - p.row0) * p.heads * D + c0;
    rf4 fy[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) fy[t] = *reinterpret_cast<const rf4*>(y + 16 * t);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      rf4 fs[4], acc[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) fs[t] = *reinterpret_cast<const rf4*>(s + 16 * c * D + 16 * t);
#pragma unroll
      for (int t = 0; t < 4; ++t) {   // four sums of sixteen keys side by side: shorter chains, smaller roundings
        acc[t] = rf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(fs[t][e], fy[t][e], acc[t], 0, 0, 0);
      }
      o[c] += (acc[0] + acc[1]) + (acc[2] + acc[3]);
    }
  }
  if constexpr (FINISH == RUNS_FINISH_SUM) {
    if (t0 + i < n)
#pragma unroll
      for (int c = 0; c < 4; ++c) *reinterpret_cast<rf4*>(p.o + row * p.o_stride + c0 + 16 * c) = o[c];
    return;
  }
  float sum = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c) sum += (o[c][0] * o[c][0] + o[c][1] * o[c][1]) + (o[c][2] * o[c][2] + o[c][3] * o[c][3]);
  sum = add_across32(add_across16(sum));
  const float rn = 1.f / sqrtf(sum / (float)D + p.eps);
  if (t0 + i >= n) return;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const rf4 gp = *reinterpret_cast<const rf4*>(p.gate + row * p.gate_stride + c0 + 16 * c);
    const rf4 nw = *reinterpret_cast<const rf4*>(p.norm_w + c0 + 16 * c);
    struct alignas(sizeof(T) * 4) Packed { T v[4]; } packed;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float gate = (FINISH == RUNS_FINISH_SILU ? gp[e] : 1.f) / (1.f + expf(-gp[e]));
      packed.v[e] = from_f32<T>(o[c][e] * rn * nw[e] * gate);
    }
    *reinterpret_cast<Packed*>((T*)p.out + row * p.out_stride + c0 + 16 * c) = packed;
  }
}

bool scan_runs_takes(const RunsArgs& p, int rule, int finish, int out_is_bf16) {
  const auto whole = [](const void* at, size_t bytes) { return (uintptr_t)at % bytes == 0; };
  const auto rows = [&](const float* at, int64_t stride) { return stride % 4 == 0 && whole(at, 16); };
  if (p.y == nullptr || p.ends == nullptr || p.moves == nullptr || p.entries < 1 || p.rows < p.entries || p.runs < 1 || p.run_rows < 16 || p.run_rows % 16 != 0) return false;
  if (!rows(p.r, p.r_stride) || !rows(p.k, p.k_stride) || !rows(p.v, p.v_stride) || !rows(p.o, p.o_stride) ||
      !rows(p.state, p.state_stride) || !whole(p.y, 16) || !whole(p.ends, 16) || !whole(p.moves, 16))
    return false;
  if (rule != RUNS_GATED && !rows(p.w, p.w_stride)) return false;
  if (rule == RUNS_DELTA && !rows(p.a, p.a_stride)) return false;
  if (rule == RUNS_BONUS && !whole(p.bonus, 16)) return false;
  return finish == RUNS_FINISH_SUM || (rows(p.gate, p.gate_stride) && whole(p.norm_w, 16) && p.out_stride % 4 == 0 &&
                                       whole(p.out, out_is_bf16 ? 8 : 16));
}

int scan_runs(const RunsArgs& p, int rule, int finish, int out_is_bf16, hipStream_t stream) {
  const int slots = scan_runs_slots(p.entries, p.rows, p.run_rows);
  if (slots > 65535) return DLI_ERR_ARGUMENT;
  const dim3 walk(p.heads, slots, rule == RUNS_BONUS || p.runs == 1 ? 1 : 2), carry(p.entries, p.heads, 4);
  if (rule == RUNS_DELTA) {
    scan_runs_walk_kernel<RUNS_DELTA><<<walk, 256, 0, stream>>>(p);
    scan_runs_carry_kernel<RUNS_DELTA><<<carry, 256, 0, stream>>>(p);
  } else if (rule == RUNS_BONUS) {
    scan_runs_walk_kernel<RUNS_BONUS><<<walk, 256, 0, stream>>>(p);
    scan_runs_carry_kernel<RUNS_BONUS><<<carry, 256, 0, stream>>>(p);
  } else {
    scan_gated_walk_kernel<<<walk, 256, 0, stream>>>(p);
    scan_runs_carry_kernel<RUNS_GATED><<<carry, 256, 0, stream>>>(p);
  }
  const dim3 done(p.heads, slots, (p.run_rows + 63) / 64);
  if (finish == RUNS_FINISH_SUM) {
    if (p.runs > 1) scan_runs_finish_kernel<float, RUNS_FINISH_SUM><<<done, 256, 0, stream>>>(p);
  } else if (finish == RUNS_FINISH_SIGMOID) {
    if (out_is_bf16) scan_runs_finish_kernel<bf16_t, RUNS_FINISH_SIGMOID><<<done, 256, 0, stream>>>(p);
    else scan_runs_finish_kernel<float, RUNS_FINISH_SIGMOID><<<done, 256, 0, stream>>>(p);
  } else {
    if (out_is_bf16) scan_runs_finish_kernel<bf16_t, RUNS_FINISH_SILU><<<done, 256, 0, stream>>>(p);
    else scan_runs_finish_kernel<float, RUNS_FINISH_SILU><<<done, 256, 0, stream>>>(p);
  }
  return dli_launch_status();
}
