// Matrix-state recurrences with heads of 64 keys and 64 values, a step's rows cut into runs that are walked side by side
// (scan_runs.hip). For the entry points of the token-by-token kernels.
#pragma once
#include "common.h"

#define RUNS_DELTA 0   // S <- diag(w) S - (a u)(u^T S) + k v^T, u = k / sqrt(sum k^2 + 1e-6);   o = S^T r
#define RUNS_BONUS 1   // o = (S + diag(bonus) k v^T)^T r;   S <- diag(w) S + k v^T
#define RUNS_GATED 2   // S <- g S;   S <- S + k (beta (v - S^T k))^T;   o = S^T r    (g and beta one value a head and token)

#define RUNS_FINISH_SUM 0       // o alone, in 32-bit
#define RUNS_FINISH_SIGMOID 1   // o / sqrt(mean(o^2) + eps) * norm_w * sigmoid(gate) to `out`
#define RUNS_FINISH_SILU 2      // the same with silu(gate)

struct RunsArgs {
  const float *r, *k, *v;            // rows; r and k: a head's 64 values for every `group` value heads
  const float* w;                    // RUNS_GATED: beta of head h at column h, g at column heads + h
  const float* a;                    // RUNS_DELTA
  const float *gate, *bonus, *norm_w;
  int64_t r_stride, k_stride, v_stride, w_stride, a_stride, gate_stride;
  float eps;
  float* state; int64_t state_stride;
  const int *q_start, *positions, *state_slots;
  float* o; int64_t o_stride;        // [rows][heads * 64]
  void* out; int64_t out_stride;
  float *y, *ends, *moves;           // scratch: [rows][heads * 64], and per slot and head 64 x 64 (moves of RUNS_BONUS: 64)
  int heads, group, run_rows, runs;  // runs of `run_rows` (a multiple of 16) rows; `runs` of them hold the longest entry
  int entries, rows, row0;           // entries, whose rows begin at row `row0` (y: at its start) and are `rows` in all
};

// Slots that hold every run of these entries: the sum of ceil(rows of an entry / run_rows) is no more.
static inline int scan_runs_slots(int entries, int rows, int run_rows) { return rows / run_rows + entries; }

// Whether these rows can be walked so (16-byte loads and stores; the caller asks before it makes the scratch).
bool scan_runs_takes(const RunsArgs& p, int rule, int finish, int out_is_bf16);
int scan_runs(const RunsArgs& p, int rule, int finish, int out_is_bf16, hipStream_t stream);
