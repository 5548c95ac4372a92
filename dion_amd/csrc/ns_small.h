// Host-side interface of the small-matrix Newton-Schulz kernel (ns_small.hip): normalisation, all iterations and the
// final store or weight update of a set of small matrices in one launch.
#pragma once
#include "common.h"

constexpr int DA_SMALL_BT = 64;           // tile edge: working matrices are padded to multiples of it
constexpr int DA_SMALL_MAX_STEPS = 8;
constexpr int DA_SMALL_CTR_STRIDE = 32;   // ints of control memory per matrix (one counter per phase)
// ints behind the counters: a line per queue (ticket word, owner word), then the status word's line
constexpr int DA_SMALL_TAIL = 9 * 32;

// One bucket of `cnt` same-shape wide matrices, mw <= nw multiples of 64, in bf16 working buffers
// x0, x1: [cnt][mw][ldx], a, b: [cnt][mw][lda].  x0 holds the staged input (not yet divided by its norm), zero outside
// the true matrix; partials: [cnt][ptiles] sums of squares of the staged input.
// tab: device table of `cnt` destination matrices (rows x cols, row pitch ld, dtype), stored transposed when rows > cols.
// vec: every destination row is whole 16-byte chunks (pitch a multiple of 8 elements, base 16-byte aligned).
// update 1: W <- r_W(r_W(W * decay) - r_bf16(X' * step)); 0: W <- X' (bf16 destinations).
struct DaNsSmallGroup {
  char *x0, *x1, *a, *b;
  long long sx, sa;              // elements between consecutive matrices
  int mw, nw, ldx, lda, cnt;
  const float* partials;
  int ptiles;
  void* const* tab;
  int dtype, rows, cols, ld, update, vec;
  float decay, step;
};

// ctl: DA_SMALL_CTR_STRIDE ints per matrix of all groups in order, then DA_SMALL_TAIL ints; cleared before the launch
// (the status word may be preset: the results are then NaN).
bool da_ns_small_applicable(const DaNsSmallGroup* g, int n, int steps);
int da_ns_small(const DaNsSmallGroup* g, int n, const float* coeffs, int steps, float eps, int* ctl, hipStream_t s);
