// Host-side interface of the small-matrix Dion kernels (dion_small.hip): the whole step of a set of small matrices in ten
// launches over all of them.
#pragma once
#include "common.h"

constexpr int DA_DS_GROUPS = 8;          // buckets together
constexpr int DA_DS_MATS = 96;           // matrices together (their pointers travel as arguments of the set-up launch)
constexpr int DA_DS_MAX_RANK = 256;

// A bucket of `cnt` same-shape matrices: X, G, M (m x n, contiguous), Q (min(m, n) x r, contiguous), host arrays of device
// pointers.  info: `cnt` device ints (or null), as da_orthonormalize.
struct DaDionSmallGroup {
  void* const* X;
  const void* const* G;
  void* const* M;
  void* const* Q;
  int cnt, m, n, r;
  float scaled_lr;
  int* info;
};
struct DaDionSmallCall {
  int x_dtype, g_dtype, m_dtype, q_dtype;
  float ef_alpha, decay, eps;
  int fail;   // test hook: start with the status word set
};

// Bytes of workspace, or 0 when they do not take these buckets (ranks, alignment of the matrices; `forced`: without
// the rule on the amount of work).
size_t da_dion_small_bytes(const DaDionSmallGroup* g, int n, const DaDionSmallCall& c, bool forced);
int da_dion_small(const DaDionSmallGroup* g, int n, const DaDionSmallCall& c, void* workspace, hipStream_t s);
