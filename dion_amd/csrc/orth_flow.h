// Host-side interface of the one-launch fp64 orthonormaliser of flagged matrices (orth_flow.hip).
#pragma once
#include "common.h"

constexpr int DA_ORTH_FLOW_CTL = 32;   // ints of control memory per matrix; another 9 * 32 for the launch

// Working memory of `batch` matrices (rows x r): P64 [batch][rows rounded up to 64][rp], rp = r rounded up to 64; slab
// [batch][slices][rp][rp]; L, T, gram [batch][rp][rp]; defect [batch][rp][rp / 32]; ctl: see above.
struct DaOrthFlow {
  double *P64, *slab, *L, *T, *gram, *defect;
  int* ctl;
};
int da_orth_flow_slices(int rows, int r);
// Whether the launch takes factors of these dimensions and is the better one for them.
bool da_orth_flow_applicable(int rows, int r);
// out[b] <- orth(P[b]) for the matrices with need[b] != 0 (out may be P); info[b] as da_orthonormalize.
int da_orth_flow(const void* P, void* out, int dtype, int batch, int rows, int r, int r_live, const int* need, int* info,
                 const DaOrthFlow& w, int fail, hipStream_t s);
