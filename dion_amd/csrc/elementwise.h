// Host-side launch descriptors for the HBM-bound passes (see elementwise.hip).
#pragma once
#include "common.h"

#define DA_MAX_PTRS 64  // matrices per launch: pointer tables travel as kernel arguments

struct DaPtrTable {
  void* p[DA_MAX_PTRS];
};

// Staging of up to DA_MAX_GROUPS buckets of same-shape matrices in one launch: momentum update (Muon) or plain cast,
// rounded into working matrices of *wide* orientation (rows <= cols), zero outside the true matrix.
struct DaStageGroup {
  void* wide;        // [cnt][mw][ldw]; null: the result of matrix b goes to dst[b], in source orientation, without padding
  float* partials;   // [cnt][da_stage_tiles(rows, cols, mw, nw)] sums of squares of the result (wide != null)
  void** xtab;       // optional: receives the dst pointers of the group's matrices
  int rows, cols;    // source matrices, row pitch ld (momentum: contiguous)
  int ld;
  int mw, nw, ldw;   // working matrices: rows, columns and pitch, all multiples of 8, >= min / max (rows, cols)
  int cnt;
};
constexpr int DA_STAGE_MATS = 80;   // matrices per launch: their pointers travel as kernel arguments
struct DaStage {
  DaStageGroup g[DA_MAX_GROUPS];
  int ngroups;
  const void* src[DA_STAGE_MATS];   // all groups' matrices in order: gradients / sources,
  void* mom[DA_STAGE_MATS];         // momentum buffers (muon), updated in place,
  void* dst[DA_STAGE_MATS];         // destinations (for xtab, or of the result itself where wide is null)
  int g_dtype, m_dtype, w_dtype;
  float mu;
  int nesterov, muon;
  // control memory of the launch behind this one: `nzero` ints to clear and a word that receives `preset`
  int* zero;
  int nzero;
  int* status;
  int preset;
};

struct DaUnstage {
  DaPtrTable x;      // destinations (rows x cols, row pitch ld)
  const void* wide;  // [batch][mw][ldw], of which the min(rows, cols) x max(rows, cols) corner is used
  int batch, rows, cols, ld;
  int mw, ldw;
  int x_dtype, w_dtype;
  float decay, step;
  int muon;
  // Stand-alone weight update: the orthogonalised matrices are wtab.p[b] (rows x cols, contiguous, source
  // orientation) instead of the batch `wide`.
  int use_wtab;
  DaPtrTable wtab;
  // Optional device word: if it is non-zero when the kernel runs, the working matrices are invalid (the launch that
  // made them gave up) and every result element is written as NaN.
  const int* poison;
};

int da_stage_tiles(int rows, int cols, int mw, int nw);
int da_stage(const DaStage& d, hipStream_t s);
// W <- W / (||W||_F + eps), the norm from `tiles` partial sums of squares per matrix
int da_normalize(void* wide, int w_dtype, long long per_matrix, int batch, const float* partials, int tiles, float eps,
                 hipStream_t s);
int da_unstage(const DaUnstage& d, hipStream_t s);
// Conditional poisoning of up to DA_MAX_UPLOADS pointer tables (numel[k] contiguous elements per matrix of table k).
constexpr int DA_MAX_UPLOADS = 6;
struct DaPtrUploads {
  DaPtrTable t[DA_MAX_UPLOADS];
  int n[DA_MAX_UPLOADS];
};
struct DaPoisonShape {
  long long numel[DA_MAX_UPLOADS];
  int f32;
};
// If *flag != 0 when the kernel runs, every element of the matrices becomes NaN.
int da_poison_multi_if(const DaPtrUploads& u, int count, const DaPoisonShape& sh, const int* flag, hipStream_t s);
