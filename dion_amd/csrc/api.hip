// C ABI entry points (declared in include/dion_amd.h) and the host-side drivers that chain
// the kernels of one Newton-Schulz / Muon bucket on a stream.
#include "../../include/dion_amd.h"
#include "common.h"
#include <cstdlib>
#include <cstring>
#include <mutex>
#include "elementwise.h"
#include "prof.h"
#include "dion.h"
#include "ns_flow.h"
#include "ns_small.h"
#include "dion_small.h"

namespace {

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Workspace carve-up for one chunk of `cb` wide matrices (mw x nw).
// Row pitch of a working matrix with n columns.  A pitch that is a multiple of 4 KiB puts every row
// of an operand tile on the same L2 channel (measured: 4096-wide bf16 operands run 17 % slower than
// with 128 bytes of padding), so such rows get 128 bytes more.
inline int padded_pitch(int n, size_t esz) { return ((size_t)n * esz) % 4096 == 0 ? n + (int)(128 / esz) : n; }

inline int round_up(int x, int g) { return (x + g - 1) / g * g; }

// Working dimension of a bf16 product of the batched kernels.  Padding is exact (zero rows and columns go through the
// iteration unchanged) and buys the K loop without bounds checks: with the padding done inside the staging and update
// passes instead of on copies, a Muon step over 14 matrices of 1021, 341 and 2731 rows / columns 1.45 -> 0.85 ms.  Whole
// 256-tiles where that costs at most 7 % more than whole 128-tiles.
inline int padded_dim(int x) {
  const int r128 = round_up(x, 128), r256 = round_up(x, 256);
  return r256 * 100LL <= r128 * 107LL ? r256 : r128;
}

// Whether the working matrices of m x n matrices are padded to whole tiles: not where that makes them more than 1.7 times as
// large (a thin matrix: the factors of a low-rank adapter).  Those keep the 8-element grid and the K loop with bounds checks,
// as their passes over memory cost more than that loop.  Muon steps, us, 8-grid : padded, by how much the padding adds:
//   x 8     224 of 16 x 4096 and of 4096 x 16   1203 : 2194 (workspace 115 : 939 MiB)     256 of 8 x 8192 (x 16)  1284 : 2456
//   x 2     224 of 64 x 4096 and of 4096 x 64   1794 : 2312 (462 : 939)                   128 of 136 x 4096 (x 1.88)  1285 : 1418
//   x 1.78  512 of 72 x 1024   655 : 753
//   x 1.64  512 of 200 x 200   720 : 631, 256 of 300 x 300   834 : 947      x 1.45  96 of 264 x 2048   1128 : 1143
//   x 1.36  24 of 1096 x 1096  1689 : 1188                                   x 1.21  4 of 648 x 10000   1388 : 1048
inline bool padding_pays(int mw, int nw) {
  return (double)padded_dim(mw) * padded_dim(nw) <= 1.7 * round_up(mw, 8) * (double)round_up(nw, 8);
}

// Whether the buckets of one grouped call all go to whole 256-tiles: a grouped product runs 256-tiles only where every member
// has them, so one member on the 128-grid costs all of them a third more per multiply-add.  (14 of 2368 x 2368 and 7 each of
// 7040 x 2368 and 2368 x 7040 with 14 of 789 x 2368, padded to 896: 22.0 ms, padded to 1024: 17.3 ms.)
template <typename Bucket, typename Count>
bool grid256(const Bucket* k, int n, Count count) {
  double nat = 0.0, big = 0.0;
  bool on = false, off = false;
  for (int i = 0; i < n; ++i) {
    const int mw = k[i].m < k[i].n ? k[i].m : k[i].n, nw = k[i].m < k[i].n ? k[i].n : k[i].m;
    if (!padding_pays(mw, nw)) continue;   // (on the 8-grid whatever the others do, and in launches of their own)
    auto cost = [&](double a, double b) { return count(k[i]) * a * a * (3.0 * b + a); };
    const int am = padded_dim(mw), an = padded_dim(nw), bm = round_up(mw, 256), bn = round_up(nw, 256);
    (am == bm && an == bn ? on : off) = true;
    nat += cost(am, an);
    big += cost(bm, bn);
  }
  return on && off && big <= 1.33 * nat;
}

// Whether the one-launch kernel for small matrices has little enough work with these buckets (`count` of each).  Matrices are
// dealt to eight queues of one XCD's workgroups each; what counts is the longest queue, in 64 x 64 x 64 stages per iteration.
// Measured against the batched launches (us per call), below the line: 912 stages (16 x 256 x 1024) 148 : 208, 1088 (512 x 512)
// 131 : 191, 1888 (512 x 1024) 173 : 222, 2280 (40 x 256 x 1024) 247 : 251, 2480 (320 x 128 x 512) 529 : 744; above it:
// 2688 (512 x 1536) 216 : 255, 2736 (48 x 256 x 1024) 262 : 259, 2880 (160 x 256 x 256) 365 : 502, 3488 (512 x 2048) 267 : 286,
// 3600 (768 x 768) 296 : 248, 3648 (64 x 256 x 1024) 341 : 278.  The line is on the safe side: the roads cross at 2700 at the
// earliest (many matrices of a middling size) and by 3600 for all.
template <typename Bucket, typename Count>
bool small_enough(const Bucket* k, int n, Count count) {
  double load[8] = {0}, worst = 0;
  int first = 0;
  for (int i = 0; i < n; ++i) {
    const int mw = round_up(k[i].m < k[i].n ? k[i].m : k[i].n, DA_SMALL_BT) / DA_SMALL_BT;
    const int nw = round_up(k[i].m < k[i].n ? k[i].n : k[i].m, DA_SMALL_BT) / DA_SMALL_BT;
    const double sym = 0.5 * mw * (mw + 1), stages = sym * nw + sym * mw + (double)mw * nw * mw;
    for (int j = 0; j < count(k[i]); ++j) load[(first + j) & 7] += stages;
    first = (first + count(k[i])) & 7;
  }
  for (int q = 0; q < 8; ++q) worst = load[q] > worst ? load[q] : worst;
  return worst <= 2500.0;
}

constexpr size_t FLOW_TAIL_BYTES = 1536;   // behind the counters of a control area: ticket, owner and status words

// The grid of the working matrices' dimensions: whole tiles of the batched products where padding pays, whole 64-tiles (the
// one-launch kernel for small matrices, ns_small.hip), whole 256-tiles where padding pays (see grid256), or 16-byte chunks only.
enum NsGrid { NS_TILES, NS_TILES64, NS_TILES256, NS_CHUNKS };

struct NsLayout {
  int mw = 0, nw = 0, tiles = 0;
  int ldx = 0, lda = 0;   // row pitches of the mw x nw iterates and of the mw x mw Gram / polynomial
  size_t esz = 0;
  size_t x_bytes = 0, a_bytes = 0, part_bytes = 0, flow_bytes = 0;  // per matrix
  size_t per_matrix = 0;
  NsLayout() {}
  NsLayout(int m, int n, int dtype, NsGrid grid = NS_TILES) {
    mw = m < n ? m : n;
    nw = m < n ? n : m;
    if (dtype == DA_BF16 && grid == NS_TILES64) { mw = round_up(mw, DA_SMALL_BT); nw = round_up(nw, DA_SMALL_BT); }
    else if (dtype != DA_BF16 || grid == NS_CHUNKS || !padding_pays(mw, nw)) { mw = round_up(mw, 8); nw = round_up(nw, 8); }
    else if (grid == NS_TILES256) { mw = round_up(mw, 256); nw = round_up(nw, 256); }
    else { mw = padded_dim(mw); nw = padded_dim(nw); }
    tiles = da_stage_tiles(m, n, mw, nw);
    esz = dtype == DA_BF16 ? 2 : 4;
    // no padding between matrices: with every pitch a multiple of 8 each one starts 16-byte aligned
    ldx = padded_pitch(nw, esz);
    lda = padded_pitch(mw, esz);
    x_bytes = (size_t)mw * ldx * esz;
    a_bytes = (size_t)mw * lda * esz;
    part_bytes = align_up((size_t)tiles * sizeof(float), 256);
    // control words of the persistent Newton-Schulz kernels: cb * flow_bytes >= da_ns_flow_ctl_bytes(cb) for cb >= 1
    // (+ 16: one slot of the table of weight pointers that the last product's epilogue updates)
    flow_bytes = DA_FLOW_CTR_STRIDE * sizeof(int) + FLOW_TAIL_BYTES + 16;
    static_assert(DA_SMALL_CTR_STRIDE <= DA_FLOW_CTR_STRIDE && DA_SMALL_TAIL * sizeof(int) + 128 <= FLOW_TAIL_BYTES,
                  "the control area serves both");
    per_matrix = 2 * x_bytes + 2 * a_bytes + part_bytes + flow_bytes;
  }
  int chunk(int batch, size_t ws_bytes) const {
    size_t c = ws_bytes / per_matrix;
    if (c > (size_t)batch) c = batch;
    if (c > DA_MAX_PTRS) c = DA_MAX_PTRS;
    return (int)c;
  }
  // whole tiles in both dimensions: the products of such matrices share launches without bounds checks
  bool whole_tiles() const { return mw % 128 == 0 && nw % 128 == 0; }
};

// Recommended workspace for a bucket: 4 GiB of matrices at most, and room for the layout of the one-launch kernel (whole
// 64-tiles, which a thin matrix does not have otherwise) where that kernel would take as many matrices at a time.
size_t ns_workspace_bytes(int batch, int m, int n, int dtype) {
  const NsLayout L(m, n, dtype);
  size_t c = ((size_t)4 << 30) / L.per_matrix;
  if (c < 1) c = 1;
  if (c > (size_t)batch) c = batch;
  if (c > DA_MAX_PTRS) c = DA_MAX_PTRS;
  size_t bytes = c * L.per_matrix;
  struct { int m, n; } shape = {m, n};
  if (dtype == DA_BF16 && small_enough(&shape, 1, [&](const decltype(shape)&) { return (int)c; })) {
    const size_t small = align_up(NsLayout(m, n, dtype, NS_TILES64).per_matrix * c, 256);
    bytes = bytes > small ? bytes : small;
  }
  return bytes;
}

struct NsBuffers {
  char *x0 = nullptr, *x1 = nullptr, *a = nullptr, *b = nullptr;
  float* partials = nullptr;
  int* flow = nullptr;
  void** xtab = nullptr;   // per-matrix destinations (the last product stores or updates them itself)
  NsBuffers() {}
  NsBuffers(const NsLayout& L, void* ws, int cb) {
    char* p = static_cast<char*>(ws);
    x0 = p; p += L.x_bytes * cb;
    x1 = p; p += L.x_bytes * cb;
    a = p; p += L.a_bytes * cb;
    b = p; p += L.a_bytes * cb;
    partials = reinterpret_cast<float*>(p); p += L.part_bytes * cb;
    flow = reinterpret_cast<int*>(p);
    xtab = reinterpret_cast<void**>(p + (DA_FLOW_CTR_STRIDE * sizeof(int) + FLOW_TAIL_BYTES) * (size_t)cb);
  }
};

// Executed multiply-adds of one launch (symmetric outputs: upper triangle incl. diagonal).
double gemm_flops(const GemmDesc& d) {
  const double mn = d.symmetric ? 0.5 * (double)d.M * ((double)d.M + 1.0) : (double)d.M * d.N;
  return 2.0 * mn * d.K * d.batch;
}

int gemm_any(const GemmDesc& d, int dtype, hipStream_t s, int kind = DA_PROF_GEMM) {
  DaProfScope prof(kind, gemm_flops(d), s);
  return dtype == DA_BF16 ? da_gemm_bf16(d, s) : da_gemm_f32(d, s);
}

// `n` products of the same form: one grouped launch in bf16, one launch each in fp32.
int gemm_group(const GemmDesc* d, int n, int dtype, hipStream_t s, int kind) {
  double flops = 0.0;
  for (int i = 0; i < n; ++i) flops += gemm_flops(d[i]);
  static const bool nogroup = getenv("DION_AMD_NO_GROUP") != nullptr;
  if (dtype == DA_BF16 && !nogroup) {
    DaProfScope prof(kind, flops, s);
    return da_gemm_bf16_grouped(d, n, s);
  }
  for (int i = 0; i < n; ++i) {
    const int rc = gemm_any(d[i], dtype, s, kind);
    if (rc) return rc;
  }
  return DA_OK;
}

// One set of wide matrices iterated together with others: `cb` matrices of layout L in buffers W.
struct NsSet {
  NsLayout L;
  NsBuffers W;
  int cb = 0;
  // Muon: the last X' = aX + BX does not store its result but applies it to the weights W.xtab[b] (x_dtype, rows x
  // cols as the optimizer holds them: transposed with respect to the wide working matrix when tall)
  int update = 0, x_dtype = 0, tall = 0, x_ld = 0;
  float decay = 1.f, step = 1.f;
};

// steps x { A = X X^T ; B = b A + c A A ; X' = a X + B X } on up to DA_MAX_GROUPS sets of wide
// matrices at once (each of the three products is one grouped launch over all sets).
// Returns in result[i] which of x0 / x1 of set i holds the final iterate, and in *poison (if asked for) a device word
// that is non-zero when the iterates are invalid (null: there is no such word).  With `updated` given and every set
// carrying its weight table, the last product applies the weight update itself where its launch allows that
// (*updated = true: result[] then holds nothing of use and the caller skips its own update pass).
int ns_iterate(const NsSet* sets, int nsets, int dtype, const float* coeffs, int steps, int faithful, hipStream_t s,
               char** result, const int** poison = nullptr, bool* updated = nullptr) {
  if (nsets < 1 || nsets > DA_MAX_GROUPS) return DA_ERR_ARG;
  if (poison) *poison = nullptr;
  if (updated) *updated = false;
  bool want_update = updated != nullptr && dtype == DA_BF16 && steps >= 1;
  for (int i = 0; i < nsets; ++i) want_update = want_update && sets[i].update;
  if (dtype == DA_BF16 && steps >= 1) {
    // many small matrices: all iterations of all sets as one persistent launch (ns_flow.hip); the sets are dealt to
    // its queues most expensive first
    DaNsFlowGroup fg[DA_MAX_GROUPS];
    int order[DA_MAX_GROUPS];
    for (int i = 0; i < nsets; ++i) order[i] = i;
    auto cost = [&](int i) { const NsLayout& L = sets[i].L; return (double)L.mw * L.mw * (3.0 * L.nw + L.mw); };
    for (int i = 1; i < nsets; ++i)
      for (int j = i; j > 0 && cost(order[j - 1]) < cost(order[j]); --j) { const int t = order[j]; order[j] = order[j - 1]; order[j - 1] = t; }
    for (int k = 0; k < nsets; ++k) {
      const NsLayout& L = sets[order[k]].L;
      const NsBuffers& W = sets[order[k]].W;
      const NsSet& S = sets[order[k]];
      fg[k] = DaNsFlowGroup{W.x0, W.x1, W.a, W.b, (long long)(L.x_bytes / L.esz), (long long)(L.a_bytes / L.esz),
                            L.mw, L.nw, L.ldx, L.lda, S.cb, W.flow,
                            want_update ? W.xtab : nullptr, S.x_dtype, S.x_ld, S.tall, S.decay, S.step};
    }
    // (the persistent kernel updates bf16 weights only: others get the separate pass)
    bool flow_update = want_update;
    for (int i = 0; i < nsets; ++i) flow_update = flow_update && sets[i].x_dtype == DA_BF16;
    if (!flow_update)
      for (int k = 0; k < nsets; ++k) fg[k].upd_tab = nullptr;
    if (da_ns_flow_applicable(fg, nsets, steps, faithful)) {
      double flops = 0.0;
      for (int i = 0; i < nsets; ++i) {
        const NsLayout& L = sets[i].L;
        flops += (double)steps * sets[i].cb * ((double)L.mw * (L.mw + 1.0) * (L.nw + L.mw) + 2.0 * L.mw * L.mw * L.nw);
      }
      DaProfScope prof(DA_PROF_NS_FLOW, flops, s);
      const int rc = da_ns_flow(fg, nsets, coeffs, steps, faithful, s);
      if (rc) return rc;
      for (int i = 0; i < nsets; ++i) result[i] = (steps & 1) ? sets[i].W.x1 : sets[i].W.x0;
      if (poison) *poison = da_ns_flow_status_word(fg);
      if (flow_update) *updated = true;
      return DA_OK;
    }
  }
  char *x[DA_MAX_GROUPS], *y[DA_MAX_GROUPS];
  for (int i = 0; i < nsets; ++i) { x[i] = sets[i].W.x0; y[i] = sets[i].W.x1; }
  for (int it = 0; it < steps; ++it) {
    const float a = coeffs[3 * it], b = coeffs[3 * it + 1], c = coeffs[3 * it + 2];
    GemmDesc g[DA_MAX_GROUPS];
    // A = X X^T   (symmetric output, k = nw)
    for (int i = 0; i < nsets; ++i) {
      const NsLayout& L = sets[i].L;
      const NsBuffers& W = sets[i].W;
      const long long sx = (long long)(L.x_bytes / L.esz), sa = (long long)(L.a_bytes / L.esz);
      g[i] = GemmDesc{};
      g[i].batch = sets[i].cb; g[i].c_dtype = dtype; g[i].faithful = faithful;
      g[i].A = x[i]; g[i].B = x[i]; g[i].C = W.a; g[i].E = nullptr;
      g[i].sA = sx; g[i].sB = sx; g[i].sC = sa; g[i].sE = 0;
      g[i].lda = L.ldx; g[i].ldb = L.ldx; g[i].ldc = L.lda; g[i].lde = 0;
      g[i].M = L.mw; g[i].N = L.mw; g[i].K = L.nw;
      g[i].a_kstrided = 0; g[i].b_kstrided = 0; g[i].symmetric = 1;
      g[i].epilogue = DA_EPI_STORE; g[i].s0 = 0.f; g[i].s1 = 1.f;
    }
    int rc = gemm_group(g, nsets, dtype, s, DA_PROF_NS_SYRK);
    if (rc) return rc;
    // B = b A + c A A^T   (A symmetric, so A A = A A^T: both operands k-contiguous)
    for (int i = 0; i < nsets; ++i) {
      const NsLayout& L = sets[i].L;
      const NsBuffers& W = sets[i].W;
      const long long sa = (long long)(L.a_bytes / L.esz);
      g[i].A = W.a; g[i].B = W.a; g[i].C = W.b; g[i].E = W.a;
      g[i].sA = sa; g[i].sB = sa; g[i].sC = sa; g[i].sE = sa;
      g[i].lda = L.lda; g[i].ldb = L.lda; g[i].ldc = L.lda; g[i].lde = L.lda;
      g[i].M = L.mw; g[i].N = L.mw; g[i].K = L.mw;
      g[i].epilogue = DA_EPI_AXPBY; g[i].s0 = b; g[i].s1 = c;
    }
    rc = gemm_group(g, nsets, dtype, s, DA_PROF_NS_POLY);
    if (rc) return rc;
    // X' = a X + B X   (B symmetric: k-contiguous; X is the k-strided operand)
    for (int i = 0; i < nsets; ++i) {
      const NsLayout& L = sets[i].L;
      const NsBuffers& W = sets[i].W;
      const long long sx = (long long)(L.x_bytes / L.esz), sa = (long long)(L.a_bytes / L.esz);
      g[i].A = W.b; g[i].B = x[i]; g[i].C = y[i]; g[i].E = x[i];
      g[i].sA = sa; g[i].sB = sx; g[i].sC = sx; g[i].sE = sx;
      g[i].lda = L.lda; g[i].ldb = L.ldx; g[i].ldc = L.ldx; g[i].lde = L.ldx;
      g[i].M = L.mw; g[i].N = L.nw; g[i].K = L.mw;
      g[i].a_kstrided = 0; g[i].b_kstrided = 1; g[i].symmetric = 0;
      g[i].epilogue = DA_EPI_AXPBY; g[i].s0 = a; g[i].s1 = 1.f;
    }
    const int plan = want_update && it + 1 == steps ? da_gemm_bf16_group_plan(g, nsets) : 0;
    if (plan > 0 && (plan & 1)) {
      for (int i = 0; i < nsets; ++i) {
        g[i].tile = plan - 1;
        g[i].upd_tab = sets[i].W.xtab; g[i].upd_dtype = sets[i].x_dtype; g[i].upd_ld = sets[i].x_ld;
        g[i].upd_transposed = sets[i].tall; g[i].upd_decay = sets[i].decay; g[i].upd_step = sets[i].step;
      }
      *updated = true;
    }
    rc = gemm_group(g, nsets, dtype, s, DA_PROF_NS_AXPY);
    if (rc) return rc;
    for (int i = 0; i < nsets; ++i) { char* t = x[i]; x[i] = y[i]; y[i] = t; }
  }
  for (int i = 0; i < nsets; ++i) result[i] = x[i];
  return DA_OK;
}

// A bucket of same-shape matrices (m x n, at most DA_MAX_GROUPS of them per call of ns_jobs): sources G (row pitch ldg),
// momentum M (null: plain cast), destinations X (row pitch ldx): the weights to update, or the result (update == 0).
struct NsJob {
  const void* const* G;
  void* const* M;
  void* const* X;
  int cnt, m, n, ldg, ldx;
  float decay, step;
};
struct NsCall {
  int x_dtype, g_dtype, compute_dtype;   // momentum has the weights' dtype
  int update;                            // 1: Muon step, 0: Newton-Schulz of the sources
  float mu;
  int nesterov;
  const float* coeffs;
  int steps;
  float eps;
  int faithful;
  NsGrid grid;                           // NS_TILES, or NS_CHUNKS for a workspace that holds no padded matrix
};

// The iterations of `n` of the staged and normalised sets, and what becomes of their results.
int ns_finish(const NsJob* jobs, const NsSet* sets, const int* order, int n, const NsCall& c, hipStream_t s) {
  const double xsz = c.x_dtype == DA_BF16 ? 2 : 4;
  NsSet part[DA_MAX_GROUPS];
  // The last product updates the weights in its epilogue where it has whole tiles of them; otherwise (and for a plain
  // result) a pass of its own follows.
  bool whole = c.update != 0;
  for (int i = 0; i < n; ++i) {
    part[i] = sets[order[i]];
    const NsJob& k = jobs[order[i]];
    const int mt = k.m < k.n ? k.m : k.n, nt = k.m < k.n ? k.n : k.m;
    whole = whole && part[i].L.mw == mt && part[i].L.nw == nt && (k.ldx & 7) == 0;
  }
  char* res[DA_MAX_GROUPS];
  const int* poison = nullptr;
  bool updated = false;
  int rc = ns_iterate(part, n, c.compute_dtype, c.coeffs, c.steps, c.faithful, s, res, &poison, whole ? &updated : nullptr);
  if (rc) return rc;
  if (updated && poison) {
    // a persistent launch that updated the weights itself: NaN in all of them if it gave up
    DaPtrUploads up{};
    DaPoisonShape shape{};
    shape.f32 = c.x_dtype == DA_F32;
    int count = 0;
    for (int i = 0; i < n; ++i) {
      const NsJob& k = jobs[order[i]];
      for (int j0 = 0; j0 < k.cnt; j0 += DA_MAX_PTRS) {
        const int cnt = k.cnt - j0 < DA_MAX_PTRS ? k.cnt - j0 : DA_MAX_PTRS;
        for (int j = 0; j < cnt; ++j) up.t[count].p[j] = k.X[j0 + j];
        up.n[count] = cnt;
        shape.numel[count] = (long long)k.m * k.n;
        if (++count == DA_MAX_UPLOADS) {
          rc = da_poison_multi_if(up, count, shape, poison, s);
          if (rc) return rc;
          count = 0;
        }
      }
    }
    return count ? da_poison_multi_if(up, count, shape, poison, s) : DA_OK;
  }
  for (int i = 0; i < n && !updated; ++i) {
    const NsJob& k = jobs[order[i]];
    const NsLayout& L = part[i].L;
    for (int j0 = 0; j0 < k.cnt; j0 += DA_MAX_PTRS) {
      const int cnt = k.cnt - j0 < DA_MAX_PTRS ? k.cnt - j0 : DA_MAX_PTRS;
      DaUnstage us{};
      for (int j = 0; j < cnt; ++j) us.x.p[j] = k.X[j0 + j];
      us.wide = res[i] + (size_t)j0 * L.x_bytes;
      us.batch = cnt; us.rows = k.m; us.cols = k.n; us.ld = k.ldx; us.mw = L.mw; us.ldw = L.ldx;
      us.x_dtype = c.x_dtype; us.w_dtype = c.compute_dtype;
      us.decay = k.decay; us.step = k.step; us.muon = c.update;
      us.poison = poison;
      // algorithmic bytes: read X (update only) and the result, write X
      DaProfScope prof(DA_PROF_UNSTAGE, (double)k.m * k.n * ((c.update ? 2 : 1) * xsz + L.esz) * cnt, s);
      rc = da_unstage(us, s);
      if (rc) return rc;
    }
  }
  return DA_OK;
}

// Whether the one-launch kernel for small matrices takes these jobs.
bool ns_small_wanted(const NsJob* jobs, int nj, const NsCall& c, size_t workspace_bytes) {
  if (c.compute_dtype != DA_BF16 || !c.faithful || c.steps < 1 || c.steps > DA_SMALL_MAX_STEPS) return false;
  if (da_ns_flow_mode() >= 0) return false;   // the caller chose between the other two
  if (!small_enough(jobs, nj, [](const NsJob& k) { return k.cnt; })) return false;
  // (a workspace sized by the queries holds this layout; a smaller one that holds the other takes the batched launches)
  size_t need = 0;
  for (int i = 0; i < nj; ++i)
    need += align_up(NsLayout(jobs[i].m, jobs[i].n, c.compute_dtype, NS_TILES64).per_matrix * (size_t)jobs[i].cnt, 256);
  return need <= workspace_bytes;
}

int ns_jobs(const NsJob* jobs, int nj, const NsCall& c, void* workspace, size_t workspace_bytes, hipStream_t s) {
  if (nj < 1 || nj > DA_MAX_GROUPS) return DA_ERR_ARG;
  const bool small = ns_small_wanted(jobs, nj, c, workspace_bytes);
  const bool all256 = grid256(jobs, nj, [](const NsJob& k) { return k.cnt; });
  // carve the workspace: every job keeps all of its matrices resident
  NsSet sets[DA_MAX_GROUPS];
  char* p = static_cast<char*>(workspace);
  int total = 0;
  for (int i = 0; i < nj; ++i) {
    const NsJob& k = jobs[i];
    NsSet& S = sets[i];
    S.L = NsLayout(k.m, k.n, c.compute_dtype, small ? NS_TILES64 : (all256 ? NS_TILES256 : c.grid));
    S.W = NsBuffers(S.L, p, k.cnt);
    S.cb = k.cnt;
    S.update = c.update; S.x_dtype = c.x_dtype; S.tall = k.m > k.n ? 1 : 0; S.x_ld = k.ldx; S.decay = k.decay; S.step = k.step;
    p += align_up(S.L.per_matrix * (size_t)k.cnt, 256);
    total += k.cnt;
  }
  int* ctl = nullptr;
  if (small) {
    // control words of all jobs in one piece: a single job's own area, else behind the last job, in the room that the
    // jobs' areas leave (FLOW_TAIL_BYTES and more per matrix, of which 8 bytes are used)
    ctl = sets[0].W.flow;
    if (nj > 1) {
      char* q = static_cast<char*>(workspace);
      for (int i = 0; i < nj; ++i) {
        NsSet& S = sets[i];
        S.W = NsBuffers(S.L, q, jobs[i].cnt);
        S.W.xtab = reinterpret_cast<void**>(S.W.flow);
        q = reinterpret_cast<char*>(S.W.xtab + jobs[i].cnt);
        q = static_cast<char*>(workspace) + align_up((size_t)(q - static_cast<char*>(workspace)), 128);
      }
      ctl = reinterpret_cast<int*>(q);
    }
  }
  const double xsz = c.x_dtype == DA_BF16 ? 2 : 4, gsz = c.g_dtype == DA_BF16 ? 2 : 4;
  // momentum update (or cast), staging in wide orientation, Frobenius partial sums
  for (int i = 0, j0 = 0; i < nj;) {
    DaStage st;
    st.ngroups = 0;
    st.g_dtype = c.g_dtype; st.m_dtype = c.x_dtype; st.w_dtype = c.compute_dtype;
    st.mu = c.mu; st.nesterov = c.nesterov; st.muon = c.update;
    st.zero = nullptr; st.nzero = 0; st.status = nullptr; st.preset = 0;
    if (small && i == 0 && j0 == 0) {
      st.zero = ctl; st.nzero = total * DA_SMALL_CTR_STRIDE + DA_SMALL_TAIL - 32;
      st.status = ctl + st.nzero; st.preset = da_ns_flow_fail() ? 1 : 0;
    }
    int mats = 0;
    double bytes = 0;
    while (i < nj && st.ngroups < DA_MAX_GROUPS && mats < DA_STAGE_MATS) {
      const NsJob& k = jobs[i];
      const NsSet& S = sets[i];
      const int n = k.cnt - j0 < DA_STAGE_MATS - mats ? k.cnt - j0 : DA_STAGE_MATS - mats;
      DaStageGroup& g = st.g[st.ngroups++];
      g.wide = S.W.x0 + (size_t)j0 * S.L.x_bytes;
      g.partials = S.W.partials + (size_t)j0 * S.L.tiles;
      g.xtab = S.W.xtab + j0;
      g.rows = k.m; g.cols = k.n; g.ld = k.ldg;
      g.mw = S.L.mw; g.nw = S.L.nw; g.ldw = S.L.ldx;
      g.cnt = n;
      for (int j = 0; j < n; ++j) {
        st.src[mats + j] = k.G[j0 + j];
        st.mom[mats + j] = k.M ? k.M[j0 + j] : nullptr;
        st.dst[mats + j] = k.X[j0 + j];
      }
      mats += n;
      // algorithmic bytes: read G (and M), write M and the working matrix
      bytes += (double)k.m * k.n * (gsz + (c.update ? 2 * xsz : 0.0) + S.L.esz) * n;
      j0 += n;
      if (j0 == k.cnt) { ++i; j0 = 0; }
    }
    DaProfScope prof(DA_PROF_STAGE, bytes, s);
    const int rc = da_stage(st, s);
    if (rc) return rc;
  }
  if (small) {
    // costliest job first, as the kernel deals them
    DaNsSmallGroup sg[DA_MAX_GROUPS];
    int order[DA_MAX_GROUPS];
    double flops = 0.0;
    for (int i = 0; i < nj; ++i) {
      const NsLayout& L = sets[i].L;
      order[i] = i;
      for (int j = i; j > 0; --j) {
        const NsLayout &A = sets[order[j - 1]].L, &B = sets[order[j]].L;
        if ((double)A.mw * A.mw * (3.0 * A.nw + A.mw) >= (double)B.mw * B.mw * (3.0 * B.nw + B.mw)) break;
        const int t = order[j]; order[j] = order[j - 1]; order[j - 1] = t;
      }
      flops += (double)c.steps * jobs[i].cnt * ((double)L.mw * (L.mw + 1.0) * (L.nw + L.mw) + 2.0 * L.mw * L.mw * L.nw);
    }
    for (int i = 0; i < nj; ++i) {
      const NsJob& k = jobs[order[i]];
      const NsSet& S = sets[order[i]];
      int vec = (k.ldx & 7) == 0;
      for (int j = 0; j < k.cnt; ++j) vec = vec && ((uintptr_t)k.X[j] & 15) == 0;
      sg[i] = DaNsSmallGroup{S.W.x0, S.W.x1, S.W.a, S.W.b, (long long)(S.L.x_bytes / 2), (long long)(S.L.a_bytes / 2),
                             S.L.mw, S.L.nw, S.L.ldx, S.L.lda, k.cnt, S.W.partials, S.L.tiles, S.W.xtab,
                             c.x_dtype, k.m, k.n, k.ldx, c.update, vec, k.decay, k.step};
    }
    DaProfScope prof(DA_PROF_NS_FLOW, flops, s);
    return da_ns_small(sg, nj, c.coeffs, c.steps, c.eps, ctl, s);
  }
  for (int i = 0; i < nj; ++i) {
    const NsLayout& L = sets[i].L;
    DaProfScope prof(DA_PROF_NORMALIZE, 2.0 * (double)jobs[i].m * jobs[i].n * L.esz * jobs[i].cnt, s);  // (padding excluded)
    const int rc = da_normalize(sets[i].W.x0, c.compute_dtype, (long long)(L.x_bytes / L.esz), jobs[i].cnt, sets[i].W.partials,
                                L.tiles, c.eps, s);
    if (rc) return rc;
  }
  // Matrices in whole tiles and others in launches of their own: one member that needs the checked K loop puts it on all
  // of a grouped launch (and keeps the persistent kernel and the update in the last epilogue from all of them).
  int order[DA_MAX_GROUPS], nwhole = 0;
  for (int pass = 0, k = 0; pass < 2; ++pass)
    for (int i = 0; i < nj; ++i)
      if ((c.compute_dtype != DA_BF16 || sets[i].L.whole_tiles()) == (pass == 0)) { order[k++] = i; nwhole += pass == 0; }
  if (nwhole) {
    const int rc = ns_finish(jobs, sets, order, nwhole, c, s);
    if (rc) return rc;
  }
  return nwhole < nj ? ns_finish(jobs, sets, order + nwhole, nj - nwhole, c, s) : DA_OK;
}

// 16-byte alignment of matrices on the 8-element grid (`chunks`); others need their elements' alignment: the staging and
// update passes look at the addresses and move such matrices with unaligned accesses.
inline bool misaligned(const void* p, bool chunks, size_t esz) { return ((uintptr_t)p & (chunks ? 15 : esz - 1)) != 0; }

bool dtype_ok(int d) { return d == DA_BF16 || d == DA_F32; }

// Run-time options (dion_amd_set_option).  -1: not set by the caller, the environment decides.
std::atomic<int> g_opt_fused_update{-1};

// Dion's error feedback and weight update, bf16 momentum: 1 as one pass over M and X where that applies, 0 as two AXPBY products,
// -1 (nobody asked for either) by one_pass_update.
// All give the same bits (dion_fused.hip uses the 32x32x16 instruction, the products 16x16x32, which form the same sums).
int update_form() {
  const int v = g_opt_fused_update.load(std::memory_order_relaxed);
  if (v >= 0) return v != 0;
  static const bool env_off = getenv("DION_AMD_NO_FUSED") != nullptr;
  return env_off ? 0 : -1;
}

// The form nobody asked for: one pass, or (false) both products in one launch, with fp32 weights one after the other.  `beside`:
// other buckets' launches run on other streams, and the pass's workgroups, one to a CU from start to end, keep them waiting.
// us a step, the pass / the products:
//   one bucket, at rank     64             128            256            384            512            1024
//   1 of 8192 x 28672       1123 / 1164    1208 / 1266    1364 / 1468    1612 / 1708    1775 / 1811    3027 / 2938
//   4 of 4096 x 4096        435 / 440      476 / 492      579 / 595      643 / 648      784 / 772      1405 / 1360
//   16 of 2048 x 2048       368 / 372      412 / 421      545 / 551      695 / 680      868 / 861      3039 / 2943
//   2 of 4096 x 14336       602 / 582      654 / 649      807 / 819      971 / 985      1098 / 1092    1994 / 1894
//   2 of 14336 x 4096       571 / 560      617 / 618      769 / 779      942 / 938      1071 / 1064    1975 / 1839
//   (48 of 768 x 768 and 12 of 3072 x 768, ranks 64 to 384: within 1 %)
//   several: a Llama-8B layer at rank 64 1118 / 1095, 256 1523 / 1473, 512 2246 / 2184;  MLP matrices of a Llama-70B layer at rank 128
//   2901 / 2779, 256 3286 / 3314, 512 4640 / 4587;  GPT-small at rank 192 701 / 684, 768 3640 / 3564.
// The shorter the products' sums, the more of their tiles is the trip to memory that the pass has under the next tile's sums.
// fp32 weights (not grouped: two output types): 947 / 970, 422 / 438.
bool one_pass_update(bool x_f32, int r, bool beside) { return x_f32 || (!beside && r < 512); }

// B = M + G inside the launch of P = B Q (the default where it applies) or as a pass of its own.
std::atomic<int> g_opt_fused_bq{-1};
bool fused_bq_enabled() {
  const int v = g_opt_fused_bq.load(std::memory_order_relaxed);
  if (v >= 0) return v != 0;
  static const bool env_off = getenv("DION_AMD_NO_FUSED_BQ") != nullptr;
  return !env_off;
}

// All small buckets together (dion_small.hip): -1 by the amount of work, 0 never, 1 whenever possible.
std::atomic<int> g_opt_dion_small{-1};

// Number of slices (1, 2 or 4) of the inner dimension `mp` for the product R = B^T P (np x r per matrix, `cb`
// matrices): workgroup rounds x 64-deep stages per tile, a 256 x 256 tile costing 4 per stage on a whole CU and a
// 128 x 128 tile 3 on half a CU; a sliced product also pays for writing and adding its fp32 partial sums.  (The times of
// an older K loop than choose_tile's; they stay because the number of slices is the order of the sums.)
int btp_slices(int np, int r, int mp, int cb) {
  int best = 1;
  double best_cost = 0.0;
  for (int s = 1; s <= DA_MAX_GROUPS; s *= 2) {
    if (s > 1 && (mp / s < 512 || mp % (s * 64) != 0)) break;
    const long long t256 = (long long)((np + 255) / 256) * ((r + 255) / 256) * cb * s;
    const long long t128 = (long long)((np + 127) / 128) * ((r + 127) / 128) * cb * s;
    const double stages = (double)(mp / s) / 64.0;
    const double big = np >= 256 && r >= 256 ? (double)((t256 + 255) / 256) * stages * 4.0 : 1e30;
    const double small = (double)((t128 + 511) / 512) * stages * 3.0;
    double cost = big < small ? big : small;
    if (s > 1) cost += 32.0 + 8.0 * s;
    if (s == 1 || cost < best_cost) { best = s; best_cost = cost; }
  }
  return best;
}

}  // namespace

extern "C" {

const char* dion_amd_version(void) { return "dion_amd 0.1 (gfx950)"; }

size_t dion_amd_ns_workspace_bytes(int batch, int m, int n, int compute_dtype) {
  if (batch <= 0 || m <= 0 || n <= 0 || !dtype_ok(compute_dtype)) return 0;
  return ns_workspace_bytes(batch, m, n, compute_dtype);
}

}  // extern "C"

namespace {

int ns_run(const void* G, int g_dtype, long long g_stride, int ldg, void* out, long long out_stride, int ldo,
           int batch, int m, int n, const float* coeffs, int steps, float eps, int compute_dtype, int faithful,
           void* workspace, size_t workspace_bytes, void* stream, NsGrid grid = NS_TILES) {
  if (!G || !out || !coeffs || !workspace || batch <= 0 || m <= 0 || n <= 0 || steps < 0) return DA_ERR_ARG;
  if (!dtype_ok(g_dtype) || !dtype_ok(compute_dtype)) return DA_ERR_DTYPE;
  const size_t gsz = g_dtype == DA_BF16 ? 2 : 4, osz = compute_dtype == DA_BF16 ? 2 : 4;
  if (ldg < n || ldo < n) return DA_ERR_ARG;
  // matrices move as 16-byte chunks where their rows allow that; only the workspace, which the library carves up
  // itself, needs 256
  const bool g_chunks = !((n | ldg) & 7), o_chunks = !((n | ldo) & 7);
  if ((g_chunks && (g_stride & 7)) || (o_chunks && (out_stride & 7))) return DA_ERR_ALIGN;
  if (misaligned(G, g_chunks && !(m & 7), gsz) || misaligned(out, o_chunks && !(m & 7), osz)) return DA_ERR_ALIGN;
  if ((uintptr_t)workspace & 255) return DA_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const NsLayout L(m, n, compute_dtype, grid);
  const int chunk = L.chunk(batch, workspace_bytes);
  if (chunk < 1) return DA_ERR_WORKSPACE;
  const NsCall call = {compute_dtype, g_dtype, compute_dtype, 0, 0.f, 0, coeffs, steps, eps, faithful, grid};
  for (int b0 = 0; b0 < batch; b0 += chunk) {
    const int cb = batch - b0 < chunk ? batch - b0 : chunk;
    const void* src[DA_MAX_PTRS];
    void* dst[DA_MAX_PTRS];
    for (int i = 0; i < cb; ++i) {
      src[i] = static_cast<const char*>(G) + (size_t)(b0 + i) * g_stride * gsz;
      dst[i] = static_cast<char*>(out) + (size_t)(b0 + i) * out_stride * osz;
    }
    const NsJob job = {src, nullptr, dst, cb, m, n, ldg, ldo, 1.f, 1.f};
    const int rc = ns_jobs(&job, 1, call, workspace, workspace_bytes, s);
    if (rc) return rc;
  }
  return DA_OK;
}

// Working memory of dion_amd_newton_schulz_static: one array per GPU, part of the library's device image (it lives
// as long as the process).  Host code never uses the array's name as an address: `static_scratch()` asks the
// runtime for the device address on the current GPU, once per device, and hands that pointer on.
// The announced size is for the matrices: the control words of the one-launch kernels, 1280 bytes a matrix beyond the
// persistent kernel's, come on top.
constexpr size_t SCRATCH_BYTES = DION_AMD_STATIC_SCRATCH_BYTES + FLOW_TAIL_BYTES - 256;
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];
constexpr int DA_MAX_DEVICES = 64;
void* g_scratch_ptr[DA_MAX_DEVICES];
std::mutex g_scratch_mutex;

int static_scratch(void** ptr) {
  int dev = -1;
  DA_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= DA_MAX_DEVICES) return DA_ERR_LIMIT;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    DA_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return DA_ERR_ARG;
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return DA_OK;
}

}  // namespace

extern "C" {

int dion_amd_newton_schulz(const void* G, int g_dtype, long long g_stride, int ldg, void* out, long long out_stride,
                           int ldo, int batch, int m, int n, const float* coeffs, int steps, float eps,
                           int compute_dtype, int faithful, void* workspace, size_t workspace_bytes, void* stream) {
  return ns_run(G, g_dtype, g_stride, ldg, out, out_stride, ldo, batch, m, n, coeffs, steps, eps, compute_dtype,
                faithful, workspace, workspace_bytes, stream);
}

size_t dion_amd_static_scratch_bytes(void) { return DION_AMD_STATIC_SCRATCH_BYTES; }

int dion_amd_newton_schulz_static(const void* G, int g_dtype, long long g_stride, int ldg, void* out,
                                  long long out_stride, int ldo, int batch, int m, int n, const float* coeffs,
                                  int steps, float eps, int compute_dtype, int faithful, void* stream) {
  if (batch <= 0 || m <= 0 || n <= 0) return DA_ERR_ARG;
  if (!dtype_ok(compute_dtype)) return DA_ERR_DTYPE;
  // one matrix's working set must fit the array (a batch then goes through it in chunks): padded to whole tiles, or else
  // without padding (648 x 10000: 32.4 MiB and 26.3)
  NsGrid grid = NS_TILES;
  if (NsLayout(m, n, compute_dtype).per_matrix > SCRATCH_BYTES) grid = NS_CHUNKS;
  if (NsLayout(m, n, compute_dtype, grid).per_matrix > SCRATCH_BYTES) return DA_ERR_LIMIT;
  void* ws = nullptr;
  const int rc = static_scratch(&ws);
  if (rc) return rc;
  return ns_run(G, g_dtype, g_stride, ldg, out, out_stride, ldo, batch, m, n, coeffs, steps, eps, compute_dtype,
                faithful, ws, SCRATCH_BYTES, stream, grid);
}

int dion_amd_syrk(const void* A, long long a_stride, int lda, void* C, long long c_stride, int ldc, int batch, int m,
                  int k, int dtype, void* stream) {
  if (!dtype_ok(dtype)) return DA_ERR_DTYPE;
  GemmDesc g{};
  g.A = A; g.B = A; g.C = C; g.E = nullptr;
  g.sA = a_stride; g.sB = a_stride; g.sC = c_stride;
  g.lda = lda; g.ldb = lda; g.ldc = ldc;
  g.M = m; g.N = m; g.K = k; g.batch = batch;
  g.symmetric = 1; g.epilogue = DA_EPI_STORE; g.s1 = 1.f; g.faithful = 0; g.c_dtype = dtype;
  return gemm_any(g, dtype, static_cast<hipStream_t>(stream));
}

int dion_amd_sym_poly(const void* A, long long a_stride, int lda, void* C, long long c_stride, int ldc, int batch,
                      int m, float alpha, float beta, int dtype, int faithful, void* stream) {
  if (!dtype_ok(dtype)) return DA_ERR_DTYPE;
  if (A == C) return DA_ERR_ARG;  // mirrored stores would race with operand loads
  GemmDesc g{};
  g.A = A; g.B = A; g.C = C; g.E = A;
  g.sA = a_stride; g.sB = a_stride; g.sC = c_stride; g.sE = a_stride;
  g.lda = lda; g.ldb = lda; g.ldc = ldc; g.lde = lda;
  g.M = m; g.N = m; g.K = m; g.batch = batch;
  g.symmetric = 1; g.any_addend = 1; g.epilogue = DA_EPI_AXPBY; g.s0 = beta; g.s1 = alpha; g.faithful = faithful; g.c_dtype = dtype;
  return gemm_any(g, dtype, static_cast<hipStream_t>(stream));
}

int dion_amd_gemm(const void* A, long long a_stride, int lda, int a_kstrided, const void* B, long long b_stride,
                  int ldb, int b_kstrided, void* C, long long c_stride, int ldc, const void* E, long long e_stride,
                  int lde, int batch, int M, int N, int K, int in_dtype, int c_dtype, int epilogue, float s0,
                  float s1, int faithful, void* stream) {
  if (!dtype_ok(in_dtype) || !dtype_ok(c_dtype)) return DA_ERR_DTYPE;
  if (epilogue != DA_EPI_STORE && epilogue != DA_EPI_AXPBY) return DA_ERR_ARG;
  GemmDesc g{};
  g.A = A; g.B = B; g.C = C; g.E = epilogue == DA_EPI_AXPBY ? E : nullptr;
  g.sA = a_stride; g.sB = b_stride; g.sC = c_stride; g.sE = e_stride;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc; g.lde = lde;
  g.M = M; g.N = N; g.K = K; g.batch = batch;
  g.a_kstrided = a_kstrided != 0; g.b_kstrided = b_kstrided != 0; g.symmetric = 0;
  g.epilogue = epilogue; g.s0 = s0; g.s1 = s1; g.faithful = faithful; g.c_dtype = c_dtype;
  return gemm_any(g, in_dtype, static_cast<hipStream_t>(stream));
}

int dion_amd_set_option(const char* name, int value) {
  if (!name) return DA_ERR_ARG;
  if (strcmp(name, "fused_update") == 0) {
    g_opt_fused_update.store(value < 0 ? -1 : (value != 0), std::memory_order_relaxed);
    return DA_OK;
  }
  if (strcmp(name, "fused_bq") == 0) {
    g_opt_fused_bq.store(value < 0 ? -1 : (value != 0), std::memory_order_relaxed);
    return DA_OK;
  }
  if (strcmp(name, "ns_flow") == 0) {
    if (value < -1 || value > 2) return DA_ERR_ARG;
    da_ns_flow_set_mode(value);
    return DA_OK;
  }
  if (strcmp(name, "edge_loop") == 0) {
    da_gemm_bf16_set_edge_loop(value);
    return DA_OK;
  }
  if (strcmp(name, "dion_small") == 0) {
    g_opt_dion_small.store(value < 0 ? -1 : (value != 0), std::memory_order_relaxed);
    return DA_OK;
  }
  if (strcmp(name, "ns_flow_fail") == 0) {
    da_ns_flow_set_fail(value != 0);
    return DA_OK;
  }
  return DA_ERR_ARG;
}

int dion_amd_ns_flow_trace_enable(int on) {
  da_ns_flow_trace_enable(on);
  return DA_OK;
}
int dion_amd_ns_flow_trace_read(void* host_dst, int max_tiles, int* tiles) {
  return da_ns_flow_trace_read(host_dst, max_tiles, tiles);
}

size_t dion_amd_muon_workspace_bytes(int batch, int m, int n) {
  if (batch <= 0 || m <= 0 || n <= 0) return 0;
  return ns_workspace_bytes(batch, m, n, DA_BF16);
}

}  // extern "C"

namespace {
int muon_check(void* const* X, const void* const* G, void* const* M, int batch, int m, int n, int x_dtype, int g_dtype) {
  const bool chunks = ((m | n) & 7) == 0;
  const size_t xsz = x_dtype == DA_BF16 ? 2 : 4, gsz = g_dtype == DA_BF16 ? 2 : 4;
  for (int i = 0; i < batch; ++i) {
    if (!X[i] || !G[i] || !M[i]) return DA_ERR_ARG;
    if (misaligned(X[i], chunks, xsz) || misaligned(G[i], chunks, gsz) || misaligned(M[i], chunks, xsz)) return DA_ERR_ALIGN;
  }
  return DA_OK;
}
}  // namespace

extern "C" {

int dion_amd_muon_step(void* const* X, const void* const* G, void* const* M, int batch, int m, int n, int x_dtype,
                       int g_dtype, float mu, int nesterov, float decay, float adjusted_lr, const float* coeffs,
                       int steps, float eps, int faithful, void* workspace, size_t workspace_bytes, void* stream) {
  if (!X || !G || !M || !coeffs || !workspace || batch <= 0 || m <= 0 || n <= 0 || steps < 0) return DA_ERR_ARG;
  if (!dtype_ok(x_dtype) || !dtype_ok(g_dtype)) return DA_ERR_DTYPE;
  if ((uintptr_t)workspace & 255) return DA_ERR_ALIGN;
  const int rc = muon_check(X, G, M, batch, m, n, x_dtype, g_dtype);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const NsLayout L(m, n, DA_BF16);
  const int chunk = L.chunk(batch, workspace_bytes);
  if (chunk < 1) return DA_ERR_WORKSPACE;
  const NsCall call = {x_dtype, g_dtype, DA_BF16, 1, mu, nesterov, coeffs, steps, eps, faithful, NS_TILES};
  for (int b0 = 0; b0 < batch; b0 += chunk) {
    const NsJob job = {G + b0, M + b0, X + b0, batch - b0 < chunk ? batch - b0 : chunk, m, n, n, n, decay, adjusted_lr};
    const int rc = ns_jobs(&job, 1, call, workspace, workspace_bytes, s);
    if (rc) return rc;
  }
  return DA_OK;
}

int dion_amd_muon_pre(const void* const* G, void* const* M, void* const* U, int batch, int m, int n, int g_dtype,
                      int m_dtype, float mu, int nesterov, void* stream) {
  if (!G || !M || !U || batch <= 0 || m <= 0 || n <= 0) return DA_ERR_ARG;
  if (!dtype_ok(g_dtype) || !dtype_ok(m_dtype)) return DA_ERR_DTYPE;
  const bool chunks = (n & 7) == 0;
  const size_t gsz = g_dtype == DA_BF16 ? 2 : 4, msz = m_dtype == DA_BF16 ? 2 : 4;
  for (int i = 0; i < batch; ++i) {
    if (!G[i] || !M[i] || !U[i]) return DA_ERR_ARG;
    if (misaligned(G[i], chunks, gsz) || misaligned(M[i], chunks, msz) || misaligned(U[i], chunks, 2)) return DA_ERR_ALIGN;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  for (int b0 = 0; b0 < batch; b0 += DA_STAGE_MATS) {
    const int cb = batch - b0 < DA_STAGE_MATS ? batch - b0 : DA_STAGE_MATS;
    DaStage st{};
    for (int i = 0; i < cb; ++i) {
      st.src[i] = G[b0 + i];
      st.mom[i] = M[b0 + i];
      st.dst[i] = U[b0 + i];
    }
    st.ngroups = 1;
    st.g[0].rows = m; st.g[0].cols = n; st.g[0].ld = n; st.g[0].cnt = cb;
    st.g_dtype = g_dtype; st.m_dtype = m_dtype; st.w_dtype = DA_BF16;
    st.mu = mu; st.nesterov = nesterov; st.muon = 1;
    DaProfScope prof(DA_PROF_STAGE, (double)m * n * (gsz + 2 * msz + 2) * cb, s);
    const int rc = da_stage(st, s);
    if (rc) return rc;
  }
  return DA_OK;
}

int dion_amd_muon_post(void* const* X, const void* const* O, int batch, int m, int n, int x_dtype, int o_dtype,
                       float decay, float adjusted_lr, void* stream) {
  if (!X || !O || batch <= 0 || m <= 0 || n <= 0) return DA_ERR_ARG;
  if (!dtype_ok(x_dtype) || !dtype_ok(o_dtype)) return DA_ERR_DTYPE;
  const bool chunks = (n & 7) == 0;
  for (int i = 0; i < batch; ++i) {
    if (!X[i] || !O[i]) return DA_ERR_ARG;
    if (misaligned(X[i], chunks, x_dtype == DA_BF16 ? 2 : 4) || misaligned(O[i], chunks, o_dtype == DA_BF16 ? 2 : 4))
      return DA_ERR_ALIGN;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const double xsz = x_dtype == DA_BF16 ? 2 : 4;
  for (int b0 = 0; b0 < batch; b0 += DA_MAX_PTRS) {
    const int cb = batch - b0 < DA_MAX_PTRS ? batch - b0 : DA_MAX_PTRS;
    DaUnstage us{};
    for (int i = 0; i < cb; ++i) {
      us.x.p[i] = X[b0 + i];
      us.wtab.p[i] = const_cast<void*>(O[b0 + i]);
    }
    us.use_wtab = 1; us.wide = nullptr;
    us.batch = cb; us.rows = m; us.cols = n; us.ld = n; us.ldw = n;
    us.x_dtype = x_dtype; us.w_dtype = o_dtype;
    us.decay = decay; us.step = adjusted_lr; us.muon = 1;
    DaProfScope prof(DA_PROF_UNSTAGE, (double)m * n * (2 * xsz + (o_dtype == DA_BF16 ? 2 : 4)) * cb, s);
    const int rc = da_unstage(us, s);
    if (rc) return rc;
  }
  return DA_OK;
}

int dion_amd_gemm_plan(int M, int N, int K, int lda, int a_kstrided, int ldb, int b_kstrided) {
  if (M <= 0 || N <= 0 || K <= 0 || lda <= 0 || ldb <= 0) return DA_ERR_ARG;
  GemmDesc g{};
  g.M = M; g.N = N; g.K = K; g.lda = lda; g.ldb = ldb; g.batch = 1;
  g.a_kstrided = a_kstrided != 0; g.b_kstrided = b_kstrided != 0;
  return da_gemm_bf16_plan(g);
}

int dion_amd_gemm_group_plan(const int* batch, const int* M, const int* N, const int* K, int n, int a_kstrided, int b_kstrided,
                             int symmetric, int epilogue) {
  if (!batch || !M || !N || !K || n <= 0 || n > DA_MAX_GROUPS) return DA_ERR_ARG;
  GemmDesc g[DA_MAX_GROUPS];
  for (int i = 0; i < n; ++i) {
    if (batch[i] <= 0 || M[i] <= 0 || N[i] <= 0 || K[i] <= 0 || (symmetric && M[i] != N[i])) return DA_ERR_ARG;
    g[i] = GemmDesc{};
    g[i].symmetric = symmetric != 0;
    g[i].batch = batch[i]; g[i].M = M[i]; g[i].N = N[i]; g[i].K = K[i];
    g[i].a_kstrided = a_kstrided != 0; g[i].b_kstrided = b_kstrided != 0;
    g[i].lda = a_kstrided ? M[i] : K[i]; g[i].ldb = b_kstrided ? N[i] : K[i];
    g[i].epilogue = epilogue;
  }
  return da_gemm_bf16_group_plan(g, n);
}

size_t dion_amd_muon_buckets_workspace_bytes(const dion_amd_muon_bucket* buckets, int nbuckets) {
  if (!buckets || nbuckets <= 0) return 0;
  size_t worst = 0;
  for (int r0 = 0; r0 < nbuckets; r0 += DA_MAX_GROUPS) {
    size_t need = 0, need_small = 0;
    const int nr = nbuckets - r0 < DA_MAX_GROUPS ? nbuckets - r0 : DA_MAX_GROUPS;
    const auto count = [](const dion_amd_muon_bucket& k) { return k.batch; };
    for (int i = r0; i < r0 + nr; ++i)
      if (buckets[i].batch <= 0 || buckets[i].m <= 0 || buckets[i].n <= 0) return 0;
    const bool all256 = grid256(buckets + r0, nr, count);
    for (int i = r0; i < r0 + nr; ++i) {
      const dion_amd_muon_bucket& k = buckets[i];
      need += align_up(NsLayout(k.m, k.n, DA_BF16, all256 ? NS_TILES256 : NS_TILES).per_matrix * (size_t)k.batch, 256);
      need_small += align_up(NsLayout(k.m, k.n, DA_BF16, NS_TILES64).per_matrix * (size_t)k.batch, 256);
    }
    if (need > worst) worst = need;
    if (need_small > worst && small_enough(buckets + r0, nr, count)) worst = need_small;
  }
  return worst;
}

int dion_amd_muon_step_buckets(const dion_amd_muon_bucket* buckets, int nbuckets, int x_dtype, int g_dtype, float mu,
                               int nesterov, const float* coeffs, int steps, float eps, int faithful,
                               void* workspace, size_t workspace_bytes, void* stream) {
  if (!buckets || nbuckets <= 0 || !coeffs || !workspace || steps < 0) return DA_ERR_ARG;
  if (!dtype_ok(x_dtype) || !dtype_ok(g_dtype)) return DA_ERR_DTYPE;
  if ((uintptr_t)workspace & 255) return DA_ERR_ALIGN;
  for (int i = 0; i < nbuckets; ++i) {
    const dion_amd_muon_bucket& k = buckets[i];
    if (!k.X || !k.G || !k.M || k.batch <= 0 || k.m <= 0 || k.n <= 0) return DA_ERR_ARG;
    const int rc = muon_check(k.X, k.G, k.M, k.batch, k.m, k.n, x_dtype, g_dtype);
    if (rc) return rc;
  }
  if (workspace_bytes < dion_amd_muon_buckets_workspace_bytes(buckets, nbuckets)) return DA_ERR_WORKSPACE;
  const NsCall call = {x_dtype, g_dtype, DA_BF16, 1, mu, nesterov, coeffs, steps, eps, faithful, NS_TILES};
  for (int r0 = 0; r0 < nbuckets; r0 += DA_MAX_GROUPS) {
    const int nr = nbuckets - r0 < DA_MAX_GROUPS ? nbuckets - r0 : DA_MAX_GROUPS;
    NsJob jobs[DA_MAX_GROUPS];
    for (int i = 0; i < nr; ++i) {
      const dion_amd_muon_bucket& k = buckets[r0 + i];
      jobs[i] = NsJob{k.G, k.M, k.X, k.batch, k.m, k.n, k.n, k.n, k.decay, k.adjusted_lr};
    }
    const int rc = ns_jobs(jobs, nr, call, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
    if (rc) return rc;
  }
  return DA_OK;
}


// ---------------------------------------------------------------------------------------
// Dion
// ---------------------------------------------------------------------------------------
}  // extern "C"

namespace {

struct DionLayout {
  // working orientation: B is mp x np with mp >= np; Q is np x r.  r is the rank rounded up to a multiple
  // of 8 (16-byte rows for every working matrix); the extra columns are zero throughout the step.
  int mp, np, r;
  size_t msz;           // bytes per element of the momentum dtype
  size_t qc, p, rb, qn, orth, sketch, part, small;  // per-matrix byte sizes
  size_t per_matrix;
  DionLayout(int m, int n, int rank, int m_dtype, int sketch_k = 0) {
    mp = m < n ? n : m;
    np = m < n ? m : n;
    r = (rank + 7) & ~7;
    msz = m_dtype == DA_BF16 ? 2 : 4;
    qc = (size_t)np * r * msz;   // exact: the orthonormaliser and the GEMMs take these as
    p = (size_t)mp * r * msz;    // contiguous batches (multiples of 128 bytes by the alignment rule)
    rb = qc;
    qn = qc;
    orth = align_up(da_orth_workspace_bytes(1, mp, r), 256);
    // (a sketched orthonormalisation keeps S P per matrix behind the orthonormaliser's own scratch)
    sketch = sketch_k > 0 ? align_up(da_orth_sketch_extra_bytes(1, sketch_k, r), 256) : 0;
    // fp32 partial sums of R = B^T P when its inner dimension is cut into DA_MAX_GROUPS slices (bf16 only)
    part = m_dtype == DA_BF16 ? (size_t)DA_MAX_GROUPS * np * r * sizeof(float) : 0;
    small = 256;  // flags, info, pointer-table slots
    per_matrix = qc + p + rb + qn + orth + sketch + part + small + 256;
  }
  size_t fixed() const { return 4 * DA_MAX_PTRS * sizeof(void*) + 2 * DA_MAX_PTRS * sizeof(int) + 1024; }
  int chunk(int batch, size_t ws_bytes) const {
    if (ws_bytes < fixed()) return 0;
    size_t c = (ws_bytes - fixed()) / per_matrix;
    if (c > (size_t)batch) c = batch;
    if (c > DA_MAX_PTRS) c = DA_MAX_PTRS;
    return (int)c;
  }
  size_t recommended(int batch) const {
    size_t c = ((size_t)6 << 30) / per_matrix;
    if (c < 1) c = 1;
    if (c > (size_t)batch) c = batch;
    if (c > DA_MAX_PTRS) c = DA_MAX_PTRS;
    return c * per_matrix + fixed();
  }
};

}  // namespace

namespace {
int dion_step_impl(void* const* X, const void* const* G, void* const* M, void* const* Q, int batch, int m, int n,
                   int rank, int x_dtype, int g_dtype, int m_dtype, int q_dtype, float ef_alpha, float decay,
                   float scaled_lr, float eps, int faithful, int power_iters, int qr_method, const void* sketch,
                   int sketch_k, int* info, void* workspace, size_t workspace_bytes, void* stream);
}  // namespace

extern "C" {

int dion_amd_dion_bq_fused(int batch, int m, int n, int rank, int m_dtype, int g_dtype) {
  if (batch <= 0 || m <= 0 || n <= 0 || rank <= 0 || rank > m || rank > n || !dtype_ok(m_dtype) || !dtype_ok(g_dtype)) return 0;
  const DionLayout L(m, n, rank, m_dtype);
  const int cb = batch < DA_MAX_PTRS ? batch : DA_MAX_PTRS;
  return fused_bq_enabled() && da_dion_bq_sum_applicable(cb, L.mp, L.np, L.r, n, m < n ? 1 : 0, m_dtype, g_dtype) ? 1 : 0;
}

size_t dion_amd_dion_workspace_bytes(int batch, int m, int n, int r, int m_dtype) {
  if (batch <= 0 || m <= 0 || n <= 0 || r <= 0 || !dtype_ok(m_dtype)) return 0;
  return DionLayout(m, n, r, m_dtype).recommended(batch);
}

size_t dion_amd_orthonormalize_workspace_bytes(int batch, int rows, int r) {
  if (batch <= 0 || rows <= 0 || r <= 0) return 0;
  return da_orth_workspace_bytes(batch, rows, r) + 256 + (size_t)batch * sizeof(int);
}

int dion_amd_orthonormalize(const void* P, void* out, int dtype, int batch, int rows, int r, int passes,
                            int* info, void* workspace, size_t workspace_bytes, void* stream) {
  return dion_amd_orthonormalize_method(P, out, dtype, batch, rows, r, passes, DA_QR_AUTO, info, workspace,
                                        workspace_bytes, stream);
}

int dion_amd_orthonormalize_method(const void* P, void* out, int dtype, int batch, int rows, int r, int passes,
                                   int qr_method, int* info, void* workspace, size_t workspace_bytes, void* stream) {
  if (!P || !out || !workspace || batch <= 0 || rows <= 0 || r <= 0 || passes < 1 || passes > 3) return DA_ERR_ARG;
  if (qr_method < 0 || qr_method > 2) return DA_ERR_ARG;
  if (!dtype_ok(dtype)) return DA_ERR_DTYPE;
  if (r > rows) return DA_ERR_ARG;
  if (workspace_bytes < dion_amd_orthonormalize_workspace_bytes(batch, rows, r)) return DA_ERR_WORKSPACE;
  if ((uintptr_t)workspace & 255) return DA_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int* inf = info;
  if (!inf) inf = reinterpret_cast<int*>(static_cast<char*>(workspace) + align_up(da_orth_workspace_bytes(batch, rows, r), 256));
  int rc = da_fill_int(inf, batch, 0, s);
  if (rc) return rc;
  DaProfScope prof(DA_PROF_DION_ORTH, 0.0, s);
  return da_orthonormalize(P, out, dtype, batch, rows, r, r, passes, qr_method, workspace, inf, s);
}

size_t dion_amd_orthonormalize_sketch_workspace_bytes(int batch, int rows, int r, int k) {
  if (batch <= 0 || rows <= 0 || r <= 0 || k <= 0) return 0;
  return align_up(dion_amd_orthonormalize_workspace_bytes(batch, rows, r), 256) + da_orth_sketch_extra_bytes(batch, k, r);
}

int dion_amd_orthonormalize_sketch(const void* P, const void* S, void* out, int dtype, int batch, int rows, int r, int k,
                                   int* info, void* workspace, size_t workspace_bytes, void* stream) {
  if (!P || !S || !out || !workspace || batch <= 0 || rows <= 0 || r <= 0 || k < r) return DA_ERR_ARG;
  if (!dtype_ok(dtype)) return DA_ERR_DTYPE;
  if (r > rows) return DA_ERR_ARG;
  // S P runs on the matrix cores of the factor's dtype: 16-byte rows for S, P and the product
  const int grid = dtype == DA_BF16 ? 7 : 3;
  if ((rows | r | k) & grid) return DA_ERR_ALIGN;
  if (workspace_bytes < dion_amd_orthonormalize_sketch_workspace_bytes(batch, rows, r, k)) return DA_ERR_WORKSPACE;
  if ((uintptr_t)workspace & 255) return DA_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  char* base = static_cast<char*>(workspace);
  const size_t own = align_up(dion_amd_orthonormalize_workspace_bytes(batch, rows, r), 256);
  int* inf = info;
  if (!inf) inf = reinterpret_cast<int*>(base + align_up(da_orth_workspace_bytes(batch, rows, r), 256));
  int rc = da_fill_int(inf, batch, 0, s);
  if (rc) return rc;
  DaProfScope prof(DA_PROF_DION_ORTH, 0.0, s);
  return da_orthonormalize_sketch(P, S, out, dtype, batch, rows, r, r, k, workspace, base + own, inf, s);
}

int dion_amd_dion_step(void* const* X, const void* const* G, void* const* M, void* const* Q, int batch, int m, int n,
                       int rank, int x_dtype, int g_dtype, int m_dtype, int q_dtype, float ef_alpha, float decay,
                       float scaled_lr, float eps, int faithful, int power_iters, int* info, void* workspace,
                       size_t workspace_bytes, void* stream) {
  return dion_amd_dion_step_qr(X, G, M, Q, batch, m, n, rank, x_dtype, g_dtype, m_dtype, q_dtype, ef_alpha, decay,
                               scaled_lr, eps, faithful, power_iters, DA_QR_AUTO, info, workspace, workspace_bytes, stream);
}

int dion_amd_dion_step_qr(void* const* X, const void* const* G, void* const* M, void* const* Q, int batch, int m, int n,
                          int rank, int x_dtype, int g_dtype, int m_dtype, int q_dtype, float ef_alpha, float decay,
                          float scaled_lr, float eps, int faithful, int power_iters, int qr_method, int* info,
                          void* workspace, size_t workspace_bytes, void* stream) {
  return dion_step_impl(X, G, M, Q, batch, m, n, rank, x_dtype, g_dtype, m_dtype, q_dtype, ef_alpha, decay, scaled_lr, eps,
                        faithful, power_iters, qr_method, nullptr, 0, info, workspace, workspace_bytes, stream);
}

size_t dion_amd_dion_sketch_workspace_bytes(int batch, int m, int n, int r, int m_dtype, int sketch_k) {
  if (batch <= 0 || m <= 0 || n <= 0 || r <= 0 || sketch_k <= 0 || !dtype_ok(m_dtype)) return 0;
  return DionLayout(m, n, r, m_dtype, sketch_k).recommended(batch);
}

int dion_amd_dion_step_sketch(void* const* X, const void* const* G, void* const* M, void* const* Q, int batch, int m,
                              int n, int rank, int x_dtype, int g_dtype, int m_dtype, int q_dtype, float ef_alpha,
                              float decay, float scaled_lr, float eps, int faithful, int power_iters, const void* sketch,
                              int sketch_k, int* info, void* workspace, size_t workspace_bytes, void* stream) {
  if (!sketch || sketch_k <= 0) return DA_ERR_ARG;
  return dion_step_impl(X, G, M, Q, batch, m, n, rank, x_dtype, g_dtype, m_dtype, q_dtype, ef_alpha, decay, scaled_lr, eps,
                        faithful, power_iters, DA_QR_AUTO, sketch, sketch_k, info, workspace, workspace_bytes, stream);
}

}  // extern "C"

namespace {

int dion_step_impl(void* const* X, const void* const* G, void* const* M, void* const* Q, int batch, int m, int n,
                   int rank, int x_dtype, int g_dtype, int m_dtype, int q_dtype, float ef_alpha, float decay,
                   float scaled_lr, float eps, int faithful, int power_iters, int qr_method, const void* sketch,
                   int sketch_k, int* info, void* workspace, size_t workspace_bytes, void* stream) {
  if (qr_method < 0 || qr_method > 2) return DA_ERR_ARG;
  if (!X || !G || !M || !Q || !workspace || batch <= 0 || m <= 0 || n <= 0 || rank <= 0) return DA_ERR_ARG;
  if (power_iters < 1 || power_iters > 64) return DA_ERR_ARG;
  if (!dtype_ok(x_dtype) || !dtype_ok(g_dtype) || !dtype_ok(m_dtype) || !dtype_ok(q_dtype)) return DA_ERR_DTYPE;
  if ((m | n) & 7) return DA_ERR_ALIGN;
  if (rank > m || rank > n) return DA_ERR_ARG;
  if ((uintptr_t)workspace & 255) return DA_ERR_ALIGN;
  for (int i = 0; i < batch; ++i) {
    if (!X[i] || !G[i] || !M[i] || !Q[i]) return DA_ERR_ARG;
    if (((uintptr_t)X[i] | (uintptr_t)G[i] | (uintptr_t)M[i] | (uintptr_t)Q[i]) & 15) return DA_ERR_ALIGN;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const DionLayout L(m, n, rank, m_dtype, sketch ? sketch_k : 0);
  const int r = L.r;   // padded rank: pitch and logical width of Qc, P, R, Qn
  if (sketch && (sketch_k < rank || (sketch_k & 7))) return DA_ERR_ARG;
  const int chunk = L.chunk(batch, workspace_bytes);
  if (chunk < 1) return DA_ERR_WORKSPACE;
  const bool transposed = m < n;
  const int mp = L.mp, np = L.np;
  const long long mn = (long long)m * n;
  const double msz = (double)L.msz, gsz = g_dtype == DA_BF16 ? 2 : 4;

  for (int b0 = 0; b0 < batch; b0 += chunk) {
    const int cb = batch - b0 < chunk ? batch - b0 : chunk;
    // ---- carve the workspace
    char* w = static_cast<char*>(workspace);
    void** tabM = reinterpret_cast<void**>(w); w += DA_MAX_PTRS * sizeof(void*);
    void** tabX = reinterpret_cast<void**>(w); w += DA_MAX_PTRS * sizeof(void*);
    w += 2 * DA_MAX_PTRS * sizeof(void*);
    int* nonzero = reinterpret_cast<int*>(w); w += DA_MAX_PTRS * sizeof(int);
    // the orthonormaliser's status words go straight to the caller's array when there is one
    int* linfo = info ? info + b0 : reinterpret_cast<int*>(w);
    w += DA_MAX_PTRS * sizeof(int);
    w = static_cast<char*>(workspace) + L.fixed();
    char* Qc = w; w += L.qc * cb;
    char* P = w; w += L.p * cb;
    char* R = w; w += L.rb * cb;
    char* Qn = w; w += L.qn * cb;
    char* orth_ws = reinterpret_cast<char*>(align_up(reinterpret_cast<uintptr_t>(w), 256));
    char* sketch_ws = orth_ws + L.orth * cb;
    float* parts = reinterpret_cast<float*>(sketch_ws + L.sketch * cb);
    const long long sQ = (long long)(L.qc / L.msz), sP = (long long)(L.p / L.msz);

    DaPtrTable tx{}, tg{}, tm{}, tq{};
    for (int i = 0; i < cb; ++i) {
      tx.p[i] = X[b0 + i]; tg.p[i] = const_cast<void*>(G[b0 + i]); tm.p[i] = M[b0 + i]; tq.p[i] = Q[b0 + i];
    }
    int rc;
    // B = M + G inside the first P = B Q (bf16 momentum and gradients, whole 256-row tiles of B)
    const bool bq_sum = fused_bq_enabled() && da_dion_bq_sum_applicable(cb, mp, np, r, n, transposed ? 1 : 0, m_dtype, g_dtype);
    {
      DaProfScope prof(DA_PROF_DION_ELEM, bq_sum ? 0.0 : (double)mn * (2 * msz + gsz) * cb, s);
      rc = da_dion_setup(tm, tabM, tx, tabX, cb, nonzero, linfo, s);
      if (rc) return rc;
      // B = M + G, kept in M   (reference dion/dion.py:794)
      if (!bq_sum) {
        rc = da_add_grad(tm, tg, m_dtype, g_dtype, mn, cb, nonzero, s);
        if (rc) return rc;
      }
      // Q in the momentum dtype   (reference dion/dion.py:1216)
      rc = da_cast_table(tq, q_dtype, Qc, m_dtype, np, rank, r, cb, s);
      if (rc) return rc;
    }
    GemmDesc g{};
    // One power iteration is the reference's batched step (dion/dion.py:801-839); more of them repeat
    // P = orth(B Q), Q = B^T P with the unnormalised R as the next Q (dion/dion_reference.py:712-730).  The
    // all-zero / NaN guard runs in every round: between rounds it only matters for an all-zero or non-finite B.
    for (int it = 0; it < power_iters; ++it) {
      g = GemmDesc{};
      g.batch = cb; g.faithful = faithful;
      // ---- P = B Q   (reference dion/dion.py:801); B is M (mp x np) or M^T when m < n
      g.Atab = const_cast<const void* const*>(tabM); g.A = nullptr; g.lda = n; g.a_kstrided = transposed ? 1 : 0;
      g.B = it == 0 ? Qc : R; g.sB = sQ; g.ldb = r; g.b_kstrided = 1;
      g.C = P; g.sC = sP; g.ldc = r; g.c_dtype = m_dtype;
      g.M = mp; g.N = r; g.K = np;
      g.epilogue = DA_EPI_STORE; g.s0 = 0.f; g.s1 = 1.f;
      if (it == 0 && bq_sum) {
        DaProfScope prof(DA_PROF_DION_BQ, gemm_flops(g), s);
        rc = da_dion_bq_sum(tm, tg, Qc, P, sQ, sP, nonzero, cb, mp, np, r, r, n, transposed ? 1 : 0, faithful, s);
        if (rc == DA_OK && r > 256) {
          // the columns of P beyond the first 256: a plain product on the B that launch left in M
          g.B = Qc + 256 * L.msz; g.C = P + 256 * L.msz; g.N = r - 256;
          rc = da_gemm_bf16(g, s);
        }
      } else {
        rc = gemm_any(g, m_dtype, s, DA_PROF_DION_BQ);
      }
      if (rc) return rc;
      // ---- orthonormalise P   (reference dion/dion.py:822, 1267-1308)
      {
        DaProfScope prof(DA_PROF_DION_ORTH, 0.0, s);
        if (sketch) {
          // sketches: [power iteration][matrix of the bucket][sketch_k][mp] in the momentum dtype
          const char* S = static_cast<const char*>(sketch) +
                          ((size_t)it * batch + b0) * (size_t)sketch_k * mp * L.msz;
          rc = da_orthonormalize_sketch(P, S, P, m_dtype, cb, mp, r, rank, sketch_k, orth_ws, sketch_ws, linfo, s);
        } else {
          rc = da_orthonormalize(P, P, m_dtype, cb, mp, r, rank, 2, qr_method, orth_ws, linfo, s);
        }
        if (rc) return rc;
        // all-zero / NaN guard on P   (reference dion/dion.py:847, 1416-1444)
        rc = da_fix(P, m_dtype, sP, cb, nonzero, s);
        if (rc) return rc;
      }
      // ---- R = B^T P   (reference dion/dion.py:839)
      g = GemmDesc{};
      g.batch = cb; g.faithful = faithful;
      g.Atab = const_cast<const void* const*>(tabM); g.lda = n; g.a_kstrided = transposed ? 0 : 1;
      g.B = P; g.sB = sP; g.ldb = r; g.b_kstrided = 1;
      g.C = R; g.sC = sQ; g.ldc = r; g.c_dtype = m_dtype;
      g.M = np; g.N = r; g.K = mp;
      g.epilogue = DA_EPI_STORE; g.s1 = 1.f;
      // A few output tiles with a long inner dimension (tall matrices at a low rank) leave most of the GPU idle:
      // cut the inner dimension into slices that run side by side as the groups of one launch and leave fp32
      // partial sums, which the fix-up pass that follows adds and rounds.
      const int slices = m_dtype == DA_BF16 ? btp_slices(np, r, mp, cb) : 1;
      if (slices > 1) {
        GemmDesc gs[DA_MAX_GROUPS];
        const int kslice = mp / slices;
        const long long pstride = (long long)cb * sQ;
        for (int k = 0; k < slices; ++k) {
          gs[k] = g;
          gs[k].K = kslice;
          gs[k].a_off = (long long)k * kslice * (g.a_kstrided ? n : 1);
          gs[k].B = P + (size_t)k * kslice * r * L.msz;
          gs[k].C = parts + k * pstride; gs[k].c_dtype = DA_F32; gs[k].faithful = 0;
        }
        rc = gemm_group(gs, slices, m_dtype, s, DA_PROF_DION_BTP);
        if (rc) return rc;
        DaProfScope prof(DA_PROF_DION_ELEM, 0.0, s);
        // (the orthonormaliser is done with its fp64 scratch: the column sums take its head)
        rc = da_fix_colsum(parts, slices, pstride, R, Qc, m_dtype, np, r, cb, nonzero, reinterpret_cast<double*>(orth_ws), s);
        if (rc) return rc;
      } else {
        rc = gemm_any(g, m_dtype, s, DA_PROF_DION_BTP);
        if (rc) return rc;
        DaProfScope prof(DA_PROF_DION_ELEM, 0.0, s);
        rc = da_fix_colsum(nullptr, 0, 0, R, Qc, m_dtype, np, r, cb, nonzero, reinterpret_cast<double*>(orth_ws), s);
        if (rc) return rc;
      }
    }  // power iterations
    // ---- error feedback, column normalisation and weight update (reference dion/dion.py:851-872)
    const int form = update_form();
    if (faithful && (form > 0 || (form < 0 && one_pass_update(x_dtype == DA_F32, r, faithful == 2))) &&
        da_dion_ef_update_applicable(mp, np, r, m_dtype)) {
      // Q_new first (it only needs R), then both rank-r updates in one pass over M and X
      {
        DaProfScope prof(DA_PROF_DION_ELEM, 0.0, s);
        rc = da_colnorm(R, Qn, m_dtype, tq, q_dtype, np, r, rank, eps, cb, reinterpret_cast<double*>(orth_ws), s);
        if (rc) return rc;
      }
      DaProfScope prof(DA_PROF_DION_EFUPD, 4.0 * (double)mp * np * r * cb, s);
      rc = da_dion_ef_update(P, R, Qn, tm, tx, cb, mp, np, r, n, transposed ? 1 : 0, x_dtype, ef_alpha, decay,
                             scaled_lr, s);
      if (rc) return rc;
      continue;
    }
    // ---- error feedback  M <- M - (1 - mu) P R^T  (or R P^T)   (reference dion/dion.py:851-853)
    GemmDesc up[2] = {GemmDesc{}, GemmDesc{}};
    for (int k = 0; k < 2; ++k) {
      GemmDesc& u = up[k];
      const char* const D = k == 0 ? R : Qn;
      u.batch = cb; u.faithful = faithful;
      if (!transposed) { u.A = P; u.sA = sP; u.B = D; u.sB = sQ; u.M = mp; u.N = np; }
      else             { u.A = D; u.sA = sQ; u.B = P; u.sB = sP; u.M = np; u.N = mp; }
      u.lda = r; u.ldb = r; u.K = r; u.ldc = n; u.lde = n;
      u.epilogue = DA_EPI_AXPBY;
    }
    up[0].Ctab = tabM; up[0].Etab = const_cast<const void* const*>(tabM); up[0].c_dtype = m_dtype;
    up[0].s0 = 1.f; up[0].s1 = ef_alpha;
    // ---- X <- (1 - lr wd) X - scaled_lr P Q_new^T  (or Q_new P^T)   (reference dion/dion.py:865-872)
    up[1].Ctab = tabX; up[1].Etab = const_cast<const void* const*>(tabX); up[1].c_dtype = x_dtype;
    up[1].s0 = decay; up[1].s1 = -scaled_lr;
    const bool together = form < 0 && m_dtype == DA_BF16 && x_dtype == DA_BF16;
    if (!together) {
      rc = gemm_any(up[0], m_dtype, s, DA_PROF_DION_EF);
      if (rc) return rc;
    }
    // ---- Q_new = column-normalised R   (reference dion/dion.py:856, 875, 1460-1491, 1533-1561)
    {
      DaProfScope prof(DA_PROF_DION_ELEM, 0.0, s);
      rc = da_colnorm(R, Qn, m_dtype, tq, q_dtype, np, r, rank, eps, cb, reinterpret_cast<double*>(orth_ws), s);
      if (rc) return rc;
    }
    rc = together ? gemm_group(up, 2, m_dtype, s, DA_PROF_DION_EFUPD) : gemm_any(up[1], m_dtype, s, DA_PROF_DION_UPD);
    if (rc) return rc;
  }
  return DA_OK;
}

}  // namespace

namespace {
// fills `g` from the caller's buckets; false: not for the kernels of small matrices
bool dion_small_groups(const dion_amd_dion_bucket* buckets, int n, DaDionSmallGroup* g) {
  if (!buckets || n < 1 || n > DA_DS_GROUPS) return false;
  for (int i = 0; i < n; ++i) {
    const dion_amd_dion_bucket& k = buckets[i];
    if (!k.X || !k.G || !k.M || !k.Q || k.batch <= 0 || k.m <= 0 || k.n <= 0 || k.r <= 0 || k.r > k.m || k.r > k.n) return false;
    for (int j = 0; j < k.batch; ++j)
      if (!k.X[j] || !k.G[j] || !k.M[j] || !k.Q[j]) return false;
    g[i] = DaDionSmallGroup{k.X, k.G, k.M, k.Q, k.batch, k.m, k.n, k.r, k.scaled_lr, k.info};
  }
  return true;
}
}  // namespace

extern "C" size_t dion_amd_dion_buckets_workspace_bytes(const dion_amd_dion_bucket* buckets, int nbuckets, int x_dtype,
                                                        int g_dtype, int m_dtype, int q_dtype) {
  if (!dtype_ok(x_dtype) || !dtype_ok(g_dtype) || !dtype_ok(m_dtype) || !dtype_ok(q_dtype)) return 0;
  const int opt = g_opt_dion_small.load(std::memory_order_relaxed);
  DaDionSmallGroup g[DA_DS_GROUPS];
  if (opt == 0 || !dion_small_groups(buckets, nbuckets, g)) return 0;
  const DaDionSmallCall c = {x_dtype, g_dtype, m_dtype, q_dtype, 0.f, 0.f, 0.f, 0};
  return da_dion_small_bytes(g, nbuckets, c, opt == 1);
}

extern "C" int dion_amd_dion_step_buckets(const dion_amd_dion_bucket* buckets, int nbuckets, int x_dtype, int g_dtype,
                                          int m_dtype, int q_dtype, float ef_alpha, float decay, float eps, void* workspace,
                                          size_t workspace_bytes, void* stream) {
  if (!workspace) return DA_ERR_ARG;
  if (!dtype_ok(x_dtype) || !dtype_ok(g_dtype) || !dtype_ok(m_dtype) || !dtype_ok(q_dtype)) return DA_ERR_DTYPE;
  DaDionSmallGroup g[DA_DS_GROUPS];
  if (!dion_small_groups(buckets, nbuckets, g)) return DA_ERR_ARG;
  if ((uintptr_t)workspace & 255) return DA_ERR_ALIGN;
  const DaDionSmallCall c = {x_dtype, g_dtype, m_dtype, q_dtype, ef_alpha, decay, eps, da_ns_flow_fail() ? 1 : 0};
  const size_t need = da_dion_small_bytes(g, nbuckets, c, true);
  if (need == 0) return DA_ERR_LIMIT;
  if (workspace_bytes < need) return DA_ERR_WORKSPACE;
  double flops = 0.0;
  for (int i = 0; i < nbuckets; ++i) flops += 8.0 * g[i].cnt * g[i].m * (double)g[i].n * g[i].r;
  DaProfScope prof(DA_PROF_DION_SMALL, flops, static_cast<hipStream_t>(stream));
  return da_dion_small(g, nbuckets, c, workspace, static_cast<hipStream_t>(stream));
}
