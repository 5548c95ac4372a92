// The Dion step (reference dion/dion.py:742-875) of a set of small matrices, all buckets at once:
//
//   B = M + G;  P = B' Q;  P <- orth(P);  R = B'^T P;  Q <- R / (||R||_col + eps);
//   M <- B - (1 - mu) P R^T;  X <- decay X - lr P Q^T              (B' = B, or B^T when m < n; mp x np, mp >= np)
//
// What bounds it: as a sequence of launches a bucket takes 40 to 60 of them (a third of which only find out that the fp64
// pass of the orthonormaliser is not needed), each a few microseconds of work: a model of 24 matrices of 256 x 256 and
// 256 x 1024 spent 0.6-0.8 ms, most of it on the host; here 0.17 ms for ten launches, of which the factorisation, a chain of
// 64-column steps, takes a third.
//
// Launches, each over all tiles of all matrices, at as many workgroups to a compute unit as its own registers and LDS allow:
//   set-up  B = M + G in place, and where any element is not zero; Q as a padded working matrix
//   BQ      P = B' Q                                      64 x 64 tiles
//   GRAM    P^T P in fp64, lower tiles, K slices as slabs of their own
//   CHAIN   P^T P = L L^T and T = L^-1 in blocks of 64, left-looking, in phases DIAG0 LOW0 DIAG1 LOW1 ..: DIAGj adds the slabs (in
//           order), forms block (j, j - 1) of L and factors and inverts block (j, j); LOWj does the rest of block column j of L and
//           of block row j of T, a task per block (factor_task).  Workgroups take tasks from eight queues, one per XCD
//           (flow_queue.h), a counter per matrix and phase says when a later one may start, and a matrix stays with one XCD.
//   PT      P T^T in fp64
//   FIXG, FIXP  only do anything for a matrix whose pivot range says that cond(P) may leave a visible defect, or with a failed
//           pivot: the closed-form second pass of da_orthonormalize in fp64 (defect measured, noise columns dropped,
//           P <- P (I - up(P^T P - I)))
//   BTP     R = B'^T P                                    64 x 64 (bf16) or 32 x 32 (fp32) tiles
//   CNORM   column norms, Q_new, Q state                  64 x 64 tiles
//   UPD     error feedback and weight update              64 x 64 tiles
// All but CHAIN used to be phases of the queues: two workgroups to a compute unit (the factorisation's registers), a matrix's tiles on
// one XCD's 64 workgroups, and a ticket and a counter for every tile.  14 bf16 matrices of 341 to 2731 rows at rank 256 and 86 (us,
// as phases / as launches): set-up 98 / 24, BQ 52 / 31, GRAM 62 / 41, PT 62 / 59, FIX 16 / 9, BTP 48 / 41, CNORM 7 / 9, UPD 155 / 67;
// the step 622 / 416, by now 407 (several states in turn; 385 on one).  24 fp32 matrices of 256 x 256 and 256 x 1024 at rank 128: 218 / 196,
// by now 188 with the element-wise groups.
// The orthonormaliser is the fp64 CholeskyQR of dion.hip for every matrix: at these sizes the fp64 products cost less than
// the launches of the two-precision road.  P, R and the products with B run on the matrix cores in the momentum's dtype with
// the instructions and the order of k of the batched kernels (v_mfma_f32_16x16x32_bf16, in the updates v_mfma_f32_32x32x16_bf16; v_mfma_f32_32x32x2_f32).
//
// Coherence in CHAIN.  What it reads is of an earlier launch or written once, and read only after its phase is complete: plain loads
// cannot meet a stale L1 line.
//
// Shapes: any m, n (rows that are no multiple of 16 bytes move with unaligned accesses), rank up to 256; the working
// matrices are padded to whole tiles and the tiles' loads fill with zeros.
#include "dion_small.h"
#include <type_traits>
#include "flow_queue.h"
#include "small_tile.h"

#pragma clang fp contract(off)

namespace {

constexpr int MAX_RT = DA_DS_MAX_RANK / 64;
// The launches behind the set-up; CHAIN is the factorisation, whose phases DIAGj (2 j), LOWj (2 j + 1) are one launch.
enum Kind { BQ, GRAM, CHAIN, PT, FIXG, FIXP, BTP, CNORM, UPD, KINDS };
constexpr int PHASES = 2 * MAX_RT;
constexpr int CTR_STRIDE = 32;     // ints per matrix: a counter per phase, then the words below
constexpr int W_NONZERO = 18, W_SICK = 19, W_BAD = 20, W_RANGE = 24;   // (W_RANGE: two doubles)
static_assert(PHASES <= W_NONZERO, "a counter per phase");
constexpr int ADD_ELEMS = 8192;
constexpr double PIVOT_RATIO = 1e-7;   // as POLISH_PIVOT_RATIO in dion.hip
constexpr int SMEM = STAGES64 + DA_DS_MAX_RANK;                  // fp64 64-tiles: two workgroups to a compute unit
constexpr int SMEM_TILE = 2 * 2 * Real<float, 64>::OPND * 4;     // two stages of two operands of fp32 64-tiles, fp64 32-tiles: four
constexpr int SMEM_UPDATE = 2 * 3 * Real<float, 64>::OPND * 4;   // of three operands: three
static_assert(SMEM_TILE >= 2 * 2 * 64 * 64 * 2 && SMEM_TILE >= 64 * 66 * 8 && SMEM_TILE >= 2 * 2 * Real<double, 32>::OPND * 8 &&
              4 * (SMEM_TILE + 1024) <= 160 * 1024, "LDS of the products");
static_assert(SMEM_UPDATE >= 2 * 3 * 64 * 64 * 2 && SMEM_UPDATE >= 2 * 64 * 66 * 4 && 3 * SMEM_UPDATE <= 160 * 1024, "LDS of the update");

struct GroupDev {
  void *const *X, *const *M, *const *Q;   // device tables
  char *P, *P2, *R, *Qn, *Qw;         // momentum dtype: [cnt][mpT * 64][rp], [cnt][npT * 64][rp]
  double* norm;                  // [cnt][nT][rp]: the column norms' shares of BTP's row tiles
  double *P64, *slab, *L, *T, *A2, *defect;   // (A2: T^T until the second pass's Gram product)
  int* words;                    // [cnt][CTR_STRIDE]
  int* info;
  int* any;                      // [cnt][mchunks]: a chunk of B with an element that is not zero
  int cnt;
  unsigned char nq[DA_QUEUES], at[DA_QUEUES];   // matrices in every queue; where their numbers begin in Args::order
  int m, n, r, rp, mp, np, mpT, npT, rT, transposed;
  int nT;
  int mchunks;                   // of ADD_ELEMS elements
  int slices, kslice;            // of the Gram products
  float scaled_lr;
};

struct Args {
  GroupDev g[DA_DS_GROUPS];
  unsigned* tickets;
  int* status;
  unsigned long long spin_limit;
  int ngroups;
  int total[DA_QUEUES];          // tasks of every queue
  unsigned char order[DA_DS_MATS];   // the matrices' numbers within their group, by group and queue
  int x_f32, q_f32;
  float ef_alpha, decay, eps;
};

// lower tiles of P^T P
__host__ __device__ inline int gram_tiles(int r, bool bf) {
  const int t = bf ? (r + 63) >> 6 : (r + 31) >> 5;
  return t * (t + 1) / 2;
}
// workgroups of a launch per matrix
__host__ __device__ inline int tiles_of(const GroupDev& G, Kind kind, bool bf) {
  const int t32 = (G.r + 31) >> 5;
  switch (kind) {
    case BQ: case PT: case FIXP: return G.mpT * G.rT;
    case GRAM: return gram_tiles(G.r, bf) * G.slices;
    case FIXG: return gram_tiles(G.r, false);
    case BTP: return bf ? G.npT * G.rT : ((G.np + 31) >> 5) * t32;
    case CNORM: return G.npT * G.rT;
    case UPD: return G.mpT * G.npT;
    default: return 0;
  }
}
// tasks of a phase of the factorisation
__host__ __device__ inline int tasks_of(const GroupDev& G, int phase) {
  return (phase >> 1) >= G.rT ? 0 : (phase & 1) ? low_tasks(G.rT, phase >> 1) : 1;
}

template <bool BF> struct MomentumType { typedef float type; };
template <> struct MomentumType<true> { typedef bf16_t type; };

// A workgroup's tile.  The tiles of a launch are dealt in eight runs, one to an XCD (which workgroups reach in turn): the tiles of a
// matrix meet in one L2.
struct Where { int g, b, task; };
template <Kind KIND, bool BF>
__device__ __forceinline__ Where my_tile(const Args& a) {
  const int q = blockIdx.x & 7, each = gridDim.x >> 3, rest = gridDim.x & 7;
  int t = q * each + min(q, rest) + (blockIdx.x >> 3), g = 0, per;
  for (;; ++g) {
    per = tiles_of(a.g[g], KIND, BF);
    if (t < a.g[g].cnt * per || g + 1 == a.ngroups) break;
    t -= a.g[g].cnt * per;
  }
  return {g, t / per, t % per};
}

struct SetupGroup {
  int end;                      // the group's last block + 1
  int first, mblocks, per;      // its first matrix; blocks of a matrix for M, for M and Q
  int m, n, r, rp, np, npR;
  char* Qw;
  int* any;
};
struct Setup {
  void* p[4][DA_DS_MATS];   // X, M, Q, G
  void** dst;               // [3][n]: X, M, Q
  int n;
  int* zero;
  int nzero, zblocks;
  int* status;
  int preset;
  int ngroups, g_f32, q_f32;
  SetupGroup g[DA_DS_GROUPS];
};
// The pointers and the counters of the step (the first blocks); B = M + G in place and the note which chunks of it are not all
// zeros; Q as a padded working matrix.  Bound by memory: 5.5 TB/s, 24 us for 14 matrices of 341 to 2731 rows (22 million elements).
template <bool BF>
__global__ __launch_bounds__(256) void dion_small_setup_kernel(Setup s) {
  typedef typename MomentumType<BF>::type E;
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < s.zblocks) {
    const int i = blockIdx.x * 256 + tid;
    if (i < s.n) {
#pragma unroll
      for (int k = 0; k < 3; ++k) s.dst[k * s.n + i] = s.p[k][i];
    }
    for (int e = i; e < s.nzero; e += s.zblocks * 256) s.zero[e] = 0;
    if (i == 0) *s.status = s.preset;
    return;
  }
  int t = blockIdx.x - s.zblocks, gi = 0, begin = 0;
  while (t >= s.g[gi].end) begin = s.g[gi++].end;
  const SetupGroup& G = s.g[gi];
  t -= begin;
  const int b = t / G.per, task = t - b * G.per, mat = G.first + b;
  if (task >= G.mblocks) {
    // ---- Q in the momentum's dtype, padded to whole tiles
    for (int h = 0; h < ADD_ELEMS / 2048; ++h) {
      const long long e = (long long)(task - G.mblocks) * ADD_ELEMS + h * 2048 + tid * 8;
      const int row = (int)(e / G.rp), col = (int)(e - (long long)row * G.rp);
      if (row >= G.npR) break;
      const int c = row < G.np ? G.r - col : 0;
      float v[8];
      if (s.q_f32) load8(static_cast<const float*>(s.p[2][mat]), (long long)row * G.r + col, c, v);
      else load8(static_cast<const bf16_t*>(s.p[2][mat]), (long long)row * G.r + col, c, v);
      store8(G.Qw + (long long)b * G.npR * G.rp * sizeof(E), !BF, e, 8, v);
    }
    return;
  }
  // ---- M + G: every load of a whole chunk on the way before the first is used
  const long long n = (long long)G.m * G.n, e0 = (long long)task * ADD_ELEMS + tid * 8;
  char* const M = static_cast<char*>(s.p[1][mat]);
  const E* const m = reinterpret_cast<const E*>(M);
  const bf16_t* const g16 = static_cast<const bf16_t*>(s.p[3][mat]);
  const float* const g32 = static_cast<const float*>(s.p[3][mat]);
  bool any = false;
  auto finish = [&](float (&mv)[8], const float (&gv)[8], long long e, int c) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      mv[i] = BF ? rbf(mv[i] + gv[i]) : mv[i] + gv[i];
      if (i < c) any |= mv[i] != 0.f;
    }
    store8(M, !BF, e, c, mv);
  };
  auto whole = [&](auto g) {
    Raw<E> mr[4];
    Raw<typename std::remove_const<typename std::remove_pointer<decltype(g)>::type>::type> gr[4];
#pragma unroll
    for (int h = 0; h < 4; ++h) { mr[h] = load_raw(m + e0 + h * 2048); gr[h] = load_raw(g + e0 + h * 2048); }
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      float mv[8], gv[8];
      unpack(mr[h], mv);
      unpack(gr[h], gv);
      finish(mv, gv, e0 + h * 2048, 8);
    }
  };
  if ((long long)(task + 1) * ADD_ELEMS <= n) {
    if (s.g_f32) whole(g32);
    else whole(g16);
  } else {
    for (int h = 0; h < 4; ++h) {
      const long long e = e0 + h * 2048;
      const int c = n - e >= 8 ? 8 : (int)(n - e);
      if (c <= 0) break;
      float mv[8], gv[8];
      load8(m, e, c, mv);
      if (s.g_f32) load8(g32, e, c, gv);
      else load8(g16, e, c, gv);
      finish(mv, gv, e, c);
    }
  }
  any = __syncthreads_or(any);
  if (tid == 0) G.any[(long long)b * G.mblocks + task] = any;
}

// P = B' Q;  R = B'^T P: a 64 x 64 tile (of R in fp32 32 x 32).  Bound by the latency of a tile's stages.
template <bool BF, bool bq>
__global__ __launch_bounds__(256, 4) void dion_small_product_kernel(Args a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  typedef typename MomentumType<BF>::type E;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_uniform(tid >> 6), wm = wave >> 1, wn = wave & 1;
  const Where w = my_tile<bq ? BQ : BTP, BF>(a);
  const GroupDev& G = a.g[w.g];
  const int b = w.b, task = w.task, rp = G.rp;
  const long long prow = (long long)b * G.mpT * 64 * rp * sizeof(E), rrow = (long long)b * G.npT * 64 * rp * sizeof(E);
  char *const P = G.P + prow, *const P2 = G.P2 + prow, *const R = G.R + rrow, *const Qw = G.Qw + rrow;
  float* const stg = reinterpret_cast<float*>(lds);
  const int rT = G.rT, rt32 = (G.r + 31) >> 5;
  if (bq && task == 0) {   // has any element of B been found not to be zero?
    bool any = false;
    for (int i = tid; i < G.mchunks; i += 256) any |= G.any[(long long)b * G.mchunks + i] != 0;
    if (__any(any) && lane == 0) __hip_atomic_store(G.words + b * CTR_STRIDE + W_NONZERO, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const bool nonzero = G.words[b * CTR_STRIDE + W_NONZERO] != 0;   // (of R: of the launch before)
  const bool turn = (G.transposed != 0) == bq;   // B' is B^T, or R takes B'^T
  auto with_layout = [&](auto body) {   // (the layout known to the compiler: no branch in the K loop)
    const E* const M = static_cast<const E*>(G.M[b]);
    const int rows = bq ? G.mp : G.np, kmax = bq ? G.np : G.mp;
    const long long last = (long long)G.m * G.n - 8;
    if (turn) body(Opnd<E, true>{M, G.n, 1, rows, kmax, last});
    else body(Opnd<E, true>{M, G.n, 0, rows, kmax, last});
  };
  const Opnd<E, false> sb = work<E>(bq ? Qw : P2, rp, 1);
  const int kend = bq ? G.np : G.mp;
  char* const C = bq ? P : R;
  // a chunk of the result: rounded and, for R, guarded (an all-zero B keeps Q)
  auto put = [&](int row0, int col0, int lr, int lc, int pitch) {
    const int row = row0 + lr, col = col0 + lc;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = row < (bq ? G.mp : G.np) ? stg[lr * pitch + lc + i] : 0.f;
    if (!bq) {
      float alt[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) alt[i] = 0.f;
      if (!nonzero) unpack(load_raw(reinterpret_cast<const E*>(Qw) + (long long)row * rp + col), alt);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = guard<BF>(v[i], nonzero, alt[i]);
#pragma unroll
      for (int i = 0; i < 8; ++i) stg[lr * pitch + lc + i] = v[i];
    }
    store8(C, !BF, (long long)row * rp + col, 8, v);
  };
  // the tile's share of the column norms
  auto norms = [&](int ti, int row0, int col0, int pitch, int tb) {
    __syncthreads();
    double* const red = reinterpret_cast<double*>(lds + 64 * 66 * 4);
    const int c = tid & (tb - 1), g = tid / tb, rows = tb * tb / 256;
    double s = 0.0;
    for (int i = g * rows; i < (g + 1) * rows; ++i) {
      const float v = row0 + i < G.np ? stg[i * pitch + c] : 0.f;
      s += (double)v * (double)v;
    }
    red[tid] = s;
    __syncthreads();
    if (tid < tb) {
      double t = 0.0;
      for (int i = 0; i < 256 / tb; ++i) t += red[i * tb + tid];
      G.norm[((long long)b * G.nT + ti) * rp + col0 + tid] = t;
    }
  };
  if (BF || bq) {
    const int ti = task / rT, tj = task - ti * rT, row0 = wave_uniform(ti) * 64, col0 = wave_uniform(tj) * 64;
    if constexpr (BF) {
      with_layout([&](const Opnd<E, true>& sa) { product_bf16(sa, sb, row0, col0, kend, lds, tid, lane, wm, wn, stg); });
    } else {
      f32x16_t acc[1];
      const Opnd<E, false> sbs[1] = {sb};
      with_layout([&](const Opnd<E, true>& sa) { tile32x2<1>(sa, sbs, row0, col0, kend, stg, tid, lane, wm, wn, acc); });
      stage_f32(acc[0], stg, lane, wm, wn);
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      put(row0, col0, (tid >> 3) + 32 * h, (tid & 7) * 8, 66);
    }
    if (!bq) norms(ti, row0, col0, 66, 64);
  } else {
    const int ti = task / rt32, tj = task - ti * rt32, row0 = wave_uniform(ti) * 32, col0 = wave_uniform(tj) * 32;
    if constexpr (!BF) with_layout([&](const Opnd<E, true>& sa) { tile16<float, 32>(sa, sb, row0, col0, 0, kend, stg, tid, lane, wm, wn); });
    if (tid < 128) put(row0, col0, tid >> 2, (tid & 3) * 8, 34);
    norms(ti, row0, col0, 34, 32);
  }
}

// One lower tile of one K slice of P^T P: 64 x 64 of a bf16 P, 32 x 32 of an fp32 one.  Bound by the fp64 matrix cores: 41 us for
// 1.8 GFLOP in bf16 (32 x 32 tiles through fp64 stages: 64).
template <bool BF>
__global__ __launch_bounds__(256, BF ? 3 : 4) void dion_small_gram_kernel(Args a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  typedef typename MomentumType<BF>::type E;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_uniform(tid >> 6), wm = wave >> 1, wn = wave & 1;
  const Where w = my_tile<GRAM, BF>(a);
  const GroupDev& G = a.g[w.g];
  const int rp = G.rp, n = gram_tiles(G.r, BF), slice = w.task / n, kbeg = slice * G.kslice;
  const E* const P = reinterpret_cast<const E*>(G.P) + (long long)w.b * G.mpT * 64 * rp;
  double *const out = G.slab + ((long long)w.b * G.slices + slice) * rp * rp, *const d = reinterpret_cast<double*>(lds);
  if constexpr (BF) {
    int ti = 0, tj = w.task - slice * n;
    while (tj > ti) tj -= ++ti;
    gram64_bf16(P + (long long)kbeg * rp, rp, ti * 64, tj * 64, min(G.kslice, G.mpT * 64 - kbeg), lds, tid, lane, wm, wn);
    for (int e = tid; e < 4096; e += 256) out[(long long)(ti * 64 + (e >> 6)) * rp + tj * 64 + (e & 63)] = d[(e >> 6) * 66 + (e & 63)];
  } else {
    int ti, tj;
    gram_tile(work<E>(P, rp, 1), w.task - slice * n, kbeg, min(kbeg + G.kslice, (G.mp + KD - 1) / KD * KD), out, rp, d, tid, lane, wm, wn, ti, tj);
  }
}

// The factorisation: phases of a matrix one after the other, tasks from the queue of its XCD.
__global__ __launch_bounds__(256, 2) void dion_small_chain_kernel(Args args) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ int sh_ticket[2];
  __shared__ int sh_start[64], sh_per[64];   // the queue's schedule: entry = phase * ngroups + group
  __shared__ unsigned char sh_at[64];
  static_assert(PHASES * DA_DS_GROUPS <= 64, "one entry each");
  const int xcd = xcc_id();

  for (int qi = 0; qi < DA_QUEUES; ++qi) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int q = (xcd + qi) & (DA_QUEUES - 1);
    const int total = args.total[q];
    if (total <= 0) continue;
    unsigned* word = args.tickets + q * DA_QUEUE_LINE;
    int slot = 0;
    if (tid == 0) sh_ticket[0] = take_ticket(word, xcd, total, false);
    __syncthreads();
    if (wave_uniform(sh_ticket[0]) < 0) {
      __syncthreads();   // thread 0 rewrites sh_ticket for the next queue
      continue;
    }
    // ---- the schedule, phase by phase, group by group: first ticket and tasks per matrix
    if (tid < 64) {
      int n = 0;
      if (tid < PHASES * args.ngroups) {
        const int k = tid / args.ngroups;
        const GroupDev& G = args.g[tid - k * args.ngroups];
        const int per = tasks_of(G, k);
        n = per * G.nq[q];
        sh_per[tid] = per;
        sh_at[tid] = G.at[q];
      }
      int sum = n;   // exclusive sums
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(sum, o);
        if (lane >= o) sum += x;
      }
      sh_start[tid] = sum - n;
    }
    while (true) {
      __syncthreads();
      int t = wave_uniform(sh_ticket[slot]);
      if (t < 0) break;
      // (opaque to the compiler: every phase's address arithmetic would move out of this loop and be spilled)
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      const int lane = tid & 63, wave = wave_uniform(tid >> 6), wm = wave >> 1, wn = wave & 1;
      const Args& a = fresh_args<Args>();
      // ---- ticket -> (phase, group, matrix, task): the last entry that starts at or before it
      const int entry = wave_uniform(__popcll(__ballot(lane < PHASES * a.ngroups && sh_start[lane] <= t)) - 1);
      t -= wave_uniform(sh_start[entry]);
      const int phase = entry / a.ngroups, per = wave_uniform(sh_per[entry]);
      const GroupDev& G = a.g[entry - phase * a.ngroups];
      const int kth = wave_uniform(t / per);
      const int task = wave_uniform(t - kth * per);
      const int b = wave_uniform((int)a.order[sh_at[entry] + kth]);
      int* words = G.words + (long long)b * CTR_STRIDE;
      const long long rr = (long long)G.rp * G.rp;
      const Factor F = {G.slab + (long long)b * G.slices * rr, G.L + b * rr, G.T + b * rr, G.A2 + b * rr, G.slices, G.r, G.rp, G.rT,
                        words + W_BAD, words + W_SICK, G.info ? G.info + b : nullptr, reinterpret_cast<double*>(words + W_RANGE), PIVOT_RATIO};
      auto wait_phase = [&](int before) {
        if (before < 0) return;
        if (tid == 0) wait_count(words + before, tasks_of(G, before), a.status, a.spin_limit);
        __syncthreads();
      };
      const bool diag = (phase & 1) == 0;
      factor_task(F, phase >> 1, diag, task, lds, tid, lane, wave, wm, wn, [&] { wait_phase(diag ? phase - 3 : phase - 2); },
                  [&] { wait_phase(diag ? phase - 2 : phase - 1); });
      // ---- publish: every wavefront's stores are acknowledged, then the matrix's counter moves
      unsigned next = DA_NO_TICKET;
      if (tid == 0) next = request_ticket(word);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (tid == 0) sh_ticket[slot ^ 1] = ticket_of(next, total);
      __syncthreads();
      if (tid == 0) __hip_atomic_fetch_add(words + phase, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);   // (in the L2)
      slot ^= 1;
    }
    __syncthreads();   // thread 0 rewrites sh_ticket for the next queue
  }
}

// P T^T in fp64 (PT; bound by the fp64 matrix cores, 59 us for 1.8 GFLOP; through LDS stages 75); for a matrix that needs it the second pass: P^T P (FIXG), P <- P (I - up(P^T P - I)) (FIXP).
template <Kind KIND, bool BF>
__global__ __launch_bounds__(256, KIND == FIXG ? 4 : KIND == PT ? 3 : 2) void dion_small_orth_kernel(Args a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  typedef typename MomentumType<BF>::type E;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_uniform(tid >> 6), wm = wave >> 1, wn = wave & 1;
  const Where w = my_tile<KIND, BF>(a);
  const GroupDev& G = a.g[w.g];
  const int b = w.b, t = w.task, rp = G.rp;
  const int* const words = G.words + (long long)b * CTR_STRIDE;
  const bool sick = words[W_SICK] != 0, nonzero = words[W_NONZERO] != 0;
  if (KIND != PT && !sick) return;   // what nearly every matrix does
  const long long rr = (long long)rp * rp, prow = (long long)b * G.mpT * 64 * rp;
  double *const P64 = G.P64 + prow, *const d = reinterpret_cast<double*>(lds);
  double* const defect = G.defect + (long long)b * rp * (2 * MAX_RT);
  if constexpr (KIND == FIXG) {
    int ti, tj;
    gram_tile(work<double>(P64, rp, 1), t, 0, (G.mp + KD - 1) / KD * KD, G.A2 + b * rr, rp, d, tid, lane, wm, wn, ti, tj);
    gram_defect(d, defect, 2 * MAX_RT, ti, tj, tid);
    return;
  }
  const int row0 = t / G.rT * 64, col0 = t % G.rT * 64;
  if constexpr (KIND == PT) {   // (T is triangular)
    direct64<false>(reinterpret_cast<const E*>(G.P) + prow + (long long)row0 * rp, rp, G.A2 + b * rr + col0, rp, col0 + 64, d, lane, wm, wn);
    if (sick) {
      for (int e = tid; e < 4096; e += 256) P64[(long long)(row0 + (e >> 6)) * rp + col0 + (e & 63)] = d[(e >> 6) * 66 + (e & 63)];
      return;
    }
  } else {
    unsigned char* const drop = reinterpret_cast<unsigned char*>(lds + STAGES64);
    find_dropped(defect, 2 * MAX_RT, G.r, rp, drop, tid);
    if (t == 0 && tid == 0 && G.info && words[W_BAD] == 0) {
      for (int c = 0; c < G.r; ++c)
        if (drop[c]) { G.info[b] = c + 1; break; }
    }
    polish_tile(P64, G.A2 + b * rr, G.r, rp, drop, row0, col0, d, tid, lane, wm, wn);
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = (tid >> 3) + 32 * h, c = (tid & 7) * 8;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = guard<BF>((float)d[r * 66 + c + i], nonzero, 0.f);
    store8(G.P2 + prow * sizeof(E), !BF, (long long)(row0 + r) * rp + col0 + c, 8, v);
  }
}

// A 64 x 64 tile of R: column norms from the tiles' shares (in order), Q_new in the momentum's dtype and as Q state.
template <bool BF>
__global__ __launch_bounds__(256) void dion_small_cnorm_kernel(Args a) {
  __shared__ double red[256];
  __shared__ float den[64];
  typedef typename MomentumType<BF>::type E;
  const int tid = threadIdx.x;
  const Where w = my_tile<CNORM, BF>(a);
  const GroupDev& G = a.g[w.g];
  const int b = w.b, task = w.task, rp = G.rp;
  const long long rrow = (long long)b * G.npT * 64 * rp * sizeof(E);
  const char* const R = G.R + rrow;
  char* const Qn = G.Qn + rrow;
  const bool poisoned = __hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  const int ti = wave_uniform(task / G.rT), row0 = ti * 64, col0 = wave_uniform(task - ti * G.rT) * 64;
  const int limit = BF ? rp : ((G.r + 31) >> 5) << 5;   // columns of R that exist
  Raw<E> rv[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    rv[h] = load_raw(reinterpret_cast<const E*>(R) + (long long)(row0 + (tid >> 3) + 32 * h) * rp + col0 + (tid & 7) * 8);
  {
    double s = 0.0;
    if (col0 + (tid & 63) < limit)
      for (int t = tid >> 6; t < G.nT; t += 4) s += G.norm[((long long)b * G.nT + t) * rp + col0 + (tid & 63)];
    red[tid] = s;
  }
  __syncthreads();
  if (tid < 64) den[tid] = sqrtf((float)(red[tid] + red[64 + tid] + red[128 + tid] + red[192 + tid])) + a.eps;
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = row0 + (tid >> 3) + 32 * h, c = (tid & 7) * 8, col = col0 + c;
    float v[8];
    unpack(rv[h], v);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] = v[i] / den[c + i];
      if (BF) v[i] = rbf(v[i]);
      if (poisoned) v[i] = __builtin_nanf("");
      if (row >= G.np || col + i >= G.r) v[i] = 0.f;   // (padding)
    }
    store8(Qn, !BF, (long long)row * rp + col, 8, v);
    store8(static_cast<char*>(G.Q[b]), a.q_f32, (long long)row * G.r + col, row < G.np ? G.r - col : 0, v);
  }
}

// Error feedback and weight update, M += ef_alpha P R^T and X = decay X - lr P Q_new^T: a 64 x 64 tile (rows of P, rows of R) per
// workgroup, three workgroups to a compute unit, the tiles of an XCD next to each other (it keeps their R and Q_new in its L2).
// Bound by the latency of a tile's loads.
template <bool BF>
__global__ __launch_bounds__(256, 3) void dion_small_update_kernel(Args a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  typedef typename MomentumType<BF>::type E;
  constexpr int MSZ = BF ? 2 : 4;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_uniform(tid >> 6), wm = wave >> 1, wn = wave & 1;
  const Where w = my_tile<UPD, BF>(a);
  const GroupDev& G = a.g[w.g];
  const int b = w.b, task = w.task;
  const int rp = G.rp;
  const char* const P2 = G.P2 + (long long)b * G.mpT * 64 * rp * MSZ;
  const char* const R = G.R + (long long)b * G.npT * 64 * rp * MSZ;
  const char* const Qn = G.Qn + (long long)b * G.npT * 64 * rp * MSZ;
  char* const M = static_cast<char*>(G.M[b]);
  float* const stg = reinterpret_cast<float*>(lds);
  const int ti = wave_uniform(task / G.npT), tj = wave_uniform(task - task / G.npT * G.npT);
  const int row0 = ti * 64, col0 = tj * 64;
  const bool turned = G.transposed != 0;
  const Opnd<E, false> sp = work<E>(P2, rp, 0), sr = work<E>(R, rp, 0), sn = work<E>(Qn, rp, 0);
  const int kend = BF ? rp : ((G.r + 31) >> 5) << 5;   // (what the tiles of BTP have written)
  char* const X = static_cast<char*>(G.X[b]);
  float* const stg2 = stg + 64 * 66;
  // a thread's chunks: stored row, eight consecutive stored columns; inside the matrix M and X are requested before the
  // products
  const int tr = turned ? col0 : row0, tc = turned ? row0 : col0;
  const bool inside = tr + 64 <= G.m && tc + 64 <= G.n;
  const long long e0 = (long long)(tr + (tid >> 3)) * G.n + tc + (tid & 7) * 8;
  Raw<E> mr[2];
  Raw<float> xr[2];      // (bf16 weights: the first quarter)
  if (inside) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const long long e = e0 + 32LL * h * G.n;
      mr[h] = load_raw(reinterpret_cast<const E*>(M) + e);
      if (a.x_f32) xr[h] = load_raw(reinterpret_cast<const float*>(X) + e);
      else xr[h].q[0] = load_raw(reinterpret_cast<const bf16_t*>(X) + e).q[0];
    }
  }
  f32x16_t acc[2];
  const Opnd<E, false> sbs[2] = {sr, sn};
  if constexpr (BF) update_bf16(sp, sbs, row0, col0, kend, lds, tid, lane, wm, wn, acc);
  else tile32x2<2>(sp, sbs, row0, col0, kend, stg, tid, lane, wm, wn, acc);
  stage_f32(acc[0], stg, lane, wm, wn);
  stage_f32(acc[1], stg2, lane, wm, wn);
  __syncthreads();
  const bool poisoned = __hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  const float lr = -G.scaled_lr;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = (tid >> 3) + 32 * h, c = (tid & 7) * 8;
    const long long e = e0 + 32LL * h * G.n;
    const int n = tr + r < G.m ? G.n - tc - c : 0;
    float mv[8], xv[8];
    if (inside) {
      unpack(mr[h], mv);
      if (a.x_f32) unpack(xr[h], xv);
      else unpack(Raw<bf16_t>{{xr[h].q[0]}}, xv);
    } else {
      load8(reinterpret_cast<const E*>(M), e, n, mv);
      if (a.x_f32) load8(reinterpret_cast<const float*>(X), e, n, xv);
      else load8(reinterpret_cast<const bf16_t*>(X), e, n, xv);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int at = turned ? (c + i) * 66 + r : r * 66 + c + i;
      // the roundings of the reference's separate tensor ops (epi_value in mfma_tile.h)
      float t1 = stg[at], t2 = stg2[at];
      if (BF) { t1 = rbf(t1); t2 = rbf(t2); }
      t1 = a.ef_alpha * t1;
      t2 = lr * t2;
      if (BF) { t1 = rbf(t1); t2 = rbf(t2); }
      mv[i] = mv[i] + t1;
      float x = a.decay * xv[i];
      if (!a.x_f32) x = rbf(x);
      xv[i] = x + t2;
      if (poisoned) mv[i] = xv[i] = __builtin_nanf("");
    }
    store8(M, !BF, e, n, mv);
    store8(X, a.x_f32, e, n, xv);
  }
}

inline size_t up256(size_t x) { return (x + 255) & ~(size_t)255; }

struct Shape {
  int mp, np, mpT, npT, rT, rp, nT, slices, kslice;
  Shape(int m, int n, int r, bool bf, int rows = 128) {
    mp = m > n ? m : n;
    np = m > n ? n : m;
    mpT = (mp + 63) / 64; npT = (np + 63) / 64; rT = (r + 63) / 64;
    rp = rT * 64;
    nT = bf ? npT : (np + 31) / 32;
    // K slices: about `rows` rows to a Gram tile, at least 128, in whole stages
    const int deep = bf ? 64 : KD;
    slices = mp / (rows > 128 ? rows : 128);
    if (slices < 1) slices = 1;
    kslice = ((mp + slices - 1) / slices + deep - 1) / deep * deep;
    slices = (mp + kslice - 1) / kslice;
  }
};

// Rows to a Gram tile for one tile to a compute unit (32 x 32 tiles: four): the fp64 matrix cores bound the launch, whose time is that of
// the unit with the most; and every K slice is a slab that the factorisation adds up.
inline int gram_rows(const DaDionSmallGroup* g, int n, bool bf) {
  long long rows = 0;
  for (int i = 0; i < n; ++i) rows += (long long)g[i].cnt * gram_tiles(g[i].r, bf) * (g[i].m > g[i].n ? g[i].m : g[i].n);
  const long long per = rows / (bf ? 256 : 1024);
  return per < 1 ? 1 : per > (1 << 30) ? 1 << 30 : (int)per;
}

inline int mchunks(int m, int n) { return (int)(((long long)m * n + ADD_ELEMS - 1) / ADD_ELEMS); }

// lays out one group at p (null: only counts); returns the bytes
size_t lay_out(GroupDev* D, const DaDionSmallGroup& g, const Shape& S, int msz, char* base) {
  size_t o = 0;
  auto take = [&](size_t n) { char* q = base ? base + o : nullptr; o += up256(n); return q; };
  const size_t c = (size_t)g.cnt, pm = c * S.mpT * 64 * S.rp, pn = c * S.npT * 64 * S.rp, rr = c * S.rp * S.rp;
  char* P = take(pm * msz);
  char* P2 = take(pm * msz);
  char* R = take(pn * msz);
  char* Qn = take(pn * msz);
  char* Qw = take(pn * msz);
  char* norm = take(c * S.nT * S.rp * 8);
  char* any = take(c * mchunks(g.m, g.n) * 4);
  double* f64[6];   // P64, slab, L, T, A2, defect
  for (int i = 0; i < 6; ++i) f64[i] = reinterpret_cast<double*>(take((i == 0 ? pm : i == 1 ? rr * S.slices : i == 5 ? c * S.rp * 2 * MAX_RT : rr) * 8));
  if (D) {
    D->any = reinterpret_cast<int*>(any); D->mchunks = mchunks(g.m, g.n);
    D->P = P; D->P2 = P2; D->R = R; D->Qn = Qn; D->Qw = Qw; D->norm = reinterpret_cast<double*>(norm); D->nT = S.nT;
    D->P64 = f64[0]; D->slab = f64[1]; D->L = f64[2]; D->T = f64[3]; D->A2 = f64[4]; D->defect = f64[5];
  }
  return o;
}

// control memory: words of all matrices, the queues' lines, the status word's line, the pointer tables
size_t control_bytes(int mats) { return up256((size_t)mats * CTR_STRIDE * 4 + (DA_QUEUES + 1) * DA_QUEUE_LINE * 4) + up256((size_t)3 * mats * 8); }

// Matrices to queues: those with the longest factorisation first, each to the queue with the least to do so far; queue[i] of matrix i,
// in the order of the groups.
void deal(const DaDionSmallGroup* g, int n, unsigned char* queue) {
  int load[DA_QUEUES] = {0}, cost[DA_DS_GROUPS], sorted[DA_DS_GROUPS], first[DA_DS_GROUPS];
  for (int i = 0, mats = 0; i < n; ++i) {
    const int rT = (g[i].r + 63) / 64;
    cost[i] = rT * rT;
    first[i] = mats;
    mats += g[i].cnt;
    int k = i;
    for (; k > 0 && cost[sorted[k - 1]] < cost[i]; --k) sorted[k] = sorted[k - 1];
    sorted[k] = i;
  }
  for (int k = 0; k < n; ++k)
    for (int j = 0; j < g[sorted[k]].cnt; ++j) {
      int q = 0;
      for (int x = 1; x < DA_QUEUES; ++x)
        if (load[x] < load[q]) q = x;
      load[q] += cost[sorted[k]];
      queue[first[sorted[k]] + j] = (unsigned char)q;
    }
}

template <bool BF>
int launch_all(const Args& a, hipStream_t s) {
  static DaOncePerDevice configured;
  int rc = configured.run([&]() -> int {
    const void* const wide[] = {reinterpret_cast<const void*>(dion_small_chain_kernel), reinterpret_cast<const void*>(dion_small_orth_kernel<FIXP, BF>)};
    for (const void* f : wide) DA_HIP_CHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM));
    return DA_OK;
  });
  auto launch = [&](void (*kernel)(Args), Kind kind, int smem) {
    long long n = kind == CHAIN ? 2 * da_cu_count() : 0;
    for (int i = 0; kind != CHAIN && i < a.ngroups; ++i) n += (long long)a.g[i].cnt * tiles_of(a.g[i], kind, BF);
    if (rc) return;
    hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(256), smem, s, a);
    rc = da_launch_status();
  };
  launch(dion_small_product_kernel<BF, true>, BQ, SMEM_TILE);
  launch(dion_small_gram_kernel<BF>, GRAM, SMEM_TILE);
  launch(dion_small_chain_kernel, CHAIN, SMEM);
  launch(dion_small_orth_kernel<PT, BF>, PT, SMEM_TILE);
  launch(dion_small_orth_kernel<FIXG, BF>, FIXG, SMEM_TILE);
  launch(dion_small_orth_kernel<FIXP, BF>, FIXP, SMEM);
  launch(dion_small_product_kernel<BF, false>, BTP, SMEM_TILE);
  launch(dion_small_cnorm_kernel<BF>, CNORM, 0);
  launch(dion_small_update_kernel<BF>, UPD, SMEM_UPDATE);
  return rc;
}

}  // namespace

size_t da_dion_small_bytes(const DaDionSmallGroup* g, int n, const DaDionSmallCall& c, bool forced) {
  if (!g || n < 1 || n > DA_DS_GROUPS) return 0;
  int mats = 0;
  size_t bytes = 0;
  // Where the line lies, in microseconds.  All buckets together: ten launches and the factorisation (45, and 35 per 64 columns of
  // rank; 70 for a factor as wide as the matrix, which takes the second pass), and per 64 x 64 tile of a matrix its passes and its
  // products.  A launch per product: what the host takes to issue a few hundred of them, 2.5 times that with shapes off the 8-grid
  // (padded copies), plus the products.  Measured, together / by buckets, layers of four d x d and two d x 4d:
  // bf16 128 x2 r 64: 74 / 503;  512 x8 r 128: 260 / 477;  512 x2 r 256: 245 / 518;  768 x1 r 192: 192 / 406;  768 x4 r 192: 360 / 508;
  // 768 x12 r 48: 460 / 503;  1024 x1 r 256: 288 / 507;  1024 x4 r 64: 283 / 511;  2048 x1 r 63: 294 / 502;
  // 256 x4 r 256: 287 / 506;  200 x1 r 200: 184 / 485;  four of 256 x 256 alone r 256: 193 / 269;  and not: 768 x12 r 192: 1002 / 711;
  // 1024 x4 r 256: 709 / 532 (2048 x1 r 256: 552 / 597 is given away);
  // fp32 256 x4 r 128: 171 / 512;  768 x4 r 48: 406 / 944;  1024 x2 r 256: 1004 / 1416;  2048 x1 r 256: 1743 / 2445;  and not 768 x12 r 192:
  // 2470 / 2345;  bf16 off the grid 1021 x4 r 255: 745 / 1863;  2043 x1 r 255: 585 / 960.
  const bool bf = c.m_dtype == DA_BF16;
  const int rows = gram_rows(g, n, bf);
  double chain = 0.0, work = 0.0, other = 0.0;
  bool padded = false, odd_full = false;
  for (int i = 0; i < n; ++i) {
    if (g[i].cnt < 1 || g[i].r < 1 || g[i].r > DA_DS_MAX_RANK || (long long)g[i].m * g[i].n > (1LL << 28) || (long long)g[i].m * g[i].n < 8) return 0;
    const Shape S(g[i].m, g[i].n, g[i].r, c.m_dtype == DA_BF16);
    for (int j = 0; j < g[i].cnt; ++j) {
      // (Nothing in these launches needs the grid any more: views 16 bytes off it, taken together, give the bits of aligned matrices in
      // the same time, 132 us for 24 of 256 x 256 and 256 x 1024 in bf16, where the road by buckets takes 428.  They are left to that
      // road, which has stepped them since one launch held all phases and a line must not be shared with another matrix.)
      if (((uintptr_t)g[i].M[j] | (uintptr_t)g[i].X[j]) & 127) return 0;
      if (((uintptr_t)g[i].G[j] | (uintptr_t)g[i].Q[j]) & 15) return 0;
    }
    const double own = 45.0 + 35.0 * S.rT + (g[i].r == S.np ? 70.0 : 0.0), tiles = (double)g[i].cnt * S.mpT * S.npT;
    chain = own > chain ? own : chain;
    work += tiles * (bf ? 0.010 + 0.0085 * S.rT : 0.020 + 0.028 * S.rT);
    other += tiles * S.rT * (bf ? 0.004 : 0.028);
    // (A full-rank factor of noise has a condition of 1e4 to 1e6, which multiplies every last-bit difference between the roads from step
    // to step.  Off the 8-grid the other road's second pass works on a padded rank, and such factors stay with it.  On the grid
    // neither road is the closer one to a step in 64 bits: 4 of 256 x 256 in bf16, first and third step, error of Q 7.95e-2 and
    // 4.76e-2 on both, the digits that differ are the fifth and later.)
    odd_full |= g[i].r == S.np && (g[i].r & 7) != 0;
    padded |= ((g[i].m | g[i].n) & 7) != 0;
    mats += g[i].cnt;
    bytes += lay_out(nullptr, g[i], Shape(g[i].m, g[i].n, g[i].r, bf, rows), c.m_dtype == DA_BF16 ? 2 : 4, nullptr);
  }
  if (mats > DA_DS_MATS) return 0;
  other += (bf ? 400.0 : 480.0) * (padded ? 2.5 : 1.0);
  if (!forced && (odd_full || chain + work > other)) return 0;
  return bytes + control_bytes(mats);
}

int da_dion_small(const DaDionSmallGroup* g, int n, const DaDionSmallCall& c, void* workspace, hipStream_t s) {
  Args a{};
  Setup su;
  const bool bf = c.m_dtype == DA_BF16;
  int mats = 0;
  char* p = static_cast<char*>(workspace);
  for (int i = 0; i < n; ++i) mats += g[i].cnt;
  if (mats > DA_DS_MATS || n > DA_DS_GROUPS) return DA_ERR_LIMIT;
  int* words = reinterpret_cast<int*>(p);
  a.tickets = reinterpret_cast<unsigned*>(words + (size_t)mats * CTR_STRIDE);
  a.status = reinterpret_cast<int*>(a.tickets + DA_QUEUES * DA_QUEUE_LINE);
  su.n = mats;
  su.zero = words;
  su.nzero = mats * CTR_STRIDE + DA_QUEUES * DA_QUEUE_LINE;
  su.status = a.status;
  su.preset = c.fail;
  su.dst = reinterpret_cast<void**>(p + up256((size_t)mats * CTR_STRIDE * 4 + (DA_QUEUES + 1) * DA_QUEUE_LINE * 4));
  p += control_bytes(mats);
  unsigned char queue[DA_DS_MATS];
  deal(g, n, queue);
  int first = 0, at = 0;
  long long adds = 0;
  const int rows = gram_rows(g, n, bf);
  for (int i = 0; i < n; ++i) {
    const Shape S(g[i].m, g[i].n, g[i].r, bf, rows);
    GroupDev& D = a.g[i];
    p += lay_out(&D, g[i], S, c.m_dtype == DA_BF16 ? 2 : 4, p);
    D.X = su.dst + first; D.M = su.dst + mats + first; D.Q = su.dst + 2 * mats + first;
    for (int j = 0; j < g[i].cnt; ++j) {
      su.p[0][first + j] = g[i].X[j];
      su.p[1][first + j] = g[i].M[j];
      su.p[2][first + j] = g[i].Q[j];
      su.p[3][first + j] = const_cast<void*>(g[i].G[j]);
    }
    D.words = words + (size_t)first * CTR_STRIDE;
    D.info = g[i].info;
    D.cnt = g[i].cnt;
    for (int q = 0; q < DA_QUEUES; ++q) {
      D.at[q] = (unsigned char)at;
      for (int j = 0; j < g[i].cnt; ++j)
        if (queue[first + j] == q) a.order[at++] = (unsigned char)j;
      D.nq[q] = (unsigned char)(at - D.at[q]);
    }
    D.m = g[i].m; D.n = g[i].n; D.r = g[i].r; D.rp = S.rp; D.mp = S.mp; D.np = S.np;
    D.mpT = S.mpT; D.npT = S.npT; D.rT = S.rT; D.transposed = g[i].m < g[i].n ? 1 : 0;
    D.slices = S.slices; D.kslice = S.kslice;
    D.scaled_lr = g[i].scaled_lr;
    SetupGroup& U = su.g[i];
    U.first = first;
    U.mblocks = D.mchunks; U.per = D.mchunks + (S.npT * 64 * S.rp + ADD_ELEMS - 1) / ADD_ELEMS;
    U.end = (int)(adds += (long long)g[i].cnt * U.per);
    U.m = g[i].m; U.n = g[i].n; U.r = g[i].r; U.rp = S.rp; U.np = S.np; U.npR = S.npT * 64;
    U.Qw = D.Qw; U.any = D.any;
    first += g[i].cnt;
  }
  a.ngroups = n;
  for (int q = 0; q < DA_QUEUES; ++q)
    for (int i = 0; i < n; ++i)
      for (int k = 0; k < PHASES; ++k) a.total[q] += a.g[i].nq[q] * tasks_of(a.g[i], k);
  a.spin_limit = 200000000ull;   // 2 s of the 100 MHz counter
  a.x_f32 = c.x_dtype == DA_F32; a.q_f32 = c.q_dtype == DA_F32;
  a.ef_alpha = c.ef_alpha; a.decay = c.decay; a.eps = c.eps;
  su.zblocks = (su.nzero + 255) / 256;
  su.ngroups = n; su.g_f32 = c.g_dtype == DA_F32; su.q_f32 = c.q_dtype == DA_F32;
  const dim3 block(256), setup((unsigned)(su.zblocks + adds));
  if (bf) hipLaunchKernelGGL(dion_small_setup_kernel<true>, setup, block, 0, s, su);
  else hipLaunchKernelGGL(dion_small_setup_kernel<false>, setup, block, 0, s, su);
  const int rc = da_launch_status();
  if (rc) return rc;
  return bf ? launch_all<true>(a, s) : launch_all<false>(a, s);
}
