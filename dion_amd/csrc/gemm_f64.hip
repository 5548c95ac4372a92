// Batched fp64 GEMM on the matrix cores (v_mfma_f64_16x16x4_f64) for the CholeskyQR
// orthonormalisation of Dion's P factor: the r x r Gram matrix P^T P (its condition number
// is the square of P's, hence fp64), the blocked Cholesky's panel / trailing updates and
// the blocked triangular solve P R^-1.
//
//   C[b] (M x N) = alpha * sum_k Aop[b](i,k) * Bop[b](j,k) + beta * E[b]
//
// 256 threads (2 x 2 wavefronts) per 64 x 64 tile; each wavefront owns 32 x 32 as 2 x 2 accumulators of 16 x 16.
// Interior tiles run a ring of two stages filled by direct-to-LDS loads (ring_loop): a stage 128 bytes deep costs a wavefront four
// load instructions and no registers, ALU work or LDS stores, and its 16 KB leave room for five workgroups on a compute unit.
// 48 Gram products of 768 x 768: 394 us with stages through registers, 375 now (63 TFLOP/s of 78.6); with rings of three and four
// stages, three and two workgroups, 453 and 532: what hides the latency here are the other workgroups.
// Other tiles go through registers, 16 k per stage, k-major LDS tiles, with the loads of the next stage in flight during the MFMAs.
// The same template is instantiated for fp32 (v_mfma_f32_16x16x4_f32; the polishing passes); the
// result may be stored as fp32 or bf16, and a block-triangular B operand shortens the sum per
// column tile.
#include "gemm_f64.h"
#include "mfma_tile.h"

namespace {

constexpr int RK = 16;             // depth of a stage through registers

// ---- the K loop of interior tiles: direct-to-LDS loads, a ring of two stages ------------------------------------------------
// A stage is 128 bytes deep: 16 k (fp64) or 32 k (fp32).  LDS layouts of an operand of R rows:
//   k-contiguous: [R][128 bytes], 16-byte chunks exchanged by (row >> 1) & 7: the 16 rows x 4 k of an operand read cover every bank once;
//   k-strided:    [depth][R elements] as in memory, chunks exchanged by k so that the k of a read fall into different banks.
template <typename T> struct Ring {
  static constexpr int D = 128 / (int)sizeof(T);                     // depth
  static constexpr int EPC = 16 / (int)sizeof(T);                    // elements of a chunk
  static constexpr int bytes(int rows) { return rows * 128; }
  // chunk exchange of a k-strided row
  static __device__ __forceinline__ int ks_chunk(int c, int k) { return sizeof(T) == 8 ? c ^ ((k & 1) << 3) : c ^ ((k & 3) << 2); }
};
// Requests one operand's stage: wavefront instruction i of R / 8 in all fills the 1 KB block i, lane p its p-th 16 bytes.
template <typename T, bool KS, int R>
struct RingAddr {
  static constexpr int PER = R / 32;          // instructions per wavefront (4 wavefronts)
  const char* base;
  unsigned off[PER];
  unsigned step;
  __device__ __forceinline__ RingAddr(const T* p, int ld, int row0, int k0, int wave, int lane) {
    typedef Ring<T> G;
    if (!KS) {
      base = reinterpret_cast<const char*>(p + (long long)row0 * ld + k0);
      step = 128u;
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int row = (i * 4 + wave) * 8 + (lane >> 3);
        off[i] = (unsigned)(row * ld) * (unsigned)sizeof(T) + (unsigned)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
      }
    } else {
      constexpr int CPR = R * (int)sizeof(T) / 16;   // chunks of a k-row
      base = reinterpret_cast<const char*>(p + (long long)k0 * ld + row0);
      step = (unsigned)(G::D * ld) * (unsigned)sizeof(T);
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int c = (i * 4 + wave) * 64 + lane, k = c / CPR;
        off[i] = (unsigned)(k * ld) * (unsigned)sizeof(T) + (unsigned)G::ks_chunk(c % CPR, k) * 16u;
      }
    }
  }
  __device__ __forceinline__ void request(unsigned lds, int wave) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      dma16(base, off[i], lds + (i * 4 + wave) * 1024);
      off[i] += step;
    }
  }
};
template <typename T, bool KS, int R> __device__ __forceinline__ T ring_read(const char* st, int row, int k) {
  if (!KS) {
    const int byte = k * (int)sizeof(T);
    return *reinterpret_cast<const T*>(st + row * 128 + (((byte >> 4) ^ ((row >> 1) & 7)) << 4) + (byte & 15));
  }
  const int byte = row * (int)sizeof(T);
  return *reinterpret_cast<const T*>(st + k * (R * (int)sizeof(T)) + (Ring<T>::ks_chunk(byte >> 4, k) << 4) + (byte & 15));
}
// a tile's operand within reach of 32-bit offsets
template <typename T, bool KS> __device__ __forceinline__ bool ring_span(int ld, int K) {
  return (long long)(KS ? K : 64) * ld * (long long)sizeof(T) + (KS ? 512 : (long long)K * (long long)sizeof(T)) < (1LL << 32);
}
// acc[TI][2] += A-rows (RA of them from m0) x B-rows (64 from n0) over KT stages from k0; lds: 2 * 128 * (RA + 64) bytes, free on
// entry.  No barrier behind the last stage.
template <typename T, bool A_KS, bool B_KS, int RA>
__device__ __forceinline__ void ring_loop(typename Mfma<T>::acc_t (&acc)[RA / 32][2], const T* A, int lda, int m0, const T* B, int ldb, int n0,
                                          int k0, int KT, char* lds, int lane, int wave, int wm, int wn) {
  typedef Ring<T> G;
  constexpr int TI = RA / 32, ST = 128 * (RA + 64);
  if (KT <= 0) return;
  RingAddr<T, A_KS, RA> ra(A, lda, m0, k0, wave, lane);
  RingAddr<T, B_KS, 64> rb(B, ldb, n0, k0, wave, lane);
  const unsigned l0 = lds_addr(lds);
  const int lc = lane & 15, lg = lane >> 4;
  ra.request(l0, wave);
  rb.request(l0 + RA * 128, wave);
  for (int kt = 0; kt < KT; ++kt) {
    dma_wait();
    __syncthreads();
    if (kt + 1 < KT) {   // into the buffer whose last readers are past the barrier
      const unsigned st = l0 + ((kt + 1) & 1) * ST;
      ra.request(st, wave);
      rb.request(st + RA * 128, wave);
    }
    const char* const sa = lds + (kt & 1) * ST;
    const char* const sb = sa + RA * 128;
#pragma unroll
    for (int ks = 0; ks < G::D / 4; ++ks) {
      const int k = ks * 4 + lg;
      T af[TI], bf[2];
#pragma unroll
      for (int i = 0; i < TI; ++i) af[i] = ring_read<T, A_KS, RA>(sa, wm * (RA / 2) + i * 16 + lc, k);
#pragma unroll
      for (int j = 0; j < 2; ++j) bf[j] = ring_read<T, B_KS, 64>(sb, wn * 32 + j * 16 + lc, k);
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = Mfma<T>::mma(af[i], bf[j], acc[i][j]);
    }
  }
}


template <bool KS, typename T>
__device__ __forceinline__ void fetch(T (&v)[4], const T* __restrict__ base, int ld, int row0, int k0,
                                      int rows, int K, int tid) {
  // the thread's 4 elements are contiguous in memory in either layout
  const int outer = KS ? k0 + (tid >> 4) : row0 + (tid >> 2);
  const int inner = KS ? row0 + (tid & 15) * 4 : k0 + (tid & 3) * 4;
  const int outer_n = KS ? K : rows, inner_n = KS ? rows : K;
  const T* p = base + (long long)outer * ld + inner;
  if (outer < outer_n && inner + 3 < inner_n && ((reinterpret_cast<uintptr_t>(p) & (2 * sizeof(T) - 1)) == 0)) {
    typedef T pair_t __attribute__((ext_vector_type(2)));   // 16 bytes (fp64) / 8 (fp32) / 4 (bf16) per access
    const pair_t lo = *reinterpret_cast<const pair_t*>(p);
    const pair_t hi = *reinterpret_cast<const pair_t*>(p + 2);
    v[0] = lo.x; v[1] = lo.y; v[2] = hi.x; v[3] = hi.y;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (outer < outer_n && inner + e < inner_n) ? p[e] : T(0);
  }
}

// A stage goes to the k-major LDS tile lds[k][row] (row pitch P).
template <bool KS, int P, typename T>
__device__ __forceinline__ void put(T* lds, const T (&v)[4], int tid) {
  if (!KS) {
    const int r = tid >> 2, k4 = (tid & 3) * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) lds[(k4 + e) * P + r] = v[e];
  } else {
    const int k = tid >> 4, r4 = (tid & 15) * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) lds[k * P + r4 + e] = v[e];
  }
}

// BT x BT output tile, 256 threads as 2 x 2 wavefronts of (BT / 2) x (BT / 2) each.  (Tiles of 128 -- half the operand bytes per flop, but
// 200 VGPRs and 64 KB of LDS in fp64, two workgroups per CU instead of five -- were 10 % slower on the orthonormaliser's large
// products and equal on the small ones.)
constexpr int BT = 64;
template <typename T, bool A_KS, bool B_KS, bool SYM>
__global__ __launch_bounds__(256) void gemm_f64_kernel(RealGemmDesc<T> d) {
  typedef typename Mfma<T>::acc_t acc_t;
  constexpr int WT = BT / 2;         // wavefront tile
  constexpr int TI = WT / 16;        // 16 x 16 accumulators per wavefront and direction
  __shared__ __attribute__((aligned(16))) char lds[2 * 128 * 128];
  T* const lds_a = reinterpret_cast<T*>(lds);
  T* const lds_b = lds_a + 2 * RK * BT;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int tiles_m = (d.M + BT - 1) / BT, tiles_n = (d.N + BT - 1) / BT;
  const bool tri = SYM || d.lower_only;
  // SYM: M == N; lower_only: M >= N, column tile c holds the tiles_m - c row tiles from the diagonal down
  const int per_batch = tri ? tiles_n * tiles_m - tiles_n * (tiles_n - 1) / 2 : tiles_m * tiles_n;
  const int split = blockIdx.y;  // split-K slice
  const int b = blockIdx.x / per_batch;
  if (d.gate && (d.gate[b] != 0) != (d.gate_want != 0)) return;
  int t = blockIdx.x - b * per_batch;
  int ti, tj;
  if (tri) {
    ti = 0;
    int len = tiles_m;
    while (t >= len) { t -= len; ++ti; --len; }
    tj = ti + t;
    if (!SYM) { const int x = ti; ti = tj; tj = x; }   // lower triangle: row tile >= column tile
  } else if (d.k_tri) {
    // longest sums (last column tiles) first
    tj = tiles_n - 1 - t / tiles_m;
    ti = t - (tiles_n - 1 - tj) * tiles_m;
  } else {
    ti = t / tiles_n;
    tj = t - ti * tiles_n;
  }
  const int m0 = ti * BT, n0 = tj * BT;
  const T* A = d.A + (long long)b * d.sA;
  const T* B = d.B + (long long)b * d.sB;
  const int Keff = d.k_tri && n0 + BT < d.K ? n0 + BT : d.K;

  acc_t acc[TI][TI];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TI; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  // double buffered: the global loads of stage s+1 are in flight while stage s is multiplied
  const int KT_all = (Keff + RK - 1) / RK;
  const int per_split = (KT_all + (int)gridDim.y - 1) / (int)gridDim.y;
  const int kt0 = split * per_split;
  const int KT = KT_all - kt0 < per_split ? KT_all - kt0 : per_split;   // may be <= 0 for the last slices
  T pa[4], pb[4];
#define DA_RFETCH(kt)                                                                               \
  do {                                                                                              \
    fetch<A_KS>(pa, A, d.lda, m0, (kt) * RK, d.M, Keff, tid);                                       \
    fetch<B_KS>(pb, B, d.ldb, n0, (kt) * RK, d.N, Keff, tid);                                       \
  } while (0)
#define DA_RPUT(buf)                                                                                \
  do {                                                                                              \
    put<A_KS, BT>(lds_a + (buf) * RK * BT, pa, tid);                                                \
    put<B_KS, BT>(lds_b + (buf) * RK * BT, pb, tid);                                                \
  } while (0)
#define DA_RMMA(sa, sb)                                                                             \
  _Pragma("unroll") for (int ks = 0; ks < RK / 4; ++ks) {                                           \
    const int k = ks * 4 + (lane >> 4);                                                             \
    T af[TI], bfv[TI];                                                                              \
    _Pragma("unroll") for (int i = 0; i < TI; ++i) af[i] = (sa)[k * BT + wm * WT + i * 16 + (lane & 15)];  \
    _Pragma("unroll") for (int j = 0; j < TI; ++j) bfv[j] = (sb)[k * BT + wn * WT + j * 16 + (lane & 15)]; \
    _Pragma("unroll") for (int i = 0; i < TI; ++i)                                                  \
      _Pragma("unroll") for (int j = 0; j < TI; ++j) acc[i][j] = Mfma<T>::mma(af[i], bfv[j], acc[i][j]);    \
  }
  // Interior tile with 16-byte aligned operand rows, whole stages, operands within reach of the loads' 32-bit offsets
  const bool interior = m0 + BT <= d.M && n0 + BT <= d.N && Keff % Ring<T>::D == 0 && kt0 * RK % Ring<T>::D == 0 && KT * RK % Ring<T>::D == 0 &&
                        ring_span<T, A_KS>(d.lda, Keff) && ring_span<T, B_KS>(d.ldb, Keff) &&
                        ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15) == 0 &&
                        (((long long)d.lda | (long long)d.ldb) * (long long)sizeof(T)) % 16 == 0;
  if (interior) {
    ring_loop<T, A_KS, B_KS, 64>(acc, A, d.lda, m0, B, d.ldb, n0, kt0 * RK, KT * RK / Ring<T>::D, lds, lane, wave, wm, wn);
  } else {

    if (KT > 0) {
      DA_RFETCH(kt0);
      DA_RPUT(0);
    }
    __syncthreads();
    for (int kt = 0; kt < KT; ++kt) {
      const T* sa = lds_a + (kt & 1) * RK * BT;
      const T* sb = lds_b + (kt & 1) * RK * BT;
      const bool more = kt + 1 < KT;
      if (more) DA_RFETCH(kt0 + kt + 1);
      DA_RMMA(sa, sb)
      if (more) DA_RPUT((kt + 1) & 1);
      __syncthreads();
    }
  }
#undef DA_RMMA
#undef DA_RFETCH
#undef DA_RPUT

  if (d.c_store != DA_STORE_NATIVE) {   // rounded once to the storage dtype; no E, no split, no mirror (checked on the host)
    char* Cc = reinterpret_cast<char*>(d.C) + (long long)b * d.sC * (d.c_store == DA_STORE_F32 ? 4 : 2);
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TI; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int m = m0 + wm * WT + i * 16 + Mfma<T>::row(v, lane);
          const int n = n0 + wn * WT + j * 16 + (lane & 15);
          if (m < d.M && n < d.N) {
            const float o = (float)((T)d.alpha * acc[i][j][v]);
            const long long at = (long long)m * d.ldc + n;
            if (d.c_store == DA_STORE_F32) reinterpret_cast<float*>(Cc)[at] = o;
            else reinterpret_cast<bf16_t*>(Cc)[at] = f2bf(o);
          }
        }
    return;
  }
  T* C = d.C + (long long)b * d.sC + (long long)split * d.split_stride;   // each K slice has an output of its own
  const T* E = d.E ? d.E + (long long)b * d.sE : nullptr;
  const bool mirror = SYM && (ti != tj);
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TI; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = m0 + wm * WT + i * 16 + Mfma<T>::row(v, lane);
        const int n = n0 + wn * WT + j * 16 + (lane & 15);
        if (m < d.M && n < d.N) {
          T o = (T)d.alpha * acc[i][j][v];
          if (E) o += (T)d.beta * E[(long long)m * d.lde + n];
          C[(long long)m * d.ldc + n] = o;
          if (mirror) C[(long long)n * d.ldc + m] = o;
        }
      }
}

template <typename T>
long long blocks_of(const RealGemmDesc<T>& d) {
  const long long tiles_m = (d.M + BT - 1) / BT, tiles_n = (d.N + BT - 1) / BT;
  return ((d.symmetric || d.lower_only) ? tiles_n * tiles_m - tiles_n * (tiles_n - 1) / 2 : tiles_m * tiles_n) * d.batch;
}

template <typename T, bool A_KS, bool B_KS, bool SYM>
int launch(const RealGemmDesc<T>& d, hipStream_t s) {
  const long long blocks = blocks_of(d);
  const bool auto_split = d.split_k < 0 && !d.E && d.c_store == DA_STORE_NATIVE;
  int split = d.split_k > 1 && !d.E ? d.split_k : 1;
  if (auto_split) split = da_auto_split(blocks, d.K);
  if (split > 1 && d.split_stride < (long long)d.sC * d.batch) return DA_ERR_ARG;
  if (blocks <= 0 || blocks > 0x7fffffffLL) return DA_ERR_LIMIT;
  hipLaunchKernelGGL((gemm_f64_kernel<T, A_KS, B_KS, SYM>), dim3((unsigned)blocks, split), dim3(256), 0, s, d);
  return da_launch_status();
}

// ---- P <- P R^-1 with R = L^T: all block columns in one launch -------------------------------------------------------------
//
//   X(:, j) = (P(:, j) - sum over k < j of X(:, k) L(j, k)^T) D_j^T,  D_j = L_jj^-1,  j in blocks of 64
//
// A workgroup owns SR rows of one matrix and walks its block columns: the sum is the K loop of the GEMM above on the X it has stored
// itself (it reads its own stores back through its compute unit's L1), the difference goes to LDS as the operand of the
// product with D_j, whose fragments come straight from memory.
//
// What bounds it: the fp64 matrix cores, and the last workgroups: SR = 32 gives a 768-row matrix 24 of them, five to a compute unit
// at a time (the registers are held to that), so that a bucket of a few dozen matrices runs in one round.  48 matrices of
// 768 x 768: 585 us, 40 TFLOP/s; as fifteen products over panels of four block columns (1 launch each) 570 us plus 85 us for the
// blocks of the panels' inverses, which are no longer needed; and as the pass over flagged matrices one launch that finds
// nothing instead of one per block column.  (Four workgroups a compute unit: 618.)
// Eight matrices at a time go to the eight XCDs (a matrix's workgroups read the same L), the up to seven that are left to all of them:
// to one XCD each they left the others idle (12 matrices of 3072 x 768: the whole orthonormaliser 1628 us, so 1508; 9: 1482 / 1284).
constexpr int SR = 32;
template <typename T, bool INTERIOR>
__device__ __forceinline__ void solve_rows_of(T* __restrict__ P, const T* __restrict__ L, const T* __restrict__ D, int rows, int r, int row0,
                                              T* lds, int tid, int lane, int wm, int wn) {
  typedef typename Mfma<T>::acc_t acc_t;
  constexpr int CB = 64;
  const int lc = lane & 15, lg = lane >> 4;
  T* const la = lds;                     // checked loop: [2][RK][SR]
  T* const lb = lds + 2 * RK * SR;       // ... [2][RK][CB]
  for (int n0 = 0; n0 < r; n0 += CB) {
    const int nb = INTERIOR || r - n0 >= CB ? CB : r - n0;
    acc_t old[2], acc[2];
    T* const own = P + (long long)(row0 + wm * 16) * r + n0 + wn * 32 + lc;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = Mfma<T>::row(v, lane);
        old[j][v] = INTERIOR || (row0 + wm * 16 + m < rows && wn * 32 + j * 16 + lc < nb) ? own[(long long)m * r + j * 16] : T(0);
        acc[j][v] = T(0);
      }
    if constexpr (INTERIOR) {
      // (what this workgroup stored is read back past nothing but its own L1: the stores are acknowledged first)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      acc_t ac2[1][2] = {{acc[0], acc[1]}};
      if (n0 > 0) ring_loop<T, false, false, SR>(ac2, P, r, row0, L, r, n0, 0, n0 / Ring<T>::D, reinterpret_cast<char*>(lds), lane, wm * 2 + wn, wm, wn);
      acc[0] = ac2[0][0];
      acc[1] = ac2[0][1];
      __syncthreads();
    } else {
      const int KT = n0 / RK;
      T pa[4], pb[4];
      auto stage_in = [&](int kt) __attribute__((always_inline)) {
        if (tid < 4 * SR) fetch<false>(pa, P, r, row0, kt * RK, rows, n0, tid);
        fetch<false>(pb, L, r, n0, kt * RK, n0 + nb, n0, tid);
      };
      auto stage_out = [&](int buf) __attribute__((always_inline)) {
        if (tid < 4 * SR) put<false, SR>(la + buf * RK * SR, pa, tid);
        put<false, CB>(lb + buf * RK * CB, pb, tid);
      };
      if (KT > 0) {
        stage_in(0);
        stage_out(0);
      }
      __syncthreads();
      for (int kt = 0; kt < KT; ++kt) {
        const T* const sa = la + (kt & 1) * RK * SR;
        const T* const sb = lb + (kt & 1) * RK * CB;
        const bool more = kt + 1 < KT;
        if (more) stage_in(kt + 1);
#pragma unroll
        for (int ks = 0; ks < RK / 4; ++ks) {
          const int k = ks * 4 + lg;
          const T af = sa[k * SR + wm * 16 + lc];
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[j] = Mfma<T>::mma(af, sb[k * CB + wn * 32 + j * 16 + lc], acc[j]);
        }
        if (more) stage_out((kt + 1) & 1);
        __syncthreads();
      }
    }
    // the difference, [column][row], then its product with D_j^T: D[n][k] at n = 32 wn + 16 j + lc, k = 4 ks + lg
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        lds[(wn * 32 + j * 16 + lc) * SR + wm * 16 + Mfma<T>::row(v, lane)] = old[j][v] - acc[j][v];
        acc[j][v] = T(0);
      }
    __syncthreads();
    const T* const dj = D + (long long)(n0 + wn * 32 + lc) * r + n0 + lg;
#pragma unroll
    for (int h = 0; h < 4; ++h) {   // (in quarters: the registers decide how many workgroups a compute unit holds)
      T df[2][CB / 16];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int ks = 0; ks < CB / 16; ++ks) {
          const int k = h * (CB / 4) + ks * 4;
          df[j][ks] = INTERIOR || (wn * 32 + j * 16 + lc < nb && k + lg < nb) ? dj[(long long)j * 16 * r + k] : T(0);
        }
#pragma unroll
      for (int ks = 0; ks < CB / 16; ++ks) {
        const T af = lds[(h * (CB / 4) + ks * 4 + lg) * SR + wm * 16 + lc];
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = Mfma<T>::mma(af, df[j][ks], acc[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = Mfma<T>::row(v, lane);
        if (INTERIOR || (row0 + wm * 16 + m < rows && wn * 32 + j * 16 + lc < nb)) own[(long long)m * r + j * 16] = acc[j][v];
      }
    __syncthreads();   // the stored columns are the next block column's operand; the buffers are free
  }
}

template <typename T>
__global__ __launch_bounds__(256, 5) void solve_rows_kernel(T* __restrict__ Pm, const T* __restrict__ Lm, const T* __restrict__ Dm, int rows,
                                                         int r, int batch, int blocks, const int* gate, int gate_want) {
  __shared__ __attribute__((aligned(16))) T lds[2 * 128 * (SR + 64) / sizeof(T)];
  static_assert(2 * 128 * (SR + 64) / sizeof(T) >= 64 * SR && 128 / sizeof(T) >= RK, "room for the difference and for the stages of the checked loop");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int b = blockIdx.x / blocks, blk = blockIdx.x - b * blocks;
  if ((int)blockIdx.x < (batch & ~7) * blocks) {
    const int idx = blockIdx.x >> 3, m = idx / blocks;
    b = m * 8 + (blockIdx.x & 7);
    blk = idx - m * blocks;
  }
  if (gate && (gate[b] != 0) != (gate_want != 0)) return;
  T* const P = Pm + (long long)b * rows * r;
  const T* const L = Lm + (long long)b * r * r;
  const T* const D = Dm + (long long)b * r * r;
  const int row0 = blk * SR;
  const bool interior = row0 + SR <= rows && r % 64 == 0 && ((reinterpret_cast<uintptr_t>(Pm) | reinterpret_cast<uintptr_t>(Lm)) & 15) == 0;
  if (interior) solve_rows_of<T, true>(P, L, D, rows, r, row0, lds, tid, lane, wave >> 1, wave & 1);
  else solve_rows_of<T, false>(P, L, D, rows, r, row0, lds, tid, lane, wave >> 1, wave & 1);
}

template <typename T>
int solve_rows(T* P, const T* L, const T* D, int batch, int rows, int r, DaGate g, hipStream_t s) {
  if (!P || !L || !D || batch <= 0 || rows <= 0 || r <= 0) return DA_ERR_ARG;
  const int blocks = (rows + SR - 1) / SR;
  const long long grid = (long long)blocks * batch;
  if (grid > 0x7fffffffLL) return DA_ERR_LIMIT;
  hipLaunchKernelGGL(solve_rows_kernel<T>, dim3((unsigned)grid), dim3(256), 0, s, P, L, D, rows, r, batch, blocks, g.flags, g.want);
  return da_launch_status();
}

// Element-wise conversions of `batch` matrices of `per` contiguous elements; blockIdx.y = matrix.
__device__ __forceinline__ bool gate_open(const int* flags, int want, int b) {
  return !flags || (flags[b] != 0) == (want != 0);
}

template <typename T, typename R>
__global__ __launch_bounds__(256) void cvt_up_kernel(const T* __restrict__ src, R* __restrict__ dst, long long per,
                                                     const int* gate, int want) {
  const long long b = blockIdx.y;
  if (!gate_open(gate, want, (int)b)) return;
  src += b * per; dst += b * per;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < per; i += (long long)gridDim.x * 256)
    dst[i] = (R)ld_as_float<T>(src + i);
}

template <typename T, typename R>
__global__ __launch_bounds__(256) void cvt_down_kernel(const R* __restrict__ src, T* __restrict__ dst, long long per,
                                                       const int* gate, int want) {
  const long long b = blockIdx.y;
  if (!gate_open(gate, want, (int)b)) return;
  src += b * per; dst += b * per;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < per; i += (long long)gridDim.x * 256)
    st_from_float<T>(dst + i, (float)src[i]);
}

// R (fp64 / fp32) -> fp32 (unless dst is null) and, if `low` is given, the same values rounded once more to bf16
template <typename R>
__global__ __launch_bounds__(256) void cvt_f32_low_kernel(const R* __restrict__ src, float* __restrict__ dst,
                                                          bf16_t* __restrict__ low, long long per, const int* gate,
                                                          int want) {
  const long long b = blockIdx.y;
  if (!gate_open(gate, want, (int)b)) return;
  src += b * per;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < per; i += (long long)gridDim.x * 256) {
    const float v = (float)src[i];
    if (dst) dst[b * per + i] = v;
    if (low) low[b * per + i] = f2bf(v);
  }
}

// fp64 -> h + l (bf16 each): h = the value rounded to bf16, l = what is left of it, rounded to bf16
__global__ __launch_bounds__(256) void cvt_hl_kernel(const double* __restrict__ src, bf16_t* __restrict__ h,
                                                     bf16_t* __restrict__ l, long long per, const int* gate, int want) {
  const long long b = blockIdx.y;
  if (!gate_open(gate, want, (int)b)) return;
  src += b * per;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < per; i += (long long)gridDim.x * 256) {
    const float v = (float)src[i];
    const bf16_t hi = f2bf(v);
    h[b * per + i] = hi;
    l[b * per + i] = f2bf(v - bf2f(hi));
  }
}

inline dim3 cvt_grid(long long per, int batch) {
  long long b = (per + 255) / 256;
  const long long cap = 8192 / batch > 0 ? 8192 / batch : 1;
  if (b > cap) b = cap;
  return dim3((unsigned)(b < 1 ? 1 : b), (unsigned)batch);
}

template <typename T>
int gemm_real(const RealGemmDesc<T>& d, hipStream_t s) {
  if (!d.A || !d.B || !d.C || d.M <= 0 || d.N <= 0 || d.K < 0 || d.batch <= 0) return DA_ERR_ARG;
  if (d.lower_only && (d.M < d.N || d.symmetric)) return DA_ERR_ARG;
  if (d.c_store != DA_STORE_NATIVE && d.c_store != DA_STORE_BF16 && d.c_store != DA_STORE_F32) return DA_ERR_DTYPE;
  if (d.c_store != DA_STORE_NATIVE && (d.E || d.split_k > 1 || d.symmetric)) return DA_ERR_ARG;
  if (d.k_tri && (d.symmetric || d.lower_only || d.split_k > 1)) return DA_ERR_ARG;
  if (d.symmetric) {
    if (d.M != d.N || !d.a_kstrided || !d.b_kstrided) return DA_ERR_ARG;  // only the Gram form A^T A
    return launch<T, true, true, true>(d, s);
  }
  if (!d.a_kstrided && !d.b_kstrided) return launch<T, false, false, false>(d, s);
  if (!d.a_kstrided && d.b_kstrided) return launch<T, false, true, false>(d, s);
  if (d.a_kstrided && !d.b_kstrided) return launch<T, true, false, false>(d, s);
  return launch<T, true, true, false>(d, s);
}

template <typename R>
int cvt_up(const void* src, int src_dtype, R* dst, long long per, int batch, DaGate g, hipStream_t s) {
  if (per <= 0 || batch <= 0 || batch > 65535) return DA_ERR_ARG;
  if (src_dtype == DA_BF16)
    hipLaunchKernelGGL((cvt_up_kernel<bf16_t, R>), cvt_grid(per, batch), dim3(256), 0, s, static_cast<const bf16_t*>(src), dst, per, g.flags, g.want);
  else if (src_dtype == DA_F32)
    hipLaunchKernelGGL((cvt_up_kernel<float, R>), cvt_grid(per, batch), dim3(256), 0, s, static_cast<const float*>(src), dst, per, g.flags, g.want);
  else
    return DA_ERR_DTYPE;
  return da_launch_status();
}

}  // namespace

int da_gemm_f64(const Gemm64Desc& d, hipStream_t s) { return gemm_real<double>(d, s); }
int da_gemm_f32s(const Gemm32Desc& d, hipStream_t s) { return gemm_real<float>(d, s); }
int da_solve_rows(double* P, const double* L, const double* D, int batch, int rows, int r, DaGate g, hipStream_t s) {
  return solve_rows<double>(P, L, D, batch, rows, r, g, s);
}
int da_solve_rows(float* P, const float* L, const float* D, int batch, int rows, int r, DaGate g, hipStream_t s) {
  return solve_rows<float>(P, L, D, batch, rows, r, g, s);
}

int da_cvt_to_f64(const void* src, int src_dtype, double* dst, long long per, int batch, DaGate g, hipStream_t s) {
  return cvt_up<double>(src, src_dtype, dst, per, batch, g, s);
}
int da_cvt_to_f32(const void* src, int src_dtype, float* dst, long long per, int batch, DaGate g, hipStream_t s) {
  return cvt_up<float>(src, src_dtype, dst, per, batch, g, s);
}
int da_cvt_from_f64(const double* src, void* dst, int dst_dtype, long long per, int batch, DaGate g, hipStream_t s) {
  if (per <= 0 || batch <= 0 || batch > 65535) return DA_ERR_ARG;
  if (dst_dtype == DA_BF16)
    hipLaunchKernelGGL((cvt_down_kernel<bf16_t, double>), cvt_grid(per, batch), dim3(256), 0, s, src, static_cast<bf16_t*>(dst), per, g.flags, g.want);
  else if (dst_dtype == DA_F32)
    hipLaunchKernelGGL((cvt_down_kernel<float, double>), cvt_grid(per, batch), dim3(256), 0, s, src, static_cast<float*>(dst), per, g.flags, g.want);
  else
    return DA_ERR_DTYPE;
  return da_launch_status();
}
int da_cvt_from_f32(const float* src, void* dst, int dst_dtype, long long per, int batch, DaGate g, hipStream_t s) {
  if (per <= 0 || batch <= 0 || batch > 65535) return DA_ERR_ARG;
  if (dst_dtype == DA_BF16)
    hipLaunchKernelGGL((cvt_down_kernel<bf16_t, float>), cvt_grid(per, batch), dim3(256), 0, s, src, static_cast<bf16_t*>(dst), per, g.flags, g.want);
  else if (dst_dtype == DA_F32)
    hipLaunchKernelGGL((cvt_down_kernel<float, float>), cvt_grid(per, batch), dim3(256), 0, s, src, static_cast<float*>(dst), per, g.flags, g.want);
  else
    return DA_ERR_DTYPE;
  return da_launch_status();
}
int da_cvt_f64_to_hl(const double* src, bf16_t* h, bf16_t* l, long long per, int batch, DaGate g, hipStream_t s) {
  if (per <= 0 || batch <= 0 || batch > 65535) return DA_ERR_ARG;
  hipLaunchKernelGGL(cvt_hl_kernel, cvt_grid(per, batch), dim3(256), 0, s, src, h, l, per, g.flags, g.want);
  return da_launch_status();
}
int da_cvt_f64_to_f32(const double* src, float* dst, bf16_t* low, long long per, int batch, DaGate g, hipStream_t s) {
  if (per <= 0 || batch <= 0 || batch > 65535) return DA_ERR_ARG;
  hipLaunchKernelGGL(cvt_f32_low_kernel<double>, cvt_grid(per, batch), dim3(256), 0, s, src, dst, low, per, g.flags, g.want);
  return da_launch_status();
}
int da_cvt_f32_to_bf16(const float* src, bf16_t* low, long long per, int batch, DaGate g, hipStream_t s) {
  if (per <= 0 || batch <= 0 || batch > 65535) return DA_ERR_ARG;
  hipLaunchKernelGGL(cvt_f32_low_kernel<float>, cvt_grid(per, batch), dim3(256), 0, s, src, static_cast<float*>(nullptr), low, per, g.flags, g.want);
  return da_launch_status();
}
