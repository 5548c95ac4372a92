// Tile products and the serial part of a factorisation for the kernels of small matrices and flagged factors (dion_small.hip, orth_flow.hip): 256 threads,
// operands from memory through registers into LDS, products on the matrix cores in bf16, fp32 and fp64.
#pragma once
#include "diag64.h"
#include "mfma_tile.h"

#pragma clang fp contract(off)

namespace {

constexpr int KD = 32;             // depth of an fp32 / fp64 stage
constexpr int STAGES64 = 2 * 2 * KD * 66 * 8;   // two stages of two fp64 operands of 64 rows: the largest user of the LDS

typedef double double2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4_un_t __attribute__((ext_vector_type(4), aligned(2)));   // an unaligned 16-byte access

// ---- operands ----------------------------------------------------------------------------------------------------------

// Element (row, k): p[row * ld + k], or p[k * ld + row] when `ks`.  EDGE: a caller's matrix of `rows` x `kmax`, of which
// anything beyond reads as zero; `last` = its elements - 8.  Otherwise a working matrix, padded to whole tiles.
template <typename E, bool EDGE> struct Opnd {
  const E* p;
  int ld, ks;
  int rows, kmax;
  long long last;
};
template <typename E> __device__ __forceinline__ Opnd<E, false> work(const void* p, int ld, int ks) {
  return Opnd<E, false>{static_cast<const E*>(p), ld, ks, 0, 0, 0};
}

// Pointers read from a table point to the compiler knows not what: a generic (flat) load counts as an LDS access as well, and every
// wait for an LDS read waits for it too.  These are global memory.
#define DA_GLOBAL __attribute__((address_space(1)))

// Eight consecutive elements as they came from memory: converted only when they go to LDS, so that the loads of the next
// stages stay in flight.
template <typename E> struct Raw { u32x4_t q[sizeof(E) / 2]; };
template <typename E> __device__ __forceinline__ Raw<E> load_raw(const E* p) {
  Raw<E> r;
#pragma unroll
  for (int i = 0; i < (int)(sizeof(E) / 2); ++i) {
    const u32x4_un_t x = *(const DA_GLOBAL u32x4_un_t*)(reinterpret_cast<const char*>(p) + 16 * i);
    r.q[i] = x;
  }
  return r;
}
template <typename T> __device__ __forceinline__ void unpack(const Raw<bf16_t>& r, T (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const unsigned w = r.q[0][i];
    v[2 * i] = (T)lo_f(w);
    v[2 * i + 1] = (T)hi_f(w);
  }
}
template <typename T> __device__ __forceinline__ void unpack(const Raw<float>& r, T (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const unsigned w = r.q[i >> 2][i & 3];
    v[i] = (T)__builtin_bit_cast(float, w);
  }
}
__device__ __forceinline__ void unpack(const Raw<double>& r, double (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const unsigned lo = r.q[i >> 1][2 * (i & 1)], hi = r.q[i >> 1][2 * (i & 1) + 1];
    v[i] = __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
  }
}
__device__ __forceinline__ float to_f(bf16_t x) { return bf2f(x); }
__device__ __forceinline__ float to_f(float x) { return x; }

// Eight elements from element offset `e`, of which n exist; the rest reads as zero.
template <typename E> __device__ __forceinline__ void load8(const E* p, long long e, int n, float (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = 0.f;
  if (n >= 8) {
    unpack(load_raw(p + e), v);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < n) v[i] = to_f(*(const DA_GLOBAL E*)(p + e + i));
  }
}

// Chunk c (eight elements) of a TB x depth-D tile: its (row, k) in the tile
template <int TB, int D>
__device__ __forceinline__ void chunk_at(int ks, int c, int& row, int& k) {
  row = ks ? (c % (TB / 8)) * 8 : c / (D / 8);
  k = ks ? c / (TB / 8) : (c % (D / 8)) * 8;
}
template <int TB, int D, typename E, bool EDGE>
__device__ __forceinline__ Raw<E> fetch_chunk(const Opnd<E, EDGE>& o, int c, int row0, int k0) {
  int row, k;
  chunk_at<TB, D>(o.ks, c, row, k);
  row += row0;
  k += k0;
  long long e = o.ks ? (long long)k * o.ld + row : (long long)row * o.ld + k;
  if (EDGE) e = e < o.last ? e : o.last;   // (inside the matrix whatever the chunk)
  return load_raw(o.p + e);
}
// what of a fetched chunk lies inside a caller's matrix; the rest becomes zero
template <int TB, int D, typename E>
__device__ __forceinline__ void mask_chunk(const Opnd<E, true>& o, Raw<E>& r, int c, int row0, int k0) {
  int row, k;
  chunk_at<TB, D>(o.ks, c, row, k);
  row += row0;
  k += k0;
  const int n = o.ks ? (k < o.kmax ? o.rows - row : 0) : (row < o.rows ? o.kmax - k : 0);
  if (n >= 8) return;
  const long long e = o.ks ? (long long)k * o.ld + row : (long long)row * o.ld + k;
  if (n > 0 && e > o.last) {   // the matrix's last elements: the load was moved back
    constexpr int W = 4 / sizeof(E);   // elements per word
#pragma unroll
    for (int i = 0; i < 8 / W; ++i) {
      unsigned w = 0;
      if (i * W < n) w = sizeof(E) == 4 ? ((const DA_GLOBAL unsigned*)(o.p + e))[i] : (unsigned)((const DA_GLOBAL unsigned short*)(o.p + e))[2 * i];
      if (sizeof(E) == 2 && i * W + 1 < n) w |= (unsigned)((const DA_GLOBAL unsigned short*)(o.p + e))[2 * i + 1] << 16;
      r.q[i >> 2][i & 3] = w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < (int)sizeof(E) * 2; ++i) {
      const unsigned w = r.q[i >> 2][i & 3];
      r.q[i >> 2][i & 3] = sizeof(E) == 4 ? (i < n ? w : 0u) : (2 * i + 1 < n ? w : 2 * i < n ? w & 0xffffu : 0u);
    }
  }
}

// ---- products of fp32 / fp64 tiles: LDS stages [k][row] with a pitch of TB + 2 (fp64) or TB + 4 (fp32) -------------------
template <typename T, int TB>
struct Real {
  static constexpr int P = TB + (sizeof(T) == 8 ? 2 : 4);
  static constexpr int OPND = KD * P;              // elements of one operand's stage
  static constexpr int NCH = TB * KD / 8;          // chunks per operand stage (at most one per thread)
};

struct NoTurn {
  template <typename V> __device__ __forceinline__ void operator()(V&, int, int) const {}
};
template <typename T, int TB, bool MASK, typename E, bool EDGE, typename Turn>
__device__ __forceinline__ void put_chunk(T* dst, const Opnd<E, EDGE>& o, Raw<E>& r, int c, int row0, int k0, Turn turn) {
  constexpr int P = Real<T, TB>::P;
  T v[8];
  if constexpr (EDGE && MASK) mask_chunk<TB, KD>(o, r, c, row0, k0);
  unpack(r, v);
  int row, k;
  chunk_at<TB, KD>(o.ks, c, row, k);
  turn(v, row0 + row, k0 + k);
  if (o.ks) {
#pragma unroll
    for (int i = 0; i < 8; ++i) dst[k * P + row + i] = v[i];
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) dst[(k + i) * P + row] = v[i];
  }
}

// The stages 0 .. n - 1 of a K loop through registers and two LDS buffers: `fetch(set, i)` requests stage i, `put(set, i, buffer,
// mask)` writes it to LDS, `acc(buffer)` multiplies.  With two register sets (AHEAD) two stages are on the way from memory while a
// third is multiplied.  The leading `full` stages need no mask, and the loop over them has no branch: where a fetch or a masked
// write is conditional the paths meet with an unknown number of loads on the way, and the compiler waits for all of them, so that every
// stage took a whole trip to memory (14 matrices of 341 to 2731 rows: P = B Q 36 -> 31 us, R = B^T P 52 -> 41).  Past the end the last
// stage is fetched again.
struct Masked { static constexpr bool value = true; };
struct Unmasked { static constexpr bool value = false; };
template <int AHEAD, typename Fetch, typename Put, typename Acc>
__device__ __forceinline__ void staged_loop(int n, int full, Fetch fetch, Put put, Acc acc) {
  const int last = n - 1;
  int i = 0;
  fetch(0, 0);
  if (AHEAD == 2) fetch(1, min(1, last));
  if (full > 0) put(0, 0, 0, Unmasked());
  else put(0, 0, 0, Masked());
  if (AHEAD == 2) {
    for (; i + 3 <= full; i += 2) {
      fetch(0, min(i + 2, last));
      __syncthreads();
      acc(0);
      put(1, i + 1, 1, Unmasked());
      fetch(1, min(i + 3, last));
      __syncthreads();
      acc(1);
      put(0, i + 2, 0, Unmasked());
    }
  } else {
    for (; i + 3 <= full; i += 2) {
      fetch(0, i + 1);
      __syncthreads();
      acc(0);
      put(0, i + 1, 1, Unmasked());
      fetch(0, i + 2);
      __syncthreads();
      acc(1);
      put(0, i + 2, 0, Unmasked());
    }
  }
  for (; i < n; i += 2) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int k = i + s;
      if (k >= n) break;
      if (k + AHEAD < n) fetch(AHEAD == 2 ? s : 0, k + AHEAD);
      __syncthreads();
      acc(s);
      if (k + 1 < n) {
        if (k + 1 < full) put(AHEAD == 2 ? s ^ 1 : 0, k + 1, s ^ 1, Unmasked());
        else put(AHEAD == 2 ? s ^ 1 : 0, k + 1, s ^ 1, Masked());
      }
    }
  }
  __syncthreads();
}
// how many of n stages, D deep from kbeg on, no chunk of which reaches past the operand's k or was loaded from another place than its
// own (fetch_chunk moves a load that would pass the matrix's end back; rows past the operand's end are read as whatever lies there,
// and the caller drops their results).  Of a caller's matrix the last stage never counts.  A k-strided chunk starts at k ld + row:
// ahead of the last k it is moved only where k ld > m n - 8, which takes rows shorter than eight elements, and then the last 7 / ld
// of the k before it are; they may lie in the stage before (ld = 3 and 65 k in stages of 64: k = 63).
template <typename E> __device__ __forceinline__ int full_stages(const Opnd<E, false>&, int, int n, int) { return n; }
template <typename E> __device__ __forceinline__ int full_stages(const Opnd<E, true>& o, int kbeg, int n, int D) {
  const int own = o.ks && o.ld < 8 ? o.kmax - 7 / o.ld : o.kmax;   // the k whose chunks lie where they belong
  return max(0, min(n - 1, (own - kbeg) / D));
}

// K loop of one TB x TB tile:  sum over k in [kbeg, kend) of A(row0 + i, k) B(col0 + j, k), for NB column operands; `mma`
// accumulates one stage of KD from the operands' LDS buffers (A first); `turn(v, col, k)` maps the chunk (col, k ..) of a column
// operand on its way to LDS.  Of fp64 64-tiles one stage is on the way (two take too many registers).
template <typename T, int TB, int NB, typename OA, typename OB, typename Mma, typename Turn>
__device__ __forceinline__ void real_loop(const OA& A, const OB (&B)[NB], int row0, int col0, int kbeg, int kend, T* lds, int tid,
                                          Mma mma, Turn turn) {
  typedef Real<T, TB> L;
  constexpr int STG = (1 + NB) * L::OPND;
  const int c = tid & (L::NCH - 1);
  const bool own = tid < L::NCH;
  const int n = (kend - kbeg + KD - 1) / KD;
  decltype(fetch_chunk<TB, KD>(A, c, row0, kbeg)) va[2];
  decltype(fetch_chunk<TB, KD>(B[0], c, col0, kbeg)) vb[2][NB];
  staged_loop<sizeof(T) == 8 && TB == 64 ? 1 : 2>(n, min(full_stages(A, kbeg, n, KD), full_stages(B[0], kbeg, n, KD)),
      [&](int s, int i) {
    const int k0 = kbeg + i * KD;
    va[s] = fetch_chunk<TB, KD>(A, c, row0, k0);
#pragma unroll
    for (int o = 0; o < NB; ++o) vb[s][o] = fetch_chunk<TB, KD>(B[o], c, col0, k0);
  },
      [&](int s, int i, int buf, auto mask) {
    const int k0 = kbeg + i * KD;
    if (own) {
      put_chunk<T, TB, decltype(mask)::value>(lds + buf * STG, A, va[s], c, row0, k0, NoTurn());
#pragma unroll
      for (int o = 0; o < NB; ++o) put_chunk<T, TB, decltype(mask)::value>(lds + buf * STG + (1 + o) * L::OPND, B[o], vb[s][o], c, col0, k0, turn);
    }
  },
      [&](int buf) { mma(lds + buf * STG); });
}

// fp64 (and fp32 in 32-tiles): v_mfma_*_16x16x4, four wavefronts of TB/2 x TB/2
template <typename T, int TB>
struct Acc16 {
  static constexpr int NBK = TB / 32, P = Real<T, TB>::P, H = TB / 2;
  typename Mfma<T>::acc_t acc[NBK][NBK];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < NBK; ++i)
#pragma unroll
      for (int j = 0; j < NBK; ++j) acc[i][j] = typename Mfma<T>::acc_t{0, 0, 0, 0};
  }
  __device__ __forceinline__ void stage(const T* sa, const T* sb, int lane, int wm, int wn) {
#pragma unroll
    for (int ks = 0; ks < KD / 4; ++ks) {
      const int k = ks * 4 + (lane >> 4);
      T af[NBK], bf[NBK];
#pragma unroll
      for (int i = 0; i < NBK; ++i) af[i] = sa[k * P + wm * H + i * 16 + (lane & 15)];
#pragma unroll
      for (int j = 0; j < NBK; ++j) bf[j] = sb[k * P + wn * H + j * 16 + (lane & 15)];
#pragma unroll
      for (int i = 0; i < NBK; ++i)
#pragma unroll
        for (int j = 0; j < NBK; ++j) acc[i][j] = Mfma<T>::mma(af[i], bf[j], acc[i][j]);
    }
  }
  // to the staging area d[row][col], pitch TB + 2; ends with a barrier
  __device__ __forceinline__ void out(T* d, int lane, int wm, int wn) const {
#pragma unroll
    for (int i = 0; i < NBK; ++i)
#pragma unroll
      for (int j = 0; j < NBK; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          d[(wm * H + i * 16 + Mfma<T>::row(v, lane)) * (TB + 2) + wn * H + j * 16 + (lane & 15)] = acc[i][j][v];
    __syncthreads();
  }
};
template <typename T, int TB, typename OA, typename OB, typename Turn = NoTurn>
__device__ __forceinline__ void tile16(const OA& A, const OB& B, int row0, int col0, int kbeg, int kend, T* lds, int tid, int lane,
                                       int wm, int wn, Turn turn = Turn()) {
  Acc16<T, TB> acc;
  acc.clear();
  const OB Bs[1] = {B};
  real_loop<T, TB, 1>(A, Bs, row0, col0, kbeg, kend, lds, tid,
                      [&](const T* st) { acc.stage(st, st + Real<T, TB>::OPND, lane, wm, wn); }, turn);
  acc.out(lds, lane, wm, wn);
}

// A 64 x 64 fp64 tile of two working matrices without LDS stages: every wavefront loads the operands of its 32 x 32 block as the
// fragments that the instruction takes, a 32-deep step ahead of the products and with no barrier between steps.  Lane l holds
// eight consecutive k of row (or column) l % 16, from 8 (l / 16) on, and the sum over k runs over them in parallel:
// k = 8 (l / 16) + s in the s-th product.  fp64 operands are k-strided (KS): 16 lanes of a load read 128 consecutive bytes; with k
// consecutive every lane reads a line of its own, and the L1's look-ups take longer than the products.
template <typename E, bool KS> struct DirectFrag {
  Raw<E> r;
  __device__ __forceinline__ void load(const E* p, int ld, int lane) { r = load_raw(p + (long long)(lane & 15) * ld + (lane >> 4) * 8); }
  __device__ __forceinline__ void get(double (&v)[8]) const { unpack(r, v); }
};
template <> struct DirectFrag<double, true> {   // (k-strided)
  double r[8];
  __device__ __forceinline__ void load(const double* p, int ld, int lane) {
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = p[(long long)((lane >> 4) * 8 + i) * ld + (lane & 15)];
  }
  __device__ __forceinline__ void get(double (&v)[8]) const {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = r[i];
  }
};
// A (the tile's first row and k = 0 at A) times B (k-strided, the tile's first column and k = 0 at B) over k < kend (a multiple of
// 64), to the staging area as tile16 leaves it.
template <bool KSA, typename E>
__device__ __forceinline__ void direct64(const E* A, int lda, const double* B, int ldb, int kend, double* d, int lane, int wm, int wn) {
  Acc16<double, 64> acc;
  acc.clear();
  DirectFrag<E, KSA> fa[2][2];
  DirectFrag<double, true> fb[2][2];
  A += wm * 32LL * (KSA ? 1 : lda);
  B += wn * 32;
  auto fetch = [&](int s, int k0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) fa[s][i].load(KSA ? A + (long long)k0 * lda + i * 16 : A + (long long)i * 16 * lda + k0, lda, lane);
#pragma unroll
    for (int j = 0; j < 2; ++j) fb[s][j].load(B + (long long)k0 * ldb + j * 16, ldb, lane);
    __builtin_amdgcn_sched_barrier(0);   // (here, and not behind the products)
  };
  auto products = [&](int s) {
    double a[2][8], b[2][8];
#pragma unroll
    for (int i = 0; i < 2; ++i) fa[s][i].get(a[i]);
#pragma unroll
    for (int j = 0; j < 2; ++j) fb[s][j].get(b[j]);
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc.acc[i][j] = Mfma<double>::mma(a[i][u], b[j][u], acc.acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  };
  fetch(0, 0);
  for (int k = 0; k < kend; k += 64) {   // (the last step is fetched twice: no load in a branch, as in staged_loop)
    fetch(1, k + 32);
    products(0);
    fetch(0, min(k + 64, kend - 32));
    products(1);
  }
  acc.out(d, lane, wm, wn);
}

// fp32, 64-tiles: one v_mfma_f32_32x32x2 block per wavefront (the order of k of gemm_f32.hip); element e of `acc` is row
// (lane & 31), column 8 (e / 4) + 4 (lane / 32) + e % 4 of the wavefront's block.  NB column operands share the row operand.
template <int NB, typename OA, typename OB>
__device__ __forceinline__ void tile32x2(const OA& A, const OB (&B)[NB], int row0, int col0, int kend, float* lds, int tid, int lane,
                                         int wm, int wn, f32x16_t (&acc)[NB]) {
  constexpr int P = Real<float, 64>::P, OPND = Real<float, 64>::OPND;
#pragma unroll
  for (int o = 0; o < NB; ++o)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[o][v] = 0.f;
  real_loop<float, 64, NB>(A, B, row0, col0, 0, kend, lds, tid, [&](const float* st) {
#pragma unroll
    for (int ks = 0; ks < KD / 2; ++ks) {
      const int k = ks * 2 + (lane >> 5);
      const float fa = st[k * P + wm * 32 + (lane & 31)];
#pragma unroll
      for (int o = 0; o < NB; ++o)
        acc[o] = __builtin_amdgcn_mfma_f32_32x32x2f32(st[(1 + o) * OPND + k * P + wn * 32 + (lane & 31)], fa, acc[o], 0, 0, 0);
    }
  }, NoTurn());
}
__device__ __forceinline__ void stage_f32(const f32x16_t& acc, float* stg, int lane, int wm, int wn) {
#pragma unroll
  for (int v = 0; v < 16; ++v)
    stg[(wm * 32 + (lane & 31)) * 66 + wn * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3)] = acc[v];
}

// ---- products of bf16 tiles: the LDS layouts of gemm_bf16_tile.h, 64-deep stages through registers -----------------------
// `acc` is called with every stage: the buffers of the row operand and of NB column operands, 8 KB each.
template <int TB, int D, bool MASK, bool EDGE>
__device__ __forceinline__ void put_bf16(char* dst, const Opnd<bf16_t, EDGE>& o, Raw<bf16_t>& r, int c, int row0, int k0) {
  if constexpr (EDGE && MASK) mask_chunk<TB, D>(o, r, c, row0, k0);
  const int q = c >> 3, ch = c & 7;   // (row or k, chunk): 8 chunks of a line either way
  *reinterpret_cast<u32x4_t*>(dst + q * 128 + (o.ks ? ks_swizzle(ch, q) : kc_swizzle(ch, q)) * 16) = r.q[0];
}
template <int NB, bool EDGE, typename Acc>
__device__ __forceinline__ void tile_bf16(const Opnd<bf16_t, EDGE>& A, const Opnd<bf16_t, false> (&B)[NB], int row0, int col0, int kend,
                                          char* lds, int tid, Acc acc) {
  constexpr int OPND = 64 * 64 * 2;
  constexpr int STG = (1 + NB) * OPND;
  const int n = (kend + 63) / 64;
  Raw<bf16_t> v[2][1 + NB][2];
  staged_loop<2>(n, full_stages(A, 0, n, 64),
      [&](int s, int i) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v[s][0][h] = fetch_chunk<64, 64>(A, tid + 256 * h, row0, i * 64);
#pragma unroll
      for (int o = 0; o < NB; ++o) v[s][1 + o][h] = fetch_chunk<64, 64>(B[o], tid + 256 * h, col0, i * 64);
    }
  },
      [&](int s, int i, int buf, auto mask) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      put_bf16<64, 64, decltype(mask)::value>(lds + buf * STG, A, v[s][0][h], tid + 256 * h, row0, i * 64);
#pragma unroll
      for (int o = 0; o < NB; ++o)
        put_bf16<64, 64, false>(lds + buf * STG + (1 + o) * OPND, B[o], v[s][1 + o][h], tid + 256 * h, col0, i * 64);
    }
  },
      [&](int buf) { acc(lds + buf * STG); });
}
// P and R: v_mfma_f32_16x16x32_bf16, four 16 x 16 blocks per wavefront, to the staging area (pitch 66)
template <bool EDGE>
__device__ __forceinline__ void product_bf16(const Opnd<bf16_t, EDGE>& A, const Opnd<bf16_t, false>& B, int row0, int col0, int kend,
                                             char* lds, int tid, int lane, int wm, int wn, float* stg) {
  f32x4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const Opnd<bf16_t, false> Bs[1] = {B};
  tile_bf16<1>(A, Bs, row0, col0, kend, lds, tid, [&](const char* st) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8_t fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        fa[i] = A.ks ? read_frag16<64, true>(st, wm * 32 + i * 16, ks, lane) : read_frag16<64, false>(st, wm * 32 + i * 16, ks, lane);
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[j] = read_frag16<64, true>(st + 8192, wn * 32 + j * 16, ks, lane);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
  });
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        stg[(wm * 32 + i * 16 + (lane & 15)) * 66 + wn * 32 + j * 16 + (lane >> 4) * 4 + v] = acc[i][j][v];
}
// A 64 x 64 tile of P^T P in fp64 over k < kend rows of a bf16 working matrix (at the tiles' first rows), to the staging area as
// tile16 leaves it.  The stages stay bf16 in the LDS, a fragment's elements become fp64 on their way into the products (as fp64 the
// LDS would carry four times the bytes, and 32 x 32 tiles twice that).  Lane l's eight k of a fragment are 8 (l / 16) on.
__device__ __forceinline__ void gram64_bf16(const bf16_t* P, int rp, int row0, int col0, int kend, char* lds, int tid, int lane, int wm,
                                            int wn) {
  Acc16<double, 64> acc;
  acc.clear();
  const Opnd<bf16_t, false> o = work<bf16_t>(P, rp, 1), Bs[1] = {o};
  tile_bf16<1>(o, Bs, row0, col0, kend, lds, tid, [&](const char* st) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      double a[2][8], b[2][8];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bf16x8_t fa = read_frag16<64, true>(st, wm * 32 + i * 16, ks, lane), fb = read_frag16<64, true>(st + 8192, wn * 32 + i * 16, ks, lane);
        unpack(Raw<bf16_t>{{__builtin_bit_cast(u32x4_t, fa)}}, a[i]);
        unpack(Raw<bf16_t>{{__builtin_bit_cast(u32x4_t, fb)}}, b[i]);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc.acc[i][j] = Mfma<double>::mma(a[i][u], b[j][u], acc.acc[i][j]);
    }
  });
  acc.out(reinterpret_cast<double*>(lds), lane, wm, wn);
}
// the updates: v_mfma_f32_32x32x16_bf16 as in the batched update kernel, both products at once
__device__ __forceinline__ void update_bf16(const Opnd<bf16_t, false>& A, const Opnd<bf16_t, false> (&B)[2], int row0, int col0,
                                            int kend, char* lds, int tid, int lane, int wm, int wn, f32x16_t (&acc)[2]) {
#pragma unroll
  for (int o = 0; o < 2; ++o)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[o][v] = 0.f;
  tile_bf16<2>(A, B, row0, col0, kend, lds, tid, [&](const char* st) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const bf16x8_t fa = read_frag<64, false>(st, wm * 32, ks, lane);
#pragma unroll
      for (int o = 0; o < 2; ++o)
        acc[o] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_frag<64, false>(st + (1 + o) * 8192, wn * 32, ks, lane), fa, acc[o], 0, 0, 0);
    }
  });
}

// ---- stores ------------------------------------------------------------------------------------------------------------

// eight values at element offset e of a matrix of dtype f32 / bf16, n of them
__device__ __forceinline__ void store8(char* p, int f32, long long e, int n, const float (&v)[8]) {
  if (n <= 0) return;
  if (f32) {
    DA_GLOBAL float* const q = (DA_GLOBAL float*)p + e;
    if (n >= 8) {
      u32x4_un_t x, y;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = __builtin_bit_cast(unsigned, v[i]);
        y[i] = __builtin_bit_cast(unsigned, v[4 + i]);
      }
      *(DA_GLOBAL u32x4_un_t*)q = x;
      *(DA_GLOBAL u32x4_un_t*)(q + 4) = y;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i < n) q[i] = v[i];
    }
  } else {
    DA_GLOBAL bf16_t* const q = (DA_GLOBAL bf16_t*)p + e;
    if (n >= 8) {
      u32x4_un_t x;
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = cvt_pk_bf16(v[2 * i], v[2 * i + 1]);
      *(DA_GLOBAL u32x4_un_t*)q = x;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i < n) q[i] = f2bf(v[i]);
    }
  }
}

// nan_to_num of the dtype; 0 for an all-zero B (reference dion/dion.py:1416-1444)
template <bool BF>
__device__ __forceinline__ float guard(float x, bool nonzero, float alt) {
  const float top = BF ? 3.3895313892515355e38f : 3.4028234663852886e38f;
  if (BF) x = rbf(x);
  if (x != x) x = 0.f;
  else if (x > top) x = top;
  else if (x < -top) x = -top;
  return nonzero ? x : alt;
}

// ---- the blocked fp64 Cholesky factorisation  P^T P = L L^T,  T = L^-1  in blocks of 64, as tasks -------------------------
// P^T P comes as lower 32 x 32 tiles in K slices (slab: [slices][rp][rp], rp = 64 rT); columns r .. rp - 1 are the identity.
struct Factor {
  const double* slab;
  double *LT, *T, *TT;         // rp x rp; the blocks of L^T above the diagonal, of T on and below it, of T^T (if wanted, or null)
  int slices, r, rp, rT;
  int *bad, *sick, *info;      // first failed pivot (column + 1); outcome: pivot range below `ratio` or a failed pivot; info may be null
  double* range;               // smallest and largest pivot so far
  double ratio;
};
// Left-looking.  DIAGj forms block (j, j - 1) of L from the inverse of the diagonal block before, takes its products off block (j, j),
// factors that and inverts the factor: the chain of the phases is one task per column of blocks, and the rest, `low_tasks` per column,
// runs beside it: blocks of column j of L from (j + 2, j) down, and blocks of block row j of T.  (With all of column j a phase
// between DIAGj and DIAG(j + 1) a column took 33 us, so 28.)
// `before` (all threads) returns when LOW(j - 2) resp. LOW(j - 1) is complete, `wait` when DIAG(j - 1) resp. DIAGj is; P^T P has been for
// long.  What a wait does not stand before is done ahead of it.
__host__ __device__ inline int low_tasks(int rT, int j) { return (rT - 2 - j > 0 ? rT - 2 - j : 0) + j; }
template <typename Before, typename Wait>
__device__ __forceinline__ void factor_task(const Factor& F, int j, bool diag, int task, char* lds, int tid, int lane, int wave, int wm,
                                            int wn, Before before, Wait wait) {
  typedef Real<double, 64> RD;
  enum Job { J_DIAG, J_LOW, J_INV };
  double* const d = reinterpret_cast<double*>(lds);
  double* const d2 = d + 64 * 66;
  static_assert(2 * 64 * 66 * 8 <= STAGES64, "two blocks");
  double *const LT = F.LT, *const T = F.T;
  const int rp = F.rp, rT = F.rT, nlow = max(0, rT - 2 - j);
  const long long rr = (long long)rp * rp;
  const Job job = diag ? J_DIAG : task < nlow ? J_LOW : J_INV;
  const int x = diag ? j : job == J_LOW ? j + 2 + task : task - nlow;
  const int jd = diag ? j - 1 : j;   // the column of blocks whose L(x, jd) is formed
  const Opnd<double, false> sd = work<double>(T + (long long)jd * 64 * rp + jd * 64, rp, 0);   // D, the inverse of its diagonal block's factor
  double2_t own[8];              // element pair u: row (tid + 256 u) / 32, columns 2 ((tid + 256 u) % 32)
  const int k = (tid & 31) * 2, i0 = tid >> 5;
  // block (x, jb) of P^T P: the slabs in slice order; beyond the rank the matrix is the identity
  auto gram_block = [&](double2_t (&w)[8], int jb) {
#pragma unroll
    for (int u = 0; u < 8; ++u) w[u] = double2_t{0.0, 0.0};
    const double* const slab = F.slab + (long long)(x * 64 + i0) * rp + jb * 64 + k;
    for (int s0 = 0; s0 < F.slices; s0 += 4) {   // four slabs on the way at a time
      double2_t y[4][8];
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (s0 + s < F.slices) {
#pragma unroll
          for (int u = 0; u < 8; ++u) y[s][u] = *reinterpret_cast<const double2_t*>(slab + (s0 + s) * rr + (long long)u * 8 * rp);
        }
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (s0 + s < F.slices) {
#pragma unroll
          for (int u = 0; u < 8; ++u) w[u] += y[s][u];
        }
    }
    const int lim = ((F.r + 31) >> 5) << 5;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int gi = x * 64 + i0 + 8 * u, gk = jb * 64 + k;
      if (gi >= F.r || gk >= lim || (gk >> 5) > (gi >> 5)) {   // (not written by GRAM)
        w[u][0] = gi >= F.r && gi == gk ? 1.0 : 0.0;
        w[u][1] = gi >= F.r && gi == gk + 1 ? 1.0 : 0.0;
      }
    }
  };
  // w += sign * the product that lies in d
  auto add = [&](double2_t (&w)[8], double sign) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      w[u][0] += sign * d[(i0 + 8 * u) * 66 + k];
      w[u][1] += sign * d[(i0 + 8 * u) * 66 + k + 1];
    }
    __syncthreads();
  };
  auto park = [&](const double2_t (&w)[8]) {   // a block out of the way of the products' registers; every thread its own elements
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      d2[(i0 + 8 * u) * 66 + k] = w[u][0];
      d2[(i0 + 8 * u) * 66 + k + 1] = w[u][1];
    }
  };
  if (job == J_LOW || (job == J_DIAG && j > 0)) {
    double2_t w[8];
    gram_block(w, jd);
    park(w);
  }
  if (job == J_DIAG) gram_block(own, j);
  before();
  if (job == J_DIAG && j > 1) {   // the columns up to j - 2 of row j
    direct64<true>(LT + j * 64, rp, LT + j * 64, rp, jd * 64, d, lane, wm, wn);
    add(own, -1.0);
  }
  wait();
  if (job == J_INV)      // sum over k of L(j, k) T(k, x), x <= k < j
    direct64<true>(LT + (long long)x * 64 * rp + j * 64, rp, T + (long long)x * 64 * rp + x * 64, rp, (j - x) * 64, d, lane, wm, wn);
  else if (jd > 0)       // sum over k < jd of L(x, k) L(jd, k)^T
    direct64<true>(LT + x * 64, rp, LT + jd * 64, rp, jd * 64, d, lane, wm, wn);
  if (jd >= 0) {
    double2_t w[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) w[u] = job == J_INV ? double2_t{0.0, 0.0} : double2_t{d2[(i0 + 8 * u) * 66 + k], d2[(i0 + 8 * u) * 66 + k + 1]};
    if (job == J_INV) add(w, 1.0);
    else if (jd > 0) add(w, -1.0);
    else __syncthreads();
    // second product, both operands to the LDS stages:  L(x, jd) = W(x, jd) D^T;   T(j, x) = -D W(j, x)
    Raw<double> dr[2];
    dr[0] = fetch_chunk<64, KD>(sd, tid, 0, 0);
    dr[1] = fetch_chunk<64, KD>(sd, tid, 0, KD);
    double* const wst = d + (job == J_INV ? RD::OPND : 0);
    double* const dst = d + (job == J_INV ? 0 : RD::OPND);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + 8 * u;
      if (job == J_INV) {
        wst[(i >> 5) * 2 * RD::OPND + (i & 31) * RD::P + k] = w[u][0];
        wst[(i >> 5) * 2 * RD::OPND + (i & 31) * RD::P + k + 1] = w[u][1];
      } else {
        wst[(k >> 5) * 2 * RD::OPND + (k & 31) * RD::P + i] = w[u][0];
        wst[(k >> 5) * 2 * RD::OPND + ((k + 1) & 31) * RD::P + i] = w[u][1];
      }
    }
    put_chunk<double, 64, false>(dst, sd, dr[0], tid, 0, 0, NoTurn());
    put_chunk<double, 64, false>(dst + 2 * RD::OPND, sd, dr[1], tid, 0, KD, NoTurn());
    __syncthreads();
    Acc16<double, 64> acc;
    acc.clear();
    acc.stage(d, d + RD::OPND, lane, wm, wn);
    acc.stage(d + 2 * RD::OPND, d + 3 * RD::OPND, lane, wm, wn);
    __syncthreads();
    acc.out(d, lane, wm, wn);
    if (job == J_INV) {
      double* const out = T + (long long)j * 64 * rp + x * 64;
      for (int e = tid; e < 4096; e += 256) out[(long long)(e >> 6) * rp + (e & 63)] = -d[(e >> 6) * 66 + (e & 63)];
    }
    double* const turned = job != J_INV ? LT + (long long)jd * 64 * rp + x * 64 : F.TT ? F.TT + (long long)x * 64 * rp + j * 64 : nullptr;
    if (turned) {
      const double sign = job == J_INV ? -1.0 : 1.0;
      for (int e = tid; e < 4096; e += 256) turned[(long long)(e >> 6) * rp + (e & 63)] = sign * d[(e & 63) * 66 + (e >> 6)];
    }
  }
  if (job != J_DIAG) return;
  // ---- the diagonal block: wavefront w holds its 16 x 16 blocks (w, 0 .. w)
  park(own);
  __syncthreads();
  Mfma<double>::acc_t S[4];
#pragma unroll
  for (int tj = 0; tj < 4; ++tj)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = wave * 16 + Mfma<double>::row(v, lane), col = tj * 16 + (lane & 15);
      S[tj][v] = tj <= wave ? (row >= col ? d2[row * 66 + col] : d2[col * 66 + row]) : 0.0;
    }
  if (j > 0) {   // less L(j, j - 1) L(j, j - 1)^T
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) {
      const double a = -d[(wave * 16 + (lane & 15)) * 66 + ks * 4 + (lane >> 4)];
#pragma unroll
      for (int tj = 0; tj < 4; ++tj)
        if (tj <= wave) S[tj] = Mfma<double>::mma(a, d[(tj * 16 + (lane & 15)) * 66 + ks * 4 + (lane >> 4)], S[tj]);
    }
  }
  __syncthreads();   // (the blocks lie where the factorisation works)
  double* const dT = d + DIAG_W;
  static_assert(2 * DIAG_W * 8 <= STAGES64, "the work area and the inverse factor");
  diag_factor64(S, d, dT, min(64, F.r - j * 64), 64, lane, wave, [&](int failed, double pmin, double pmax) {
    if (lane != 0) return;
    int bad = failed ? j * 64 + failed : 0;
    if (j > 0) {
      const int before = __hip_atomic_load(F.bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (before) bad = before;
      pmin = fmin(pmin, __hip_atomic_load(F.range, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      pmax = fmax(pmax, __hip_atomic_load(F.range + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    }
    __hip_atomic_store(F.bad, bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(F.range, pmin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(F.range + 1, pmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (j == rT - 1) {
      const bool healthy = bad == 0 && pmin >= F.ratio * pmax && pmax > 0.0;
      __hip_atomic_store(F.sick, healthy ? 0 : 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (F.info) *F.info = bad;
    }
  });
  double* const Dw = T + (long long)j * 64 * rp + j * 64;
  for (int e = tid; e < 4096; e += 256) Dw[(long long)(e >> 6) * rp + (e & 63)] = dT[(e & 63) * DIAG_P + (e >> 6)];
  if (F.TT) {
    double* const Dt = F.TT + (long long)j * 64 * rp + j * 64;
    for (int e = tid; e < 4096; e += 256) Dt[(long long)(e >> 6) * rp + (e & 63)] = dT[(e >> 6) * DIAG_P + (e & 63)];
  }
}

// One lower 32 x 32 tile (number t of t32 (t32 + 1) / 2) of S^T S over rows [kbeg, kend) of S, into out (pitch rp) and d (pitch 34)
template <typename OP>
__device__ __forceinline__ void gram_tile(const OP& S, int t, int kbeg, int kend, double* out, int rp, double* d, int tid, int lane, int wm,
                                          int wn, int& ti, int& tj) {
  int i = 0;
  while (t > i) { t -= i + 1; ++i; }
  ti = wave_uniform(i);
  tj = wave_uniform(t);
  tile16<double, 32>(S, S, ti * 32, tj * 32, kbeg, kend, d, tid, lane, wm, wn);
  for (int e = tid; e < 1024; e += 256) out[(long long)(ti * 32 + (e >> 5)) * rp + tj * 32 + (e & 31)] = d[(e >> 5) * 34 + (e & 31)];
}
// the tile's share of || column of S^T S - I ||^2, by rows and (symmetric) by columns: defect[column][32-tile]
__device__ __forceinline__ void gram_defect(const double* d, double* defect, int pitch, int ti, int tj, int tid) {
  if (tid >= 64) return;
  const int i = tid & 31;
  double s = 0.0;
  for (int k = 0; k < 32; ++k) {
    const double v = (tid < 32 ? d[i * 34 + k] : d[k * 34 + i]) - (ti == tj && i == k ? 1.0 : 0.0);
    s += v * v;
  }
  const int c = (tid < 32 ? ti : tj) * 32 + i, t = tid < 32 ? tj : ti;
  if (tid < 32 || ti != tj) defect[(long long)c * pitch + t] = s;
}
// drop[c]: column c came from a noise-level pivot (columns 0 .. rp - 1)
__device__ __forceinline__ void find_dropped(const double* defect, int pitch, int r, int rp, unsigned char* drop, int tid) {
  for (int c = tid; c < rp; c += 256) {
    double s = 0.0;
    if (c < r)
      for (int t = 0; t < ((r + 31) >> 5); ++t) s += defect[(long long)c * pitch + t];
    drop[c] = !(s <= 0.25) ? 1 : 0;
  }
  __syncthreads();
}
// A 64 x 64 tile of S V into d, V = I - up(S^T S - I) without the dropped columns; V^T is formed from the lower tiles of S^T S
// on the way to LDS
__device__ __forceinline__ void polish_tile(const double* S, const double* gram, int r, int rp, const unsigned char* drop, int row0, int col0,
                                            double* d, int tid, int lane, int wm, int wn) {
  tile16<double, 64>(work<double>(S, rp, 0), work<double>(gram, rp, 0), row0, col0, 0, col0 + 64, d, tid, lane, wm, wn,
                     [&](double (&v)[8], int c, int k) {
    const bool gone = drop[c] != 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const double y = v[i];
      const bool on = k + i == c;
      double u = k + i < c ? -y : (on ? 1.5 - 0.5 * y : 0.0);
      if (c >= r) u = on ? 1.0 : 0.0;                 // beyond the rank: the identity
      if (gone) u = 0.0;                              // a dropped column comes out as zero
      else if (drop[k + i]) u = on ? 1.0 : 0.0;       // and gives no correction
      v[i] = u;
    }
  });
}

}  // namespace
