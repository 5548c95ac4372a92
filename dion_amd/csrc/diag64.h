// The serial part of the blocked Cholesky factorisations (cholesky.hip in fp32, small_tile.h): a 64 x 64 diagonal block S = L L^T and
// T = L^-1 by one workgroup of four wavefronts, fp64 or fp32.
//
// What bounds it: the chain of 64 dependent columns -- pivot, reciprocal square root, one column of L, update of the next column --
// and what is put between its links.  Four panels of 16 columns.  The first wavefront factors a panel without LDS and without a
// barrier between the columns: lane = row, sixteen columns in registers, the diagonal block once in every sixteen lanes so that a
// column's multipliers are DPP operands of the multiply-adds (row_newbcast; through v_readlane and scalar registers it took twice
// the instructions), the 48 rows below it and the identity, which becomes the inverse of the diagonal block, in a second set
// that the same multipliers serve.  Between panels the other three wavefronts update a tile each of the next panel on the matrix
// cores; while it is factored, the tiles further right, and they form a block column each of T below the diagonal,
// left-looking: T(i, c) = T(i, i) V, V = -sum of L(i, k) T(k, c), a product's accumulators being the next one's operand as they are.
// Measured, one workgroup: fp64 19 800 cycles (8.2 us; 10 600 of them the columns), fp32 16 100 (6.7 us).  Sixteen steps of 4
// columns, each with a round trip through LDS, a barrier and rank-4 updates of S and of the whole inverse, took 33 700 in
// fp64, and 46 400 the first time (cold instruction cache; now 22 200): 24 fp32 matrices of 256 x 256 and
// 256 x 1024 at rank 128 under Dion 241.9 -> 217.8 us a step; GPT-small's 72 at rank 192 725 -> 696 us.
// (The fp64 steps of cholesky.hip keep their own, see there.)
#pragma once
#include "gemm_f64.h"

namespace {

constexpr int DIAG_P = 65;                       // LDS pitch of every 64-wide array here
constexpr int DIAG_W = 64 * DIAG_P;              // elements of the work area
static_assert(DA_CHOL_NB == 64, "four panels of 16");

template <typename T> __device__ __forceinline__ T rsqrt_seed(T p);
template <> __device__ __forceinline__ double rsqrt_seed<double>(double p) { return __builtin_amdgcn_rsq(p); }
template <> __device__ __forceinline__ float rsqrt_seed<float>(float p) { return __builtin_amdgcn_rsqf(p); }
// a positive normal number (false for NaN, infinities, zero and denormals, which the estimate does not handle)
__device__ __forceinline__ bool usable_pivot(double p) { return __builtin_amdgcn_class(p, 0x100); }
__device__ __forceinline__ bool usable_pivot(float p) { return __builtin_amdgcn_classf(p, 0x100); }

// Lane K of every 16 lanes, to all sixteen of them (DPP row_newbcast), and acc += that lane's `src` times `mul`.  A lane's register
// is read through DPP two wait states after its write at the earliest, which nobody watches over in assembly: bcast16 waits
// itself, and what fma16 broadcasts comes from scale16.
template <int K> __device__ __forceinline__ double bcast16(double x) {
  double r;
  asm("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(x), "n"(K));
  return r;
}
template <int K> __device__ __forceinline__ float bcast16(float x) {
  float r;
  asm("s_nop 1\n\tv_mov_b32_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(x), "n"(K));
  return r;
}
__device__ __forceinline__ double scale16(double x, double y) {
  double r;
  asm("v_mul_f64 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(x), "v"(y));
  return r;
}
__device__ __forceinline__ float scale16(float x, float y) {
  float r;
  asm("v_mul_f32 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(x), "v"(y));
  return r;
}
template <int K> __device__ __forceinline__ void fma16(double& acc, double src, double mul) {
  asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(src), "v"(mul), "n"(K));
}
template <int K> __device__ __forceinline__ void fma16(float& acc, float src, float mul) {
  asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(src), "v"(mul), "n"(K));
}

// Column J of a panel and what follows from it for the columns right of it.  d: the panel's diagonal block, lane lc of every 16 holds
// row lc; a: other rows that the panel's factor is divided out of.  On return a[J] holds minus the rows' entries of column J.
// pv: the pivot of the lane's own column.
template <int K, int J, typename T> __device__ __forceinline__ void panel_update(T (&d)[16], T (&a)[16], T l, T nd, T na) {
  if constexpr (K < 16) {
    fma16<K>(d[K], l, nd);
    fma16<K>(a[K], l, na);
    panel_update<K + 1, J>(d, a, l, nd, na);
  }
}
template <int J, typename T> __device__ __forceinline__ void panel_columns(T (&d)[16], T (&a)[16], T& pv, int mine) {
#pragma clang fp contract(fast)
  if constexpr (J < 16) {
    const T piv = bcast16<J>(d[J]);
    // 1 / sqrt from the hardware estimate (fp32: 1 ulp; fp64: 2^-27 and one step of third order): the library's square root and
    // division are four times as long
    T rs = rsqrt_seed<T>(piv);
    if (sizeof(T) == 8) {
      const T err = T(1) - piv * rs * rs;
      rs = rs + rs * err * (T(0.5) + T(0.375) * err);
    }
    rs = usable_pivot(piv) ? rs : T(0);
    pv = mine == J ? piv : pv;
    const T l = scale16(d[J], rs), na = -(a[J] * rs), nd = -l;
    a[J] = na;
    panel_update<J + 1, J>(d, a, l, nd, na);
    panel_columns<J + 1>(d, a, pv, mine);
  }
}

__device__ __forceinline__ double lane_value(double x, int lane) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)u, lane), hi = __builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
  return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
__device__ __forceinline__ float lane_value(float x, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}
// smallest lo and largest hi of every sixteen lanes
template <int K, typename T> __device__ __forceinline__ void row_range(T lo, T hi, T& pmin, T& pmax) {
  if constexpr (K < 16) {
    const T x = bcast16<K>(lo), y = bcast16<K>(hi);
    pmin = x < pmin ? x : pmin;
    pmax = y > pmax ? y : pmax;
    row_range<K + 1>(lo, hi, pmin, pmax);
  }
}

// S: wavefront w holds the 16 x 16 tiles (w, 0 .. w) of the block in accumulator layout (rows and columns beyond the matrix: the
// identity).  dT receives the inverse factor, transposed: dT[k * DIAG_P + x] = T[x][k], zero above the diagonal and in rows and
// columns >= keep.  work: DIAG_W elements.  Both are free on entry (a barrier behind their last use) and dT is complete on return
// (a barrier is the last thing done).  A pivot that is not positive zeroes its column.  pivots(failed, pmin, pmax), called by all
// lanes of the first wavefront: 1 + the first column < live whose pivot is not positive (0: none) and the range of the others.
template <typename T, typename Pivots>
__device__ __forceinline__ void diag_factor64(const typename Mfma<T>::acc_t (&S)[4], T* work, T* dT, int live, int keep, int lane, int wave,
                                              Pivots pivots) {
  typedef typename Mfma<T>::acc_t acc_t;
  const int lc = lane & 15, lg = lane >> 4;
  // work[column][row]: what is left of S, in finished panels -L below the diagonal blocks
  auto at = [&](int rt, int ct, int i, int k) -> T& { return work[(ct * 16 + k) * DIAG_P + rt * 16 + i]; };
  auto t_at = [&](int rt, int ct, int i, int k) -> T& { return dT[(ct * 16 + k) * DIAG_P + rt * 16 + i]; };
  auto get = [&](int rt, int ct) __attribute__((always_inline)) {   // a tile in accumulator layout
    acc_t x;
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] = at(rt, ct, Mfma<T>::row(v, lane), lc);
    return x;
  };
  auto put = [&](int rt, int ct, const acc_t& x) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < 4; ++v) at(rt, ct, Mfma<T>::row(v, lane), lc) = x[v];
  };
  // x - L(rt, p) L(ct, p)^T
  auto update = [&](int p, int rt, int ct, acc_t x) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) x = Mfma<T>::mma(-at(rt, p, lc, ks * 4 + lg), at(ct, p, lc, ks * 4 + lg), x);
    return x;
  };
#pragma unroll
  for (int tj = 0; tj < 4; ++tj)
    if (tj <= wave) put(wave, tj, S[tj]);
  __syncthreads();
  if (wave == 0) {
    T pv = T(0);                                    // lane i: pivot of column i
#pragma unroll 1
    for (int p = 0; p < 4; ++p) {
      const int base = 16 * p;
      // the sixteen-lane groups 0 .. 2 - p take the tiles of rows below the panel, the last group minus the identity: its rows become
      // the columns of the inverse of the panel's diagonal block
      T d[16], a[16];
      const int row = base + 16 + lane;
      const T* const col = work + base * DIAG_P;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        d[j] = col[j * DIAG_P + base + lc];
        a[j] = col[j * DIAG_P + (row < 64 ? row : base + lc)];
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) a[j] = lg == 3 ? (lc == j ? T(-1) : T(0)) : a[j];
      panel_columns<0>(d, a, pv, lane - base);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (the stores may not move above the loads of other lanes)
      __builtin_amdgcn_wave_barrier();
      if (lg == 3 || row < 64) {
        T* const to = lg == 3 ? &t_at(p, p, 0, lc) : &work[base * DIAG_P + row];
        const int step = lg == 3 ? 1 : DIAG_P;
#pragma unroll
        for (int j = 0; j < 16; ++j) to[j * step] = a[j];
      }
      __syncthreads();                              // panel p of L and T(p, p)
      if (p < 3) __syncthreads();                   // the next panel of S
    }
    // the smallest and the largest pivot: over every sixteen lanes through DPP, then over the four groups
    const bool ok = usable_pivot(pv), counts = lane < live;
    const unsigned long long failed = __ballot(counts && !ok);
    const T lo = ok && counts ? pv : T(3e38), hi = ok && counts ? pv : T(0);
    T pmin = lo, pmax = hi;
    row_range<0>(lo, hi, pmin, pmax);
    T mn = pmin, mx = pmax;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const T x = lane_value(pmin, 16 * g), y = lane_value(pmax, 16 * g);
      mn = x < mn ? x : mn;
      mx = y > mx ? y : mx;
    }
    pivots(failed ? __ffsll((long long)failed) : 0, mn, mx);
  } else {
    const int c = wave - 1;
    for (int e = c * 64 + lane; e < 6 * 256; e += 192) {   // the blocks of T above the diagonal
      const int blk = e >> 8, ct = blk < 1 ? 1 : blk < 3 ? 2 : 3, rt = blk - (ct * (ct - 1) >> 1);
      t_at(rt, ct, e & 15, (e >> 4) & 15) = T(0);
    }
    acc_t V[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      __syncthreads();                              // panel p of L and T(p, p)
      if (p < 3) {
        if (p + 1 + c < 4) put(p + 1 + c, p + 1, update(p, p + 1 + c, p + 1, get(p + 1 + c, p + 1)));
        __syncthreads();                            // the next panel of S
      }
      // the tiles right of it
      if (p == 0) {
        const int rt = c == 0 ? 2 : 3, ct = c == 2 ? 3 : 2;
        put(rt, ct, update(0, rt, ct, get(rt, ct)));
      } else if (p == 1 && c == 2) {
        put(3, 3, update(1, 3, 3, get(3, 3)));
      }
      if (p == c) {
#pragma unroll
        for (int i = p + 1; i < 4; ++i) {
          V[i] = acc_t{0, 0, 0, 0};
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) V[i] = Mfma<T>::mma(at(i, p, lc, ks * 4 + lg), t_at(p, p, ks * 4 + lg, lc), V[i]);
        }
      } else if (p > c) {
        acc_t t = {0, 0, 0, 0};
#pragma unroll
        for (int v = 0; v < 4; ++v) t = Mfma<T>::mma(t_at(p, p, lc, Mfma<T>::row(v, lane)), V[p][v], t);
#pragma unroll
        for (int v = 0; v < 4; ++v) t_at(p, c, Mfma<T>::row(v, lane), lc) = t[v];
#pragma unroll
        for (int i = p + 1; i < 4; ++i)
#pragma unroll
          for (int v = 0; v < 4; ++v) V[i] = Mfma<T>::mma(at(i, p, lc, Mfma<T>::row(v, lane)), t[v], V[i]);
      }
    }
  }
  __syncthreads();
  if (keep < 64) {
    for (int e = wave * 64 + lane; e < (64 - keep) * 64; e += 256) dT[(e & 63) * DIAG_P + keep + (e >> 6)] = T(0);   // (rows; the columns are zero above them)
    __syncthreads();
  }
}

}  // namespace
