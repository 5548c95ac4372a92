// HBM-bound passes around the Newton-Schulz iteration (all single-pass, 16-byte accesses):
//
//   stage       : source matrices of several buckets -> bf16/f32 working matrices in *wide*
//                 orientation (rows <= cols; tall sources are transposed through an LDS tile),
//                 fused with either a plain dtype cast (stand-alone Newton-Schulz) or Muon's
//                 momentum / Nesterov update, plus per-tile partial sums of squares for
//                 the Frobenius norm.  Shapes off the 8-element grid are read and written in
//                 place with unaligned 16-byte accesses; the working matrices are padded with zeros.
//   normalize   : X <- X / (||X||_F + eps) with the reference's rounding points, the norm from
//                 a fixed-order sum of the partial sums.
//   unstage     : wide working matrix -> destination orientation; either a plain store
//                 (stand-alone Newton-Schulz) or Muon's weight-decay + scaled update.
//
// Rounding follows the reference op by op (reference dion/muon.py:536-550, 569-573,
// 633-638); the translation unit must be compiled with -ffp-contract=off.
#include "common.h"
#include "elementwise.h"

namespace {

constexpr int TS = 64;  // tile edge of the transposing passes; 256 threads, 16 elements (two 8-wide chunks) per thread
constexpr int RT = 32, CT = 256;   // tile of the passes that keep the orientation: 32 rows x 256 columns

template <typename T> struct Vec8;
template <> struct Vec8<bf16_t> {
  static __device__ __forceinline__ void load(const bf16_t* p, float (&v)[8]) {
    const uint4 r = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = bf2f((bf16_t)(w[i] & 0xffffu));
      v[2 * i + 1] = bf2f((bf16_t)(w[i] >> 16));
    }
  }
  static __device__ __forceinline__ void store(bf16_t* p, const float (&v)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = (uint32_t)f2bf(v[2 * i]) | ((uint32_t)f2bf(v[2 * i + 1]) << 16);
    *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
  }
  // streaming variants: data that is not touched again before it would fall out of the caches anyway
  static __device__ __forceinline__ void load_nt(const bf16_t* p, float (&v)[8]) {
    typedef unsigned u4_t __attribute__((ext_vector_type(4)));
    const u4_t w = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(p));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned x = w[i];
      v[2 * i] = __builtin_bit_cast(float, x << 16);
      v[2 * i + 1] = __builtin_bit_cast(float, x & 0xffff0000u);
    }
  }
  static __device__ __forceinline__ void store_nt(bf16_t* p, const float (&v)[8]) {
    typedef unsigned u4_t __attribute__((ext_vector_type(4)));
    u4_t w;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = (uint32_t)f2bf(v[2 * i]) | ((uint32_t)f2bf(v[2 * i + 1]) << 16);
    __builtin_nontemporal_store(w, reinterpret_cast<u4_t*>(p));
  }
  static __device__ __forceinline__ float round(float x) { return rbf(x); }
};
template <> struct Vec8<float> {
  static __device__ __forceinline__ void load(const float* p, float (&v)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(p);
    const float4 b = *reinterpret_cast<const float4*>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
  static __device__ __forceinline__ void store(float* p, const float (&v)[8]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
  }
  static __device__ __forceinline__ void load_nt(const float* p, float (&v)[8]) {
    typedef float f4_t __attribute__((ext_vector_type(4)));
    const f4_t a = __builtin_nontemporal_load(reinterpret_cast<const f4_t*>(p));
    const f4_t b = __builtin_nontemporal_load(reinterpret_cast<const f4_t*>(p) + 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = a[i], y = b[i];
      v[i] = x;
      v[4 + i] = y;
    }
  }
  static __device__ __forceinline__ void store_nt(float* p, const float (&v)[8]) {
    typedef float f4_t __attribute__((ext_vector_type(4)));
    const f4_t a = {v[0], v[1], v[2], v[3]}, b = {v[4], v[5], v[6], v[7]};
    __builtin_nontemporal_store(a, reinterpret_cast<f4_t*>(p));
    __builtin_nontemporal_store(b, reinterpret_cast<f4_t*>(p) + 1);
  }
  static __device__ __forceinline__ float round(float x) { return x; }
};

__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float s = 0.f;
  if (threadIdx.x == 0) s = (red[0] + red[1]) + (red[2] + red[3]);
  return s;  // valid in thread 0
}

// Eight consecutive elements of a row of which `n` exist (n <= 0: none).  VEC: every chunk is whole and 16-byte aligned;
// otherwise they move as unaligned 16-byte accesses, a row's last chunk element by element.
typedef unsigned u32x4_un_t __attribute__((ext_vector_type(4), aligned(2)));   // an unaligned 16-byte access
template <typename T, bool VEC>
__device__ __forceinline__ void load8(const T* p, int n, float (&v)[8]) {
  if (VEC) {
    if (n > 0) Vec8<T>::load_nt(p, v);
  } else if (n >= 8) {
    const u32x4_un_t x = *reinterpret_cast<const u32x4_un_t*>(p);
    if constexpr (sizeof(T) == 4) {
      const u32x4_un_t y = *reinterpret_cast<const u32x4_un_t*>(p + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned xe = x[e], ye = y[e];
        v[e] = __builtin_bit_cast(float, xe);
        v[4 + e] = __builtin_bit_cast(float, ye);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned xe = x[e];
        v[2 * e] = __builtin_bit_cast(float, xe << 16);
        v[2 * e + 1] = __builtin_bit_cast(float, xe & 0xffff0000u);
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = 0.f;
      if (e < n) v[e] = ld_as_float<T>(p + e);
    }
  }
}
template <typename T, bool VEC>
__device__ __forceinline__ void store8(T* p, int n, const float (&v)[8]) {
  if (VEC) {
    if (n > 0) Vec8<T>::store_nt(p, v);
  } else if (n >= 8) {
    u32x4_un_t x;
    if constexpr (sizeof(T) == 4) {
      u32x4_un_t y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = __builtin_bit_cast(unsigned, v[e]);
        y[e] = __builtin_bit_cast(unsigned, v[4 + e]);
      }
      *reinterpret_cast<u32x4_un_t*>(p + 4) = y;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = (unsigned)f2bf(v[2 * e]) | ((unsigned)f2bf(v[2 * e + 1]) << 16);
    }
    *reinterpret_cast<u32x4_un_t*>(p) = x;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < n) st_from_float<T>(p + e, v[e]);
  }
}

// ---------------------------------------------------------------------------------------
// stage
// ---------------------------------------------------------------------------------------
struct StageArgs {
  DaStage d;
  int blk0[DA_MAX_GROUPS + 1];   // first block of each group
  int mat0[DA_MAX_GROUPS];       // first matrix of each group in the pointer arrays
  int tiles[DA_MAX_GROUPS];      // blocks per matrix
};

// VEC: the rows of every group are whole, 16-byte aligned chunks
template <typename TG, typename TM, typename TW, bool VEC>
__global__ __launch_bounds__(256, VEC ? 5 : 4) void stage_kernel(StageArgs a) {
  __shared__ float red[4];
  __shared__ float tile[TS][TS + 1];
  const int tid = threadIdx.x;
  if (a.d.zero) {
    for (int i = blockIdx.x * 256 + tid; i < a.d.nzero; i += gridDim.x * 256) a.d.zero[i] = 0;
    if (blockIdx.x == 0 && tid == 0) *a.d.status = a.d.preset;
  }
  int grp = 0;
#pragma unroll
  for (int q = 1; q < DA_MAX_GROUPS; ++q)
    if (q < a.d.ngroups && (int)blockIdx.x >= a.blk0[q]) grp = q;
  const DaStageGroup& g = a.d.g[grp];
  const int blk = (int)blockIdx.x - a.blk0[grp];
  const int b = __builtin_amdgcn_readfirstlane(blk / a.tiles[grp]);
  const int t = blk - b * a.tiles[grp];
  const int mat = a.mat0[grp] + b;
  const int rows = g.rows, cols = g.cols;
  const bool muon = a.d.muon != 0, nesterov = a.d.nesterov != 0;
  const float mu = a.d.mu;
  const TG* G = static_cast<const TG*>(a.d.src[mat]);
  TM* M = muon ? static_cast<TM*>(a.d.mom[mat]) : nullptr;
  TW* W = g.wide ? static_cast<TW*>(g.wide) + (long long)b * g.mw * g.ldw : static_cast<TW*>(a.d.dst[mat]);
  if (t == 0 && tid == 0 && g.xtab) g.xtab[b] = a.d.dst[mat];

  // one chunk: momentum update (momentum stored back) or plain cast; returns the rounded result in u
  auto update = [&](int i, int j, int n, const float (&gv)[8], float (&m)[8], float (&u)[8]) {
    if (muon) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float ge = Vec8<TM>::round(gv[e]);                // G.to(M.dtype)
        float me = Vec8<TM>::round(m[e] * mu);                  // M *= mu
        me = Vec8<TM>::round(me + ge);                          // M += G
        m[e] = me;
        float ue = me;
        if (nesterov) ue = Vec8<TM>::round(Vec8<TM>::round(me * mu) + ge);  // U = M*mu; U += G
        u[e] = Vec8<TW>::round(ue);                             // U.to(bf16)
      }
      store8<TM, VEC>(M + (long long)i * cols + j, n, m);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) u[e] = Vec8<TW>::round(gv[e]);
    }
  };

  float ss = 0.f;
  const bool tall = g.wide && rows > cols;
  if (!tall) {
    // No transpose: a tile is RT rows x CT columns, a wavefront's 16-byte accesses cover whole 512-byte row
    // segments, and all of a thread's loads are requested before the first is used.
    const int rows_p = g.wide ? g.mw : rows, cols_p = g.wide ? g.nw : cols;
    const int tiles_cw = (cols_p + CT - 1) / CT;
    const int wi = t / tiles_cw, wj = t % tiles_cw;
    constexpr int NC = RT * CT / 8 / 256;   // chunks per thread
    float gv[NC][8], m[NC][8];
    int nv[NC];
#pragma unroll
    for (int it = 0; it < NC; ++it) {
      const int c = tid + 256 * it;
      const int i = wi * RT + c / (CT / 8), j = wj * CT + (c % (CT / 8)) * 8;
      nv[it] = i < rows ? cols - j : 0;
      if (nv[it] > 0) {
        load8<TG, VEC>(G + (long long)i * g.ld + j, nv[it], gv[it]);
        if (muon) load8<TM, VEC>(M + (long long)i * cols + j, nv[it], m[it]);
      }
    }
#pragma unroll
    for (int it = 0; it < NC; ++it) {
      const int c = tid + 256 * it;
      const int i = wi * RT + c / (CT / 8), j = wj * CT + (c % (CT / 8)) * 8;
      if (i >= rows_p || j >= cols_p) continue;
      float u[8];
      if (nv[it] > 0) {
        update(i, j, nv[it], gv[it], m[it], u);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += u[e] * u[e];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] = 0.f;
      }
      if (g.wide) Vec8<TW>::store(W + (long long)i * g.ldw + j, u);
      else store8<TW, VEC>(W + (long long)i * cols + j, nv[it], u);
    }
  } else {
    const int tiles_c = (g.mw + TS - 1) / TS;   // tiles over the source's columns
    const int ti = t / tiles_c, tj = t % tiles_c;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int c = tid + 256 * it;        // chunk id within tile: 64 rows x 8 chunks
      const int r = c >> 3, cc = (c & 7) * 8;
      const int i = ti * TS + r, j = tj * TS + cc;
      const int n = i < rows ? cols - j : 0;
      float u[8];
      if (n > 0) {
        float gv[8], m[8];
        load8<TG, VEC>(G + (long long)i * g.ld + j, n, gv);
        if (muon) load8<TM, VEC>(M + (long long)i * cols + j, n, m);
        update(i, j, n, gv, m, u);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += u[e] * u[e];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] = 0.f;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) tile[cc + e][r] = u[e];  // tile[source col][source row]
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int c = tid + 256 * it;
      const int p = c >> 3, qq = (c & 7) * 8;   // wide row p = source col, wide cols = source rows
      const int wi = tj * TS + p, wj = ti * TS + qq;
      if (wi < g.mw && wj < g.nw) {
        float u[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] = tile[p][qq + e];
        Vec8<TW>::store(W + (long long)wi * g.ldw + wj, u);
      }
    }
  }
  if (!g.wide) return;   // (uniform over the workgroup)
  const float s = block_sum(ss, red);
  if (tid == 0) g.partials[(long long)b * a.tiles[grp] + t] = s;
}

// x / d for a divisor shared by many elements: with rd = RN(1 / d), one residual step on the estimate x * rd gives
// the correctly rounded quotient (three fused operations instead of the dozen of a full division; the pass is
// otherwise bound by its arithmetic).  |x| <= d here (d is the matrix's Frobenius norm plus eps), so nothing
// overflows; a divisor whose reciprocal is zero or not finite takes the plain division (the caller's branch).
__device__ __forceinline__ float div_by(float x, float d, float rd) {
  const float q = x * rd;
  const float rem = __builtin_fmaf(-q, d, x);
  return __builtin_fmaf(rem, rd, q);
}

// The divisor of a matrix from its partial sums of squares, round(round(sqrt(sum)) + eps) in bf16 mode: a fixed-order
// fp64 sum, so every workgroup of the matrix arrives at the same bits.
__device__ __forceinline__ float divisor_of(const float* partials, int n, float eps, int bf16_mode, double* red) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += (double)partials[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  const float nrm = sqrtf((float)red[0]);
  return bf16_mode ? rbf(rbf(nrm) + eps) : nrm + eps;
}

// The divisor is formed here from the matrix's partial sums (n per matrix).
template <typename TW>
__global__ __launch_bounds__(256) void normalize_kernel(TW* W, long long per_matrix, const float* partials, int n, float eps,
                                                        int bf16_mode) {
  const int b = blockIdx.y;
  __shared__ double red[256];
  const float d = divisor_of(partials + (long long)b * n, n, eps, bf16_mode, red);
  const float rd = 1.f / d;
  const bool fast = __builtin_isfinite(rd) && rd != 0.f;   // (the same for the whole matrix)
  TW* p = W + (long long)b * per_matrix;
  // four 16-byte chunks per thread and trip, all requested before the first is used
  for (long long i0 = (long long)blockIdx.x * 8192; i0 < per_matrix; i0 += (long long)gridDim.x * 8192) {
    float v[4][8];
    bool ok[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const long long i = i0 + (q * 256 + threadIdx.x) * 8;
      ok[q] = i < per_matrix;
      if (ok[q]) Vec8<TW>::load(p + i, v[q]);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (!ok[q]) continue;
      const long long i = i0 + (q * 256 + threadIdx.x) * 8;
      if (fast) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[q][e] = div_by(v[q][e], d, rd);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[q][e] = v[q][e] / d;
      }
      Vec8<TW>::store(p + i, v[q]);
    }
  }
}

// ---------------------------------------------------------------------------------------
// unstage
// ---------------------------------------------------------------------------------------
template <typename TX, typename TW>
struct UnstageArgs {
  DaPtrTable x;       // destinations, one pointer per matrix (rows x cols, row-major, pitch ld)
  const TW* wide;     // [batch][mw][ldw], columns < nw used
  int rows, cols, ld, mw, ldw;
  float decay;        // 1 - lr * weight_decay
  float step;         // adjusted learning rate
  int muon;           // 1: X <- X*decay - wide*step ; 0: X <- wide
  int use_wtab;       // 1: source b is wtab.p[b] (rows x cols contiguous); never with TALL
  DaPtrTable wtab;
  const int* poison;  // optional device word: non-zero = the working matrices are invalid, the result becomes NaN
};

// VEC: the rows of x (and of wtab's matrices) are whole, 16-byte aligned chunks
template <typename TX, typename TW, bool TALL, bool VEC>
__global__ __launch_bounds__(256) void unstage_kernel(UnstageArgs<TX, TW> a) {
  __shared__ float tile[TALL ? TS : 1][TS + 1];
  const bool poisoned = a.poison != nullptr && *a.poison != 0;
  const float nan = __builtin_nanf("");
  const int b = blockIdx.y;
  const int tiles_c = (a.cols + TS - 1) / TS;
  const int ti = blockIdx.x / tiles_c, tj = blockIdx.x % tiles_c;
  const int tid = threadIdx.x;
  TX* X = static_cast<TX*>(a.x.p[b]);
  const TW* W = a.use_wtab ? static_cast<const TW*>(a.wtab.p[b]) : a.wide + (long long)b * a.mw * a.ldw;

  if (!TALL) {
    const int tiles_cw = (a.cols + CT - 1) / CT;
    const int wi = blockIdx.x / tiles_cw, wj = blockIdx.x % tiles_cw;
    constexpr int NC = RT * CT / 8 / 256;
    float u[NC][8], x[NC][8];
    int nv[NC];
#pragma unroll
    for (int it = 0; it < NC; ++it) {
      const int c = tid + 256 * it;
      const int i = wi * RT + c / (CT / 8), j = wj * CT + (c % (CT / 8)) * 8;
      nv[it] = i < a.rows ? a.cols - j : 0;
      if (nv[it] > 0) {
        // (the rows of a working matrix are whole chunks, zero behind the last column)
        if (a.use_wtab) load8<TW, VEC>(W + (long long)i * a.ldw + j, nv[it], u[it]);
        else Vec8<TW>::load(W + (long long)i * a.ldw + j, u[it]);
        if (a.muon) load8<TX, VEC>(X + (long long)i * a.ld + j, nv[it], x[it]);
        if (poisoned) {
#pragma unroll
          for (int e = 0; e < 8; ++e) u[it][e] = nan;
        }
      }
    }
#pragma unroll
    for (int it = 0; it < NC; ++it) {
      if (nv[it] <= 0) continue;
      const int c = tid + 256 * it;
      const int i = wi * RT + c / (CT / 8), j = wj * CT + (c % (CT / 8)) * 8;
      TX* xp = X + (long long)i * a.ld + j;
      if (a.muon) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float xd = Vec8<TX>::round(x[it][e] * a.decay);    // X *= 1 - lr*wd
          const float t = Vec8<TW>::round(u[it][e] * a.step);      // U * adjusted_lr (U's dtype)
          x[it][e] = xd - t;                                       // X -= U ; rounded by the store
        }
        store8<TX, VEC>(xp, nv[it], x[it]);
      } else {
        store8<TX, VEC>(xp, nv[it], u[it]);
      }
    }
    return;
  }
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int c = tid + 256 * it;
    const int p = c >> 3, qq = (c & 7) * 8;
    const int wi = tj * TS + p, wj = ti * TS + qq;
    float u[8];
    if (wi < a.cols && wj < a.rows) Vec8<TW>::load(W + (long long)wi * a.ldw + wj, u);
    else {
#pragma unroll
      for (int e = 0; e < 8; ++e) u[e] = 0.f;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) tile[qq + e][p] = u[e];  // tile[source row][source col]
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int c = tid + 256 * it;
    const int r = c >> 3, cc = (c & 7) * 8;
    const int i = ti * TS + r, j = tj * TS + cc;
    const int n = i < a.rows ? a.cols - j : 0;
    if (n <= 0) continue;
    float u[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) u[e] = tile[r][cc + e];
    if (poisoned) {
#pragma unroll
      for (int e = 0; e < 8; ++e) u[e] = nan;
    }
    TX* xp = X + (long long)i * a.ld + j;
    if (a.muon) {
      float x[8];
      load8<TX, VEC>(xp, n, x);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float xd = Vec8<TX>::round(x[e] * a.decay);    // X *= 1 - lr*wd
        const float t = Vec8<TW>::round(u[e] * a.step);      // U * adjusted_lr (U's dtype)
        x[e] = xd - t;                                       // X -= U ; rounded by the store
      }
      store8<TX, VEC>(xp, n, x);
    } else {
      store8<TX, VEC>(xp, n, u);
    }
  }
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// The vector form is for rows of whole 16-byte chunks at 16-byte aligned addresses: a matrix off the 8-element grid may start
// anywhere (33 rows of 64 elements: whole chunks, but wherever the caller's view begins).
template <typename TG, typename TM, typename TW>
int stage_launch(const StageArgs& a, hipStream_t s) {
  bool vec = true;
  for (int i = 0, mat = 0; i < a.d.ngroups; ++i) {
    const DaStageGroup& g = a.d.g[i];
    vec = vec && !((g.ld | g.cols) & 7);
    for (int b = 0; vec && b < g.cnt; ++b)
      vec = aligned16(a.d.src[mat + b]) && (!a.d.muon || aligned16(a.d.mom[mat + b])) && (g.wide || aligned16(a.d.dst[mat + b]));
    mat += g.cnt;
  }
  const dim3 grid((unsigned)a.blk0[DA_MAX_GROUPS]);
  if (vec) hipLaunchKernelGGL((stage_kernel<TG, TM, TW, true>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((stage_kernel<TG, TM, TW, false>), grid, dim3(256), 0, s, a);
  return da_launch_status();
}

template <typename TG, typename TM>
int stage_dispatch_w(const StageArgs& a, hipStream_t s) {
  return a.d.w_dtype == DA_BF16 ? stage_launch<TG, TM, bf16_t>(a, s) : stage_launch<TG, TM, float>(a, s);
}

template <typename TX, typename TW>
int unstage_launch(const DaUnstage& d, hipStream_t s) {
  bool vec = !((d.ld | (d.use_wtab ? d.ldw : 0) | d.cols) & 7);
  for (int b = 0; vec && b < d.batch; ++b) vec = aligned16(d.x.p[b]) && (!d.use_wtab || aligned16(d.wtab.p[b]));
  UnstageArgs<TX, TW> a{d.x, static_cast<const TW*>(d.wide), d.rows, d.cols, d.ld, d.mw, d.ldw, d.decay, d.step, d.muon, d.use_wtab, d.wtab, d.poison};
  const bool tall = d.rows > d.cols && !d.use_wtab;
  const int tiles = tall ? ((a.rows + TS - 1) / TS) * ((a.cols + TS - 1) / TS)
                         : ((a.rows + RT - 1) / RT) * ((a.cols + CT - 1) / CT);
  dim3 grid(tiles, d.batch);
  if (tall && vec) hipLaunchKernelGGL((unstage_kernel<TX, TW, true, true>), grid, dim3(256), 0, s, a);
  else if (tall) hipLaunchKernelGGL((unstage_kernel<TX, TW, true, false>), grid, dim3(256), 0, s, a);
  else if (vec) hipLaunchKernelGGL((unstage_kernel<TX, TW, false, true>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((unstage_kernel<TX, TW, false, false>), grid, dim3(256), 0, s, a);
  return da_launch_status();
}

}  // namespace

// Workgroups (and partial sums of squares) per matrix of da_stage: transposing tiles for a tall source.
int da_stage_tiles(int rows, int cols, int mw, int nw) {
  return rows > cols ? ((nw + TS - 1) / TS) * ((mw + TS - 1) / TS) : ((mw + RT - 1) / RT) * ((nw + CT - 1) / CT);
}

int da_stage(const DaStage& d, hipStream_t s) {
  if (d.ngroups < 1 || d.ngroups > DA_MAX_GROUPS) return DA_ERR_LIMIT;
  if (d.nzero > 0 && (!d.zero || !d.status)) return DA_ERR_ARG;
  StageArgs a;
  a.d = d;
  long long blocks = 0;
  int mats = 0;
  for (int i = 0; i < d.ngroups; ++i) {
    const DaStageGroup& g = d.g[i];
    if (g.cnt < 1 || g.rows < 1 || g.cols < 1) return DA_ERR_ARG;
    if (g.wide && ((g.mw | g.nw | g.ldw) & 7)) return DA_ERR_ALIGN;
    a.blk0[i] = (int)blocks;
    a.mat0[i] = mats;
    a.tiles[i] = g.wide ? da_stage_tiles(g.rows, g.cols, g.mw, g.nw) : ((g.rows + RT - 1) / RT) * ((g.cols + CT - 1) / CT);
    blocks += (long long)a.tiles[i] * g.cnt;
    mats += g.cnt;
    if (mats > DA_STAGE_MATS || blocks > 0x7fffffffLL) return DA_ERR_LIMIT;
  }
  for (int i = d.ngroups; i <= DA_MAX_GROUPS; ++i) a.blk0[i] = (int)blocks;
  const int gd = d.g_dtype, md = d.muon ? d.m_dtype : d.g_dtype;
  if (gd == DA_BF16 && md == DA_BF16) return stage_dispatch_w<bf16_t, bf16_t>(a, s);
  if (gd == DA_F32 && md == DA_BF16) return stage_dispatch_w<float, bf16_t>(a, s);
  if (gd == DA_BF16 && md == DA_F32) return stage_dispatch_w<bf16_t, float>(a, s);
  if (gd == DA_F32 && md == DA_F32) return stage_dispatch_w<float, float>(a, s);
  return DA_ERR_DTYPE;
}

int da_normalize(void* wide, int w_dtype, long long per_matrix, int batch, const float* partials, int tiles, float eps,
                 hipStream_t s) {
  if (per_matrix & 7) return DA_ERR_ALIGN;
  if (!partials) return DA_ERR_ARG;
  long long blocks = (per_matrix + 8191) / 8192;
  if (blocks > 2048) blocks = 2048;
  dim3 grid((unsigned)blocks, batch);
  if (w_dtype == DA_BF16)
    hipLaunchKernelGGL(normalize_kernel<bf16_t>, grid, dim3(256), 0, s, static_cast<bf16_t*>(wide), per_matrix, partials,
                       tiles, eps, 1);
  else
    hipLaunchKernelGGL(normalize_kernel<float>, grid, dim3(256), 0, s, static_cast<float*>(wide), per_matrix, partials, tiles,
                       eps, 0);
  return da_launch_status();
}

namespace {
// every element of the matrices becomes NaN if *flag != 0 (the launch that produced them gave up)
__global__ __launch_bounds__(256) void poison_multi_kernel(DaPtrUploads u, DaPoisonShape sh, const int* flag) {
  if (*flag == 0) return;
  const int k = blockIdx.z;
  if ((int)blockIdx.y >= u.n[k]) return;
  const float nan = __builtin_nanf("");
  void* p = u.t[k].p[blockIdx.y];
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < sh.numel[k]; i += (long long)gridDim.x * 256) {
    if (sh.f32) static_cast<float*>(p)[i] = nan;
    else static_cast<bf16_t*>(p)[i] = f2bf(nan);
  }
}
}  // namespace

int da_poison_multi_if(const DaPtrUploads& u, int count, const DaPoisonShape& sh, const int* flag, hipStream_t s) {
  if (!flag || count < 1 || count > DA_MAX_UPLOADS) return DA_ERR_ARG;
  hipLaunchKernelGGL(poison_multi_kernel, dim3(64, DA_MAX_PTRS, (unsigned)count), dim3(256), 0, s, u, sh, flag);
  return da_launch_status();
}

int da_unstage(const DaUnstage& d, hipStream_t s) {
  if (d.batch <= 0 || d.batch > DA_MAX_PTRS) return DA_ERR_LIMIT;
  if (!d.use_wtab && (d.ldw & 7)) return DA_ERR_ALIGN;
  if (d.x_dtype == DA_BF16 && d.w_dtype == DA_BF16) return unstage_launch<bf16_t, bf16_t>(d, s);
  if (d.x_dtype == DA_F32 && d.w_dtype == DA_BF16) return unstage_launch<float, bf16_t>(d, s);
  if (d.x_dtype == DA_F32 && d.w_dtype == DA_F32) return unstage_launch<float, float>(d, s);
  if (d.x_dtype == DA_BF16 && d.w_dtype == DA_F32) return unstage_launch<bf16_t, float>(d, s);
  return DA_ERR_DTYPE;
}
