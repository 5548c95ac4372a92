// Newton-Schulz on a set of small matrices in ONE launch: division by the Frobenius norm, all iterations
//
//   A = X X^T ;  B = b A + c A A ;  X' = a X + B X                        (reference dion/muon.py:633-645)
//
// and the store of the result, or the weight update it is for.
//
// What bounds it: a chain of 3 dependent products per iteration, each far too small for the chip (256 x 768: 10 to 48
// tiles of 64 x 64, 4 to 12 stages of k).  Launched product by product every link costs a launch (4-5 us from launch to
// drain) and a K loop that waits for one stage at a time (9-11 us per product, 165 us for the whole call).  Here the
// links are counters in device memory, and a tile keeps three stages of k in flight.
//
// Split.  Workgroups of 256 threads, two per compute unit, take tiles from eight queues, one per XCD; every matrix
// belongs to one queue, so all tiles of a matrix, producers and consumers, meet in one L2: a finished tile waits for its
// stores to be acknowledged (they are then in that L2) and moves its matrix's counter, and every load of what this launch
// wrote goes past the L1.  The first XCD that takes a ticket of a queue owns it.  Tickets run (phase, matrix, tile): a tile's
// producers hold smaller tickets of the same queue, so a waiting workgroup waits only for workgroups that are running,
// whatever the placement.  Ready workgroups of the next phase are already waiting when a phase ends: tickets and address
// arithmetic stay off the critical path.
//
// Every wait is bounded: after `spin_limit` ticks of the 100 MHz counter a workgroup sets the status word and goes on
// without what it waited for; waits end at once from then on, and the last product's tiles store NaN when they find the
// status word set.  It is set before the counter of the tile that went on, so no tile that depends on that one
// (directly or not) can miss it.
//
// Tiles are 64 x 64 (K in 64-deep stages), or 32 x 32 (128-deep stages) for the symmetric products of a launch that has
// few of them: a 64-tile's stage costs 0.3 us, most of it LDS traffic (16 KB in, 32 KB of fragment reads), and an XCD has
// 32 compute units for the 10 tiles of a 256-row product.  Either way four LDS buffers of 16 KB, two workgroups per compute
// unit, three stages in flight (eight buffers and one workgroup measured no faster).  Operand layouts, swizzles, MFMA
// instruction, order of k and rounding-faithful epilogue arithmetic are those of gemm_bf16_tile.h, so the products have the
// same bits as the batched kernel's.
#include "ns_small.h"
#include "flow_queue.h"
#include "gemm_bf16_tile.h"

namespace {

typedef Cfg<64, 2, 2> Sm;
constexpr int BT = DA_SMALL_BT;
constexpr int NQ = DA_QUEUES;
constexpr int NST = 4;                     // LDS stage buffers
constexpr int STAGE = 2 * BT * BK * 2;     // bytes of one stage: both operands
constexpr int PITCH = BT + 4;              // floats per row of the epilogue's staging area
constexpr int NORM_ELEMS = 8192;           // elements per normalisation task
static_assert(Sm::NT == 256 && Sm::TMI == 2 && Sm::TNJ == 2 && Sm::NCH == 2, "the K loop below is written for this shape");
static_assert(BT * PITCH * 4 <= 4 * STAGE, "the epilogue stages through the K loop's buffers");

struct GroupDev {
  char *x0, *x1, *a, *b;
  long long sx, sa;
  const float* partials;
  void* const* tab;
  int* counters;             // [cnt][DA_SMALL_CTR_STRIDE]
  int ldx, lda;
  int tm, tn, tnorm, ptiles;
  int cnt, first;            // matrices; index of the first one in the dealing order
  int dtype, rows, cols, ld, update, vec;
  float decay, step;
};

struct SmallArgs {
  GroupDev g[DA_MAX_GROUPS];
  float coeffs[3 * DA_SMALL_MAX_STEPS];
  unsigned* tickets;         // [NQ][DA_QUEUE_LINE]
  int* status;
  unsigned long long spin_limit;
  float eps;
  int ngroups, steps;
  int sym32;                 // the symmetric products in 32 x 32 tiles
};

__device__ __forceinline__ int in_queue(const GroupDev& G, int q) { return da_in_queue(G.first, G.cnt, q); }
// tasks per matrix: kind 0 normalisation, 1 / 2 the symmetric products, 3 X'
__device__ __forceinline__ int tasks_of(const GroupDev& G, int kind, int sym32) {
  if (kind == 0) return G.tnorm;
  if (kind == 3) return G.tm * G.tn;
  return sym32 ? G.tm * (2 * G.tm + 1) : G.tm * (G.tm + 1) / 2;
}

struct Item { int phase, kind, g, b, t; };

// ticket t of queue q; phase 0: normalisation, phase 1 + 3 it + p: product p of iteration it
__device__ __forceinline__ Item decode(const SmallArgs& a, int q, int t) {
  int n0 = 0, ns = 0, nx = 0;
  for (int g = 0; g < a.ngroups; ++g) {
    const int nq = in_queue(a.g[g], q);
    n0 += nq * tasks_of(a.g[g], 0, a.sym32);
    ns += nq * tasks_of(a.g[g], 1, a.sym32);
    nx += nq * tasks_of(a.g[g], 3, a.sym32);
  }
  Item r;
  if (t < n0) {
    r.phase = 0; r.kind = 0;
  } else {
    t -= n0;
    const int per_it = 2 * ns + nx;
    const int it = t / per_it;
    t -= it * per_it;
    int p = 0;
    if (t >= ns) { t -= ns; p = 1; }
    if (p == 1 && t >= ns) { t -= ns; p = 2; }
    r.phase = 1 + 3 * it + p;
    r.kind = 1 + p;
  }
  // X X^T takes the groups costliest first (the order they are given in), the products behind it cheapest first
  r.g = 0; r.b = 0; r.t = 0;
  bool found = false;
  for (int i = 0; i < a.ngroups; ++i) {
    const int g = r.kind <= 1 ? i : a.ngroups - 1 - i;
    const GroupDev& G = a.g[g];
    const int nq = in_queue(G, q), per = tasks_of(G, r.kind, a.sym32);
    if (found) continue;
    if (t < nq * per || i + 1 == a.ngroups) {
      const int k = t / per;
      found = true;
      r.g = g;
      r.t = t - k * per;
      r.b = ((q - G.first) & 7) + 8 * k;     // the k-th matrix of the group whose dealing index is q modulo 8
    } else {
      t -= nq * per;
    }
  }
  return r;
}

// Waits until at most the loads of n stages behind the one needed are in flight: four direct-to-LDS loads each, completed
// in the order issued.
__device__ __forceinline__ void wait_stages(int n) {
  if (n >= 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  else if (n == 1) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  else dma_wait();
}

// acc += A-rows (m0 ...) x B-rows (n0 ...) over KT 64-deep stages, direct-to-LDS loads NST - 1 stages ahead.
template <bool B_KS>
__device__ __forceinline__ void small_k_loop(Sm::acc_t (&acc)[2][2], const bf16_t* A, int lda, const bf16_t* B, int ldb,
                                             int dim_m, int dim_n, int m0, int n0, int KT, char* lds, int tid, int lane,
                                             int wave, int wm, int wn) {
  StageAddr<Sm, false> sa(A, lda, m0, tid, dim_m);
  StageAddr<Sm, B_KS> sb(B, ldb, n0, tid, dim_n);
  const unsigned ts_a = (unsigned)(sa.tstep * 2), ts_b = (unsigned)(sb.tstep * 2);
  unsigned koff_a = 0, koff_b = 0;
  auto issue = [&](int kt) {
    const unsigned st = lds_addr(lds) + (unsigned)(kt % NST) * STAGE;
#pragma unroll
    for (int i = 0; i < 2; ++i) dma16_l2(sa.dbase, sa.doff + i * sa.dstep + koff_a, st + (i * 4 + wave) * 1024);
#pragma unroll
    for (int i = 0; i < 2; ++i) dma16_l2(sb.dbase, sb.doff + i * sb.dstep + koff_b, st + STAGE / 2 + (i * 4 + wave) * 1024);
    koff_a += ts_a;
    koff_b += ts_b;
  };
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.f;
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < KT) issue(s);
  for (int kt = 0; kt < KT; ++kt) {
    wait_stages(min(KT - 1 - kt, NST - 2));
    __syncthreads();
    if (kt + NST - 1 < KT) issue(kt + NST - 1);   // into the buffer whose last readers are past the barrier above
    const char* st = lds + (kt % NST) * STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8_t fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[i] = read_frag16<BT, false>(st, wm * 32 + i * 16, ks, lane);
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[j] = read_frag16<BT, B_KS>(st + STAGE / 2, wn * 32 + j * 16, ks, lane);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
  }
  __syncthreads();
}

// The same for a 32 x 32 tile of a product of two k-contiguous operands (one 16 x 16 block per wavefront), 128-deep stages
// of two 8 KB halves; an odd last half is loaded twice so that every stage has its four loads, and used once.
__device__ __forceinline__ void small_k_loop32(f32x4_t& acc, const bf16_t* A, int ld, int m0, int n0, int KT, char* lds,
                                               int lane, int wave, int wm, int wn) {
  const char* pa = reinterpret_cast<const char*>(A + (long long)m0 * ld);
  const char* pb = reinterpret_cast<const char*>(A + (long long)n0 * ld);
  const int drow = wave * 8 + (lane >> 3);
  const unsigned off = (unsigned)(drow * ld + kc_swizzle(lane & 7, drow) * 8) * 2u;
  const int KS = (KT + 1) >> 1;
  auto issue = [&](int s) {
    const unsigned st = lds_addr(lds) + (unsigned)(s % NST) * STAGE + wave * 1024;
    const unsigned k0 = (unsigned)s * 256u, k1 = 2 * s + 1 < KT ? k0 + 128u : k0;
    dma16_l2(pa, off + k0, st);
    dma16_l2(pb, off + k0, st + 4096);
    dma16_l2(pa, off + k1, st + 8192);
    dma16_l2(pb, off + k1, st + 12288);
  };
#pragma unroll
  for (int v = 0; v < 4; ++v) acc[v] = 0.f;
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < KS) issue(s);
  for (int s = 0; s < KS; ++s) {
    wait_stages(min(KS - 1 - s, NST - 2));
    __syncthreads();
    if (s + NST - 1 < KS) issue(s + NST - 1);
    const char* st = lds + (s % NST) * STAGE;
    bf16x8_t fa[4], fb[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      fa[k] = read_frag16<32, false>(st + (k >> 1) * 8192, wm * 16, k & 1, lane);
      fb[k] = read_frag16<32, false>(st + (k >> 1) * 8192 + 4096, wn * 16, k & 1, lane);
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[0], fa[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[1], fa[1], acc, 0, 0, 0);
    if (2 * s + 1 < KT) {
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[2], fa[2], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[3], fa[3], acc, 0, 0, 0);
    }
  }
  __syncthreads();
}

__device__ __forceinline__ u32x4_t pack8(const float (&v)[8]) {
  u32x4_t o;
#pragma unroll
  for (int q = 0; q < 4; ++q) o[q] = cvt_pk_bf16(v[2 * q], v[2 * q + 1]);
  return o;
}

// Destination row access: 8 elements at column c of a row of `cols` elements; `vec`: 16-byte aligned whole chunks.
struct Dest {
  char* p;
  int rows, cols, ld, f32, vec;
  __device__ __forceinline__ int valid(int r, int c) const { return r < rows ? min(8, cols - c) : 0; }
  __device__ __forceinline__ void load(int r, int c, float (&w)[8]) const {
    const int n = valid(r, c);
    const char* q = p + ((long long)r * ld + c) * (f32 ? 4 : 2);
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = 0.f;
    if (n <= 0) return;
    if (vec && n == 8) {
      const u32x4_t x = ldg16(q);
      if (f32) {
        const u32x4_t y = ldg16(q + 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned xe = x[e], ye = y[e];   // (copied out: bit_cast of a vector element lvalue reads element 0)
          w[e] = __builtin_bit_cast(float, xe);
          w[4 + e] = __builtin_bit_cast(float, ye);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) { w[2 * e] = lo_f(x[e]); w[2 * e + 1] = hi_f(x[e]); }
      }
      return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < n) w[e] = f32 ? reinterpret_cast<const float*>(q)[e] : bf2f(reinterpret_cast<const bf16_t*>(q)[e]);
  }
  __device__ __forceinline__ void store(int r, int c, const float (&w)[8]) const {
    const int n = valid(r, c);
    char* q = p + ((long long)r * ld + c) * (f32 ? 4 : 2);
    if (n <= 0) return;
    if (vec && n == 8) {
      if (f32) {
        u32x4_t x, y;
#pragma unroll
        for (int e = 0; e < 4; ++e) { x[e] = __builtin_bit_cast(unsigned, w[e]); y[e] = __builtin_bit_cast(unsigned, w[4 + e]); }
        stg16(q, x);
        stg16(q + 16, y);
      } else {
        stg16(q, pack8(w));
      }
      return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < n) {
        if (f32) reinterpret_cast<float*>(q)[e] = w[e];
        else reinterpret_cast<bf16_t*>(q)[e] = f2bf(w[e]);
      }
  }
};

__global__ __launch_bounds__(256, 2) void ns_small_kernel(SmallArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ int sh_ticket[2];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = wave_uniform(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int xcd = xcc_id();

  for (int qi = 0; qi < NQ; ++qi) {
    const int q = (xcd + qi) & (NQ - 1);
    int total = 0, norms = 0;
    for (int g = 0; g < a.ngroups; ++g) {
      const int nq = in_queue(a.g[g], q);
      norms += nq * tasks_of(a.g[g], 0, a.sym32);
      total += nq * (2 * tasks_of(a.g[g], 1, a.sym32) + tasks_of(a.g[g], 3, a.sym32));
    }
    total = total * a.steps + norms;
    if (total <= 0) continue;
    int slot = 0;
    if (tid == 0) sh_ticket[0] = take_ticket(a.tickets + q * DA_QUEUE_LINE, xcd, total, false);
    while (true) {
      __syncthreads();
      const int t = wave_uniform(sh_ticket[slot]);
      if (t < 0) break;
      Item w = decode(a, q, t);
      // (the divisions run on the vector unit: back into scalar registers, or every address below is per lane)
      w.phase = wave_uniform(w.phase); w.kind = wave_uniform(w.kind); w.g = wave_uniform(w.g);
      w.b = wave_uniform(w.b); w.t = wave_uniform(w.t);
      const GroupDev& G = a.g[w.g];
      int* ctr = G.counters + (long long)w.b * DA_SMALL_CTR_STRIDE + w.phase;
      const int it = (w.phase - 1) / 3;
      if (tid == 0) {
        if (w.phase > 0) {
          // the product this tile reads must be complete for its matrix
          const int want = tasks_of(G, w.phase == 1 ? 0 : (w.kind == 1 ? 3 : w.kind - 1), a.sym32);
          wait_count(ctr - 1, want, a.status, a.spin_limit);
        }
      }
      __syncthreads();

      int next = -1;   // (thread 0) the next ticket, asked for when this task is on its way: not earlier, or a waiting
                       // workgroup would hold two tasks of a phase while others have none
      auto ask = [&]() {
        if (tid == 0) next = take_ticket(a.tickets + q * DA_QUEUE_LINE, xcd, total, true);
      };
      if (w.kind == 0) {
        // ---- X <- X / (||X||_F + eps), the divisor from the matrix's partial sums (the order and the roundings of
        // normalize_kernel in elementwise.hip)
        double* red = reinterpret_cast<double*>(lds);
        const float* part = G.partials + (long long)w.b * G.ptiles;
        const long long per = (long long)G.tm * BT * G.ldx;
        char* X = G.x0 + (long long)w.b * G.sx * 2;
        const long long i0 = (long long)w.t * NORM_ELEMS + tid * 8;
        u32x4_t v[4];
        bool ok[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          ok[k] = i0 + k * 2048 < per;
          if (ok[k]) v[k] = ldg16(X + (i0 + k * 2048) * 2);
        }
        ask();
        double sum = 0.0;
        for (int i = tid; i < G.ptiles; i += 256) sum += (double)part[i];
        red[tid] = sum;
        __syncthreads();
        if (G.ptiles > 64) {   // (at most 64 partial sums: the upper three quarters are zero)
          for (int o = 128; o > 32; o >>= 1) {
            if (tid < o) red[tid] += red[tid + o];
            __syncthreads();
          }
        }
        sum = red[lane];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_down(sum, o, 64);
        const float nrm = sqrtf((float)__shfl(sum, 0, 64));
        const float d = rbf(rbf(nrm) + a.eps);
        const float rd = 1.f / d;
        const bool fast = __builtin_isfinite(rd) && rd != 0.f;
        auto div = [&](float x) {
          if (!fast) return x / d;
          const float y = x * rd;
          return __builtin_fmaf(__builtin_fmaf(-y, d, x), rd, y);
        };
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (!ok[k]) continue;
          u32x4_t o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = cvt_pk_bf16(div(lo_f(v[k][e])), div(hi_f(v[k][e])));
          stg16(X + (i0 + k * 2048) * 2, o);
        }
      } else {
        // ---- one tile of a product
        const float ca = a.coeffs[3 * it], cb = a.coeffs[3 * it + 1], cc = a.coeffs[3 * it + 2];
        const char* xcur = ((it & 1) ? G.x1 : G.x0) + (long long)w.b * G.sx * 2;
        char* xnext = ((it & 1) ? G.x0 : G.x1) + (long long)w.b * G.sx * 2;
        char* pa = G.a + (long long)w.b * G.sa * 2;
        char* pb = G.b + (long long)w.b * G.sa * 2;
        int ti, tj;
        const bool t32 = w.kind != 3 && a.sym32 != 0;
        if (w.kind == 3) {
          ti = w.t / G.tn;
          tj = w.t - ti * G.tn;
        } else {
          ti = 0;
          int rem = w.t, len = t32 ? 2 * G.tm : G.tm;
          while (rem >= len) { rem -= len; ++ti; --len; }
          tj = ti + rem;
        }
        ti = wave_uniform(ti);
        tj = wave_uniform(tj);
        char* C = w.kind == 3 ? xnext : (w.kind == 2 ? pb : pa);
        const int ldc = w.kind == 3 ? G.ldx : G.lda;
        const bool mirror = w.kind != 3 && ti != tj;
        if (t32) {
          const int m0 = ti * 32, n0 = tj * 32;
          // the first 128 threads own one 8-element chunk of the tile each
          const int cr = tid >> 2, c8 = (tid & 3) * 8;
          const bool own = tid < 128;
          u32x4_t ev;
          if (w.kind == 2 && own) ev = ldg16_l2(pa + ((long long)(m0 + cr) * G.lda + n0 + c8) * 2);
          f32x4_t acc;
          small_k_loop32(acc, reinterpret_cast<const bf16_t*>(w.kind == 1 ? xcur : pa), w.kind == 1 ? G.ldx : G.lda, m0, n0,
                         w.kind == 1 ? G.tn : G.tm, lds, lane, wave, wm, wn);
          ask();
          float* stg = reinterpret_cast<float*>(lds);
          *reinterpret_cast<float4*>(stg + (wm * 16 + (lane & 15)) * 36 + wn * 16 + (lane >> 4) * 4) =
              make_float4(acc[0], acc[1], acc[2], acc[3]);
          __syncthreads();
          if (own) {
            float* sp = stg + cr * 36 + c8;
            const float4 a0 = *reinterpret_cast<const float4*>(sp);
            const float4 a1 = *reinterpret_cast<const float4*>(sp + 4);
            const float v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
            u32x4_t pk = pack8(v);
            if (w.kind == 2) {
#pragma unroll
              for (int e = 0; e < 4; ++e) pk[e] = epi_pair<true, true, false>(cb, cc, v[2 * e], v[2 * e + 1], ev[e]);
            }
            stg16(C + ((long long)(m0 + cr) * ldc + n0 + c8) * 2, pk);
            if (mirror) {
              *reinterpret_cast<float4*>(sp) = make_float4(lo_f(pk[0]), hi_f(pk[0]), lo_f(pk[1]), hi_f(pk[1]));
              *reinterpret_cast<float4*>(sp + 4) = make_float4(lo_f(pk[2]), hi_f(pk[2]), lo_f(pk[3]), hi_f(pk[3]));
            }
          }
          if (mirror) {
            __syncthreads();
            if (own) {
              float v[8];
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] = stg[(c8 + e) * 36 + cr];
              stg16(C + ((long long)(n0 + cr) * ldc + m0 + c8) * 2, pack8(v));
            }
          }
        } else {
        const int m0 = ti * BT, n0 = tj * BT;
        const bool last = w.kind == 3 && it + 1 == a.steps;
        const bool turned = last && G.rows > G.cols;
        const Dest dst = {last ? static_cast<char*>(G.tab[w.b]) : nullptr, G.rows, G.cols, G.ld, G.dtype == DA_F32, G.vec};
        // a thread's two 8-element chunks of the tile: row cr + 32 h, columns cc8 ...; requested before the K loop
        const int cr = tid >> 3, c8 = (tid & 7) * 8;
        u32x4_t ev[2];
        float wv[2][8];
        const char* E = w.kind == 3 ? xcur : pa;
        const int lde = w.kind == 3 ? G.ldx : G.lda;
        if (w.kind != 1) {
#pragma unroll
          for (int h = 0; h < 2; ++h) ev[h] = ldg16_l2(E + ((long long)(m0 + cr + 32 * h) * lde + n0 + c8) * 2);
        }
        if (last && G.update) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if (turned) dst.load(n0 + cr + 32 * h, m0 + c8, wv[h]);
            else dst.load(m0 + cr + 32 * h, n0 + c8, wv[h]);
          }
        }
        Sm::acc_t acc[2][2];
        const int mw = G.tm * BT, nw = G.tn * BT;
        if (w.kind == 3)
          small_k_loop<true>(acc, reinterpret_cast<const bf16_t*>(pb), G.lda, reinterpret_cast<const bf16_t*>(xcur), G.ldx, mw,
                             nw, m0, n0, G.tm, lds, tid, lane, wave, wm, wn);
        else if (w.kind == 2)
          small_k_loop<false>(acc, reinterpret_cast<const bf16_t*>(pa), G.lda, reinterpret_cast<const bf16_t*>(pa), G.lda, mw,
                              mw, m0, n0, G.tm, lds, tid, lane, wave, wm, wn);
        else
          small_k_loop<false>(acc, reinterpret_cast<const bf16_t*>(xcur), G.ldx, reinterpret_cast<const bf16_t*>(xcur), G.ldx,
                              mw, mw, m0, n0, G.tn, lds, tid, lane, wave, wm, wn);
        ask();
        // ---- epilogue through LDS
        float* stg = reinterpret_cast<float*>(lds);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            *reinterpret_cast<float4*>(stg + (wm * 32 + i * 16 + (lane & 15)) * PITCH + wn * 32 + j * 16 + (lane >> 4) * 4) =
                make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
        __syncthreads();
        const bool poisoned = last && __hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
        auto finish = [&](int r, int c, u32x4_t pk, const float (&x)[8]) {   // a chunk of the result at its destination
          float o[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            float u = (e & 1) ? hi_f(pk[e >> 1]) : lo_f(pk[e >> 1]);
            if (poisoned) u = __builtin_nanf("");
            if (G.update) {
              float xd = x[e] * G.decay;
              if (G.dtype != DA_F32) xd = rbf(xd);
              u = xd - rbf(u * G.step);     // (rounded to the weights' dtype by the store)
            }
            o[e] = u;
          }
          dst.store(r, c, o);
        };
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          float* sp = stg + (cr + 32 * h) * PITCH + c8;
          const float4 a0 = *reinterpret_cast<const float4*>(sp);
          const float4 a1 = *reinterpret_cast<const float4*>(sp + 4);
          const float v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
          u32x4_t pk;
          if (w.kind == 1) {
            pk = pack8(v);
          } else if (w.kind == 2) {
#pragma unroll
            for (int e = 0; e < 4; ++e) pk[e] = epi_pair<true, true, false>(cb, cc, v[2 * e], v[2 * e + 1], ev[h][e]);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) pk[e] = epi_pair<true, true, true>(ca, 1.f, v[2 * e], v[2 * e + 1], ev[h][e]);
          }
          if (!last) stg16(C + ((long long)(m0 + cr + 32 * h) * ldc + n0 + c8) * 2, pk);
          else if (!turned) finish(m0 + cr + 32 * h, n0 + c8, pk, wv[h]);
          if (mirror || turned) {
            *reinterpret_cast<float4*>(sp) = make_float4(lo_f(pk[0]), hi_f(pk[0]), lo_f(pk[1]), hi_f(pk[1]));
            *reinterpret_cast<float4*>(sp + 4) = make_float4(lo_f(pk[2]), hi_f(pk[2]), lo_f(pk[3]), hi_f(pk[3]));
          }
        }
        if (mirror || turned) {
          __syncthreads();
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = stg[(c8 + e) * PITCH + cr + 32 * h];
            const u32x4_t pk = pack8(v);
            if (mirror) stg16(C + ((long long)(n0 + cr + 32 * h) * ldc + m0 + c8) * 2, pk);
            else finish(n0 + cr + 32 * h, m0 + c8, pk, wv[h]);
          }
        }
        }
      }
      // ---- publish: every wavefront's stores are acknowledged, then the matrix's counter moves
      if (tid == 0) sh_ticket[slot ^ 1] = next;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);   // (executed in the L2)
      slot ^= 1;
    }
    __syncthreads();   // thread 0 rewrites sh_ticket for the next queue
  }
}

}  // namespace

bool da_ns_small_applicable(const DaNsSmallGroup* g, int n, int steps) {
  if (n < 1 || n > DA_MAX_GROUPS || steps < 1 || steps > DA_SMALL_MAX_STEPS) return false;
  for (int i = 0; i < n; ++i) {
    if (g[i].cnt < 1 || g[i].mw % BT || g[i].nw % BT || g[i].mw > g[i].nw) return false;
    // 32-bit byte offsets inside a tile's operand panels
    if ((long long)g[i].mw * g[i].ldx * 2 >= (1LL << 31) || (long long)g[i].mw * g[i].lda * 2 >= (1LL << 31)) return false;
  }
  return true;
}

int da_ns_small(const DaNsSmallGroup* g, int n, const float* coeffs, int steps, float eps, int* ctl, hipStream_t s) {
  if (!g || !coeffs || !ctl || !da_ns_small_applicable(g, n, steps)) return DA_ERR_ARG;
  SmallArgs a{};
  int first = 0;
  long long tickets = 0;
  for (int i = 0; i < n; ++i) {
    const DaNsSmallGroup& G = g[i];
    if (!G.x0 || !G.x1 || !G.a || !G.b || !G.partials || !G.tab || G.ptiles < 1) return DA_ERR_ARG;
    if ((G.ldx & 7) || (G.lda & 7) || (G.sx & 7) || (G.sa & 7)) return DA_ERR_ALIGN;
    if (G.dtype != DA_BF16 && (G.dtype != DA_F32 || !G.update)) return DA_ERR_DTYPE;
    const bool tall = G.rows > G.cols;
    if ((tall ? G.cols : G.rows) > G.mw || (tall ? G.rows : G.cols) > G.nw) return DA_ERR_ARG;
    GroupDev& D = a.g[i];
    D.x0 = G.x0; D.x1 = G.x1; D.a = G.a; D.b = G.b;
    D.sx = G.sx; D.sa = G.sa; D.ldx = G.ldx; D.lda = G.lda;
    D.partials = G.partials; D.ptiles = G.ptiles; D.tab = G.tab;
    D.counters = ctl + (size_t)first * DA_SMALL_CTR_STRIDE;
    D.tm = G.mw / BT; D.tn = G.nw / BT;
    D.tnorm = (int)(((long long)G.mw * G.ldx + NORM_ELEMS - 1) / NORM_ELEMS);
    D.cnt = G.cnt; D.first = first;
    D.dtype = G.dtype; D.rows = G.rows; D.cols = G.cols; D.ld = G.ld; D.update = G.update;
    D.vec = G.vec;
    D.decay = G.decay; D.step = G.step;
    first += G.cnt;
    tickets += (long long)G.cnt * (D.tnorm + steps * (D.tm * (D.tm + 1) + D.tm * D.tn));
  }
  if (tickets >= (1LL << 27)) return DA_ERR_LIMIT;
  for (int i = 0; i < 3 * steps; ++i) a.coeffs[i] = coeffs[i];
  a.ngroups = n; a.steps = steps; a.eps = eps;
  int* tail = ctl + (size_t)first * DA_SMALL_CTR_STRIDE;
  a.tickets = reinterpret_cast<unsigned*>(tail);
  a.status = tail + NQ * DA_QUEUE_LINE;
  a.spin_limit = 200000000ull;   // 2 s of the 100 MHz counter
  // 32-tiles for the symmetric products while those of every queue fit one and a half rounds of its 64 workgroups
  long long most = 0;
  for (int q = 0; q < NQ; ++q) {
    long long sym = 0;
    for (int i = 0; i < n; ++i) sym += (long long)((a.g[i].first + a.g[i].cnt - q + 7) / 8 - (a.g[i].first - q + 7) / 8) * a.g[i].tm * (2 * a.g[i].tm + 1);
    most = sym > most ? sym : most;
  }
  if (most <= 96) a.sym32 = 1;
  static DaOncePerDevice configured;
  const int rc = configured.run([&]() -> int {
    DA_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(ns_small_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, NST * STAGE));
    return DA_OK;
  });
  if (rc) return rc;
  hipLaunchKernelGGL(ns_small_kernel, dim3(2 * (unsigned)da_cu_count()), dim3(Sm::NT), NST * STAGE, s, a);
  return da_launch_status();
}
