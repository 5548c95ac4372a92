// The fp64 pass of the orthonormaliser and its polishing step for the matrices of a bucket that the fp32 pass left too large a
// defect in, as ONE launch (reference dion/dion.py:1267-1308: P <- P R^-1 with P = Q R).
//
// What bounds it: nothing, as a rule -- no matrix is flagged and the launch returns at once (5 us).  As a launch per product the
// same took 28 to 60 launches that each found out for themselves that there is nothing to do: 75 us of a bucket of rank 192,
// and the host's time to issue them (72 bf16 matrices, rank 192: a step 835 -> 727 us).  For a flagged matrix it is the scheme of dion_small.hip: tasks
// from eight queues, one per XCD (flow_queue.h), a matrix stays with one XCD, counters say when a phase may start:
//   GRAM   P^T P in fp64, lower 32 x 32 tiles, K slices as slabs of their own
//   DIAGj, LOWj   blocked Cholesky factor and its inverse, left-looking (factor_task)
//   PT     S = P L^-T in fp64
//   FIX    the closed form of a second pass: S^T S, columns from noise-level pivots dropped, out = S (I - up(S^T S - I))
// A flagged matrix keeps one XCD busy: large ones are left to the launches per product, which spread over the chip
// (da_orth_flow_applicable).
#include "orth_flow.h"
#include "flow_queue.h"
#include "small_tile.h"

#pragma clang fp contract(off)

namespace {

constexpr int MAX_RT = 62, MAX_BATCH = 256;
constexpr int CTR_GRAM = 0, CTR_FACTOR = 1, CTR_PT = 2, W_GRAM2 = 3, W_BAD = 4, W_SICK = 5, W_RANGE = 6;   // (W_RANGE: two doubles)
constexpr int SMEM = STAGES64 + MAX_RT * 64;

struct Args {
  const char* P;
  char* out;
  const int* need;
  int* info;
  DaOrthFlow w;
  int* words;
  unsigned* tickets;
  int* status;
  unsigned long long spin_limit;
  int batch, rows, r, r_live, rT, mT, slices, kslice;
};

template <bool BF> struct FactorType { typedef float type; };
template <> struct FactorType<true> { typedef bf16_t type; };

template <bool BF>
__global__ __launch_bounds__(256, 2) void orth_flow_kernel(Args args) {
  typedef typename FactorType<BF>::type E;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ int sh_ticket[2], sh_any;
  __shared__ int sh_start[128], sh_per[128];   // the schedule: GRAM, DIAG0, LOW0, DIAG1, .., PT, FIX
  __shared__ unsigned char sh_flag[MAX_BATCH], sh_list[MAX_BATCH / DA_QUEUES];
  const int xcd = xcc_id();
  {
    const int tid = threadIdx.x;
    if (tid == 0) sh_any = 0;
    __syncthreads();
    const int f = tid < args.batch && args.need[tid] != 0;
    sh_flag[tid] = (unsigned char)f;
    if (f) sh_any = 1;
    __syncthreads();
    if (!sh_any) return;
  }
  const int rT = args.rT, rp = rT * 64, t32 = (args.r_live + 31) >> 5, ng = t32 * (t32 + 1) / 2, entries = 2 * rT + 3;
  for (int qi = 0; qi < DA_QUEUES; ++qi) {
    const int q = (xcd + qi) & (DA_QUEUES - 1);
    int nf = 0;
    for (int b = q; b < args.batch; b += DA_QUEUES) nf += sh_flag[b];
    nf = wave_uniform(nf);
    if (nf == 0) continue;
    {
      const int tid = threadIdx.x, lane = tid & 63;
      if (tid == 0) {
        int k = 0;
        for (int b = q; b < args.batch; b += DA_QUEUES)
          if (sh_flag[b]) sh_list[k++] = (unsigned char)(b >> 3);
      }
      if (tid < 128) {
        const int per = tid >= entries ? 0 : tid == 0 ? ng * args.slices : tid == entries - 2 ? args.mT * rT : tid == entries - 1 ? ng + args.mT * rT
                        : (tid & 1) ? 1 : low_tasks(rT, (tid - 1) >> 1);
        sh_per[tid] = per;
        sh_start[tid] = per * nf;
      }
      __syncthreads();
      if (tid < 64) {   // exclusive sums of 128 entries by one wavefront
        const int lo = sh_start[2 * lane], hi = sh_start[2 * lane + 1];
        int sum = lo + hi;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int x = __shfl_up(sum, o);
          if (lane >= o) sum += x;
        }
        sh_start[2 * lane] = sum - lo - hi;
        sh_start[2 * lane + 1] = sum - hi;
        if (lane == 63) sh_any = sum;
      }
      __syncthreads();
    }
    const int total = wave_uniform(sh_any);
    unsigned* word = args.tickets + q * DA_QUEUE_LINE;
    int slot = 0;
    if (threadIdx.x == 0) sh_ticket[0] = take_ticket(word, xcd, total, false);
    while (true) {
      __syncthreads();
      int t = wave_uniform(sh_ticket[slot]);
      if (t < 0) break;
      // (opaque to the compiler: every phase's address arithmetic would move out of this loop and be spilled)
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      const int lane = tid & 63, wave = wave_uniform(tid >> 6), wm = wave >> 1, wn = wave & 1;
      const Args& a = fresh_args<Args>();
      // ---- ticket -> (entry, matrix, task): the last entry that starts at or before it
      const int entry = wave_uniform(__popcll(__ballot(sh_start[lane] <= t)) + __popcll(__ballot(sh_start[64 + lane] <= t)) - 1);
      t -= wave_uniform(sh_start[entry]);
      const int per = wave_uniform(sh_per[entry]);
      const int kth = wave_uniform(t / per), task = wave_uniform(t - kth * per);
      const long long b = wave_uniform((int)sh_list[kth] * DA_QUEUES + q);
      int* const words = a.words + b * DA_ORTH_FLOW_CTL;
      const bool gram = entry == 0, pt = entry == entries - 2, fix = entry == entries - 1;
      if (tid == 0 && !gram) {
        const int j = (entry - 1) >> 1;
        if (fix) {
          wait_count(words + CTR_PT, a.mT * rT, a.status, a.spin_limit);
          if (task >= ng) wait_count(words + W_GRAM2, ng, a.status, a.spin_limit);
        } else if (entry == 1) {
          wait_count(words + CTR_GRAM, ng * a.slices, a.status, a.spin_limit);
        } else {
          // one counter for the phases, rT - 1 tasks to a column (the last: rT): DIAG(j - 1) and what is before it, LOW(j - 2)
          // included, which no later task could stand in for; LOWj likewise
          wait_count(words + CTR_FACTOR, pt ? (rT - 1) * (rT - 1) + rT : ((entry & 1) ? j - 1 : j) * (rT - 1) + 1, a.status, a.spin_limit);
        }
      }
      __syncthreads();
      unsigned next = DA_NO_TICKET;
      const long long rr = (long long)rp * rp, last = (long long)a.rows * a.r - 8;
      const E* const P = reinterpret_cast<const E*>(a.P) + b * ((long long)a.rows * a.r);
      double* const S = a.w.P64 + b * ((long long)a.mT * 64 * rp);
      double* const defect = a.w.defect + b * ((long long)rp * 2 * rT);
      double* const d = reinterpret_cast<double*>(lds);
      int* counter = words + CTR_FACTOR;
      if (gram) {
        counter = words + CTR_GRAM;
        const int slice = wave_uniform(task / ng), kbeg = slice * a.kslice;
        const Opnd<E, true> p = {P, a.r, 1, a.r, a.rows, last};
        int ti, tj;
        gram_tile(p, task - slice * ng, kbeg, min(kbeg + a.kslice, (a.rows + KD - 1) / KD * KD), a.w.slab + (b * a.slices + slice) * rr, rp,
                  d, tid, lane, wm, wn, ti, tj);
        if (tid == 0) next = request_ticket(word);
      } else if (fix && task < ng) {
        counter = words + W_GRAM2;
        int ti, tj;
        gram_tile(work<double>(S, rp, 1), task, 0, (a.rows + KD - 1) / KD * KD, a.w.gram + b * rr, rp, d, tid, lane, wm, wn, ti, tj);
        if (tid == 0) next = request_ticket(word);
        gram_defect(d, defect, 2 * rT, ti, tj, tid);
      } else if (pt || fix) {
        const int t2 = fix ? task - ng : task, row0 = wave_uniform(t2 / rT) * 64, col0 = wave_uniform(t2 % rT) * 64;
        if (pt) {   // S = P T^T (T is triangular)
          counter = words + CTR_PT;
          const Opnd<E, true> p = {P, a.r, 0, a.rows, a.r, last};
          tile16<double, 64>(p, work<double>(a.w.T + b * rr, rp, 0), row0, col0, 0, col0 + 64, d, tid, lane, wm, wn);
        } else {
          unsigned char* const drop = reinterpret_cast<unsigned char*>(lds + STAGES64);
          find_dropped(defect, 2 * rT, a.r_live, rp, drop, tid);
          if (t2 == 0 && tid == 0 && __hip_atomic_load(words + W_BAD, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
            for (int c = 0; c < a.r_live; ++c)
              if (drop[c]) { a.info[b] = c + 1; break; }
          }
          polish_tile(S, a.w.gram + b * rr, a.r_live, rp, drop, row0, col0, d, tid, lane, wm, wn);
        }
        if (tid == 0) next = request_ticket(word);
        if (pt) {
          for (int e = tid; e < 4096; e += 256) S[(long long)(row0 + (e >> 6)) * rp + col0 + (e & 63)] = row0 + (e >> 6) < a.rows ? d[(e >> 6) * 66 + (e & 63)] : 0.0;
        } else {
          const bool poisoned = __hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
          char* const out = a.out + b * ((long long)a.rows * a.r) * (long long)sizeof(E);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int rw = row0 + (tid >> 3) + 32 * h, c = (tid & 7) * 8;
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = poisoned ? __builtin_nanf("") : (float)d[(rw - row0) * 66 + c + i];
            store8(out, !BF, (long long)rw * a.r + col0 + c, rw < a.rows ? a.r - col0 - c : 0, v);
          }
        }
      } else {
        const Factor F = {a.w.slab + b * a.slices * rr, a.w.L + b * rr, a.w.T + b * rr, nullptr, a.slices, a.r_live, rp, rT,
                          words + W_BAD, words + W_SICK, a.info + b, reinterpret_cast<double*>(words + W_RANGE), 0.0};
        factor_task(F, (entry - 1) >> 1, (entry & 1) != 0, task, lds, tid, lane, wave, wm, wn, [] {}, [] {});
        if (tid == 0) next = request_ticket(word);
      }
      // ---- publish: every wavefront's stores are acknowledged, then the counter moves
      if (tid == 0) sh_ticket[slot ^ 1] = ticket_of(next, total);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);   // (in the L2)
      slot ^= 1;
    }
    __syncthreads();   // the next queue's schedule
  }
}

__global__ __launch_bounds__(256) void orth_flow_setup_kernel(int* words, int n, int* status, int preset) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) words[i] = 0;
  if (i == 0) *status = preset;
}

}  // namespace

int da_orth_flow_slices(int rows, int r) {
  // enough Gram tasks for an XCD's 32 compute units, at least 128 rows each
  const int t32 = (r + 31) / 32, tiles = t32 * (t32 + 1) / 2;
  int slices = (64 + tiles - 1) / tiles;
  if (slices > rows / 128) slices = rows / 128;
  if (slices < 1) slices = 1;
  const int kslice = ((rows + slices - 1) / slices + KD - 1) / KD * KD;
  return (rows + kslice - 1) / kslice;
}

// Where the line lies: a flagged matrix has one XCD to itself at best, the launches per product the whole chip.  A full-rank
// factor of a fresh Q is flagged (12 of 3072 x 768 each in two buckets: 13.4 ms a step in one launch, 6.8 ms in many), so the
// work per matrix is kept to what one XCD does in about half a millisecond.
bool da_orth_flow_applicable(int rows, int r) {
  return (r + 63) / 64 <= MAX_RT && (long long)rows * r >= 8 && (double)rows * r * r <= 4e8;
}

int da_orth_flow(const void* P, void* out, int dtype, int batch, int rows, int r, int r_live, const int* need, int* info,
                 const DaOrthFlow& w, int fail, hipStream_t s) {
  if (!da_orth_flow_applicable(rows, r)) return DA_ERR_LIMIT;
  static DaOncePerDevice configured;
  int rc = configured.run([&]() -> int {
    DA_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(orth_flow_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize, SMEM));
    DA_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(orth_flow_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize, SMEM));
    return DA_OK;
  });
  if (rc) return rc;
  const long long esz = dtype == DA_BF16 ? 2 : 4, per = (long long)rows * r;
  for (int b0 = 0; b0 < batch; b0 += MAX_BATCH) {
    Args a{};
    a.rT = (r + 63) / 64;
    a.mT = (rows + 63) / 64;
    const long long rp = a.rT * 64, rr = rp * rp;
    a.slices = da_orth_flow_slices(rows, r);
    a.kslice = ((rows + a.slices - 1) / a.slices + KD - 1) / KD * KD;
    a.P = static_cast<const char*>(P) + b0 * per * esz;
    a.out = static_cast<char*>(out) + b0 * per * esz;
    a.need = need + b0;
    a.info = info + b0;
    a.w = {w.P64 + b0 * (long long)a.mT * 64 * rp, w.slab + b0 * rr * a.slices, w.L + b0 * rr, w.T + b0 * rr, w.gram + b0 * rr,
           w.defect + b0 * rp * 2 * a.rT, w.ctl};
    a.batch = batch - b0 < MAX_BATCH ? batch - b0 : MAX_BATCH;
    a.words = w.ctl;
    a.tickets = reinterpret_cast<unsigned*>(w.ctl + a.batch * DA_ORTH_FLOW_CTL);
    a.status = reinterpret_cast<int*>(a.tickets + DA_QUEUES * DA_QUEUE_LINE);
    a.spin_limit = 500000000ull;   // 5 s of the 100 MHz counter
    a.rows = rows; a.r = r; a.r_live = r_live;
    const int n = a.batch * DA_ORTH_FLOW_CTL + DA_QUEUES * DA_QUEUE_LINE;
    hipLaunchKernelGGL(orth_flow_setup_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a.words, n, a.status, fail);
    rc = da_launch_status();
    if (rc) return rc;
    const dim3 grid(2 * (unsigned)da_cu_count());
    if (dtype == DA_BF16) hipLaunchKernelGGL(orth_flow_kernel<true>, grid, dim3(256), SMEM, s, a);
    else hipLaunchKernelGGL(orth_flow_kernel<false>, grid, dim3(256), SMEM, s, a);
    rc = da_launch_status();
    if (rc) return rc;
  }
  return DA_OK;
}
