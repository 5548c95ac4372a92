// Ticket queues of the kernels for small matrices that run a chain of phases (ns_small.hip, dion_small.hip): eight queues, one per XCD.
#pragma once
#include "common.h"

constexpr int DA_QUEUES = 8;          // = XCDs
constexpr int DA_QUEUE_LINE = 32;     // ints: every queue's words have a 128-byte line of their own

namespace {

__host__ __device__ inline int ceil8(int x) { return (x + 7) >> 3; }   // x >= -7
// how many of the matrices first .. first + cnt - 1 (in dealing order) belong to queue q
__host__ __device__ inline int da_in_queue(int first, int cnt, int q) { return ceil8(first + cnt - q) - ceil8(first - q); }

// The kernel's arguments (its first and only parameter, of type A), opaque to the compiler: read again where they are used.  Hoisted
// out of a persistent loop they take more scalar registers than there are, and are spilled.
template <typename A>
__device__ __forceinline__ const A& fresh_args() {
  typedef const __attribute__((address_space(4))) A* ptr_t;
  ptr_t p = (ptr_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const A*)p;
}

__device__ __forceinline__ int xcc_id() { return (int)(__builtin_amdgcn_s_getreg(20 | (3 << 11)) & 7u); }
__device__ __forceinline__ unsigned long long now_ticks() { return __builtin_amdgcn_s_memrealtime(); }

// Next ticket of a queue for a workgroup on XCD `xcd`, or -1: the queue is used up or belongs to another XCD.  word[0] is
// the ticket counter, word[1] the owner (XCD + 1): the first XCD that asks.  Only the owner's workgroups touch the
// counter, so its atomics need no more than the XCD's own L2 (workgroup scope: no sc1 bit): of agent scope they take
// 130 ns each, one after the other, 8 us for the 64 tiles of a 512 x 512 product.
__device__ __forceinline__ int take_ticket(unsigned* word, int xcd, int total, bool owned) {
  const unsigned me = (unsigned)(xcd + 1);
  if (!owned) {
    unsigned cur = __hip_atomic_load(word + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (cur == 0) {
      unsigned expect = 0;
      cur = __hip_atomic_compare_exchange_strong(word + 1, &expect, me, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT) ? me : expect;
    }
    if (cur != me) return -1;
  }
  const unsigned idx = __hip_atomic_fetch_add(word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  return idx < (unsigned)total ? (int)idx : -1;
}

// The same in two halves, for a workgroup that owns the queue: the answer to a request is looked at (ticket_of) only when
// the ticket is handed on, and not where it is asked for, in front of the stores of a task, where it holds the asking
// wavefront, and at the next barrier the other three, for a round trip to the L2 (14 bf16 matrices of 1021, 341 and 2731
// rows / columns under Dion: 684 -> 674 us).  The address goes through a vector register: for a wave-uniform one the compiler
// adds up the lanes' requests, broadcasts the answer and waits for it on the spot.
constexpr unsigned DA_NO_TICKET = ~0u;
__device__ __forceinline__ unsigned request_ticket(unsigned* word) {
  typedef __attribute__((address_space(1))) unsigned global_word_t;
  unsigned off = 0;
  asm volatile("" : "+v"(off));
  return __hip_atomic_fetch_add((global_word_t*)word + off, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int ticket_of(unsigned idx, int total) { return idx < (unsigned)total ? (int)idx : -1; }

// (one thread) waits until *ctr >= want.  Bounded: after `limit` ticks of the 100 MHz counter, or when another workgroup
// has given up, *status is set and the wait ends.
__device__ __forceinline__ void wait_count(const int* ctr, int want, int* status, unsigned long long limit) {
  unsigned spins = 0;
  unsigned long long t0 = 0;
  while (__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < want) {
    // (the status word and the clock every 32nd time only: each load is a round trip to the L2)
    if ((spins++ & 31) != 31) continue;
    if (t0 == 0) t0 = now_ticks();
    if (now_ticks() - t0 > limit || __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
      __hip_atomic_store(status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      break;
    }
  }
}

}  // namespace
