// Copies from memory straight into LDS (no registers on the way), asked for ahead and waited for by count.
//
// A wave's copy brings 64 pieces of 16 bytes: lane l's piece comes from byte `from + scalar` of the buffer, `from` the
// lane's own and `scalar` the wave's, and goes to LDS byte `to` + 16 l.  A lane whose offset lies at or beyond the
// buffer's end brings zeros, which is how rows, columns and k-blocks that do not exist are filled in: COPY_NOTHING is
// beyond the end of every buffer made here.
//
// The copy is written as an instruction because the compiler, which cannot tell a ring's slots apart, would wait for
// every copy in flight before any LDS read.  It has no output register, so nothing can be overwritten by one in
// flight; its two waits (for M0) stand in the same block.  What the compiler counts for its own loads stays right: copies
// it does not know of only make its waits longer.  Who uses this waits with `copies_arrived` and a barrier before a
// slot is read, and lets no wave write a slot that another may still read.  No wave ends, or uses the ring's LDS for
// something else, with copies of its own in flight: what was asked for last is waited for with copies_arrived<0>, also
// where nobody wants it.
#pragma once
#include "common.h"

typedef int i32x4_t __attribute__((ext_vector_type(4)));
#define COPY_NOTHING 0xfffffff0u

// A buffer of `bytes` bytes (4 GB less a few at most: fits_copy_buffer).
__device__ __forceinline__ i32x4_t copy_buffer(const void* base, size_t bytes) {
  const uint64_t a = (uint64_t)base;
  return i32x4_t{(int)(uint32_t)a, (int)(uint32_t)((a >> 32) & 0xffffu), (int)(uint32_t)bytes, BUFFER_WORD3};
}
static inline bool fits_copy_buffer(size_t bytes) { return bytes <= (size_t)COPY_NOTHING; }

__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}

__device__ __forceinline__ void copy16_to_lds(i32x4_t buffer, uint32_t from, uint32_t scalar, uint32_t to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(to), "v"(from), "s"(buffer), "s"(scalar)
               : "memory", "m0");
}

// Two copies of neighbouring kilobytes: the second one's bytes come from `from1` + 1024 and go to `to` + 1024 (the
// instruction's offset counts on both sides).  The five states waited for are those between a vector instruction that
// writes a scalar register and a memory instruction that reads it: the buffer may come straight from v_readfirstlane.
__device__ __forceinline__ void copy_pair_to_lds(i32x4_t buffer, uint32_t from0, uint32_t from1, uint32_t to) {
  asm volatile(
      "s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %3, 0 offen lds\n\tbuffer_load_dwordx4 %2, %3, 0 offen offset:1024 lds"
      :
      : "s"(to), "v"(from0), "v"(from1), "s"(buffer)
      : "memory", "m0");
}

// Every copy of this wave but the newest N has arrived, and its LDS reads are done: with a barrier behind it, what all
// waves copied can be read, and what all waves have read may be written.
template <int N>
__device__ __forceinline__ void copies_arrived() {
  static_assert(N >= 0 && N < 64, "the counter holds six bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void ring_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
