// lds_dma.hpp -- device helpers of the kernels that stage through LDS with
// buffer loads that have an LDS destination (grouped.hip, few.hip).
#pragma once
#include "int4_common.hpp"

namespace cai4 {
namespace {

typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef __attribute__((address_space(3))) void lds_void;

CAI4_DEV rsrc_t rsrc(const void *base, size_t bytes) {
  const int n = bytes > 0x7FFFFFFFu ? 0x7FFFFFFF : (int)bytes;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, n, 0x00020000);
}

// The same with the (wave-uniform) base and size forced into scalar registers.
CAI4_DEV rsrc_t rsrc_scalar(const void *base, size_t bytes) {
  const uint64_t b = (uint64_t)base;
  // (readfirstlane returns int: without the cast its sign would fill the high half)
  const uint64_t u = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32;
  const int n = __builtin_amdgcn_readfirstlane(bytes > 0x7FFFFFFFu ? 0x7FFFFFFF : (int)bytes);
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(u), (short)0, n, 0x00020000);
}

// Wait until at most n of this wave's vector-memory loads are outstanding and
// its LDS reads have returned, then barrier.  Inline asm with a memory
// clobber: neither LDS reads nor the LDS-destination loads move across it.
template <int n>
CAI4_DEV void dma_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(n) : "memory");
}

// One global -> LDS buffer load (16 or 4 bytes per lane, lane i at M0 +
// bytes * i) from byte voff + soff.  Inline asm: the compiler cannot tell the
// stage buffers apart and would make LDS reads of any stage wait for the
// newest prefetch.  A lane's row limit is in voff (soff only steps along K).
// The load reads M0 one wait state after a scalar write of it at the earliest;
// the compiler knows that rule for its own instructions and not for asm, and
// sets M0 right before: the s_nop is that wait state.
template <int bytes>
CAI4_DEV void lds_dma(rsrc_t r, uint32_t lds, uint32_t voff, uint32_t soff) {
  if constexpr (bytes == 16)
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"{m0}"(lds), "v"(voff),
                 "s"(r), "s"(soff)
                 : "memory");
  else
    asm volatile("s_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"{m0}"(lds), "v"(voff),
                 "s"(r), "s"(soff)
                 : "memory");
}

// A read of LDS at byte address at + off.  The constant off is a pointer step,
// not integer arithmetic, so that it becomes the instruction's offset.
template <class T>
CAI4_DEV T lds_at(uint32_t at, int off) {
  typedef const __attribute__((address_space(3))) uint8_t *bytes_t;
  return *reinterpret_cast<const __attribute__((address_space(3))) T *>(
      reinterpret_cast<bytes_t>(at) + off);
}

constexpr uint32_t kDmaOOB = 0x80000000u;  // an offset past every range: no data moves

}  // namespace
}  // namespace cai4
