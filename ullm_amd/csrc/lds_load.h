// Loads that write shared memory themselves, and the waits and the barrier that go with them.  The loads are issued in
// inline assembly: the compiler, which cannot tell which of such loads a read of shared memory depends on, would
// otherwise wait for all of them before every read.  The waits stand in the code, by count (a wave's loads complete in
// order).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// 16 bytes per lane from `src` to shared memory at lds_base + 16 * lane (lds_base the same in the whole wave).
// The instruction takes the place in shared memory from M0, which the compiler keeps for itself and warns
// about; nothing else in kernels that call this uses it.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load16_to_lds(const void* src, unsigned char* lds_base) {
#ifdef __HIP_DEVICE_COMPILE__
  typedef __attribute__((address_space(3))) unsigned char lds_byte_t;
  const unsigned at = (unsigned)__builtin_amdgcn_readfirstlane((int)(uintptr_t)(lds_byte_t*)lds_base);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(at) : "memory", "m0");
#else
  __builtin_amdgcn_global_load_lds(src, lds_base, 16, 0, 0);
#endif
}
// The same for what is read once and need not stay in the caches.
__device__ __forceinline__ void load16_to_lds_once(const void* src, unsigned char* lds_base) {
#ifdef __HIP_DEVICE_COMPILE__
  typedef __attribute__((address_space(3))) unsigned char lds_byte_t;
  const unsigned at = (unsigned)__builtin_amdgcn_readfirstlane((int)(uintptr_t)(lds_byte_t*)lds_base);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" : : "v"(src), "s"(at) : "memory", "m0");
#endif
}
// The same from base + off bytes (base the same in the whole wave), to the place `at` of shared memory (lds_place).
__device__ __forceinline__ void load16_to_lds_from(const void* base, unsigned off, unsigned at) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(at) : "memory", "m0");
#endif
}
// The same for what is read once and need not stay in the caches.
__device__ __forceinline__ void load16_to_lds_from_once(const void* base, unsigned off, unsigned at) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" : : "v"(off), "s"(base), "s"(at) : "memory", "m0");
#endif
}
#pragma clang diagnostic pop
__device__ __forceinline__ unsigned lds_place(unsigned char* p) {
#ifdef __HIP_DEVICE_COMPILE__
  typedef __attribute__((address_space(3))) unsigned char lds_byte_t;
  return (unsigned)__builtin_amdgcn_readfirstlane((int)(uintptr_t)(lds_byte_t*)p);
#else
  return 0;
#endif
}
// at most N of this wave's loads are still on their way
template <int N>
__device__ __forceinline__ void loads_left() {
  static_assert(N >= 0 && N < 64, "the counter has six bits");
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
#endif
}
// This wave's reads of shared memory have returned.
__device__ __forceinline__ void reads_done() {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
#endif
}
// Every wave of the block has read what it read of shared memory before this and may write it from here on; loads on
// their way stay on their way.
__device__ __forceinline__ void bare_barrier() {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
#endif
}
