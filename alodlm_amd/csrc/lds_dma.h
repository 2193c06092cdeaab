// Direct global->LDS loads (global_load_lds_dword[x4]) issued from inline
// assembly.
//
// Lane i of one instruction writes the i-th slot (4 or 16 bytes) after the
// LDS base held in M0.  The compiler is not told about these loads: left to
// itself it cannot prove that later transposed LDS reads
// (ds_read_b64_tr_b16) do not alias the pending writes, and it then waits for
// every outstanding load (vmcnt(0)) before each such read, which cancels any
// prefetch.  Kernels using these helpers therefore wait for their own loads
// explicitly (s_waitcnt vmcnt(n) before the barrier that publishes a tile).
// Loads the compiler does not count only make its own vmcnt waits more
// conservative, never less.  M0 is saved and restored around each global load;
// the buffer loads name it as an input.
#pragma once

#include <stdint.h>

#define ALODLM_LDS_AS __attribute__((address_space(3)))

// LDS byte address of a pointer into a __shared__ array, made wave-uniform.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(ALODLM_LDS_AS const void*)p);
}

// 16 bytes per lane from the per-lane address g.
__device__ __forceinline__ void dma16_v(const void* g, uint32_t lds) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %2\n\t"
      "global_load_lds_dwordx4 %1, off\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(g), "s"(lds)
      : "memory");
}

// 16 bytes per lane from the wave-uniform base plus the lane's 32-bit offset.
__device__ __forceinline__ void dma16_s(const void* base, uint32_t off, uint32_t lds) {
  uint32_t saved;
  const uint64_t b = (uint64_t)(uintptr_t)base;
  // readfirstlane returns int: go through uint32_t so the low word is
  // zero-extended, never sign-extended into the high word
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  const uint64_t ub = ((uint64_t)hi << 32) | (uint64_t)lo;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "global_load_lds_dwordx4 %1, %2\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(off), "s"(ub), "s"(lds)
      : "memory");
}

// dma16_s for data read once: non-temporal (streamed past the caches' normal
// retention), so it does not evict operands that other workgroups re-read.
__device__ __forceinline__ void dma16_s_nt(const void* base, uint32_t off, uint32_t lds) {
  uint32_t saved;
  const uint64_t b = (uint64_t)(uintptr_t)base;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  const uint64_t ub = ((uint64_t)hi << 32) | (uint64_t)lo;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "global_load_lds_dwordx4 %1, %2 nt\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(off), "s"(ub), "s"(lds)
      : "memory");
}

// 4 bytes per lane from the per-lane address g.
__device__ __forceinline__ void dma4_v(const void* g, uint32_t lds) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %2\n\t"
      "global_load_lds_dword %1, off\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(g), "s"(lds)
      : "memory");
}

// A buffer of `bytes` bytes at p (wave-uniform) for the loads below, whose range
// check returns zeros past its end.
typedef int v4i_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4i_t buffer_of(const void* p, int64_t bytes) {
  const uint64_t b = (uint64_t)(uintptr_t)p;
  v4i_t r;
  r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  r.y = __builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
  r.z = __builtin_amdgcn_readfirstlane((int)(uint32_t)bytes);
  r.w = 0x00020000;
  return r;
}

// 16 (4) bytes per lane from the buffer's byte voff (+ soff) into the lane's slot
// after the LDS byte address m0v.
__device__ __forceinline__ void dma16_buf(v4i_t rsrc, uint32_t voff, uint32_t soff, uint32_t m0v) {
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds"
               ::"v"(voff), "s"(rsrc), "s"(soff), "{m0}"(m0v) : "memory");
}
__device__ __forceinline__ void dma16_buf(v4i_t rsrc, uint32_t voff, uint32_t m0v) {
  asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(rsrc), "{m0}"(m0v) : "memory");
}
__device__ __forceinline__ void dma4_buf(v4i_t rsrc, uint32_t voff, uint32_t m0v) {
  asm volatile("buffer_load_dword %0, %1, 0 offen lds" ::"v"(voff), "s"(rsrc), "{m0}"(m0v) : "memory");
}
