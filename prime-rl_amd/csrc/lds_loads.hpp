// Global -> LDS loads, counted waits, counted stores and MFMA shapes shared by the GEMM kernels that stage through LDS (dense,
// split reduction, narrow, deep, wide and ring tiles).
#pragma once

#include "common.hpp"

namespace moe_i8 {

constexpr int kStepBytes = 128;  // reduction bytes of a row fetched and multiplied at a time

// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding: vmcnt = bits 3:0 and
// 15:14; expcnt 6:4 and lgkmcnt 11:8 left at their maximum).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

// Waits until at most n * kPer of this wavefront's vector-memory operations are pending, n <= kMost.
template <int kPer, int kMost>
__device__ __forceinline__ void wait_groups(int n) {
  if constexpr (kMost == 0) {
    wait_vmcnt<0>();
  } else {
    if (n >= kMost)
      wait_vmcnt<kPer * kMost>();
    else
      wait_groups<kPer, kMost - 1>(n);
  }
}

__device__ __forceinline__ uint64_t uniform_address(const void* base) {
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  // readfirstlane yields a signed int: go through uint32_t so that the low half is not sign-extended
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
  return (uint64_t)lo | ((uint64_t)hi << 32);
}

// 16 bytes per lane from global memory straight into LDS: lane i lands at lds_addr + 16 * i
// (lds_addr is wave-uniform and goes through M0).  The source is a wave-uniform base plus an unsigned
// 32-bit byte offset per lane.  Inline assembly, so that the waits are the explicit counted ones.
__device__ __forceinline__ void load_to_lds_16(const void* base, uint32_t offset, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"((uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(offset), "s"(uniform_address(base))
               : "memory", "m0");
}
// The same with the non-temporal hint, for rows that nothing else reads.
__device__ __forceinline__ void load_to_lds_16_stream(const void* base, uint32_t offset, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
               :
               : "s"((uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(offset), "s"(uniform_address(base))
               : "memory", "m0");
}
// 4 bytes per lane from any address of the lane's own
__device__ __forceinline__ void load_to_lds_4(const void* addr, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
               :
               : "s"((uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(reinterpret_cast<uint64_t>(addr))
               : "memory", "m0");
}
// A store through to memory by those of the active lanes that are in `lanes`, issued even if that is none of them, so that the
// waits can count it (where the branches around it are the same for all lanes: a branch that no lane takes is jumped over as
// a whole).  The lanes that were active before are active again afterwards.  (The two wait states behind it: a store of more
// than 8 bytes reads its data that late, and the compiler, which keeps a write of them away from its own stores, does not know
// of this one.)
__device__ __forceinline__ void store16_through(void* to, const uint4& v, uint64_t lanes) {
  uint64_t active;
  lanes = uniform_address(reinterpret_cast<const void*>(lanes));
  asm volatile("s_and_saveexec_b64 %0, %3\n\tglobal_store_dwordx4 %1, %2, off sc1\n\ts_mov_b64 exec, %0\n\ts_nop 1"
               : "=&s"(active)
               : "v"(reinterpret_cast<uint64_t>(to)), "v"(v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w}), "s"(lanes)
               : "memory", "scc");
}
// The same into the caches, or past them with the non-temporal hint.
template <bool NT>
__device__ __forceinline__ void store16_lanes(void* to, const uint4& v, uint64_t lanes) {
  uint64_t active;
  lanes = uniform_address(reinterpret_cast<const void*>(lanes));
  const v4i x{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
  if constexpr (NT)
    asm volatile("s_and_saveexec_b64 %0, %3\n\tglobal_store_dwordx4 %1, %2, off nt\n\ts_mov_b64 exec, %0\n\ts_nop 1"
                 : "=&s"(active) : "v"(reinterpret_cast<uint64_t>(to)), "v"(x), "s"(lanes) : "memory", "scc");
  else
    asm volatile("s_and_saveexec_b64 %0, %3\n\tglobal_store_dwordx4 %1, %2, off\n\ts_mov_b64 exec, %0\n\ts_nop 1"
                 : "=&s"(active) : "v"(reinterpret_cast<uint64_t>(to)), "v"(x), "s"(lanes) : "memory", "scc");
}
// through: written through to memory instead of left in the L2.  (The two wait states behind that store: a store of more than
// 8 bytes reads its data that late, and the compiler, which keeps a write of them away from its own stores, does not know of
// this one.)
__device__ __forceinline__ void store16(void* to, const v4i& v, bool through) {
  if (through)
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" :: "v"(reinterpret_cast<uint64_t>(to)), "v"(v) : "memory");
  else
    *reinterpret_cast<v4i*>(to) = v;
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)((const __attribute__((address_space(3))) char*)p);
}

// A row of a stage is eight 16-byte chunks; chunk c of row r sits at position c ^ swizzle_of_row(r), so that
// the operand reads (many rows, one chunk) spread over all banks.
__device__ __forceinline__ int swizzle_of_row(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// v_mfma_i32_32x32x32_i8 and v_mfma_i32_16x16x64_i8.  Operand lane l: row l % MF, chunk l / MF of the
// instruction's reduction bytes; result lane l: column l % MF, rows 4 * (l / MF) + r (+ 8 * q for 32).
template <int MF>
struct Mfma;
template <>
struct Mfma<32> {
  typedef v16i Acc;
  static constexpr int kRegs = 16;
  static constexpr int kSub = 4;  // MFMAs per 128 reduction bytes
  static __device__ __forceinline__ Acc mul(v4i a, v4i b, Acc c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }
};
template <>
struct Mfma<16> {
  typedef v4i Acc;
  static constexpr int kRegs = 4;
  static constexpr int kSub = 2;
  static __device__ __forceinline__ Acc mul(v4i a, v4i b, Acc c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0); }
};

}  // namespace moe_i8
