// Shared by the prefill and the decode kernels: loads from global memory straight into LDS (no staging registers)
// and exchanges between the lanes of a wavefront.
#ifndef FP_PREFILL_COMMON_H
#define FP_PREFILL_COMMON_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fp {

// 16 bytes per lane from global memory to LDS at `lds` + lane * 16 (`lds` wavefront-uniform).
// Written as inline assembly on purpose: while the compiler knows of such a load in flight it turns
// every wait for an LDS read into a wait for all of them, which serialises the operand reads of a
// main loop against its MFMAs.  The code that issues these loads waits for them itself (vmcnt(0)
// before the barrier that publishes a tile).  Nothing else in these kernels uses M0.
__device__ __forceinline__ void load_to_lds(const char* src, char* lds) {
  const uint32_t base = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds)));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(base), "v"(src) : "memory");
}

// The same with the address split into a wavefront-uniform base (scalar registers) and a 32-bit offset per lane.
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t offset, char* lds) {
  const uint32_t m0v = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds)));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(m0v), "v"(offset), "s"(base) : "memory");
}

// Both forms with the place in LDS as a number in two parts, a wavefront's own and a constant (lds_address of an array, plus bytes): a pointer
// that a loop keeps is 64 bits of scalar registers and a test for null at every load, and a sum for every load of a loop a register each.
__device__ __forceinline__ uint32_t lds_address(const char* array) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)array));
}
__device__ __forceinline__ void load_to_lds(const char* src, uint32_t own, uint32_t constant) {
  asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off"
               : : "s"(own), "s"(constant), "v"(src) : "memory", "scc");
}
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t offset, uint32_t own, uint32_t constant) {
  asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
               : : "s"(own), "s"(constant), "v"(offset), "s"(base) : "memory", "scc");
}

// Both forms for rows that are read once (non-temporal, so that they do not displace what the caches hold).
__device__ __forceinline__ void load_to_lds_nt(const char* src, char* lds) {
  const uint32_t base = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds)));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" : : "s"(base), "v"(src) : "memory");
}
__device__ __forceinline__ void load_to_lds_nt(const char* base, uint32_t offset, char* lds) {
  const uint32_t m0v = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds)));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" : : "s"(m0v), "v"(offset), "s"(base) : "memory");
}

// v_permlane32_swap exchanges the upper half of its first operand with the lower half of its second.  Of one value twice, both
// operands hold both halves' values afterwards, in every lane; of two values, the sum of the operands is the first value's total in the
// lower half and the second's in the upper.  No trip through LDS as a shuffle takes it.  (Inline assembly: the compiler's builtin returned
// the first operand for both.  The no-ops are the wait states between a vector write, the swap and the next vector read.)
__device__ __forceinline__ void swap_lane_halves(float& a, float& b) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
// max(x of lane l, x of lane l ^ 32) in both lanes
__device__ __forceinline__ float max_across_lane_halves(float x) {
  float y = x;
  swap_lane_halves(x, y);
  return fmaxf(x, y);
}

// Largest x of the wavefront, in scalar registers: lane exchanges inside rows of 16, then one lane of each, no trip through LDS.
__device__ __forceinline__ int wave_max(int x) {
  x = max(x, __builtin_amdgcn_update_dpp(x, x, 0xB1, 0xf, 0xf, true));   // quad_perm [1,0,3,2]
  x = max(x, __builtin_amdgcn_update_dpp(x, x, 0x4E, 0xf, 0xf, true));   // quad_perm [2,3,0,1]
  x = max(x, __builtin_amdgcn_update_dpp(x, x, 0x141, 0xf, 0xf, true));  // row_half_mirror
  x = max(x, __builtin_amdgcn_update_dpp(x, x, 0x140, 0xf, 0xf, true));  // row_mirror
  return max(max(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
             max(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}

}  // namespace fp
#endif
