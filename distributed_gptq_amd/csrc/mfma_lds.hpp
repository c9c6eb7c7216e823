// What the 4-wave MFMA kernels (the Hessian's Gram tiles, the dense product)
// share: direct-to-LDS copies, bare barriers and waits, and the MFMA as
// inline asm with the accumulators pinned to AGPRs.
#pragma once

#include "common.hpp"

namespace gptq {
namespace {

typedef __attribute__((address_space(3))) void lds_void;

// The accumulators stay in AGPRs and the fragments in VGPRs (with the builtin
// the register allocator moved accumulators through VGPRs and spilled);
// volatile keeps the MFMAs in program order with the LDS reads and copies.
template <bool kBF16>
__device__ __forceinline__ void mfma32_asm(f32x16& acc, const u32x4& a, const u32x4& b) {
  if constexpr (kBF16)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

template <bool kBF16>
__device__ __forceinline__ void mfma16_asm(f32x4& acc, const u32x4& a, const u32x4& b) {
  if constexpr (kBF16)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// The wait states between the last MFMA and a read of its result (the
// compiler does not see the asm MFMAs' results as MFMA results).
__device__ __forceinline__ void mfma_settle() { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory"); }

// A wave-uniform 64-bit value through readfirstlane, which takes and returns
// int: each half is widened as unsigned, so that a low half with bit 31 set
// does not sign-extend into the high half.
__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(v))));
  const uint32_t hi =
      static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(v >> 32))));
  return static_cast<uint64_t>(hi) << 32 | lo;
}

// One 16-byte-per-lane copy into LDS from base + voff + soff, zeros at and past nrec
// bytes.  base and nrec are wave-uniform (the descriptor stays in SGPRs).
// (Target builtins sit in a __device__ function, not in the kernel body: in
// the kernel body the host pass dropped the kernel's launch stub.)
__device__ __forceinline__ void lds_copy16(const uint16_t* base, uint32_t nrec, uint8_t* lds, uint32_t voff,
                                           int soff = 0) {
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      reinterpret_cast<uint16_t*>(uniform_u64(reinterpret_cast<uint64_t>(base))), static_cast<short>(0),
      __builtin_amdgcn_readfirstlane(static_cast<int>(nrec)), 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)lds, 16, voff, soff, 0, 0);
}

__device__ __forceinline__ void bare_barrier() { asm volatile("s_barrier" ::: "memory"); }

// s_waitcnt for "at most N vector-memory operations outstanding" (gfx9
// encoding: vmcnt bits 3:0 and 15:14; expcnt and lgkmcnt left at "no wait")
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N < 64, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// s_waitcnt for "at most N LDS / scalar-memory operations outstanding"
template <int N>
__device__ __forceinline__ void wait_lgkm() {
  static_assert(N < 16, "lgkmcnt immediate");
  __builtin_amdgcn_s_waitcnt(0xC07F | (N << 8));
}

}  // namespace
}  // namespace gptq
