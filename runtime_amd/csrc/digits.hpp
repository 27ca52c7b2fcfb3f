// Device code shared by the digit GEMMs (gemm_mx.hip, gemm_i8.hip).
//
// Number range.  The kernels' sums are true magnitudes in f32, which serves
// ordinary values.  Where a row's 128-group is so small that a factor of its
// products would be subnormal, or so large that a sum could overflow although
// the weights leave most of it out, the split kernel stores a NaN with a code in
// its payload as the factor that meets every sum of the group.  That makes the
// row's totals NaN; a block that finds one computes its tiles again, straight
// from memory, in an arithmetic for any range.  Ordinary calls pay one addition
// per total for it.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

namespace mfh {

// 16 bytes per lane, from base + offset (uniform base, the lane's byte offset)
// to the LDS bytes [lds, lds + 1024) of the wave.  The caller waits (vmcnt)
// and synchronises before the bytes are read.  (m0 is the compiler's to reserve: it
// sets it anew before each use of its own.)
__device__ __forceinline__ void copy_to_lds(const uint8_t *base, uint32_t offset, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %0\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds), "v"(offset), "s"(base)
                 : "memory");
}

// The lane, for code off the hot path: no register of the caller's stays live for
// it.
__device__ __forceinline__ uint32_t cold_lane()
{
    uint32_t lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lane));
    return lane;
}

// A NaN that stands for the group's own code (0: a non-finite value, whose row
// stays NaN; below 2^22), and the code of such a NaN.
constexpr uint32_t kNanBits = 0x7fc00000u;
__device__ __forceinline__ float nan_of(uint32_t code) { return __uint_as_float(kNanBits | code); }
__device__ __forceinline__ bool is_code(uint32_t bits)
{
    return (bits & kNanBits) == kNanBits && (bits & ~kNanBits);
}

}  // namespace mfh
