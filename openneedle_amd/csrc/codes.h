// Code-dword decoding shared by the FP32 GEMV kernels.
#pragma once

#include "common.h"

namespace nd {

// (x byte BYTE) & mask, one SDWA op; mask lives in an SGPR.
template <int BYTE>
__device__ __forceinline__ uint32_t and_byte(uint32_t mask, uint32_t x) {
    uint32_t r;
    if constexpr (BYTE == 0)
        asm("v_and_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_0"
            : "=v"(r) : "s"(mask), "v"(x));
    else if constexpr (BYTE == 1)
        asm("v_and_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_1"
            : "=v"(r) : "s"(mask), "v"(x));
    else if constexpr (BYTE == 2)
        asm("v_and_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_2"
            : "=v"(r) : "s"(mask), "v"(x));
    else
        asm("v_and_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_3"
            : "=v"(r) : "s"(mask), "v"(x));
    return r;
}

// Byte offsets of the 8 table entries addressed by one code dword, in code
// order: off[2m] from nibble 2m, off[2m+1] from nibble 2m+1.
template <int KIND>
__device__ __forceinline__ void slot_offsets_sdwa(uint32_t wd, uint32_t mask, uint32_t off[8]) {
    constexpr int kRot = KIND == kNib ? 2 : 3;                      // log2(entry bytes)
    const uint32_t X = __builtin_amdgcn_alignbit(wd, wd, 32 - kRot);  // rotate left: even nibbles
    const uint32_t Y = __builtin_amdgcn_alignbit(wd, wd, 4 - kRot);   // rotate right: odd nibbles
    off[0] = and_byte<0>(mask, X);
    off[1] = and_byte<0>(mask, Y);
    off[2] = and_byte<1>(mask, X);
    off[3] = and_byte<1>(mask, Y);
    off[4] = and_byte<2>(mask, X);
    off[5] = and_byte<2>(mask, Y);
    off[6] = and_byte<3>(mask, X);
    off[7] = and_byte<3>(mask, Y);
}

}  // namespace nd
