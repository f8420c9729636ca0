// Device helpers that the convolutions share: the reduction of a wave's
// largest magnitude and its report for the next layer.
#pragma once
#include "azh_conv_iface.hpp"

#include <hip/hip_runtime.h>

namespace azh {

namespace {

// The largest of a wave's values, in every lane (as a scalar): a DPP
// reduction to lane 63.
__device__ __forceinline__ unsigned waveMax(unsigned v) {
#define AZH_DPP_MAX(CTRL, ROWS) v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false))
    AZH_DPP_MAX(0x111, 0xf);   // row_shr:1
    AZH_DPP_MAX(0x112, 0xf);   // row_shr:2
    AZH_DPP_MAX(0x114, 0xf);   // row_shr:4
    AZH_DPP_MAX(0x118, 0xf);   // row_shr:8
    AZH_DPP_MAX(0x142, 0xa);   // row_bcast:15 into rows 1 and 3
    AZH_DPP_MAX(0x143, 0xc);   // row_bcast:31 into rows 2 and 3
#undef AZH_DPP_MAX
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// The byte (BoardScales) of a largest magnitude (bits): its biased exponent,
// at least 1 for anything but zero.
__device__ __forceinline__ unsigned scaleByte(unsigned top) { return top ? max(top >> 23, 1u) : 0u; }

// Writes the wave's byte for board b (BoardScales) of its lanes' largest
// magnitude, top (bits).
__device__ __forceinline__ void reportScale(const BoardScales& s, unsigned top, int b, int part) {
    top = waveMax(top);
    if (s.out && (threadIdx.x & 63) == 0) s.out[(size_t)b * s.stride + part] = (uint8_t)scaleByte(top);
}

} // namespace

} // namespace azh
