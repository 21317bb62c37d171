// SPDX-License-Identifier: MIT
// Lane exchanges inside a wavefront as operand modifiers (DPP): the
// instruction that uses one takes no extra step, where __shfl goes through
// the LDS pipe (ds_bpermute).  Every lane that is read must be active.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pmh {

enum : int { kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140, kDppRowShr = 0x110,
             kDppRowRor = 0x120, kDppRowBcast15 = 0x142, kDppRowBcast31 = 0x143, kDppNewBcast = 0x150 };
template <int kCtrl>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x) {
    return uint32_t(__builtin_amdgcn_update_dpp(0, int(x), kCtrl, 0xf, 0xf, true));
}
template <int kCtrl>
__device__ __forceinline__ float dpp_f32(float x) { return __uint_as_float(dpp_u32<kCtrl>(__float_as_uint(x))); }
// The value of lane kLane of each 16-lane row.
template <int kLane>
__device__ __forceinline__ float row_bcast(float x) { return dpp_f32<kDppNewBcast + kLane>(x); }

}  // namespace pmh
