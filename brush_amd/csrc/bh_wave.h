// bh_wave.h — wave64 scans over DPP lane moves.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace bh {

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROW_MASK, 0xF, true);
}

// The value of lane K of the lane's quad (lanes 4 q .. 4 q + 3), or of its
// neighbour at distance 1 or 2 in the quad.
template <int K>
__device__ __forceinline__ uint32_t quad_u32(uint32_t x) {
    return dpp_u32<K * 0x55, 0xF>(x);
}
template <int K>
__device__ __forceinline__ float quad_f32(float x) {
    return __uint_as_float(quad_u32<K>(__float_as_uint(x)));
}
__device__ __forceinline__ uint32_t quad_xor1_u32(uint32_t x) { return dpp_u32<0xB1, 0xF>(x); }
__device__ __forceinline__ uint32_t quad_xor2_u32(uint32_t x) { return dpp_u32<0x4E, 0xF>(x); }

// x for the quad's lane 0, y, z and w for lanes 1, 2 and 3.
__device__ __forceinline__ float quad_pick(float x, float y, float z, float w) {
    x = __builtin_amdgcn_inverse_ballot_w64(0x2222222222222222ull) ? y : x;
    x = __builtin_amdgcn_inverse_ballot_w64(0x4444444444444444ull) ? z : x;
    return __builtin_amdgcn_inverse_ballot_w64(0x8888888888888888ull) ? w : x;
}

// Inclusive wave64 scans: shifts within 16-lane rows, then row broadcasts of
// lanes 15 and 31 into the following rows.
__device__ __forceinline__ uint32_t wave_incl_add_u32(uint32_t x) {
    x += dpp_u32<0x111, 0xF>(x);  // row_shr:1
    x += dpp_u32<0x112, 0xF>(x);  // row_shr:2
    x += dpp_u32<0x114, 0xF>(x);  // row_shr:4
    x += dpp_u32<0x118, 0xF>(x);  // row_shr:8
    x += dpp_u32<0x142, 0xA>(x);  // row_bcast:15 into rows 1 and 3
    x += dpp_u32<0x143, 0xC>(x);  // row_bcast:31 into rows 2 and 3
    return x;
}
__device__ __forceinline__ uint32_t wave_incl_max_u32(uint32_t x) {
    x = max(x, dpp_u32<0x111, 0xF>(x));
    x = max(x, dpp_u32<0x112, 0xF>(x));
    x = max(x, dpp_u32<0x114, 0xF>(x));
    x = max(x, dpp_u32<0x118, 0xF>(x));
    x = max(x, dpp_u32<0x142, 0xA>(x));
    x = max(x, dpp_u32<0x143, 0xC>(x));
    return x;
}

// The or of x over the wave, in every lane (a scalar).
__device__ __forceinline__ uint32_t wave_or_u32(uint32_t x) {
    x |= dpp_u32<0x111, 0xF>(x);
    x |= dpp_u32<0x112, 0xF>(x);
    x |= dpp_u32<0x114, 0xF>(x);
    x |= dpp_u32<0x118, 0xF>(x);
    x |= dpp_u32<0x142, 0xA>(x);
    x |= dpp_u32<0x143, 0xC>(x);
    return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

}  // namespace bh
