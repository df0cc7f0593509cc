// Sums and exchanges between the lanes of a wave without LDS instructions (gfx950: 64 lanes, rows of 16).
#pragma once

#include <hip/hip_runtime.h>

namespace nuto_amd
{

// DPP control words: exchanges within a quad, rotations within a row of 16 lanes
constexpr int kDppXor1 = 0xB1;   // quad_perm [1, 0, 3, 2]
constexpr int kDppXor2 = 0x4E;   // quad_perm [2, 3, 0, 1]
constexpr int kDppRor4 = 0x124;  // row_ror:4
constexpr int kDppRor8 = 0x128;  // row_ror:8

// v of the lane that the DPP control word selects
template <int CTRL>
__device__ inline double LaneDpp(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// v + v of lane ^ 16 / lane ^ 32, the lower row's (half's) value first: v_permlane{16,32}_swap of a
// register with itself leaves the even rows' (lower half's) values in one result and the odd rows' in
// the other
__device__ inline double AddXor16(double v)
{
    const long long b = __double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)b, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
    return __longlong_as_double(((long long)hi[0] << 32) | lo[0]) + __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}
__device__ inline double AddXor32(double v)
{
    const long long b = __double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)b, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
    return __longlong_as_double(((long long)hi[0] << 32) | lo[0]) + __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}

// v summed over the 16 lanes of the wave with the same lane & 3, known to each of them
__device__ inline double QuadLaneSum(double v)
{
    v += LaneDpp<kDppRor8>(v);
    v += LaneDpp<kDppRor4>(v);
    return AddXor32(AddXor16(v));
}

// v summed over the 64 lanes, known to every lane
__device__ inline double WaveSum(double v)
{
    v += LaneDpp<kDppXor1>(v);
    v += LaneDpp<kDppXor2>(v);
    return QuadLaneSum(v);
}

}  // namespace nuto_amd
