// Hex8 cells on groups of 8 lanes with the trilinear interpolation done axis by axis.
//
// Lane m of a group stands for one corner of the reference cube: for the node there and for the 2x2x2
// Gauss point next to it. Between a node value and an integration point value lie three one-dimensional
// steps, each a weighted sum with the lane across one axis: 6 exchanges per component for the value and
// the three reference derivatives at every point, 8 or 9 for the transposed sums, against 8 exchanges
// and 32 products when every lane adds the 8 nodes itself. The corners are numbered so that each
// exchange is one DPP operand (no LDS): across x lane ^ 1, across y lane ^ 2, across z lane ^ 7.
#pragma once

#include <hip/hip_runtime.h>

#include "lanes.hpp"

namespace nuto_amd
{

constexpr int kDppXor7 = 0x141;  // row_half_mirror

struct CornerLane
{
    int node;           // local node of this lane (InterpolationBrickLinear.cpp:37-52 order)
    int ip;             // integration point next to it (xi fastest)
    double hx, hy, hz;  // derivative of the linear function that is 1 at this corner: +-1/2 per axis
};

__device__ inline CornerLane CornerOf(int lane)
{
    const int z = (lane >> 2) & 1, x = (lane & 1) ^ z, y = ((lane >> 1) & 1) ^ z;
    CornerLane c;
    c.node = 4 * z + (y ? 3 - x : x);
    c.ip = x + 2 * y + 4 * z;
    c.hx = x ? 0.5 : -0.5;
    c.hy = y ? 0.5 : -0.5;
    c.hz = z ? 0.5 : -0.5;
    return c;
}

constexpr double kNear = 0.5 * (1.0 + 0.57735026918962573);  // linear shape values at the Gauss points
constexpr double kFar = 0.5 * (1.0 - 0.57735026918962573);

template <int CTRL>
__device__ inline double Across(double v)
{
    return fma(kFar, LaneDpp<CTRL>(v), kNear * v);
}

// value and reference gradient at this lane's integration point of the field with node values v
__device__ inline void NodesToPoint(const CornerLane& c, double v, double& value, double grad[3])
{
    const double vx = LaneDpp<kDppXor1>(v);
    const double a = fma(kFar, vx, kNear * v), dx = c.hx * (v - vx);
    const double ay = LaneDpp<kDppXor2>(a);
    const double b = fma(kFar, ay, kNear * a), dy = c.hy * (a - ay);
    const double bz = LaneDpp<kDppXor7>(b);
    value = fma(kFar, bz, kNear * b);
    grad[0] = Across<kDppXor7>(Across<kDppXor2>(dx));
    grad[1] = Across<kDppXor7>(dy);
    grad[2] = c.hz * (b - bz);
}

// sum over the 8 integration points of g . dN/dxi + q N of this lane's node
template <bool VALUE>
__device__ inline double PointsToNode(const CornerLane& c, const double g[3], double q)
{
    double w = c.hz * (g[2] + LaneDpp<kDppXor7>(g[2]));
    if (VALUE)
        w += Across<kDppXor7>(q);
    const double x = Across<kDppXor2>(Across<kDppXor7>(g[0]));
    const double y = Across<kDppXor7>(g[1]);
    w = fma(c.hy, y + LaneDpp<kDppXor2>(y), Across<kDppXor2>(w));
    return fma(c.hx, x + LaneDpp<kDppXor1>(x), Across<kDppXor1>(w));
}

// v summed over the 8 lanes of the group, known to each of them
__device__ inline double CornerSum(double v)
{
    v += LaneDpp<kDppXor1>(v);
    v += LaneDpp<kDppXor2>(v);
    return v + LaneDpp<kDppXor7>(v);
}

}  // namespace nuto_amd
