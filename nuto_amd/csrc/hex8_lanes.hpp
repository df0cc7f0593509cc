// Hex8 cells on groups of 8 lanes with the trilinear interpolation done axis by axis.
//
// Lane m of a group stands for one corner of the reference cube: for the node there and for the 2x2x2
// Gauss point next to it. Between a node value and an integration point value lie three one-dimensional
// steps, each a weighted sum with the lane across one axis: 6 exchanges per component for the value and
// the three reference derivatives at every point, 8 or 9 for the transposed sums, against 8 exchanges
// and 32 products when every lane adds the 8 nodes itself. The corners are numbered so that each
// exchange is one DPP operand (no LDS): across x lane ^ 1, across y lane ^ 2, across z lane ^ 7.
//
// The linear shape functions at the two Gauss points of an axis are near = (1 + g) / 2 and far = (1 - g) / 2
// (g = sqrt(1/3)), the derivatives +-1/2. The functions leave the common factors to the caller: a step is
// v + (far / near) v', one fused operation, and a derivative a signed difference, so a value comes out
// divided by kValueScale = near^3 and a derivative by kGradScale = near^2 / 2. The caller puts the factors
// into a coefficient that it multiplies with anyway.
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
    double sx, sy, sz;  // sides of the corner: +-1 per axis
};

__device__ inline CornerLane CornerOf(int lane)
{
    const int z = (lane >> 2) & 1, x = (lane & 1) ^ z, y = ((lane >> 1) & 1) ^ z;
    CornerLane c;
    c.node = 4 * z + (y ? 3 - x : x);
    c.ip = x + 2 * y + 4 * z;
    c.sx = x ? 1.0 : -1.0;
    c.sy = y ? 1.0 : -1.0;
    c.sz = z ? 1.0 : -1.0;
    return c;
}

constexpr double kNear = 0.5 * (1.0 + 0.57735026918962573);
constexpr double kFarNear = 0.26794919243112271;  // far / near = 2 - sqrt(3)
constexpr double kValueScale = kNear * kNear * kNear;
constexpr double kGradScale = 0.5 * kNear * kNear;

// v / near of the step across the axis of the exchange
template <int CTRL>
__device__ inline double Across(double v)
{
    return fma(kFarNear, LaneDpp<CTRL>(v), v);
}

// reference gradient / kGradScale at this lane's integration point of the field with node values v
__device__ inline void NodesToPoint(const CornerLane& c, double v, double grad[3])
{
    const double vx = LaneDpp<kDppXor1>(v);
    const double a = fma(kFarNear, vx, v), dx = c.sx * (v - vx);
    const double ay = LaneDpp<kDppXor2>(a);
    const double b = fma(kFarNear, ay, a), dy = c.sy * (a - ay);
    grad[0] = Across<kDppXor7>(Across<kDppXor2>(dx));
    grad[1] = Across<kDppXor7>(dy);
    grad[2] = c.sz * (b - LaneDpp<kDppXor7>(b));
}

// value / kValueScale at this lane's integration point
__device__ inline double NodesToValue(double v)
{
    return Across<kDppXor7>(Across<kDppXor2>(Across<kDppXor1>(v)));
}

// sum over the 8 integration points of g . dN/dxi + q N of this lane's node, for g kGradScale and q kValueScale
// given
template <bool VALUE>
__device__ inline double PointsToNode(const CornerLane& c, const double g[3], double q)
{
    const double z = g[2] + LaneDpp<kDppXor7>(g[2]);
    double w = VALUE ? fma(c.sz, z, Across<kDppXor7>(q)) : c.sz * z;
    const double x = Across<kDppXor2>(Across<kDppXor7>(g[0]));
    const double y = Across<kDppXor7>(g[1]);
    w = fma(c.sy, y + LaneDpp<kDppXor2>(y), Across<kDppXor2>(w));
    return fma(c.sx, x + LaneDpp<kDppXor1>(x), Across<kDppXor1>(w));
}

// sum over the 8 integration points of q N of this lane's node, for q kValueScale given
__device__ inline double ValuesToNode(double q)
{
    return Across<kDppXor1>(Across<kDppXor2>(Across<kDppXor7>(q)));
}

// sums over the 8 integration points of h dN/dxi_k of this lane's node, k = 0, 1, 2, for h kGradScale given
__device__ inline void ValuesToGradients(const CornerLane& c, double h, double d[3])
{
    const double hz = LaneDpp<kDppXor7>(h);
    const double z = fma(kFarNear, hz, h), zs = h + hz;
    const double zy = LaneDpp<kDppXor2>(z);
    const double y = fma(kFarNear, zy, z), ys = z + zy, yz = Across<kDppXor2>(zs);
    d[0] = c.sx * (y + LaneDpp<kDppXor1>(y));
    d[1] = c.sy * Across<kDppXor1>(ys);
    d[2] = c.sz * Across<kDppXor1>(yz);
}

// sum_n N_n v[n] at this lane's integration point, the nodes in local order, each N_n the product
// ((1/8 f_0) f_1) f_2: bit for bit the sum over the nodes of the shape tables. `v`: the cell's 8 node values
// (LDS). For the nonlocal strain, whose comparison with the history must come out alike in every kernel.
__device__ inline double NodeSum(const CornerLane& c, const double* v)
{
    const double near = 1.0 + 0.57735026918962573, far = 1.0 - 0.57735026918962573;
    const double fx[2] = {c.sx < 0.0 ? near : far, c.sx < 0.0 ? far : near};
    const double fy[2] = {c.sy < 0.0 ? near : far, c.sy < 0.0 ? far : near};
    const double fz[2] = {c.sz < 0.0 ? near : far, c.sz < 0.0 ? far : near};
    double s = 0.0;
#pragma unroll
    for (int n = 0; n < 8; n++)
        s = fma(0.125 * fx[((n + 1) >> 1) & 1] * fy[(n >> 1) & 1] * fz[n >> 2], v[n], s);
    return s;
}

// v summed over the 8 lanes of the group, known to each of them
__device__ inline double CornerSum(double v)
{
    v += LaneDpp<kDppXor1>(v);
    v += LaneDpp<kDppXor2>(v);
    return v + LaneDpp<kDppXor7>(v);
}

}  // namespace nuto_amd
