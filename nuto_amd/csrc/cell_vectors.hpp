// Vectors assembled in two steps: every cell's vector once, then the sum over the cells of each node.
#pragma once

#include <hip/hip_runtime.h>

#include "assemble_rows.hpp"

namespace nuto_amd
{

// R from the cells' vectors cv[cell][node][F]: one lane per (dof node, component) adds the node's
// incident cells in group order (the order setFromTriplets and the serial loop of
// SimpleAssembler.cpp:49-57 use). Components beyond DIM are the field of slot 1 (row nU + node). The F
// lanes of a node read F consecutive doubles per cell; four cells are in flight at a time.
template <int NND, int DIM, int F>
__global__ void __launch_bounds__(256) kGatherCellVectors(const RowArgs A, const double* __restrict__ cv,
                                                          double* __restrict__ R)
{
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    const int p = (int)(t / F), c = (int)(t % F);
    if (p >= A.nNodes)
        return;
    const int beg = A.incPtr[p], end = A.incPtr[p + 1];
    double sum = 0.0;
    for (int k = beg; k < end; k += 4)
    {
        double v[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
        {
            const int kk = k + i < end ? k + i : end - 1;  // past the last cell: the last, unused
            v[i] = cv[((size_t)A.incCell[kk] * NND + A.incLocal[kk]) * F + c];
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            sum = k + i < end ? sum + v[i] : sum;
    }
    R[c < DIM ? (size_t)p * DIM + c : (size_t)A.nU + p] = sum;
}

template <int NND, int DIM, int F>
inline void LaunchGatherCellVectors(const RowArgs& a, const double* cv, double* R, hipStream_t stream)
{
    const long long n = (long long)a.nNodes * F;
    if (n > 0)
        hipLaunchKernelGGL((kGatherCellVectors<NND, DIM, F>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a,
                           cv, R);
}

}  // namespace nuto_amd
