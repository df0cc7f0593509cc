// Row assembly of elements with few nodes and points (quad4; tet4) without staged cell matrices: a wave owns
// the rows of 16 (quad4) or 8 (tet4) consecutive dof nodes.
//
// The rows of consecutive nodes are one segment of the CSR; it is built in LDS and written once, in
// consecutive stores. Four (eight) lanes per node take its incident cells in turn: each forms the row blocks of one
// cell (CellRows, the integration of the row-owner kernel), then they add theirs to the segment one after
// the other, so every entry sums its cells in group order as setFromTriplets does (SimpleAssembler.cpp:149-155).
// A node's blocks of all its cells would fit one lane, as in kAssembleRows, but that kernel has a quarter of
// the lanes and reads and rewrites each entry in memory, 8 bytes at a time; a cell matrix kernel and a gather
// (kCellMatrices, kGatherRowsWave) write and read 8 ND^2 bytes per cell more.
// Measured, R + K of 40,000 quad4 cells, linear elasticity: row-owner kernel 26.5 us, tiles 10.7 us (14 MB
// moved; 2526 waves, bound by the chain of the gathers and the four turns); tet4, 1350 cells, local damage, with 4
// lanes per node 33 us, with 8 27 us, 33,000 cells 35.3 and 33.9 us.
#pragma once

#include <hip/hip_runtime.h>

#include "assemble_rows.hpp"

namespace nuto_amd
{

// lanes per node (an inner node of a quad4 mesh has 4 cells, of a tet4 mesh about 24), nodes per wave
constexpr int TileLanes(int dim)
{
    return dim == 2 ? 4 : 8;
}
constexpr int TileNodes(int dim)
{
    return 64 / TileLanes(dim);
}
constexpr size_t kTileMaxLds = 40 * 1024;      // segments beyond this leave too few waves per CU

// Rows of the nodes [p0, p1); dynamic LDS: the largest segment of kTileNodes consecutive nodes. Three waves
// per SIMD (at most 168 VGPRs): left alone, tet4 with local damage takes 176 and two, 546,750 cells 234 us
// instead of 213 us.
template <int KIND, int DIM, int NNC, int NND, int NIP, bool WR>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(KIND == kLocalDamage ? 3 : 1)))
kNodeTile(const RowArgs A, int p0, int p1)
{
    static_assert(KIND != kGradientDamage, "one dof type");
    constexpr int kTileLanes = TileLanes(DIM), kTileNodes = TileNodes(DIM);
    extern __shared__ double seg[];
    __shared__ double sR[kTileNodes * DIM];
    const int lane = (int)threadIdx.x;
    const int node = lane / kTileLanes, j = lane % kTileLanes;
    const int first = p0 + (int)blockIdx.x * kTileNodes;
    const int end = first + kTileNodes < p1 ? first + kTileNodes : p1;
    const int p = first + node < end ? first + node : end - 1;
    const bool own = first + node < end;
    const int k0 = A.rowPtr[first * DIM], len = A.rowPtr[end * DIM] - k0;
    for (int k = lane; k < len; k += 64)
        seg[k] = 0.0;
    if (WR && lane < kTileNodes * DIM)
        sR[lane] = 0.0;
    const int beg = A.incPtr[p], last = own ? A.incPtr[p + 1] : beg;
    const int L = (A.adjPtr[p + 1] - A.adjPtr[p]) * DIM;
    double* rows = seg + (A.rowPtr[p * DIM] - k0);
    __syncthreads();
    for (int r0 = beg; __any(r0 < last); r0 += kTileLanes)
    {
        const int r = r0 + j;
        const bool mine = r < last;
        double kacc[NND][DIM * DIM], racc[DIM];
#pragma unroll
        for (int b = 0; b < NND; b++)
#pragma unroll
            for (int i = 0; i < DIM * DIM; i++)
                kacc[b][i] = 0.0;
#pragma unroll
        for (int i = 0; i < DIM; i++)
            racc[i] = 0.0;
        int slot[NND];
        if (mine)
        {
#pragma unroll
            for (int b = 0; b < NND; b++)
                slot[b] = A.slot[(size_t)r * NND + b] & 0x7fff;
            CellNodes<KIND, DIM, NNC, NND> cell;
            LoadCellNodes<KIND, DIM, NNC, NND>(A, A.incCell[r], cell);
            CellRows<KIND, DIM, NNC, NND, NIP, NND, WR, true>(A, cell, A.incLocal[r], 0, kacc, racc);
        }
#pragma unroll
        for (int jj = 0; jj < kTileLanes; jj++)
        {
            if (mine && j == jj)
            {
#pragma unroll
                for (int b = 0; b < NND; b++)
#pragma unroll
                    for (int i = 0; i < DIM; i++)
#pragma unroll
                        for (int k = 0; k < DIM; k++)
                            rows[i * L + DIM * slot[b] + k] += kacc[b][i * DIM + k];
                if constexpr (WR)
                {
#pragma unroll
                    for (int i = 0; i < DIM; i++)
                        sR[node * DIM + i] += racc[i];
                }
            }
            __syncthreads();
        }
    }
    for (int k = lane; k < len; k += 64)
        __builtin_nontemporal_store(seg[k], A.K + k0 + k);
    if (WR && lane < (end - first) * DIM)
        A.R[(size_t)first * DIM + lane] = sR[lane];
}

}  // namespace nuto_amd
