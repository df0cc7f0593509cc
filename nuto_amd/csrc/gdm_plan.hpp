// The hex8 gradient-damage plan of a context: the node kernel's tables, the geometry records and the
// launches (gdm_hex8.hip; the kernels are in gdm_hex8.hpp and gdm_hex8_vectors.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdlib>

#include "assemble_rows.hpp"
#include "devbuf.hpp"
#include "elements.hpp"
#include "mesh.hpp"

namespace nuto_amd
{

namespace gdm8
{
constexpr int kMaxInc = 8;   // incident cells per node
constexpr int kMaxAdj = 32;  // neighbours per node
constexpr int kGeo = 10;     // doubles per (cell, IP) geometry record: J^-1 (row-major), detJ * w
// per (cell, IP) state record of the pre-pass (kGdmHex8Ip): with e'' = [e0, e1, e2, e3/2, e4/2, e5/2]
// (tensor strain) the stress, t = s omega' kappa' d sigma / d omega and m = d eps_eq / d eps are all
// of the form alpha [1, 1, 1, 0, 0, 0] + beta e'', so B_a^T of each is alpha g_a + beta (e'' g_a)
constexpr int kSr = 18;
// with the decreasing nonlocal interaction two more, the factor g and g' omega' kappa' (padded to an odd
// number of 16-byte chunks)
template <bool DEC>
constexpr int kSrOf = DEC ? 22 : kSr;
constexpr int rGi = 18;   // g(omega)
constexpr int rDg = 19;   // dg / d omega * d omega / d kappa * d kappa / d eeq
constexpr int rEps = 0;   // e'' (6)
constexpr int rSig = 6;   // s alpha_sigma, s beta_sigma
constexpr int rT = 8;     // alpha_t, beta_t (s and kValueScale included)
constexpr int rM = 10;    // s alpha_m, s beta_m (kGradScale included, as in the next two)
constexpr int rC1 = 12;   // FULL: s (1 - omega); UNILATERAL: s (3K (1 - omega H) - 2G (1 - omega)) / 3
constexpr int rC2 = 13;   // UNILATERAL: s G (1 - omega); FULL: 0
constexpr int rRe = 14;   // s (eeq - eps_eq)
constexpr int rGe = 15;   // s c grad eeq (3)
constexpr int kPs = 17;      // doubles per partial block (odd: 64 lanes spread over the banks)
constexpr int kTab = 57;     // per-IP table row: w, dNc[8][3], N[8], dNd[8][3]

constexpr int kRed = 1160;  // doubles of the reduction: partial blocks 64 x kPs, R sums 32, 8 unused, slot map 32

}  // namespace gdm8

// Per-node tables of the node kernel (built once per pattern, see GdmHex8Plan::Prepare), stored in
// traversal order: position s holds the node order[s] (nodes sorted along a Morton curve).
struct GdmHex8Tables
{
    const int4* nodeHead;           // [pos]: node p, first CSR entry of its displacement rows, their
                                    //        length 4 nA, first CSR entry of its eeq row
    const int* nodeCell;            // [pos][8]: r-th incident cell (group order), -1 past the last
    const unsigned char* nodeLa;    // [pos][8]: local index of the node in that cell
    const unsigned char* nodeSlot;  // [pos][8][8]: neighbour slot (column block) of local node j
    const double* geo;              // [cell][ip][kGeo] geometry records
    const double* ipState;          // [cell][ip][kSrOf] pre-pass state records (nullptr: recompute)
    const double* geoCell;          // [cell][kGeo] IP 0's geometry record (affine meshes, else nullptr)
    int xcdMap;                     // 1: contiguous node ranges per XCD
    int pBegin, pEnd;               // launch indices [pBegin, pEnd)
    const int* order;               // launch index -> position (nullptr: the index is the position)
};

struct GdmHex8Plan
{
    bool ready = false;
    int nNodes = 0;
    int grid = 0;     // workgroups: one per node (rounded up to a multiple of 8 with the XCD mapping)
    int xcdMap = 1;   // contiguous node ranges per XCD (env NUTO_AMD_GDM_XCD_MAP=0 switches it off)
    DevBuf nodeHead, nodeCell, nodeLa, nodeSlot, geo;
    DevBuf posOf;        // node -> table position (Morton order; NUTO_AMD_GDM_ORDER=0: node order, empty)
    DevBuf ipState;      // pre-pass state records, or cell vectors (Work)
    DevBuf geoCell;      // affine meshes: IP 0's geometry record per cell
    DevBuf extra;        // nodes beyond the kernel's bounds (more than 8 cells or 32 neighbours)
    int nExtra = 0;      // ... assembled by the generic row-owner kernel
    int prepass = -1;     // NUTO_AMD_GDM_PREPASS=0 / 1: never / always run the pre-pass; -1: by the mesh's size
    bool affine = false;  // every cell affine: one J^-1 per cell
    bool decreasing = false;  // NonlocalInteraction::Decreasing: longer pre-pass records
    int nCells = 0;

    void Release()
    {
        ready = false;
        nNodes = 0;
        for (DevBuf* b : {&nodeHead, &nodeCell, &nodeLa, &nodeSlot, &geo, &ipState, &posOf, &geoCell, &extra})
            b->Release();
        nExtra = 0;
    }

    bool Usable(int kind, int coordType, int dofType, int nip) const
    {
        return ready && kind == kGradientDamage && coordType == kHex8 && dofType == kHex8 && nip == 8;
    }

    // Builds the per-node tables from the node graph and the geometry records from the device
    // coordinates (x, y, z by coordinate node, cconn) and the IP table. Returns false (plan not
    // used) when the mesh exceeds the kernel's bounds; a HIP failure is returned through `err`.
    bool Prepare(int kind, int coordType, int dofType, int nip, const NodeGraph& g, int nCells,
                 int nCoord, const double* x, const double* y, const double* z, const int* cconn, const double* tab,
                 const int* rowPtr, int nRows, bool decreasingInteraction, hipStream_t stream, hipError_t& err);

    GdmHex8Tables Tables() const
    {
        return GdmHex8Tables{nodeHead.As<int4>(), nodeCell.As<int>(),
                             nodeLa.As<unsigned char>(), nodeSlot.As<unsigned char>(), geo.As<double>(),
                             ipState.p ? ipState.As<double>() : nullptr, geoCell.p ? geoCell.As<double>() : nullptr,
                             xcdMap, 0, nNodes, nullptr};
    }

    // doubles of a pre-pass record
    int RecordDoubles() const
    {
        return decreasing ? gdm8::kSrOf<true> : gdm8::kSrOf<false>;
    }

    // doubles of the pre-pass state records (written in full by kGdmHex8Ip before the node kernel reads them)
    size_t StateDoubles() const
    {
        return prepass ? (size_t)nCells * 8 * RecordDoubles() : 0;
    }

    // K (and R, wr). state: device memory of StateDoubles() doubles for the pre-pass records (nullptr: the
    // plan's own)
    void Launch(const RowArgs& a, bool wr, hipStream_t stream, double* state = nullptr) const;

    // The plan's device memory: the pre-pass records of a matrix assembly (StateDoubles), or the cell
    // vectors of a residual or an adjoint (32 doubles per cell, less than the records)
    double* Work() const
    {
        return ipState.As<double>();
    }

    // K (and R) rows of the nodes beyond the node kernel's bounds (the generic row-owner body)
    void LaunchExtras(const RowArgs& a, bool wr, hipStream_t stream) const;

    // R + K of the nodes [first, end) only (one mesh of a batch), plain block order; the nodes beyond
    // the bounds are not visited (LaunchExtras covers them for the whole plan)
    void LaunchRange(const RowArgs& a, int first, int end, hipStream_t stream) const;

    // The residual into `vec` (layout of R)
    void LaunchVector(const RowArgs& a, double* vec, hipStream_t stream) const;

    // K^T lambda into `vec` and, unless null, dR/dtheta^T lambda into `dtheta` (3 x nCells)
    void LaunchAdjoint(const RowArgs& a, const double* lam, double* vec, double* dtheta, hipStream_t stream) const;
};

}  // namespace nuto_amd
