// Integration-point work of a cell without its matrix: the cell's vector R_e (Cell::Integrate of
// MomentumBalance::Gradient or GradientDamage::Gradient, Cell.h:105-119), the history update
// (GradientDamage::Update, GradientDamage.h:122-125; EvolutionImplicit::Update,
// LocalIsotropicDamage.h:130-133) and the fields of Cell::Eval (Cell.h:80-93).
//
// One workgroup takes as many whole cells as its threads have points: their coordinates and node values go to
// LDS once, lane (cell, IP) forms the point's state, and for R_e lane (cell, node) adds the points in rule order
// from LDS. A point is evaluated once; the row-owner kernel evaluates it for every node of its cell. The sum
// over the cells is kGatherCellVectors. Bound by the latency of the gathers and the two passes over LDS. Where
// a cell has one point (kOwn) its lane is the only reader of its nodes, which then stay in registers.
// Measured on 47,880 ten-node tetrahedra with local damage: residual 267 us by the row-owner kernel, 22 +
// 10 us (gather) here; history 15 -> 13 us, stresses 17 -> 15 us (one lane per point with its own gathers
// before). 2993 waves, three per SIMD: the chain of loads, not a rate, is what is left.
#pragma once

#include <hip/hip_runtime.h>

#include "assemble_rows.hpp"
#include "cell_fields.hpp"

namespace nuto_amd
{

enum PointOutput : int
{
    kPointVector,   // R_e[cell][node][F]
    kPointHistory,  // kappa[cellId + ip * ld] = max(history, equivalent strain) (local damage)
    kPointField     // field[(cell * NIP + ip) * components]
};

// o[DIM i + m] = s sum_k sigma_ik J^-1_mk: sigma g_a = (this) dN_a/dxi
template <int DIM>
__device__ inline void PointTerms(double s, const double* sig, const double inv[DIM][DIM], double* o)
{
    double t[DIM][DIM];
    if constexpr (DIM == 2)
    {
        t[0][0] = sig[0];
        t[1][1] = sig[1];
        t[0][1] = t[1][0] = sig[2];
    }
    else
    {
        t[0][0] = sig[0];
        t[1][1] = sig[1];
        t[2][2] = sig[2];
        t[1][2] = t[2][1] = sig[3];
        t[0][2] = t[2][0] = sig[4];
        t[0][1] = t[1][0] = sig[5];
    }
#pragma unroll
    for (int i = 0; i < DIM; i++)
#pragma unroll
        for (int m = 0; m < DIM; m++)
        {
            double v = 0.0;
#pragma unroll
            for (int k = 0; k < DIM; k++)
                v += t[i][k] * inv[m][k];
            o[DIM * i + m] = s * v;
        }
}

// threads of a workgroup: four waves where a lane has a cell (fewer workgroups to dispatch; 384,000 tet4 cells with
// local damage: history 12.1 us with a wave and LDS, 8.8 with a wave and registers, 8.1 with four waves; kappa 13.2,
// 9.0, 8.4 us), and where a wave's whole cells would leave more than a fifth of its lanes idle (25 points; 10^6
// quad4 cells: strain 414 -> 334 us). Elsewhere one wave: four take longer at their barriers (27 points, 125,000
// hex8 cells: strain 114 -> 131 us).
constexpr int PointThreads(int nip)
{
    return nip == 1 || 64 % nip * 5 > 64 ? 256 : 64;
}

// kappa = max(history, eeq) of gradient damage. It needs no geometry: a lane per cell, the grid's second
// dimension the point, so that the shape values are scalars and the history, stored point by point, is read and
// written in consecutive lanes. Measured, kCellPoints / this kernel: 13,824 cells with 64 points 23.1 / 7.1 us,
// with 27 points 10.6 / 5.5 us, 64,000 cells with 8 points 7.9 / 5.1 us.
template <int NNC, int NND, int NIP>
__global__ void __launch_bounds__(256) kNonlocalHistory(const RowArgs A, double* __restrict__ out)
{
    constexpr int S = 1 + NNC * 3 + NND + NND * 3;  // IP table row: w, dNc, N, dNd
    const int cell = (int)blockIdx.x * 256 + (int)threadIdx.x, ip = (int)blockIdx.y;
    if (cell >= A.nCells)
        return;
    const double* Nd = A.tab + ip * S + 1 + NNC * 3;
    double eN = 0.0;
#pragma unroll
    for (int b = 0; b < NND; b++)
        eN = fma(Nd[b], A.e[A.dconn[(size_t)cell * NND + b]], eN);
    const int cid = A.cellId ? A.cellId[cell] : cell;
    const size_t at = (size_t)cid + (size_t)ip * A.kappaLd;
    const double kh = A.kappa[at];
    out[at] = kh < eN ? eN : kh;
}

template <int KIND, int DIM, int NNC, int NND, int NIP, int OUT>
__global__ void __launch_bounds__(PointThreads(NIP)) kCellPoints(const RowArgs A, int field, double* __restrict__ out)
{
    constexpr int NT = PointThreads(NIP);
    constexpr int CPW = NT / NIP;                       // cells per workgroup
    constexpr bool kOwn = NIP == 1;                     // a lane has its cell to itself: nodes in registers
    constexpr bool GD = KIND == kGradientDamage;
    constexpr int F = GD ? DIM + 1 : DIM;               // values per node
    constexpr int S = 1 + NNC * DIM + NND + NND * DIM;  // IP table row: w, dNc, N, dNd
    constexpr int NV = DIM == 2 ? 3 : 6;
    constexpr int SX = NNC * DIM | 1, SU = NND * F | 1;  // odd strides: consecutive cells on other banks
    constexpr int PR = GD ? DIM * DIM + DIM + 1 : (DIM == 2 ? 5 : 9);  // doubles per point in LDS (odd)
    static_assert(CPW >= 1, "a workgroup holds a cell's points");
    constexpr int IN = kOwn ? 0 : CPW * (SX + SU), RES = OUT == kPointHistory ? 1 : CPW * NIP * PR;
    __shared__ double pool[IN > RES ? IN : RES];  // the cells' nodes, then the points' results
    double* sX = pool;
    double* sU = pool + CPW * SX;
    double* sP = pool;
    const int lane = (int)threadIdx.x;
    const int cell0 = (int)blockIdx.x * CPW;
    const int nc = A.nCells - cell0 < CPW ? A.nCells - cell0 : CPW;
    const LawParams& P = A.P;
    static_assert(!(GD && OUT == kPointHistory), "kNonlocalHistory");
    // every node number, then every node value is loaded before the first of them is waited for
    constexpr int ITX = (CPW * NNC + NT - 1) / NT, ITU = (CPW * NND + NT - 1) / NT;
    double rX[kOwn ? NNC * DIM : 1], rU[kOwn ? NND * F : 1];
    if constexpr (kOwn)
    {
        const size_t cell = (size_t)cell0 + (lane < nc ? lane : 0);
        int nx[NNC], nu[NND];
#pragma unroll
        for (int k = 0; k < NNC; k++)
            nx[k] = A.cconn[cell * NNC + k];
#pragma unroll
        for (int k = 0; k < NND; k++)
            nu[k] = A.dconn[cell * NND + k];
#pragma unroll
        for (int k = 0; k < NNC; k++)
        {
            rX[k * DIM] = A.x[nx[k]];
            rX[k * DIM + 1] = A.y[nx[k]];
            if constexpr (DIM == 3)
                rX[k * DIM + 2] = A.z[nx[k]];
        }
#pragma unroll
        for (int k = 0; k < NND; k++)
        {
#pragma unroll
            for (int i = 0; i < DIM; i++)
                rU[k * F + i] = A.u[(size_t)nu[k] * DIM + i];
            if constexpr (GD)
                rU[k * F + DIM] = A.e[nu[k]];
        }
    }
    else
    {
        int nx[ITX], nu[ITU];
        double x[ITX][DIM], v[ITU][F];
#pragma unroll
        for (int i = 0; i < ITX; i++)
            nx[i] = A.cconn[(size_t)cell0 * NNC + (lane + NT * i < nc * NNC ? lane + NT * i : 0)];
#pragma unroll
        for (int i = 0; i < ITU; i++)
            nu[i] = A.dconn[(size_t)cell0 * NND + (lane + NT * i < nc * NND ? lane + NT * i : 0)];
#pragma unroll
        for (int i = 0; i < ITX; i++)
        {
            x[i][0] = A.x[nx[i]];
            x[i][1] = A.y[nx[i]];
            if constexpr (DIM == 3)
                x[i][2] = A.z[nx[i]];
        }
#pragma unroll
        for (int i = 0; i < ITU; i++)
        {
#pragma unroll
            for (int k = 0; k < DIM; k++)
                v[i][k] = A.u[(size_t)nu[i] * DIM + k];
            if constexpr (GD)
                v[i][DIM] = A.e[nu[i]];
        }
#pragma unroll
        for (int i = 0; i < ITX; i++)
        {
            const int k = lane + NT * i;
            if (k < nc * NNC)
            {
#pragma unroll
                for (int m = 0; m < DIM; m++)
                    sX[k / NNC * SX + k % NNC * DIM + m] = x[i][m];
            }
        }
#pragma unroll
        for (int i = 0; i < ITU; i++)
        {
            const int k = lane + NT * i;
            if (k < nc * NND)
            {
#pragma unroll
                for (int m = 0; m < F; m++)
                    sU[k / NND * SU + k % NND * F + m] = v[i][m];
            }
        }
        __syncthreads();
    }

    const int cl = lane / NIP, ip = lane - cl * NIP;
    double o[PR];  // the point's results
    if (cl < nc)
    {
        const int cell = cell0 + cl;
        const double* t = A.tab + ip * S;
        const double* dNc = t + 1;
        const double* Nd = dNc + NNC * DIM;
        const double* dNd = Nd + NND;
        const double* X = kOwn ? rX : sX + cl * SX;
        const double* U = kOwn ? rU : sU + cl * SU;
        double eN = 0.0;
        if constexpr (GD)
        {
#pragma unroll
            for (int b = 0; b < NND; b++)
                eN = fma(Nd[b], U[b * F + DIM], eN);
        }
        double eps[NV], inv[DIM][DIM], ge[3] = {0.0, 0.0, 0.0}, s = 0.0;
        double J[DIM][DIM];
        NodalGradient<DIM, NNC, DIM>(X, dNc, J);
        s = Inverse<DIM>(J, inv) * t[0];
        if constexpr (DIM == 2 || GD)
        {
#pragma unroll
            for (int i = 0; i < NV; i++)
                eps[i] = 0.0;
#pragma unroll
            for (int b = 0; b < NND; b++)
            {
                double g[DIM];
                Grad<DIM, NND>(dNd, b, inv, g);
                const double* u = U + b * F;
                AddStrain<DIM>(g, u, eps);
                if constexpr (GD)
                {
#pragma unroll
                    for (int i = 0; i < 3; i++)
                        ge[i] += g[i] * u[DIM];
                }
            }
        }
        else
        {
            double R[DIM][DIM];
            // five nodes at a time on twenty: all at once the shape derivatives take 350 registers and leave one
            // wave per SIMD (64,000 hex20 cells, stress 152 -> 105 us); a residual of few cells would wait longer
            NodalGradient<DIM, NND, F, NND == 20 && OUT != kPointVector ? 5 : NND>(U, dNd, R);
            StrainOfGradient(&R[0][0], inv, eps);
        }

        const double E = A.thE ? A.thE[cell] : P.E;
        if constexpr (KIND == kLinearElastic)
        {
            double sig[NV];
            if constexpr (DIM == 2)
            {
                double C11, C12, C33;
                if (P.plane_state == 0)
                {
                    const double f = E / (1.0 - P.nu * P.nu);
                    C11 = f;
                    C12 = f * P.nu;
                    C33 = f * 0.5 * (1.0 - P.nu);
                }
                else
                {
                    const double f = E / ((1.0 + P.nu) * (1.0 - 2.0 * P.nu));
                    C11 = f * (1.0 - P.nu);
                    C12 = f * P.nu;
                    C33 = E / (2.0 * (1.0 + P.nu));
                }
                sig[0] = C11 * eps[0] + C12 * eps[1];
                sig[1] = C12 * eps[0] + C11 * eps[1];
                sig[2] = C33 * eps[2];
            }
            else
            {
                const double f = E / ((1.0 + P.nu) * (1.0 - 2.0 * P.nu));
                const double lam = f * P.nu, mu = E / (2.0 * (1.0 + P.nu));
                const double tr = eps[0] + eps[1] + eps[2];
                for (int i = 0; i < 3; i++)
                    sig[i] = lam * tr + 2.0 * mu * eps[i];
                for (int i = 3; i < 6; i++)
                    sig[i] = mu * eps[i];
            }
            if constexpr (OUT == kPointVector)
                PointTerms<DIM>(s, sig, inv, o);
            else
            {
                // strain or stress (the caller rejects the damage fields)
#pragma unroll
                for (int i = 0; i < NV; i++)
                    o[i] = field == kIpStrain ? eps[i] : sig[i];
            }
        }
        else
        {
            const int cid = A.cellId ? A.cellId[cell] : cell;
            const size_t at = (size_t)cid + (size_t)ip * A.kappaLd;
            double d[6];
            const double eq = Mises3(eps, P.nu, P.k, d);
            const double drive = GD ? eN : eq;
            const double kh = A.kappa[at];
            const double kap = kh < drive ? drive : kh;
            if constexpr (OUT == kPointHistory)
            {
                out[at] = kap;
                return;
            }
            double om = 0.0, dom = 0.0;
            DamageStress3 ds;
            if (OUT == kPointVector || field == kIpStress || field == kIpDamage)
            {
                const double k0 = A.thE ? A.thFt[cell] / E : P.kappa0;
                const double beta = A.thE ? A.thFt[cell] / A.thGf[cell] : P.beta;
                DamageExp(kap, k0, beta, P.alpha, om, dom);
                ElasticDamage3(eps, om, E, P.nu, P.damage_application, ds);
            }
            if constexpr (OUT == kPointVector)
            {
                PointTerms<DIM>(s, ds.sig, inv, o);
                if constexpr (GD)
                {
                    double gi, dgi;
                    NonlocalFactor(P, om, gi, dgi);
                    const double c = s * P.c * gi;
#pragma unroll
                    for (int k = 0; k < 3; k++)
                        o[9 + k] = c * (ge[0] * inv[k][0] + ge[1] * inv[k][1] + ge[2] * inv[k][2]);
                    o[12] = s * (eN - eq);
                }
            }
            else if (field <= kIpStress)
            {
#pragma unroll
                for (int i = 0; i < 6; i++)
                    o[i] = field == kIpStrain ? eps[i] : ds.sig[i];
            }
            else
                o[0] = field == kIpKappa ? kap : (field == kIpDamage ? om : eq);
        }
    }
    if constexpr (OUT == kPointHistory)
        return;
    if constexpr (kOwn && OUT == kPointField)
    {
        if (field > kIpStress)
        {
            if (cl < nc)
                out[cell0 + cl] = o[0];
            return;
        }
    }
    if constexpr (!kOwn)
        __syncthreads();  // the results overwrite the nodes
    if (cl < nc)
    {
#pragma unroll
        for (int i = 0; i < PR; i++)
            sP[lane * PR + i] = o[i];
    }
    __syncthreads();
    if constexpr (OUT == kPointField)
    {
        // the block's values are contiguous: written with consecutive lanes on consecutive doubles
        const int w = field <= kIpStress ? NV : 1;
        double* dst = out + (size_t)cell0 * NIP * w;
        for (int k = lane; k < nc * NIP * w; k += NT)
            dst[k] = sP[(k / w) * PR + k % w];
        return;
    }
    // R_e: the points' reference-space terms against dN_a/dxi (and N_a), in rule order
    for (int k = lane; k < nc * NND; k += NT)
    {
        const int c = k / NND, a = k - c * NND;
        double r[F];
#pragma unroll
        for (int i = 0; i < F; i++)
            r[i] = 0.0;
        for (int q = 0; q < NIP; q++)
        {
            const double* pt = sP + (c * NIP + q) * PR;
            const double* Nd = A.tab + q * S + 1 + NNC * DIM;
            const double* dN = Nd + NND + a * DIM;
            double d[DIM];
#pragma unroll
            for (int m = 0; m < DIM; m++)
                d[m] = dN[m];
#pragma unroll
            for (int i = 0; i < DIM; i++)
#pragma unroll
                for (int m = 0; m < DIM; m++)
                    r[i] += pt[i * DIM + m] * d[m];
            if constexpr (GD)
            {
#pragma unroll
                for (int m = 0; m < DIM; m++)
                    r[DIM] += pt[9 + m] * d[m];
                r[DIM] += pt[12] * Nd[a];
            }
        }
        double* dst = out + ((size_t)cell0 * NND + k) * F;
#pragma unroll
        for (int i = 0; i < F; i++)
            dst[i] = r[i];
    }
}

}  // namespace nuto_amd
