// Outputs of a cell group besides R and K: the diagonally lumped mass matrix and the names of the fields
// at the integration points (cell_points.hpp).
//
// kLumpedMass: SimpleAssembler::BuildDiagonallyLumpedMatrix (SimpleAssembler.cpp:67-98) with the
//   integrand DynamicMomentumBalance::Hessian2 = N^T N rho (DynamicMomentumBalance.h:22-30) on dof
//   type slot 0. Row-owner form like the assembly kernel: one lane per dof node, its incident cells
//   in group order, so the per-node sum runs in cell order without atomics.
#pragma once

#include <hip/hip_runtime.h>

#include "assemble_rows.hpp"

namespace nuto_amd
{

// fields of nuto_eval_ip (values per IP: strain and stress NV = 3 (2D) or 6 (3D), the others 1)
enum IpField : int
{
    kIpStrain = 0,    // B u, engineering Voigt (Nabla::Strain, DifferentialOperators.h:24-86)
    kIpStress = 1,    // the law's stress at that strain (and damage)
    kIpKappa = 2,     // GradientDamage::Kappa = max(history, eeq) (GradientDamage.h:126-129);
                      // local damage: max(history, eps_eq(strain)) (EvolutionImplicit)
    kIpDamage = 3,    // DamageLawExponential::Damage(kappa) (DamageLawExponential.h:39-45)
    kIpEqStrain = 4,  // ModifiedMisesStrainNorm::Value(strain) (ModifiedMisesStrainNorm.h:70-84)
};

// J = X dN/dxi of the coordinate element of `cell` at one IP, its inverse and determinant
// (Jacobian.h:16-48)
template <int DIM, int NNC>
__device__ inline double CellJacobian(const RowArgs& A, int cell, const double* dNc, double inv[DIM][DIM])
{
    double X[NNC][DIM];
#pragma unroll
    for (int k = 0; k < NNC; k++)
    {
        const int n = A.cconn[(size_t)cell * NNC + k];
        X[k][0] = A.x[n];
        X[k][1] = A.y[n];
        if constexpr (DIM == 3)
            X[k][2] = A.z[n];
    }
    double J[DIM][DIM];
    NodalGradient<DIM, NNC, DIM>(&X[0][0], dNc, J);
    return Inverse<DIM>(J, inv);
}

// Lumped mass of dof node p: over the incident cells in group order, the cell's consistent-mass
// diagonal entry m_p = sum_ip ((N_p N_p) rho detJ) w (first IP assigns, Cell.h:105-119), times
// (sum of all entries of the cell's block / sum of its diagonal) / ncomp. The block has ncomp
// identical copies of the nodal mass matrix, so the two sums are ncomp sum_ip ((sum_a N_a)^2 rho
// detJ) w and ncomp sum_a m_a, and their ratio needs no ncomp. Every component of p gets the
// same value.
template <int DIM, int NNC, int NND, int NIP>
__global__ void __launch_bounds__(64) kLumpedMass(const RowArgs A, double rho, double* __restrict__ M)
{
    constexpr int S = 1 + NNC * DIM + NND + NND * DIM;
    const int p = blockIdx.x * 64 + threadIdx.x;
    if (p >= A.nNodes)
        return;
    double acc = 0.0;
    for (int r = A.incPtr[p]; r < A.incPtr[p + 1]; ++r)
    {
        const int cell = A.incCell[r];
        const int la = A.incLocal[r];
        double m[NND];
        double full = 0.0;
        for (int ip = 0; ip < NIP; ip++)
        {
            const double* t = A.tab + ip * S;
            const double w = t[0];
            const double* dNc = t + 1;
            const double* Nd = dNc + NNC * DIM;
            double inv[DIM][DIM];
            const double detJ = CellJacobian<DIM, NNC>(A, cell, dNc, inv);
            double sN = 0.0;
#pragma unroll
            for (int b = 0; b < NND; b++)
            {
                const double v = (((Nd[b] * Nd[b]) * rho) * detJ) * w;
                m[b] = ip == 0 ? v : m[b] + v;
                sN += Nd[b];
            }
            const double f = (((sN * sN) * rho) * detJ) * w;
            full = ip == 0 ? f : full + f;
        }
        double diag = 0.0;
#pragma unroll
        for (int b = 0; b < NND; b++)
            diag += m[b];
        double mp = 0.0;
#pragma unroll
        for (int b = 0; b < NND; b++)
            mp = b == la ? m[b] : mp;
        acc += mp * ((full / diag) / DIM);
    }
#pragma unroll
    for (int c = 0; c < DIM; c++)
        M[(size_t)p * DIM + c] = acc;
}

}  // namespace nuto_amd
