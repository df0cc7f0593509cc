// Vectors of the hex8 gradient-damage integrand: the residual R = BuildVector(GradientDamage<3>::Gradient)
// (SimpleAssembler.cpp:38-65, GradientDamage.h:70-90) and its vector-Jacobian product with a cotangent
// lambda (length n_rows, layout of R):
//   d_state = (dR / d(u, eeq))^T lambda = K^T lambda   (K = BuildMatrix(Hessian0), GradientDamage.h:92-120)
//   d_theta = (dR / d theta)^T lambda for the per-cell fields theta = (E, f_t, G_f)
//             (kappa0 = f_t / E, beta = f_t / G_f, DamageLawExponential.h:32-37)
// without forming K. The history kappa is a constant of the residual.
//
// Per IP (weight s = detJ w) the residual has the stress sigma, the nonlocal gradient c grad eeq and the
// value eeq - eps_eq; its adjoint, with eps_l = B_u lambda_u, g_l = B_e lambda_e, l_N = N lambda_e, has
//   tau    = (d sigma / d eps) eps_l - l_N (d eps_eq / d eps)       (K_uu^T, K_eu^T parts)
//   c g_l, and the value omega' kappa' (d sigma / d omega . eps_l) + l_N   (K_ue^T, K_ee^T)
//   d_E    += s (sigma / E . eps_l + (d sigma / d omega . eps_l) (d omega / d kappa0) (-kappa0 / E))
//   d_ft   += s (d sigma / d omega . eps_l) (d omega / d kappa0 / E + d omega / d beta / G_f)
//   d_Gf   += s (d sigma / d omega . eps_l) (d omega / d beta) (-beta / G_f)
// (d sigma / d eps is symmetric, LinearElasticDamage.h:74-82; eps_eq and R_e do not depend on theta).
// Both then integrate the same way, d_u,a += s B_a^T tau, d_e,a += s (N_a value + g_a . gradient).
//
// Two kernels: kGdmHex8CellVec evaluates every integration point once, sums the cell's vector over its
// points and writes it (32 doubles per cell) and d_theta; kGatherCellVectors adds the cells' entries of
// every dof node in group order. Nothing limits the number of cells or neighbours of a node. The adjoint of a
// small mesh takes one kernel, kGdmHex8NodeVec.
// Measured on 262,144 cells, affine: adjoint 66 us for the cells + 23 us for the gather, residual 41 + 23
// us (120 and 110 MB moved; the vector arithmetic, about 650 and 450 instructions per wave, takes as long
// as the memory). With every node's workgroup evaluating the points of its own 8 cells the adjoint took
// 665 us and the residual, from records of the points, 318 us.
#pragma once

#include "cell_vectors.hpp"
#include "gdm_hex8.hpp"

namespace nuto_amd
{

// What lane (r, m) reads of its cell: the state and lambda at the lane's node q, the history at its point and the
// material (scalar parameters map to f_t = kappa0 E, G_f = f_t / beta)
struct CellPoint
{
    double v[4], l[4], kh, E, k0, beta, gf;
};

template <bool ADJ>
__device__ inline void LoadCellPoint(const RowArgs& A, const CornerLane& c, int cell, int q,
                                     const double* __restrict__ lam, CellPoint& o)
{
    const LawParams& P = A.P;
    const int hist = A.cellId ? A.cellId[cell] : cell;
    o.kh = A.kappa[(size_t)hist + (size_t)c.ip * A.kappaLd];
    o.E = P.E;
    o.k0 = P.kappa0;
    o.beta = P.beta;
    o.gf = o.k0 * o.E / o.beta;
    if (A.thE)
    {
        o.E = A.thE[cell];
        const double ft = A.thFt[cell];
        o.gf = A.thGf[cell];
        o.k0 = ft / o.E;
        o.beta = ft / o.gf;
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
        o.v[i] = A.u[(size_t)q * 3 + i];
    o.v[3] = A.e[q];
    if constexpr (ADJ)
    {
#pragma unroll
        for (int i = 0; i < 3; i++)
            o.l[i] = lam[(size_t)q * 3 + i];
        o.l[3] = lam[(size_t)A.nU + q];
    }
}

// The cell's vector at the lane's node, summed over the cell's points, into res. sE: eeq of the cell's nodes (LDS,
// written before a barrier); g: the geometry record of the lane's point. ADJ: the cell's d_theta (nCells apart) goes
// to dtheta, if given, from the lane with `own`.
template <bool FULLDMG, bool ADJ>
__device__ inline void CellVectorTerms(const LawParams& P, const CornerLane& c, const CellPoint& pt, const double* sE,
                                       const double* g, double* __restrict__ dtheta, size_t nCells, bool own,
                                       double res[4])
{
    using namespace gdm8;
    const double *v = pt.v, *l = pt.l;
    const double kh = pt.kh, E = pt.E, k0 = pt.k0, beta = pt.beta, gf = pt.gf;
    const double inv[3][3] = {{g[0], g[1], g[2]}, {g[3], g[4], g[5]}, {g[6], g[7], g[8]}};
    const double s = g[9];
    const double m3K = P.cK * E, m2G = P.cG * E;
    double inv0[3][3];  // J^-1 with the gradients' factor
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int k = 0; k < 3; k++)
            inv0[i][k] = kGradScale * inv[i][k];
    double Hu[3][3], he[3];
#pragma unroll
    for (int i = 0; i < 3; i++)
        NodesToPoint(c, v[i], Hu[i]);
    NodesToPoint(c, v[3], he);
    // kappa' jumps where eeq meets the history, as it does at every loading point after an update: eeq is bit
    // for bit the value that the update and the matrix kernels form, so that all take the same side and a
    // residual does not change with the update
    const double eN = NodeSum(c, sE);
    GdmIp st;
    GdmIpState<FULLDMG>(Hu, he, eN, inv0, kh, m3K, m2G, k0, beta, P, st);

    double sig[6], grad[3], value;  // s times the stress-like, gradient-like and value terms
    if constexpr (ADJ)
    {
        double Hl[3][3], hl[3], m[6];
#pragma unroll
        for (int i = 0; i < 3; i++)
            NodesToPoint(c, l[i], Hl[i]);
        NodesToPoint(c, l[3], hl);
        const double lN = kValueScale * NodesToValue(l[3]);
        GdmMisesDerivative(st, P, m);
        double Gl[3][3];
#pragma unroll
        for (int i = 0; i < 3; i++)
            GradOf(Hl[i], inv0, Gl[i]);
        const double el[6] = {Gl[0][0], Gl[1][1], Gl[2][2], Gl[1][2] + Gl[2][1], Gl[2][0] + Gl[0][2],
                              Gl[0][1] + Gl[1][0]};
        const double elV = (el[0] + el[1] + el[2]) * kThird;
        const double sVl = (1.0 - st.om * st.H) * m3K * elV;
        double dsel = 0.0, sgel = 0.0;
#pragma unroll
        for (int i = 0; i < 6; i++)
        {
            sig[i] = s * ((i < 3 ? sVl + st.d2G * (el[i] - elV) : 0.5 * st.d2G * el[i]) - lN * m[i]);
            dsel += st.dsw[i] * el[i];
            sgel += st.sig[i] * el[i];
        }
        GradOf(hl, inv0, grad);
#pragma unroll
        for (int i = 0; i < 3; i++)
            grad[i] *= s * P.c;
        value = s * (st.dom * st.dk * dsel + lN);
        if (dtheta)
        {
            // d omega / d kappa0 and d omega / d beta of DamageLawExponential (zero below kappa0)
            double dwk = 0.0, dwb = 0.0;
            if (!(st.kap < k0))
            {
                const double ik = 1.0 / st.kap;
                const double ex = exp(beta * (k0 - st.kap));
                dwk = -ik * (1.0 - P.alpha + P.alpha * ex) - k0 * ik * P.alpha * beta * ex;
                dwb = -k0 * ik * P.alpha * ex * (k0 - st.kap);
            }
            const double t0 = CornerSum(s * (sgel / E + dsel * dwk * (-k0 / E)));
            const double t1 = CornerSum(s * dsel * (dwk / E + dwb / gf));
            const double t2 = CornerSum(s * dsel * dwb * (-beta / gf));
            if (own)
            {
                dtheta[0] = t0;
                dtheta[nCells] = t1;
                dtheta[2 * nCells] = t2;
            }
        }
    }
    else
    {
        double gi = 1.0, dgi;
        if (P.interaction != 0)
            NonlocalFactor(P, st.om, gi, dgi);
#pragma unroll
        for (int i = 0; i < 6; i++)
            sig[i] = s * st.sig[i];
#pragma unroll
        for (int i = 0; i < 3; i++)
            grad[i] = s * P.c * gi * st.ge[i];
        value = s * (st.eN - st.eq);
    }
    // sigma g_a = (sigma J^-T) dN_a/dxi: the reference-space terms of this point, then the node's sums
    const double S[3][3] = {{sig[0], sig[5], sig[4]}, {sig[5], sig[1], sig[3]}, {sig[4], sig[3], sig[2]}};
    double p[3];
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
#pragma unroll
        for (int k = 0; k < 3; k++)
            p[k] = S[i][0] * inv0[k][0] + S[i][1] * inv0[k][1] + S[i][2] * inv0[k][2];
        res[i] = PointsToNode<false>(c, p, 0.0);
    }
#pragma unroll
    for (int k = 0; k < 3; k++)
        p[k] = grad[0] * inv0[k][0] + grad[1] * inv0[k][1] + grad[2] * inv0[k][2];
    res[3] = PointsToNode<true>(c, p, kValueScale * value);
}

// One wave per 8 cells (lane (r, m): cell 8 w + r, corner m). The geometry records of the wave's cells are
// contiguous and pass through LDS, so that they are read with 16 contiguous bytes per lane; the 4
// values of the lane's node go to out[cell][node][4].
template <bool FULLDMG, bool AFF, bool ADJ>
__global__ void __launch_bounds__(64) kGdmHex8CellVec(const RowArgs A, const GdmHex8Tables T,
                                                       const double* __restrict__ lam, double* __restrict__ out,
                                                       double* __restrict__ dtheta)
{
    using namespace gdm8;
    constexpr int kPerCell = AFF ? kGeo / 2 : 8 * kGeo / 2;  // 16-byte chunks of geometry per cell
    __shared__ __align__(16) double stage[16 * kPerCell];
    __shared__ double sE[64];  // eeq of the cells' nodes
    const int lane = (int)threadIdx.x, r = lane >> 3;
    const CornerLane c = CornerOf(lane);
    const long long cell0 = (long long)blockIdx.x * 8;
    const int nc = (int)(A.nCells - cell0 < 8 ? A.nCells - cell0 : 8);  // cells of this block, >= 1
    const bool valid = r < nc;
    const int cell = (int)cell0 + (valid ? r : 0);
    const int q = A.dconn[(size_t)cell * 8 + c.node];
    {
        const double2* src =
            reinterpret_cast<const double2*>(AFF ? T.geoCell + cell0 * kGeo : T.geo + cell0 * 8 * kGeo);
        double2* dst = reinterpret_cast<double2*>(stage);
#pragma unroll
        for (int i = 0; i < (8 * kPerCell + 63) / 64; i++)
        {
            const int k = lane + 64 * i;
            if (k < nc * kPerCell)
                dst[k] = src[k];
        }
    }
    CellPoint pt;
    LoadCellPoint<ADJ>(A, c, cell, q, lam, pt);
    sE[8 * r + c.node] = pt.v[3];
    __syncthreads();
    double g[kGeo];
    {
        const double2* gs = reinterpret_cast<const double2*>(stage + (AFF ? r : r * 8 + c.ip) * kGeo);
#pragma unroll
        for (int k = 0; k < kGeo / 2; k++)
        {
            const double2 w = gs[k];
            g[2 * k] = w.x;
            g[2 * k + 1] = w.y;
        }
    }
    double res[4];
    CellVectorTerms<FULLDMG, ADJ>(A.P, c, pt, sE + 8 * r, g, dtheta ? dtheta + cell : nullptr, A.nCells,
                                  valid && (lane & 7) == 0, res);
    if (valid)
    {
        double2* dst = reinterpret_cast<double2*>(out + ((size_t)cell * 8 + c.node) * 4);
        dst[0] = make_double2(res[0], res[1]);
        dst[1] = make_double2(res[2], res[3]);
    }
}

// The adjoint in one launch, for small meshes: one wave per dof node, lane (r, m) corner m of the r-th cell
// incident to it. Every cell is evaluated for each of its 8 nodes, but up to 16 waves per CU the time is about
// the latency of one wave, and a second launch costs more. d_theta is the entry of the wave whose node is the
// cell's local node 0. Measured, the whole call, one launch / two: 27 to 4096 nodes 10.3 / 12.8 us, 4913 nodes
// 11.5 / 12.8 us, 6859 nodes 14.6 / 12.8 us.
constexpr int kNodeVecNodes = 16 * 256;
template <bool FULLDMG, bool AFF>
__global__ void __launch_bounds__(64) kGdmHex8NodeVec(const RowArgs A, const GdmHex8Tables T,
                                                       const double* __restrict__ lam, double* __restrict__ vec,
                                                       double* __restrict__ dtheta)
{
    using namespace gdm8;
    __shared__ double sE[64], sV[32];
    const int pos = NodeOfBlock(T);
    if (pos < 0)
        return;
    const int lane = (int)threadIdx.x, r = lane >> 3;
    const CornerLane c = CornerOf(lane);
    const NodeTab tab = LoadNodeTab(T, pos, r, c);
    const int p = T.nodeHead[pos].x;
    const bool valid = tab.cell >= 0;
    const int cell = valid ? tab.cell : 0;
    if (lane < 32)
        sV[lane] = 0.0;
    if (A.nCells > 0)
    {
        NodeRecord<false> rec;
        LoadNodeRecord<false, AFF, false>(A, T, tab, c, rec);
        CellPoint pt;
        LoadCellPoint<true>(A, c, cell, A.dconn[(size_t)cell * 8 + c.node], lam, pt);
        sE[8 * r + c.node] = pt.v[3];
        __syncthreads();
        double res[4];
        const bool own = valid && c.node == tab.la;  // this lane's corner is the node
        CellVectorTerms<FULLDMG, true>(A.P, c, pt, sE + 8 * r, rec.g, dtheta ? dtheta + cell : nullptr, A.nCells,
                                       own && tab.la == 0, res);
        if (own)
        {
#pragma unroll
            for (int k = 0; k < 4; k++)
                sV[4 * r + k] = res[k];
        }
    }
    __syncthreads();
    if (lane < 4)
    {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 8; k++)
            s += sV[4 * k + lane];
        vec[lane < 3 ? (size_t)p * 3 + lane : (size_t)A.nU + p] = s;
    }
}

// The residual (ADJ false: lam and dtheta unused) or the adjoint into `vec` (layout of R). `work`: 32
// doubles per cell of device memory, written in full before they are read.
template <bool ADJ>
inline void LaunchGdmHex8Vector(const GdmHex8Plan& plan, const RowArgs& a, const double* lam, double* vec,
                                double* dtheta, double* work, hipStream_t stream)
{
    const GdmHex8Tables t = plan.Tables();
    const bool full = a.P.damage_application == 0;
    if constexpr (ADJ)
    {
        if (plan.nExtra == 0 && plan.nNodes <= kNodeVecNodes)
        {
            const dim3 grid((unsigned)plan.grid), block(64);
            if (plan.nNodes == 0)
                return;
            if (full && plan.affine)
                hipLaunchKernelGGL((kGdmHex8NodeVec<true, true>), grid, block, 0, stream, a, t, lam, vec, dtheta);
            else if (full)
                hipLaunchKernelGGL((kGdmHex8NodeVec<true, false>), grid, block, 0, stream, a, t, lam, vec, dtheta);
            else if (plan.affine)
                hipLaunchKernelGGL((kGdmHex8NodeVec<false, true>), grid, block, 0, stream, a, t, lam, vec, dtheta);
            else
                hipLaunchKernelGGL((kGdmHex8NodeVec<false, false>), grid, block, 0, stream, a, t, lam, vec, dtheta);
            return;
        }
    }
    if (a.nCells > 0)
    {
        const dim3 grid((unsigned)((a.nCells + 7) / 8)), block(64);
        if (full && plan.affine)
            hipLaunchKernelGGL((kGdmHex8CellVec<true, true, ADJ>), grid, block, 0, stream, a, t, lam, work, dtheta);
        else if (full)
            hipLaunchKernelGGL((kGdmHex8CellVec<true, false, ADJ>), grid, block, 0, stream, a, t, lam, work, dtheta);
        else if (plan.affine)
            hipLaunchKernelGGL((kGdmHex8CellVec<false, true, ADJ>), grid, block, 0, stream, a, t, lam, work, dtheta);
        else
            hipLaunchKernelGGL((kGdmHex8CellVec<false, false, ADJ>), grid, block, 0, stream, a, t, lam, work, dtheta);
    }
    LaunchGatherCellVectors<8, 3, 4>(a, work, vec, stream);
}

}  // namespace nuto_amd
