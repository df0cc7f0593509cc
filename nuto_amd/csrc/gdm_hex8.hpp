// Hex8 gradient-damage R+K kernel (the hot path): one 64-lane workgroup per dof node p.
//
// Lanes are (r, m) with r = the r-th cell incident to p (group order) and m = a corner of the cell
// (hex8_lanes.hpp): the integration point there and the column node b there.
//   blocks   lane (r, m): the 4x4 block (a_r, b) of cell r's element matrix for p's rows (a_r = local index
//            of p), summed over the 8 IPs (Cell.h:108-117) by exchanges between the 8 lanes: CellBlock
//   reduce   slot q of p's neighbourhood = sum over r (cell order, the order setFromTriplets
//            uses, SimpleAssembler.cpp:149-155) of the blocks that land on q
//   write    p's three displacement rows (contiguous) and its eeq row, coalesced, written once.
// R is reduced the same way (its IP terms over the lanes, then the cells in order). No atomics: the
// result is deterministic, and every nonzero and R entry is written exactly once per assembly.
//
// Block algebra (per IP, weight s = detJ * w; g = dN/dX; FULL damage application):
//   uu = lambda' S + mu' S^T + mu' tr(S) I with S = sum_ip s (1-omega) g_a g_b^T,
//        lambda' = (3K - 2G) / 3, mu' = G  (LinearElasticDamage::DstressDstrain, H = 1)
//   ue = sum_ip (B_a^T t) N_b, t = s * omega' * kappa' * dSigma/dOmega
//   eu = -sum_ip N_a B_b^T (s * d eps_eq / d eps)
//   ee = sum_ip s N_a N_b + c s g_a . g_b
// UNILATERAL damage application keeps the volumetric factor per IP, so uu is accumulated in the
// general form c1 g_a g_b^T + c2 g_b g_a^T + c2 (g_a . g_b) I.
//
// AFF: every cell of the mesh is affine, one J^-1 per cell; otherwise J^-1 per IP. PRE: the IP states come
// from the pre-pass kGdmHex8Ip; otherwise every node's workgroup evaluates its cells' IPs itself (8 times
// the physics, one launch less), with the same functions on the same operands, so that both give the same
// bits. GdmHex8Plan::Launch says when.
//
// What bounds it: the FP64 and exchange instructions of the vector units, 672 per wave with AFF (333
// FP64), with the latency of the record gather and of the reduction's LDS reads behind them (4 waves per
// SIMD: 9.3 KB of LDS per workgroup). Summing the blocks from records in LDS instead (each lane reading
// the 8 points' records of its cell) took 732 instructions and kept the LDS busy 78 % of the time.
// Measured, R + K: 1,000,000 affine cells 2.39 -> 2.08 ms, 146,969 jittered cells 0.479 -> 0.374 ms.
//
// Usable when every node has at most 8 incident cells and at most 32 neighbours (structured hex
// meshes: 8 and 27) and the coordinate and dof layers share their nodes; other meshes use the
// generic row-owner kernel.
//
// Gathers are two dependent loads deep: per-node incidence tables padded to 8 cells (cell, local index,
// neighbour slots), then the cell's geometry and state records. The geometry of every (cell, IP) - J^-1 and
// detJ * w (Jacobian.h:35-47, Cell.h:108-117) - depends on the coordinates only; it is computed once per
// pattern by kGdmHex8Geometry with the same arithmetic and stored (80 bytes per IP).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "assemble_rows.hpp"
#include "gdm_plan.hpp"
#include "hex8_lanes.hpp"
#include "laws.hpp"
#include "morton.hpp"

namespace nuto_amd
{

namespace gdm8
{
constexpr double kGauss = 0.57735026918962573;  // sqrt(1/3), the 2-point Gauss abscissa
constexpr double kThird = 1.0 / 3.0;
constexpr double kSixth = 1.0 / 6.0;

// dN_n/dxi and N_n of hex8 node n (InterpolationBrickLinear.cpp:42-57 order) at 2x2x2 Gauss point
// ip (xi fastest, IntegrationTypeTensorProduct.cpp:28-38): products of the factors 1 +- g
__device__ inline void ShapeAt(int n, int ip, double d[3], double& N)
{
    const int sx = ((n + 1) >> 1) & 1, sy = (n >> 1) & 1, sz = n >> 2;
    const double f0 = (sx == (ip & 1)) ? 1.0 + kGauss : 1.0 - kGauss;
    const double f1 = (sy == ((ip >> 1) & 1)) ? 1.0 + kGauss : 1.0 - kGauss;
    const double f2 = (sz == (ip >> 2)) ? 1.0 + kGauss : 1.0 - kGauss;
    const double e = 0.125;
    d[0] = (sx ? e : -e) * f1 * f2;
    d[1] = (sy ? e : -e) * f0 * f2;
    d[2] = (sz ? e : -e) * f0 * f1;
    N = e * f0 * f1 * f2;
}

// In the functions below that the pre-pass and the node kernel share, every fused multiply-add is named and
// the compiler's own contraction is off: a record gives the same bits whichever kernel evaluates it.
__device__ inline double Dot3(double a0, double a1, double a2, double b0, double b1, double b2)
{
    return fma(a2, b2, fma(a1, b1, a0 * b0));
}

__device__ inline void ElasticFactors(const LawParams& P, double E, double& m3K, double& m2G)
{
#pragma clang fp contract(off)
    m3K = P.cK * E;
    m2G = P.cG * E;
}

// g = J^-T d  (dN/dX = dN/dxi J^-1, Jacobian.h:100-103)
__device__ inline void GradOf(const double d[3], const double inv[3][3], double g[3])
{
#pragma unroll
    for (int c = 0; c < 3; c++)
        g[c] = fma(d[2], inv[2][c], fma(d[1], inv[1][c], d[0] * inv[0][c]));
}
}  // namespace gdm8

// Integration-point state of GradientDamage<3> (GradientDamage.h:70-135) from the displacement
// gradient w.r.t. xi (Hu), the nonlocal-strain gradient w.r.t. xi (he), the nonlocal strain (eN),
// J^-1 and the history kappa.
struct GdmIp
{
    double eps[6];   // engineering strain, Voigt [xx, yy, zz, yz, zx, xy]
    double ge[3];    // grad eeq
    double eN;       // eeq at the IP
    double dk;       // d kappa / d eeq
    double kap, om, dom;  // kappa, damage and its derivative
    double H;        // 1, or 0 for UNILATERAL application under volumetric compression
    double d2G;      // (1 - omega) 2G
    double sig[6], dsw[6];  // stress and d stress / d omega
    double I1, Am, eq;      // modified Mises: I1, sqrt term, value
};

template <bool FULLDMG>
__device__ inline void GdmIpState(const double Hu[3][3], const double he[3], double eN, const double inv[3][3],
                                  double kh, double m3K, double m2G, double k0, double beta, const LawParams& P,
                                  GdmIp& o)
{
#pragma clang fp contract(off)
    using namespace gdm8;
    // displacement gradient Gu = Hu J^-1
    double Gu[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
        GradOf(Hu[i], inv, Gu[i]);
    o.eps[0] = Gu[0][0];
    o.eps[1] = Gu[1][1];
    o.eps[2] = Gu[2][2];
    o.eps[3] = Gu[1][2] + Gu[2][1];
    o.eps[4] = Gu[2][0] + Gu[0][2];
    o.eps[5] = Gu[0][1] + Gu[1][0];
    GradOf(he, inv, o.ge);
    o.eN = eN;
    // kappa = max(history, eeq), d kappa / d eeq (GradientDamage.h:127-135)
    o.kap = kh < eN ? eN : kh;
    o.dk = eN >= kh ? 1.0 : 0.0;
    // DamageLawExponential (DamageLawExponential.h:39-52)
    o.om = 0.0;
    o.dom = 0.0;
    if (!(o.kap < k0))
    {
        const double ik = 1.0 / o.kap;
        const double ex = exp(beta * (k0 - o.kap));
        const double rr = k0 * ik;
        o.om = fma(-rr, fma(P.alpha, ex, 1.0 - P.alpha), 1.0);
        o.dom = rr * fma((ik + beta) * P.alpha, ex, (1.0 - P.alpha) * ik);
    }
    // LinearElasticDamage<3> stress and dStress/dOmega (LinearElasticDamage.h:65-91)
    const double* eps = o.eps;
    const double eV = (eps[0] + eps[1] + eps[2]) * kThird;
    o.H = (!FULLDMG && eV < 0.0) ? 0.0 : 1.0;
    const double sV = fma(-o.om, o.H, 1.0) * m3K * eV;
    o.d2G = (1.0 - o.om) * m2G;
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
        const double dev = eps[i] - eV;
        o.sig[i] = fma(o.d2G, dev, sV);
        o.dsw[i] = fma(-m2G, dev, -m3K * eV * o.H);
    }
#pragma unroll
    for (int i = 3; i < 6; i++)
    {
        o.sig[i] = 0.5 * o.d2G * eps[i];
        o.dsw[i] = -0.5 * m2G * eps[i];
    }
    // ModifiedMisesStrainNorm<3> value (ModifiedMisesStrainNorm.h:136-146)
    o.I1 = eps[0] + eps[1] + eps[2];
    const double a0 = eps[0] - eps[1], a1 = eps[1] - eps[2], a2 = eps[2] - eps[0];
    const double J2 =
        fma(0.25, Dot3(eps[3], eps[4], eps[5], eps[3], eps[4], eps[5]), Dot3(a0, a1, a2, a0, a1, a2) * kSixth);
    o.Am = sqrt(fma(P.K1 * P.K1 * o.I1, o.I1, P.K2 * J2));
    o.eq = fma(P.K1, o.I1, o.Am);
}

// d eps_eq / d eps of the modified Mises norm (ModifiedMisesStrainNorm.h:231-268, A == 0 branch)
__device__ inline void GdmMisesDerivative(const GdmIp& o, const LawParams& P, double m[6])
{
    using namespace gdm8;
    const double* eps = o.eps;
    if (o.Am == 0.0)
    {
        m[0] = m[1] = m[2] = P.K1;
        m[3] = m[4] = m[5] = 0.0;
    }
    else
    {
        const double h = 0.5 / o.Am;
        const double t2 = 2.0 * P.K1 * P.K1 * o.I1;
        m[0] = P.K1 + h * (t2 + P.K2 * (2.0 * eps[0] - eps[1] - eps[2]) * kThird);
        m[1] = P.K1 + h * (t2 + P.K2 * (2.0 * eps[1] - eps[0] - eps[2]) * kThird);
        m[2] = P.K1 + h * (t2 + P.K2 * (2.0 * eps[2] - eps[0] - eps[1]) * kThird);
        m[3] = h * P.K2 * 0.5 * eps[3];
        m[4] = h * P.K2 * 0.5 * eps[4];
        m[5] = h * P.K2 * 0.5 * eps[5];
    }
}

// Table position of this workgroup, -1 past the end. Workgroups are dispatched round-robin over the
// 8 XCDs; with xcdMap, XCD x takes the x-th contiguous eighth of the traversal, which follows space
// (Morton order), so the nodes one XCD works on at a time share their cells' records in its L2.
// Launches over a node range (one mesh of a batch) index by node and map it through `order`.
__device__ inline int NodeOfBlock(const GdmHex8Tables& T)
{
    int i = blockIdx.x;
    if (T.xcdMap)
    {
        const int per = (int)((gridDim.x + 7) >> 3);
        i = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    }
    i += T.pBegin;
    if (i >= T.pEnd)
        return -1;
    return T.order ? T.order[i] : i;
}

// Table entries of lane (r, m) for the node at a position: its r-th cell (-1 past the last), its local index
// there and the neighbour slot of node c.node of that cell
struct NodeTab
{
    int cell, la, slot;
};

__device__ inline NodeTab LoadNodeTab(const GdmHex8Tables& T, int pos, int r, const CornerLane& c)
{
    const size_t pr = (size_t)pos * 8 + r;
    return NodeTab{T.nodeCell[pr], T.nodeLa[pr], T.nodeSlot[pr * 8 + c.node]};
}

// Geometry and state record of the lane's cell at its IP, and the cell's E. Lanes past the node's last cell
// take cell 0's: their blocks are never read and their R terms are zeroed.
template <bool DEC>
struct NodeRecord
{
    double g[gdm8::kGeo], sr[gdm8::kSrOf<DEC>], E;
};

template <bool PRE, bool AFF, bool DEC>
__device__ inline void LoadNodeRecord(const RowArgs& A, const GdmHex8Tables& T, const NodeTab& tab, const CornerLane& c,
                                      NodeRecord<DEC>& f)
{
    using namespace gdm8;
    constexpr int kN = kSrOf<DEC>, kUse = DEC ? 20 : kSr;  // record stride, doubles read
    const int cell = tab.cell < 0 ? 0 : tab.cell;
    const double2* gr =
        reinterpret_cast<const double2*>(AFF ? T.geoCell + (size_t)cell * kGeo : T.geo + ((size_t)cell * 8 + c.ip) * kGeo);
#pragma unroll
    for (int k = 0; k < kGeo / 2; k++)
    {
        const double2 v = gr[k];
        f.g[2 * k] = v.x;
        f.g[2 * k + 1] = v.y;
    }
    if constexpr (PRE)
    {
        const double2* sp = reinterpret_cast<const double2*>(T.ipState + ((size_t)cell * 8 + c.ip) * kN);
#pragma unroll
        for (int k = 0; k < kUse / 2; k++)
        {
            const double2 v = sp[k];
            f.sr[2 * k] = v.x;
            f.sr[2 * k + 1] = v.y;
        }
    }
    f.E = A.thE ? A.thE[cell] : A.P.E;
}

// The pre-pass state record of an integration point (kSrOf doubles)
template <bool FULLDMG, bool DEC>
__device__ inline void StateRecord(const GdmIp& st, double s, double m3K, double m2G, const LawParams& P, double* rec)
{
#pragma clang fp contract(off)
    using namespace gdm8;
    const double eV = st.I1 * kThird;
    const double sV = fma(-st.om, st.H, 1.0) * m3K * eV;
    double am = P.K1, bm = 0.0;  // m = am [1,1,1,0,0,0] + bm e'' (A == 0: m = K1 [1,1,1,0,0,0])
    if (st.Am != 0.0)
    {
        const double h = 0.5 / st.Am;
        am = fma(-h * P.K2 * st.I1, kThird, fma(h, 2.0 * P.K1 * P.K1 * st.I1, P.K1));
        bm = h * P.K2;
    }
    const double ct = kValueScale * s * st.dom * st.dk, sg = kGradScale * s;
    rec[rEps] = st.eps[0];
    rec[rEps + 1] = st.eps[1];
    rec[rEps + 2] = st.eps[2];
    rec[rEps + 3] = 0.5 * st.eps[3];
    rec[rEps + 4] = 0.5 * st.eps[4];
    rec[rEps + 5] = 0.5 * st.eps[5];
    rec[rSig] = s * fma(-st.d2G, eV, sV);
    rec[rSig + 1] = s * st.d2G;
    rec[rT] = -ct * (m3K * st.H - m2G) * eV;
    rec[rT + 1] = -ct * m2G;
    rec[rM] = sg * am;
    rec[rM + 1] = sg * bm;
    rec[rC1] = FULLDMG ? sg * (1.0 - st.om) : sg * fma(m3K, fma(-st.om, st.H, 1.0), -st.d2G) * kThird;
    rec[rC2] = FULLDMG ? 0.0 : 0.5 * sg * st.d2G;
    rec[rRe] = s * (st.eN - st.eq);
    rec[rGe] = s * P.c * st.ge[0];
    rec[rGe + 1] = s * P.c * st.ge[1];
    rec[rGe + 2] = s * P.c * st.ge[2];
    if constexpr (DEC)
    {
        double gi, dgi;
        NonlocalFactor(P, st.om, gi, dgi);
        rec[rGi] = gi;
        rec[rDg] = dgi * st.dom * st.dk;
        rec[kSrOf<DEC> - 2] = rec[kSrOf<DEC> - 1] = 0.0;
    }
}

// Material of a cell (per-cell fields: E, kappa0 = f_t / E, beta = f_t / G_f)
__device__ inline void GdmMaterial(const RowArgs& A, int cell, double& E, double& k0, double& beta)
{
    E = A.P.E;
    k0 = A.P.kappa0;
    beta = A.P.beta;
    if (A.thE)
    {
        E = A.thE[cell];
        k0 = A.thFt[cell] / E;
        beta = A.thFt[cell] / A.thGf[cell];
    }
}

// The state of (cell, c.ip) from the node values v = (u, eeq) of node c.node in each lane of the cell's
// group; sE: 8 doubles of LDS of the group (written by the caller before a barrier: eeq in local node order)
template <bool FULLDMG>
__device__ inline void GdmCellState(const RowArgs& A, const CornerLane& c, int cell, const double v[4], const double* sE,
                                    const double inv[3][3], GdmIp& st, double& m3K, double& m2G)
{
    double E, k0, beta;
    GdmMaterial(A, cell, E, k0, beta);
    gdm8::ElasticFactors(A.P, E, m3K, m2G);
    const int hist = A.cellId ? A.cellId[cell] : cell;
    const double kh = A.kappa[(size_t)hist + (size_t)c.ip * A.kappaLd];
    double Hu[3][3], he[3], inv0[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
        NodesToPoint(c, v[i], Hu[i]);
#pragma unroll
        for (int k = 0; k < 3; k++)
            inv0[i][k] = kGradScale * inv[i][k];
    }
    NodesToPoint(c, v[3], he);
    GdmIpState<FULLDMG>(Hu, he, NodeSum(c, sE), inv0, kh, m3K, m2G, k0, beta, A.P, st);
}

// the sum over the 8 lanes of a group, ((t0 + t1) + (t2 + t3)) + ((t4 + t5) + (t6 + t7)), valid in its lane 0
__device__ inline double GroupSum0(double v)
{
    v += LaneDpp<kDppXor1>(v);
    v += LaneDpp<kDppXor2>(v);
    v += LaneDpp<0x104>(v);  // row_shl:4: lane i + 4
    return v;
}

// Block (a_r, c.node) of cell r for the rows of node a (local index la), summed over the cell's IPs, from
// the state record sr and geometry g of this lane's IP: acc[4 i + k], i = row component (0..2
// displacement rows, 3 eeq row), k = column component. Each term is a field over the IPs (formed here from
// a's shape data) times N_b or dN_b/dxi, summed to the 8 nodes b by the group's exchanges; with one J^-1
// per cell (AFF) S = (sum s (1-w) g_a dN_b/dxi^T) J^-1, otherwise J^-1 goes into the field. Rv: the R terms
// of node a at this IP, s B_a^T sigma and s (N_a (eeq - eps_eq) + c g_a . grad eeq).
// DEC: the nonlocal term carries g(omega), and K_ee the term c (grad eeq . g_a) g' omega' kappa' N_b, which
// joins s N_a N_b.
template <bool FULLDMG, bool AFF, bool DEC>
__device__ inline void CellBlock(const CornerLane& c, const double* sr, const double* g, int la, double m3K, double m2G,
                                 const LawParams& P, double acc[16], double Rv[4])
{
#pragma clang fp contract(off)
    using namespace gdm8;
    const double inv[3][3] = {{g[0], g[1], g[2]}, {g[3], g[4], g[5]}, {g[6], g[7], g[8]}};
    const double s = g[9];
    double da[3], Na, ga[3];
    ShapeAt(la, c.ip, da, Na);
    GradOf(da, inv, ga);
    const double E[3][3] = {{sr[rEps], sr[rEps + 5], sr[rEps + 4]},
                            {sr[rEps + 5], sr[rEps + 1], sr[rEps + 3]},
                            {sr[rEps + 4], sr[rEps + 3], sr[rEps + 2]}};
    const double gdot = Dot3(ga[0], ga[1], ga[2], sr[rGe], sr[rGe + 1], sr[rGe + 2]);
    const double cs = kGradScale * P.c * (DEC ? s * sr[DEC ? rGi : 0] : s);
    Rv[3] = fma(Na, sr[rRe], DEC ? sr[DEC ? rGi : 0] * gdot : gdot);
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
        // e'' g_a: B_a^T of the Voigt vector e''
        const double Eg = Dot3(E[i][0], E[i][1], E[i][2], ga[0], ga[1], ga[2]);
        Rv[i] = fma(sr[rSig], ga[i], sr[rSig + 1] * Eg);
        acc[4 * i + 3] = ValuesToNode(fma(sr[rT], ga[i], sr[rT + 1] * Eg));  // ue: (B_a^T t) N_b
    }
    double p[3];
    {
        // eu: -N_a s (B_b^T m), m = alpha [1, 1, 1, 0, 0, 0] + beta e''
        const double am = -Na * sr[rM], bm = -Na * sr[rM + 1];
#pragma unroll
        for (int i = 0; i < 3; i++)
        {
#pragma unroll
            for (int k = 0; k < 3; k++)
                p[k] = fma(am, inv[k][i], bm * Dot3(E[i][0], E[i][1], E[i][2], inv[k][0], inv[k][1], inv[k][2]));
            acc[12 + i] = PointsToNode<false>(c, p, 0.0);
        }
    }
    // ee: s N_a N_b + c s g_a . g_b
#pragma unroll
    for (int k = 0; k < 3; k++)
        p[k] = cs * Dot3(ga[0], ga[1], ga[2], inv[k][0], inv[k][1], inv[k][2]);
    acc[15] = PointsToNode<true>(c, p, kValueScale * (DEC ? fma(s, Na, sr[DEC ? rDg : 0] * gdot) : s * Na));
    // S = sum h g_a g_b^T for the factor h of the displacement block
    auto gram = [&](double h, double S[3][3]) {
#pragma unroll
        for (int i = 0; i < 3; i++)
        {
            const double f = h * ga[i];
            if constexpr (AFF)
            {
                double d[3];
                ValuesToGradients(c, f, d);
                GradOf(d, inv, S[i]);
            }
            else
            {
#pragma unroll
                for (int j = 0; j < 3; j++)
                {
#pragma unroll
                    for (int k = 0; k < 3; k++)
                        p[k] = f * inv[k][j];
                    S[i][j] = PointsToNode<false>(c, p, 0.0);
                }
            }
        }
    };
    double S[3][3];
    if constexpr (FULLDMG)
    {
        // uu = lambda' S + mu' S^T + mu' tr(S) I
        gram(sr[rC1], S);
        const double lam = (m3K - m2G) * kThird, mu = 0.5 * m2G;
        const double tr = mu * (S[0][0] + S[1][1] + S[2][2]);
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int k = 0; k < 3; k++)
            {
                acc[4 * i + k] = fma(lam, S[i][k], mu * S[k][i]);
                if (i == k)
                    acc[4 * i + k] += tr;
            }
    }
    else
    {
        // uu = S1 + S2^T + tr(S2) I with the factors c1 and c2
        gram(sr[rC2], S);
        const double tr = S[0][0] + S[1][1] + S[2][2];
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int k = 0; k < 3; k++)
                acc[4 * i + k] = S[k][i] + (i == k ? tr : 0.0);
        gram(sr[rC1], S);
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int k = 0; k < 3; k++)
                acc[4 * i + k] += S[i][k];
    }
}

// K is written once and not read again here: streaming (non-temporal) stores keep the records,
// which are re-read, in the caches.
typedef double D2v __attribute__((ext_vector_type(2)));

// Stores n consecutive doubles from LDS to dst, the 64 lanes writing consecutive 16-byte pairs (a
// leading double when dst is not 16-byte aligned, a trailing one when the rest is odd).
__device__ inline void StoreRows(double* dst, const double* src, int n, int lane)
{
    const int head = (reinterpret_cast<unsigned long long>(dst) & 15) ? 1 : 0;
    if (head && lane == 0)
        __builtin_nontemporal_store(src[0], dst);
    const int np = (n - head) >> 1;
    for (int k = lane; k < np; k += 64)
        __builtin_nontemporal_store(D2v{src[head + 2 * k], src[head + 2 * k + 1]},
                                    reinterpret_cast<D2v*>(dst + head + 2 * k));
    if (((n - head) & 1) && lane == 0)
        __builtin_nontemporal_store(src[n - 1], dst + n - 1);
}

// The rows of node p (one 64-lane workgroup); `state` is the workgroup's LDS (kRed doubles): partial
// blocks, R sums and the slot map.
template <bool WR, bool FULLDMG, bool PRE, bool AFF, bool DEC>
__device__ inline void NodeBody(const RowArgs& A, const GdmHex8Tables& T, int pos, double* state)
{
    using namespace gdm8;
    const int lane = threadIdx.x;
    const int r = lane >> 3, m = lane & 7;
    const CornerLane c = CornerOf(lane);
    const LawParams& P = A.P;
    const NodeTab tab = LoadNodeTab(T, pos, r, c);
    // node p at table position pos; its rows: 3 displacement rows (consecutive in the CSR) and the
    // eeq row, each 4 nA long
    const int4 head = T.nodeHead[pos];
    const int p = head.x, ru0 = head.y, L = head.z, re0 = head.w;
    const int nA = L >> 2;
    const bool valid = tab.cell >= 0;  // r < number of cells incident to p
    const int slot = tab.slot;

    double Rv[4] = {0.0, 0.0, 0.0, 0.0};
    double acc[16];
    if (A.nCells > 0)
    {
        NodeRecord<DEC> rec;
        LoadNodeRecord<PRE, AFF, DEC>(A, T, tab, c, rec);
        double m3K, m2G;
        ElasticFactors(P, rec.E, m3K, m2G);
        if constexpr (!PRE)
        {
            const int cell = valid ? tab.cell : 0;
            const int q = A.dconn[(size_t)cell * 8 + c.node];
            const double v[4] = {A.u[(size_t)q * 3], A.u[(size_t)q * 3 + 1], A.u[(size_t)q * 3 + 2], A.e[q]};
            state[8 * r + c.node] = v[3];
            __syncthreads();
            const double* g = rec.g;
            const double inv[3][3] = {{g[0], g[1], g[2]}, {g[3], g[4], g[5]}, {g[6], g[7], g[8]}};
            GdmIp st;
            GdmCellState<FULLDMG>(A, c, cell, v, state + 8 * r, inv, st, m3K, m2G);
            StateRecord<FULLDMG, DEC>(st, g[9], m3K, m2G, P, rec.sr);
        }
        CellBlock<FULLDMG, AFF, DEC>(c, rec.sr, rec.g, tab.la, m3K, m2G, P, acc, Rv);
        if (!valid)
            Rv[0] = Rv[1] = Rv[2] = Rv[3] = 0.0;
    }
    // R: per cell over its IPs (butterfly within the cell's 8 lanes), then over the cells in order
    if (WR)
    {
#pragma unroll
        for (int k = 0; k < 4; k++)
            Rv[k] = GroupSum0(Rv[k]);  // stored by lane m == 0
    }
    __syncthreads();

    // ---- partial blocks, R sums and the slot map to LDS ----------------------------------------------
    double* part = state;               // [r][m][kPs]
    double* rcell = state + 64 * kPs;  // [4][r]: R terms summed over the IPs of cell r
    // slotOf[q][r] = lane of neighbour q in cell r, 0xFF if q is not a node of cell r
    unsigned char(*slotOf)[kMaxInc] = reinterpret_cast<unsigned char(*)[kMaxInc]>(rcell + 32);
    {
        reinterpret_cast<unsigned int*>(slotOf)[lane] = 0xFFFFFFFFu;  // 64 x 4 bytes = the whole map
#pragma unroll
        for (int i = 0; i < 16; i++)
            part[lane * kPs + i] = acc[i];
    }
    if (WR && m == 0)
    {
#pragma unroll
        for (int k = 0; k < 4; k++)
            rcell[k * 8 + r] = Rv[k];
    }
    __syncthreads();
    if (valid)
        slotOf[slot][r] = (unsigned char)lane;
    __syncthreads();

    // ---- reduce: lane (q, half) sums its 8 block entries over the cells in order and writes them ----
    // (only the cells that hold q are read: the lanes of absent (cell, q) pairs sit out that step, so
    // the LDS reads are the 64 partial blocks, not 8 per neighbour). Row layout: the three
    // displacement rows of p are consecutive in the CSR (4 nA columns each), then the eeq row.
    {
        const int q = lane >> 1, h = lane & 1;
        double sum[8];
#pragma unroll
        for (int k = 0; k < 8; k++)
            sum[k] = 0.0;
        if (q < nA)
        {
            const unsigned long long row = *reinterpret_cast<const unsigned long long*>(&slotOf[q][0]);
#pragma unroll
            for (int rr = 0; rr < 8; rr++)
            {
                const unsigned b = (unsigned)(row >> (8 * rr)) & 0xFFu;
                if (b != 0xFFu)
                {
                    const double* src = part + (int)b * kPs + h * 8;
#pragma unroll
                    for (int k = 0; k < 8; k++)
                        sum[k] += src[k];
                }
            }
        }
        __syncthreads();  // the rows below overwrite the partial blocks
        // p's rows in CSR order in LDS: [3 L] displacement rows, then [L] the eeq row. Block entry
        // (i, c): i = row component (0..2 displacement rows, 3 eeq row), c = column component
        // (0..2 displacement columns, 3 eeq column)
        double* rows = state;
        if (q < nA)
        {
#pragma unroll
            for (int k = 0; k < 8; k++)
            {
                const int e = h * 8 + k;
                const int i = e >> 2, c = e & 3;
                rows[i * L + (c < 3 ? 3 * q + c : 3 * nA + q)] = sum[k];
            }
        }
        __syncthreads();
        StoreRows(A.K + ru0, rows, 3 * L, lane);
        StoreRows(A.K + re0, rows + 3 * L, L, lane);
    }
    if (WR && lane < 4)
    {
        const double* t = rcell + lane * 8;
        double s = 0.0;
#pragma unroll
        for (int rr = 0; rr < 8; rr++)
            s += t[rr];
        if (lane < 3)
            A.R[(size_t)p * 3 + lane] = s;
        else
            A.R[(size_t)A.nU + p] = s;
    }
}

// 4 waves per SIMD (<= 128 VGPRs; the LDS allows 17 workgroups per CU)
template <bool WR, bool FULLDMG, bool PRE, bool AFF, bool DEC>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
kGdmHex8Node(const RowArgs A, const GdmHex8Tables T)
{
    __shared__ __align__(16) double state[gdm8::kRed];
    const int pos = NodeOfBlock(T);
    if (pos < 0)
        return;
    NodeBody<WR, FULLDMG, PRE, AFF, DEC>(A, T, pos, state);
}

// Pre-pass: the state of every (cell, IP) once, for the node kernel (which would otherwise evaluate
// it in each of the cell's 8 node workgroups). Lane (c, ip) of 8-lane group c; node j of the cell is
// gathered by lane (c, j); the lanes exchange their values (NodesToPoint), as in the node kernel.
// AFF: affine cells, IP 0's geometry (T.geoCell) at every IP.
// Workgroup w handles cells 8w .. 8w + 7 (lane (r, j): cell 8w + r, IP j). Their geometry and their
// records are contiguous blocks in memory; both pass through LDS so that every global load and
// store of them is 16 contiguous bytes per lane across the wave (the address and data paths, not
// the arithmetic, bound this kernel).
template <bool FULLDMG, bool AFF, bool DEC>
__global__ void __launch_bounds__(64) kGdmHex8Ip(const RowArgs A, const GdmHex8Tables T, double* __restrict__ out)
{
    using namespace gdm8;
    constexpr int kN = kSrOf<DEC>;
    __shared__ __align__(16) double stage[64 * kN];  // the block's geometry, then its records
    __shared__ double sE[64];  // eeq of the cells' nodes
    const int lane = threadIdx.x;
    const int r = lane >> 3;
    const CornerLane c = CornerOf(lane);
    const long long cell0 = (long long)blockIdx.x * 8;
    const int nc = (int)(A.nCells - cell0 < 8 ? A.nCells - cell0 : 8);  // cells of this block, >= 1
    const int cell = (int)cell0 + (r < nc ? r : 0);  // groups past the last cell repeat the first (not stored)
    {
        constexpr int kPerCell = AFF ? kGeo / 2 : 8 * kGeo / 2;  // 16-byte chunks of geometry per cell
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
    const int q = A.dconn[(size_t)cell * 8 + c.node];
    const double v[4] = {A.u[(size_t)q * 3], A.u[(size_t)q * 3 + 1], A.u[(size_t)q * 3 + 2], A.e[q]};
    sE[8 * r + c.node] = v[3];
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
    const double inv[3][3] = {{g[0], g[1], g[2]}, {g[3], g[4], g[5]}, {g[6], g[7], g[8]}};
    GdmIp st;
    double m3K, m2G, rec[kN];
    GdmCellState<FULLDMG>(A, c, cell, v, sE + 8 * r, inv, st, m3K, m2G);
    StateRecord<FULLDMG, DEC>(st, g[9], m3K, m2G, A.P, rec);
    __syncthreads();  // the records overwrite the geometry
    {
        // record (r, ip) at row r * 8 + ip: 9 or 11 chunks (odd), consecutive lanes on distinct bank groups
        double* dst = stage + (r * 8 + c.ip) * kN;
#pragma unroll
        for (int k = 0; k < kN; k += 2)
            *reinterpret_cast<double2*>(dst + k) = make_double2(rec[k], rec[k + 1]);
    }
    __syncthreads();
    {
        constexpr int kPerCell = 8 * kN / 2;  // 16-byte chunks of records per cell
        const double2* src = reinterpret_cast<const double2*>(stage);
        double2* dst = reinterpret_cast<double2*>(out + cell0 * 8 * kN);
#pragma unroll
        for (int i = 0; i < (8 * kPerCell + 63) / 64; i++)
        {
            const int k = lane + 64 * i;
            if (k < nc * kPerCell)
                dst[k] = src[k];
        }
    }
}

// Geometry of every (cell, IP): J = sum_n X_n dN_n/dxi^T over the coordinate nodes in local
// order (Jacobian.h:16-48), J^-1 and detJ (Jacobian.h:35-47), detJ * w (Cell.h:108-117).
__global__ void __launch_bounds__(256) kGdmHex8Geometry(const double* x, const double* y, const double* z,
                                                         const int* cconn, const double* tab, int nCells,
                                                         double* geo)
{
    using namespace gdm8;
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;  // (cell, ip)
    if (t >= (long long)nCells * 8)
        return;
    const int c = (int)(t >> 3), ip = (int)(t & 7);
    double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
    for (int n = 0; n < 8; n++)
    {
        double d[3], Nv;
        ShapeAt(n, ip, d, Nv);
        const int cn = cconn[(size_t)c * 8 + n];
        const double X[3] = {x[cn], y[cn], z[cn]};
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int k = 0; k < 3; k++)
                J[i][k] += X[i] * d[k];
    }
    double inv[3][3];
    const double detJ = Inverse<3>(J, inv);
    double* g = geo + (size_t)t * kGeo;
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++)
            g[3 * a + b] = inv[a][b];
    g[9] = detJ * tab[ip * kTab];
}

// Counts the cells that are not parallelepipeds (0 means every cell is affine and the node kernel
// may keep one J^-1 per cell). For a parallelepiped J is the same at every point of the cell; the
// J^-1 computed at the 8 IPs then differ only by rounding, so a cell counts as affine when they
// agree to 1e-13 of its largest entry and detJ w to 1e-13 of IP 0's (equal weights, as in 2x2x2
// Gauss). IP 0's geometry is then used for all IPs: a relative change of order 1e-16 in the results.
__global__ void __launch_bounds__(256) kGdmHex8CountNonAffine(const double* geo, int nCells, int* count)
{
    using namespace gdm8;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= nCells)
        return;
    const double* g0 = geo + (size_t)c * 8 * kGeo;
    double scale = 0.0;
    for (int k = 0; k < 9; k++)
        scale = fmax(scale, fabs(g0[k]));
    bool same = true;
    for (int ip = 1; ip < 8; ip++)
    {
        for (int k = 0; k < 9; k++)
            same = same && (fabs(g0[ip * kGeo + k] - g0[k]) <= 1e-13 * scale);
        same = same && (fabs(g0[ip * kGeo + 9] - g0[9]) <= 1e-13 * fabs(g0[9]));
    }
    if (!same)
        atomicAdd(count, 1);
}

// Nodes sorted along a Morton (Z-order) curve of their coordinates (MortonSort): each node takes
// the coordinates of its first incident cell's coordinate node (hex8 dof nodes are the coordinate
// nodes); nodes without cells go first.
inline hipError_t MortonOrder(const NodeGraph& g, int nCells, int nCoord, const double* x, const double* y,
                              const double* z, const int* cconn, hipStream_t stream, std::vector<int>& order)
{
    std::vector<double> hx(nCoord), hy(nCoord), hz(nCoord);
    std::vector<int> hc((size_t)nCells * 8);
    hipError_t err;
    if ((err = hipMemcpyAsync(hx.data(), x, nCoord * sizeof(double), hipMemcpyDeviceToHost, stream)) != hipSuccess ||
        (err = hipMemcpyAsync(hy.data(), y, nCoord * sizeof(double), hipMemcpyDeviceToHost, stream)) != hipSuccess ||
        (err = hipMemcpyAsync(hz.data(), z, nCoord * sizeof(double), hipMemcpyDeviceToHost, stream)) != hipSuccess ||
        (err = hipMemcpyAsync(hc.data(), cconn, hc.size() * sizeof(int), hipMemcpyDeviceToHost, stream)) !=
            hipSuccess ||
        (err = hipStreamSynchronize(stream)) != hipSuccess)
        return err;
    const int n = g.nNodes;
    std::vector<double> pts((size_t)n * 3, 0.0);
    std::vector<char> valid(n, 0);
    for (int p = 0; p < n; p++)
    {
        if (g.incPtr[p + 1] == g.incPtr[p])
            continue;
        const int k = g.incPtr[p];
        const int c = hc[(size_t)g.incCell[k] * 8 + g.incLocal[k]];
        pts[(size_t)p * 3] = hx[c];
        pts[(size_t)p * 3 + 1] = hy[c];
        pts[(size_t)p * 3 + 2] = hz[c];
        valid[p] = 1;
    }
    MortonSort(n, 3, pts.data(), order, valid.data());
    return hipSuccess;
}

}  // namespace nuto_amd
