// Constrained linear solve on the device: ConstrainedSystemSolver::Solve / SolveTrialState
// (Solve.cpp:8-78) with the unit constraint matrix C of Constraints::BuildUnitConstraintMatrix
// (Constraints.cpp:89-137).
//
// The reduced system (C^T K C) u = C^T f is never formed, and its vectors are not stored in the reduced
// numbering: every Krylov vector has the full length, independent dof j at its own position and zeros
// at the dependent dofs. C then only fills the dependent entries of a product's input from the
// equations' terms, C^T adds the dependent rows of the result to the terms' dofs; without terms (all
// equations x = rhs, the usual case) both are the mask that the K product applies when it writes. So an
// operator application is one pass over K instead of three kernels with two more passes over the
// vectors.
//
// Solvers: Jacobi-preconditioned conjugate gradients and BiCGSTAB (the iterative solvers NuTo selects
// by name, EigenSparseSolve.cpp:44-49, whose default preconditioner is the diagonal). An iteration is
// two (CG) or three (BiCGSTAB) kernels in small systems, three or five in larger ones (kFormNodes). Dot
// products ride on the kernels that make their operands: each block leaves its partial sum, and every
// block of the next kernel adds the partials itself, all in the same fixed order, so solves are
// bit-reproducible and no kernel exists only to finish a reduction (but for the K product of the largest
// systems, kFoldRows). A kernel loads all that does not depend on those sums, the test of the status
// included, before it waits for them. The scalars, the convergence test and the iteration count stay on the device
// (KrylovState); once the test is met the remaining launches return at once. The host queues
// kSolveChunk iterations at a time and reads the state of a chunk while the next one runs, so the
// device never waits for it.
// Measured, per iteration: BiCGSTAB in a load step on 1536 hex8 gradient-damage cells (K of 5.8 MB) 61
// us with 14 kernels and a host read, 23 us with five kernels, 15.3 us with three (the two products 5.8 us
// each, the update 3.7 us, without gaps between them); conjugate gradients on 24,480 elastic tet10 cells (K
// of 69 MB) 55 us with 9 kernels and a host read, 29 us with three.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <vector>

#include "devbuf.hpp"
#include "lanes.hpp"

namespace nuto_amd
{

constexpr int kDotBlocks = 1024;    // blocks (= partial sums) of the vector kernels
constexpr int kSpmvBlocks = 2048;   // blocks of the K product: 8 of 4 waves on each of 256 CUs
constexpr int kSolveChunk = 4;      // iterations the host queues before it reads a state

// Up to this size a wave of the K product has one node, and an iteration takes as long as its chain of
// launches and dependent loads: there the product forms its input vector where it gathers it, and the
// kernels that made the vectors are left out. In larger systems the product is bound by its reads, and two
// or three gathers in place of one cost more than a pass over the vectors. Measured, us per iteration with
// stored / formed vectors, hex8 gradient damage (K of 4 rows per node): CG 125 nodes 12.0 / 9.3, 2025 nodes
// 13.6 / 11.1, 9261 nodes 16.0 / 15.4, 226,981 nodes 234 / 248; BiCGSTAB 18.6 / 16.1, 20.4 / 17.5, 27.6 / 28.5,
// 465 / 530; elastic hex8, 15,625 nodes: 17.5 / 17.0 and 30.5 / 33.3.
constexpr int kFormNodes = 4 * kSpmvBlocks;

// From this many rows on a wave of the K product has one node, and one more kernel adds the many blocks'
// partials up to kFoldBlocks: waves that stride over the nodes keep the partials few, but 2048 blocks of 72
// VGPRs are one and a third rounds of resident blocks, and a wave that ends early leaves its place empty.
// Below, the fold's launch costs more than that. Measured, us per iteration, striding / one node per wave:
// hex8 gradient damage (4 rows per node), BiCGSTAB 157,216 rows 67.0 / 68.3, 202,612 rows 85.7 / 82.5,
// 4,121,204 rows 2122 / 1687, CG there 1064 / 857; elastic hex8, BiCGSTAB 151,959 rows 62.3 / 63.1, 206,763
// rows 79.6 / 78.0, 3,090,903 rows 1451 / 1219; elastic quad4 181,202 rows 70.3 / 72.7, 722,402 rows 235 / 225.
constexpr int kFoldRows = 24 * 4 * kSpmvBlocks;
constexpr int kFoldBlocks = 512;

enum SolveStatus : int
{
    kRunning = 0,
    kDone = 1,
    kRestart = 2  // BiCGSTAB: rho is tiny, the host recomputes the residual (rare)
};

// Scalars of a running solve. Two copies are used in turn: the first kernel of iteration s reads copy
// s & 1 and writes copy (s + 1) & 1, the other kernels of the iteration use the latter; no block then
// reads a field that another block of the same kernel writes.
struct KrylovState
{
    double rr, bb, rho, alpha, w, r0sq;  // (r . r), (b . b); CG: rho = (r . z)
    int status, iters;
};

// sums of N per-lane values over the 256 lanes of a block, known to every lane: within each wave, then
// the four waves in order
template <int N>
__device__ inline void BlockSum(double v[N], double* sh)
{
    const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < N; i++)
    {
        v[i] = WaveSum(v[i]);
        if (lane == 0)
            sh[i * 4 + wave] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; i++)
        v[i] = (sh[i * 4] + sh[i * 4 + 1]) + (sh[i * 4 + 2] + sh[i * 4 + 3]);
    __syncthreads();  // sh may be used again
}

// the N sums whose per-block partials are part[i * np + block] (np <= MAX), known to every lane; every
// load is issued before the first sum waits for one
template <int N, int MAX>
__device__ inline void SumPartials(const double* __restrict__ part, int np, double v[N], double* sh)
{
    constexpr int STEPS = MAX / 256;
    double t[N][STEPS];
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int j = 0; j < STEPS; j++)
        {
            const int k = (int)threadIdx.x + 256 * j;
            t[i][j] = part[i * np + (k < np ? k : np - 1)];
        }
#pragma unroll
    for (int i = 0; i < N; i++)
    {
        v[i] = 0.0;
#pragma unroll
        for (int j = 0; j < STEPS; j++)
            v[i] = (int)threadIdx.x + 256 * j < np ? v[i] + t[i][j] : v[i];
    }
    BlockSum<N>(v, sh);
}

// the block's partials of N sums
template <int N>
__device__ inline void StorePartials(double v[N], double* __restrict__ part, double* sh)
{
    BlockSum<N>(v, sh);
    if (threadIdx.x == 0)
    {
#pragma unroll
        for (int i = 0; i < N; i++)
            part[i * gridDim.x + blockIdx.x] = v[i];
    }
}

// What the first kernel of an iteration needs: its launch number seq (copy seq & 1 of the state is read, the
// other written), the iteration `it`, the partials of the dots that the iteration before left, the
// tolerance. first: the state of a new solve; forced: no tests (the iteration after a restart, whose
// (r . r) becomes |r0|^2); check: the test alone, no iteration follows. tell: where the host reads the
// outcome (pinned memory, or nullptr): the kernel writes it there itself, since a copy command between the
// kernels holds the stream up for longer than an iteration of a small system takes.
struct StepArgs
{
    int seq, it;
    bool first, forced, check;
    double tol2;
    const double* part;
    int np;
    KrylovState* st;
    KrylovState* tell;
};

__device__ inline void Tell(KrylovState* host, double rr, double bb, int status, int iters)
{
    if (!host)
        return;
    host->rr = rr;
    host->bb = bb;
    host->status = status;
    host->iters = iters;
}

// CG: the test |r|^2 < tol^2 |b|^2, then beta = (r . z) / (r . z of the iteration before); false when the
// solve has ended
__device__ inline bool CgStep(const StepArgs& a, double* sh, double& beta)
{
    const KrylovState* in = a.st + (a.seq & 1);
    KrylovState* out = a.st + ((a.seq + 1) & 1);
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    const int status = in->status, iters = in->iters;
    const double oldRr = in->rr, oldRho = in->rho, oldBb = in->bb;
    double s[2];
    SumPartials<2, kDotBlocks>(a.part, a.np, s, sh);
    if (status != kRunning)
    {
        if (lead)
        {
            out->rr = oldRr;
            out->bb = oldBb;
            out->status = status;
            out->iters = iters;
            Tell(a.tell, oldRr, oldBb, status, iters);
        }
        return false;
    }
    const double bb = a.first ? s[0] : oldBb;
    const bool done = s[0] < fmax(a.tol2 * bb, 1e-300);
    if (lead)
    {
        const int now = done ? kDone : kRunning;
        const int before = done && a.it > 0 ? a.it - 1 : a.it;  // the iterations before the converging one
        out->rr = s[0];
        out->bb = bb;
        out->rho = s[1];
        out->status = now;
        out->iters = before;
        Tell(a.tell, s[0], bb, now, before);
    }
    beta = a.first ? 0.0 : s[1] / oldRho;
    return !done;
}

// BiCGSTAB: the tests !(|r|^2 > tol^2 |b|^2) and |rho| < eps^2 |r0|^2 (a restart, done by the host), then
// beta; false when the solve has ended or waits for the restart
__device__ inline bool BicgStep(const StepArgs& a, double* sh, double& beta)
{
    const KrylovState* in = a.st + (a.seq & 1);
    KrylovState* out = a.st + ((a.seq + 1) & 1);
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    const int status = in->status, iters = in->iters;
    const double oldRr = in->rr, oldBb = in->bb, oldRho = in->rho, alpha = in->alpha, w = in->w, oldR0 = in->r0sq;
    double s[2];
    SumPartials<2, kDotBlocks>(a.part, a.np, s, sh);
    if (status == kDone || (status == kRestart && !a.forced))
    {
        if (lead)
        {
            out->rr = oldRr;
            out->bb = oldBb;
            out->rho = oldRho;
            out->alpha = alpha;
            out->w = w;
            out->r0sq = oldR0;
            out->status = status;
            out->iters = iters;
            Tell(a.tell, oldRr, oldBb, status, iters);
        }
        return false;
    }
    const double bb = a.first ? s[0] : oldBb, r0sq = a.first || a.forced ? s[0] : oldR0;
    int now = kRunning;
    if (!a.forced)
    {
        const double eps2 = 2.220446049250313e-16 * 2.220446049250313e-16;
        if (!(s[0] > a.tol2 * bb))
            now = kDone;
        else if (!a.check && fabs(s[1]) < eps2 * r0sq)
            now = kRestart;
    }
    if (lead)
    {
        const double rr = a.forced ? oldRr : s[0];  // after a restart the residual's norm is the one that was tested
        Tell(a.tell, rr, bb, now, a.it);
        out->rr = rr;
        out->bb = bb;
        out->rho = now == kRestart ? oldRho : s[1];  // the restarted iteration's beta divides by the last rho
        out->alpha = alpha;
        out->w = w;
        out->r0sq = r0sq;
        out->status = now;
        out->iters = a.it;
    }
    beta = (s[1] / oldRho) * (alpha / w);
    return now == kRunning;
}

// Dots of the K product: none, (d . y) (CG: p . q, BiCGSTAB: r0 . v), or (y . y) and (d . y)
// (BiCGSTAB: t . t, t . s)
enum SpmvDots : int
{
    kNoDots = 0,
    kOneDot = 1,
    kTwoDots = 2
};

// The vector that the K product multiplies: x itself, or formed entry by entry where it is gathered (every
// block forms the entries it needs; `own` receives the vector before the preconditioner at the block's rows):
// CG p = x + beta x2 (z, the last p), BiCGSTAB invd p with p = x + beta x2 (r, the last p - w v) or invd s with
// s = x - alpha x2 (r, v)
enum SpmvInput : int
{
    kStored = 0,
    kCgDirection = 1,
    kBicgDirection = 2,
    kBicgHalfStep = 3
};
struct FormedInput
{
    const double *x, *x2, *invd;
    double* own;
    StepArgs step;            // the directions: the iteration begins here
    const double* dotPart;    // the half step: partials of (r0 . v)
    int nDot;
};

// y = A x for a CSR matrix, 16 lanes per row: lane l sums the entries l, l + 16, ... of its row in
// order, then the partial sums are added by an xor butterfly (a fixed order). For numberings whose
// node structure the kernel below does not cover.
__global__ void __launch_bounds__(256) kCsrSpmv(int nRows, const int* __restrict__ rowPtr, const int* __restrict__ col,
                                                const double* __restrict__ val, const double* __restrict__ x,
                                                double* __restrict__ y)
{
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long r = t / 16;
    const int l = (int)(t % 16);
    double s = 0.0;
    if (r < nRows)
        for (int k = rowPtr[r] + l; k < rowPtr[r + 1]; k += 16)
            s += val[k] * x[col[k]];
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1)
        s += __shfl_xor(s, m, 16);
    if (r < nRows && l == 0)
        y[r] = s;
}

// y = K x for the assembled monolithic K: the C0 field-0 rows of dof node p (rows C0 p + i) and its
// field-1 row (nU + p, when C1 = 1) hold the same L columns, so one wave per node reads each x entry
// once for all of them. Lane l sums the entries l, l + 64, ... of each row in order; the 64 partial
// sums are added by exchanges in which the lanes share out the rows, a fixed order, without LDS.
// A wave strides over the nodes (so that the dots' partials stay few; not in the largest systems, kFoldRows)
// and keeps the next node's first 128 entries of every row in flight while it works on this one's, and
// the row offsets of the node after that: only the gather of x is waited for. mask (one byte per node,
// bit i: row i is a dependent dof) zeroes those rows of y; DOTS: the block's partial sums of the dots over
// its rows.
// Bound by the reads of the values; in small systems by the latency of its launch and of its dependent
// loads. IN != kStored: the kernel that would make x is left out, see SpmvInput; the first node's entries
// are in flight while the block adds the partials.
template <int C0, int C1, int DOTS, int IN>
__global__ void __launch_bounds__(256) kNodeSpmv(int nNodes, int nU, const int* __restrict__ rowPtr,
                                                 const int* __restrict__ col, const double* __restrict__ val,
                                                 const double* __restrict__ x, double* __restrict__ y,
                                                 const unsigned char* __restrict__ mask, const double* __restrict__ d,
                                                 double* __restrict__ part, KrylovState* __restrict__ st,
                                                 const FormedInput in)
{
    constexpr int F = C0 + C1;
    __shared__ double sh[8];
    const int status = IN == kStored && DOTS != kNoDots ? st->status : kRunning;
    const int l = (int)(threadIdx.x & 63);
    const int step = (int)gridDim.x * 4;
    const int last = nNodes - 1;
    int p = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    double dots[2] = {0.0, 0.0};
    // row offsets of a node: its field-0 rows begin at r0, L entries each, its field-1 row at re
    struct Head
    {
        int r0, L, re;
    };
    auto head = [&](int q) {
        const int c = q < last ? q : last;  // past the end: the last node's, unused
        Head h;
        h.r0 = rowPtr[C0 * c];
        h.L = rowPtr[C0 * c + 1] - h.r0;
        h.re = C1 ? rowPtr[nU + c] : 0;
        return h;
    };
    // entries l and l + 64 of every row (lanes past the end: the last entry, unused)
    int ca, cb;
    double va[F], vb[F];
    auto load = [&](const Head& h) {
        const int ka = l < h.L ? l : h.L - 1, kb = l + 64 < h.L ? l + 64 : h.L - 1;
        ca = col[h.r0 + ka];
        cb = col[h.r0 + kb];
#pragma unroll
        for (int i = 0; i < C0; i++)
        {
            va[i] = val[h.r0 + i * h.L + ka];
            vb[i] = val[h.r0 + i * h.L + kb];
        }
        if constexpr (C1 == 1)
        {
            va[C0] = val[h.re + ka];
            vb[C0] = val[h.re + kb];
        }
    };
    Head now = head(p), next = head(p + step);
    if (p < nNodes && now.L > 0)
        load(now);
    if (status != kRunning)
        return;
    double f = 0.0;  // beta or -alpha
    if constexpr (IN == kCgDirection)
    {
        if (!CgStep(in.step, sh, f))
            return;
    }
    if constexpr (IN == kBicgDirection)
    {
        if (!BicgStep(in.step, sh, f))
            return;
    }
    if constexpr (IN == kBicgHalfStep)
    {
        const int status = st->status;
        const double rho = st->rho;
        double rv[1];
        SumPartials<1, kSpmvBlocks>(in.dotPart, in.nDot, rv, sh);
        if (status != kRunning)
            return;
        const double alpha = rho / rv[0];
        if (blockIdx.x == 0 && threadIdx.x == 0)
            st->alpha = alpha;
        f = -alpha;
    }
    auto entry = [&](int j) {
        if constexpr (IN == kStored)
            return x[j];
        else if constexpr (IN == kCgDirection)
            return fma(f, in.x2[j], in.x[j]);
        else
            return in.invd[j] * fma(f, in.x2[j], in.x[j]);
    };
    for (; p < nNodes; p += step)
    {
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
        const Head h = now;
        // this lane's row of y after the exchanges
        const int row = l < C0 ? C0 * p + l : nU + p;
        const bool dep = mask && ((mask[p] >> (l & 7)) & 1);
        const bool formsD = IN == kCgDirection || IN == kBicgHalfStep;  // d is the formed vector
        const double dr = DOTS != kNoDots && !formsD && l < F ? d[row] : 0.0;
        const double ov = IN != kStored && l < F ? fma(f, in.x2[row], in.x[row]) : 0.0;
        const double dv = formsD ? ov : dr;
        double xa = 0.0, xb = 0.0, wa[F], wb[F];
        if (h.L > 0)
        {
            xa = entry(ca);
            xb = entry(cb);
#pragma unroll
            for (int i = 0; i < F; i++)
            {
                wa[i] = va[i];
                wb[i] = vb[i];
            }
        }
        now = next;
        if (p + step < nNodes && now.L > 0)
            load(now);
        next = head(p + 2 * step);
        if (h.L > 0)
        {
#pragma unroll
            for (int i = 0; i < F; i++)
            {
                acc[i] = l < h.L ? wa[i] * xa : 0.0;
                acc[i] = l + 64 < h.L ? acc[i] + wb[i] * xb : acc[i];
            }
        }
        for (int k = l + 128; k < h.L; k += 64)
        {
            const double xk = entry(col[h.r0 + k]);
#pragma unroll
            for (int i = 0; i < C0; i++)
                acc[i] += val[h.r0 + i * h.L + k] * xk;
            if constexpr (C1 == 1)
                acc[C0] += val[h.re + k] * xk;
        }
        // lanes with l & 1 keep rows 1, 3, the others rows 0, 2; then l & 2 selects between the two
        double a;
        {
            const bool odd = l & 1;
            a = (odd ? acc[1] : acc[0]) + LaneDpp<kDppXor1>(odd ? acc[0] : acc[1]);
            if constexpr (F > 2)
            {
                const double b = (odd ? acc[3] : acc[2]) + LaneDpp<kDppXor1>(odd ? acc[2] : acc[3]);
                const bool hi = l & 2;
                a = (hi ? b : a) + LaneDpp<kDppXor2>(hi ? a : b);
            }
            else
                a += LaneDpp<kDppXor2>(a);
            a = QuadLaneSum(a);
        }
        if (l < F)
        {
            a = dep ? 0.0 : a;
            y[row] = a;
            if constexpr (IN != kStored)
                in.own[row] = ov;
            if constexpr (DOTS == kOneDot)
                dots[0] += a * dv;
            if constexpr (DOTS == kTwoDots)
            {
                dots[0] += a * a;
                dots[1] += a * dv;
            }
        }
    }
    if constexpr (DOTS != kNoDots)
        StorePartials<DOTS>(dots, part, sh);
}

// the dots of a finished product y (the path with constraint terms, whose C^T changes y after the
// K product)
template <int DOTS>
__global__ void __launch_bounds__(256) kSpmvDots(long long n, const double* __restrict__ y, const double* __restrict__ d,
                                                 double* __restrict__ part, const KrylovState* __restrict__ st)
{
    __shared__ double sh[8];
    if (st->status != kRunning)
        return;
    double v[2] = {0.0, 0.0};
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    {
        if constexpr (DOTS == kTwoDots)
        {
            v[0] += y[i] * y[i];
            v[1] += y[i] * d[i];
        }
        else
            v[0] += y[i] * d[i];
    }
    StorePartials<DOTS>(v, part, sh);
}

// The constraint equations on full-length vectors. Dependent dof dep[q] of equation q is
// sum val x[dof] over terms [ptr[q], ptr[q + 1]) (coefficients of C, signs included); indDof are the
// independent dofs that appear in terms, with the equations they appear in.
struct ConstraintView
{
    int nEq = 0, nTermDofs = 0;
    const int* dep = nullptr;
    const int* ptr = nullptr;     // per equation: its terms
    const int* dof = nullptr;
    const double* val = nullptr;
    const int* tDof = nullptr;    // independent dofs with terms
    const int* tPtr = nullptr;    // per such dof: the dependent dofs whose rows it collects
    const int* tDep = nullptr;
    const double* tVal = nullptr;
};

// C on a full-length vector: the dependent entries from the independent ones
__global__ void __launch_bounds__(256) kFillDependent(ConstraintView c, double* __restrict__ x)
{
    const int q = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (q >= c.nEq)
        return;
    double s = 0.0;
    for (int k = c.ptr[q]; k < c.ptr[q + 1]; k++)
        s += c.val[k] * x[c.dof[k]];
    x[c.dep[q]] = s;
}

// C^T on a full-length vector, first part: the dependent rows added to the terms' dofs
__global__ void __launch_bounds__(256) kCollectDependent(ConstraintView c, double* __restrict__ y)
{
    const int j = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (j >= c.nTermDofs)
        return;
    double s = y[c.tDof[j]];
    for (int k = c.tPtr[j]; k < c.tPtr[j + 1]; k++)
        s += c.tVal[k] * y[c.tDep[k]];
    y[c.tDof[j]] = s;
}

// second part: zeros at the dependent dofs
__global__ void __launch_bounds__(256) kClearDependent(ConstraintView c, double* __restrict__ y)
{
    const int q = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (q < c.nEq)
        y[c.dep[q]] = 0.0;
}

// invd[i] = 1 / diag(C^T K C) at the independent dofs (1 where the diagonal is zero), 0 at the
// dependent ones. diag of column j of C = sum over its entries (a, c_a), (b, c_b) of c_a c_b K(a, b)
// (column j of C = row j of C^T; K's columns are ascending in every row: binary search)
__global__ void __launch_bounds__(256) kInvDiag(int n, const int* __restrict__ rev, const int* __restrict__ ctRow,
                                                const int* __restrict__ ctCol, const double* __restrict__ ctVal,
                                                const int* __restrict__ kRow, const int* __restrict__ kCol,
                                                const double* __restrict__ kVal, double* __restrict__ invd)
{
    const int i = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (i >= n)
        return;
    const int j = rev[i];
    if (j < 0)
    {
        invd[i] = 0.0;
        return;
    }
    double s = 0.0;
    for (int p = ctRow[j]; p < ctRow[j + 1]; p++)
    {
        const int a = ctCol[p];
        for (int q = ctRow[j]; q < ctRow[j + 1]; q++)
        {
            const int b = ctCol[q];
            int lo = kRow[a], hi = kRow[a + 1];
            while (lo < hi)
            {
                const int mid = (lo + hi) >> 1;
                if (kCol[mid] < b)
                    lo = mid + 1;
                else
                    hi = mid;
            }
            if (lo < kRow[a + 1] && kCol[lo] == b)
                s += ctVal[p] * ctVal[q] * kVal[lo];
        }
    }
    invd[i] = s != 0.0 ? 1.0 / s : 1.0;
}

// (C^T f)_i at independent dof i (row j = rev[i] of C^T), 0 at a dependent one
__device__ inline double CtRow(int i, const int* __restrict__ rev, const int* __restrict__ ctRow,
                               const int* __restrict__ ctCol, const double* __restrict__ ctVal,
                               const double* __restrict__ f)
{
    const int j = rev[i];
    if (j < 0)
        return 0.0;
    double s = 0.0;
    for (int k = ctRow[j]; k < ctRow[j + 1]; k++)
        s += ctVal[k] * f[ctCol[k]];
    return s;
}

// partial sums of |C^T f|^2
__global__ void __launch_bounds__(256) kReducedNorm(int n, const int* __restrict__ rev, const int* __restrict__ ctRow,
                                                    const int* __restrict__ ctCol, const double* __restrict__ ctVal,
                                                    const double* __restrict__ f, double* __restrict__ part)
{
    __shared__ double sh[8];
    double v[1] = {0.0};
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    {
        const double b = CtRow((int)i, rev, ctRow, ctCol, ctVal, f);
        v[0] += b * b;
    }
    StorePartials<1>(v, part, sh);
}

// one block: out[0 .. N) = the sums of the partials
template <int N>
__global__ void __launch_bounds__(256) kSumPartials(int np, const double* __restrict__ part, double* __restrict__ out)
{
    __shared__ double sh[8];
    double v[N];
    SumPartials<N, kDotBlocks>(part, np, v, sh);
    if (threadIdx.x == 0)
    {
#pragma unroll
        for (int i = 0; i < N; i++)
            out[i] = v[i];
    }
}

// out[N][gridDim.x] = the sums of consecutive runs of the K product's partials part[N][np]
template <int N>
__global__ void __launch_bounds__(256) kFoldPartials(int np, const double* __restrict__ part, double* __restrict__ out,
                                                     const KrylovState* __restrict__ st)
{
    __shared__ double sh[8];
    if (st->status != kRunning)
        return;
    const int run = (np + (int)gridDim.x - 1) / (int)gridDim.x;
    const int beg = (int)blockIdx.x * run, end = beg + run < np ? beg + run : np;
    double v[N];
#pragma unroll
    for (int i = 0; i < N; i++)
    {
        v[i] = 0.0;
        for (int k = beg + (int)threadIdx.x; k < end; k += 256)
            v[i] += part[(size_t)i * np + k];
    }
    StorePartials<N>(v, out, sh);
}

// Start of a solve from x = 0: b = C^T f, r = b, and for BiCGSTAB r0 = b, p = v = 0 with the partials
// of (r . r) and (r0 . r), for CG z = invd b with those of (r . r) and (r . z); the state
template <bool CG>
__global__ void __launch_bounds__(256) kKrylovStart(int n, const int* __restrict__ rev, const int* __restrict__ ctRow,
                                                    const int* __restrict__ ctCol, const double* __restrict__ ctVal,
                                                    const double* __restrict__ f, const double* __restrict__ invd,
                                                    double* __restrict__ b, double* __restrict__ x, double* __restrict__ r,
                                                    double* __restrict__ r0, double* __restrict__ p,
                                                    double* __restrict__ v, double* __restrict__ part,
                                                    KrylovState* __restrict__ st)
{
    __shared__ double sh[8];
    double s[2] = {0.0, 0.0};
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    {
        const double bi = CtRow((int)i, rev, ctRow, ctCol, ctVal, f);
        x[i] = 0.0;
        r[i] = bi;
        p[i] = 0.0;
        if constexpr (CG)
        {
            const double zi = invd[i] * bi;
            r0[i] = zi;  // CG: the preconditioned residual z
            s[1] += bi * zi;
        }
        else
        {
            b[i] = bi;
            r0[i] = bi;
            v[i] = 0.0;
            s[1] += bi * bi;
        }
        s[0] += bi * bi;
    }
    StorePartials<2>(s, part, sh);
    if (blockIdx.x == 0 && threadIdx.x == 0)
        st[0] = KrylovState{0.0, 0.0, 1.0, 1.0, 1.0, 0.0, kRunning, 0};
}

// First kernel of CG iteration `it` where the K product does not begin the iteration itself: p = z + beta p.
// `check`: the test alone (after the last iteration that the caller allows).
__global__ void __launch_bounds__(256) kCgP(int n, const StepArgs a, const double* __restrict__ z, double* __restrict__ p)
{
    __shared__ double sh[8];
    double beta;
    if (!CgStep(a, sh, beta) || a.check)
        return;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
        p[i] = fma(beta, p[i], z[i]);
}

// CG's alpha = (r . z) / (p . q), x += alpha p, r -= alpha q, z = invd r, and the partials of (r . r)
// and (r . z)
__global__ void __launch_bounds__(256) kCgUpdate(int n, const double* __restrict__ dotPart, int np,
                                                 const double* __restrict__ p, const double* __restrict__ q,
                                                 double* __restrict__ x, double* __restrict__ r,
                                                 const double* __restrict__ invd, double* __restrict__ z,
                                                 double* __restrict__ part, const KrylovState* __restrict__ st)
{
    __shared__ double sh[8];
    // the operands of a lane's first entry are in flight while the block adds the partials
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long i0 = i < n ? i : n - 1;
    double pi = p[i0], qi = q[i0], xi = x[i0], ri = r[i0], di = invd[i0];
    const int status = st->status;
    const double rho = st->rho;
    double pq[1];
    SumPartials<1, kSpmvBlocks>(dotPart, np, pq, sh);
    if (status != kRunning)
        return;
    const double alpha = rho / pq[0];
    double s[2] = {0.0, 0.0};
    while (i < n)
    {
        x[i] = fma(alpha, pi, xi);
        ri = fma(-alpha, qi, ri);
        r[i] = ri;
        const double zi = di * ri;
        z[i] = zi;
        s[0] = fma(ri, ri, s[0]);
        s[1] = fma(ri, zi, s[1]);
        i += (long long)gridDim.x * 256;
        if (i < n)
        {
            pi = p[i];
            qi = q[i];
            xi = x[i];
            ri = r[i];
            di = invd[i];
        }
    }
    StorePartials<2>(s, part, sh);
}

// First kernel of a BiCGSTAB iteration where the K product does not begin it itself: p = r + beta (p - w v),
// y = invd p. check: the tests alone.
__global__ void __launch_bounds__(256) kBicgP(int n, const StepArgs a, const double* __restrict__ r,
                                              const double* __restrict__ v, const double* __restrict__ invd,
                                              double* __restrict__ p, double* __restrict__ y)
{
    __shared__ double sh[8];
    double beta;
    const double w = a.st[a.seq & 1].w;
    if (!BicgStep(a, sh, beta) || a.check)
        return;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    {
        const double pi = fma(beta, fma(-w, v[i], p[i]), r[i]);
        p[i] = pi;
        y[i] = invd[i] * pi;
    }
}

// BiCGSTAB's alpha = rho / (r0 . v), s = r - alpha v, z = invd s
__global__ void __launch_bounds__(256) kBicgS(int n, const double* __restrict__ dotPart, int np,
                                              const double* __restrict__ r, const double* __restrict__ v,
                                              const double* __restrict__ invd, double* __restrict__ s,
                                              double* __restrict__ z, KrylovState* __restrict__ st)
{
    __shared__ double sh[8];
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long i0 = i < n ? i : n - 1;
    double vi = v[i0], ri = r[i0], di = invd[i0];
    const int status = st->status;
    const double rho = st->rho;
    double d[1];
    SumPartials<1, kSpmvBlocks>(dotPart, np, d, sh);
    if (status != kRunning)
        return;
    const double alpha = rho / d[0];
    if (blockIdx.x == 0 && threadIdx.x == 0)
        st->alpha = alpha;
    while (i < n)
    {
        const double si = fma(-alpha, vi, ri);
        s[i] = si;
        z[i] = di * si;
        i += (long long)gridDim.x * 256;
        if (i < n)
        {
            vi = v[i];
            ri = r[i];
            di = invd[i];
        }
    }
}

// BiCGSTAB's w = (t . s) / (t . t) (0 when t = 0), x += alpha y + w z, r = s - w t, and the partials of
// (r . r) and (r0 . r). FORM: y = invd p and z = invd s are formed here, and h = p - w v is left for the
// next direction.
template <bool FORM>
__global__ void __launch_bounds__(256) kBicgUpdate(int n, const double* __restrict__ dotPart, int np,
                                                   const double* __restrict__ y, const double* __restrict__ z,
                                                   double* __restrict__ x, const double* __restrict__ s,
                                                   const double* __restrict__ t, double* __restrict__ r,
                                                   const double* __restrict__ r0, double* __restrict__ part,
                                                   KrylovState* __restrict__ st, const double* __restrict__ invd,
                                                   const double* __restrict__ p, const double* __restrict__ v,
                                                   double* __restrict__ h)
{
    __shared__ double sh[8];
    // the operands of a lane's first entry are in flight while the block adds the partials
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long i0 = i < n ? i : n - 1;
    double si = s[i0], ti = t[i0], xi = x[i0], r0i = r0[i0];
    double a = FORM ? p[i0] : y[i0], b = FORM ? v[i0] : z[i0], di = FORM ? invd[i0] : 0.0;
    const int status = st->status;
    const double alpha = st->alpha;
    double d[2];
    SumPartials<2, kSpmvBlocks>(dotPart, np, d, sh);
    if (status != kRunning)
        return;
    const double w = d[0] > 0.0 ? d[1] / d[0] : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0)
        st->w = w;
    double q[2] = {0.0, 0.0};
    while (i < n)
    {
        const double yi = FORM ? di * a : a, zi = FORM ? di * si : b;
        if constexpr (FORM)
            h[i] = fma(-w, b, a);
        x[i] = fma(w, zi, fma(alpha, yi, xi));
        const double ri = fma(-w, ti, si);
        r[i] = ri;
        q[0] = fma(ri, ri, q[0]);
        q[1] = fma(r0i, ri, q[1]);
        i += (long long)gridDim.x * 256;
        if (i < n)
        {
            si = s[i];
            ti = t[i];
            xi = x[i];
            r0i = r0[i];
            a = FORM ? p[i] : y[i];
            b = FORM ? v[i] : z[i];
            di = FORM ? invd[i] : 0.0;
        }
    }
    StorePartials<2>(q, part, sh);
}

// BiCGSTAB restart: r = r0 = b - t (t = A x) and the partials of (r . r), twice (rho = (r0 . r))
__global__ void __launch_bounds__(256) kBicgRestart(int n, const double* __restrict__ b, const double* __restrict__ t,
                                                    double* __restrict__ r, double* __restrict__ r0,
                                                    double* __restrict__ part)
{
    __shared__ double sh[8];
    double q[2] = {0.0, 0.0};
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    {
        const double ri = b[i] - t[i];
        r[i] = ri;
        r0[i] = ri;
        q[0] += ri * ri;
        q[1] += ri * ri;
    }
    StorePartials<2>(q, part, sh);
}

// y = a x + b y (x, y of length n); a zero factor leaves its operand unread (y = 0 with a = b = 0)
__global__ void __launch_bounds__(256) kAxpby(long long n, double a, const double* __restrict__ x, double b,
                                              double* __restrict__ y)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n)
        y[i] = (a == 0.0 ? 0.0 : a * x[i]) + (b == 0.0 ? 0.0 : b * y[i]);
}

// delta[dep[e]] = rhsNew[e] - rhsOld[e] (dependent dofs are distinct)
__global__ void __launch_bounds__(256) kScatterDelta(int nEq, const int* __restrict__ dep,
                                                     const double* __restrict__ rhsOld,
                                                     const double* __restrict__ rhsNew, double* __restrict__ delta)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e < nEq)
        delta[dep[e]] = rhsNew[e] - (rhsOld ? rhsOld[e] : 0.0);
}

// Device CSR view
struct Csr
{
    int nRows = 0;
    const int* row = nullptr;
    const int* col = nullptr;
    const double* val = nullptr;
};

// node structure of an assembled K (rows per node of field 0 and 1), for the node product
struct NodeRows
{
    int nNodes = 0, nU = 0, c0 = 0, c1 = 0;
};

// What the caller keeps between solves on one stream: the vectors, the states, and the pinned copies of
// the states that the host reads with the events that say when they have arrived
struct SolveBuffers
{
    double* work = nullptr;          // ReducedSolver::WorkDoubles
    KrylovState* host = nullptr;     // 2, pinned
    hipEvent_t arrived[2] = {nullptr, nullptr};
};

// Krylov solver on the operator C^T K C in full-length form
class ReducedSolver
{
public:
    // doubles of the workspace: 11 vectors of a solve (x and the preconditioner's diagonal included) and
    // 2 of its caller, the partial sums of the vector kernels and of the K product, the two states, and the
    // partials of one block per four nodes (a node has two rows at least)
    static size_t WorkDoubles(long long n)
    {
        return 13 * (size_t)n + 2 * kDotBlocks + 2 * kSpmvBlocks + 32 + (n >= kFoldRows ? 2 * (size_t)(n / 8 + 1) : 0);
    }
    ReducedSolver(hipStream_t s, Csr K, Csr Ct, const int* rev, const unsigned char* mask, ConstraintView cons,
                  NodeRows nodes, const SolveBuffers& buf)
        : mS(s), mK(K), mCt(Ct), mRev(rev), mMask(mask), mCons(cons), mN(K.nRows), mNodes(nodes), mBuf(buf)
    {
        vecs = buf.work;
        part = vecs + 13 * (size_t)mN;
        dotPart = part + 2 * kDotBlocks;
        state = reinterpret_cast<KrylovState*>(dotPart + 2 * kSpmvBlocks);
        blockPart = dotPart + 2 * kSpmvBlocks + 32;
        const bool known = (nodes.c0 == 3 && nodes.c1 <= 1) || (nodes.c0 == 2 && nodes.c1 == 0);
        mNode = nodes.nNodes > 0 && known;
        mFused = mNode && cons.nTermDofs == 0;
    }
    // vector k of the workspace: x (the result of Solve) is 0, 10 and 11 are the caller's
    double* Vec(int k) const
    {
        return vecs + (size_t)k * mN;
    }

    // y = K x (no constraints)
    void SpmvK(const double* x, double* y)
    {
        Product<kNoDots>(x, y, nullptr, nullptr, nullptr);
    }
    void Axpby(long long n, double a, const double* x, double b, double* y)
    {
        if (n > 0)
            hipLaunchKernelGGL(kAxpby, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, mS, n, a, x, b, y);
    }
    // |C^T v|^2 (one host read)
    double ReducedNorm2(const double* v, hipError_t& err)
    {
        if (mN == 0)
            return 0.0;
        const int g = Grid();
        double* out = reinterpret_cast<double*>(state);
        hipLaunchKernelGGL(kReducedNorm, dim3(g), dim3(256), 0, mS, mN, mRev, mCt.row, mCt.col, mCt.val, v, part);
        hipLaunchKernelGGL(kSumPartials<1>, dim3(1), dim3(256), 0, mS, g, part, out);
        if ((err = hipGetLastError()) != hipSuccess ||
            (err = hipMemcpyAsync(mBuf.host, out, sizeof(double), hipMemcpyDeviceToHost, mS)) != hipSuccess ||
            (err = hipStreamSynchronize(mS)) != hipSuccess)
            return 0.0;
        return mBuf.host[0].rr;
    }

    // The solve from x = 0 with right-hand side C^T f: x = C u in Vec(0). CG: stops when
    // |r|^2 < tol^2 |b|^2, `iters` counts the iterations before the converging one; BiCGSTAB: when
    // !(|r|^2 > tol^2 |b|^2). Both after maxIt iterations at the latest.
    hipError_t Solve(bool cg, const double* f, double tol, int maxIt, int& iters, double& relRes)
    {
        iters = 0;
        relRes = 0.0;
        if (mN == 0)
            return hipSuccess;
        double *x = Vec(0), *invd = Vec(1), *b = Vec(2), *R = Vec(3), *R0 = Vec(4), *P = Vec(5), *V = Vec(6),
               *Y = Vec(7), *Z = Vec(8), *T = Vec(9);
        double* S = Vec(12);
        const dim3 g((unsigned)Grid()), blk(256);
        const int np = Grid();
        const double tol2 = tol * tol;
        hipLaunchKernelGGL(kInvDiag, dim3((unsigned)((mN + 255) / 256)), blk, 0, mS, mN, mRev, mCt.row, mCt.col,
                           mCt.val, mK.row, mK.col, mK.val, invd);
        const bool formed = Formed();
        double* H = Y;  // BiCGSTAB, formed: p - w v
        if (cg)
            hipLaunchKernelGGL(kKrylovStart<true>, g, blk, 0, mS, mN, mRev, mCt.row, mCt.col, mCt.val, f, invd, b, x, R,
                               R0, P, V, part, state);
        else
            hipLaunchKernelGGL(kKrylovStart<false>, g, blk, 0, mS, mN, mRev, mCt.row, mCt.col, mCt.val, f, invd, b, x,
                               R, R0, formed ? H : P, V, part, state);
        int it = 0, seq = 0, restarts = 0, queued = 0;
        bool first = true, forced = false;
        KrylovState last{};
        hipError_t err = hipGetLastError();
        while (err == hipSuccess)
        {
            // a chunk of iterations, then the test alone once the caller's limit is reached
            const int end = std::min(it + kSolveChunk, maxIt);
            for (; it < end; it++, seq++)
            {
                KrylovState* st = state + ((seq + 1) & 1);
                KrylovState* tell = it + 1 == end && end < maxIt ? mBuf.host + (queued & 1) : nullptr;
                const StepArgs step{seq, it, first, forced, false, tol2, part, np, state, tell};
                first = forced = false;
                if (cg)
                {
                    double* p = P;
                    int nd;
                    if (formed)
                    {
                        // the product reads the last p at other rows than it writes: two copies in turn
                        double* old = it & 1 ? Y : P;
                        p = it & 1 ? P : Y;
                        nd = NodeProduct<kOneDot, kCgDirection>(nullptr, V, mMask, nullptr, dotPart, st,
                                                                {R0, old, nullptr, p, step, nullptr, 0});
                    }
                    else
                    {
                        hipLaunchKernelGGL(kCgP, g, blk, 0, mS, mN, step, R0, P);
                        nd = Product<kOneDot>(P, V, P, st, dotPart);
                    }
                    hipLaunchKernelGGL(kCgUpdate, g, blk, 0, mS, mN, dotPart, nd, p, V, x, R, invd, R0, part, st);
                    continue;
                }
                if (formed)
                {
                    double* part2 = Z;  // 2 sums per block; dotPart is read by the kernel that writes these
                    int nd = NodeProduct<kOneDot, kBicgDirection>(nullptr, V, mMask, R0, dotPart, st,
                                                                  {R, H, invd, P, step, nullptr, 0});
                    nd = NodeProduct<kTwoDots, kBicgHalfStep>(nullptr, T, mMask, nullptr, part2, st,
                                                              {R, V, invd, S, {}, dotPart, nd});
                    hipLaunchKernelGGL(kBicgUpdate<true>, g, blk, 0, mS, mN, part2, nd, nullptr, nullptr, x, S, T, R, R0,
                                       part, st, invd, P, V, H);
                    continue;
                }
                hipLaunchKernelGGL(kBicgP, g, blk, 0, mS, mN, step, R, V, invd, P, Y);
                int nd = Product<kOneDot>(Y, V, R0, st, dotPart);
                hipLaunchKernelGGL(kBicgS, g, blk, 0, mS, mN, dotPart, nd, R, V, invd, S, Z, st);
                nd = Product<kTwoDots>(Z, T, S, st, dotPart);
                hipLaunchKernelGGL(kBicgUpdate<false>, g, blk, 0, mS, mN, dotPart, nd, Y, Z, x, S, T, R, R0, part, st,
                                   nullptr, nullptr, nullptr, nullptr);
            }
            const bool atEnd = it >= maxIt;
            if (atEnd)
            {
                const StepArgs step{seq, it, first, forced, true, tol2, part, np, state, mBuf.host + (queued & 1)};
                if (cg)
                    hipLaunchKernelGGL(kCgP, dim3(1), blk, 0, mS, mN, step, R0, P);
                else
                    hipLaunchKernelGGL(kBicgP, dim3(1), blk, 0, mS, mN, step, R, V, invd, P, Y);
                seq++;
            }
            const int slot = queued & 1;
            if ((err = hipGetLastError()) != hipSuccess ||
                (err = hipEventRecord(mBuf.arrived[slot], mS)) != hipSuccess)
                break;
            queued++;
            // the state of the chunk before this one, or of this one where nothing more can be queued
            const int read = atEnd ? slot : 1 - slot;
            if (queued == 1 && !atEnd)
                continue;
            if ((err = hipEventSynchronize(mBuf.arrived[read])) != hipSuccess)
                break;
            last = mBuf.host[read];
            if (last.status == kDone)
                break;
            if (last.status == kRestart)
            {
                // the launches queued after the test returned at once: wait for them, then restart with the
                // current residual r = b - A x at the iteration that was not begun
                if ((err = hipStreamSynchronize(mS)) != hipSuccess)
                    break;
                it = last.iters;
                if (restarts++ == 0)
                    it = 0;
                Operator(x, T);
                hipLaunchKernelGGL(kBicgRestart, g, blk, 0, mS, mN, b, T, R, R0, part);
                forced = true;
                queued = 0;
                if (it < maxIt)
                    continue;
            }
            if (atEnd)
                break;
        }
        // the pinned states must not be written after this returns
        const hipError_t end = hipStreamSynchronize(mS);
        if (err == hipSuccess)
            err = end;
        iters = last.iters;
        relRes = last.bb > 0.0 || last.bb != last.bb ? std::sqrt(last.rr / last.bb) : 0.0;
        if (cg && last.status == kDone && last.iters == 0 && last.rr == last.bb)
            relRes = 0.0;  // converged before the first iteration
        return err;
    }

private:
    int Grid() const
    {
        return std::max(1, std::min(kDotBlocks, (mN + 255) / 256));
    }
    // whether the K products form the vectors they multiply
    bool Formed() const
    {
        const char* v = std::getenv("NUTO_AMD_SOLVE_FORM");  // 0 / 1: never / wherever possible (tests)
        if (!mFused || (v && v[0] == '0'))
            return false;
        return (v && v[0] == '1') || mNodes.nNodes <= kFormNodes;
    }
    // y = C^T K C x for a full-length x whose dependent entries this fills
    void Operator(double* x, double* y)
    {
        if (mFused)
            NodeProduct<kNoDots, kStored>(x, y, mMask, nullptr, nullptr, nullptr);
        else
            Constrained(x, y);
    }
    void Constrained(double* x, double* y)
    {
        const ConstraintView& c = mCons;
        const dim3 ge((unsigned)((c.nEq + 255) / 256)), gt((unsigned)((c.nTermDofs + 255) / 256)), blk(256);
        if (c.nEq > 0)
            hipLaunchKernelGGL(kFillDependent, ge, blk, 0, mS, c, x);
        Product<kNoDots>(x, y, nullptr, nullptr, nullptr);
        if (c.nTermDofs > 0)
            hipLaunchKernelGGL(kCollectDependent, gt, blk, 0, mS, c, y);
        if (c.nEq > 0)
            hipLaunchKernelGGL(kClearDependent, ge, blk, 0, mS, c, y);
    }
    // DOTS: the operator C^T K C with the dots' partials in `out`, their number returned; kNoDots: K alone
    template <int DOTS>
    int Product(const double* x, double* y, const double* d, KrylovState* st, double* out)
    {
        if constexpr (DOTS == kNoDots)
        {
            if (mNode)
                NodeProduct<kNoDots, kStored>(x, y, nullptr, nullptr, nullptr, nullptr);
            else if (mN > 0)
                hipLaunchKernelGGL(kCsrSpmv, dim3((unsigned)(((long long)mN * 16 + 255) / 256)), dim3(256), 0, mS, mN,
                                   mK.row, mK.col, mK.val, x, y);
            return 0;
        }
        else
        {
            if (mFused)
                return NodeProduct<DOTS, kStored>(x, y, mMask, d, out, st);
            Constrained(const_cast<double*>(x), y);
            hipLaunchKernelGGL(kSpmvDots<DOTS>, dim3((unsigned)Grid()), dim3(256), 0, mS, (long long)mN, y, d, out, st);
            return Grid();
        }
    }
    template <int DOTS, int IN>
    int NodeProduct(const double* x, double* y, const unsigned char* mask, const double* d, double* out,
                    KrylovState* st, const FormedInput& in = {})
    {
        const NodeRows& nr = mNodes;
        const int all = (nr.nNodes + 3) / 4;
        const bool fold = IN == kStored && mN >= kFoldRows;
        const int g = fold ? all : std::min(kSpmvBlocks, all);
        double* const sums = out;
        if (fold && DOTS != kNoDots)
            out = blockPart;
        const dim3 grid((unsigned)g), block(256);
        if (nr.c0 == 3 && nr.c1 == 1)
            hipLaunchKernelGGL((kNodeSpmv<3, 1, DOTS, IN>), grid, block, 0, mS, nr.nNodes, nr.nU, mK.row, mK.col, mK.val, x,
                               y, mask, d, out, st, in);
        else if (nr.c0 == 3)
            hipLaunchKernelGGL((kNodeSpmv<3, 0, DOTS, IN>), grid, block, 0, mS, nr.nNodes, nr.nU, mK.row, mK.col, mK.val, x,
                               y, mask, d, out, st, in);
        else
            hipLaunchKernelGGL((kNodeSpmv<2, 0, DOTS, IN>), grid, block, 0, mS, nr.nNodes, nr.nU, mK.row, mK.col, mK.val, x,
                               y, mask, d, out, st, in);
        if constexpr (DOTS != kNoDots)
        {
            if (fold)
            {
                hipLaunchKernelGGL(kFoldPartials<DOTS>, dim3(kFoldBlocks), block, 0, mS, g, blockPart, sums, st);
                return kFoldBlocks;
            }
        }
        return g;
    }

    hipStream_t mS;
    Csr mK, mCt;
    const int* mRev;
    const unsigned char* mMask;
    ConstraintView mCons;
    int mN;
    NodeRows mNodes;
    SolveBuffers mBuf;
    bool mNode = false, mFused = false;
    double *vecs = nullptr, *part = nullptr, *dotPart = nullptr, *blockPart = nullptr;
    KrylovState* state = nullptr;
};

}  // namespace nuto_amd
