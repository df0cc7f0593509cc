// Set-up and launches of the hex8 gradient-damage kernels (gdm_plan.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <vector>

#include "gdm_hex8.hpp"
#include "gdm_hex8_vectors.hpp"
#include "gdm_plan.hpp"

namespace nuto_amd
{

bool GdmHex8Plan::Prepare(int kind, int coordType, int dofType, int nip, const NodeGraph& g, int nCells,
             int nCoord, const double* x, const double* y, const double* z, const int* cconn, const double* tab,
             const int* rowPtr, int nRows, bool decreasingInteraction, hipStream_t stream, hipError_t& err)
{
    Release();
    err = hipSuccess;
    if (kind != kGradientDamage || coordType != kHex8 || dofType != kHex8 || nip != 8)
        return false;
    const int n = g.nNodes;
    if (nRows != 4 * n)  // 3 displacement rows and 1 eeq row per node
        return false;
    // nodes beyond the kernel's bounds stay out of the tables (the generic kernel assembles them)
    std::vector<char> out(n, 0);
    std::vector<int> extraNodes;
    for (int p = 0; p < n; p++)
    {
        if (g.incPtr[p + 1] - g.incPtr[p] > gdm8::kMaxInc || g.adjPtr[p + 1] - g.adjPtr[p] > gdm8::kMaxAdj)
        {
            out[p] = 1;
            extraNodes.push_back(p);
        }
    }
    if (n > 0 && (int)extraNodes.size() == n)
        return false;
    // traversal order: position s holds node ord[s]
    std::vector<int> ord(n);
    bool reordered = false;
    const char* ordEnv = std::getenv("NUTO_AMD_GDM_ORDER");
    if (n > 0 && nCells > 0 && !(ordEnv && ordEnv[0] == '0'))
    {
        if ((err = MortonOrder(g, nCells, nCoord, x, y, z, cconn, stream, ord)) != hipSuccess)
            return false;
        reordered = true;
    }
    else
    {
        for (int s = 0; s < n; s++)
            ord[s] = s;
    }
    if (!extraNodes.empty())
    {
        // drop the outside nodes from the traversal; they keep position -1
        ord.erase(std::remove_if(ord.begin(), ord.end(), [&](int p) { return out[p] != 0; }), ord.end());
        reordered = true;
    }
    const int nIn = (int)ord.size();
    // CSR rows: displacement rows 3p .. 3p + 2, eeq row 3n + p
    std::vector<int> rp((size_t)4 * n + 1);
    if ((err = hipMemcpyAsync(rp.data(), rowPtr, rp.size() * sizeof(int), hipMemcpyDeviceToHost, stream)) !=
            hipSuccess ||
        (err = hipStreamSynchronize(stream)) != hipSuccess)
        return false;
    std::vector<int4> head(nIn);
    std::vector<int> cell((size_t)nIn * 8, -1), pos(reordered ? n : 0, -1);
    std::vector<unsigned char> la((size_t)nIn * 8, 0), slot((size_t)nIn * 64, 0);
    for (int s = 0; s < nIn; s++)
    {
        const int p = ord[s];
        head[s] = make_int4(p, rp[(size_t)3 * p], rp[(size_t)3 * p + 1] - rp[(size_t)3 * p], rp[(size_t)3 * n + p]);
        if (reordered)
            pos[p] = s;
        for (int k = g.incPtr[p], r = 0; k < g.incPtr[p + 1]; k++, r++)
        {
            const size_t pr = (size_t)s * 8 + r;
            cell[pr] = g.incCell[k];
            la[pr] = g.incLocal[k];
            for (int j = 0; j < 8; j++)
                slot[pr * 8 + j] = (unsigned char)(g.slot[(size_t)k * 8 + j] & 0x7fff);
        }
    }
    if ((err = nodeHead.Upload(head.data(), head.size() * sizeof(int4), stream)) != hipSuccess ||
        (reordered && (err = posOf.Upload(pos.data(), pos.size() * sizeof(int), stream)) != hipSuccess) ||
        (err = nodeCell.Upload(cell.data(), cell.size() * sizeof(int), stream)) != hipSuccess ||
        (err = nodeLa.Upload(la.data(), la.size(), stream)) != hipSuccess ||
        (!extraNodes.empty() &&
         (err = extra.Upload(extraNodes.data(), extraNodes.size() * sizeof(int), stream)) != hipSuccess) ||
        (err = nodeSlot.Upload(slot.data(), slot.size(), stream)) != hipSuccess ||
        (err = geo.Alloc((size_t)nCells * 8 * gdm8::kGeo * sizeof(double))) != hipSuccess)
    {
        Release();
        return false;
    }
    if (nCells > 0)
    {
        const long long items = (long long)nCells * 8;
        hipLaunchKernelGGL(kGdmHex8Geometry, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, stream, x, y,
                           z, cconn, tab, nCells, geo.As<double>());
        if ((err = hipGetLastError()) != hipSuccess || (err = hipStreamSynchronize(stream)) != hipSuccess)
        {
            Release();
            return false;
        }
    }
    const char* pre = std::getenv("NUTO_AMD_GDM_PREPASS");
    prepass = pre ? (pre[0] == '0' ? 0 : 1) : -1;
    const char* aff = std::getenv("NUTO_AMD_GDM_AFFINE");
    affine = false;
    if (nCells > 0 && !(aff && aff[0] == '0'))
    {
        DevBuf cnt;
        int h = -1;
        if ((err = cnt.Alloc(sizeof(int))) != hipSuccess ||
            (err = hipMemsetAsync(cnt.p, 0, sizeof(int), stream)) != hipSuccess)
        {
            Release();
            return false;
        }
        hipLaunchKernelGGL(kGdmHex8CountNonAffine, dim3((unsigned)((nCells + 255) / 256)), dim3(256), 0, stream,
                           geo.As<double>(), nCells, cnt.As<int>());
        if ((err = hipGetLastError()) != hipSuccess ||
            (err = hipMemcpyAsync(&h, cnt.p, sizeof(int), hipMemcpyDeviceToHost, stream)) != hipSuccess ||
            (err = hipStreamSynchronize(stream)) != hipSuccess)
        {
            Release();
            return false;
        }
        affine = h == 0;
        if (affine && ((err = geoCell.Alloc((size_t)nCells * gdm8::kGeo * sizeof(double))) != hipSuccess ||
                       (err = hipMemcpy2DAsync(geoCell.p, gdm8::kGeo * sizeof(double), geo.p,
                                               8 * gdm8::kGeo * sizeof(double), gdm8::kGeo * sizeof(double),
                                               nCells, hipMemcpyDeviceToDevice, stream)) != hipSuccess ||
                       (err = hipStreamSynchronize(stream)) != hipSuccess))
        {
            Release();
            return false;
        }
    }
    decreasing = decreasingInteraction;
    if ((err = ipState.Alloc((size_t)nCells * 8 * RecordDoubles() * sizeof(double))) != hipSuccess)
    {
        Release();
        return false;
    }
    this->nCells = nCells;
    nNodes = nIn;
    nExtra = (int)extraNodes.size();
    const char* env = std::getenv("NUTO_AMD_GDM_XCD_MAP");
    xcdMap = env ? std::atoi(env) : 1;
    grid = xcdMap ? (nNodes + 7) / 8 * 8 : nNodes;
    ready = true;
    return true;
}

template <bool FULLDMG, bool PRE, bool DEC>
static void LaunchNodes(const RowArgs& a, const GdmHex8Tables& t, bool affine, bool wr, int grid, hipStream_t stream)
{
    if (wr && affine)
        hipLaunchKernelGGL((kGdmHex8Node<true, FULLDMG, PRE, true, DEC>), dim3(grid), dim3(64), 0, stream, a, t);
    else if (wr)
        hipLaunchKernelGGL((kGdmHex8Node<true, FULLDMG, PRE, false, DEC>), dim3(grid), dim3(64), 0, stream, a, t);
    else if (affine)
        hipLaunchKernelGGL((kGdmHex8Node<false, FULLDMG, PRE, true, DEC>), dim3(grid), dim3(64), 0, stream, a, t);
    else
        hipLaunchKernelGGL((kGdmHex8Node<false, FULLDMG, PRE, false, DEC>), dim3(grid), dim3(64), 0, stream, a, t);
}

// all nodes of the plan; state: the pre-pass records' memory (nullptr: no pre-pass)
template <bool FULLDMG, bool DEC>
static void LaunchT(const GdmHex8Plan& plan, const RowArgs& a, bool wr, double* state, hipStream_t stream)
{
    GdmHex8Tables t = plan.Tables();
    if (!state)
    {
        LaunchNodes<FULLDMG, false, DEC>(a, t, plan.affine, wr, plan.grid, stream);
        return;
    }
    t.ipState = state;
    if (plan.nCells > 0)
    {
        const dim3 grid((unsigned)((plan.nCells + 7) / 8));
        if (plan.affine)
            hipLaunchKernelGGL((kGdmHex8Ip<FULLDMG, true, DEC>), grid, dim3(64), 0, stream, a, t, state);
        else
            hipLaunchKernelGGL((kGdmHex8Ip<FULLDMG, false, DEC>), grid, dim3(64), 0, stream, a, t, state);
    }
    LaunchNodes<FULLDMG, true, DEC>(a, t, plan.affine, wr, plan.grid, stream);
}

// A mesh whose nodes' workgroups are all on the chip at once (16 per CU) takes one launch without the
// pre-pass: its time is the latency of one workgroup, which the pre-pass would only precede. Measured, R + K,
// with / without pre-pass: 125 nodes 9.7 / 7.0 us, 3375 nodes 14.7 / 12.6 us (affine) and 16.0 / 12.5 us
// (jittered); 9261 nodes 24.4 / 24.1 and 28.2 / 24.7 us, 24,389 nodes 47.7 / 56.1 and 52.8 / 55.9 us.
constexpr int kOneLaunchNodes = 16 * 256;

void GdmHex8Plan::Launch(const RowArgs& a, bool wr, hipStream_t stream, double* state) const
{
    if (nNodes > 0)
    {
        const bool pre = prepass < 0 ? nNodes > kOneLaunchNodes : prepass != 0;
        double* records = !pre ? nullptr : (state ? state : Work());
        const bool full = a.P.damage_application == 0;
        if (full && decreasing)
            LaunchT<true, true>(*this, a, wr, records, stream);
        else if (full)
            LaunchT<true, false>(*this, a, wr, records, stream);
        else if (decreasing)
            LaunchT<false, true>(*this, a, wr, records, stream);
        else
            LaunchT<false, false>(*this, a, wr, records, stream);
    }
    LaunchExtras(a, wr, stream);
}

void GdmHex8Plan::LaunchExtras(const RowArgs& a, bool wr, hipStream_t stream) const
{
    if (nExtra > 0)
    {
        const dim3 grid((unsigned)((nExtra + 63) / 64));
        const int* list = extra.As<int>();
        if (wr)
            hipLaunchKernelGGL((kAssembleRowsList<kGradientDamage, 3, 8, 8, 8, 4, true, true>), grid, dim3(64), 0,
                               stream, a, list, nExtra);
        else
            hipLaunchKernelGGL((kAssembleRowsList<kGradientDamage, 3, 8, 8, 8, 4, false, true>), grid, dim3(64), 0,
                               stream, a, list, nExtra);
    }
}

void GdmHex8Plan::LaunchRange(const RowArgs& a, int first, int end, hipStream_t stream) const
{
    if (end <= first)
        return;
    GdmHex8Tables t = Tables();
    t.xcdMap = 0;
    t.pBegin = first;
    t.pEnd = end;
    t.order = posOf.p ? posOf.As<int>() : nullptr;  // launch index = node
    // without the pre-pass, which runs over all cells of the plan
    if (a.P.damage_application == 0)
        LaunchNodes<true, false, false>(a, t, affine, true, end - first, stream);
    else
        LaunchNodes<false, false, false>(a, t, affine, true, end - first, stream);
}

void GdmHex8Plan::LaunchVector(const RowArgs& a, double* vec, hipStream_t stream) const
{
    LaunchGdmHex8Vector<false>(*this, a, nullptr, vec, nullptr, Work(), stream);
}

void GdmHex8Plan::LaunchAdjoint(const RowArgs& a, const double* lam, double* vec, double* dtheta,
                                hipStream_t stream) const
{
    LaunchGdmHex8Vector<true>(*this, a, lam, vec, dtheta, Work(), stream);
}

}  // namespace nuto_amd
