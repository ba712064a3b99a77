// Host side of the C ABI declared in include/optcuts_gpu.h: context, HBM
// layout, sparsity-pattern and slot-map construction, and the
// device-resident Newton step. Kernels live in oc_kernels.hip.
#include "../../include/optcuts_gpu.h"
#include "oc_air_mesh.hpp"
#include "oc_amg.hpp"
#include "oc_amg_structure.hpp"
#include "oc_common.hpp"
#include "oc_gnn.hpp"
#include "oc_ic0.hpp"
#include "oc_io.hpp"
#include "oc_kernels.hpp"
#include "oc_system_pattern.hpp"

#include <algorithm>
#include <atomic>
#include <array>
#include <chrono>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <iterator>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

namespace {

using oc::PcgCtrl;
using oc::TriSet;

// Device allocation owned by the context. Grows, never shrinks.
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    ~DevBuf()
    {
        if (p) (void)hipFree(p);
    }
    hipError_t ensure(size_t b)
    {
        if (b <= bytes && p) return hipSuccess;
        if (p) {
            (void)hipFree(p);
            p = nullptr;
            bytes = 0;
        }
        const size_t nb = b < 256 ? 256 : b;
        hipError_t e = hipMalloc(&p, nb);
        if (e == hipSuccess) bytes = nb;
        return e;
    }
    template <typename T>
    T* as() const
    {
        return static_cast<T*>(p);
    }
};

// Full symmetric 2x2-block CSR over nV vertices.
struct BlockPattern : oc::HostPattern {
    DevBuf dRowPtr, dColIdx, dDiagPos, dVals, dMinv;
    int vals32 = 0;  // dVals holds float blocks (room for double blocks is always allocated)
    bool pcgSmall = false;  // Jacobi-PCG runs in one workgroup (pcg_small_fits)
};

}  // namespace

struct oc_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    char arch[64] = {0};

    // ---- per-iteration traces (energyValPerIter.txt, gradientPerIter.txt) ----
    FILE* trE = nullptr;
    FILE* trG = nullptr;
    double trSeam = 0.0;
    // the seam column recomputed per line from the cohesive edges (oc_trace_set_seams)
    bool trSeams = false;
    int trFracture = 0, trNCoh = 0;
    double trInitSeamLen = 0.0;
    std::vector<int> trCohE;
    DevBuf dTrCohE;

    // ---- mesh block (block 0) -----------------------------------------------
    int nV = 0, nF = 0;
    std::vector<int> Fh;            // nF x 3
    std::vector<double> Vh;         // nV x 3 rest positions
    std::vector<int> fixedSorted;   // mesh fixed vertices, ascending
    std::vector<unsigned char> fixedMaskMesh;
    double surfaceArea = 0.0, avgEdgeLen = 0.0;
    // mesh-only gather lists (Energy interface)
    std::vector<int> mvcPtr, mvcSrc;
    DevBuf dMvcPtr, dMvcSrc;
    // split-query pre-screen: per-vertex keys, and the mesh's boundary flags
    // and neighbour counts (built on first use for the mesh of meshGen topoGen)
    DevBuf dDivGrad, dCohE, dSeam;
    DevBuf dMrgA, dMrgB, dMrgOff, dMrgTri, dMrgCorner, dMrgStatus, dMrgPos;  // merge-query screen
    // avgEdgeLen summed in igl::avg_edge_length's order (the device reduction's order differs in the last bits;
    // the merge screen's eps must be the reference's to the bit), for the mesh of meshGen refAelGen
    double refAvgEdgeLen = 0.0;
    unsigned long refAelGen = 0;
    unsigned long topoGen = 0;
    std::vector<unsigned char> isBnd;
    std::vector<int> nbrCount;
    std::vector<long long> tripOff;  // per mesh triangle
    std::vector<unsigned char> vFree;
    long long nTripElem = 0;
    DevBuf dTripOff, dVFree;

    // ---- air block (block 1) -------------------------------------------------
    int nVair = 0, nFair = 0, nBnd = 0;
    double wScaf = 0.0, airAreaThres = 0.0;
    std::vector<int> FairLocal;         // nFair x 3 in air-mesh numbering
    std::vector<int> airL2G;            // air vertex -> combined vertex (localVI2Global)
    DevBuf dAirL2G, dAirUV2;            // the same on the device; air-vertex UV copy-out
    std::vector<int> FairGlobal;        // nFair x 3 in combined numbering
    std::vector<unsigned char> airFixedGlobal;  // per combined vertex: fixed in the air mesh

    // ---- combined triangle storage (mesh then air) ----------------------------
    DevBuf dF0, dF1, dF2, dTriArea, dA2, dE0, dE1, dE01;
    DevBuf dVrest, dTmpVrest, dTmpF;
    DevBuf dMeshSums, dAirSums;  // 3 doubles each
    DevBuf dUV;                  // combined vertices x 2
    DevBuf dUVspare;             // the other UV buffer of an air-mesh change
    DevBuf dFixedMaskMesh;

    // scratch
    DevBuf dPartials, dCounters, dScalars, dOrdMin, dLsOut, dEelem, dElemG, dElemH, dG, dTmpVec, dDir, dLsDec;
    // pinned host words the Newton step reads back asynchronously (the gradient norm, the line-search outcome),
    // and the event that marks the gradient norm's arrival
    double* mail = nullptr;
    hipEvent_t evGsq = nullptr;
    PcgCtrl* pcgMail = nullptr;  // pinned: control records of the last two parts of a PCG's first batch
    hipEvent_t evPcg[2] = {nullptr, nullptr};
    DevBuf dTrI, dTrJ, dTrV;

    // ---- Newton system (combined) ---------------------------------------------
    bool sysReady = false;
    int nVt = 0, nFt = 0;
    BlockPattern sys;
    oc::SystemMaps sm;  // upper blocks of sys and their assembly map
    oc::HostPattern sysSpare;  // the previous build's pattern and maps: storage for the next build
    oc::SystemMaps smSpare;
    std::vector<int> FtBuf;  // combined triangle list (mesh, then air) of the last build
    std::vector<int> vcPtr, vcSrc;
    // what sys and sm were built from: the mesh (meshGen of oc_set_mesh) and
    // the mesh vertices in air triangles; rows of the other mesh vertices are
    // reused when only the air mesh changed
    unsigned long meshGen = 0, sysMeshGen = 0;
    bool sysBuilt = false;
    std::vector<unsigned char> sysAirTouched;
    std::vector<unsigned char> fixedMaskSys;
    std::vector<double> fixedDiag;
    DevBuf dUbRow, dUbCol, dUbPosU, dUbPosL, dUbCPtr, dUbCSrc, dVcPtr, dVcSrc, dFixedMaskSys, dFixedDiag;
    double a0 = 1.0, relGL2Tol = 1e-12, targetGRes = 0.0;
    int allowEDecRelTol = 1;
    double lastE = 0.0, lastESD = 0.0, lastEScaf = 0.0;
    // oc_newton_set_forcing: after a step shorter than looseBelow (the injectivity bound held it back, so the
    // direction's accuracy is mostly unused) the next solve runs to max(pcgTol, looseTol); 0 turns it off
    double looseTol = 0.0, looseBelow = 0.0, lastStep = 1.0;
    int nPrecond = OC_PRECOND_JACOBI;
    double pcgTol = 1e-10;
    int pcgMaxIter = 10000;
    int pcgHint = 0;  // iterations of the previous Newton step's solve (first-batch size)
    int amgSkip = 0;  // Newton steps left that go to Jacobi-PCG directly after multigrid failed
    int amgFailStreak = 0;  // consecutive multigrid steps whose whole fallback chain ended in Jacobi-PCG
    // host wall times (ms) of the last set-up and air-mesh update, for oc_setup_times
    double tSetup[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    bool airLimited = false;  // the last step's injectivity bound came from an air triangle
    bool amgPending = false;  // multigrid selected, its structure not yet built for the current pattern
    int airSinceRemesh = 0;   // oc_scaffold_update calls since the air mesh was last re-meshed
    // Mixed form with the learned factor: element terms of the Newton system
    // (gradient, Hessian) in FP64 from the step whose FP32-assembled system
    // broke the solve until the next oc_newton_init
    bool elemFp64 = false;

    int precision = OC_PRECISION_FP64;  // requested for the next oc_newton_init
    int sysPrecision = OC_PRECISION_FP64;
    oc::Amg<double> amg64;  // multigrid preconditioner, FP64 hierarchy
    oc::Amg<float> amg32;   // FP32 hierarchy (mixed form)
    oc::AmgBase* amg = nullptr;
    bool amgValid = false;
    // After an air re-mesh the multigrid structure of the previous Newton pattern is kept (kAmgRemapMax times
    // in a row, then rebuilt): the Newton matrix is mapped onto that pattern (amgPat) before each numeric set-up
    oc::HostPattern amgPat;                   // the pattern the current multigrid structure was built for
    const oc::AmgBase* amgPatOwner = nullptr;  // the hierarchy holding that structure
    bool amgOnOld = false;                    // amgPat differs from the Newton pattern: values go through the map
    int amgRemaps = 0;                        // air re-meshes since the structure was last built
    bool amgRebuild = false;                  // a solve on a kept structure needed a fallback: rebuild it
    DevBuf dAmgOldRowPtr, dAmgMap, dAmgDropPtr, dAmgDrop, dAmgOldDiag, dAmgVals;
    std::vector<int> amgMapH, amgDropPtrH, amgDropH;  // host side of the map (kept for its memory)
    bool amgPatUploaded = false;                      // dAmgOldRowPtr / dAmgOldDiag hold amgPat
    oc_gnn* learned = nullptr;             // bound by oc_newton_set_learned (not owned)
    // iterative refinement (oc_newton_set_refinement): at most irMax passes of PCG on the FP32-rounded Newton
    // matrix dVals32, each on the FP64 residual of the accumulated solution dXir
    int irMax = 0;
    DevBuf dVals32, dXir, dRir, dIrPart;
    DevBuf dPcgSmall;                         // slot-major blocks of the one-workgroup PCG
    // block IC(0) of the Newton matrix: the preconditioner of OC_PRECOND_IC0, and the learned form's fallback
    // (its structure then built when first needed for the current pattern)
    oc::Ic0 ic0;
    bool ic0Struct = false;
    oc::Preconditioner* ext = nullptr;     // the external preconditioner of the Newton PCG, if any

    // ---- PCG workspace ---------------------------------------------------------
    DevBuf dX, dR, dR1, dZ, dP0, dP1, dQ, dB, dCtrl, dPcgPart;
    // PCG iterations replayed from captured HIP graphs (an even iteration,
    // an odd one, an even+odd pair, a run of pairs), valid for the buffers
    // and sizes recorded in pcgSig
    bool pcgGraphs = true;
    std::vector<uintptr_t> pcgSig;
    hipGraphExec_t pcgG[4] = {nullptr, nullptr, nullptr, nullptr};
    long long pcgGraphBuilds = 0;
    void clear_pcg_graphs()
    {
        for (auto& g : pcgG)
            if (g) {
                (void)hipGraphExecDestroy(g);
                g = nullptr;
            }
        pcgSig.clear();
    }
    int lastIters = 0;
    double lastRelRes = 0.0;

    // ---- batched charts (contiguous vertex / triangle ranges of the mesh) ----------
    int nCharts = 0;  // 0: one problem
    std::vector<int> chartV, chartF;        // nCharts + 1 range starts
    std::vector<int> chartBlk;              // chart-aligned triangle blocks of chart c: [chartBlk[c], chartBlk[c+1])
    std::vector<double> chartTarget, chartLastE, chartGsq, chartStep;
    std::vector<int> chartState;            // 0 active, 1 gradient converged, 2 line search stopped
    DevBuf dChartV, dChartF, dChartBlk, dBlkRange, dBlkChart, dVChart, dTriChart, dChartArea, dChartActive,
        dChartAlpha, dChartOrdMin, dChartOut, dChartGsq;

    // ---- Tutte initial map --------------------------------------------------------
    BlockPattern tut;
    oc::Amg<double> amgTut;

    // ---- LinSysSolver drop-in ---------------------------------------------------
    BlockPattern sol;
    int solN = 0;
    std::vector<int> solIa, solJa, solDst, solMir;
    std::vector<double> solA;
    DevBuf dSolA, dSolDst, dSolMir, dSolB, dSolX;
    int solPrecond = OC_PRECOND_JACOBI;
    double solTol = 1e-10;
    int solMaxIter = 100000;
    bool solFactorized = false;
    // multigrid for the drop-in: structure per pattern, hierarchy per factorize; near-null space from the
    // coordinates of oc_solver_set_coords (rigid motions), translations only until they are set
    oc::Amg<double> amgSol;
    std::vector<unsigned char> solFixed;
    bool solAmgStruct = false;
    DevBuf dSolUV;
    bool solHaveUV = false;
    int solFallback = 0;  // what the last solve fell back to (0 none, 1 safe-interval multigrid, 2 Jacobi)
    oc::Ic0 ic0Sol;         // IC(0) of the drop-in (structure per pattern)
    bool solIc0Struct = false;

    const char* fail(const std::string& m)
    {
        err = m;
        return err.c_str();
    }
};

#define OC_HIP(ctx, call)                                                                       \
    do {                                                                                        \
        hipError_t e_ = (call);                                                                 \
        if (e_ != hipSuccess) {                                                                 \
            (ctx)->err = std::string(#call) + ": " + hipGetErrorString(e_);                     \
            return OC_ERR_HIP;                                                                  \
        }                                                                                       \
    } while (0)

#define OC_ARG(ctx, cond, msg)           \
    do {                                 \
        if (!(cond)) {                   \
            (ctx)->err = (msg);          \
            return OC_ERR_ARG;           \
        }                                \
    } while (0)

namespace {

constexpr int kMaxPartialBlocks = 1 << 16;
constexpr int kRzRecords = 2048;  // r.z partial records of an external preconditioner
constexpr size_t kMailBytes = 4096;  // pinned read-back words of a context
constexpr int kAmgSkip = 3;          // steps without multigrid after it failed on a step
#ifndef OC_AMG_REMAP_MAX
#define OC_AMG_REMAP_MAX 4
#endif
constexpr int kAmgRemapMax = OC_AMG_REMAP_MAX;  // air re-meshes on one multigrid structure before it is rebuilt
#ifndef OC_AMG_KEEP_DROP
#define OC_AMG_KEEP_DROP 0.003
#endif
// a kept multigrid structure is rebuilt once the Newton pattern has this share of its blocks outside it
constexpr double kAmgKeepDrop = OC_AMG_KEEP_DROP;
constexpr int kMaxTimedLevels = 16;  // oc_time_kernel 10 + l: Chebyshev step on multigrid level l
#ifndef OC_AIR_LIMIT_RATIO
#define OC_AIR_LIMIT_RATIO 0.5
#endif
constexpr double kAirLimitRatio = OC_AIR_LIMIT_RATIO;  // air bound below this share of the mesh's: re-mesh

int ensure_scratch(oc_ctx* c, long nItems)
{
    const long blocks = oc::grid_for(nItems);
    // 3*kLSCand compensated pairs per block is the widest publisher
    OC_HIP(c, c->dPartials.ensure(sizeof(double) * (size_t)blocks * 2 * 3 * oc::kLSCand + 4096));
    if (!c->dCounters.p) {
        OC_HIP(c, c->dCounters.ensure(sizeof(unsigned int) * 64));
        OC_HIP(c, hipMemsetAsync(c->dCounters.p, 0, c->dCounters.bytes, c->stream));
    }
    if (!c->dScalars.p) {
        OC_HIP(c, c->dScalars.ensure(sizeof(double) * 64));
        OC_HIP(c, hipMemsetAsync(c->dScalars.p, 0, c->dScalars.bytes, c->stream));
    }
    OC_HIP(c, c->dOrdMin.ensure(sizeof(unsigned long long) * 8));
    OC_HIP(c, c->dLsOut.ensure(sizeof(double) * 4 * oc::kLSCand));
    OC_HIP(c, c->dLsDec.ensure(sizeof(oc::LsDecision)));
    (void)kMaxPartialBlocks;
    return OC_OK;
}

// counters: [0] features mesh, [1] features air, [2] element esum, [3] gather grad,
//           [4] line search, [5] inversion count (plain counter)
unsigned int* counter(oc_ctx* c, int k) { return c->dCounters.as<unsigned int>() + k; }
// scalars: [0..2] scratch sums, [4..5] esum, [6] gsq
double* scalar(oc_ctx* c, int k) { return c->dScalars.as<double>() + k; }

TriSet mesh_set(oc_ctx* c, int uniform)
{
    TriSet T;
    T.nF = c->nF;
    T.nFmesh = c->nF;
    T.f0 = c->dF0.as<int>();
    T.f1 = c->dF1.as<int>();
    T.f2 = c->dF2.as<int>();
    T.triArea = c->dTriArea.as<double>();
    T.A2 = c->dA2.as<double>();
    T.E0 = c->dE0.as<double>();
    T.E1 = c->dE1.as<double>();
    T.E01 = c->dE01.as<double>();
    T.surfaceArea = c->dMeshSums.as<double>();
    if (c->nCharts > 0) {
        T.surfaceArea = c->dChartArea.as<double>();
        T.triChart = c->dTriChart.as<int>();
    }
    T.uniformMesh = uniform;
    T.sMesh = 1.0;
    T.sAir = 1.0;
    return T;
}

TriSet system_set(oc_ctx* c)
{
    TriSet T = mesh_set(c, 0);
    T.nF = c->nF + c->nFair;
    T.sMesh = c->a0;
    T.sAir = c->nFair ? c->wScaf / (double)c->nFair : 0.0;
    return T;
}

using oc::build_vertex_lists;

template <typename T>
int upload(oc_ctx* c, DevBuf& d, const std::vector<T>& h)
{
    OC_HIP(c, d.ensure(sizeof(T) * (h.size() ? h.size() : 1)));
    if (!h.empty()) OC_HIP(c, hipMemcpyAsync(d.p, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice, c->stream));
    return OC_OK;
}

// Build the full block pattern from a per-vertex neighbour relation (each
// row sorted, unique, including the diagonal) restricted by the fixed mask:
// fixed rows keep only the diagonal, free rows drop fixed columns.
void build_block_pattern(BlockPattern& P, int nV, const std::vector<std::vector<int>>& rows,
                         const std::vector<unsigned char>& fixedMask)
{
    P.nV = nV;
    P.rowPtr.assign(nV + 1, 0);
    P.colIdx.clear();
    P.diagPos.assign(nV, -1);
    for (int u = 0; u < nV; ++u) {
        if (fixedMask[u]) {
            P.diagPos[u] = (int)P.colIdx.size();
            P.colIdx.push_back(u);
        } else {
            for (int w : rows[u]) {
                if (w != u && fixedMask[w]) continue;
                if (w == u) P.diagPos[u] = (int)P.colIdx.size();
                P.colIdx.push_back(w);
            }
        }
        P.rowPtr[u + 1] = (int)P.colIdx.size();
    }
}

int upload_pattern(oc_ctx* c, BlockPattern& P)
{
    if (upload(c, P.dRowPtr, P.rowPtr)) return OC_ERR_HIP;
    if (upload(c, P.dColIdx, P.colIdx)) return OC_ERR_HIP;
    if (upload(c, P.dDiagPos, P.diagPos)) return OC_ERR_HIP;
    OC_HIP(c, P.dVals.ensure(sizeof(double) * 4 * (size_t)std::max<long>(1, P.nnzb())));
    OC_HIP(c, P.dMinv.ensure(sizeof(double) * 4 * (size_t)std::max(1, P.nV)));
    P.pcgSmall = oc::pcg_small_fits(P.nV, P.rowPtr.data());
    return OC_OK;
}

int ensure_pcg(oc_ctx* c, int nV)
{
    const size_t b = sizeof(double) * 2 * (size_t)std::max(1, nV);
    OC_HIP(c, c->dX.ensure(b));
    OC_HIP(c, c->dR.ensure(b));
    OC_HIP(c, c->dZ.ensure(b));
    OC_HIP(c, c->dP0.ensure(b));
    OC_HIP(c, c->dP1.ensure(b));
    OC_HIP(c, c->dQ.ensure(b));
    OC_HIP(c, c->dB.ensure(b));
    if (!c->dCtrl.p) {
        OC_HIP(c, c->dCtrl.ensure(sizeof(PcgCtrl)));
        OC_HIP(c, hipMemsetAsync(c->dCtrl.p, 0, sizeof(PcgCtrl), c->stream));
    }
    OC_HIP(c, c->dPcgPart.ensure(sizeof(double) * (4 * (size_t)std::max(oc::pcg_grid_update(nV), oc::pcg_grid_spmv(nV)) +
                                                   (size_t)oc::pcg_grid_spmv(nV) + kRzRecords)));
    OC_HIP(c, c->dPcgSmall.ensure(oc::pcg_small_bytes(nV)));
    return ensure_scratch(c, 2L * nV);
}

// PCG on pattern P for right-hand side b (device), solution in c->dX.
// Iterations are queued in batches; ctrl is read back between batches.
// vals (null: P's own values) and vals32: the matrix the iterations multiply by, on P's pattern.
int run_pcg(oc_ctx* c, BlockPattern& P, const double* b, double relTol, int maxIter, int& iters, double& relRes,
            oc::Preconditioner* amg = nullptr, int hint = 0, const void* vals = nullptr, int vals32 = 0)
{
    const int nV = P.nV;
    const void* V = vals ? vals : P.dVals.p;
    const int V32 = vals ? vals32 : P.vals32;
    PcgCtrl* ctrl = c->dCtrl.as<PcgCtrl>();
    PcgCtrl h{};
    h.tol2 = relTol * relTol;
    h.maxit = maxIter;
    OC_HIP(c, hipMemcpyAsync(&ctrl->tol2, &h.tol2, sizeof(double), hipMemcpyHostToDevice, c->stream));
    OC_HIP(c, hipMemcpyAsync(&ctrl->maxit, &h.maxit, sizeof(int), hipMemcpyHostToDevice, c->stream));
    const auto result = [&] {
        iters = h.iter;
        relRes = h.bb > 0.0 ? std::sqrt(h.rr / h.bb) : 0.0;
        if (h.done == 3) {
            c->err = "PCG breakdown (p^T A p <= 0)";
            return OC_ERR_BREAKDOWN;
        }
        if (h.done == 2) {
            c->err = "PCG reached maxIter before the tolerance";
            return OC_ERR_NOT_CONVERGED;
        }
        return OC_OK;
    };
    if (!amg && P.pcgSmall) {
        // iterations per launch, which bounds its length: 2.5-6 ms with rows of at most 8 blocks, 13 at the rule's limit
        constexpr int kSpan = 1024;
        for (int it = 0; !h.done; it += kSpan) {
            oc::launch_pcg_small(c->stream, nV, P.dRowPtr.as<int>(), P.dColIdx.as<int>(), V, V32, b,
                                 P.dMinv.as<double>(), c->dX.as<double>(), c->dR.as<double>(), c->dP0.as<double>(),
                                 c->dPcgSmall.p, it, it + kSpan, ctrl);
            OC_HIP(c, hipGetLastError());
            OC_HIP(c, hipMemcpyAsync(&h, ctrl, sizeof(PcgCtrl), hipMemcpyDeviceToHost, c->stream));
            OC_HIP(c, hipStreamSynchronize(c->stream));
        }
        return result();
    }
    const bool fused = amg && amg->update_records() > 0;
    const int GU = fused ? amg->update_records() : oc::pcg_grid_update(nV), GS = oc::pcg_grid_spmv(nV);
    double* partU[2] = {c->dPcgPart.as<double>(), c->dPcgPart.as<double>() + 2 * (size_t)GU};
    double* partS = c->dPcgPart.as<double>() + 4 * (size_t)GU;
    double* partRZ = partS + GS;
    const double* Minv = amg ? nullptr : P.dMinv.as<double>();
    // A multigrid's first smoothing step runs in the kernels that write the residual, and its first kernel stops the
    // iteration when that residual is within the tolerance (the V-cycle on a converged residual has no use).
    const oc::FirstStep first = amg ? amg->first_step() : oc::FirstStep{};
    const auto precondition = [&](const double* pu) {
        const oc::PcgStage stage{pu + 1, GU, 2, ctrl};
        amg->apply(c->stream, c->dR.as<double>(), c->dZ.as<double>(), partRZ, &ctrl->done, first.d ? &stage : nullptr);
    };
    oc::launch_pcg_init(c->stream, nV, b, Minv, c->dX.as<double>(), c->dR.as<double>(), c->dZ.as<double>(), partU[0],
                        GU, ctrl, first);
    if (amg) precondition(partU[0]);
    double* pbuf[2] = {c->dP0.as<double>(), c->dP1.as<double>()};
    double* rbuf[2] = {c->dR.as<double>(), c->dR1.as<double>()};  // a fused update alternates
    // One iteration's launches. The kernels take the iteration number from
    // the control record, so the launches depend only on its parity (which
    // buffers alternate) and every iteration of one parity is the same graph.
    const auto enqueue = [&](int par) {
        double* pOld = pbuf[par];
        double* pNew = pbuf[par ^ 1];
        const double* pu = partU[par];
        if (amg)
            oc::launch_pcg_spmv(c->stream, nV, P.dRowPtr.as<int>(), P.dColIdx.as<int>(), V, V32,
                                c->dZ.as<double>(), pOld, pNew, c->dQ.as<double>(), partRZ, amg->rz_records(), 1,
                                pu + 1, GU, 2, partS, ctrl);
        else
            oc::launch_pcg_spmv(c->stream, nV, P.dRowPtr.as<int>(), P.dColIdx.as<int>(), V, V32,
                                c->dZ.as<double>(), pOld, pNew, c->dQ.as<double>(), pu, GU, 2, pu + 1, GU, 2, partS,
                                ctrl);
        if (fused) {
            amg->update_apply(c->stream,
                              oc::PcgUpdate{pNew, c->dQ.as<double>(), rbuf[par], c->dX.as<double>(), rbuf[par ^ 1],
                                            partS, GS, partU[par ^ 1], ctrl},
                              c->dZ.as<double>(), partRZ);
            return;
        }
        oc::launch_pcg_update(c->stream, nV, pNew, c->dQ.as<double>(), Minv, c->dX.as<double>(), c->dR.as<double>(),
                              c->dZ.as<double>(), partS, partU[par ^ 1], ctrl, first);
        if (amg) precondition(partU[par ^ 1]);
    };
    // Graphs: 0 an even iteration, 1 an odd one, 2 an even+odd pair, 3 a run
    // of kChain pairs. They name these buffers and sizes; anything else
    // recaptures them.
    constexpr int kChain = 8;
    if (c->pcgGraphs) {
        const uintptr_t sig[] = {(uintptr_t)nV,           (uintptr_t)P.dRowPtr.p, (uintptr_t)P.dColIdx.p,
                                 (uintptr_t)V,            (uintptr_t)V32,         (uintptr_t)Minv,
                                 (uintptr_t)c->dX.p,      (uintptr_t)c->dR.p,     (uintptr_t)c->dZ.p,
                                 (uintptr_t)c->dR1.p,
                                 (uintptr_t)c->dP0.p,     (uintptr_t)c->dP1.p,    (uintptr_t)c->dQ.p,
                                 (uintptr_t)c->dPcgPart.p, (uintptr_t)ctrl,       (uintptr_t)amg,
                                 amg ? (uintptr_t)amg->generation() : 0, amg ? (uintptr_t)amg->rz_records() : 0};
        const size_t ns = sizeof(sig) / sizeof(sig[0]);
        if (c->pcgSig.size() != ns || !std::equal(sig, sig + ns, c->pcgSig.begin())) {
            c->clear_pcg_graphs();
            c->pcgSig.assign(sig, sig + ns);
        }
    }
    const auto graph = [&](int kind) -> hipGraphExec_t {
        if (c->pcgG[kind]) return c->pcgG[kind];
        if (hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) return nullptr;
        if (kind == 0 || kind == 2) enqueue(0);
        if (kind == 1 || kind == 2) enqueue(1);
        if (kind == 3)
            for (int q = 0; q < 2 * kChain; ++q) enqueue(q & 1);
        hipGraph_t g = nullptr;
        if (hipStreamEndCapture(c->stream, &g) != hipSuccess || !g) return nullptr;
        hipGraphExec_t ex = nullptr;
        const hipError_t e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) return nullptr;
        c->pcgG[kind] = ex;
        ++c->pcgGraphBuilds;
        return ex;
    };
    // Queues iterations [it, it + n): replayed graphs, or launches one by one
    // (graphs off, or a capture that failed, which turns them off).
    const auto queue = [&](int it, int n) -> hipError_t {
        for (int k = 0; k < n;) {
            const int par = (it + k) & 1;
            const int kind = par ? 1 : (n - k >= 2 * kChain ? 3 : (n - k >= 2 ? 2 : 0));
            const int span = kind == 3 ? 2 * kChain : (kind == 2 ? 2 : 1);
            hipGraphExec_t ex = c->pcgGraphs ? graph(kind) : nullptr;
            if (c->pcgGraphs && !ex) {
                c->pcgGraphs = false;
                c->clear_pcg_graphs();
                (void)hipGetLastError();
            }
            if (ex) {
                const hipError_t e = hipGraphLaunch(ex, c->stream);
                if (e != hipSuccess) return e;
            } else {
                for (int q = 0; q < span; ++q) enqueue((par + q) & 1);
            }
            k += span;
        }
        return hipGetLastError();
    };
    int it = 0;
    // Iterations are queued in batches and the control record read back after
    // each. Queued iterations past convergence still launch (and return at
    // once), so the first batch is sized by the caller's hint (the previous
    // solve's iteration count, +1 for the converging check unless the preconditioner makes it at the end of the
    // iteration), then grows.
    int batch = hint > 0 ? hint + (first.d ? 0 : 1) : (amg ? 8 : 32);
    int next = amg ? 2 : 32;
    const int maxBatch = amg ? 32 : 512;
    // A long first batch goes out in parts, each once the part before the last has reported, so the queue never runs dry
    // and at most two parts of eight run past the end: a Newton step may need a hundredth of the previous one's
    // iterations, and every launch past the end costs 2-3 us (a step of 4 iterations after one of 1,013 at 200k faces:
    // 5.4 ms queued whole, 2.8 in four parts, 1.5 in eight; a step of 449 learned iterations the same to 1% with all).
    constexpr int kParts = 8;
    const int part = std::max((batch + kParts - 1) / kParts + 2 * kChain - 1, 4 * kChain) & ~(2 * kChain - 1);
    for (int k = 0; batch > part && !h.done; ++k) {
        const int slot = k & 1;
        OC_HIP(c, queue(it, part));
        it += part;
        batch -= part;
        OC_HIP(c, hipMemcpyAsync(&c->pcgMail[slot], ctrl, sizeof(PcgCtrl), hipMemcpyDeviceToHost, c->stream));
        OC_HIP(c, hipEventRecord(c->evPcg[slot], c->stream));
        if (k > 0) {
            OC_HIP(c, hipEventSynchronize(c->evPcg[slot ^ 1]));
            h = c->pcgMail[slot ^ 1];
        }
    }
    // what was queued past the end is over before the caller goes on: it may free or capture anew what those launches name
    if (h.done) OC_HIP(c, hipStreamSynchronize(c->stream));
    while (!h.done) {
        OC_HIP(c, queue(it, batch));
        it += batch;
        OC_HIP(c, hipMemcpyAsync(&h, ctrl, sizeof(PcgCtrl), hipMemcpyDeviceToHost, c->stream));
        OC_HIP(c, hipStreamSynchronize(c->stream));
        batch = next;
        if (next < maxBatch) next *= 2;
    }
    return result();
}

int ensure_tri_storage(oc_ctx* c, int nFtot)
{
    const size_t i4 = sizeof(int) * (size_t)std::max(1, nFtot), d8 = sizeof(double) * (size_t)std::max(1, nFtot);
    // grow preserving the mesh part
    auto grow = [&](DevBuf& b, size_t bytes, size_t keep) -> hipError_t {
        if (b.p && b.bytes >= bytes) return hipSuccess;
        DevBuf nb;
        hipError_t e = nb.ensure(bytes);
        if (e != hipSuccess) return e;
        if (b.p && keep) {
            e = hipMemcpyAsync(nb.p, b.p, std::min(keep, b.bytes), hipMemcpyDeviceToDevice, c->stream);
            if (e != hipSuccess) return e;
            e = hipStreamSynchronize(c->stream);
            if (e != hipSuccess) return e;
        }
        std::swap(b.p, nb.p);
        std::swap(b.bytes, nb.bytes);
        return hipSuccess;
    };
    const size_t ki = sizeof(int) * (size_t)c->nF, kd = sizeof(double) * (size_t)c->nF;
    OC_HIP(c, grow(c->dF0, i4, ki));
    OC_HIP(c, grow(c->dF1, i4, ki));
    OC_HIP(c, grow(c->dF2, i4, ki));
    OC_HIP(c, grow(c->dTriArea, d8, kd));
    OC_HIP(c, grow(c->dA2, d8, kd));
    OC_HIP(c, grow(c->dE0, d8, kd));
    OC_HIP(c, grow(c->dE1, d8, kd));
    OC_HIP(c, grow(c->dE01, d8, kd));
    return OC_OK;
}

int upload_tri_ids(oc_ctx* c, int offset, int n, const int* F)
{
    std::vector<int> a(n), b(n), d(n);
    for (int t = 0; t < n; ++t) {
        a[t] = F[3 * t];
        b[t] = F[3 * t + 1];
        d[t] = F[3 * t + 2];
    }
    if (n == 0) return OC_OK;
    OC_HIP(c, hipMemcpyAsync(c->dF0.as<int>() + offset, a.data(), sizeof(int) * n, hipMemcpyHostToDevice, c->stream));
    OC_HIP(c, hipMemcpyAsync(c->dF1.as<int>() + offset, b.data(), sizeof(int) * n, hipMemcpyHostToDevice, c->stream));
    OC_HIP(c, hipMemcpyAsync(c->dF2.as<int>() + offset, d.data(), sizeof(int) * n, hipMemcpyHostToDevice, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));  // host vectors go out of scope
    return OC_OK;
}

int energy_sums(oc_ctx* c, const TriSet& T, double* Emesh, double* Eair, int f32 = 0)
{
    if (ensure_scratch(c, T.nF)) return OC_ERR_HIP;
    oc::launch_element(c->stream, T, c->dUV.as<double>(), nullptr, nullptr, nullptr, 0, c->dPartials.as<double>(),
                       scalar(c, 4), f32);
    OC_HIP(c, hipGetLastError());
    double e[2];
    OC_HIP(c, hipMemcpyAsync(e, scalar(c, 4), sizeof(e), hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    *Emesh = e[0];
    *Eair = e[1];
    return OC_OK;
}

int count_inverted(oc_ctx* c, const TriSet& T, unsigned int* n)
{
    OC_HIP(c, hipMemsetAsync(counter(c, 5), 0, sizeof(unsigned int), c->stream));
    oc::launch_count_inverted(c->stream, T, c->dUV.as<double>(), counter(c, 5));
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipMemcpyAsync(n, counter(c, 5), sizeof(unsigned int), hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return OC_OK;
}

int step_bound(oc_ctx* c, const TriSet& T, const double* dDir, double cap, double* out)
{
    unsigned long long* om = c->dOrdMin.as<unsigned long long>();
    oc::launch_set_u64(c->stream, om, oc::dbl_to_ordered_host(cap));
    oc::launch_step_bound(c->stream, T, c->dUV.as<double>(), dDir, om, cap);
    OC_HIP(c, hipGetLastError());
    unsigned long long r;
    OC_HIP(c, hipMemcpyAsync(&r, om, sizeof(r), hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    *out = oc::ordered_to_dbl_host(r);
    return OC_OK;
}

// Numeric multigrid hierarchy for the current Newton matrix (safe: the
// guaranteed smoother interval).
void amg_numeric(oc_ctx* c, int safe)
{
    const double* vals = c->sys.dVals.as<double>();
    if (c->amgOnOld) {
        oc::launch_remap_blocks(c->stream, c->amgPat.nV, c->dAmgOldRowPtr.as<int>(), c->dAmgMap.as<int>(),
                                c->dAmgDropPtr.as<int>(), c->dAmgDrop.as<int>(), c->dAmgOldDiag.as<int>(),
                                c->sys.dVals.as<double>(), c->dAmgVals.as<double>());
        vals = c->dAmgVals.as<double>();
    }
    c->amg->numeric(c->stream, vals, c->dUV.as<double>(), safe);
}

int amg_structure(oc_ctx* c);
int amg_remap(oc_ctx* c);

// Block IC(0) structure of the current Newton pattern.
int ic0_structure(oc_ctx* c)
{
    std::string e;
    if (c->ic0.setup(c->stream, c->nVt, c->sys.rowPtr, c->sys.colIdx, e) != 0) {
        c->err = e;
        return OC_ERR_HIP;
    }
    if (c->ic0.rz_records() > kRzRecords) {
        c->err = "IC(0): too many partial records";
        return OC_ERR_STATE;
    }
    c->ic0Struct = true;
    return OC_OK;
}

double ms_since(std::chrono::steady_clock::time_point t0)
{
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

// airOnly: only the air triangles changed since the last build (a re-mesh of oc_scaffold_update), so the
// multigrid structure may be kept.
int build_system(oc_ctx* c, bool airOnly = false)
{
    const auto tb0 = std::chrono::steady_clock::now();
    const int nVt = c->nV + (c->nFair ? c->nVair - c->nBnd : 0);
    oc::AmgBase* const amgTarget =
        c->nPrecond != OC_PRECOND_AMG ? nullptr
        : c->sysPrecision == OC_PRECISION_MIXED ? static_cast<oc::AmgBase*>(&c->amg32)
                                                : static_cast<oc::AmgBase*>(&c->amg64);
    const bool keepAmg = airOnly && amgTarget && c->amgValid && c->amg == amgTarget && !c->amgRebuild &&
                         c->amgPatOwner == amgTarget && c->amgPat.nV == nVt && c->amgRemaps < kAmgRemapMax;
    const int nFt = c->nF + c->nFair;
    c->nVt = nVt;
    c->nFt = nFt;
    std::vector<int>& Ft = c->FtBuf;
    Ft.resize(3 * (size_t)nFt);
    std::copy(c->Fh.begin(), c->Fh.end(), Ft.begin());
    std::copy(c->FairGlobal.begin(), c->FairGlobal.end(), Ft.begin() + 3 * (size_t)c->nF);

    c->fixedMaskSys.assign(nVt, 0);
    for (int v : c->fixedSorted) c->fixedMaskSys[v] = 1;
    const double sAir = c->nFair ? c->wScaf / (double)c->nFair : 0.0;
    c->fixedDiag.assign(nVt, 0.0);
    for (int v : c->fixedSorted) {
        c->fixedDiag[v] = c->a0;
        if (c->nFair && !c->airFixedGlobal.empty() && c->airFixedGlobal[v]) c->fixedDiag[v] += sAir;
    }
    // vertex -> (triangle*3 + corner) lists in triangle order (the gradient
    // gathers use them, and so does everything below)
    build_vertex_lists(nVt, nFt, Ft.data(), c->vcPtr, c->vcSrc);
    c->tSetup[0] = ms_since(tb0);
    auto tp = std::chrono::steady_clock::now();
    // Pattern and slot maps. After an air-mesh change on the same mesh (the
    // scaffold is rebuilt every Newton iteration, Optimizer.cpp:251-257, and
    // re-patterned, :522-530), the rows of mesh vertices outside the old and
    // the new air triangles are copied from the previous build.
    std::vector<unsigned char> touched(c->nV, 0);
    for (int v : c->FairGlobal)
        if (v < c->nV) touched[v] = 1;
    std::vector<unsigned char> keep;
    if (c->sysBuilt && c->sysMeshGen == c->meshGen && c->sysAirTouched.size() == (size_t)c->nV) {
        keep.resize(c->nV);
        for (int v = 0; v < c->nV; ++v) keep[v] = !touched[v] && !c->sysAirTouched[v];
    }
    // built into the spare pattern and maps (the build before last's, whose memory is reused), then swapped in
    oc::build_system_maps(nVt, Ft, c->fixedMaskSys.data(), c->vcPtr, c->vcSrc, c->sysSpare, c->smSpare,
                          keep.empty() ? nullptr : &c->sys, keep.empty() ? nullptr : &c->sm,
                          keep.empty() ? nullptr : keep.data(), (int)keep.size());
    std::swap(static_cast<oc::HostPattern&>(c->sys), c->sysSpare);
    std::swap(c->sm, c->smSpare);
    c->sysBuilt = true;
    c->sysMeshGen = c->meshGen;
    c->sysAirTouched = std::move(touched);
    c->tSetup[1] = ms_since(tp);
    tp = std::chrono::steady_clock::now();
    if (upload_pattern(c, c->sys)) return OC_ERR_HIP;
    // The PCG matrix stays FP64 in both precisions: rounding the assembled
    // Hessian to FP32 can make it indefinite along its near-null directions
    // (rigid rotation about the fixed vertex), which breaks CG. The mixed
    // form's FP32 lives in the element terms and the preconditioner.
    c->sys.vals32 = 0;
    if (upload(c, c->dUbRow, c->sm.ubRow) || upload(c, c->dUbCol, c->sm.ubCol) ||
        upload(c, c->dUbPosU, c->sm.ubPosU) || upload(c, c->dUbPosL, c->sm.ubPosL) ||
        upload(c, c->dUbCPtr, c->sm.ubCPtr) || upload(c, c->dUbCSrc, c->sm.ubCSrc) ||
        upload(c, c->dVcPtr, c->vcPtr) || upload(c, c->dVcSrc, c->vcSrc) ||
        upload(c, c->dFixedMaskSys, c->fixedMaskSys) || upload(c, c->dFixedDiag, c->fixedDiag))
        return OC_ERR_HIP;
    OC_HIP(c, c->dElemG.ensure(sizeof(double) * 6 * (size_t)std::max(1, nFt)));
    OC_HIP(c, c->dElemH.ensure(sizeof(double) * 24 * (size_t)std::max(1, nFt)));
    OC_HIP(c, c->dG.ensure(sizeof(double) * 2 * (size_t)std::max(1, nVt)));
    OC_HIP(c, c->dTmpVec.ensure(sizeof(double) * 2 * (size_t)std::max(1, nVt)));
    if (ensure_pcg(c, nVt)) return OC_ERR_HIP;
    if (ensure_scratch(c, std::max(std::max(nFt, nVt), (int)c->sm.ubRow.size()))) return OC_ERR_HIP;
    OC_HIP(c, hipStreamSynchronize(c->stream));
    c->tSetup[2] = ms_since(tp);
    tp = std::chrono::steady_clock::now();
    c->amgValid = false;
    c->amg64.drop_values();  // upload_pattern (or amg_remap below) may have replaced the buffer it reads
    c->amg = nullptr;
    c->ext = nullptr;
    c->tSetup[3] = c->tSetup[4] = 0.0;
    if (c->nPrecond == OC_PRECOND_LEARNED) {
        if (!c->learned) {
            c->err = "OC_PRECOND_LEARNED needs a network (oc_newton_set_learned)";
            return OC_ERR_STATE;
        }
        std::string e;
        if (c->learned->net.set_pattern(c->stream, nVt, c->sys.rowPtr, c->sys.colIdx, c->fixedMaskSys, e) != 0) {
            c->err = e;
            return OC_ERR_HIP;
        }
        c->learned->rowPtr.clear();  // the network's pattern now belongs to this context
        OC_HIP(c, c->dR1.ensure(sizeof(double) * 2 * (size_t)std::max(1, nVt)));  // its update alternates residuals
        if (c->learned->net.rz_records() > kRzRecords) {
            c->err = "learned preconditioner: too many partial records";
            return OC_ERR_STATE;
        }
        c->ext = &c->learned->net;
        c->tSetup[4] = ms_since(tp);
    }
    c->ic0Struct = false;
    if (c->nPrecond == OC_PRECOND_IC0) {
        if (int st = ic0_structure(c)) return st;
        c->ext = &c->ic0;
    }
    c->amgPending = false;
    if (c->nPrecond == OC_PRECOND_AMG) {
        c->amg = c->sysPrecision == OC_PRECISION_MIXED ? static_cast<oc::AmgBase*>(&c->amg32)
                                                      : static_cast<oc::AmgBase*>(&c->amg64);
        // while multigrid is being skipped after a failure, its structure is built when it is next used
        if (c->amgSkip > 0) c->amgPending = true;
        else if (keepAmg) {
            const int st = amg_remap(c);
            if (st > 0) return st;
            if (st < 0)  // too far from the kept pattern
                if (int st2 = amg_structure(c)) return st2;
        } else if (int st = amg_structure(c)) return st;
    }
    OC_HIP(c, hipStreamSynchronize(c->stream));
    if (c->nPrecond == OC_PRECOND_AMG) c->tSetup[3] = ms_since(tp);
    c->tSetup[5] = ms_since(tb0);
    c->sysReady = true;
    return OC_OK;
}

// The multigrid structure (aggregates, prolongator pattern, product maps) of the current Newton pattern.
int amg_structure(oc_ctx* c)
{
    std::string e;
    // the rows an air mesh can change (air vertices and the mesh vertices in air triangles) are aggregated
    // last, so the hierarchy away from the air mesh keeps its numbering and is copied after a re-mesh
    std::vector<unsigned char> late;
    if (c->nFair) {
        late.assign(c->nVt, 0);
        for (int v : c->FairGlobal) late[v] = 1;
    }
    c->amgPatOwner = nullptr;
    c->amgOnOld = false;
    c->amgRebuild = false;
    if (c->amg->setup(c->stream, c->nVt, c->sys.rowPtr, c->sys.colIdx, c->fixedMaskSys, e,
                      late.empty() ? nullptr : &late) != 0) {
        c->err = e;
        return OC_ERR_HIP;
    }
    c->ext = c->amg;
    if (c->ext->rz_records() > kRzRecords) {
        c->err = "AMG: too many partial records";
        return OC_ERR_STATE;
    }
    c->amgPat = static_cast<const oc::HostPattern&>(c->sys);
    c->amgPatOwner = c->amg;
    c->amgPatUploaded = false;
    c->amgRemaps = 0;
    c->amgValid = true;
    c->amgPending = false;
    return OC_OK;
}

// Keeps the multigrid structure built for amgPat (same rows as the current Newton pattern, which differs from
// it only in rows an air re-mesh touched): per block of amgPat the block of the current pattern with the same
// (row, column) or -1, and per row the current blocks that amgPat lacks. amg_numeric maps the Newton matrix
// through them (launch_remap_blocks: the lacking blocks go onto the diagonal by their Frobenius norms, which
// keeps the mapped matrix symmetric positive definite), so the preconditioner is that of a nearby matrix; the
// PCG products stay on the Newton matrix itself. Returns -1, keeping nothing, when more than kAmgKeepDrop of
// amgPat's block count lies outside it (the caller then builds the structure anew).
int amg_remap(oc_ctx* c)
{
    const oc::HostPattern& O = c->amgPat;
    const oc::HostPattern& N = c->sys;
    const int n = O.nV;
    std::vector<int>& map = c->amgMapH;
    std::vector<int>& dropPtr = c->amgDropPtrH;
    std::vector<int>& drop = c->amgDropH;
    map.resize(O.colIdx.size());
    dropPtr.assign(n + 1, 0);
    // pass 1 (rows in parallel): the map, and per row the count of current blocks the kept pattern lacks
    std::atomic<bool> bad{false};
    const int nt = oc::setup_threads((long)O.colIdx.size());
    const int nch = nt > 1 ? 8 * nt : 1;
    oc::parallel_row_chunks(n, nch, [&](int, int r0, int r1) {
        for (int u = r0; u < r1; ++u) {
            int i = O.rowPtr[u], j = N.rowPtr[u], nd = 0;
            const int ie = O.rowPtr[u + 1], je = N.rowPtr[u + 1];
            while (i < ie || j < je) {
                if (j == je || (i < ie && O.colIdx[i] < N.colIdx[j])) map[i++] = -1;
                else if (i == ie || N.colIdx[j] < O.colIdx[i]) { ++nd; ++j; }
                else map[i++] = j++;
            }
            dropPtr[u + 1] = nd;
            if (O.diagPos[u] < 0 || map[O.diagPos[u]] < 0) bad = true;
        }
    });
    if (bad) return -1;
    for (int u = 0; u < n; ++u) dropPtr[u + 1] += dropPtr[u];
    if ((double)dropPtr[n] > kAmgKeepDrop * (double)O.nnzb()) return -1;
    drop.resize(std::max(1, dropPtr[n]));  // one unread entry when empty keeps the upload non-empty
    // pass 2: the lacking blocks of each row, in column order
    oc::parallel_row_chunks(n, nch, [&](int, int r0, int r1) {
        for (int u = r0; u < r1; ++u) {
            int i = O.rowPtr[u], j = N.rowPtr[u], q = dropPtr[u];
            const int ie = O.rowPtr[u + 1], je = N.rowPtr[u + 1];
            while (j < je) {
                if (i < ie && O.colIdx[i] < N.colIdx[j]) ++i;
                else if (i == ie || N.colIdx[j] < O.colIdx[i]) drop[q++] = j++;
                else { ++i; ++j; }
            }
        }
    });
    // the kept pattern's rows and diagonal positions go up once per structure
    if (!c->amgPatUploaded) {
        if (upload(c, c->dAmgOldRowPtr, O.rowPtr) || upload(c, c->dAmgOldDiag, O.diagPos)) return OC_ERR_HIP;
        c->amgPatUploaded = true;
    }
    if (upload(c, c->dAmgMap, map) || upload(c, c->dAmgDropPtr, dropPtr) || upload(c, c->dAmgDrop, drop))
        return OC_ERR_HIP;
    OC_HIP(c, c->dAmgVals.ensure(sizeof(double) * 4 * (size_t)std::max<long>(1, O.nnzb())));
    OC_HIP(c, hipStreamSynchronize(c->stream));  // the host maps end with this call
    c->ext = c->amg;
    c->amgOnOld = true;
    ++c->amgRemaps;
    c->amgValid = true;
    c->amgPending = false;
    return OC_OK;
}

int system_energy(oc_ctx* c, double* E, double* Emesh, double* Eair)
{
    TriSet T = system_set(c);
    double em, ea;
    if (int st = energy_sums(c, T, &em, &ea, c->sysPrecision == OC_PRECISION_MIXED)) return st;
    *Emesh = em;
    *Eair = c->nFair ? ea * (c->wScaf / (double)c->nFair) : 0.0;
    *E = c->a0 * em + *Eair;
    return OC_OK;
}

// Split-query keys at the current UV into c->dDivGrad (mesh vertices): the
// element pass's weighted gradient rows (w = triArea / surfaceArea, as
// SymDirichletEnergy::computeLocalGradient), then their per-vertex spread.
int div_grad_keys(oc_ctx* c)
{
    if (ensure_scratch(c, c->nF)) return OC_ERR_HIP;
    OC_HIP(c, c->dDivGrad.ensure(sizeof(double) * (size_t)c->nV));
    oc::launch_element(c->stream, mesh_set(c, 0), c->dUV.as<double>(), nullptr, c->dElemG.as<double>(), nullptr, 0,
                       nullptr, nullptr);
    oc::launch_div_grad(c->stream, c->nV, c->dMvcPtr.as<int>(), c->dMvcSrc.as<int>(), c->dElemG.as<double>(),
                        c->dDivGrad.as<double>());
    OC_HIP(c, hipGetLastError());
    return OC_OK;
}

// E_se / virtualRadius at the current UV: TriMesh::computeSeamSparsity(E_se, !fractureMode) over the cohesive
// edges of oc_trace_set_seams plus initSeamLen, divided by sqrt(surfaceArea / pi) (TriMesh.cpp:404,1542-1558;
// Optimizer.cpp:708-710).
int seam_term(oc_ctx* c, double* out)
{
    double s = 0.0;
    if (c->trNCoh > 0) {
        if (ensure_scratch(c, c->trNCoh)) return OC_ERR_HIP;
        oc::launch_seam_len(c->stream, c->trNCoh, c->dTrCohE.as<int>(), c->dVrest.as<double>(), c->dUV.as<double>(),
                            c->avgEdgeLen, !c->trFracture, c->dPartials.as<double>(), c->dSeam.as<double>());
        OC_HIP(c, hipGetLastError());
        OC_HIP(c, hipMemcpyAsync(&s, c->dSeam.p, sizeof(double), hipMemcpyDeviceToHost, c->stream));
        OC_HIP(c, hipStreamSynchronize(c->stream));
    }
    *out = (s + c->trInitSeamLen) / std::sqrt(c->surfaceArea / M_PI);
    return OC_OK;
}

// One energyValPerIter.txt line (Optimizer::writeEnergyValToFile, Optimizer.cpp:706-728): in fracture mode the
// first column is lastEnergyVal + (1 - energyParams[0]) E_se, else lastEnergyVal; then E_SD, E_se, a0. Without
// oc_trace_set_seams the seam column is the caller's constant (oc_trace_set_seam).
int write_energy_trace(oc_ctx* c, double E, double Esd)
{
    double seam = c->trSeam, col0 = E;
    if (c->trSeams) {
        if (int st = seam_term(c, &seam)) return st;
        if (c->trFracture) col0 = E + (1.0 - c->a0) * seam;
    }
    oc::io::trace_energy_line(c->trE, col0, Esd, seam, c->a0);
    return OC_OK;
}

// Boundary flags and neighbour counts of the mesh (TriMesh::computeFeatures
// builds vNeighbor and the directed-edge map edge2Tri, TriMesh.cpp:437-446;
// isBoundaryVert, TriMesh.cpp:2069-2083, asks for a neighbour w with (v, w) or
// (w, v) missing from edge2Tri). Around vertex v the directed edges leaving it
// end at the corners after v and those entering it start at the corners
// before v, so v is on the boundary when those two sets differ.
void mesh_topology(oc_ctx* c)
{
    if (c->topoGen == c->meshGen && (int)c->isBnd.size() == c->nV) return;
    const int nV = c->nV;
    c->isBnd.assign(nV, 0);
    c->nbrCount.assign(nV, 0);
    oc::parallel_row_chunks(nV, oc::setup_threads(3L * c->nF), [&](int, int r0, int r1) {
        std::vector<int> nx, pv, un;
        for (int v = r0; v < r1; ++v) {
            nx.clear();
            pv.clear();
            for (int q = c->mvcPtr[v]; q < c->mvcPtr[v + 1]; ++q) {
                const int t = c->mvcSrc[q] / 3, k = c->mvcSrc[q] % 3;
                nx.push_back(c->Fh[3 * (size_t)t + (k + 1) % 3]);
                pv.push_back(c->Fh[3 * (size_t)t + (k + 2) % 3]);
            }
            std::sort(nx.begin(), nx.end());
            nx.erase(std::unique(nx.begin(), nx.end()), nx.end());
            std::sort(pv.begin(), pv.end());
            pv.erase(std::unique(pv.begin(), pv.end()), pv.end());
            un.clear();
            std::set_union(nx.begin(), nx.end(), pv.begin(), pv.end(), std::back_inserter(un));
            c->nbrCount[v] = (int)un.size();
            c->isBnd[v] = nx != pv;
        }
    });
    c->topoGen = c->meshGen;
}

}  // namespace

// ---- scratch of the no-allocation entry point (oc_energy_noalloc) --------------------------------------------
// The energy reduction's workgroup records (2 compensated sums = 4 doubles each, up to kStaticBlocks workgroups of
// kBlock triangles) and its two finished sums, in a file-scope device array: 2 MiB + 64 B held on every device the
// library runs on. Host code reaches each device's copy only through the address hipGetSymbolAddress returns for
// it (looked up once per device, at the first context on that device).
namespace {
constexpr int kStaticBlocks = 1 << 16;
constexpr long kStaticMaxTri = (long)kStaticBlocks * oc::kBlock;  // 16,777,216 triangles
constexpr size_t kStaticRecordDoubles = 4 * (size_t)kStaticBlocks;
}  // namespace
static __device__ __align__(256) double scratch[kStaticRecordDoubles + 8];

namespace {
std::mutex g_scratchMu;
std::vector<double*> g_scratchPtr;  // per device

// With `device` current: its copy of `scratch`, looked up on the first call for the device.
int static_scratch_setup(int device)
{
    std::lock_guard<std::mutex> g(g_scratchMu);
    if ((int)g_scratchPtr.size() <= device) g_scratchPtr.resize(device + 1, nullptr);
    if (g_scratchPtr[device]) return OC_OK;
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return OC_ERR_HIP;
    g_scratchPtr[device] = static_cast<double*>(p);
    return OC_OK;
}

double* static_scratch(int device)
{
    std::lock_guard<std::mutex> g(g_scratchMu);
    return device < (int)g_scratchPtr.size() ? g_scratchPtr[device] : nullptr;
}
}  // namespace

// =====================================================================================
extern "C" {

int oc_ctx_create(int device, oc_ctx** out)
{
    if (!out) return OC_ERR_ARG;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= device || device < 0) return OC_ERR_NO_DEVICE;
    if (hipSetDevice(device) != hipSuccess) return OC_ERR_NO_DEVICE;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return OC_ERR_NO_DEVICE;
    oc_ctx* c = new oc_ctx();
    c->device = device;
    std::snprintf(c->arch, sizeof(c->arch), "%s", prop.gcnArchName);
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return OC_ERR_HIP;
    }
    if (hipHostMalloc((void**)&c->mail, kMailBytes + 2 * sizeof(PcgCtrl), hipHostMallocDefault) != hipSuccess ||
        hipEventCreateWithFlags(&c->evGsq, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c->evPcg[0], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c->evPcg[1], hipEventDisableTiming) != hipSuccess || static_scratch_setup(device)) {
        (void)oc_ctx_destroy(c);
        return OC_ERR_HIP;
    }
    c->pcgMail = reinterpret_cast<PcgCtrl*>(c->mail + kMailBytes / sizeof(double));
    *out = c;
    return OC_OK;
}

int oc_ctx_destroy(oc_ctx* c)
{
    if (!c) return OC_ERR_ARG;
    (void)oc_trace_close(c);
    (void)hipSetDevice(c->device);
    if (c->stream) {
        (void)hipStreamSynchronize(c->stream);
        c->clear_pcg_graphs();
        (void)hipStreamDestroy(c->stream);
    }
    for (hipEvent_t e : {c->evGsq, c->evPcg[0], c->evPcg[1]})
        if (e) (void)hipEventDestroy(e);
    if (c->mail) (void)hipHostFree(c->mail);
    delete c;
    return OC_OK;
}

const char* oc_last_error(const oc_ctx* c) { return c ? c->err.c_str() : "null context"; }

int oc_trace_close(oc_ctx* c)
{
    if (!c) return OC_ERR_ARG;
    int bad = 0;
    for (FILE** f : {&c->trE, &c->trG})
        if (*f) {
            bad |= std::fclose(*f);
            *f = nullptr;
        }
    if (bad) {
        c->err = "oc_trace_close: write error";
        return OC_ERR_STATE;
    }
    return OC_OK;
}

int oc_trace_open(oc_ctx* c, const char* folder)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, folder != nullptr, "oc_trace_open: null folder");
    (void)oc_trace_close(c);
    std::string base(folder);
    if (!base.empty() && base.back() != '/') base += '/';
    c->trE = std::fopen((base + "energyValPerIter.txt").c_str(), "w");
    c->trG = std::fopen((base + "gradientPerIter.txt").c_str(), "w");
    if (!c->trE || !c->trG) {
        (void)oc_trace_close(c);
        c->err = "oc_trace_open: cannot create the trace files in " + base;
        return OC_ERR_ARG;
    }
    return OC_OK;
}

int oc_trace_set_seam(oc_ctx* c, double seamTerm)
{
    if (!c) return OC_ERR_ARG;
    c->trSeam = seamTerm;
    c->trSeams = false;
    return OC_OK;
}

int oc_trace_set_seams(oc_ctx* c, int nCoh, const int* cohE, double initSeamLen, int fractureMode)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && nCoh >= 0 && (nCoh == 0 || cohE), "oc_trace_set_seams: bad arguments");
    for (long k = 0; k < 4L * nCoh; ++k) OC_ARG(c, cohE[k] < c->nV, "oc_trace_set_seams: vertex id out of range");
    (void)hipSetDevice(c->device);
    c->trCohE.assign(cohE, cohE + 4 * (size_t)nCoh);
    if (upload(c, c->dTrCohE, c->trCohE)) return OC_ERR_HIP;
    OC_HIP(c, c->dSeam.ensure(sizeof(double)));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    c->trNCoh = nCoh;
    c->trInitSeamLen = initSeamLen;
    c->trFracture = fractureMode ? 1 : 0;
    c->trSeams = true;
    return OC_OK;
}

int oc_device_arch(const oc_ctx* c, char* buf, int buflen)
{
    if (!c || !buf || buflen <= 0) return OC_ERR_ARG;
    std::snprintf(buf, buflen, "%s", c->arch);
    return OC_OK;
}

int oc_set_mesh(oc_ctx* c, int nV, const double* Vrest, int nF, const int* F, int nFixed, const int* fixedV,
                double areaThres)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, nV > 0 && nF > 0 && Vrest && F && nFixed >= 0 && (nFixed == 0 || fixedV), "oc_set_mesh: bad sizes");
    for (long k = 0; k < 3L * nF; ++k) OC_ARG(c, F[k] >= 0 && F[k] < nV, "oc_set_mesh: vertex index out of range");
    for (int k = 0; k < nFixed; ++k) OC_ARG(c, fixedV[k] >= 0 && fixedV[k] < nV, "oc_set_mesh: fixed id out of range");
    (void)hipSetDevice(c->device);
    c->sysReady = false;
    c->nFair = 0;
    c->nVair = 0;
    c->nBnd = 0;
    c->FairGlobal.clear();
    c->airFixedGlobal.clear();
    c->nCharts = 0;
    c->nV = nV;
    c->nF = nF;
    ++c->meshGen;
    c->sysBuilt = false;
    c->Fh.assign(F, F + 3 * (size_t)nF);
    c->Vh.assign(Vrest, Vrest + 3 * (size_t)nV);
    c->fixedSorted.assign(fixedV, fixedV + nFixed);
    std::sort(c->fixedSorted.begin(), c->fixedSorted.end());
    c->fixedSorted.erase(std::unique(c->fixedSorted.begin(), c->fixedSorted.end()), c->fixedSorted.end());
    c->fixedMaskMesh.assign(nV, 0);
    for (int v : c->fixedSorted) c->fixedMaskMesh[v] = 1;

    if (int st = ensure_tri_storage(c, nF)) return st;
    if (int st = upload_tri_ids(c, 0, nF, F)) return st;
    // features (areaThres applies to every triangle of this block)
    OC_HIP(c, c->dVrest.ensure(sizeof(double) * 3 * (size_t)nV));
    OC_HIP(c, hipMemcpyAsync(c->dVrest.p, Vrest, sizeof(double) * 3 * (size_t)nV, hipMemcpyHostToDevice, c->stream));
    if (ensure_scratch(c, nF)) return OC_ERR_HIP;
    OC_HIP(c, c->dMeshSums.ensure(sizeof(double) * 4));
    oc::launch_rest_features(c->stream, nF, c->dF0.as<int>(), c->dF1.as<int>(), c->dF2.as<int>(),
                             c->dVrest.as<double>(), areaThres, c->dTriArea.as<double>(), c->dA2.as<double>(),
                             c->dE0.as<double>(), c->dE1.as<double>(), c->dE01.as<double>(),
                             c->dPartials.as<double>(), c->dMeshSums.as<double>());
    OC_HIP(c, hipGetLastError());
    double sums[3];
    OC_HIP(c, hipMemcpyAsync(sums, c->dMeshSums.p, sizeof(sums), hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    c->surfaceArea = sums[0];
    c->avgEdgeLen = sums[1] / (3.0 * nF);
    if (sums[2] > 0.0) {
        c->err = "a rest triangle has zero area";
        return OC_ERR_DEGENERATE;
    }
    // mesh-only gather lists and reference triplet offsets
    build_vertex_lists(nV, nF, F, c->mvcPtr, c->mvcSrc);
    c->tripOff.resize(nF);
    c->vFree.resize(nF);
    long long off = 0;
    for (int t = 0; t < nF; ++t) {
        unsigned char m = 0;
        int nfree = 0;
        for (int k = 0; k < 3; ++k)
            if (!c->fixedMaskMesh[F[3 * t + k]]) {
                m |= (unsigned char)(1u << k);
                ++nfree;
            }
        c->vFree[t] = m;
        c->tripOff[t] = off;
        off += 4LL * nfree * nfree;
    }
    c->nTripElem = off;
    if (upload(c, c->dMvcPtr, c->mvcPtr) || upload(c, c->dMvcSrc, c->mvcSrc) || upload(c, c->dTripOff, c->tripOff) ||
        upload(c, c->dVFree, c->vFree) || upload(c, c->dFixedMaskMesh, c->fixedMaskMesh))
        return OC_ERR_HIP;
    OC_HIP(c, c->dUV.ensure(sizeof(double) * 2 * (size_t)nV));
    OC_HIP(c, hipMemsetAsync(c->dUV.p, 0, sizeof(double) * 2 * (size_t)nV, c->stream));
    OC_HIP(c, c->dElemG.ensure(sizeof(double) * 6 * (size_t)nF));
    OC_HIP(c, c->dG.ensure(sizeof(double) * 2 * (size_t)nV));
    OC_HIP(c, c->dEelem.ensure(sizeof(double) * (size_t)nF));
    OC_HIP(c, c->dDir.ensure(sizeof(double) * 2 * (size_t)nV));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return OC_OK;
}

int oc_set_uv(oc_ctx* c, const double* UV)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0, "oc_set_uv: no mesh");
    OC_ARG(c, UV != nullptr, "oc_set_uv: null UV");
    (void)hipSetDevice(c->device);
    OC_HIP(c, hipMemcpyAsync(c->dUV.p, UV, sizeof(double) * 2 * (size_t)c->nV, hipMemcpyHostToDevice, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return OC_OK;
}

int oc_get_uv(oc_ctx* c, double* UV)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && UV, "oc_get_uv: no mesh");
    (void)hipSetDevice(c->device);
    OC_HIP(c, hipMemcpyAsync(UV, c->dUV.p, sizeof(double) * 2 * (size_t)c->nV, hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return OC_OK;
}

int oc_mesh_stats(oc_ctx* c, double* surfaceArea, double* avgEdgeLen)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0, "oc_mesh_stats: no mesh");
    if (surfaceArea) *surfaceArea = c->surfaceArea;
    if (avgEdgeLen) *avgEdgeLen = c->avgEdgeLen;
    return OC_OK;
}

int oc_energy(oc_ctx* c, int uniformWeight, double* E)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && E, "oc_energy: no mesh");
    (void)hipSetDevice(c->device);
    double em, ea;
    if (int st = energy_sums(c, mesh_set(c, uniformWeight), &em, &ea)) return st;
    *E = em;
    return OC_OK;
}

int oc_energy_noalloc(oc_ctx* c, int uniformWeight, double* E)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && E, "oc_energy_noalloc: no mesh");
    OC_ARG(c, (long)c->nF <= kStaticMaxTri,
           "oc_energy_noalloc: more than 16,777,216 triangles (the static scratch holds 65,536 workgroup records)");
    double* p = static_scratch(c->device);
    if (!p) {
        c->err = "oc_energy_noalloc: the static scratch of this device was not found";
        return OC_ERR_STATE;
    }
    (void)hipSetDevice(c->device);
    // the same kernels as oc_energy: per-workgroup records, then the one-workgroup finisher; every record is
    // written before it is read, so nothing needs clearing between calls
    double* sums = p + kStaticRecordDoubles;
    oc::launch_element(c->stream, mesh_set(c, uniformWeight), c->dUV.as<double>(), nullptr, nullptr, nullptr, 0, p,
                       sums);
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipMemcpyAsync(c->mail, sums, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    *E = c->mail[0];
    return OC_OK;
}

int oc_energy_per_elem(oc_ctx* c, int uniformWeight, double* Eelem)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && Eelem, "oc_energy_per_elem: no mesh");
    (void)hipSetDevice(c->device);
    oc::launch_element(c->stream, mesh_set(c, uniformWeight), c->dUV.as<double>(), c->dEelem.as<double>(), nullptr,
                       nullptr, 0, nullptr, nullptr);
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipMemcpyAsync(Eelem, c->dEelem.p, sizeof(double) * (size_t)c->nF, hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return OC_OK;
}

int oc_gradient(oc_ctx* c, int uniformWeight, double* g)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && g, "oc_gradient: no mesh");
    (void)hipSetDevice(c->device);
    if (ensure_scratch(c, c->nV)) return OC_ERR_HIP;
    oc::launch_element(c->stream, mesh_set(c, uniformWeight), c->dUV.as<double>(), nullptr, c->dElemG.as<double>(),
                       nullptr, 0, nullptr, nullptr);
    oc::launch_gather_grad(c->stream, c->nV, c->dMvcPtr.as<int>(), c->dMvcSrc.as<int>(),
                           c->dFixedMaskMesh.as<unsigned char>(), c->dElemG.as<double>(), c->dG.as<double>(),
                           c->dPartials.as<double>(), nullptr);
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipMemcpyAsync(g, c->dG.p, sizeof(double) * 2 * (size_t)c->nV, hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return OC_OK;
}

int oc_hessian_triplets(oc_ctx* c, int uniformWeight, long long capacity, int* I, int* J, double* V,
                        long long* count)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && count, "oc_hessian_triplets: no mesh");
    const long long total = c->nTripElem + 2LL * (long long)c->fixedSorted.size();
    *count = total;
    if (!I) return OC_OK;
    OC_ARG(c, J && V && capacity >= total, "oc_hessian_triplets: capacity too small");
    (void)hipSetDevice(c->device);
    const size_t ne = (size_t)std::max<long long>(1, c->nTripElem);
    OC_HIP(c, c->dTrI.ensure(sizeof(int) * ne));
    OC_HIP(c, c->dTrJ.ensure(sizeof(int) * ne));
    OC_HIP(c, c->dTrV.ensure(sizeof(double) * ne));
    oc::launch_triplets(c->stream, mesh_set(c, uniformWeight), c->dUV.as<double>(), c->dTripOff.as<long long>(),
                        c->dVFree.as<unsigned char>(), c->dTrI.as<int>(), c->dTrJ.as<int>(), c->dTrV.as<double>());
    OC_HIP(c, hipGetLastError());
    if (c->nTripElem) {
        OC_HIP(c, hipMemcpyAsync(I, c->dTrI.p, sizeof(int) * c->nTripElem, hipMemcpyDeviceToHost, c->stream));
        OC_HIP(c, hipMemcpyAsync(J, c->dTrJ.p, sizeof(int) * c->nTripElem, hipMemcpyDeviceToHost, c->stream));
        OC_HIP(c, hipMemcpyAsync(V, c->dTrV.p, sizeof(double) * c->nTripElem, hipMemcpyDeviceToHost, c->stream));
    }
    OC_HIP(c, hipStreamSynchronize(c->stream));
    long long o = c->nTripElem;
    for (int v : c->fixedSorted)
        for (int d = 0; d < 2; ++d) {
            I[o] = J[o] = 2 * v + d;
            V[o] = 1.0;
            ++o;
        }
    return OC_OK;
}

int oc_element_terms(oc_ctx* c, int precision, double* E, double* G, double* H)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0, "oc_element_terms: no mesh");
    OC_ARG(c, precision == OC_PRECISION_FP64 || precision == OC_PRECISION_MIXED, "oc_element_terms: bad precision");
    (void)hipSetDevice(c->device);
    const size_t nF = (size_t)c->nF;
    const int f32 = precision == OC_PRECISION_MIXED;
    OC_HIP(c, c->dElemH.ensure(sizeof(double) * 24 * nF));
    oc::launch_element(c->stream, mesh_set(c, 0), c->dUV.as<double>(), c->dEelem.as<double>(), c->dElemG.as<double>(),
                       H ? c->dElemH.p : nullptr, 1, nullptr, nullptr, f32);
    OC_HIP(c, hipGetLastError());
    if (E) OC_HIP(c, hipMemcpyAsync(E, c->dEelem.p, sizeof(double) * nF, hipMemcpyDeviceToHost, c->stream));
    if (G) OC_HIP(c, hipMemcpyAsync(G, c->dElemG.p, sizeof(double) * 6 * nF, hipMemcpyDeviceToHost, c->stream));
    std::vector<double> blk;
    if (H) {
        blk.resize(24 * nF);
        if (f32) {
            std::vector<float> b32(24 * nF);
            OC_HIP(c, hipMemcpyAsync(b32.data(), c->dElemH.p, sizeof(float) * 24 * nF, hipMemcpyDeviceToHost,
                                     c->stream));
            OC_HIP(c, hipStreamSynchronize(c->stream));
            std::copy(b32.begin(), b32.end(), blk.begin());
        } else {
            OC_HIP(c, hipMemcpyAsync(blk.data(), c->dElemH.p, sizeof(double) * 24 * nF, hipMemcpyDeviceToHost,
                                     c->stream));
        }
    }
    OC_HIP(c, hipStreamSynchronize(c->stream));
    if (H) {
        // upper 2x2 blocks (vertex pairs (0,0) (0,1) (0,2) (1,1) (1,2) (2,2), each [xx, xy, yx, yy]) -> full 6x6
        static const int bi[6] = {0, 0, 0, 1, 1, 2}, bj[6] = {0, 1, 2, 1, 2, 2};
        for (size_t t = 0; t < nF; ++t) {
            double* M = H + 36 * t;
            for (int b = 0; b < 6; ++b)
                for (int r = 0; r < 2; ++r)
                    for (int q = 0; q < 2; ++q) {
                        const double v = blk[24 * t + 4 * b + 2 * r + q];
                        M[(2 * bi[b] + r) * 6 + 2 * bj[b] + q] = v;
                        M[(2 * bj[b] + q) * 6 + 2 * bi[b] + r] = v;
                    }
        }
    }
    return OC_OK;
}

int oc_init_step_size(oc_ctx* c, const double* dir, double* stepSize)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && dir && stepSize, "oc_init_step_size: no mesh");
    (void)hipSetDevice(c->device);
    if (ensure_scratch(c, c->nF)) return OC_ERR_HIP;
    OC_HIP(c, hipMemcpyAsync(c->dDir.p, dir, sizeof(double) * 2 * (size_t)c->nV, hipMemcpyHostToDevice, c->stream));
    double r;
    if (int st = step_bound(c, mesh_set(c, 0), c->dDir.as<double>(), *stepSize, &r)) return st;
    *stepSize = r;
    return OC_OK;
}

int oc_check_inversion(oc_ctx* c, int* ok)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && ok, "oc_check_inversion: no mesh");
    (void)hipSetDevice(c->device);
    if (ensure_scratch(c, c->nF)) return OC_ERR_HIP;
    unsigned int n = 0;
    if (int st = count_inverted(c, mesh_set(c, 0), &n)) return st;
    *ok = (n == 0) ? 1 : 0;
    return OC_OK;
}

int oc_pcg_graphs(oc_ctx* c, int enable)
{
    if (!c) return OC_ERR_ARG;
    (void)hipSetDevice(c->device);
    OC_HIP(c, hipStreamSynchronize(c->stream));
    c->clear_pcg_graphs();
    c->pcgGraphs = enable != 0;
    return OC_OK;
}

int oc_pcg_graph_builds(oc_ctx* c, long long* n)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, n, "oc_pcg_graph_builds: no result pointer");
    *n = c->pcgGraphBuilds;
    return OC_OK;
}

int oc_seam_sparsity(oc_ctx* c, int nCoh, const int* cohE, double initSeamLen, int triSoup, double* sparsity)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && nCoh >= 0 && (nCoh == 0 || cohE) && sparsity, "oc_seam_sparsity: bad arguments");
    for (long k = 0; k < 4L * nCoh; ++k)
        OC_ARG(c, cohE[k] < c->nV, "oc_seam_sparsity: cohesive vertex id out of range");
    (void)hipSetDevice(c->device);
    if (ensure_scratch(c, std::max(1, nCoh))) return OC_ERR_HIP;
    OC_HIP(c, c->dCohE.ensure(sizeof(int) * 4 * (size_t)std::max(1, nCoh)));
    OC_HIP(c, c->dSeam.ensure(sizeof(double)));
    if (nCoh)
        OC_HIP(c, hipMemcpyAsync(c->dCohE.p, cohE, sizeof(int) * 4 * (size_t)nCoh, hipMemcpyHostToDevice, c->stream));
    oc::launch_seam_len(c->stream, nCoh, c->dCohE.as<int>(), c->dVrest.as<double>(), c->dUV.as<double>(),
                        c->avgEdgeLen, triSoup, c->dPartials.as<double>(), c->dSeam.as<double>());
    OC_HIP(c, hipGetLastError());
    double s = 0.0;
    OC_HIP(c, hipMemcpyAsync(&s, c->dSeam.p, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    *sparsity = s + initSeamLen;
    return OC_OK;
}

int oc_info_write(oc_ctx* c, const char* path, int vertAmtInput, int nFInitial, int iterNum, int topoIter,
                  double lambdaInit, const double* timings, int nInitSeams, const int* initSeams)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && path && timings && nInitSeams >= 0 && (nInitSeams == 0 || initSeams),
           "oc_info_write: bad arguments");
    (void)hipSetDevice(c->device);
    const int nV = c->nV, nF = c->nF;
    std::vector<double> UV(2 * (size_t)nV);
    OC_HIP(c, hipMemcpyAsync(UV.data(), c->dUV.p, sizeof(double) * UV.size(), hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    // distortion: energyTerms[0]->computeEnergyVal at the result (main.cpp:372-373)
    double distortion, unused;
    if (int st = energy_sums(c, mesh_set(c, 0), &distortion, &unused)) return st;
    // seam length (main.cpp:360-370): half the boundary length in pure distortion mode (energyParams[0] == 1),
    // else computeSeamSparsity(!fractureMode) over the cohesive edges of oc_trace_set_seams
    const double virtualRadius = std::sqrt(c->surfaceArea / M_PI);
    double seamTerm = 0.0;  // seamLen / virtualRadius
    const double* Vr = c->Vh.data();
    auto restLen = [&](int a, int b) {
        const double dx = Vr[3 * (size_t)a] - Vr[3 * (size_t)b], dy = Vr[3 * (size_t)a + 1] - Vr[3 * (size_t)b + 1],
                     dz = Vr[3 * (size_t)a + 2] - Vr[3 * (size_t)b + 2];
        return std::sqrt(dx * dx + dy * dy + dz * dz);
    };
    if (c->a0 == 1.0) {
        // TriMesh::computeBoundaryLen (TriMesh.cpp:1533-1541): directed edges whose reverse is no edge
        std::vector<std::pair<int, int>> he;
        he.reserve(3 * (size_t)nF);
        for (int t = 0; t < nF; ++t)
            for (int k = 0; k < 3; ++k) he.emplace_back(c->Fh[3 * (size_t)t + k], c->Fh[3 * (size_t)t + (k + 1) % 3]);
        std::vector<std::pair<int, int>> sorted(he);
        std::sort(sorted.begin(), sorted.end());
        sorted.erase(std::unique(sorted.begin(), sorted.end()), sorted.end());
        double seamLen = 0.0;
        for (const auto& e : sorted)
            if (!std::binary_search(sorted.begin(), sorted.end(), std::make_pair(e.second, e.first)))
                seamLen += restLen(e.second, e.first);
        seamLen /= 2.0;
        seamTerm = seamLen / virtualRadius;
    } else if (c->trSeams) {
        if (int st = seam_term(c, &seamTerm)) return st;
    }
    // TriMesh::computeStandardStretch (TriMesh.cpp:1585-1652) with IglUtils::computeDeformationGradient and
    // mapTriangleTo2D (IglUtils.cpp:172-194)
    double l2 = 0.0, sinf = -DBL_MAX, shear = 0.0, cinf = DBL_MAX, areaUV = 0.0, area = 0.0;
    for (int t = 0; t < nF; ++t) {
        const int* f = &c->Fh[3 * (size_t)t];
        double e0[3], e1[3];
        for (int d = 0; d < 3; ++d) {
            e0[d] = Vr[3 * (size_t)f[1] + d] - Vr[3 * (size_t)f[0] + d];
            e1[d] = Vr[3 * (size_t)f[2] + d] - Vr[3 * (size_t)f[0] + d];
        }
        const double e0n = std::sqrt(e0[0] * e0[0] + e0[1] * e0[1] + e0[2] * e0[2]);
        const double cx = e0[1] * e1[2] - e0[2] * e1[1], cy = e0[2] * e1[0] - e0[0] * e1[2],
                     cz = e0[0] * e1[1] - e0[1] * e1[0];
        const double x1 = e0n, x2x = (e0[0] * e1[0] + e0[1] * e1[1] + e0[2] * e1[2]) / e0n,
                     x2y = std::sqrt(cx * cx + cy * cy + cz * cz) / e0n;
        const double u01[2] = {UV[2 * (size_t)f[1]] - UV[2 * (size_t)f[0]], UV[2 * (size_t)f[1] + 1] - UV[2 * (size_t)f[0] + 1]};
        const double u02[2] = {UV[2 * (size_t)f[2]] - UV[2 * (size_t)f[0]], UV[2 * (size_t)f[2] + 1] - UV[2 * (size_t)f[0] + 1]};
        const double u01Len = std::sqrt(u01[0] * u01[0] + u01[1] * u01[1]);
        // U = [[u01Len, u01.u02 / u01Len], [0, (u01 x u02) / u01Len]], Vm = [[x1, x2x], [0, x2y]], F = Vm U^-1
        const double U00 = u01Len, U01 = (u01[0] * u02[0] + u01[1] * u02[1]) / u01Len,
                     U11 = (u01[0] * u02[1] - u01[1] * u02[0]) / u01Len;
        const double invdet = 1.0 / (U00 * U11);  // Eigen's 2x2 inverse: cofactors times 1/det
        const double I00 = U11 * invdet, I01 = -U01 * invdet, I11 = U00 * invdet;
        const double F00 = x1 * I00, F01 = x1 * I01 + x2x * I11, F10 = 0.0, F11 = x2y * I11;
        const double a = F00 * F00 + F10 * F10, b = F00 * F01 + F10 * F11, cc = F01 * F01 + F11 * F11;
        const double t0 = a + cc, t1 = std::sqrt((a - cc) * (a - cc) + 4. * b * b);
        const double tau = std::sqrt((t0 + t1) / 2.), gamma = std::sqrt((t0 - t1) / 2.);
        const double triArea = 0.5 * std::sqrt(cx * cx + cy * cy + cz * cz);  // TriMesh.cpp:364-367
        l2 += t0 / 2.0 * triArea;
        if (tau > sinf) sinf = tau;
        shear += b * b / a / cc * triArea;
        if (gamma < cinf) cinf = gamma;
        areaUV += 0.5 * (u01[0] * u02[1] - u01[1] * u02[0]);
        area += triArea;
    }
    l2 = std::sqrt(l2 / c->surfaceArea);
    shear = std::sqrt(shear / c->surfaceArea);
    const double scale = std::sqrt(areaUV / c->surfaceArea);
    l2 *= scale;
    sinf *= scale;
    cinf *= scale;
    (void)area;
    FILE* fp = std::fopen(path, "w");
    if (!fp) {
        c->err = std::string("oc_info_write: cannot create ") + path;
        return OC_ERR_ARG;
    }
    static const char* lbl[13] = {"topo", "desc", "scaf", "enUp", "mtrComp", "mtrAssem", "symFac", "numFac",
                                  "backSolve", "lineSearch", "bSplit", "iSplit", "cMerge"};
    std::fprintf(fp, "%d %d\n", vertAmtInput, nFInitial);
    std::fprintf(fp, "%d %d 0 0 %g %g\n", iterNum, topoIter, lambdaInit, 1.0 - c->a0);
    std::fprintf(fp, "0.0 0.0 %g %g", timings[0], timings[1]);
    for (int k = 0; k < 13; ++k) std::fprintf(fp, " %s%g", lbl[k], timings[2 + k]);
    std::fprintf(fp, "\n%g %g\n", distortion, seamTerm);
    std::fprintf(fp, "%g %g %g %g\n", l2, sinf, shear, cinf);
    std::fprintf(fp, "initialSeams %d\n", nInitSeams);
    // Eigen's default matrix output: every entry right-aligned to the widest entry, one space apart
    int width = 0;
    for (long k = 0; k < 4L * nInitSeams; ++k) width = std::max(width, std::snprintf(nullptr, 0, "%d", initSeams[k]));
    for (int r = 0; r < nInitSeams; ++r) {
        for (int q = 0; q < 4; ++q) std::fprintf(fp, q ? " %*d" : "%*d", width, initSeams[4 * (size_t)r + q]);
        if (r + 1 < nInitSeams) std::fputc('\n', fp);
    }
    std::fputc('\n', fp);
    const bool ok = std::ferror(fp) == 0;
    std::fclose(fp);
    if (!ok) {
        c->err = std::string("oc_info_write: write error on ") + path;
        return OC_ERR_ARG;
    }
    return OC_OK;
}

int oc_div_grad_per_vert(oc_ctx* c, double* out)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && out, "oc_div_grad_per_vert: no mesh");
    (void)hipSetDevice(c->device);
    if (int st = div_grad_keys(c)) return st;
    OC_HIP(c, hipMemcpyAsync(out, c->dDivGrad.p, sizeof(double) * (size_t)c->nV, hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return OC_OK;
}

int oc_split_candidates(oc_ctx* c, int splitInterior, double filterExpIn, const double* vertWeight, int capacity,
                        int* cand, int* nCand, int* nSorted)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && nCand && nSorted && capacity >= 0 && (capacity == 0 || cand),
           "oc_split_candidates: bad arguments");
    (void)hipSetDevice(c->device);
    if (int st = div_grad_keys(c)) return st;
    std::vector<double> dg(c->nV);
    OC_HIP(c, hipMemcpyAsync(dg.data(), c->dDivGrad.p, sizeof(double) * (size_t)c->nV, hipMemcpyDeviceToHost,
                             c->stream));
    mesh_topology(c);
    OC_HIP(c, hipStreamSynchronize(c->stream));
    // std::map<double, int> semantics: keys ascending, a later vertex with an
    // equal key replaces the earlier one. The (key, vertex) pairs are
    // distinct, so their sorted order is unique; it is built as sorted row
    // chunks merged pairwise, on the host workers.
    const int nth = oc::setup_threads(4L * c->nV);
    std::vector<std::vector<std::pair<double, int>>> part(nth);
    std::vector<char> nanKey(nth, 0);
    oc::parallel_row_chunks(c->nV, nth, [&](int ch, int r0, int r1) {
        auto& out = part[ch];
        for (int v = r0; v < r1; ++v) {
            if (c->nbrCount[v] <= 2) continue;
            if (splitInterior) {
                if (c->isBnd[v]) continue;
                bool toBound = false;
                for (int q = c->mvcPtr[v]; q < c->mvcPtr[v + 1] && !toBound; ++q) {
                    const int t = c->mvcSrc[q] / 3;
                    for (int k = 0; k < 3; ++k) toBound = toBound || c->isBnd[c->Fh[3 * (size_t)t + k]];
                }
                if (toBound) continue;
            } else if (!c->isBnd[v]) {
                continue;
            }
            const double key = -dg[v] / (vertWeight ? vertWeight[v] : 1.0);
            if (std::isnan(key)) nanKey[ch] = 1;
            out.push_back({key, v});
        }
        std::sort(out.begin(), out.end());
    });
    for (char b : nanKey)
        if (b) {
            c->err = "oc_split_candidates: a split key is NaN (degenerate or inverted triangles)";
            return OC_ERR_DEGENERATE;
        }
    std::vector<size_t> bound(1, 0);
    for (auto& p : part) bound.push_back(bound.back() + p.size());
    std::vector<std::pair<double, int>> keys(bound.back());
    for (int ch = 0; ch < nth; ++ch) std::copy(part[ch].begin(), part[ch].end(), keys.begin() + bound[ch]);
    for (size_t w = 1; w < (size_t)nth; w *= 2) {  // merge runs [i, i+w) and [i+w, i+2w) of chunks
        const int nm = (int)((nth + 2 * w - 1) / (2 * w));
        oc::parallel_row_chunks(nm, nm, [&](int j, int, int) {
            const size_t a = 2 * w * j, b = std::min(a + w, (size_t)nth), e = std::min(a + 2 * w, (size_t)nth);
            if (b < e)
                std::inplace_merge(keys.begin() + bound[a], keys.begin() + bound[b], keys.begin() + bound[e]);
        });
    }
    size_t m = 0;
    for (size_t i = 0; i < keys.size(); ++i) {
        if (i + 1 < keys.size() && keys[i + 1].first == keys[i].first) continue;
        keys[m++] = keys[i];
    }
    keys.resize(m);
    *nSorted = (int)m;
    *nCand = 0;
    if (m == 0) return OC_OK;
    int amt = splitInterior ? static_cast<int>(std::pow((double)m, filterExpIn))
                            : static_cast<int>(std::pow((double)m, 0.8) * 1.0);
    if (amt < 2) amt = 2;
    const int n = std::min<int>(amt, (int)m);
    *nCand = n;
    for (int i = 0; i < n && i < capacity; ++i) cand[i] = keys[i].second;
    return OC_OK;
}

int oc_merge_candidates(oc_ctx* c, int nCoh, const int* cohE, int* status, double* mergedPos, int* nCand)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0 && nCoh >= 0 && (nCoh == 0 || (cohE && status && mergedPos)) && nCand,
           "oc_merge_candidates: bad arguments");
    for (long k = 0; k < 4L * nCoh; ++k)
        OC_ARG(c, cohE[k] >= 0 && cohE[k] < c->nV, "oc_merge_candidates: cohesive vertex out of range");
    (void)hipSetDevice(c->device);
    // zipper-bottom rows and their triangle lists: for each merge vertex v, the triangle holding the directed
    // edge (v, w) for every neighbour w in ascending order (vNeighbor, edge2Tri; the last triangle when two hold
    // the same directed edge, as the map assignment leaves it)
    std::vector<int> rowOf, rA, rB, off(1, 0), tl, cl;
    std::vector<std::array<int, 3>> inc;
    for (int r = 0; r < nCoh; ++r) {
        const int* row = cohE + 4 * (size_t)r;
        int fork;
        if (row[0] == row[2]) fork = 0;
        else if (row[1] == row[3]) fork = 1;
        else {
            status[r] = 1;
            mergedPos[2 * (size_t)r] = mergedPos[2 * (size_t)r + 1] = 0.0;
            continue;
        }
        const int va = row[1 - fork], vb = row[3 - fork];
        for (int v : {va, vb}) {
            inc.clear();
            for (int q = c->mvcPtr[v]; q < c->mvcPtr[v + 1]; ++q) {
                const int t = c->mvcSrc[q] / 3, k = c->mvcSrc[q] % 3;
                inc.push_back({c->Fh[3 * (size_t)t + (k + 1) % 3], t, k});
            }
            std::sort(inc.begin(), inc.end());
            for (size_t i = 0; i < inc.size(); ++i) {
                if (i + 1 < inc.size() && inc[i + 1][0] == inc[i][0]) continue;
                tl.push_back(inc[i][1]);
                cl.push_back(inc[i][2]);
            }
        }
        rowOf.push_back(r);
        rA.push_back(va);
        rB.push_back(vb);
        off.push_back((int)tl.size());
    }
    const int n = (int)rowOf.size();
    *nCand = 0;
    if (n == 0) return OC_OK;
    if (c->refAelGen != c->meshGen) {  // igl::avg_edge_length (avg_edge_length.cpp:17-30): half-edges in face order
        double el = 0.0;
        for (int t = 0; t < c->nF; ++t)
            for (int j = 0; j < 3; ++j) {
                const double* p = &c->Vh[3 * (size_t)c->Fh[3 * (size_t)t + j]];
                const double* q = &c->Vh[3 * (size_t)c->Fh[3 * (size_t)t + (j + 1) % 3]];
                const double dx = p[0] - q[0], dy = p[1] - q[1], dz = p[2] - q[2];
                el += std::sqrt(dx * dx + dy * dy + dz * dz);
            }
        c->refAvgEdgeLen = el / (double)(3L * c->nF);
        c->refAelGen = c->meshGen;
    }
    if (upload(c, c->dMrgA, rA) || upload(c, c->dMrgB, rB) || upload(c, c->dMrgOff, off) ||
        upload(c, c->dMrgTri, tl) || upload(c, c->dMrgCorner, cl))
        return OC_ERR_HIP;
    OC_HIP(c, c->dMrgStatus.ensure(sizeof(int) * (size_t)n));
    OC_HIP(c, c->dMrgPos.ensure(sizeof(double) * 2 * (size_t)n));
    oc::launch_merge_screen(c->stream, n, c->dMrgA.as<int>(), c->dMrgB.as<int>(), c->dMrgOff.as<int>(),
                            c->dMrgTri.as<int>(), c->dMrgCorner.as<int>(), c->dF0.as<int>(), c->dF1.as<int>(),
                            c->dF2.as<int>(), c->dUV.as<double>(), 1.0e-6 * c->refAvgEdgeLen, c->dMrgStatus.as<int>(),
                            c->dMrgPos.as<double>());
    OC_HIP(c, hipGetLastError());
    std::vector<int> st(n);
    std::vector<double> mp(2 * (size_t)n);
    OC_HIP(c, hipMemcpyAsync(st.data(), c->dMrgStatus.p, sizeof(int) * n, hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipMemcpyAsync(mp.data(), c->dMrgPos.p, sizeof(double) * 2 * n, hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    for (int i = 0; i < n; ++i) {
        const int r = rowOf[i];
        status[r] = st[i];
        mergedPos[2 * (size_t)r] = mp[2 * (size_t)i];
        mergedPos[2 * (size_t)r + 1] = mp[2 * (size_t)i + 1];
        *nCand += st[i] == 0;
    }
    return OC_OK;
}

int oc_set_air_mesh(oc_ctx* c, int nVair, const double* airUV, int nFair, const int* Fair, int nBnd, const int* bnd,
                    double areaThres, double wScaf)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0, "oc_set_air_mesh: no mesh");
    OC_ARG(c, c->nCharts == 0 || nFair == 0, "oc_set_air_mesh: not available with batched charts");
    (void)hipSetDevice(c->device);
    c->sysReady = false;
    if (nFair == 0) {
        c->nFair = c->nVair = c->nBnd = 0;
        c->FairGlobal.clear();
        c->airFixedGlobal.clear();
        return OC_OK;
    }
    OC_ARG(c, nVair > 0 && airUV && Fair && nBnd >= 0 && nBnd <= nVair && (nBnd == 0 || bnd) && wScaf >= 0.0,
           "oc_set_air_mesh: bad sizes");
    for (int k = 0; k < nBnd; ++k) OC_ARG(c, bnd[k] >= 0 && bnd[k] < c->nV, "oc_set_air_mesh: bnd out of range");
    for (long k = 0; k < 3L * nFair; ++k) OC_ARG(c, Fair[k] >= 0 && Fair[k] < nVair, "oc_set_air_mesh: bad Fair");
    const int nVt = c->nV + nVair - nBnd;
    c->nVair = nVair;
    c->nFair = nFair;
    c->nBnd = nBnd;
    c->wScaf = wScaf;
    std::vector<int> l2g(nVair);
    for (int l = 0; l < nVair; ++l) l2g[l] = l < nBnd ? bnd[l] : c->nV + l - nBnd;
    c->FairGlobal.resize(3 * (size_t)nFair);
    for (long k = 0; k < 3L * nFair; ++k) c->FairGlobal[k] = l2g[Fair[k]];
    c->FairLocal.assign(Fair, Fair + 3 * (size_t)nFair);
    c->airAreaThres = areaThres;
    c->airSinceRemesh = 0;
    c->airLimited = false;
    c->airL2G = l2g;
    if (upload(c, c->dAirL2G, c->airL2G)) return OC_ERR_HIP;
    OC_HIP(c, c->dAirUV2.ensure(sizeof(double) * 2 * (size_t)nVair));
    c->airFixedGlobal.assign(nVt, 0);
    for (int l = 0; l < nBnd; ++l)
        if (c->fixedMaskMesh[bnd[l]]) c->airFixedGlobal[bnd[l]] = 1;

    if (int st = ensure_tri_storage(c, c->nF + nFair)) return st;
    // air rest features from its own rest shape (UV, z = 0) and local indices
    std::vector<double> vr(3 * (size_t)nVair);
    for (int l = 0; l < nVair; ++l) {
        vr[3 * l] = airUV[2 * l];
        vr[3 * l + 1] = airUV[2 * l + 1];
        vr[3 * l + 2] = 0.0;
    }
    if (upload(c, c->dTmpVrest, vr)) return OC_ERR_HIP;
    if (int st = upload_tri_ids(c, c->nF, nFair, Fair)) return st;  // local ids first, for the features
    OC_HIP(c, c->dAirSums.ensure(sizeof(double) * 4));
    if (ensure_scratch(c, nFair)) return OC_ERR_HIP;
    const int o = c->nF;
    oc::launch_rest_features(c->stream, nFair, c->dF0.as<int>() + o, c->dF1.as<int>() + o, c->dF2.as<int>() + o,
                             c->dTmpVrest.as<double>(), areaThres, c->dTriArea.as<double>() + o,
                             c->dA2.as<double>() + o, c->dE0.as<double>() + o, c->dE1.as<double>() + o,
                             c->dE01.as<double>() + o, c->dPartials.as<double>(), c->dAirSums.as<double>());
    OC_HIP(c, hipGetLastError());
    double sums[3];
    OC_HIP(c, hipMemcpyAsync(sums, c->dAirSums.p, sizeof(sums), hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    if (sums[2] > 0.0) {
        c->err = "an air-mesh triangle has zero area";
        return OC_ERR_DEGENERATE;
    }
    if (int st = upload_tri_ids(c, c->nF, nFair, c->FairGlobal.data())) return st;
    // combined UV: keep the mesh part, append the interior air vertices (two buffers alternate, so an air-mesh
    // change allocates only when the combined size outgrows them)
    DevBuf& nu = c->dUVspare;
    OC_HIP(c, nu.ensure(sizeof(double) * 2 * (size_t)nVt));
    OC_HIP(c, hipMemcpyAsync(nu.p, c->dUV.p, sizeof(double) * 2 * (size_t)c->nV, hipMemcpyDeviceToDevice, c->stream));
    if (nVair > nBnd)
        OC_HIP(c, hipMemcpyAsync(nu.as<double>() + 2 * (size_t)c->nV, airUV + 2 * (size_t)nBnd,
                                 sizeof(double) * 2 * (size_t)(nVair - nBnd), hipMemcpyHostToDevice, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    std::swap(c->dUV.p, nu.p);
    std::swap(c->dUV.bytes, nu.bytes);
    return OC_OK;
}

// ---- LinSysSolver drop-in ------------------------------------------------------------
int oc_solver_set_pattern(oc_ctx* c, int nV, const int* nbrPtr, const int* nbr, int nFixed, const int* fixedV,
                          int* nnz)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, nV > 0 && nbrPtr && nbr && nFixed >= 0 && (nFixed == 0 || fixedV), "oc_solver_set_pattern: bad args");
    (void)hipSetDevice(c->device);
    std::vector<unsigned char> isFixed(nV, 0);
    for (int k = 0; k < nFixed; ++k) {
        OC_ARG(c, fixedV[k] >= 0 && fixedV[k] < nV, "oc_solver_set_pattern: fixed id out of range");
        isFixed[fixedV[k]] = 1;
    }
    // reference upper CSR (LinSysSolver.hpp:37-135), 0-based
    std::vector<int>& ia = c->solIa;
    std::vector<int>& ja = c->solJa;
    ia.assign(2 * (size_t)nV + 1, 0);
    ja.clear();
    std::vector<std::vector<int>> rows(nV);
    for (int v = 0; v < nV; ++v) {
        std::vector<int> nb(nbr + nbrPtr[v], nbr + nbrPtr[v + 1]);
        for (int w : nb) OC_ARG(c, w >= 0 && w < nV, "oc_solver_set_pattern: neighbour out of range");
        std::sort(nb.begin(), nb.end());
        nb.erase(std::unique(nb.begin(), nb.end()), nb.end());
        if (!isFixed[v]) {
            std::vector<int> rowx = {2 * v, 2 * v + 1};
            for (int w : nb)
                if (!isFixed[w] && w > v) {
                    rowx.push_back(2 * w);
                    rowx.push_back(2 * w + 1);
                }
            for (int x : rowx) ja.push_back(x);
            ia[2 * v + 1] = ia[2 * v] + (int)rowx.size();
            for (size_t k = 1; k < rowx.size(); ++k) ja.push_back(rowx[k]);
            ia[2 * v + 2] = ia[2 * v + 1] + (int)rowx.size() - 1;
        } else {
            ja.push_back(2 * v);
            ja.push_back(2 * v + 1);
            ia[2 * v + 1] = ia[2 * v] + 1;
            ia[2 * v + 2] = ia[2 * v + 1] + 1;
        }
    }
    // block rows of the full symmetric matrix
    for (int i = 0; i < 2 * nV; ++i)
        for (int k = ia[i]; k < ia[i + 1]; ++k) {
            const int u = i / 2, w = ja[k] / 2;
            rows[u].push_back(w);
            rows[w].push_back(u);
        }
    for (int v = 0; v < nV; ++v) {
        auto& r = rows[v];
        r.push_back(v);
        std::sort(r.begin(), r.end());
        r.erase(std::unique(r.begin(), r.end()), r.end());
    }
    std::vector<unsigned char> noFixed(nV, 0);  // the rows above already exclude fixed couplings
    build_block_pattern(c->sol, nV, rows, noFixed);
    const int nnzU = (int)ja.size();
    c->solDst.resize(nnzU);
    c->solMir.resize(nnzU);
    for (int i = 0; i < 2 * nV; ++i)
        for (int k = ia[i]; k < ia[i + 1]; ++k) {
            const int j = ja[k];
            const int u = i / 2, w = j / 2, ri = i % 2, cj = j % 2;
            const int P = c->sol.find(u, w);
            c->solDst[k] = 4 * P + 2 * ri + cj;
            if (u != w) c->solMir[k] = 4 * c->sol.find(w, u) + 2 * cj + ri;
            else c->solMir[k] = (ri != cj) ? 4 * P + 2 * cj + ri : -1;
        }
    c->solN = 2 * nV;
    c->solA.assign(nnzU, 0.0);
    c->solFixed = isFixed;
    c->solAmgStruct = false;
    c->solIc0Struct = false;
    c->solHaveUV = false;
    if (upload_pattern(c, c->sol)) return OC_ERR_HIP;
    if (upload(c, c->dSolDst, c->solDst) || upload(c, c->dSolMir, c->solMir)) return OC_ERR_HIP;
    OC_HIP(c, c->dSolA.ensure(sizeof(double) * (size_t)std::max(1, nnzU)));
    OC_HIP(c, c->dSolB.ensure(sizeof(double) * 2 * (size_t)nV));
    OC_HIP(c, c->dSolX.ensure(sizeof(double) * 2 * (size_t)nV));
    OC_HIP(c, c->dSolUV.ensure(sizeof(double) * 2 * (size_t)nV));
    OC_HIP(c, hipMemsetAsync(c->dSolUV.p, 0, sizeof(double) * 2 * (size_t)nV, c->stream));
    if (ensure_pcg(c, nV)) return OC_ERR_HIP;
    OC_HIP(c, hipStreamSynchronize(c->stream));
    c->solFactorized = false;
    if (nnz) *nnz = nnzU;
    return OC_OK;
}

int oc_solver_get_pattern(oc_ctx* c, int* ia, int* ja)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->solN > 0 && ia && ja, "oc_solver_get_pattern: no pattern");
    std::copy(c->solIa.begin(), c->solIa.end(), ia);
    std::copy(c->solJa.begin(), c->solJa.end(), ja);
    return OC_OK;
}

static int upload_sol_a_impl(oc_ctx* c);
static int upload_sol_a(oc_ctx* c) { return upload_sol_a_impl(c); }

int oc_solver_update_a(oc_ctx* c, long long nT, const int* I, const int* J, const double* V)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->solN > 0, "oc_solver_update_a: no pattern");
    OC_ARG(c, nT >= 0 && (nT == 0 || (I && J && V)), "oc_solver_update_a: bad triplets");
    (void)hipSetDevice(c->device);
    std::fill(c->solA.begin(), c->solA.end(), 0.0);
    const int* ia = c->solIa.data();
    const int* ja = c->solJa.data();
    for (long long k = 0; k < nT; ++k) {
        const int i = I[k], j = J[k];
        if (i > j) continue;
        if (i < 0 || j >= c->solN) {
            c->err = "oc_solver_update_a: triplet index out of range";
            return OC_ERR_PATTERN;
        }
        const int* b = ja + ia[i];
        const int* e = ja + ia[i + 1];
        const int* p = std::lower_bound(b, e, j);
        if (p == e || *p != j) {
            c->err = "oc_solver_update_a: triplet outside the pattern";
            return OC_ERR_PATTERN;
        }
        c->solA[p - ja] += V[k];
    }
    return upload_sol_a(c);
}

static int upload_sol_a_impl(oc_ctx* c)
{
    const int nnz = (int)c->solA.size();
    OC_HIP(c, hipMemcpyAsync(c->dSolA.p, c->solA.data(), sizeof(double) * nnz, hipMemcpyHostToDevice, c->stream));
    OC_HIP(c, hipMemsetAsync(c->sol.dVals.p, 0, sizeof(double) * 4 * (size_t)c->sol.nnzb(), c->stream));
    oc::launch_expand_upper(c->stream, nnz, c->dSolA.as<double>(), c->dSolDst.as<int>(), c->dSolMir.as<int>(),
                            c->sol.dVals.as<double>());
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipStreamSynchronize(c->stream));
    c->solFactorized = false;
    return OC_OK;
}

int oc_solver_set_a(oc_ctx* c, const double* a)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->solN > 0 && a, "oc_solver_set_a: no pattern");
    (void)hipSetDevice(c->device);
    std::copy(a, a + c->solA.size(), c->solA.begin());
    return upload_sol_a(c);
}

int oc_solver_get_a(oc_ctx* c, double* a)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->solN > 0 && a, "oc_solver_get_a: no pattern");
    std::copy(c->solA.begin(), c->solA.end(), a);
    return OC_OK;
}

int oc_solver_analyze_pattern(oc_ctx* c)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->solN > 0, "oc_solver_analyze_pattern: no pattern");
    return OC_OK;
}

int oc_solver_factorize(oc_ctx* c)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->solN > 0, "oc_solver_factorize: no pattern");
    (void)hipSetDevice(c->device);
    oc::launch_jacobi_from_bsr(c->stream, c->sol.nV, c->sol.dDiagPos.as<int>(), c->sol.dVals.as<double>(),
                               c->sol.dMinv.as<double>(), c->solPrecond == OC_PRECOND_BLOCK_JACOBI);
    OC_HIP(c, hipGetLastError());
    if (c->solPrecond == OC_PRECOND_AMG) {
        if (!c->solAmgStruct) {
            std::string e;
            if (c->amgSol.setup(c->stream, c->sol.nV, c->sol.rowPtr, c->sol.colIdx, c->solFixed, e) != 0) {
                c->err = "oc_solver_factorize: " + e;
                return OC_ERR_HIP;
            }
            c->solAmgStruct = true;
        }
        c->amgSol.numeric(c->stream, c->sol.dVals.as<double>(), c->dSolUV.as<double>());
        OC_HIP(c, hipGetLastError());
    }
    if (c->solPrecond == OC_PRECOND_IC0) {
        if (!c->solIc0Struct) {
            std::string e;
            if (c->ic0Sol.setup(c->stream, c->sol.nV, c->sol.rowPtr, c->sol.colIdx, e) != 0) {
                c->err = "oc_solver_factorize: " + e;
                return OC_ERR_HIP;
            }
            c->solIc0Struct = true;
        }
        c->ic0Sol.numeric(c->stream, c->sol.dVals.as<double>());
        OC_HIP(c, hipGetLastError());
    }
    OC_HIP(c, hipStreamSynchronize(c->stream));
    c->solFactorized = true;
    return OC_OK;
}

int oc_solver_set_coords(oc_ctx* c, const double* UV)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->solN > 0 && UV, "oc_solver_set_coords: no pattern");
    (void)hipSetDevice(c->device);
    OC_HIP(c, hipMemcpyAsync(c->dSolUV.p, UV, sizeof(double) * c->solN, hipMemcpyHostToDevice, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    c->solHaveUV = true;
    c->solFactorized = false;
    return OC_OK;
}

int oc_solver_solve(oc_ctx* c, const double* rhs, double* x)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->solN > 0 && rhs && x, "oc_solver_solve: no pattern");
    if (!c->solFactorized) {
        c->err = "oc_solver_solve: factorize first";
        return OC_ERR_STATE;
    }
    (void)hipSetDevice(c->device);
    OC_HIP(c, hipMemcpyAsync(c->dSolB.p, rhs, sizeof(double) * c->solN, hipMemcpyHostToDevice, c->stream));
    int it;
    double rr;
    c->solFallback = 0;
    int st;
    if (c->solPrecond == OC_PRECOND_AMG) {
        // multigrid; on a breakdown (an indefinite V-cycle from a low eigenvalue estimate) the hierarchy is
        // rebuilt with the guaranteed Gershgorin interval, then Jacobi-PCG takes over
        st = run_pcg(c, c->sol, c->dSolB.as<double>(), c->solTol, c->solMaxIter, it, rr, &c->amgSol);
        if (st == OC_ERR_BREAKDOWN) {
            int it2;
            c->amgSol.numeric(c->stream, c->sol.dVals.as<double>(), c->dSolUV.as<double>(), 1);
            OC_HIP(c, hipGetLastError());
            c->solFallback = 1;
            st = run_pcg(c, c->sol, c->dSolB.as<double>(), c->solTol, c->solMaxIter, it2, rr, &c->amgSol);
            it += it2;
        }
        if (st == OC_ERR_BREAKDOWN) {
            int it2;
            c->solFallback = 2;
            st = run_pcg(c, c->sol, c->dSolB.as<double>(), c->solTol, c->solMaxIter, it2, rr);
            it += it2;
        }
    } else if (c->solPrecond == OC_PRECOND_IC0) {
        // block IC(0); on a breakdown Jacobi-PCG takes over
        st = run_pcg(c, c->sol, c->dSolB.as<double>(), c->solTol, c->solMaxIter, it, rr, &c->ic0Sol);
        if (st == OC_ERR_BREAKDOWN) {
            int it2;
            c->solFallback = 2;
            st = run_pcg(c, c->sol, c->dSolB.as<double>(), c->solTol, c->solMaxIter, it2, rr);
            it += it2;
        }
    } else {
        st = run_pcg(c, c->sol, c->dSolB.as<double>(), c->solTol, c->solMaxIter, it, rr);
    }
    c->lastIters = it;
    c->lastRelRes = rr;
    if (st != OC_OK && st != OC_ERR_NOT_CONVERGED) return st;
    OC_HIP(c, hipMemcpyAsync(x, c->dX.p, sizeof(double) * c->solN, hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return st;
}

int oc_solver_multiply(oc_ctx* c, const double* x, double* Ax)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->solN > 0 && x && Ax, "oc_solver_multiply: no pattern");
    (void)hipSetDevice(c->device);
    OC_HIP(c, hipMemcpyAsync(c->dSolB.p, x, sizeof(double) * c->solN, hipMemcpyHostToDevice, c->stream));
    oc::launch_spmv(c->stream, c->sol.nV, c->sol.dRowPtr.as<int>(), c->sol.dColIdx.as<int>(),
                    c->sol.dVals.p, 0, c->dSolB.as<double>(), c->dSolX.as<double>());
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipMemcpyAsync(Ax, c->dSolX.p, sizeof(double) * c->solN, hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return OC_OK;
}

int oc_solver_apply_precond(oc_ctx* c, const double* r, double* z)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->solN > 0 && r && z, "oc_solver_apply_precond: no pattern");
    if (!c->solFactorized) {
        c->err = "oc_solver_apply_precond: factorize first";
        return OC_ERR_STATE;
    }
    (void)hipSetDevice(c->device);
    OC_HIP(c, c->dPcgPart.ensure(sizeof(double) * (size_t)kRzRecords));
    OC_HIP(c, hipMemcpyAsync(c->dSolB.p, r, sizeof(double) * c->solN, hipMemcpyHostToDevice, c->stream));
    oc::Preconditioner* M = c->solPrecond == OC_PRECOND_AMG ? static_cast<oc::Preconditioner*>(&c->amgSol)
                            : c->solPrecond == OC_PRECOND_IC0 ? static_cast<oc::Preconditioner*>(&c->ic0Sol)
                                                               : nullptr;
    if (!M) {
        c->err = "oc_solver_apply_precond: OC_PRECOND_AMG or OC_PRECOND_IC0 only";
        return OC_ERR_STATE;
    }
    M->apply(c->stream, c->dSolB.as<double>(), c->dSolX.as<double>(), c->dPcgPart.as<double>(), nullptr);
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipMemcpyAsync(z, c->dSolX.p, sizeof(double) * c->solN, hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return OC_OK;
}

int oc_ic0_set_sweeps(oc_ctx* c, int factorSweeps, int applySweeps)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, factorSweeps >= 0 && factorSweeps <= 100000 && applySweeps >= 0 && applySweeps <= 100000,
           "oc_ic0_set_sweeps: bad sweep counts");
    c->ic0.set_sweeps(factorSweeps, applySweeps);
    c->ic0Sol.set_sweeps(factorSweeps, applySweeps);
    c->solFactorized = false;
    return OC_OK;
}

int oc_amg_set_tail(oc_ctx* c, int maxNodes)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, maxNodes >= -1 && maxNodes <= 100000, "oc_amg_set_tail: bad node count");
    for (oc::AmgBase* a : {static_cast<oc::AmgBase*>(&c->amg64), static_cast<oc::AmgBase*>(&c->amg32),
                           static_cast<oc::AmgBase*>(&c->amgTut), static_cast<oc::AmgBase*>(&c->amgSol)})
        a->set_tail_max(maxNodes);
    c->solFactorized = false;
    return OC_OK;
}

int oc_solver_set_params(oc_ctx* c, int precond, double relTol, int maxIter)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, (precond == OC_PRECOND_JACOBI || precond == OC_PRECOND_BLOCK_JACOBI || precond == OC_PRECOND_AMG ||
               precond == OC_PRECOND_IC0) &&
                  relTol > 0.0 && maxIter > 0,
           "oc_solver_set_params: bad parameters");
    c->solPrecond = precond;
    c->solTol = relTol;
    c->solMaxIter = maxIter;
    c->solFactorized = false;
    return OC_OK;
}

int oc_solver_last_stats(oc_ctx* c, int* iters, double* relResidual)
{
    if (!c) return OC_ERR_ARG;
    if (iters) *iters = c->lastIters;
    if (relResidual) *relResidual = c->lastRelRes;
    return OC_OK;
}

int oc_solver_last_fallback(oc_ctx* c, int* fallback)
{
    if (!c || !fallback) return OC_ERR_ARG;
    *fallback = c->solFallback;
    return OC_OK;
}

// ---- Tutte initial map (main.cpp:1317-1364) -----------------------------------------
namespace {

// Boundary topology of a triangle mesh for the Tutte map: triangle edge
// (F(f,i), F(f,i+1)) is a boundary edge when no other triangle holds it
// (triangle_triangle_adjacency.cpp); vertex -> triangles in ascending order
// (vertex_triangle_adjacency.cpp); edge-connected components numbered in order
// of their lowest triangle (facet_components.cpp).
struct LoopTopology {
    int nV = 0, nF = 0, nComp = 0;
    const int* F = nullptr;
    std::vector<int> tt;           // 3 per triangle: neighbour across edge i, -1 on the boundary
    std::vector<char> faceHasBnd;  // triangle has a boundary edge
    std::vector<int> vfPtr, vf;
    std::vector<int> comp;  // per triangle

    // 0, or -1 for an edge held by three or more triangles
    int build(int nV_, int nF_, const int* F_)
    {
        nV = nV_;
        nF = nF_;
        F = F_;
        struct E {
            int a, b, f, i;
        };
        std::vector<E> es;
        es.reserve(3 * (size_t)nF);
        for (int f = 0; f < nF; ++f)
            for (int i = 0; i < 3; ++i) {
                int a = F[3 * (size_t)f + i], b = F[3 * (size_t)f + (i + 1) % 3];
                if (a > b) std::swap(a, b);
                es.push_back(E{a, b, f, i});
            }
        std::sort(es.begin(), es.end(), [](const E& x, const E& y) {
            return x.a != y.a ? x.a < y.a : (x.b != y.b ? x.b < y.b : (x.f != y.f ? x.f < y.f : x.i < y.i));
        });
        tt.assign(3 * (size_t)nF, -1);
        for (size_t k = 0; k < es.size();) {
            size_t e = k + 1;
            while (e < es.size() && es[e].a == es[k].a && es[e].b == es[k].b) ++e;
            if (e - k > 2) return -1;
            if (e - k == 2) {
                tt[3 * (size_t)es[k].f + es[k].i] = es[k + 1].f;
                tt[3 * (size_t)es[k + 1].f + es[k + 1].i] = es[k].f;
            }
            k = e;
        }
        faceHasBnd.assign(nF, 0);
        for (int f = 0; f < nF; ++f)
            for (int i = 0; i < 3; ++i)
                if (tt[3 * (size_t)f + i] < 0) faceHasBnd[f] = 1;
        vfPtr.assign(nV + 1, 0);
        vf.resize(3 * (size_t)nF);
        for (int f = 0; f < nF; ++f)
            for (int i = 0; i < 3; ++i) vfPtr[F[3 * (size_t)f + i] + 1]++;
        for (int v = 0; v < nV; ++v) vfPtr[v + 1] += vfPtr[v];
        std::vector<int> fill(vfPtr.begin(), vfPtr.end() - 1);
        for (int f = 0; f < nF; ++f)
            for (int i = 0; i < 3; ++i) vf[fill[F[3 * (size_t)f + i]]++] = f;
        comp.assign(nF, -1);
        nComp = 0;
        std::vector<int> queue;
        for (int g = 0; g < nF; ++g) {
            if (comp[g] >= 0) continue;
            comp[g] = nComp;
            queue.assign(1, g);
            while (!queue.empty()) {
                const int f = queue.back();
                queue.pop_back();
                for (int i = 0; i < 3; ++i) {
                    const int h = tt[3 * (size_t)f + i];
                    if (h >= 0 && comp[h] < 0) {
                        comp[h] = nComp;
                        queue.push_back(h);
                    }
                }
            }
            ++nComp;
        }
        return 0;
    }

    // Loops of the triangles of component `which` (-1: all triangles) as
    // libigl's boundary_loop walks them (boundary_loop.cpp): a loop starts at
    // the smallest unvisited border vertex and moves on through the first
    // triangle (ascending) whose boundary edge leaves the current vertex to an
    // unvisited one. `starts` lists the border vertices of those triangles in
    // ascending order; `unvisited` is all zero on entry and on return.
    void walk(int which, const std::vector<int>& starts, std::vector<char>& unvisited,
              std::vector<std::vector<int>>& loops) const
    {
        for (int v : starts) unvisited[v] = 1;
        for (int start : starts) {
            if (!unvisited[start]) continue;
            std::vector<int> loop(1, start);
            unvisited[start] = 0;
            for (;;) {
                const int v = loop.back();
                int next = -1;
                for (int q = vfPtr[v]; q < vfPtr[v + 1] && next < 0; ++q) {
                    const int f = vf[q];
                    if (!faceHasBnd[f] || (which >= 0 && comp[f] != which)) continue;
                    int loc = 0;
                    while (F[3 * (size_t)f + loc] != v) ++loc;
                    const int vn = F[3 * (size_t)f + (loc + 1) % 3];
                    if (unvisited[vn] && tt[3 * (size_t)f + loc] < 0) next = vn;
                }
                if (next < 0) break;
                loop.push_back(next);
                unvisited[next] = 0;
            }
            loops.push_back(std::move(loop));
        }
    }

    // The loops the Tutte map pins: layout 0 = the first longest loop of each
    // component (main.cpp:1486-1512), layout 1 = every loop (main.cpp:1313-1317).
    // Returns -1 - k when component k has no boundary.
    int tutte_loops(int layout, std::vector<std::vector<int>>& out) const
    {
        out.clear();
        std::vector<char> unvisited(nV, 0);
        if (layout == 1) {
            std::vector<char> mark(nV, 0);
            for (int f = 0; f < nF; ++f)
                for (int i = 0; i < 3; ++i)
                    if (tt[3 * (size_t)f + i] < 0)
                        mark[F[3 * (size_t)f + i]] = mark[F[3 * (size_t)f + (i + 1) % 3]] = 1;
            std::vector<int> starts;
            for (int v = 0; v < nV; ++v)
                if (mark[v]) starts.push_back(v);
            walk(-1, starts, unvisited, out);
            return out.empty() ? -1 : 0;
        }
        std::vector<std::vector<int>> starts(nComp);
        for (int f = 0; f < nF; ++f)
            for (int i = 0; i < 3; ++i)
                if (tt[3 * (size_t)f + i] < 0) {
                    starts[comp[f]].push_back(F[3 * (size_t)f + i]);
                    starts[comp[f]].push_back(F[3 * (size_t)f + (i + 1) % 3]);
                }
        std::vector<std::vector<int>> loops;
        for (int k = 0; k < nComp; ++k) {
            auto& st = starts[k];
            std::sort(st.begin(), st.end());
            st.erase(std::unique(st.begin(), st.end()), st.end());
            loops.clear();
            walk(k, st, unvisited, loops);
            if (loops.empty()) return -1 - k;
            size_t best = 0;
            for (size_t b = 1; b < loops.size(); ++b)
                if (loops[best].size() < loops[b].size()) best = b;
            out.push_back(std::move(loops[best]));
        }
        return 0;
    }
};

}  // namespace

int oc_tutte(oc_ctx* c, int layout, int precond, double relTol, int maxIter, double* UVout, int* nLoops,
             int* nBnd, int* iters)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0, "oc_tutte: no mesh");
    OC_ARG(c, (layout == OC_TUTTE_COMPONENTS || layout == OC_TUTTE_ALL_LOOPS) && relTol > 0.0 && maxIter > 0 &&
                  (precond == OC_PRECOND_JACOBI || precond == OC_PRECOND_AMG),
           "oc_tutte: bad parameters");
    (void)hipSetDevice(c->device);
    const int nV = c->nV, nF = c->nF;
    LoopTopology topo;
    if (topo.build(nV, nF, c->Fh.data()) != 0) {
        c->err = "oc_tutte: an edge is shared by more than two triangles";
        return OC_ERR_ARG;
    }
    std::vector<std::vector<int>> loops;
    const int lr = topo.tutte_loops(layout, loops);
    if (lr != 0) {
        c->err = layout == OC_TUTTE_ALL_LOOPS
                     ? std::string("oc_tutte: the mesh has no boundary")
                     : "oc_tutte: component " + std::to_string(-1 - lr) + " has no boundary";
        return OC_ERR_STATE;
    }
    // loop k on the unit circle by arc length of the rest positions
    // (map_vertices_to_circle.cpp), shifted by (k % d, k / d) * 2.1 with d the
    // smallest integer with d * d >= number of loops (main.cpp:1335-1357)
    auto dist = [&](int a, int b) {
        double s2 = 0.0;
        for (int j = 0; j < 3; ++j) {
            const double d = c->Vh[3 * (size_t)a + j] - c->Vh[3 * (size_t)b + j];
            s2 += d * d;
        }
        return std::sqrt(s2);
    };
    int grid = 0;
    do {
        ++grid;
    } while (grid * grid < (int)loops.size());
    std::vector<double> bc(2 * (size_t)nV, 0.0);
    std::vector<unsigned char> isB(nV, 0);
    int nb = 0;
    for (size_t k = 0; k < loops.size(); ++k) {
        const std::vector<int>& bnd = loops[k];
        const int n = (int)bnd.size();
        std::vector<double> len(n, 0.0);
        for (int i = 1; i < n; ++i) len[i] = len[i - 1] + dist(bnd[i - 1], bnd[i]);
        const double total = len[n - 1] + dist(bnd[0], bnd[n - 1]);
        const double xo = (double)(k % grid) * 2.1, yo = (double)(k / grid) * 2.1;
        for (int i = 0; i < n; ++i) {
            if (isB[bnd[i]]) {
                c->err = "oc_tutte: vertex " + std::to_string(bnd[i]) + " lies on two boundary loops";
                return OC_ERR_ARG;
            }
            const double a = len[i] * 2.0 * M_PI / total;
            bc[2 * (size_t)bnd[i]] = std::cos(a) + xo;
            bc[2 * (size_t)bnd[i] + 1] = std::sin(a) + yo;
            isB[bnd[i]] = 1;
        }
        nb += n;
    }
    // Q = -L for the uniform Laplacian (IglUtils.cpp:39-60): per triangle +1 on
    // both directions of each edge, -2 per corner, negated; igl::harmonic with
    // k = 1 solves Q_II W_I = -Q_IB bc (harmonic.cpp, min_quad_with_fixed).
    std::vector<std::vector<int>> rows(nV);
    for (int t = 0; t < nF; ++t)
        for (int a = 0; a < 3; ++a)
            for (int b = 0; b < 3; ++b) rows[c->Fh[3 * (size_t)t + a]].push_back(c->Fh[3 * (size_t)t + b]);
    for (int v = 0; v < nV; ++v) {
        auto& r = rows[v];
        r.push_back(v);
        std::sort(r.begin(), r.end());
        r.erase(std::unique(r.begin(), r.end()), r.end());
    }
    BlockPattern& P = c->tut;
    build_block_pattern(P, nV, rows, isB);
    rows.clear();
    std::vector<double> q(P.nnzb(), 0.0), b(2 * (size_t)nV, 0.0);
    for (int t = 0; t < nF; ++t) {
        const int* f = &c->Fh[3 * (size_t)t];
        for (int e = 0; e < 3; ++e) {
            const int u = f[e], w = f[(e + 1) % 3];
            for (int dir = 0; dir < 2; ++dir) {
                const int r = dir ? w : u, col = dir ? u : w;
                if (isB[r]) continue;
                if (isB[col]) {  // known boundary value: to the right-hand side
                    b[2 * (size_t)r] += bc[2 * (size_t)col];
                    b[2 * (size_t)r + 1] += bc[2 * (size_t)col + 1];
                } else {
                    q[P.find(r, col)] -= 1.0;
                }
            }
            if (!isB[u]) q[P.diagPos[u]] += 2.0;
        }
    }
    for (int v = 0; v < nV; ++v)
        if (!isB[v] && q[P.diagPos[v]] == 0.0) {
            c->err = "oc_tutte: vertex " + std::to_string(v) + " is in no triangle";
            return OC_ERR_ARG;
        }
    for (int v = 0; v < nV; ++v)
        if (isB[v]) {
            q[P.diagPos[v]] = 1.0;
            b[2 * (size_t)v] = bc[2 * (size_t)v];
            b[2 * (size_t)v + 1] = bc[2 * (size_t)v + 1];
        }
    std::vector<double> vals(4 * (size_t)P.nnzb());
    for (long k = 0; k < P.nnzb(); ++k) {
        vals[4 * k] = q[k];
        vals[4 * k + 1] = 0.0;
        vals[4 * k + 2] = 0.0;
        vals[4 * k + 3] = q[k];
    }
    if (upload_pattern(c, P)) return OC_ERR_HIP;
    P.vals32 = 0;
    OC_HIP(c, hipMemcpyAsync(P.dVals.p, vals.data(), sizeof(double) * vals.size(), hipMemcpyHostToDevice, c->stream));
    if (ensure_pcg(c, nV)) return OC_ERR_HIP;
    OC_HIP(c, hipMemcpyAsync(c->dB.p, b.data(), sizeof(double) * b.size(), hipMemcpyHostToDevice, c->stream));
    oc::launch_jacobi_from_bsr(c->stream, nV, P.dDiagPos.as<int>(), P.dVals.as<double>(), P.dMinv.as<double>(), 0);
    oc::Preconditioner* pre = nullptr;
    if (precond == OC_PRECOND_AMG) {
        std::string e;
        if (c->amgTut.setup(c->stream, nV, P.rowPtr, P.colIdx, isB, e) != 0) {
            c->err = e;
            return OC_ERR_HIP;
        }
        // rigid-motion near-null space at the boundary-initialised positions,
        // staged in the solution buffer (the solve starts from zero after it)
        OC_HIP(c, hipMemcpyAsync(c->dX.p, bc.data(), sizeof(double) * bc.size(), hipMemcpyHostToDevice, c->stream));
        c->amgTut.numeric(c->stream, P.dVals.as<double>(), c->dX.as<double>());
        pre = &c->amgTut;
    }
    OC_HIP(c, hipGetLastError());
    int it = 0;
    double rr = 0.0;
    int st = run_pcg(c, P, c->dB.as<double>(), relTol, maxIter, it, rr, pre);
    if (iters) *iters = it;
    if (st != OC_OK) return st;
    // boundary values exactly as placed (the solve meets them to its tolerance)
    std::vector<double> uv(2 * (size_t)nV);
    OC_HIP(c, hipMemcpyAsync(uv.data(), c->dX.p, sizeof(double) * uv.size(), hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    for (int v = 0; v < nV; ++v)
        if (isB[v]) {
            uv[2 * (size_t)v] = bc[2 * (size_t)v];
            uv[2 * (size_t)v + 1] = bc[2 * (size_t)v + 1];
        }
    OC_HIP(c, hipMemcpyAsync(c->dUV.p, uv.data(), sizeof(double) * uv.size(), hipMemcpyHostToDevice, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    if (UVout) std::copy(uv.begin(), uv.end(), UVout);
    if (nBnd) *nBnd = nb;
    if (nLoops) *nLoops = (int)loops.size();
    c->sysReady = false;
    return OC_OK;
}

// ---- batched charts -------------------------------------------------------------------
int oc_set_charts(oc_ctx* c, int nCharts, const int* vertexStart, const int* faceStart)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0, "oc_set_charts: no mesh");
    OC_ARG(c, c->nFair == 0, "oc_set_charts: not available with an air mesh");
    OC_ARG(c, nCharts >= 1 && vertexStart && faceStart, "oc_set_charts: bad arguments");
    OC_ARG(c, vertexStart[0] == 0 && vertexStart[nCharts] == c->nV && faceStart[0] == 0 &&
                  faceStart[nCharts] == c->nF,
           "oc_set_charts: ranges must cover all vertices and triangles");
    for (int k = 0; k < nCharts; ++k)
        OC_ARG(c, vertexStart[k + 1] > vertexStart[k] && faceStart[k + 1] > faceStart[k],
               "oc_set_charts: every chart needs vertices and triangles");
    std::vector<int> vChart(c->nV), triChart(c->nF);
    for (int k = 0; k < nCharts; ++k) {
        for (int v = vertexStart[k]; v < vertexStart[k + 1]; ++v) vChart[v] = k;
        for (int t = faceStart[k]; t < faceStart[k + 1]; ++t) {
            triChart[t] = k;
            for (int j = 0; j < 3; ++j) {
                const int v = c->Fh[3 * (size_t)t + j];
                OC_ARG(c, v >= vertexStart[k] && v < vertexStart[k + 1],
                       "oc_set_charts: a triangle uses a vertex of another chart");
            }
        }
    }
    (void)hipSetDevice(c->device);
    c->sysReady = false;
    c->chartV.assign(vertexStart, vertexStart + nCharts + 1);
    c->chartF.assign(faceStart, faceStart + nCharts + 1);
    // chart-aligned triangle blocks
    std::vector<int2> blk;
    std::vector<int> blkChart;
    c->chartBlk.assign(nCharts + 1, 0);
    for (int k = 0; k < nCharts; ++k) {
        for (int t0 = faceStart[k]; t0 < faceStart[k + 1]; t0 += oc::kBlock) {
            int2 r;
            r.x = t0;
            r.y = std::min(t0 + oc::kBlock, faceStart[k + 1]);
            blk.push_back(r);
            blkChart.push_back(k);
        }
        c->chartBlk[k + 1] = (int)blk.size();
    }
    if (upload(c, c->dChartV, c->chartV) || upload(c, c->dChartF, c->chartF) || upload(c, c->dChartBlk, c->chartBlk) ||
        upload(c, c->dBlkChart, blkChart) || upload(c, c->dVChart, vChart) || upload(c, c->dTriChart, triChart))
        return OC_ERR_HIP;
    OC_HIP(c, c->dBlkRange.ensure(sizeof(int2) * blk.size()));
    OC_HIP(c, hipMemcpyAsync(c->dBlkRange.p, blk.data(), sizeof(int2) * blk.size(), hipMemcpyHostToDevice, c->stream));
    const size_t nC = (size_t)nCharts;
    OC_HIP(c, c->dChartArea.ensure(sizeof(double) * nC));
    OC_HIP(c, c->dChartActive.ensure(nC));
    OC_HIP(c, c->dChartAlpha.ensure(sizeof(double) * nC));
    OC_HIP(c, c->dChartOrdMin.ensure(sizeof(unsigned long long) * nC));
    OC_HIP(c, c->dChartOut.ensure(sizeof(double) * 2 * oc::kLSCand * nC));
    OC_HIP(c, c->dChartGsq.ensure(sizeof(double) * nC));
    if (ensure_scratch(c, (long)c->nF + (long)oc::kBlock * nCharts)) return OC_ERR_HIP;
    // per-chart surface areas (the weight of chart c's triangles is area / its chart's area)
    oc::launch_chart_seg_sum(c->stream, nCharts, c->dChartF.as<int>(), c->dTriArea.as<double>(),
                             c->dChartArea.as<double>());
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipStreamSynchronize(c->stream));
    c->nCharts = nCharts;
    return OC_OK;
}

int oc_charts_state(oc_ctx* c, double* E_SD, double* gradSq, double* step, int* state)
{
    if (!c) return OC_ERR_ARG;
    if (c->nCharts == 0 || c->chartState.empty()) {
        c->err = "oc_charts_state: no batched charts initialised (oc_set_charts, oc_newton_init)";
        return OC_ERR_STATE;
    }
    for (int k = 0; k < c->nCharts; ++k) {
        if (E_SD) E_SD[k] = c->chartLastE[k] / c->a0;
        if (gradSq) gradSq[k] = c->chartGsq[k];
        if (step) step[k] = c->chartStep[k];
        if (state) state[k] = c->chartState[k];
    }
    return OC_OK;
}

// ---- Newton driver ------------------------------------------------------------------
int oc_newton_init(oc_ctx* c, double a0, double relGL2Tol, int allowEDecRelTol, int precond, double pcgRelTol,
                   int pcgMaxIter, double* E0)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0, "oc_newton_init: no mesh");
    OC_ARG(c, a0 > 0.0 && relGL2Tol > 0.0 && pcgRelTol > 0.0 && pcgMaxIter > 0 &&
                  (precond == OC_PRECOND_JACOBI || precond == OC_PRECOND_BLOCK_JACOBI || precond == OC_PRECOND_AMG ||
                   precond == OC_PRECOND_LEARNED || precond == OC_PRECOND_IC0),
           "oc_newton_init: bad parameters");
    (void)hipSetDevice(c->device);
    c->a0 = a0;
    c->relGL2Tol = relGL2Tol;
    c->allowEDecRelTol = allowEDecRelTol;
    c->nPrecond = precond;
    c->pcgTol = pcgRelTol;
    c->pcgMaxIter = pcgMaxIter;
    c->pcgHint = 0;
    c->amgSkip = 0;
    c->amgFailStreak = 0;
    c->lastStep = 0.0;  // the first solve counts as following a short step
    c->elemFp64 = false;
    c->sysPrecision = c->precision;
    // Optimizer constructor: exit(-1) on an inverted initial map (Optimizer.cpp:65-67)
    if (ensure_scratch(c, c->nF + c->nFair)) return OC_ERR_HIP;
    unsigned int ninv = 0;
    if (int st = count_inverted(c, mesh_set(c, 0), &ninv)) return st;
    if (ninv) {
        c->err = "inverted triangle in the initial UV map";
        return OC_ERR_INVERTED;
    }
    if (int st = build_system(c)) return st;
    c->targetGRes = a0 * (double)(c->nV - (int)c->fixedSorted.size()) / (double)c->nV * relGL2Tol;
    if (int st = system_energy(c, &c->lastE, &c->lastESD, &c->lastEScaf)) return st;
    if (c->nCharts > 0) {
        // per-chart targetGRes (Optimizer.cpp:675-678) and energies
        const int nC = c->nCharts;
        c->chartTarget.assign(nC, 0.0);
        for (int k = 0; k < nC; ++k) {
            int nFix = 0;
            for (int v : c->fixedSorted) nFix += v >= c->chartV[k] && v < c->chartV[k + 1];
            const int nVc = c->chartV[k + 1] - c->chartV[k];
            c->chartTarget[k] = a0 * (double)(nVc - nFix) / (double)nVc * relGL2Tol;
        }
        oc::launch_element(c->stream, mesh_set(c, 0), c->dUV.as<double>(), c->dEelem.as<double>(), nullptr, nullptr, 0,
                           nullptr, nullptr);
        oc::launch_chart_seg_sum(c->stream, nC, c->dChartF.as<int>(), c->dEelem.as<double>(),
                                 c->dChartGsq.as<double>());
        OC_HIP(c, hipGetLastError());
        c->chartLastE.assign(nC, 0.0);
        OC_HIP(c, hipMemcpyAsync(c->chartLastE.data(), c->dChartGsq.p, sizeof(double) * nC, hipMemcpyDeviceToHost,
                                 c->stream));
        OC_HIP(c, hipStreamSynchronize(c->stream));
        double e = 0.0;
        for (double& x : c->chartLastE) {
            x *= a0;
            e += x;
        }
        c->chartState.assign(nC, 0);
        c->chartGsq.assign(nC, 0.0);
        c->chartStep.assign(nC, 0.0);
        c->lastE = e;
    }
    if (E0) *E0 = c->lastE;
    if (c->trE && c->nCharts == 0)
        if (int st = write_energy_trace(c, c->lastE, c->lastESD)) return st;
    return OC_OK;
}

int oc_newton_rebuild(oc_ctx* c, double* E)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, c->nV > 0, "oc_newton_rebuild: no mesh");
    if (!c->sysBuilt || c->nCharts > 0) {
        c->err = "oc_newton_rebuild: needs an oc_newton_init of this mesh (single problem)";
        return OC_ERR_STATE;
    }
    (void)hipSetDevice(c->device);
    // Optimizer::solve rebuilds the scaffold after a step (Optimizer.cpp:251-257); the next iteration only
    // re-patterns the system (:522-530). Parameters, trace files, the previous solve's iteration count and the
    // precision escalation of the mixed learned form carry over.
    if (ensure_scratch(c, c->nF + c->nFair)) return OC_ERR_HIP;
    if (int st = build_system(c)) return st;
    if (int st = system_energy(c, &c->lastE, &c->lastESD, &c->lastEScaf)) return st;
    if (E) *E = c->lastE;
    return OC_OK;
}

int oc_air_mesh_get(oc_ctx* c, double* airUV, int* Fair)
{
    if (!c) return OC_ERR_ARG;
    if (c->nFair == 0) {
        c->err = "oc_air_mesh_get: no air mesh";
        return OC_ERR_STATE;
    }
    (void)hipSetDevice(c->device);
    if (airUV) {
        oc::launch_uv_gather(c->stream, c->nVair, c->dAirL2G.as<int>(), c->dUV.as<double>(), nullptr,
                             c->dAirUV2.as<double>());
        OC_HIP(c, hipGetLastError());
        OC_HIP(c, hipMemcpyAsync(airUV, c->dAirUV2.p, sizeof(double) * 2 * (size_t)c->nVair, hipMemcpyDeviceToHost,
                                 c->stream));
        OC_HIP(c, hipStreamSynchronize(c->stream));
    }
    if (Fair) std::copy(c->FairLocal.begin(), c->FairLocal.end(), Fair);
    return OC_OK;
}

int oc_scaffold_update(oc_ctx* c, int mode, double minAngleDeg, int maxInterval, double* E, int* flips)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, mode == OC_SCAFFOLD_REFRESH || mode == OC_SCAFFOLD_REMESH_WHEN_NEEDED || mode == OC_SCAFFOLD_REMESH,
           "oc_scaffold_update: unknown mode");
    if (c->nFair == 0 || !c->sysBuilt || c->nCharts > 0) {
        c->err = "oc_scaffold_update: needs an air mesh and an oc_newton_init";
        return OC_ERR_STATE;
    }
    (void)hipSetDevice(c->device);
    hipStream_t s = c->stream;
    long nFlips = 0;
    ++c->airSinceRemesh;
    const auto tu0 = std::chrono::steady_clock::now();
    c->tSetup[6] = 0.0;
    if (mode != OC_SCAFFOLD_REFRESH) {
        std::vector<double> P(2 * (size_t)c->nVair);
        oc::launch_uv_gather(s, c->nVair, c->dAirL2G.as<int>(), c->dUV.as<double>(), nullptr,
                             c->dAirUV2.as<double>());
        OC_HIP(c, hipGetLastError());
        OC_HIP(c, hipMemcpyAsync(P.data(), c->dAirUV2.p, sizeof(double) * P.size(), hipMemcpyDeviceToHost, s));
        OC_HIP(c, hipStreamSynchronize(s));
        if (mode == OC_SCAFFOLD_REMESH || c->airLimited || (maxInterval > 0 && c->airSinceRemesh >= maxInterval) ||
            (minAngleDeg > 0.0 && oc::air_min_angle(P, c->FairLocal) < minAngleDeg * M_PI / 180.0)) {
            c->airLimited = false;
            c->airSinceRemesh = 0;
            nFlips = oc::lawson_flips(P, c->FairLocal, 64L * c->nFair + 1024);
            c->tSetup[6] = ms_since(tu0);
            if (nFlips > 0) {
                for (size_t k = 0; k < c->FairLocal.size(); ++k) c->FairGlobal[k] = c->airL2G[c->FairLocal[k]];
                if (int st = upload_tri_ids(c, c->nF, c->nFair, c->FairGlobal.data())) return st;
                c->sysReady = false;
                if (int st = build_system(c, true)) return st;
            }
        }
    }
    // the air mesh's rest shape becomes its current UV (z = 0), as a freshly built air mesh has
    // (Scaffold.cpp:174-177); triangles below areaThres_AM take the equilateral clamp
    const int nVt = c->nVt;
    OC_HIP(c, c->dTmpVrest.ensure(sizeof(double) * 3 * (size_t)nVt));
    oc::launch_uv_gather(s, nVt, nullptr, c->dUV.as<double>(), c->dTmpVrest.as<double>(), nullptr);
    const int o = c->nF;
    oc::launch_rest_features(s, c->nFair, c->dF0.as<int>() + o, c->dF1.as<int>() + o, c->dF2.as<int>() + o,
                             c->dTmpVrest.as<double>(), c->airAreaThres, c->dTriArea.as<double>() + o,
                             c->dA2.as<double>() + o, c->dE0.as<double>() + o, c->dE1.as<double>() + o,
                             c->dE01.as<double>() + o, c->dPartials.as<double>(), c->dAirSums.as<double>());
    OC_HIP(c, hipGetLastError());
    double sums[3];
    OC_HIP(c, hipMemcpyAsync(sums, c->dAirSums.p, sizeof(sums), hipMemcpyDeviceToHost, s));
    OC_HIP(c, hipStreamSynchronize(s));
    if (sums[2] > 0.0) {
        c->err = "oc_scaffold_update: an air-mesh triangle has zero area";
        return OC_ERR_DEGENERATE;
    }
    if (int st = system_energy(c, &c->lastE, &c->lastESD, &c->lastEScaf)) return st;
    if (E) *E = c->lastE;
    if (flips) *flips = (int)nFlips;
    c->tSetup[7] = ms_since(tu0);
    return OC_OK;
}

int oc_amg_levels(oc_ctx* c, int capacity, int* nLevels, long long* rows, long long* blocks, int* blockSize)
{
    if (!c || !nLevels || capacity < 0) return OC_ERR_ARG;
    if (!c->amgValid) {
        *nLevels = 0;
        return OC_OK;
    }
    *nLevels = c->amg->levels();
    for (int l = 0; l < *nLevels && l < capacity; ++l) {
        if (rows) rows[l] = c->amg->level_rows(l);
        if (blocks) blocks[l] = c->amg->level_blocks(l);
        if (blockSize) blockSize[l] = c->amg->level_block_size(l);
    }
    return OC_OK;
}

int oc_setup_times(oc_ctx* c, double* ms)
{
    if (!c || !ms) return OC_ERR_ARG;
    std::copy(c->tSetup, c->tSetup + 8, ms);
    ms[8] = c->amgValid && c->amgOnOld ? (double)c->amgRemaps : 0.0;
    return OC_OK;
}

int oc_newton_set_learned(oc_ctx* c, oc_gnn* net)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, !net || net->device == c->device, "oc_newton_set_learned: network on another device");
    c->learned = net;
    c->sysReady = false;  // the next oc_newton_init binds it
    return OC_OK;
}

int oc_newton_set_precision(oc_ctx* c, int precision)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, precision == OC_PRECISION_FP64 || precision == OC_PRECISION_MIXED,
           "oc_newton_set_precision: unknown precision");
    c->precision = precision;
    return OC_OK;
}

int oc_newton_set_forcing(oc_ctx* c, double looseTol, double stepBelow)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, looseTol >= 0.0 && looseTol < 1.0 && stepBelow >= 0.0, "oc_newton_set_forcing: bad parameters");
    c->looseTol = looseTol;
    c->looseBelow = stepBelow;
    return OC_OK;
}

int oc_newton_set_refinement(oc_ctx* c, int maxPasses)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, maxPasses >= 0 && maxPasses <= 100, "oc_newton_set_refinement: maxPasses must be in [0, 100]");
    c->irMax = maxPasses;
    return OC_OK;
}

namespace {
// Element pass + Hessian assembly of the Newton system in the driver's precision.
// FP32 element terms in the Newton system (mixed form, not escalated)
bool system_f32(const oc_ctx* c) { return c->sysPrecision == OC_PRECISION_MIXED && !c->elemFp64; }

void system_element_pass(oc_ctx* c, const TriSet& T)
{
    const int f32 = system_f32(c);
    oc::launch_element(c->stream, T, c->dUV.as<double>(), nullptr, c->dElemG.as<double>(), c->dElemH.p, 1, nullptr,
                       nullptr, f32);
}

void system_assemble(oc_ctx* c);

// The preconditioner's numeric set-up for the assembled Newton matrix (no host synchronisation).
int launch_precond_setup(oc_ctx* c, oc_iter_stats* S)
{
    if ((c->amgPending || (c->amgRebuild && c->amgValid)) && c->amgSkip == 0)
        if (int st = amg_structure(c)) return st;
    // The multigrid hierarchy is rebuilt for every Newton matrix: reusing the
    // previous one stays a valid (SPD) preconditioner but, measured at 200k
    // faces, early Newton steps change the matrix enough to multiply the PCG
    // iterations (12 -> 733), which costs more than the set-up saved.
    if (c->amgValid && c->amgSkip == 0) {
        amg_numeric(c, 0);
        ++S->precond_setups;
    }
    if (c->nPrecond == OC_PRECOND_LEARNED) c->learned->net.forward(c->stream, c->sys.dVals.p, c->sys.vals32);
    if (c->nPrecond == OC_PRECOND_IC0) c->ic0.numeric(c->stream, c->sys.dVals.as<double>());
    return OC_OK;
}

// Jacobi-PCG for the direction (the fallback of every preconditioner), with the truncated-Newton rule when it
// meets negative curvature; iterations are added to it.
int jacobi_direction(oc_ctx* c, oc_iter_stats* S, int& it, double& rr)
{
    int it2 = 0;
    int st = run_pcg(c, c->sys, c->dB.as<double>(), c->pcgTol, std::max(c->pcgMaxIter, 200000), it2, rr, nullptr);
    it += it2;
    if (st == OC_ERR_BREAKDOWN) {
        // Negative curvature along p (the assembled matrix is not positive
        // definite): truncated Newton. The iterate before the breakdown
        // minimises the quadratic model over the Krylov space so far and is
        // a descent direction; with no iterate, steepest descent.
        if (it2 == 0)
            OC_HIP(c, hipMemcpyAsync(c->dX.p, c->dB.p, sizeof(double) * 2 * (size_t)c->sys.nV,
                                     hipMemcpyDeviceToDevice, c->stream));
        S->pcg_fallback = 3;
        st = OC_OK;
    }
    return st;
}

// Newton direction H d = b (b in c->dB, d in c->dX) with the selected
// preconditioner and its fallbacks; fills the PCG fields of S. setupLaunched:
// launch_precond_setup was already queued for this matrix.
// Sum of the residual-norm records (fixed order, so the result does not depend on timing).
int residual_sq(oc_ctx* c, long n, const double* b, const double* y, double* r, double& out)
{
    const int g = oc::launch_residual_norm(c->stream, n, b, y, r, c->dIrPart.as<double>());
    OC_HIP(c, hipGetLastError());
    std::vector<double> h(g);
    OC_HIP(c, hipMemcpyAsync(h.data(), c->dIrPart.p, sizeof(double) * g, hipMemcpyDeviceToHost, c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    double sum = 0.0;
    for (double v : h) sum += v;
    out = sum;
    return OC_OK;
}

// Mixed-precision iterative refinement of the Newton solve A x = b (A FP64): the PCG iterations multiply by the
// FP32 rounding of A (half the matrix traffic) and the residual and the solution are kept in FP64. (A diagonal
// guard on the rounding, 4 * 2^-24 times each row's absolute sum, keeps A32 definite but was measured to stall
// the refinement on the near-null rigid rotation; it is left off.)
//   x = 0, r = b;  pass k: PCG on A32 d = r to tol_k = min(0.5, pcgTol |b| / |r|) (a breakdown keeps the
//   iterate it reached), x += d, r = b - A x in FP64;  until |r| <= pcgTol |b|, irMax passes, the iteration
//   cap or a pass that does not halve |r|. The result is in dX; relRes is the FP64 residual. Returns OC_OK,
//   OC_ERR_NOT_CONVERGED (cap, passes spent or stagnation) or OC_ERR_BREAKDOWN (a first pass with no iteration).
int refined_pcg(oc_ctx* c, int& iters, double& relRes, int& passes)
{
    hipStream_t s = c->stream;
    BlockPattern& P = c->sys;
    const long n = 2L * P.nV;
    OC_HIP(c, c->dVals32.ensure(sizeof(float) * 4 * (size_t)std::max<long>(1, P.nnzb())));
    OC_HIP(c, c->dXir.ensure(sizeof(double) * (size_t)n));
    OC_HIP(c, c->dRir.ensure(sizeof(double) * (size_t)n));
    OC_HIP(c, c->dIrPart.ensure(sizeof(double) * (size_t)oc::grid_for(n)));
    oc::launch_round_blocks(s, P.nV, P.dRowPtr.as<int>(), P.dDiagPos.as<int>(), P.dVals.as<double>(),
                            c->dVals32.as<float>(), 0.0);
    double bb = 0.0, rrTrue = 0.0;
    if (int st = residual_sq(c, n, c->dB.as<double>(), nullptr, c->dRir.as<double>(), bb)) return st;
    iters = 0;
    passes = 0;
    relRes = 0.0;
    if (bb == 0.0) {
        oc::launch_scale_copy(s, n, 0.0, c->dB.as<double>(), c->dX.as<double>());
        return OC_OK;
    }
    rrTrue = bb;
    double rrPrev = bb;
    int st = OC_ERR_NOT_CONVERGED;
    while (passes < c->irMax && iters < c->pcgMaxIter) {
        const double tolK = std::min(0.5, c->pcgTol * std::sqrt(bb / rrTrue));
        int it = 0;
        double rr = 0.0;
        const int sp = run_pcg(c, P, c->dRir.as<double>(), tolK, c->pcgMaxIter - iters, it, rr, c->ext,
                               passes == 0 ? c->pcgHint : 0, c->dVals32.p, 1);
        if (sp != OC_OK && sp != OC_ERR_NOT_CONVERGED && sp != OC_ERR_BREAKDOWN) return sp;
        iters += it;
        ++passes;
        if (it == 0) {
            if (passes == 1) return OC_ERR_BREAKDOWN;
            break;
        }
        // x += d (the first pass starts x from d); r = b - A x
        if (passes == 1)
            OC_HIP(c, hipMemcpyAsync(c->dXir.p, c->dX.p, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
        else
            oc::launch_axpy_commit(s, n, 1.0, c->dX.as<double>(), c->dXir.as<double>());
        oc::launch_spmv(s, P.nV, P.dRowPtr.as<int>(), P.dColIdx.as<int>(), P.dVals.p, 0, c->dXir.as<double>(),
                        c->dTmpVec.as<double>());
        if (int e = residual_sq(c, n, c->dB.as<double>(), c->dTmpVec.as<double>(), c->dRir.as<double>(), rrTrue))
            return e;
        if (rrTrue <= c->pcgTol * c->pcgTol * bb) {
            st = OC_OK;
            break;
        }
        if (sp == OC_ERR_NOT_CONVERGED) break;  // the iteration cap
        // stagnation: the FP32 rounding perturbs the Newton matrix's near-null directions (the rigid rotation
        // about the fixed vertex) by more than the refinement can correct; the iterate so far is kept
        if (rrTrue > 0.25 * rrPrev) break;
        rrPrev = rrTrue;
    }
    if (passes > 0)
        OC_HIP(c, hipMemcpyAsync(c->dX.p, c->dXir.p, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    relRes = std::sqrt(rrTrue / bb);
    return st;
}

int solve_direction(oc_ctx* c, oc_iter_stats* S, bool setupLaunched = false)
{
    hipStream_t s = c->stream;
    if (!setupLaunched)
        if (int st = launch_precond_setup(c, S)) return st;
    int it = 0;
    double rr = 0.0;
    if ((c->amgValid || c->amgPending) && c->amgSkip > 0) {
        // multigrid failed on a recent step (and no set-up was launched): Jacobi-PCG directly
        --c->amgSkip;
        S->pcg_fallback = 5;
        const int st = jacobi_direction(c, S, it, rr);
        S->pcg_iters = it;
        S->pcg_rel_res = rr;
        return st != OC_OK && st != OC_ERR_NOT_CONVERGED ? st : OC_OK;
    }
    // the PCG tolerance of this step (looser after a step the injectivity bound cut short)
    const double pcgTol = c->looseTol > 0.0 && c->lastStep < c->looseBelow ? std::max(c->pcgTol, c->looseTol)
                                                                          : c->pcgTol;
    int st;
    if (c->irMax > 0) {
        int passes = 0;
        st = refined_pcg(c, it, rr, passes);
        S->ir_passes = passes;
    } else {
        st = run_pcg(c, c->sys, c->dB.as<double>(), pcgTol, c->pcgMaxIter, it, rr, c->ext, c->pcgHint);
    }
    c->pcgHint = st == OC_OK ? it : 0;
    if (!c->ext && st == OC_ERR_BREAKDOWN) {
        // Jacobi-PCG met p.Ap <= 0: the Newton matrix is singular along p (one triangle whose only fixed vertex
        // leaves it free to rotate, or FP32 element Hessians that left it slightly indefinite). Truncated Newton
        // with the iterate so far (steepest descent when there is none), as the fallback chain below.
        if (it == 0)
            OC_HIP(c, hipMemcpyAsync(c->dX.p, c->dB.p, sizeof(double) * 2 * (size_t)c->sys.nV,
                                     hipMemcpyDeviceToDevice, s));
        S->pcg_fallback = 3;
        st = OC_OK;
    }
    if (c->ext && st == OC_ERR_NOT_CONVERGED && it > 0 && c->nPrecond == OC_PRECOND_AMG) {
        // Multigrid-PCG at its iteration cap without a breakdown: inexact (truncated) Newton with the iterate so
        // far, which minimises the quadratic model over the Krylov space and so is a descent direction. Retrying
        // with a safer hierarchy or Jacobi-PCG only spends time on systems the cap already judged hard.
        S->pcg_iters_first = it;
        S->pcg_fallback = 6;
        st = OC_OK;
    }
    // a multigrid structure kept across air re-meshes is rebuilt for the next solve once one needed more
    c->amgRebuild = c->amgRebuild || (c->amgOnOld && (st != OC_OK || S->pcg_fallback != 0));
    if (c->ext && st != OC_OK) {
        // The preconditioned solve broke down or hit its cap. With the
        // learned factor in the mixed form the likely cause is the matrix
        // itself: FP32 element Hessians, each PSD to FP32 rounding, can sum to
        // a matrix slightly indefinite along its near-null directions, which
        // the long Krylov runs of that preconditioner find. The matrix is then
        // rebuilt from FP64 element terms at the same UV (the right-hand side
        // stays), the factor predicted again, and the solve retried; later
        // steps of this solve build their Newton system from FP64 element
        // terms directly (the line search keeps FP32 energies). (With
        // multigrid the FP32-stored hierarchy is what loses definiteness, and
        // the FP64 rebuild was measured not to help.) Multigrid retries with
        // its guaranteed (Gershgorin) smoother interval; what still fails falls
        // back to Jacobi-PCG at the same tolerance.
        S->pcg_iters_first = it;
        S->pcg_fallback = 2;
        if (system_f32(c)) {
            c->elemFp64 = true;
            system_element_pass(c, system_set(c));
            system_assemble(c);
            if (c->nPrecond == OC_PRECOND_LEARNED) {
                c->learned->net.forward(s, c->sys.dVals.p, c->sys.vals32);
            } else if (c->nPrecond == OC_PRECOND_IC0) {
                c->ic0.numeric(s, c->sys.dVals.as<double>());
            } else if (c->amgValid) {
                amg_numeric(c, 0);
                ++S->precond_setups;
            }
            int it2 = 0;
            st = run_pcg(c, c->sys, c->dB.as<double>(), pcgTol, c->pcgMaxIter, it2, rr, c->ext);
            it += it2;
            if (st == OC_ERR_NOT_CONVERGED && it2 > 0 && c->nPrecond == OC_PRECOND_AMG) st = OC_OK;
            if (st == OC_OK) S->pcg_fallback = 4;
        }
        if (st != OC_OK && c->amgValid) {
            amg_numeric(c, 1);
            ++S->precond_setups;
            int it2 = 0;
            st = run_pcg(c, c->sys, c->dB.as<double>(), pcgTol, c->pcgMaxIter, it2, rr, c->ext);
            it += it2;
            if (st == OC_OK) S->pcg_fallback = 1;
        }
        if (st != OC_OK && c->nPrecond == OC_PRECOND_LEARNED) {
            // the learned factor failed: block IC(0)-PCG at the same tolerance before Jacobi-PCG
            if (c->ic0Struct || (st = ic0_structure(c)) == OC_OK) {
                c->ic0.numeric(s, c->sys.dVals.as<double>());
                int it2 = 0;
                st = run_pcg(c, c->sys, c->dB.as<double>(), pcgTol, c->pcgMaxIter, it2, rr, &c->ic0);
                it += it2;
                if (st == OC_OK) S->pcg_fallback = 7;
            }
        }
        if (st != OC_OK) {
            st = jacobi_direction(c, S, it, rr);
            // multigrid whose attempts ended in Jacobi-PCG on two consecutive steps is skipped for the next
            // kAmgSkip steps (retried afterwards): on maps whose Newton matrices it cannot precondition (the Tutte
            // map of a cut genus-3 surface squeezes triangles to 1e-4 of the mean area) its attempts would be paid
            // on every step; a single failure (one hard step of an otherwise easy solve) skips nothing
            if (c->amgValid && ++c->amgFailStreak >= 2) c->amgSkip = kAmgSkip;
        }
    }
    if (c->nPrecond == OC_PRECOND_AMG && S->pcg_fallback != 2) c->amgFailStreak = 0;
    S->pcg_iters = it;
    S->pcg_rel_res = rr;
    if (st != OC_OK && st != OC_ERR_NOT_CONVERGED) return st;
    return OC_OK;
}

void system_assemble(oc_ctx* c);
// One Newton iteration of every active chart (batched charts): the element
// pass, assembly and PCG run once over the union of the charts (the system is
// block diagonal, so the solve is the per-chart solves at once); gradient
// norms, step bounds, line-search energies, step sizes, commits and stop
// tests are per chart, exactly as separate Optimizer::solve(1) calls would
// make them (Optimizer.cpp:206-231, 575-652).
int newton_step_charts(oc_ctx* c, oc_iter_stats* S, int* done)
{
    const TriSet T = system_set(c);
    const int nVt = c->nVt, nC = c->nCharts;
    hipStream_t s = c->stream;
    system_element_pass(c, T);
    oc::launch_gather_grad(s, nVt, c->dVcPtr.as<int>(), c->dVcSrc.as<int>(), c->dFixedMaskSys.as<unsigned char>(),
                           c->dElemG.as<double>(), c->dG.as<double>(), c->dPartials.as<double>(), scalar(c, 6));
    oc::launch_chart_gsq(s, nC, c->dChartV.as<int>(), c->dG.as<double>(), c->dChartGsq.as<double>());
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipMemcpyAsync(c->chartGsq.data(), c->dChartGsq.p, sizeof(double) * nC, hipMemcpyDeviceToHost, s));
    OC_HIP(c, hipStreamSynchronize(s));
    std::vector<unsigned char> act(nC, 0);
    int nAct = 0;
    double gsum = 0.0, esum = 0.0;
    for (int k = 0; k < nC; ++k) {
        gsum += c->chartGsq[k];
        esum += c->chartLastE[k];
        if (c->chartState[k] == 0 && c->chartGsq[k] < c->chartTarget[k]) c->chartState[k] = 1;  // :215-221
        act[k] = c->chartState[k] == 0;
        nAct += act[k];
    }
    S->grad_sq = gsum;
    S->E_total = esum;
    S->E_SD = esum / c->a0;
    if (nAct == 0) {
        S->converged = 1;
        *done = 1;
        return OC_OK;
    }
    OC_HIP(c, hipMemcpyAsync(c->dChartActive.p, act.data(), nC, hipMemcpyHostToDevice, s));
    system_assemble(c);
    oc::launch_chart_rhs(s, nVt, c->dVChart.as<int>(), c->dChartActive.as<unsigned char>(), c->dG.as<double>(),
                         c->dB.as<double>());
    if (int st = solve_direction(c, S)) return st;
    const double* dir = c->dX.as<double>();
    // per-chart injectivity bound (cap 1)
    const int nBlk = c->chartBlk[nC];
    std::vector<unsigned long long> om(nC, oc::dbl_to_ordered_host(1.0));
    OC_HIP(c, hipMemcpyAsync(c->dChartOrdMin.p, om.data(), sizeof(unsigned long long) * nC, hipMemcpyHostToDevice,
                             s));
    oc::launch_chart_step_bound(s, T, c->dUV.as<double>(), dir, nBlk, c->dBlkRange.as<int2>(),
                                c->dBlkChart.as<int>(), c->dChartOrdMin.as<unsigned long long>(), 1.0);
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipMemcpyAsync(om.data(), c->dChartOrdMin.p, sizeof(unsigned long long) * nC, hipMemcpyDeviceToHost,
                             s));
    OC_HIP(c, hipStreamSynchronize(s));
    // line search, each chart with its own rule state
    constexpr int K = oc::kLSCand;
    std::vector<double> alpha(nC, 0.0), alphaCommit(nC, 0.0), testE(nC, 0.0), base(nC, 0.0);
    std::vector<int> kNext(nC, 0), phase(nC, 0), fin(nC, 1), stopped(nC, 0);
    int halvings = 0;
    for (int k = 0; k < nC; ++k)
        if (act[k]) {
            alpha[k] = alphaCommit[k] = oc::ordered_to_dbl_host(om[k]) * 0.99;
            fin[k] = 0;
        }
    std::vector<double> out(2 * K * (size_t)nC), aDev(nC);
    for (;;) {
        bool any = false;
        for (int k = 0; k < nC; ++k) {
            // each unfinished chart fetches K candidates from its next index
            aDev[k] = fin[k] ? 0.0 : alpha[k];
            any = any || !fin[k];
        }
        if (!any) break;
        OC_HIP(c, hipMemcpyAsync(c->dChartAlpha.p, aDev.data(), sizeof(double) * nC, hipMemcpyHostToDevice, s));
        oc::launch_chart_linesearch(s, T, c->dUV.as<double>(), dir, nBlk, c->dBlkRange.as<int2>(),
                                    c->dBlkChart.as<int>(), c->dChartAlpha.as<double>(), nC, c->dChartBlk.as<int>(),
                                    c->dPartials.as<double>(), c->dChartOut.as<double>());
        OC_HIP(c, hipGetLastError());
        OC_HIP(c, hipMemcpyAsync(out.data(), c->dChartOut.p, sizeof(double) * out.size(), hipMemcpyDeviceToHost, s));
        OC_HIP(c, hipStreamSynchronize(s));
        for (int k = 0; k < nC; ++k) {
            if (fin[k]) continue;
            const double lastE = c->chartLastE[k];
            for (int j = 0; j < K && !fin[k]; ++j) {
                // candidate j is alpha[k] / 2^j, the value alpha[k] takes after j halvings
                const double E = c->a0 * out[(size_t)k * 2 * K + j];
                const bool inv = out[(size_t)k * 2 * K + K + j] > 0.0;
                testE[k] = E;
                if (phase[k] == 0 && !(E > lastE)) phase[k] = 1;  // energy test passed: inversion guard next
                if (phase[k] == 1 && !inv) {                       // (:615-629)
                    fin[k] = 1;
                    break;
                }
                const double na = alpha[k] / 2.0;
                ++halvings;
                if (na == 0.0) {
                    stopped[k] = 1;
                    fin[k] = 1;
                    alpha[k] = 0.0;
                    break;
                }
                alpha[k] = na;
                alphaCommit[k] = na;
            }
        }
    }
    for (int k = 0; k < nC; ++k) aDev[k] = act[k] ? alphaCommit[k] : 0.0;
    OC_HIP(c, hipMemcpyAsync(c->dChartAlpha.p, aDev.data(), sizeof(double) * nC, hipMemcpyHostToDevice, s));
    oc::launch_chart_commit(s, nVt, c->dVChart.as<int>(), c->dChartAlpha.as<double>(), dir, c->dUV.as<double>());
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipStreamSynchronize(s));
    int nLeft = 0;
    double esumNew = 0.0, amax = 0.0;
    for (int k = 0; k < nC; ++k) {
        c->chartStep[k] = act[k] ? alpha[k] : 0.0;
        if (act[k]) {
            const double dec = c->chartLastE[k] - testE[k];
            bool st = stopped[k] != 0;
            if (c->allowEDecRelTol && (dec / c->chartLastE[k] < 1.0e-6 * alpha[k]) && (alpha[k] > 1.0e-3)) st = true;
            c->chartLastE[k] = testE[k];
            if (st) c->chartState[k] = 2;
            amax = std::max(amax, alpha[k]);
        }
        esumNew += c->chartLastE[k];
        nLeft += c->chartState[k] == 0;
    }
    S->E_total = esumNew;
    S->E_SD = esumNew / c->a0;
    S->step = amax;
    c->lastStep = amax;
    S->halvings = halvings;
    S->stopped = nLeft == 0;
    *done = nLeft == 0;
    return OC_OK;
}

void system_assemble(oc_ctx* c)
{
    const int nUB = (int)c->sm.ubRow.size();
    const int bj = c->nPrecond == OC_PRECOND_BLOCK_JACOBI;
    if (system_f32(c))
        oc::launch_assemble<float>(c->stream, nUB, c->dUbRow.as<int>(), c->dUbCol.as<int>(), c->dUbPosU.as<int>(),
                                   c->dUbPosL.as<int>(), c->dUbCPtr.as<int>(), c->dUbCSrc.as<int>(),
                                   c->dFixedMaskSys.as<unsigned char>(), c->dFixedDiag.as<double>(),
                                   c->dElemH.as<float>(), c->sys.dVals.p, c->sys.vals32, c->sys.dMinv.as<double>(), bj);
    else
        oc::launch_assemble<double>(c->stream, nUB, c->dUbRow.as<int>(), c->dUbCol.as<int>(), c->dUbPosU.as<int>(),
                                    c->dUbPosL.as<int>(), c->dUbCPtr.as<int>(), c->dUbCSrc.as<int>(),
                                    c->dFixedMaskSys.as<unsigned char>(), c->dFixedDiag.as<double>(),
                                    c->dElemH.as<double>(), c->sys.dVals.p, c->sys.vals32, c->sys.dMinv.as<double>(),
                                    bj);
}
}  // namespace

int oc_newton_step(oc_ctx* c, oc_iter_stats* S, int* done)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, S && done, "oc_newton_step: null output");
    if (!c->sysReady) {
        c->err = "oc_newton_step: call oc_newton_init first";
        return OC_ERR_STATE;
    }
    (void)hipSetDevice(c->device);
    std::memset(S, 0, sizeof(*S));
    *done = 0;
    if (c->nCharts > 0) return newton_step_charts(c, S, done);
    const TriSet T = system_set(c);
    const int nVt = c->nVt;
    hipStream_t s = c->stream;
    const int f32 = c->sysPrecision == OC_PRECISION_MIXED;
    // gradient (and element Hessians in the same pass)
    system_element_pass(c, T);
    oc::launch_gather_grad(s, nVt, c->dVcPtr.as<int>(), c->dVcSrc.as<int>(), c->dFixedMaskSys.as<unsigned char>(),
                           c->dElemG.as<double>(), c->dG.as<double>(), c->dPartials.as<double>(), scalar(c, 6),
                           c->dB.as<double>());
    OC_HIP(c, hipGetLastError());
    // ||g||^2 travels to the host while the Newton system is assembled and the preconditioner set up (work
    // that is simply dropped on the one step whose gradient test succeeds)
    OC_HIP(c, hipMemcpyAsync(c->mail, scalar(c, 6), sizeof(double), hipMemcpyDeviceToHost, s));
    OC_HIP(c, hipEventRecord(c->evGsq, s));
    system_assemble(c);
    if (int st = launch_precond_setup(c, S)) return st;
    OC_HIP(c, hipGetLastError());
    OC_HIP(c, hipEventSynchronize(c->evGsq));
    const double gsq = c->mail[0];
    S->grad_sq = gsq;
    S->E_total = c->lastE;
    S->E_SD = c->lastESD;
    S->E_scaf = c->lastEScaf;
    if (c->trG) {  // Optimizer.cpp:211-214: |g|^2 and the SD term's own |g_SD|^2
        double gsd = gsq / (c->a0 * c->a0);
        if (c->nFair) {
            // dTmpVec (2 nVt) and the partial records (nVt rows) were sized by the system build
            oc::launch_element(s, mesh_set(c, 0), c->dUV.as<double>(), nullptr, c->dElemG.as<double>(), nullptr, 0,
                               nullptr, nullptr);
            oc::launch_gather_grad(s, c->nV, c->dMvcPtr.as<int>(), c->dMvcSrc.as<int>(),
                                   c->dFixedMaskMesh.as<unsigned char>(), c->dElemG.as<double>(),
                                   c->dTmpVec.as<double>(), c->dPartials.as<double>(), scalar(c, 8));
            OC_HIP(c, hipGetLastError());
            OC_HIP(c, hipMemcpyAsync(&gsd, scalar(c, 8), sizeof(double), hipMemcpyDeviceToHost, s));
            OC_HIP(c, hipStreamSynchronize(s));
        }
        oc::io::trace_grad_line(c->trG, gsq, gsd);
    }
    if (gsq < c->targetGRes) {  // Optimizer.cpp:215-221
        S->converged = 1;
        *done = 1;
        return OC_OK;
    }
    // direction: H d = -g (system assembled and preconditioner set up above)
    if (int st = solve_direction(c, S, true)) return st;
    const double* dir = c->dX.as<double>();
    // line search (Optimizer.cpp:575-652) on the device: the injectivity bound, the energies at the first
    // kLSCand halvings from 0.99 x the bound, the reference's rule applied to them and the step committed, then
    // one read-back; more halvings than that continue on the host below
    constexpr int K = oc::kLSCand;
    unsigned long long* om = c->dOrdMin.as<unsigned long long>();
    unsigned long long* omAir = c->nFair ? om + 1 : nullptr;  // the air and the mesh triangles' own bounds
    oc::launch_set_u64(s, om, oc::dbl_to_ordered_host(1.0), omAir ? 3 : 1);
    oc::launch_step_bound(s, T, c->dUV.as<double>(), dir, om, 1.0, omAir);
    const double* esum = nullptr;
    if (c->nFair) {  // the scaffold changed: the energy is recomputed (Optimizer.cpp:588-592)
        oc::launch_element(s, T, c->dUV.as<double>(), nullptr, nullptr, nullptr, 0, c->dPartials.as<double>(),
                           scalar(c, 4), f32);
        esum = scalar(c, 4);
    }
    oc::LsDecision* dDec = c->dLsDec.as<oc::LsDecision>();
    oc::launch_linesearch(s, T, c->dUV.as<double>(), dir, 0.0, 0, c->dPartials.as<double>(), c->dLsOut.as<double>(),
                          f32, om, oc::LsDecide{dDec, om, omAir, esum, c->lastE});
    oc::launch_ls_commit(s, dDec, 2L * nVt, dir, c->dUV.as<double>());
    OC_HIP(c, hipGetLastError());
    double* cand = c->mail;
    oc::LsDecision* D = reinterpret_cast<oc::LsDecision*>(c->mail + 4 * K);
    OC_HIP(c, hipMemcpyAsync(cand, c->dLsOut.p, sizeof(double) * 4 * K, hipMemcpyDeviceToHost, s));
    OC_HIP(c, hipMemcpyAsync(D, dDec, sizeof(oc::LsDecision), hipMemcpyDeviceToHost, s));
    OC_HIP(c, hipStreamSynchronize(s));
    double lastE = c->lastE, lastEScafStart = c->lastEScaf;
    if (c->nFair) {
        lastE = c->lastE = D->lastE;
        c->lastESD = D->lastESD;
        lastEScafStart = c->lastEScaf = D->lastEScaf;
    }
    const double stepSize = D->bound * 0.99;
    // the air mesh held the step back: its triangles' bound is below kAirLimitRatio of what the mesh alone
    // allows (capped at a full step)
    c->airLimited = c->nFair > 0 && D->airBound < kAirLimitRatio * std::min(1.0, D->meshBound);
    int k0 = 0;  // first index of the candidates held in cand
    auto fetch = [&](int kstart) -> int {
        oc::launch_linesearch(s, T, c->dUV.as<double>(), dir, stepSize, kstart, c->dPartials.as<double>(),
                              c->dLsOut.as<double>(), f32);
        OC_HIP(c, hipGetLastError());
        OC_HIP(c, hipMemcpyAsync(cand, c->dLsOut.p, sizeof(double) * 4 * K, hipMemcpyDeviceToHost, s));
        OC_HIP(c, hipStreamSynchronize(s));
        k0 = kstart;
        return OC_OK;
    };
    auto get = [&](int k, double* E, double* Esd, double* Es, bool* inv) -> int {
        if (k0 < 0 || k < k0 || k >= k0 + K)
            if (int e = fetch(k)) return e;
        const int j = k - k0;
        *E = cand[j];
        *Esd = cand[K + j];
        *Es = cand[2 * K + j] * T.sAir;
        *inv = cand[3 * K + j] > 0.0;
        return OC_OK;
    };
    bool stopped = false;
    int k = 0;
    double alpha = stepSize;     // current trial step
    double alphaCommit = alpha;  // step of the UV left in place
    double testE, testESD, testES;
    bool inv;
    int halvings = 0;
    if (D->status != 1) {
        // decided and committed on the device
        stopped = D->status == 2;
        alpha = D->alpha;
        alphaCommit = D->alphaCommit;
        testE = D->testE;
        testESD = D->testESD;
        testES = D->testES;
        halvings = D->halvings;
    } else {
        // more than kLSCand halvings: the rule continues on the host from the first candidate
        if (int e = get(0, &testE, &testESD, &testES, &inv)) return e;
        while (testE > lastE) {
            const double na = alpha / 2.0;
            ++halvings;
            if (na == 0.0) {
                stopped = true;
                alpha = 0.0;
                break;
            }
            alpha = na;
            alphaCommit = alpha;
            ++k;
            if (int e = get(k, &testE, &testESD, &testES, &inv)) return e;
        }
        // post-check of inversions (Optimizer.cpp:615-629)
        while (!stopped && inv) {
            const double na = alpha / 2.0;
            ++halvings;
            if (na == 0.0) {
                stopped = true;
                alpha = 0.0;
                break;
            }
            alpha = na;
            alphaCommit = alpha;
            ++k;
            if (int e = get(k, &testE, &testESD, &testES, &inv)) return e;
        }
        oc::launch_axpy_commit(s, 2L * nVt, alphaCommit, dir, c->dUV.as<double>());
        OC_HIP(c, hipGetLastError());
    }
    double lastEDec = lastE - testE;
    if (c->nFair) lastEDec += (-lastEScafStart + testES);
    if (c->allowEDecRelTol && (lastEDec / lastE < 1.0e-6 * alpha) && (alpha > 1.0e-3)) stopped = true;
    c->lastE = testE;
    c->lastESD = testESD;
    c->lastEScaf = testES;
    OC_HIP(c, hipStreamSynchronize(s));
    S->E_total = testE;
    S->E_SD = testESD;
    S->E_scaf = testES;
    S->step = alpha;
    c->lastStep = alpha;
    S->halvings = halvings;
    S->stopped = stopped ? 1 : 0;
    *done = stopped ? 1 : 0;
    if (c->trE && !stopped)  // Optimizer.cpp:645-648
        if (int st = write_energy_trace(c, testE, testESD)) return st;
    return OC_OK;
}

int oc_time_kernel(oc_ctx* c, int which, int reps, double* ms)
{
    if (!c) return OC_ERR_ARG;
    OC_ARG(c, ms && reps > 0 && which >= 0 && which <= 9 + kMaxTimedLevels, "oc_time_kernel: bad args");
    if (which >= 10 && (!c->amgValid || which - 10 + 1 >= c->amg->levels())) {
        c->err = "oc_time_kernel: no multigrid level with a transfer at that depth";
        return OC_ERR_STATE;
    }
    if ((which == 7 || which == 8) && !c->ext) {
        c->err = "oc_time_kernel: no multigrid, learned or IC(0) preconditioner is active";
        return OC_ERR_STATE;
    }
    if (which == 9 && !c->amgValid) {
        c->err = "oc_time_kernel: the multigrid preconditioner is not active";
        return OC_ERR_STATE;
    }
    if (!c->sysReady) {
        c->err = "oc_time_kernel: call oc_newton_init first";
        return OC_ERR_STATE;
    }
    (void)hipSetDevice(c->device);
    hipStream_t s = c->stream;
    if (c->amgValid && !c->amg->has_values()) amg_numeric(c, 0);  // no step since oc_newton_init
    const TriSet T = system_set(c);
    PcgCtrl* ctrl = c->dCtrl.as<PcgCtrl>();
    // Timing copies of the partial records: the update reads a live p.q record
    // and the SpMV a live (r.z, r.r) record; the kernels write into scratch
    // records so the values they read stay fixed across repetitions.
    const int GU = oc::pcg_grid_update(c->nVt), GS = oc::pcg_grid_spmv(c->nVt);
    // size the partial records before any pointer into them is taken
    if (ensure_scratch(c, std::max<long>(4L * GU + 2L * GS, 2L * c->nVt))) return OC_ERR_HIP;
    double* tp = c->dPartials.as<double>();
    double* tU = tp;                         // 2*GU read by spmv
    double* tS = tp + 2 * (size_t)GU;        // GS   read by update
    double* tUo = tS + GS;                   // 2*GU written by update
    double* tSo = tUo + 2 * (size_t)GU;      // GS   written by spmv
    auto spmv = [&]() {
        oc::launch_pcg_spmv(s, c->nVt, c->sys.dRowPtr.as<int>(), c->sys.dColIdx.as<int>(), c->sys.dVals.p,
                            c->sys.vals32, c->dZ.as<double>(), c->dP0.as<double>(), c->dP1.as<double>(),
                            c->dQ.as<double>(), tU, GU, 2, tU + 1, GU, 2, tSo, ctrl);
    };
    auto update = [&]() {
        oc::launch_pcg_update(s, c->nVt, c->dP1.as<double>(), c->dQ.as<double>(), c->sys.dMinv.as<double>(),
                              c->dTmpVec.as<double>(), c->dR.as<double>(), c->dZ.as<double>(), tS, tUo, ctrl);
    };
    auto launch = [&]() {
        switch (which) {
        case 0:
            system_element_pass(c, T);
            break;
        case 1:
            system_assemble(c);
            break;
        case 2:
            spmv();
            update();
            break;
        case 3:
            oc::launch_linesearch(s, T, c->dUV.as<double>(), c->dX.as<double>(), 0.5, 0, c->dPartials.as<double>(),
                                  c->dLsOut.as<double>(), c->sysPrecision == OC_PRECISION_MIXED);
            break;
        case 4:
            oc::launch_step_bound(s, T, c->dUV.as<double>(), c->dX.as<double>(), c->dOrdMin.as<unsigned long long>(),
                                  1.0);
            break;
        case 5:
            spmv();
            break;
        case 6:
            update();
            break;
        case 7:
            c->ext->apply(s, c->dR.as<double>(), c->dTmpVec.as<double>(), c->dPartials.as<double>(), nullptr);
            break;
        case 8:
            if (c->amgValid) amg_numeric(c, 0);
            else if (c->nPrecond == OC_PRECOND_IC0) c->ic0.numeric(s, c->sys.dVals.as<double>());
            else
                c->learned->net.forward(s, c->sys.dVals.p, c->sys.vals32);
            break;
        case 9:
            c->amg->lanczos0_step(s);
            break;
        default:  // 10 + l: one Chebyshev step of the V-cycle on multigrid level l
            c->amg->cheb_step_level(s, which - 10);
            break;
        }
    };
    if (which == 7) OC_HIP(c, c->dTmpVec.ensure(sizeof(double) * 2 * (size_t)c->nVt));
    if (which == 9) c->amg->lanczos0_prepare(s);
    if (which == 2 || which == 5 || which == 6) {
        // Keep the PCG kernels doing full work on the current system: a
        // private copy of x (dTmpVec) so the last direction is not
        // disturbed, done cleared, iteration cap out of reach.
        OC_HIP(c, c->dTmpVec.ensure(sizeof(double) * 2 * (size_t)c->nVt));
        OC_HIP(c, hipMemcpyAsync(c->dTmpVec.p, c->dX.p, sizeof(double) * 2 * (size_t)c->nVt,
                                 hipMemcpyDeviceToDevice, s));
        PcgCtrl h{};
        OC_HIP(c, hipMemcpyAsync(&h, ctrl, sizeof(PcgCtrl), hipMemcpyDeviceToHost, s));
        OC_HIP(c, hipStreamSynchronize(s));
        h.done = 0;
        h.iter = 1;
        h.itNext = h.itCur = 1;
        h.maxit = 1 << 30;
        h.tol2 = 0.0;
        h.bb = 1.0;
        h.rzSlot[0] = h.rzSlot[1] = 1.0;
        OC_HIP(c, hipMemcpyAsync(ctrl, &h, sizeof(PcgCtrl), hipMemcpyHostToDevice, s));
        // records: (r.z, r.r) = (1, 1) so the SpMV neither stops nor breaks down; p.q = 1
        std::vector<double> rec(2 * (size_t)GU + GS, 0.0);
        rec[0] = 1.0;
        rec[1] = 1.0;
        rec[2 * (size_t)GU] = 1.0;
        OC_HIP(c, hipMemcpyAsync(tU,rec.data(), sizeof(double) * rec.size(), hipMemcpyHostToDevice, s));
        OC_HIP(c, hipStreamSynchronize(s));
    }
    hipEvent_t e0, e1;
    OC_HIP(c, hipEventCreate(&e0));
    OC_HIP(c, hipEventCreate(&e1));
    launch();  // warm
    OC_HIP(c, hipStreamSynchronize(s));
    // back-to-back launches between one pair of events: the per-launch
    // average then excludes the event round trips. Single-kernel timings
    // replay the launches from a captured graph, as the PCG iterations run:
    // launched one by one from the host, a small coarse-level kernel would
    // measure the host's launch rate instead of its own duration.
    hipGraphExec_t gx = nullptr;
    if (which == 5 || which == 6 || which >= 9) {
        hipGraph_t g = nullptr;
        if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) == hipSuccess) {
            for (int r = 0; r < reps; ++r) launch();
            if (hipStreamEndCapture(s, &g) == hipSuccess && g) {
                if (hipGraphInstantiate(&gx, g, nullptr, nullptr, 0) != hipSuccess) gx = nullptr;
                (void)hipGraphDestroy(g);
            }
        }
        (void)hipGetLastError();
        if (gx) {  // one untimed replay
            OC_HIP(c, hipGraphLaunch(gx, s));
            OC_HIP(c, hipStreamSynchronize(s));
        }
    }
    OC_HIP(c, hipEventRecord(e0, s));
    if (gx) OC_HIP(c, hipGraphLaunch(gx, s));
    else
        for (int r = 0; r < reps; ++r) launch();
    OC_HIP(c, hipEventRecord(e1, s));
    OC_HIP(c, hipEventSynchronize(e1));
    if (gx) (void)hipGraphExecDestroy(gx);
    float t = 0.f;
    OC_HIP(c, hipEventElapsedTime(&t, e0, e1));
    *ms = (double)t / reps;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    OC_HIP(c, hipGetLastError());
    if (which == 2 || which == 5 || which == 6) {
        // leave the solver state re-armed for the next Newton step
        PcgCtrl h{};
        OC_HIP(c, hipMemcpyAsync(&h, ctrl, sizeof(PcgCtrl), hipMemcpyDeviceToHost, s));
        OC_HIP(c, hipStreamSynchronize(s));
        h.done = 1;
        OC_HIP(c, hipMemcpyAsync(ctrl, &h, sizeof(PcgCtrl), hipMemcpyHostToDevice, s));
        OC_HIP(c, hipStreamSynchronize(s));
    }
    return OC_OK;
}

int oc_newton_get_system(oc_ctx* c, int* rowPtr, int* colIdx, double* vals, double* rhs, unsigned char* fixedMask)
{
    if (!c) return OC_ERR_ARG;
    if (!c->sysReady) {
        c->err = "oc_newton_get_system: call oc_newton_init first";
        return OC_ERR_STATE;
    }
    (void)hipSetDevice(c->device);
    const BlockPattern& P = c->sys;
    if (rowPtr) std::copy(P.rowPtr.begin(), P.rowPtr.end(), rowPtr);
    if (colIdx) std::copy(P.colIdx.begin(), P.colIdx.end(), colIdx);
    if (fixedMask) std::copy(c->fixedMaskSys.begin(), c->fixedMaskSys.end(), fixedMask);
    const size_t nv = 4 * (size_t)P.nnzb();
    if (vals) {
        if (P.vals32) {
            std::vector<float> f(nv);
            OC_HIP(c, hipMemcpyAsync(f.data(), P.dVals.p, sizeof(float) * nv, hipMemcpyDeviceToHost, c->stream));
            OC_HIP(c, hipStreamSynchronize(c->stream));
            for (size_t i = 0; i < nv; ++i) vals[i] = f[i];
        } else {
            OC_HIP(c, hipMemcpyAsync(vals, P.dVals.p, sizeof(double) * nv, hipMemcpyDeviceToHost, c->stream));
        }
    }
    if (rhs) OC_HIP(c, hipMemcpyAsync(rhs, c->dB.p, sizeof(double) * 2 * (size_t)c->nVt, hipMemcpyDeviceToHost,
                                      c->stream));
    OC_HIP(c, hipStreamSynchronize(c->stream));
    return OC_OK;
}

int oc_system_sizes(oc_ctx* c, long long* nF, long long* nV, long long* nnzBlocks, long long* nUpperBlocks)
{
    if (!c) return OC_ERR_ARG;
    if (nF) *nF = c->sysReady ? c->nFt : c->nF;
    if (nV) *nV = c->sysReady ? c->nVt : c->nV;
    if (nnzBlocks) *nnzBlocks = c->sysReady ? c->sys.nnzb() : 0;
    if (nUpperBlocks) *nUpperBlocks = c->sysReady ? (long long)c->sm.ubRow.size() : 0;
    return OC_OK;
}

}  // extern "C"
