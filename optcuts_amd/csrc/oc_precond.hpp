// Interface of an external PCG preconditioner (multigrid, learned factor).
#pragma once

#include <hip/hip_runtime.h>

namespace oc {

// The iteration number lives here, not in launch arguments, so that every
// iteration of one parity launches identical arguments (graph replay):
// k_pcg_init sets itNext = 0; k_pcg_spmv reads itNext and records it in itCur
// (and iter); k_pcg_update (or update_apply()) reads itCur and sets itNext = itCur + 1. A field is
// written by workgroup 0 alone and read by later kernels; only done is read in the launch that may set it
// (k_pcg_spmv, a multigrid's first kernel): there each thread reads it first and acts on it behind the record sums, from
// which every workgroup takes the same decision as the one that set it. Once the PCG is over, k_pcg_spmv leaves -1 in
// itCur and the update -1 in itNext, each written by one kernel and read by the other: launches queued past the end
// return on it at once (behind the sums, such an iteration of Jacobi-PCG at 200k faces took 9 us instead of 5).
struct PcgCtrl {
    double bb, tol2, rr, pad0;
    double rzSlot[2];
    int iter, maxit, done, itNext;
    int itCur, pad1, pad2, pad3;
};

// The damped first smoothing step of a multigrid preconditioner, d = Dinv r / theta for the row's 2x2 blocks Dinv
// and theta of the interval that ends at *lam: row-local, so the PCG kernel that writes r computes it on the way.
struct FirstStep {
    const void* Dinv = nullptr;  // 4 values per row, float when f32
    const double* lam = nullptr;
    void* d = nullptr;  // 2 values per row of the same type; null: the preconditioner has no such step
    int f32 = 0;
};

// What a PCG hands to apply() so that the preconditioner's first kernel decides convergence itself: the records of
// r.r (record b at partRr[b * sRr]) and the control record.
struct PcgStage {
    const double* partRr = nullptr;
    int nRr = 0, sRr = 0;
    PcgCtrl* ctrl = nullptr;
};

// The PCG update of one iteration (alpha = rz / sum of the p.q records, x += alpha p, rNew = rOld - alpha q) with its
// records (value 2b + 1 of partU: r.r), for a preconditioner that does it in its first kernel.
struct PcgUpdate {
    const double *p, *q, *rOld;
    double *x, *rNew;
    const double* partS;
    int nPartS;
    double* partU;
    PcgCtrl* ctrl;
};

// Chebyshev parameters on [lmax/30, lmax], lmax = 1.1 * lambda estimate
struct ChebP {
    double theta, delta, sigma;
};
__device__ __forceinline__ ChebP cheb_params(double lam)
{
    const double lmax = 1.1 * lam, lmin = lmax / 30.0;
    ChebP p;
    p.theta = 0.5 * (lmax + lmin);
    p.delta = 0.5 * (lmax - lmin);
    p.sigma = p.theta / p.delta;
    return p;
}

struct Preconditioner {
    virtual ~Preconditioner() = default;
    // z = M^-1 r for FP64 vectors on the stream; writes rz_records()
    // per-workgroup partial sums of r.z into rzPart. Every kernel returns at
    // once while *stop is nonzero (a converged PCG); stop may be null. pcg
    // (may be null; given only to a preconditioner with a first_step(), whose
    // direction the caller has then written): stop at once, setting
    // pcg->ctrl->done, when the residual is within the tolerance.
    virtual void apply(hipStream_t s, const double* r, double* z, double* rzPart, const int* stop,
                       const PcgStage* pcg = nullptr) = 0;
    virtual int rz_records() const = 0;
    virtual FirstStep first_step() const { return {}; }
    // Records of an update made by update_apply(), which then stands for the
    // PCG's update and apply(); 0: not offered.
    virtual int update_records() const { return 0; }
    virtual void update_apply(hipStream_t, const PcgUpdate&, double* /*z*/, double* /*rzPart*/) {}
    // Changes whenever the device buffers apply() launches on may have
    // changed (a new set-up); launches captured into a graph stay valid while
    // it holds.
    unsigned long generation() const { return generation_; }

protected:
    unsigned long generation_ = 0;
};

}  // namespace oc
