// SPDX-License-Identifier: GPL-3.0-or-later
// HEM handle shared by the flash plugin and the device-resident step.
#ifndef REACTIVE_AMD_HEM_INTERNAL_H
#define REACTIVE_AMD_HEM_INTERNAL_H
#include <hip/hip_runtime.h>
#include <cstdint>
#include <vector>
#include "flash_device.h"
#include "flash_step.h"

namespace ramd {

struct HemHandle {
    int ns = 0, nl = 0, device = 0;
    bool analytic = false;  // the model's analytic-Jacobian mode (FP64 flash)
    bool boundary = false;  // the model's boundary search (boundaryRecovery = 1)
    bool prune = false;     // the model's stable-gas pruning (stableGasPrune = 1)
    // one species with its liquid: the mixed flash looks its candidates up in the saturation table
    bool pure() const { return ns == 1 && nl == 1 && !prune; }
    int arithmetic = 0;     // equilibrium flash of host batches: REACTIVE_AMD_FLASH_FP64 or _MIXED
    size_t capacity = 0, deviceBytes = 0, modelBytes = 0;
    void* model = nullptr;  // HemModel<ns> in device memory
    // phases residuals candidates stable failures fd successes analytic, then
    // (mixed arithmetic) FP32 phases and deferred cells
    unsigned long long* totals = nullptr;
    // mixed arithmetic: candidate sets and lists (allocated on the first
    // mixed batch), the last batch's FP32 phase evaluations and deferred cells
    MixedScratch mixed;
    uint64_t lastSinglePhases = 0, lastQueued = 0;
    // host-path staging (allocated on the first host batch)
    bool hostReady = false;
    double *dq = nullptr, *de = nullptr;
    ThermoOut* dguess = nullptr;
    HemOutputDev* dout = nullptr;
    uint32_t* dorder = nullptr;
    HemCapillaryDev* dcap = nullptr;      // host-path capillary staging
    std::vector<uint32_t> hostOrder;
    std::vector<uint8_t> hostKey;
    std::vector<HemOutputDev> hostOut;
    hipStream_t stream = nullptr;
    hipEvent_t events[4] = {};
    std::vector<void*> allocations;

    ~HemHandle();
    void* allocate(size_t bytes);
    void ensureHostPath();
    // Flash count cells named by order (or 0..count-1) on stream s; q, e,
    // guess, capillary and out are indexed by cell.  Totals: phases,
    // residuals, candidates, stable, failures, fd Jacobians, successes,
    // analytic Jacobians.
    // With partials (slots of 8 counters, at least one per 64 cells), the
    // workgroups write their sums there instead of adding them to totals.
    // Returns the workgroups launched.
    unsigned launch(const double* q, const double* e, const ThermoOut* guess, const uint32_t* order, size_t count,
                    const HemCapillaryDev* capillary, HemOutputDev* out, hipStream_t s,
                    unsigned long long* partials = nullptr, unsigned slots = 0);
    // The equilibrium flash of the same cells in mixed arithmetic: FP32
    // candidate search, FP64 refinement and the deferred queue; totals as
    // launch's plus totals[8] FP32 phases and totals[9] deferred cells.
    void launchMixed(const double* q, const double* e, const ThermoOut* guess, const uint32_t* order, size_t count,
                     HemOutputDev* out, hipStream_t s);
};

HemHandle* createHem(const void* raw, size_t bytes, size_t capacity, bool hostPath);

}  // namespace ramd
#endif
