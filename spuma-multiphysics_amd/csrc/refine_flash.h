// SPDX-License-Identifier: GPL-3.0-or-later
// FP64 refinement of the mixed flash's candidates, one cell per lane: the
// resident step's and the HEM batch's.  Launched by step.hip and hem.hip;
// those of two species by two.hip (built otherwise, see lane_flash.h).
#ifndef RAMD_REFINE_FLASH_H
#define RAMD_REFINE_FLASH_H
#include "flash_step.h"

namespace ramd {

// Mixed precision, second half: FP64 refinement, stability and selection of
// the listed cells' candidates.  Deferred cells go to the queue, or, where
// the candidates came from the saturation table, to the list of cells to
// search.  A list counted on the device is swept in rounds.
template <int NS, int NL>
__global__ __launch_bounds__(256, RAMD_REFINE_MIN_WAVES) void stepRefineKernel(const HemModel<NS>* __restrict__ globalModel,
                                                       FlashCells cells, CellList list,
                                                       const CandidateSet* __restrict__ sets,
                                                       ThermoOut* __restrict__ out, double* __restrict__ pOut,
                                                       double* __restrict__ cOut, double* __restrict__ rOut,
                                                       uint16_t* __restrict__ cost,
                                                       unsigned long long* __restrict__ counters,
                                                       uint32_t* __restrict__ queue, unsigned* __restrict__ queueCount,
                                                       uint32_t* __restrict__ search, unsigned* __restrict__ searchCount,
                                                       uint8_t* __restrict__ failMark) {
    const uint32_t count = list.size();
    if (blockIdx.x * blockDim.x >= count) return;  // uniform per workgroup
    const HemModel<NS>& model = workgroupModel(globalModel);
    uint32_t failed = 0, phases = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
        const uint32_t c = list.cells[i];
        if (!cells.flashed(c)) continue;
        Counts n = {0, 0, 0, 0, 0, 0, 0};
        Flash<NS, NL, double, true, false, false, kModelLds> f(model, n);
        cells.load<NS>(f, c);
        EvalT<double, true> result;
        zeroEval(result);
        bool deferred = false;
        const bool ok = f.refine(sets[c], result, &deferred);
        if (deferred) {
            if (sets[c].flags & kDirect) search[atomicAdd(searchCount, 1u)] = c;
            else queue[atomicAdd(queueCount, 1u)] = c;
        } else {
            storeCell(ok, result, cells.seeds[c], c, out, pOut, cOut, rOut);
            if (!ok && failMark) failMark[c] = 1;
            failed += ok ? 0u : 1u;
            if (cost) cost[c] = uint16_t(n.phases < 65535u ? n.phases : 65535u);
        }
        phases += n.phases;
    }
    countFlash(failed, phases, counters);
}

// Mixed arithmetic, second half: FP64 refinement, stability and selection of
// the listed cells' candidates; deferred cells go to the queue, or, where the
// candidates came from the saturation table, to the list of cells to search.
template <int NS, int NL>
__global__ __launch_bounds__(64, RAMD_REFINE_MIN_WAVES) void hemRefineKernel(const HemModel<NS>* __restrict__ globalModel,
                                                     FlashCells cells, CellList list,
                                                     const CandidateSet* __restrict__ sets,
                                                     HemOutputDev* __restrict__ out,
                                                     unsigned long long* __restrict__ totals,
                                                     uint32_t* __restrict__ queue, unsigned* __restrict__ queueCount,
                                                     uint32_t* __restrict__ search,
                                                     unsigned* __restrict__ searchCount) {
    const uint32_t count = list.size();
    if (blockIdx.x * 64u >= count) return;  // uniform per workgroup
    const HemModel<NS>& model = workgroupModel(globalModel);
    Counts n = {0, 0, 0, 0, 0, 0, 0};
    uint32_t succeeded = 0;
    for (uint32_t i = blockIdx.x * 64u + threadIdx.x; i < count; i += gridDim.x * 64u) {
        const uint32_t c = list.cells[i];
        Flash<NS, NL, double, true, false, false, kModelLds> f(model, n);
        cells.load<NS>(f, c);
        EvalT<double, true> result;
        zeroEval(result);
        bool deferred = false;
        const bool ok = f.refine(sets[c], result, &deferred);
        if (deferred) {
            if (sets[c].flags & kDirect) search[atomicAdd(searchCount, 1u)] = c;
            else queue[atomicAdd(queueCount, 1u)] = c;
        } else {
            storeHemCell(ok, result, out[c]);
            succeeded += ok ? 1u : 0u;
        }
    }
    addTotals(n, succeeded, totals);
}

// The launches of two.hip.
void launchStepRefineTwo(int nl, const void* model, const FlashCells& cells, const CellList& list,
                         const CandidateSet* sets, const FlashSink& sink, uint32_t* queue, unsigned* queueCount,
                         unsigned grid, unsigned block, hipStream_t stream);
void launchHemRefineTwo(int nl, const void* model, const FlashCells& cells, const CellList& list,
                        const CandidateSet* sets, const FlashSink& sink, uint32_t* queue, unsigned* queueCount,
                        unsigned grid, hipStream_t stream);

}  // namespace ramd
#endif
