// SPDX-License-Identifier: GPL-3.0-or-later
// FP64 flashes of two species: one cell per wave (group_flash.h), and the
// mixed flash's refinement (refine_flash.h) and deferred cells.  Built as
// lanes.hip is (see lane_flash.h): these solvers keep masks of finished lanes
// among the scalars that do not fit.
#include <hip/hip_runtime.h>
#include "group_flash.h"
#include "refine_flash.h"

namespace ramd {

void launchGroupFlashTwo(int nl, bool analytic, bool capillaryFlash, const void* model, const FlashCells& cells,
                         const uint32_t* order, uint32_t count, const HemCapillaryDev* capillary,
                         const FlashSink& sink, hipStream_t stream) {
#define RAMD_GROUP(NL_, RJ_, CAP_)                                                                                \
    hipLaunchKernelGGL((groupFlashKernel<2, NL_, RJ_, CAP_>), dim3(count), dim3(64), 0, stream,                    \
                       static_cast<const HemModel<2>*>(model), cells, order, capillary, sink)
#define RAMD_GROUP_MODES(CAP_)                     \
    if (nl == 0) RAMD_GROUP(0, false, CAP_);       \
    else if (!analytic) RAMD_GROUP(1, false, CAP_); \
    else RAMD_GROUP(1, true, CAP_);
    if (capillaryFlash) { RAMD_GROUP_MODES(true) }
    else { RAMD_GROUP_MODES(false) }
#undef RAMD_GROUP_MODES
#undef RAMD_GROUP
    RAMD_HIP(hipGetLastError());
}

void launchRefineQueueTwo(int nl, const void* model, const FlashCells& cells, const uint32_t* queue,
                          const unsigned* queueCount, const CandidateSet* sets, const FlashSink& sink,
                          hipStream_t stream) {
    const auto* m = static_cast<const HemModel<2>*>(model);
    if (nl == 0) {
        hipLaunchKernelGGL((refineQueueKernel<2, 0, false>), dim3(RAMD_QUEUE_BLOCKS), dim3(64), 0, stream, m, cells,
                           queue, queueCount, sets, sink);
    } else {
        hipLaunchKernelGGL((refineQueueKernel<2, 1, true>), dim3(RAMD_WIDE_CELLS), dim3(kQueueThreads), 0, stream, m,
                           cells, queue, queueCount, sets, sink);
        hipLaunchKernelGGL((refineQueueKernel<2, 1, false>), dim3(RAMD_QUEUE_BLOCKS), dim3(64), 0, stream, m, cells,
                           queue, queueCount, sets, sink);
    }
    RAMD_HIP(hipGetLastError());
}

void launchStepRefineTwo(int nl, const void* model, const FlashCells& cells, const CellList& list,
                         const CandidateSet* sets, const FlashSink& sink, uint32_t* queue, unsigned* queueCount,
                         unsigned grid, unsigned block, hipStream_t stream) {
#define RAMD_STEP_REFINE(NL_)                                                                                     \
    hipLaunchKernelGGL((stepRefineKernel<2, NL_>), dim3(grid), dim3(block), 0, stream,                              \
                       static_cast<const HemModel<2>*>(model), cells, list, sets, sink.out, sink.p, sink.c, sink.r, \
                       sink.cost, sink.counters, queue, queueCount, nullptr, nullptr, sink.failMark)
    if (nl == 0) RAMD_STEP_REFINE(0);
    else RAMD_STEP_REFINE(1);
#undef RAMD_STEP_REFINE
    RAMD_HIP(hipGetLastError());
}

void launchHemRefineTwo(int nl, const void* model, const FlashCells& cells, const CellList& list,
                        const CandidateSet* sets, const FlashSink& sink, uint32_t* queue, unsigned* queueCount,
                        unsigned grid, hipStream_t stream) {
#define RAMD_HEM_REFINE(NL_)                                                                                      \
    hipLaunchKernelGGL((hemRefineKernel<2, NL_>), dim3(grid), dim3(64), 0, stream,                                  \
                       static_cast<const HemModel<2>*>(model), cells, list, sets, sink.hem, sink.totals, queue,    \
                       queueCount, nullptr, nullptr)
    if (nl == 0) RAMD_HEM_REFINE(0);
    else RAMD_HEM_REFINE(1);
#undef RAMD_HEM_REFINE
    RAMD_HIP(hipGetLastError());
}

}  // namespace ramd
