// SPDX-License-Identifier: GPL-3.0-or-later
// Launches of the FP64 flashes of one cell per wave (group_flash.h).
#include <hip/hip_runtime.h>
#include "group_flash.h"

namespace ramd {

void launchGroupFlash(int ns, int nl, bool analytic, bool boundary, const void* model, const FlashCells& cells,
                      const uint32_t* order, uint32_t count, const HemCapillaryDev* capillary, const FlashSink& sink,
                      hipStream_t stream) {
    if (ns == 2)
        return launchGroupFlashTwo(nl, analytic, capillary || boundary, model, cells, order, count, capillary, sink,
                                   stream);
#define RAMD_GROUP(NL_, RJ_, CAP_)                                                                                \
    hipLaunchKernelGGL((groupFlashKernel<1, NL_, RJ_, CAP_>), dim3(count), dim3(64), 0, stream,                    \
                       static_cast<const HemModel<1>*>(model), cells, order, capillary, sink)
#define RAMD_GROUP_MODES(CAP_)                     \
    if (nl == 0) RAMD_GROUP(0, false, CAP_);       \
    else if (!analytic) RAMD_GROUP(1, false, CAP_); \
    else RAMD_GROUP(1, true, CAP_);
    if (capillary || boundary) { RAMD_GROUP_MODES(true) }
    else { RAMD_GROUP_MODES(false) }
#undef RAMD_GROUP_MODES
#undef RAMD_GROUP
    RAMD_HIP(hipGetLastError());
}

void launchRefineQueue(int ns, int nl, const void* model, const FlashCells& cells, const uint32_t* queue,
                       const unsigned* queueCount, const CandidateSet* sets, const FlashSink& sink, hipStream_t stream) {
    if (ns == 2) return launchRefineQueueTwo(nl, model, cells, queue, queueCount, sets, sink, stream);
    const auto* m = static_cast<const HemModel<1>*>(model);
    if (nl == 0) {
        hipLaunchKernelGGL((refineQueueKernel<1, 0, false>), dim3(RAMD_QUEUE_BLOCKS), dim3(64), 0, stream, m, cells,
                           queue, queueCount, sets, sink);
    } else {
        hipLaunchKernelGGL((refineQueueKernel<1, 1, true>), dim3(RAMD_WIDE_CELLS), dim3(kQueueThreads), 0, stream, m,
                           cells, queue, queueCount, sets, sink);
        hipLaunchKernelGGL((refineQueueKernel<1, 1, false>), dim3(RAMD_QUEUE_BLOCKS), dim3(64), 0, stream, m, cells,
                           queue, queueCount, sets, sink);
    }
    RAMD_HIP(hipGetLastError());
}

}  // namespace ramd
