// SPDX-License-Identifier: GPL-3.0-or-later
// Launches of the FP64 flashes of one cell per wave (group_flash.h).
#include <hip/hip_runtime.h>
#include "group_flash.h"

namespace ramd {

void launchGroupFlash(int ns, int nl, bool analytic, bool boundary, const void* model, const FlashCells& cells,
                      const uint32_t* order, uint32_t count, const HemCapillaryDev* capillary, const FlashSink& sink,
                      hipStream_t stream) {
#define RAMD_GROUP(NS_, NL_, RJ_, CAP_)                                                                            \
    hipLaunchKernelGGL((groupFlashKernel<NS_, NL_, RJ_, CAP_>), dim3(count), dim3(64), 0, stream,                  \
                       static_cast<const HemModel<NS_>*>(model), cells, order, capillary, sink)
#define RAMD_GROUP_SPECIES(CAP_)                                   \
    if (ns == 1 && nl == 0) RAMD_GROUP(1, 0, false, CAP_);         \
    else if (ns == 1 && !analytic) RAMD_GROUP(1, 1, false, CAP_);  \
    else if (ns == 1) RAMD_GROUP(1, 1, true, CAP_);                \
    else if (!analytic) RAMD_GROUP(2, 1, false, CAP_);             \
    else RAMD_GROUP(2, 1, true, CAP_);
    if (ns == 2 && nl == 0)
        return launchGasGroupFlash(capillary || boundary, model, cells, order, count, capillary, sink, stream);
    if (capillary || boundary) { RAMD_GROUP_SPECIES(true) }
    else { RAMD_GROUP_SPECIES(false) }
#undef RAMD_GROUP_SPECIES
#undef RAMD_GROUP
    RAMD_HIP(hipGetLastError());
}

void launchRefineQueue(int ns, int nl, const void* model, const FlashCells& cells, const uint32_t* queue,
                       const unsigned* queueCount, const CandidateSet* sets, const FlashSink& sink, hipStream_t stream) {
#define RAMD_QUEUE(NS_, NL_)                                                                                      \
    if (NL_) hipLaunchKernelGGL((refineQueueKernel<NS_, NL_, true>), dim3(RAMD_WIDE_CELLS), dim3(kQueueThreads), 0, \
                       stream, static_cast<const HemModel<NS_>*>(model), cells, queue, queueCount, sets, sink);   \
    hipLaunchKernelGGL((refineQueueKernel<NS_, NL_, false>), dim3(RAMD_QUEUE_BLOCKS), dim3(64), 0, stream,         \
                       static_cast<const HemModel<NS_>*>(model), cells, queue, queueCount, sets, sink)
    if (ns == 1 && nl == 0) { RAMD_QUEUE(1, 0); }
    else if (ns == 1) { RAMD_QUEUE(1, 1); }
    else if (nl == 0) launchGasRefineQueue(model, cells, queue, queueCount, sets, sink, stream);
    else { RAMD_QUEUE(2, 1); }
#undef RAMD_QUEUE
    RAMD_HIP(hipGetLastError());
}

}  // namespace ramd
