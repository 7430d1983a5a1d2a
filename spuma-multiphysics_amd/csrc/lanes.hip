// SPDX-License-Identifier: GPL-3.0-or-later
// FP64 flashes of one cell per lane of two species, the analytic-Jacobian mode
// and the capillary / boundary-search flash (see lane_flash.h).
#include <hip/hip_runtime.h>
#include "lane_flash.h"

namespace ramd {

void launchLaneStep(int ns, int nl, bool analytic, const void* model, const FlashCells& cells, const uint32_t* order,
                    uint32_t count, const FlashSink& sink, unsigned blocks, unsigned block, hipStream_t stream) {
#define RAMD_STEP_FLASH(NS_, NL_, RJ_)                                                                            \
    hipLaunchKernelGGL((stepFlashKernel<NS_, NL_, RJ_>), dim3(blocks), dim3(block), 0, stream,                     \
                       static_cast<const HemModel<NS_>*>(model), cells, order, count, sink.out, sink.p, sink.c,    \
                       sink.r, sink.cost, sink.counters, sink.failMark)
    if (ns == 1) RAMD_STEP_FLASH(1, 1, true);
    else if (nl == 0) RAMD_STEP_FLASH(2, 0, false);
    else if (!analytic) RAMD_STEP_FLASH(2, 1, false);
    else RAMD_STEP_FLASH(2, 1, true);
#undef RAMD_STEP_FLASH
    RAMD_HIP(hipGetLastError());
}

void launchLaneHem(int ns, int nl, bool analytic, bool boundary, const void* model, const FlashCells& cells,
                   const uint32_t* order, uint32_t count, const HemCapillaryDev* capillary, HemOutputDev* out,
                   unsigned long long* totals, unsigned long long* partials, hipStream_t stream) {
    const unsigned blocks = unsigned((size_t(count) + 63) / 64);
#define RAMD_HEM_LAUNCH(NS_, NL_, RJ_, CAP_)                                                                       \
    hipLaunchKernelGGL((hemFlashKernel<NS_, NL_, RJ_, CAP_>), dim3(blocks), dim3(64), 0, stream,                   \
                       static_cast<const HemModel<NS_>*>(model), cells, order, count, capillary, out, totals, partials)
    if (capillary || boundary) {
        if (ns == 1 && nl == 0) RAMD_HEM_LAUNCH(1, 0, false, true);
        else if (ns == 1 && !analytic) RAMD_HEM_LAUNCH(1, 1, false, true);
        else if (ns == 1) RAMD_HEM_LAUNCH(1, 1, true, true);
        else if (nl == 0) RAMD_HEM_LAUNCH(2, 0, false, true);
        else if (!analytic) RAMD_HEM_LAUNCH(2, 1, false, true);
        else RAMD_HEM_LAUNCH(2, 1, true, true);
    } else {
        if (ns == 1) RAMD_HEM_LAUNCH(1, 1, true, false);
        else if (nl == 0) RAMD_HEM_LAUNCH(2, 0, false, false);
        else if (!analytic) RAMD_HEM_LAUNCH(2, 1, false, false);
        else RAMD_HEM_LAUNCH(2, 1, true, false);
    }
#undef RAMD_HEM_LAUNCH
    RAMD_HIP(hipGetLastError());
}

}  // namespace ramd
