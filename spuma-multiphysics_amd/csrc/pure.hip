// SPDX-License-Identifier: GPL-3.0-or-later
// FP64 refinement of a pure fluid's two-phase points, in registers.
//
// The directed search leaves one two-phase point for most cells of a pure
// fluid, within about 1e-7 of the root, and its refinement is the same short
// sequence for all of them: two or three evaluations of both phases, the
// Jacobian's response, the sound speeds.  The general refinement runs it
// through calls that keep the flash and three evaluation records on the
// stack; here it is one inlined loop (Flash::activeLean), same operations and
// same results.  Cells that leave the sequence go to the general refinement.
#include <hip/hip_runtime.h>
#include "flash_step.h"

// One wave per SIMD: 380 registers and 368 bytes of stack.  A 160^3 flash's
// refinements take 5.3 ms with the leftovers' general refinement (7.4 ms as
// the general refinement alone); with two waves per SIMD and a second record
// for line searches, 1,536 bytes of stack and 9.6 ms.
#ifndef RAMD_TWO_PHASE_MIN_WAVES
#define RAMD_TWO_PHASE_MIN_WAVES 1
#endif

namespace ramd {

template <int NS>
__global__ __launch_bounds__(64, RAMD_TWO_PHASE_MIN_WAVES) void refineTwoPhaseKernel(
    const HemModel<NS>* __restrict__ globalModel, FlashCells cells, const uint32_t* __restrict__ order, uint32_t count,
    const CandidateSet* __restrict__ sets, FlashSink sink, SearchScratch scratch, uint32_t* __restrict__ search,
    unsigned* __restrict__ searchCount) {
    const HemModel<NS>& model = workgroupModel(globalModel);
    const uint32_t i = blockIdx.x * 64u + threadIdx.x;
    Counts n = {0, 0, 0, 0, 0, 0, 0};
    uint32_t succeeded = 0;
    const uint32_t c = i < count ? order[i] : 0u;
    if (i < count && cells.flashed(c)) {
        const uint32_t flags = sets[c].flags;
        if (!(flags & kSingle)) {
            EvalT<double, true> result;
            zeroEval(result);
            Flash<NS, 1, double, true, false, false, kModelLds> f(model, n);
            cells.load<NS>(f, c);
            if (!sets[c].count) {
                search[atomicAdd(searchCount, 1u)] = c;
            } else if (f.refineTwoPhase(sets[c].c[0], result)) {
                succeeded = 1;
                if (sink.hem) {
                    storeHemCell(true, result, sink.hem[c]);
                } else {
                    storeCell(true, result, cells.seeds[c], c, sink.out, sink.p, sink.c, sink.r);
                    if (sink.cost) sink.cost[c] = uint16_t(n.phases < 65535u ? n.phases : 65535u);
                }
            } else {
                n = {0, 0, 0, 0, 0, 0, 0};
                scratch.single[atomicAdd(scratch.singleCount, 1u)] = c;
            }
        }
    }
    if (sink.hem) addTotals(n, succeeded, sink.totals);
    else countFlash(0u, n.phases, sink.counters);
}

void launchRefineTwoPhase(const void* model, const FlashCells& cells, const uint32_t* order, uint32_t count,
                          const CandidateSet* sets, const FlashSink& sink, const SearchScratch& scratch, uint32_t* search,
                          unsigned* searchCount, hipStream_t stream) {
    hipLaunchKernelGGL((refineTwoPhaseKernel<1>), dim3(unsigned((size_t(count) + 63) / 64)), dim3(64), 0, stream,
                       static_cast<const HemModel<1>*>(model), cells, order, count, sets, sink, scratch, search,
                       searchCount);
    RAMD_HIP(hipGetLastError());
}

}  // namespace ramd
