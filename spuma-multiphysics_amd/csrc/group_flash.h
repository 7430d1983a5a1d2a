// SPDX-License-Identifier: GPL-3.0-or-later
// FP64 flashes of one cell per wave: small batches and the mixed flash's
// deferred cells.
//
// On one lane a cell's search is a chain of several hundred phase
// evaluations, of tens of thousands for the cells that go through all their
// restarts, and a batch lasts as long as the longest chain of its waves: a
// 257-cell batch 30 ms, 20,000 binary cells 1.4 s, with the chip idle.  Here
// the cell's starts run on the wave's eight groups of eight lanes, and each
// group shares its line searches and finite differences (the flash's GROUP
// mode), so the chain is one start's Newton iterations.  Bound by the latency
// of those iterations; in a batch large enough to fill the chip with one cell
// per lane, the lanes a cell's own starts leave idle cost more than that.
//
// Launched by group.hip; those of two species by two.hip (built otherwise,
// see lane_flash.h).
#ifndef RAMD_GROUP_FLASH_H
#define RAMD_GROUP_FLASH_H
#include "flash_step.h"

namespace ramd {

// A cell's result and counts, from lane 0.
template <class E>
__device__ inline void storeGroup(const FlashSink& sink, bool ok, const E& result, const FlashCells& cells, uint32_t c,
                                  const Counts& n) {
    const bool lead = threadIdx.x == 0;
    if (sink.hem) {
        if (lead) storeHemCell(ok, result, sink.hem[c]);
        if (sink.partials) {
            if (lead) {
                unsigned long long* slot = sink.partials + size_t(blockIdx.x) * 8;
                slot[0] = n.phases; slot[1] = n.residuals; slot[2] = n.candidates; slot[3] = n.stable;
                slot[4] = n.failures; slot[5] = n.fd; slot[6] = ok ? 1 : 0; slot[7] = n.analytic;
            }
        } else {
            const Counts none = {0, 0, 0, 0, 0, 0, 0};
            addTotals(lead ? n : none, lead && ok ? 1u : 0u, sink.totals);
        }
    } else {
        if (lead) {
            storeCell(ok, result, cells.seeds[c], c, sink.out, sink.p, sink.c, sink.r);
            if (!ok && sink.failMark) sink.failMark[c] = 1;
            if (sink.cost) sink.cost[c] = uint16_t(n.phases < 65535u ? n.phases : 65535u);
        }
        countFlash(lead && !ok ? 1u : 0u, lead ? n.phases : 0u, sink.counters);
    }
}

template <int NS, int NL, bool RJ, bool CAP>
__global__ __launch_bounds__(64, RAMD_REFINE_MIN_WAVES) void groupFlashKernel(
    const HemModel<NS>* __restrict__ globalModel, FlashCells cells, const uint32_t* __restrict__ order,
    const HemCapillaryDev* __restrict__ capillary, FlashSink sink) {
    const uint32_t c = order ? order[blockIdx.x] : blockIdx.x;
    if (!cells.flashed(c)) return;  // uniform per workgroup
    const HemModel<NS>& model = workgroupModel(globalModel);
    Counts n = {0, 0, 0, 0, 0, 0, 0};
    using F = Flash<NS, NL, double, false, RJ, CAP, kModelLds, 8>;
    F f(model, n);
    cells.load<NS>(f, c);
    typename F::E result;
    zeroEval(result);
    const bool ok = runHemCell<CAP, NL>(f, cells.seeds[c], capillary ? capillary + c : nullptr, result);
    storeGroup(sink, ok, result, cells, c, n);
}

// The deferred cells (full FP64 search, FP64 restarts, or a frozen
// candidate's solve from the cell's guess) refined again without deferral.
// queueCount is read on the device (the launch does not depend on it).
// Three waves per cell: the first refines, and all three run the twenty
// restarts of a cell that needs them: three rounds of eight on one wave, 90 ms
// in a flash of 40^3 binary cells, now 57.
constexpr int kQueueThreads = 192;
static_assert(kQueueThreads / 8 >= kRestarts, "a group per restart");
template <int NS, int NL, bool WIDE>
__global__ __launch_bounds__(WIDE ? kQueueThreads : 64, RAMD_REFINE_MIN_WAVES) void refineQueueKernel(
    const HemModel<NS>* __restrict__ globalModel, FlashCells cells, const uint32_t* __restrict__ queue,
    const unsigned* __restrict__ queueCount, const CandidateSet* __restrict__ sets, FlashSink sink) {
    const unsigned count = *queueCount;
    if (blockIdx.x >= count || (NL > 0 && count <= RAMD_WIDE_CELLS) != WIDE) return;  // uniform per workgroup
    const HemModel<NS>& model = workgroupModel(globalModel);
    using F = Flash<NS, NL, double, true, false, false, kModelLds, 8, WIDE>;
    __shared__ typename F::Wide wide;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    for (unsigned i = blockIdx.x; i < count; i += gridDim.x) {  // uniform per workgroup
        const uint32_t c = queue[i];
        Counts n = {0, 0, 0, 0, 0, 0, 0};
        F f(model, n);
        cells.load<NS>(f, c);
        if (WIDE) f.wide = &wide;
        if (!WIDE || wave == 0) {
            EvalT<double, true> result;
            zeroEval(result);
            const bool ok = f.refine(sets[c], result);
            if (WIDE) f.wideDone();
            storeGroup(sink, ok, result, cells, c, n);
        } else {
            f.wideWorker();
        }
        if (WIDE) __syncthreads();  // before the next cell's first call
    }
}

// The launches of two.hip: two species.
void launchGroupFlashTwo(int nl, bool analytic, bool capillaryFlash, const void* model, const FlashCells& cells,
                         const uint32_t* order, uint32_t count, const HemCapillaryDev* capillary,
                         const FlashSink& sink, hipStream_t stream);
void launchRefineQueueTwo(int nl, const void* model, const FlashCells& cells, const uint32_t* queue,
                          const unsigned* queueCount, const CandidateSet* sets, const FlashSink& sink,
                          hipStream_t stream);

}  // namespace ramd
#endif
