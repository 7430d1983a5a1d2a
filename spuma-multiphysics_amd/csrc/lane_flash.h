// SPDX-License-Identifier: GPL-3.0-or-later
// FP64 flashes of one cell per lane: the resident step's and the HEM batch's.
//
// The pure fluid's reference arithmetic is launched by step.hip and hem.hip;
// two species, the analytic-Jacobian mode and the capillary flash come from
// lanes.hip, whose compilation differs (build.sh): these kernels hold more
// scalars than the registers take, and the ordinary allocation of the
// registers that keep the rest let one lane's spills overwrite another's.
// (Two species' flashes of one cell per wave, group_flash.h, and their
// refinement, refine_flash.h, are built so in two.hip.)
// That allocation costs the pure fluid's flash 30 % (64^3 cells, two steps:
// 312 ms, 418 with it).
#ifndef RAMD_LANE_FLASH_H
#define RAMD_LANE_FLASH_H
#include "flash_step.h"

namespace ramd {

// Plain FP64 flash of the cells in `order`; RJ: the model's
// analytic-Jacobian mode.
template <int NS, int NL, bool RJ>
__global__ __launch_bounds__(256, RAMD_FLASH_MIN_WAVES) void stepFlashKernel(const HemModel<NS>* __restrict__ globalModel,
                                                      FlashCells cells,
                                                      const uint32_t* __restrict__ order, uint32_t count,
                                                      ThermoOut* __restrict__ out,
                                                      double* __restrict__ pOut, double* __restrict__ cOut,
                                                      double* __restrict__ rOut, uint16_t* __restrict__ cost,
                                                      unsigned long long* __restrict__ counters,
                                                      uint8_t* __restrict__ failMark) {
    const HemModel<NS>& model = workgroupModel(globalModel);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    Counts n = {0, 0, 0, 0, 0, 0};
    uint32_t failed = 0;
    if (i < count && cells.flashed(order[i])) {
        const uint32_t c = order[i];
        using F = Flash<NS, NL, double, false, RJ, false, kModelLds>;
        F f(model, n);
        cells.load<NS>(f, c);
        typename F::E result;
        zeroEval(result);
        const bool ok = f.run(result);
        storeCell(ok, result, cells.seeds[c], c, out, pOut, cOut, rOut);
        if (!ok && failMark) failMark[c] = 1;
        failed = ok ? 0u : 1u;
        if (cost) cost[c] = uint16_t(n.phases < 65535u ? n.phases : 65535u);
    }
    countFlash(failed, n.phases, counters);
}

// One cell per lane (runHemCell).  RJ: the model's analytic-Jacobian mode
// (analyticJacobian = 1); CAP: the capillary / boundary-search flash, for
// capillary input and boundaryRecovery models.
template <int NS, int NL, bool RJ, bool CAP>
__global__ __launch_bounds__(64, RAMD_FLASH_MIN_WAVES) void hemFlashKernel(const HemModel<NS>* __restrict__ globalModel,
                                                     FlashCells cells, const uint32_t* __restrict__ order, uint32_t count,
                                                     const HemCapillaryDev* __restrict__ capillary,
                                                     HemOutputDev* __restrict__ out,
                                                     unsigned long long* __restrict__ totals,
                                                     unsigned long long* __restrict__ partials) {
    const HemModel<NS>& model = workgroupModel(globalModel);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    Counts n = {0, 0, 0, 0, 0, 0, 0};
    uint32_t succeeded = 0;
    if (i < count) {
        const uint32_t c = order ? order[i] : i;
        using F = Flash<NS, NL, double, false, RJ, CAP, kModelLds>;
        F f(model, n);
        cells.load<NS>(f, c);
        typename F::E result;
        zeroEval(result);
        const bool ok = runHemCell<CAP, NL>(f, cells.seeds[c], capillary ? capillary + c : nullptr, result);
        storeHemCell(ok, result, out[c]);
        succeeded = ok ? 1u : 0u;
    }
    if (partials) {  // one 64-lane workgroup: its eight sums go to its own slot
        const uint32_t s0 = waveSum(n.phases), s1 = waveSum(n.residuals), s2 = waveSum(n.candidates);
        const uint32_t s3 = waveSum(n.stable), s4 = waveSum(n.failures), s5 = waveSum(n.fd);
        const uint32_t s6 = waveSum(succeeded), s7 = waveSum(n.analytic);
        if (threadIdx.x == 0) {
            unsigned long long* slot = partials + size_t(blockIdx.x) * 8;
            slot[0] = s0; slot[1] = s1; slot[2] = s2; slot[3] = s3;
            slot[4] = s4; slot[5] = s5; slot[6] = s6; slot[7] = s7;
        }
    } else if (totals) {
        addTotals(n, succeeded, totals);
    }
}

// The launches of lanes.hip: every model but a pure fluid's reference flash.
void launchLaneStep(int ns, int nl, bool analytic, const void* model, const FlashCells& cells, const uint32_t* order,
                    uint32_t count, const FlashSink& sink, unsigned blocks, unsigned block, hipStream_t stream);
void launchLaneHem(int ns, int nl, bool analytic, bool boundary, const void* model, const FlashCells& cells,
                   const uint32_t* order, uint32_t count, const HemCapillaryDev* capillary, HemOutputDev* out,
                   unsigned long long* totals, unsigned long long* partials, hipStream_t stream);

}  // namespace ramd
#endif
