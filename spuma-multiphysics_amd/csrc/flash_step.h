// SPDX-License-Identifier: GPL-3.0-or-later
// Per-cell helpers shared by the resident step's flash kernels (step.hip)
// and the single-precision search kernel (search.hip).
#ifndef REACTIVE_AMD_FLASH_STEP_H
#define REACTIVE_AMD_FLASH_STEP_H
#include <hip/hip_runtime.h>
#include <cstring>
#include "hip_common.h"
#include "flash_device.h"

// Tuning knobs (compile-time): the model image in LDS, and the minimum waves
// per SIMD the register allocation targets for the FP64 flash kernels (3:
// 168 VGPRs, at 160^3 17 % faster than 2) and for the mixed flash's FP64
// refinement kernels (2: at 3 the refinement ran 8 % slower).
#ifndef RAMD_MODEL_LDS
#define RAMD_MODEL_LDS 1
#endif
#ifndef RAMD_FLASH_MIN_WAVES
#define RAMD_FLASH_MIN_WAVES 3
#endif
#ifndef RAMD_REFINE_MIN_WAVES
#define RAMD_REFINE_MIN_WAVES 2
#endif
// Persistent grid of the deferred queue, in single-wave workgroups that take
// one cell at a time: sixteen per CU, more than stay resident, so that a wave
// that finishes its cell is replaced at once.  (Against 1024: 160^3 pure N2O
// step 135.8 -> 132.5 ms with 2,537 deferred cells per flash, binary N2O/N2
// 96^3 2242 -> 1788 ms, when a flash deferred that many.)
#ifndef RAMD_QUEUE_BLOCKS
#define RAMD_QUEUE_BLOCKS 4096
#endif
// A queue of up to this many deferred cells gives each a workgroup of three
// waves for its restarts, a longer one a wave.
#ifndef RAMD_WIDE_CELLS
#define RAMD_WIDE_CELLS 4096
#endif
// FP64 batches of up to this many cells run one cell per wave, its starts on
// groups of eight lanes (group_flash.h); larger ones one cell per lane.
// Measured, per lane and per wave: pure, 16,384 cells 43.2 and 14.9 ms, 65,536
// cells 51.4 and 54.1, where the line lies; binary, 65,536 cells 1,708 and 453
// ms: two species cross later, at a size not measured.
#ifndef RAMD_GROUP_CELLS
#define RAMD_GROUP_CELLS 65536
#endif

namespace ramd {

// Flashes of the kernels read the workgroup's LDS model copy directly.
constexpr bool kModelLds = RAMD_MODEL_LDS != 0;

// The workgroup's copy of the model image: tables are read from LDS rather
// than global memory.  Every thread of the workgroup must call this (it
// synchronises the workgroup).
template <int NS>
__device__ inline const HemModel<NS>& workgroupModel(const HemModel<NS>* __restrict__ global) {
#if RAMD_MODEL_LDS
    static_assert(sizeof(HemModel<NS>) % 4 == 0, "model image in 4-byte words");
    HemModel<NS>& local = sharedModel<NS>();
    const uint32_t* src = reinterpret_cast<const uint32_t*>(global);
    uint32_t* dst = reinterpret_cast<uint32_t*>(&local);
    for (uint32_t w = threadIdx.x; w < sizeof(HemModel<NS>) / 4; w += blockDim.x) dst[w] = src[w];
    __syncthreads();
    return local;
#else
    return *global;
#endif
}

// The inputs of a flash batch, by cell.  The resident step's: conserved SoA
// q[k stride + c], e = rhoE - |rho u|^2 / (2 rho) (ReactiveFoam.C:727-728, in
// FP64) and the step-start seeds.  A HEM batch's (energy non-null): species
// masses q[c ns + k] and the given internal energies.
struct FlashCells {
    const double* q;
    size_t stride;
    const double* energy;
    const ThermoOut* seeds;
    const double* gate;   // the step's dt: nothing is flashed unless positive (null: always)
    const uint32_t* rep;  // exact reuse: only cells that represent themselves (null: all)
    __device__ inline bool flashed(uint32_t c) const { return !(gate && !(*gate > 0)) && !(rep && rep[c] != c); }
    template <int NS, class F>
    __device__ inline void load(F& f, uint32_t c) const {
        using R = decltype(f.energy);
        if (energy) {
            for (int k = 0; k < NS; ++k) f.q[k] = R(q[size_t(c) * NS + k]);
            f.energy = R(energy[c]);
        } else {
            double rho = 0;
            for (int k = 0; k < NS; ++k) {
                const double mass = q[size_t(k) * stride + c];
                f.q[k] = R(mass);
                rho += mass;
            }
            const double m0 = q[size_t(NS) * stride + c], m1 = q[size_t(NS + 1) * stride + c];
            const double m2 = q[size_t(NS + 2) * stride + c], E = q[size_t(NS + 3) * stride + c];
            f.energy = R(E - .5 * (m0 * m0 + m1 * m1 + m2 * m2) / rho);
        }
        const ThermoOut& g = seeds[c];
        f.guessP = R(g.p);
        f.guessT = R(g.T);
        f.guessLiquid = R(g.liquidMass[0]);
    }
    // Inputs a single-precision search takes up, with some of the condensable.
    template <int NS>
    __device__ inline bool valid(uint32_t c, int condensable) const;
};
template <int NS, class R = double>
struct FlashInput {
    R q[NS], energy, guessP, guessT, guessLiquid;
};
template <int NS>
__device__ inline bool FlashCells::valid(uint32_t c, int condensable) const {
    FlashInput<NS, float> f;
    load<NS>(f, c);
    float rho = 0;
    bool ok = fin(f.energy);
    for (int k = 0; k < NS; ++k) {
        rho += f.q[k];
        ok = ok && fin(f.q[k]) && f.q[k] >= 0;
    }
    return ok && rho > 0 && f.q[condensable] > 0;
}
// Cells of a launch: `count` of them, or as many as *counted says.
struct CellList {
    const uint32_t* cells;
    uint32_t count;
    const unsigned* counted;
    __device__ inline uint32_t size() const { return counted ? *counted : count; }
};

// Commits a flash result, or keeps the step-start state of a failed cell
// (the reference commits nothing for it); p, c_frozen and rho go to the SoA
// arrays the next transport stage reads.
template <bool A, bool RJ, bool C>
__device__ inline void storeCell(bool ok, const EvalT<double, A, RJ, C>& result, const ThermoOut& g, uint32_t c,
                                 ThermoOut* __restrict__ out, double* __restrict__ pOut, double* __restrict__ cOut,
                                 double* __restrict__ rOut) {
    if (ok) {
        writeOut(result, out[c]);
        pOut[c] = result.p;
        cOut[c] = result.cf;
        rOut[c] = result.rho;
    } else {
        out[c] = g;
        pOut[c] = g.p;
        cOut[c] = g.soundFrozen;
        rOut[c] = g.rho;
    }
}

// Flash output record, byte-compatible with ReactiveGpuHemOutputV1 (184 B).
struct HemOutputDev {
    ThermoOut state;
    int success, reserved;
};
// Per-cell capillary input, byte-compatible with ReactiveGpuHemCapillaryInputV2
// (24 B): the interface's color and pressure jump, and equilibrium 1 for the
// UV equilibrium with the boundary search, 0 for the frozen inventory.
struct HemCapillaryDev {
    double color, pressureJump;
    int equilibrium, pad;
};
// A flash result into the batch's output record (zero state where it failed).
template <class E>
__device__ inline void storeHemCell(bool ok, const E& result, HemOutputDev& o) {
    if (ok) writeOut(result, o.state);
    else std::memset(&o.state, 0, sizeof(o.state));
    o.success = ok ? 1 : 0;
    o.reserved = 0;
}
// Adds one wavefront's work counters (phases, residuals, candidates, stable,
// failures, fd Jacobians, successes, analytic Jacobians) to totals: one
// 64-bit atomic per counter per wavefront.
__device__ inline void addTotals(const Counts& n, uint32_t succeeded, unsigned long long* __restrict__ totals) {
    const uint32_t s0 = waveSum(n.phases), s1 = waveSum(n.residuals), s2 = waveSum(n.candidates);
    const uint32_t s3 = waveSum(n.stable), s4 = waveSum(n.failures), s5 = waveSum(n.fd);
    const uint32_t s6 = waveSum(succeeded), s7 = waveSum(n.analytic);
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&totals[0], (unsigned long long)s0);
        atomicAdd(&totals[1], (unsigned long long)s1);
        atomicAdd(&totals[2], (unsigned long long)s2);
        atomicAdd(&totals[3], (unsigned long long)s3);
        atomicAdd(&totals[4], (unsigned long long)s4);
        atomicAdd(&totals[5], (unsigned long long)s5);
        atomicAdd(&totals[6], (unsigned long long)s6);
        atomicAdd(&totals[7], (unsigned long long)s7);
    }
}
// One cell of a HEM batch by flash f (g: its seed, x: its capillary input or
// null).  Without capillary input the equilibrium UV flash (recover,
// reactiveDeviceFlash.h:564-567).  With it (recoverCapillary, :572-590) the
// cell's interface (color, pressure jump) held during the solve, then the UV
// equilibrium with the boundary search (equilibrium = 1) or the frozen
// inventory at the seed's liquid masses (0); a cell whose color or jump the
// reference rejects (its status 2) fails.
template <bool CAP, int NL, class F>
__device__ inline bool runHemCell(F& f, const ThermoOut& g, const HemCapillaryDev* x, typename F::E& result) {
    if (!x) return f.run(result);
    if constexpr (CAP) {
        if (!fin(x->color) || x->color < 0 || x->color > 1 || !fin(x->pressureJump) ||
            (x->pressureJump != 0 && NL != 1))
            return false;
        f.color = x->color;
        f.jump = x->pressureJump;
        if (x->equilibrium != 0) return f.run(result, true);
    }
    return f.frozen(NL ? g.liquidMass[0] : 0.0, result, 0, g.liquidMass[1]);
}

__device__ inline void countFlash(uint32_t failed, uint32_t phases, unsigned long long* __restrict__ counters) {
    const uint32_t sumFailed = waveSum(failed), sumPhases = waveSum(phases);
    if ((threadIdx.x & 63) == 0) {
        if (sumFailed) atomicAdd(&counters[0], (unsigned long long)sumFailed);
        atomicAdd(&counters[1], (unsigned long long)sumPhases);
    }
}

// ---- one cell per wave (group_flash.h) -------------------------------------
// Where a cell's result and counts go: a HEM batch's records and totals (or a
// slot of eight sums per workgroup in partials), or the step's arrays.
struct FlashSink {
    HemOutputDev* hem;
    unsigned long long *totals, *partials;
    ThermoOut* out;
    double *p, *c, *r;
    uint16_t* cost;
    unsigned long long* counters;
    uint8_t* failMark;
};
// FP64 flash of the cells in `order` (null: 0 .. count - 1); capillary (may be
// null) by cell; analytic, boundary: the model's modes.
void launchGroupFlash(int ns, int nl, bool analytic, bool boundary, const void* model, const FlashCells& cells,
                      const uint32_t* order, uint32_t count, const HemCapillaryDev* capillary, const FlashSink& sink,
                      hipStream_t stream);
// The deferred cells of the mixed flash: refined again without deferral.
void launchRefineQueue(int ns, int nl, const void* model, const FlashCells& cells, const uint32_t* queue,
                       const unsigned* queueCount, const CandidateSet* sets, const FlashSink& sink, hipStream_t stream);

// ---- candidates of the mixed flash (search.hip) ---------------------------
// FP64 refinement of a directed search's two-phase points.  Cells without a
// point go to the list `search`; one-phase cells, and those whose point takes
// more than full Newton steps, are left to refine(), in scratch.single.
void launchRefineTwoPhase(const void* model, const FlashCells& cells, const uint32_t* order, uint32_t count,
                          const CandidateSet* sets, const FlashSink& sink, const SearchScratch& scratch,
                          uint32_t* search, unsigned* searchCount, hipStream_t stream);
// The table of a one-species model with its liquid.
void launchSaturation(const void* model, SaturationTable* table, hipStream_t stream);
// The directed search of every cell in `order`: sets of one candidate or none, flagged kDirect.
void launchDirect(const void* model, const SaturationTable* table, const FlashCells& cells, const uint32_t* order,
                  uint32_t count, const SearchScratch& scratch, CandidateSet* sets, uint16_t* cost,
                  unsigned long long* phases, hipStream_t stream);
// Single-precision search, one cell per lane in workgroups of `block` lanes
// (64, 128 or 256); candidate sets and evaluation counts by cell.
void launchSearch(int ns, int nl, const void* model, const FlashCells& cells, const uint32_t* order, uint32_t count,
                  CandidateSet* sets, uint16_t* cost, unsigned long long* phases, hipStream_t stream, unsigned block);
// The same search, one start per lane, for models without stable-gas pruning;
// stride: the list's largest length; directed: the sets are the directed
// search's, whose flags leave out some of the frozen solves.
void launchSearchStarts(int ns, int nl, const void* model, const FlashCells& cells, const CellList& list, size_t stride,
                        const SearchScratch& scratch, bool directed, CandidateSet* sets, uint16_t* cost,
                        unsigned long long* phases, hipStream_t stream);

}  // namespace ramd
#endif
