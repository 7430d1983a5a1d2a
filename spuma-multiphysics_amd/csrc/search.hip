// SPDX-License-Identifier: GPL-3.0-or-later
// Candidates of the mixed flash: the single-precision search and, for a pure
// fluid, the saturation table that directs it.  This file alone is
// compiled with -freciprocal-math -fapprox-func (build.sh): it only chooses
// and seeds candidates, every accepted result is recomputed by the FP64
// refinement, so it may use the hardware reciprocal and transcendental
// approximations.  Non-finite values keep their IEEE meaning (no finite-math
// assumption), so the search's NaN and range checks hold.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "flash_step.h"

// Minimum waves per SIMD the register allocation of the search kernels targets
// (5: 96 VGPRs; at 160^3 3-4 % faster than 4, 6 and 8 slower: more stack).
#ifndef RAMD_SEARCH_MIN_WAVES
#define RAMD_SEARCH_MIN_WAVES 5
#endif
// The same for the pure fluid's lean solves, which keep their state in registers.
#ifndef RAMD_LEAN_MIN_WAVES
#define RAMD_LEAN_MIN_WAVES 4
#endif
// Phase evaluations after which a start's solve by one lane is given up.
#ifndef RAMD_SLOW_PHASES
#define RAMD_SLOW_PHASES 64
#endif
// A list of up to this many such starts runs on groups of eight lanes, a
// longer one a start per lane (searchSlowKernel).
#ifndef RAMD_SLOW_GROUPS
#define RAMD_SLOW_GROUPS 196608
#endif

namespace ramd {

// ---- the whole search of a cell on one lane: models with stable-gas
// pruning, whose seeds run only where the gas solve says so.
template <int NS, int NL>
__global__ __launch_bounds__(256, RAMD_SEARCH_MIN_WAVES) void searchKernel(
    const HemModel<NS>* __restrict__ globalModel, FlashCells cells, const uint32_t* __restrict__ order,
    uint32_t count, CandidateSet* __restrict__ sets, uint16_t* __restrict__ cost,
    unsigned long long* __restrict__ phases) {
    const HemModel<NS>& model = workgroupModel(globalModel);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    Counts n = {0, 0, 0, 0, 0, 0, 0};
    if (i < count && cells.flashed(order[i])) {
        const uint32_t c = order[i];
        Flash<NS, NL, float, true, false, false, kModelLds> f(model, n);
        cells.load<NS>(f, c);
        CandidateSet set;
        f.searchRecord(set);
        sets[c] = set;
        if (cost) cost[c] = uint16_t(n.phases < 65535u ? n.phases : 65535u);
    }
    const uint32_t sum = waveSum(n.phases);
    if ((threadIdx.x & 63) == 0) atomicAdd(phases, (unsigned long long)sum);
}

// ---- the search, one start per lane.  A cell's all-gas, all-liquid and
// five seed solves are independent, so they run side by side: wave (block, s)
// runs start s of 64 cells, and a wave is as long as the longest of its 64
// solves rather than the longest sum of seven (and of the twenty restarts,
// which now run only for the cells that need them, see below).  Bound by the
// latency of the few solves that crawl, not by arithmetic: a 12^3 box's
// search took 18 ms sequentially.  With two species and a liquid, starts that crawl (past
// RAMD_SLOW_PHASES phase evaluations; one that arrives takes about 25) are
// given up and listed for searchSlowKernel.
template <int NS, int NL>
__global__ __launch_bounds__(64, RAMD_SEARCH_MIN_WAVES) void searchStartsKernel(
    const HemModel<NS>* __restrict__ globalModel, FlashCells cells, CellList list, size_t stride,
    const CandidateSet* __restrict__ directed, StartRecord* __restrict__ records, uint32_t* __restrict__ slow,
    unsigned* __restrict__ slowCount, unsigned long long* __restrict__ phases) {
    const uint32_t count = list.size();
    if (blockIdx.x * 64u >= count) return;  // uniform per workgroup
    const HemModel<NS>& model = workgroupModel(globalModel);
    uint32_t total = 0;
    for (uint32_t base = blockIdx.x * 64u; base < count; base += gridDim.x * 64u) {
        const uint32_t i = base + threadIdx.x;
        if (i < count && cells.flashed(list.cells[i])) {
            Counts n = {0, 0, 0, 0, 0, 0, 0};
            Flash<NS, NL, float, true, false, false, kModelLds> f(model, n);
            cells.load<NS>(f, list.cells[i]);
            StartRecord r;
            if (NS > 1 && NL && stride <= size_t(1) << 29) f.phaseLimit = RAMD_SLOW_PHASES;  // (an entry's position)
            if (blockIdx.y >= 2) r.bits = f.searchSeed(int(blockIdx.y), r.x);
            else if (directed && (directed[list.cells[i]].flags & (blockIdx.y ? kNotLiquid : kNotGas))) r.bits = 0;
            else r.bits = f.searchFrozen(blockIdx.y == 1, r.x);
            if (NS > 1 && NL && f.overrun) {
                slow[atomicAdd(slowCount, 1u)] = i * 8u + blockIdx.y;
                continue;
            }
            r.bits |= n.phases << 2;
            records[size_t(blockIdx.y) * stride + i] = r;
            total += n.phases;
        }
    }
    const uint32_t sum = waveSum(total);
    if (threadIdx.x == 0) atomicAdd(phases, (unsigned long long)sum);
}

// The listed (list position, start) pairs, each on GROUP lanes.  On a group
// of eight a line search tries eight fractions at a time and the difference
// Jacobian its six points, as the solve of one lane would one after the
// other, with the same result.  A crawling start's latency (ninety iterations of
// up to thirty fractions) is what the search of a small or mid-size batch
// waits for: a 40^3 binary box's search (57,000 crawling starts a flash) 37
// ms on groups, 68 with a start per lane.  A list that fills the chip with
// one start per lane is bound by its evaluations instead, of which a group
// makes several times as many: 160^3 (3.7 million) 1,500 ms on groups, 1,130
// per lane.  The line: 56^3 (156,000) 75 and 80 ms, 64^3 (234,000) 105 and 93.
// A pure fluid's few starts without a table point (47^3 cells) end as soon on
// one lane, 3.2 ms against 3.6, and are not listed.  Both kernels are launched
// and the count on the device chooses.
template <int NS, int NL, int GROUP>
__global__ __launch_bounds__(64, RAMD_SEARCH_MIN_WAVES) void searchSlowKernel(
    const HemModel<NS>* __restrict__ globalModel, FlashCells cells, CellList list, size_t stride,
    StartRecord* __restrict__ records, const uint32_t* __restrict__ slow, const unsigned* __restrict__ slowCount,
    unsigned long long* __restrict__ phases) {
    constexpr uint32_t kEach = 64u / GROUP;  // starts per wave
    const uint32_t count = *slowCount;
    if (blockIdx.x * kEach >= count || (count <= RAMD_SLOW_GROUPS) != (GROUP > 1)) return;  // uniform per workgroup
    const HemModel<NS>& model = workgroupModel(globalModel);
    uint32_t total = 0;
    for (uint32_t base = blockIdx.x * kEach; base < count; base += gridDim.x * kEach) {
        const uint32_t k = base + threadIdx.x / GROUP;
        if (k < count) {
            const uint32_t i = slow[k] / 8u, start = slow[k] % 8u;
            Counts n = {0, 0, 0, 0, 0, 0, 0};
            Flash<NS, NL, float, true, false, false, kModelLds, GROUP> f(model, n);
            cells.load<NS>(f, list.cells[i]);
            StartRecord r;
            r.bits = start >= 2 ? f.searchSeed(int(start), r.x) : f.searchFrozen(start == 1, r.x);
            r.bits |= n.phases << 2;
            if (threadIdx.x % GROUP == 0) {
                records[size_t(start) * stride + i] = r;
                total += n.phases;
            }
        }
    }
    const uint32_t sum = waveSum(total);
    if (threadIdx.x == 0) atomicAdd(phases, (unsigned long long)sum);
}

// The seven records of a cell in search order into its candidate set; cells
// without a stable one go to the restart list.
template <int NS>
__global__ __launch_bounds__(256) void searchMergeKernel(const HemModel<NS>* __restrict__ model, FlashCells cells,
                                                         CellList list, size_t stride,
                                                         const StartRecord* __restrict__ records,
                                                         CandidateSet* __restrict__ sets,
                                                         uint16_t* __restrict__ cost,
                                                         uint32_t* __restrict__ restarts,
                                                         unsigned* __restrict__ restartCount) {
    const uint32_t count = list.size();
    const double top = lo(model->Tmax, model->liquidTc * (1 - 1e-10)), bottom = hi(model->Tmin, model->liquidTmin);
    const bool restartable = model->nl && top > bottom;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < count; i += gridDim.x * 256u) {
        const uint32_t c = list.cells[i];
        if (!cells.flashed(c)) continue;
        CandidateSet set;
        set.count = set.flags = 0;
        bool have = false;
        uint32_t evaluations = 0;
        for (int s = 0; s < kStarts; ++s) {
            const StartRecord r = records[size_t(s) * stride + i];
            evaluations += r.bits >> 2;
            have = have || (r.bits & kStartStable);
            if (r.bits & kStartFound)
                noteCandidate(set, s == 0 ? kGasCandidate : s == 1 ? kLiquidCandidate : kSeedCandidate,
                              int16_t(s < 2 ? 0 : s - 2), r.x, s >= 2);
        }
        // (a cell whose inputs no solve accepts has no candidates and no restarts)
        if (!have && restartable && cells.valid<NS>(c, model->condensable)) {
            set.flags |= kRestartsSearched;
            restarts[atomicAdd(restartCount, 1u)] = c;
        }
        sets[c] = set;
        if (cost) cost[c] = uint16_t(evaluations < 65535u ? evaluations : 65535u);
    }
}

// The twenty restarts of the listed cells, a cell per workgroup of three
// waves and a restart per group of eight lanes (as searchSlowKernel), appended
// to the cells' sets in search order.  40^3 binary cells: 40 ms with a restart
// per lane, 14.5 so; 47^3 cells of a pure fluid: 0.44 and 0.11 ms
// (160^3: 0.41 and 0.70, of 11 ms a flash).
template <int NS, int NL>
__global__ __launch_bounds__(192, RAMD_SEARCH_MIN_WAVES) void searchRestartsKernel(
    const HemModel<NS>* __restrict__ globalModel, FlashCells cells, CellList list, CandidateSet* __restrict__ sets,
    uint16_t* __restrict__ cost, unsigned long long* __restrict__ phases) {
    const uint32_t count = list.size();
    if (blockIdx.x >= count) return;  // uniform per workgroup
    const HemModel<NS>& model = workgroupModel(globalModel);
    __shared__ StartRecord found[kRestarts];
    uint32_t total = 0;
    const uint32_t s = threadIdx.x / 8u;
    for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {  // uniform per workgroup
        if (s < kRestarts) {
            Counts n = {0, 0, 0, 0, 0, 0, 0};
            Flash<NS, NL, float, true, false, false, kModelLds, 8> f(model, n);
            cells.load<NS>(f, list.cells[i]);
            StartRecord r;
            r.bits = f.searchSeed(kStarts + int(s), r.x);
            r.bits |= n.phases << 2;
            if (threadIdx.x % 8u == 0) {
                found[s] = r;
                total += n.phases;
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t c = list.cells[i];
            CandidateSet set = sets[c];
            uint32_t evaluations = 0;
            for (int k = 0; k < kRestarts; ++k) {
                const StartRecord r = found[k];
                evaluations += r.bits >> 2;
                if (r.bits & kStartFound) noteCandidate(set, kRestartCandidate, int16_t(k), r.x, true);
            }
            sets[c] = set;
            if (cost) {
                evaluations += cost[c];
                cost[c] = uint16_t(evaluations < 65535u ? evaluations : 65535u);
            }
        }
        __syncthreads();
    }
    const uint32_t sum = waveSum(total);
    if (threadIdx.x % 64u == 0) atomicAdd(phases, (unsigned long long)sum);
}

// ---- a pure fluid's search, directed by its saturation curve --------------
//
// At a given (rho, e) a pure fluid has one equilibrium: two phases where some
// saturation temperature T has v_l(T) < 1/rho < v_v(T) and the lever rule's
// energy equal to e, one phase elsewhere.  Which it is, and where, is looked
// up: T by bisection in a table of the saturation curve, or, outside the
// dome, by Newton's method on e(T) at fixed rho.  The reference accepts a
// cell only where one of its solves arrives, so one has to be seen to: for
// one phase its own solve, for two any seed (of the step-start temperature,
// or of a restart temperature: those run only if no other start finds a
// stable point, and here none could).  The seed nearest the known liquid
// fraction arrives in about 90 % of the two-phase cells of a seeded box, and
// of the rest the restart nearest the known point in as many as all twenty
// restarts together; the second try runs over a compacted list.  The
// refinement then confirms the point with the FP64 solver and stability
// test, as it does a searched candidate.  A cell whose solves do not arrive
// or whose point is not confirmed (and every cell the table says too little
// about: colder than the table, near the critical point or the dome's edge,
// outside the model's range) runs the whole search, but for the frozen
// solves that cannot lead to the known point.
__global__ void saturationInitKernel(SaturationTable* __restrict__ table) {
    if (threadIdx.x == 0) table->count = kSaturationRows;
}
// One node per thread: ln p by Newton on mu_l = mu_v (d(mu / RT) / d ln p = z),
// kept between the pressures known to be too low (no liquid) and too high
// (no vapour).  The first node without a solution ends the table.
template <int NS>
__global__ __launch_bounds__(64) void saturationKernel(const HemModel<NS>* __restrict__ globalModel,
                                                       SaturationTable* __restrict__ table) {
    const HemModel<NS>& model = workgroupModel(globalModel);
    const int i = int(blockIdx.x * 64 + threadIdx.x);
    if (i >= kSaturationRows) return;
    const double T0 = hi(model.Tmin, model.liquidTmin);
    const double dT = (lo(model.Tmax, model.liquidTc) - T0) / kSaturationRows, T = T0 + i * dT;
    if (i == 0) {
        table->T0 = T0;
        table->dT = dT;
    }
    Counts n = {0, 0, 0, 0, 0, 0, 0};
    Flash<NS, 1, double, false, false, false, kModelLds> f(model, n);
    const double Tc = model.liquid.Tc[0], pc = kOmegaB * kR * Tc / model.liquid.b[0];
    double low = ::log(model.pmin) - 20, high = ::log(pc);
    double x = clamp(high + 5.373 * (1 + (model.liquid.kappa[0] - .37464) / 1.54226) * (1 - Tc / T), low, high);
    bool found = false;
    PRState g, l;
    for (int it = 0; it < 60 && !found; ++it) {
        const double p = ::exp(x);
        const double Y[NS] = {1};
        double muG[NS], muL[1];
        if (f.gasTP(T, p, Y, g, muG) != kOk) high = x;
        else if (f.liquidTP(T, p, l, muL) != kOk) low = x;
        else {
            const double RT = kR * T, difference = (muL[0] - muG[0]) / RT, slope = p * (l.V - g.V) / RT;
            if (difference > 0) low = x;
            else high = x;
            const double next = x - difference / slope;
            found = ::fabs(next - x) < 1e-11;
            x = next > low && next < high ? next : .5 * (low + high);
            continue;
        }
        x = .5 * (low + high);
    }
    if (!found || !(g.rho < l.rho)) {
        atomicMin(&table->count, i);
        return;
    }
    table->row[i] = {1 / l.rho, 1 / g.rho, l.e, g.e, x};
}

// Newton's method on e(T) = u at fixed density (single precision).
template <int NS>
__device__ inline bool temperatureAt(const Table<NS>& t, float V, float u, float low, float high, float& T,
                                     uint32_t& evaluations) {
    const float b = float(t.b[0]), W = float(t.W[0]), Rg = float(kR), sq2 = float(kSqrt2);
    const float L = m_log((V + (1 + sq2) * b) / (V + (1 - sq2) * b)) / (2 * sq2 * b);
    const float one[1] = {1};
    for (int it = 0; it < 20; ++it) {
        MixT<float> mx;
        float cpR, hRT, sR;
        ++evaluations;
        if (mixing(t, T, one, mx) != kOk) return false;
        nasa(region(t, 0, T), T, cpR, hRT, sR);
        const float F = Rg * T * (hRT - 1) + L * (T * mx.da - mx.aa) - u * W;
        const float cv = Rg * (cpR - 1) + L * T * mx.d2a;
        const float step = F / cv;
        if (!(cv > 0) || !fin(step)) return false;
        const float next = clamp(T - step, low, high);
        const bool done = ab(next - T) <= 3e-6f * T;
        T = next;
        if (done) return T > low && T < high;
    }
    return false;
}

// Where a saturated state's energy passes the cell's, or the dome ends: both
// are crossed once as T rises at fixed v.
__device__ inline bool saturationPast(const SaturationRow& r, double v, double u, bool& outside) {
    outside = v <= r.vl || v >= r.vv;
    const double x = (v - r.vl) / (r.vv - r.vl);
    return outside || r.el + x * (r.ev - r.el) > u;
}
// Liquid fractions (and energies, in units of the vaporisation energy) this
// close to the dome's edge are left to the search, whose candidates on both
// sides of the edge the refinement compares.
constexpr double kDomeEdge = 1e-3;

// The cell's equilibrium point into its set (count 0: not known).
template <int NS>
__device__ inline void directCandidate(const HemModel<NS>& m, const SaturationTable& table, double rho, double energy,
                                        double guessT, CandidateSet& set, uint32_t& evaluations) {
    set.count = 0;
    set.flags = kDirect;
    if (!fin(energy) || !(rho > 0) || !fin(rho)) return;
    const double v = 1 / rho, u = energy / rho;
    const int rows = table.count;
    if (rows < 2) return;
    int low = -1, high = rows;
    bool outside = false, highOutside = false;
    while (high - low > 1) {
        const int mid = (low + high) >> 1;
        if (saturationPast(table.row[mid], v, u, outside)) { high = mid; highOutside = outside; }
        else low = mid;
    }
    if (high == rows) return;             // near the critical point, or above it
    if (low < 0 && !highOutside) return;  // colder than the table
    if (!highOutside) {  // two phases, between the rows low and low + 1
        const SaturationRow a = table.row[low], b = table.row[high];
        const double ea = a.el + (v - a.vl) / (a.vv - a.vl) * (a.ev - a.el);
        const double eb = b.el + (v - b.vl) / (b.vv - b.vl) * (b.ev - b.el);
        const double w = clamp((u - ea) / (eb - ea), 0., 1.);
        const double vl = a.vl + w * (b.vl - a.vl), vv = a.vv * ::exp(w * ::log(b.vv / a.vv));
        const double liquid = (vv - v) / (vv - vl);
        if (liquid > kDomeEdge) set.flags |= kNotGas;
        if (liquid < 1 - kDomeEdge) set.flags |= kNotLiquid;
        if (!(liquid > kDomeEdge && liquid < 1 - kDomeEdge)) return;
        const float at[3] = {float(a.lnp + w * (b.lnp - a.lnp)), float(::log(table.T0 + (low + w) * table.dT)),
                             float(liquid)};
        noteCandidate(set, kSeedCandidate, 0, at, false);
        return;
    }
    if (low >= 0) {
        // the dome ends between the rows: one phase where its edge lies well below the cell's energy
        const SaturationRow& r = table.row[high];
        const bool vapour = v >= r.vv;
        if (u < (vapour ? r.ev : r.el) + kDomeEdge * (r.ev - r.el)) {
            set.flags |= vapour ? kNotLiquid : kNotGas;
            return;
        }
    }
    const SaturationRow& r = table.row[high];
    const bool vapour = v >= r.vv;
    float T = float(clamp(guessT, m.Tmin, m.Tmax));
    const double V = v * m.gas.W[0];
    if (!(V > m.gas.b[0]) || !temperatureAt(m.gas, float(V), float(u), float(m.Tmin), float(m.Tmax), T, evaluations))
        return;
    const double one[1] = {1};
    Mix mx;
    if (mixing(m.gas, double(T), one, mx) != kOk) return;
    const double p = kR * T / (V - mx.b) - mx.aa / (V * V + 2 * V * mx.b - mx.b * mx.b);
    if (!(p >= m.pmin && p <= m.pmax)) return;
    const float at[3] = {float(::log(p)), m_log(T), 0.f};
    noteCandidate(set, vapour || T >= float(m.liquidTc) ? kGasCandidate : kLiquidCandidate, 0, at, false);
}

// The liquid fraction of seed j for a flash input.
template <int NS>
__device__ inline float seedFraction(const FlashInput<NS>& at, int j) {
    return j == 0 ? clamp(float(at.guessLiquid / at.q[0]), 0.f, 1.f) : j == 1 ? .5f : j == 2 ? .95f : j == 3 ? .1f : .9999f;
}
template <int NS>
__device__ inline int nearestSeed(const FlashInput<NS>& at, float liquid, int first) {
    int nearest = first;
    for (int j = first + 1; j < 5; ++j)
        if (ab(seedFraction(at, j) - liquid) < ab(seedFraction(at, nearest) - liquid)) nearest = j;
    return nearest;
}

// Looks every cell up and runs the two-phase cells' nearest seed; those it
// does not arrive for go to `again`, the one-phase cells to `single`.  The
// seed's solve is inlined and keeps its state in registers (Flash::activeLean);
// through the general solver's calls it waited for the stack for 75 % of its
// cycles: 160^3 cells 4.5 -> 3.1 ms with both lists.
template <int NS>
__global__ __launch_bounds__(64, RAMD_LEAN_MIN_WAVES) void directKernel(
    const HemModel<NS>* __restrict__ globalModel, const SaturationTable* __restrict__ table, FlashCells cells,
    const uint32_t* __restrict__ order, uint32_t count, CandidateSet* __restrict__ sets, uint16_t* __restrict__ cost,
    unsigned long long* __restrict__ phases, SearchScratch scratch) {
    const HemModel<NS>& model = workgroupModel(globalModel);
    const uint32_t i = blockIdx.x * 64u + threadIdx.x;
    Counts n = {0, 0, 0, 0, 0, 0, 0};
    if (i < count && cells.flashed(order[i])) {
        const uint32_t c = order[i];
        CandidateSet set;
        FlashInput<NS> at;
        cells.load<NS>(at, c);
        directCandidate<NS>(model, *table, at.q[0], at.energy, at.guessT, set, n.phases);
        if (set.count && set.c[0].kind != kSeedCandidate) {
            set.flags |= kSingle;
            scratch.single[atomicAdd(scratch.singleCount, 1u)] = c;
        } else if (set.count) {
            Flash<NS, 1, float, true, false, false, kModelLds> f(model, n);
            cells.load<NS>(f, c);
            if (!f.seedArrives(2 + nearestSeed(at, set.c[0].x[2], 0))) {
                set.count = 0;
                scratch.again[atomicAdd(scratch.againCount, 1u)] = c;
            }
        }
        CandidateSet& o = sets[c];
        o.count = set.count;
        o.flags = set.flags;
        o.c[0] = set.c[0];
        if (cost) cost[c] = uint16_t(n.phases < 65535u ? n.phases : 65535u);
    }
    const uint32_t sum = waveSum(n.phases);
    if (threadIdx.x == 0) atomicAdd(phases, (unsigned long long)sum);
}

// SINGLE: the listed one-phase cells' frozen solve.  Otherwise the second try
// of the listed two-phase cells: the restart nearest the known point in
// temperature and liquid fraction (their sets hold the point with a count of
// zero).
template <int NS, bool SINGLE>
__global__ __launch_bounds__(64, SINGLE ? RAMD_SEARCH_MIN_WAVES : RAMD_LEAN_MIN_WAVES) void directListKernel(
    const HemModel<NS>* __restrict__ globalModel, FlashCells cells, CellList list, CandidateSet* __restrict__ sets,
    uint16_t* __restrict__ cost, unsigned long long* __restrict__ phases) {
    const uint32_t count = list.size();
    if (blockIdx.x * 64u >= count) return;  // uniform per workgroup
    const HemModel<NS>& model = workgroupModel(globalModel);
    uint32_t total = 0;
    for (uint32_t base = blockIdx.x * 64u; base < count; base += gridDim.x * 64u) {
        const uint32_t i = base + threadIdx.x;
        if (i < count) {
            const uint32_t c = list.cells[i];
            Counts n = {0, 0, 0, 0, 0, 0, 0};
            Flash<NS, 1, float, true, false, false, kModelLds> f(model, n);
            cells.load<NS>(f, c);
            if constexpr (SINGLE) {
                float x[3];
                if (!(f.searchFrozen(sets[c].c[0].kind == kLiquidCandidate, x) & kStartFound)) sets[c].count = 0;
            } else {
                FlashInput<NS> at;
                cells.load<NS>(at, c);
                const float T = m_exp(sets[c].c[0].x[1]);
                int t = 0;
                for (int k = 1; k < 4; ++k)
                    if (ab(f.restartTemperature(k) - T) < ab(f.restartTemperature(t) - T)) t = k;
                if (f.seedArrives(kStarts + 5 * t + nearestSeed(at, sets[c].c[0].x[2], 1))) sets[c].count = 1;
            }
            total += n.phases;
            if (cost) {
                const uint32_t evaluations = n.phases + cost[c];
                cost[c] = uint16_t(evaluations < 65535u ? evaluations : 65535u);
            }
        }
    }
    const uint32_t sum = waveSum(total);
    if (threadIdx.x == 0) atomicAdd(phases, (unsigned long long)sum);
}

// ---- launches --------------------------------------------------------------
#define RAMD_SPECIES(LAUNCH)                         \
    if (ns == 1 && nl == 0) { LAUNCH(1, 0); }        \
    else if (ns == 1) { LAUNCH(1, 1); }              \
    else if (nl == 0) { LAUNCH(2, 0); }              \
    else { LAUNCH(2, 1); }

void launchSaturation(const void* model, SaturationTable* table, hipStream_t stream) {
    hipLaunchKernelGGL(saturationInitKernel, dim3(1), dim3(64), 0, stream, table);
    hipLaunchKernelGGL((saturationKernel<1>), dim3((kSaturationRows + 63) / 64), dim3(64), 0, stream,
                       static_cast<const HemModel<1>*>(model), table);
    RAMD_HIP(hipGetLastError());
}

void launchSearch(int ns, int nl, const void* model, const FlashCells& cells, const uint32_t* order, uint32_t count,
                  CandidateSet* sets, uint16_t* cost, unsigned long long* phases, hipStream_t stream, unsigned block) {
    const unsigned blocks = unsigned((size_t(count) + block - 1) / block);
#define RAMD_SEARCH(NS_, NL_)                                                                                \
    hipLaunchKernelGGL((searchKernel<NS_, NL_>), dim3(blocks), dim3(block), 0, stream,                        \
                       static_cast<const HemModel<NS_>*>(model), cells, order, count, sets, cost, phases)
    RAMD_SPECIES(RAMD_SEARCH)
#undef RAMD_SEARCH
    RAMD_HIP(hipGetLastError());
}

// Waves of a launch over a list counted on the device: enough to fill the
// chip at the search's five waves per SIMD; a longer list takes more rounds.
constexpr unsigned kListWaves = 5120;

void launchDirect(const void* model, const SaturationTable* table, const FlashCells& cells, const uint32_t* order,
                  uint32_t count, const SearchScratch& scratch, CandidateSet* sets, uint16_t* cost,
                  unsigned long long* phases, hipStream_t stream) {
    const unsigned waves = unsigned((size_t(count) + 63) / 64);
    hipLaunchKernelGGL((directKernel<1>), dim3(waves), dim3(64), 0, stream, static_cast<const HemModel<1>*>(model),
                       table, cells, order, count, sets, cost, phases, scratch);
    hipLaunchKernelGGL((directListKernel<1, false>), dim3(std::min(kListWaves, waves)), dim3(64), 0, stream,
                       static_cast<const HemModel<1>*>(model), cells,
                       CellList{scratch.again, 0, scratch.againCount}, sets, cost, phases);
    hipLaunchKernelGGL((directListKernel<1, true>), dim3(std::min(kListWaves, waves)), dim3(64), 0, stream,
                       static_cast<const HemModel<1>*>(model), cells,
                       CellList{scratch.single, 0, scratch.singleCount}, sets, cost, phases);
    RAMD_HIP(hipGetLastError());
}

void launchSearchStarts(int ns, int nl, const void* model, const FlashCells& cells, const CellList& list, size_t stride,
                        const SearchScratch& scratch, bool directed, CandidateSet* sets, uint16_t* cost,
                        unsigned long long* phases, hipStream_t stream) {
    const unsigned waves = unsigned((stride + 63) / 64);
    const unsigned blocks = list.counted ? std::min(waves, kListWaves / kStarts) : waves;
#define RAMD_STARTS(NS_, NL_)                                                                                \
    hipLaunchKernelGGL((searchStartsKernel<NS_, NL_>), dim3(blocks, kStarts), dim3(64), 0, stream,            \
                       static_cast<const HemModel<NS_>*>(model), cells, list, stride,                                   \
                       directed ? sets : nullptr, scratch.records, scratch.restarts, scratch.slowCount, phases); \
    if constexpr (NS_ > 1 && NL_ > 0) {                                                                       \
        const size_t slow = std::min(stride * kStarts, size_t(RAMD_SLOW_GROUPS));                             \
        hipLaunchKernelGGL((searchSlowKernel<NS_, NL_, 8>), dim3(unsigned(std::min(size_t(kListWaves), (slow + 7) / 8))), \
                           dim3(64), 0, stream, static_cast<const HemModel<NS_>*>(model), cells, list, stride, \
                           scratch.records, scratch.restarts, scratch.slowCount, phases);                     \
        if (stride * kStarts > RAMD_SLOW_GROUPS)                                                              \
            hipLaunchKernelGGL((searchSlowKernel<NS_, NL_, 1>), dim3(kListWaves), dim3(64), 0, stream,         \
                               static_cast<const HemModel<NS_>*>(model), cells, list, stride, scratch.records, \
                               scratch.restarts, scratch.slowCount, phases);                                  \
    }                                                                                                         \
    hipLaunchKernelGGL((searchMergeKernel<NS_>), dim3(std::min(2048u, (waves + 3) / 4)), dim3(256), 0, stream, \
                       static_cast<const HemModel<NS_>*>(model), cells, list, stride, scratch.records, sets, cost, \
                       scratch.restarts, scratch.restartCount);                                              \
    hipLaunchKernelGGL((searchRestartsKernel<NS_, NL_>),                                                      \
                       dim3(unsigned(std::min(size_t(kListWaves), stride))), dim3(192), 0, stream,            \
                       static_cast<const HemModel<NS_>*>(model), cells,                                       \
                       CellList{scratch.restarts, 0, scratch.restartCount}, sets, cost, phases)
    RAMD_SPECIES(RAMD_STARTS)
#undef RAMD_STARTS
    RAMD_HIP(hipGetLastError());
}
#undef RAMD_SPECIES

}  // namespace ramd
