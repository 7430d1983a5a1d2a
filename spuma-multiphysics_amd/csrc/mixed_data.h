// SPDX-License-Identifier: GPL-3.0-or-later
// What the mixed flash keeps per cell between its kernels, and the device
// buffers that hold it (plain data; nothing here needs a device).
#ifndef REACTIVE_AMD_MIXED_DATA_H
#define REACTIVE_AMD_MIXED_DATA_H
#include <cstddef>
#include <cstdint>

namespace ramd {

// Candidates of the single-precision search, in search order.
enum CandidateKind : int16_t { kGasCandidate = 0, kLiquidCandidate = 1, kSeedCandidate = 2, kRestartCandidate = 3 };
struct Candidate {
    float x[3];     // ln p, ln T, liquid fraction (0 for the gas and all-liquid candidates)
    int16_t kind;   // CandidateKind
    int16_t index;  // seed j, or 5 t + j for restart temperature t
};
constexpr int kMaxCandidates = 6;
enum CandidateFlags : uint32_t {
    kRestartsSearched = 1u,  // the search ran the restart temperatures
    kOverflow = 2u,          // more distinct candidates than the set holds
    kSeedsPruned = 4u,       // the stable-gas pruning skipped the seeds
    kDirect = 8u,            // the directed search's (saturation table): one candidate or none
    kNotGas = 16u,           // with kDirect: the all-gas solve cannot lead to the equilibrium
    kNotLiquid = 32u,        // with kDirect: nor can the all-liquid one
    kSingle = 64u,           // with kDirect: the point has one phase
};
enum StartBits : uint32_t {
    kStartFound = 1u,   // converged, or stalled near convergence
    kStartStable = 2u,  // converged and stable in single precision
};
constexpr int kStarts = 7, kRestarts = 20;  // all gas, all liquid, five seeds; the seeds from four temperatures
struct CandidateSet {
    uint32_t count, flags;
    Candidate c[kMaxCandidates];
};
static_assert(sizeof(CandidateSet) == 104, "candidate set layout");

// One start's outcome: the point, kStart* bits and the evaluations above them.
struct StartRecord {
    float x[3];
    uint32_t bits;
};
// Saturated liquid and vapour at evenly spaced temperatures: specific volumes
// and energies, ln p.  Interpolated between 2,048 rows over N2O's 161 K they
// lie within 1e-6 of the curve except next to the critical point, inside the
// refinement's one or two Newton steps.
constexpr int kSaturationRows = 2048;
struct SaturationRow {
    double vl, vv, el, ev, lnp;
};
struct SaturationTable {
    int count, pad;
    double T0, dT;
    SaturationRow row[kSaturationRows];
};

// Scratch of the search: kStarts records per listed cell (record s of list
// position i at s stride + i), the cells to restart (two species: before that
// the slow starts, up to kStarts per listed cell), and the directed search's
// two-phase cells to try again and one-phase cells; the counts are zero on
// entry.
struct SearchScratch {
    StartRecord* records;
    uint32_t *restarts, *again, *single;
    unsigned *restartCount, *againCount, *singleCount, *slowCount;
};
// Counts of the mixed flash's lists, in one array that a kernel clears before
// every flash.
enum ListCount : int {
    kDeferredCount = 0,  // cells whose refinement is deferred
    kSearchCount,        // cells the saturation table leaves to the search
    kRestartCount,       // cells to restart
    kAgainCount,         // two-phase cells the directed search tries again
    kSingleCount,        // one-phase cells
    kSlowCount,          // slow starts
    kListCounts
};

// The buffers of the mixed flash of `cells` cells, made on its first use.
struct MixedScratch {
    CandidateSet* sets = nullptr;
    uint32_t* queue = nullptr;  // deferred cells
    unsigned* counts = nullptr;
    // a pure fluid's saturation table, and the cells it left to the search
    SaturationTable* saturation = nullptr;
    bool tableMade = false;
    uint32_t* searchList = nullptr;
    SearchScratch search = {};

    // alloc(p, n): n elements of device memory into p, where p is null, or an
    // exception.  Every call goes through all the buffers, so that a call
    // after one that ran out of memory makes the rest of them.
    template <class Alloc>
    void need(int ns, bool prune, bool pure, size_t cells, Alloc alloc) {
        alloc(queue, cells);
        alloc(counts, size_t(kListCounts));
        if (!prune) {
            // one record per start and cell; a pure fluid searches only the cells its table leaves
            alloc(search.records, kStarts * cells);
            alloc(search.restarts, (ns > 1 ? kStarts : 1) * cells);
            search.restartCount = counts + kRestartCount;
            search.slowCount = counts + kSlowCount;
        }
        if (pure) {
            alloc(searchList, cells);
            alloc(search.again, cells);
            search.againCount = counts + kAgainCount;
            alloc(search.single, cells);
            search.singleCount = counts + kSingleCount;
            alloc(saturation, size_t(1));
        }
        alloc(sets, cells);
    }
};

}  // namespace ramd
#endif
