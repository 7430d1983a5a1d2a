// SPDX-License-Identifier: GPL-3.0-or-later
// Batched HEM UV flash plugin for gfx950: the reactive_gpu_hem_* ABI
// (src/reactiveThermo/reactiveGpuHem.h:40-84) over the device flash of
// flash_device.h.
//
// Execution: one work-item per cell in 64-lane workgroups (one wavefront),
// cells visited in heavy-first bucket order (the reference's scheduling key,
// src/reactiveTransport/reactiveHemBucket.h:13-18): liquid-active cells run
// the long seeded searches, so they go first and cheap gas cells fill the
// tail.  Work counters are reduced per wavefront and accumulated with one
// 64-bit atomic per counter per wavefront.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <array>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "hip_common.h"
#include "flash_device.h"
#include "model_image.h"
#include "hem_internal.h"
#include "flash_step.h"
#include "lane_flash.h"
#include "refine_flash.h"
#include "reactive_gpu_hem.h"
#include "reactive_amd.h"

namespace ramd {

static_assert(sizeof(ThermoOut) == sizeof(ReactiveThermoState), "state layout");
static_assert(sizeof(HemCapillaryDev) == sizeof(ReactiveGpuHemCapillaryInputV2) &&
                  offsetof(HemCapillaryDev, equilibrium) == offsetof(ReactiveGpuHemCapillaryInputV2, equilibrium),
              "capillary input layout");
static_assert(sizeof(HemOutputDev) == sizeof(ReactiveGpuHemOutputV1) &&
                  offsetof(HemOutputDev, success) == offsetof(ReactiveGpuHemOutputV1, success),
              "output layout");

__global__ void clearCountsKernel(unsigned* __restrict__ counts) {
    if (threadIdx.x < kListCounts) counts[threadIdx.x] = 0;
}

// totals[k] = sum over b < blocks of partials[b * width + k], k < width: one
// 64-lane workgroup, a fixed summation order (no atomics, nothing cleared).
__global__ __launch_bounds__(64) void reducePartialsKernel(const unsigned long long* __restrict__ partials,
                                                          unsigned blocks, int width,
                                                          unsigned long long* __restrict__ totals) {
    for (int k = 0; k < width; ++k) {
        unsigned long long sum = 0;
        for (unsigned b = threadIdx.x; b < blocks; b += 64) sum += partials[size_t(b) * width + k];
        for (int offset = 32; offset > 0; offset >>= 1) sum += __shfl_xor(sum, offset, 64);
        if (threadIdx.x == 0) totals[k] = sum;
    }
}

__global__ void zeroTotalsKernel(unsigned long long* totals, int n) {
    if (threadIdx.x < n) totals[threadIdx.x] = 0;
}
__global__ void queueCountKernel(const unsigned* __restrict__ count, unsigned long long* __restrict__ total) {
    if (threadIdx.x == 0) *total = *count;
}

// Scheduling key (reactiveHemBucket.h:13-18).
inline unsigned bucketKey(const double* q, int ns, int activeLiquids) {
    unsigned present = 0, dominant = 0;
    for (int k = 0; k < ns; ++k) {
        if (q[k] > 0) ++present;
        if (q[k] > q[dominant]) dominant = unsigned(k);
    }
    const unsigned liquids = activeLiquids < 0 ? 0u : (activeLiquids > 3 ? 3u : unsigned(activeLiquids));
    return (liquids << 6) | ((present > 7 ? 7u : present) << 3) | (dominant > 7 ? 7u : dominant);
}

HemHandle::~HemHandle() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (auto e : events)
        if (e) (void)hipEventDestroy(e);
    for (void* p : allocations) (void)hipFree(p);
    if (stream) (void)hipStreamDestroy(stream);
}

void* HemHandle::allocate(size_t bytes) {
    void* p = nullptr;
    RAMD_HIP(hipMalloc(&p, bytes));
    allocations.push_back(p);
    deviceBytes += bytes;
    return p;
}

void HemHandle::ensureHostPath() {
    if (hostReady) return;
    dq = static_cast<double*>(allocate(capacity * ns * sizeof(double)));
    de = static_cast<double*>(allocate(capacity * sizeof(double)));
    dguess = static_cast<ThermoOut*>(allocate(capacity * sizeof(ThermoOut)));
    dout = static_cast<HemOutputDev*>(allocate(capacity * sizeof(HemOutputDev)));
    dorder = static_cast<uint32_t*>(allocate(capacity * sizeof(uint32_t)));
    hostOrder.resize(capacity);
    hostKey.resize(capacity);
    hostOut.resize(capacity);
    hostReady = true;
}

unsigned HemHandle::launch(const double* q, const double* e, const ThermoOut* g, const uint32_t* order, size_t count,
                           const HemCapillaryDev* capillary, HemOutputDev* out, hipStream_t s,
                           unsigned long long* partials, unsigned slots) {
    if (!count) return 0;
    const unsigned blocks = unsigned((count + 63) / 64);
    if (!partials) hipLaunchKernelGGL(zeroTotalsKernel, dim3(1), dim3(64), 0, s, totals, 8);
    const FlashCells cells = {q, 0, e, g, nullptr, nullptr};
    if (count <= RAMD_GROUP_CELLS && (!partials || count <= slots)) {
        FlashSink sink = {};
        sink.hem = out;
        sink.totals = totals;
        sink.partials = partials;
        launchGroupFlash(ns, nl, analytic, boundary, model, cells, order, uint32_t(count), capillary, sink, s);
        return unsigned(count);
    }
#define RAMD_HEM_LAUNCH(NS_, NL_)                                                                                  \
    hipLaunchKernelGGL((hemFlashKernel<NS_, NL_, false, false>), dim3(blocks), dim3(64), 0, s,                     \
                       static_cast<const HemModel<NS_>*>(model), cells, order, uint32_t(count), capillary, out,    \
                       totals, partials)
    if (capillary || boundary || ns != 1 || (nl && analytic))
        launchLaneHem(ns, nl, analytic, boundary, model, cells, order, uint32_t(count), capillary, out, totals, partials, s);
    else if (nl == 0) RAMD_HEM_LAUNCH(1, 0);
    else RAMD_HEM_LAUNCH(1, 1);
#undef RAMD_HEM_LAUNCH
    RAMD_HIP(hipGetLastError());
    return blocks;
}

void HemHandle::launchMixed(const double* q, const double* e, const ThermoOut* g, const uint32_t* order,
                            size_t count, HemOutputDev* out, hipStream_t s) {
    if (!count) return;
    mixed.need(ns, prune, pure(), capacity, [this](auto*& p, size_t n) {
        if (!p) p = static_cast<std::remove_reference_t<decltype(p)>>(allocate(n * sizeof(*p)));
    });
    if (mixed.saturation && !mixed.tableMade) {
        launchSaturation(model, mixed.saturation, s);
        mixed.tableMade = true;
    }
    const SearchScratch& scratch = mixed.search;
    SaturationTable* const saturation = mixed.saturation;
    CandidateSet* const sets = mixed.sets;
    uint32_t *const queue = mixed.queue, *const searchList = mixed.searchList;
    unsigned *const queueCount = mixed.counts + kDeferredCount, *const searchCount = mixed.counts + kSearchCount;
    const unsigned blocks = unsigned((count + 63) / 64);
    const FlashCells cells = {q, 0, e, g, nullptr, nullptr};
    const CellList whole = {order, uint32_t(count), nullptr}, left = {searchList, 0, searchCount};
    const CellList first = saturation ? CellList{scratch.single, 0, scratch.singleCount} : whole;
    FlashSink sink = {};
    sink.hem = out;
    sink.totals = totals;
    hipLaunchKernelGGL(zeroTotalsKernel, dim3(1), dim3(64), 0, s, totals, 10);
    hipLaunchKernelGGL(clearCountsKernel, dim3(1), dim3(64), 0, s, mixed.counts);
    if (saturation) launchDirect(model, saturation, cells, order, uint32_t(count), scratch, sets, nullptr, totals + 8, s);
    else if (prune) launchSearch(ns, nl, model, cells, order, uint32_t(count), sets, nullptr, totals + 8, s, 64);
    else launchSearchStarts(ns, nl, model, cells, whole, count, scratch, false, sets, nullptr, totals + 8, s);
    if (saturation)
        launchRefineTwoPhase(model, cells, order, uint32_t(count), sets, sink, scratch, searchList, searchCount, s);
    const auto refine = [&](const CellList& list, unsigned grid) {
        if (ns == 2) return launchHemRefineTwo(nl, model, cells, list, sets, sink, queue, queueCount, grid, s);
#define RAMD_HEM_REFINE(NL_)                                                                                      \
    hipLaunchKernelGGL((hemRefineKernel<1, NL_>), dim3(grid), dim3(64), 0, s, static_cast<const HemModel<1>*>(model), \
                       cells, list, sets, out, totals, queue, queueCount, searchList, searchCount)
        if (nl == 0) RAMD_HEM_REFINE(0);
        else RAMD_HEM_REFINE(1);
#undef RAMD_HEM_REFINE
    };
    refine(first, blocks);
    if (saturation) {
        launchSearchStarts(ns, nl, model, cells, left, count, scratch, true, sets, nullptr, totals + 8, s);
        refine(left, std::min(2048u, blocks));
    }
    launchRefineQueue(ns, nl, model, cells, queue, queueCount, sets, sink, s);
    hipLaunchKernelGGL(queueCountKernel, dim3(1), dim3(64), 0, s, queueCount, totals + 9);
    RAMD_HIP(hipGetLastError());
}

// The process's default flash arithmetic: REACTIVE_AMD_HEM_ARITHMETIC=mixed
// selects the mixed flash, anything else (or nothing) plain FP64.  Read once,
// so the numerical policy a driver hashes and the handles it creates agree.
static int defaultArithmetic() {
    static const int mode = [] {
        const char* v = std::getenv("REACTIVE_AMD_HEM_ARITHMETIC");
        return v && std::strcmp(v, "mixed") == 0 ? REACTIVE_AMD_FLASH_MIXED : REACTIVE_AMD_FLASH_FP64;
    }();
    return mode;
}

HemHandle* createHem(const void* raw, size_t bytes, size_t capacity, bool hostPath) {
    using namespace image;
    require(raw && bytes == sizeof(Model) && capacity && capacity <= UINT32_MAX, "Invalid HIP HEM model/capacity");
    Model m;
    std::memcpy(static_cast<void*>(&m), raw, sizeof(m));
    require(validModel(m), "Invalid HIP HEM model tables or domain");
    require(m.ns == 1 || m.ns == 2, "This HEM build supports 1 or 2 gas species");
    require(m.nl <= 1, "This HEM build supports at most one pure liquid");
    require(!(m.nl && m.condensedKind[0]), "Solid condensed phases are not provided by this HEM build");
    int devices = 0;
    RAMD_HIP(hipGetDeviceCount(&devices));
    require(devices > 0, "No HIP device");
    std::unique_ptr<HemHandle> h(new HemHandle);
    h->ns = m.ns;
    h->nl = m.nl;
    h->analytic = m.analyticJacobian != 0;
    h->boundary = m.boundaryRecovery != 0;
    h->prune = m.stableGasPrune != 0;
    h->arithmetic = defaultArithmetic();
    h->capacity = capacity;
    h->device = currentDevice();
    RAMD_HIP(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
    for (auto& e : h->events) RAMD_HIP(hipEventCreate(&e));
    if (m.ns == 1) {
        HemModel<1> d;
        buildDeviceModel<1>(m, d);
        h->model = h->allocate(sizeof(d));
        RAMD_HIP(hipMemcpy(h->model, &d, sizeof(d), hipMemcpyHostToDevice));
    } else {
        HemModel<2> d;
        buildDeviceModel<2>(m, d);
        h->model = h->allocate(sizeof(d));
        RAMD_HIP(hipMemcpy(h->model, &d, sizeof(d), hipMemcpyHostToDevice));
    }
    h->totals = static_cast<unsigned long long*>(h->allocate(10 * sizeof(unsigned long long)));
    h->modelBytes = h->deviceBytes;
    if (hostPath) h->ensureHostPath();
    return h.release();
}

// Host-array batch (reactiveGpuHem.cuh:227-349 semantics).
int runHost(HemHandle* h, const double* q, const double* energy, const ReactiveGpuHemCapillaryInputV2* capillary,
            size_t count, ReactiveThermoState* states, int* success, ReactiveGpuHemProfileV1* profile) {
    require(h && q && energy && states && success && profile && profile->abiVersion == 1 &&
                profile->structBytes == sizeof(*profile),
            "Invalid HIP HEM batch arguments");
    require(count && count <= h->capacity, "HIP HEM batch exceeds capacity");
    if (capillary) {
        for (size_t c = 0; c < count; ++c) {
            const auto& x = capillary[c];
            require(fin(x.color) && x.color >= 0 && x.color <= 1 && fin(x.pressureJump) &&
                        (x.equilibrium == 0 || x.equilibrium == 1),
                    "Invalid HIP HEM capillary cell input");  // reactiveGpuHem.cuh:237-243
        }
    }
    RAMD_HIP(hipSetDevice(h->device));
    h->ensureHostPath();
    if (capillary && !h->dcap)
        h->dcap = static_cast<HemCapillaryDev*>(h->allocate(h->capacity * sizeof(HemCapillaryDev)));
    const auto begin = std::chrono::steady_clock::now();
    // stable counting sort on the scheduling key, heavy buckets first
    std::array<size_t, 256> counts{};
    for (size_t c = 0; c < count; ++c) {
        const unsigned key = bucketKey(q + c * h->ns, h->ns, states[c].activeLiquids);
        h->hostKey[c] = uint8_t(key);
        ++counts[key];
    }
    std::array<size_t, 256> offset{};
    size_t next = 0;
    for (int b = 255; b >= 0; --b) { offset[b] = next; next += counts[b]; }
    for (size_t c = 0; c < count; ++c) h->hostOrder[offset[h->hostKey[c]]++] = uint32_t(c);
    hipStream_t s = h->stream;
    RAMD_HIP(hipEventRecord(h->events[0], s));
    RAMD_HIP(hipMemcpyAsync(h->dq, q, count * h->ns * sizeof(double), hipMemcpyHostToDevice, s));
    RAMD_HIP(hipMemcpyAsync(h->de, energy, count * sizeof(double), hipMemcpyHostToDevice, s));
    RAMD_HIP(hipMemcpyAsync(h->dguess, states, count * sizeof(ThermoOut), hipMemcpyHostToDevice, s));
    RAMD_HIP(hipMemcpyAsync(h->dorder, h->hostOrder.data(), count * sizeof(uint32_t), hipMemcpyHostToDevice, s));
    if (capillary)
        RAMD_HIP(hipMemcpyAsync(h->dcap, capillary, count * sizeof(HemCapillaryDev), hipMemcpyHostToDevice, s));
    RAMD_HIP(hipEventRecord(h->events[1], s));
    // the mixed arithmetic runs the equilibrium flash without the boundary search
    const bool mixed = !capillary && !h->boundary && h->arithmetic == REACTIVE_AMD_FLASH_MIXED;
    if (mixed) h->launchMixed(h->dq, h->de, h->dguess, h->dorder, count, h->dout, s);
    else h->launch(h->dq, h->de, h->dguess, h->dorder, count, capillary ? h->dcap : nullptr, h->dout, s);
    RAMD_HIP(hipEventRecord(h->events[2], s));
    RAMD_HIP(hipMemcpyAsync(h->hostOut.data(), h->dout, count * sizeof(HemOutputDev), hipMemcpyDeviceToHost, s));
    unsigned long long totals[10] = {};
    RAMD_HIP(hipMemcpyAsync(totals, h->totals, sizeof(totals), hipMemcpyDeviceToHost, s));
    RAMD_HIP(hipEventRecord(h->events[3], s));
    RAMD_HIP(hipEventSynchronize(h->events[3]));
    float upload = 0, kernel = 0, download = 0;
    RAMD_HIP(hipEventElapsedTime(&upload, h->events[0], h->events[1]));
    RAMD_HIP(hipEventElapsedTime(&kernel, h->events[1], h->events[2]));
    RAMD_HIP(hipEventElapsedTime(&download, h->events[2], h->events[3]));
    ReactiveGpuHemProfileV1 p{};
    p.abiVersion = 1;
    p.structBytes = sizeof(p);
    p.batches = 1;
    p.submitted = count;
    for (size_t c = 0; c < count; ++c) {
        const HemOutputDev& o = h->hostOut[c];
        success[c] = o.success;
        if (o.success) {
            std::memcpy(&states[c], &o.state, sizeof(ReactiveThermoState));
            ++p.succeeded;
        }
    }
    p.deviceFailures = count - p.succeeded;
    // the mixed arithmetic counts its FP32 search's phase evaluations too
    p.phaseEvaluations = totals[0] + (mixed ? totals[8] : 0);
    h->lastSinglePhases = mixed ? totals[8] : 0;
    h->lastQueued = mixed ? totals[9] : 0;
    p.residualEvaluations = totals[1];
    p.flashCandidates = totals[2];
    p.stableCandidates = totals[3];
    p.finiteDifferenceJacobians = totals[5];
    p.analyticJacobians = totals[7];
    p.transferBytes = count * (h->ns * sizeof(double) + sizeof(double) + sizeof(ThermoOut) + sizeof(uint32_t) +
                               sizeof(HemOutputDev) + (capillary ? sizeof(int) : 0)) +
                      sizeof(totals);
    p.deviceBytes = h->deviceBytes;
    p.hostBytes = h->capacity * (sizeof(HemOutputDev) + sizeof(uint32_t) + sizeof(uint8_t));
    p.wallSeconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - begin).count();
    p.kernelSeconds = kernel / 1000.;
    p.copySeconds = (upload + download) / 1000.;
    *profile = p;
    return 0;
}

// ---- device scratch of the allocation-free resident batch
// (reactive_gpu_hem_run_resident_noalloc_v1).  One slot of 8 counters per
// 64-cell workgroup of a launch, then the 8 batch totals: 1 MiB + 64 B on
// every device the library runs on, held until the process ends.  Every slot
// a call reads, the same call has written first, so nothing is cleared
// between calls; calls that overlap on one device share it and race.
constexpr unsigned kNoAllocBlocks = 16384;
constexpr size_t kNoAllocMaxCells = size_t(kNoAllocBlocks) * 64;  // 1,048,576 cells per call
static __device__ __align__(256) unsigned long long scratch[size_t(kNoAllocBlocks) * 8 + 8];

// scratch's address on `device` (the host-side name of the array is only a
// stand-in): looked up once per device with that device current.
unsigned long long* scratchAddress(int device) {
    constexpr int kDevices = 64;
    static std::mutex lock;
    static unsigned long long* address[kDevices] = {};
    require(device >= 0 && device < kDevices, "HIP device index beyond the allocation-free batch's table");
    std::lock_guard<std::mutex> guard(lock);
    if (!address[device]) {
        void* ptr = nullptr;
        RAMD_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        address[device] = static_cast<unsigned long long*>(ptr);
    }
    return address[device];
}

}  // namespace ramd

using namespace ramd;

extern "C" {

// "" (plain FP64, separate rounding) or, with the mixed arithmetic as the
// process default, the FP32 combined policy (reactiveGpuHem.h:37); both are
// strings reactiveThermo.cpp:294-301 accepts.
const char* reactive_gpu_hem_numerical_policy_v1(void) {
    return defaultArithmetic() == REACTIVE_AMD_FLASH_MIXED ? "fp32-cubic-newton-fp64-accept-v2:experimental" : "";
}

int reactive_amd_hem_set_arithmetic(void* raw, int mode) {
    if (!raw) return -1;
    if (mode != REACTIVE_AMD_FLASH_FP64 && mode != REACTIVE_AMD_FLASH_MIXED) return 1;
    static_cast<HemHandle*>(raw)->arithmetic = mode;
    return 0;
}

int reactive_amd_hem_mixed_report(void* raw, uint64_t* singlePhaseEvaluations, uint64_t* queuedCells) {
    if (!raw) return -1;
    if (!singlePhaseEvaluations || !queuedCells) return 1;
    const HemHandle* h = static_cast<const HemHandle*>(raw);
    *singlePhaseEvaluations = h->lastSinglePhases;
    *queuedCells = h->lastQueued;
    return 0;
}

void* reactive_gpu_hem_create_v1(const void* model, size_t bytes, size_t capacity, char* error, size_t size) {
    try {
        return createHem(model, bytes, capacity, true);
    } catch (const std::exception& e) {
        writeError(error, size, e.what());
        return nullptr;
    }
}

void* reactive_gpu_hem_create_resident_v1(const void* model, size_t bytes, size_t capacity, char* error, size_t size) {
    try {
        return createHem(model, bytes, capacity, false);
    } catch (const std::exception& e) {
        writeError(error, size, e.what());
        return nullptr;
    }
}

size_t reactive_gpu_hem_device_bytes_v1(void* raw) { return raw ? static_cast<HemHandle*>(raw)->deviceBytes : 0; }

void reactive_gpu_hem_destroy_v1(void* raw) { delete static_cast<HemHandle*>(raw); }

int reactive_gpu_hem_run_v1(void* raw, const double* q, const double* energy, size_t count, ReactiveThermoState* states,
                            int* success, ReactiveGpuHemProfileV1* profile, char* error, size_t size) {
    try {
        return runHost(static_cast<HemHandle*>(raw), q, energy, nullptr, count, states, success, profile);
    } catch (const std::exception& e) {
        writeError(error, size, e.what());
        return 1;
    }
}

int reactive_gpu_hem_run_v2(void* raw, const double* q, const double* energy,
                            const ReactiveGpuHemCapillaryInputV2* capillary, size_t count, ReactiveThermoState* states,
                            int* success, ReactiveGpuHemProfileV1* profile, char* error, size_t size) {
    if (!capillary) {
        writeError(error, size, "Null HIP HEM capillary input");
        return 1;
    }
    try {
        return runHost(static_cast<HemHandle*>(raw), q, energy, capillary, count, states, success, profile);
    } catch (const std::exception& e) {
        writeError(error, size, e.what());
        return 1;
    }
}

int reactive_gpu_hem_initialize_tp_v1(void*, double*, double*, const ReactiveGpuHemCapillaryInputV2*, size_t,
                                      ReactiveThermoState*, int*, ReactiveGpuHemProfileV1*, char* error, size_t size) {
    writeError(error, size, "reactive_gpu_hem_initialize_tp_v1: capillary primitive initialisation is not provided "
                            "by the MI355X HEM build");
    return 1;
}

int reactive_gpu_hem_run_resident_v1(void* raw, const double* q, const double* energy, const ReactiveThermoState* seed,
                                     const ReactiveGpuHemCapillaryInputV2* capillary, const uint32_t* order,
                                     size_t count, ReactiveGpuHemOutputV1* output, ReactiveGpuHemProfileV1* profile,
                                     char* error, size_t size) {
    try {
        require(raw && q && energy && seed && capillary && order && output && profile && profile->abiVersion == 1 &&
                    profile->structBytes == sizeof(*profile),
                "Invalid resident HIP HEM batch arguments");
        HemHandle* h = static_cast<HemHandle*>(raw);
        require(count && count <= h->capacity, "Resident HIP HEM batch exceeds capacity");
        const auto begin = std::chrono::steady_clock::now();
        RAMD_HIP(hipSetDevice(h->device));
        hipStream_t s = h->stream;
        // every input is device memory indexed by global cell; as in the
        // reference (reactiveGpuHem.cuh:360-380), a cell whose interface input
        // recoverCapillary rejects fails on its own
        const auto* cap = reinterpret_cast<const HemCapillaryDev*>(capillary);
        RAMD_HIP(hipEventRecord(h->events[0], s));
        h->launch(q, energy, reinterpret_cast<const ThermoOut*>(seed), order, count, cap,
                  reinterpret_cast<HemOutputDev*>(output), s);
        RAMD_HIP(hipEventRecord(h->events[1], s));
        unsigned long long totals[8] = {};
        RAMD_HIP(hipMemcpyAsync(totals, h->totals, sizeof(totals), hipMemcpyDeviceToHost, s));
        RAMD_HIP(hipEventRecord(h->events[2], s));
        RAMD_HIP(hipEventSynchronize(h->events[2]));
        float kernel = 0, download = 0;
        RAMD_HIP(hipEventElapsedTime(&kernel, h->events[0], h->events[1]));
        RAMD_HIP(hipEventElapsedTime(&download, h->events[1], h->events[2]));
        ReactiveGpuHemProfileV1 p{};
        p.abiVersion = 1;
        p.structBytes = sizeof(p);
        p.batches = 1;
        p.submitted = count;
        p.succeeded = totals[6];
        p.deviceFailures = count - totals[6];
        p.phaseEvaluations = totals[0];
        p.residualEvaluations = totals[1];
        p.flashCandidates = totals[2];
        p.stableCandidates = totals[3];
        p.finiteDifferenceJacobians = totals[5];
        p.analyticJacobians = totals[7];
        p.transferBytes = sizeof(totals);
        p.deviceBytes = h->deviceBytes;
        p.wallSeconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - begin).count();
        p.kernelSeconds = kernel / 1000.;
        p.copySeconds = download / 1000.;
        *profile = p;
        return 0;
    } catch (const std::exception& e) {
        writeError(error, size, e.what());
        return 1;
    }
}

// Same contract and results as reactive_gpu_hem_run_resident_v1, without any
// device allocation: the work counters go to the library's static scratch.
int reactive_gpu_hem_run_resident_noalloc_v1(void* raw, const double* q, const double* energy,
                                             const ReactiveThermoState* seed,
                                             const ReactiveGpuHemCapillaryInputV2* capillary, const uint32_t* order,
                                             size_t count, ReactiveGpuHemOutputV1* output,
                                             ReactiveGpuHemProfileV1* profile, char* error, size_t size) {
    try {
        require(raw && q && energy && seed && capillary && order && output && profile && profile->abiVersion == 1 &&
                    profile->structBytes == sizeof(*profile),
                "Invalid resident HIP HEM batch arguments");
        HemHandle* h = static_cast<HemHandle*>(raw);
        require(count && count <= h->capacity, "Resident HIP HEM batch exceeds capacity");
        require(count <= kNoAllocMaxCells, "reactive_gpu_hem_run_resident_noalloc_v1: a batch holds at most "
                                           "1048576 cells (the size of its static device scratch)");
        const auto begin = std::chrono::steady_clock::now();
        RAMD_HIP(hipSetDevice(h->device));
        unsigned long long* partials = scratchAddress(h->device);
        unsigned long long* totalsDev = partials + size_t(kNoAllocBlocks) * 8;
        hipStream_t s = h->stream;
        const auto* cap = reinterpret_cast<const HemCapillaryDev*>(capillary);
        RAMD_HIP(hipEventRecord(h->events[0], s));
        const unsigned blocks = h->launch(q, energy, reinterpret_cast<const ThermoOut*>(seed), order, count, cap,
                                          reinterpret_cast<HemOutputDev*>(output), s, partials, kNoAllocBlocks);
        hipLaunchKernelGGL(reducePartialsKernel, dim3(1), dim3(64), 0, s, partials, blocks, 8, totalsDev);
        RAMD_HIP(hipGetLastError());
        RAMD_HIP(hipEventRecord(h->events[1], s));
        unsigned long long totals[8] = {};
        RAMD_HIP(hipMemcpyAsync(totals, totalsDev, sizeof(totals), hipMemcpyDeviceToHost, s));
        RAMD_HIP(hipEventRecord(h->events[2], s));
        RAMD_HIP(hipEventSynchronize(h->events[2]));
        float kernel = 0, download = 0;
        RAMD_HIP(hipEventElapsedTime(&kernel, h->events[0], h->events[1]));
        RAMD_HIP(hipEventElapsedTime(&download, h->events[1], h->events[2]));
        ReactiveGpuHemProfileV1 p{};
        p.abiVersion = 1;
        p.structBytes = sizeof(p);
        p.batches = 1;
        p.submitted = count;
        p.succeeded = totals[6];
        p.deviceFailures = count - totals[6];
        p.phaseEvaluations = totals[0];
        p.residualEvaluations = totals[1];
        p.flashCandidates = totals[2];
        p.stableCandidates = totals[3];
        p.finiteDifferenceJacobians = totals[5];
        p.analyticJacobians = totals[7];
        p.transferBytes = sizeof(totals);
        p.deviceBytes = h->deviceBytes;
        p.wallSeconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - begin).count();
        p.kernelSeconds = kernel / 1000.;
        p.copySeconds = download / 1000.;
        *profile = p;
        return 0;
    } catch (const std::exception& e) {
        writeError(error, size, e.what());
        return 1;
    }
}

}
