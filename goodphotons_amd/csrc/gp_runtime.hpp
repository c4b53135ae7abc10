// Host runtime internals shared by the C ABI implementation files.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/goodphotons.h"
#include "gp_kernels.hpp"
#include "gp_types.hpp"

namespace gp {

// Pinned host memory through which results leave the device and inputs reach it, in slots
// filled and emptied in turn. A copy between the device and a caller's pageable array goes
// through the runtime's own staging in small pieces, one after the other (1 MB: 430 us,
// 32 MB into fresh pages: 7.8 ms, 14 times the pinned copy); here the device fills a slot
// while the host empties another.
// One ring per process, used by one call at a time and allocated by the first. It and up to
// kKeep of device scratch stay for the process (a program that rebuilds its only scene would
// otherwise allocate 16 MB of pinned memory for every scene: 0.9 ms of a 3.1 ms rebuild);
// larger scratch goes with the last scene or film (StagingUse).
struct Staging {
    static constexpr size_t kSlot = size_t(2) << 20;
    static constexpr int kSlots = 8;
    std::mutex mu;                  // held for a whole transfer
    char* host = nullptr;           // kSlots * kSlot
    hipEvent_t ev[kSlots] = {};     // the device is done with the slot
    std::atomic<int> users{0};
    gp_status ready();              // allocates (mu held)
    // Device scratch of a call that holds mu, grown to `bytes` and kept up to kScratch.
    static constexpr size_t kScratch = size_t(128) << 20;
    char* scratch = nullptr;
    size_t scratchBytes = 0;
    gp_status scratchFor(size_t bytes, char** out);
    static constexpr size_t kKeep = size_t(16) << 20;
    void trim(size_t most);         // drops scratch larger than that
};
Staging& staging();
struct StagingUse {
    StagingUse();
    ~StagingUse();
    StagingUse(const StagingUse&) = delete;
    StagingUse& operator=(const StagingUse&) = delete;
};

}  // namespace gp

struct gp_scene {
    int64_t nTris = 0;
    int64_t nNodes = 0;                // four-wide nodes on the device
    int depth = 0;                     // child-pair levels of the built tree
    int stackNeed = 0;                 // traversal stack entries a ray can need (3 per four-wide level)
    // ray-binning grid over the triangle-centroid box: cell = (x - binLo) * binScale
    float binLo[3] = {0.f, 0.f, 0.f};
    float binScale[3] = {0.f, 0.f, 0.f};
    float4* dNodes = nullptr;
    float4* dTris = nullptr;
    float4* dTrin = nullptr;
    gp::DevMaterial* dMats = nullptr;
    gp::DevEmitter* dEms = nullptr;
    double* dCdfs = nullptr;
    double* dEmCdf = nullptr;
    int32_t* dGuides = nullptr;        // per emitter kCdfGuide + 1 CDF guide entries
    gp::DevMirrorPlane* dMirrors = nullptr;   // flat mirror planes (camera connections through them)
    float* dSpec = nullptr;            // samples of the scene's sampled spectra
    int nMirrors = 0;
    int nEm = 0;
    double totalPower = 0.0;
    double basePower = 0.0;
    int64_t deviceBytes = 0;
    double buildMs = 0.0;
    // host copies for camera-distance bounds (empty when the tree was built on the
    // device: the bound is then computed there and cached per eye position)
    std::vector<float> pairs;          // 16 floats per pair node (host copy of the built tree)
    std::vector<float> leafTris;       // 9 floats per triangle, leaf order
    std::vector<std::array<double, 12>> emitQuads;   // origin, u, v, normal
    int builder = GP_BVH_HOST_SAH;
    mutable std::map<std::array<double, 3>, double> eyeDist2;

    gp::StagingUse staging;

    gp_scene() = default;
    gp_scene(const gp_scene&) = delete;
    gp_scene& operator=(const gp_scene&) = delete;
    ~gp_scene();   // frees the device tables
};

struct gp_film {
    int32_t rx = 0, ry = 0;
    int64_t maxPhotons = 0;
    unsigned long long* d = nullptr;
    double scale = 0.0;                 // contribution -> integer units (0 = not yet fixed)
    unsigned long long qmax = 0;        // largest single splat value
    double splatBudget = 0.0;           // photons*(maxDepth+1) the scale was sized for
    double splatUsed = 0.0;

    gp::StagingUse staging;

    gp_film() = default;
    gp_film(const gp_film&) = delete;
    gp_film& operator=(const gp_film&) = delete;
    ~gp_film();    // frees d (a stream-ordered film clears d after its asynchronous free)
};

namespace gp {

gp_status fail(gp_status s, const std::string& msg);
#define GP_HIP(call)                                                                         \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess)                                                                \
            return ::gp::fail(GP_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

struct DeviceState {
    bool ok = false;
    gp_status status = GP_ERR_NO_DEVICE;
    std::string why;
    int id = 0;
    int cus = 0;
    size_t ldsPerBlock = 0;
    std::string name, arch;
    hipStream_t stream = nullptr;       // engine work
    hipStream_t copyStream = nullptr;   // result downloads that overlap engine work
};
DeviceState& device();
gp_status requireDevice();

// memcpy of results into a caller's array, in pieces: one of megabytes goes past the caches,
// and into fresh pages, which the kernel has just cleared there, that takes half as long again
// (5.5 MB 157 -> 105 us, 34 MB 1.70 -> 1.13 ms).
inline void copyOut(void* dst, const void* src, size_t bytes) {
    constexpr size_t kPiece = size_t(256) << 10;
    for (size_t at = 0; at < bytes; at += kPiece)
        std::memcpy((char*)dst + at, (const char*)src + at, std::min(kPiece, bytes - at));
}

// Moves `items` items of `each` bytes from the device: fill(slot, first, count) enqueues on
// s what writes items [first, first + count) to the pinned slot, drain(slot, first, count)
// takes them on the host. Returns when all are drained. One thread drains: what is left of
// a copy is its page faults in the caller's fresh array, and four threads brought 118 MB of
// frames from 12.6 to 10.9 ms only.
// stagedDownLocked: for a caller that holds g.mu and has called g.ready().
template <class Fill, class Drain>
gp_status stagedDownLocked(Staging& g, size_t items, size_t each, hipStream_t s, Fill&& fill, Drain&& drain) {
    const size_t per = std::max<size_t>(1, Staging::kSlot / each), chunks = (items + per - 1) / per;
    hipError_t e = hipSuccess;
    if (chunks == 1) {   // an event would cost a small copy more than it orders
        e = fill(g.host, 0, items);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e == hipSuccess) drain((const char*)g.host, 0, items);
    }
    for (size_t c = 0, d = 0; chunks > 1 && d < chunks && e == hipSuccess;) {
        const bool down = c == chunks || c - d == Staging::kSlots;
        const size_t chunk = down ? d++ : c++, first = chunk * per, count = std::min(per, items - first);
        const size_t k = chunk % Staging::kSlots;
        char* slot = g.host + k * Staging::kSlot;
        if (down) {
            e = hipEventSynchronize(g.ev[k]);
            if (e == hipSuccess) drain((const char*)slot, first, count);
        } else {
            e = fill(slot, first, count);
            if (e == hipSuccess) e = hipEventRecord(g.ev[k], s);
        }
    }
    if (e != hipSuccess) {
        hipStreamSynchronize(s);   // nothing may still write to the slots
        return fail(GP_ERR_HIP, std::string("staged copy: ") + hipGetErrorString(e));
    }
    return GP_OK;
}
template <class Fill, class Drain>
gp_status stagedDown(size_t items, size_t each, hipStream_t s, Fill&& fill, Drain&& drain) {
    Staging& g = staging();
    std::lock_guard<std::mutex> lock(g.mu);
    const gp_status st = g.ready();
    return st != GP_OK ? st : stagedDownLocked(g, items, each, s, fill, drain);
}
// Plain copy of device memory to a caller's array, after the work on s.
gp_status copyDownLocked(Staging& g, void* dst, const void* src, size_t bytes, hipStream_t s);
gp_status copyDown(void* dst, const void* src, size_t bytes, hipStream_t s);

// Film words -> the doubles of gp_film_download: pixels [0, n) of `film` to xyz (3 n, may be
// null) and hits (n, may be null), word * inv and word.
void launchFilmTotals(const unsigned long long* film, size_t n, double inv, double* xyz, double* hits, hipStream_t s);
// The same on the host.
void wordsToTotals(const long long* words, size_t n, double inv, double* xyz, double* hits);
// Those doubles into a caller's arrays (either may be null), after the work on s. Up to
// kHostTotals pixels the host converts a copy of the words: a kernel that writes to pinned
// memory takes longer than so small a copy (kernel -> host, whole calls: 1024 pixels 16.8 ->
// 13.5 us, 2025 17.9 -> 15.9; 4096 pixels 20.8 by the kernel, 17 for the copy alone).
constexpr size_t kHostTotals = 3072;
gp_status downloadTotals(const gp_film& f, double* xyz, double* hits, hipStream_t s);

// Camera basis as the reference's Camera::lookAt (src/camera.h:110-129), in double.
struct CamBasis {
    double eye[3], u[3], v[3], w[3];
    double tanHalfX, tanHalfY, pixelArea;
    int resX, resY;
};
bool cameraBasis(const gp_camera_desc& c, CamBasis& out);

// Smallest distance from point p to any triangle or emitter quad of the scene.
double sceneMinDistance(const gp_scene& s, const double p[3]);

// Kernel timing slots: schedule, emit, extend, shade, connect (+ mirror), binning.
constexpr int kKernelSlots = 6;

constexpr size_t kCtrlStride = (sizeof(Ctrl) + 255) & ~size_t(255);

// Wavefront engine: device queues, control block, job table, graphs.
struct Engine {
    std::mutex mu;
    gp_tuning tun{};
    bool tunSet = false;
    unsigned capacity = 0;
    unsigned segCap = 0;                // path slots per queue segment
    int spillDepth = 0;
    size_t spillThreads = 0;
    Queues q{};
    LaunchShape ls{};
    Ctrl* dCtrl = nullptr;
    Ctrl* hCtrl = nullptr;              // pinned
    DevJob* dJobs = nullptr;
    unsigned long long* dJobAcc = nullptr;       // kMaxJobs * kSegs * kAccRow, behind dCtrl
    DevCamera* dJobCams = nullptr;               // kMaxJobs * kMaxCams
    int camCap = 1;                              // cameras per job the connection queue is sized for
    // job slot 0's accumulator rows as of the last readCtrl
    const unsigned long long* traceRows() const { return (const unsigned long long*)((const char*)hCtrl + kCtrlStride); }
    void initCtrl();                            // zero the host control block, set capacities
    void* bufs[40] = {};
    int nbufs = 0;
    int parity = 0;
    hipGraphExec_t graph = nullptr;
    int graphIters = 0;
    int graphLds = 0;
    int graphShape = 0;
    int graphBinned = 0;
    int graphEmitOrder = 0;
    // k_mirror runs in each iteration while a job of a scene with flat mirrors is live
    // (set by the caller before runIterations; the graph is re-captured on a change)
    bool mirrorActive = false;
    bool graphMirror = false;
    bool mirrorQueue = false;           // the mirror-vertex queue has been requested once
    // The control block holds one trace or one server's jobs at a time. `owner` is the
    // server whose jobs are in the engine (live or with chunks in flight); `epoch` counts
    // re-initialisations, so a server sees that a trace used the engine since its last
    // step and starts from a fresh control block.
    const void* owner = nullptr;
    uint64_t epoch = 0;
    // per-kernel HIP-event timing (tuning.profile), slots as gp_trace_stats.kernel_ms
    std::vector<std::array<hipEvent_t, 2>> pending[kKernelSlots];
    double kernelMs[kKernelSlots] = {};
    uint64_t kernelLaunches[kKernelSlots] = {};
    void resetProfile();
    gp_status collectProfile();

    // What a call asks of the engine: launch grids, queue and spill sizes, kernel variants, and
    // what of it has to be allocated. same: nothing changes; otherwise ensure() drops the
    // graph and may re-allocate, so no chunk may be in flight.
    struct Shape {
        LaunchShape ls{};
        unsigned segCap = 0;
        int cams = 0;
        size_t threads = 0;             // of the closest-hit kernel (spill rows)
        int connLds = 0, needSpill = 0, useSpill = 0, connUseSpill = 0, binned = 0;
        bool queues = false, mirrorAlloc = false, binAlloc = false, spillAlloc = false, same = false;
    };
    Shape shapeFor(unsigned cap, int lds, int stackNeed, int cams, bool mirrors) const;
    // stackNeed: traversal stack entries the traced scenes can need (gp_scene::stackNeed);
    // mirrors: allocate the mirror-vertex queue (kept from then on, like the camera count)
    gp_status ensure(unsigned cap, int lds, int stackNeed, int cams = 1, bool mirrors = false);
    void release();
    void releaseQueues();
    void releaseSpill();
    template <class F>
    gp_status timed(int k, const Sink& s, F&& launch);
    gp_status enqueueEmit(const LaunchShape& sh, Sink& s);
    gp_status enqueueBounce(const LaunchShape& sh, Sink& s);
    // Runs a trace whose n photons fit the path queue, from k_start_trace (once) to the
    // last path's end; reads the control block and slot 0's rows back. Every live path
    // advances one segment per iteration, so maxDepth iterations end it; the host looks
    // for an earlier end every chunkIterations(). Grids are sized for n, and only the first
    // iteration schedules and emits: with five kernels an iteration on grids for the full
    // queue a 5000-photon render of the box spent 64 us an iteration on empty workgroups.
    gp_status traceOnce(unsigned n, int cams, int maxDepth);
    int onceIterations = 0;
    // Whether a trace of n photons runs as one k_flight launch, and that run. Mirror planes,
    // traversal statistics, kernel timing and ray binning belong to the wavefront's kernels.
    bool flies(uint64_t n, int cams, int stackNeed, int maxDepth) const;
    gp_status fly(unsigned n, int maxDepth);
    gp_status enqueueIterations(int n, Sink& s);    // tracks parity
    gp_status runIterations(int n);           // graph replay when possible
    // Whether new photons of a trace, or of a server's jobs (the largest and all of them), are
    // emitted in sorted order (set by the caller before runIterations). A trace of more photons
    // than the queue holds sorts a part of them in every iteration, and small parts do not pay
    // for that. 2^22 photons, 8 segments deep, index order -> sorted, ms:
    //   queue           2^16           2^18           2^19           2^20           2^21
    //   box             14.6 -> 16.2   5.59 -> 6.14   4.65 -> 4.71   3.64 -> 3.60   3.53 -> 3.39
    //   glass, prism    27.7 -> 29.8   9.72 -> 11.4   7.05 -> 7.42   5.80 -> 5.69   5.22 -> 4.77
    //   soup 100K tri.  59.6 -> 60.9   18.8 -> 19.8   15.0 -> 15.3   12.5 -> 12.6   11.3 -> 11.2
    //   icosphere 1.3M  50.2 -> 51.6   16.3 -> 16.8   10.2 -> 10.5   7.39 -> 7.35   6.26 -> 6.05
    bool wantsEmitOrder(uint64_t photons) const {
        return photons >= kEmitOrderJobMin && capacity >= std::min<uint64_t>(photons, 2 * kEmitOrderJobMin);
    }
    bool wantsEmitOrder(uint64_t largest, uint64_t all) const {
        return all >= kEmitOrderServerMin && wantsEmitOrder(largest);
    }
    void setEmitOrder(bool on) { q.emitOrder = on ? 1 : 0; }
    gp_status readCtrl();                     // synchronous copy of the control block and slot 0's rows
};
Engine& engine();
gp_tuning defaultTuning();
// Iterations between host reads of the control block: iters_per_graph, rounded down
// to even when graphs are replayed (a graph covers both queue parities).
inline int chunkIterations(const gp_tuning& t) {
    return t.use_graph ? std::max(2, t.iters_per_graph & ~1) : std::max(1, t.iters_per_graph);
}
unsigned segmentBound(unsigned cap, unsigned blocks, unsigned threads);
// Whether the wavefront bins its rays: with gp_tuning.ray_sort = 1. Automatic (2) does
// not: with new photons emitted in sorted order and survivors sorted per workgroup, the
// full sort costs more than it gains on every scene measured (whole traces, queue order
// against binned: 8K-triangle glass scene 28.2 vs 31.4 ms, icospheres of 5K / 82K / 1.3M /
// 5.2M 15.1 vs 17.8 / 18.9 vs 21.7 / 13.7 vs 15.4 / 55.2 vs 57.5 ms, soups of 20K / 60K /
// 300K / 1M 4.8 vs 5.4 / 8.3 vs 8.7 / 13.9 vs 14.2 / 13.3 vs 13.8 ms).
bool binningFor(const gp_tuning& t);
// Sums the kSegs accumulator rows of one job: ledger[5] (fixed point) and
// counters[kAccCounters] (the quantities from kAccPhotons on).
void sumAccRows(const unsigned long long* rows, unsigned long long ledger[5], unsigned long long* counters);
// Adds summed counters into a stats record.
void addCounters(const unsigned long long* counters, gp_trace_stats& st);

// Job record for slot `slot` over cameras cams[0..nCams) and their films; the camera
// records (to be placed at J.cams) are written to camsOut.
gp_status fillJob(const gp_scene* s, const gp_camera_desc* cams, gp_film* const* films, int nCams,
                  const gp_trace_params& p, int slot, DevJob& J, DevCamera* camsOut);
// gp_trace_shared; without mayFly a small trace runs the wavefront's kernels too.
gp_status traceShared(gp_scene* s, int nCams, const gp_camera_desc* cams, gp_film* const* films,
                      const gp_trace_params* p, gp_energy* energy, gp_trace_stats* stats, bool mayFly);
gp_status prepareFilm(gp_film* film, const gp_scene* s, const CamBasis& cb,
                      const gp_trace_params& p);

// Flat mirror planes of a scene description: mirror triangles grouped by plane, at
// most kMaxMirrorPlanes (the largest total areas), boxes padded.
void buildMirrorPlanes(const gp_scene_desc* d, std::vector<DevMirrorPlane>& out);

}  // namespace gp
