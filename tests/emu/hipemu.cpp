// Test infrastructure only: runtime of the CPU emulation build (see hipemu.hpp).
#include "hipemu.hpp"

#include <dlfcn.h>
#include <condition_variable>
#include <map>
#include <memory>
#include <mutex>
#include <semaphore>
#include <span>
#include <string>
#include <thread>
#include <vector>

thread_local dim3 threadIdx, blockIdx;
dim3 blockDim, gridDim;

namespace {

enum State { Runnable, AtColl, AtSync, Done };
enum Kind { KBallot, KShfl, KSync, KSyncOr };

struct Lane {
    std::binary_semaphore go{0};
    State st = Runnable;
    Kind kind = KBallot;
    void* site = nullptr;
    long long arg = 0;
    int src = 0;
    long long result = 0;
    unsigned tid = 0;
};

// The lanes of the running block. Their threads are kept from block to block (blocks run
// one at a time) and end with the process.
struct Block {
    std::vector<std::unique_ptr<Lane>> lanes;
    std::binary_semaphore back{0};
    const std::function<void()>* fn = nullptr;
    unsigned bx = 0;
    int nLanes = 0;
};
Block& block() {
    static Block* b = new Block();   // never destroyed: the threads wait in it
    return *b;
}

thread_local Lane* gLane = nullptr;
thread_local unsigned gYields = 0;   // preemption points passed in this block

void yieldLane(Lane& L) {
    block().back.release();
    L.go.acquire();
}

void laneThread(Lane* L) {
    Block& B = block();
    gLane = L;
    while (true) {
        L->go.acquire();
        threadIdx = dim3(L->tid, 0, 0);
        blockIdx = dim3(B.bx, 0, 0);
        gYields = 0;
        (*B.fn)();
        L->st = Done;
        B.back.release();
    }
}

void runBlock(const std::function<void()>& fn, unsigned bx, unsigned nthreads) {
    Block& B = block();
    B.nLanes = (int)nthreads;
    B.fn = &fn;
    B.bx = bx;
    while (B.lanes.size() < nthreads) {
        B.lanes.emplace_back(new Lane());
        B.lanes.back()->tid = (unsigned)B.lanes.size() - 1;
        std::thread(laneThread, B.lanes.back().get()).detach();
    }
    const std::span<std::unique_ptr<Lane>> lanes(B.lanes.data(), nthreads);
    for (auto& lp : lanes) lp->st = Runnable;
    while (true) {
        // run every runnable lane until it blocks or finishes
        bool any = false;
        for (auto& lp : lanes) {
            Lane& L = *lp;
            if (L.st == Runnable) {
                any = true;
                L.go.release();
                B.back.acquire();
            }
        }
        (void)any;
        bool preempted = false;
        for (auto& lp : lanes) preempted = preempted || lp->st == Runnable;
        if (preempted) continue;
        // resolve collectives per wave per site
        bool progress = false;
        const int nw = (B.nLanes + 63) / 64;
        for (int w = 0; w < nw; ++w) {
            std::map<void*, std::vector<Lane*>> groups;
            for (int l = w * 64; l < std::min(B.nLanes, w * 64 + 64); ++l) {
                Lane& L = *lanes[l];
                if (L.st == AtColl) groups[L.site].push_back(&L);
            }
            for (auto& kv : groups) {
                auto& g = kv.second;
                const Kind k = g[0]->kind;
                for (Lane* L : g)
                    if (L->kind != k) { fprintf(stderr, "EMU: mixed collectives at one site\n"); abort(); }
                if (k == KBallot) {
                    unsigned long long m = 0;
                    for (Lane* L : g) if (L->arg) m |= 1ull << (L->tid & 63);
                    for (Lane* L : g) { L->result = (long long)m; L->st = Runnable; }
                } else {
                    std::map<unsigned, long long> val;
                    for (Lane* L : g) val[L->tid & 63] = L->arg;
                    for (Lane* L : g) {
                        unsigned src = L->src >= 0 ? (unsigned)L->src : ((L->tid & 63) ^ (unsigned)(-1 - L->src));
                        src &= 63;
                        auto it = val.find(src);
                        if (it == val.end()) {
                            fprintf(stderr, "EMU: shfl from inactive lane %u (block %u)\n", src, blockIdx.x);
                            abort();
                        }
                        L->result = it->second;
                    }
                    for (Lane* L : g) L->st = Runnable;
                }
                progress = true;
            }
        }
        if (progress) continue;
        int done = 0, sync = 0;
        for (auto& lp : lanes) {
            if (lp->st == Done) ++done;
            else if (lp->st == AtSync) ++sync;
        }
        if (done == B.nLanes) break;
        if (sync + done == B.nLanes && sync > 0) {
            if (done) { fprintf(stderr, "EMU: barrier with %d exited lanes\n", done); abort(); }
            void* site = nullptr;
            long long orv = 0;
            for (auto& lp : lanes) {
                if (lp->st != AtSync) continue;
                if (!site) site = lp->site;
                orv |= lp->arg;
            }
            for (auto& lp : lanes)
                if (lp->st == AtSync) { lp->result = orv != 0; lp->st = Runnable; }
            continue;
        }
        fprintf(stderr, "EMU: deadlock (done %d, at barrier %d)\n", done, sync);
        abort();
    }
}

struct Rec {
    std::string name;
    std::function<void()> fn;
    dim3 g, b;
};

// one launch at a time, whichever thread makes it (blockDim, shared memory)
std::mutex gRun;
// streams, events, counts
std::mutex gState;
std::map<std::string, long long> gLaunches;
long long gStreamSyncs = 0, gEventRecords = 0;
void (*gOnGraph)() = nullptr;

bool async() {
    static const bool on = getenv("EMU_ASYNC") && atoi(getenv("EMU_ASYNC")) != 0;
    return on;
}

}  // namespace

struct EmuStream {
    bool capturing = false, invalid = false;
    std::vector<Rec> captured;
    unsigned long long enqueued = 0, done = 0;   // pieces of work given and waited for
};
struct EmuEvent {
    EmuStream* s = nullptr;
    unsigned long long at = 0;
};
struct EmuGraph {
    std::vector<Rec> recs;
    EmuStream* s = nullptr;   // last launch
    unsigned long long at = 0;
};

static EmuStream gNullStream;
static EmuStream* streamOf(hipStream_t s) { return s ? s : &gNullStream; }
static EmuStream* gCapturing = nullptr;   // the stream under capture, if any

// A synchronous call: ends a capture in an error, whichever stream is captured.
static void synchronous() {
    std::lock_guard<std::mutex> lock(gState);
    if (gCapturing) gCapturing->invalid = true;
}

unsigned long long emu_ballot(int pred, void* site) {
    Lane& L = *gLane;
    L.kind = KBallot; L.arg = pred ? 1 : 0; L.site = site; L.st = AtColl;
    yieldLane(L);
    return (unsigned long long)L.result;
}
int emu_shfl_i(int v, int src, void* site) {
    Lane& L = *gLane;
    L.kind = KShfl; L.arg = v; L.src = src; L.site = site; L.st = AtColl;
    yieldLane(L);
    return (int)L.result;
}
unsigned emu_lane() { return gLane->tid & 63; }
// With EMU_PREEMPT=k, a lane gives up the baton at every k-th preemption point, so the
// lanes of a block interleave inside loops that have no collectives (as waves do).
void emu_maybe_yield() {
    static const int every = getenv("EMU_PREEMPT") ? atoi(getenv("EMU_PREEMPT")) : 0;
    if (!every || !gLane) return;
    if (++gYields % (unsigned)every) return;
    Lane& L = *gLane;
    L.st = Runnable;
    yieldLane(L);
}
void emu_sync(void* site) {
    Lane& L = *gLane;
    L.kind = KSync; L.arg = 0; L.site = site; L.st = AtSync;
    yieldLane(L);
}
int emu_sync_or(int pred, void* site) {
    Lane& L = *gLane;
    L.kind = KSyncOr; L.arg = pred ? 1 : 0; L.site = site; L.st = AtSync;
    yieldLane(L);
    return (int)L.result;
}

static void runRec(const Rec& r) {
    std::lock_guard<std::mutex> run(gRun);
    {
        std::lock_guard<std::mutex> lock(gState);
        ++gLaunches[r.name];
    }
    gridDim = r.g;
    blockDim = r.b;
    for (unsigned bx = 0; bx < r.g.x; ++bx) runBlock(r.fn, bx, r.b.x);
}

// The kernel's symbol where it has one (launchers pass kernels on under other names).
static std::string kernelName(const char* given, void* kernel) {
    Dl_info info;
    return dladdr(kernel, &info) && info.dli_sname && info.dli_saddr == kernel ? info.dli_sname : given;
}

void emu_launch(const char* given, void* kernel, std::function<void()> fn, dim3 g, dim3 b, hipStream_t st) {
    EmuStream* s = streamOf(st);
    const std::string name = kernelName(given, kernel);
    {
        std::lock_guard<std::mutex> lock(gState);
        if (s->capturing) {
            s->captured.push_back({name, fn, g, b});
            return;
        }
        ++s->enqueued;
    }
    runRec({name, fn, g, b});
}

// Work on a stream that cannot be recorded here (the library captures kernels only).
static hipError_t enqueueOther(hipStream_t st) {
    EmuStream* s = streamOf(st);
    std::lock_guard<std::mutex> lock(gState);
    if (s->capturing) {
        s->invalid = true;
        return hipErrorStreamCaptureUnsupported;
    }
    ++s->enqueued;
    return hipSuccess;
}

void emu_on_graph(void (*cb)()) { gOnGraph = cb; }
long long emu_launches(const char* part) {
    std::lock_guard<std::mutex> lock(gState);
    long long n = 0;
    for (auto& kv : gLaunches)
        if (kv.first.find(part) != std::string::npos) n += kv.second;
    return n;
}
long long emu_stream_syncs() {
    std::lock_guard<std::mutex> lock(gState);
    return gStreamSyncs;
}
long long emu_event_records() {
    std::lock_guard<std::mutex> lock(gState);
    return gEventRecords;
}

static int gEmuCus() {
    const char* e = getenv("EMU_CUS");
    return e ? atoi(e) : 2;
}
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* symbol) { *p = const_cast<void*>(symbol); return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->name, "CPU emulator");
    std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    p->multiProcessorCount = gEmuCus();
    p->sharedMemPerBlock = 160 * 1024;
    p->warpSize = 64;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = size_t(8) << 30; *t = size_t(16) << 30; return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : "emulated error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipPeekAtLastError() { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
// fresh device memory holds garbage on the GPU: fill it so reads of unwritten words
// show up (EMU_FILL, default 0xA5)
hipError_t hipMalloc(void** p, size_t n) {
    *p = malloc(n ? n : 1);
    if (!*p) return hipErrorOutOfMemory;
    const char* f = getenv("EMU_FILL");
    std::memset(*p, f ? atoi(f) : 0xA5, n);
    return hipSuccess;
}
static long long gAsyncAllowed = -1;
void emu_fail_async_allocations(long long allowed) { gAsyncAllowed = allowed; }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) {
    if (gAsyncAllowed == 0) return hipErrorOutOfMemory;
    if (gAsyncAllowed > 0) --gAsyncAllowed;
    return hipMalloc(p, n);
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipFreeAsync(void* p, hipStream_t) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
static hipError_t copyNow(void* d, const void* s, size_t n) { if (n) std::memmove(d, s, n); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { synchronous(); return copyNow(d, s, n); }
hipError_t hipMemcpy2D(void* d, size_t dpitch, const void* s, size_t spitch, size_t width, size_t height,
                       hipMemcpyKind) {
    if (width > dpitch || width > spitch) return hipErrorInvalidValue;
    for (size_t r = 0; r < height; ++r)
        std::memmove((char*)d + r * dpitch, (const char*)s + r * spitch, width);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    const hipError_t e = enqueueOther(st);
    return e != hipSuccess ? e : copyNow(d, s, n);
}
hipError_t hipMemset(void* d, int v, size_t n) { synchronous(); std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
    const hipError_t e = enqueueOther(st);
    if (e == hipSuccess) std::memset(d, v, n);
    return e;
}
hipError_t hipStreamCreate(hipStream_t* s) { *s = new EmuStream(); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s) { delete s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t st) {
    EmuStream* s = streamOf(st);
    std::lock_guard<std::mutex> lock(gState);
    ++gStreamSyncs;
    if (s->capturing) {
        s->invalid = true;
        return hipErrorStreamCaptureUnsupported;
    }
    s->done = s->enqueued;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = new EmuEvent(); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
    const hipError_t r = enqueueOther(st);
    if (r != hipSuccess) return r;
    std::lock_guard<std::mutex> lock(gState);
    ++gEventRecords;
    e->s = streamOf(st);
    e->at = e->s->enqueued;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    std::lock_guard<std::mutex> lock(gState);
    if (e->s && e->s->done < e->at) e->s->done = e->at;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    std::lock_guard<std::mutex> lock(gState);
    return async() && e->s && e->at > e->s->done ? hipErrorNotReady : hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
static void onGraph() {
    if (void (*cb)() = gOnGraph) {
        gOnGraph = nullptr;
        cb();
    }
}
hipError_t hipStreamBeginCapture(hipStream_t st, hipStreamCaptureMode) {
    EmuStream* s = streamOf(st);
    {
        std::lock_guard<std::mutex> lock(gState);
        s->capturing = true;
        s->invalid = false;
        s->captured.clear();
        gCapturing = s;
    }
    onGraph();
    return hipSuccess;
}
hipError_t hipGraphCreate(hipGraph_t* g, unsigned) {
    *g = new EmuGraph();
    onGraph();
    return hipSuccess;
}
hipError_t hipGraphAddKernelNode(hipGraphNode_t* node, hipGraph_t g, const hipGraphNode_t* deps, size_t n,
                                 const hipKernelNodeParams* p) {
    // nodes are numbered from 1 in the order of addition
    const size_t last = g->recs.size();
    if ((last == 0) != (n == 0) || n > 1 || (n == 1 && (size_t)deps[0] != last)) return hipErrorInvalidValue;
    g->recs.push_back({kernelName("node", p->func.at), p->func.bind(p->kernelParams), p->gridDim, p->blockDim});
    *node = (hipGraphNode_t)(last + 1);
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t st, hipGraph_t* g) {
    EmuStream* s = streamOf(st);
    std::lock_guard<std::mutex> lock(gState);
    s->capturing = false;
    gCapturing = nullptr;
    if (s->invalid) { *g = nullptr; return hipErrorStreamCaptureInvalidated; }
    *g = new EmuGraph{s->captured};
    s->captured.clear();
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
    *e = new EmuGraph{g->recs};
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t st) {
    const hipError_t r = enqueueOther(st);
    if (r != hipSuccess) return r;
    e->s = streamOf(st);
    e->at = e->s->enqueued;
    for (auto& rec : e->recs) runRec(rec);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    if (async() && e->s && e->at > e->s->done) {
        fprintf(stderr, "EMU: graph destroyed while it runs\n");
        abort();
    }
    delete e;
    return hipSuccess;
}
