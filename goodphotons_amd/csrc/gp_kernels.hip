// Wavefront forward light-tracing kernels for CDNA4 (gfx950).
//
// One iteration of the wavefront:
//   k_schedule  (1 block)  refill free queue slots from the jobs' photon budgets (a trace
//                          that fits the queue starts with k_start_trace instead and
//                          emits once)
//   k_emit_keys, k_bin_chunks, k_bin_scan, k_emit_perm  (large traces) sort the new photons
//   k_emit                 emission + hero bundle + direct light->camera connection
//   k_bin_*                (gp_tuning.ray_sort only) counting sort of the paths by
//                          origin cell and direction octant into a third queue
//   k_extend               closest hit for every live path (four-wide nodes, LDS stack)
//   k_shade                material scatter, Russian roulette, camera connection,
//                          survivors placed in the other queue sorted within the workgroup
//   k_connect              any-hit for every connection; unoccluded ones splat into
//                          the int64 fixed-point film with 64-bit atomics
//   k_flight               (small traces, instead of all the others) whole paths in registers
//   k_mirror               (scenes with flat mirrors only) camera connections of the
//                          queued vertices through each mirror plane
// All kernels are fixed-grid and grid-stride over counts that live on the device,
// so an iteration needs no host round trip and can be captured in a hipGraph.
//
// Per path the arithmetic follows the reference's Renderer::tracePhotonHero /
// tracePhotonHeroLoop (src/render.h:2252-2631), connectGeom / connectHero
// (:499-577) and refractOrReflect (:2657-2694), in float32.
#include <hip/hip_runtime.h>

#include <tuple>

#include "gp_device.hpp"
#include "gp_kernels.hpp"

namespace gp {

namespace {

constexpr float kInvPi = 0.318309886183791f;

__device__ __forceinline__ unsigned long long toFixed(double v, double scale) {
    double q = v * scale;
    return q > 0.0 ? (unsigned long long)__double2ll_rn(q) : 0ull;
}

__device__ __forceinline__ unsigned long long shflXor64(unsigned long long v, int m) {
    unsigned lo = (unsigned)v, hi = (unsigned)(v >> 32);
    lo = __shfl_xor(lo, m);
    hi = __shfl_xor(hi, m);
    return ((unsigned long long)hi << 32) | lo;
}

// Per-job sums (ledger terms, counters) without contended global atomics: each lane
// keeps a register sum for the job it is currently on; when its job changes the sum
// goes into a per-workgroup LDS table (one row per job slot), and the table is added
// to global memory once per workgroup. A queue holding one job never touches the
// table until the end; a mixed queue pays LDS atomics, not global ones.
template <int K>
struct JobAcc {
    int job = -1;
    unsigned long long v[K] = {};
};

template <int K>
__device__ __forceinline__ void initJobTable(unsigned long long* tab, int nJobs) {
    for (int r = threadIdx.x; r < nJobs * K; r += blockDim.x) tab[r] = 0ull;
    __syncthreads();
}

template <int K>
__device__ __forceinline__ void spill(JobAcc<K>& a, unsigned long long* tab) {
    if (a.job >= 0)
        for (int k = 0; k < K; ++k)
            if (a.v[k]) atomicAdd(&tab[a.job * K + k], a.v[k]);
    for (int k = 0; k < K; ++k) a.v[k] = 0;
}

template <int K>
__device__ __forceinline__ void accumulate(JobAcc<K>& a, int job, unsigned long long* tab) {
    if (a.job != job) {
        spill(a, tab);
        a.job = job;
    }
}

// Called by every thread of the workgroup (converged).
template <int K, class Addr>
__device__ __forceinline__ void flushJobTable(JobAcc<K>& a, unsigned long long* tab, int nJobs, Addr addr) {
    spill(a, tab);
    __syncthreads();
    for (int r = threadIdx.x; r < nJobs * K; r += blockDim.x) {
        const unsigned long long v = tab[r];
        if (v) atomicAdd(addr(r / K, r % K), v);
    }
}

// Ledger and counter sums go to the job's row (blockIdx.x % kSegs): eight rows on
// eight cache lines, so the per-workgroup flushes of a launch spread over eight
// addresses instead of serialising on one.
struct AccAddr {
    const DevJob* jobs;
    int base;   // first index of this kernel's quantities in the row
    __device__ unsigned long long* operator()(int j, int k) const {
        return jobs[j].acc + (size_t)(blockIdx.x % kSegs) * kAccRow + base + k;
    }
};

// Logical index -> slot of a segmented queue. `pre` is the prefix of the segment
// counts (wave-uniform); the segment is the last one whose prefix is <= i, which
// skips empty segments.
struct SegMap {
    unsigned pre[kSegs];
    unsigned cap;
    __device__ __forceinline__ unsigned slot(unsigned i) const {
        unsigned base = 0, off = i;
#pragma unroll
        for (int g = 1; g < kSegs; ++g)
            if (i >= pre[g]) { base = (unsigned)g * cap; off = i - pre[g]; }
        return base + off;
    }
    // The same slot through a per-workgroup LDS table tab[g] = g * cap - pre[g]
    // (initSegTab): the segment is counted with compares against the wave-uniform
    // prefixes and the one per-lane lookup is an LDS read, so no uniform value has to
    // be copied into vector registers (slot's selects need them there).
    __device__ __forceinline__ unsigned slotTab(unsigned i, const unsigned* tab) const {
        unsigned g = 0;
#pragma unroll
        for (int k = 1; k < kSegs; ++k) g += (i >= pre[k]) ? 1u : 0u;
        return i + tab[g];
    }
};

// Fills the LDS table of SegMap::slotTab; the caller synchronises the workgroup before
// the first lookup.
__device__ __forceinline__ void initSegTab(const SegMap& m, unsigned* tab) {
#pragma unroll
    for (int g = 0; g < kSegs; ++g)
        if (threadIdx.x == (unsigned)g) tab[g] = (unsigned)g * m.cap - m.pre[g];
}

__device__ __forceinline__ unsigned loadSegMap(const unsigned (*cnt)[kLine], unsigned cap, SegMap& m) {
    unsigned acc = 0;
#pragma unroll
    for (int g = 0; g < kSegs; ++g) {
        m.pre[g] = acc;
        // a segment that overflowed (the trace then fails with GP_ERR_CAPACITY) still
        // maps only its own slots
        acc += min(cnt[g][0], cap);
    }
    m.cap = cap;
    return acc;
}

// Append to this workgroup's segment (blockIdx.x % kSegs) of a segmented queue;
// returns the slot, or ~0u (and raises the overflow flag) if the segment is full.
__device__ __forceinline__ unsigned segAppend(unsigned (*cnt)[kLine], unsigned cap, bool pred,
                                              unsigned* overflow) {
    const unsigned g = blockIdx.x % kSegs;
    const unsigned off = waveAppend(&cnt[g][0], pred);
    if (pred && off >= cap) {
        *overflow = 1u;
        return ~0u;
    }
    return g * cap + off;
}

// Workgroups are dispatched to the eight XCDs round-robin (workgroup b to XCD b % 8),
// and each XCD has its own L2. Renumbering b as (b % 8) * (G / 8) + b / 8 gives every
// XCD a contiguous eighth of each grid-stride round (and adjacent numbers to the
// workgroups of one XCD). Identity when the grid G is not a multiple of 8.
constexpr unsigned kXcds = 8;
__device__ __forceinline__ unsigned xcdBlock() {
    const unsigned G = gridDim.x, b = blockIdx.x;
    return (G % kXcds) ? b : (b % kXcds) * (G / kXcds) + b / kXcds;
}

// Ray-binning key of a ray: the Morton code of its origin's cell in the job's
// kBinCellsPerAxis^3 grid over the triangle-centroid box, then its direction octant.
__device__ __forceinline__ unsigned spread3(unsigned v) {
    return (v & 1u) | ((v & 2u) << 2) | ((v & 4u) << 4);
}

__device__ __forceinline__ unsigned binCell(float x, float lo, float scale) {
    // fmaxf returns 0 for a NaN cell coordinate
    const float f = fminf(fmaxf((x - lo) * scale, 0.0f), (float)(kBinCellsPerAxis - 1));
    return (unsigned)f;
}

__device__ __forceinline__ unsigned short binKey(const DevJob& J, F3 o, F3 d) {
    const unsigned m = spread3(binCell(o.x, J.binLo[0], J.binScale[0])) |
                       (spread3(binCell(o.y, J.binLo[1], J.binScale[1])) << 1) |
                       (spread3(binCell(o.z, J.binLo[2], J.binScale[2])) << 2);
    const unsigned oct = (d.x < 0.0f ? 1u : 0u) | (d.y < 0.0f ? 2u : 0u) | (d.z < 0.0f ? 4u : 0u);
    return (unsigned short)((m << 3) | oct);
}

// Camera connection of a diffuse (or emitter) vertex at p with shading normal n (flat
// triangles: n is also the oriented geometric normal, so the reference's terminator
// factor and adjoint correction are exactly 1).
struct ConnGeom {
    F3 wdir;
    float dist, cosSurf, denom;
    int pix;
};

// The connection's geometry; whether p lies in the camera's view and the camera in front
// of the surface.
__device__ __forceinline__ bool connectGeom(const DevCamera& K, F3 p, F3 n, ConnGeom& g) {
    const F3 eye = load3(K.eye);
    F3 toCam = eye - p;
    g.dist = sqrtf(dot(toCam, toCam));
    g.wdir = toCam * (1.0f / g.dist);
    g.cosSurf = dot(n, g.wdir);
    F3 dd = p - eye;
    float cz = dot(dd, load3(K.w));
    float ix = (dot(dd, load3(K.u)) / cz) / K.tanHalfX;
    float iy = (dot(dd, load3(K.v)) / cz) / K.tanHalfY;
    int px = (int)((ix * 0.5f + 0.5f) * (float)K.resX);
    int py = (int)((iy * 0.5f + 0.5f) * (float)K.resY);
    px = min(max(px, 0), K.resX - 1);
    py = min(max(py, 0), K.resY - 1);
    float dist2 = dot(dd, dd);
    float cosCam = cz / sqrtf(dist2);
    g.denom = dist2 * (K.pixelArea * cosCam * cosCam * cosCam);
    g.pix = py * K.resX + px;
    return g.cosSurf > 0.0f && cz > 1e-9f && ix >= -1.0f && ix < 1.0f && iy >= -1.0f && iy < 1.0f;
}

__device__ __forceinline__ void connectRecord(const ConnGeom& g, unsigned tagJobCam, F3 p, F3 n, const float* lam,
                                              const float* beta, const float* rho, int nUp, float4& co, float4& cd,
                                              float4& cx) {
    float X = 0.f, Y = 0.f, Z = 0.f;
    for (int i = 0; i < nUp; ++i) {
        float c = beta[i] * (rho[i] * kInvPi) * g.cosSurf / g.denom;
        F3 w = cie(lam[i]);
        X += w.x * c;
        Y += w.y * c;
        Z += w.z * c;
    }
    F3 org = p + n * kRayEps;
    co = make_float4(org.x, org.y, org.z, (g.dist - 2.0f * kRayEps) - kRayEps);
    cd = make_float4(g.wdir.x, g.wdir.y, g.wdir.z, __int_as_float(g.pix));
    cx = make_float4(X, Y, Z, __int_as_float(tagJobCam | ((unsigned)nUp << 16)));
}

__device__ __forceinline__ bool makeConnection(const DevCamera& K, unsigned tagJobCam, F3 p, F3 n,
                                               const float* lam, const float* beta, const float* rho,
                                               int nUp, float4& co, float4& cd, float4& cx) {
    ConnGeom g;
    if (!connectGeom(K, p, n, g)) return false;
    connectRecord(g, tagJobCam, p, n, lam, beta, rho, nUp, co, cd, cx);
    return true;
}

// Connections are appended in two steps, so that one atomic reserves room for all cameras of
// a wave (k_emit) or workgroup (k_shade): same-address atomics take 12 ns each, and a wave's
// append for every camera held up both. Six cameras: k_shade 1915 -> 1452 us, k_emit 646 ->
// 408 us; one camera: k_shade 13.3 -> 12.9 ms on the glass scene, 1137 -> 1087 us on the box.
// First the cameras the vertex connects to (bit k: camera k; lanes without a vertex pass
// nCams = 0); called by all lanes of the wave.
__device__ __forceinline__ unsigned connectMask(const DevCamera* cams, int nCams, F3 p, F3 n) {
    unsigned mask = 0;
    for (int k = 0; __any(k < nCams); ++k) {
        ConnGeom g;
        if (k < nCams && connectGeom(cams[k], p, n, g)) mask |= 1u << k;
    }
    return mask;
}

// The wave's connections.
__device__ __forceinline__ unsigned connectCount(unsigned mask) {
    unsigned total = 0;
    for (int k = 0; __any((mask >> k) != 0u); ++k) total += (unsigned)__popcll(__ballot((mask >> k) & 1u));
    return total;
}

// Then their records, from `off` of the workgroup's segment on.
__device__ __forceinline__ void connectWrite(const Queues& q, Ctrl* c, const DevCamera* cams, unsigned mask,
                                             unsigned off, unsigned job, F3 p, F3 n, const float* lam,
                                             const float* beta, const float* rho, int nUp) {
    const unsigned seg = blockIdx.x % kSegs;
    for (int k = 0; __any((mask >> k) != 0u); ++k) {
        const bool conn = (mask >> k) & 1u;
        const unsigned long long lanes = __ballot(conn);
        const unsigned at = off + __builtin_amdgcn_mbcnt_hi((unsigned)(lanes >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((unsigned)lanes, 0u));
        off += (unsigned)__popcll(lanes);
        if (!conn) continue;
        if (at >= q.connSegCap) {
            c->overflow = 1u;
            continue;
        }
        ConnGeom g;
        (void)connectGeom(cams[k], p, n, g);
        float4 co, cd, cx;
        connectRecord(g, connTag(job, 0u, (unsigned)k), p, n, lam, beta, rho, nUp, co, cd, cx);
        const unsigned ci = seg * q.connSegCap + at;
        q.co[ci] = co;
        q.cd[ci] = cd;
        q.cx[ci] = cx;
    }
}

// A vertex to connect to its job's cameras through the scene's flat mirrors, queued
// for k_mirror (weights w: the albedo at a surface vertex, 1 at the emitter). Called
// by all active lanes of the wave.
__device__ __forceinline__ void queueMirrorVertex(const Queues& q, Ctrl* c, bool pred, unsigned job, F3 p,
                                                  F3 n, const float* lam, const float* beta,
                                                  const float* w, int nUp) {
    if (!__any(pred)) return;
    const unsigned mi = segAppend(c->mirrorCount, q.mirrorSegCap, pred, &c->overflow);
    if (pred && mi != ~0u) {
        q.mv[0][mi] = make_float4(p.x, p.y, p.z, __int_as_float((int)(job | ((unsigned)nUp << 16))));
        q.mv[1][mi] = make_float4(n.x, n.y, n.z, 0.f);
        q.mv[2][mi] = make_float4(lam[0], lam[1], lam[2], lam[3]);
        q.mv[3][mi] = make_float4(beta[0] * w[0], beta[1] * w[1], beta[2] * w[2], beta[3] * w[3]);
    }
}

}  // namespace

// ------------------------------------------------------------------ schedule
// One workgroup of kMaxJobs threads: thread k owns position k of the priority order.
// Photons still to emit per job are scanned (inclusive prefix in LDS) and each job
// takes what fits in the free queue slots after the jobs ahead of it. The emitted
// photons are then placed after the survivors of each segment, filling segments in
// order; the segments' free room adds up to at least the free capacity, so the
// number emitted depends only on the total number of survivors.
__global__ void __launch_bounds__(kMaxJobs) k_schedule(Queues q, int cur) {
    __shared__ unsigned sScan[kMaxJobs];
    Ctrl* c = q.ctrl;
    const int k = threadIdx.x;
    const int n = c->nOrder;
    const unsigned it = c->iter;
    unsigned alive = 0;
#pragma unroll
    for (int g = 0; g < kSegs; ++g) alive += c->pathCount[cur][g][0];
    const unsigned freeSlots = c->capacity > alive ? c->capacity - alive : 0u;
    int j = -1;
    unsigned rem = 0;
    if (k < n) {
        j = c->order[k];
        const unsigned long long nx = c->nextPhoton[j], en = c->endPhoton[j];
        const unsigned long long r = (c->active[j] && en > nx) ? en - nx : 0ull;
        rem = r > (unsigned long long)freeSlots ? freeSlots : (unsigned)r;
    }
    sScan[k] = rem;
    __syncthreads();
    for (int off = 1; off < kMaxJobs; off <<= 1) {
        unsigned v = (k >= off) ? sScan[k - off] : 0u;
        __syncthreads();
        if (k >= off) sScan[k] = min(sScan[k] + v, 0x7fffffffu);
        __syncthreads();
    }
    const unsigned before = (k > 0) ? sScan[k - 1] : 0u;
    if (k < n) {
        const unsigned room = freeSlots > before ? freeSlots - before : 0u;
        const unsigned take = rem < room ? rem : room;
        const unsigned start = before < freeSlots ? before : freeSlots;
        c->emitPrefix[k] = start;
        c->emitJob[k] = j;
        c->emitStart[k] = c->nextPhoton[j];
        if (take) {
            c->nextPhoton[j] += take;
            if (c->nextPhoton[j] == c->endPhoton[j]) c->lastEmitIter[j] = (int)it;
        }
    }
    __syncthreads();
    if (k == 0) {
        const unsigned total = (n > 0) ? min(sScan[n - 1], freeSlots) : 0u;
        c->emitPrefix[n] = total;
        c->nEmit = total;
        unsigned left = total, placed = 0;
        for (int g = 0; g < kSegs; ++g) {
            const unsigned cnt = c->pathCount[cur][g][0];
            const unsigned room = c->segCap > cnt ? c->segCap - cnt : 0u;
            const unsigned e = left < room ? left : room;
            c->segBase[g] = cnt;
            c->segEmit[g] = placed;
            c->pathCount[cur][g][0] = cnt + e;
            c->pathCount[cur ^ 1][g][0] = 0;
            c->connCount[g][0] = 0;
            c->mirrorCount[g][0] = 0;
            placed += e;
            left -= e;
        }
        c->segEmit[kSegs] = placed;
        if (left) c->overflow = 1u;
        c->iter = it + 1;
    }
}

// ------------------------------------------------------------------ emit
// Position in the emission order of emission slot s (largest k with emitPrefix[k] <= s).
__device__ __forceinline__ int emitPosition(const Ctrl* c, int nOrder, unsigned s) {
    int lo = 0, hi = nOrder;
    while (lo + 1 < hi) {
        const int mid = (lo + hi) >> 1;
        if (c->emitPrefix[mid] <= s) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Emitter of a photon by the job's power CDF; draws only where there are several.
__device__ __forceinline__ int pickEmitter(const DevJob& J, Rng& rng) {
    if (J.nEm <= 1) return 0;
    const double u = rng.uniformD();
    int lo = 0, hi = J.nEm - 1;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (J.emCdf[mid] < u) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// Contiguous share [lo, hi) of column `col` of n items.
__device__ __forceinline__ void binRange(unsigned n, unsigned col, unsigned cols, unsigned& lo, unsigned& hi) {
    lo = (unsigned)(((unsigned long long)n * col) / cols);
    hi = (unsigned)(((unsigned long long)n * (col + 1)) / cols);
}

// Emission order. The key of a photon is the Morton code of the two uniform draws that
// place it on what spreads its rays most: the direction of a cosine emitter (the draws
// map to the hemisphere with equal area, so the keys fill evenly), the origin of a
// collimated one. With several jobs or emitters the leading bits keep those apart.
// The photon's stream is seeded again for it: the draws cost less than storing them.
__device__ __forceinline__ unsigned spread2(unsigned v) {
    v = (v | (v << 4)) & 0x0f0fu;
    v = (v | (v << 2)) & 0x3333u;
    return (v | (v << 1)) & 0x5555u;
}

__device__ __forceinline__ unsigned emitOrderKey(const Queues& q, const Ctrl* c, int nOrder, unsigned s) {
    const int k = nOrder > 1 ? emitPosition(c, nOrder, s) : 0;
    const DevJob& J = q.jobs[c->emitJob[k]];
    Rng rng = seedPhoton(J.seedBase + (c->emitStart[k] + (s - c->emitPrefix[k])), J.salt);
    const int ei = pickEmitter(J, rng);
    unsigned a = rng.next(), b = rng.next();
    if (!J.ems[ei].collimated) {
        a = rng.next();
        b = rng.next();
    }
    int bits = kBinBits;
    unsigned key = 0;
    if (nOrder > 1) {
        bits -= 4;
        key = ((unsigned)k & 15u) << bits;
    }
    if (J.nEm > 1) {
        bits -= 2;
        key |= ((unsigned)ei & 3u) << bits;
    }
    const unsigned z = (spread2(a >> 24) << 1) | spread2(b >> 24);   // 16 bits
    return key | (z >> (16 - bits));
}

// Keys of column blockIdx.x's emission slots and their histogram.
__global__ void __launch_bounds__(kBinThreads) k_emit_keys(Queues q) {
    __shared__ unsigned h[kBins];
    const Ctrl* c = q.ctrl;
    const unsigned n = c->nEmit;
    if (n < kEmitOrderMin) return;
    const int nOrder = c->nOrder;
    for (int b = threadIdx.x; b < kBins; b += blockDim.x) h[b] = 0u;
    __syncthreads();
    unsigned lo, hi;
    binRange(n, blockIdx.x, kEmitCols, lo, hi);
    for (unsigned s = lo + threadIdx.x; s < hi; s += blockDim.x) {
        const unsigned key = emitOrderKey(q, c, nOrder, s);
        q.emitKey[s] = (unsigned short)key;
        atomicAdd(&h[key], 1u);
    }
    __syncthreads();
    unsigned* out = q.emitHist + (size_t)blockIdx.x * kBins;
    for (int b = threadIdx.x; b < kBins; b += blockDim.x) out[b] = h[b];
}

// Emission slots in key order: emitPerm[sorted position] = slot. Only these 4 bytes per
// photon are scattered; k_emit reads them in order and writes its paths in order.
__global__ void __launch_bounds__(kBinThreads) k_emit_perm(Queues q) {
    __shared__ unsigned slot[kBins];
    const unsigned n = q.ctrl->nEmit;
    if (n < kEmitOrderMin) return;
    const unsigned col = blockIdx.x, ch = col / (kEmitCols / kBinChunks);
    const unsigned* colHist = q.emitHist + (size_t)col * kBins;
    const unsigned* chunk = q.emitChunk + (size_t)ch * kBins;
    for (int b = threadIdx.x; b < kBins; b += blockDim.x) slot[b] = q.emitTotal[b] + chunk[b] + colHist[b];
    __syncthreads();
    unsigned lo, hi;
    binRange(n, col, kEmitCols, lo, hi);
    for (unsigned s = lo + threadIdx.x; s < hi; s += blockDim.x) {
        const unsigned at = atomicAdd(&slot[q.emitKey[s]], 1u);
        if (at < n) q.emitPerm[at] = s;   // always: both passes read the same keys
    }
}

// Photon `idx` of job J: where it leaves the light and in which direction, its bundle of
// wavelengths and their weights. False for a photon without power at its wavelength.
__device__ __forceinline__ bool emitPhoton(const DevJob& J, unsigned long long idx, Rng& rng, F3& org, F3& en,
                                           F3& dir, float* lam, float* beta) {
    rng = seedPhoton(J.seedBase + idx, J.salt);
    const int ei = pickEmitter(J, rng);
    const DevEmitter& E = J.ems[ei];
    float u1 = rng.uniform();
    float u2 = rng.uniform();
    org = load3(E.origin) + load3(E.u) * u1 + load3(E.v) * u2;
    en = load3(E.normal);
    dir = E.collimated ? load3(E.beam) : cosineDir(en, rng);
    const int C = J.heroC;
    double ub = rng.uniformD();
    double pdf0;
    lam[0] = (float)invertCdf(E.cdf, E.guide, ub, pdf0);
    for (int i = 1; i < C; ++i) {
        double uu = ub + (double)i / (double)C;
        if (uu >= 1.0) uu -= 1.0;
        double pd;
        lam[i] = (float)invertCdf(E.cdf, E.guide, uu, pd);
    }
    const float b = J.basePower / (float)C;
    for (int i = 0; i < C; ++i) beta[i] = b;
    return pdf0 > 0.0;
}

// Launch bound: five waves per SIMD (96 registers, no spills; -2% k_emit time on c2).
__global__ void __launch_bounds__(256, 5) k_emit(Queues q, int cur) {
    Ctrl* c = q.ctrl;
    const unsigned nEmit = c->nEmit;
    const int nOrder = c->nOrder;
    const int nJobs = c->nJobs;
    // emission position `at` goes to segment g (segEmit[g] <= at < segEmit[g + 1]), after
    // that segment's segBase[g] survivors
    SegMap em;
    unsigned emBase[kSegs];
#pragma unroll
    for (int g = 0; g < kSegs; ++g) {
        em.pre[g] = c->segEmit[g];
        emBase[g] = c->segBase[g];
    }
    em.cap = q.segCap;
    __shared__ unsigned long long eTab[kMaxJobs], pTab[kMaxJobs * 2];
    initJobTable<1>(eTab, nJobs);
    initJobTable<2>(pTab, nJobs);
    JobAcc<1> eacc;   // emitted
    JobAcc<2> pacc;   // photons, direct camera connections
    AccAddr ea{q.jobs, kAccEnergy};
    AccAddr pa{q.jobs, kAccPhotons};
    const unsigned stride = gridDim.x * blockDim.x;
    const bool ordered = q.emitOrder && nEmit >= kEmitOrderMin;
    for (unsigned at = blockIdx.x * blockDim.x + threadIdx.x; at < nEmit; at += stride) {
        const unsigned s = ordered ? q.emitPerm[at] : at;   // emission slot; `at` places the path
        const int k = nOrder > 1 ? emitPosition(c, nOrder, s) : 0;
        const int j = c->emitJob[k];
        const DevJob& J = q.jobs[j];
        const unsigned long long idx = c->emitStart[k] + (s - c->emitPrefix[k]);
        float lam[kMaxHero] = {0.f, 0.f, 0.f, 0.f};
        float beta[kMaxHero] = {0.f, 0.f, 0.f, 0.f};
        F3 org, en, dir;
        Rng rng;
        const int C = J.heroC;
        const bool dead = !emitPhoton(J, idx, rng, org, en, dir, lam, beta);
        const float b = beta[0];
        accumulate(eacc, j, eTab);
        accumulate(pacc, j, pTab);
        pacc.v[0] += 1;
        if (!dead) eacc.v[0] += toFixed((double)b * (double)C, J.energyScale);
        {
            const float one[kMaxHero] = {1.f, 1.f, 1.f, 1.f};
            const unsigned mask = connectMask(J.cams, dead ? 0 : J.nCams, org, en);
            const unsigned room = connectCount(mask);
            unsigned off = 0;
            if (room) {
                const unsigned first = (unsigned)__ffsll((long long)__ballot(true)) - 1u;
                if (laneId() == first) off = atomicAdd(&c->connCount[blockIdx.x % kSegs][0], room);
                off = __shfl(off, (int)first);
                connectWrite(q, c, J.cams, mask, off, (unsigned)j, org, en, lam, beta, one, C);
            }
            pacc.v[1] += (unsigned)__popcll(mask);
            queueMirrorVertex(q, c, !dead && J.nMirrors > 0, (unsigned)j, org, en, lam, beta, one, C);
        }
        F3 o = org + dir * kRayEps;
        unsigned slot = 0;
        {
            unsigned off = at, g0 = 0;
#pragma unroll
            for (int g = 1; g < kSegs; ++g)
                if (at >= em.pre[g]) { g0 = (unsigned)g; off = at - em.pre[g]; }
            unsigned b = emBase[0];
#pragma unroll
            for (int g = 1; g < kSegs; ++g)
                if (g0 == (unsigned)g) b = emBase[g];
            slot = g0 * q.segCap + b + off;
        }
        q.ro[cur][slot] = make_float4(o.x, o.y, o.z, 0.f);
        q.rd[cur][slot] = make_float4(dir.x, dir.y, dir.z, 0.f);
        q.lam[cur][slot] = make_float4(lam[0], lam[1], lam[2], lam[3]);
        q.beta[cur][slot] = make_float4(beta[0], beta[1], beta[2], beta[3]);
        unsigned meta = packMeta((unsigned)j, 0u, (unsigned)C) | (dead ? 0x80000000u : 0u);
        q.st[cur][slot] = make_uint4((unsigned)rng.state, (unsigned)(rng.state >> 32), (unsigned)idx, meta);
        if (q.binned) q.key[cur][slot] = dead ? (unsigned short)0 : binKey(J, o, dir);
    }
    flushJobTable(eacc, eTab, nJobs, ea);
    flushJobTable(pacc, pTab, nJobs, pa);
}

// ------------------------------------------------------------------ extend
// STATS: also count the traversal statistics (node visits, triangle tests) per job.
// BIN: read the binned queue (ray binning) instead of queue `cur`.
// The traversal waits on dependent node loads, so resident waves are what hides the
// latency. Segments are counted by k_shade (same paths), so outside the statistics
// variant the kernel's LDS is the traversal stack alone (SD * 512 bytes per one-wave
// workgroup), and the launch bound asks for six waves per SIMD (at most 80 registers;
// the compiler applies it where the LDS allows six: SD = 8, two spilled registers in
// the spilling binned variant). Measured on c2, closest-hit time per 2^28 photons:
// 148.3 ms at SD 16 and five waves, 144.2 at SD 8 and five, 140.6 at SD 8 and six;
// seven or eight waves spill inside the loop (187 / 202 ms).
template <int SD, bool SPILL, bool STATS, bool BIN>
__global__ void __launch_bounds__(kExtendThreads, 6) k_extend(Queues q, int cur) {
    constexpr int NA = STATS ? 2 : 1;   // node visits, triangle tests
    __shared__ int2 sStk[SD * kExtendThreads];
    __shared__ unsigned segTab[kSegs];
    SegMap sm;
    const unsigned n = loadSegMap(q.ctrl->pathCount[cur], q.segCap, sm);
    if (q.resetCounts && blockIdx.x == 0 && threadIdx.x < kSegs) {
        // nothing else of this kernel touches these; the last readers ran before it
        q.ctrl->pathCount[cur ^ 1][threadIdx.x][0] = 0u;
        q.ctrl->connCount[threadIdx.x][0] = 0u;
        q.ctrl->mirrorCount[threadIdx.x][0] = 0u;
    }
    if constexpr (!BIN) {
        initSegTab(sm, segTab);
        __syncthreads();
    }
    const unsigned stride = gridDim.x * blockDim.x;
    const unsigned gtid = blockIdx.x * blockDim.x + threadIdx.x;
    Stack<SD, true, SPILL, kExtendThreads> stk{sStk + threadIdx.x, nullptr,
                                               SPILL ? q.spill + (size_t)gtid * q.spillDepth : nullptr, 0};
    const int nJobs = q.ctrl->nJobs;
    __shared__ unsigned long long sTab[STATS ? kMaxJobs * NA : 1];
    if constexpr (STATS) initJobTable<NA>(sTab, nJobs);
    JobAcc<NA> sacc;
    AccAddr sa{q.jobs, kAccNodeVisits};
    for (unsigned li = gtid; li < n; li += stride) {
        const unsigned i = BIN ? li : sm.slotTab(li, segTab);
        const uint4 s4 = BIN ? bitcast4(q.pb[5 * (size_t)i + 4]) : q.st[cur][i];
        int best = -1;
        float t = INFINITY;
        if (!(s4.w & 0x80000000u)) {
            const int j = (int)(s4.w & 0xffffu);
            const DevJob& J = q.jobs[j];
            const float4 o = BIN ? q.pb[5 * (size_t)i] : q.ro[cur][i];
            const float4 d = BIN ? q.pb[5 * (size_t)i + 1] : q.rd[cur][i];
            RayPre r = prepareRay(xyz(o), xyz(d));
            float tmax = INFINITY;
            TravCount<STATS> tc;
            best = traceClosest<SD, SPILL>(J.nodes, J.tris, r, kRayEps, tmax, stk, tc);
            t = tmax;
            if constexpr (STATS) {
                accumulate(sacc, j, sTab);
                sacc.v[0] += tc.nodes;
                sacc.v[1] += tc.tri;
            }
        }
        q.hit[i] = make_float2(t, __int_as_float(best));
    }
    if constexpr (STATS) flushJobTable(sacc, sTab, nJobs, sa);
}

// ------------------------------------------------------------------ shade
// BIN: read the binned queue (ray binning) instead of queue `cur` and store the
// survivors' bin keys.
// Each round of the workgroup places its survivors sorted by kLocalKeys local keys (five
// Morton bits of the origin's cell, then the direction octant) in one run of its
// segment: a counting sort in LDS, one queue atomic per workgroup and round instead of
// one per wave. Paths that follow sorted ones start close together, so the octant then
// separates them well: closest-hit time on the glass scene 25.7 -> 22.8 ms per 2^26
// photons (without ray binning), 2.5 -> 2.3 ms on the box.
constexpr int kLocalKeys = 256;
__device__ __forceinline__ unsigned localKey(unsigned key) { return ((key >> 7) << 3) | (key & 7u); }

// What a path's hit at p (triangle `tri`, arriving along d) does: the scatter in place
// (wavelengths, weights, stream), the vertex to connect to the cameras, and whether the
// path goes on (from no along nd). led: absorbed, escaped, residual.
struct Vertex {
    bool diffuse = false;
    F3 n{0.f, 0.f, 0.f};
    float beta[kMaxHero] = {0.f, 0.f, 0.f, 0.f}, rho[kMaxHero] = {0.f, 0.f, 0.f, 0.f};
};

__device__ __forceinline__ bool scatterHit(const DevJob& J, F3 p, F3 d, int tri, unsigned photon, int bounce,
                                           Rng& rng, const float* lam, float* beta, int& nUp,
                                           unsigned long long* led, Vertex& v, F3& no, F3& nd) {
    auto activeSum = [&]() {
        double s = 0.0;
        for (int k = 0; k < nUp; ++k) s += (double)beta[k];
        return s;
    };
    const float4 tn = J.trin[tri];
    const F3 gn = xyz(tn);
    const DevMaterial& M = J.mats[__float_as_int(tn.w)];
    const F3 n = (dot(d, gn) < 0.0f) ? gn : -gn;
    rng.inc = photonInc(J.seedBase + photon, J.salt);
    const bool roulette = bounce >= J.rrDepth;
    bool alive = true;
    if (M.type == 1) {
        // Dielectric: de-hero, then Fresnel reflect or Snell refract (exterior
        // index 1). The side is read off the geometric normal (entering when the
        // ray runs against it), as the reference does.
        if (nUp > 1) {
            beta[0] *= (float)J.heroC;
            nUp = 1;
        }
        const float eta_g = specEval(M.ior, lam[0]);
        const bool entering = dot(d, gn) < 0.0f;
        const F3 nl = entering ? gn : -gn;
        const float n1 = entering ? 1.0f : eta_g;
        const float n2 = entering ? eta_g : 1.0f;
        const float eta = n1 / n2;
        const float cosI = -dot(d, nl);
        const float sin2t = eta * eta * (1.0f - cosI * cosI);
        F3 out;
        bool refracted = false;
        if (sin2t > 1.0f) {
            out = reflectDir(d, nl);
        } else {
            const float cosT = sqrtf(1.0f - sin2t);
            const float rs = (n1 * cosI - n2 * cosT) / (n1 * cosI + n2 * cosT);
            const float rp = (n1 * cosT - n2 * cosI) / (n1 * cosT + n2 * cosI);
            const float R = 0.5f * (rs * rs + rp * rp);
            if (rng.uniform() < R) {
                out = reflectDir(d, nl);
            } else {
                out = d * eta + nl * (eta * cosI - cosT);
                refracted = true;
            }
        }
        out = normalize(out);
        if (M.roughness > 1e-3f) {
            F3 pert = glossyDir(out, M.roughness, rng);
            bool ok = refracted ? (dot(pert, nl) < 0.0f) : (dot(pert, nl) > 0.0f);
            if (ok) out = pert;
        }
        no = p + out * kRayEps;
        nd = out;
    } else {
        float c[kMaxHero] = {0.f, 0.f, 0.f, 0.f};
        float q0 = 0.0f;
        for (int k = 0; k < nUp; ++k) {
            float r = specEval(M.reflect, lam[k]);
            c[k] = r < 0.0f ? 0.0f : (r > 1.0f ? 1.0f : r);
            q0 = (k == 0 || c[k] > q0) ? c[k] : q0;
        }
        const bool diffuse = (M.type == 0);
        if (diffuse) {
            v.diffuse = true;
            v.n = n;
            for (int k = 0; k < kMaxHero; ++k) { v.beta[k] = beta[k]; v.rho[k] = c[k]; }
        }
        if (roulette) {
            if (rng.uniform() >= q0) {
                led[0] += toFixed(activeSum(), J.energyScale);
                alive = false;
            } else {
                double ab = 0.0;
                for (int k = 0; k < nUp; ++k) {
                    float w = c[k] / q0;
                    ab += (double)beta[k] * (double)(1.0f - w);
                    beta[k] *= w;
                }
                led[0] += toFixed(ab, J.energyScale);
            }
        } else {
            if (!(q0 > 0.0f)) {
                led[0] += toFixed(activeSum(), J.energyScale);
                alive = false;
            } else {
                double ab = 0.0;
                for (int k = 0; k < nUp; ++k) {
                    ab += (double)beta[k] * (double)(1.0f - c[k]);
                    beta[k] *= c[k];
                }
                led[0] += toFixed(ab, J.energyScale);
            }
        }
        if (alive) {
            F3 wo;
            if (diffuse) {
                wo = cosineDir(n, rng);
            } else if (M.type == 2) {
                wo = reflectDir(d, n);
            } else {
                wo = glossyDir(reflectDir(d, n), M.roughness, rng);
                if (dot(wo, n) <= 0.0f) {
                    led[0] += toFixed(activeSum(), J.energyScale);
                    alive = false;
                }
            }
            no = p + n * kRayEps;
            nd = wo;
        }
    }
    if (alive && bounce + 1 >= J.maxDepth) {
        led[2] += toFixed(activeSum(), J.energyScale);
        alive = false;
    }
    return alive;
}

template <bool BIN>
__global__ void __launch_bounds__(kShadeThreads, 4) k_shade(Queues q, int cur) {
    const int nxt = cur ^ 1;
    Ctrl* ctl = q.ctrl;
    SegMap sm;
    const unsigned n = loadSegMap(ctl->pathCount[cur], q.segCap, sm);
    __shared__ unsigned segTab[kSegs];
    if constexpr (!BIN) initSegTab(sm, segTab);   // initJobTable's barrier covers it
    const unsigned stride = gridDim.x * blockDim.x;
    const int nJobs = ctl->nJobs;
    __shared__ unsigned long long eTab[kMaxJobs * 4];
    initJobTable<4>(eTab, nJobs);
    // absorbed, escaped, residual -> ledger entries 1, 3, 4; the closest-hit queries of
    // the paths (every live path of the queue was traced by k_extend) -> segments
    JobAcc<4> eacc;
    AccAddr ea{q.jobs, kAccEnergy};
    auto eaddr = [&](int j, int k) {
        return ea(j, k == 0 ? 1 : (k == 1 ? 3 : (k == 2 ? 4 : kAccSegments - kAccEnergy)));
    };
    __shared__ unsigned keyHist[2][kLocalKeys], waveSum[kLocalKeys / 64], runBase;
    __shared__ unsigned waveConn[kShadeThreads / 64];   // connections, then each wave's first slot
    if (threadIdx.x < kLocalKeys) keyHist[0][threadIdx.x] = 0u;
    __syncthreads();
    const unsigned seg = blockIdx.x % kSegs;
    unsigned buf = 0;
    // rounds are workgroup-uniform (the sort has barriers)
    for (unsigned base = blockIdx.x * blockDim.x; base < n; base += stride, buf ^= 1u) {
        const unsigned li = base + threadIdx.x;
        const bool have = li < n;
        const unsigned i = BIN ? (have ? li : base) : sm.slotTab(have ? li : base, segTab);
        const float4* rec = q.pb + 5 * (size_t)i;   // binned record (BIN only)
        const uint4 s4 = BIN ? bitcast4(rec[4]) : q.st[cur][i];
        bool alive = false;
        unsigned short bkey = 0;
        // diffuse vertex to connect to the cameras after shading
        int camN = 0;
        bool mirrorsToo = false;
        const DevCamera* cams = nullptr;
        unsigned cjob = 0;
        int cUp = 0;
        F3 cp{0.f, 0.f, 0.f}, cn{0.f, 0.f, 0.f};
        float cbeta[kMaxHero] = {0.f, 0.f, 0.f, 0.f}, crho[kMaxHero] = {0.f, 0.f, 0.f, 0.f};
        F3 no, nd;
        float lam[kMaxHero], beta[kMaxHero];
        unsigned meta = s4.w;
        Rng rng;
        rng.state = (uint64_t)s4.x | ((uint64_t)s4.y << 32);
        if (have && !(meta & 0x80000000u)) {
            const int j = (int)(meta & 0xffffu);
            const int bounce = (int)((meta >> 16) & 0xffu);
            int nUp = (int)((meta >> 24) & 7u);
            const DevJob& J = q.jobs[j];
            accumulate(eacc, j, eTab);
            eacc.v[3] += 1;
            const float4 l4 = BIN ? rec[2] : q.lam[cur][i], b4 = BIN ? rec[3] : q.beta[cur][i];
            lam[0] = l4.x; lam[1] = l4.y; lam[2] = l4.z; lam[3] = l4.w;
            beta[0] = b4.x; beta[1] = b4.y; beta[2] = b4.z; beta[3] = b4.w;
            auto activeSum = [&]() {
                double s = 0.0;
                for (int k = 0; k < nUp; ++k) s += (double)beta[k];
                return s;
            };
            const float2 h = q.hit[i];
            const int tri = __float_as_int(h.y);
            if (tri < 0) {
                eacc.v[1] += toFixed(activeSum(), J.energyScale);
            } else {
                const float4 o4 = BIN ? rec[0] : q.ro[cur][i], d4 = BIN ? rec[1] : q.rd[cur][i];
                const F3 d = xyz(d4);
                const F3 p = xyz(o4) + d * h.x;
                Vertex v;
                alive = scatterHit(J, p, d, tri, s4.z, bounce, rng, lam, beta, nUp, eacc.v, v, no, nd);
                if (v.diffuse) {
                    camN = J.nCams;
                    mirrorsToo = J.nMirrors > 0;
                    cams = J.cams;
                    cjob = (unsigned)j;
                    cUp = nUp;
                    cp = p;
                    cn = v.n;
                    for (int k = 0; k < kMaxHero; ++k) { cbeta[k] = v.beta[k]; crho[k] = v.rho[k]; }
                }
                if (alive) bkey = binKey(J, no, nd);
                meta = packMeta((unsigned)j, (unsigned)(bounce + 1), (unsigned)nUp);
            }
        }
        const unsigned camMask = connectMask(cams, camN, cp, cn);
        const unsigned room = connectCount(camMask);
        if ((threadIdx.x & 63u) == 0u) waveConn[threadIdx.x >> 6] = room;
        queueMirrorVertex(q, ctl, mirrorsToo, cjob, cp, cn, lam, cbeta, crho, cUp);
        // survivors: rank within the key, exclusive scan of the keys, one run per round
        // (the other histogram is cleared for the next round meanwhile)
        unsigned* hist = keyHist[buf];
        const unsigned lk = localKey(bkey);
        const unsigned rank = alive ? atomicAdd(&hist[lk], 1u) : 0u;
        __syncthreads();
        if (threadIdx.x < kLocalKeys) {
            // after the barrier: every wave has read the last round's ranks in it
            keyHist[buf ^ 1u][threadIdx.x] = 0u;
            const unsigned lane = threadIdx.x & 63u, own = hist[threadIdx.x];
            unsigned sum = own;
            for (unsigned off = 1; off < 64; off <<= 1) {
                const unsigned v = __shfl(sum, (int)(lane >= off ? lane - off : lane));
                sum += lane >= off ? v : 0u;
            }
            hist[threadIdx.x] = sum - own;
            if (lane == 63u) waveSum[threadIdx.x >> 6] = sum;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned total = 0;
            for (int k = 0; k < kLocalKeys / 64; ++k) {
                const unsigned v = waveSum[k];
                waveSum[k] = total;
                total += v;
            }
            runBase = total ? atomicAdd(&ctl->pathCount[nxt][seg][0], total) : 0u;
        }
        if (threadIdx.x == 64) {
            unsigned total = 0;
            for (int k = 0; k < kShadeThreads / 64; ++k) total += waveConn[k];
            unsigned at = total ? atomicAdd(&ctl->connCount[seg][0], total) : 0u;
            for (int k = 0; k < kShadeThreads / 64; ++k) {
                const unsigned v = waveConn[k];
                waveConn[k] = at;
                at += v;
            }
        }
        __syncthreads();
        connectWrite(q, ctl, cams, camMask, waveConn[threadIdx.x >> 6], cjob, cp, cn, lam, cbeta, crho, cUp);
        const unsigned off = runBase + waveSum[lk >> 6] + hist[lk] + rank;
        if (alive && off >= q.segCap) {
            ctl->overflow = 1u;
            alive = false;
        }
        if (alive) {
            const unsigned pi = seg * q.segCap + off;
            q.ro[nxt][pi] = make_float4(no.x, no.y, no.z, 0.f);
            q.rd[nxt][pi] = make_float4(nd.x, nd.y, nd.z, 0.f);
            q.lam[nxt][pi] = make_float4(lam[0], lam[1], lam[2], lam[3]);
            q.beta[nxt][pi] = make_float4(beta[0], beta[1], beta[2], beta[3]);
            q.st[nxt][pi] = make_uint4((unsigned)rng.state, (unsigned)(rng.state >> 32), s4.z, meta);
            if constexpr (BIN) q.key[nxt][pi] = bkey;
        }
    }
    flushJobTable(eacc, eTab, nJobs, eaddr);
}

// ------------------------------------------------------------------ connect
// Splat table: a per-workgroup open-addressing table in LDS keyed by (job, camera,
// pixel).
// Unoccluded connections add their integer X, Y, Z and hit count into it with LDS
// 64-bit atomics. When a connection finds no slot within kSplatProbe probes, the
// workgroup flushes the whole table to the film and starts a fresh one, so every
// film update goes through the table. Two properties of the memory system shape
// this:
//   - film atomics are limited by requests, not operations: four lanes adding the
//     four words of one pixel in one instruction cost one request, four lanes each
//     adding to their own pixel cost four (measured ~91 vs ~23 G atomics/s on
//     MI355X), so the flush hands (slot, word) pairs to consecutive lanes;
//   - atomics on one address serialise (~12 ns each), and pixels that many
//     connections hit (the emitter's direct view, caustic foci) would queue on a few
//     addresses; the table sums them first.
// Integer sums are order-independent, so the film is bit-identical to splatting
// each connection directly.
constexpr int kSplatSlots = 256;
constexpr int kSplatProbe = 8;
constexpr unsigned long long kSplatEmpty = ~0ull;

// Slot of `key` (claimed if absent) within maxProbe linear probes, or -1.
template <int SLOTS = kSplatSlots>
__device__ __forceinline__ int splatSlot(unsigned long long* sKey, unsigned long long key, int maxProbe) {
    const unsigned h = (unsigned)((key * 0x9E3779B97F4A7C15ull) >> 56);
    for (int p = 0; p < maxProbe; ++p) {
        const int s = (int)((h + (unsigned)p) & (SLOTS - 1));
        unsigned long long cur = __hip_atomic_load(&sKey[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (cur == kSplatEmpty) cur = atomicCAS(&sKey[s], kSplatEmpty, key);
        if (cur == kSplatEmpty || cur == key) return s;
    }
    return -1;
}

__device__ __forceinline__ void splatAdd(unsigned long long* sVal, int s, unsigned long long X,
                                         unsigned long long Y, unsigned long long Z, unsigned long long H) {
    if (X) atomicAdd(&sVal[4 * s + 0], X);
    if (Y) atomicAdd(&sVal[4 * s + 1], Y);
    if (Z) atomicAdd(&sVal[4 * s + 2], Z);
    atomicAdd(&sVal[4 * s + 3], H);
}

// Called by every thread of the workgroup after a barrier: adds every occupied
// slot into its film, lane t taking word t % 4 of slot t / 4 (+ 64 per pass).
template <int SLOTS = kSplatSlots>
__device__ __forceinline__ void flushSplats(const DevJob* jobs, const unsigned long long* sKey,
                                            const unsigned long long* sVal) {
    const int w = threadIdx.x & 3;
    for (int s = threadIdx.x >> 2; s < SLOTS; s += blockDim.x >> 2) {
        const unsigned long long key = sKey[s];
        if (key == kSplatEmpty) continue;
        const unsigned long long v = sVal[4 * s + w];
        if (v) {
            const unsigned jc = (unsigned)(key >> 32);
            unsigned long long* f = (unsigned long long*)jobs[jc / kMaxCams].cams[jc % kMaxCams].film;
            atomicAdd(f + 4 * (size_t)(key & 0xffffffffull) + w, v);
        }
    }
}

template <int SLOTS = kSplatSlots>
__device__ __forceinline__ void clearSplats(unsigned long long* sKey, unsigned long long* sVal) {
    for (int k = threadIdx.x; k < SLOTS; k += blockDim.x) {
        sKey[k] = kSplatEmpty;
        sVal[4 * k + 0] = 0; sVal[4 * k + 1] = 0; sVal[4 * k + 2] = 0; sVal[4 * k + 3] = 0;
    }
}

// Launch bound: six waves per SIMD where the LDS allows it (the default 8-entry stack:
// 22.8 KB per workgroup; 80 registers, five spilled): k_connect 26.7 -> 25.6 ms on c2
// against five waves with a 16-entry stack.
template <int SD, bool SPILL, bool STATS>
__global__ void __launch_bounds__(kTravThreads, 6) k_connect(Queues q) {
    constexpr int NA = STATS ? 4 : 2;   // connections, splats[, node visits, triangle tests]
    __shared__ int sStk[SD * kTravThreads];
    __shared__ unsigned long long sKey[kSplatSlots];
    __shared__ unsigned long long sVal[kSplatSlots * 4];
    clearSplats(sKey, sVal);
    SegMap sm;
    const unsigned n = loadSegMap(q.ctrl->connCount, q.connSegCap, sm);
    __shared__ unsigned segTab[kSegs];
    initSegTab(sm, segTab);   // initJobTable's barrier covers it
    const unsigned stride = gridDim.x * blockDim.x;
    const unsigned gtid = blockIdx.x * blockDim.x + threadIdx.x;
    Stack<SD, false, SPILL> stk{nullptr, sStk + threadIdx.x,
                                SPILL ? q.spill + (size_t)gtid * q.spillDepth : nullptr, 0};
    const int nJobs = q.ctrl->nJobs;
    __shared__ unsigned long long cTab[kMaxJobs * NA];
    initJobTable<NA>(cTab, nJobs);   // (its barrier also orders clearSplats)
    JobAcc<NA> cacc;
    AccAddr ca{q.jobs, kAccConnections};
    // Rounds are workgroup-uniform so the table can be flushed between them.
    for (unsigned base = blockIdx.x * blockDim.x; base < n; base += stride) {
        const unsigned li = base + threadIdx.x;
        bool pending = false;
        unsigned long long key = 0, X = 0, Y = 0, Z = 0, H = 0;
        if (li < n) {
            const unsigned i = sm.slotTab(li, segTab);
            const float4 co = q.co[i], cd = q.cd[i], cx = q.cx[i];
            const unsigned tag = (unsigned)__float_as_int(cx.w);
            const int j = (int)(tag & 0xffffu);
            const int cam = (int)((tag >> 19) & 15u);
            const DevJob& J = q.jobs[j];
            accumulate(cacc, j, cTab);
            cacc.v[0] += 1;
            RayPre r = prepareRay(xyz(co), xyz(cd));
            TravCount<STATS> tc;
            const bool occ = traceAny<SD, SPILL>(J.nodes, J.tris, r, kRayEps, co.w, stk, tc);
            if constexpr (STATS) {
                cacc.v[2] += tc.nodes;
                cacc.v[3] += tc.tri;
            }
            if (!occ) {
                cacc.v[1] += 1;
                const DevCamera& K = J.cams[cam];
                const unsigned pix = (unsigned)__float_as_int(cd.w);
                X = min(toFixed((double)cx.x, K.filmScale), K.filmQmax);
                Y = min(toFixed((double)cx.y, K.filmScale), K.filmQmax);
                Z = min(toFixed((double)cx.z, K.filmScale), K.filmQmax);
                H = (unsigned long long)((tag >> 16) & 7u);
                key = ((unsigned long long)(j * kMaxCams + cam) << 32) | pix;
                const int s = splatSlot(sKey, key, kSplatProbe);
                if (s >= 0) splatAdd(sVal, s, X, Y, Z, H);
                else pending = true;
            }
        }
        if (__syncthreads_or(pending)) {
            flushSplats(q.jobs, sKey, sVal);
            __syncthreads();
            clearSplats(sKey, sVal);
            __syncthreads();
            // Only the pending keys, at most one per thread, go into the empty table
            // before the barrier below lets any thread start the next round, so a full
            // scan always finds its key or a free slot. (Without the barrier, waves
            // racing ahead could fill the table first.) A failed scan still falls
            // back to the film itself rather than index the table with -1.
            if (pending) {
                const int s = splatSlot(sKey, key, kSplatSlots);
                if (s >= 0) {
                    splatAdd(sVal, s, X, Y, Z, H);
                } else {
                    const unsigned jc = (unsigned)(key >> 32);
                    unsigned long long* f =
                        (unsigned long long*)q.jobs[jc / kMaxCams].cams[jc % kMaxCams].film +
                        4 * (size_t)(key & 0xffffffffull);
                    if (X) atomicAdd(f + 0, X);
                    if (Y) atomicAdd(f + 1, Y);
                    if (Z) atomicAdd(f + 2, Z);
                    atomicAdd(f + 3, H);
                }
            }
            __syncthreads();
        }
    }
    flushJobTable(cacc, cTab, nJobs, ca);   // ends with a barrier-ordered read of cTab
    __syncthreads();
    flushSplats(q.jobs, sKey, sVal);
}

// ------------------------------------------------------------------ flight
// A whole small trace in one launch: each lane carries a photon from the light to the end
// of its path, and connects its vertices on the way. A lane whose path has ended takes its
// next photon (gtid, gtid + stride, ...) once a quarter of the wave's live lanes waits for
// one, so that the emission code does not run for a lane or two at a time. Between
// iterations of the wavefront a path goes through 200 bytes of memory and three launches;
// here it stays in registers (128 of them: four waves per SIMD).
// The wavefront's kernels are bound by launches and dependent loads while a trace does not
// fill the chip: the 5000-photon preview of the box spent 470 of its 590 us in 26 kernels.
// `lanes` of each wave carry photons: a trace of few photons is spread over more waves, so
// that a wave's time is the longest of fewer paths.
// One wave per workgroup, with a splat table of its own that is flushed only at the end: a
// splat that finds no slot is added to its film by four lanes, one per word. Any hit and
// closest hit use the lane's own stack column one after the other. Lanes of a wave may be in
// different traversals, so both keep to the same words: entry k of lane t at int2 64 k + t and
// at int 128 k + 2 t. (int entries of stride 64 would lie in other lanes' columns: lanes
// popped each other's words as nodes when k_mirror once did that.)
constexpr int kFlightSlots = 64;

// Keeps the LDS accesses of a wave's lanes on either side apart. The hardware runs them in
// program order; the fence keeps the compiler to it also where the two sides use one array
// under different types (stack entries, staged words), which it may otherwise take for
// different memory. No instruction of its own.
__device__ __forceinline__ void waveFence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Adds the splats of the lanes with `pending` to their films, four lanes per splat. The
// records are staged in the stack array `stk` (no traversal is running: the whole wave is
// here).
__device__ __forceinline__ void splatDirect(int2* stk, bool pending, unsigned long long* at, unsigned long long X,
                                            unsigned long long Y, unsigned long long Z, unsigned long long H) {
    const unsigned long long mask = __ballot(pending);
    if (mask == 0ull) return;
    waveFence();
    const unsigned lane = threadIdx.x;
    unsigned long long* col = (unsigned long long*)stk;
    const unsigned rank = __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
    if (pending) {
        col[0 * kFlightThreads + rank] = X;
        col[1 * kFlightThreads + rank] = Y;
        col[2 * kFlightThreads + rank] = Z;
        col[3 * kFlightThreads + rank] = H;
        col[4 * kFlightThreads + rank] = (unsigned long long)at;
    }
    waveFence();
    const unsigned count = (unsigned)__popcll(mask);
    for (unsigned b = 0; b < count; b += 16) {
        const unsigned r = b + (lane >> 2);
        if (r < count) {
            const unsigned long long v = col[(lane & 3u) * kFlightThreads + r];
            if (v) atomicAdd((unsigned long long*)col[4 * kFlightThreads + r] + (lane & 3u), v);
        }
    }
    waveFence();
}

template <int SD, bool SPILL>
__global__ void __launch_bounds__(kFlightThreads, 4) k_flight(Queues q, unsigned n, unsigned lanes) {
    static_assert(SD >= 5, "splatDirect stages five words per lane");
    __shared__ int2 sStk[SD * kFlightThreads];
    __shared__ unsigned long long sKey[kFlightSlots];
    __shared__ unsigned long long sVal[kFlightSlots * 4];
    __shared__ unsigned long long sAcc[kAccRow];
    __shared__ unsigned sLongest;   // segments of the longest path
    clearSplats<kFlightSlots>(sKey, sVal);
    if (threadIdx.x < kAccRow) sAcc[threadIdx.x] = 0ull;
    if (threadIdx.x == 0) sLongest = 0u;
    __syncthreads();
    const DevJob& J = q.jobs[0];
    const unsigned gtid = blockIdx.x * blockDim.x + threadIdx.x;
    int2* spill = SPILL ? q.spill + (size_t)gtid * q.spillDepth : nullptr;
    const unsigned stride = gridDim.x * lanes;
    unsigned next = threadIdx.x < lanes ? min(blockIdx.x * lanes + threadIdx.x, n) : n;
    unsigned long long led[3] = {}, emitted = 0;   // absorbed, escaped, residual; emitted
    unsigned photons = 0, direct = 0, segments = 0, connections = 0, splats = 0;
    bool alive = false;
    F3 o{0.f, 0.f, 0.f}, d{0.f, 0.f, 0.f};
    float lam[kMaxHero] = {0.f, 0.f, 0.f, 0.f}, beta[kMaxHero] = {0.f, 0.f, 0.f, 0.f};
    Rng rng{};
    unsigned photon = 0;
    int bounce = 0, nUp = 0;
    TravCount<false> tc;
    while (true) {
        const unsigned live = (unsigned)__popcll(__ballot(alive));
        const unsigned waiting = (unsigned)__popcll(__ballot(!alive && next < n));
        if (live + waiting == 0) break;
        F3 vp{0.f, 0.f, 0.f};
        Vertex v;
        int vUp = 0;
        bool atLight = false;
        if (alive) {
            Stack<SD, true, SPILL, kFlightThreads> stk{sStk + threadIdx.x, nullptr, spill, 0};
            float t = INFINITY;
            const int tri = traceClosest<SD, SPILL>(J.nodes, J.tris, prepareRay(o, d), kRayEps, t, stk, tc);
            ++segments;
            if (tri < 0) {
                double s = 0.0;
                for (int k = 0; k < nUp; ++k) s += (double)beta[k];
                led[1] += toFixed(s, J.energyScale);
                alive = false;
            } else {
                vp = o + d * t;
                F3 no{0.f, 0.f, 0.f}, nd{0.f, 0.f, 0.f};
                vUp = nUp;
                alive = scatterHit(J, vp, d, tri, photon, bounce, rng, lam, beta, nUp, led, v, no, nd);
                o = no;
                d = nd;
                ++bounce;
            }
            if (!alive) atomicMax(&sLongest, (unsigned)bounce + (tri < 0 ? 1u : 0u));
        } else if (next < n && 4 * waiting >= live) {
            for (int k = 0; k < kMaxHero; ++k) { lam[k] = 0.f; beta[k] = 0.f; }
            photon = next;
            next = n - next > stride ? next + stride : n;
            F3 dir;
            alive = emitPhoton(J, photon, rng, vp, v.n, dir, lam, beta);
            ++photons;
            o = vp + dir * kRayEps;
            d = dir;
            bounce = 0;
            nUp = vUp = J.heroC;
            if (alive) {
                emitted += toFixed((double)beta[0] * (double)J.heroC, J.energyScale);
                atLight = v.diffuse = true;
                for (int k = 0; k < kMaxHero; ++k) { v.beta[k] = beta[k]; v.rho[k] = 1.0f; }
            }
        }
        __syncthreads();   // one wave: the lanes are together from here to the next photon
        const int nCams = v.diffuse ? J.nCams : 0;
        for (int k = 0; __any(k < nCams); ++k) {
            bool pending = false;
            unsigned long long *at = nullptr, X = 0, Y = 0, Z = 0, H = 0;
            if (k < nCams) {
                const DevCamera& K = J.cams[k];
                float4 co, cd, cx;
                if (makeConnection(K, 0u, vp, v.n, lam, v.beta, v.rho, vUp, co, cd, cx)) {
                    ++connections;
                    direct += atLight ? 1u : 0u;
                    Stack<SD, false, SPILL, 2 * kFlightThreads> stk{nullptr, (int*)(sStk + threadIdx.x), spill, 0};
                    if (!traceAny<SD, SPILL>(J.nodes, J.tris, prepareRay(xyz(co), xyz(cd)), kRayEps, co.w, stk, tc)) {
                        ++splats;
                        const unsigned pix = (unsigned)__float_as_int(cd.w);
                        X = min(toFixed((double)cx.x, K.filmScale), K.filmQmax);
                        Y = min(toFixed((double)cx.y, K.filmScale), K.filmQmax);
                        Z = min(toFixed((double)cx.z, K.filmScale), K.filmQmax);
                        H = (unsigned long long)vUp;
                        const int s = splatSlot<kFlightSlots>(sKey, ((unsigned long long)k << 32) | pix, kSplatProbe);
                        if (s >= 0) {
                            splatAdd(sVal, s, X, Y, Z, H);
                        } else {
                            pending = true;
                            at = (unsigned long long*)K.film + 4 * (size_t)pix;
                        }
                    }
                }
            }
            splatDirect(sStk, pending, at, X, Y, Z, H);
        }
    }
    auto add = [&](int k, unsigned long long x) {
        if (x) atomicAdd(&sAcc[k], x);
    };
    add(kAccEnergy + 0, emitted);
    add(kAccEnergy + 1, led[0]);
    add(kAccEnergy + 3, led[1]);
    add(kAccEnergy + 4, led[2]);
    add(kAccPhotons, photons);
    add(kAccDirect, direct);
    add(kAccSegments, segments);
    add(kAccConnections, connections);
    add(kAccSplats, splats);
    __syncthreads();
    if (threadIdx.x < kAccRow && sAcc[threadIdx.x])
        atomicAdd(J.acc + (size_t)(blockIdx.x % kSegs) * kAccRow + threadIdx.x, sAcc[threadIdx.x]);
    if (threadIdx.x == 0) atomicMax(&q.ctrl->iter, sLongest);
    flushSplats<kFlightSlots>(q.jobs, sKey, sVal);
}

// ------------------------------------------------------------------ mirrors
// Camera connections through flat mirrors (the reference's connectSpecularPlane,
// src/render.h:1334-1376, GPU twin src/render_cuda.cu:5004-5052). Mirroring the eye
// in the plane turns vertex -> mirror -> eye into the straight segment from the
// vertex to the eye's image, so the mirror point R is a plane intersection and the
// specular geometry factor is 1 / D^2 over the unfolded length D. The geometry is
// solved in double; the two legs are traced in float: the light side must be clear
// (any hit), and the eye's closest hit must be a mirror triangle at R (within
// 1e-4 (1 + |R - eye|)), whose reflectance tints the splat.
// One wave per workgroup, in two steps: the wave's lanes solve the geometry of their
// vertices against the scene's planes (outer) and the job's cameras (inner), most of which
// end there, and list the rest in LDS; 64 listed connections are then traced together. The
// two legs run on the lane's own stack column one after the other, as in k_flight, and
// splats go through its per-wave table. As one thread per vertex in 256-thread workgroups,
// solving and tracing under each other's masks with 199 registers and 52 KB of LDS (two
// waves per SIMD) and a film atomic per word, the mirror box (2^20 photons) spent 1370 us
// here, now 626 us.
struct MirrorSolve {
    double wP[3];       // vertex -> mirror point, unit
    double dP;          // vertex -> mirror point distance
    double wE[3];       // eye -> mirror point, unit
    double dE;          // eye -> mirror point distance
    double weight;      // (cos at the vertex / pi) / (D^2 * pixel solid angle)
    unsigned pix;       // film pixel of the mirror point
};

__device__ __forceinline__ bool solveMirror(const DevMirrorPlane& P, const DevCamera& K, const double p[3],
                                            const double np[3], MirrorSolve& o) {
    const double e[3] = {(double)K.eye[0], (double)K.eye[1], (double)K.eye[2]};
    const double pd = P.n[0] * p[0] + P.n[1] * p[1] + P.n[2] * p[2];
    const double se = (P.n[0] * e[0] + P.n[1] * e[1] + P.n[2] * e[2]) - P.d;
    const double sp = pd - P.d;
    if (!(se * sp > 0.0)) return false;   // eye and vertex on the same face
    double w[3];
    for (int a = 0; a < 3; ++a) w[a] = (e[a] - P.n[a] * (2.0 * se)) - p[a];
    const double D = sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
    if (D < 1e-9) return false;
    const double inv = 1.0 / D;
    for (int a = 0; a < 3; ++a) w[a] *= inv;
    const double cosSurf = np[0] * w[0] + np[1] * w[1] + np[2] * w[2];
    if (!(cosSurf > 0.0)) return false;
    const double denom = P.n[0] * w[0] + P.n[1] * w[1] + P.n[2] * w[2];
    if (fabs(denom) < 1e-12) return false;
    const double dP = (P.d - pd) / denom;
    if (dP <= 1e-7 || dP >= D - 1e-7) return false;
    double R[3];
    for (int a = 0; a < 3; ++a) {
        R[a] = p[a] + w[a] * dP;
        if (R[a] < P.lo[a] || R[a] > P.hi[a]) return false;
    }
    // pinhole projection of R (Camera::project / pixelSolidAngle)
    const double d[3] = {R[0] - e[0], R[1] - e[1], R[2] - e[2]};
    const double cz = d[0] * K.w[0] + d[1] * K.w[1] + d[2] * K.w[2];
    if (!(cz > 1e-9)) return false;
    const double ix = ((d[0] * K.u[0] + d[1] * K.u[1] + d[2] * K.u[2]) / cz) / (double)K.tanHalfX;
    const double iy = ((d[0] * K.v[0] + d[1] * K.v[1] + d[2] * K.v[2]) / cz) / (double)K.tanHalfY;
    if (!(ix >= -1.0 && ix < 1.0 && iy >= -1.0 && iy < 1.0)) return false;
    const int px = min(max((int)((ix * 0.5 + 0.5) * (double)K.resX), 0), K.resX - 1);
    const int py = min(max((int)((iy * 0.5 + 0.5) * (double)K.resY), 0), K.resY - 1);
    const double dist2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    const double cosCam = cz / sqrt(dist2);
    const double omega = (double)K.pixelArea * cosCam * cosCam * cosCam;
    if (!(omega > 0.0)) return false;
    const double dE = D - dP;
    for (int a = 0; a < 3; ++a) {
        o.wP[a] = w[a];
        o.wE[a] = (R[a] - e[a]) * (1.0 / dE);
    }
    o.dP = dP;
    o.dE = dE;
    o.weight = (cosSurf / 3.141592653589793) / (D * D * omega);
    o.pix = (unsigned)(py * K.resX + px);
    return true;
}

template <int SD, bool SPILL>
__global__ void __launch_bounds__(kFlightThreads, 4) k_mirror(Queues q) {
    static_assert(SD >= 5, "splatDirect stages five words per lane");
    __shared__ int2 sStk[SD * kFlightThreads];
    __shared__ unsigned long long sKey[kFlightSlots];
    __shared__ unsigned long long sVal[kFlightSlots * 4];
    __shared__ unsigned long long sCand[2 * kFlightThreads];   // vertex, plane << 32, camera << 40
    __shared__ unsigned cTab[kMaxJobs * 2];   // ray queries, splats (legs not in the statistics)
    clearSplats<kFlightSlots>(sKey, sVal);
    SegMap sm;
    const unsigned n = loadSegMap(q.ctrl->mirrorCount, q.mirrorSegCap, sm);
    const int nJobs = q.ctrl->nJobs;
    for (int r = threadIdx.x; r < nJobs * 2; r += kFlightThreads) cTab[r] = 0u;
    __syncthreads();
    TravCount<false> tc;
    const unsigned lane = threadIdx.x, stride = gridDim.x * kFlightThreads;
    int2* spill = SPILL ? q.spill + (size_t)(blockIdx.x * kFlightThreads + lane) * q.spillDepth : nullptr;
    auto vertexAt = [&](unsigned i, double p[3], double np[3]) -> unsigned {
        const float4 a = q.mv[0][i], b = q.mv[1][i];
        p[0] = (double)a.x; p[1] = (double)a.y; p[2] = (double)a.z;
        np[0] = (double)b.x; np[1] = (double)b.y; np[2] = (double)b.z;
        return (unsigned)__float_as_int(a.w);
    };
    unsigned held = 0;                               // listed connections
    unsigned base = blockIdx.x * kFlightThreads;     // this wave's vertices, plane and camera to solve
    int m = 0, k = 0;
    while (true) {
        while (held < kFlightThreads && base < n) {
            const unsigned li = base + lane;
            const unsigned i = sm.slot(li < n ? li : base);
            double p[3], np[3];
            const DevJob& J = q.jobs[vertexAt(i, p, np) & 0xffffu];
            const int nM = li < n ? J.nMirrors : 0, nC = J.nCams;
            MirrorSolve g;
            const bool ok = m < nM && k < nC && solveMirror(J.mirrors[m], J.cams[k], p, np, g);
            const unsigned long long mask = __ballot(ok);
            const unsigned rank = __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
            if (ok) sCand[held + rank] = i | ((unsigned long long)m << 32) | ((unsigned long long)k << 40);
            held += (unsigned)__popcll(mask);
            ++k;
            if (!__any(m < nM && k < nC)) {
                k = 0;
                ++m;
                if (!__any(m < nM)) {
                    m = 0;
                    base += stride;
                    if (base < stride) base = n;   // past 2^32
                }
            }
        }
        if (held == 0) break;
        __syncthreads();
        const unsigned count = min(held, (unsigned)kFlightThreads);
        bool pending = false;
        unsigned long long *at = nullptr, X = 0, Y = 0, Z = 0, H = 0;
        if (lane < count) {
            const unsigned long long cand = sCand[lane];
            const unsigned i = (unsigned)cand;
            const int cam = (int)(cand >> 40);
            double p[3], np[3];
            const unsigned tag = vertexAt(i, p, np);
            const int j = (int)(tag & 0xffffu);
            const DevJob& J = q.jobs[j];
            const DevCamera& K = J.cams[cam];
            MirrorSolve g;
            bool ok = solveMirror(J.mirrors[(cand >> 32) & 0xffu], K, p, np, g);   // solved before
            unsigned queries = 0;
            if (ok) {
                queries = 1;
                const F3 wl{(float)g.wP[0], (float)g.wP[1], (float)g.wP[2]};
                const F3 ol{(float)(p[0] + g.wP[0] * 1e-6), (float)(p[1] + g.wP[1] * 1e-6),
                            (float)(p[2] + g.wP[2] * 1e-6)};
                Stack<SD, false, SPILL, 2 * kFlightThreads> as{nullptr, (int*)(sStk + lane), spill, 0};
                ok = !traceAny<SD, SPILL>(J.nodes, J.tris, prepareRay(ol, wl), kRayEps,
                                          (float)((g.dP - 2e-6) - 1e-6), as, tc);
            }
            int tri = -1;
            if (ok) {
                ++queries;
                Stack<SD, true, SPILL, kFlightThreads> cs{sStk + lane, nullptr, spill, 0};
                float th = INFINITY;
                tri = traceClosest<SD, SPILL>(
                    J.nodes, J.tris, prepareRay(load3(K.eye), F3{(float)g.wE[0], (float)g.wE[1], (float)g.wE[2]}),
                    kRayEps, th, cs, tc);
                ok = tri >= 0 && !(fabs((double)th - g.dE) > 1e-4 * (1.0 + g.dE));
            }
            if (queries) atomicAdd(&cTab[2 * j], queries);
            if (ok) {
                const DevMaterial& M = J.mats[__float_as_int(J.trin[tri].w)];
                if (M.type == 2) {   // only Mirror is a planar mirror here
                    atomicAdd(&cTab[2 * j + 1], 1u);
                    const float4 l4 = q.mv[2][i], w4 = q.mv[3][i];
                    const float lam[kMaxHero] = {l4.x, l4.y, l4.z, l4.w};
                    const float bw[kMaxHero] = {w4.x, w4.y, w4.z, w4.w};
                    const int nUp = (int)((tag >> 16) & 7u);
                    double x = 0.0, y = 0.0, z = 0.0;
                    for (int c = 0; c < nUp; ++c) {
                        float r = specEval(M.reflect, lam[c]);
                        r = r < 0.0f ? 0.0f : (r > 1.0f ? 1.0f : r);
                        const double contrib = (double)bw[c] * g.weight * (double)r;
                        if (!(contrib > 0.0)) continue;
                        const F3 cw = cie(lam[c]);
                        x += (double)cw.x * contrib;
                        y += (double)cw.y * contrib;
                        z += (double)cw.z * contrib;
                        ++H;
                    }
                    if (H) {
                        X = min(toFixed(x, K.filmScale), K.filmQmax);
                        Y = min(toFixed(y, K.filmScale), K.filmQmax);
                        Z = min(toFixed(z, K.filmScale), K.filmQmax);
                        const unsigned long long key = ((unsigned long long)(j * kMaxCams + cam) << 32) | g.pix;
                        const int s = splatSlot<kFlightSlots>(sKey, key, kSplatProbe);
                        if (s >= 0) {
                            splatAdd(sVal, s, X, Y, Z, H);
                        } else {
                            pending = true;
                            at = (unsigned long long*)K.film + 4 * (size_t)g.pix;
                        }
                    }
                }
            }
        }
        __syncthreads();   // one wave: together again
        splatDirect(sStk, pending, at, X, Y, Z, H);
        held -= count;
        const unsigned long long rest = sCand[kFlightThreads + lane];
        __syncthreads();
        if (lane < held) sCand[lane] = rest;
        __syncthreads();
    }
    __syncthreads();
    AccAddr ca{q.jobs, kAccConnections};
    for (int r = threadIdx.x; r < nJobs * 2; r += kFlightThreads)
        if (cTab[r]) atomicAdd(ca(r / 2, r % 2), (unsigned long long)cTab[r]);
    flushSplats<kFlightSlots>(q.jobs, sKey, sVal);
}

// ------------------------------------------------------------------ ray binning
// Counting sort of queue `cur` into the binned queue by the 12-bit keys the emission
// and shading kernels stored (binKey). Column c (workgroup xcdBlock() of C = q.binCols) owns the
// contiguous logical range [n c / C, n (c + 1) / C). The order inside a (column,
// bin) run is that of LDS atomics; nothing downstream depends on it (films, ledgers
// and counters are integer sums).
// Histogram of column xcdBlock() into binHist[col][*].
__global__ void __launch_bounds__(kBinThreads) k_bin_count(Queues q, int cur) {
    __shared__ unsigned h[kBins];
    for (int b = threadIdx.x; b < kBins; b += blockDim.x) h[b] = 0u;
    __syncthreads();
    SegMap sm;
    const unsigned n = loadSegMap(q.ctrl->pathCount[cur], q.segCap, sm);
    const unsigned col = xcdBlock();
    unsigned lo, hi;
    binRange(n, col, (unsigned)q.binCols, lo, hi);
    const unsigned short* __restrict__ keys = q.key[cur];
    // the mask bounds the LDS index (keys have 12 bits; both passes read the same words)
    for (unsigned li = lo + threadIdx.x; li < hi; li += blockDim.x) atomicAdd(&h[keys[sm.slot(li)] & (kBins - 1)], 1u);
    __syncthreads();
    unsigned* out = q.binHist + (size_t)col * kBins;
    for (int b = threadIdx.x; b < kBins; b += blockDim.x) out[b] = h[b];
}

// Tables of one counting sort: hist[cols][kBins], chunk[kBinChunks][kBins], total[kBins].
struct BinTables {
    unsigned* hist;
    unsigned* chunk;
    unsigned* total;
    int cols;
};

// Per bin: exclusive prefix of the columns inside each of the kBinChunks column
// chunks (in place), the chunks' exclusive prefix (binChunk[chunk][bin]) and the
// bin's total (binTotal[bin]). A workgroup takes 32 bins x kBinChunks chunks at a
// time, grid-stride over the kBins / 32 groups.
__global__ void __launch_bounds__(256) k_bin_chunks(BinTables t) {
    const unsigned per = (unsigned)t.cols / kBinChunks;
    __shared__ unsigned part[kBinChunks][32];
    const unsigned bl = threadIdx.x & 31u, ch = threadIdx.x >> 5;
    for (unsigned grp = blockIdx.x; grp < kBins / 32; grp += gridDim.x) {
        const unsigned bin = grp * 32u + bl;
        unsigned run = 0;
        // eight columns loaded before any is rewritten, then the rest one at a time
        unsigned c = ch * per;
        const unsigned cEnd = (ch + 1) * per;
        for (; c + 8 <= cEnd; c += 8) {
            unsigned v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = t.hist[(size_t)(c + k) * kBins + bin];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                t.hist[(size_t)(c + k) * kBins + bin] = run;
                run += v[k];
            }
        }
        for (; c < cEnd; ++c) {
            unsigned* e = t.hist + (size_t)c * kBins + bin;
            const unsigned v = *e;
            *e = run;
            run += v;
        }
        part[ch][bl] = run;
        __syncthreads();
        if (ch == 0) {
            unsigned acc = 0;
            for (unsigned k = 0; k < kBinChunks; ++k) {
                t.chunk[(size_t)k * kBins + bin] = acc;
                acc += part[k][bl];
            }
            t.total[bin] = acc;
        }
        __syncthreads();
    }
}

// Exclusive scan of the kBins totals in place (one workgroup of 1024 threads).
constexpr int kBinScanThreads = kBins < 1024 ? kBins : 1024;
__global__ void __launch_bounds__(kBinScanThreads) k_bin_scan(BinTables bt) {
    constexpr int kPer = kBins / kBinScanThreads;
    __shared__ unsigned sum[kBinScanThreads];
    const unsigned t = threadIdx.x;
    unsigned v[kPer], acc = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        v[k] = bt.total[t * kPer + k];
        acc += v[k];
    }
    sum[t] = acc;
    __syncthreads();
    for (unsigned off = 1; off < kBinScanThreads; off <<= 1) {
        const unsigned add = t >= off ? sum[t - off] : 0u;
        __syncthreads();
        sum[t] += add;
        __syncthreads();
    }
    unsigned base = t ? sum[t - 1] : 0u;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        bt.total[t * kPer + k] = base;
        base += v[k];
    }
}

__device__ __forceinline__ void scatterWave(float4* __restrict__ out, float4* st, unsigned lane, unsigned dst,
                                            const float4& o, const float4& d, const float4& l, const float4& b,
                                            const uint4& s) {
    // Lane L stages its record at st[5 L ..]; then round k stores float4 64 k + L,
    // element e of record r = (64 k + L) / 5, at the destination of lane r: a store
    // instruction writes about 13 whole records (80 contiguous bytes each) instead of
    // one 16-byte piece of 64 records.
    st[5 * lane + 0] = o;
    st[5 * lane + 1] = d;
    st[5 * lane + 2] = l;
    st[5 * lane + 3] = b;
    st[5 * lane + 4] = bitcast4f(s);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (unsigned k = 0; k < 5; ++k) {
        const unsigned f = 64u * k + lane, r = f / 5u, e = f - 5u * r;
        const unsigned t = (unsigned)__shfl((int)dst, (int)r);
        const float4 v = st[f];
        if (t != ~0u) out[5 * (size_t)t + e] = v;
    }
    __builtin_amdgcn_wave_barrier();
}

// Moves column xcdBlock()'s paths to their bins' slots of the binned queue.
__global__ void __launch_bounds__(kBinThreads) k_bin_scatter(Queues q, int cur) {
    __shared__ unsigned slot[kBins];
    __shared__ float4 stage[kBinThreads / 64][5 * 64];
    const unsigned col = xcdBlock();
    const unsigned ch = col / ((unsigned)q.binCols / kBinChunks);
    const unsigned* colHist = q.binHist + (size_t)col * kBins;
    const unsigned* chunk = q.binChunk + (size_t)ch * kBins;
    for (int b = threadIdx.x; b < kBins; b += blockDim.x) slot[b] = q.binTotal[b] + chunk[b] + colHist[b];
    __syncthreads();
    SegMap sm;
    const unsigned n = loadSegMap(q.ctrl->pathCount[cur], q.segCap, sm);
    const unsigned room = kSegs * q.segCap;
    unsigned lo, hi;
    binRange(n, col, (unsigned)q.binCols, lo, hi);
    const unsigned short* __restrict__ keys = q.key[cur];
    const uint4* __restrict__ sst = q.st[cur];
    const float4* __restrict__ sro = q.ro[cur];
    const float4* __restrict__ srd = q.rd[cur];
    const float4* __restrict__ slam = q.lam[cur];
    const float4* __restrict__ sbeta = q.beta[cur];
    float4* __restrict__ out = q.pb;
    const unsigned lane = threadIdx.x & 63u;
    float4* st = stage[threadIdx.x >> 6];
    // two paths per lane and step, both loaded before either is stored; the loop is
    // wave-uniform (a lane past the end loads its wave's first path and stores nothing)
    for (unsigned wb = lo + (threadIdx.x & ~63u); wb < hi; wb += 2 * blockDim.x) {
        const unsigned li = wb + lane, lj = li + blockDim.x;
        const bool v0 = li < hi, v1 = lj < hi;
        const unsigned i0 = sm.slot(v0 ? li : wb), i1 = sm.slot(v1 ? lj : wb);
        const unsigned k0 = keys[i0] & (kBins - 1), k1 = keys[i1] & (kBins - 1);
        const uint4 s0 = sst[i0], s1 = sst[i1];
        const float4 o0 = sro[i0], o1 = sro[i1], d0 = srd[i0], d1 = srd[i1];
        const float4 l0 = slam[i0], l1 = slam[i1], b0 = sbeta[i0], b1 = sbeta[i1];
        unsigned t0 = v0 ? atomicAdd(&slot[k0], 1u) : ~0u;
        unsigned t1 = v1 ? atomicAdd(&slot[k1], 1u) : ~0u;
        if ((v0 && t0 >= room) || (v1 && t1 >= room)) {   // impossible: the two passes read the same keys
            q.ctrl->overflow = 1u;
            t0 = t0 >= room ? ~0u : t0;
            t1 = t1 >= room ? ~0u : t1;
        }
        scatterWave(out, st, lane, t0, o0, d0, l0, b0, s0);
        scatterWave(out, st, lane, t1, o1, d1, l1, b1, s1);
    }
}

// ------------------------------------------------------------------ probes
// One-wave workgroups and six waves per SIMD, as k_extend: 400,003 rays into a soup of
// 50,000 triangles take 549 us, 578 in 256-thread workgroups with 16 LDS entries (five waves,
// and a last round of workgroups that filled a quarter of the chip).
template <int SD, bool SPILL>
__global__ void __launch_bounds__(kExtendThreads, 6) k_probe_closest(const float4* nodes, const float4* tris,
                                                                    const float* rays, unsigned n, float tmin,
                                                                    int* prim, float* tout, int2* spill,
                                                                    int spillDepth) {
    __shared__ int2 sStk[SD * kExtendThreads];
    const unsigned stride = gridDim.x * blockDim.x, gtid = blockIdx.x * blockDim.x + threadIdx.x;
    Stack<SD, true, SPILL, kExtendThreads> stk{sStk + threadIdx.x, nullptr,
                                               SPILL ? spill + (size_t)gtid * spillDepth : nullptr, 0};
    for (unsigned i = gtid; i < n; i += stride) {
        const float* rp = rays + 6 * (size_t)i;
        RayPre r = prepareRay(F3{rp[0], rp[1], rp[2]}, F3{rp[3], rp[4], rp[5]});
        float tmax = INFINITY;
        TravCount<false> tc;
        int best = traceClosest<SD, SPILL>(nodes, tris, r, tmin, tmax, stk, tc);
        prim[i] = best >= 0 ? __float_as_int(tris[3 * best].w) : -1;
        tout[i] = best >= 0 ? tmax : INFINITY;
    }
}

template <int SD, bool SPILL>
__global__ void __launch_bounds__(kExtendThreads, 6) k_probe_any(const float4* nodes, const float4* tris,
                                                                const float* rays, const float* tmax, unsigned n,
                                                                float tmin, unsigned char* occ, int2* spill,
                                                                int spillDepth) {
    __shared__ int sStk[SD * kExtendThreads];
    const unsigned stride = gridDim.x * blockDim.x, gtid = blockIdx.x * blockDim.x + threadIdx.x;
    Stack<SD, false, SPILL, kExtendThreads> stk{nullptr, sStk + threadIdx.x,
                                                SPILL ? spill + (size_t)gtid * spillDepth : nullptr, 0};
    for (unsigned i = gtid; i < n; i += stride) {
        const float* rp = rays + 6 * (size_t)i;
        RayPre r = prepareRay(F3{rp[0], rp[1], rp[2]}, F3{rp[3], rp[4], rp[5]});
        TravCount<false> tc;
        occ[i] = traceAny<SD, SPILL>(nodes, tris, r, tmin, tmax[i], stk, tc) ? 1 : 0;
    }
}

// ------------------------------------------------------------------ job table
// Installs a job into slot a.slot: its record, photon range, emission state and zeroed
// ledger rows. A job without photons is complete once maxDepth iterations have run
// from now, like a job whose last photon was emitted in the current iteration.
__global__ void __launch_bounds__(256) k_install_job(Queues q, JobInstall a) {
    Ctrl* c = q.ctrl;
    const int slot = a.slot;
    if (threadIdx.x == 0) {
        const_cast<DevJob*>(q.jobs)[slot] = a.job;
        const_cast<DevCamera*>(a.job.cams)[0] = a.cam;
        c->nextPhoton[slot] = a.next;
        c->endPhoton[slot] = a.end;
        c->lastEmitIter[slot] = (a.end > a.next) ? -1 : (int)c->iter;
        c->active[slot] = 1;
    }
    for (int k = threadIdx.x; k < kSegs * kAccRow; k += blockDim.x) a.job.acc[k] = 0ull;
}

// Starts a trace: the control block, job slot 0, its cameras and zeroed ledger rows from
// the kernel's arguments (one launch instead of three copies and a fill). With `once` the
// whole budget fits the path queue: all photons are laid out over the segments as
// k_schedule would in iteration 0, and the later iterations need no k_schedule or k_emit.
__global__ void __launch_bounds__(256) k_start_trace(Queues q, TraceStart a) {
    Ctrl* c = q.ctrl;
    unsigned* words = (unsigned*)c;
    for (unsigned k = threadIdx.x; k < sizeof(Ctrl) / sizeof(unsigned); k += blockDim.x) words[k] = 0u;
    for (int k = threadIdx.x; k < kSegs * kAccRow; k += blockDim.x) a.job.acc[k] = 0ull;
    __syncthreads();
    c->lastEmitIter[threadIdx.x] = -1;
    if (threadIdx.x < (unsigned)a.nCams) const_cast<DevCamera*>(a.job.cams)[threadIdx.x] = a.cams[threadIdx.x];
    __syncthreads();
    if (threadIdx.x != 0) return;
    const_cast<DevJob*>(q.jobs)[0] = a.job;
    c->nJobs = 1;
    c->nOrder = 1;
    c->capacity = a.capacity;
    c->segCap = q.segCap;
    c->connSegCap = q.connSegCap;
    c->mirrorSegCap = q.mirrorSegCap;
    c->endPhoton[0] = a.photons;
    c->active[0] = 1;
    if (a.once) {
        const unsigned n = (unsigned)a.photons;
        unsigned placed = 0;
        for (int g = 0; g < kSegs; ++g) {
            const unsigned e = min(n - placed, q.segCap);
            c->segEmit[g] = placed;
            c->pathCount[0][g][0] = e;
            placed += e;
        }
        c->segEmit[kSegs] = placed;
        c->nEmit = n;
        c->emitPrefix[1] = n;
        c->nextPhoton[0] = a.photons;
        c->lastEmitIter[0] = 0;
        c->iter = 1;
    }
}

__global__ void __launch_bounds__(kMaxJobs) k_set_order(Queues q, OrderUpdate a) {
    Ctrl* c = q.ctrl;
    c->order[threadIdx.x] = a.order[threadIdx.x];
    if (threadIdx.x == 0) {
        c->nOrder = a.nOrder;
        c->nJobs = a.nJobs;
        if (a.clearSlot >= 0) c->active[a.clearSlot] = 0;
    }
}

__global__ void k_fill64(unsigned long long* p, size_t n, unsigned long long v) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// ------------------------------------------------------------------ launchers
// Launches on the sink's stream, or appends the kernel to its graph. The arguments are
// copied either way.
template <class... P, class... A>
static void enqueue(Sink& k, void (*kernel)(P...), dim3 grid, dim3 block, const A&... a) {
    if (!k.graph) {
        hipLaunchKernelGGL(kernel, grid, block, 0, k.stream, a...);
        return;
    }
    std::tuple<P...> args(a...);
    hipKernelNodeParams n{};
    n.func = (decltype(n.func))kernel;
    n.gridDim = grid;
    n.blockDim = block;
    hipGraphNode_t node = nullptr;
    const hipError_t e = std::apply(
        [&](P&... x) {
            void* at[] = {(void*)&x...};
            n.kernelParams = at;
            return hipGraphAddKernelNode(&node, k.graph, k.last ? &k.last : nullptr, k.last ? 1 : 0, &n);
        },
        args);
    if (e != hipSuccess) k.error = e;
    k.last = node;
}

void launchSchedule(const Queues& q, int cur, Sink& k) {
    enqueue(k, k_schedule, dim3(1), dim3(kMaxJobs), q, cur);
}
void launchEmit(const Queues& q, int cur, const LaunchShape& ls, Sink& k) {
    enqueue(k, k_emit, dim3(ls.emit), dim3(256), q, cur);
}
void launchShade(const Queues& q, int cur, const LaunchShape& ls, Sink& k) {
    if (q.binned) enqueue(k, k_shade<true>, dim3(ls.shade), dim3(kShadeThreads), q, cur);
    else enqueue(k, k_shade<false>, dim3(ls.shade), dim3(kShadeThreads), q, cur);
}
// Kernel instances by LDS stack depth and spill use.
#define GP_BY_STACK(LDS, SPILL, CALL) \
    do {                                   \
        if (SPILL) {                       \
            switch (LDS) {                 \
                case 8: CALL(8, true); break;   \
                case 24: CALL(24, true); break; \
                case 32: CALL(32, true); break; \
                default: CALL(16, true); break; \
            }                              \
        } else {                           \
            switch (LDS) {                 \
                case 8: CALL(8, false); break;   \
                case 24: CALL(24, false); break; \
                case 32: CALL(32, false); break; \
                default: CALL(16, false); break; \
            }                              \
        }                                  \
    } while (0)

// The closest-hit kernel also has a 12-entry stack (6 KB of LDS per one-wave
// workgroup: six waves per SIMD still fit): c2 closest-hit time 139.0 ms against 140.9
// at 8 entries, 176.7 against 191.6 in queue order.
#define GP_BY_STACK_EXT(LDS, SPILL, CALL)  \
    do {                                   \
        if ((LDS) == 12) {                 \
            if (SPILL) CALL(12, true);     \
            else CALL(12, false);          \
        } else {                           \
            GP_BY_STACK(LDS, SPILL, CALL); \
        }                                  \
    } while (0)

void launchExtend(const Queues& q, int cur, const LaunchShape& ls, Sink& k) {
    const dim3 grid(ls.extend);
#define GP_CALL(SD, SP) enqueue(k, k_extend<SD, SP, false, false>, grid, dim3(kExtendThreads), q, cur)
#define GP_CALLS(SD, SP) enqueue(k, k_extend<SD, SP, true, false>, grid, dim3(kExtendThreads), q, cur)
#define GP_CALLB(SD, SP) enqueue(k, k_extend<SD, SP, false, true>, grid, dim3(kExtendThreads), q, cur)
#define GP_CALLSB(SD, SP) enqueue(k, k_extend<SD, SP, true, true>, grid, dim3(kExtendThreads), q, cur)
    if (q.binned) {
        if (q.stats) GP_BY_STACK_EXT(q.lds, q.useSpill, GP_CALLSB);
        else GP_BY_STACK_EXT(q.lds, q.useSpill, GP_CALLB);
    } else {
        if (q.stats) GP_BY_STACK_EXT(q.lds, q.useSpill, GP_CALLS);
        else GP_BY_STACK_EXT(q.lds, q.useSpill, GP_CALL);
    }
#undef GP_CALLSB
#undef GP_CALLB
#undef GP_CALLS
#undef GP_CALL
}
void launchEmitOrder(const Queues& q, Sink& k) {
    static_assert(kEmitCols % kBinChunks == 0, "emission columns split into the scan's chunks");
    const BinTables bt{q.emitHist, q.emitChunk, q.emitTotal, kEmitCols};
    enqueue(k, k_emit_keys, dim3(kEmitCols), dim3(kBinThreads), q);
    enqueue(k, k_bin_chunks, dim3(kBins / 32), dim3(kBinChunks * 32), bt);
    enqueue(k, k_bin_scan, dim3(1), dim3(kBinScanThreads), bt);
    enqueue(k, k_emit_perm, dim3(kEmitCols), dim3(kBinThreads), q);
}
void launchBin(const Queues& q, int cur, Sink& k) {
    enqueue(k, k_bin_count, dim3(q.binCols), dim3(kBinThreads), q, cur);
    const BinTables bt{q.binHist, q.binChunk, q.binTotal, q.binCols};
    enqueue(k, k_bin_chunks, dim3(std::min(kBins / 32, q.binCols)), dim3(kBinChunks * 32), bt);
    enqueue(k, k_bin_scan, dim3(1), dim3(kBinScanThreads), bt);
    enqueue(k, k_bin_scatter, dim3(q.binCols), dim3(kBinThreads), q, cur);
}
void launchConnect(const Queues& q, const LaunchShape& ls, Sink& k) {
#define GP_CALL(SD, SP) enqueue(k, k_connect<SD, SP, false>, dim3(ls.connect), dim3(kTravThreads), q)
#define GP_CALLS(SD, SP) enqueue(k, k_connect<SD, SP, true>, dim3(ls.connect), dim3(kTravThreads), q)
    if (q.stats) GP_BY_STACK(q.connLds, q.connUseSpill, GP_CALLS);
    else GP_BY_STACK(q.connLds, q.connUseSpill, GP_CALL);
#undef GP_CALLS
#undef GP_CALL
}
void launchFlight(const Queues& q, unsigned n, unsigned lanes, int blocks, hipStream_t s) {
#define GP_CALL(SD, SP) hipLaunchKernelGGL((k_flight<SD, SP>), dim3(blocks), dim3(kFlightThreads), 0, s, q, n, lanes)
    GP_BY_STACK_EXT(q.lds, q.useSpill, GP_CALL);
#undef GP_CALL
}
void launchMirror(const Queues& q, const LaunchShape& ls, Sink& k) {
#define GP_CALL(SD, SP) enqueue(k, k_mirror<SD, SP>, dim3(ls.mirror), dim3(kFlightThreads), q)
    GP_BY_STACK(q.connLds, q.connUseSpill, GP_CALL);
#undef GP_CALL
}
void launchProbeClosest(const float4* nodes, const float4* tris, const float* rays, unsigned n, float tmin,
                        int* prim, float* t, int2* spill, int spillDepth, int lds, int blocks, hipStream_t s) {
#define GP_CALL(SD, SP) hipLaunchKernelGGL((k_probe_closest<SD, SP>), dim3(blocks), dim3(kExtendThreads), 0, s, nodes, tris, rays, n, tmin, prim, t, spill, spillDepth)
    GP_BY_STACK_EXT(lds, spillDepth > 0, GP_CALL);
#undef GP_CALL
}
void launchProbeAny(const float4* nodes, const float4* tris, const float* rays, const float* tmax, unsigned n,
                    float tmin, unsigned char* occ, int2* spill, int spillDepth, int lds, int blocks,
                    hipStream_t s) {
#define GP_CALL(SD, SP) hipLaunchKernelGGL((k_probe_any<SD, SP>), dim3(blocks), dim3(kExtendThreads), 0, s, nodes, tris, rays, tmax, n, tmin, occ, spill, spillDepth)
    GP_BY_STACK_EXT(lds, spillDepth > 0, GP_CALL);
#undef GP_CALL
}
#undef GP_BY_STACK
void launchInstallJob(const Queues& q, const JobInstall& a, hipStream_t s) {
    hipLaunchKernelGGL(k_install_job, dim3(1), dim3(256), 0, s, q, a);
}
void launchStartTrace(const Queues& q, const TraceStart& a, hipStream_t s) {
    static_assert(kMaxJobs == 256, "one thread per job slot");
    hipLaunchKernelGGL(k_start_trace, dim3(1), dim3(256), 0, s, q, a);
}
void launchSetOrder(const Queues& q, const OrderUpdate& a, hipStream_t s) {
    hipLaunchKernelGGL(k_set_order, dim3(1), dim3(kMaxJobs), 0, s, q, a);
}
void launchFill64(unsigned long long* p, size_t n, unsigned long long v, hipStream_t s) {
    if (n == 0) return;
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill64, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
}

}  // namespace gp
