// Plain-old-data layouts shared by the host runtime and the CDNA4 kernels.
// Everything the kernels read lives in HBM in these forms:
//   BVH        four-wide nodes, 128 B each (four slot boxes in SoA form + four links)
//   triangles  3 x float4 per triangle in leaf order (vertices; .w = prim id,
//              material id), plus 1 x float4 geometric normal (.w = material)
//   paths      structure-of-arrays queues of float4/uint4 (80 B per path), split
//              into kSegs segments, each with its own append counter
//   hits       one float2 per path (t, leaf-order triangle index)
//   camera     connections: 3 x float4 per record (48 B)
//   mirrors    vertices to connect through flat mirrors: 4 x float4 per record (64 B)
//   films      int64 fixed-point (X, Y, Z, hits) per pixel, 32 B
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace gp {

constexpr int kMaxHero = 4;           // wavelengths per path (hero + 3)
constexpr int kMaxJobs = 256;         // job slots in one wavefront
constexpr int kLambdaBins = 470;      // 1-nm bins over [360, 830)
constexpr int kCdfGuide = 64;         // guide-table cells over [0, 1) for the CDF inversion
constexpr float kRayEps = 1e-6f;      // origin offset and tmin, as the reference CPU path
constexpr int kLeafMax = 4;           // triangles per BVH leaf
// Queues are split into kSegs segments, each appended to through its own counter
// (its own 128-byte line): workgroup b appends to segment b % kSegs. Same-address
// atomics serialise (~12 ns each on MI355X), so eight counters instead of one cut
// the append cost of a launch eightfold; and because a segment only receives the
// items of every eighth workgroup, its fill is bounded without any assumption about
// where the hardware places workgroups.
constexpr int kSegs = 8;
constexpr int kLine = 32;             // u32 per 128-byte line
constexpr int kAccRow = 16;           // u64 per per-segment ledger/counter row
// Quantities of a per-job accumulator row (u64 index in the row).
constexpr int kAccEnergy = 0;         // emitted, absorbed, sensor, escaped, residual (fixed point)
constexpr int kAccPhotons = 5;        // photons emitted
constexpr int kAccDirect = 6;         // camera connections queued at the emission points
constexpr int kAccSegments = 7;       // closest-hit queries of the paths
constexpr int kAccNodeVisits = 8;     // their four-wide node visits (traversal statistics only)
constexpr int kAccTriTests = 9;       // their triangle tests (traversal statistics only)
constexpr int kAccConnections = 10;   // connection ray queries
constexpr int kAccSplats = 11;        // connections that reached the film
constexpr int kAccAnyNodeVisits = 12; // camera shadow rays' node visits (traversal statistics only)
constexpr int kAccAnyTriTests = 13;   // camera shadow rays' triangle tests (traversal statistics only)
constexpr int kAccCounters = 9;       // counters [kAccPhotons, kAccPhotons + kAccCounters)

// Ray binning (gp_tuning.ray_sort): before the closest-hit kernel, the paths of an
// iteration are reordered by a 12-bit key, the Morton code of the origin's cell in an
// 8 x 8 x 8 grid over the job's triangle-centroid box followed by the direction
// octant, so that the lanes of a wave trace similar rays.
// A counting sort: binCols workgroups (4 per CU, at most kBinCols) each count their
// contiguous share of the queue into a histogram column, the columns are scanned in
// (bin, column) order, and each workgroup scatters its share to the bins' ranges.
constexpr int kBinBits = 12;
constexpr int kBins = 1 << kBinBits;
constexpr int kBinCols = 1024;        // most histogram columns (workgroups of the count/scatter)
constexpr int kBinChunks = 8;         // column chunks per bin in the scan
constexpr int kBinColStep = 8;        // the column count is a multiple of this (and of kBinChunks)
constexpr int kBinThreads = 1024;     // threads of a count/scatter workgroup (one column)
constexpr int kBinCellsPerAxis = 8;
// Emission order: an iteration's new photons are emitted sorted by where they leave the
// light and in which direction (a counting sort over kBins keys in kEmitCols columns,
// one 1024-thread workgroup each), so that the lanes of a wave trace similar rays and the
// surface points they reach, with everything that starts there, stay close together.
// Whole renders, index order -> sorted: 5.24M-triangle icosphere (2^28 photons, 1024^2)
// 219.0 -> 204.0 ms, closest-hit kernel 147 -> 131; glass sphere and prism (2^26, 512^2)
// 66.9 -> 62.7 ms; the box (2^22) 4.73 -> 4.64 ms.
// The four sorting kernels take about 35 us in an iteration that emits and 12 us in one that
// does not. A trace of one refill is sorted once: from kEmitOrderJobMin photons on it gains
// or, on the box, costs 1%; fewer photons fly. Index order -> sorted, ms:
//   photons              2^19           2^20           2^21           2^22
//   box                  1.00 -> 1.01   1.32 -> 1.29   1.97 -> 1.90   3.38 -> 3.23
//   glass, prism         2.71 -> 2.44   2.87 -> 2.77   3.89 -> 3.57   5.73 -> 5.08
//   soup 100K tri.       5.00 -> 4.91   5.83 -> 5.75   7.45 -> 7.19   10.5 -> 10.0
//   icosphere 1.3M       3.04 -> 3.07   3.45 -> 3.37   4.11 -> 3.89   5.45 -> 4.99
// A server runs them in every iteration of a chunk, so the photons of all its jobs have to
// pay for those that emit nothing. Sorted / index order over five scenes and depths of 3, 8
// and 16, mean (least .. most):
//   one job     2^19 1.09 (1.02 .. 1.17)   2^20 1.06 (1.01 .. 1.15)   2^21 1.01 (0.95 .. 1.10)
//   four jobs   2^19 1.03 (0.99 .. 1.12)   2^20 0.99 (0.91 .. 1.07)
//   in all      3 * 2^20 1.00 (0.92 .. 1.09)   2^22 0.98 (0.90 .. 1.06)
// hence kEmitOrderServerMin; sixteen jobs of 2^18, as many photons, gain nothing (1.005).
// Refills of fewer than kEmitOrderMin (a few photons to each of the 4096 keys) keep index
// order. The macros let a CPU test sort a few thousand photons.
#ifndef GP_EMIT_COLS
#define GP_EMIT_COLS 256
#define GP_EMIT_ORDER_MIN (1u << 16)
#define GP_EMIT_ORDER_JOB_MIN (1u << 19)
#define GP_EMIT_ORDER_SERVER_MIN (1u << 22)
#endif
constexpr int kEmitCols = GP_EMIT_COLS;
constexpr unsigned kEmitOrderMin = GP_EMIT_ORDER_MIN;
constexpr uint64_t kEmitOrderJobMin = GP_EMIT_ORDER_JOB_MIN;         // the trace, or a server's largest job
constexpr uint64_t kEmitOrderServerMin = GP_EMIT_ORDER_SERVER_MIN;   // a server's jobs in all

// A trace that the chip holds at once flies (k_flight) instead of running the wavefront.
// kFlightWaves: resident waves of k_flight per CU. Per-trace times, wavefront -> flight, on
// 256 CUs (262144 resident lanes), us:
//   photons         4096          65536         262144        393216        524445
//   box             501 -> 231    550 -> 327    668 -> 461    768 -> 765    869 -> 903
//   glass, prism    1288 -> 372   1644 -> 646   1856 -> 892   1962 -> 1262  2078 -> 1497
//   soup 100K tri.  2509 -> 525   3659 -> 1103  4133 -> 1507  4245 -> 2251  4412 -> 2634
//   icosphere 1.3M  2181 -> 515   3366 -> 907   3905 -> 1252  4070 -> 1838  4277 -> 1929
// so a box loses past one and a half photons per lane.
// Several cameras: a lane traces its vertex to one after the other, while the wavefront's
// k_connect gets them all at once. How soon that loses depends on what an iteration costs the
// wavefront: little in a small tree (box, 8 segments deep):
//   cameras, photons    3, 65536      4, 30000      6, 4096       6, 30000      16, 4096
//                       618 -> 542    618 -> 550    601 -> 547    669 -> 775    843 -> 1307
// more in a deep one, where paths of few segments do not fill it and lose (soup of 100K):
//   cameras, photons    6, 12000      12, 4096      12, 30000     16, 30000
//   3 segments          1684 -> 1391  1802 -> 1704  1871 -> 3269  1913 -> 4048
//   8 segments          3588 -> 1601  3366 -> 2606  4200 -> 4210  4356 -> 5019
// Over 1 to 16 cameras, 1 to 16 segments, 1000 to 393216 photons and six scenes (36 triangles
// to 1.3 M) no trace that flies by the rule takes longer than the wavefront did when each
// camera's connections were appended by an atomic of their own (0.99 at most); a few of one to
// three segments take up to 1.36 times what today's takes. Paths of up to 16 segments move the
// limits by up to twice, as they cost the wavefront twice the iterations. Left out: deep trees of which
// little is seen (the icosphere gains up to 4x with 8 to 16 cameras past the limit), which
// nothing known before a trace tells from the soup.
constexpr int kFlightWaves = 16;
constexpr int kFlightSmallTree = 12;   // stack entries (four levels of the four-wide tree)
inline bool flightFits(uint64_t photons, int cams, int stackNeed, int maxDepth, int cus) {
    const double n = (double)photons, c = cams, lanes = (double)cus * kFlightWaves * 64;
    const double more = std::min(std::max(maxDepth, 8), 16) / 8.0;
    if (n * (2.0 + c) > 4.5 * lanes) return false;   // one camera: 1.5 photons a lane
    if (stackNeed <= kFlightSmallTree) return cams <= 6 && n * c * std::sqrt(c) <= 1.5 * lanes * more;
    if (maxDepth < 8) return n * c * c * c * std::sqrt(c) <= 24.0 * lanes;
    return n * std::pow(c, 1.75) <= 7.0 * lanes * more;
}

// Leaf links are negative: ~((first << 3) | (count - 1)).
inline constexpr int leafCode(int first, int count) { return ~((first << 3) | (count - 1)); }

struct DevSpectrum {
    int32_t kind;
    int32_t n;           // sampled: number of samples
    const float* tab;    // sampled: the samples (the scene's device table)
    float p[6];          // sampled: p[0] first sample's wavelength, p[1] samples per nm
    float band_lo, band_hi;
};  // 48 B

struct DevMaterial {
    int32_t type;
    float roughness;
    int32_t pad[2];
    DevSpectrum reflect;
    DevSpectrum ior;
};  // 112 B

struct DevEmitter {
    float origin[3], u[3], v[3], normal[3], beam[3];
    int32_t collimated;
    float power;        // integral(SPD) * area * pi
    int32_t pad;
    const double* cdf;  // kLambdaBins + 1 entries, normalised
    const int32_t* guide;  // kCdfGuide + 1 entries: guide[k] = last bin with cdf <= k / kCdfGuide
};

constexpr int kMaxCams = 16;          // cameras one job splats into (shared photon flight)
constexpr int kMaxMirrorPlanes = 64;  // flat mirror surfaces one scene connects through

// One flat mirror surface: the coplanar mirror triangles of a plane, reduced to the
// plane (unit normal n, dot(n, x) = d) and the padded box of its triangles. The
// connection geometry is solved in double, so the plane is stored in double.
struct DevMirrorPlane {
    double n[3];
    double d;
    double lo[3], hi[3];
};  // 80 B

// Pinhole camera and the film it splats into (Camera::lookAt basis, float).
struct DevCamera {
    float eye[3], u[3], v[3], w[3];
    float tanHalfX, tanHalfY, pixelArea;
    int32_t resX, resY;
    int32_t pad;
    long long* film;             // res*4 int64
    double filmScale;            // contribution -> integer units
    unsigned long long filmQmax; // saturation value of one splat
};

// One job = one (scene, cameras + films, photon budget). A single gp_trace is one job;
// the batched and serving paths run many jobs in the same queues. Every photon of a
// job connects to each of its cameras.
struct DevJob {
    // scene
    const float4* nodes;
    const float4* tris;
    const float4* trin;
    const DevMaterial* mats;
    const DevEmitter* ems;
    const double* emCdf;     // power CDF over emitters (n_em entries)
    int32_t nEm;
    float basePower;         // photon power: the single emitter's, else the total
    // cameras
    const DevCamera* cams;   // nCams entries
    int32_t nCams;
    int32_t nMirrors;        // flat mirror planes of the scene (0: no mirror connections)
    const DevMirrorPlane* mirrors;
    // kSegs rows of kAccRow u64 (layout: the kAcc* indices above); workgroup b adds
    // into row b % kSegs
    unsigned long long* acc;
    double energyScale;
    // path settings
    unsigned long long seedBase, salt;
    int32_t heroC, maxDepth, rrDepth, pad0;
    // ray binning: origin cell = (o - binLo) * binScale, clamped to the grid
    float binLo[3], binScale[3];
};

// Connection tag (float bits of the record's 4th word): job slot in bits 0..15,
// live wavelengths in 16..18, camera in 19..22.
inline constexpr unsigned connTag(unsigned job, unsigned nUp, unsigned cam) {
    return job | (nUp << 16) | (cam << 19);
}

// Device-side wavefront control block.
struct Ctrl {
    unsigned int pathCount[2][kSegs][kLine];   // per segment of path queue 0 / 1 (one line each)
    unsigned int connCount[kSegs][kLine];      // per segment of the connection queue
    unsigned int mirrorCount[kSegs][kLine];    // per segment of the mirror-vertex queue
    unsigned int nEmit;         // photons emitted this iteration
    unsigned int iter;          // iterations run
    int32_t nJobs;              // job slots in use are below this
    unsigned int capacity;      // path queue capacity (total over segments)
    unsigned int segCap;        // path slots per segment
    unsigned int connSegCap;    // connection slots per segment
    unsigned int overflow;      // set by a kernel that found a segment full (never expected)
    unsigned int mirrorSegCap;  // mirror-vertex slots per segment
    unsigned int segBase[kSegs];        // survivors already in each segment (emission goes after)
    unsigned int segEmit[kSegs + 1];    // prefix of this iteration's emission over segments
    unsigned int pad2[7];
    // per job
    unsigned long long nextPhoton[kMaxJobs];   // next photon index to emit (job-relative)
    unsigned long long endPhoton[kMaxJobs];    // one past the last photon
    int32_t lastEmitIter[kMaxJobs];            // iteration that emitted the job's last photon
    int32_t active[kMaxJobs];                  // 1 = emitting / in flight
    int32_t order[kMaxJobs];                   // job slots in emission priority order
    int32_t nOrder;                            // entries of `order` in use
    int32_t pad3[3];
    // this iteration's emission, indexed by position k in `order`
    unsigned int emitPrefix[kMaxJobs + 1];     // prefix of photons emitted before order[k]
    int32_t emitJob[kMaxJobs];                 // = order[k]
    unsigned long long emitStart[kMaxJobs];    // first photon index emitted for order[k]
};

// Path metadata word (uint4.w of the state array).
//   bits  0..15 job slot, 16..23 bounce, 24..26 live wavelengths, 31 dead
inline constexpr unsigned packMeta(unsigned job, unsigned bounce, unsigned nUp) {
    return job | (bounce << 16) | (nUp << 24);
}

}  // namespace gp
