// Device BVH builder (linear BVH, collapsed into four-wide nodes) and the device-side
// eye-to-scene distance used when the tree never exists on the host.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/goodphotons.h"

namespace gp {

struct DeviceBvh {
    float4* nodes = nullptr;   // nPairs four-wide nodes x 8 float4 (node i = pair node i collapsed)
    float4* tris = nullptr;    // 3 float4 per triangle, leaf order
    float4* trin = nullptr;    // normal + material per triangle, leaf order
    int64_t nPairs = 0;
    int depth = 0;             // pair nodes on the longest root-to-leaf path
    int stackNeed = 0;         // traversal stack bound: 3 per four-wide level
    double buildMs = 0.0;
};

// A caller's triangles on the device, as uploaded, and the bounds of their box centres.
struct DeviceTris {
    float* verts = nullptr;    // 9 floats per triangle; one allocation with mats behind it
    int32_t* mats = nullptr;
    int64_t n = 0;
    float centerLo[3] = {}, centerHi[3] = {};

    DeviceTris() = default;
    DeviceTris(const DeviceTris&) = delete;
    DeviceTris& operator=(const DeviceTris&) = delete;
    ~DeviceTris();
};

// Uploads and checks n triangles (GP_ERR_INVALID: a material id outside [0, nMats) or a
// vertex that is not finite) and reduces their bounds. Synchronous.
gp_status scanTrisDevice(const float* verts, const int32_t* mats, int64_t n, int nMats, DeviceTris& out);

// Synchronous.
gp_status buildBvhDevice(const DeviceTris& in, DeviceBvh& out);

// Smallest squared distance from p to any of n triangles (3 float4 each), in double.
gp_status deviceMinDistance2(const float4* dTris, int64_t n, const double p[3], double& d2);

}  // namespace gp
