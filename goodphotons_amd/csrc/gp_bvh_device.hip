// Device BVH builder: a linear BVH (Karras, "Maximizing parallelism in the
// construction of BVHs, octrees, and k-d trees", HPG 2012) emitted in the child-pair
// layout and collapsed into the four-wide nodes the traversal reads.
//
// The vertices and material ids are uploaded as the caller holds them; one kernel checks
// them and reduces the bounds of the box centres (scanTrisDevice), and the tree's kernels
// read them from there.
//
//   1. Morton code (21 bits per axis) of each triangle's box centre in the scene's
//      centre bounds; sort (code, index) pairs (rocPRIM radix sort).
//   2. One thread per internal node i finds the sorted range it covers and its split
//      from the longest common prefixes of neighbouring codes (equal codes are told
//      apart by their positions, so the tree is a valid binary tree for any input).
//   3. Every node covers a contiguous sorted range, so its box is the union of a few
//      entries of a binary tree of boxes over the sorted leaves (a segment tree built a
//      workgroup at a time): no node waits for its children.
//   4. Every internal node whose range holds more than kLeafMax primitives becomes a
//      pair node; a child with at most kLeafMax primitives becomes a leaf over its
//      contiguous sorted range. Triangles are gathered into sorted (leaf) order,
//      with their normals.
//   5. Pair node i becomes four-wide node i, whose slots are its grandchildren (a
//      leaf child keeps its own slot), so links keep their indices; the root is
//      node 0, and nodes at odd pair levels are built but never reached.
//
// Boxes are padded and rounded outward exactly like the host builder's (1e-6 pad),
// so traversal stays conservative; closest-hit results do not depend on the tree.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <cstring>

#include "gp_bvh_device.hpp"
#include "gp_runtime.hpp"

namespace gp {
namespace {

constexpr double kPadD = 1e-6;

struct KNode {
    int left, right;     // child index; leaf children are encoded as -(k + 1)
    int first, last;     // sorted primitive range
};

__device__ __forceinline__ unsigned long long spread21(unsigned v) {
    unsigned long long x = v & 0x1fffffu;
    x = (x | (x << 32)) & 0x1f00000000ffffull;
    x = (x | (x << 16)) & 0x1f0000ff0000ffull;
    x = (x | (x << 8)) & 0x100f00f00f00f00full;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}

// Outward rounding of a double to float (as the host builder's down()/up()).
__device__ __forceinline__ float roundDown(double v) {
    float f = (float)v;
    return ((double)f > v) ? nextafterf(f, -FLT_MAX) : f;
}
__device__ __forceinline__ float roundUp(double v) {
    float f = (float)v;
    return ((double)f < v) ? nextafterf(f, FLT_MAX) : f;
}

// Padded box of input triangle t (nine floats per triangle, input order).
__device__ __forceinline__ void triBox(const float* __restrict__ verts, int t, float lo[3], float hi[3]) {
    const float* v = verts + 9 * (size_t)t;
    for (int k = 0; k < 3; ++k) {
        const double l = fmin(fmin((double)v[k], (double)v[3 + k]), (double)v[6 + k]) - kPadD;
        const double h = fmax(fmax((double)v[k], (double)v[3 + k]), (double)v[6 + k]) + kPadD;
        lo[k] = roundDown(l);
        hi[k] = roundUp(h);
    }
}

// Unsigned words that order like the floats.
__device__ __forceinline__ unsigned orderedBits(float f) {
    const unsigned u = (unsigned)__float_as_int(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Checks the triangles and reduces the bounds of their box centres into out[7] (zeroed):
// maxima of the complemented ordered lower bounds, of the ordered upper bounds, and flags
// (1: a material id out of range, 2: a vertex that is not finite). Reads 40 bytes a
// triangle once. The host loops over the same data, with the 64 bytes a triangle that they
// prepared and uploaded, took 8 of the 12.7 ms of a 400,000-triangle rebuild. At most 256
// workgroups, so that the seven same-address atomics of each stay under 20 us.
__global__ void __launch_bounds__(256) k_scan_tris(const float* __restrict__ verts, const int* __restrict__ mats,
                                                   size_t n, int nMats, unsigned* __restrict__ out) {
    __shared__ unsigned red[7];
    if (threadIdx.x < 7) red[threadIdx.x] = 0u;
    __syncthreads();
    unsigned r[6] = {0u, 0u, 0u, 0u, 0u, 0u}, flags = 0u;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += stride) {
        const float* v = verts + 9 * t;
        const int m = mats[t];
        if (m < 0 || m >= nMats) flags |= 1u;
        for (int k = 0; k < 3; ++k) {
            const float a = v[k], b = v[3 + k], c = v[6 + k];
            if (!(fabsf(a) <= FLT_MAX && fabsf(b) <= FLT_MAX && fabsf(c) <= FLT_MAX)) flags |= 2u;
            const float ctr = 0.5f * (fminf(fminf(a, b), c) + fmaxf(fmaxf(a, b), c));
            const unsigned u = orderedBits(ctr);
            r[k] = max(r[k], ~u);
            r[3 + k] = max(r[3 + k], u);
        }
    }
    for (int k = 0; k < 6; ++k) atomicMax(&red[k], r[k]);
    if (flags) atomicOr(&red[6], flags);
    __syncthreads();
    if (threadIdx.x < 6) atomicMax(&out[threadIdx.x], red[threadIdx.x]);
    if (threadIdx.x == 6 && red[6]) atomicOr(&out[6], red[6]);
}

__global__ void k_morton(const float* __restrict__ verts, int n, float3 lo, float3 inv,
                         unsigned long long* __restrict__ keys, unsigned* __restrict__ vals) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float bl[3], bh[3];
    triBox(verts, i, bl, bh);
    const float cx = 0.5f * (bl[0] + bh[0]), cy = 0.5f * (bl[1] + bh[1]), cz = 0.5f * (bl[2] + bh[2]);
    auto q = [](float c, float l, float s) {
        float u = (c - l) * s;
        u = fminf(fmaxf(u, 0.0f), 1.0f);
        return (unsigned)fminf(u * 2097152.0f, 2097151.0f);
    };
    const unsigned ux = q(cx, lo.x, inv.x), uy = q(cy, lo.y, inv.y), uz = q(cz, lo.z, inv.z);
    keys[i] = (spread21(ux) << 2) | (spread21(uy) << 1) | spread21(uz);
    vals[i] = (unsigned)i;
}

// longest common prefix of sorted keys i and j (positions break ties), -1 outside
__device__ __forceinline__ int lcp(const unsigned long long* __restrict__ k, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    const unsigned long long a = k[i], b = k[j];
    if (a == b) return 64 + __clz((unsigned)(i ^ j));
    return __clzll(a ^ b);
}

__global__ void k_karras(const unsigned long long* __restrict__ keys, int n, KNode* __restrict__ nodes,
                         int* __restrict__ parent) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int d = (lcp(keys, n, i, i + 1) - lcp(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = lcp(keys, n, i, i - d);
    long long lmax = 2;
    while (lcp(keys, n, i, (int)(i + lmax * d)) > dmin) lmax <<= 1;
    long long l = 0;
    for (long long t = lmax >> 1; t >= 1; t >>= 1)
        if (lcp(keys, n, i, (int)(i + (l + t) * d)) > dmin) l += t;
    const int j = (int)(i + l * d);
    const int dnode = lcp(keys, n, i, j);
    long long s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (lcp(keys, n, i, (int)(i + (s + t) * d)) > dnode) s += t;
    } while (t > 1);
    const int gamma = (int)(i + s * d) + min(d, 0);
    KNode nd;
    nd.first = min(i, j);
    nd.last = max(i, j);
    if (nd.first == gamma) {
        nd.left = -(gamma + 1);
    } else {
        nd.left = gamma;
        parent[gamma] = i;
    }
    if (nd.last == gamma + 1) {
        nd.right = -(gamma + 2);
    } else {
        nd.right = gamma + 1;
        parent[gamma + 1] = i;
    }
    if (i == 0) parent[0] = -1;   // the root is no node's child
    nodes[i] = nd;
}

// box[6] of every sorted leaf
__global__ void k_leaf_boxes(const float* __restrict__ verts, const unsigned* __restrict__ order, int n,
                             float* __restrict__ leafBox) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    float lo[3], hi[3];
    triBox(verts, (int)order[k], lo, hi);
    for (int a = 0; a < 3; ++a) {
        leafBox[6 * (size_t)k + a] = lo[a];
        leafBox[6 * (size_t)k + 3 + a] = hi[a];
    }
}

// Binary tree of boxes over the sorted leaves: entry i of level k is the union of the
// leaves [i 2^k, (i + 1) 2^k) below n. Level 0 is leafBox; level k >= 1 starts at off[k].
constexpr int kMaxLevels = 30;   // triangles < 2^28
struct BoxLevels {
    unsigned size[kMaxLevels];
    unsigned off[kMaxLevels];
    int count;
};

__device__ __forceinline__ void growBox(float b[6], const float* __restrict__ p) {
    for (int a = 0; a < 3; ++a) {
        b[a] = fminf(b[a], p[a]);
        b[3 + a] = fmaxf(b[3 + a], p[3 + a]);
    }
}

// Levels base + 1 .. base + kBoxStep from level `base`: a workgroup folds 2^kBoxStep
// entries, level by level, through LDS.
constexpr int kBoxStep = 9;
__global__ void __launch_bounds__(1 << (kBoxStep - 1)) k_box_levels(BoxLevels L, int base,
                                                                  const float* __restrict__ leafBox,
                                                                  float* __restrict__ up) {
    __shared__ float sh[1 << (kBoxStep - 1)][6];
    const float* src = base ? up + 6 * (size_t)L.off[base] : leafBox;
    const unsigned t = threadIdx.x;
    for (int s = 1; s <= kBoxStep && base + s < L.count; ++s) {
        const unsigned width = 1u << (kBoxStep - s);          // entries of level base + s here
        const unsigned e = blockIdx.x * width + t;            // entry of that level
        const bool have = t < width && e < L.size[base + s];
        float b[6];
        if (have) {
            const bool two = 2 * e + 1 < L.size[base + s - 1];
            const float* l = s == 1 ? src + 12 * (size_t)e : sh[2 * t];
            for (int a = 0; a < 6; ++a) b[a] = l[a];
            if (two) growBox(b, s == 1 ? l + 6 : sh[2 * t + 1]);
        }
        __syncthreads();   // the level below is read
        if (have) {
            float* o = up + 6 * (size_t)(L.off[base + s] + e);
            for (int a = 0; a < 6; ++a) { sh[t][a] = b[a]; o[a] = b[a]; }
        }
        __syncthreads();
    }
}

// Box of every internal node: the union over its sorted range, at most two entries of
// each level. A climb from the leaves in which the second child to arrive merges the boxes
// needs a device-wide fence at each node, which writes back an XCD's whole L2: 2500 us for
// 400,000 triangles, against 14 us for this, 17 us for the levels and 28 us for k_height.
__global__ void k_node_boxes(BoxLevels L, const KNode* __restrict__ nodes, int nInner,
                             const float* __restrict__ leafBox, const float* __restrict__ up,
                             float* __restrict__ box) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nInner) return;
    const KNode nd = nodes[i];
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    unsigned l = (unsigned)nd.first, r = (unsigned)nd.last + 1u;
    for (int k = 0; l < r; ++k, l >>= 1, r >>= 1) {
        const float* lev = k ? up + 6 * (size_t)L.off[k] : leafBox;
        if (l & 1u) growBox(b, lev + 6 * (size_t)l++);
        if (r & 1u) growBox(b, lev + 6 * (size_t)--r);
    }
    for (int a = 0; a < 6; ++a) box[6 * (size_t)i + a] = b[a];
}

// Pair-node levels of the tree: the longest chain of ancestors above a pair node without
// pair-node children. height[0] (zeroed) receives the maximum.
__global__ void __launch_bounds__(256) k_height(const KNode* __restrict__ nodes, const int* __restrict__ parent,
                                                int nInner, int* __restrict__ height) {
    __shared__ int best;
    if (threadIdx.x == 0) best = 0;
    __syncthreads();
    auto isPair = [&](int c) { return c >= 0 && nodes[c].last - nodes[c].first + 1 > kLeafMax; };
    int mine = 0;
    const int stride = (int)(gridDim.x * blockDim.x);
    for (int64_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nInner; i += stride) {
        const KNode nd = nodes[i];
        if (nd.last - nd.first + 1 <= kLeafMax || isPair(nd.left) || isPair(nd.right)) continue;
        int h = 0;
        for (int p = (int)i; p >= 0; p = parent[p]) ++h;
        mine = max(mine, h);
    }
    if (mine) atomicMax(&best, mine);
    __syncthreads();
    if (threadIdx.x == 0 && best) atomicMax(height, best);
}

__device__ __forceinline__ int childLink(const KNode* __restrict__ nodes, int c) {
    if (c < 0) return leafCode(-c - 1, 1);
    const KNode cn = nodes[c];
    const int cnt = cn.last - cn.first + 1;
    return cnt <= kLeafMax ? leafCode(cn.first, cnt) : c;
}

__global__ void k_emit_pairs(const KNode* __restrict__ nodes, int n, const float* __restrict__ leafBox,
                             const float* __restrict__ box, float4* __restrict__ pairs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const KNode nd = nodes[i];
    if (nd.last - nd.first + 1 <= kLeafMax) return;   // collapsed into its parent's leaf
    const float* bl = nd.left < 0 ? leafBox + 6 * (size_t)(-nd.left - 1) : box + 6 * (size_t)nd.left;
    const float* br = nd.right < 0 ? leafBox + 6 * (size_t)(-nd.right - 1) : box + 6 * (size_t)nd.right;
    const int ll = childLink(nodes, nd.left), rl = childLink(nodes, nd.right);
    float4* q = pairs + 4 * (size_t)i;
    q[0] = make_float4(bl[0], bl[1], bl[2], __int_as_float(ll));
    q[1] = make_float4(bl[3], bl[4], bl[5], __int_as_float(rl));
    q[2] = make_float4(br[0], br[1], br[2], 0.0f);
    q[3] = make_float4(br[3], br[4], br[5], 0.0f);
}

// Four-wide node i from pair node i (see step 5; the layout is collapse4's in
// gp_bvh.hpp). `nodes` is null for the single pair of a lone leaf.
__global__ void k_collapse4(const KNode* __restrict__ nodes, int nInner, const float4* __restrict__ pairs,
                            float4* __restrict__ quads) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nInner) return;
    if (nodes) {
        const KNode nd = nodes[i];
        if (nd.last - nd.first + 1 <= kLeafMax) return;   // no pair node here
    }
    float lo[3][4], hi[3][4];
    int link[4];
    int n = 0;
    for (int side = 0; side < 2; ++side) {
        const float4* p = pairs + 4 * (size_t)i;
        const float4 a = side ? p[2] : p[0], b = side ? p[3] : p[1];
        const int c = __float_as_int(side ? p[1].w : p[0].w);
        if (c < 0) {
            lo[0][n] = a.x; lo[1][n] = a.y; lo[2][n] = a.z;
            hi[0][n] = b.x; hi[1][n] = b.y; hi[2][n] = b.z;
            link[n++] = c;
        } else {
            const float4* q = pairs + 4 * (size_t)c;
            for (int g = 0; g < 2; ++g) {
                const float4 ga = g ? q[2] : q[0], gb = g ? q[3] : q[1];
                lo[0][n] = ga.x; lo[1][n] = ga.y; lo[2][n] = ga.z;
                hi[0][n] = gb.x; hi[1][n] = gb.y; hi[2][n] = gb.z;
                link[n++] = __float_as_int(g ? q[1].w : q[0].w);
            }
        }
    }
    for (int k = n; k < 4; ++k) {   // unused slot: far point box, linked to slot 0
        for (int a = 0; a < 3; ++a) { lo[a][k] = 1e30f; hi[a][k] = 1e30f; }
        link[k] = link[0];
    }
    float4* o = quads + 8 * (size_t)i;
    for (int a = 0; a < 3; ++a) {
        o[2 * a] = make_float4(lo[a][0], lo[a][1], lo[a][2], lo[a][3]);
        o[2 * a + 1] = make_float4(hi[a][0], hi[a][1], hi[a][2], hi[a][3]);
    }
    o[6] = make_float4(__int_as_float(link[0]), __int_as_float(link[1]), __int_as_float(link[2]),
                       __int_as_float(link[3]));
    o[7] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// a scene of <= kLeafMax triangles: one leaf, tested through a pair with itself
__global__ void k_lone_leaf(const float* __restrict__ leafBox, int n, float4* __restrict__ pairs) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (int k = 0; k < n; ++k)
        for (int a = 0; a < 3; ++a) {
            lo[a] = fminf(lo[a], leafBox[6 * k + a]);
            hi[a] = fmaxf(hi[a], leafBox[6 * k + 3 + a]);
        }
    const int code = leafCode(0, n);
    pairs[0] = make_float4(lo[0], lo[1], lo[2], __int_as_float(code));
    pairs[1] = make_float4(hi[0], hi[1], hi[2], __int_as_float(code));
    pairs[2] = make_float4(lo[0], lo[1], lo[2], 0.0f);
    pairs[3] = make_float4(hi[0], hi[1], hi[2], 0.0f);
}

// Triangles and their geometric normals in sorted order, from the input arrays (the
// normal as the host builder's scene upload computes it: in double, no contraction).
__global__ void k_gather(const float* __restrict__ verts, const int* __restrict__ mats,
                         const unsigned* __restrict__ order, int n, float4* __restrict__ tris,
                         float4* __restrict__ trin) {
#pragma clang fp contract(off)
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int t = (int)order[k];
    const float* v = verts + 9 * (size_t)t;
    const float mat = __int_as_float(mats[t]);
    tris[3 * (size_t)k + 0] = make_float4(v[0], v[1], v[2], __int_as_float(t));
    tris[3 * (size_t)k + 1] = make_float4(v[3], v[4], v[5], mat);
    tris[3 * (size_t)k + 2] = make_float4(v[6], v[7], v[8], 0.f);
    const double e1[3] = {(double)v[3] - v[0], (double)v[4] - v[1], (double)v[5] - v[2]};
    const double e2[3] = {(double)v[6] - v[0], (double)v[7] - v[1], (double)v[8] - v[2]};
    double c[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
    const double l = sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
    if (l > 0) { c[0] /= l; c[1] /= l; c[2] /= l; } else { c[0] = 0; c[1] = 0; c[2] = 1; }
    trin[k] = make_float4((float)c[0], (float)c[1], (float)c[2], mat);
}

// ---- eye-to-scene distance (brute force, double; Ericson 5.1.5)
__device__ double dsub(double a, double b) { return a - b; }
__device__ double pointTriDist2D(const double p[3], const double a[3], const double b[3], const double c[3]) {
#pragma clang fp contract(off)
    double ab[3], ac[3], ap[3];
    for (int i = 0; i < 3; ++i) { ab[i] = b[i] - a[i]; ac[i] = c[i] - a[i]; ap[i] = p[i] - a[i]; }
    auto dot = [](const double* x, const double* y) { return x[0] * y[0] + x[1] * y[1] + x[2] * y[2]; };
    auto dist2 = [&](const double* x) {
        double d[3] = {p[0] - x[0], p[1] - x[1], p[2] - x[2]};
        return dot(d, d);
    };
    double q[3];
    const double d1 = dot(ab, ap), d2 = dot(ac, ap);
    if (d1 <= 0 && d2 <= 0) return dist2(a);
    double bp[3] = {p[0] - b[0], p[1] - b[1], p[2] - b[2]};
    const double d3 = dot(ab, bp), d4 = dot(ac, bp);
    if (d3 >= 0 && d4 <= d3) return dist2(b);
    const double vc = d1 * d4 - d3 * d2;
    if (vc <= 0 && d1 >= 0 && d3 <= 0) {
        const double v = d1 / (d1 - d3);
        for (int i = 0; i < 3; ++i) q[i] = a[i] + v * ab[i];
        return dist2(q);
    }
    double cp[3] = {p[0] - c[0], p[1] - c[1], p[2] - c[2]};
    const double d5 = dot(ab, cp), d6 = dot(ac, cp);
    if (d6 >= 0 && d5 <= d6) return dist2(c);
    const double vb = d5 * d2 - d1 * d6;
    if (vb <= 0 && d2 >= 0 && d6 <= 0) {
        const double w = d2 / (d2 - d6);
        for (int i = 0; i < 3; ++i) q[i] = a[i] + w * ac[i];
        return dist2(q);
    }
    const double va = d3 * d6 - d5 * d4;
    if (va <= 0 && (d4 - d3) >= 0 && (d5 - d6) >= 0) {
        const double w = (d4 - d3) / ((d4 - d3) + (d5 - d6));
        for (int i = 0; i < 3; ++i) q[i] = b[i] + w * (c[i] - b[i]);
        return dist2(q);
    }
    const double denom = 1.0 / (va + vb + vc);
    const double v = vb * denom, w = vc * denom;
    for (int i = 0; i < 3; ++i) q[i] = a[i] + ab[i] * v + ac[i] * w;
    return dist2(q);
}

__global__ void k_min_dist2(const float4* __restrict__ tris, size_t n, double px, double py, double pz,
                            unsigned long long* __restrict__ best) {
    __shared__ unsigned long long sBest;
    if (threadIdx.x == 0) sBest = ~0ull;
    __syncthreads();
    const double p[3] = {px, py, pz};
    unsigned long long mine = ~0ull;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += stride) {
        const float4 a = tris[3 * t], b = tris[3 * t + 1], c = tris[3 * t + 2];
        const double da[3] = {a.x, a.y, a.z}, db[3] = {b.x, b.y, b.z}, dc[3] = {c.x, c.y, c.z};
        const double d2 = pointTriDist2D(p, da, db, dc);
        const unsigned long long bits = (unsigned long long)__double_as_longlong(d2);
        mine = bits < mine ? bits : mine;
    }
    atomicMin(&sBest, mine);
    __syncthreads();
    if (threadIdx.x == 0) atomicMin(best, sBest);
}

struct DevBuf {
    void* p = nullptr;
    ~DevBuf() { if (p) hipFree(p); }
};

int blocks(int64_t n) { return (int)std::max<int64_t>(1, (n + 255) / 256); }

}  // namespace

DeviceTris::~DeviceTris() {
    if (verts) hipFree(verts);
}

gp_status scanTrisDevice(const float* verts, const int32_t* mats, int64_t n, int nMats, DeviceTris& out) {
    hipStream_t s = device().stream;
    const size_t vb = sizeof(float) * 9 * (size_t)n, mb = sizeof(int32_t) * (size_t)n;
    const size_t words = ((vb + mb + 255) & ~size_t(255));   // the reduced words behind both arrays
    hipError_t e = hipMalloc((void**)&out.verts, words + 8 * sizeof(unsigned));
    if (e != hipSuccess) {
        out.verts = nullptr;
        return fail(GP_ERR_OOM, std::string("scene upload: hipMalloc: ") + hipGetErrorString(e));
    }
    out.mats = (int32_t*)((char*)out.verts + vb);
    out.n = n;
    unsigned* red = (unsigned*)((char*)out.verts + words);
    GP_HIP(hipMemcpyAsync(out.verts, verts, vb, hipMemcpyHostToDevice, s));
    GP_HIP(hipMemcpyAsync(out.mats, mats, mb, hipMemcpyHostToDevice, s));
    launchFill64((unsigned long long*)red, 4, 0ull, s);
    hipLaunchKernelGGL(k_scan_tris, dim3(std::min(256, blocks(n))), dim3(256), 0, s, (const float*)out.verts,
                       (const int*)out.mats, (size_t)n, nMats, red);
    GP_HIP(hipGetLastError());
    unsigned r[8];
    GP_HIP(hipMemcpyAsync(r, red, sizeof r, hipMemcpyDeviceToHost, s));
    GP_HIP(hipStreamSynchronize(s));
    if (r[6] & 1u) return fail(GP_ERR_INVALID, "triangle material id out of range");
    if (r[6] & 2u) return fail(GP_ERR_INVALID, "non-finite vertex");
    auto toFloat = [](unsigned u) {
        u = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
        float f;
        std::memcpy(&f, &u, sizeof f);
        return f;
    };
    for (int a = 0; a < 3; ++a) {
        out.centerLo[a] = toFloat(~r[a]);
        out.centerHi[a] = toFloat(r[3 + a]);
    }
    return GP_OK;
}

gp_status buildBvhDevice(const DeviceTris& in, DeviceBvh& out) {
    hipStream_t s = device().stream;
    const int n = (int)in.n;
    auto t0 = std::chrono::steady_clock::now();
    float3 lo = make_float3(in.centerLo[0], in.centerLo[1], in.centerLo[2]);
    auto invExt = [](float l, float h) { return h > l ? 1.0f / (h - l) : 0.0f; };
    float3 inv = make_float3(invExt(in.centerLo[0], in.centerHi[0]), invExt(in.centerLo[1], in.centerHi[1]),
                             invExt(in.centerLo[2], in.centerHi[2]));
    const size_t inner = (size_t)std::max(1, n - 1);
    BoxLevels L{};
    unsigned upper = 0;
    L.size[0] = (unsigned)n;
    L.count = 1;
    while (L.size[L.count - 1] > 1) {
        L.size[L.count] = (L.size[L.count - 1] + 1) / 2;
        L.off[L.count] = upper;
        upper += L.size[L.count++];
    }
    size_t tempBytes = 0;
    GP_HIP(rocprim::radix_sort_pairs(nullptr, tempBytes, (unsigned long long*)nullptr, (unsigned long long*)nullptr,
                                     (unsigned*)nullptr, (unsigned*)nullptr, (size_t)n, 0u, 63u, s));
    // one allocation holds every temporary (a dozen allocations and frees of their own took
    // more than the tree's kernels)
    size_t need = 0;
    auto part = [&](size_t bytes) {
        const size_t at = need;
        need += (std::max<size_t>(bytes, 16) + 255) & ~size_t(255);
        return at;
    };
    const size_t oKeys = part(sizeof(unsigned long long) * n), oKeys2 = part(sizeof(unsigned long long) * n);
    const size_t oVals = part(sizeof(unsigned) * n), oVals2 = part(sizeof(unsigned) * n);
    const size_t oLeaf = part(sizeof(float) * 6 * (size_t)n), oUp = part(sizeof(float) * 6 * (size_t)upper);
    const size_t oNodes = part(sizeof(KNode) * inner), oParent = part(sizeof(int) * inner);
    const size_t oBox = part(sizeof(float) * 6 * inner), oPairs = part(sizeof(float4) * 4 * inner);
    const size_t oHeight = part(sizeof(unsigned long long)), oTemp = part(tempBytes);
    DevBuf arena;
    {
        hipError_t e = hipMalloc(&arena.p, need);
        if (e != hipSuccess) {
            arena.p = nullptr;
            return fail(GP_ERR_OOM, std::string("BVH build: hipMalloc: ") + hipGetErrorString(e));
        }
    }
    auto at = [&](size_t o) { return (void*)((char*)arena.p + o); };
    unsigned long long *keys = (unsigned long long*)at(oKeys), *skeys = (unsigned long long*)at(oKeys2);
    unsigned *vals = (unsigned*)at(oVals), *order = (unsigned*)at(oVals2);
    float *leafBox = (float*)at(oLeaf), *up = (float*)at(oUp), *box = (float*)at(oBox);
    float4* pairs = (float4*)at(oPairs);
    hipLaunchKernelGGL(k_morton, dim3(blocks(n)), dim3(256), 0, s, (const float*)in.verts, n, lo, inv, keys, vals);
    GP_HIP(hipGetLastError());
    GP_HIP(rocprim::radix_sort_pairs(at(oTemp), tempBytes, keys, skeys, vals, order, (size_t)n, 0u, 63u, s));
    hipLaunchKernelGGL(k_leaf_boxes, dim3(blocks(n)), dim3(256), 0, s, (const float*)in.verts, (const unsigned*)order,
                       n, leafBox);
    GP_HIP(hipGetLastError());

    struct Out {
        void* p = nullptr;
        bool keep = false;
        ~Out() { if (!keep && p) hipFree(p); }
    } quads, tris, trin;
    if (hipMalloc(&quads.p, inner * 8 * sizeof(float4)) != hipSuccess) {
        quads.p = nullptr;
        return fail(GP_ERR_OOM, "BVH build: node allocation failed");
    }
    int height = 1;
    if (n <= kLeafMax) {
        hipLaunchKernelGGL(k_lone_leaf, dim3(1), dim3(64), 0, s, (const float*)leafBox, n, pairs);
        hipLaunchKernelGGL(k_collapse4, dim3(1), dim3(64), 0, s, (const KNode*)nullptr, 1, (const float4*)pairs,
                           (float4*)quads.p);
        GP_HIP(hipGetLastError());
    } else {
        KNode* nodes = (KNode*)at(oNodes);
        int *parent = (int*)at(oParent), *dHeight = (int*)at(oHeight);
        launchFill64((unsigned long long*)dHeight, 1, 0ull, s);
        hipLaunchKernelGGL(k_karras, dim3(blocks(n - 1)), dim3(256), 0, s, (const unsigned long long*)skeys, n, nodes,
                           parent);
        for (int base = 0; base + 1 < L.count; base += kBoxStep)
            hipLaunchKernelGGL(k_box_levels, dim3((L.size[base] + (1u << kBoxStep) - 1) >> kBoxStep),
                               dim3(1 << (kBoxStep - 1)), 0, s, L, base, (const float*)leafBox, up);
        hipLaunchKernelGGL(k_node_boxes, dim3(blocks(n - 1)), dim3(256), 0, s, L, (const KNode*)nodes, n - 1,
                           (const float*)leafBox, (const float*)up, box);
        hipLaunchKernelGGL(k_height, dim3(std::min(256, blocks(n - 1))), dim3(256), 0, s, (const KNode*)nodes,
                           (const int*)parent, n - 1, dHeight);
        hipLaunchKernelGGL(k_emit_pairs, dim3(blocks(n - 1)), dim3(256), 0, s, (const KNode*)nodes, n,
                           (const float*)leafBox, (const float*)box, pairs);
        hipLaunchKernelGGL(k_collapse4, dim3(blocks(n - 1)), dim3(256), 0, s, (const KNode*)nodes, n - 1,
                           (const float4*)pairs, (float4*)quads.p);
        GP_HIP(hipGetLastError());
        GP_HIP(hipMemcpyAsync(&height, dHeight, sizeof(int), hipMemcpyDeviceToHost, s));
    }
    if (hipMalloc(&tris.p, sizeof(float4) * 3 * (size_t)n) != hipSuccess) tris.p = nullptr;
    if (hipMalloc(&trin.p, sizeof(float4) * (size_t)n) != hipSuccess) trin.p = nullptr;
    if (!tris.p || !trin.p) {
        hipStreamSynchronize(s);   // the height is still being written
        return fail(GP_ERR_OOM, "BVH build: triangle allocation failed");
    }
    hipLaunchKernelGGL(k_gather, dim3(blocks(n)), dim3(256), 0, s, (const float*)in.verts, (const int*)in.mats,
                       (const unsigned*)order, n, (float4*)tris.p, (float4*)trin.p);
    hipError_t ge = hipGetLastError();
    hipError_t se = hipStreamSynchronize(s);
    if (ge != hipSuccess || se != hipSuccess)
        return fail(GP_ERR_HIP, std::string("BVH build: ") + hipGetErrorString(ge != hipSuccess ? ge : se));
    quads.keep = tris.keep = trin.keep = true;
    out.nodes = (float4*)quads.p;
    out.tris = (float4*)tris.p;
    out.trin = (float4*)trin.p;
    out.nPairs = (int64_t)inner;
    out.depth = std::max(1, height);
    out.stackNeed = 3 * ((out.depth + 1) / 2);   // four-wide levels: pair levels 1, 3, 5, ...
    out.buildMs = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return GP_OK;
}

gp_status deviceMinDistance2(const float4* dTris, int64_t n, const double p[3], double& d2) {
    hipStream_t s = device().stream;
    DevBuf best;
    GP_HIP(hipMalloc(&best.p, sizeof(unsigned long long)));
    GP_HIP(hipMemsetAsync(best.p, 0xff, sizeof(unsigned long long), s));
    const int g = (int)std::min<int64_t>(4096, std::max<int64_t>(1, (n + 255) / 256));
    hipLaunchKernelGGL(k_min_dist2, dim3(g), dim3(256), 0, s, dTris, (size_t)n, p[0], p[1], p[2],
                       (unsigned long long*)best.p);
    GP_HIP(hipGetLastError());
    unsigned long long bits = 0;
    GP_HIP(hipMemcpyAsync(&bits, best.p, sizeof bits, hipMemcpyDeviceToHost, s));
    GP_HIP(hipStreamSynchronize(s));
    std::memcpy(&d2, &bits, sizeof d2);
    return GP_OK;
}

}  // namespace gp
