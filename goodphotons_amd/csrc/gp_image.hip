// Film -> image on the device: scene-linear sRGB (the PFM buffer) and the 8-bit sRGB
// tone map with the p99 auto-exposure anchor, from the int64 fixed-point film.
//
// Follows the reference's filmToLinear / filmToRgb8 (src/main.cpp:10282-10348) and
// xyzToLinearSrgb / srgbGamma (src/color.h:41-53), without the optional denoiser.
// Everything is computed in double with the reference's evaluation order and no FMA
// contraction, starting from the same doubles gp_film_download hands out
// ((double)q * (1 / scale)), so the output equals the CPU reduction of the downloaded
// film bit for bit.
//
// The anchor is an exact order statistic: the element at (size_t)(0.99 (n - 1)) of
// max(r, g, b, 0) over the pixels. It is found by a 5-pass radix select over the
// bit patterns of those non-negative doubles (which order like the values): each
// pass builds an 8192-bin histogram of the next 13 of their 63 bits (11 in the last)
// among the keys that match the bits chosen so far, and one workgroup picks the bin
// holding the k-th key. Eight passes of one byte each took 215 us at 1920 x 1080,
// 65 us now: the first byte is the same for nearly every key (all sign and
// exponent), so its histogram was one LDS address, while 13 bits reach into the mantissa.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>

#include "gp_runtime.hpp"

namespace gp {
namespace {

constexpr double kAbsExposureGain = 6.0;   // absolute-EV sensor gain (main.cpp:10265)

// sum of ybar over 360..830 nm in 1-nm steps (color.h:32-39)
double cieYIntegralHost() {
    auto lobe = [](double x, double mu, double s1, double s2) {
        double t = (x - mu) * ((x < mu) ? s1 : s2);
        return std::exp(-0.5 * t * t);
    };
    double s = 0;
    for (double w = 360.0; w <= 830.0; w += 1.0)
        s += 0.821 * lobe(w, 568.8, 0.0213, 0.0247) + 0.286 * lobe(w, 530.9, 0.0613, 0.0322);
    return s;
}

__device__ __forceinline__ void linearPixel(const long long* __restrict__ film, size_t i, double inv,
                                            double norm, double& r, double& g, double& b) {
#pragma clang fp contract(off)
    const double x = ((double)film[4 * i + 0] * inv) * norm;
    const double y = ((double)film[4 * i + 1] * inv) * norm;
    const double z = ((double)film[4 * i + 2] * inv) * norm;
    r = 3.2406 * x - 1.5372 * y - 0.4986 * z;
    g = -0.9689 * x + 1.8758 * y + 0.0415 * z;
    b = 0.0557 * x - 0.2040 * y + 1.0570 * z;
}

__device__ __forceinline__ double srgbGamma(double c) {
#pragma clang fp contract(off)
    c = c > 0.0 ? c : 0.0;
    return (c <= 0.0031308) ? 12.92 * c : 1.055 * pow(c, 1.0 / 2.4) - 0.055;
}

// Linear sRGB as float (PFM order: the film's own rows): thread i computes channel i % 3 of
// pixel i / 3, so that a wave stores contiguous floats (to pinned host memory).
__global__ void __launch_bounds__(256) k_linear(const long long* __restrict__ film, size_t npix, double inv,
                                                double norm, float* __restrict__ lin) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < 3 * npix; i += stride) {
        double c[3];
        linearPixel(film, i / 3, inv, norm, c[0], c[1], c[2]);
        const unsigned k = (unsigned)(i % 3);
        lin[i] = (float)(k == 0 ? c[0] : (k == 1 ? c[1] : c[2]));
    }
}

// Keys of the anchor.
__global__ void __launch_bounds__(256) k_keys(const long long* __restrict__ film, size_t npix, double inv,
                                              double norm, unsigned long long* __restrict__ keys) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < npix; i += stride) {
        double r, g, b;
        linearPixel(film, i, inv, norm, r, g, b);
        double m = r > g ? r : g;
        m = m > b ? m : b;
        // every value <= 0 is the same key (+0.0), so -0.0 cannot sort last
        keys[i] = m > 0.0 ? (unsigned long long)__double_as_longlong(m) : 0ull;
    }
}

struct SelectState {
    unsigned long long prefix;   // bits chosen so far
    unsigned long long mask;     // which bits are chosen
    unsigned long long k;        // rank still sought among keys matching the prefix
    unsigned long long pad;
};

constexpr int kSelBits = 13, kSelBins = 1 << kSelBits, kSelPasses = 5;
inline int selShift(int pass) { return std::max(0, 63 - kSelBits * (pass + 1)); }

constexpr int kHistThreads = 512;
__global__ void __launch_bounds__(kHistThreads) k_select_hist(const unsigned long long* __restrict__ keys, size_t n,
                                                              const SelectState* st, int shift,
                                                              unsigned* __restrict__ hist) {
    __shared__ unsigned h[kSelBins];
    for (int b = threadIdx.x; b < kSelBins; b += kHistThreads) h[b] = 0;
    __syncthreads();
    const unsigned long long prefix = st->prefix, mask = st->mask;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const unsigned long long key = keys[i];
        // in the last pass the upper two of these bits are chosen already, the same in all
        if ((key & mask) == prefix) atomicAdd(&h[(key >> shift) & (kSelBins - 1)], 1u);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < kSelBins; b += kHistThreads)
        if (h[b]) atomicAdd(&hist[b], h[b]);
}

// One workgroup: find the bin holding rank k, narrow the prefix, clear hist.
constexpr int kPickThreads = 1024;
__global__ void __launch_bounds__(kPickThreads) k_select_pick(SelectState* st, int shift, unsigned* hist) {
    constexpr int kPer = kSelBins / kPickThreads;
    __shared__ unsigned long long scan[kPickThreads];
    const int t = threadIdx.x;
    unsigned c[kPer];
    unsigned long long sum = 0;
    for (int k = 0; k < kPer; ++k) {
        c[k] = hist[t * kPer + k];
        hist[t * kPer + k] = 0;
        sum += c[k];
    }
    scan[t] = sum;
    __syncthreads();
    for (int off = 1; off < kPickThreads; off <<= 1) {
        const unsigned long long v = t >= off ? scan[t - off] : 0ull;
        __syncthreads();
        scan[t] += v;
        __syncthreads();
    }
    const unsigned long long k = st->k;
    unsigned long long before = t > 0 ? scan[t - 1] : 0ull;
    __syncthreads();
    for (int j = 0; j < kPer; ++j) {
        if (c[j] > 0 && before <= k && k < before + c[j]) {
            st->k = k - before;
            st->prefix |= (unsigned long long)(t * kPer + j) << shift;
            st->mask |= (unsigned long long)(kSelBins - 1) << shift;
        }
        before += c[j];
    }
}

// exposure from the anchor (main.cpp:10305-10338); out[0] = eAuto, out[1] = exposure
__global__ void k_exposure(const SelectState* st, double anchor, double expComp, int absolute, double* out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double eAuto;
    if (absolute) {
        eAuto = kAbsExposureGain;
    } else if (anchor > 0.0) {
        eAuto = anchor;
    } else {
        const double p99 = __longlong_as_double((long long)st->prefix);
        eAuto = (p99 > 0) ? 0.9 / p99 : 1.0;
    }
    out[0] = eAuto;
    out[1] = eAuto * (expComp > 0.0 ? expComp : 1.0);
}

// 8-bit sRGB, row 0 = image top (the film's last row)
__global__ void k_rgb8(const long long* __restrict__ film, int W, int H, double inv, double norm,
                       const double* __restrict__ expo, unsigned char* __restrict__ out) {
#pragma clang fp contract(off)
    const double exposure = expo[1];
    const size_t npix = (size_t)W * H;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t d = (size_t)blockIdx.x * blockDim.x + threadIdx.x; d < npix; d += stride) {
        const int y = (int)(d / (size_t)W), x = (int)(d % (size_t)W);
        const size_t src = (size_t)(H - 1 - y) * W + x;
        double c[3];
        linearPixel(film, src, inv, norm, c[0], c[1], c[2]);
        for (int k = 0; k < 3; ++k) {
            double v = srgbGamma(c[k] * exposure) * 255.0 + 0.5;
            v = v < 0.0 ? 0.0 : (v > 255.0 ? 255.0 : v);
            out[3 * d + k] = (unsigned char)v;
        }
    }
}

// Starts a select: the rank sought, empty prefix, zeroed histogram (a kernel rather
// than a host copy and memset, so the allocation-free entry point records only
// kernels on the stream).
__global__ void __launch_bounds__(256) k_select_init(SelectState* st, unsigned* hist, unsigned long long k) {
    for (int b = threadIdx.x; b < kSelBins; b += blockDim.x) hist[b] = 0;
    if (threadIdx.x == 0) *st = SelectState{0, 0, k, 0};
}

// Scratch memory of the allocation-free tone map (gp_film_tonemap_noalloc): the
// select state, histogram and exposure, then the anchor keys (8 B per pixel) and the
// 8-bit image (3 B per pixel) of a film of at most kNoAllocMaxPixels pixels. Each GPU
// holds its own copy for the life of the process; host code reaches it only through
// the address hipGetSymbolAddress returns on that device (noAllocScratch).
constexpr size_t kNoAllocMaxPixels = size_t(1) << 22;   // 2048 x 2048
constexpr size_t kNoAllocHead = 65536;                  // SelectState, bins, 2 doubles
constexpr size_t kNoAllocKeys = kNoAllocMaxPixels * sizeof(unsigned long long);
constexpr size_t kNoAllocBytes = kNoAllocHead + kNoAllocKeys + kNoAllocMaxPixels * 3;
static_assert(sizeof(SelectState) + kSelBins * sizeof(unsigned) + 2 * sizeof(double) <= kNoAllocHead, "head");
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kNoAllocMaxDevices = 64;
std::mutex gScratchMu;
void* gScratchPtr[kNoAllocMaxDevices] = {};

// The device address of `scratch` on the current device, looked up once per device
// (with that device current) and kept.
gp_status noAllocScratch(int dev, unsigned char** out) {
    if (dev < 0 || dev >= kNoAllocMaxDevices) return fail(GP_ERR_NO_DEVICE, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(gScratchMu);
    if (!gScratchPtr[dev]) {
        int cur = -1;
        GP_HIP(hipGetDevice(&cur));
        if (cur != dev) GP_HIP(hipSetDevice(dev));
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != dev) hipSetDevice(cur);
        if (e != hipSuccess || !p)
            return fail(GP_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        gScratchPtr[dev] = p;
    }
    *out = (unsigned char*)gScratchPtr[dev];
    return GP_OK;
}

gp_status filmNorm(const gp_film* f, int64_t nPhotons, double& inv, double& norm) {
    if (!f) return fail(GP_ERR_INVALID, "null film");
    if (nPhotons <= 0) return fail(GP_ERR_INVALID, "n_photons must be positive");
    inv = f->scale > 0 ? 1.0 / f->scale : 0.0;
    norm = 1.0 / ((double)nPhotons * cieYIntegralHost());
    return GP_OK;
}

// Film words to doubles, written straight to pinned host memory (gp_film_download) or to
// device memory (a server's films): thread i converts word i of the pixels' X, Y, Z and, past
// those, of their hit counts, so that the stores of a wave are contiguous in either array.
// Bound by the link to the host (52 GB/s) where it writes there; the same multiply on the
// host, over int64 words copied to pageable memory first, took 8 ms of a 1024 x 1024 render.
__global__ void __launch_bounds__(256) k_film_totals(const long long* __restrict__ film, size_t n, double inv,
                                                     double* __restrict__ xyz, double* __restrict__ hits) {
    const size_t stride = (size_t)gridDim.x * blockDim.x, first = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (xyz)
        for (size_t i = first; i < 3 * n; i += stride) xyz[i] = (double)film[4 * (i / 3) + i % 3] * inv;
    if (hits)
        for (size_t i = first; i < n; i += stride) hits[i] = (double)film[4 * i + 3];
}

int gridFor(size_t n) {
    size_t b = (n + 255) / 256;
    return (int)(b < 4096 ? (b > 0 ? b : 1) : 4096);
}

// The tone map's kernels: select state, histogram and exposure in `head`, then keys and image.
// Returns where the exposure (automatic, applied) is.
const double* enqueueTonemap(const gp_film* film, double inv, double norm, double anchor, double expComp, int absolute,
                             unsigned char* head, unsigned long long* keys, unsigned char* img, hipStream_t s) {
    const int W = film->rx, H = film->ry;
    const size_t npix = (size_t)W * H;
    SelectState* st = (SelectState*)head;
    unsigned* hist = (unsigned*)(head + sizeof(SelectState));
    double* expo = (double*)((char*)hist + kSelBins * sizeof(unsigned));
    const long long* d = (const long long*)film->d;
    // the previous call's state may still be there: start the select afresh
    hipLaunchKernelGGL(k_select_init, dim3(1), dim3(256), 0, s, st, hist,
                       (unsigned long long)(size_t)(0.99 * (double)(npix - 1)));
    if (!absolute && !(anchor > 0.0)) {
        hipLaunchKernelGGL(k_keys, dim3(gridFor(npix)), dim3(256), 0, s, d, npix, inv, norm, keys);
        const unsigned g = (unsigned)std::min<size_t>(512, (npix + kHistThreads - 1) / kHistThreads);
        for (int pass = 0; pass < kSelPasses; ++pass) {
            hipLaunchKernelGGL(k_select_hist, dim3(g), dim3(kHistThreads), 0, s, (const unsigned long long*)keys, npix,
                               (const SelectState*)st, selShift(pass), hist);
            hipLaunchKernelGGL(k_select_pick, dim3(1), dim3(kPickThreads), 0, s, st, selShift(pass), hist);
        }
    }
    hipLaunchKernelGGL(k_exposure, dim3(1), dim3(64), 0, s, (const SelectState*)st, anchor, expComp, absolute, expo);
    hipLaunchKernelGGL(k_rgb8, dim3(gridFor(npix)), dim3(256), 0, s, d, W, H, inv, norm, (const double*)expo, img);
    return expo;
}

}  // namespace

void launchFilmTotals(const unsigned long long* film, size_t n, double inv, double* xyz, double* hits, hipStream_t s) {
    // 512 workgroups keep the link busy and leave the rest of the chip to other streams
    const size_t b = std::min<size_t>(512, std::max<size_t>(1, (3 * n + 255) / 256));
    hipLaunchKernelGGL(k_film_totals, dim3((unsigned)b), dim3(256), 0, s, (const long long*)film, n, inv, xyz, hits);
}

}  // namespace gp

using namespace gp;

extern "C" {

gp_status gp_film_to_linear(gp_film* film, int64_t n_photons, float* rgb) {
    double inv, norm;
    gp_status st = filmNorm(film, n_photons, inv, norm);
    if (st != GP_OK) return st;
    if (!rgb) return fail(GP_ERR_INVALID, "null output");
    if ((st = requireDevice()) != GP_OK) return st;
    const size_t npix = (size_t)film->rx * film->ry;
    hipStream_t s = device().stream;
    return stagedDown(
        npix, 3 * sizeof(float), s,
        [&](char* slot, size_t first, size_t n) {
            hipLaunchKernelGGL(k_linear, dim3(std::min(1024, gridFor(3 * n))), dim3(256), 0, s,
                               (const long long*)film->d + 4 * first, n, inv, norm, (float*)slot);
            return hipGetLastError();
        },
        [&](const char* slot, size_t first, size_t n) {
            copyOut(rgb + 3 * first, slot, n * 3 * sizeof(float));
        });
}

gp_status gp_film_tonemap(gp_film* film, int64_t n_photons, double exposure_comp, int32_t absolute,
                          double* anchor, uint8_t* rgb8, double* exposure_out) {
    double inv, norm;
    gp_status st = filmNorm(film, n_photons, inv, norm);
    if (st != GP_OK) return st;
    if (!rgb8) return fail(GP_ERR_INVALID, "null output");
    if ((st = requireDevice()) != GP_OK) return st;
    const size_t npix = (size_t)film->rx * film->ry;
    hipStream_t s = device().stream;
    Staging& g = staging();
    std::lock_guard<std::mutex> lock(g.mu);
    if ((st = g.ready()) != GP_OK) return st;
    struct Trim {
        Staging& g;
        ~Trim() { g.trim(Staging::kScratch); }
    } trim{g};
    char* base = nullptr;
    if ((st = g.scratchFor(kNoAllocHead + npix * (sizeof(unsigned long long) + 3), &base)) != GP_OK) return st;
    unsigned char* img = (unsigned char*)base + kNoAllocHead + npix * sizeof(unsigned long long);
    const double* expo = enqueueTonemap(film, inv, norm, anchor ? *anchor : 0.0, exposure_comp, (int)absolute,
                                        (unsigned char*)base, (unsigned long long*)(base + kNoAllocHead), img, s);
    GP_HIP(hipGetLastError());
    if ((st = copyDownLocked(g, rgb8, img, npix * 3, s)) != GP_OK) return st;
    double e[2];
    if ((st = copyDownLocked(g, e, expo, sizeof e, s)) != GP_OK) return st;
    if (anchor && !absolute && !(*anchor > 0.0)) *anchor = e[0];
    if (exposure_out) *exposure_out = e[1];
    return GP_OK;
}

gp_status gp_film_tonemap_noalloc(gp_film* film, int64_t n_photons, double exposure_comp, int32_t absolute,
                                  double* anchor, uint8_t* rgb8, double* exposure_out) {
    double inv, norm;
    gp_status st = filmNorm(film, n_photons, inv, norm);
    if (st != GP_OK) return st;
    if (!rgb8) return fail(GP_ERR_INVALID, "null output");
    if ((st = requireDevice()) != GP_OK) return st;
    const int W = film->rx, H = film->ry;
    const size_t npix = (size_t)W * H;
    if (npix > kNoAllocMaxPixels)
        return fail(GP_ERR_CAPACITY, "gp_film_tonemap_noalloc: film of " + std::to_string(npix) +
                                         " pixels exceeds its scratch limit of 4194304 (2048 x 2048)");
    unsigned char* base = nullptr;
    if ((st = noAllocScratch(device().id, &base)) != GP_OK) return st;
    unsigned char* img = base + kNoAllocHead + kNoAllocKeys;
    hipStream_t s = device().stream;
    const double* expo = enqueueTonemap(film, inv, norm, anchor ? *anchor : 0.0, exposure_comp, (int)absolute, base,
                                        (unsigned long long*)(base + kNoAllocHead), img, s);
    GP_HIP(hipGetLastError());
    double e[2];
    GP_HIP(hipMemcpyAsync(rgb8, img, npix * 3, hipMemcpyDeviceToHost, s));
    GP_HIP(hipMemcpyAsync(e, expo, sizeof e, hipMemcpyDeviceToHost, s));
    GP_HIP(hipStreamSynchronize(s));
    if (anchor && !absolute && !(*anchor > 0.0)) *anchor = e[0];
    if (exposure_out) *exposure_out = e[1];
    return GP_OK;
}

}  // extern "C"
