// Input scan of the drop-in validation (include/ohm_sw.h, ohm_scan_inputs).
//
// The reference validates a call with several torch reductions and host
// copies: the numerical domain and the mask marker (orihime/operator.py
// :249-386: no +inf, no NaN, every finite score within `bound` of 0 unless it
// is the legacy marker), the mask sentinel's per-pair maximum (:334-386), and
// the lengths range (src/sw_affine/torch_hip.cpp:69-99).  Here one pass over
// the padded scores gathers all of it into four counts and the per-pair
// maxima, so the host reads back one small block once per call.
//
// The pass is bound by HBM reads, so everything else is kept off it: a lane
// compares the largest magnitude of each 16-byte load with the domain bound
// once and looks at single cells only where that fails, and a workgroup
// scans a long run of one pair, reduces it through LDS and issues one atomic
// per result.  (One atomic maximum per 1024 cells, from every wave of a grid
// with a workgroup per 4096 cells, serialised on the pairs' few words: the
// scan of [16, 4096, 4096] took 2.99 ms, 0.36 TB/s; now 0.19 ms, 5.6 TB/s,
// and [256, 512, 512] 41 us instead of 273.)
//
// No host synchronisation, no memset (graph-capturable).  Batches of up to
// kSmallCells cells run as one workgroup and one launch; larger ones as
// scan_init, which clears the counts and seeds the maxima, and scan_kernel,
// which merges with integer atomics (counts: adds; maxima: a signed maximum
// for non-negative floats, an unsigned minimum of the bits for negative
// ones, so the result does not depend on the order).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>

#include "ohm_sw.h"

namespace ohm {
void set_error(const std::string& msg);
}

namespace {

constexpr int kScanThreads = 256;
constexpr int kSmallThreads = 1024;
constexpr int kScanRun = 4;  // 16-byte loads a lane has in flight
// Workgroups of a large scan: 8 per CU keep enough loads in flight on every
// XCD; more only add atomics.
constexpr int64_t kScanGroups = 2048;
// Up to this size one workgroup (4.5 us at 32 K cells, 5.5 at 64 K) beats
// the two launches (5.7 us at any smaller size than 640 K cells; the three
// launches before took 8.4-9.3).
constexpr int64_t kSmallCells = 1 << 16;
constexpr int kSmallPairs = 64;

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // scores are 4-byte aligned

struct Found {
    int pinf, bad, ninf;  // +inf cells, NaN or out-of-domain cells, -inf cells
    float mx;             // largest cell that is not NaN
};
__device__ __forceinline__ Found nothing() { return {0, 0, 0, -__builtin_inff()}; }

__device__ __forceinline__ uint32_t magnitude(float x) { return __builtin_bit_cast(uint32_t, x) & 0x7fffffffu; }

// One cell, classified on the bits (the
// library is built without NaN semantics for float compares).
__device__ __forceinline__ void classify(Found& f, float x, float marker, uint32_t lim) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x), m = u & 0x7fffffffu;
    const bool is_nan = m > 0x7f800000u;
    f.pinf += u == 0x7f800000u;
    f.ninf += u == 0xff800000u;
    f.bad += is_nan || (m >= lim && m < 0x7f800000u && x != marker);
    if (!is_nan) f.mx = fmaxf(f.mx, x);
}

// `n` cells from `base` by `nthr` threads.  lim: a magnitude is in the domain
// when its bits are below.
__device__ __forceinline__ void scan_cells(Found& f, const float* __restrict__ base, int64_t n, int t, int nthr,
                                           float marker, uint32_t lim) {
    const int64_t step = (int64_t)nthr * 4;
    const int64_t body = n / (step * kScanRun) * (step * kScanRun);
    for (int64_t i = (int64_t)t * 4; i < body; i += step * kScanRun) {
        f4u v[kScanRun];
#pragma unroll
        for (int q = 0; q < kScanRun; ++q) v[q] = *reinterpret_cast<const f4u*>(base + i + q * step);
#pragma unroll
        for (int q = 0; q < kScanRun; ++q) {
            uint32_t m = 0;
#pragma unroll
            for (int c = 0; c < 4; ++c) m = max(m, magnitude(v[q][c]));
            if (m < lim) {
                f.mx = fmaxf(f.mx, fmaxf(fmaxf(v[q][0], v[q][1]), fmaxf(v[q][2], v[q][3])));
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) classify(f, v[q][c], marker, lim);
            }
        }
    }
    for (int64_t i = body + t; i < n; i += nthr) classify(f, base[i], marker, lim);
}

__device__ __forceinline__ int wave_add(int v) {
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ float wave_fmax(float v) {
    for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

// The workgroup's results in thread 0 (NW waves; red: NW records).  Every
// thread calls it; the trailing barrier lets `red` be used again.
template <int NW>
__device__ __forceinline__ Found combine(Found f, Found* red, int t) {
    f.pinf = wave_add(f.pinf);
    f.bad = wave_add(f.bad);
    f.ninf = wave_add(f.ninf);
    f.mx = wave_fmax(f.mx);
    if ((t & 63) == 0) red[t >> 6] = f;
    __syncthreads();
    if (t == 0) {
        for (int w = 1; w < NW; ++w) {
            f.pinf += red[w].pinf;
            f.bad += red[w].bad;
            f.ninf += red[w].ninf;
            f.mx = fmaxf(f.mx, red[w].mx);
        }
    }
    __syncthreads();
    return f;
}

__device__ __forceinline__ int bad_lengths(const int32_t* lengths, int b, int L1, int L2) {
    const int l1 = lengths[2 * b], l2 = lengths[2 * b + 1];
    return (l1 < 0 || l1 > L1) + (l2 < 0 || l2 > L2);
}

// counts: [0] +inf cells, [1] NaN or out-of-domain finite cells, [2] -inf
// cells, [3] lengths entries outside [0, L1] x [0, L2].
__global__ __launch_bounds__(256) void scan_init(int32_t* counts, float* pair_max, int B) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < 4) counts[t] = 0;
    if (t < B) pair_max[t] = -__builtin_inff();
}

// One-dimensional grid of B * nblk workgroups: workgroup x scans cells
// [run * (x % nblk), + run) of pair x / nblk (whole pair boxes of the padded
// layout: the cells past a pair's lengths are scanned too, as the reference
// does).
__global__ __launch_bounds__(kScanThreads) void scan_kernel(const float* __restrict__ scores,
                                                            const int32_t* __restrict__ lengths,
                                                            int64_t cells, int64_t run, int nblk, int L1, int L2,
                                                            uint32_t lim, float marker, int32_t* counts,
                                                            float* pair_max) {
    __shared__ Found red[kScanThreads / 64];
    const int b = blockIdx.x / nblk, blk = blockIdx.x % nblk;
    const int t = threadIdx.x;
    if (blk == 0 && t == 0 && lengths) {
        const int bad = bad_lengths(lengths, b, L1, L2);
        if (bad) atomicAdd(&counts[3], bad);
    }
    const int64_t start = min(run * blk, cells), n = min(run, cells - start);
    Found f = nothing();
    scan_cells(f, scores + (int64_t)b * cells + start, n, t, kScanThreads, marker, lim);
    f = combine<kScanThreads / 64>(f, red, t);
    if (t == 0) {
        if (f.pinf) atomicAdd(&counts[0], f.pinf);
        if (f.bad) atomicAdd(&counts[1], f.bad);
        if (f.ninf) atomicAdd(&counts[2], f.ninf);
        // float maximum on the bits: non-negative floats order as signed
        // integers, negative ones inversely as unsigned
        const uint32_t u = __builtin_bit_cast(uint32_t, f.mx);
        if (!(u & 0x80000000u)) atomicMax(reinterpret_cast<int*>(pair_max) + b, (int)u);
        else if (u != 0xff800000u) atomicMin(reinterpret_cast<uint32_t*>(pair_max) + b, u);
    }
}

// A small batch (B <= kSmallPairs) in one launch: a pair is cut into `parts`
// slices, a wave scans a slice at a time.
__global__ __launch_bounds__(kSmallThreads) void scan_small_kernel(const float* __restrict__ scores,
                                                                   const int32_t* __restrict__ lengths, int B,
                                                                   int64_t cells, int parts, int L1, int L2,
                                                                   uint32_t lim, float marker, int32_t* counts,
                                                                   float* pair_max) {
    constexpr int kWaves = kSmallThreads / 64;
    __shared__ Found red[kWaves];
    __shared__ float s_max[kSmallPairs > kWaves ? kSmallPairs : kWaves];  // B * parts slices
    __shared__ int s_bad;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    if (t == 0) s_bad = 0;
    __syncthreads();
    if (lengths && t < B) {
        const int bad = bad_lengths(lengths, t, L1, L2);
        if (bad) atomicAdd(&s_bad, bad);
    }
    const int64_t run = (cells + parts - 1) / parts;
    Found all = nothing();
    for (int u = wv; u < B * parts; u += kWaves) {
        const int b = u / parts;
        const int64_t start = min(run * (u % parts), cells), n = min(run, cells - start);
        Found f = nothing();
        scan_cells(f, scores + (int64_t)b * cells + start, n, lane, 64, marker, lim);
        f.mx = wave_fmax(f.mx);
        if (lane == 0) s_max[u] = f.mx;
        all.pinf += f.pinf;
        all.bad += f.bad;
        all.ninf += f.ninf;
    }
    all = combine<kWaves>(all, red, t);  // (its barriers order s_max and s_bad too)
    if (t < B) {
        float mx = s_max[t * parts];
        for (int q = 1; q < parts; ++q) mx = fmaxf(mx, s_max[t * parts + q]);
        pair_max[t] = mx;
    }
    if (t == 0) {
        counts[0] = all.pinf;
        counts[1] = all.bad;
        counts[2] = all.ninf;
        counts[3] = s_bad;
    }
}

ohm_status fail(ohm_status st, const std::string& msg) {
    ohm::set_error(msg);
    return st;
}

}  // namespace

extern "C" ohm_status ohm_scan_inputs(const float* scores, const int32_t* lengths, int32_t B,
                                      int32_t L1, int32_t L2, float bound, float marker,
                                      int32_t* counts, float* pair_max, void* stream) {
    if (B < 0 || L1 < 0 || L2 < 0) return fail(OHM_EINVAL, "negative batch size or length");
    if (!counts) return fail(OHM_EINVAL, "counts is null");
    if (B > 0 && !pair_max) return fail(OHM_EINVAL, "pair_max is null");
    const int64_t cells = (int64_t)L1 * L2;
    if (B > 0 && cells > 0 && !scores) return fail(OHM_EINVAL, "scores is null");
    hipStream_t s = static_cast<hipStream_t>(stream);
    // in the domain: finite and magnitude <= bound (bits order as magnitudes;
    // a negative bound admits nothing, -0 the zeros, a NaN bound every finite
    // cell)
    uint32_t lim = 0x7f800000u;
    if (bound < 0.0f) {
        lim = 0;
    } else if (bound < 3.4028234663852886e38f) {
        const float size = std::fabs(bound);  // (-0: its sign bit is no magnitude)
        std::memcpy(&lim, &size, sizeof lim);
        ++lim;
    }
    if (B <= kSmallPairs && B * cells <= kSmallCells) {
        constexpr int kWaves = kSmallThreads / 64;
        const int parts = B > 0 ? std::max(1, kWaves / B) : 1;
        hipLaunchKernelGGL(scan_small_kernel, dim3(1), dim3(kSmallThreads), 0, s, scores, lengths, B, cells, parts, L1,
                           L2, lim, marker, counts, pair_max);
    } else {
        // runs of whole workgroup iterations, about kScanGroups of them in all
        constexpr int64_t per = (int64_t)kScanThreads * 4 * kScanRun;
        const int64_t want = (kScanGroups + B - 1) / B;
        const int64_t run = std::max<int64_t>(per, ((cells + want - 1) / want + per - 1) / per * per);
        const int64_t nblk = std::max<int64_t>(1, (cells + run - 1) / run);
        if (nblk * B > 0x7fffffff) return fail(OHM_EINVAL, "batch too large for one scan launch");
        hipLaunchKernelGGL(scan_init, dim3((unsigned)((B + 255) / 256)), dim3(256), 0, s, counts, pair_max, B);
        hipLaunchKernelGGL(scan_kernel, dim3((unsigned)(nblk * B)), dim3(kScanThreads), 0, s, scores, lengths, cells,
                           run, (int)nblk, L1, L2, lim, marker, counts, pair_max);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(OHM_ELAUNCH, std::string("scan kernels: ") + hipGetErrorString(e));
    return OHM_OK;
}
