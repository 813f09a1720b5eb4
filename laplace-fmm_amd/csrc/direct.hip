// direct.hip -- FP64 all-pairs sums on the GPU (the reference's
// fmm::gpu::ComputeExact, src/common/simple_math.cu:9-22 and :24-130, with the
// pair terms of src/common/simple_math.h:120-151 and their device forms
// :197-208).
//
// 3D pair:
//   q / max(|r|, 1e-4)  and  q r / max(|r|, 1e-4)^3   (r = x_i - x_j)
// evaluated as q * rsqrt(max(|r|^2, 1e-8)), the reference's device form.
// 2D pair: q * 0.5 log max(|dz|^2, 1e-8) and q conj(dz) / max(|dz|^2, 1e-8).
// With `exclude` the pair j == i is skipped (single-set calls only).
#include "device_common.h"
#include "direct.h"

#include <algorithm>
#include <mutex>

namespace lfmm {

namespace {

constexpr int kTile = 256;

// 1 / sqrt(r2): v_rsq_f64 (relative error 5e-8) refined by one third-order
// step: with e = 1 - r2 y^2, y (1 + e / 2 + 3 e^2 / 8) leaves 5/16 e^3, far
// below the rounding of the last operation
__device__ __forceinline__ double rsqrt_full(double r2)
{
    const double y = __builtin_amdgcn_rsq(r2);
    const double e = fma(-(r2 * y), y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// All pairs, targets first .. end - 1.  A workgroup of 1024 threads owns 2 LT of
// them, two per lane (LT lanes), and cuts the sources into 1024 / LT interleaved
// slices, one per group of LT lanes; the slices' sums are added in a fixed order
// at the end (shuffles within a wave, then LDS over the waves).  So 512 targets
// and more fill the chip without a buffer for partial sums: one thread per target
// ran 4,096 targets on 16 of 256 CUs (123 ms against 1,048,576 sources).  Fewer
// than 512 leave CUs idle.
// Bound by FP64 vector issue: 19 operations and v_rsq_f64 per 3D pair.  With
// LT >= 64 a wave's source is uniform and arrives by scalar loads; below, two
// targets per lane halve the L1 reads per pair, which one target per lane
// would be bound by (64 lanes x 32 bytes at 64 bytes per cycle).
template <int DIM>
struct DirectSum;
template <>
struct DirectSum<3> {
    double p = 0.0, fx = 0.0, fy = 0.0, fz = 0.0;
    __device__ __forceinline__ void add(const double4& t, double sx, double sy, double sz, double q)
    {
        const double dx = t.x - sx, dy = t.y - sy, dz = t.z - sz;
        const double r2 = fmax(fma(dx, dx, fma(dy, dy, dz * dz)), 1.e-8);
        const double ir = rsqrt_full(r2);
        const double qi = q * ir;
        p += qi;
        const double q3 = qi * (ir * ir);
        fx = fma(q3, dx, fx);
        fy = fma(q3, dy, fy);
        fz = fma(q3, dz, fz);
    }
};
template <>
struct DirectSum<2> {
    double p = 0.0, fx = 0.0, fy = 0.0, fz = 0.0;  // fz unused
    __device__ __forceinline__ void add(const double4& t, double sx, double sy, double, double q)
    {
        // packed 2D records are (x, y, 0, q)
        const double dx = t.x - sx, dy = t.y - sy;
        const double r2 = fmax(fma(dx, dx, dy * dy), 1.e-8);
        p = fma(q * 0.5, log(r2), p);
        const double qr = q / r2;
        fx = fma(qr, dx, fx);
        fy = fma(-qr, dy, fy);
    }
};

constexpr int kDirectThreads = 1024;

template <int DIM, int LT, bool EXCLUDE>
__global__ void __launch_bounds__(kDirectThreads) k_direct(const double4* __restrict__ tgt, int64_t first,
                                                          int64_t end, const double4* __restrict__ src, int64_t ns,
                                                          double* __restrict__ pot, double* __restrict__ field)
{
    constexpr int S = kDirectThreads / LT, NW = kDirectThreads / 64;
    // per wave the sums of its targets (LT <= 64: 2 LT; above: 2 per lane)
    constexpr int WT = LT < 64 ? LT : 64;
    __shared__ double4 part[S > 1 ? 2 * NW * WT : 1];
    const int lt = threadIdx.x & (LT - 1), lane = threadIdx.x & 63;
    int64_t i[2];
    double4 t[2];
    DirectSum<DIM> a[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        i[u] = first + (int64_t)blockIdx.x * (2 * LT) + u * LT + lt;
        t[u] = i[u] < end ? tgt[i[u]] : make_double4(0.0, 0.0, 0.0, 0.0);
    }
    auto pair = [&](int64_t j, double sx, double sy, double sz, double q) {
#pragma unroll
        for (int u = 0; u < 2; ++u) a[u].add(t[u], sx, sy, sz, EXCLUDE && j == i[u] ? 0.0 : q);
    };
    if constexpr (LT >= 64) {
        typedef const double __attribute__((address_space(4))) scalar;
        scalar* p = (scalar*)(uintptr_t)src;
        const int s = __builtin_amdgcn_readfirstlane((int)threadIdx.x / LT);
#pragma unroll 4
        for (int64_t j = s; j < ns; j += S) pair(j, p[4 * j], p[4 * j + 1], p[4 * j + 2], p[4 * j + 3]);
    } else {
#pragma unroll 4
        for (int64_t j = threadIdx.x / LT; j < ns; j += S) {
            const double4 r = src[j];
            pair(j, r.x, r.y, r.z, r.w);
        }
    }
    if constexpr (S > 1) {
        // slices of one wave, then the waves in order
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            for (int off = 32; off >= WT; off >>= 1) {
                a[u].p += __shfl_xor(a[u].p, off);
                a[u].fx += __shfl_xor(a[u].fx, off);
                a[u].fy += __shfl_xor(a[u].fy, off);
                if constexpr (DIM == 3) a[u].fz += __shfl_xor(a[u].fz, off);
            }
            if (lane < WT)
                part[((threadIdx.x >> 6) * 2 + u) * WT + lane] = make_double4(a[u].p, a[u].fx, a[u].fy, a[u].fz);
        }
        __syncthreads();
        if (threadIdx.x >= LT) return;
        // wave w holds target lanes (w WT) mod LT ..
        constexpr int STEP = LT <= 64 ? 1 : LT / 64;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            a[u] = DirectSum<DIM>();
#pragma unroll 1
            for (int w = LT <= 64 ? 0 : (int)(threadIdx.x >> 6); w < NW; w += STEP) {
                const double4 v = part[(w * 2 + u) * WT + (lt & (WT - 1))];
                a[u].p += v.x;
                a[u].fx += v.y;
                a[u].fy += v.z;
                a[u].fz += v.w;
            }
        }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        if (i[u] >= end) continue;
        if (pot) pot[i[u]] = a[u].p;
        if (field) {
            field[DIM * i[u]] = a[u].fx;
            field[DIM * i[u] + 1] = a[u].fy;
            if constexpr (DIM == 3) field[DIM * i[u] + 2] = a[u].fz;
        }
    }
}

// Few targets, many sources: block (x, y) sums targets x * kTile .. over
// source chunk y into part[y * nt + i] = (pot, field); k_direct3d_join adds
// the chunks in order.  Spreads a sampled check (hundreds of targets against
// millions of sources) over the whole GPU.
__global__ void __launch_bounds__(kTile) k_direct3d_part(const double4* __restrict__ tgt, int64_t nt,
                                                        const double4* __restrict__ src, int64_t ns, int64_t chunk,
                                                        double4* __restrict__ part)
{
    __shared__ double4 tile[kTile];
    const int64_t i = (int64_t)blockIdx.x * kTile + threadIdx.x;
    const double4 t = i < nt ? tgt[i] : make_double4(0.0, 0.0, 0.0, 0.0);
    const int64_t j_beg = (int64_t)blockIdx.y * chunk, j_end = min(ns, j_beg + chunk);
    double p = 0.0, fx = 0.0, fy = 0.0, fz = 0.0;
    for (int64_t base = j_beg; base < j_end; base += kTile) {
        __syncthreads();
        const int64_t j0 = base + threadIdx.x;
        tile[threadIdx.x] = j0 < j_end ? src[j0] : make_double4(0.0, 0.0, 0.0, 0.0);
        __syncthreads();
        const int cnt = (int)min<int64_t>(kTile, j_end - base);
        for (int j = 0; j < cnt; ++j) {
            const double4 s = tile[j];
            const double dx = t.x - s.x, dy = t.y - s.y, dz = t.z - s.z;
            const double r2 = fmax(fma(dx, dx, fma(dy, dy, dz * dz)), 1.e-8);
            const double ir = rsqrt_full(r2);
            const double qi = s.w * ir;
            p += qi;
            const double q3 = qi * ir * ir;
            fx = fma(q3, dx, fx);
            fy = fma(q3, dy, fy);
            fz = fma(q3, dz, fz);
        }
    }
    if (i < nt) part[(int64_t)blockIdx.y * nt + i] = make_double4(p, fx, fy, fz);
}

__global__ void __launch_bounds__(256) k_direct3d_join(const double4* __restrict__ part, int64_t nt, int splits,
                                                      double* __restrict__ pot, double* __restrict__ field)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nt) return;
    double p = 0.0, fx = 0.0, fy = 0.0, fz = 0.0;
    for (int y = 0; y < splits; ++y) {
        const double4 v = part[(int64_t)y * nt + i];
        p += v.x;
        fx += v.y;
        fy += v.z;
        fz += v.w;
    }
    if (pot) pot[i] = p;
    if (field) {
        field[3 * i] = fx;
        field[3 * i + 1] = fy;
        field[3 * i + 2] = fz;
    }
}

// Field of vector charges from the fields of their components: with
// E_c = sum_j q_j^c r / |r|^3, sum_j q_j x r / |r|^3 = (E_2.z - E_3.y,
// E_3.x - E_1.z, E_1.y - E_2.x) (the reference's forces_cross,
// src/cuda/multipole3d.cu:765-776).  Written over e3.
__global__ void __launch_bounds__(256) k_cross_fields(const double* __restrict__ e1, const double* __restrict__ e2,
                                                     double* __restrict__ e3, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double a0 = e1[3 * i], a1 = e1[3 * i + 1], a2 = e1[3 * i + 2];
    const double b0 = e2[3 * i], b1 = e2[3 * i + 1], b2 = e2[3 * i + 2];
    const double c0 = e3[3 * i], c1 = e3[3 * i + 1], c2 = e3[3 * i + 2];
    (void)a0;
    (void)b1;
    (void)c2;
    e3[3 * i] = b2 - c1;
    e3[3 * i + 1] = c0 - a2;
    e3[3 * i + 2] = a1 - b0;
}

}  // namespace

hipError_t launch_cross_fields(const double* e1, const double* e2, double* e3, int64_t n, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_cross_fields, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, e1, e2, e3, n);
    return hipGetLastError();
}

template <int DIM, int LT>
static hipError_t direct_lt(const double4* tgt, int64_t first, int64_t end, const double4* src, int64_t ns, bool exclude,
                            double* pot, double* field, hipStream_t st)
{
    const dim3 grid((unsigned)((end - first + 2 * LT - 1) / (2 * LT))), block(kDirectThreads);
    if (exclude)
        hipLaunchKernelGGL((k_direct<DIM, LT, true>), grid, block, 0, st, tgt, first, end, src, ns, pot, field);
    else
        hipLaunchKernelGGL((k_direct<DIM, LT, false>), grid, block, 0, st, tgt, first, end, src, ns, pot, field);
    return hipGetLastError();
}

// A CU holds one workgroup (1024 threads; 3D: 126 registers), so the targets go
// in rounds of 256 workgroups, and a round that is not full takes as long as a
// full one.  Each launch therefore takes whole rounds at the largest LT that fills
// one, and what is left goes on in smaller rounds, down to 512 targets, unless
// less than a launch's time is gained.  One launch at one LT lost up to half:
// 200,000 sources and 530,000 targets 149 -> 76 ms (one thread per target:
// 99), 270,000 75 -> 38 (59), 4,097 1.36 -> 0.86 (4,096: 0.78).
constexpr int64_t kDirectRound = 512;      // targets of a round at LT = 1
constexpr int64_t kDirectGain = 8000000;   // pairs in 8 us (2D: 28 us)

template <int DIM>
static hipError_t direct_dim(const double4* tgt, int64_t nt, const double4* src, int64_t ns, bool exclude, double* pot,
                             double* field, hipStream_t st)
{
    int least = 1;  // no more slices than there are sources for
    while (least < kDirectThreads && kDirectThreads / least > ns) least *= 2;
    for (int64_t at = 0; at < nt;) {
        const int64_t left = nt - at;
        int lt = least;
        while (lt < kDirectThreads && left >= kDirectRound * 2 * lt) lt *= 2;
        const int64_t round = kDirectRound * lt, rest = left % round;
        int64_t end = nt;
        if (left > round && rest > 0) {
            const int64_t small = kDirectRound * least;
            const int64_t gained = round - rest - (small - rest % small) % small;
            if (gained > kDirectGain / std::max<int64_t>(ns, 1)) end = nt - rest;
        }
        hipError_t e = hipErrorInvalidValue;
        switch (lt) {
#define X(n) case n: e = direct_lt<DIM, n>(tgt, at, end, src, ns, exclude, pot, field, st); break;
            X(1) X(2) X(4) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024)
#undef X
        }
        if (e != hipSuccess) return e;
        at = end;
    }
    return hipSuccess;
}

hipError_t launch_direct(int dim, const double4* tgt, int64_t nt, const double4* src, int64_t ns, bool exclude_self,
                         double* pot, double* field, hipStream_t st)
{
    if (nt <= 0) return hipSuccess;
    return dim == 3 ? direct_dim<3>(tgt, nt, src, ns, exclude_self, pot, field, st)
                    : direct_dim<2>(tgt, nt, src, ns, exclude_self, pot, field, st);
}

int direct3d_split_count(int64_t nt, int64_t ns)
{
    if (nt <= 0 || ns <= 0) return 1;
    const int64_t tblocks = (nt + kTile - 1) / kTile;
    const int64_t want = (2048 + tblocks - 1) / tblocks;        // about 8 workgroups per CU
    const int64_t most = (ns + 4 * kTile - 1) / (4 * kTile);    // at least 4 tiles per chunk
    return (int)std::max<int64_t>(1, std::min<int64_t>({want, most, 65535}));
}

hipError_t launch_direct3d_split(const double4* tgt, int64_t nt, const double4* src, int64_t ns, double* pot,
                                 double* field, double4* part, int splits, hipStream_t st)
{
    if (nt <= 0) return hipSuccess;
    const int64_t chunk = ((ns + splits - 1) / splits + kTile - 1) / kTile * kTile;
    const dim3 grid((unsigned)((nt + kTile - 1) / kTile), (unsigned)splits);
    hipLaunchKernelGGL(k_direct3d_part, grid, dim3(kTile), 0, st, tgt, nt, src, ns, chunk, part);
    hipLaunchKernelGGL(k_direct3d_join, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, st, part, nt, splits, pot,
                       field);
    return hipGetLastError();
}

// ---- the allocation-free direct sum (lfmm_direct3d_noalloc)
// The packed (x, y, z, q) records of one call's sources and targets live in
// this fixed array, one copy per GPU, held until the process ends.  Host code
// never passes the array's name to a kernel (in host code it is a stand-in,
// not a device address): each device's address comes from
// hipGetSymbolAddress once, with that device current (noalloc_scratch_init,
// from lfmm_create), and is used from then on.
constexpr int64_t kNoAllocRecords = (int64_t)(kNoAllocScratchBytes / sizeof(double4));
static __device__ __align__(256) double4 scratch[kNoAllocRecords];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double4* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

hipError_t noalloc_scratch_init(int device)
{
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (g_scratch_ptr[device]) return hipSuccess;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[device] = (double4*)p;
    return hipSuccess;
}

double4* noalloc_scratch(int device)
{
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> g(g_scratch_mu);
    return g_scratch_ptr[device];
}

}  // namespace lfmm
