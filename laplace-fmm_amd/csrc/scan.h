// scan.h -- device-wide exclusive sums over a computed input, the result
// handed to a functor: flags are counted, and lists written, without arrays of
// flags or sums in between.
//
// Tiles of 4,096 values.  One tile: one launch.  Up to kScanDirect tiles two:
// the tiles' sums, then every workgroup adds the sums before its own itself
// (at most 4 loads per thread, in L2) instead of waiting for a third launch;
// beyond that a workgroup between them scans the sums, since those loads grow
// with the square of the tiles.  Latency-bound at the tree's sizes (65,536
// particles): three launches of 256 threads took 4.4 + 2.8 + 4.4 us and the
// gaps between them, one now takes 4.7; several tiles 4.5 + 4.7.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace lfmm {

constexpr int kScanThreads = 1024;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanThreads * kScanItems;
constexpr int kScanDirect = 4096;

// LDS slot of a tile's element: threads' elements start 5 words apart
__host__ __device__ constexpr int scan_slot(int i) { return i + i / kScanItems; }

template <typename T>
__device__ inline T wave_incl_scan(T v)
{
    const int lane = threadIdx.x & 63;
    for (int off = 1; off < 64; off <<= 1) {
        const T t = __shfl_up(v, off);
        if (lane >= off) v += t;
    }
    return v;
}

// Exclusive scan of one value per thread of the workgroup; total: their sum.
// The call before it and after it may use the same LDS.
template <int THREADS, typename T>
__device__ inline T block_excl_scan(T v, T& total)
{
    __shared__ T wsum[THREADS / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const T inc = wave_incl_scan(v);
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    T off = 0, tot = 0;
    for (int i = 0; i < THREADS / 64; ++i) {
        if (i < w) off += wsum[i];
        tot += wsum[i];
    }
    __syncthreads();
    total = tot;
    return off + inc - v;
}

template <typename In>
__global__ void __launch_bounds__(kScanThreads) k_scan_reduce(In in, int64_t n, uint32_t* __restrict__ sums)
{
    const int64_t base = blockIdx.x * (int64_t)kScanTile;
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        const int64_t j = base + i * kScanThreads + threadIdx.x;
        if (j < n) s += in(j);
    }
    uint32_t tot;
    block_excl_scan<kScanThreads>(s, tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// in place: sums[i] = the sums before i, sums[nb] = all (one workgroup)
static __global__ void __launch_bounds__(1024) k_scan_top(uint32_t* __restrict__ sums, int nb)
{
    const int per = (nb + 1023) / 1024;
    const int b0 = threadIdx.x * per;
    uint32_t s = 0;
    for (int i = 0; i < per; ++i)
        if (b0 + i < nb) s += sums[b0 + i];
    uint32_t tot;
    uint32_t run = block_excl_scan<1024>(s, tot);
    for (int i = 0; i < per; ++i)
        if (b0 + i < nb) {
            const uint32_t t = sums[b0 + i];
            sums[b0 + i] = run;
            run += t;
        }
    if (threadIdx.x == 0) sums[nb] = tot;
}

// The sums before this workgroup's tile; scanned: sums holds them already.
__device__ inline uint32_t scan_before(const uint32_t* __restrict__ sums, bool scanned)
{
    if (blockIdx.x == 0) return 0;
    if (scanned) return sums[blockIdx.x];
    uint32_t s = 0, tot;
    for (int i = threadIdx.x; i < (int)blockIdx.x; i += kScanThreads) s += sums[i];
    block_excl_scan<kScanThreads>(s, tot);
    return tot;
}

// out(j, sum of in(0 .. j - 1)) for every j < n
template <typename In, typename Out>
__global__ void __launch_bounds__(kScanThreads) k_scan_down(In in, Out out, int64_t n, const uint32_t* __restrict__ sums,
                                                            int scanned)
{
    __shared__ uint32_t tile[scan_slot(kScanTile)];
    const int64_t base = blockIdx.x * (int64_t)kScanTile;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        const int k = i * kScanThreads + threadIdx.x;
        tile[scan_slot(k)] = base + k < n ? in(base + k) : 0u;
    }
    const uint32_t before = scan_before(sums, scanned != 0);
    __syncthreads();
    uint32_t loc[kScanItems];
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        loc[i] = tile[scan_slot(threadIdx.x * kScanItems + i)];
        s += loc[i];
    }
    uint32_t tot;
    uint32_t run = block_excl_scan<kScanThreads>(s, tot) + before;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        tile[scan_slot(threadIdx.x * kScanItems + i)] = run;
        run += loc[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        const int k = i * kScanThreads + threadIdx.x;
        if (base + k < n) out(base + k, tile[scan_slot(k)]);
    }
}

// ws: scan_ws_elems(n) words
template <typename In, typename Out>
hipError_t scan_apply(In in, Out out, int64_t n, uint32_t* ws, hipStream_t st)
{
    const int64_t nb = (n + kScanTile - 1) / kScanTile;
    if (n < 0 || nb >= (int64_t)1 << 22) return hipErrorInvalidValue;  // 2^32 threads in a launch
    if (nb == 0) return hipSuccess;
    const dim3 grid((unsigned)nb), block(kScanThreads);
    if (nb > 1) hipLaunchKernelGGL((k_scan_reduce<In>), grid, block, 0, st, in, n, ws);
    const int scanned = nb > kScanDirect ? 1 : 0;
    if (scanned) hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, st, ws, (int)nb);
    hipLaunchKernelGGL((k_scan_down<In, Out>), grid, block, 0, st, in, out, n, (const uint32_t*)ws, scanned);
    return hipGetLastError();
}

struct ScanLoad {
    const uint32_t* p;
    __device__ uint32_t operator()(int64_t j) const { return p[j]; }
};
struct ScanStore {
    uint32_t* p;
    __device__ void operator()(int64_t j, uint32_t before) const { p[j] = before; }
};

}  // namespace lfmm
