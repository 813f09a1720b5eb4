// p2p.hip -- near-field pair sums (P2P), several targets per lane.
//
// The reference's near field (src/cpu/multipole3d.cpp:964-1151, GPU
// src/cuda/multipole3d.cu:568-576; pair term src/common/simple_math.h:130-139):
// phi_i += q_j / max(r, 1e-4), E_i += q_j (x_i - x_j) / max(r, 1e-4)^3 over
// the 27 neighbour leaves, self pair included.
//
// Each lane owns TPL consecutive targets of one leaf (they share the neighbour
// list) and every 32-byte source record it loads feeds TPL pair terms: 4 where
// leaves hold 64 particles and more on average, else 2 (past a leaf's end a
// lane repeats its last target, computed but not written).  Lanes are listed
// per leaf: lane slot_begin[leaf] + k owns targets leaf_begin[leaf] + TPL k ...
// + TPL k + TPL - 1.
//
// Bound by vector issue: 18 FP64 operations and v_rsq_f64 per pair.  A lane
// walks the near ranges of its leaf as one list, so a wave runs as long as its
// longest leaf total, on a uniform count: per source one compare (the range's
// end), one pointer step and two loads.  The bounds of the next range are
// loaded a range ahead; a lane past its list reads a zero charge, so nothing
// is masked.  That record sits in its own leaf (pad): far from it, at the origin
// say, r^2 could overflow, and 0 times that sum's NaN would enter the results.
#include "device_common.h"
#include "ops3d.h"
#include "tree.h"

#include <algorithm>

namespace lfmm {

namespace {

// 1 / sqrt(r2): v_rsq_f64 (relative error ~5e-8) refined by one Newton step:
// relative error <= 4.3e-15 (measured over 4M arguments in [1e-9, 10]), 1e-4
// of the FMM's own error at any order, for 3 fewer FP64 operations per pair
// than a second step
__device__ __forceinline__ double rsqrt_nf(double r2)
{
    const double y = __builtin_amdgcn_rsq(r2);
    const double hr = 0.5 * r2;
    return y * fma(-hr * y, y, 1.5);
}

// Every WIDTH leaves are ordered by the sources of their near lists, so that
// the leaves of a wave end together: leaf l is pos[l] in lane order,
// cnt[pos]: its lanes.  pad[l]: a zero charge at leaf l's first particle.
template <int TPL, int WIDTH>
__global__ void __launch_bounds__(512) k_pair_counts(const int32_t* __restrict__ leaf_begin,
                                                    const int32_t* __restrict__ near_total, int nleaf,
                                                    uint32_t* __restrict__ cnt, int32_t* __restrict__ pos,
                                                    const double4* __restrict__ src, double4* __restrict__ pad)
{
    __shared__ uint64_t key[512];
    const int base = blockIdx.x * blockDim.x, l = base + threadIdx.x;
    // past the last leaf: sorts last
    const uint64_t mine = l < nleaf ? ((uint64_t)(uint32_t)near_total[l] << 32) | threadIdx.x : ~0ull;
    int leaf = l;
    if constexpr (WIDTH > 1) {  // bitonic
        key[threadIdx.x] = mine;
        for (int w = 2; w <= WIDTH; w *= 2)
            for (int h = w / 2; h > 0; h /= 2) {
                __syncthreads();
                const int i = threadIdx.x, j = i ^ h;
                if (j > i) {
                    const uint64_t a = key[i], b = key[j];
                    if ((a > b) == (w == WIDTH || (i & w) == 0)) {
                        key[i] = b;
                        key[j] = a;
                    }
                }
            }
        __syncthreads();
        leaf = base + (int)(uint32_t)key[threadIdx.x];
    }
    if (l >= nleaf) return;
    const double4 first = src[leaf_begin[l]];
    pad[l] = make_double4(first.x, first.y, first.z, 0.0);
    pos[leaf] = l;
    cnt[l] = (uint32_t)((leaf_begin[leaf + 1] - leaf_begin[leaf] + TPL - 1) / TPL);
}

template <int TPL>
__global__ void __launch_bounds__(256) k_pair_lanes(const int32_t* __restrict__ leaf_of,
                                                   const int32_t* __restrict__ leaf_begin,
                                                   const int32_t* __restrict__ pos,
                                                   const uint32_t* __restrict__ slot_begin, int64_t n,
                                                   int32_t* __restrict__ lanes)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int leaf = leaf_of[s];
    const int64_t k = s - leaf_begin[leaf];
    if (k % TPL == 0) lanes[slot_begin[pos[leaf]] + k / TPL] = (int32_t)s;
}

// a source record, read by global (not flat) loads
typedef double rec4 __attribute__((ext_vector_type(4)));
typedef const rec4 __attribute__((address_space(1)))* rec4_ptr;

// max(x, floor) for an x from an arithmetic instruction: fmax would quiet
// floor again in every pass of the loop
__device__ __forceinline__ double max_nf(double x, double floor)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(floor));
    return r;
}

// Output of one target: the sums of its pairs and far field, in the input's
// order and units.  The self pair (clamped at 1e-4) is in the sums; its field
// term is exactly zero.
__device__ __forceinline__ void p2p_write(const LeafArgs& a, int64_t s, double q, double sc, double ph, double fx,
                                          double fy, double fz)
{
    const int64_t o = a.perm[s];
    if (o >= a.n_out) return;
    const double self = a.exclude_self ? rsqrt_nf(1.e-8 * (sc * sc)) : 0.0;
    const double sc2 = sc * sc;
    if (a.pot) a.pot[o] = (ph - q * self) * sc;
    if (a.field) {
        a.field[3 * o] = fx * sc2;
        a.field[3 * o + 1] = fy * sc2;
        a.field[3 * o + 2] = fz * sc2;
    }
}

// parts > 1: part j of a leaf's source list goes to part_out[j * n + s], added
// in order by k_p2p_join.
template <int TPL>
__global__ void __launch_bounds__(256) k_p2p_multi(LeafArgs a, const int32_t* __restrict__ lanes,
                                                  const uint32_t* __restrict__ slot_begin,
                                                  const uint32_t* __restrict__ cnt, int parts,
                                                  const double4* __restrict__ pad, double4* __restrict__ part_out)
{
    const int blk = xcd_local_block(blockIdx.x, gridDim.x);
    const int part = blk % parts;
    const int64_t i = (int64_t)(blk / parts) * blockDim.x + threadIdx.x;
    const int64_t total = (int64_t)slot_begin[a.nleaf - 1] + cnt[a.nleaf - 1];
    const bool active = i < total;
    const int64_t s0 = active ? lanes[i] : 0;
    const int leaf = a.leaf_of[s0];
    const int64_t e = active ? a.leaf_begin[leaf + 1] : 0;
    // targets s0 .. s0 + TPL - 1 of the leaf; past its end the last one is
    // repeated (computed, not written)
    double4 t[TPL];
    double ph[TPL], fx[TPL], fy[TPL], fz[TPL];
#pragma unroll
    for (int u = 0; u < TPL; ++u) {
        const int64_t s = max(min(s0 + u, e - 1), (int64_t)0);
        t[u] = a.src[s];
        ph[u] = fx[u] = fy[u] = fz[u] = 0.0;
        if (a.far && parts == 1) {  // far field from k_l2p
            const double4 f = a.far[s];
            ph[u] = f.x;
            fx[u] = f.y;
            fy[u] = f.z;
            fz[u] = f.w;
        }
    }
    // near-source ranges: 27 entries per leaf (uniform tree) or a CSR list
    const int2* nr = a.nbr + (a.nbr_off ? (int64_t)a.nbr_off[leaf] : (int64_t)leaf * 27);
    const int nrc = active ? a.near_runs[leaf] : 0;
    const double sc = a.leaf_scale ? a.leaf_scale[leaf] : 1.0;
    const double r2min = 1.e-8 * (sc * sc);  // (1e-4 in the system's units)^2
    // this part of the list: its first source's range and offset there
    const int all = active ? a.near_total[leaf] : 0;
    const int first = (int)((int64_t)all * part / parts);
    int nsrc = (int)((int64_t)all * (part + 1) / parts) - first;
    const int left = nsrc;
    // sources of the wave's longest list
    for (int off = 32; off > 0; off >>= 1) nsrc = max(nsrc, __shfl_xor(nsrc, off));
    nsrc = __builtin_amdgcn_readfirstlane(nsrc);
    const rec4_ptr src = (rec4_ptr)(uintptr_t)a.src, zero = (rec4_ptr)(uintptr_t)(pad + leaf);
    rec4_ptr p = zero, end = zero;  // the lane's current range; before the first: at its end
    int64_t step = sizeof(rec4);
    int k = 0, todo = left;  // ranges taken, sources not yet in a taken range
    int2 rn = nrc > 0 ? nr[0] : make_int2(0, 0);
    for (int skip = first; skip > 0 && k < nrc;) {
        const int len = rn.y - rn.x;
        if (skip < len) {
            rn.x += skip;
            break;
        }
        skip -= len;
        rn = nr[min(++k, nrc - 1)];
    }
    auto next = [&]() -> rec4 {
        if (p == end) {
            if (todo > 0) {
                const int len = min(rn.y - rn.x, todo);
                p = src + rn.x;
                end = p + len;
                todo -= len;
                rn = nr[min(++k, nrc - 1)];
            } else {  // past its list: the leaf's zero charge from here on
                p = zero;
                end = src;  // never reached: the step is 0
                step = 0;
            }
        }
        const rec4 q = *p;
        p = (rec4_ptr)((uintptr_t)p + step);
        return q;
    };
    auto pairs = [&](const rec4& q) {
#pragma unroll
        for (int u = 0; u < TPL; ++u) {
            const double dx = t[u].x - q.x, dy = t[u].y - q.y, dz = t[u].z - q.z;
            const double r2 = max_nf(fma(dx, dx, fma(dy, dy, dz * dz)), r2min);
            const double ir = rsqrt_nf(r2);
            const double qi = q.w * ir;
            const double qi3 = qi * (ir * ir);
            ph[u] += qi;
            fx[u] = fma(dx, qi3, fx[u]);
            fy[u] = fma(dy, qi3, fy[u]);
            fz[u] = fma(dz, qi3, fz[u]);
        }
    };
    // two sources ahead of their pairs: the next record is in flight while
    // one is used
    rec4 qa = next();
    for (int it = 0; it < nsrc; it += 2) {
        const rec4 qb = next();
        pairs(qa);
        qa = next();
        pairs(qb);
    }
#pragma unroll
    for (int u = 0; u < TPL; ++u) {
        if (s0 + u >= e) break;
        if (parts > 1) part_out[(int64_t)part * a.n + s0 + u] = make_double4(ph[u], fx[u], fy[u], fz[u]);
        else p2p_write(a, s0 + u, t[u].w, sc, ph[u], fx[u], fy[u], fz[u]);
    }
}

__global__ void __launch_bounds__(256) k_p2p_join(LeafArgs a, const double4* __restrict__ part_out, int parts)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= a.n) return;
    double4 v = a.far ? a.far[s] : make_double4(0.0, 0.0, 0.0, 0.0);
    for (int j = 0; j < parts; ++j) {
        const double4 w = part_out[(int64_t)j * a.n + s];
        v.x += w.x;
        v.y += w.y;
        v.z += w.z;
        v.w += w.w;
    }
    const double sc = a.leaf_scale ? a.leaf_scale[a.leaf_of[s]] : 1.0;
    p2p_write(a, s, a.src[s].w, sc, v.x, v.y, v.z, v.w);
}

inline int nblk(int64_t n, int t) { return (int)((n + t - 1) / t); }

}  // namespace

// upper bound on the lane count: sum over leaves of ceil(count / tpl)
inline int64_t lane_bound(int64_t n, int64_t nleaf, int tpl) { return (n + (tpl - 1) * nleaf) / tpl + 1; }

// targets per lane: 4 halves the source loads per pair and the lane setup, but
// wastes more of a lane at a leaf's end
inline int p2p_tpl(int64_t n, int64_t nleaf) { return n >= 64 * nleaf ? 4 : 2; }

// Parts of every source list.  A wave runs its longest list, so few waves
// leave the chip idle (50,000 particles in 64 leaves: 195 waves for 1,024
// SIMDs; 4.7 ms in one part, 0.6 in 64) or end unevenly (400,000 in 512: 8.6
// -> 4.9 ms).  16 waves per SIMD keep all of them busy to the end (8: 3% less
// on 1M particles in 4,096 leaves).  A part of a list of average length has at
// least 128 sources (256: 65,536 particles in 4,096 leaves 0.081 -> 0.128 ms); shorter
// lists are split as often.
static int p2p_parts(int64_t n, int64_t nleaf)
{
    const int64_t waves = n / (64 * p2p_tpl(n, nleaf)) + 1;
    const int64_t near = std::min<int64_t>(27, nleaf) * n / nleaf;
    return (int)std::max<int64_t>(1, std::min<int64_t>({16384 / waves, near / 128, 64}));
}

static int64_t p2p_head_elems(int64_t n, int64_t nleaf) { return (lane_bound(n, nleaf, 2) + 3 * nleaf + 7) / 8 * 8; }

int64_t p2p_ws_elems(int64_t n, int64_t nleaf)
{
    const int parts = p2p_parts(n, nleaf);
    return p2p_head_elems(n, nleaf) + (nleaf + (parts > 1 ? parts * n : 0)) * (int64_t)(sizeof(double4) / sizeof(int32_t));
}

template <int TPL>
static hipError_t p2p_launch(const LeafArgs& a, int32_t* ws, uint32_t* scan_ws, hipStream_t st)
{
    // ws: cnt, slot_begin, pos [nleaf each], lanes [lane_bound], then pad [nleaf] and the parts' sums
    uint32_t* cnt = (uint32_t*)ws;
    uint32_t* slot = cnt + a.nleaf;
    int32_t* pos = (int32_t*)(slot + a.nleaf);
    int32_t* lanes = pos + a.nleaf;
    const int parts = p2p_parts(a.n, a.nleaf);
    double4* pad = (double4*)(ws + p2p_head_elems(a.n, a.nleaf));
    double4* part_out = parts > 1 ? pad + a.nleaf : nullptr;
    // Leaves ordered by their source counts end together in a wave (lanes in
    // use on 4M uniform particles: 90 -> 97%), at the price of locality:
    // adaptive lists differ most (512: 4M clustered particles 4.3 -> 3.6 ms),
    // uniform ones less (256: 4M particles 1.95 -> 1.74 ms); with few, large leaves only
    // near neighbours are exchanged (400,000 particles in 512 leaves: 5.4 ms
    // unordered, 4.9 with 32, 6.2 with 256), or none (64 leaves).
    const dim3 grid(nblk(a.nleaf, 512)), block(512);
    if (a.nbr_off)
        hipLaunchKernelGGL((k_pair_counts<TPL, 512>), grid, block, 0, st, a.leaf_begin, a.near_total, a.nleaf, cnt, pos,
                           a.src, pad);
    else if (a.nleaf >= 2048)
        hipLaunchKernelGGL((k_pair_counts<TPL, 256>), grid, block, 0, st, a.leaf_begin, a.near_total, a.nleaf, cnt, pos,
                           a.src, pad);
    else if (a.nleaf >= 256)
        hipLaunchKernelGGL((k_pair_counts<TPL, 32>), grid, block, 0, st, a.leaf_begin, a.near_total, a.nleaf, cnt, pos,
                           a.src, pad);
    else
        hipLaunchKernelGGL((k_pair_counts<TPL, 1>), grid, block, 0, st, a.leaf_begin, a.near_total, a.nleaf, cnt, pos,
                           a.src, pad);
    hipError_t e = exclusive_scan(cnt, slot, a.nleaf, scan_ws, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_pair_lanes<TPL>), dim3(nblk(a.n, 256)), dim3(256), 0, st, a.leaf_of, a.leaf_begin, pos, slot,
                       a.n, lanes);
    const int64_t bound = lane_bound(a.n, a.nleaf, TPL);
    hipLaunchKernelGGL((k_p2p_multi<TPL>), dim3(nblk(bound, 256) * parts), dim3(256), 0, st, a, lanes, slot, cnt, parts,
                       pad, part_out);
    if (parts > 1) hipLaunchKernelGGL(k_p2p_join, dim3(nblk(a.n, 256)), dim3(256), 0, st, a, part_out, parts);
    return hipGetLastError();
}

hipError_t launch_p2p(const LeafArgs& a, int32_t* ws, uint32_t* scan_ws, hipStream_t st)
{
    if (a.n <= 0 || a.nleaf <= 0) return hipSuccess;
    return p2p_tpl(a.n, a.nleaf) == 4 ? p2p_launch<4>(a, ws, scan_ws, st) : p2p_launch<2>(a, ws, scan_ws, st);
}

}  // namespace lfmm
