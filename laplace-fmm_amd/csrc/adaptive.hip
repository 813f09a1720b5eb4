// adaptive.hip -- adaptive octree and its interaction lists on the GPU.
//
// Start: the uniform tree of the deepest level any box needs (every box of
// it holds at most leaf_max particles), built by build_tree with parent
// indices.  A uniform box belongs to the adaptive tree iff its parent holds
// more than leaf_max particles (then so does every ancestor); it is a leaf
// iff it holds at most leaf_max particles or sits on the deepest level.  The
// kept boxes of each level are compacted in key order; leaves are listed
// globally in particle (Morton) order, where they tile [0, n).
//
// Lists (definitions in adaptive.h):
//   U  per leaf: the leaf itself, the leaves of its level or coarser that
//      hold one of its 26 neighbour cells (walk up the levels from the cell),
//      and the finer leaves that found it that way (pairs transposed by a
//      stable sort, so every list has a fixed order)
//   X  per box b (levels >= 2): the coarser leaves that hold a neighbour cell
//      of b's parent and do not touch b
//   W  per leaf: the X pairs transposed (stable sort by leaf)
// Every list keeps a deterministic order, so the sums of a solve do not
// depend on timing.
#include "adaptive.h"
#include "api_internal.h"
#include "device_common.h"
#include "scan.h"
#include "tree.h"

namespace lfmm {

namespace {

inline int nblk(int64_t n, int t) { return (int)((n + t - 1) / t); }

__device__ inline int ad_level(const AdLevels& A, int g)
{
    int l = 0;
    while (l + 1 < A.depth && g >= A.off[l + 1]) ++l;
    return l;
}

__device__ inline int ad_find(const AdLevels& A, int l, uint64_t key)
{
    return find_box(key, A.lut[l], A.keys + A.off[l], A.off[l + 1] - A.off[l]);
}

// The leaf (gid) that holds cell (x, y, z) of level l, at level l or above;
// -2 when a box with children holds the cell at level l (finer leaves below
// it); -1 when no particle lies in the cell.
__device__ inline int ad_cover(const AdLevels& A, int l, int x, int y, int z)
{
    for (int lv = l; lv >= 0; --lv) {
        const int sh = l - lv;
        const int j = ad_find(A, lv, morton3((uint32_t)x >> sh, (uint32_t)y >> sh, (uint32_t)z >> sh));
        if (j >= 0) {
            const int g = A.off[lv] + j;
            if (A.box2leaf[g] >= 0) return g;
            return lv == l ? -2 : -1;
        }
    }
    return -1;
}

// The uniform levels the adaptive tree is cut from, concatenated: level l's
// boxes are off[l] .. off[l + 1] - 1, its begin and first arrays (one entry
// more per level) start at off[l] + l.  All levels together can hold several
// times the particles (a deep tree of a dense clump in an even background).
struct UniLevels {
    int depth;
    int64_t off[kAdMaxLevels + 1];
    const uint64_t* keys;
    const int32_t* child;
    const int32_t* first;
    const int32_t* parent;
};

__device__ inline int uni_level(const UniLevels& U, int64_t j)
{
    int l = 0;
    while (l + 1 < U.depth && j >= U.off[l + 1]) ++l;
    return l;
}

// what the list kernels report to the host
struct AdInfo {
    int32_t loff[kAdMaxLevels + 1];  // first box of each level
    uint32_t max_leaf;
    int32_t ioff[kAdMaxLevels + 1];  // boxes with children before each level
    uint32_t nleaf, fine_pairs, x_pairs, u_total, n_total;
    uint32_t xseg[kAdMaxLevels + 1];
};

// 1 for a box that is kept: its parent holds more than leaf_max particles
struct AdKeep {
    UniLevels U;
    int leaf_max, min_leaf_level;
    __device__ uint32_t operator()(int64_t j) const
    {
        if (j >= U.off[U.depth]) return 0u;
        const int l = uni_level(U, j);
        if (l == 0 || l <= min_leaf_level) return 1u;
        const int32_t* f = U.first + U.off[l - 1] + (l - 1) + U.parent[j];
        return f[1] - f[0] > leaf_max ? 1u : 0u;
    }
};

struct AdKeepOut {
    UniLevels U;
    uint32_t* kex;
    AdInfo* host;
    __device__ void operator()(int64_t j, uint32_t before) const
    {
        kex[j] = before;
        for (int l = 0; l <= U.depth; ++l)
            if (j == U.off[l]) host->loff[l] = (int32_t)before;
    }
};

// The kept boxes: numbered level by level (kex), so child and leaf numbers
// follow from the scan.  child: level l's kept boxes start at A.off[l] + l.
__global__ void __launch_bounds__(256) k_ad_fill(UniLevels U, AdLevels A, const uint32_t* __restrict__ kex, int leaf_max,
                                                 int min_leaf_level, uint64_t* __restrict__ keys_all,
                                                 int2* __restrict__ range_all, int32_t* __restrict__ child,
                                                 int32_t* __restrict__ box2leaf, int32_t* __restrict__ tag)
{
    const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (j < U.depth) child[A.off[j + 1] + j] = j + 1 < U.depth ? A.off[j + 2] - A.off[j + 1] : 0;
    if (j >= U.off[U.depth]) return;
    const int g = (int)kex[j];
    if ((int)kex[j + 1] == g) return;
    const int l = uni_level(U, j);
    const bool last = l + 1 == U.depth;
    const int b = U.first[j + l], e = U.first[j + l + 1];
    const uint64_t key = U.keys[j];
    keys_all[g] = key;
    range_all[g] = make_int2(b, e);
    // a leaf's uniform children are not kept: its child range is empty
    child[g + l] = last ? 0 : (int)kex[U.off[l + 1] + U.child[j + l]] - A.off[l + 1];
    const bool leaf = last || (l >= min_leaf_level && e - b <= leaf_max);
    box2leaf[g] = leaf ? 0 : -1;
    if (leaf) tag[b] = g;  // its first particle
    if (A.lut[l]) const_cast<int32_t*>(A.lut[l])[key] = g - A.off[l];
}

struct AdTagged {
    const int32_t* tag;
    __device__ uint32_t operator()(int64_t s) const { return tag[s] >= 0 ? 1u : 0u; }
};

struct AdLeafOut {
    AdLevels A;
    const int32_t* tag;
    int64_t n;
    int32_t* box2leaf;
    int32_t* leaf_begin;
    int32_t* leaf_gid;
    uint64_t* leaf_key;
    int32_t* leaf_lvl;
    int32_t* leaf_of;
    uint32_t* nleaf;
    AdInfo* host;
    __device__ void operator()(int64_t s, uint32_t before) const
    {
        const int g = tag[s];
        const int i = (int)before + (g >= 0 ? 1 : 0) - 1;  // particle 0 always starts a leaf
        leaf_of[s] = i;
        if (g >= 0) {
            leaf_begin[i] = (int32_t)s;
            leaf_gid[i] = g;
            leaf_key[i] = A.keys[g];
            leaf_lvl[i] = ad_level(A, g);
            box2leaf[g] = i;
        }
        if (s == n - 1) {
            leaf_begin[i + 1] = (int32_t)n;
            *nleaf = (uint32_t)(i + 1);
            host->nleaf = (uint32_t)(i + 1);
        }
    }
};

// The list kernels give a leaf or box half a wave: lane o < 27 looks up cell
// o, a vote over the half gives each found cell its place, and the half's
// reads and writes are consecutive (a thread per leaf kept its 27 cells in
// scratch memory and wrote rows 27 apart).
constexpr int kHalf = 32;
constexpr int kHalves = 256 / kHalf;  // per workgroup

__device__ inline uint32_t half_ballot(bool v) { return (uint32_t)(__ballot(v) >> (threadIdx.x & 32)); }
__device__ inline int half_rank(uint32_t m) { return __popc(m & ((1u << (threadIdx.x & 31)) - 1u)); }

// true where an earlier lane of the half holds the same c (c < 0: never)
__device__ inline bool seen_before(int c)
{
    const int o = threadIdx.x & 31;
    bool seen = false;
#pragma unroll
    for (int k = 0; k < 27; ++k) seen |= __shfl(c, k, kHalf) == c && k < o;
    return seen && c >= 0;
}

// U lists, first part: per leaf, the 27 cells around it (offset order) mapped
// to the leaf holding each at its level or coarser; a coarser leaf that holds
// several cells is kept at its first cell.  nbr27 = leaf index or -1.
__global__ void __launch_bounds__(256) k_ad_u1(AdLevels A, const int32_t* __restrict__ leaf_gid,
                                               const int32_t* __restrict__ leaf_lvl,
                                               const int32_t* __restrict__ leaf_begin, const uint32_t* __restrict__ nleaf,
                                               int32_t* __restrict__ nbr27, uint32_t* __restrict__ nu1,
                                               uint32_t* __restrict__ ncoarse, uint32_t* __restrict__ max_leaf)
{
    const int i = blockIdx.x * kHalves + threadIdx.x / kHalf, o = threadIdx.x & 31;
    const bool live = i < (int)*nleaf;
    block_max_u32(live ? (uint32_t)(leaf_begin[i + 1] - leaf_begin[i]) : 0u, max_leaf);
    int r = -1;
    bool coarse = false;
    if (live && o < 27) {
        const int g = leaf_gid[i], l = leaf_lvl[i];
        const uint64_t key = A.keys[g];
        const int cx = (int)compact3(key >> 2) + o / 9 - 1, cy = (int)compact3(key >> 1) + (o / 3) % 3 - 1,
                  cz = (int)compact3(key) + o % 3 - 1;
        const int side = 1 << l;
        if (o == 13) r = g;
        else if (cx >= 0 && cy >= 0 && cz >= 0 && cx < side && cy < side && cz < side) r = max(ad_cover(A, l, cx, cy, cz), -1);
        coarse = r >= 0 && r < A.off[l];
    }
    if (seen_before(r) && coarse) r = -1;
    const uint32_t found = half_ballot(r >= 0), up = half_ballot(r >= 0 && coarse);
    if (!live) return;
    if (o < 27) nbr27[(int64_t)i * 27 + o] = r >= 0 ? A.box2leaf[r] : -1;
    if (o == 0) {
        nu1[i] = (uint32_t)__popc(found);
        ncoarse[i] = (uint32_t)__popc(up);
    }
}

// (coarse leaf, this leaf) pairs for the transposition, in leaf order
__global__ void __launch_bounds__(256) k_ad_u_pairs(const int32_t* __restrict__ nbr27, const int32_t* __restrict__ leaf_lvl,
                                                    int nleaf, const uint32_t* __restrict__ coff,
                                                    uint64_t* __restrict__ pk, uint32_t* __restrict__ pv,
                                                    uint32_t* __restrict__ finecnt)
{
    const int i = blockIdx.x * kHalves + threadIdx.x / kHalf, o = threadIdx.x & 31;
    const int j = i < nleaf && o < 27 ? nbr27[(int64_t)i * 27 + o] : -1;
    const bool up = j >= 0 && leaf_lvl[j] < leaf_lvl[i];
    const uint32_t m = half_ballot(up);
    if (!up) return;
    const uint32_t w = coff[i] + half_rank(m);
    pk[w] = (uint64_t)j;
    pv[w] = (uint32_t)i;
    atomicAdd(&finecnt[j], 1u);
}

__global__ void __launch_bounds__(256) k_ad_u_fill(const int32_t* __restrict__ nbr27, const int32_t* __restrict__ leaf_begin,
                                                   int nleaf, const uint32_t* __restrict__ uoff,
                                                   const uint32_t* __restrict__ fine_off,
                                                   const uint32_t* __restrict__ finecnt,
                                                   const uint32_t* __restrict__ fine_leaf, int2* __restrict__ urng)
{
    const int i = blockIdx.x * kHalves + threadIdx.x / kHalf, o = threadIdx.x & 31;
    const int j = i < nleaf && o < 27 ? nbr27[(int64_t)i * 27 + o] : -1;
    const uint32_t m = half_ballot(j >= 0);
    if (i >= nleaf) return;
    const uint32_t w = uoff[i];
    if (j >= 0) urng[w + half_rank(m)] = make_int2(leaf_begin[j], leaf_begin[j + 1]);
    const uint32_t fb = fine_off[i], fc = finecnt[i], wf = w + __popc(m);
    for (uint32_t k = o; k < fc; k += kHalf) {
        const int f = (int)fine_leaf[fb + k];
        urng[wf + k] = make_int2(leaf_begin[f], leaf_begin[f + 1]);
    }
}

// X lists: per box of levels >= 2 (t = gid - g2), the leaves coarser than it
// that hold a neighbour cell of its parent and do not touch it.
__global__ void __launch_bounds__(256) k_ad_x(AdLevels A, int g2, int total, int32_t* __restrict__ x27,
                                              uint32_t* __restrict__ xcnt)
{
    const int t = blockIdx.x * kHalves + threadIdx.x / kHalf, o = threadIdx.x & 31;
    int c = -1;
    if (t < total - g2 && o < 27) {
        const int g = g2 + t;
        const int l = ad_level(A, g);
        const uint64_t key = A.keys[g];
        const int x = (int)compact3(key >> 2), y = (int)compact3(key >> 1), z = (int)compact3(key);
        const int cx = (x >> 1) + o / 9 - 1, cy = (y >> 1) + (o / 3) % 3 - 1, cz = (z >> 1) + o % 3 - 1;
        const int pside = 1 << (l - 1);
        if (cx >= 0 && cy >= 0 && cz >= 0 && cx < pside && cy < pside && cz < pside) c = ad_cover(A, l - 1, cx, cy, cz);
        if (c >= 0) {
            // c: a leaf at level lc <= l - 1; in units of level-l cells it
            // spans [c * s, (c + 1) * s) per axis
            const int lc = ad_level(A, c);
            const uint64_t ck = A.keys[c];
            const int s = 1 << (l - lc);
            const int ax = (int)compact3(ck >> 2) * s, ay = (int)compact3(ck >> 1) * s, az = (int)compact3(ck) * s;
            const bool touch = x <= ax + s && x + 1 >= ax && y <= ay + s && y + 1 >= ay && z <= az + s && z + 1 >= az;
            if (touch) c = -1;
        }
    }
    const bool seen = seen_before(c);
    const bool take = c >= 0 && !seen;
    const uint32_t m = half_ballot(take);
    if (t >= total - g2) return;
    if (take) x27[(int64_t)t * 27 + half_rank(m)] = A.box2leaf[c];
    if (o == 0) xcnt[t] = (uint32_t)__popc(m);
}

__global__ void __launch_bounds__(256) k_ad_x_fill(const int32_t* __restrict__ x27, const uint32_t* __restrict__ xcnt,
                                                   const uint32_t* __restrict__ xoff, int nb,
                                                   const int32_t* __restrict__ leaf_begin, int g2,
                                                   int2* __restrict__ xrng, uint64_t* __restrict__ wk,
                                                   uint32_t* __restrict__ wv, uint32_t* __restrict__ wcnt,
                                                   int32_t* __restrict__ xlist, const uint32_t* __restrict__ lex,
                                                   const int32_t* __restrict__ box2leaf)
{
    const int t = blockIdx.x * kHalves + threadIdx.x / kHalf;
    const uint32_t k = threadIdx.x & 31;
    if (t >= nb) return;
    const uint32_t c = xcnt[t];
    if (k >= c) return;
    if (k == 0 && box2leaf[g2 + t] < 0) xlist[lex[t]] = t;  // P2L for boxes with children only
    const uint32_t w = xoff[t] + k;
    const int j = x27[(int64_t)t * 27 + k];
    xrng[w] = make_int2(leaf_begin[j], leaf_begin[j + 1]);
    wk[w] = (uint64_t)j;
    wv[w] = (uint32_t)(g2 + t);
    atomicAdd(&wcnt[j], 1u);
}

// Near lists of the pair kernel: the U list, then the leaf's X sources (a
// leaf target: direct sums, cheaper and exact), then the W boxes of at most
// direct_max particles (direct sums instead of M2P).
__global__ void __launch_bounds__(256) k_ad_near_count(const int32_t* __restrict__ leaf_gid, int nleaf,
                                                       const uint32_t* __restrict__ u_off,
                                                       const uint32_t* __restrict__ x_off, int g2,
                                                       const uint32_t* __restrict__ w_off,
                                                       const int32_t* __restrict__ w_gid, const int2* __restrict__ range,
                                                       int direct_max, uint32_t* __restrict__ ncnt)
{
    const int i = blockIdx.x * kHalves + threadIdx.x / kHalf;
    const uint32_t o = threadIdx.x & 31;
    if (i >= nleaf) return;
    uint32_t c = 0;
    if (w_gid)
        for (uint32_t k = w_off[i] + o; k < w_off[i + 1]; k += kHalf) {
            const int2 r = range[w_gid[k]];
            c += (r.y - r.x <= direct_max) ? 1u : 0u;
        }
    for (int off = 16; off > 0; off >>= 1) c += (uint32_t)__shfl_xor((int)c, off, kHalf);
    if (o != 0) return;
    const int g = leaf_gid[i];
    c += u_off[i + 1] - u_off[i];
    if (x_off && g >= g2) c += x_off[g - g2 + 1] - x_off[g - g2];
    ncnt[i] = c;
}

__global__ void __launch_bounds__(256) k_ad_near_fill(const int32_t* __restrict__ leaf_gid, int nleaf,
                                                      const uint32_t* __restrict__ u_off, const int2* __restrict__ u_rng,
                                                      const uint32_t* __restrict__ x_off, const int2* __restrict__ x_rng,
                                                      int g2, const uint32_t* __restrict__ w_off,
                                                      const int32_t* __restrict__ w_gid, const int2* __restrict__ range,
                                                      int direct_max, const uint32_t* __restrict__ n_off,
                                                      int2* __restrict__ n_rng, int32_t* __restrict__ n_sources,
                                                      int32_t* __restrict__ n_runs, int32_t* __restrict__ m2p_gid,
                                                      int32_t* __restrict__ m2p_count)
{
    const int i = blockIdx.x * kHalves + threadIdx.x / kHalf;
    const uint32_t o = threadIdx.x & 31;
    if (i >= nleaf) return;
    const int g = leaf_gid[i];
    uint32_t w = n_off[i];
    int sum = 0;
    auto copy = [&](const int2* from, uint32_t c) {
        for (uint32_t k = o; k < c; k += kHalf) {
            const int2 r = from[k];
            n_rng[w + k] = r;
            sum += r.y - r.x;
        }
        w += c;
    };
    copy(u_rng + u_off[i], u_off[i + 1] - u_off[i]);
    if (x_off && g >= g2) copy(x_rng + x_off[g - g2], x_off[g - g2 + 1] - x_off[g - g2]);
    uint32_t big = 0;  // W boxes left to M2P
    if (w_gid)
        for (uint32_t b = w_off[i], e = w_off[i + 1]; b < e; b += kHalf) {  // the half stays together
            const int gw = b + o < e ? w_gid[b + o] : -1;
            const int2 r = gw >= 0 ? range[gw] : make_int2(0, 0);
            const bool take = gw >= 0 && r.y - r.x <= direct_max;
            const uint32_t m = half_ballot(take), mb = half_ballot(gw >= 0 && !take);
            if (gw >= 0 && !take) m2p_gid[w_off[i] + big + half_rank(mb)] = gw;
            big += __popc(mb);
            if (take) {
                n_rng[w + half_rank(m)] = r;
                sum += r.y - r.x;
            }
            w += __popc(m);
        }
    for (int off = 16; off > 0; off >>= 1) sum += __shfl_xor(sum, off, kHalf);
    if (o == 0) {
        n_sources[i] = sum;
        n_runs[i] = (int32_t)(w - n_off[i]);
        m2p_count[i] = (int32_t)big;
    }
}

// boxes with children: numbered within their level (slot, -1: none) and
// listed (list: index at the level, levels one after another)
struct AdInner {
    const int32_t* box2leaf;
    int64_t n;
    __device__ uint32_t operator()(int64_t g) const { return g < n && box2leaf[g] < 0 ? 1u : 0u; }
};

struct AdInnerOut {
    AdLevels A;
    const int32_t* box2leaf;
    int64_t n;
    uint32_t* before_all;
    int32_t* list;
    AdInfo* host;
    __device__ void operator()(int64_t g, uint32_t before) const
    {
        before_all[g] = before;
        for (int l = 0; l <= A.depth; ++l)
            if (g == A.off[l]) host->ioff[l] = (int32_t)before;
        if (g < n && box2leaf[g] < 0) list[before] = (int32_t)g - A.off[ad_level(A, (int)g)];
    }
};

__global__ void __launch_bounds__(256) k_ad_slots(AdLevels A, const int32_t* __restrict__ box2leaf, int n,
                                                  const uint32_t* __restrict__ before, int32_t* __restrict__ slot)
{
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < n) slot[g] = box2leaf[g] < 0 ? (int32_t)(before[g] - before[A.off[ad_level(A, g)]]) : -1;
}

// ---- inputs and outputs of the scans: counts of `live` entries (then zeros)
// into offsets; the total goes to the host
struct AdCount {
    const uint32_t* c;
    const uint32_t* live;  // null: the static bound n
    int64_t n;
    __device__ uint32_t operator()(int64_t j) const { return j < (live ? (int64_t)*live : n) ? c[j] : 0u; }
};

struct AdSum2 {
    const uint32_t *a, *b;
    int64_t n;
    __device__ uint32_t operator()(int64_t j) const { return j < n ? a[j] + b[j] : 0u; }
};

// boxes whose X list runs as P2L: those with children (a leaf takes its X
// sources in its near list instead)
struct AdP2l {
    const uint32_t* c;
    const int32_t* box2leaf;  // of the first box with an X list
    int64_t n;
    __device__ uint32_t operator()(int64_t j) const { return j < n && c[j] && box2leaf[j] < 0 ? 1u : 0u; }
};

struct AdOffsets {
    uint32_t* off;
    int64_t n;
    uint32_t* total;  // host, or null
    const uint32_t* max_leaf = nullptr;
    uint32_t* max_out = nullptr;  // host
    __device__ void operator()(int64_t j, uint32_t before) const
    {
        off[j] = before;
        if (j == n && total) *total = before;
        if (j == n && max_leaf) *max_out = *max_leaf;
    }
};

struct AdP2lOut {
    AdLevels A;
    uint32_t* off;
    int g2;
    AdInfo* host;
    __device__ void operator()(int64_t j, uint32_t before) const
    {
        off[j] = before;
        for (int l = 2; l <= A.depth; ++l)
            if (j + g2 == A.off[l]) host->xseg[l] = before;
    }
};

// sum over leaves of (particles) x (particles in its U list)
__global__ void __launch_bounds__(256) k_ad_pairs(const int32_t* __restrict__ leaf_begin, const uint32_t* __restrict__ u_off,
                                                  const int2* __restrict__ u_rng, int64_t nleaf,
                                                  unsigned long long* __restrict__ out)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    unsigned long long c = 0, rd = 0;
    if (i < nleaf) {
        unsigned long long t = 0;
        for (uint32_t k = u_off[i]; k < u_off[i + 1]; ++k) t += (unsigned long long)(u_rng[k].y - u_rng[k].x);
        c = t * (unsigned long long)(leaf_begin[i + 1] - leaf_begin[i]);
        rd = t;
    }
    for (int off = 32; off > 0; off >>= 1) {
        c += (unsigned long long)__shfl_xor((long long)c, off);
        rd += (unsigned long long)__shfl_xor((long long)rd, off);
    }
    if ((threadIdx.x & 63) == 0 && c) atomicAdd(out, c);
    if ((threadIdx.x & 63) == 0 && rd) atomicAdd(out + 1, rd);
}

int bits_for(int64_t v)
{
    int b = 1;
    while (b < 63 && ((int64_t)1 << b) <= v) ++b;
    return b;
}

// A forest leaf's system: its ancestor cell (2a, 2b, 2c) at the system level
// holds system (a side + b) side + c; out = that system's length scale.
__global__ void __launch_bounds__(256) k_forest_leaf_scale(const uint64_t* __restrict__ leaf_key,
                                                           const int32_t* __restrict__ leaf_lvl, int64_t nleaf,
                                                           int level, int side, const double* __restrict__ sys_scale,
                                                           double* __restrict__ out)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= nleaf) return;
    const int lv = leaf_lvl[i];
    const uint64_t k = lv >= level ? leaf_key[i] >> (3 * (lv - level)) : 0;
    const int a = (int)(compact3(k >> 2) >> 1), b = (int)(compact3(k >> 1) >> 1), c = (int)(compact3(k) >> 1);
    out[i] = (lv >= level && a < side && b < side && c < side) ? sys_scale[(a * side + b) * side + c] : 1.0;
}

}  // namespace

}  // namespace lfmm

namespace lfmm::host {

AdLevels Tree::view() const
{
    AdLevels A{};
    A.depth = depth;
    for (int l = 0; l <= depth; ++l) A.off[l] = loff[l];
    A.keys = keys_all;
    for (int l = 0; l < depth; ++l) A.lut[l] = lut[l];
    A.box2leaf = box2leaf;
    A.range = range_all;
    return A;
}

// out[0 .. n]: exclusive sums of the n + 1 values in(j)
template <typename In, typename Out>
static int scan_to(Arena& A, const In& in, const Out& out, int64_t n, hipStream_t st)
{
    uint32_t* ws = take<uint32_t>(A, scan_ws_elems(n + 1));
    if (!ws) return LFMM_ERR_NOMEM;
    LFMM_HIP(scan_apply(in, out, n + 1, ws, st));
    return LFMM_OK;
}

// Three reads of the host wait for the GPU: the kept boxes, the leaves with the
// sizes of both pair lists, the near lists' sizes.  Everything that does not
// size an array runs between them on bounds known to the host.
int build_adaptive(lfmm_ctx* ctx, int leaf_max, Tree& T, int min_leaf_level)
{
    static_assert(sizeof(AdInfo) <= kHostInfoBytes, "the host page holds it");
    hipStream_t st = ctx->stream;
    Arena& A = ctx->arena;
    AdInfo* info = (AdInfo*)ctx->host_info;
    const int depth = T.depth;
    const int64_t n = T.n;
    if (depth > kAdMaxLevels || leaf_max < 1) return LFMM_ERR_INVALID;
    if ((int)T.uparent.size() != depth) return LFMM_ERR_INVALID;
    int rc;

    // ---- kept boxes and their numbering
    UniLevels U{};
    U.depth = depth;
    for (int l = 0; l < depth; ++l) U.off[l + 1] = U.off[l] + T.cnt[l];
    const int64_t utotal = U.off[depth];
    U.keys = T.lkeys[0];
    U.child = T.lbegin[0];
    U.first = T.ufirst[0];
    U.parent = T.uparent[0];
    uint32_t* kex = take<uint32_t>(A, utotal + 1);
    if (!kex) return LFMM_ERR_NOMEM;
    rc = scan_to(A, AdKeep{U, leaf_max, min_leaf_level}, AdKeepOut{U, kex, info}, utotal, st);
    if (rc != LFMM_OK) return rc;
    LFMM_HIP(hipStreamSynchronize(st));
    T.loff.assign(info->loff, info->loff + depth + 1);
    for (int l = 0; l < depth; ++l)
        if (T.loff[l + 1] <= T.loff[l]) return LFMM_ERR_INVALID;  // every level holds a box (the depth needs it)
    const int total = T.loff[depth];
    T.keys_all = take<uint64_t>(A, total);
    T.range_all = take<int2>(A, total);
    T.box2leaf = take<int32_t>(A, total);
    int32_t* child = take<int32_t>(A, total + depth);
    int32_t* tag = take<int32_t>(A, n);
    int64_t dense = 0;
    for (int l = 2; l < depth && l <= lut_max_level(3); ++l) dense += (int64_t)1 << (3 * l);
    int32_t* lut = dense > 0 ? take<int32_t>(A, dense) : nullptr;
    if (!T.keys_all || !T.range_all || !T.box2leaf || !child || !tag || (dense > 0 && !lut)) return LFMM_ERR_NOMEM;
    LFMM_HIP(fill_u32((uint32_t*)tag, n, 0xffffffffu, st));
    if (dense > 0) LFMM_HIP(fill_u32((uint32_t*)lut, dense, 0xffffffffu, st));
    // the tree's level arrays describe the kept boxes from here on
    for (int l = 0; l < depth; ++l) {
        T.cnt[l] = T.loff[l + 1] - T.loff[l];
        T.lkeys[l] = T.keys_all + T.loff[l];
        T.lbegin[l] = child + T.loff[l] + l;
        T.lut[l] = nullptr;
        if (l >= 2 && l <= lut_max_level(3)) {
            T.lut[l] = lut;
            lut += (int64_t)1 << (3 * l);
        }
    }
    T.adaptive = true;
    const AdLevels V = T.view();
    hipLaunchKernelGGL(k_ad_fill, dim3(nblk(utotal, 256)), dim3(256), 0, st, U, V, kex, leaf_max, min_leaf_level,
                       T.keys_all, T.range_all, child, T.box2leaf, tag);

    // ---- global leaf list (particle order); at most `total` leaves
    T.leaf_begin = take<int32_t>(A, total + 1);
    T.leaf_gid = take<int32_t>(A, total);
    T.leaf_key = take<uint64_t>(A, total);
    T.leaf_lvl = take<int32_t>(A, total);
    uint32_t* nleaf = take<uint32_t>(A, 1);
    if (!T.leaf_begin || !T.leaf_gid || !T.leaf_key || !T.leaf_lvl || !nleaf) return LFMM_ERR_NOMEM;
    rc = scan_to(A, AdTagged{tag}, AdLeafOut{V, tag, n, T.box2leaf, T.leaf_begin, T.leaf_gid, T.leaf_key, T.leaf_lvl,
                                             T.leaf_of, nleaf, info}, n - 1, st);
    if (rc != LFMM_OK) return rc;

    // ---- same-level and coarser leaves of the U lists; X lists
    int32_t* nbr27 = take<int32_t>(A, (int64_t)total * 27);
    uint32_t* nu1 = take<uint32_t>(A, total);
    uint32_t* nco = take<uint32_t>(A, total);
    uint32_t* coff = take<uint32_t>(A, total + 1);
    uint32_t* most = T.umax;  // 0: cleared with the counts
    uint32_t* fcnt = take<uint32_t>(A, 2 * (int64_t)total);  // finer touching leaves, then W boxes, per leaf
    uint32_t* wcnt = fcnt + total;
    if (!nbr27 || !nu1 || !nco || !coff || !fcnt) return LFMM_ERR_NOMEM;
    LFMM_HIP(fill_u32(most, 1, 0u, st));
    LFMM_HIP(fill_u32(fcnt, 2 * (int64_t)total, 0u, st));
    hipLaunchKernelGGL(k_ad_u1, dim3(nblk(total, kHalves)), dim3(256), 0, st, V, T.leaf_gid, T.leaf_lvl, T.leaf_begin,
                       nleaf, nbr27, nu1, nco, most);
    rc = scan_to(A, AdCount{nco, nleaf, 0}, AdOffsets{coff, total, &info->fine_pairs, most, &info->max_leaf}, total, st);
    if (rc != LFMM_OK) return rc;
    uint32_t* inner_before = take<uint32_t>(A, total + 1);
    T.inner_list = take<int32_t>(A, total);
    T.inner_slot = take<int32_t>(A, total);
    if (!inner_before || !T.inner_list || !T.inner_slot) return LFMM_ERR_NOMEM;
    rc = scan_to(A, AdInner{T.box2leaf, total}, AdInnerOut{V, T.box2leaf, total, inner_before, T.inner_list, info}, total, st);
    if (rc != LFMM_OK) return rc;
    hipLaunchKernelGGL(k_ad_slots, dim3(nblk(total, 256)), dim3(256), 0, st, V, T.box2leaf, total, inner_before, T.inner_slot);
    const int g2 = depth > 2 ? T.loff[2] : total;
    const int nb = total - g2;
    int32_t* x27 = nullptr;
    uint32_t *xcnt = nullptr, *lex = nullptr;
    info->x_pairs = 0;
    if (nb > 0) {
        x27 = take<int32_t>(A, (int64_t)nb * 27);
        xcnt = take<uint32_t>(A, nb);
        lex = take<uint32_t>(A, nb + 1);
        T.x_off = take<uint32_t>(A, nb + 1);
        if (!x27 || !xcnt || !lex || !T.x_off) return LFMM_ERR_NOMEM;
        hipLaunchKernelGGL(k_ad_x, dim3(nblk(nb, kHalves)), dim3(256), 0, st, V, g2, total, x27, xcnt);
        rc = scan_to(A, AdCount{xcnt, nullptr, nb}, AdOffsets{T.x_off, nb, &info->x_pairs}, nb, st);
        if (rc != LFMM_OK) return rc;
        rc = scan_to(A, AdP2l{xcnt, T.box2leaf + g2, nb}, AdP2lOut{V, lex, g2, info}, nb, st);
        if (rc != LFMM_OK) return rc;
    }
    LFMM_HIP(hipStreamSynchronize(st));
    const int64_t nl = T.nleaf = info->nleaf;
    T.max_leaf = info->max_leaf;
    T.ioff.assign(info->ioff, info->ioff + depth + 1);
    const int64_t npairs = info->fine_pairs;
    T.x_pairs = info->x_pairs;
    T.xseg.assign(depth + 1, 0);
    if (nb > 0) std::copy(info->xseg + 2, info->xseg + depth + 1, T.xseg.begin() + 2);

    // ---- finer leaves of the U lists, W lists: the pairs transposed
    uint32_t* fine_leaf = nullptr;
    if (npairs > 0) {
        uint64_t* pk = take<uint64_t>(A, npairs);
        uint32_t* pv = take<uint32_t>(A, npairs);
        void* sws = A.alloc((size_t)sort_ws_bytes(npairs));
        if (!pk || !pv || !sws) return LFMM_ERR_NOMEM;
        hipLaunchKernelGGL(k_ad_u_pairs, dim3(nblk(nl, kHalves)), dim3(256), 0, st, nbr27, T.leaf_lvl, (int)nl, coff, pk, pv,
                           fcnt);
        uint64_t* sk = pk;
        LFMM_HIP(radix_sort(pk, pv, npairs, bits_for(nl), sws, st, &sk, &fine_leaf));
    }
    uint32_t* foff = take<uint32_t>(A, nl + 1);
    T.u_off = take<uint32_t>(A, nl + 1);
    T.w_off = take<uint32_t>(A, nl + 1);
    if (!foff || !T.u_off || !T.w_off) return LFMM_ERR_NOMEM;
    rc = scan_to(A, AdCount{fcnt, nullptr, nl}, AdOffsets{foff, nl, nullptr}, nl, st);
    if (rc != LFMM_OK) return rc;
    rc = scan_to(A, AdSum2{nu1, fcnt, nl}, AdOffsets{T.u_off, nl, &info->u_total}, nl, st);
    if (rc != LFMM_OK) return rc;
    if (nb > 0) {
        const int64_t xp = T.x_pairs;
        T.x_rng = take<int2>(A, xp);
        T.xlist = take<int32_t>(A, T.xseg[depth]);
        uint64_t* wk = take<uint64_t>(A, xp);
        uint32_t* wv = take<uint32_t>(A, xp);
        void* sws = A.alloc((size_t)sort_ws_bytes(std::max<int64_t>(xp, 1)));
        if (!T.x_rng || !T.xlist || !wk || !wv || !sws) return LFMM_ERR_NOMEM;
        T.w_gid = (int32_t*)wv;
        if (xp > 0) {
            hipLaunchKernelGGL(k_ad_x_fill, dim3(nblk(nb, kHalves)), dim3(256), 0, st, x27, xcnt, T.x_off, nb, T.leaf_begin,
                               g2, T.x_rng, wk, wv, wcnt, T.xlist, lex, T.box2leaf);
            uint64_t* sk = wk;
            uint32_t* sv = wv;
            LFMM_HIP(radix_sort(wk, wv, xp, bits_for(nl), sws, st, &sk, &sv));
            T.w_gid = (int32_t*)sv;
        }
    }
    rc = scan_to(A, AdCount{wcnt, nullptr, nl}, AdOffsets{T.w_off, nl, nullptr}, nl, st);
    if (rc != LFMM_OK) return rc;

    // ---- near lists of the pair kernel: U, plus the X and small W pairs
    // that run as direct sums
    const uint32_t* xo = T.x_pairs > 0 ? T.x_off : nullptr;
    const int32_t* wg = T.x_pairs > 0 ? T.w_gid : nullptr;
    uint32_t* ncnt = take<uint32_t>(A, nl);
    T.n_off = take<uint32_t>(A, nl + 1);
    if (!ncnt || !T.n_off) return LFMM_ERR_NOMEM;
    hipLaunchKernelGGL(k_ad_near_count, dim3(nblk(nl, kHalves)), dim3(256), 0, st, T.leaf_gid, (int)nl, T.u_off, xo, g2,
                       T.w_off, wg, T.range_all, kDirectMax, ncnt);
    rc = scan_to(A, AdCount{ncnt, nullptr, nl}, AdOffsets{T.n_off, nl, &info->n_total}, nl, st);
    if (rc != LFMM_OK) return rc;
    LFMM_HIP(hipStreamSynchronize(st));
    T.u_total = info->u_total;
    T.n_total = info->n_total;
    T.u_rng = take<int2>(A, T.u_total);
    T.n_rng = take<int2>(A, T.n_total);
    T.n_sources = take<int32_t>(A, nl);
    T.n_runs = take<int32_t>(A, nl);
    T.m2p_gid = take<int32_t>(A, T.x_pairs);
    T.m2p_count = take<int32_t>(A, nl);
    if (!T.u_rng || !T.n_rng || !T.n_sources || !T.n_runs || !T.m2p_gid || !T.m2p_count) return LFMM_ERR_NOMEM;
    hipLaunchKernelGGL(k_ad_u_fill, dim3(nblk(nl, kHalves)), dim3(256), 0, st, nbr27, T.leaf_begin, (int)nl, T.u_off, foff,
                       fcnt, fine_leaf, T.u_rng);
    hipLaunchKernelGGL(k_ad_near_fill, dim3(nblk(nl, kHalves)), dim3(256), 0, st, T.leaf_gid, (int)nl, T.u_off, T.u_rng, xo,
                       T.x_rng, g2, T.w_off, wg, T.range_all, kDirectMax, T.n_off, T.n_rng, T.n_sources, T.n_runs,
                       T.m2p_gid, T.m2p_count);
    LFMM_HIP(hipGetLastError());
    return LFMM_OK;
}

int forest_leaf_scale(lfmm_ctx* ctx, const Tree& T, const ForestSpec& fs, double* out)
{
    if (T.nleaf > 0)
        hipLaunchKernelGGL(k_forest_leaf_scale, dim3(nblk(T.nleaf, 256)), dim3(256), 0, ctx->stream, T.leaf_key,
                           T.leaf_lvl, T.nleaf, fs.level, fs.side, fs.sys_scale, out);
    LFMM_HIP(hipGetLastError());
    return LFMM_OK;
}

int ad_count_pairs(const int32_t* leaf_begin, const uint32_t* u_off, const int2* u_rng, int64_t nleaf,
                   unsigned long long* ws, int64_t* pairs, int64_t* reads, hipStream_t st)
{
    LFMM_HIP(fill_u32((uint32_t*)ws, 4, 0u, st));
    hipLaunchKernelGGL(k_ad_pairs, dim3(nblk(nleaf, 256)), dim3(256), 0, st, leaf_begin, u_off, u_rng, nleaf, ws);
    unsigned long long h[2] = {0, 0};
    LFMM_HIP(hipMemcpyAsync(h, ws, 16, hipMemcpyDeviceToHost, st));
    LFMM_HIP(hipStreamSynchronize(st));
    *pairs = (int64_t)h[0];
    if (reads) *reads = (int64_t)h[1];
    return LFMM_OK;
}

}  // namespace lfmm::host
