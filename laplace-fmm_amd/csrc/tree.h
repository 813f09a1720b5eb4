// tree.h -- host entry points of the GPU octree build (tree.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>
#include <vector>

namespace lfmm {

constexpr int kMaxLevels = 32;
constexpr int kHostInfoBytes = 4096;  // pinned host memory that build kernels write for the host

// What the host reads of a build: level sizes, the fullest boxes and the
// level that fits leaf_max (see count_levels), geom[0..4].
struct LevelInfo {
    uint32_t count[kMaxLevels];
    uint32_t most[3];
    double geom[5];
};

// Level arrays (l <= leaf level): keys and begin have count[l] (+ 1) entries;
// begin: first child, at the leaves first particle; optional: first = first
// particle, parent = box number one level up, lut = dense key -> box (holds -1
// everywhere).  leaf_of[particle] = its leaf.
struct LevelOut {
    uint64_t* keys[kMaxLevels];
    int32_t* begin[kMaxLevels];
    int32_t* first[kMaxLevels];
    int32_t* parent[kMaxLevels];
    int32_t* lut[kMaxLevels];
    uint32_t count[kMaxLevels];
    int32_t* leaf_of;
};

// dim = 2 (quadtree, x << 1 | y keys) or 3 (octree).
// geom[5] = {shift_x, shift_y, shift_z, scale, 1 if a coordinate is not finite};
// part needs 7 * 1024 doubles.
hipError_t extent(int dim, const double* pos, int64_t stride, int64_t n, double* part, double* geom, hipStream_t st);
// v: 0 .. n - 1; clear[0 .. 2] = 0
hipError_t keys(int dim, const double* pos, int64_t stride, int64_t n, int bits, const double* geom, uint64_t* k,
                uint32_t* v, uint32_t* clear, hipStream_t st);
int64_t scan_ws_elems(int64_t n);
// out[j] = in[0] + .. + in[j - 1]; ws: scan_ws_elems(n).  May be in place.
hipError_t exclusive_scan(const uint32_t* in, uint32_t* out, int64_t n, uint32_t* ws, hipStream_t st);
int64_t sort_ws_bytes(int64_t n);
// Stable LSD radix sort of (keys, vals) on the low `bits` bits; results land
// in *keys_res / *vals_res (either the inputs or the workspace).
hipError_t radix_sort(uint64_t* keys, uint32_t* vals, int64_t n, int bits, void* ws, hipStream_t st,
                      uint64_t** keys_res, uint32_t** vals_res);
// (x, y, z, q) records from a strided view (q = 0 when q is null; z = 0 in 2D).
hipError_t pack_points(int dim, const double* pos, int64_t ps, const double* q, int64_t qs, int64_t n, double4* out,
                       hipStream_t st);
// Per-leaf source/target partition of the sorted order (q != 0 first).
hipError_t partition_leaves(const int32_t* begin, int64_t nleaf, uint32_t* order, const double* q, int64_t qs,
                            hipStream_t st);
hipError_t gather_sources(int dim, const double* pos, int64_t pstride, const double* q, int64_t qstride,
                          const uint32_t* order, int64_t n, double4* src, hipStream_t st);
// Levels of sorted keys of level key_level.  count_levels: sizes to *host
// (pinned; there once the stream is waited for), with the fullest box of
// key_level and of the level above (most[0], most[1]) and, for leaf_max > 0, the
// smallest level at which no box holds more than leaf_max particles (most[2];
// key_level + 1: none); most: 3 words, 0 before; sums [level_tiles(n) *
// (key_level + 1)].  emit_levels then fills the arrays of levels 0 ..
// leaf_level <= key_level, and leaf_order puts the particles of every leaf
// back in input order (needed where leaf_level < key_level).
int64_t level_tiles(int64_t n);
hipError_t count_levels(int dim, const uint64_t* keys, int64_t n, int key_level, int leaf_max, uint32_t* sums,
                        const double* geom, uint32_t* most, LevelInfo* host, hipStream_t st);
hipError_t emit_levels(int dim, const uint64_t* keys, int64_t n, int key_level, int leaf_level, const uint32_t* sums,
                       const LevelOut& out, hipStream_t st);
hipError_t leaf_order(const int32_t* leaf_of, const int32_t* begin, int64_t n, const uint32_t* in, uint32_t* out,
                      hipStream_t st);
// Exact M2L and near-field pair counts of a built tree (report only); ws
// holds 2 + depth counters, m2l_per_level (optional) depth entries;
// p2p_reads (optional): the particles of every leaf's near list, summed over
// the leaves.  Synchronises.
hipError_t count_ops(int dim, const std::vector<uint64_t*>& keys, const std::vector<int32_t*>& begin,
                     const std::vector<int32_t*>& lut, const std::vector<int64_t>& cnt, unsigned long long* ws,
                     int64_t* m2l_ops, int64_t* p2p_pairs, int64_t* m2l_per_level, hipStream_t st,
                     int64_t* p2p_reads = nullptr);
// nbr[leaf][0 .. runs[leaf]) (3^dim entries per leaf) = particle ranges of the
// neighbour leaves, joined where they touch; total[leaf] their particles;
// pad[leaf] (optional) = a zero charge at the leaf's first particle
hipError_t launch_leaf_ranges(int dim, const uint64_t* leaf_key, const int32_t* leaf_begin, int nleaf, int level,
                              const int32_t* lut, int2* nbr, int32_t* total, int32_t* runs, hipStream_t st,
                              const double4* src = nullptr, double4* pad = nullptr);
// p[0..n) = v with a fill kernel (safe inside stream capture)
hipError_t fill_u32(uint32_t* p, int64_t n, uint32_t v, hipStream_t st);
}  // namespace lfmm
