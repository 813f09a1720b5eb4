// ops2d.h -- argument blocks and launchers of the 2D operator kernels (ops2d.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "lfmm_internal.h"

namespace lfmm {

// Device copies of Pack2d, and of what the FP32 M2L takes from OpTables2d.
struct Tables2d {
    const double* m2l;
    const double* src;
    const double* out;
    const double2* log;
    const double* m2m;
    const double* l2l;
    const double2* down;
    const double2* up;
    const double2* zero;       // an expansion of zeros
    const LogEntry2d* pair_log;
    const float2* m2l32;       // [40][N][N] M2L rounded to FP32 (mixed M2L)
    const int* dir_vec;        // [40][2]
    const int* class_dirs;     // [4][27]
};

struct P2M2dArgs {
    const double4* src;        // sorted (x, y, 0, q)
    const int32_t* leaf_begin;
    const uint64_t* leaf_key;
    int nleaf;
    int level;
    const double* geom;        // {shift x, y, -, scale}
    int N;
    double2* outer;
};

struct M2M2dArgs {
    int N;
    int num_parents;           // boxes at the parent level
    const int32_t* child_begin;
    const uint64_t* child_keys;
    const double2* src;        // multipoles of the child level
    double2* dst;              // multipoles of the parent level
};

struct M2L2dArgs {
    int level;                 // target level
    int num_parents;           // boxes at level - 1
    const int32_t* child_begin;
    const uint64_t* child_keys;   // keys at `level`
    const int32_t* lut;        // dense key -> box table at `level`, or null
    int size;                  // boxes at `level`
    double log_h;              // log of the box edge at `level`
    const double2* src;        // multipoles at `level`
    double2* dst;              // locals at `level` (written)
};

// FP64 M2L of several levels in one launch
constexpr int kM2l2dLevels = 31;
struct M2L2dLevels {
    M2L2dArgs level[kM2l2dLevels];
    int first[kM2l2dLevels + 1];  // first workgroup of each; set by the launch
    int count;
};

struct L2L2dArgs {
    int N;
    int num_parents;
    const int32_t* child_begin;
    const uint64_t* child_keys;
    const double2* src;        // locals of the parents
    double2* dst;              // locals of the children (added to)
};

struct Leaf2dArgs {
    const double4* src;
    const int32_t* leaf_of;
    const uint64_t* leaf_key;
    const int32_t* leaf_begin;
    int nleaf;
    int level;
    const double* geom;
    const int2* nbr;           // near-source ranges, 9 entries per leaf
    const int32_t* near_total; // their particles
    const int32_t* near_runs;  // and how many there are
    const double4* pad;        // per leaf: a zero charge at its first particle
    bool wide;                 // squared distances may overflow
    const double2* local;      // normalised locals of the leaves, or null
    int N;
    const uint32_t* perm;
    int64_t n;
    int64_t n_out;
    int exclude_self;
    double* pot;
    double* field;             // (re, im) of the complex force per output
};

hipError_t launch_p2m2d(const P2M2dArgs& a, hipStream_t st);
hipError_t launch_m2m2d(const M2M2dArgs& a, const Tables2d& T, hipStream_t st);
hipError_t launch_m2l2d(int N, M2L2dLevels& a, const Tables2d& T, hipStream_t st);
hipError_t launch_m2l2d_f32(int N, const M2L2dArgs& a, const Tables2d& T, hipStream_t st);
hipError_t launch_l2l2d(const L2L2dArgs& a, const Tables2d& T, hipStream_t st);
hipError_t launch_leaf2d(const Leaf2dArgs& a, const Tables2d& T, hipStream_t st);

}  // namespace lfmm
