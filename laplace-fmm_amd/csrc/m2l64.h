// m2l64.h -- shared declarations of the FP64 matrix-core M2L (m2l64_kernels.h).
#pragma once
#include "lfmm_internal.h"
#include "ops3d.h"

#include <vector>

namespace lfmm {

// Operators of the FP64 matrix-core M2L (m2l64_kernels.h) in 4 x 4 blocks.
// Degree n has m64_chunks(n + 1) chunks of 4 orders, order m has
// m64_chunks(N - m) chunks of 4 degrees, counted down from N - 1.
constexpr int m64_chunks(int x) { return (x + 3) / 4; }
constexpr int m64_rot_base(int n)  // first block of degree n
{
    int r = 0;
    for (int i = 0; i < n; ++i) r += m64_chunks(i + 1) * m64_chunks(i + 1);
    return r;
}
constexpr int m64_blocks(int N) { return m64_rot_base(N); }
// the same with the degrees stored from N - 1 down
constexpr int m64_rot_at(int N, int n) { return m64_blocks(N) - m64_rot_base(n + 1); }
constexpr int m64_tr_base(int N, int m)  // first block of order m
{
    int r = 0;
    for (int i = 0; i < m; ++i) r += m64_chunks(N - i) * m64_chunks(N - i);
    return r;
}
// registers of set (a, b): degrees N-1-4a-s, orders 4b+g, s and g < m64_set
constexpr int m64_set(int N, int a, int b) { return N - 4 * a - 4 * b < 0 ? 0 : (N - 4 * a - 4 * b > 4 ? 4 : N - 4 * a - 4 * b); }
constexpr int kM64Groups = 64;    // operator groups per child class (L2L, at most 60 of the M2L), padded
constexpr int kM64Steps = kDirsPerClass + 1;
constexpr int kM64GroupMax = 8;   // directions per group
constexpr int m64_nw(int) { return 4; }                        // waves per workgroup
constexpr int m64_tile(int N) { return 8 * m64_nw(N); }        // targets per workgroup
constexpr int kM64MinTerms = 14;                               // smaller expansions: m2lv_kernels.h

// M2L steps of one target child class, grouped by operator (m2l64.cpp); both
// FP64 M2L kernels walk them.
struct M2LSteps {
    // class 8: the M2M of a parent, its children as sources of neighbour parent 13
    std::vector<int> steps;     // [9][kM64Steps] (direction, 8 * neighbour parent + source class; -1: L2L)
    std::vector<int> groups;    // [9][kM64Groups] (theta, translation, first step, end)
    int nsteps[9] = {};
};
void pack_m2l_steps(const OpTables& T, M2LSteps& out);
struct M2LStepTables {
    const int2* steps;
    const int4* groups;
    const double2* zero;        // an expansion of zeros
    int nsteps[9];
};

// The tables in the operand layout of the FP64 matrix-core M2L (m2l64.cpp).
struct M64Pack {
    std::vector<double> rot;    // [theta][block pair][P, Q][16] (even, odd block)
    std::vector<double> trans;  // [kNumTrans][block pair][16] (even, odd)
    std::vector<double> ephi;   // [kNumDirs][2][4 * chunks] (cos, sin)
};
void pack_m2l64(const OpTables& T, M64Pack& out);

struct M64Tables {
    const double2* rot;      // [theta][block pair][P, Q][16] (even, odd block)
    const double2* trans;    // [kNumTrans][block pair][16] (even block, odd block)
    const double2* ephi;     // [dir][2][4 * chunks]
};

struct M64Level {
    RtrLevel L;
    const int32_t* plut;     // key -> box at level - 1 (dense), or null
    const uint64_t* pkeys;   // keys at level - 1
    int psize;               // boxes at level - 1
    const double2* packed;   // class-major sources (launch_m2lv_pack), or null
    int slots;
};

// FP64 M2L of one level with the L2L of parent_local (m2l64_kernels.h), N >=
// kM64MinTerms; tiles / ctile in tiles of m64_tile targets
hipError_t launch_m2l64(int N, const M2LStepTables& S, const M64Tables& T, const M64Level& A, hipStream_t st);

}  // namespace lfmm
