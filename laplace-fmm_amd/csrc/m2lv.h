// m2lv.h -- shared declarations of the FP64 M2L on the vector units
// (m2lv_kernels.h).
#pragma once
#include "m2l64.h"

namespace lfmm {

constexpr int kM2lvMaxTerms = kM64MinTerms - 1;                // state and two operator tables fit the LDS
// Waves per workgroup: 4 up to 9 terms (2 or more workgroups per CU fit the
// LDS; 4M uniform particles, 9 terms: 6.6 ms against 6.7 with 8 waves), above
// that 8 (the one workgroup of a CU then has 2 waves per SIMD; 11 terms: 13.5
// against 16.3 ms, before the packed sources)
constexpr int m2lv_nw(int N) { return N <= 9 ? 4 : 8; }
constexpr int kM2lvTile = 64;                                  // targets per workgroup, one per lane

// Work partition of a step over the waves of a workgroup: degrees (rotations)
// and orders (translation) by cost over 4 SIMDs, longest first, each SIMD's
// share then over its NW / 4 waves (wave w runs on SIMD w % 4).
template <int N, int NW>
struct M2lvPart {
    int deg[N > 0 ? N : 1] = {};
    int ord[N > 0 ? N : 1] = {};
    constexpr M2lvPart()
    {
        int simd[4] = {}, wave[NW] = {};
        for (int n = N - 1; n >= 0; --n) deg[n] = take(simd, wave, (n + 1) * (n + 1) + n * n + 8 * n + 4);
        for (int i = 0; i < 4; ++i) simd[i] = 0;
        for (int i = 0; i < NW; ++i) wave[i] = 0;
        for (int k = 0; k < N; ++k) {  // order 1 costs the most: order 0 has no imaginary part
            const int m = k == 0 ? (N > 1 ? 1 : 0) : (k == 1 ? 0 : k);
            ord[m] = take(simd, wave, (m > 0 ? 2 : 1) * (N - m) * (N - m));
        }
    }
    constexpr int take(int* simd, int* wave, int cost)
    {
        int s = 0;
        for (int i = 1; i < 4; ++i)
            if (simd[i] < simd[s]) s = i;
        int w = s;
        for (int i = s; i < NW; i += 4)
            if (wave[i] < wave[w]) w = i;
        simd[s] += cost;
        wave[w] += cost;
        return w;
    }
};

// Operator streams: a wave's coefficients in the order of use, 16 per
// register.  They come in blocks that serve one asm statement and never
// straddle registers.  Rotation of degree n: rows 2r, 2r + 1, per k the block
// P_2r, P_2r+1, Q_2r, Q_2r+1 (Q for row, k > 0; rows up to n).  Translation of
// order m: output degrees m + 2r, m + 2r + 1, per input degree m + i their two
// coefficients.  Registers of the waves follow one another.
constexpr int m2lv_rot_block(int n, int r, int k)
{
    const int rows = 2 * r + 1 <= n ? 2 : 1;
    return rows + (k > 0 ? rows - (r == 0 ? 1 : 0) : 0);
}
template <int N, int NW>
struct M2lvLayout {
    static constexpr int H = (N + 1) / 2;
    short rot[N][H][N] = {};          // block positions in the wave's stream; bit 14: the register's last block
    short tr[N][H][N] = {};
    int rot_reg[NW + 1] = {};         // first register of each wave's stream
    int tr_reg[NW + 1] = {};
    constexpr M2lvLayout()
    {
        constexpr M2lvPart<N, NW> P{};
        for (int w = 0; w < NW; ++w) {
            int p = 0;
            short* last = nullptr;
            auto place = [&](short& at, int size) {
                if (p % 16 + size > 16) p = (p / 16 + 1) * 16;
                if (last && p / 16 != *last / 16) *last |= 1 << 14;
                at = (short)p;
                last = &at;
                p += size;
            };
            for (int n = N - 1; n >= 0; --n)
                if (P.deg[n] == w)
                    for (int r = 0; 2 * r <= n; ++r)
                        for (int k = 0; k <= n; ++k) place(rot[n][r][k], m2lv_rot_block(n, r, k));
            rot_reg[w + 1] = rot_reg[w] + (p + 15) / 16;
            p = 0;
            last = nullptr;
            for (int m = 0; m < N; ++m)
                if (P.ord[m] == w)
                    for (int r = 0; 2 * r < N - m; ++r)
                        for (int i = 0; i < N - m; ++i) place(tr[m][r][i], 2 * r + 1 < N - m ? 2 : 1);
            tr_reg[w + 1] = tr_reg[w] + (p + 15) / 16;
        }
    }
};
constexpr int m2lv_pos(int at) { return at & 0x3fff; }
constexpr bool m2lv_last(int at) { return (at & 0x4000) != 0; }

struct M2lvPack {
    std::vector<double> rot;    // [theta][register][16]
    std::vector<double> trans;  // [kNumTrans][register][16]
    std::vector<double> ephi;   // [kNumDirs][2][16] (cos, sin)
    int rot_regs = 0, tr_regs = 0;
};
void pack_m2lv(const OpTables& T, M2lvPack& out);  // N <= kM2lvMaxTerms

struct M2lvTables {
    const double* rot;
    const double* trans;
    const double* ephi;
};

// Class-major copy of a level's multipoles (stride coefficients per box) for
// launch_m2lv: packed[(class * nx + coefficient) * slots + parent], zeros for
// absent children and from slot num_parents on.
inline int m2lv_slots(int64_t parents) { return (int)((parents + 8) / 8 * 8); }
hipError_t launch_m2lv_pack(const RtrLevel& L, int nx, double2* packed, hipStream_t st);
// op: M2LV_M2L, M2LV_M2M (A.L as for launch_rtr) or M2LV_L2L
enum { M2LV_M2L = 0, M2LV_M2M = 1, M2LV_L2L = 2 };
hipError_t launch_m2lv(int N, int op, const M2LStepTables& S, const M2lvTables& V, const M64Level& A, hipStream_t st);

}  // namespace lfmm
