// m2l64_kernels.h -- FP64 M2L (fused with L2L) of 14 terms and more on the
// matrix cores: the rotate / axial-translate / rotate-back operator (reference
// M2L :152-190, L2L :192-226 and Downward :328-349 of src/cpu/multipole3d.cpp)
// as chains of v_mfma_f64_4x4x4 products.  Compiled once per expansion size.
//
// The 4 blocks of an instruction take 16 columns: 8 targets x (real,
// imaginary part), so one operator register holds P for the real and Q for
// the imaginary lanes.  Lane l, K index and result row l / 16: the result of
// one product chain is an operand of the next without any exchange, except
// that the rotations contract over orders and the translation over degrees; a
// 4 x 4 transpose over the lane groups (v_permlane32/16_swap) turns one into
// the other.  A wave keeps the whole state of its 8 targets in registers
// (N = 18: 100 doubles, and 100 accumulators), the operators of a group of
// directions with one polar angle and distance sit in LDS (65 KB at N = 18).
//
// What bounds it: a 4 x 4 x 4 FP64 product blocks the SIMD's vector unit for
// 16 cycles (measured; no overlap with other vector work), so products (2/3
// of the time at N = 18), transposes and the azimuthal factors add up; with
// one wave per SIMD the source loads are only partly hidden.  524,288 uniform
// particles, 18 terms: 34.6 ms with the operators by scalar loads on the
// vector units (whose LDS state left one wave per SIMD waiting for them),
// 8.0 ms here; v_mfma_f64_16x16x4 reached 46 TFLOP/s against 74 for 4x4x4.
// Smaller expansions run on the vector units (m2lv_kernels.h): there the same
// kernel needs 10.5 ms at 13 terms and 1M clustered particles against 9.5.
#pragma once
#include "device_common.h"
#include "m2l64.h"
#include "m2l_children.h"
#include "ops3d_kernels.h"

#include <algorithm>

namespace lfmm {

__device__ __forceinline__ double m64_mfma(double a, double b, double c)
{
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

// (a, b): lanes 32..63 of a <-> lanes 0..31 of b
__device__ __forceinline__ void m64_swap32(double& a, double& b)
{
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}

// (a, b): 16-lane rows 1, 3 of a <-> rows 0, 2 of b
__device__ __forceinline__ void m64_swap16(double& a, double& b)
{
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]);
    b = __hiloint2double((int)hi[1], (int)lo[1]);
}

// Transposes registers r[0..V-1] against the lane groups (lane / 16):
// afterwards group s of r[g] holds what group g of r[s] held.  Lane groups
// >= V of the results are finite leftovers (their operator entries are zero).
template <int V>
__device__ __forceinline__ void m64_transpose(double (&r)[4])
{
    if constexpr (V == 2) {
        m64_swap16(r[0], r[1]);
    } else if constexpr (V >= 3) {
        if constexpr (V == 3) r[3] = r[1];
        m64_swap32(r[0], r[2]);
        m64_swap32(r[1], r[3]);
        m64_swap16(r[0], r[1]);
        m64_swap16(r[2], r[3]);
    }
}

template <int N>
struct M64Buf {  // one group's operators in LDS, in 16-byte units
    static constexpr int pairs = (m64_blocks(N) + 1) / 2;
    static constexpr int rot = 32 * pairs;
    static constexpr int trans = 16 * pairs;
    static constexpr int ephi = 8 * m64_chunks(N);
    static constexpr int units = rot + trans + kM64GroupMax * ephi;
};

constexpr int kAhead = 4;  // operator reads in flight

// the other lane of a (re, im) pair: lane ^ 8
__device__ __forceinline__ double m64_partner(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x128, 0xf, 0xf, true);  // row_ror:8
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x128, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

template <int N, int NW>
__global__ void __launch_bounds__(64 * NW, 1) k_m2l64(M2LStepTables S, M64Tables T, M64Level A)
{
    constexpr int NX = tri(N);
    constexpr int NT = 64 * NW;
    constexpr int TILE = 8 * NW;
    constexpr int CB = m64_chunks(N);  // chunks of 4 orders (m = 4b + g) or of 4 degrees (n = N - 1 - 4a - s)
    using B = M64Buf<N>;
    const RtrLevel& L = A.L;
    __shared__ double2 tab[2][B::units];
    __shared__ int2 kids[27][TILE];  // per neighbour parent: first child, child classes present
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, im = (lane >> 3) & 1;
    const int blk = xcd_local_block(blockIdx.x, gridDim.x);
    int tile, c, part = 0, pbeg = 0, pend = L.num_parents;
    if (L.csorted) {
        c = blk & 7;
        tile = blk >> 3;
        if (tile >= L.ctile[c + 1] - L.ctile[c]) return;  // the whole block
        pbeg = L.coff[c];
        pend = L.coff[c + 1];
    } else {
        const int per_tile = 8 * L.dsplit;
        tile = blk / per_tile;
        const int r = blk - tile * per_tile;
        part = r >> 3;
        c = r & 7;
    }
    pbeg += tile * TILE;
    m64_children<TILE, NT>(A, pbeg, pend, kids);
    const int tj = w * 8 + (lane & 7);
    const int P = pbeg + tj < pend ? (L.plist ? L.plist[pbeg + tj] : pbeg + tj) : -1;
    const int64_t SX = L.stride > 0 ? L.stride : NX;
    __syncthreads();
    // box of class s under neighbour parent k (ks = 8 k + s), -1: none
    auto box_of = [&](int ks) -> int {
        const int2 v = kids[ks >> 3][tj];
        return (v.y >> (ks & 7)) & 1 ? v.x + __popc(v.y & ((1 << (ks & 7)) - 1)) : -1;
    };
    const int tgt = box_of(13 * 8 + c);
    // Steps are grouped by operator (theta, translation); a group's tables
    // stay in LDS for its steps.  Step 0 of group 0 is the L2L.
    const int g_first = L.parent_local ? 0 : 1;
    const auto groups = m64_scalar((const m64_i4*)S.groups) + c * kM64Groups;  // (theta, translation, first step, end)
    const auto steps = m64_scalar((const m64_i2*)S.steps) + c * kM64Steps;     // (direction, 8 * neighbour parent + source class)
    const int s_first = groups[g_first].z, ns = S.nsteps[c] - s_first;
    const int d_beg = s_first + part * ns / L.dsplit, d_end = s_first + (part + 1) * ns / L.dsplit;
    int gi = g_first;
    while (groups[gi].w <= d_beg) ++gi;
    // source of this lane's target at a step (-1: none)
    auto source_of = [&](int d) -> int {
        const int ks = steps[d].y;
        return tgt < 0 ? -1 : (ks < 0 ? P : box_of(ks));
    };
    // a group's operators: global -> registers -> LDS
    constexpr int U = (B::units + NT - 1) / NT;
    m64_v2 stage[U];
    auto stage_load = [&](m64_i4 gr) {
        const double2* rot = T.rot + (int64_t)gr.x * B::rot;
        const double2* tr = T.trans + (int64_t)gr.y * B::trans;
        sfor<0, U>([&](auto I) {
            constexpr int i = decltype(I)::value;
            const int u = i * NT + (int)threadIdx.x;
            const double2* p = rot + u;
            if (i * NT + NT - 1 >= B::rot && u >= B::rot) p = tr + (u - B::rot);
            if (i * NT + NT - 1 >= B::rot + B::trans && u >= B::rot + B::trans) {
                const int e = u - B::rot - B::trans, k = e / B::ephi;
                p = T.ephi + steps[min(gr.z + k, gr.w - 1)].x * B::ephi + (e - k * B::ephi);
            }
            if (i * NT + NT - 1 < B::units || u < B::units) stage[i] = *(const m64_v2*)p;
        });
    };
    auto stage_store = [&](double2* dst) {
        sfor<0, U>([&](auto I) {
            constexpr int i = decltype(I)::value;
            const int u = i * NT + (int)threadIdx.x;
            if (i * NT + NT - 1 < B::units || u < B::units) *(m64_v2*)(dst + u) = stage[i];
        });
    };
    // The state of a step, one double per lane and register: target lane % 8,
    // real (lane / 8 even) or imaginary part.  Registers come in sets of 4
    // degrees (n = N-1-4a-s) x 4 orders (m = 4b+g): x[a][b][s] with order g
    // in lane group g, or, transposed, x[a][b][g] with degree s in group s.
    double x[CB][CB][4];
    // source coefficients of degree n (past m = n, entry n repeated: its
    // operator columns are zero)
    auto load_degree = [&](auto NN, const double* sp) {
        constexpr int n = decltype(NN)::value;
        sfor<0, n / 4 + 1>([&](auto BI) {
            constexpr int b = decltype(BI)::value, r = n - 4 * b;
            x[(N - 1 - n) / 4][b][(N - 1 - n) % 4] = sp[2 * (tri(n) + 4 * b + (r >= 3 ? g : min(g, r)))];
        });
    };
    auto load_all = [&](const double* sp) {
        sfor<0, N>([&](auto KK) { load_degree(std::integral_constant<int, N - 1 - decltype(KK)::value>{}, sp); });
    };
    auto pointer_of = [&](int idx, bool l2l) -> const double* {
        return (const double*)(idx < 0 ? S.zero : (l2l ? L.parent_local : L.src) + (int64_t)idx * SX) + im;
    };

    double acc[N][CB];
    sfor<0, N>([&](auto NN) {
        sfor<0, decltype(NN)::value / 4 + 1>([&](auto BI) { acc[decltype(NN)::value][decltype(BI)::value] = 0.0; });
    });

    m64_i4 gr = groups[gi];
    stage_load(gr);
    bool any;
    {
        const int idx = source_of(d_beg);
        load_all(pointer_of(idx, d_beg == 0));
        any = __ballot(idx >= 0) != 0ull;
    }
    stage_store(tab[0]);
    lds_barrier();
    int buf = 0;
    for (int d = d_beg; d < d_end; ++d) {
        const double2* __restrict__ t = tab[buf];
        // the next group's tables are staged during a group's first step here
        const bool stage_now = (d == d_beg || d == gr.z) && gr.w < d_end;
        if (stage_now) stage_load(groups[gi + 1]);
        const int nidx = d + 1 < d_end ? source_of(d + 1) : -1;
        const double* nsp = pointer_of(nidx, false);
        if (any) {
            // The step's operator blocks, two per 16-byte read, are read in
            // consumption order, kAhead reads before their products.
            constexpr int R = m64_blocks(N), RP = B::pairs, Q = 3 * RP;
            const double2* __restrict__ trot = t + im * 16 + g * 4 + (lane & 3);
            const double2* __restrict__ ttr = t + B::rot + g * 4 + (lane & 3);
            const double2* __restrict__ teph = t + B::rot + B::trans + (d - gr.z) * B::ephi + im * (4 * CB) + g;
            double2 ring[kAhead];
            auto fetch = [&](auto QI) {
                constexpr int q = decltype(QI)::value;
                if constexpr (q < RP) ring[q % kAhead] = trot[32 * q];
                else if constexpr (q < 2 * RP) ring[q % kAhead] = ttr[16 * (q - RP)];
                else if constexpr (q < Q) ring[q % kAhead] = trot[32 * (q - 2 * RP)];
            };
            auto operand = [&](auto KI, auto BASE) -> double {
                constexpr int k = decltype(KI)::value;
                const double2 v = ring[(decltype(BASE)::value + k / 2) % kAhead];
                return (k & 1) ? v.y : v.x;
            };
            auto after = [&](auto KI, auto BASE) {  // the products of block k are issued
                constexpr int k = decltype(KI)::value;
                if constexpr ((k & 1) || k == R - 1)
                    fetch(std::integral_constant<int, decltype(BASE)::value + k / 2 + kAhead>{});
                __builtin_amdgcn_sched_barrier(0x6);  // VALU and SALU may cross
            };
            sfor<0, kAhead>(fetch);
            double2 eph[CB];
            auto load_eph = [&]() {
                sfor<0, CB>([&](auto BI) { eph[decltype(BI)::value] = teph[4 * decltype(BI)::value]; });
            };
            load_eph();
            auto transpose_set = [&](auto AI, auto BI) {
                constexpr int a = decltype(AI)::value, b = decltype(BI)::value;
                constexpr int v = m64_set(N, a, b);
                if constexpr (v > 1) m64_transpose<v>(x[a][b]);
            };
            // ---- Rz(phi), Ry(theta), degrees from the top: a set of degrees
            // is transposed while the next set's products run
            auto phi = [&](auto NN) {
                constexpr int n = decltype(NN)::value, a = (N - 1 - n) / 4, s = (N - 1 - n) % 4;
                sfor<0, n / 4 + 1>([&](auto BI) {
                    constexpr int b = decltype(BI)::value;
                    const double v = x[a][b][s];
                    x[a][b][s] = fma(v, eph[b].x, m64_partner(v) * eph[b].y);
                });
            };
            phi(std::integral_constant<int, N - 1>{});
            sfor<0, N>([&](auto KK) {
                constexpr int n = N - 1 - decltype(KK)::value;
                constexpr int ch = n / 4 + 1, a = (N - 1 - n) / 4, s = (N - 1 - n) % 4;
                if constexpr (n > 0) phi(std::integral_constant<int, n - 1>{});
                double y[ch];
                sfor<0, ch * ch>([&](auto JJ) {
                    constexpr int b = decltype(JJ)::value / ch, bo = decltype(JJ)::value % ch;
                    constexpr std::integral_constant<int, m64_rot_at(N, n) + decltype(JJ)::value> k{};
                    constexpr std::integral_constant<int, 0> base{};
                    y[bo] = m64_mfma(operand(k, base), x[a][b][s], b == 0 ? 0.0 : y[bo]);
                    after(k, base);
                });
                sfor<0, ch>([&](auto BO) { x[a][decltype(BO)::value][s] = y[decltype(BO)::value]; });
                if constexpr (s == 3 || n == 0) sfor<0, CB>([&](auto BI) { transpose_set(std::integral_constant<int, a>{}, BI); });
            });
            // ---- axial translation, orders from 0: one product chain per order
            sfor<0, N>([&](auto MM) {
                constexpr int m = decltype(MM)::value;
                constexpr int ct = (N - 1 - m) / 4 + 1, b = m / 4, gm = m % 4;
                double y[ct];
                sfor<0, ct * ct>([&](auto JJ) {
                    constexpr int ai = decltype(JJ)::value / ct, ao = decltype(JJ)::value % ct;
                    constexpr std::integral_constant<int, m64_tr_base(N, m) + decltype(JJ)::value> k{};
                    constexpr std::integral_constant<int, RP> base{};
                    y[ao] = m64_mfma(operand(k, base), x[ai][b][gm], ai == 0 ? 0.0 : y[ao]);
                    after(k, base);
                });
                sfor<0, ct>([&](auto AO) { x[decltype(AO)::value][b][gm] = y[decltype(AO)::value]; });
                if constexpr (gm == 3 || m == N - 1) sfor<0, CB>([&](auto AI) { transpose_set(AI, std::integral_constant<int, b>{}); });
            });
            // ---- Ry(-theta), Rz(-phi), accumulate, degrees from the top; a
            // degree's registers then take the next step's sources
            asm volatile("" ::: "memory");
            load_eph();
            sfor<0, N>([&](auto KK) {
                constexpr int n = N - 1 - decltype(KK)::value;
                constexpr int ch = n / 4 + 1, a = (N - 1 - n) / 4, s = (N - 1 - n) % 4;
                double y[ch];
                sfor<0, ch * ch>([&](auto JJ) {
                    constexpr int b = decltype(JJ)::value / ch, bo = decltype(JJ)::value % ch;
                    constexpr std::integral_constant<int, m64_rot_at(N, n) + decltype(JJ)::value> k{};
                    constexpr std::integral_constant<int, 2 * RP> base{};
                    y[bo] = m64_mfma(operand(k, base), x[a][b][s], b == 0 ? 0.0 : y[bo]);
                    after(k, base);
                });
                load_degree(std::integral_constant<int, n>{}, nsp);
                sfor<0, ch>([&](auto BO) {
                    constexpr int bo = decltype(BO)::value;
                    acc[n][bo] = fma(y[bo], eph[bo].x, fma(-m64_partner(y[bo]), eph[bo].y, acc[n][bo]));
                });
            });
        } else {
            load_all(nsp);
        }
        if (stage_now) stage_store(tab[buf ^ 1]);
        any = __ballot(nidx >= 0) != 0ull;
        if (d + 1 == gr.w && d + 1 < d_end) {
            lds_barrier();
            gr = groups[++gi];
            buf ^= 1;
        }
    }
    if (tgt >= 0) {
        double* out = (double*)(L.dsplit > 1 ? L.partial + ((int64_t)part * L.size + tgt) * NX : L.dst + (int64_t)tgt * SX) + im;
        // coefficients beyond this launch's order are zero
        for (int64_t i = NX + g; i < SX; i += 4) out[2 * i] = 0.0;
        const double sg = (g & 1) ? -1.0 : 1.0;  // (-1)^m (see pack_m2l64)
        sfor<0, N>([&](auto NN) {
            constexpr int n = decltype(NN)::value;
            sfor<0, n / 4 + 1>([&](auto BI) {
                constexpr int b = decltype(BI)::value;
                if (4 * b + 3 <= n || 4 * b + g <= n) out[2 * (tri(n) + 4 * b + g)] = sg * acc[n][b];
            });
        });
    }
}

template <int N>
hipError_t do_m2l64(const M2LStepTables& S, const M64Tables& T, const M64Level& A, hipStream_t st)
{
    const RtrLevel& L = A.L;
    int blocks = 0;
    if (L.csorted) {
        if (L.dsplit != 1 || !L.plist || L.coff[8] != L.num_parents) return hipErrorInvalidValue;
        int mt = 0;
        for (int c = 0; c < 8; ++c) {
            const int t = L.ctile[c + 1] - L.ctile[c];
            if (t != (L.coff[c + 1] - L.coff[c] + m64_tile(N) - 1) / m64_tile(N)) return hipErrorInvalidValue;
            mt = std::max(mt, t);
        }
        blocks = 8 * mt;
    } else {
        if (L.tiles != (L.num_parents + m64_tile(N) - 1) / m64_tile(N)) return hipErrorInvalidValue;
        blocks = L.tiles * 8 * L.dsplit;
    }
    if (blocks > 0) hipLaunchKernelGGL((k_m2l64<N, m64_nw(N)>), dim3(blocks), dim3(64 * m64_nw(N)), 0, st, S, T, A);
    return hipGetLastError();
}

}  // namespace lfmm
