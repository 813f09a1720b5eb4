// m2lv_kernels.h -- FP64 M2L (fused with L2L), M2M and L2L of up to 13 terms on
// the vector units: the rotate / axial-translate / rotate-back operator
// (reference M2M :115-150, M2L :152-190, L2L :192-226 and Downward :328-349 of
// src/cpu/multipole3d.cpp).  Compiled once per expansion size.
//
// A workgroup owns 64 targets, one per lane, and walks their interaction
// directions.  The state of a direction lives in LDS as [coefficient][lane]
// and goes through three phases, each split over the waves at compile time:
//   A  Rz(phi), Ry(theta)                by source degree
//   B  axial translation                 by order
//   C  Ry(-theta), Rz(-phi), accumulate  by target degree (registers)
//
// What bounds it is FP64 vector issue (N = 13: 4,400 products per 64 targets
// and direction), if the coefficients, each used for one product per lane,
// arrive in time.  As scalar operands they do not: scalar loads complete in
// any order, so a wave waits for all of them, and at 13 terms the kernel
// spent 53% of its time waiting with 20% vector issue.  Here a coefficient
// register holds 16 coefficients, one per lane of each 16-lane row, read from
// LDS by one instruction (128 bytes); v_fmac_f64_dpp row_newbcast broadcasts
// one of them per product at full rate (measured 4.2 cycles per wave).  The
// products are inline assembly because the compiler does not fold the
// broadcast (v_mov_b64_dpp) into the product; a coefficient register is only
// ever written by an LDS read, never by a vector instruction just before it.
// Directions with one polar angle and distance share their tables (3.7 on
// average), so the tables are staged, and double-buffered, per such group.
// On large, mostly full levels the sources are packed class-major
// (m2lv_pack.hip): one box per lane costs the L1 64 tag lookups per load.
//
// Measured, 4M uniform particles (M2L of all levels; before, with scalar
// operands): 9 terms 8.3 -> 6.6 ms, 11 terms 16.2 -> 11.0 ms, 13 terms 49.0 -> 16.9
// ms (33 TFLOP/s algorithmic); the packing adds 0.2 ms.  The vector units are busy
// about half of the time; the rest is the phase barriers (5%), the source
// loads (13%) and dependent issue with 2 waves per SIMD.
#pragma once
#include "device_common.h"
#include "m2l_children.h"
#include "m2lv.h"
#include "rowbc.h"
#include "ops3d_kernels.h"

#include <algorithm>

namespace lfmm {

#define LFMM_BC(I) " row_newbcast:" I " row_mask:0xf bank_mask:0xf"
// Products with entries I, I + 1, .. of c.  Two rows of a rotation:
// re0 += P0 x, re1 += P1 x, im0 += Q0 y, im1 += Q1 y.
template <int I>
__device__ __forceinline__ void rot4_bc(double& re0, double& re1, double& im0, double& im1, double c, double x, double y)
{
    asm("v_fmac_f64_dpp %0, %4, %5" LFMM_BC("%7") "\n\tv_fmac_f64_dpp %1, %4, %5" LFMM_BC("%8")
        "\n\tv_fmac_f64_dpp %2, %4, %6" LFMM_BC("%9") "\n\tv_fmac_f64_dpp %3, %4, %6" LFMM_BC("%10")
        : "+&v"(re0), "+&v"(re1), "+&v"(im0), "+&v"(im1)
        : "v"(c), "v"(x), "v"(y), "n"(I), "n"(I + 1), "n"(I + 2), "n"(I + 3));
}
// rows 0 (no imaginary part) and 1
template <int I>
__device__ __forceinline__ void rot3_bc(double& re0, double& re1, double& im1, double c, double x, double y)
{
    asm("v_fmac_f64_dpp %0, %3, %4" LFMM_BC("%6") "\n\tv_fmac_f64_dpp %1, %3, %4" LFMM_BC("%7")
        "\n\tv_fmac_f64_dpp %2, %3, %5" LFMM_BC("%8")
        : "+&v"(re0), "+&v"(re1), "+&v"(im1)
        : "v"(c), "v"(x), "v"(y), "n"(I), "n"(I + 1), "n"(I + 2));
}
// a += c_I x, b += c_J y
template <int I, int J>
__device__ __forceinline__ void pair_bc(double& a, double& b, double c, double x, double y)
{
    asm("v_fmac_f64_dpp %0, %2, %3" LFMM_BC("%5") "\n\tv_fmac_f64_dpp %1, %2, %4" LFMM_BC("%6")
        : "+&v"(a), "+&v"(b)
        : "v"(c), "v"(x), "v"(y), "n"(I), "n"(J));
}
#undef LFMM_BC


// per neighbour parent of a target: its slot (packed sources) or its first
// child and the child classes present
template <bool PACKED>
using m2lv_near_t = std::conditional_t<PACKED, int, int2>;

template <int N, int NW>
struct M2lvBuf {  // one group's operators in LDS, in doubles
    static constexpr M2lvLayout<N, NW> LY{};
    static constexpr int rot = 16 * LY.rot_reg[NW];
    static constexpr int trans = 16 * LY.tr_reg[NW];
    static constexpr int size = rot + trans;
};

// A stream of coefficient registers read `ahead` registers before use.
template <int REGS>
struct M2lvStream {
    static constexpr int ahead = 4;
    const double* p;
    double ring[ahead];
    __device__ __forceinline__ explicit M2lvStream(const double* q) : p(q)
    {
        sfor<0, ahead>([&](auto R) {
            constexpr int r = decltype(R)::value;
            if constexpr (r < REGS) ring[r] = p[16 * r];
        });
    }
    template <int AT>
    __device__ __forceinline__ double reg() const
    {
        return ring[(m2lv_pos(AT) / 16) % ahead];
    }
    template <int AT>
    __device__ __forceinline__ void used()  // the block at AT
    {
        constexpr int r = m2lv_pos(AT) / 16;
        if constexpr (m2lv_last(AT) && r + ahead < REGS) ring[r % ahead] = p[16 * (r + ahead)];
        if constexpr (m2lv_last(AT)) __builtin_amdgcn_sched_barrier(0);
    }
};

// Rows 2R, 2R + 1 of the rotation of degree n: (re, im)[0..1] += P, Q rows.
template <int N, int NW, int n, int R, int REGS>
__device__ __forceinline__ void m2lv_rows(M2lvStream<REGS>& S, const double2 (&v)[n + 1], double (&re)[2], double (&im)[2])
{
    constexpr M2lvLayout<N, NW> LY{};
    sfor<0, n + 1>([&](auto K) {
        constexpr int k = decltype(K)::value, at = LY.rot[n][R][k], i = m2lv_pos(at) % 16;
        constexpr bool two = 2 * R + 1 <= n;
        const double c = S.template reg<at>();
        if constexpr (k == 0) {
            if constexpr (two) pair_bc<i, i + 1>(re[0], re[1], c, v[0].x, v[0].x);
            else fmac_bc<i>(re[0], c, v[0].x);
        } else if constexpr (R == 0) {
            if constexpr (two) rot3_bc<i>(re[0], re[1], im[1], c, v[k].x, v[k].y);
            else fmac_bc<i>(re[0], c, v[k].x);
        } else {
            if constexpr (two) rot4_bc<i>(re[0], re[1], im[0], im[1], c, v[k].x, v[k].y);
            else pair_bc<i, i + 1>(re[0], im[0], c, v[k].x, v[k].y);
        }
        S.template used<at>();
    });
}

// OP: M2L with the L2L, or one of the other two operators of this form alone:
// M2M (targets: parents, steps: their 8 children) and L2L (one step).  With
// scalar coefficients (k_rtr) a step took 12 us however few the boxes; here,
// 13 terms, 4M clustered particles: M2M 2.40 -> 1.12 ms, L2L 0.79 -> 0.51.
template <int N, int NW, int W, bool PACKED, int OP>
__device__ __forceinline__ void m2lv_wave(const M2LStepTables& T, const M2lvTables& V, const M64Level& A, double2* state,
                                          double (*tab)[M2lvBuf<N, NW>::size], m2lv_near_t<PACKED> (*near)[kM2lvTile],
                                          int c, int part, int pbeg, int pend)
{
    constexpr int NX = tri(N);
    constexpr M2lvPart<N, NW> PT{};
    constexpr M2lvLayout<N, NW> LY{};
    using B = M2lvBuf<N, NW>;
    constexpr int RR = LY.rot_reg[W + 1] - LY.rot_reg[W], TR = LY.tr_reg[W + 1] - LY.tr_reg[W];
    const RtrLevel& L = A.L;
    const int lane = threadIdx.x & 63, l16 = lane & 15;
    const int P = pbeg + lane < pend ? (L.plist ? L.plist[pbeg + lane] : pbeg + lane) : -1;
    const int64_t SX = L.stride > 0 ? L.stride : NX;
    // source box (packed: slot) of class s under neighbour parent k (ks = 8 k + s), -1: none
    auto box_of = [&](int ks) -> int {
        const auto v = near[ks >> 3][lane];
        if constexpr (PACKED) return v;
        else return (v.y >> (ks & 7)) & 1 ? v.x + __popc(v.y & ((1 << (ks & 7)) - 1)) : -1;
    };
    int tgt = -1;
    if constexpr (OP == M2LV_M2M) {
        // a parent without children (a leaf of the adaptive tree) keeps its P2M
        if (P >= 0 && L.child_begin[P + 1] > L.child_begin[P]) tgt = P;
    } else if (P >= 0) {
        for (int i = L.child_begin[P]; i < L.child_begin[P + 1]; ++i)
            if ((int)(L.child_keys[i] & 7u) == c) tgt = i;
    }
    const int g_first = OP == M2LV_M2L && !L.parent_local ? 1 : 0;
    const auto groups = m64_scalar((const m64_i4*)T.groups) + c * kM64Groups;  // (theta, translation, first step, end)
    const auto steps = m64_scalar((const m64_i2*)T.steps) + c * kM64Steps;     // (direction, 8 * neighbour parent + source class)
    const int s_first = groups[g_first].z, ns = OP == M2LV_L2L ? 1 : T.nsteps[c] - s_first;
    const int d_beg = s_first + part * ns / L.dsplit, d_end = s_first + (part + 1) * ns / L.dsplit;
    int gi = g_first;
    while (groups[gi].w <= d_beg) ++gi;
    auto source_of = [&](int ks) -> int { return tgt < 0 ? -1 : (ks < 0 ? P : box_of(ks)); };
    // a group's operators: global -> registers -> LDS
    constexpr int NT = 64 * NW, U = (B::size / 2 + NT - 1) / NT;
    m64_v2 stage[U];
    auto stage_load = [&](m64_i4 gr) {
        const double* rot = V.rot + (int64_t)gr.x * B::rot;
        const double* tr = V.trans + (int64_t)gr.y * B::trans;
        sfor<0, U>([&](auto I) {
            constexpr int i = decltype(I)::value;
            const int u = 2 * (i * NT + (int)threadIdx.x);
            const double* p = u < B::rot ? rot + u : tr + (u - B::rot);
            if (u < B::size) stage[i] = *(const m64_v2*)p;
        });
    };
    auto stage_store = [&](double* dst) {
        sfor<0, U>([&](auto I) {
            constexpr int i = decltype(I)::value;
            const int u = 2 * (i * NT + (int)threadIdx.x);
            if (u < B::size) *(m64_v2*)(dst + u) = stage[i];
        });
    };
    // the wave's source degrees, loaded a step ahead.  Packed sources: one
    // row of slots per class and coefficient, a slot of zeros at the end.
    double2 pf[NX];
    auto each_source = [&](auto&& f) {
        sfor<0, N>([&](auto KK) {
            constexpr int n = N - 1 - decltype(KK)::value;
            if constexpr (PT.deg[n] == W)
                sfor<0, n + 1>([&](auto K) { f(std::integral_constant<int, tri(n) + decltype(K)::value>{}); });
        });
    };
    auto load_boxes = [&](const double2* base, int idx) {
        const double2* sp = idx < 0 ? T.zero : base + (int64_t)idx * SX;
        each_source([&](auto I) { pf[decltype(I)::value] = sp[decltype(I)::value]; });
    };
    auto load_sources = [&](int ks, int idx) {
        if constexpr (PACKED) {
            const double2* row = A.packed + (int64_t)(ks & 7) * NX * A.slots;
            const uint32_t at = (uint32_t)(idx < 0 ? A.slots - 1 : idx);
            each_source([&](auto I) { pf[decltype(I)::value] = row[decltype(I)::value * (int64_t)A.slots + at]; });
        } else {
            load_boxes(L.src, idx);
        }
    };
    double ec, es;  // cos k phi, sin k phi in lane k of every 16
    auto load_phi = [&](int dir) {
        ec = V.ephi[dir * 32 + l16];
        es = V.ephi[dir * 32 + 16 + l16];
    };
    double2 acc[NX];
    sfor<0, NX>([&](auto I) { acc[decltype(I)::value] = make_double2(0.0, 0.0); });

    m64_i4 gr = groups[gi];
    stage_load(gr);
    m64_i2 st = steps[d_beg];
    const int idx0 = source_of(st.y);
    if (st.y < 0) load_boxes(L.parent_local, idx0);
    else load_sources(st.y, idx0);
    load_phi(st.x);
    bool any = __ballot(idx0 >= 0) != 0ull;  // the same lanes in every wave: uniform over the workgroup
    stage_store(tab[0]);
    lds_barrier();
    int buf = 0;
    for (int d = d_beg; d < d_end; ++d) {
        const double* __restrict__ t = tab[buf];
        // the next group's tables are staged during a group's first step here
        const bool stage_now = (d == d_beg || d == gr.z) && gr.w < d_end;
        if (stage_now) stage_load(groups[gi + 1]);
        st = steps[min(d + 1, d_end - 1)];
        const int nidx = d + 1 < d_end ? source_of(st.y) : -1;
        if (any) {
            {   // ---- Rz(phi), then Ry(theta), by degree
                M2lvStream<RR> S(t + 16 * LY.rot_reg[W] + l16);
                sfor<0, N>([&](auto KK) {
                    constexpr int n = N - 1 - decltype(KK)::value;
                    if constexpr (PT.deg[n] == W) {
                        double2 v[n + 1];
                        v[0] = pf[tri(n)];
                        sfor<1, n + 1>([&](auto K) {
                            constexpr int k = decltype(K)::value;
                            const double2 s = pf[tri(n) + k];
                            const double ck = bc<k>(ec);
                            v[k].x = s.x * ck;
                            v[k].y = s.y * ck;
                            fnmac_bc<k>(v[k].x, es, s.y);
                            fmac_bc<k>(v[k].y, es, s.x);
                        });
                        __builtin_amdgcn_sched_barrier(0);
                        sfor<0, n / 2 + 1>([&](auto R) {
                            constexpr int m = 2 * decltype(R)::value;
                            double re[2] = {0.0, 0.0}, im[2] = {0.0, 0.0};
                            m2lv_rows<N, NW, n, m / 2>(S, v, re, im);
                            state[(tri(n) + m) * kM2lvTile + lane] = make_double2(re[0], im[0]);
                            if constexpr (m < n) state[(tri(n) + m + 1) * kM2lvTile + lane] = make_double2(re[1], im[1]);
                        });
                    }
                });
            }
            load_sources(st.y & 0xff, nidx);  // complete under the next two phases
            lds_barrier();
            {   // ---- axial translation, by order
                M2lvStream<TR> S(t + B::rot + 16 * LY.tr_reg[W] + l16);
                sfor<0, N>([&](auto MM) {
                    constexpr int m = decltype(MM)::value;
                    if constexpr (PT.ord[m] == W) {
                        double2 x[N - m];
                        sfor<0, N - m>([&](auto I) {
                            constexpr int i = decltype(I)::value;
                            x[i] = state[(tri(m + i) + m) * kM2lvTile + lane];
                        });
                        sfor<0, (N - m + 1) / 2>([&](auto R) {
                            constexpr int j = 2 * decltype(R)::value;
                            constexpr bool two = j + 1 < N - m;
                            double re[2] = {0.0, 0.0}, im[2] = {0.0, 0.0};
                            sfor<0, N - m>([&](auto I) {
                                constexpr int i = decltype(I)::value, at = LY.tr[m][j / 2][i], e = m2lv_pos(at) % 16;
                                const double cr = S.template reg<at>();
                                if constexpr (m == 0) {
                                    if constexpr (two) pair_bc<e, e + 1>(re[0], re[1], cr, x[i].x, x[i].x);
                                    else fmac_bc<e>(re[0], cr, x[i].x);
                                } else {
                                    if constexpr (two) tr4_bc<e>(re[0], im[0], re[1], im[1], cr, x[i].x, x[i].y);
                                    else pair_bc<e, e>(re[0], im[0], cr, x[i].x, x[i].y);
                                }
                                S.template used<at>();
                            });
                            state[(tri(m + j) + m) * kM2lvTile + lane] = make_double2(re[0], im[0]);
                            if constexpr (two) state[(tri(m + j + 1) + m) * kM2lvTile + lane] = make_double2(re[1], im[1]);
                        });
                    }
                });
            }
            lds_barrier();
            {   // ---- Ry(-theta), Rz(-phi), accumulate, by degree
                M2lvStream<RR> S(t + 16 * LY.rot_reg[W] + l16);
                sfor<0, N>([&](auto KK) {
                    constexpr int n = N - 1 - decltype(KK)::value;
                    if constexpr (PT.deg[n] == W) {
                        double2 v[n + 1];
                        sfor<0, n + 1>([&](auto K) {
                            constexpr int k = decltype(K)::value;
                            v[k] = state[(tri(n) + k) * kM2lvTile + lane];
                        });
                        sfor<0, n / 2 + 1>([&](auto R) {
                            constexpr int m = 2 * decltype(R)::value;
                            double re[2] = {m == 0 ? acc[tri(n)].x : 0.0, 0.0}, im[2] = {0.0, 0.0};
                            m2lv_rows<N, NW, n, m / 2>(S, v, re, im);
                            if constexpr (m == 0) acc[tri(n)].x = re[0];
                            sfor<(m == 0 ? 1 : 0), (m < n ? 2 : 1)>([&](auto Q) {
                                constexpr int q = decltype(Q)::value;
                                double2& o = acc[tri(n) + m + q];
                                fmac_bc<m + q>(o.x, ec, re[q]);
                                fmac_bc<m + q>(o.y, ec, im[q]);
                                fmac_bc<m + q>(o.x, es, im[q]);
                                fnmac_bc<m + q>(o.y, es, re[q]);
                            });
                        });
                    }
                });
            }
        } else {
            load_sources(st.y & 0xff, nidx);
        }
        load_phi(st.x);
        if (stage_now) stage_store(tab[buf ^ 1]);
        const bool last = d + 1 == gr.w;
        if (any || last) lds_barrier();
        any = __ballot(nidx >= 0) != 0ull;
        if (last && d + 1 < d_end) {
            gr = groups[++gi];
            buf ^= 1;
        }
    }
    double mx = 0.0;
    if (tgt >= 0) {
        const int at = OP == M2LV_M2M && L.plist ? pbeg + lane : tgt;  // of a part: list entry or box
        double2* out = L.dsplit > 1 ? L.partial + ((int64_t)part * L.size + at) * NX : L.dst + (int64_t)tgt * SX;
        if constexpr (W == 0)  // coefficients beyond this launch's order are zero
            for (int64_t i = NX; i < SX; ++i) out[i] = make_double2(0.0, 0.0);
        sfor<0, N>([&](auto NN) {
            constexpr int n = decltype(NN)::value;
            if constexpr (PT.deg[n] == W)
                sfor<0, n + 1>([&](auto M) {  // (-1)^m: see pack_m2lv
                    constexpr int m = decltype(M)::value;
                    const double2 v = acc[tri(n) + m];
                    out[tri(n) + m] = (m & 1) ? make_double2(-v.x, -v.y) : v;
                    if constexpr (OP == M2LV_M2M) mx = fmax(mx, fmax(fabs(v.x), fabs(v.y)));
                });
        });
    }
    if constexpr (OP == M2LV_M2M)
        if (L.absmax && L.dsplit == 1) wave_absmax(mx, L.absmax);  // of parts: with their sum
}

template <int N, int NW, bool PACKED, int OP = M2LV_M2L>
__global__ void __launch_bounds__(64 * NW, 2) k_m2lv(M2LStepTables T, M2lvTables V, M64Level A)
{
    using B = M2lvBuf<N, NW>;
    __shared__ double2 state[tri(N) * kM2lvTile];
    __shared__ __align__(16) double tab[2][B::size];
    __shared__ m2lv_near_t<PACKED> near[27][kM2lvTile];
    const RtrLevel& L = A.L;
    const int blk = xcd_local_block(blockIdx.x, gridDim.x);
    int tile, c, part = 0, pbeg = 0, pend = L.num_parents;
    if constexpr (OP == M2LV_M2M) {
        tile = blk / L.dsplit;
        part = blk - tile * L.dsplit;
        c = 8;  // of the step tables
    } else if (L.csorted) {
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
    pbeg += tile * kM2lvTile;
    if constexpr (PACKED) m64_parents<kM2lvTile, 64 * NW>(A, pbeg, pend, near);
    else if constexpr (OP == M2LV_M2L) m64_children<kM2lvTile, 64 * NW>(A, pbeg, pend, near);
    else if constexpr (OP == M2LV_M2M) m64_children<kM2lvTile, 64 * NW, 13, 14>(A, pbeg, pend, near);
    __syncthreads();
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    sfor<0, NW>([&](auto WW) {
        constexpr int W = decltype(WW)::value;
        if (w == W) m2lv_wave<N, NW, W, PACKED, OP>(T, V, A, state, tab, near, c, part, pbeg, pend);
    });
}

template <int N>
hipError_t do_m2lv(int op, const M2LStepTables& T, const M2lvTables& V, const M64Level& A, hipStream_t st)
{
    constexpr int NW = m2lv_nw(N);
    const RtrLevel& L = A.L;
    const int tiles = (L.num_parents + kM2lvTile - 1) / kM2lvTile;
    int blocks = 0;
    if (op == M2LV_M2M) {
        if (L.csorted || L.dsplit < 1 || L.dsplit > 8) return hipErrorInvalidValue;
        blocks = tiles * L.dsplit;
    } else if (L.csorted) {
        if (L.dsplit != 1 || !L.plist || L.coff[8] != L.num_parents) return hipErrorInvalidValue;
        int mt = 0;
        for (int c = 0; c < 8; ++c) {
            const int t = L.ctile[c + 1] - L.ctile[c];
            if (t != (L.coff[c + 1] - L.coff[c] + kM2lvTile - 1) / kM2lvTile) return hipErrorInvalidValue;
            mt = std::max(mt, t);
        }
        blocks = 8 * mt;
    } else {
        if (L.tiles != tiles || (op == M2LV_L2L && L.dsplit != 1)) return hipErrorInvalidValue;
        blocks = L.tiles * 8 * L.dsplit;
    }
    if (blocks <= 0) return hipSuccess;
    const dim3 grid(blocks), block(64 * NW);
    if (op == M2LV_M2M) hipLaunchKernelGGL((k_m2lv<N, NW, false, M2LV_M2M>), grid, block, 0, st, T, V, A);
    else if (op == M2LV_L2L) hipLaunchKernelGGL((k_m2lv<N, NW, false, M2LV_L2L>), grid, block, 0, st, T, V, A);
    else if (A.packed) hipLaunchKernelGGL((k_m2lv<N, NW, true>), grid, block, 0, st, T, V, A);
    else hipLaunchKernelGGL((k_m2lv<N, NW, false>), grid, block, 0, st, T, V, A);
    return hipGetLastError();
}

}  // namespace lfmm
