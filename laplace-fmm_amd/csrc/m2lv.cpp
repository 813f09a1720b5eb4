// m2lv.cpp -- host packing of the FP64 operator tables into the coefficient
// streams of the vector M2L (m2lv_kernels.h), and its dispatch over N.
#include "m2lv.h"

namespace lfmm {

template <int N> hipError_t do_m2lv(int op, const M2LStepTables& S, const M2lvTables& V, const M64Level& A, hipStream_t st);

#define LFMM_M2LV_TERMS(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13)

hipError_t launch_m2lv(int N, int op, const M2LStepTables& S, const M2lvTables& V, const M64Level& A, hipStream_t st)
{
    switch (N) {
#define X(n) case n: return do_m2lv<n>(op, S, V, A, st);
        LFMM_M2LV_TERMS(X)
#undef X
    default: return hipErrorInvalidValue;
    }
}

// The inverse rotation is Ry(-theta)_{mu m} = (-1)^(mu + m) Ry(theta)_{mu m}:
// (-1)^m is folded into the translation's output rows of order m, (-1)^mu
// into the kernel's final store, so both rotations read one stream.
template <int N>
static void pack(const OpTables& T, M2lvPack& out)
{
    constexpr int NW = m2lv_nw(N);
    constexpr M2lvPart<N, NW> P{};
    constexpr M2lvLayout<N, NW> LY{};
    out.rot_regs = LY.rot_reg[NW];
    out.tr_regs = LY.tr_reg[NW];
    out.rot.assign((size_t)T.num_theta * out.rot_regs * 16, 0.0);
    out.trans.assign((size_t)kNumTrans * out.tr_regs * 16, 0.0);
    out.ephi.assign((size_t)kNumDirs * 32, 0.0);
    for (int t = 0; t < T.num_theta; ++t)
        for (int n = 0; n < N; ++n) {
            const double* pq = &T.rot[((size_t)t * rot_size(N) + rot_base(n)) * 2];
            double* stream = &out.rot[((size_t)t * out.rot_regs + LY.rot_reg[P.deg[n]]) * 16];
            for (int r = 0; 2 * r <= n; ++r)
                for (int k = 0; k <= n; ++k) {
                    double* o = stream + m2lv_pos(LY.rot[n][r][k]);
                    for (int q = 0; q < 2; ++q)
                        for (int m = 2 * r; m <= n && m < 2 * r + 2; ++m)
                            if (q == 0 || (m > 0 && k > 0)) *o++ = pq[2 * (m * (n + 1) + k) + q];
                }
        }
    for (int t = 0; t < kNumTrans; ++t)
        for (int m = 0; m < N; ++m) {
            const int len = N - m;
            const double* tt = &T.trans[(size_t)t * tr_size(N) + tr_base(N, m)];
            double* stream = &out.trans[((size_t)t * out.tr_regs + LY.tr_reg[P.ord[m]]) * 16];
            for (int r = 0; 2 * r < len; ++r)
                for (int i = 0; i < len; ++i)
                    for (int j = 2 * r; j < len && j < 2 * r + 2; ++j)
                        stream[m2lv_pos(LY.tr[m][r][i]) + j - 2 * r] = (m & 1) ? -tt[j * len + i] : tt[j * len + i];
        }
    for (int d = 0; d < kNumDirs; ++d)
        for (int k = 0; k < N; ++k) {
            out.ephi[(size_t)d * 32 + k] = T.ephi[((size_t)d * N + k) * 2];
            out.ephi[(size_t)d * 32 + 16 + k] = T.ephi[((size_t)d * N + k) * 2 + 1];
        }
}

void pack_m2lv(const OpTables& T, M2lvPack& out)
{
    switch (T.N) {
#define X(n) case n: pack<n>(T, out); break;
        LFMM_M2LV_TERMS(X)
#undef X
    default: break;
    }
}

}  // namespace lfmm
