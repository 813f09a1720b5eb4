// m2l64.cpp -- host packing of the FP64 operator tables into the 4 x 4 blocks
// and the step lists of the matrix-core M2L (m2l64_kernels.h).
#include "m2l64.h"

namespace lfmm {

template <int N> hipError_t do_m2l64(const M2LStepTables& S, const M64Tables& T, const M64Level& A, hipStream_t st);

hipError_t launch_m2l64(int N, const M2LStepTables& S, const M64Tables& T, const M64Level& A, hipStream_t st)
{
    switch (N) {
#define X(n) case n: return do_m2l64<n>(S, T, A, st);
        X(14) X(15) X(16) X(17) X(18)
#undef X
    default: return hipErrorInvalidValue;
    }
}

// Block entries are stored [k][i] (K index, row): lane l of a wave takes entry
// 4 (l / 16) + l % 4, the A-operand element of v_mfma_f64_4x4x4.
// The inverse rotation is Ry(-theta)_{mu m} = (-1)^(mu + m) Ry(theta)_{mu m}:
// (-1)^m is folded into the rows of the translation blocks of order m, and
// (-1)^mu into the kernel's final store, so both rotations read one table.
void pack_m2l64(const OpTables& T, M64Pack& out)
{
    const int N = T.N, blocks = m64_blocks(N), chunks = m64_chunks(N);
    const int pairs = (blocks + 1) / 2;
    out.rot.assign((size_t)T.num_theta * pairs * 64, 0.0);
    for (int t = 0; t < T.num_theta; ++t)
        for (int n = 0; n < N; ++n) {
            const int ch = m64_chunks(n + 1);
            const double* pq = &T.rot[((size_t)t * rot_size(N) + rot_base(n)) * 2];
            for (int m = 0; m <= n; ++m)
                for (int k = 0; k <= n; ++k) {
                    const int q = m64_rot_at(N, n) + (k / 4) * ch + m / 4;
                    double* e = &out.rot[((size_t)t * pairs + q / 2) * 64 + ((k % 4) * 4 + m % 4) * 2 + (q & 1)];
                    e[0] = pq[2 * (m * (n + 1) + k)];
                    e[32] = pq[2 * (m * (n + 1) + k) + 1];
                }
        }
    out.trans.assign((size_t)kNumTrans * pairs * 32, 0.0);
    for (int t = 0; t < kNumTrans; ++t)
        for (int m = 0; m < N; ++m) {
            const int ct = m64_chunks(N - m), L = N - m;
            const double* tt = &T.trans[(size_t)t * tr_size(N) + tr_base(N, m)];
            for (int j = 0; j < L; ++j)  // degree m + j, chunk position from the top
                for (int i = 0; i < L; ++i) {
                    const int pj = L - 1 - j, pi = L - 1 - i;
                    const int q = m64_tr_base(N, m) + (pi / 4) * ct + pj / 4;
                    const double v = tt[j * L + i];
                    out.trans[((size_t)t * pairs + q / 2) * 32 + ((pi % 4) * 4 + pj % 4) * 2 + (q & 1)] =
                        (m & 1) ? -v : v;
                }
        }
    // Rz(phi): part = part cos + other part * (-sin for the real, sin for the
    // imaginary part)
    out.ephi.assign((size_t)kNumDirs * chunks * 16, 0.0);
    for (int d = 0; d < kNumDirs; ++d)
        for (int k = 0; k < N; ++k)
            for (int im = 0; im < 2; ++im) {
                const double* cs = &T.ephi[((size_t)d * N + k) * 2];
                double* e = &out.ephi[((size_t)d * 2 + im) * chunks * 8 + 2 * k];
                e[0] = cs[0];
                e[1] = im ? cs[1] : -cs[1];
            }
}

// Steps: the L2L, then the class's directions by operator group (same
// polar angle and distance), the groups by their first direction in the
// class's list.  A group is one |x|, |y| pair and one z, so its sources lie
// in one or two child classes and the list's source-class-major order
// (whose sources stay cache-resident) holds for the groups.
void pack_m2l_steps(const OpTables& T, M2LSteps& out)
{
    out.steps.assign((size_t)9 * kM64Steps * 2, -1);
    out.groups.assign((size_t)9 * kM64Groups * 4, 0);
    for (int c = 0; c < 8; ++c) {
        const int* dirs = &T.class_dirs[c * kDirsPerClass];
        int* st = &out.steps[(size_t)c * kM64Steps * 2];
        int* gr = &out.groups[(size_t)c * kM64Groups * 4];
        int ns = 0, ng = 0;
        auto open = [&](int d, int tr) {
            int* g = gr + 4 * ng++;
            g[0] = T.dir_theta[d];
            g[1] = tr;
            g[2] = ns;
        };
        open(kDiagBase + 7 - c, kTransL2L);
        st[0] = kDiagBase + 7 - c;
        gr[3] = ++ns;
        std::vector<char> used(kDirsPerClass, 0);
        for (int i = 0; i < kDirsPerClass; ++i) {
            if (used[i]) continue;
            open(dirs[i], T.dir_trans[dirs[i]]);
            const int first = ns;
            for (int j = i; j < kDirsPerClass && ns - first < kM64GroupMax; ++j) {
                const int d = dirs[j];
                if (used[j] || T.dir_theta[d] != T.dir_theta[dirs[i]] || T.dir_trans[d] != T.dir_trans[dirs[i]]) continue;
                used[j] = 1;
                int k = 0, s = 0;
                for (int ax = 0; ax < 3; ++ax) {  // child coordinate c + d along each axis, x first
                    const int v = ((c >> (2 - ax)) & 1) + T.dir_vec[4 * d + ax];
                    k = 3 * k + (v >> 1) + 1;
                    s = 2 * s + (v & 1);
                }
                st[2 * ns] = d;
                st[2 * ns + 1] = 8 * k + s;
                ++ns;
            }
            gr[4 * ng - 1] = ns;
        }
        out.nsteps[c] = ns;
    }
    int* st = &out.steps[(size_t)8 * kM64Steps * 2];
    int* gr = &out.groups[(size_t)8 * kM64Groups * 4];
    int ns = 0, ng = 0;
    std::vector<char> used(8, 0);
    for (int i = 0; i < 8; ++i) {
        if (used[i]) continue;
        int* g = gr + 4 * ng++;
        g[0] = T.dir_theta[kDiagBase + i];
        g[1] = kTransM2M;
        g[2] = ns;
        for (int s = i; s < 8; ++s) {
            if (used[s] || T.dir_theta[kDiagBase + s] != g[0]) continue;
            used[s] = 1;
            st[2 * ns] = kDiagBase + s;
            st[2 * ns + 1] = 8 * 13 + s;
            ++ns;
        }
        g[3] = ns;
    }
    out.nsteps[8] = ns;
}

}  // namespace lfmm
