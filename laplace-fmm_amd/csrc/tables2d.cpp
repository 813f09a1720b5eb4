// tables2d.cpp -- host operator tables of the 2D (complex-series) FMM.
//
// Expansions are stored normalised per level, with h the box edge:
//   multipole  at_k = a_k / h^k,   local  bt_k = b_k h^k,
// where a, b are the reference's coefficients (src/cpu/multipole.cpp:22-97:
// a_0 = sum q, a_k = -sum q (z - c)^k / k; the local expansion is evaluated
// as Re sum b_k (z - c)^k).  With this scaling every translation depends only
// on an integer box offset d (complex, in box units):
//   M2M (child class c, delta = child centre - parent centre in child edges)
//     bt_j = 2^-j [ sum_{s=1..j} at_s delta^(j-s) C(j-1, s-1) - at_0 delta^j / j ],  bt_0 = at_0
//   M2L (d = source centre - target centre, in box edges)
//     bt_0 = at_0 (log h + conj(log(-d))) + sum_{j>=1} (-1)^j at_j / d^j
//     bt_l = [ -at_0 / l + sum_{j>=1} (-1)^j at_j C(l+j-1, j-1) / d^j ] / d^l
//   L2L (parent -> child class c): bt_k = sum_{j>=k} at_j 2^-j C(j, k) delta^(j-k)
// (reference M2M :38-53, M2L :66-84, L2L :86-97).  The level term at_0 log h
// of the M2L is added in the kernel.  All tables are computed in long double.
#include "lfmm_internal.h"

#include <cmath>
#include <complex>
#include <cstring>

namespace lfmm {

using ld = long double;
using cld = std::complex<ld>;

static ld binom_l(int n, int k)
{
    if (k < 0 || k > n) return 0;
    ld r = 1;
    for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
    return r;
}

static cld cpow_l(cld z, int e)
{
    cld r = 1;
    for (int i = 0; i < e; ++i) r *= z;
    return r;
}

static void put(std::vector<double>& v, size_t i, cld z)
{
    v[2 * i] = (double)z.real();
    v[2 * i + 1] = (double)z.imag();
}

// child class c = (x bit << 1) | y bit of the child's Morton key
static cld child_offset(int c) { return cld((c & 2) ? 0.5L : -0.5L, (c & 1) ? 0.5L : -0.5L); }

void build_op_tables_2d(int N, OpTables2d& T)
{
    T.N = N;
    T.dir_vec.clear();
    for (int dx = -3; dx <= 3; ++dx)
        for (int dy = -3; dy <= 3; ++dy) {
            if (std::abs(dx) <= 1 && std::abs(dy) <= 1) continue;
            T.dir_vec.push_back(dx);
            T.dir_vec.push_back(dy);
        }
    const int ND = (int)T.dir_vec.size() / 2;  // 40
    T.class_dirs.assign(4 * kDirsPerClass2d, -1);
    for (int c = 0; c < 4; ++c) {
        const int cx = (c >> 1) & 1, cy = c & 1;
        int cnt = 0;
        for (int d = 0; d < ND; ++d) {
            const int x = T.dir_vec[2 * d], y = T.dir_vec[2 * d + 1];
            if (x < -2 - cx || x > 3 - cx || y < -2 - cy || y > 3 - cy) continue;
            T.class_dirs[c * kDirsPerClass2d + cnt++] = d;
        }
    }
    T.m2l.assign((size_t)ND * N * N * 2, 0.0);
    std::vector<cld> pw(2 * N);  // z^k
    for (int d = 0; d < ND; ++d) {
        const cld z((ld)T.dir_vec[2 * d], (ld)T.dir_vec[2 * d + 1]);
        pw[0] = 1;
        for (int k = 1; k < 2 * N; ++k) pw[k] = pw[k - 1] * z;
        for (int l = 0; l < N; ++l)
            for (int j = 0; j < N; ++j) {
                cld v;
                const ld sj = (j & 1) ? -1.0L : 1.0L;
                if (l == 0 && j == 0) v = std::conj(std::log(-z));
                else if (l == 0) v = sj / pw[j];
                else if (j == 0) v = -1.0L / ((ld)l * pw[l]);
                else v = sj * binom_l(l + j - 1, j - 1) / pw[l + j];
                put(T.m2l, ((size_t)d * N + l) * N + j, v);
            }
    }
}

void build_shift_tables_2d(OpTables2d& T)
{
    const int N = T.N;
    T.m2m.assign((size_t)4 * N * N * 2, 0.0);
    T.l2l.assign((size_t)4 * N * N * 2, 0.0);
    for (int c = 0; c < 4; ++c) {
        const cld dl = child_offset(c);
        for (int j = 0; j < N; ++j) {
            const ld sc = ldexpl(1.0L, -j);
            for (int s = 0; s < N; ++s) {
                cld v = 0;
                if (j == 0 && s == 0) v = 1;
                else if (j >= 1 && s == 0) v = -sc * cpow_l(dl, j) / (ld)j;
                else if (s >= 1 && s <= j) v = sc * cpow_l(dl, j - s) * binom_l(j - 1, s - 1);
                put(T.m2m, ((size_t)c * N + j) * N + s, v);
            }
        }
        for (int k = 0; k < N; ++k)
            for (int j = 0; j < N; ++j) {
                const cld v = (j >= k) ? ldexpl(1.0L, -j) * binom_l(j, k) * cpow_l(dl, j - k) : cld(0);
                put(T.l2l, ((size_t)c * N + k) * N + j, v);
            }
    }
}

// M2L: bt = diag(d^-l) B diag((-1)^j d^-j) at with one real B for every
// direction (B_lj = C(l+j-1, j-1), column 0: -1/l, row 0: 1), apart from
// bt_0 += at_0 (log h + conj(log(-d))).  M2M and L2L: child offsets are
// i^r e, so a child enters M2M as i^(r (j-s)), which depends on (j - s) mod 4
// alone: the children's four sums with weights i^(r m) go through one real
// matrix, and the L2L is the transpose.
void pack_2d(const OpTables2d& T, Pack2d& P)
{
    const int N = T.N;
    const int ND = (int)T.dir_vec.size() / 2, NB = m2l2d_blocks(N), pairs = m2l2d_pairs(N), regs = m2l2d_regs(N);
    P.m2l.assign((size_t)NB * regs * 16, 0.0);
    for (int l = 0; l < N; ++l)
        for (int j = 0; j < N; ++j) {
            ld v = 0;
            if (l == 0) v = j == 0 ? 0 : 1;
            else v = j == 0 ? -1.0L / (ld)l : binom_l(l + j - 1, j - 1);
            const int b = l / (2 * pairs), r = l - b * 2 * pairs;
            P.m2l[(size_t)b * regs * 16 + (size_t)(r / 2) * 2 * N + 2 * j + r % 2] = (double)v;
        }
    P.src.assign((size_t)ND * 64, 0.0);
    P.out.assign((size_t)ND * NB * 32, 0.0);
    P.log.assign((size_t)ND * 2, 0.0);
    for (int d = 0; d < ND; ++d) {
        const cld z((ld)T.dir_vec[2 * d], (ld)T.dir_vec[2 * d + 1]);
        for (int k = 0; k < N; ++k) {
            const cld w = 1.0L / cpow_l(z, k);
            P.src[(size_t)d * 64 + k] = (double)((k & 1) ? -w.real() : w.real());
            P.src[(size_t)d * 64 + 32 + k] = (double)((k & 1) ? -w.imag() : w.imag());
            const int b = k / (2 * pairs), r = k - b * 2 * pairs;
            P.out[((size_t)d * NB + b) * 32 + r] = (double)w.real();
            P.out[((size_t)d * NB + b) * 32 + 16 + r] = (double)w.imag();
        }
        const cld lg = std::conj(std::log(-z));
        P.log[2 * d] = (double)lg.real();
        P.log[2 * d + 1] = (double)lg.imag();
    }
    const cld e = child_offset(3);
    P.m2m.assign((size_t)N * N, 0.0);
    P.l2l.assign((size_t)N * N, 0.0);
    P.down.assign((size_t)N * 2, 0.0);
    P.up.assign((size_t)N * 2, 0.0);
    for (int k = 0; k < N; ++k) {
        for (int j = 0; j < N; ++j) {
            P.m2m[(size_t)k * N + j] = (double)(j == 0 ? (k == 0 ? 1.0L : -1.0L / (ld)k) : binom_l(k - 1, j - 1));
            P.l2l[(size_t)k * N + j] = (double)binom_l(j, k);
        }
        const cld a = cpow_l(e / 2.0L, k), b = 1.0L / cpow_l(e, k);
        P.down[2 * k] = (double)a.real();
        P.down[2 * k + 1] = (double)a.imag();
        P.up[2 * k] = (double)b.real();
        P.up[2 * k + 1] = (double)b.imag();
    }
}

void pack_log_2d(std::vector<LogEntry2d>& t)
{
    auto start = [](int i) {
        const uint64_t u = (uint64_t)(uint32_t)(kLog2dFirst + i * 0x2000) << 32;
        double v;
        std::memcpy(&v, &u, sizeof v);
        return v;
    };
    t.resize(kLog2dEntries);
    for (int i = 0; i < kLog2dEntries; ++i) {
        const double inv = i == kLog2dOne ? 1.0 : std::rint(512.0 / (start(i) + start(i + 1))) / 256.0;
        const ld log_c = -std::log((ld)inv);
        const double hi = std::ldexp(std::rint(std::ldexp((double)log_c, 42)), -42);
        t[i] = {hi, (float)inv, (float)(log_c - hi)};
    }
}

}  // namespace lfmm
