// host_check.cpp -- exercises the host-side C++ of the library without a
// GPU: the FP64 table builders (3D and 2D), their packed forms unpacked again
// as the kernels read them, the dense and split-fp16 M2L operators, the arena,
// the exact-file reader and writer, ReadError's statistics, and the argument
// checks every entry point runs before device work.  Built
// together with the library's host sources under AddressSanitizer and
// UndefinedBehaviorSanitizer (make sanitize); any report aborts the run.
// Prints "host_check ok" and exits 0 when every check holds.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "lfmm.h"
#include "api_internal.h"
#include "lfmm_internal.h"
#include "m2l64.h"
#include "m2lv.h"

#include <complex>
#include <utility>

namespace {

int failures = 0;

void expect(bool ok, const char* what, int detail = 0)
{
    if (!ok) {
        std::printf("FAILED: %s (%d)\n", what, detail);
        ++failures;
    }
}

// d^j(beta) is orthogonal: d d^T = I.
void check_wigner()
{
    for (int j = 0; j <= 24; ++j) {
        const int n = 2 * j + 1;
        std::vector<double> d((size_t)n * n);
        expect(lfmm_host_wigner_d(j, 0.37 + 0.1 * j, d.data()) == LFMM_OK, "wigner status", j);
        double worst = 0.0;
        for (int a = 0; a < n; ++a)
            for (int b = 0; b < n; ++b) {
                double s = 0.0;
                for (int k = 0; k < n; ++k) s += d[(size_t)a * n + k] * d[(size_t)b * n + k];
                worst = std::fmax(worst, std::fabs(s - (a == b ? 1.0 : 0.0)));
            }
        expect(worst < 1e-11, "wigner orthogonality", j);
    }
    expect(lfmm_host_wigner_d(-1, 0.1, nullptr) == LFMM_ERR_INVALID, "wigner bad j");
    expect(lfmm_host_wigner_d(65, 0.1, nullptr) == LFMM_ERR_INVALID, "wigner j cap");
}

// The tables of the expansion sizes at the ends of the range and of the
// sizes the solves use most, built once per size; the C entry points that
// copy them out are exercised at one size each (every call rebuilds).
void check_tables_3d()
{
    for (int N : {1, 2, 3, 9, 13, LFMM_MAX_TERMS_3D}) {
        lfmm::OpTables T;
        lfmm::build_op_tables(N, T);
        for (const std::vector<double>* t : {&T.rot, &T.ephi, &T.trans, &T.knm}) {
            expect(!t->empty(), "op table size", N);
            for (double v : *t) expect(std::isfinite(v), "op table finite", N);
        }
        for (int d : T.dir_theta) expect(d >= 0 && d < T.num_theta, "dir_theta", N);
        for (int d : T.class_dirs) expect(d >= 0 && d < lfmm::kNumM2LDirs, "class_dirs", N);
        std::vector<double> K((size_t)N * N * N * N);
        for (int dir : {0, 57, 188, lfmm::kNumM2LDirs - 1}) {
            lfmm::m2l_dense_matrix(T, dir, K.data());
            for (double v : K) expect(std::isfinite(v), "m2l dense finite", N);
        }
        std::vector<uint16_t> pk;
        std::vector<int> kpre;
        double kinv = 0.0;
        lfmm::pack_m2l16(T, pk, kinv, kpre);
        const int tiles = (N * N + 31) / 32;
        expect(!pk.empty() && kinv > 0.0, "m2l16 pack", N);
        expect(kpre.size() == (size_t)lfmm::kNumM2LDirs * tiles * 2, "m2l16 prefix count", N);
        for (size_t i = 0; i + 1 < kpre.size(); i += 2)
            expect(kpre[i] >= 0 && kpre[i + 1] >= 0 && kpre[i + 1] <= kpre[i] + 32 * tiles, "m2l16 prefixes", N);
    }
    const int N = 5;
    for (int which = 0; which < 8; ++which) {
        const int64_t count = lfmm_host_op_tables(N, which, nullptr, 0);
        expect(count > 0, "op table count", which);
        if (count <= 0) continue;
        std::vector<double> buf((size_t)count);  // 8-byte slots hold either element size
        expect(lfmm_host_op_tables(N, which, buf.data(), count) == count, "op table copy", which);
    }
    std::vector<double> K((size_t)N * N * N * N);
    expect(lfmm_host_m2l_dense(N, 7, K.data()) == LFMM_OK, "m2l dense entry");
    double kinv = 0.0;
    const int64_t np = lfmm_host_m2l16_pack(N, nullptr, 0, &kinv, nullptr);
    expect(np > 0, "m2l16 pack entry size");
    std::vector<uint16_t> pk((size_t)(np > 0 ? np : 1));
    std::vector<int32_t> kpre((size_t)lfmm::kNumM2LDirs * 2);
    expect(lfmm_host_m2l16_pack(N, pk.data(), np, &kinv, kpre.data()) == np, "m2l16 pack entry");
    expect(lfmm_host_op_tables(0, 0, nullptr, 0) < 0, "op tables N=0");
    expect(lfmm_host_op_tables(19, 0, nullptr, 0) < 0, "op tables N=19");
    expect(lfmm_host_op_tables(5, 8, nullptr, 0) < 0, "op tables bad kind");
    expect(lfmm_host_m2l_dense(5, lfmm::kNumM2LDirs, nullptr) != LFMM_OK, "m2l dense bad dir");
}

// The step lists: the L2L, then every direction of the class once, in groups of
// one operator that follow one another; the source of a step is the cell
// (child + direction) as (neighbour parent, class).  List 8: the 8 children.
void check_m2l_steps(const lfmm::OpTables& T)
{
    using namespace lfmm;
    M2LSteps S;
    pack_m2l_steps(T, S);
    expect(S.steps.size() == (size_t)9 * kM64Steps * 2 && S.groups.size() == (size_t)9 * kM64Groups * 4, "step list sizes");
    for (int c = 0; c < 9; ++c) {
        const int n = S.nsteps[c];
        expect(n == (c < 8 ? kDirsPerClass + 1 : 8), "step count", c);
        std::vector<int> seen(kNumDirs, 0);
        int at = 0, g = 0;
        for (; g < kM64Groups && at < n; ++g) {
            const int* gr = &S.groups[((size_t)c * kM64Groups + g) * 4];
            expect(gr[2] == at && gr[3] > at && gr[3] - at <= kM64GroupMax && gr[3] <= n, "group range", c);
            if (gr[2] != at || gr[3] <= at || gr[3] > n) return;
            for (; at < gr[3]; ++at) {
                const int d = S.steps[((size_t)c * kM64Steps + at) * 2], ks = S.steps[((size_t)c * kM64Steps + at) * 2 + 1];
                expect(d >= 0 && d < kNumDirs, "step direction", c);
                if (d < 0 || d >= kNumDirs) return;
                ++seen[d];
                const int trans = c == 8 ? kTransM2M : ks < 0 ? kTransL2L : T.dir_trans[d];
                expect(T.dir_theta[d] == gr[0] && trans == gr[1], "group operator", c);
                if (c == 8) expect(ks == 8 * 13 + d - kDiagBase, "child of a parent", c);
                else if (ks < 0) expect(at == 0 && d == kDiagBase + 7 - c, "L2L step", c);
                else
                    for (int ax = 0; ax < 3; ++ax) {
                        const int parent = (ks / 8) / (ax == 0 ? 9 : ax == 1 ? 3 : 1) % 3 - 1;
                        const int child = (c >> (2 - ax)) & 1, source = (ks >> (2 - ax)) & 1;
                        expect(2 * parent + source == child + T.dir_vec[4 * d + ax], "step source", c);
                    }
            }
        }
        expect(at == n, "steps in groups", c);
        for (int i = 0; i < (c < 8 ? kDirsPerClass : 8); ++i)
            expect(seen[c < 8 ? T.class_dirs[c * kDirsPerClass + i] : kDiagBase + i] == 1, "direction once", c);
    }
}

// The streams of the vector M2L, read as its kernel does: the blocks of a wave
// one after another, 16 coefficients to a register, a flag on the last block of
// every register but the final one.
template <int N>
void check_m2lv(const lfmm::OpTables& T)
{
    using namespace lfmm;
    constexpr int NW = m2lv_nw(N);
    constexpr M2lvPart<N, NW> P{};
    constexpr M2lvLayout<N, NW> LY{};
    M2lvPack V;
    pack_m2lv(T, V);
    expect(V.rot.size() == (size_t)T.num_theta * 16 * LY.rot_reg[NW], "m2lv rotation size", N);
    expect(V.trans.size() == (size_t)kNumTrans * 16 * LY.tr_reg[NW], "m2lv translation size", N);
    expect(V.ephi.size() == (size_t)kNumDirs * 32, "m2lv azimuth size", N);
    for (int w = 0; w < NW; ++w) {
        int reg = 0, next = 0, flagged = 1;
        auto block = [&](int at, int size) {
            const int p = m2lv_pos(at);
            if (p / 16 != reg || next == 0) expect(next == 0 ? p == 0 : p == 16 * (reg + 1) && flagged, "m2lv register", N);
            else expect(p == next && !flagged, "m2lv block", N);
            expect(p % 16 + size <= 16, "m2lv block in a register", N);
            reg = p / 16;
            next = p + size;
            flagged = m2lv_last(at);
        };
        for (int n = N - 1; n >= 0; --n)
            if (P.deg[n] == w)
                for (int r = 0; 2 * r <= n; ++r)
                    for (int k = 0; k <= n; ++k) block(LY.rot[n][r][k], m2lv_rot_block(n, r, k));
        expect(next == 0 || (!flagged && reg + 1 == LY.rot_reg[w + 1] - LY.rot_reg[w]), "m2lv rotation registers", N);
        reg = next = 0;
        flagged = 1;
        for (int m = 0; m < N; ++m)
            if (P.ord[m] == w)
                for (int r = 0; 2 * r < N - m; ++r)
                    for (int i = 0; i < N - m; ++i) block(LY.tr[m][r][i], 2 * r + 1 < N - m ? 2 : 1);
        expect(next == 0 || (!flagged && reg + 1 == LY.tr_reg[w + 1] - LY.tr_reg[w]), "m2lv translation registers", N);
    }
    for (int t = 0; t < T.num_theta; ++t)
        for (int n = 0; n < N; ++n)
            for (int m = 0; m <= n; ++m)
                for (int k = 0; k <= n; ++k) {
                    const double* pq = &T.rot[((size_t)t * rot_size(N) + rot_base(n) + m * (n + 1) + k) * 2];
                    const double* b = &V.rot[((size_t)t * LY.rot_reg[NW] + LY.rot_reg[P.deg[n]]) * 16 + m2lv_pos(LY.rot[n][m / 2][k])];
                    const int rows = (m | 1) <= n ? 2 : 1;
                    expect(b[m % 2] == pq[0], "m2lv P", N);
                    if (k > 0 && m > 0) expect(b[rows + (m < 2 ? 0 : m % 2)] == pq[1], "m2lv Q", N);
                }
    for (int t = 0; t < kNumTrans; ++t)
        for (int m = 0; m < N; ++m)
            for (int j = 0; j < N - m; ++j)
                for (int i = 0; i < N - m; ++i) {
                    const double v = T.trans[(size_t)t * tr_size(N) + tr_base(N, m) + j * (N - m) + i];
                    const double* b = &V.trans[((size_t)t * LY.tr_reg[NW] + LY.tr_reg[P.ord[m]]) * 16 + m2lv_pos(LY.tr[m][j / 2][i])];
                    expect(b[j % 2] == ((m & 1) ? -v : v), "m2lv translation", N);
                }
    for (int d = 0; d < kNumDirs; ++d)
        for (int k = 0; k < N; ++k)
            for (int s = 0; s < 2; ++s)
                expect(V.ephi[(size_t)d * 32 + 16 * s + k] == T.ephi[((size_t)d * N + k) * 2 + s], "m2lv azimuth", N);
}

// The 4 x 4 blocks of the matrix-core M2L: every entry in its place, all others 0.
void check_m2l64(const lfmm::OpTables& T)
{
    using namespace lfmm;
    const int N = T.N, pairs = (m64_blocks(N) + 1) / 2;
    M64Pack M;
    pack_m2l64(T, M);
    expect(M.rot.size() == (size_t)T.num_theta * pairs * 64 && M.trans.size() == (size_t)kNumTrans * pairs * 32 &&
               M.ephi.size() == (size_t)kNumDirs * m64_chunks(N) * 16, "m2l64 sizes", N);
    auto take = [&](std::vector<double>& v, size_t at, double want, const char* what) {
        expect(at < v.size() && v[at] == want, what, N);
        if (at < v.size()) v[at] = 0.0;
    };
    for (int t = 0; t < T.num_theta; ++t)
        for (int n = 0; n < N; ++n)
            for (int m = 0; m <= n; ++m)
                for (int k = 0; k <= n; ++k) {
                    const int q = m64_rot_at(N, n) + (k / 4) * m64_chunks(n + 1) + m / 4;
                    const double* pq = &T.rot[((size_t)t * rot_size(N) + rot_base(n) + m * (n + 1) + k) * 2];
                    const size_t at = ((size_t)t * pairs + q / 2) * 64 + ((k % 4) * 4 + m % 4) * 2 + q % 2;
                    take(M.rot, at, pq[0], "m2l64 P");
                    take(M.rot, at + 32, pq[1], "m2l64 Q");
                }
    for (int t = 0; t < kNumTrans; ++t)
        for (int m = 0; m < N; ++m)
            for (int j = m; j < N; ++j)
                for (int i = m; i < N; ++i) {  // degrees, chunks from the top
                    const int q = m64_tr_base(N, m) + (N - 1 - i) / 4 * m64_chunks(N - m) + (N - 1 - j) / 4;
                    const double v = T.trans[(size_t)t * tr_size(N) + tr_base(N, m) + (j - m) * (N - m) + i - m];
                    take(M.trans, ((size_t)t * pairs + q / 2) * 32 + ((N - 1 - i) % 4 * 4 + (N - 1 - j) % 4) * 2 + q % 2,
                         (m & 1) ? -v : v, "m2l64 translation");
                }
    for (int d = 0; d < kNumDirs; ++d)
        for (int k = 0; k < N; ++k) {
            const double* cs = &T.ephi[((size_t)d * N + k) * 2];
            const size_t at = (size_t)d * m64_chunks(N) * 16 + 2 * k;
            for (int im = 0; im < 2; ++im) {
                take(M.ephi, at + im * m64_chunks(N) * 8, cs[0], "m2l64 cos");
                take(M.ephi, at + im * m64_chunks(N) * 8 + 1, im ? cs[1] : -cs[1], "m2l64 sin");
            }
        }
    for (const std::vector<double>* v : {&M.rot, &M.trans, &M.ephi})
        for (double x : *v) expect(x == 0.0, "m2l64 padding", N);
}

template <int... I>
void check_m2lv_sizes(std::integer_sequence<int, I...>)
{
    (..., [] {
        lfmm::OpTables T;
        lfmm::build_op_tables(I + 1, T);
        check_m2lv<I + 1>(T);
        check_m2l_steps(T);
    }());
}

void check_packed_3d()
{
    check_m2lv_sizes(std::make_integer_sequence<int, lfmm::kM2lvMaxTerms>{});
    for (int N = lfmm::kM64MinTerms; N <= lfmm::kMaxTerms3d; ++N) {
        lfmm::OpTables T;
        lfmm::build_op_tables(N, T);
        check_m2l64(T);
        check_m2l_steps(T);
    }
}

// The factored 2D operators multiplied out against the matrices: products of
// three rounded factors, so 4 rounding errors per entry.
void check_packed_2d(const lfmm::OpTables2d& T)
{
    using cd = std::complex<double>;
    const int N = T.N, NB = lfmm::m2l2d_blocks(N), rows = 2 * lfmm::m2l2d_pairs(N);
    lfmm::Pack2d K;
    lfmm::pack_2d(T, K);
    expect(K.m2l.size() == (size_t)NB * lfmm::m2l2d_regs(N) * 16 && NB * rows >= N && rows <= 16 &&
               lfmm::m2l2d_regs(N) * 16 >= rows * N, "2d packed sizes", N);
    auto close = [&](cd a, cd b) { return std::abs(a - b) <= 1e-15 * std::abs(b); };
    auto entry = [](const std::vector<double>& v, size_t i) { return cd(v[2 * i], v[2 * i + 1]); };
    for (int d = 0; d < lfmm::kNumM2LDirs2d; ++d)
        for (int l = 0; l < N; ++l) {
            const int b = l / rows, r = l % rows;
            const cd out(K.out[((size_t)d * NB + b) * 32 + r], K.out[((size_t)d * NB + b) * 32 + 16 + r]);
            for (int j = 0; j < N; ++j) {
                const double e = K.m2l[(size_t)b * lfmm::m2l2d_regs(N) * 16 + r / 2 * 2 * N + 2 * j + r % 2];
                const cd src(K.src[(size_t)d * 64 + j], K.src[(size_t)d * 64 + 32 + j]);
                const cd v = l == 0 && j == 0 ? e + entry(K.log, d) : out * e * src;
                expect(close(v, entry(T.m2l, ((size_t)d * N + l) * N + j)), "2d m2l factors", N);
            }
        }
    const cd turn[4] = {{1, 0}, {0, 1}, {-1, 0}, {0, -1}};
    const int quarter[4] = {2, 1, 3, 0};  // child class c lies at i^quarter (1 + i) / 2
    for (int c = 0; c < 4; ++c)
        for (int a = 0; a < N; ++a)
            for (int b = 0; b < N; ++b) {
                const size_t i = ((size_t)c * N + a) * N + b;
                const cd up = b <= a ? entry(K.down, a) * K.m2m[a * N + b] * turn[quarter[c] * (a - b) & 3] * entry(K.up, b) : 0.0;
                expect(close(up, entry(T.m2m, i)), "2d m2m factors", N);
                const cd dn = b >= a ? entry(K.up, a) * K.l2l[a * N + b] * turn[quarter[c] * (b - a) & 3] * entry(K.down, b) : 0.0;
                expect(close(dn, entry(T.l2l, i)), "2d l2l factors", N);
            }
}

// Entries of the pair logarithm: r = m / c - 1 within 2^-7 over each interval,
// none at 1, log c to 2^-64.
void check_log_2d()
{
    std::vector<lfmm::LogEntry2d> t;
    lfmm::pack_log_2d(t);
    expect(t.size() == (size_t)lfmm::kLog2dEntries, "log table size");
    for (int i = 0; i < (int)t.size(); ++i) {
        auto start = [&](int k) {
            const int hi = lfmm::kLog2dFirst + k * 0x2000;
            return std::ldexp(1.0 + (hi & 0xfffff) * 0x1p-20, (hi >> 20) - 1023);
        };
        const double a = start(i), b = start(i + 1), inv = t[i].inv;
        expect(std::fabs(a * inv - 1.0) <= 0x1p-7 && std::fabs(b * inv - 1.0) <= 0x1p-7, "log interval", i);
        expect(a < 1.0 && b > 1.0 ? i == lfmm::kLog2dOne && inv == 1.0 && t[i].hi == 0.0 && t[i].lo == 0.0f : a != 1.0,
               "log at 1", i);
        expect(std::rint(t[i].hi * 0x1p42) == t[i].hi * 0x1p42, "log grid", i);
        expect(std::fabs((double)((long double)t[i].hi + t[i].lo + std::log((long double)inv))) <= 0x1p-64, "log value", i);
    }
}

void check_tables_2d()
{
    for (int N = 1; N <= LFMM_MAX_TERMS_2D; ++N) {
        lfmm::OpTables2d T;
        lfmm::build_op_tables_2d(N, T);
        lfmm::build_shift_tables_2d(T);
        expect(T.m2l.size() == (size_t)lfmm::kNumM2LDirs2d * N * N * 2, "2d m2l size", N);
        for (double v : T.m2l) expect(std::isfinite(v), "2d m2l finite", N);
        for (double v : T.m2m) expect(std::isfinite(v), "2d m2m finite", N);
        for (double v : T.l2l) expect(std::isfinite(v), "2d l2l finite", N);
        check_packed_2d(T);
    }
    check_log_2d();
}

void check_exact_files(const std::string& dir)
{
    const int widths[4] = {1, 2, 1, 3};
    for (int kind = 0; kind < 4; ++kind) {
        const int64_t n = 257;
        const int w = widths[kind];
        std::vector<double> v((size_t)(n * w)), back((size_t)(n * w), 0.0);
        for (int64_t i = 0; i < n * w; ++i) v[(size_t)i] = std::sin(0.7 * (double)i) * std::pow(10.0, (double)(i % 9) - 4);
        const std::string path = dir + "/" + lfmm_exact_filename(kind);
        expect(lfmm_write_exact(path.c_str(), kind, n, v.data()) == LFMM_OK, "write exact", kind);
        expect(lfmm_read_exact(path.c_str(), kind, n, back.data()) == n, "read exact count", kind);
        for (int64_t i = 0; i < n * w; ++i) expect(back[(size_t)i] == v[(size_t)i], "exact round trip", kind);
        // asking for more values than the file holds returns what is there
        std::vector<double> more((size_t)((n + 10) * w), 0.0);
        expect(lfmm_read_exact(path.c_str(), kind, n + 10, more.data()) == n, "short file", kind);
        double mx = -1.0, l2 = -1.0, rel = -1.0;
        expect(lfmm_error_stats(kind, n, v.data(), v.data(), &mx, &l2, &rel) == LFMM_OK, "error stats", kind);
        expect(mx == 0.0 && rel == 0.0, "error stats of equal data", kind);
        std::remove(path.c_str());
    }
    expect(lfmm_read_exact((dir + "/missing.txt").c_str(), 0, 4, nullptr) < 0, "missing file");
    expect(lfmm_write_exact(nullptr, 0, 1, nullptr) != LFMM_OK, "write null path");
    expect(lfmm_error_stats(7, 1, nullptr, nullptr, nullptr, nullptr, nullptr) != LFMM_OK, "stats bad kind");
}

// A buffer that cannot be had leaves the arena's next allocation where it was.
void check_arena()
{
    std::vector<char> mem(4096);
    lfmm::host::Arena A;
    A.chunks.push_back({mem.data(), mem.size()});
    expect(A.alloc(1000) == mem.data(), "arena first");
    expect(A.try_alloc((size_t)1 << 60) == nullptr, "arena too large");
    expect(A.try_alloc(1000) == mem.data() + 1024 && A.alloc(2048) == mem.data() + 2048, "arena goes on");
    expect(A.used == 4096 && A.peak == 4096, "arena use");
}

// Entry points given a null context fail with LFMM_ERR_INVALID before any
// device work.
void check_null_context()
{
    double buf[16] = {};
    lfmm_points3d pts{4, buf, 3, buf, 1};
    const int bad = LFMM_ERR_INVALID;
    expect(lfmm_fmm3d(nullptr, &pts, nullptr, 1e-8, 5, 3, 0, 0, 0, buf, buf, nullptr) == bad, "fmm3d null ctx");
    expect(lfmm_fmm2d(nullptr, &pts, nullptr, 1e-8, 5, 3, 0, 0, 0, buf, buf, nullptr) == bad, "fmm2d null ctx");
    expect(lfmm_fmm3d_vec(nullptr, &pts, nullptr, 1e-8, 5, 3, 0, 0, 0, buf, nullptr) == bad, "fmm3d_vec null ctx");
    expect(lfmm_direct3d(nullptr, &pts, nullptr, 0, 0u, buf, buf) == bad, "direct3d null ctx");
    expect(lfmm_direct2d(nullptr, &pts, nullptr, 0, 0u, buf, buf) == bad, "direct2d null ctx");
    expect(lfmm_direct3d_vec(nullptr, &pts, nullptr, 0, buf) == bad, "direct3d_vec null ctx");
    expect(lfmm_direct3d_noalloc(nullptr, &pts, nullptr, 0u, buf, buf) == bad, "direct3d_noalloc null ctx");
    expect(lfmm_set_stream(nullptr, nullptr) == bad, "set_stream null ctx");
    expect(lfmm_trim(nullptr) == bad, "trim null ctx");
    expect(lfmm_tree3d(nullptr, &pts, 3, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr) == bad, "tree3d");
    expect(lfmm_tree2d(nullptr, &pts, 3, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr) == bad, "tree2d");
    const int64_t off[2] = {0, 4};
    expect(lfmm_fmm3d_batch(nullptr, 1, off, buf, buf, 1e-8, 5, 3, 0, 0, 0u, 1, buf, buf, nullptr) == bad,
           "batch null ctx");
    expect(lfmm_set_order_model(nullptr, nullptr, 0.9, 1e-6, 16) == bad, "set_order_model null ctx");
    lfmm_destroy(nullptr);
    for (int s = -1; s <= 10; ++s) expect(lfmm_strerror(s) != nullptr, "strerror", s);
    expect(lfmm_version() != nullptr, "version");
}

}  // namespace

int main(int argc, char** argv)
{
    const std::string dir = argc > 1 ? argv[1] : ".";
    check_wigner();
    check_tables_3d();
    check_packed_3d();
    check_tables_2d();
    check_exact_files(dir);
    check_arena();
    check_null_context();
    if (failures) {
        std::printf("host_check: %d failures\n", failures);
        return 1;
    }
    std::printf("host_check ok\n");
    return 0;
}
