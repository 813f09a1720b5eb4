// ops2d.hip -- FP64 operator kernels of the 2D (complex-series) FMM, gfx950.
//
//   k_p2m2d    P2M, thread per leaf                    (reference Multipole, src/cpu/multipole.cpp:22-36)
//   k_m2m2d    M2M, thread per (parent, coefficient)    (M2M :38-53, Upward :155-177)
//   k_m2l2d    M2L of all levels, lane per target       (M2L :66-84, Downward :179-231)
//   k_m2l2d32  the same with FP32 per-direction sums added in FP64
//   k_l2l2d    L2L, thread per (parent, coefficient)    (L2L :86-97)
//   k_leaf2d   L2P + P2P over the 3x3 neighbourhood, thread per particle,
//              results scattered to input order       (ComputePotentials / ComputeForces :233-449)
//
// Expansions are normalised per level (tables2d.cpp), so every operator is a
// fixed complex matrix per integer box offset or child class, factored into one
// real matrix between complex diagonals (pack_2d).
#include "device_common.h"
#include "lfmm_internal.h"
#include "m2l_children.h"
#include "ops2d.h"
#include "rowbc.h"


namespace lfmm {

__device__ inline double2 cmul2(double2 a, double2 b)
{
    return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}

__global__ void __launch_bounds__(256) k_p2m2d(P2M2dArgs a)
{
    const int leaf = blockIdx.x * blockDim.x + threadIdx.x;
    if (leaf >= a.nleaf) return;
    const uint64_t key = a.leaf_key[leaf];
    const double scale = a.geom[3];
    const double cx = box_centre(compact2(key >> 1), a.level, scale, a.geom[0]);
    const double cy = box_centre(compact2(key), a.level, scale, a.geom[1]);
    const double ih = ldexp(1.0, a.level) / scale;
    double2 acc[kMaxTerms2d];
#pragma unroll
    for (int k = 0; k < kMaxTerms2d; ++k) acc[k] = make_double2(0.0, 0.0);
    const int b = a.leaf_begin[leaf], e = a.leaf_begin[leaf + 1];
    for (int p = b; p < e; ++p) {
        const double4 s = a.src[p];
        const double ux = (s.x - cx) * ih, uy = (s.y - cy) * ih, q = s.w;
        double wx = q * ux, wy = q * uy;  // q u^k
        acc[0].x += q;
#pragma unroll
        for (int k = 1; k < kMaxTerms2d; ++k) {
            if (k < a.N) {
                acc[k].x += wx;
                acc[k].y += wy;
                const double t = wx * ux - wy * uy;
                wy = wx * uy + wy * ux;
                wx = t;
            }
        }
    }
    double2* out = a.outer + (int64_t)leaf * a.N;
    out[0] = acc[0];
#pragma unroll
    for (int k = 1; k < kMaxTerms2d; ++k)
        if (k < a.N) out[k] = make_double2(-acc[k].x / k, -acc[k].y / k);
}

// exponent of i in a child's offset: i^r (1 + i)/2
__device__ inline int turn_of(int c) { return c == 3 ? 0 : c == 1 ? 1 : c == 0 ? 2 : 3; }

constexpr int kPairs2d = 256;  // (parent, coefficient) threads of a workgroup

// The four sums y_m = sum over the children of i^(r m) at_s e^-s go to LDS once
// per source coefficient; an output coefficient then takes one real product
// per source, where the children's complex matrices took 16 products (1M
// particles of 21 terms, 6 levels: 139 -> 60 us).
__global__ void __launch_bounds__(kPairs2d) k_m2m2d(M2M2dArgs a, Tables2d T)
{
    __shared__ double2 y[4 * kPairs2d];
    const int N = a.N, per = kPairs2d / N;
    const int p = threadIdx.x / N, j = threadIdx.x - p * N;
    const int P = blockIdx.x * per + p;
    const bool live = p < per && P < a.num_parents;
    if (live) {
        double2 m[4];
        for (int k = 0; k < 4; ++k) m[k] = make_double2(0.0, 0.0);
        for (int ch = a.child_begin[P]; ch < a.child_begin[P + 1]; ++ch) {
            const int r = turn_of((int)(a.child_keys[ch] & 3u));
            double2 x = a.src[(int64_t)ch * N + j];
            for (int k = 0; k < 4; ++k) {  // x i^(r k)
                m[k].x += x.x;
                m[k].y += x.y;
                for (int t = 0; t < r; ++t) x = make_double2(-x.y, x.x);
            }
        }
        const double2 e = T.up[j];
        for (int k = 0; k < 4; ++k) y[(p * 4 + k) * N + j] = cmul2(m[k], e);
    }
    __syncthreads();
    if (!live) return;
    double2 v = make_double2(0.0, 0.0);
    const double2* q = y + p * 4 * N;
    for (int s = 0; s <= j; ++s) {
        const double2 x = q[((j - s) & 3) * N + s];
        const double c = T.m2m[j * N + s];
        v.x = fma(c, x.x, v.x);
        v.y = fma(c, x.y, v.y);
    }
    a.dst[(int64_t)P * N + j] = cmul2(v, T.down[j]);
}

// The transpose: the parent's coefficients by distance mod 4, one real product
// each, and the children take the four sums with weights i^(r m).
__global__ void __launch_bounds__(kPairs2d) k_l2l2d(L2L2dArgs a, Tables2d T)
{
    __shared__ double2 xs[kPairs2d];
    const int N = a.N, per = kPairs2d / N;
    const int p = threadIdx.x / N, k = threadIdx.x - p * N;
    const int P = blockIdx.x * per + p;
    const bool live = p < per && P < a.num_parents;
    if (live) xs[threadIdx.x] = cmul2(a.src[(int64_t)P * N + k], T.down[k]);
    __syncthreads();
    if (!live) return;
    double2 z[4];
    for (int m = 0; m < 4; ++m) z[m] = make_double2(0.0, 0.0);
    for (int j = k; j < N; j += 4)
#pragma unroll
        for (int m = 0; m < 4; ++m)
            if (j + m < N) {
                const double c = T.l2l[k * N + j + m];
                const double2 x = xs[p * N + j + m];
                z[m].x = fma(c, x.x, z[m].x);
                z[m].y = fma(c, x.y, z[m].y);
            }
    const double2 e = T.up[k];
    for (int ch = a.child_begin[P]; ch < a.child_begin[P + 1]; ++ch) {
        const int r = turn_of((int)(a.child_keys[ch] & 3u));
        // i^(r m): 1; i^r; (-1)^r; i^-r
        const double s2 = (r & 1) ? -1.0 : 1.0;
        double2 v = make_double2(z[0].x + s2 * z[2].x, z[0].y + s2 * z[2].y);
        double2 w = make_double2(z[1].x + s2 * z[3].x, z[1].y + s2 * z[3].y);
        for (int t = 0; t < r; ++t) w = make_double2(-w.y, w.x);
        v = cmul2(make_double2(v.x + w.x, v.y + w.y), e);
        double2* o = a.dst + (int64_t)ch * N + k;
        *o = make_double2(o->x + v.x, o->y + v.y);
    }
}

// M2L into the class-c children of 64 consecutive parents, one lane per target,
// one wave per (class, parent tile, row block): every level in one launch,
// since the levels' M2L are independent and a coarse level, 27 dependent
// gathers for each of a few waves, takes as long as a full one.
// Bound by FP64 issue: a source coefficient is scaled once (5 operations), then
// each row takes 2 products with a real entry that is the same for every
// direction and target: the wave keeps the entries of its rows in registers, 16
// to each, and broadcasts them by row_newbcast.  (As complex entries per
// direction, read from LDS, it was 4 products and a 16-byte LDS read each, and a
// launch per level: 1M particles of 21 terms, 0.82 -> 0.22 ms.)  Two row blocks from 12 terms
// on and three from 25: more waves, and their accumulators and entries fit beside
// the source.
template <int N>
__global__ void __launch_bounds__(64) k_m2l2d(M2L2dLevels A, Tables2d T)
{
    constexpr int NB = m2l2d_blocks(N), NP = m2l2d_pairs(N), REGS = m2l2d_regs(N);
    const int blk = blockIdx.x;
    int li = 0;
    while (blk >= A.first[li + 1]) ++li;
    const M2L2dArgs& a = A.level[li];
    const int g = xcd_local_block(blk - A.first[li], A.first[li + 1] - A.first[li]);
    const int b = g % NB, c = g / NB & 3, tile = g / (4 * NB);
    const int lane = threadIdx.x, l16 = lane & 15;
    const int P = tile * 64 + lane;
    int t = -1;
    if (P < a.num_parents)
        for (int i = a.child_begin[P]; i < a.child_begin[P + 1]; ++i)
            if ((int)(a.child_keys[i] & 3u) == c) t = i;
    const uint64_t key = t < 0 ? 0 : a.child_keys[t];
    const int tx = (int)compact2(key >> 1), ty = (int)compact2(key);
    const int side = 1 << a.level;
    const auto dirs = m64_scalar((const int*)T.class_dirs) + c * kDirsPerClass2d;
    const auto vec = m64_scalar((const m64_i2*)T.dir_vec);
    const auto lg = m64_scalar((const m64_v2*)T.log);
    auto source_of = [&](int k) -> int {
        const m64_i2 d = vec[dirs[k]];
        const int sx = tx + d.x, sy = ty + d.y;
        if (t < 0 || sx < 0 || sy < 0 || sx >= side || sy >= side) return -1;
        return find_box(morton2(sx, sy), a.lut, a.child_keys, a.size);
    };
    double ent[REGS];
#pragma unroll
    for (int i = 0; i < REGS; ++i) ent[i] = T.m2l[(b * REGS + i) * 16 + l16];
    double2 acc[2 * NP];
#pragma unroll
    for (int i = 0; i < 2 * NP; ++i) acc[i] = make_double2(0.0, 0.0);
    int s = source_of(0);
    for (int k = 0; k < kDirsPerClass2d; ++k) {
        const int d = dirs[k];
        const bool any = __ballot(s >= 0) != 0ull;
        const double2* xs = s < 0 ? T.zero : a.src + (int64_t)s * N;
        if (k + 1 < kDirsPerClass2d) s = source_of(k + 1);
        if (!any) continue;
        double2 v[N];
#pragma unroll
        for (int j = 0; j < N; ++j) v[j] = xs[j];
        constexpr int W = (N + 15) / 16;
        double wr[W], wi[W];
#pragma unroll
        for (int i = 0; i < W; ++i) {
            wr[i] = T.src[d * 64 + 16 * i + l16];
            wi[i] = T.src[d * 64 + 32 + 16 * i + l16];
        }
        const double orr = T.out[(d * NB + b) * 32 + l16], oi = T.out[(d * NB + b) * 32 + 16 + l16];
        if (b == 0) {  // at_0 (log h + conj(log(-d)))
            const m64_v2 q = lg[d];
            const double lr = q.x + a.log_h;
            acc[0].x = fma(v[0].x, lr, fma(-v[0].y, q.y, acc[0].x));
            acc[0].y = fma(v[0].x, q.y, fma(v[0].y, lr, acc[0].y));
        }
        sfor2<1, N>([&](auto J) {
            constexpr int j = decltype(J)::value;
            const double2 x = v[j];
            const double w = bc<j % 16>(wr[j / 16]);
            v[j].x = x.x * w;
            v[j].y = x.y * w;
            fnmac_bc<j % 16>(v[j].x, wi[j / 16], x.y);
            fmac_bc<j % 16>(v[j].y, wi[j / 16], x.x);
        });
        sfor2<0, NP>([&](auto R) {
            constexpr int r = decltype(R)::value;
            double re[2] = {0.0, 0.0}, im[2] = {0.0, 0.0};
            sfor2<0, N>([&](auto J) {
                constexpr int j = decltype(J)::value, at = r * 2 * N + 2 * j;
                tr4_bc<at % 16>(re[0], im[0], re[1], im[1], ent[at / 16], v[j].x, v[j].y);
            });
            sfor2<0, 2>([&](auto Q) {
                constexpr int q = decltype(Q)::value, i = 2 * r + q;
                fmac_bc<i>(acc[i].x, orr, re[q]);
                fmac_bc<i>(acc[i].y, orr, im[q]);
                fnmac_bc<i>(acc[i].x, oi, im[q]);
                fmac_bc<i>(acc[i].y, oi, re[q]);
            });
        });
    }
    if (t < 0) return;
    double2* out = a.dst + (int64_t)t * N + b * 2 * NP;
#pragma unroll
    for (int i = 0; i < 2 * NP; ++i)
        if (b * 2 * NP + i < N) out[i] = acc[i];
}

// M2L of one level with each direction's sum over the source coefficients
// formed in FP32 (FP32 operator, sources rounded on load) and added to the FP64
// accumulator; the level term (coefficient 0) stays FP64.  One lane per target
// of class c, one workgroup per (class, 256 parents, block of LB output
// coefficients): the rows it needs of the class's 27 operators are staged in
// LDS once and read as broadcasts.
constexpr int m2l2d_lb(int N) { return (N + 3) / 4; }

template <int N>
__global__ void __launch_bounds__(256) k_m2l2d32(M2L2dArgs a, Tables2d T)
{
    constexpr int LB = m2l2d_lb(N), NB = (N + LB - 1) / LB, ROWS = LB * N;
    __shared__ float2 mop[kDirsPerClass2d * ROWS];
    const int c = blockIdx.x & 3;
    const int rest = (int)(blockIdx.x >> 2);
    const int l0 = (rest % NB) * LB;
    for (int i = threadIdx.x; i < kDirsPerClass2d * ROWS; i += 256) {
        const int k = i / ROWS, r = (i % ROWS) / N, j = i % N;
        const int d = T.class_dirs[c * kDirsPerClass2d + k];
        const int l = l0 + r;
        mop[i] = l < N ? T.m2l32[((int64_t)d * N + l) * N + j] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    const int P = (rest / NB) * 256 + (int)threadIdx.x;
    int t = -1;
    if (P < a.num_parents)
        for (int i = a.child_begin[P]; i < a.child_begin[P + 1]; ++i)
            if ((int)(a.child_keys[i] & 3u) == c) t = i;
    if (t < 0) return;  // no barriers below: lanes may leave
    const uint64_t key = a.child_keys[t];
    const int tx = (int)compact2(key >> 1), ty = (int)compact2(key);
    const int side = 1 << a.level;
    double2 acc[LB];
#pragma unroll
    for (int r = 0; r < LB; ++r) acc[r] = make_double2(0.0, 0.0);
    for (int k = 0; k < kDirsPerClass2d; ++k) {
        const int d = T.class_dirs[c * kDirsPerClass2d + k];
        const int sx = tx + T.dir_vec[2 * d], sy = ty + T.dir_vec[2 * d + 1];
        if (sx < 0 || sy < 0 || sx >= side || sy >= side) continue;
        const int s = find_box(morton2(sx, sy), a.lut, a.child_keys, a.size);
        if (s < 0) continue;
        const double2* xs = a.src + (int64_t)s * N;
        double2 x[N];
#pragma unroll
        for (int j = 0; j < N; ++j) x[j] = xs[j];
        if (l0 == 0) {  // level term at_0 log h of the normalised M2L
            acc[0].x = fma(x[0].x, a.log_h, acc[0].x);
            acc[0].y = fma(x[0].y, a.log_h, acc[0].y);
        }
        const float2* m = mop + k * ROWS;
        float xr[N], xi[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            xr[j] = (float)x[j].x;
            xi[j] = (float)x[j].y;
        }
#pragma unroll
        for (int r = 0; r < LB; ++r) {
            float ax = 0.f, ay = 0.f;
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const float2 mv = m[r * N + j];
                ax = fmaf(mv.x, xr[j], fmaf(-mv.y, xi[j], ax));
                ay = fmaf(mv.x, xi[j], fmaf(mv.y, xr[j], ay));
            }
            acc[r].x += (double)ax;
            acc[r].y += (double)ay;
        }
    }
    double2* out = a.dst + (int64_t)t * N;
#pragma unroll
    for (int r = 0; r < LB; ++r)
        if (l0 + r < N) out[l0 + r] = acc[r];
}

// log(x) of a normal x > 0 by a table (P.T.P. Tang, ACM TOMS 16 (1990) 378;
// pack_log_2d): x = 2^e m, r = m/c - 1 exact but for its last bit, e log 2 + log c
// exact in its first part, |r| <= 2^-7 and a series to r^7 (the next term is 2^-59
// of the first).  Within 0.52 ulp everywhere, next to 1 included (1e7 arguments
// against 113 bits), as the library function, for about half its operations.
__device__ __forceinline__ double log_tab(double x, const LogEntry2d* tab)
{
    const int d = __double2hiint(x) - kLog2dFirst, e = d >> 20;
    const double m = __hiloint2double(__double2hiint(x) - (e << 20), __double2loint(x));
    const LogEntry2d t = tab[(d >> 13) & (kLog2dEntries - 1)];
    const double r = fma(m, (double)t.inv, -1.0);
    double p = fma(r, 1.0 / 7.0, -1.0 / 6.0);
    p = fma(r, p, 0.2);
    p = fma(r, p, -0.25);
    p = fma(r, p, 1.0 / 3.0);
    p = fma(r, p, -0.5);
    // log 2 in two parts: 42 bits, so that its product with e is exact, and the rest
    const double h = fma((double)e, 0x1.62e42fefa38p-1, t.hi), w = h + r;
    const double lo = fma((double)e, 0x1.ef35793c7673p-45, ((h - w) + r) + (double)t.lo);
    return w + fma(r * r, p, lo);
}

// Pair term of the reference 2D kernels (src/common/simple_math.h:119-128):
// q log(max(|dz|, 1e-4)) and q conj(dz) / max(|dz|^2, 1e-8), self pair included.
// Bound by vector issue.  A lane walks the near ranges of its leaf as one list
// (leaves of a wave would wait for each other at every range), one source
// ahead; past its end it reads a zero charge in its own leaf (at the origin, say,
// the squared distance could overflow, and 0 times its logarithm is no zero).  1M
// particles, 16 per leaf, 150M pairs: 0.76 ms with the library's log and division and
// a loop per neighbour, 0.32 so (0.25 with a logarithm that cancels next to 1 and an
// uncorrected quotient).  WIDE: distances whose square overflows, within a leaf too: a
// lane past its list adds nothing.
typedef double pt2d __attribute__((ext_vector_type(4)));
typedef const pt2d __attribute__((address_space(1)))* pt2d_ptr;

template <bool EXCLUDE, bool WIDE>
__global__ void __launch_bounds__(256) k_leaf2d(Leaf2dArgs a, Tables2d T)
{
    __shared__ LogEntry2d tab[kLog2dEntries];
    if (threadIdx.x < kLog2dEntries) tab[threadIdx.x] = T.pair_log[threadIdx.x];
    __syncthreads();
    const int64_t i = xcd_local_block(blockIdx.x, gridDim.x) * (int64_t)blockDim.x + threadIdx.x;
    const int64_t s = min(i, a.n - 1);
    const int64_t o = a.perm[s];
    const bool live = i < a.n && o < a.n_out;
    const int leaf = a.leaf_of[s];
    const double4 t = a.src[s];
    double ph = 0.0, fx = 0.0, fy = 0.0;
    const int all = live ? a.near_total[leaf] : 0;
    int todo = all, nsrc = all;
    for (int off = 32; off > 0; off >>= 1) nsrc = max(nsrc, __shfl_xor(nsrc, off));
    nsrc = __builtin_amdgcn_readfirstlane(nsrc);
    const pt2d_ptr src = (pt2d_ptr)(uintptr_t)a.src, zero = (pt2d_ptr)(uintptr_t)(a.pad + leaf);
    const int2* nr = a.nbr + (int64_t)leaf * 9;
    const int nrc = a.near_runs[leaf];
    pt2d_ptr p = zero, end = zero;
    int64_t step = sizeof(pt2d);
    int k = 0;
    int2 rn = nr[0];
    bool self = false;
    auto next = [&]() -> pt2d {
        if (p == end) {
            if (todo > 0) {
                p = src + rn.x;
                end = src + rn.y;
                todo -= rn.y - rn.x;
                rn = nr[min(++k, nrc - 1)];
            } else {  // past its list
                p = zero;
                end = src;  // never reached: the step is 0
                step = 0;
            }
        }
        const pt2d q = *p;
        if constexpr (EXCLUDE) self = p == src + s;
        p = (pt2d_ptr)((uintptr_t)p + step);
        return q;
    };
    pt2d q = next();
    for (int it = 0; it < nsrc; ++it) {
        const double dx = t.x - q.x, dy = t.y - q.y;
        const double w = EXCLUDE && self ? 0.0 : q.w;
        q = next();
        const double nz = fmax(fma(dx, dx, dy * dy), 1.e-8);
        if constexpr (WIDE) {
            if (it >= all) continue;
            const double qi = w / nz;
            ph += w * log(nz);
            fx = fma(qi, dx, fx);
            fy = fma(-qi, dy, fy);
        } else {
            // w / nz: v_rcp_f64 (relative error 4.7e-8) and one Newton step, then
            // the quotient's own residual: correctly rounded (8.6e9 quotients
            // compared with the division; w y alone: a quarter were not); the
            // fixup keeps infinite charges
            double y = __builtin_amdgcn_rcp(nz);
            y = fma(y, fma(-nz, y, 1.0), y);
            const double q0 = w * y;
            const double qi = __builtin_amdgcn_div_fixup(fma(fma(-nz, q0, w), y, q0), nz, w);
            ph = fma(w, log_tab(nz, tab), ph);
            fx = fma(qi, dx, fx);
            fy = fma(-qi, dy, fy);
        }
    }
    if (!live) return;
    ph *= 0.5;
    if (a.local) {  // L2P by Horner: P(u) = sum bt_k u^k, P'(u)
        const uint64_t key = a.leaf_key[leaf];
        const double scale = a.geom[3];
        const double ih = ldexp(1.0, a.level) / scale;
        const double ux = (t.x - box_centre(compact2(key >> 1), a.level, scale, a.geom[0])) * ih;
        const double uy = (t.y - box_centre(compact2(key), a.level, scale, a.geom[1])) * ih;
        const double2* b = a.local + (int64_t)leaf * a.N;
        double2 v = b[a.N - 1], d = make_double2(0.0, 0.0);
        for (int j = a.N - 2; j >= 0; --j) {
            d = make_double2(d.x * ux - d.y * uy + v.x, d.x * uy + d.y * ux + v.y);
            const double2 bj = b[j];
            v = make_double2(v.x * ux - v.y * uy + bj.x, v.x * uy + v.y * ux + bj.y);
        }
        ph += v.x;
        fx += d.x * ih;
        fy += d.y * ih;
    }
    if (a.pot) a.pot[o] = ph;
    if (a.field) {
        a.field[2 * o] = fx;
        a.field[2 * o + 1] = fy;
    }
}

static inline unsigned nblk(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

hipError_t launch_p2m2d(const P2M2dArgs& a, hipStream_t st)
{
    if (a.N < 1 || a.N > kMaxTerms2d) return hipErrorInvalidValue;
    if (a.nleaf > 0) hipLaunchKernelGGL(k_p2m2d, dim3(nblk(a.nleaf, 256)), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_m2m2d(const M2M2dArgs& a, const Tables2d& T, hipStream_t st)
{
    if (a.N < 1 || a.N > kMaxTerms2d) return hipErrorInvalidValue;
    if (a.num_parents > 0)
        hipLaunchKernelGGL(k_m2m2d, dim3(nblk(a.num_parents, kPairs2d / a.N)), dim3(kPairs2d), 0, st, a, T);
    return hipGetLastError();
}

hipError_t launch_l2l2d(const L2L2dArgs& a, const Tables2d& T, hipStream_t st)
{
    if (a.N < 1 || a.N > kMaxTerms2d) return hipErrorInvalidValue;
    if (a.num_parents > 0)
        hipLaunchKernelGGL(k_l2l2d, dim3(nblk(a.num_parents, kPairs2d / a.N)), dim3(kPairs2d), 0, st, a, T);
    return hipGetLastError();
}

template <int N>
hipError_t m2l2d_n(M2L2dLevels& a, const Tables2d& T, hipStream_t st)
{
    a.first[0] = 0;
    for (int i = 0; i < a.count; ++i)
        a.first[i + 1] = a.first[i] + 4 * m2l2d_blocks(N) * (int)nblk(a.level[i].num_parents, 64);
    if (a.first[a.count] > 0) hipLaunchKernelGGL(k_m2l2d<N>, dim3((unsigned)a.first[a.count]), dim3(64), 0, st, a, T);
    return hipGetLastError();
}

template <int N>
hipError_t m2l2d_f32_n(const M2L2dArgs& a, const Tables2d& T, hipStream_t st)
{
    constexpr int NB = (N + m2l2d_lb(N) - 1) / m2l2d_lb(N);
    const dim3 grid((unsigned)(4 * NB * ((a.num_parents + 255) / 256)));
    if (a.num_parents > 0) hipLaunchKernelGGL(k_m2l2d32<N>, grid, dim3(256), 0, st, a, T);
    return hipGetLastError();
}

#define LFMM_TERMS2D(X)                                                                                            \
    X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) X(17) X(18) X(19) X(20) \
        X(21) X(22) X(23) X(24) X(25) X(26) X(27) X(28) X(29) X(30)

hipError_t launch_m2l2d(int N, M2L2dLevels& a, const Tables2d& T, hipStream_t st)
{
    if (a.count < 0 || a.count > kM2l2dLevels) return hipErrorInvalidValue;
    switch (N) {
#define X(n) case n: return m2l2d_n<n>(a, T, st);
        LFMM_TERMS2D(X)
#undef X
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_m2l2d_f32(int N, const M2L2dArgs& a, const Tables2d& T, hipStream_t st)
{
    switch (N) {
#define X(n) case n: return m2l2d_f32_n<n>(a, T, st);
        LFMM_TERMS2D(X)
#undef X
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_leaf2d(const Leaf2dArgs& a, const Tables2d& T, hipStream_t st)
{
    if (a.n <= 0) return hipSuccess;
    const dim3 grid(nblk(a.n, 256)), block(256);
    if (a.wide) {
        if (a.exclude_self) hipLaunchKernelGGL((k_leaf2d<true, true>), grid, block, 0, st, a, T);
        else hipLaunchKernelGGL((k_leaf2d<false, true>), grid, block, 0, st, a, T);
    } else {
        if (a.exclude_self) hipLaunchKernelGGL((k_leaf2d<true, false>), grid, block, 0, st, a, T);
        else hipLaunchKernelGGL((k_leaf2d<false, false>), grid, block, 0, st, a, T);
    }
    return hipGetLastError();
}

}  // namespace lfmm
