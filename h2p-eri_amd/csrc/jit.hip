// On-the-fly B and D blocks (a BD_JIT = 1 handle) on the GPU.
//
// The reference's BD_JIT mode (src/H2ERI_matvec.c:411-568 intermediate
// products, :761-879 near field, :911 and :928 the switch) stores U only and
// evaluates every coupling block B_ij and near-field block D_ij from the
// shell pairs at each matvec, through H2ERI_calc_ERI_pairs_to_mat
// (src/CMS.c:387-451).  Here the blocks' products with their inputs are
// evaluated on the device without ever forming an integral:
//
//  * Sides.  A list of shell pairs is one side of a node: its full leaf rows,
//    or its skeleton rows (J_row).  Side rules of the reference's three
//    coupling cases (src/H2ERI_matvec.c:455-545): node n is on its skeleton
//    side against an admissible partner m when level(n) >= level(m), else on
//    its full side (n is then a leaf).  Full rows are x-indexed and receive
//    the near field (the leaf itself and its inadmissible partners, both
//    orientations) and the coupling products of case (2)/(3) leaves;
//    skeleton rows are y1 of the node.  Every output row has one writer: a
//    block (n, m) is evaluated once from each side, against the reference's
//    once with a bi-GEMV, in exchange for no atomics and a fixed summation
//    order (bit-reproducible results).
//  * The product of a block with its input in a Hermite Gaussian basis.  In
//    McMurchie-Davidson form (Helgaker, Jorgensen & Olsen, Molecular
//    Electronic-Structure Theory, eqs. 9.5.x and 9.9.33)
//    (ab|cd) = sum_{ij} 2 pi^{5/2} / (p q sqrt(p+q)) K_i K_j
//              sum_{tuv} E^{ab}_{tuv} sum_{tau nu phi} (-1)^{tau+nu+phi}
//              E^{cd}_{tau nu phi} R_{t+tau, u+nu, v+phi}(alpha, PQ),
//    and sum_cd (ab|cd) x_cd separates: the input is first contracted with
//    the ket's E into a Hermite density H_j per primitive (once per side,
//    not once per bra), each bra primitive i collects the Hermite potential
//    V_i = sum_j R H_j / sqrt(p+q), and the rows are E^{ab} V_i (the density
//    form of the J build: Ahmadi & Almlof, Chem. Phys. Lett. 246, 364 (1995);
//    White & Head-Gordon, J. Chem. Phys. 104, 2620 (1996)).  A primitive
//    quartet costs its Boys values, the R recursion and one product of
//    nherm(L_ab) x nherm(L_cd) terms; no Cartesian component is formed.
//  * Centres.  The primitives of a side with equal exponent sum, centre and
//    total order are one Hermite centre (contracted s shells of one atom
//    share their exponents: 289 s-s primitives of a C-C pair in cc-pVDZ are
//    81 centres).
//  * R^{(n)}_{000} = (-2 alpha)^n F_n(alpha |PQ|^2), R^{(n)}_{t+1,u,v} =
//    t R^{(n+1)}_{t-1,u,v} + X_PQ R^{(n+1)}_{t,u,v}, in registers, with the
//    Boys function from a table in LDS.  Shells up to d (cc-pVDZ); the
//    primitive pairs, centres and conventions are the host engine's (first
//    shell of a pair = N, row index n * nbf(M) + m, lexicographic
//    Cartesians).
//  * Sweeps: the up sweep (y0 = U^T x, children first) and the down sweep
//    (parents first) are one launch per tree level over the nodes of that
//    level, with U in FP64.
//
// Sequence of one matvec: zero y1 and the row outputs, up sweep, Hermite
// densities of every side (they need y0), potentials, rows, down sweep (it
// needs y1), y = down-sweep rows + block rows.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstring>
#include <map>
#include <numeric>
#include <thread>
#include <unordered_map>
#include <utility>
#include <vector>

#include "h2eri_internal.h"

namespace h2e {

static const int JIT_LMAX = 2;      // shell angular momentum (d)
static const int JIT_OMAX = 4;      // order of a pair (la + lb)
static const int JIT_NORD = JIT_OMAX + 1;
static const int JIT_NLT = 2 * JIT_OMAX + 1;   // total orders of a quartet
static const int JIT_WPG = 4;       // waves (tasks) per workgroup of the potential kernels

// Boys table: T in [0, 40) in 640 intervals of 1/16; per interval eight
// doubles, the seven coefficients of F_m in powers of (T0 - T), T0 the
// interval's midpoint, and exp(-T0).  40,960 bytes per order, four tables to
// the 160 KB of LDS of a CU.
static const int JIT_BGRID = 640;
static const int JIT_BROW = 8;
static const double JIT_BTMAX = 40.0;

// One wave's work: the potential of n centres (from global centre c0, order
// la) against the centres of order lb in segments [s0, s1), bw = 2^lbw lanes
// per centre group (64 / bw slices share the segments' centres); partial
// potentials nherm(la) x bw into part[poff].
struct JitTask {
    int cls;        // la * JIT_NORD + lb
    int c0, n, lbw;
    int s0, s1;
    long long poff;
};
// Centres [c0, c0 + n) of order la: the sum of its tasks' partials, in order.
struct JitChunk {
    int la, c0, n, lbw;
    int t0, t1;     // in ctask
};

// Everything the kernels read or write; the pointers are device or, in the
// emulator, host arrays.
struct JitView {
    int N, ncen, nent;
    const int *pinfo;     // per shell pair: la, lb, primitive pairs, first primitive
    const double *pgeo;   // per shell pair: A (3), B (3)
    const double *prim;   // per primitive pair: p, P (3), K, 1/(2p)
    const double *boys;   // Boys tables by total order
    const int *kl_pair, *kl_moff;     // per side entry: shell pair, its row map
    const int *kmap;                  // index per row (< N: x / y, else y0 / y1; -1: not used)
    const int *e_c0, *ecen;           // per entry: first of its primitives' centres in ecen
    const int *cptr, *cent, *cprim;   // per centre: its contributions (entry, primitive)
    const double *cgeo;               // per centre: p, P (3)
    int coff[JIT_NORD + 1];           // first centre of each order
    long long hoff[JIT_NORD];         // its first Hermite coefficient
    double *H, *V;                    // Hermite densities and potentials by centre
    const JitTask *tasks;
    const int *segs;                  // (first, end) centre per segment
    const JitChunk *chunks;
    const long long *cpoff;           // per chunk and task: its partials in part
    double *part;
    const int *oent;                  // entries with output rows, by class
    const double *X, *Y0;             // inputs: index < N in X, else Y0[index - N]
    double *YJ, *Y1;                  // outputs: index < N in YJ, else Y1[index - N]
};

__host__ __device__ constexpr int jit_ncart(int L) { return (L + 1) * (L + 2) / 2; }
__host__ __device__ constexpr int jit_nherm(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
// index of the Hermite triple (t, u, v) among all triples of total order
// <= t+u+v, lexicographic within an order
__host__ __device__ constexpr int jit_herm(int t, int u, int v) {
    const int k = t + u + v, a = k - t;
    return k * (k + 1) * (k + 2) / 6 + a * (a + 1) / 2 + v;
}
// exponent in direction dir of the k-th lexicographic Cartesian component of order L
__host__ __device__ constexpr int jit_cexp(int L, int k, int dir) {
    int a = 0;
    while ((a + 1) * (a + 2) / 2 <= k) a++;
    const int lx = L - a, ly = a - (k - a * (a + 1) / 2);
    return dir == 0 ? lx : (dir == 1 ? ly : L - lx - ly);
}
// Components of the Hermite triple of index h (inverse of jit_herm).
__host__ __device__ constexpr int jit_hcomp(int h, int which) {
    for (int k = 0; k <= 8; k++)
        for (int t = k; t >= 0; t--)
            for (int u = k - t; u >= 0; u--)
                if (jit_herm(t, u, k - t - u) == h) return which == 0 ? t : (which == 1 ? u : k - t - u);
    return 0;
}
template <int H1, int H2>
struct JitSum {   // index of the triple sum and the sign of the ket triple
    static constexpr int t1 = jit_hcomp(H1, 0), u1 = jit_hcomp(H1, 1), w1 = jit_hcomp(H1, 2);
    static constexpr int t2 = jit_hcomp(H2, 0), u2 = jit_hcomp(H2, 1), w2 = jit_hcomp(H2, 2);
    static constexpr int idx = jit_herm(t1 + t2, u1 + u2, w1 + w2);
    static constexpr bool neg = ((t2 + u2 + w2) & 1) != 0;
};

// 1 / sqrt(x), x > 0.  On the device one third-order step from v_rsq_f64
// (good to 2^-23): with e = 1 - x y^2, y (1 + e/2 + 3 e^2 / 8) is off by
// e^3 (2^-66) besides its rounding.
__host__ __device__ inline double jit_rsqrt(double x) {
#ifdef __HIP_DEVICE_COMPILE__
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
#else
    return 1.0 / sqrt(x);
#endif
}

// Position of coefficient pair k (0..3) of interval gi in its table: the
// pairs of a row are permuted by the row number, so that lanes at different
// rows read different LDS banks (rows are 16 of the 64 banks wide; unpermuted,
// a pair of every row would sit in the same 16 banks).
__host__ __device__ inline int jit_bpos(int gi, int k) { return gi * JIT_BROW + ((2 * k) ^ (((gi >> 2) & 3) * 2)); }

// F_0..F_M at T into F: the table's polynomial for F_M and downward
// recursion F_{m-1} = (2T F_m + e^-T) / (2m - 1) below T = 40; above, F_0 =
// sqrt(pi/T)/2 (erfc(sqrt 40) is 4e-19) and upward recursion.  There e^-T is
// 3e-10 of F_8 at T = 40 and 4e-19 of it at 64, and below an ulp of F_0 and
// F_1 throughout.
template <int M>
__host__ __device__ inline void jit_boys(double T, const double *bt, double *F) {
    if (T < JIT_BTMAX) {
        const int gi = (int)(T * 16.0);
        const double d = fma((double)gi, 0.0625, 0.03125) - T;
        struct D2 { double x, y; };
        const D2 a = *reinterpret_cast<const D2 *>(bt + jit_bpos(gi, 0)), b = *reinterpret_cast<const D2 *>(bt + jit_bpos(gi, 1));
        const D2 c = *reinterpret_cast<const D2 *>(bt + jit_bpos(gi, 2)), e = *reinterpret_cast<const D2 *>(bt + jit_bpos(gi, 3));
        F[M] = fma(fma(fma(fma(fma(fma(e.x, d, c.y), d, c.x), d, b.y), d, b.x), d, a.y), d, a.x);
        if constexpr (M > 0) {
            // e^-T = e^-T0 e^d, |d| <= 1/32: the omitted d^8/8! is 2e-17
            const double ed = fma(fma(fma(fma(fma(fma(fma(d, 1.0 / 5040, 1.0 / 720), d, 1.0 / 120), d, 1.0 / 24), d,
                                          1.0 / 6), d, 0.5), d, 1.0), d, 1.0);
            const double eT = e.y * ed, T2 = 2.0 * T;
#pragma unroll
            for (int m = M; m > 0; m--) F[m - 1] = fma(T2, F[m], eT) * (1.0 / (2 * m - 1));
        }
    } else {
        const double r = jit_rsqrt(T);
        F[0] = 0.88622692545275801365 * r;   // sqrt(pi) / 2
        if constexpr (M > 0) {
            const double i2T = 0.5 * r * r;
            double eT = 0.0;
            if constexpr (M > 1)
                if (T < 64.0) eT = exp(-T);
#pragma unroll
            for (int m = 0; m < M; m++) F[m + 1] = fma((double)(2 * m + 1), F[m], -eT) * i2T;
        }
    }
}

// The in-place Hermite recursion for a fixed total order LT, in registers:
// for n = LT-1 .. 0 the entries of order <= LT-n in decreasing index (so
// the orders an entry reads still hold R^{(n+1)}), then R^{(n)}_{000}.
template <int H>
struct JitStep {   // R_h = X_dir R_{h1} + c R_{h2}
    static constexpr int t = jit_hcomp(H, 0), u = jit_hcomp(H, 1), w = jit_hcomp(H, 2);
    static constexpr int dir = t > 0 ? 0 : (u > 0 ? 1 : 2);
    static constexpr int c = dir == 0 ? t - 1 : (dir == 1 ? u - 1 : w - 1);
    static constexpr int h1 = dir == 0 ? jit_herm(t - 1, u, w) : (dir == 1 ? jit_herm(t, u - 1, w) : jit_herm(t, u, w - 1));
    static constexpr int h2 = c <= 0 ? -1 : (dir == 0 ? jit_herm(t - 2, u, w) : (dir == 1 ? jit_herm(t, u - 2, w) : jit_herm(t, u, w - 2)));
};
template <int H>
__host__ __device__ inline void jit_rdesc(double *r, const double *xyz) {
    if constexpr (H >= 1) {
        using S = JitStep<H>;
        if constexpr (S::h2 >= 0) r[H] = fma(xyz[S::dir], r[S::h1], (double)S::c * r[S::h2]);
        else r[H] = xyz[S::dir] * r[S::h1];
        jit_rdesc<H - 1>(r, xyz);
    }
}
template <int LT, int N>
__host__ __device__ inline void jit_rlevel(double *r, const double *xyz, const double *Fs) {
    if constexpr (N >= 0) {
        jit_rdesc<jit_nherm(LT - N) - 1>(r, xyz);
        r[0] = Fs[N];
        jit_rlevel<LT, N - 1>(r, xyz, Fs);
    }
}

template <int H1, int... H2>
__host__ __device__ inline void jit_vrow(const double *R, const double *H, double &V, std::integer_sequence<int, H2...>) {
    ((V = fma(R[JitSum<H1, H2>::idx], H[H2], V)), ...);
}
template <int LB, int... H1>
__host__ __device__ inline void jit_vall(const double *R, const double *H, double *V, std::integer_sequence<int, H1...>) {
    (jit_vrow<H1>(R, H, V[H1], std::make_integer_sequence<int, jit_nherm(LB)>{}), ...);
}
// V += R H / sqrt(p+q) of one bra centre (exponent p, position P, order LA)
// and one ket centre (kg: q, Q; Hermite density Hk, order LB).
template <int LA, int LB>
__host__ __device__ inline void jit_pair(double p, double Px, double Py, double Pz, double q, double Qx, double Qy,
                                         double Qz, const double *Hk, const double *bt, double *V) {
    constexpr int LT = LA + LB;
    const double xyz[3] = {Px - Qx, Py - Qy, Pz - Qz};
    const double s = jit_rsqrt(p + q);
    const double alpha = p * q * (s * s);
    const double T = alpha * fma(xyz[0], xyz[0], fma(xyz[1], xyz[1], xyz[2] * xyz[2]));
    double F[LT + 1];
    jit_boys<LT>(T, bt, F);
    double f = s;
#pragma unroll
    for (int n = 0; n <= LT; n++) { F[n] *= f; f *= -2.0 * alpha; }
    double R[jit_nherm(LT)];
    R[0] = F[LT];
    jit_rlevel<LT, LT - 1>(R, xyz, F);
    jit_vall<LB>(R, Hk, V, std::make_integer_sequence<int, jit_nherm(LA)>{});
}

// Hermite expansion coefficients of one primitive pair along one direction,
// for a fixed (LA, LB): e[i][j][t], zero for t > i + j.  E^{00}_0 = 1: the
// exponential factor is in the pair prefactor K.  Two-term recurrences
// E^{i+1,j}_t = E^{ij}_{t-1} / (2p) + X_PA E^{ij}_t + (t+1) E^{ij}_{t+1}, and
// the same in j with X_PB.  (Trip counts are constant, so that every index is
// one after unrolling.)
template <int LA, int LB>
__host__ __device__ inline void jit_hermite_e(double xpa, double xpb, double i2p, double (&e)[LA + 1][LB + 1][LA + LB + 1]) {
    constexpr int NT = LA + LB + 1;
#pragma unroll
    for (int i = 0; i <= LA; i++)
#pragma unroll
        for (int j = 0; j <= LB; j++)
#pragma unroll
            for (int t = 0; t < NT; t++) e[i][j][t] = 0.0;
    e[0][0][0] = 1.0;
#pragma unroll
    for (int i = 0; i < LA; i++)
#pragma unroll
        for (int t = 0; t < NT; t++)
            if (t <= i + 1)
                e[i + 1][0][t] = (t > 0 ? i2p * e[i][0][t > 0 ? t - 1 : 0] : 0.0) + (t <= i ? xpa * e[i][0][t] : 0.0) +
                                 (t + 1 <= i ? (t + 1) * e[i][0][t + 1 < NT ? t + 1 : 0] : 0.0);
#pragma unroll
    for (int i = 0; i <= LA; i++)
#pragma unroll
        for (int j = 0; j < LB; j++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                if (t <= i + j + 1)
                    e[i][j + 1][t] = (t > 0 ? i2p * e[i][j][t > 0 ? t - 1 : 0] : 0.0) + (t <= i + j ? xpb * e[i][j][t] : 0.0) +
                                     (t + 1 <= i + j ? (t + 1) * e[i][j][t + 1 < NT ? t + 1 : 0] : 0.0);
}
template <int LA, int LB>
struct JitE {
    double x[LA + 1][LB + 1][LA + LB + 1], y[LA + 1][LB + 1][LA + LB + 1], z[LA + 1][LB + 1][LA + LB + 1];
    // E tables of primitive pr of the pair at geo, the x table times f
    __host__ __device__ inline void make(const double *pr, const double *geo, double f) {
        jit_hermite_e<LA, LB>(pr[1] - geo[0], pr[1] - geo[3], pr[5], x);
        jit_hermite_e<LA, LB>(pr[2] - geo[1], pr[2] - geo[4], pr[5], y);
        jit_hermite_e<LA, LB>(pr[3] - geo[2], pr[3] - geo[5], pr[5], z);
#pragma unroll
        for (int i = 0; i <= LA; i++)
#pragma unroll
            for (int j = 0; j <= LB; j++)
#pragma unroll
                for (int t = 0; t <= LA + LB; t++) x[i][j][t] *= f;
    }
};
// Cartesian component AB of class (LA, LB) and Hermite triple H: whether H is
// in the component's box, and its E product.
template <int LA, int LB, int AB, int H>
struct JitBox {
    static constexpr int ia = AB / jit_ncart(LB), ib = AB % jit_ncart(LB);
    static constexpr int ax = jit_cexp(LA, ia, 0), ay = jit_cexp(LA, ia, 1), az = jit_cexp(LA, ia, 2);
    static constexpr int bx = jit_cexp(LB, ib, 0), by = jit_cexp(LB, ib, 1), bz = jit_cexp(LB, ib, 2);
    static constexpr int t = jit_hcomp(H, 0), u = jit_hcomp(H, 1), w = jit_hcomp(H, 2);
    static constexpr bool in = t <= ax + bx && u <= ay + by && w <= az + bz;
    static constexpr bool neg = ((t + u + w) & 1) != 0;
    static __host__ __device__ inline double e(const JitE<LA, LB> &E) { return E.x[ax][bx][t] * E.y[ay][by][u] * E.z[az][bz][w]; }
};
template <int LA, int LB, int AB, int... H>
__host__ __device__ inline void jit_dens_ab(const JitE<LA, LB> &E, double x, double *Hc, std::integer_sequence<int, H...>) {
    ([&] {
        using B = JitBox<LA, LB, AB, H>;
        if constexpr (B::in) Hc[H] = fma(B::neg ? -x : x, B::e(E), Hc[H]);
    }(), ...);
}
template <int LA, int LB, int... AB>
__host__ __device__ inline void jit_dens_all(const JitE<LA, LB> &E, const JitView &v, const int *km, double *Hc,
                                             std::integer_sequence<int, AB...>) {
    ([&] {
        const int k = km[AB];   // k < 0: the row is not used
        const double x = k < 0 ? 0.0 : (k < v.N ? v.X[k] : v.Y0[k - v.N]);
        jit_dens_ab<LA, LB, AB>(E, x, Hc, std::make_integer_sequence<int, jit_nherm(LA + LB)>{});
    }(), ...);
}
// Hermite density of one contribution: entry e (class LA, LB), primitive pr;
// 2 pi^{5/2} K / q and the ket's signs are in it.
template <int LA, int LB>
__host__ __device__ inline void jit_dens(const JitView &v, int e, int b, const double *pr, double *Hc) {
    JitE<LA, LB> E;
    E.make(pr, v.pgeo + 6 * (size_t)b, 4.0 * M_PI * M_PI * sqrt(M_PI) * pr[5] * pr[4]);
    jit_dens_all<LA, LB>(E, v, v.kmap + v.kl_moff[e], Hc, std::make_integer_sequence<int, jit_ncart(LA) * jit_ncart(LB)>{});
}
// Hermite density of centre c of order L: its contributions in order.
template <int L>
__host__ __device__ inline void jit_density(const JitView &v, int c) {
    double Hc[jit_nherm(L)];
#pragma unroll
    for (int h = 0; h < jit_nherm(L); h++) Hc[h] = 0.0;
    for (int k = v.cptr[c]; k < v.cptr[c + 1]; k++) {
        const int e = v.cent[k], b = v.kl_pair[e];
        const double *pr = v.prim + 6 * (size_t)v.cprim[k];
        if constexpr (L == 0) jit_dens<0, 0>(v, e, b, pr, Hc);
        if constexpr (L == 1) { if (v.pinfo[4 * b] == 0) jit_dens<0, 1>(v, e, b, pr, Hc); else jit_dens<1, 0>(v, e, b, pr, Hc); }
        if constexpr (L == 2) {
            const int la = v.pinfo[4 * b];
            if (la == 0) jit_dens<0, 2>(v, e, b, pr, Hc);
            else if (la == 1) jit_dens<1, 1>(v, e, b, pr, Hc);
            else jit_dens<2, 0>(v, e, b, pr, Hc);
        }
        if constexpr (L == 3) { if (v.pinfo[4 * b] == 1) jit_dens<1, 2>(v, e, b, pr, Hc); else jit_dens<2, 1>(v, e, b, pr, Hc); }
        if constexpr (L == 4) jit_dens<2, 2>(v, e, b, pr, Hc);
    }
    double *o = v.H + v.hoff[L] + (long long)(c - v.coff[L]) * jit_nherm(L);
#pragma unroll
    for (int h = 0; h < jit_nherm(L); h++) o[h] = Hc[h];
}

// One thread per centre, workgroups of one order, the highest (and slowest)
// first.  The E tables of order 4 take 256 VGPRs and 30 AGPRs, so one wave per
// SIMD: 1,024 fit, C30H62 has 1,236 (77,249 centres; 31 us).
__global__ void __launch_bounds__(256) jit_density_kernel(JitView v) {
    int b = blockIdx.x, L = JIT_OMAX;
    for (; L > 0; L--) {
        const int nb = (v.coff[L + 1] - v.coff[L] + 255) / 256;
        if (b < nb) break;
        b -= nb;
    }
    const int c = v.coff[L] + b * 256 + threadIdx.x;
    if (c >= v.coff[L + 1]) return;
    switch (L) {
    case 0: jit_density<0>(v, c); break;
    case 1: jit_density<1>(v, c); break;
    case 2: jit_density<2>(v, c); break;
    case 3: jit_density<3>(v, c); break;
    default: jit_density<4>(v, c); break;
    }
}

// Rows of entry e (class LA, LB) from the potentials of its primitives'
// centres: primitives sub, sub + NS, ... on this lane; NS lanes share an
// entry and add their rows in a fixed order.
template <int LA, int LB, int AB, int... H>
__host__ __device__ inline double jit_row_ab(const JitE<LA, LB> &E, const double *Vc, std::integer_sequence<int, H...>) {
    double s = 0.0;
    ([&] {
        using B = JitBox<LA, LB, AB, H>;
        if constexpr (B::in) s = fma(B::e(E), Vc[H], s);
    }(), ...);
    return s;
}
template <int LA, int LB, int... AB>
__host__ __device__ inline void jit_row_all(const JitE<LA, LB> &E, const double *Vc, double *acc, std::integer_sequence<int, AB...>) {
    ((acc[AB] += jit_row_ab<LA, LB, AB>(E, Vc, std::make_integer_sequence<int, jit_nherm(LA + LB)>{})), ...);
}
template <int LA, int LB, int NS>
__host__ __device__ inline void jit_rows(const JitView &v, int e, int b, int sub) {
    constexpr int L = LA + LB, NAB = jit_ncart(LA) * jit_ncart(LB), NH = jit_nherm(L);
    double acc[NAB];
#pragma unroll
    for (int k = 0; k < NAB; k++) acc[k] = 0.0;
    const int np = v.pinfo[4 * b + 2], p0 = v.pinfo[4 * b + 3], ec = v.e_c0[e];
    for (int k = sub; k < np; k += NS) {
        const double *pr = v.prim + 6 * (size_t)(p0 + k);
        const double *Vp = v.V + v.hoff[L] + (long long)(v.ecen[ec + k] - v.coff[L]) * NH;
        double Vc[NH];
#pragma unroll
        for (int h = 0; h < NH; h++) Vc[h] = Vp[h];
        JitE<LA, LB> E;
        E.make(pr, v.pgeo + 6 * (size_t)b, 2.0 * pr[5] * pr[4]);
        jit_row_all<LA, LB>(E, Vc, acc, std::make_integer_sequence<int, NAB>{});
    }
    const int *om = v.kmap + v.kl_moff[e];
#pragma unroll
    for (int k = 0; k < NAB; k++) {
        double a = acc[k];
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
        for (int s = 1; s < NS; s <<= 1) a += __shfl_xor(a, s, NS);
#endif
        if (k % NS == sub) {
            const int o = om[k];
            if (o >= 0) {
                if (o < v.N) v.YJ[o] = a;
                else v.Y1[o - v.N] = a;
            }
        }
    }
}
template <int NS>
__host__ __device__ inline void jit_rows_any(const JitView &v, int e, int sub) {
    const int b = v.kl_pair[e];
    switch (v.pinfo[4 * b] * 3 + v.pinfo[4 * b + 1]) {
    case 0: jit_rows<0, 0, NS>(v, e, b, sub); break;
    case 1: jit_rows<0, 1, NS>(v, e, b, sub); break;
    case 2: jit_rows<0, 2, NS>(v, e, b, sub); break;
    case 3: jit_rows<1, 0, NS>(v, e, b, sub); break;
    case 4: jit_rows<1, 1, NS>(v, e, b, sub); break;
    case 5: jit_rows<1, 2, NS>(v, e, b, sub); break;
    case 6: jit_rows<2, 0, NS>(v, e, b, sub); break;
    case 7: jit_rows<2, 1, NS>(v, e, b, sub); break;
    default: jit_rows<2, 2, NS>(v, e, b, sub); break;
    }
}
// Eight lanes per entry; entries are sorted by class, so a wave's eight
// entries take one path.  256 VGPRs and 86 AGPRs, one wave per SIMD (C30H62:
// 3,584 waves, 28 us).
static const int JIT_RLANES = 8;
__global__ void __launch_bounds__(256) jit_rows_kernel(JitView v, int nout) {
    const int i = (blockIdx.x * 256 + threadIdx.x) / JIT_RLANES;
    // whole lane groups leave together: the shuffles stay within a group
    if (i < nout) jit_rows_any<JIT_RLANES>(v, v.oent[i], threadIdx.x % JIT_RLANES);
}

// The potential kernels, bound by FP64 vector issue: C30H62 has 5.4e8 pairs
// of centres (1.08e9 primitive quartets) at 45 (s-s) to about 2,000 (order 4
// with 4) vector instructions, 104 on average (8.8e8 of whole waves, idle
// lanes among them): 1.5 ms at one per SIMD and four cycles.  The three
// launches take 1.18 + 0.63 + 0.20 ms (total orders <= 2, 3 and 4, >= 5), in
// place of 255 ms when every quartet formed its Cartesian components.
// Counters: vector instructions issue in 86%, 77% and 54% of their SIMD
// cycles, 70%, 82% and 87% of them FP64 arithmetic.  The last one keeps 474
// registers (one wave per SIMD, so latency shows) and moves 114 VGPRs through
// AGPRs; the first loses 16% of its LDS cycles to bank conflicts of the
// table.  One wave per task, lanes over bra centres (their
// exponent, position and potential in registers), a loop over the ket
// centres, which are the same for every lane: their data come through scalar
// loads and feed the FMAs from scalar registers.  A task whose centres fill
// less than half a wave gives each centre 64 / bw lanes, which take the ket
// centres in turn and add their potentials at the end in a fixed order.
template <int LA, int LB, bool UNI>
__device__ __forceinline__ void jit_potential(const JitView &v, const JitTask &t, const double *__restrict__ cgeo,
                                              const double *__restrict__ Hall, const int *__restrict__ segs,
                                              const double *bt) {
    constexpr int NA = jit_nherm(LA), NB = jit_nherm(LB);
    const int lane = threadIdx.x & 63, bw = 1 << t.lbw;
    const int b = lane & (bw - 1), sl = UNI ? 0 : lane >> t.lbw, ns = UNI ? 1 : 64 >> t.lbw;
    const double *bg = cgeo + 4 * (long long)(t.c0 + min(b, t.n - 1));   // lanes past the tile repeat its last centre
    const double p = bg[0], Px = bg[1], Py = bg[2], Pz = bg[3];
    double V[NA];
#pragma unroll
    for (int h = 0; h < NA; h++) V[h] = 0.0;
    const double *Hb = Hall + v.hoff[LB] - (long long)v.coff[LB] * NB;
    for (int sg = t.s0; sg < t.s1; sg++) {
        const int k0 = segs[2 * sg], k1 = segs[2 * sg + 1];
        for (int j = k0 + sl; j < k1; j += ns) {
            const double *g = cgeo + 4 * (long long)j;
            jit_pair<LA, LB>(p, Px, Py, Pz, g[0], g[1], g[2], g[3], Hb + (long long)j * NB, bt, V);
        }
    }
    if constexpr (!UNI) {
#pragma unroll
        for (int h = 0; h < NA; h++)
            for (int s = bw; s < 64; s <<= 1) V[h] += __shfl_xor(V[h], s, 64);
    }
    if (lane < t.n) {
        double *o = v.part + t.poff + lane;
#pragma unroll
        for (int h = 0; h < NA; h++) o[(long long)h * bw] = V[h];
    }
}

// Groups of classes by total order LT, one kernel each: 0 LT <= 2, 1 LT 3 and
// 4, 2 LT >= 5 (up to 165 Hermite integrals per lane).  The tasks of a
// workgroup share a class, so its Boys table is one order's.
__host__ __device__ constexpr int jit_group(int LT) { return LT <= 2 ? 0 : (LT <= 4 ? 1 : 2); }
template <int G, int LA, int LB>
__device__ __forceinline__ void jit_run(const JitView &v, const JitTask &t, const double *__restrict__ cgeo,
                                        const double *__restrict__ H, const int *__restrict__ segs, const double *bt) {
    if constexpr (jit_group(LA + LB) == G) {
        if (G < 2 && t.lbw == 6) jit_potential<LA, LB, true>(v, t, cgeo, H, segs, bt);
        else jit_potential<LA, LB, false>(v, t, cgeo, H, segs, bt);
    }
}
template <int G, int... C>
__device__ __forceinline__ void jit_dispatch(const JitView &v, const JitTask &t, const double *__restrict__ cgeo,
                                             const double *__restrict__ H, const int *__restrict__ segs,
                                             const double *bt, std::integer_sequence<int, C...>) {
    ([&] { if constexpr (jit_group(C / JIT_NORD + C % JIT_NORD) == G) {
        if (t.cls == C) jit_run<G, C / JIT_NORD, C % JIT_NORD>(v, t, cgeo, H, segs, bt);
    } }(), ...);
}
template <int G> constexpr int jit_waves() { return G == 0 ? 4 : (G == 1 ? 2 : 1); }
template <int G>
__global__ void __launch_bounds__(64 * JIT_WPG, jit_waves<G>())
jit_potential_kernel(JitView v, const JitTask *__restrict__ tasks, const double *__restrict__ cgeo,
                     const double *__restrict__ H, const int *__restrict__ segs, const double *__restrict__ boys) {
    __shared__ double2 bt[JIT_BGRID * JIT_BROW / 2];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const JitTask t = tasks[JIT_WPG * blockIdx.x + wave];
    const int LT = t.cls / JIT_NORD + t.cls % JIT_NORD;
    const double2 *src = reinterpret_cast<const double2 *>(boys + (long long)LT * JIT_BGRID * JIT_BROW);
#pragma unroll
    for (int k = threadIdx.x; k < JIT_BGRID * JIT_BROW / 2; k += 64 * JIT_WPG) bt[k] = src[k];
    __syncthreads();
    if (t.n == 0) return;   // padding of the workgroup
    jit_dispatch<G>(v, t, cgeo, H, segs, reinterpret_cast<const double *>(bt),
                    std::make_integer_sequence<int, JIT_NORD * JIT_NORD>{});
}

// V of the centres of chunk g: the partials of its tasks, in order.
__host__ __device__ inline void jit_reduce(const JitView &v, const JitChunk &g, int lane, int NL) {
    const int nh = jit_nherm(g.la), bw = 1 << g.lbw;
    double *o = v.V + v.hoff[g.la] + (long long)(g.c0 - v.coff[g.la]) * nh;
    for (int q = lane; q < nh * bw; q += NL) {
        const int h = q >> g.lbw, b = q & (bw - 1);
        if (b >= g.n) continue;
        double s = 0.0;
        #pragma unroll 8
        for (int k = g.t0; k < g.t1; k++) s += v.part[v.cpoff[k] + q];
        o[(long long)b * nh + h] = s;
    }
}
__global__ void __launch_bounds__(256) jit_reduce_kernel(JitView v) { jit_reduce(v, v.chunks[blockIdx.x], threadIdx.x, 256); }

// The sweeps, one launch per tree level.  They are bound by the read of U
// (once each); a level near the root has few nodes, so a node is spread over
// workgroups by columns (up) and rows (down).
//
// Up sweep: y0[n] = U_n^T in_n, the input rows from x (leaves) or from the
// children's y0 (index map uin).  A workgroup takes 64 columns of a node
// (lanes; a wave reads 512 bytes of a row), its 16 waves split the rows with
// eight loads in flight, inputs staged in LDS; partial sums added in a fixed
// order.  C30H62 (4 levels, 128 MB of U): 4 x 13.5 us; with one workgroup
// of four waves per node 4 x 190 us.
static const int JIT_URB = 1024;   // input rows staged at a time
__global__ void __launch_bounds__(1024) jit_up_kernel(const int *__restrict__ items, const long long *__restrict__ uoff,
                                                      const int *__restrict__ unr, const int *__restrict__ unc,
                                                      const int *__restrict__ uin0, const int *__restrict__ y0off,
                                                      const int *__restrict__ uin, const double *__restrict__ U,
                                                      const double *__restrict__ X, double *__restrict__ Y0, int N) {
    __shared__ double xin[JIT_URB];
    __shared__ double red[16][64];
    const int n = items[2 * blockIdx.x], c0 = items[2 * blockIdx.x + 1];
    const int nr = unr[n], ncl = unc[n], w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const double *Un = U + uoff[n] + min(c0 + lane, ncl - 1);   // lanes past the last column repeat it
    const int *in = uin + uin0[n];
    double s = 0.0;
    for (int rb = 0; rb < nr; rb += JIT_URB) {
        const int m = min(JIT_URB, nr - rb);
        __syncthreads();
        for (int r = threadIdx.x; r < m; r += 1024) {
            const int k = in[rb + r];
            xin[r] = k < N ? X[k] : Y0[k - N];
        }
        __syncthreads();
        int r = w;
        for (; r + 7 * 16 < m; r += 8 * 16) {
            double u[8];
#pragma unroll
            for (int k = 0; k < 8; k++) u[k] = Un[(size_t)(rb + r + 16 * k) * ncl];
#pragma unroll
            for (int k = 0; k < 8; k++) s = fma(u[k], xin[r + 16 * k], s);
        }
        for (; r < m; r += 16) s = fma(Un[(size_t)(rb + r) * ncl], xin[r], s);
    }
    red[w][lane] = s;
    __syncthreads();
    for (int h = 8; h > 0; h >>= 1) {
        if (w < h) red[w][lane] += red[w + h][lane];
        __syncthreads();
    }
    if (w == 0 && c0 + lane < ncl) Y0[y0off[n] + c0 + lane] = red[0][lane];
}

// Down sweep: t = U_n y1[n]; row r goes to its leaf row of yd (index < N) or
// is added to the child's y1 (index - N; a child has one parent).  A
// workgroup takes 64 rows of a node, a wave four rows at a time with its
// lanes over the columns.  C30H62: 4 x 12.7 us; with a thread per row 4 x 133 us.
static const int JIT_DROWS = 64;
__global__ void __launch_bounds__(256) jit_down_kernel(const int *__restrict__ items, const long long *__restrict__ uoff,
                                                       const int *__restrict__ unr, const int *__restrict__ unc,
                                                       const int *__restrict__ uin0, const int *__restrict__ y0off,
                                                       const int *__restrict__ uin, const double *__restrict__ U,
                                                       double *__restrict__ YD, double *__restrict__ Y1, int N) {
    const int n = items[2 * blockIdx.x], r0 = items[2 * blockIdx.x + 1];
    const int nr = unr[n], ncl = unc[n], w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const double *Un = U + uoff[n];
    const double *y1 = Y1 + y0off[n];
    const int *out = uin + uin0[n];
    const int re = min(r0 + JIT_DROWS, nr);
    for (int r = r0 + 4 * w; r < re; r += 16) {
        const double *row[4];
        double s[4];
#pragma unroll
        for (int k = 0; k < 4; k++) { row[k] = Un + (size_t)min(r + k, re - 1) * ncl; s[k] = 0.0; }
        for (int c = lane; c < ncl; c += 64) {
            const double y = y1[c];
#pragma unroll
            for (int k = 0; k < 4; k++) s[k] = fma(row[k][c], y, s[k]);
        }
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) s[k] += __shfl_xor(s[k], d, 64);
        if (lane < 4 && r + lane < re) {
            const double v = lane == 0 ? s[0] : (lane == 1 ? s[1] : (lane == 2 ? s[2] : s[3]));
            const int k = out[r + lane];
            if (k < N) YD[k] = v;
            else Y1[k - N] += v;
        }
    }
}

__global__ void jit_zero_kernel(double *__restrict__ a, long long n) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        a[i] = 0.0;
}

__global__ void jit_add_kernel(const double *__restrict__ a, const double *__restrict__ b, double *__restrict__ y, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = a[i] + b[i];
}

// ---------------------------------------------------------------------------
// Host plan
// ---------------------------------------------------------------------------
struct JitPlan {
    int N = 0, nY = 0, num_sp = 0, max_level = 0;
    std::vector<int> pinfo;
    std::vector<double> pgeo, prim;
    std::vector<int> kl_start, kl_count, kl_pair, kl_moff, kmap;
    // Hermite centres, order by order, and their contributions
    std::vector<int> e_c0, ecen, cptr, cent, cprim;
    std::vector<double> cgeo;
    int coff[JIT_NORD + 1] = {};
    long long hoff[JIT_NORD] = {}, nherm = 0;
    // tasks: group g in [gtask[g], gtask[g + 1]), whole workgroups
    std::vector<JitTask> tasks;
    std::vector<JitChunk> chunks;
    std::vector<int> segs, ctask, oent;
    std::vector<long long> cpoff;
    int gtask[4] = {};
    long long npart = 0;
    int ntask = 0;   // without the padding
    std::vector<double> boys;
    // sweeps
    std::vector<long long> uoff;
    std::vector<int> unr, unc, uin0, y0off, uin;
    std::vector<double> U;
    std::vector<std::vector<int>> level_nodes;   // nodes with a non-empty U, per level
    // work per matvec
    double quartets = 0, prim_quartets = 0, eri_values = 0;
    double cost_b = 0, cost_d = 0;   // planned task cost of coupling and near-field blocks
};

// The Boys tables of the potential kernels (JIT_BROW): per order M and
// interval the Taylor coefficients F_{M+k}(T0) / k!, k = 0..8, with the last
// two replaced by their best lower-degree polynomials on |d| <= 1/32 (from
// the Chebyshev polynomials T_8 and T_7); what is left out is below
// (1/32)^7 / (64 7!) F_{M+7}, 1e-16 of F_M for M <= 8.
static void jit_boys_tables(std::vector<double> &out) {
    const int top = 2 * JIT_OMAX + 8;
    out.assign((size_t)JIT_NLT * JIT_BGRID * JIT_BROW, 0.0);
    for (int gi = 0; gi < JIT_BGRID; gi++) {
        const long double T = (gi + 0.5L) / 16.0L, eT = expl(-T);
        long double F[2 * JIT_OMAX + 9];
        long double term = 1.0L / (2 * top + 1), sum = term;
        for (int k = 1; k < 2000 && term >= sum * 1e-21L; k++) {
            term *= 2.0L * T / (long double)(2 * top + 2 * k + 1);
            sum += term;
        }
        F[top] = eT * sum;
        for (int m = top; m > 0; m--) F[m - 1] = (2.0L * T * F[m] + eT) / (long double)(2 * m - 1);
        for (int M = 0; M < JIT_NLT; M++) {
            long double c[9], fact = 1.0L;
            for (int k = 0; k <= 8; k++) { c[k] = F[M + k] / fact; fact *= (long double)(k + 1); }
            const long double r = 1.0L / 32.0L, r2 = r * r;
            c[6] += c[8] * r2 * 2.0L;
            c[4] -= c[8] * r2 * r2 * 160.0L / 128.0L;
            c[2] += c[8] * r2 * r2 * r2 * 32.0L / 128.0L;
            c[0] -= c[8] * r2 * r2 * r2 * r2 / 128.0L;
            c[5] += c[7] * r2 * 112.0L / 64.0L;
            c[3] -= c[7] * r2 * r2 * 56.0L / 64.0L;
            c[1] += c[7] * r2 * r2 * r2 * 7.0L / 64.0L;
            double *tab = out.data() + (size_t)M * JIT_BGRID * JIT_BROW;
            for (int k = 0; k < 8; k++) tab[jit_bpos(gi, k >> 1) + (k & 1)] = (double)(k < 7 ? c[k] : eT);
        }
    }
}

static bool jit_plan(H2ERI_p h, JitPlan &J) {
    HostState *hs = host_state(h);
    const int np = h->num_sp, n_node = h->n_node, N = h->krnl_mat_size;
    if (!h->BD_JIT || !h->U || (int)hs->pairs.size() != np || np <= 0) {
        set_error(ERR_ARG, "on-the-fly B/D: no BD_JIT representation with shell-pair data");
        return false;
    }
    if (!h->J_pair || !h->J_row || !h->pt_cluster || !h->mat_cluster || !h->sp_bfp_sidx || !h->node_level) {
        set_error(ERR_ARG, "on-the-fly B/D: tree or skeleton lists missing");
        return false;
    }
    J.N = N;
    J.num_sp = np;
    J.max_level = h->max_level;
    // ---- shell pairs
    J.pinfo.resize(4 * (size_t)np);
    J.pgeo.resize(6 * (size_t)np);
    for (int i = 0; i < np; i++) {
        const PairView pv = pair_view(hs->pairs[i]);
        if (pv.la > JIT_LMAX || pv.lb > JIT_LMAX || pv.la < 0 || pv.lb < 0) {
            set_error(ERR_UNSUPPORTED, "on-the-fly B/D: shell pair %d has angular momentum above d", i);
            return false;
        }
        if (pv.np > 1296) {   // 36 x 36 primitives: the interface's limit
            set_error(ERR_UNSUPPORTED, "on-the-fly B/D: shell pair %d has %d primitive pairs (at most 1296)", i, pv.np);
            return false;
        }
        if (jit_ncart(pv.la) * jit_ncart(pv.lb) != h->sp_nbfp[i] ||
            h->sp_bfp_sidx[i + 1] - h->sp_bfp_sidx[i] != h->sp_nbfp[i]) {
            set_error(ERR_ARG, "on-the-fly B/D: shell pair %d rows disagree with sp_nbfp", i);
            return false;
        }
        J.pinfo[4 * i] = pv.la;
        J.pinfo[4 * i + 1] = pv.lb;
        J.pinfo[4 * i + 2] = pv.np;
        J.pinfo[4 * i + 3] = (int)(J.prim.size() / 6);
        for (int d = 0; d < 3; d++) { J.pgeo[6 * i + d] = pv.A[d]; J.pgeo[6 * i + 3 + d] = pv.B[d]; }
        for (int k = 0; k < pv.np; k++) {
            J.prim.push_back(pv.p[k]);
            for (int d = 0; d < 3; d++) J.prim.push_back(pv.P[3 * k + d]);
            J.prim.push_back(pv.K[k]);
            J.prim.push_back(0.5 / pv.p[k]);
        }
    }
    if (J.prim.size() / 6 >= (size_t)INT32_MAX) { set_error(ERR_UNSUPPORTED, "on-the-fly B/D: too many primitive pairs"); return false; }
    // ---- nodes: ranks, y0 offsets, U and the sweep index maps
    auto rank = [&](int n) { return h->U[n] ? h->U[n]->ncol : 0; };
    auto urows = [&](int n) { return h->U[n] ? h->U[n]->nrow : 0; };
    J.y0off.assign(n_node, 0);
    J.unr.assign(n_node, 0);
    J.unc.assign(n_node, 0);
    J.uin0.assign(n_node, 0);
    J.uoff.assign(n_node, 0);
    long long ny = 0;
    for (int n = 0; n < n_node; n++) { J.y0off[n] = (int)ny; ny += rank(n); }
    if (ny + N >= INT32_MAX) { set_error(ERR_UNSUPPORTED, "on-the-fly B/D: index space too large"); return false; }
    J.nY = (int)ny;
    J.level_nodes.assign(h->max_level + 1, {});
    for (int n = 0; n < n_node; n++) {
        const int nr = urows(n), nc = rank(n);
        J.uin0[n] = (int)J.uin.size();
        if (nr == 0 || nc == 0) continue;
        const H2E_dense_mat_p Un = h->U[n];
        J.unr[n] = nr;
        J.unc[n] = nc;
        J.uoff[n] = (long long)J.U.size();
        for (int r = 0; r < nr; r++)
            for (int c = 0; c < nc; c++) J.U.push_back(Un->data[(size_t)r * Un->ld + c]);
        if (h->n_child[n] == 0) {
            const int s0 = h->mat_cluster[2 * n], s1 = h->mat_cluster[2 * n + 1];
            if (s1 - s0 + 1 != nr || s0 < 0 || s1 >= N) {
                set_error(ERR_ARG, "on-the-fly B/D: leaf %d has %d U rows for %d x rows", n, nr, s1 - s0 + 1);
                return false;
            }
            for (int r = 0; r < nr; r++) J.uin.push_back(s0 + r);
        } else {
            int tot = 0;
            for (int k = 0; k < h->n_child[n]; k++) {
                const int ch = h->children[(size_t)n * 8 + k];   // 8 child slots per node
                for (int r = 0; r < rank(ch); r++) J.uin.push_back(N + J.y0off[ch] + r);
                tot += rank(ch);
            }
            if (tot != nr) {
                set_error(ERR_ARG, "on-the-fly B/D: node %d has %d U rows for %d child ranks", n, nr, tot);
                return false;
            }
        }
        const int lv = h->node_level[n];
        if (lv < 0 || lv > h->max_level) { set_error(ERR_ARG, "on-the-fly B/D: node %d level %d", n, lv); return false; }
        J.level_nodes[lv].push_back(n);
    }
    // ---- partner lists: 2n = full rows of leaf n, 2n + 1 = skeleton rows of n
    auto is_leaf = [&](int n) { return h->n_child[n] == 0; };
    J.kl_start.assign(2 * (size_t)n_node, 0);
    J.kl_count.assign(2 * (size_t)n_node, 0);
    std::vector<std::vector<int>> skel_pos(n_node);   // row of the concatenated J_pair rows -> skeleton index
    for (int n = 0; n < n_node; n++) {
        if (is_leaf(n)) {
            J.kl_start[2 * n] = (int)J.kl_pair.size();
            for (int b = h->pt_cluster[2 * n]; b <= h->pt_cluster[2 * n + 1]; b++) {
                J.kl_pair.push_back(b);
                J.kl_moff.push_back((int)J.kmap.size());
                for (int c = 0; c < h->sp_nbfp[b]; c++) J.kmap.push_back(h->sp_bfp_sidx[b] + c);
            }
            J.kl_count[2 * n] = (int)J.kl_pair.size() - J.kl_start[2 * n];
        }
        const H2E_int_vec_p jp = h->J_pair[n], jr = h->J_row[n];
        if (!jp || !jr || rank(n) == 0) continue;
        if (jr->length != rank(n)) {
            set_error(ERR_ARG, "on-the-fly B/D: node %d has %d skeleton rows for rank %d", n, jr->length, rank(n));
            return false;
        }
        int tot = 0;
        for (int k = 0; k < jp->length; k++) tot += h->sp_nbfp[jp->data[k]];
        std::vector<int> &pos = skel_pos[n];
        pos.assign(tot, -1);
        for (int j = 0; j < jr->length; j++) {
            if (jr->data[j] < 0 || jr->data[j] >= tot) { set_error(ERR_ARG, "on-the-fly B/D: node %d skeleton row", n); return false; }
            pos[jr->data[j]] = j;
        }
        J.kl_start[2 * n + 1] = (int)J.kl_pair.size();
        int rr = 0;
        for (int k = 0; k < jp->length; k++) {
            const int b = jp->data[k];
            bool any = false;
            for (int c = 0; c < h->sp_nbfp[b]; c++) any |= pos[rr + c] >= 0;
            if (any) {
                J.kl_pair.push_back(b);
                J.kl_moff.push_back((int)J.kmap.size());
                for (int c = 0; c < h->sp_nbfp[b]; c++)
                    J.kmap.push_back(pos[rr + c] >= 0 ? N + J.y0off[n] + pos[rr + c] : -1);
            }
            rr += h->sp_nbfp[b];
        }
        J.kl_count[2 * n + 1] = (int)J.kl_pair.size() - J.kl_start[2 * n + 1];
    }
    // ---- partners
    std::vector<std::vector<int>> adm(n_node), nearf(n_node);
    for (int i = 0; i < h->n_r_adm_pair; i++) {
        const int n0 = h->r_adm_pairs[2 * i], n1 = h->r_adm_pairs[2 * i + 1];
        adm[n0].push_back(n1);
        adm[n1].push_back(n0);
    }
    for (int i = 0; i < h->n_leaf_node; i++) nearf[h->height_nodes[i]].push_back(h->height_nodes[i]);
    for (int i = 0; i < h->n_r_inadm_pair; i++) {
        const int n0 = h->r_inadm_pairs[2 * i], n1 = h->r_inadm_pairs[2 * i + 1];
        nearf[n0].push_back(n1);
        nearf[n1].push_back(n0);
    }
    auto lv = [&](int n) { return h->node_level[n]; };
    // ---- target sides and the sides they take
    struct Target { int list, n_near; std::vector<int> src; };   // the first n_near sources are near field
    std::vector<Target> targets;
    std::vector<char> used(2 * (size_t)n_node, 0);
    for (int n = 0; n < n_node; n++) {
        if (is_leaf(n)) {   // full rows: near field and case (2)/(3) coupling with n uncompressed
            Target t;
            t.list = 2 * n;
            for (int m : nearf[n]) {
                if (!is_leaf(m)) { set_error(ERR_ARG, "on-the-fly B/D: near-field partner %d is not a leaf", m); return false; }
                t.src.push_back(2 * m);
            }
            t.n_near = (int)t.src.size();
            for (int m : adm[n])
                if (lv(n) < lv(m)) t.src.push_back(2 * m + 1);
            if (!t.src.empty()) targets.push_back(t);
        }
        Target t;   // skeleton rows: partners at the same or a coarser level
        t.list = 2 * n + 1;
        t.n_near = 0;
        for (int m : adm[n]) {
            if (lv(n) < lv(m)) continue;
            if (lv(m) < lv(n) && !is_leaf(m)) {
                set_error(ERR_ARG, "on-the-fly B/D: coarser admissible partner %d of %d is not a leaf", m, n);
                return false;
            }
            t.src.push_back(lv(m) >= lv(n) ? 2 * m + 1 : 2 * m);
        }
        if (t.src.empty()) continue;
        if (!h->J_pair[n] || rank(n) == 0) {
            set_error(ERR_ARG, "on-the-fly B/D: node %d has coupling blocks and no skeleton", n);
            return false;
        }
        targets.push_back(t);
    }
    for (const Target &t : targets) {
        used[t.list] = 1;
        for (int L : t.src) used[L] = 1;
    }
    // ---- Hermite centres: primitives of one side with equal order, exponent
    // sum (bitwise) and centre (to rounding: (a A + b A) / p of one atom's
    // primitives depends on their order) are one centre
    const size_t ne = J.kl_pair.size();
    J.e_c0.assign(ne + 1, 0);
    for (size_t e = 0; e < ne; e++) J.e_c0[e + 1] = J.e_c0[e] + J.pinfo[4 * J.kl_pair[e] + 2];
    J.ecen.assign((size_t)J.e_c0[ne], -1);
    struct Cen { double g[4]; };
    std::vector<Cen> cen[JIT_NORD];
    std::vector<int> lc0[JIT_NORD];   // per list: its first centre of the order (lists in order, then the end)
    struct Key {
        long long a, x, y, z;
        bool operator==(const Key &o) const { return a == o.a && x == o.x && y == o.y && z == o.z; }
    };
    struct KeyHash {
        size_t operator()(const Key &k) const {
            unsigned long long s = (unsigned long long)k.a;
            for (long long w : {k.x, k.y, k.z}) s = (s ^ (unsigned long long)w) * 0x9e3779b97f4a7c15ULL, s ^= s >> 29;
            return (size_t)s;
        }
    };
    for (int l = 0; l < JIT_NORD; l++) lc0[l].assign(2 * (size_t)n_node + 1, 0);
    for (int L = 0; L < 2 * n_node; L++) {
        for (int l = 0; l < JIT_NORD; l++) lc0[l][L] = (int)cen[l].size();
        if (!used[L]) continue;
        std::unordered_map<Key, int, KeyHash> at[JIT_NORD];
        for (int e = J.kl_start[L]; e < J.kl_start[L] + J.kl_count[L]; e++) {
            const int b = J.kl_pair[e], l = J.pinfo[4 * b] + J.pinfo[4 * b + 1];
            for (int k = 0; k < J.pinfo[4 * b + 2]; k++) {
                const double *pr = J.prim.data() + 6 * (size_t)(J.pinfo[4 * b + 3] + k);
                Key key;
                memcpy(&key.a, &pr[0], sizeof(double));
                const double grid = 17592186044416.0;   // 2^44 per bohr
                key.x = llround(pr[1] * grid);
                key.y = llround(pr[2] * grid);
                key.z = llround(pr[3] * grid);
                auto it = at[l].find(key);
                bool same = it != at[l].end();
                if (same)
                    for (int d = 0; d < 3; d++) {
                        const double P = cen[l][it->second].g[1 + d];
                        same = same && std::fabs(P - pr[1 + d]) <= 8 * 2.22e-16 * std::fabs(P);
                    }
                int id = same ? it->second : (int)cen[l].size();
                if (!same) {
                    if (it == at[l].end()) at[l].emplace(key, id);
                    cen[l].push_back(Cen{{pr[0], pr[1], pr[2], pr[3]}});
                }
                J.ecen[J.e_c0[e] + k] = id;   // within its order, for now
            }
        }
    }
    long long nc = 0;
    for (int l = 0; l < JIT_NORD; l++) {
        lc0[l][2 * (size_t)n_node] = (int)cen[l].size();
        J.coff[l] = (int)nc;
        J.hoff[l] = J.nherm;
        nc += (long long)cen[l].size();
        J.nherm += (long long)cen[l].size() * jit_nherm(l);
        if (nc >= INT32_MAX) { set_error(ERR_UNSUPPORTED, "on-the-fly B/D: too many primitives"); return false; }
        for (const Cen &c : cen[l]) J.cgeo.insert(J.cgeo.end(), c.g, c.g + 4);
    }
    J.coff[JIT_NORD] = (int)nc;
    // contributions of every centre, in entry order
    J.cptr.assign((size_t)nc + 1, 0);
    for (size_t e = 0; e < ne; e++) {
        const int b = J.kl_pair[e], l = J.pinfo[4 * b] + J.pinfo[4 * b + 1];
        for (int i = J.e_c0[e]; i < J.e_c0[e + 1]; i++)
            if (J.ecen[i] >= 0) { J.ecen[i] += J.coff[l]; J.cptr[J.ecen[i] + 1]++; }
    }
    for (long long c = 0; c < nc; c++) J.cptr[c + 1] += J.cptr[c];
    J.cent.resize((size_t)J.cptr[nc]);
    J.cprim.resize((size_t)J.cptr[nc]);
    {
        std::vector<int> pos(J.cptr.begin(), J.cptr.end() - 1);
        for (size_t e = 0; e < ne; e++)
            for (int i = J.e_c0[e]; i < J.e_c0[e + 1]; i++)
                if (J.ecen[i] >= 0) {
                    const int q = pos[J.ecen[i]]++;
                    J.cent[q] = (int)e;
                    J.cprim[q] = J.pinfo[4 * J.kl_pair[e] + 3] + (i - J.e_c0[e]);
                }
    }
    auto count = [&](int L, int l) { return lc0[l][L + 1] - lc0[l][L]; };
    // ---- work
    double cost[JIT_NORD][JIT_NORD];   // vector instructions of one pair of centres, roughly
    for (int la = 0; la < JIT_NORD; la++)
        for (int lb = 0; lb < JIT_NORD; lb++) {
            const int LT = la + lb;
            double rec = 0;
            for (int n = 1; n <= LT; n++) rec += jit_nherm(n) - 1;
            cost[la][lb] = (45.0 + (LT > 0 ? 12.0 + 3.0 * LT : 0.0) + 1.4 * rec + (double)jit_nherm(la) * jit_nherm(lb)) *
                           (jit_group(LT) == 2 ? 1.3 : 1.0);
        }
    double total = 0;
    std::vector<double> le(2 * (size_t)n_node), lp(2 * (size_t)n_node, 0.0), lr(2 * (size_t)n_node, 0.0);
    for (int L = 0; L < 2 * n_node; L++) {
        le[L] = J.kl_count[L];
        for (int e = J.kl_start[L]; e < J.kl_start[L] + J.kl_count[L]; e++) {
            lp[L] += J.pinfo[4 * J.kl_pair[e] + 2];
            lr[L] += h->sp_nbfp[J.kl_pair[e]];
        }
    }
    for (const Target &t : targets)
        for (size_t i = 0; i < t.src.size(); i++) {
            const int S = t.src[i];
            J.quartets += le[t.list] * le[S];
            J.prim_quartets += lp[t.list] * lp[S];
            J.eri_values += lr[t.list] * lr[S];
            double c = 0;
            for (int la = 0; la < JIT_NORD; la++)
                for (int lb = 0; lb < JIT_NORD; lb++) c += cost[la][lb] * count(t.list, la) / 64.0 * count(S, lb);
            total += c;
            ((int)i < t.n_near ? J.cost_d : J.cost_b) += c;
        }
    // ---- tasks: the centres of a target in chunks of 64, each against the
    // sources' centres of one order, cut into runs of bounded cost: a wave's
    // share of the pass when 16 waves of every CU take four tasks each, and at
    // least 32 centres per lane (below that the table load and the first
    // loads show)
    const double cap = total / (256.0 * 16 * 4);
    struct TaskRec { JitTask t; double cost; };
    std::vector<TaskRec> recs;
    for (const Target &t : targets)
        for (int la = 0; la < JIT_NORD; la++) {
            const int c0 = J.coff[la] + lc0[la][t.list], c1 = c0 + count(t.list, la);
            std::map<std::pair<int, int>, std::vector<std::pair<int, int>>> cuts;   // (lb, lbw): its runs of segments
            for (int c = c0; c < c1; c += 64) {
                const int n = std::min(64, c1 - c);
                int lbw = 2;
                while ((1 << lbw) < n) lbw++;
                JitChunk ch{la, c, n, lbw, (int)J.ctask.size(), 0};
                const int ns = 64 >> lbw;
                for (int lb = 0; lb < JIT_NORD; lb++) {
                    auto key = std::make_pair(lb, lbw);
                    auto it = cuts.find(key);
                    if (it == cuts.end()) {
                        std::vector<std::pair<int, int>> sg;   // contiguous sources joined
                        long long tot = 0;
                        for (int S : t.src) {
                            const int k0 = J.coff[lb] + lc0[lb][S], k1 = k0 + count(S, lb);
                            if (k0 == k1) continue;
                            tot += k1 - k0;
                            if (!sg.empty() && sg.back().second == k0) sg.back().second = k1;
                            else sg.push_back({k0, k1});
                        }
                        std::vector<std::pair<int, int>> runs;
                        const long long per_min = 32LL * ns;
                        long long per = std::max((long long)(cap / cost[la][lb]) * ns, per_min);
                        const long long nrun = std::max(1LL, (tot + per - 1) / per);
                        per = (tot + nrun - 1) / nrun;
                        per = (per + ns - 1) / ns * ns;
                        long long left = per;
                        int s0 = (int)J.segs.size() / 2;
                        for (auto s : sg)
                            while (s.first < s.second) {
                                const int take = (int)std::min<long long>(left, s.second - s.first);
                                J.segs.push_back(s.first);
                                J.segs.push_back(s.first + take);
                                s.first += take;
                                left -= take;
                                if (left == 0) {
                                    runs.push_back({s0, (int)J.segs.size() / 2});
                                    s0 = (int)J.segs.size() / 2;
                                    left = per;
                                }
                            }
                        if (s0 < (int)J.segs.size() / 2) runs.push_back({s0, (int)J.segs.size() / 2});
                        it = cuts.emplace(key, runs).first;
                    }
                    for (const auto &r : it->second) {
                        double iters = 0;
                        for (int s = r.first; s < r.second; s++) iters += (J.segs[2 * s + 1] - J.segs[2 * s] + ns - 1) / ns;
                        J.ctask.push_back((int)recs.size());
                        recs.push_back(TaskRec{JitTask{la * JIT_NORD + lb, c, n, lbw, r.first, r.second, J.npart}, iters * cost[la][lb]});
                        J.npart += (long long)jit_nherm(la) << lbw;
                    }
                }
                ch.t1 = (int)J.ctask.size();
                J.chunks.push_back(ch);
            }
        }
    J.ntask = (int)recs.size();
    // workgroups of four tasks of one class, longest first within each launch
    std::vector<int> by(recs.size());
    std::iota(by.begin(), by.end(), 0);
    std::stable_sort(by.begin(), by.end(), [&](int x, int y) {
        if (recs[x].t.cls != recs[y].t.cls) return recs[x].t.cls < recs[y].t.cls;
        return recs[x].cost > recs[y].cost;
    });
    struct Wg { int first, n, group; double cost; };
    std::vector<Wg> wgs;
    for (size_t i = 0; i < by.size();) {
        size_t e = i;
        const int cls = recs[by[i]].t.cls;
        while (e < by.size() && e - i < (size_t)JIT_WPG && recs[by[e]].t.cls == cls) e++;
        wgs.push_back(Wg{(int)i, (int)(e - i), jit_group(cls / JIT_NORD + cls % JIT_NORD), recs[by[i]].cost});
        i = e;
    }
    std::stable_sort(wgs.begin(), wgs.end(), [](const Wg &x, const Wg &y) {
        return x.group != y.group ? x.group < y.group : x.cost > y.cost;
    });
    std::vector<int> newid(recs.size());
    for (const Wg &w : wgs) {
        for (int k = 0; k < JIT_WPG; k++) {
            JitTask t = recs[by[w.first + std::min(k, w.n - 1)]].t;
            if (k < w.n) newid[by[w.first + k]] = (int)J.tasks.size();
            else t.n = 0;
            J.tasks.push_back(t);
        }
        J.gtask[w.group + 1] = (int)J.tasks.size();
    }
    for (int g = 0; g < 3; g++) J.gtask[g + 1] = std::max(J.gtask[g + 1], J.gtask[g]);
    for (int &t : J.ctask) t = newid[t];
    for (int t : J.ctask) J.cpoff.push_back(J.tasks[t].poff);
    // ---- entries with output rows, by class, longest first
    for (const Target &t : targets)
        for (int e = J.kl_start[t.list]; e < J.kl_start[t.list] + J.kl_count[t.list]; e++) J.oent.push_back(e);
    std::stable_sort(J.oent.begin(), J.oent.end(), [&](int x, int y) {
        const int *a = &J.pinfo[4 * J.kl_pair[x]], *b = &J.pinfo[4 * J.kl_pair[y]];
        if (a[0] * 3 + a[1] != b[0] * 3 + b[1]) return a[0] * 3 + a[1] < b[0] * 3 + b[1];
        return a[2] > b[2];
    });
    // ---- every index within its array
    const long long space = (long long)N + J.nY;
    for (int k : J.kmap)
        if (k < -1 || k >= space) { set_error(ERR_ARG, "on-the-fly B/D: row index %d out of range", k); return false; }
    for (int k : J.uin)
        if (k < 0 || k >= space) { set_error(ERR_ARG, "on-the-fly B/D: sweep index %d out of range", k); return false; }
    for (size_t e = 0; e < ne; e++)
        if (J.kl_pair[e] < 0 || J.kl_pair[e] >= np || J.kl_moff[e] + h->sp_nbfp[J.kl_pair[e]] > (long long)J.kmap.size()) {
            set_error(ERR_ARG, "on-the-fly B/D: partner entry %zu out of range", e);
            return false;
        }
    for (int i = 0; i < np; i++)
        if ((size_t)(J.pinfo[4 * i + 3] + J.pinfo[4 * i + 2]) * 6 > J.prim.size()) {
            set_error(ERR_ARG, "on-the-fly B/D: primitives of pair %d out of range", i);
            return false;
        }
    for (const JitTask &t : J.tasks) {
        const int la = t.cls / JIT_NORD, lb = t.cls % JIT_NORD;
        bool ok = t.cls >= 0 && la < JIT_NORD && t.n >= 0 && t.n <= (1 << t.lbw) && t.lbw <= 6 && t.c0 >= J.coff[la] &&
                  t.c0 + t.n <= J.coff[la + 1] && t.s0 >= 0 && t.s1 * 2 <= (int)J.segs.size() &&
                  t.poff + ((long long)jit_nherm(la) << t.lbw) <= J.npart;
        for (int s = t.s0; ok && s < t.s1; s++)
            ok = J.segs[2 * s] >= J.coff[lb] && J.segs[2 * s] <= J.segs[2 * s + 1] && J.segs[2 * s + 1] <= J.coff[lb + 1];
        if (!ok) { set_error(ERR_ARG, "on-the-fly B/D: task out of range"); return false; }
    }
    for (const JitChunk &c : J.chunks) {
        bool ok = c.t0 >= 0 && c.t0 <= c.t1 && c.t1 <= (int)J.ctask.size() && c.c0 >= J.coff[c.la] && c.c0 + c.n <= J.coff[c.la + 1];
        for (int k = c.t0; ok && k < c.t1; k++)
            ok = J.ctask[k] >= 0 && J.ctask[k] < (int)J.tasks.size() && J.tasks[J.ctask[k]].c0 == c.c0 && J.tasks[J.ctask[k]].lbw == c.lbw;
        if (!ok) { set_error(ERR_ARG, "on-the-fly B/D: chunk out of range"); return false; }
    }
    for (int e : J.oent)
        for (int i = J.e_c0[e]; i < J.e_c0[e + 1]; i++) {
            const int l = J.pinfo[4 * J.kl_pair[e]] + J.pinfo[4 * J.kl_pair[e] + 1];
            if (J.ecen[i] < J.coff[l] || J.ecen[i] >= J.coff[l + 1]) { set_error(ERR_ARG, "on-the-fly B/D: centre out of range"); return false; }
        }
    jit_boys_tables(J.boys);
    return true;
}

// ---------------------------------------------------------------------------
// Device state
// ---------------------------------------------------------------------------
struct JitState {
    JitPlan P;
    bool ready = false;
    int *d_ints = nullptr;      // every int array, one allocation
    double *d_dbls = nullptr;   // pgeo, prim, Boys tables, centres, U
    long long *d_uoff = nullptr;
    JitTask *d_tasks = nullptr;
    JitChunk *d_chunks = nullptr;
    double *Y0 = nullptr, *Y1 = nullptr, *YJ = nullptr, *YD = nullptr, *part = nullptr, *HV = nullptr;
    JitView view{};
    const int *d_unr = nullptr, *d_unc = nullptr, *d_uin0 = nullptr, *d_y0off = nullptr, *d_uin = nullptr;
    const double *d_U = nullptr;
    // work items per level: (node, first column) up, (node, first row) down
    std::vector<const int *> d_up, d_down;
    std::vector<int> n_up, n_down;
    size_t bytes = 0;   // device memory held
    std::vector<hipEvent_t> ev;   // phase timing: 6 per vector
};

#define JIT_HIP(expr)                                                                                       \
    do {                                                                                                    \
        hipError_t e_ = (expr);                                                                             \
        if (e_ != hipSuccess) {                                                                             \
            set_error(ERR_DEVICE, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
            return false;                                                                                   \
        }                                                                                                   \
    } while (0)

void jit_release(JitState *&js) {
    if (!js) return;
    for (hipEvent_t e : js->ev) (void)hipEventDestroy(e);
    void *ps[] = {js->d_ints, js->d_dbls, js->d_uoff, js->d_tasks, js->d_chunks, js->Y0, js->Y1, js->part, js->HV};
    for (void *p : ps)
        if (p) (void)hipFree(p);
    delete js;
    js = nullptr;
}

size_t jit_resident_bytes(const JitState *js) { return js ? js->bytes : 0; }

// The plan's scalars and, at the given array bases, its pointers.
static void jit_view_counts(const JitPlan &P, JitView &v) {
    v.N = P.N;
    v.ncen = P.coff[JIT_NORD];
    v.nent = (int)P.kl_pair.size();
    for (int l = 0; l <= JIT_NORD; l++) v.coff[l] = P.coff[l];
    for (int l = 0; l < JIT_NORD; l++) v.hoff[l] = P.hoff[l];
}

bool jit_upload(H2ERI_p h, JitState *&js) {
    if (js && js->ready) return true;
    jit_release(js);
    js = new JitState();
    JitPlan &P = js->P;
    if (!jit_plan(h, P)) { jit_release(js); return false; }
    // int arrays, concatenated
    std::vector<const std::vector<int> *> iv = {&P.pinfo, &P.kl_pair, &P.kl_moff, &P.kmap, &P.e_c0, &P.ecen,
                                                &P.cptr, &P.cent, &P.cprim, &P.segs, &P.oent,
                                                &P.unr, &P.unc, &P.uin0, &P.y0off, &P.uin};
    std::vector<int> ints;
    std::vector<size_t> ioff;
    for (auto *v : iv) { ioff.push_back(ints.size()); ints.insert(ints.end(), v->begin(), v->end()); }
    std::vector<size_t> up_off, down_off;
    for (auto &l : P.level_nodes) {
        up_off.push_back(ints.size());
        for (int n : l)
            for (int c = 0; c < P.unc[n]; c += 64) { ints.push_back(n); ints.push_back(c); }
        down_off.push_back(ints.size());
        for (int n : l)
            for (int r = 0; r < P.unr[n]; r += JIT_DROWS) { ints.push_back(n); ints.push_back(r); }
        js->n_up.push_back((int)(down_off.back() - up_off.back()) / 2);
        js->n_down.push_back((int)(ints.size() - down_off.back()) / 2);
    }
    ints.push_back(0);
    std::vector<double> dbls;
    auto put = [&](const std::vector<double> &a) {
        dbls.resize((dbls.size() + 31) & ~(size_t)31, 0.0);   // 256-byte starts
        const size_t o = dbls.size();
        dbls.insert(dbls.end(), a.begin(), a.end());
        return o;
    };
    const size_t o_geo = put(P.pgeo), o_prim = put(P.prim), o_boys = put(P.boys), o_cen = put(P.cgeo), o_U = put(P.U);
    dbls.push_back(0.0);
    JIT_HIP(hipMalloc(&js->d_ints, ints.size() * sizeof(int)));
    JIT_HIP(hipMemcpy(js->d_ints, ints.data(), ints.size() * sizeof(int), hipMemcpyHostToDevice));
    JIT_HIP(hipMalloc(&js->d_dbls, dbls.size() * sizeof(double)));
    JIT_HIP(hipMemcpy(js->d_dbls, dbls.data(), dbls.size() * sizeof(double), hipMemcpyHostToDevice));
    std::vector<long long> lls(P.uoff);   // U offsets, then the partials' offsets
    lls.insert(lls.end(), P.cpoff.begin(), P.cpoff.end());
    lls.push_back(0);
    JIT_HIP(hipMalloc(&js->d_uoff, lls.size() * sizeof(long long)));
    JIT_HIP(hipMemcpy(js->d_uoff, lls.data(), lls.size() * sizeof(long long), hipMemcpyHostToDevice));
    JIT_HIP(hipMalloc(&js->d_tasks, (P.tasks.size() + 1) * sizeof(JitTask)));
    JIT_HIP(hipMemcpy(js->d_tasks, P.tasks.data(), P.tasks.size() * sizeof(JitTask), hipMemcpyHostToDevice));
    JIT_HIP(hipMalloc(&js->d_chunks, (P.chunks.size() + 1) * sizeof(JitChunk)));
    JIT_HIP(hipMemcpy(js->d_chunks, P.chunks.data(), P.chunks.size() * sizeof(JitChunk), hipMemcpyHostToDevice));
    const size_t ny = (size_t)std::max(P.nY, 1), nn = (size_t)std::max(P.N, 1), nh = (size_t)P.nherm + 1;
    JIT_HIP(hipMalloc(&js->Y0, ny * sizeof(double)));
    JIT_HIP(hipMalloc(&js->Y1, (ny + 2 * nn) * sizeof(double)));   // Y1, YJ, YD: cleared together
    js->YJ = js->Y1 + ny;
    js->YD = js->YJ + nn;
    JIT_HIP(hipMalloc(&js->HV, 2 * nh * sizeof(double)));
    JIT_HIP(hipMalloc(&js->part, ((size_t)P.npart + 1) * sizeof(double)));
    js->bytes = ints.size() * sizeof(int) + dbls.size() * sizeof(double) + lls.size() * sizeof(long long) +
                P.tasks.size() * sizeof(JitTask) + P.chunks.size() * sizeof(JitChunk) +
                (2 * ny + 2 * nn + 2 * nh + (size_t)P.npart) * sizeof(double);
    const int *I = js->d_ints;
    JitView &v = js->view;
    jit_view_counts(P, v);
    v.pinfo = I + ioff[0];
    v.kl_pair = I + ioff[1];
    v.kl_moff = I + ioff[2];
    v.kmap = I + ioff[3];
    v.e_c0 = I + ioff[4];
    v.ecen = I + ioff[5];
    v.cptr = I + ioff[6];
    v.cent = I + ioff[7];
    v.cprim = I + ioff[8];
    v.segs = I + ioff[9];
    v.oent = I + ioff[10];
    js->d_unr = I + ioff[11];
    js->d_unc = I + ioff[12];
    js->d_uin0 = I + ioff[13];
    js->d_y0off = I + ioff[14];
    js->d_uin = I + ioff[15];
    v.cpoff = js->d_uoff + P.uoff.size();
    for (size_t o : up_off) js->d_up.push_back(I + o);
    for (size_t o : down_off) js->d_down.push_back(I + o);
    v.pgeo = js->d_dbls + o_geo;
    v.prim = js->d_dbls + o_prim;
    v.boys = js->d_dbls + o_boys;
    v.cgeo = js->d_dbls + o_cen;
    js->d_U = js->d_dbls + o_U;
    v.H = js->HV;
    v.V = js->HV + nh;
    v.tasks = js->d_tasks;
    v.chunks = js->d_chunks;
    v.part = js->part;
    v.Y0 = js->Y0;
    v.Y1 = js->Y1;
    v.YJ = js->YJ;
    js->ready = true;
    return true;
}

template <int G>
static void jit_launch_potential(const JitPlan &P, const JitView &v, hipStream_t s) {
    const int t0 = P.gtask[G], nwg = (P.gtask[G + 1] - t0) / JIT_WPG;
    if (nwg > 0)
        hipLaunchKernelGGL(jit_potential_kernel<G>, dim3(nwg), dim3(64 * JIT_WPG), 0, s, v, v.tasks + t0, v.cgeo, v.H, v.segs, v.boys);
}

bool jit_matvec(H2ERI_p h, JitState *js, int nvec, const double *X, double *Y, void *stream, double *ms5) {
    if (!js || !js->ready) { set_error(ERR_ARG, "on-the-fly B/D: not uploaded"); return false; }
    hipStream_t s = (hipStream_t)stream;
    const JitPlan &P = js->P;
    const int N = P.N;
    if (ms5)
        while (js->ev.size() < 6 * (size_t)nvec) {
            hipEvent_t e;
            JIT_HIP(hipEventCreate(&e));
            js->ev.push_back(e);
        }
    auto mark = [&](int k, int i) -> bool {
        if (ms5) JIT_HIP(hipEventRecord(js->ev[6 * k + i], s));
        return true;
    };
    for (int k = 0; k < nvec; k++) {
        const double *x = X + (size_t)k * N;
        double *y = Y + (size_t)k * N;
        if (!mark(k, 0)) return false;
        const long long nz = (long long)std::max(P.nY, 1) + 2LL * std::max(N, 1);   // Y1, YJ, YD
        hipLaunchKernelGGL(jit_zero_kernel, dim3((unsigned)std::min<long long>(1024, (nz + 255) / 256)), dim3(256), 0, s, js->Y1, nz);
        JIT_HIP(hipGetLastError());
        if (!mark(k, 1)) return false;
        for (int L = P.max_level; L >= 0; L--) {
            if (js->n_up[L] == 0) continue;
            hipLaunchKernelGGL(jit_up_kernel, dim3(js->n_up[L]), dim3(1024), 0, s, js->d_up[L], js->d_uoff, js->d_unr,
                               js->d_unc, js->d_uin0, js->d_y0off, js->d_uin, js->d_U, x, js->Y0, N);
            JIT_HIP(hipGetLastError());
        }
        if (!mark(k, 2)) return false;
        JitView v = js->view;
        v.X = x;
        unsigned ndens = 0;
        for (int l = 0; l < JIT_NORD; l++) ndens += (unsigned)(P.coff[l + 1] - P.coff[l] + 255) / 256;
        if (ndens > 0) hipLaunchKernelGGL(jit_density_kernel, dim3(ndens), dim3(256), 0, s, v);
        JIT_HIP(hipGetLastError());
        jit_launch_potential<2>(P, v, s);
        jit_launch_potential<1>(P, v, s);
        jit_launch_potential<0>(P, v, s);
        JIT_HIP(hipGetLastError());
        if (!P.chunks.empty()) hipLaunchKernelGGL(jit_reduce_kernel, dim3((unsigned)P.chunks.size()), dim3(256), 0, s, v);
        const int nout = (int)P.oent.size();
        if (nout > 0)
            hipLaunchKernelGGL(jit_rows_kernel, dim3((unsigned)(((long long)nout * JIT_RLANES + 255) / 256)), dim3(256), 0, s, v, nout);
        JIT_HIP(hipGetLastError());
        if (!mark(k, 3)) return false;
        for (int L = 0; L <= P.max_level; L++) {
            if (js->n_down[L] == 0) continue;
            hipLaunchKernelGGL(jit_down_kernel, dim3(js->n_down[L]), dim3(256), 0, s, js->d_down[L], js->d_uoff, js->d_unr,
                               js->d_unc, js->d_uin0, js->d_y0off, js->d_uin, js->d_U, js->YD, js->Y1, N);
            JIT_HIP(hipGetLastError());
        }
        if (!mark(k, 4)) return false;
        hipLaunchKernelGGL(jit_add_kernel, dim3((N + 255) / 256), dim3(256), 0, s, js->YD, js->YJ, y, N);
        JIT_HIP(hipGetLastError());
        if (!mark(k, 5)) return false;
    }
    if (ms5) {   // per phase: up sweep, B and D tasks (split by planned cost), down sweep, vector work
        JIT_HIP(hipEventSynchronize(js->ev[6 * (size_t)nvec - 1]));
        const double fb = P.cost_b + P.cost_d > 0 ? P.cost_b / (P.cost_b + P.cost_d) : 0.0;
        for (int k = 0; k < nvec; k++) {
            float t[5];
            for (int i = 0; i < 5; i++) JIT_HIP(hipEventElapsedTime(&t[i], js->ev[6 * k + i], js->ev[6 * k + i + 1]));
            ms5[0] += t[1];
            ms5[1] += t[2] * fb;
            ms5[2] += t[3];
            ms5[3] += t[2] * (1.0 - fb);
            ms5[4] += t[0] + t[4];
        }
    }
    (void)h;
    return true;
}

// ---------------------------------------------------------------------------
// Host emulation (tests)
// ---------------------------------------------------------------------------
template <int LA, int LB>
static void jit_potential_host(const JitView &v, const JitTask &t, const double *bt) {
    constexpr int NA = jit_nherm(LA), NB = jit_nherm(LB);
    const int bw = 1 << t.lbw, ns = 64 >> t.lbw;
    const double *Hb = v.H + v.hoff[LB] - (long long)v.coff[LB] * NB;
    for (int b = 0; b < t.n; b++) {
        const double *bg = v.cgeo + 4 * (size_t)(t.c0 + b);
        std::vector<double> V((size_t)NA * ns, 0.0);
        for (int sg = t.s0; sg < t.s1; sg++)
            for (int sl = 0; sl < ns; sl++)
                for (int j = v.segs[2 * sg] + sl; j < v.segs[2 * sg + 1]; j += ns) {
                    const double *g = v.cgeo + 4 * (size_t)j;
                    jit_pair<LA, LB>(bg[0], bg[1], bg[2], bg[3], g[0], g[1], g[2], g[3], Hb + (long long)j * NB, bt, &V[(size_t)NA * sl]);
                }
        for (int k = 0; k < NA; k++) {
            double s = 0.0;
            for (int sl = 0; sl < ns; sl++) s += V[(size_t)NA * sl + k];
            v.part[t.poff + (long long)k * bw + b] = s;
        }
    }
}
template <int... C>
static void jit_potential_host_any(const JitView &v, const JitTask &t, const double *bt, std::integer_sequence<int, C...>) {
    ([&] { if (t.cls == C) jit_potential_host<C / JIT_NORD, C % JIT_NORD>(v, t, bt); }(), ...);
}
template <int L>
static void jit_density_host(const JitView &v) {
    for (int c = v.coff[L]; c < v.coff[L + 1]; c++) jit_density<L>(v, c);
}

}  // namespace h2e

using namespace h2e;

extern "C" {

// Host execution of the on-the-fly matvec (tests only): the device's
// densities, pair terms and rows on the host, the sweeps as plain loops.
// Returns 0, or -1 with the error set.
int H2ERI_jit_emulate(H2ERI_p h, const double *x, double *y) {
    if (!h || !x || !y) { set_error(ERR_ARG, "jit_emulate: null argument"); return -1; }
    JitPlan P;
    if (!jit_plan(h, P)) return -1;
    const int N = P.N;
    std::vector<double> Y0(std::max(P.nY, 1), 0.0), Y1(std::max(P.nY, 1), 0.0), YJ(N, 0.0), YD(N, 0.0);
    for (int L = P.max_level; L >= 0; L--)
        for (int n : P.level_nodes[L]) {
            const double *Un = P.U.data() + P.uoff[n];
            const int *in = P.uin.data() + P.uin0[n];
            for (int c = 0; c < P.unc[n]; c++) {
                double part[4] = {0, 0, 0, 0};
                for (int r = 0; r < P.unr[n]; r++) {
                    const int k = in[r];
                    part[r & 3] += Un[(size_t)r * P.unc[n] + c] * (k < N ? x[k] : Y0[k - N]);
                }
                Y0[P.y0off[n] + c] = (part[0] + part[1]) + (part[2] + part[3]);
            }
        }
    JitView v{};
    jit_view_counts(P, v);
    v.pinfo = P.pinfo.data(); v.pgeo = P.pgeo.data(); v.prim = P.prim.data(); v.boys = P.boys.data();
    v.kl_pair = P.kl_pair.data(); v.kl_moff = P.kl_moff.data(); v.kmap = P.kmap.data();
    v.e_c0 = P.e_c0.data(); v.ecen = P.ecen.data(); v.cptr = P.cptr.data(); v.cent = P.cent.data(); v.cprim = P.cprim.data();
    v.cgeo = P.cgeo.data(); v.tasks = P.tasks.data(); v.segs = P.segs.data(); v.chunks = P.chunks.data();
    v.cpoff = P.cpoff.data(); v.oent = P.oent.data();
    std::vector<double> part((size_t)P.npart + 1, 0.0), HV(2 * (size_t)P.nherm + 2, 0.0);
    v.part = part.data();
    v.H = HV.data();
    v.V = HV.data() + P.nherm + 1;
    v.X = x; v.Y0 = Y0.data(); v.YJ = YJ.data(); v.Y1 = Y1.data();
    jit_density_host<0>(v);
    jit_density_host<1>(v);
    jit_density_host<2>(v);
    jit_density_host<3>(v);
    jit_density_host<4>(v);
    const int ntask = (int)P.tasks.size();
    std::atomic<int> next(0);
    auto worker = [&]() {
        for (int t = next++; t < ntask; t = next++) {
            const JitTask &tk = P.tasks[t];
            if (tk.n == 0) continue;
            const int LT = tk.cls / JIT_NORD + tk.cls % JIT_NORD;
            jit_potential_host_any(v, tk, v.boys + (size_t)LT * JIT_BGRID * JIT_BROW,
                                   std::make_integer_sequence<int, JIT_NORD * JIT_NORD>{});
        }
    };
    const int nth = std::max(1, std::min(16, (int)std::thread::hardware_concurrency()));
    std::vector<std::thread> pool;
    for (int i = 1; i < nth; i++) pool.emplace_back(worker);
    worker();
    for (auto &th : pool) th.join();
    for (const JitChunk &c : P.chunks) jit_reduce(v, c, 0, 1);
    for (int e : P.oent) jit_rows_any<1>(v, e, 0);
    for (int L = 0; L <= P.max_level; L++)
        for (int n : P.level_nodes[L]) {
            const double *Un = P.U.data() + P.uoff[n];
            const int *out = P.uin.data() + P.uin0[n];
            for (int r = 0; r < P.unr[n]; r++) {
                double s = 0.0;
                for (int c = 0; c < P.unc[n]; c++) s += Un[(size_t)r * P.unc[n] + c] * Y1[P.y0off[n] + c];
                const int k = out[r];
                if (k < N) YD[k] = s;
                else Y1[k - N] += s;
            }
        }
    for (int i = 0; i < N; i++) y[i] = YD[i] + YJ[i];
    return 0;
}

// Work of one on-the-fly matvec: out4 = {tasks, shell quartets, primitive
// quartets, integral values}, each block counted from both sides.  Host only.
// Returns 0 or -1.
int H2ERI_jit_stats(H2ERI_p h, double *out4) {
    if (!h || !out4) { set_error(ERR_ARG, "jit_stats: null argument"); return -1; }
    JitPlan P;
    if (!jit_plan(h, P)) return -1;
    out4[0] = (double)P.ntask;
    out4[1] = P.quartets;
    out4[2] = P.prim_quartets;
    out4[3] = P.eri_values;
    return 0;
}

// B and D blocks stored dense (on = 0) or compressed to [U | V^T] where it
// pays (on = 1, the default), from the next H2ERI_build_H2 on.
void H2ERI_set_block_compression(H2ERI_p h, const int on) {
    if (!h) { set_error(ERR_ARG, "set_block_compression: null handle"); return; }
    host_state(h)->bd_dense = on == 0;
}

}  // extern "C"
