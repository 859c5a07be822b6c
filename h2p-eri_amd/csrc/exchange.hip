// Exchange matrix through the H2 representation on the MI355X:
//
//   K_mq = sum_{n,p} (mn|pq) D_np            (src/H2ERI_build_exchange.c:1356-1450)
//
// The reference evaluates K with partial multi-column H2 products, one per
// (N,Q) shell pair (:1021-1353), with gathered inputs (:609-688) and an atomic
// scatter of the outputs into K (:691-771).  This device version evaluates
// the same sum block by block of A_H2 instead:
//
//   A_H2 = sum_i D_ii + sum_{(i,j)} [F_ij + F_ij^T],   F_ij = L_ij R_ij^T
//
// - diagonal near-field blocks are applied once;
// - every reduced admissible (B) or inadmissible (D) pair is applied with its
//   transpose (src/H2ERI_matvec.c:299-407,572-660).
// L and R come from the expanded nested bases (P_n = U of a leaf, or
// blockdiag(P of children) U of an inner node) and the block's core (dense C,
// or U V^T for a low-rank block), as listed at build_terms.
//
// Row x of A_H2 is the basis-function pair (a_x, b_x) of a screened shell
// pair, stored with the smaller shell first.  When the two shells differ,
// the row stands for both (ab| and (ba|; a same-shell pair has one row per
// ordered (a,b).  For a term with rows in node i and columns in node j, the
// contraction factorises through the basis-function sets B(i), B(j) of the
// two nodes:
//
//   G[n][t][q] = sum_{c in j, (p,q) orientation of c} R[c][t] D[n][p]   (ket, n in B(i), q in B(j))
//   K[m][q]   += sum_{r in i, (m,n) orientation of r} sum_t L[r][t] G[n][t][q]   (bra)
//
// For big nodes this costs kk (|B(i)| m_j + m_i |B(j)|) rather than the
// m_i m_j kk of forming F.  Dense near-field blocks are contracted directly.
//
// Accumulation and symmetry:
// - For symmetric D the transpose terms give the transpose of the F terms:
//   K = K1 + K1^T + K_diag.
// - Contributions go into K1 and K_diag with FP64 atomic adds, as the
//   reference's scatter does (:767), so the last bits of K depend on the
//   order of the adds.
// - The L and R products of the cores, the ket and the bra are FP64 MFMA
//   tiles (v_mfma_f64_16x16x4f64) with FP64 accumulation.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <numeric>
#include <type_traits>

#include "h2eri_internal.h"

namespace h2e {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

enum KSrc { KS_PB = 0, KS_CB = 1, KS_SC = 2 };

struct KTerm {
    int direct;           // 1: dense core contracted directly (identity bases on both sides)
    int diag;             // 1: diagonal near-field block (into K_diag), 0: into K1
    int ni, nj;           // node-list ids of the row and column ranges
    int m0, m1, kk;
    int Lsrc, Lld;        // L[r][t] = src[Loff + r*Lld + t]   (direct: C[r][c] = src[Loff + r*Lld + c])
    long long Loff;
    int Rsrc, Rrs, Rcs;   // R[c][t] = src[Roff + c*Rrs + t*Rcs]
    long long Roff;
};

struct KGemm {           // out (m x n, ld ldo) = A (m x k, PB, ld lda) * X (k x n, CB, ld ldx)
    long long Aoff, Xoff, Ooff;
    int m, n, k, lda, ldx, ldo;
};

struct KTask {           // one workgroup: term and tile origin
    int term;
    int e0;               // block: first column slot; direct: first (m,q) index
    int t0;               // block: split of local m
    int pad_;
};

struct KGemmTask {
    int g, row0, col0, pad_;
};

struct KNode {           // per row/column range: basis-function set and the orientation lists
    int bf_off, nbf;      // B(node) = bfidx[bf_off .. bf_off + nbf)
    int q_ptr;            // byQ CSR rows: qptr[q_ptr .. q_ptr + nbf]   entries (column c, p)
    int m_ptr;            // byM CSR rows: mptr[m_ptr .. m_ptr + nbf]   entries (row r, local n)
    int g_ptr;            // merged lists of pairs of column slots: gptr[g_ptr + 2 g]   entries (p, columns c of the two),
                          // gptr[g_ptr + 2 g + 1] of their fours (the first ones) have every entry in both
    int c_off, ngrp;      // functions q of the 2 ngrp column slots: bfidx[c_off + slot] (-1: none)
    int b_ptr;            // bra block lists: bptr[b_ptr + ((split * steps of 16 n) + step) * 8 + wave], and the next one
    int nsplit;           // splits of the functions m
    int ssz;              // functions m per split: the nbf functions in nsplit = ceil(nbf / KM) even parts
};

static const int KWG = 256;
// Workgroups are dispatched to the 8 XCDs round-robin by id, and each XCD has
// its own L2.  This bijection of [0, n) hands out runs of C consecutive tasks
// of the list, run j to XCD j mod 8 (the tail of fewer than 8 runs is split
// into 8 contiguous ranges), so tasks next to each other in the list, which
// share L rows and D, read them through one L2.
__device__ inline int xcd_task(int bid, int n, int C) {
    const int full = n / (8 * C);
    const int x = bid & 7, k = bid >> 3;
    if (bid < full * 8 * C) return ((k / C) * 8 + x) * C + k % C;
    const int n2 = n - full * 8 * C, k2 = (bid - full * 8 * C) >> 3, q = n2 >> 3, r = n2 & 7;
    return full * 8 * C + x * q + min(x, r) + k2;
}
static const int KRUN = 8;      // consecutive tasks per XCD
static const int KQ = 16;       // column slots q per task (eight pairs)
static const int KNQ = 8;      // fours of a pair's entries whose R operands stay in registers
static const int KGN = 258;     // doubles per function n of the G tile (16 t x 16 q, and two that shift the LDS banks)
static const int KGT = 16 * KGN;
static const int KBWG = 512;    // threads of a block task (8 waves)
static const int KPAD = 32;     // readable doubles past every operand array
// Most local functions m of a task (its K block in LDS): 352, the G tile and
// the node's function offsets take 79,616 bytes, two workgroups per CU; the
// functions of a larger node are cut into even splits, each of which forms
// its G again.
static const int KM = 352;
static const int KNMAX = 4096;  // most functions of a row node whose list is in LDS (the 32-bit form)
// LDS of a block task: G tile, K block and, in the 32-bit form, the row node's
// functions
static size_t kblock_lds(int m, int n, bool wide) { return (size_t)(KGT + (m + 1) * KQ) * 8 + (wide ? 0 : (size_t)n * 4); }
// A bra entry: row r, and the byte of m's row in the K block (16 bits; the row
// past the last is a sink for rows of a block without an entry) under local n
// (4 bits) and flags of the block.
static const int KMORE = 16;          // the wave's next block is of the same functions m
static const int KFIRST = 32;         // the block before is not
static const int KEMPTY = 64;         // no entry at all
static const int KCHAIN = 3;          // most blocks in a row of the same m

// Operand addresses are a uniform base and a byte offset O per lane: 32 bits,
// or 64 where an operand array of a term or D is larger than 4 GB (or a node
// has more functions than the LDS should list).
struct __attribute__((packed, aligned(8))) KU2 { double x, y; };   // 16 bytes at 8-byte alignment
template <typename O>
__device__ __forceinline__ void kload4(const double *p, O byte, double (&o)[4]) {
    const KU2 *q = reinterpret_cast<const KU2 *>(reinterpret_cast<const char *>(p) + byte);
    const KU2 a = q[0], b = q[1];
    o[0] = a.x; o[1] = a.y; o[2] = b.x; o[3] = b.y;
}
template <typename O>
__device__ __forceinline__ double kload(const double *p, O byte) {
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(p) + byte);
}

static const int KNS = 2;       // fours read at a time past them

// byte offset of a row: 24-bit factors (checked on the host) in the 32-bit form
__device__ __forceinline__ unsigned krow(int r, unsigned ld) { return __umul24(r, ld); }
__device__ __forceinline__ unsigned long long krow(int r, unsigned long long ld) { return (unsigned long long)r * ld; }

// f(integral constant of min(n, KNQ)): straight-line code for every length
template <typename F>
__device__ __forceinline__ void kfours(int n, F f) {
    switch (min(n, KNQ)) {
    case 0: break;
    case 1: f(std::integral_constant<int, 1>()); break;
    case 2: f(std::integral_constant<int, 2>()); break;
    case 3: f(std::integral_constant<int, 3>()); break;
    case 4: f(std::integral_constant<int, 4>()); break;
    case 5: f(std::integral_constant<int, 5>()); break;
    case 6: f(std::integral_constant<int, 6>()); break;
    case 7: f(std::integral_constant<int, 7>()); break;
    default: f(std::integral_constant<int, KNQ>()); break;
    }
}

// One block term's share of K: a workgroup takes 16 column slots q of the
// column node and a split of the row node's functions m, and walks the inner
// index t in steps of 16 and, for each, the functions n of the row node in
// steps of 16:
//   ket  G[n][t][q] = sum over the entries (c, p) of q of R[c][t] D[p][n]
//        into LDS: a wave takes two q, one MFMA tile (16 t x 16 n) each.  The
//        two entry lists are merged on p, so that one D operand serves both;
//        an entry a function does not have meets a zero D operand.  D is
//        symmetric (the entry point's contract): D[p][n] lets the 16 lanes of
//        an entry read along a row.  The R operands of the first 32 entries
//        stay in registers over all steps of n: a step loads one D operand
//        per two MFMAs.  Entries past them are read again in every step.
//   bra  K[m][q] += sum over the entries (r, m) of n of L[r][t] G[n][t][q]:
//        the entries of every n in blocks of 16 rows, dealt to the waves; the
//        functions n of a shell have the same m, so up to three of them add
//        up in one tile, which is added into the K block in LDS with FP64 LDS
//        atomics (tiles of different shells may share an m).  Its operands are one
//        stream over all steps: the next two blocks' rows are in flight, across
//        the barriers too, and their indices two further ahead.
// At the end the K block is added into K with FP64 global atomics.
//
// What bounds it: FP64 MFMA issue together with VALU issue, which it does not
// overlap: an MFMA takes 64 cycles of its SIMD, at most 62 TFLOP/s on this
// card, and every VALU instruction beside it adds about two (twelve per MFMA:
// 44 TFLOP/s).  C30H62 issues 189 GFLOP of MFMAs, half of them padding (the
// entries of an n come in sixteens, those of a q in fours): 3.05 ms of the
// 5.15, the MFMA units busy in 48% of the cycles.  (H2O)64, whose ranks of
// about 13 fill a step of 16 t badly, issues 1,073 GFLOP for 460: 42% of its
// 33.3 ms.
// So the loops are kept short of VALU work: fours that both functions have
// meet their D operands unmasked, rows without an entry add into a sink
// instead of being masked, K block bytes and flags are in the lists.  Masks,
// index arithmetic and register copies in the loops: 5.50 ms.
// What is left beside it, from timing builds of the 5.50 ms form: a wave waits
// at a step's two barriers for the one with most work (0.6 ms), the loads of a
// new t (0.2) and the LDS atomics (0.15).  Operand latency is covered there:
// rows padded to whole 128-byte lines
// (5.55 ms), a second block in flight (5.52) and the next step's D in
// registers (5.63) changed nothing or cost.  16 waves per CU (128 VGPRs, two
// workgroups by LDS): 40 entries in registers spill (5.86 ms against 5.64).
// K per build with G in HBM between two kernels / G in LDS, R read in every
// step of n and neighbouring functions paired in order / R in registers and
// balanced slots / this one: C10H22 2.77 / 1.52 / 1.16 / 1.08 ms, C30H62
// 13.1 / 7.37 / 5.64 / 5.15 ms.
template <typename O>
__global__ __launch_bounds__(KBWG, 4) void kx_block(const KTask *__restrict__ tasks, const KTerm *__restrict__ terms,
                                                    const KNode *__restrict__ nodes, const int *__restrict__ bfidx,
                                                    const int *__restrict__ gptr, const int4 *__restrict__ ge,
                                                    const int *__restrict__ bptr, const int2 *__restrict__ brow,
                                                    const double *__restrict__ PB, const double *__restrict__ CB,
                                                    const double *__restrict__ SC, const double *__restrict__ D,
                                                    double *__restrict__ KA, int nacc, int nbf) {
    extern __shared__ double lds[];
    const KTask tk = tasks[xcd_task(blockIdx.x, gridDim.x, KRUN)];   // term, first q, split
    const KTerm t = terms[tk.term];
    const KNode ni = nodes[t.ni], nj = nodes[t.nj];
    double *Gt = lds, *Kb = lds + KGT;
    int *nof = reinterpret_cast<int *>(Kb + (ni.ssz + 1) * KQ);   // function of every local n (32-bit form)
    const int q0 = tk.e0, split = tk.t0, ml0 = split * ni.ssz;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int l16 = lane & 15, kl = lane >> 4;
    const int mlN = min(ni.ssz, ni.nbf - ml0);
    for (int i = threadIdx.x; i < mlN * KQ; i += KBWG) Kb[i] = 0.0;
    if (sizeof(O) == 4)
        for (int i = threadIdx.x; i < ni.nbf; i += KBWG) nof[i] = bfidx[ni.bf_off + i];
    auto func = [&](int n) { return sizeof(O) == 4 ? nof[n] : bfidx[ni.bf_off + n]; };
    __syncthreads();
    const double *L = (t.Lsrc == KS_PB ? PB : (t.Lsrc == KS_CB ? CB : SC)) + t.Loff;
    const double *R = (t.Rsrc == KS_PB ? PB : (t.Rsrc == KS_CB ? CB : SC)) + t.Roff;
    const int kk = t.kk, nstep = (ni.nbf + 15) >> 4;
    const O Rrs = (O)t.Rrs * 8, Rcs = (O)t.Rcs * 8, Lld = (O)t.Lld * 8, Dld = (O)nbf * 8;

    // ---- ket: entries in fours; pairs come longest first, and the waves of
    // one SIMD (w, w + 4) take a long and a short one
    const int grp = (q0 >> 1) + (w < 4 ? w : 11 - w), qw = 2 * (grp - (q0 >> 1));
    const bool gok = grp < nj.ngrp;
    const int *gp = gptr + nj.g_ptr + 2 * grp;
    const int ga = gok ? gp[0] : 0, gs = gok ? (gp[2] - ga) >> 2 : 0, gfull = gok ? gp[1] : 0;
    double ra[KNQ][2];      // R operands of the entries of the two q
    O pd[KNQ];              // rows of D
    unsigned has0 = 0, has1 = 0;   // entry i of the lane's exists for the first / second q
    auto ket_rows = [&](int t0) {   // rows of t past the last repeat it (their G is stored as zero)
        const O to = (O)min(t0 + l16, kk - 1) * Rcs;
        kfours(gs, [&](auto N) {
            int4 x[N];
            #pragma unroll
            for (int i = 0; i < N; i++) x[i] = ge[ga + 4 * i + kl];
            has0 = has1 = 0;
            #pragma unroll
            for (int i = 0; i < N; i++) {
                ra[i][0] = kload(R, (O)max(x[i].x, 0) * Rrs + to);
                ra[i][1] = kload(R, (O)max(x[i].y, 0) * Rrs + to);
                pd[i] = (O)x[i].z * Dld;
                has0 |= x[i].x >= 0 ? 1u << i : 0u;
                has1 |= x[i].y >= 0 ? 1u << i : 0u;
            }
        });
    };
    // ---- bra stream: pairs of blocks of the wave's list of the step, steps, t0.
    // A set of operands is loaded where its last use lies, so that no copy of
    // registers waits for the load.
    const int *bp = bptr + ni.b_ptr + split * nstep * 8 + w;
    int bi = bp[0], be = bp[1], bs = 0, bt = 0, xt = 0;   // position of the rows xr; t of the operands loaded next
    int2 xr[2];                    // rows loaded next (row, local m | (local n | KMORE) << 24)
    int om[2];                     // local m and n of the operands in flight
    double ol[2][4];
    const unsigned xo = l16 * 8;
    auto bra_index = [&](int j) {
        xr[j] = *reinterpret_cast<const int2 *>(reinterpret_cast<const char *>(brow + (long long)(bi + j) * 16) + xo);
    };
    auto bra_load = [&](int j) {
        kload4(L, krow(xr[j].x, Lld) + (O)(xt + 4 * kl) * 8, ol[j]);
        // a copy that keeps xr free for the load below (sharing its register would
        // put a copy that waits for that load at the end of the loop)
        asm volatile("v_mov_b32 %0, %1" : "=v"(om[j]) : "v"(xr[j].y));
        bra_index(j);
    };
    auto bra_next = [&]() {
        xt = bt;
        bi += 2;
        if (bi == be) {
            if (++bs == nstep) {
                bs = 0;
                bt = bt + 16 < kk ? bt + 16 : 0;
            }
            bi = bp[8 * bs];
            be = bp[8 * bs + 1];
        }
    };
    bra_index(0);
    bra_index(1);
    bra_next();
    bra_load(0);
    bra_load(1);

    for (int t0 = 0; t0 < kk; t0 += 16) {
        ket_rows(t0);
        for (int st = 0; st < nstep; st++) {
            const int b0 = bp[8 * st], b1 = bp[8 * st + 1];
            const O no = (O)func(min(16 * st + l16, ni.nbf - 1)) * 8;   // n past the last repeat it (not used)
            d4 acc[2];
            acc[0] = acc[1] = d4{0.0, 0.0, 0.0, 0.0};
            auto ket = [&](auto N, auto same) {
                double d[N];
                #pragma unroll
                for (int i = 0; i < N; i++) d[i] = kload(D, pd[i] + no);
                #pragma unroll
                for (int i = 0; i < N - 1; i++) {
                    acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ra[i][0], same || has0 >> i & 1 ? d[i] : 0.0, acc[0], 0, 0, 0);
                    acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ra[i][1], same || has1 >> i & 1 ? d[i] : 0.0, acc[1], 0, 0, 0);
                }
                acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ra[N - 1][0], has0 >> (N - 1) & 1 ? d[N - 1] : 0.0, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ra[N - 1][1], has1 >> (N - 1) & 1 ? d[N - 1] : 0.0, acc[1], 0, 0, 0);
            };
            if (gfull >= min(gs, KNQ) - 1) kfours(gs, [&](auto N) { ket(N, std::true_type()); });
            else kfours(gs, [&](auto N) { ket(N, std::false_type()); });
            for (int s = KNQ; s < gs; s += KNS) {   // entries past the registers
                const O to = (O)min(t0 + l16, kk - 1) * Rcs;
                int4 x[KNS];
                double a[KNS][2], d[KNS];
                #pragma unroll
                for (int u = 0; u < KNS; u++) {
                    x[u] = ge[ga + 4 * min(s + u, gs - 1) + kl];
                    if (s + u >= gs) x[u].x = x[u].y = -1;
                }
                #pragma unroll
                for (int u = 0; u < KNS; u++) {
                    a[u][0] = kload(R, (O)max(x[u].x, 0) * Rrs + to);
                    a[u][1] = kload(R, (O)max(x[u].y, 0) * Rrs + to);
                    d[u] = kload(D, (O)x[u].z * Dld + no);
                }
                #pragma unroll
                for (int u = 0; u < KNS; u++) {
                    acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][0], x[u].x >= 0 ? d[u] : 0.0, acc[0], 0, 0, 0);
                    acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][1], x[u].y >= 0 ? d[u] : 0.0, acc[1], 0, 0, 0);
                }
            }
            if (t0 + 16 > kk) {   // zero past the last t: what the bra's loads find there does not count
                #pragma unroll
                for (int r = 0; r < 4; r++)
                    if (t0 + kl + 4 * r >= kk) acc[0][r] = acc[1][r] = 0.0;
            }
            #pragma unroll
            for (int r = 0; r < 4; r++)
                *reinterpret_cast<double2 *>(Gt + l16 * KGN + (4 * kl + r) * 16 + qw) = make_double2(acc[0][r], acc[1][r]);
            __syncthreads();
            // MFMA u takes the inner indices t = 4 k + u, which lie at k + 4 u of the
            // G tile: its 64 values are one run of LDS
            d4 x;
            for (int b = b0; b < b1; b += 2) {
                bra_next();
                #pragma unroll
                for (int j = 0; j < 2; j++) {
                    const int nf = __builtin_amdgcn_readfirstlane(om[j]) >> 16;   // local n and flags
                    if (!(nf & KEMPTY)) {
                        const double *g = Gt + (nf & 15) * KGN + lane;
                        if (nf & KFIRST) x = __builtin_amdgcn_mfma_f64_16x16x4f64(ol[j][0], g[0], d4{0.0, 0.0, 0.0, 0.0}, 0, 0, 0);
                        else x = __builtin_amdgcn_mfma_f64_16x16x4f64(ol[j][0], g[0], x, 0, 0, 0);
                        #pragma unroll
                        for (int u = 1; u < 4; u++) x = __builtin_amdgcn_mfma_f64_16x16x4f64(ol[j][u], g[64 * u], x, 0, 0, 0);
                        if (!(nf & KMORE)) {   // else the next block has the same m
                            int m[4];
                            #pragma unroll
                            for (int r = 0; r < 4; r++) m[r] = __shfl(om[j], kl + 4 * r);   // lane e of the wave holds entry e's
                            #pragma unroll
                            for (int r = 0; r < 4; r++)
                                atomicAdd(reinterpret_cast<double *>(reinterpret_cast<char *>(Kb) + ((m[r] & 0xffff) | xo)), x[r]);
                        }
                    }
                    bra_load(j);
                }
            }
            __syncthreads();
        }
    }
    double *Kout = KA + (size_t)nbf * nbf * (2 * (blockIdx.x % nacc) + (t.diag ? 1 : 0));
    for (int i = threadIdx.x; i < mlN * KQ; i += KBWG) {
        const int slot = q0 + (i & (KQ - 1));
        const int q = slot < 2 * nj.ngrp ? bfidx[nj.c_off + slot] : -1;
        const double v = Kb[i];
        if (q >= 0 && v != 0.0) unsafeAtomicAdd(Kout + (size_t)func(ml0 + i / KQ) * nbf + q, v);
    }
}

// Dense core with identity bases: K[m][q] += sum_{(r,n)} sum_{(c,p)} C[r][c] D[n][p].
// One wave per (m, q), its lanes over the (row, column) entry pairs: a
// thread per (m, q) walked up to a thousand dependent gathers (C30H62: 890 us
// for 1 MFLOP).
__global__ __launch_bounds__(KWG) void kx_direct(const KTask *__restrict__ tasks, const KTerm *__restrict__ terms,
                                                  const KNode *__restrict__ nodes, const int *__restrict__ bfidx,
                                                  const int *__restrict__ qptr, const int2 *__restrict__ qent,
                                                  const int *__restrict__ mptr, const int2 *__restrict__ ment,
                                                  const double *__restrict__ CB, const double *__restrict__ D,
                                                  double *__restrict__ KA, int nbf) {
    const KTask tk = tasks[blockIdx.x];
    const KTerm t = terms[tk.term];
    const KNode ni = nodes[t.ni], nj = nodes[t.nj];
    const int e = tk.e0 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (e >= ni.nbf * nj.nbf) return;   // whole wave
    const int ml = e / nj.nbf, ql = e - ml * nj.nbf;
    const double *C = CB + t.Loff;
    const int q0 = qptr[nj.q_ptr + ql], nq = qptr[nj.q_ptr + ql + 1] - q0;
    const int r0 = mptr[ni.m_ptr + ml], nr = mptr[ni.m_ptr + ml + 1] - r0;
    double acc = 0.0;
    for (long long k = lane; k < (long long)nr * nq; k += 64) {
        const int j = (int)(k / nq), i = (int)(k - (long long)j * nq);
        const int2 rn = ment[r0 + j], cp = qent[q0 + i];
        acc = fma(C[(long long)rn.x * t.Lld + cp.x], D[(size_t)bfidx[ni.bf_off + rn.y] * nbf + cp.y], acc);
    }
    for (int d = 32; d > 0; d >>= 1) acc += __shfl_xor(acc, d, 64);
    const int m = bfidx[ni.bf_off + ml], q = bfidx[nj.bf_off + ql];
    if (lane == 0) unsafeAtomicAdd(KA + (t.diag ? (size_t)nbf * nbf : 0) + (size_t)m * nbf + q, acc);
}

// Grouped FP64 GEMM on MFMA: a 64 x 64 output tile per workgroup, wave w owns
// rows [16w, 16w+16) and four 16 x 16 column tiles.  Operand layout of
// v_mfma_f64_16x16x4f64 (checked on gfx950): lane l holds A[l%16][l/16] and
// B[l/16][l%16]; output register r of lane l is C[l/16 + 4r][l%16].
__global__ __launch_bounds__(KWG) void kx_gemm(const KGemmTask *__restrict__ tasks, const KGemm *__restrict__ gemms,
                                                const double *__restrict__ PB, const double *__restrict__ CB,
                                                double *__restrict__ SC) {
    const KGemmTask tk = tasks[blockIdx.x];
    const KGemm g = gemms[tk.g];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ar = tk.row0 + 16 * w + (lane & 15);
    const int kl = lane >> 4;
    const double *A = PB + g.Aoff;
    const double *X = CB + g.Xoff;
    d4 acc[4];
    #pragma unroll
    for (int c = 0; c < 4; c++) acc[c] = d4{0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < g.k; k0 += 4) {
        const int kk = k0 + kl;
        const double a = (ar < g.m && kk < g.k) ? A[(long long)ar * g.lda + kk] : 0.0;
        #pragma unroll
        for (int c = 0; c < 4; c++) {
            const int col = tk.col0 + 16 * c + (lane & 15);
            const double b = (kk < g.k && col < g.n) ? X[(long long)kk * g.ldx + col] : 0.0;
            acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[c], 0, 0, 0);
        }
    }
    #pragma unroll
    for (int c = 0; c < 4; c++) {
        const int col = tk.col0 + 16 * c + (lane & 15);
        #pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = tk.row0 + 16 * w + (lane >> 4) + 4 * r;
            if (row < g.m && col < g.n) SC[g.Ooff + (long long)row * g.ldo + col] = acc[c][r];
        }
    }
}

// Density screening (src/H2ERI_build_exchange.c:774-838): block (N,P) of D
// takes part in K only when some |D_np|, n in N and p in P, exceeds
// DTOL = 1e-10 (:790).  The reference restricts every P list to dlist[N]
// (:410-417,1397-1398), which sums over the kept blocks only; here every
// other block is written as zeros into Ds, the density the kernels read.
// One thread per block; the threads of a row of blocks read consecutive
// columns of the same rows of D.
__global__ void kx_dlist(const int *__restrict__ sbf, int nshell, const double *__restrict__ D, double *__restrict__ Ds,
                         int nbf) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)nshell * nshell) return;
    const int n = (int)(idx / nshell), p = (int)(idx - (long long)n * nshell);
    const int r0 = sbf[n], r1 = sbf[n + 1], c0 = sbf[p], c1 = sbf[p + 1];
    bool keep = false;
    for (int i = r0; i < r1; i++)
        for (int j = c0; j < c1; j++) keep |= fabs(D[(size_t)i * nbf + j]) > 1e-10;
    for (int i = r0; i < r1; i++)
        for (int j = c0; j < c1; j++) Ds[(size_t)i * nbf + j] = keep ? D[(size_t)i * nbf + j] : 0.0;
}

__global__ void kx_zero(double *__restrict__ p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t s = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += s) p[i] = 0.0;
}

// K = K1 + K1^T + K_diag, each summed over its nacc copies in order; 32 x 32
// tiles, K1^T through LDS.
__global__ __launch_bounds__(256) void kx_final(const double *__restrict__ KA, int nacc, double *__restrict__ K, int nbf) {
    __shared__ double tr[32][33];
    const size_t n2 = (size_t)nbf * nbf;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
    for (int k = ty; k < 32; k += 8) {   // the transposed tile: rows c0.., columns r0..
        const int r = c0 + k, c = r0 + tx;
        double s = 0.0;
        if (r < nbf && c < nbf)
            for (int a = 0; a < nacc; a++) s += KA[2 * n2 * a + (size_t)r * nbf + c];
        tr[k][tx] = s;
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
        const int r = r0 + k, c = c0 + tx;
        if (r >= nbf || c >= nbf) continue;
        const size_t i = (size_t)r * nbf + c;
        double s1 = 0.0, sd = 0.0;
        for (int a = 0; a < nacc; a++) { s1 += KA[2 * n2 * a + i]; sd += KA[2 * n2 * a + n2 + i]; }
        K[i] = (s1 + tr[tx][k]) + sd;
    }
}

// ---------------------------------------------------------------------------
// Host plan
// ---------------------------------------------------------------------------
struct KPlan {
    std::vector<double> PB, CB;
    std::vector<KTerm> terms;
    std::vector<KGemm> gemms;
    std::vector<KNode> nodes;
    std::vector<int> bfidx, qptr, mptr, bptr, gptr;
    // bra blocks: 16 (row r, byte of m in the K block | (local n within the step | flags) << 16) each, the
    // last row repeated with the sink's byte past a block's entries
    std::vector<int2> qent, ment, brow;
    std::vector<int4> ge;   // ket entries: columns c of the two q (-1: none), p
    std::vector<KTask> block, direct;
    std::vector<KGemmTask> gtasks;
    long long nSC = 0;      // L / R products (computed once)
    int nacc = 1;           // copies of the K accumulators
    int mmax = 1, nmax = 1, smax = 1;   // of the row nodes of block terms: most functions m of a split, functions, splits
    bool wide = false;      // 64-bit offsets (kx_block)
    double flops = 0;
    size_t block_lds() const { return kblock_lds(mmax, nmax, wide); }
};

// Default bound of the K accumulators (bytes): workgroups add into one of
// several copies of (K1, K_diag), up to KACC_MAX as the bound allows, so that
// the atomics of the eight XCDs meet less on one address; kx_final adds the
// copies.  C30H62 4.6 MB, (H2O)64 20 MB per matrix.
static const double KACC_BUDGET_DEFAULT = 2.0 * 1024.0 * 1024.0 * 1024.0;
static const int KACC_MAX = 4;

struct KState {
    KPlan P;
    bool ready = false;
    double budget = KACC_BUDGET_DEFAULT;   // bytes of the accumulators (H2ERI_set_exchange_scratch)
    bool wide = false;      // 64-bit offsets whatever the sizes (H2ERI_set_exchange_wide)
    double *PB = nullptr, *CB = nullptr, *SC = nullptr, *KA = nullptr, *D = nullptr, *K = nullptr;
    double *Ds = nullptr;   // the density after screening (the kernels' D)
    int *sbf = nullptr;     // shell_bf_sidx
    KTerm *terms = nullptr;
    KGemm *gemms = nullptr;
    KNode *nodes = nullptr;
    int *bfidx = nullptr, *qptr = nullptr, *mptr = nullptr, *bptr = nullptr, *gptr = nullptr;
    int2 *qent = nullptr, *ment = nullptr, *brow = nullptr;
    int4 *ge = nullptr;
    KTask *block = nullptr, *direct = nullptr;
    KGemmTask *gtasks = nullptr;
    size_t resident = 0;
};

static void kfree(void *&p) {
    if (p) { (void)hipFree(p); p = nullptr; }
}

static void kstate_release(KState *k) {
    void **ps[] = {(void **)&k->PB, (void **)&k->CB, (void **)&k->SC, (void **)&k->KA, (void **)&k->D,
                   (void **)&k->K, (void **)&k->terms, (void **)&k->gemms, (void **)&k->nodes, (void **)&k->bfidx,
                   (void **)&k->qptr, (void **)&k->mptr, (void **)&k->qent, (void **)&k->ment, (void **)&k->bptr,
                   (void **)&k->brow, (void **)&k->gptr, (void **)&k->ge,
                   (void **)&k->block, (void **)&k->direct, (void **)&k->gtasks, (void **)&k->Ds, (void **)&k->sbf};
    for (void **p : ps) kfree(*p);
    k->ready = false;
    k->resident = 0;
    k->P = KPlan();
}

struct KBuilder {
    H2ERI_p h;
    KPlan &P;
    double budget;                   // bytes of the K accumulators
    std::vector<int> ra, rb;
    std::vector<char> sw;
    std::vector<int> bf_shell;       // shell of every basis function
    std::vector<long long> pb_off;   // expanded basis of each tree node in PB (-1: none)
    std::vector<int> node_list;      // tree node -> KNode id (-1: not built)

    KBuilder(H2ERI_p h_, KPlan &p_, const KState *k)
        : h(h_), P(p_), budget(k ? k->budget : KACC_BUDGET_DEFAULT) { P.wide = k && k->wide; }

    int rank_of(int n) const { return h->U[n] ? h->U[n]->ncol : 0; }
    int rows_of(int n) const { return h->mat_cluster[2 * n + 1] - h->mat_cluster[2 * n] + 1; }

    bool pair_rows() {
        const int N = h->krnl_mat_size, np = h->num_sp;
        ra.assign(N, -1); rb.assign(N, -1); sw.assign(N, 0);
        bf_shell.assign(h->num_bf, -1);
        for (int s = 0; s < h->nshell; s++)
            for (int k = h->shell_bf_sidx[s]; k < h->shell_bf_sidx[s + 1] && k < h->num_bf; k++) bf_shell[k] = s;
        for (int i = 0; i < np; i++) {
            const int s0 = h->sp_shell_idx[i], s1 = h->sp_shell_idx[i + np];
            const int f0 = h->shell_bf_sidx[s0], n0 = h->shell_bf_sidx[s0 + 1] - f0;
            const int f1 = h->shell_bf_sidx[s1], n1 = h->shell_bf_sidx[s1 + 1] - f1;
            for (int j = 0; j < n1; j++)
                for (int k = 0; k < n0; k++) {
                    const int x = h->sp_bfp_sidx[i] + j * n0 + k;
                    if (x < 0 || x >= N) { set_error(ERR_ARG, "exchange: shell-pair layout out of range"); return false; }
                    ra[x] = f0 + k; rb[x] = f1 + j; sw[x] = s0 != s1;
                }
        }
        for (int x = 0; x < N; x++)
            if (ra[x] < 0) { set_error(ERR_ARG, "exchange: row %d belongs to no shell pair", x); return false; }
        return true;
    }

    // expanded nested bases of every node with a basis, leaves first
    void expand_bases() {
        const int nn = h->n_node, nl = h->n_leaf_node;
        pb_off.assign(nn, -1);
        for (int lv = h->max_level; lv >= 0; lv--)
            for (int j = 0; j < h->level_n_node[lv]; j++) {
                const int node = h->level_nodes[(size_t)lv * nl + j];
                const int k = rank_of(node);
                if (k == 0 || h->U[node]->nrow == 0) continue;
                const int s = h->mat_cluster[2 * node], m = rows_of(node);
                const long long off = (long long)P.PB.size();
                P.PB.resize(P.PB.size() + (size_t)m * k, 0.0);
                double *Pn = P.PB.data() + off;
                const H2E_dense_mat_p U = h->U[node];
                if (h->n_child[node] == 0) {
                    if (U->nrow != m) continue;
                    for (int r = 0; r < m; r++) memcpy(Pn + (size_t)r * k, U->data + (size_t)r * U->ld, sizeof(double) * k);
                } else {
                    int uoff = 0;
                    for (int c = 0; c < h->n_child[node]; c++) {
                        const int ch = h->children[(size_t)node * h->max_child + c];
                        const int kc = rank_of(ch);
                        if (kc > 0 && pb_off[ch] >= 0) {
                            const double *Pc = P.PB.data() + pb_off[ch];
                            const int cs = h->mat_cluster[2 * ch] - s, cm = rows_of(ch);
                            for (int row = 0; row < cm; row++)
                                for (int l = 0; l < kc; l++) {
                                    const double a = Pc[(size_t)row * kc + l];
                                    const double *urow = U->data + (size_t)(uoff + l) * U->ld;
                                    double *o = Pn + (size_t)(cs + row) * k;
                                    for (int t = 0; t < k; t++) o[t] += a * urow[t];
                                }
                        }
                        uoff += kc;
                    }
                }
                pb_off[node] = off;
            }
    }

    // Column slots of a node: pairs of functions q and their entries merged on
    // p, in fours.  Functions of one shell share their partners, so pairs are
    // taken within a shell first; the functions left over meet the one whose
    // list leaves the fewest entries single.  Long lists are cut (the parts
    // are slots of their own and add into the same q) and pairs come longest
    // first, so that the eight waves of a task have lists of about one length:
    // with pairs of neighbours in order the longest list of a task was twice
    // the mean (C30H62: 175 GFLOP of ket steps for 90 GFLOP of entries, 97 for
    // 71 with the pairs sorted and uncut).  The cut is the one with the
    // fewest MFMAs per step of n: `bra` per task and two per four of the
    // longest list, four past those in registers.
    void column_pairs(KNode &kn, const std::vector<int> &bfs, const std::vector<std::vector<int2>> &byq, double bra) {
        const int nb = (int)bfs.size();
        struct Pair { int a, b; std::vector<int4> e; };
        std::vector<Pair> pairs;
        std::vector<int> single;
        for (int i = 0; i < nb;) {
            int j = i + 1;
            while (j < nb && bf_shell[bfs[j]] == bf_shell[bfs[i]]) j++;
            for (; i + 1 < j; i += 2) pairs.push_back(Pair{i, i + 1, {}});
            if (i < j) single.push_back(i++);
        }
        std::vector<std::vector<int>> ps(nb);   // partners p, sorted
        for (int i = 0; i < nb; i++) {
            for (const int2 &e : byq[i]) ps[i].push_back(e.y);
            std::sort(ps[i].begin(), ps[i].end());
        }
        std::stable_sort(single.begin(), single.end(), [&](int x, int y) { return ps[x].size() > ps[y].size(); });
        std::vector<char> used(single.size(), 0);
        for (size_t i = 0; i < single.size(); i++) {
            if (used[i]) continue;
            const std::vector<int> &x = ps[single[i]];
            size_t best = 0, cost = 0, seen = 0;
            for (size_t j = i + 1; j < single.size() && seen < 64; j++) {
                if (used[j]) continue;
                seen++;
                const std::vector<int> &y = ps[single[j]];
                size_t k = 0, l = 0, common = 0;
                while (k < x.size() && l < y.size()) {
                    if (x[k] == y[l]) { common++; k++; l++; }
                    else if (x[k] < y[l]) k++;
                    else l++;
                }
                const size_t c = x.size() + y.size() - 2 * common;
                if (best == 0 || c < cost) { best = j; cost = c; }
            }
            if (best) used[best] = 1;
            pairs.push_back(Pair{single[i], best ? single[best] : -1, {}});
        }
        for (Pair &p : pairs) {
            // columns of each partner p, of both functions: more than one where a
            // shell pair is stored in both orders (or twice)
            struct Cols { std::vector<int> c[2]; };
            std::map<int, Cols> at;
            for (int j = 0; j < 2; j++)
                if ((j == 0 ? p.a : p.b) >= 0)
                    for (const int2 &e : byq[j == 0 ? p.a : p.b]) at[e.y].c[j].push_back(e.x);
            for (int both = 1; both >= 0; both--)   // entries that both have come first
                for (const auto &e : at) {
                    const std::vector<int> &x = e.second.c[0], &y = e.second.c[1];
                    const size_t nboth = std::min(x.size(), y.size()), n = both ? nboth : std::max(x.size(), y.size());
                    for (size_t k = both ? 0 : nboth; k < n; k++)
                        p.e.push_back(make_int4(k < x.size() ? x[k] : -1, k < y.size() ? y[k] : -1, e.first, 0));
                }
        }
        // lengths in fours of the parts for a cut of `cap` fours, longest first
        auto parts = [&](int cap) {
            std::vector<std::pair<int, int>> v;   // length, pair
            for (int i = 0; i < (int)pairs.size(); i++) {
                const int n4 = ((int)pairs[i].e.size() + 3) / 4, np = (n4 + cap - 1) / cap;
                for (int k = 0; k < np; k++) v.push_back({n4 * (k + 1) / np - n4 * k / np, i});
            }
            std::stable_sort(v.begin(), v.end(), [](const std::pair<int, int> &x, const std::pair<int, int> &y) { return x.first > y.first; });
            return v;
        };
        std::vector<std::pair<int, int>> v;
        double cost = 0.0;
        for (int cap : {4, 5, 6, 7, 8, 9, 10, 11, 12, 14, 16, 20, 24, 32, 48, 64, 1 << 28}) {
            std::vector<std::pair<int, int>> w = parts(cap);
            double c = 0.0;
            for (size_t g = 0; g < w.size(); g += KQ / 2) c += bra + 2.0 * w[g].first + 2.0 * std::max(0, w[g].first - KNQ);
            if (v.empty() || c < cost) { v = w; cost = c; }
        }
        kn.g_ptr = (int)P.gptr.size();
        kn.c_off = (int)P.bfidx.size();
        kn.ngrp = (int)v.size();
        std::vector<size_t> at(pairs.size(), 0);
        for (const auto &g : v) {
            const Pair &p = pairs[g.second];
            P.gptr.push_back((int)P.ge.size());
            int full = 0;
            for (int k = 0; k < 4 * g.first; k++) {
                const size_t i = at[g.second]++;
                P.ge.push_back(i < p.e.size() ? p.e[i] : make_int4(-1, -1, 0, 0));
                if (full == k && P.ge.back().x >= 0 && P.ge.back().y >= 0) full++;
            }
            P.gptr.push_back(full / 4);
            P.bfidx.push_back(bfs[p.a]);
            P.bfidx.push_back(p.b >= 0 ? bfs[p.b] : -1);
        }
        P.gptr.push_back((int)P.ge.size());
    }

    // basis-function set and orientation lists of a tree node's row range
    int list_of(int node) {
        if (node_list[node] >= 0) return node_list[node];
        const int s = h->mat_cluster[2 * node], m = rows_of(node);
        std::vector<int> bfs;
        bfs.reserve(2 * m);
        for (int r = 0; r < m; r++) { bfs.push_back(ra[s + r]); bfs.push_back(rb[s + r]); }
        std::sort(bfs.begin(), bfs.end());
        bfs.erase(std::unique(bfs.begin(), bfs.end()), bfs.end());
        const int nb = (int)bfs.size();
        std::vector<int> loc(h->num_bf, -1);
        for (int i = 0; i < nb; i++) loc[bfs[i]] = i;
        KNode kn;
        kn.bf_off = (int)P.bfidx.size();
        kn.nbf = nb;
        P.bfidx.insert(P.bfidx.end(), bfs.begin(), bfs.end());
        // byQ: ket orientations (p,q) of each row c; byM: bra orientations (m,n) of each row r
        std::vector<std::vector<int2>> byq(nb), bym(nb);
        for (int r = 0; r < m; r++) {
            const int x = s + r, a = ra[x], b = rb[x];
            byq[loc[b]].push_back(make_int2(r, a));
            bym[loc[a]].push_back(make_int2(r, loc[b]));
            if (sw[x]) {
                byq[loc[a]].push_back(make_int2(r, b));
                bym[loc[b]].push_back(make_int2(r, loc[a]));
            }
        }
        kn.q_ptr = (int)P.qptr.size();
        for (int i = 0; i < nb; i++) { P.qptr.push_back((int)P.qent.size()); P.qent.insert(P.qent.end(), byq[i].begin(), byq[i].end()); }
        P.qptr.push_back((int)P.qent.size());
        kn.m_ptr = (int)P.mptr.size();
        for (int i = 0; i < nb; i++) { P.mptr.push_back((int)P.ment.size()); P.ment.insert(P.ment.end(), bym[i].begin(), bym[i].end()); }
        P.mptr.push_back((int)P.ment.size());
        // bra: for each local n the (row, local m) entries, sorted by m; per
        // split of ssz functions m (at most KM, even parts so that no split is
        // a sliver) and step of 16 n, blocks of up to 16 entries dealt to the
        // eight waves, an even number each (empty ones make up for it)
        std::vector<std::vector<int2>> byn(nb);
        for (int ml = 0; ml < nb; ml++)
            for (const int2 &e : bym[ml]) byn[e.y].push_back(make_int2(e.x, ml));
        kn.nsplit = (nb + KM - 1) / KM;
        kn.ssz = kn.nsplit > 0 ? (nb + kn.nsplit - 1) / kn.nsplit : KM;
        kn.b_ptr = (int)P.bptr.size();
        int nblk = 0;   // not empty
        for (int sp = 0; sp < kn.nsplit; sp++)
            for (int n0 = 0; n0 < nb; n0 += 16) {
                // runs of functions n of one shell, whose lists hold the same m: a
                // chain takes the same 16 entries of each, in one accumulator
                struct Chain { int nl, nn, e0, cnt; };
                std::vector<Chain> ch;
                auto range = [&](int nl) {   // entries of the split
                    int a = 0, b = 0;
                    while (a < (int)byn[nl].size() && byn[nl][a].y < sp * kn.ssz) a++;
                    for (b = a; b < (int)byn[nl].size() && byn[nl][b].y < (sp + 1) * kn.ssz;) b++;
                    return std::make_pair(a, b);
                };
                const int n1 = std::min(n0 + 16, nb);
                for (int nl = n0, nn; nl < n1; nl += nn) {
                    const auto r = range(nl);
                    for (nn = 1; nn < KCHAIN && nl + nn < n1; nn++) {
                        const auto q = range(nl + nn);
                        if (bf_shell[bfs[nl + nn]] != bf_shell[bfs[nl]] || q.second - q.first != r.second - r.first) break;
                        bool same = true;
                        for (int k = 0; same && k < r.second - r.first; k++)
                            same = byn[nl + nn][q.first + k].y == byn[nl][r.first + k].y;
                        if (!same) break;
                    }
                    for (int e = r.first; e < r.second; e += 16)
                        ch.push_back(Chain{nl, nn, e - r.first, std::min(16, r.second - e)});
                }
                // to the wave with the fewest blocks, long chains first
                std::stable_sort(ch.begin(), ch.end(), [](const Chain &x, const Chain &y) { return x.nn > y.nn; });
                std::vector<Chain> wv[8];
                int load[8] = {0};
                for (const Chain &c : ch) {
                    const int w = (int)(std::min_element(load, load + 8) - load);
                    load[w] += c.nn;
                    nblk += c.nn;
                    wv[w].push_back(c);
                }
                for (int w = 0; w < 8; w++) {
                    P.bptr.push_back((int)P.brow.size() / 16);
                    if (load[w] == 0 || load[w] % 2) wv[w].push_back(Chain{n0, 1, 0, 0});
                    if (load[w] == 0) wv[w].push_back(Chain{n0, 1, 0, 0});
                    for (const Chain &c : wv[w])
                        for (int k = 0; k < c.nn; k++) {
                            const int a0 = range(c.nl + k).first + c.e0;
                            const int nf = (c.nl + k - n0) | (k + 1 < c.nn ? KMORE : 0) | (k == 0 ? KFIRST : 0) | (c.cnt == 0 ? KEMPTY : 0);
                            for (int e = 0; e < 16; e++) {
                                const int2 a = c.cnt ? byn[c.nl + k][a0 + std::min(e, c.cnt - 1)] : make_int2(0, 0);
                                P.brow.push_back(make_int2(a.x, (e < c.cnt ? a.y - sp * kn.ssz : kn.ssz) * KQ * 8 | nf << 16));
                            }
                        }
                }
            }
        P.bptr.push_back((int)P.brow.size() / 16);
        // a step of n costs a wave about four MFMAs per bra block
        column_pairs(kn, bfs, byq, 4.0 * nblk / (8.0 * kn.nsplit * ((nb + 15) / 16)));
        P.nodes.push_back(kn);
        node_list[node] = (int)P.nodes.size() - 1;
        return node_list[node];
    }

    struct Core { bool lr; long long C, U, VT; int nrow, ncol, k; };
    Core store_core(H2E_dense_mat_p b) {
        Core c{false, -1, -1, -1, b->nrow, b->ncol, 0};
        const long long off = (long long)P.CB.size();
        if (b->ld >= 0) {
            P.CB.insert(P.CB.end(), b->data, b->data + (size_t)b->nrow * b->ncol);
            c.C = off;
        } else {
            c.lr = true;
            c.k = -b->ld;
            P.CB.insert(P.CB.end(), b->data, b->data + (size_t)(b->nrow + b->ncol) * c.k);
            c.U = off;
            c.VT = off + (long long)b->nrow * c.k;
        }
        return c;
    }
    long long salloc(long long n) {
        const long long o = P.nSC;
        P.nSC += (n + 31) & ~31LL;
        return o;
    }
    long long gemm(long long Aoff, int lda, int m, int k, long long Xoff, int ldx, int n) {
        KGemm g;
        g.Aoff = Aoff; g.lda = lda; g.m = m; g.k = k; g.Xoff = Xoff; g.ldx = ldx; g.n = n;
        g.Ooff = salloc((long long)m * n);
        g.ldo = n;
        P.gemms.push_back(g);
        P.flops += 2.0 * m * n * k;
        return g.Ooff;
    }

    // one term: rows of node n0 (basis side if bas0) x columns of node n1 (bas1), core b
    void add_term(int n0, bool bas0, int n1, bool bas1, H2E_dense_mat_p b, int diag) {
        if (!b || b->nrow == 0 || b->ncol == 0) return;
        const int m0 = rows_of(n0), m1 = rows_of(n1);
        const int k0 = bas0 ? rank_of(n0) : m0, k1 = bas1 ? rank_of(n1) : m1;
        if (b->nrow != k0 || b->ncol != k1) return;   // not part of A_H2
        if ((bas0 && pb_off[n0] < 0) || (bas1 && pb_off[n1] < 0)) return;
        const Core c = store_core(b);
        KTerm t;
        memset(&t, 0, sizeof(t));
        t.diag = diag;
        t.ni = list_of(n0);
        t.nj = list_of(n1);
        t.m0 = m0; t.m1 = m1;
        if (!bas0 && !bas1 && !c.lr) {            // dense near-field block: direct contraction
            t.direct = 1;
            t.kk = m1;
            t.Lsrc = KS_CB; t.Loff = c.C; t.Lld = m1;
            P.terms.push_back(t);
            return;
        }
        if (!c.lr) {
            if (bas0 && bas1) {        // L = P0 C, R = P1
                t.kk = k1;
                t.Lsrc = KS_SC; t.Loff = gemm(pb_off[n0], k0, m0, k0, c.C, k1, k1); t.Lld = k1;
                t.Rsrc = KS_PB; t.Roff = pb_off[n1]; t.Rrs = k1; t.Rcs = 1;
            } else if (bas0) {         // L = P0, R = C^T
                t.kk = k0;
                t.Lsrc = KS_PB; t.Loff = pb_off[n0]; t.Lld = k0;
                t.Rsrc = KS_CB; t.Roff = c.C; t.Rrs = 1; t.Rcs = m1;
            } else {                   // L = C, R = P1
                t.kk = k1;
                t.Lsrc = KS_CB; t.Loff = c.C; t.Lld = k1;
                t.Rsrc = KS_PB; t.Roff = pb_off[n1]; t.Rrs = k1; t.Rcs = 1;
            }
        } else {
            const int k = c.k;
            t.kk = k;
            if (bas0) { t.Lsrc = KS_SC; t.Loff = gemm(pb_off[n0], k0, m0, k0, c.U, k, k); t.Lld = k; }
            else { t.Lsrc = KS_CB; t.Loff = c.U; t.Lld = k; }
            if (bas1) { t.Rsrc = KS_SC; t.Roff = gemm(pb_off[n1], k1, m1, k1, c.VT, k, k); t.Rrs = k; t.Rcs = 1; }
            else { t.Rsrc = KS_CB; t.Roff = c.VT; t.Rrs = k; t.Rcs = 1; }
        }
        P.terms.push_back(t);
    }

    bool build() {
        if (h->num_bf <= 0 || !h->sp_shell_idx || !h->shell_bf_sidx) { set_error(ERR_ARG, "exchange needs shell-pair metadata"); return false; }
        if (h->BD_JIT) { set_error(ERR_UNSUPPORTED, "H2ERI_build_exchange does not support BD_JIT representations"); return false; }
        if (!pair_rows()) return false;
        expand_bases();
        node_list.assign(h->n_node, -1);
        const int nl = h->n_leaf_node;
        for (int i = 0; i < nl; i++) add_term(h->height_nodes[i], false, h->height_nodes[i], false, h->c_D_blks[i], 1);
        for (int i = 0; i < h->n_r_inadm_pair; i++)
            add_term(h->r_inadm_pairs[2 * i], false, h->r_inadm_pairs[2 * i + 1], false, h->c_D_blks[nl + i], 0);
        for (int i = 0; i < h->n_r_adm_pair; i++) {
            const int n0 = h->r_adm_pairs[2 * i], n1 = h->r_adm_pairs[2 * i + 1];
            const int l0 = h->node_level[n0], l1 = h->node_level[n1];
            add_term(n0, l0 >= l1, n1, l1 >= l0, h->c_B_blks[i], 0);
        }
        // launch task lists
        for (int g = 0; g < (int)P.gemms.size(); g++)
            for (int r0 = 0; r0 < P.gemms[g].m; r0 += 64)
                for (int c0 = 0; c0 < P.gemms[g].n; c0 += 64) P.gtasks.push_back(KGemmTask{g, r0, c0, 0});
        // block tasks: 16 functions q by a split of the functions m, the terms
        // with the most work first (a workgroup's time goes with the steps of
        // n, t and entries)
        std::vector<std::pair<double, int>> order;
        for (int ti = 0; ti < (int)P.terms.size(); ti++) {
            const KTerm &t = P.terms[ti];
            const KNode &ni = P.nodes[t.ni], &nj = P.nodes[t.nj];
            if (t.direct) {
                const long long ne = (long long)ni.nbf * nj.nbf;
                for (long long e0 = 0; e0 < ne; e0 += KWG / 64) P.direct.push_back(KTask{ti, (int)e0, 0, 0});
                continue;
            }
            P.mmax = std::max(P.mmax, ni.ssz);
            P.nmax = std::max(P.nmax, ni.nbf);
            P.smax = std::max(P.smax, ni.nsplit);
            const double reach = std::max({(double)t.m1 * t.Rrs + (double)t.kk * t.Rcs, (double)t.m0 * t.Lld + t.kk + KPAD,
                                           (double)h->num_bf * h->num_bf});
            if (reach * 8.0 >= 4294967296.0 || ni.nbf > KNMAX || t.m0 >= 1 << 24 || t.Lld >= 1 << 21) P.wide = true;
            const double steps = (double)((ni.nbf + 15) / 16) * ((t.kk + 15) / 16);
            order.push_back({steps * (4.0 + (double)t.m1 / nj.nbf + (double)t.m0 / ni.nbf), ti});
        }
        std::stable_sort(order.begin(), order.end(), [](const std::pair<double, int> &a, const std::pair<double, int> &b) { return a.first > b.first; });
        for (const auto &o : order) {
            const KNode &ni = P.nodes[P.terms[o.second].ni], &nj = P.nodes[P.terms[o.second].nj];
            for (int ql0 = 0; ql0 < 2 * nj.ngrp; ql0 += KQ)
                for (int sp = 0; sp < ni.nsplit; sp++) P.block.push_back(KTask{o.second, ql0, sp, 0});
        }
        const double acc = 16.0 * (double)h->num_bf * h->num_bf;   // bytes of one (K1, K_diag)
        P.nacc = std::max(1, (int)std::min((double)KACC_MAX, budget / acc));
        return validate();
    }

    // every access of every kernel checked on the host before any launch
    bool validate() const {
        const long long nPB = (long long)P.PB.size(), nCB = (long long)P.CB.size(), nSC = P.nSC;
        const int nbf = h->num_bf;
        auto size_of = [&](int src) { return src == KS_PB ? nPB : (src == KS_CB ? nCB : nSC); };
        for (const KGemm &g : P.gemms) {
            const bool ok = g.m > 0 && g.n > 0 && g.k > 0 && g.Aoff >= 0 && g.Aoff + (long long)(g.m - 1) * g.lda + g.k <= nPB &&
                            g.Xoff >= 0 && g.Xoff + (long long)(g.k - 1) * g.ldx + g.n <= nCB && g.Ooff >= 0 &&
                            g.Ooff + (long long)(g.m - 1) * g.ldo + g.n <= nSC && g.lda >= g.k && g.ldx >= g.n && g.ldo >= g.n;
            if (!ok) { set_error(ERR_ARG, "exchange plan check failed: gemm"); return false; }
        }
        for (const KNode &n : P.nodes) {
            bool ok = n.bf_off >= 0 && n.bf_off + n.nbf <= (long long)P.bfidx.size() && n.q_ptr + n.nbf < (long long)P.qptr.size() &&
                      n.m_ptr + n.nbf < (long long)P.mptr.size() && n.g_ptr + 2LL * n.ngrp < (long long)P.gptr.size() &&
                      n.c_off >= 0 && n.c_off + 2LL * n.ngrp <= (long long)P.bfidx.size();
            for (int i = 0; ok && i < n.nbf; i++) ok = P.bfidx[n.bf_off + i] >= 0 && P.bfidx[n.bf_off + i] < nbf;
            for (int i = 0; ok && i < 2 * n.ngrp; i++) ok = P.bfidx[n.c_off + i] >= -1 && P.bfidx[n.c_off + i] < nbf;
            if (!ok) { set_error(ERR_ARG, "exchange plan check failed: node lists"); return false; }
            // the column slots of a function hold each of its entries once
            std::vector<int> live(nbf, 0);
            for (int i = 0; i < 2 * n.ngrp; i++) {
                const int q = P.bfidx[n.c_off + i], g = n.g_ptr + 2 * (i >> 1);
                for (int j = P.gptr[g]; j < P.gptr[g + 2]; j++) {
                    const bool has = ((i & 1) ? P.ge[j].y : P.ge[j].x) >= 0;
                    if (has && q < 0) ok = false;
                    else if (has) live[q]++;
                }
            }
            for (int i = 0; ok && i < n.nbf; i++)
                ok = live[P.bfidx[n.bf_off + i]] == P.qptr[n.q_ptr + i + 1] - P.qptr[n.q_ptr + i];
            if (!ok) { set_error(ERR_ARG, "exchange plan check failed: column slots"); return false; }
        }
        for (const KTerm &t : P.terms) {
            const KNode &ni = P.nodes[t.ni], &nj = P.nodes[t.nj];
            bool ok = t.kk > 0 && (long long)ni.nbf * nj.nbf < (1LL << 31);
            // entries: columns < m1, p < nbf; rows < m0, local n < |B(i)|
            for (int j = P.qptr[nj.q_ptr]; ok && j < P.qptr[nj.q_ptr + nj.nbf]; j++)
                ok = P.qent[j].x >= 0 && P.qent[j].x < t.m1 && P.qent[j].y >= 0 && P.qent[j].y < nbf;
            for (int g = 0; ok && g < nj.ngrp; g++) {
                const int ga = P.gptr[nj.g_ptr + 2 * g], gb = P.gptr[nj.g_ptr + 2 * g + 2], full = P.gptr[nj.g_ptr + 2 * g + 1];
                ok = ga >= 0 && ga <= gb && gb <= (int)P.ge.size() && (gb - ga) % 4 == 0 && full >= 0 && 4 * full <= gb - ga;
                for (int j = ga; ok && j < gb; j++)
                    ok = P.ge[j].z >= 0 && P.ge[j].z < nbf && P.ge[j].x < t.m1 && P.ge[j].y < t.m1 &&
                         (j >= ga + 4 * full || (P.ge[j].x >= 0 && P.ge[j].y >= 0));
            }
            for (int j = P.mptr[ni.m_ptr]; ok && j < P.mptr[ni.m_ptr + ni.nbf]; j++)
                ok = P.ment[j].x >= 0 && P.ment[j].x < t.m0 && P.ment[j].y >= 0 && P.ment[j].y < ni.nbf;
            // bra blocks: at least one per step and wave, rows below m0, m within
            // the split (the splits cover every local m)
            const int nst = (ni.nbf + 15) / 16;
            ok = ok && ni.nsplit >= 1 && ni.ssz >= 1 && ni.ssz <= KM && (long long)ni.nsplit * ni.ssz >= ni.nbf && ni.b_ptr >= 0 &&
                 ni.b_ptr + (long long)ni.nsplit * nst * 8 < (long long)P.bptr.size();
            for (int k = 0; ok && k < ni.nsplit * nst * 8; k++) {
                const int sp = k / (nst * 8);
                const int b0 = P.bptr[ni.b_ptr + k], b1 = P.bptr[ni.b_ptr + k + 1];
                ok = b0 >= 0 && b0 < b1 && (b1 - b0) % 2 == 0 && b1 <= (int)(P.brow.size() / 16);
                const int rows = std::min((sp + 1) * ni.ssz, ni.nbf) - sp * ni.ssz;
                for (int e = 16 * b0; ok && e < 16 * b1; e++) {
                    const int m = P.brow[e].y & 0xffff, nf = P.brow[e].y >> 16;
                    ok = P.brow[e].x >= 0 && P.brow[e].x < t.m0 && nf >= 0 && nf < 128 && nf == P.brow[e & ~15].y >> 16 &&
                         m % (KQ * 8) == 0 && (m / (KQ * 8) < rows || m / (KQ * 8) == ni.ssz);
                    // a chain begins where none goes on, and goes on in a block of the
                    // same list with the same m
                    if (ok && (nf & KMORE)) ok = e + 16 < 16 * b1 && (P.brow[e + 16].y & 0xffff) == m && !(P.brow[e + 16].y >> 16 & (KFIRST | KEMPTY));
                    if (ok && !(nf & KFIRST)) ok = e >= 16 * b0 + 16 && (P.brow[e - 16].y >> 16 & KMORE);
                }
            }
            ok = ok && t.Loff >= 0 && t.Loff + (long long)(t.m0 - 1) * t.Lld + t.kk <= size_of(t.Lsrc);
            if (!t.direct) {
                const long long last = t.Roff + (long long)(t.m1 - 1) * t.Rrs + (long long)(t.kk - 1) * t.Rcs;
                ok = ok && t.Roff >= 0 && last < size_of(t.Rsrc);
            }
            if (!ok) { set_error(ERR_ARG, "exchange plan check failed: term"); return false; }
        }
        // block tasks: each within its term
        bool ok = true;
        for (size_t i = 0; ok && i < P.block.size(); i++) {
            const KTask &k = P.block[i];
            ok = k.term >= 0 && k.term < (int)P.terms.size() && !P.terms[k.term].direct;
            if (!ok) break;
            const KNode &ni = P.nodes[P.terms[k.term].ni], &nj = P.nodes[P.terms[k.term].nj];
            ok = k.e0 >= 0 && k.e0 < 2 * nj.ngrp && k.e0 % KQ == 0 && k.t0 >= 0 && k.t0 < ni.nsplit;
        }
        if (!ok) { set_error(ERR_ARG, "exchange plan check failed: tasks"); return false; }
        return true;
    }
};

}  // namespace

static KState *kstate(H2ERI_p h) { return (KState *)h->thread_Kmat_workbuf; }

void exchange_release(H2ERI_p h) {
    KState *k = kstate(h);
    if (!k) return;
    device_release_graph_kind(h, 2);   // a captured exchange graph refers to the buffers freed here
    kstate_release(k);
    delete k;
    h->thread_Kmat_workbuf = nullptr;
}

#define KHIP(expr)                                                                                           \
    do {                                                                                                     \
        hipError_t e_ = (expr);                                                                              \
        if (e_ != hipSuccess) {                                                                              \
            set_error(ERR_DEVICE, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
            return false;                                                                                    \
        }                                                                                                    \
    } while (0)

static bool k_upload(H2ERI_p h) {
    if (!h->U || !h->c_B_blks || !h->c_D_blks) { set_error(ERR_ARG, "no H2 representation built or loaded"); return false; }
    if (!h->shell_bf_sidx || h->nshell <= 0) { set_error(ERR_ARG, "the exchange build needs shell metadata"); return false; }
    if (!h->thread_Kmat_workbuf) h->thread_Kmat_workbuf = (void **)new KState();
    KState *k = kstate(h);
    if (k->ready) return true;
    kstate_release(k);
    KBuilder b(h, k->P, k);
    if (!b.build()) return false;
    const KPlan &P = k->P;
    const int nbf = h->num_bf;
    auto up = [&](void **dst, const void *src, size_t bytes) -> bool {
        if (bytes == 0) bytes = 64;
        KHIP(hipMalloc(dst, bytes));
        if (src) KHIP(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
        k->resident += bytes;
        return true;
    };
    const size_t nn2 = (size_t)nbf * nbf;
    // operand arrays end in KPAD zeros: the bra's loads of four t run past a row's end
    k->P.PB.resize(P.PB.size() + KPAD, 0.0);
    k->P.CB.resize(P.CB.size() + KPAD, 0.0);
    if (!up((void **)&k->PB, P.PB.data(), P.PB.size() * 8) || !up((void **)&k->CB, P.CB.data(), P.CB.size() * 8) ||
        !up((void **)&k->SC, nullptr, ((size_t)P.nSC + KPAD) * 8) ||
        !up((void **)&k->KA, nullptr, nn2 * 16 * P.nacc) || !up((void **)&k->D, nullptr, nn2 * 8) ||
        !up((void **)&k->K, nullptr, nn2 * 8) || !up((void **)&k->Ds, nullptr, nn2 * 8) ||
        !up((void **)&k->sbf, h->shell_bf_sidx, (size_t)(h->nshell + 1) * 4) ||
        !up((void **)&k->terms, P.terms.empty() ? nullptr : P.terms.data(), P.terms.size() * sizeof(KTerm)) ||
        !up((void **)&k->gemms, P.gemms.empty() ? nullptr : P.gemms.data(), P.gemms.size() * sizeof(KGemm)) ||
        !up((void **)&k->nodes, P.nodes.empty() ? nullptr : P.nodes.data(), P.nodes.size() * sizeof(KNode)) ||
        !up((void **)&k->bfidx, P.bfidx.data(), P.bfidx.size() * 4) || !up((void **)&k->qptr, P.qptr.data(), P.qptr.size() * 4) ||
        !up((void **)&k->mptr, P.mptr.data(), P.mptr.size() * 4) ||
        !up((void **)&k->bptr, P.bptr.data(), P.bptr.size() * 4) ||
        !up((void **)&k->brow, P.brow.empty() ? nullptr : P.brow.data(), P.brow.size() * sizeof(int2)) ||
        !up((void **)&k->qent, P.qent.empty() ? nullptr : P.qent.data(), P.qent.size() * sizeof(int2)) ||
        !up((void **)&k->ment, P.ment.empty() ? nullptr : P.ment.data(), P.ment.size() * sizeof(int2)) ||
        !up((void **)&k->gptr, P.gptr.data(), P.gptr.size() * 4) ||
        !up((void **)&k->ge, P.ge.empty() ? nullptr : P.ge.data(), P.ge.size() * sizeof(int4)) ||
        !up((void **)&k->block, P.block.empty() ? nullptr : P.block.data(), P.block.size() * sizeof(KTask)) ||
        !up((void **)&k->direct, P.direct.empty() ? nullptr : P.direct.data(), P.direct.size() * sizeof(KTask)) ||
        !up((void **)&k->gtasks, P.gtasks.empty() ? nullptr : P.gtasks.data(), P.gtasks.size() * sizeof(KGemmTask)))
        return false;
    // one limit for the process: the most any plan asks for, not this one's
    for (const void *f : {reinterpret_cast<const void *>(&kx_block<unsigned>), reinterpret_cast<const void *>(&kx_block<unsigned long long>)})
        KHIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kblock_lds(KM, KNMAX, false)));
    // (zeros also between the products, whose rows end where the next begins)
    KHIP(hipMemset(k->SC, 0, ((size_t)P.nSC + KPAD) * 8));
    // L / R products do not depend on D: computed once at upload
    if (!P.gtasks.empty()) {
        hipLaunchKernelGGL(kx_gemm, dim3((unsigned)P.gtasks.size()), dim3(KWG), 0, 0, k->gtasks, k->gemms, k->PB, k->CB, k->SC);
        KHIP(hipGetLastError());
        KHIP(hipDeviceSynchronize());
    }
    k->ready = true;
    return true;
}

static bool k_run(H2ERI_p h, const double *D_dev, double *K_dev, hipStream_t s) {
    if (!k_upload(h)) return false;
    KState *k = kstate(h);
    const KPlan &P = k->P;
    const int nbf = h->num_bf;
    const size_t nn2 = (size_t)nbf * nbf;
    const unsigned zb = (unsigned)std::min<size_t>((nn2 + 255) / 256, 2048);
    const long long nblk = (long long)h->nshell * h->nshell;
    hipLaunchKernelGGL(kx_dlist, dim3((unsigned)((nblk + 255) / 256)), dim3(256), 0, s, k->sbf, h->nshell, D_dev, k->Ds, nbf);
    D_dev = k->Ds;
    hipLaunchKernelGGL(kx_zero, dim3(zb), dim3(256), 0, s, k->KA, nn2 * 2 * P.nacc);
    KHIP(hipGetLastError());
    // the blocks add into the accumulators with atomics
    if (!P.block.empty())
        hipLaunchKernelGGL(P.wide ? kx_block<unsigned long long> : kx_block<unsigned>, dim3((unsigned)P.block.size()), dim3(KBWG),
                           P.block_lds(), s, k->block, k->terms, k->nodes, k->bfidx, k->gptr, k->ge, k->bptr, k->brow,
                           k->PB, k->CB, k->SC, D_dev, k->KA, P.nacc, nbf);
    if (!P.direct.empty())
        hipLaunchKernelGGL(kx_direct, dim3((unsigned)P.direct.size()), dim3(KWG), 0, s, k->direct, k->terms, k->nodes,
                           k->bfidx, k->qptr, k->qent, k->mptr, k->ment, k->CB, D_dev, k->KA, nbf);
    KHIP(hipGetLastError());
    const unsigned nt = (unsigned)(nbf + 31) / 32;
    hipLaunchKernelGGL(kx_final, dim3(nt, nt), dim3(256), 0, s, k->KA, P.nacc, K_dev, nbf);
    KHIP(hipGetLastError());
    return true;
}

bool exchange_prepare(H2ERI_p h) { return k_upload(h); }

bool exchange_enqueue(H2ERI_p h, const double *D_dev, double *K_dev, void *stream) {
    return k_run(h, D_dev, K_dev, (hipStream_t)stream);
}

}  // namespace h2e

using namespace h2e;

extern "C" {

// Density screening list on the host (src/H2ERI_build_exchange.c:774-838):
// dlist_sidx[N]..dlist_sidx[N+1] lists, in increasing order, the shells P
// whose block (N,P) of D has some |D_np| > 1e-10 (:790).  The device build
// applies the same rule to its copy of D.
void H2ERI_exchange_dlist(H2ERI_p h, const double *den_mat) {
    if (!h || !den_mat) { set_error(ERR_ARG, "H2ERI_exchange_dlist: null argument"); return; }
    if (!h->shell_bf_sidx || h->nshell <= 0) { set_error(ERR_ARG, "H2ERI_exchange_dlist: needs shell-pair metadata (a molecule)"); return; }
    const int ns = h->nshell, nbf = h->num_bf;
    const int *sbf = h->shell_bf_sidx;
    std::vector<std::vector<int>> rows(ns);
    #pragma omp parallel for schedule(dynamic)
    for (int n = 0; n < ns; n++)
        for (int p = 0; p < ns; p++) {
            bool keep = false;
            for (int i = sbf[n]; i < sbf[n + 1] && !keep; i++)
                for (int j = sbf[p]; j < sbf[p + 1]; j++)
                    if (std::fabs(den_mat[(size_t)i * nbf + j]) > 1e-10) { keep = true; break; }
            if (keep) rows[n].push_back(p);
        }
    free(h->dlist_sidx);
    free(h->dlist);
    h->dlist_sidx = (int *)malloc(sizeof(int) * (ns + 1));
    size_t len = 0;
    for (int n = 0; n < ns; n++) len += rows[n].size();
    h->dlist = (int *)malloc(sizeof(int) * (len > 0 ? len : 1));
    if (!h->dlist_sidx || !h->dlist) { set_error(ERR_ALLOC, "H2ERI_exchange_dlist: allocation failed"); return; }
    h->dlist_sidx[0] = 0;
    for (int n = 0; n < ns; n++) {
        std::copy(rows[n].begin(), rows[n].end(), h->dlist + h->dlist_sidx[n]);
        h->dlist_sidx[n + 1] = h->dlist_sidx[n] + (int)rows[n].size();
    }
}

void H2ERI_build_exchange(H2ERI_p h, const double *den_mat, double *K_mat) {
    if (!h || !den_mat || !K_mat) { set_error(ERR_ARG, "H2ERI_build_exchange: null argument"); return; }
    H2ERI_exchange_dlist(h, den_mat);   // the reference's side effect on the handle
    if (has_error()) return;
    if (!k_upload(h)) return;
    KState *k = kstate(h);
    const size_t nn2 = (size_t)h->num_bf * h->num_bf;
    if (hipMemcpy(k->D, den_mat, nn2 * 8, hipMemcpyHostToDevice) != hipSuccess) { set_error(ERR_DEVICE, "copy D"); return; }
    if (!k_run(h, k->D, k->K, nullptr)) return;
    if (hipMemcpy(K_mat, k->K, nn2 * 8, hipMemcpyDeviceToHost) != hipSuccess) { set_error(ERR_DEVICE, "copy K"); return; }
    h->n_matvec++;
}

void H2ERI_build_exchange_dev(H2ERI_p h, const double *den_dev, double *K_dev, void *stream) {
    if (!h || !den_dev || !K_dev) { set_error(ERR_ARG, "H2ERI_build_exchange_dev: null argument"); return; }
    k_run(h, den_dev, K_dev, (hipStream_t)stream);
}

// Builds the exchange plan on the device now (otherwise done by the first
// call); the reference allocates its per-thread K work buffers here.
void H2ERI_exchange_workbuf_init(H2ERI_p h) {
    if (h) k_upload(h);
}

void H2ERI_exchange_workbuf_free(H2ERI_p h) {
    if (h) exchange_release(h);
}

// Builds the exchange plan on the host only (no HIP call) and checks every
// access of its kernels; out4 as H2ERI_exchange_stats with out4[2] the bytes
// the plan would make resident.  Returns the number of terms, -1 on failure.
int H2ERI_exchange_plan_check(H2ERI_p h, double *out4) {
    if (!h || !h->U || !h->c_B_blks || !h->c_D_blks) { set_error(ERR_ARG, "exchange_plan_check: nothing built"); return -1; }
    KPlan P;
    KBuilder b(h, P, kstate(h));
    if (!b.build()) return -1;
    if (out4) {
        const double nn2 = (double)h->num_bf * h->num_bf;
        out4[0] = P.flops;
        out4[1] = (double)P.terms.size();
        const double nacc = 2.0 * P.nacc * nn2;
        // as k_upload: operands and their padding, accumulators, D, K and the
        // screened D, lists, terms, tasks (an empty array takes 64 bytes)
        const double operands = (double)P.PB.size() + (double)P.CB.size() + (double)P.nSC + 3.0 * KPAD;
        out4[2] = 8.0 * (operands + nacc + 3.0 * nn2);
        auto add = [&](size_t n, size_t size) { out4[2] += n > 0 ? (double)n * (double)size : 64.0; };
        for (const auto *v : {&P.bfidx, &P.qptr, &P.mptr, &P.gptr, &P.bptr}) add(v->size(), sizeof(int));
        for (const auto *v : {&P.qent, &P.ment, &P.brow}) add(v->size(), sizeof(int2));
        add(P.ge.size(), sizeof(int4));
        add(P.terms.size(), sizeof(KTerm));
        add(P.gemms.size(), sizeof(KGemm));
        add(P.nodes.size(), sizeof(KNode));
        add(P.gtasks.size(), sizeof(KGemmTask));
        for (const auto *v : {&P.block, &P.direct}) add(v->size(), sizeof(KTask));
        add((size_t)h->nshell + 1, sizeof(int));
        out4[3] = (double)P.nSC + nacc;
    }
    return (int)P.terms.size();
}

// Shape of the block tasks (host only, tests): out4 = {LDS bytes of a
// workgroup, most functions of a row node of a block term, most splits of one,
// 1 when operand offsets take 64 bits}.  Returns 0, -1 on failure.
int H2ERI_exchange_plan_shape(H2ERI_p h, double *out4) {
    if (!h || !out4 || !h->U || !h->c_B_blks || !h->c_D_blks) { set_error(ERR_ARG, "exchange_plan_shape: nothing built"); return -1; }
    KPlan P;
    KBuilder b(h, P, kstate(h));
    if (!b.build()) return -1;
    out4[0] = (double)P.block_lds();
    out4[1] = P.nmax;
    out4[2] = P.smax;
    out4[3] = P.wide ? 1.0 : 0.0;
    return 0;
}

// Work figures of the exchange plan: out4 = {GEMM flops at upload, terms,
// device bytes resident, scratch doubles}.
void H2ERI_exchange_stats(H2ERI_p h, double *out4) {
    if (!h || !out4 || !k_upload(h)) return;
    KState *k = kstate(h);
    out4[0] = k->P.flops;
    out4[1] = (double)k->P.terms.size();
    out4[2] = (double)k->resident;
    out4[3] = (double)k->P.nSC + 2.0 * k->P.nacc * (double)h->num_bf * h->num_bf;
}

// Bound of the exchange build's K accumulators in bytes (additive, tuning):
// at least one copy of (K1, K_diag) whatever the bound.  Releases the
// exchange plan (rebuilt by the next K build).
void H2ERI_set_exchange_scratch(H2ERI_p h, const double bytes) {
    if (!h || !(bytes >= 1024.0)) { set_error(ERR_ARG, "H2ERI_set_exchange_scratch: at least 1024 bytes"); return; }
    if (!h->thread_Kmat_workbuf) h->thread_Kmat_workbuf = (void **)new KState();
    KState *k = kstate(h);
    if (k->budget == bytes) return;
    device_release_graph_kind(h, 2);
    kstate_release(k);
    k->budget = bytes;
}

// The block kernel's 64-bit form for every size (on = 1; tests): plans take it
// by themselves where offsets need it.  Releases the exchange plan.
void H2ERI_set_exchange_wide(H2ERI_p h, const int on) {
    if (!h) { set_error(ERR_ARG, "H2ERI_set_exchange_wide: null handle"); return; }
    if (!h->thread_Kmat_workbuf) h->thread_Kmat_workbuf = (void **)new KState();
    KState *k = kstate(h);
    if (k->wide == (on != 0)) return;
    device_release_graph_kind(h, 2);
    kstate_release(k);
    k->wide = on != 0;
}

}  // extern "C"
