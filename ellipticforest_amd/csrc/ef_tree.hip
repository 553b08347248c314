// ef_tree.hip -- gfx950 kernels of the tree levels of the HPS path: the 4-to-1 merges of
// the build stage (HPSAlgorithm::merge4to1 and its steps, src/HPSAlgorithm.hpp:497-518,
// 707-1009) and the family steps of the upward and downward sweeps (upwards4to1 :529-551,
// split1to4 :562-577), batched over whole tree levels.
//
// The reference forms X, S_RHS and H element by element, calls dgesv for S = X^-1 S_RHS and
// dgemm for T = blkdiag + H S (Matrix.hpp:827-953), one family at a time.  Here:
//  * X is inverted once per merge (blocked Gauss-Jordan in natural order with the multipliers
//    checked, going on with partial pivoting where one is large; every O(m^3) step a batched
//    MFMA product), so the upward sweep's mergeW_ is a product with X^-1 instead of a
//    re-factorisation per solve;
//  * S = X^-1 S_RHS and T = blkdiag + H S read S_RHS and H straight out of the children's
//    DtN maps (they are blocks of them, with signs), skipping their zero blocks;
//  * the sweeps' products run on register-resident batched GEMM kernels whose waves read their
//    operands in the v_mfma_f64_16x16x4_f64 layouts, the build's larger ones on tiles in LDS.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "ef_host.hpp"
#include "ef_kernels.hpp"
#include "ef_tree.hpp"

namespace efk {

typedef double td4 __attribute__((ext_vector_type(4)));
typedef double td2 __attribute__((ext_vector_type(2)));
// loads through the global address space: the descriptors' pointers are generic, and a generic
// (FLAT) load also counts against the LDS counter, so the compiler waits for every load in
// flight before each use -- which defeats the GEMM's software pipeline
__device__ inline td2 gld2(const double* p) { return *(const EF_GLOBAL td2*)gmem(p); }
__device__ inline double gld(const double* p) { return *gmem(p); }

typedef float tf4 __attribute__((ext_vector_type(4)));

__device__ inline td4 mfma_f64(double a, double b, td4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// v_mfma_f32_16x16x4_f32: the same operand layout (lane l: A[l%16][l/16], B[l/16][l%16]);
// the accumulator holds rows 4 (l/16) + v of column l%16 (the f64 instruction: rows 4 v + l/16)
__device__ inline tf4 mfma_f32(double a, double b, tf4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32((float)a, (float)b, c, 0, 0, 0);
}
template <bool F32>
using GemmAcc = std::conditional_t<F32, tf4, td4>;
template <bool F32>
__device__ inline GemmAcc<F32> mfma_acc(double a, double b, GemmAcc<F32> c) {
    if constexpr (F32) return mfma_f32(a, b, c);
    else return mfma_f64(a, b, c);
}

// lane `src`'s value of x in every lane (src uniform)
__device__ inline double readlane_f64(double x, int src) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), src);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(x), src);
    return __hiloint2double(hi, lo);
}



// ---------------------------------------------------------------------------------------
// Batched GEMM
// ---------------------------------------------------------------------------------------
// A B over k in [0, K) into this wave's 32 x (16 TN) block.  a0p / a1p: the lane's two
// A rows (r and r + 16, clamped into the matrix); bp[j]: B column (clamped) of column tile j.
// Within each block of 16 k values lane group q takes k = kb + 4q + s at MFMA step s: A is
// read as two 16-byte vectors per lane and row (a 128-byte row segment per lane group), B as
// one row segment of 16 consecutive columns per lane group and step.
// block-gather mode of segment 0: row offsets of each block's segment (hDiff: the two children's
// segments, subtracted; g: the side's segment alone)
// (MODE 1 subtracts the d1 segment, MODE 2 reads the d2 segment alone; MODE 0: B contiguous
// along k, MODE 3: B strided along k)
struct DiffRows {
    int dn, kbase;  // block size; absolute row of the segment's first k
    long long d2[4], d1[4];
};

// The factors alpha of a product's two segments are signs, applied to the accumulators once per segment
// (A scaled as it is loaded took a multiplication per MFMA on the unit the f64 MFMAs run on).
template <bool F32, int TN>
__device__ inline void flip_sign(GemmAcc<F32> (&acc)[2][TN]) {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = -acc[i][j];
}

template <int RT, int TN, bool F32, int MODE, int PD>
__device__ inline void gemm_segment(const double* __restrict__ a0p, const double* __restrict__ a1p,
                                    const double* const (&bp)[TN], long long ldb, int K,
                                    GemmAcc<F32> (&acc)[2][TN], const DiffRows& dr) {
    constexpr bool DIFF = MODE == 1 || MODE == 2;
    const int q = (int)(threadIdx.x & 63) >> 4;
    // hDiff rows: absolute row ka lies in interface block r = ka / dn; both children's offsets
    auto drow = [&](int ka, long long& o2, long long& o1) {
        const int r = ka / dr.dn, i = ka - r * dr.dn;
        o2 = pick4(dr.d2, r) + i;
        o1 = pick4(dr.d1, r) + i;
    };
    // the operands of block kb: A rows (two 16-byte vectors per row) and B columns
    // MODE 1 keeps both children's rows and subtracts them in the products: a subtraction at
    // load time would wait for the loads as soon as they are issued
    struct Blk {
        td2 x0, x1, y0, y1;
        double b[TN][4];
        double c[MODE == 1 ? TN : 1][4];
    };
    auto load = [&](int kb, Blk& o) {
        const int k = kb + 4 * q;
        o.x0 = gld2(a0p + k);
        o.x1 = gld2(a0p + k + 2);
        if (RT == 2) {
            o.y0 = gld2(a1p + k);
            o.y1 = gld2(a1p + k + 2);
        }
        if (DIFF) {  // four consecutive rows lie in one block (dn % 4 == 0)
            long long o2, o1;
            drow(dr.kbase + k, o2, o1);
            if (MODE == 1) {
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const td2 u0 = gld2(bp[j] + o2), u1 = gld2(bp[j] + o2 + 2);
                    const td2 v0 = gld2(bp[j] + o1), v1 = gld2(bp[j] + o1 + 2);
                    o.b[j][0] = u0[0]; o.b[j][1] = u0[1]; o.b[j][2] = u1[0]; o.b[j][3] = u1[1];
                    o.c[j][0] = v0[0]; o.c[j][1] = v0[1]; o.c[j][2] = v1[0]; o.c[j][3] = v1[1];
                }
            } else {
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const td2 u0 = gld2(bp[j] + o2), u1 = gld2(bp[j] + o2 + 2);
                    o.b[j][0] = u0[0]; o.b[j][1] = u0[1]; o.b[j][2] = u1[0]; o.b[j][3] = u1[1];
                }
            }
        } else if (MODE == 0) {  // B contiguous along k: two 16-byte vectors per column
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const td2 u0 = gld2(bp[j] + k), u1 = gld2(bp[j] + k + 2);
                o.b[j][0] = u0[0]; o.b[j][1] = u0[1]; o.b[j][2] = u1[0]; o.b[j][3] = u1[1];
            }
        } else {
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int s = 0; s < 4; s++) o.b[j][s] = gld(bp[j] + (long long)(k + s) * ldb);
        }
    };
    auto mma = [&](const Blk& o) {
        const double a0[4] = {o.x0[0], o.x0[1], o.x1[0], o.x1[1]};
        double a1[4] = {0.0, 0.0, 0.0, 0.0};
        if (RT == 2) {
            a1[0] = o.y0[0]; a1[1] = o.y0[1]; a1[2] = o.y1[0]; a1[3] = o.y1[1];
        }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const double bv = MODE == 1 ? o.b[j][s] - o.c[MODE == 1 ? j : 0][s] : o.b[j][s];
                acc[0][j] = mfma_acc<F32>(a0[s], bv, acc[0][j]);
                if (RT == 2) acc[1][j] = mfma_acc<F32>(a1[s], bv, acc[1][j]);
            }
    };
    const int nfull = K / 16;
    int kb = 0;
    if (nfull > 0) {
        // software pipeline of depth PD: block b lives in buf[b % PD]; while block b's MFMAs run,
        // blocks b + 1 .. b + PD - 1 are in flight, and block b + PD is issued into the slot b
        // frees -- no buffer is copied to another (a copy waits for its loads).  Measured at 64
        // right-hand sides, adaptive Poisson sweep GEMMs: PD = 2 0.871 ms, 3 0.969 ms, 4 0.996 ms
        // (more registers, fewer waves per SIMD); a cur/next pair with a copy 0.948 ms.  The split-K
        // kernel, whose waves are few and whose ranges are short, takes PD = 3.
        // The steady-state loop issues its loads unconditionally, so the loop head sees one
        // order of outstanding loads and waits for the older block only (a conditional load
        // there makes the wait counts cover both blocks).
        Blk buf[PD];
        if (nfull >= PD) {
#pragma unroll
            for (int j = 0; j < PD; j++) load(16 * j, buf[j]);
            int i = 0;
            for (; i + 2 * PD <= nfull; i += PD) {
#pragma unroll
                for (int j = 0; j < PD; j++) {
                    mma(buf[j]);
                    load(16 * (i + j + PD), buf[j]);
                }
            }
            // PD <= nfull - i < 2 PD: one round with the last loads, then the blocks left
#pragma unroll
            for (int j = 0; j < PD; j++) {
                mma(buf[j]);
                if (i + j + PD < nfull) load(16 * (i + j + PD), buf[j]);
            }
            i += PD;
#pragma unroll
            for (int j = 0; j < PD - 1; j++)
                if (i + j < nfull) mma(buf[j]);
        } else {
#pragma unroll
            for (int j = 0; j < PD - 1; j++)
                if (j < nfull) load(16 * j, buf[j]);
#pragma unroll
            for (int j = 0; j < PD - 1; j++)
                if (j < nfull) mma(buf[j]);
        }
        kb = 16 * nfull;
    }
    if (kb < K) {  // partial last block: k >= K contributes zero (addresses clamped to K - 1)
        const int k = kb + 4 * q;
        double a0[4], a1[4], b[TN][4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const bool ok = k + s < K;
            const int kk = ok ? k + s : K - 1;
            const double x = gld(a0p + kk);
            a0[s] = ok ? x : 0.0;
            if (RT == 2) {
                const double y = gld(a1p + kk);
                a1[s] = ok ? y : 0.0;
            }
            if (DIFF) {
                long long o2, o1;
                drow(dr.kbase + kk, o2, o1);
#pragma unroll
                for (int j = 0; j < TN; j++) b[j][s] = MODE == 1 ? gld(bp[j] + o2) - gld(bp[j] + o1) : gld(bp[j] + o2);
            } else {
#pragma unroll
                for (int j = 0; j < TN; j++) b[j][s] = gld(bp[j] + (long long)kk * ldb);
            }
        }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                acc[0][j] = mfma_acc<F32>(a0[s], b[j][s], acc[0][j]);
                if (RT == 2) acc[1][j] = mfma_acc<F32>(a1[s], b[j][s], acc[1][j]);
            }
    }
}

template <int RT, int TN, bool F32>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8)))
tree_gemm_kernel(const TreeGemm* __restrict__ probs,
                                                         const int* __restrict__ start,
                                                         const int* __restrict__ wprob, int nwaves) {
    const int w = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (w >= nwaves) return;  // uniform per wave
    const int lo = __builtin_amdgcn_readfirstlane(wprob[w]);  // the wave's problem (a table, not a search)
    const TreeGemm p = probs[lo];
    const int lane = threadIdx.x & 63, q = lane >> 4, r = lane & 15;
    constexpr int RW = 16 * RT, CW = 16 * TN;
    const int tm = (p.M + RW - 1) / RW, tn = (p.N + CW - 1) / CW;
    const int t = w - start[lo];
    const int row0 = (t / tn) * RW, col0 = (t % tn) * CW;
    int rows[RT];
#pragma unroll
    for (int i = 0; i < RT; i++) rows[i] = min(row0 + 16 * i + r, p.M - 1);
    int cj[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) cj[j] = min(col0 + 16 * j + r, p.N - 1);
    GemmAcc<F32> acc[2][TN];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = GemmAcc<F32>{0, 0, 0, 0};
    // this wave sums both segments over their whole k range (split-K launches run on
    // tree_gemm_split_kernel)
    const int kb0 = 0, ke0 = p.K0, kb1 = 0, ke1 = p.K1;
    // C (when the product adds to it) loaded before the products, so its latency overlaps
    // them; rows and columns clamped as the stores are guarded
    double cv[RT][TN][4];
    bool keep[TN];  // (a value that is not kept is dropped after the products: no wait before them)
    const bool has_c = p.C != nullptr;
    if (has_c) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int cb = p.cn > 0 ? cj[j] / p.cn : 0;
            const double* cp = p.cn > 0 ? (cb == p.cb1 ? p.C1 : p.C) + (cj[j] - cb * p.cn) : p.C + (long long)cj[j] * p.ccs;
            keep[j] = p.cn == 0 || cb == p.cb0 || cb == p.cb1;
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    cv[i][j][v] = gld(cp + (long long)min(row0 + 16 * i + (F32 ? 4 * q + v : 4 * v + q), p.M - 1) * p.ldc);
        }
    }
    DiffRows dr;
    dr.dn = p.dn;
    dr.kbase = kb0;
#pragma unroll
    for (int r4 = 0; r4 < 4; r4++) { dr.d2[r4] = p.d2[r4]; dr.d1[r4] = p.d1[r4]; }
    if (ke0 > kb0) {
        const double* bp[TN];
        if (p.dn > 0) {  // hDiff mode: column bases, rows resolved per interface block
#pragma unroll
            for (int j = 0; j < TN; j++) bp[j] = p.B0 + (long long)cj[j] * p.bcs;
            const double* a0 = p.A0 + (long long)rows[0] * p.lda0 + kb0;
            const double* a1 = p.A0 + (long long)rows[RT - 1] * p.lda0 + kb0;
            if (p.dsub) gemm_segment<RT, TN, F32, 1, 2>(a0, a1, bp, 1, ke0 - kb0, acc, dr);
            else gemm_segment<RT, TN, F32, 2, 2>(a0, a1, bp, 1, ke0 - kb0, acc, dr);
        } else {
#pragma unroll
            for (int j = 0; j < TN; j++) bp[j] = p.B0 + (long long)kb0 * p.ldb0 + (long long)cj[j] * p.bcs;
            const double* a0 = p.A0 + (long long)rows[0] * p.lda0 + kb0;
            const double* a1 = p.A0 + (long long)rows[RT - 1] * p.lda0 + kb0;
            if (p.ldb0 == 1) gemm_segment<RT, TN, F32, 0, 2>(a0, a1, bp, 1, ke0 - kb0, acc, dr);
            else gemm_segment<RT, TN, F32, 3, 2>(a0, a1, bp, p.ldb0, ke0 - kb0, acc, dr);
        }
    }
    if (ke1 > kb1) {
        if (p.alpha0 != p.alpha1) flip_sign<F32>(acc);
        const double* bp[TN];
#pragma unroll
        for (int j = 0; j < TN; j++) bp[j] = p.B1 + (long long)kb1 * p.ldb1 + (long long)cj[j] * p.bcs;
        const double* a0 = p.A1 + (long long)rows[0] * p.lda1 + kb1;
        const double* a1 = p.A1 + (long long)rows[RT - 1] * p.lda1 + kb1;
        if (p.ldb1 == 1) gemm_segment<RT, TN, F32, 0, 2>(a0, a1, bp, 1, ke1 - kb1, acc, dr);
        else gemm_segment<RT, TN, F32, 3, 2>(a0, a1, bp, p.ldb1, ke1 - kb1, acc, dr);
    }
    if ((ke1 > kb1 ? p.alpha1 : p.alpha0) < 0.0) flip_sign<F32>(acc);
    // with RT = 1 only the first accumulator row holds products
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = row0 + 16 * i + (F32 ? 4 * q + v : 4 * v + q), col = col0 + 16 * j + r;
                if (row < p.M && col < p.N) {
                    double o = (double)acc[i][j][v];
                    if (has_c) o += keep[j] ? p.beta * cv[i][j][v] : 0.0;
                    *gmem(p.D + (long long)row * p.ldd + (long long)col * p.dcs) = o;
                }
            }
}

template __global__ void tree_gemm_kernel<1, 1, false>(const TreeGemm*, const int*, const int*, int);
template __global__ void tree_gemm_kernel<1, 2, false>(const TreeGemm*, const int*, const int*, int);
template __global__ void tree_gemm_kernel<2, 2, false>(const TreeGemm*, const int*, const int*, int);
template __global__ void tree_gemm_kernel<1, 1, true>(const TreeGemm*, const int*, const int*, int);
template __global__ void tree_gemm_kernel<1, 2, true>(const TreeGemm*, const int*, const int*, int);
template __global__ void tree_gemm_kernel<2, 2, true>(const TreeGemm*, const int*, const int*, int);

// The build's S and T products of merges with n >= 32 (row-major operands, K a multiple of 16, M and N of
// the tile): one workgroup per (32 WR) x (32 WC) tile of D, its WR x WC waves a 32 x 32 block each, A and
// B staged through LDS in blocks of 16 k values, two blocks' loads in flight during the MFMAs of the
// one before.  Bound: the f64 matrix cores.  One wave per 32 x 32 block reading its own operands
// (tree_gemm_kernel) asks the L1 for 32 bytes per cycle and CU at full matrix rate and holds 2 waves per
// SIMD; LDS tiles halve that and 4 waves fit.  n = 512, T (34 GFLOP): 724 us (47 TFLOP/s) -> 554
// (62; the card's large matrix product reaches 72); 256 merges of n = 32: S 48 -> 42, T 97 -> 78 us; S and
// T of 1,024 leaves of 32^2: 2.32 -> 1.79 ms.  Of that: one block in flight instead of two 604 us
// for the n = 512 product; workgroups in launch order, so that each XCD's L2 sees every tile, 578.
// Each element sums its k range in tree_gemm_kernel's order.
template <int WR, int WC>
__global__ void __launch_bounds__(256) tree_gemm_lds_kernel(const TreeGemm* __restrict__ probs,
                                                            const int* __restrict__ start,
                                                            const int* __restrict__ gprob, int ngroups) {
    static_assert(WR * WC == 4, "four waves");
    constexpr int TR = 32 * WR, TC = 32 * WC;
    constexpr int LA = 18, LB = TC + 4;  // LDS rows of A and B in doubles: each read covers every bank once
    __shared__ __attribute__((aligned(16))) double sa[2][TR * LA];
    __shared__ __attribute__((aligned(16))) double sb[2][16 * LB];
    const int bid = (int)blockIdx.x, n8 = ngroups / 8;
    if (bid >= ngroups) return;  // uniform per workgroup
    // (consecutive workgroups go to the 8 XCDs in turn: each gets a run of consecutive tiles)
    const int g = bid < 8 * n8 ? (bid & 7) * n8 + (bid >> 3) : bid;
    const int lo = __builtin_amdgcn_readfirstlane(gprob[g]);
    const TreeGemm p = probs[lo];
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, r = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = g - start[lo], tm = p.M / TR;
    const int row0 = (t % tm) * TR, col0 = (t / tm) * TC;
    const int wr = 32 * (wave / WC), wc = 32 * (wave % WC);
    GemmAcc<false> acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = GemmAcc<false>{0, 0, 0, 0};
    const int nb0 = p.K0 / 16, nb = nb0 + p.K1 / 16;
    struct Blk {
        td2 x[WR], y[WC];
    };
    // a lane's share of a block: WR vectors of A (eight to a row), WC of B (16 WC to a row)
    auto load = [&](int b, Blk& o) {  // block b of the concatenated k range (past its end: the last one again)
        b = min(b, nb - 1);
        const bool s1 = b >= nb0;  // uniform
        const int k = 16 * (s1 ? b - nb0 : b);
        const double* A = (s1 ? p.A1 : p.A0) + k;
        const double* B = (s1 ? p.B1 : p.B0) + col0;
        const int lda = s1 ? p.lda1 : p.lda0, ldb = s1 ? p.ldb1 : p.ldb0;
#pragma unroll
        for (int v = 0; v < WR; v++) o.x[v] = gld2(A + (long long)(row0 + 32 * v + (tid >> 3)) * lda + 2 * (tid & 7));
#pragma unroll
        for (int v = 0; v < WC; v++) {
            const int e = tid + 256 * v;
            o.y[v] = gld2(B + (long long)(k + e / (16 * WC)) * ldb + 2 * (e % (16 * WC)));
        }
    };
    auto stage = [&](int slot, const Blk& o) {
#pragma unroll
        for (int v = 0; v < WR; v++) *(td2*)&sa[slot][(32 * v + (tid >> 3)) * LA + 2 * (tid & 7)] = o.x[v];
#pragma unroll
        for (int v = 0; v < WC; v++) {
            const int e = tid + 256 * v;
            *(td2*)&sb[slot][e / (16 * WC) * LB + 2 * (e % (16 * WC))] = o.y[v];
        }
    };
    Blk buf[2];
    load(0, buf[0]);
    load(1, buf[1]);
    stage(0, buf[0]);
    __syncthreads();
    for (int b0 = 0; b0 < nb; b0 += 2) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int b = b0 + h;
            if (b >= nb) break;  // uniform
            if (b == nb0 && p.alpha0 != p.alpha1) flip_sign<false>(acc);
            load(b + 2, buf[h]);
            const double* la = &sa[h][(wr + r) * LA + 4 * q];
            const double* lb = &sb[h][4 * q * LB + wc + r];
            double a[2][4], v[2][4];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const td2 u0 = *(const td2*)(la + 16 * i * LA), u1 = *(const td2*)(la + 16 * i * LA + 2);
                a[i][0] = u0[0]; a[i][1] = u0[1]; a[i][2] = u1[0]; a[i][3] = u1[1];
            }
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int s = 0; s < 4; s++) v[j][s] = lb[s * LB + 16 * j];
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int i = 0; i < 2; i++) acc[i][j] = mfma_f64(a[i][s], v[j][s], acc[i][j]);
            stage(1 - h, buf[1 - h]);  // (block b - 1 was read from that slot: every wave is past the barrier after it)
            __syncthreads();
        }
    }
    if ((p.K1 > 0 ? p.alpha1 : p.alpha0) < 0.0) flip_sign<false>(acc);
    // C: a wave's columns lie in one column block (cn a multiple of 32)
    const int cb = p.cn > 0 ? (col0 + wc) / p.cn : 0;
    const double* C = p.C;
    if (p.cn > 0) C = cb == p.cb0 ? p.C - (long long)cb * p.cn : cb == p.cb1 ? p.C1 - (long long)cb * p.cn : nullptr;
    if (C) {  // uniform
        double cv[2][2][4];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    cv[i][j][v] = gld(C + (long long)(row0 + wr + 16 * i + 4 * v + q) * p.ldc + col0 + wc + 16 * j + r);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[i][j][v] += p.beta * cv[i][j][v];
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = row0 + wr + 16 * i + 4 * v + q, col = col0 + wc + 16 * j + r;
                *gmem(p.D + (long long)row * p.ldd + col) = acc[i][j][v];
            }
}

template __global__ void tree_gemm_lds_kernel<1, 4>(const TreeGemm*, const int*, const int*, int);
template __global__ void tree_gemm_lds_kernel<2, 2>(const TreeGemm*, const int*, const int*, int);
template __global__ void tree_gemm_lds_kernel<4, 1>(const TreeGemm*, const int*, const int*, int);

// Split-K inside the workgroup: workgroup g computes the 16 x 16 output tile g - start[p] of
// problem p = gprob[g]; its wave w sums chunk w, k in [w kc, (w + 1) kc), of the concatenated k
// range of the two segments (a chunk may span both), and wave 0 adds the chunks' partials in
// chunk order, then beta C.  The chunks depend on the problem only, never on N, so a column's
// result does not depend on the batch; nothing goes through HBM between the chunks and no second
// launch sums them.  blockDim = 64 x (the launch's largest chunk count, <= 16).
__global__ void __launch_bounds__(1024) tree_gemm_split_kernel(const TreeGemm* __restrict__ probs,
                                                                const int* __restrict__ start,
                                                                const int* __restrict__ gprob, int ngroups) {
    __shared__ double part[16][4][64];  // [chunk][accumulator slot][lane], 32 KiB
    const int g = (int)blockIdx.x;
    if (g >= ngroups) return;  // uniform per workgroup
    const int lo = __builtin_amdgcn_readfirstlane(gprob[g]);
    const TreeGemm p = probs[lo];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int q = lane >> 4, r = lane & 15;
    const int tn = (p.N + 15) / 16;
    const int t = g - start[lo];
    const int row0 = (t / tn) * 16, col0 = (t % tn) * 16;
    const int rowc = min(row0 + r, p.M - 1), cj = min(col0 + r, p.N - 1);
    GemmAcc<false> acc[2][1];
    acc[0][0] = GemmAcc<false>{0, 0, 0, 0};
    acc[1][0] = GemmAcc<false>{0, 0, 0, 0};
    const int K = p.K0 + p.K1, kbeg = wave * p.kc, kend = min(kbeg + p.kc, K);
    // wave 0 loads C before its products (it alone writes D)
    double cv[4] = {0.0, 0.0, 0.0, 0.0};
    if (wave == 0 && p.C) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = min(row0 + 4 * v + q, p.M - 1);
            cv[v] = gld(p.C + (long long)row * p.ldc + (long long)cj * p.ccs);
        }
    }
    if (kbeg < K) {  // uniform per wave
        const int kb0 = min(kbeg, p.K0), ke0 = min(kend, p.K0);
        const int kb1 = max(kbeg, p.K0) - p.K0, ke1 = max(kend, p.K0) - p.K0;
        DiffRows dr;
        dr.dn = p.dn;
        dr.kbase = kb0;
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) { dr.d2[r4] = p.d2[r4]; dr.d1[r4] = p.d1[r4]; }
        if (ke0 > kb0) {
            const double* bp[1];
            const double* a0 = p.A0 + (long long)rowc * p.lda0 + kb0;
            if (p.dn > 0) {
                bp[0] = p.B0 + (long long)cj * p.bcs;
                if (p.dsub) gemm_segment<1, 1, false, 1, 3>(a0, a0, bp, 1, ke0 - kb0, acc, dr);
                else gemm_segment<1, 1, false, 2, 3>(a0, a0, bp, 1, ke0 - kb0, acc, dr);
            } else {
                bp[0] = p.B0 + (long long)kb0 * p.ldb0 + (long long)cj * p.bcs;
                if (p.ldb0 == 1) gemm_segment<1, 1, false, 0, 3>(a0, a0, bp, 1, ke0 - kb0, acc, dr);
                else gemm_segment<1, 1, false, 3, 3>(a0, a0, bp, p.ldb0, ke0 - kb0, acc, dr);
            }
        }
        if (ke1 > kb1) {
            if (p.alpha0 != p.alpha1) flip_sign<false>(acc);
            const double* bp[1] = {p.B1 + (long long)kb1 * p.ldb1 + (long long)cj * p.bcs};
            const double* a1 = p.A1 + (long long)rowc * p.lda1 + kb1;
            if (p.ldb1 == 1) gemm_segment<1, 1, false, 0, 3>(a1, a1, bp, 1, ke1 - kb1, acc, dr);
            else gemm_segment<1, 1, false, 3, 3>(a1, a1, bp, p.ldb1, ke1 - kb1, acc, dr);
        }
        if ((ke1 > kb1 ? p.alpha1 : p.alpha0) < 0.0) flip_sign<false>(acc);
    }
    if (wave > 0) {
#pragma unroll
        for (int v = 0; v < 4; v++) part[wave][v][lane] = acc[0][0][v];
    }
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int row = row0 + 4 * v + q, col = col0 + r;
        if (row < p.M && col < p.N) {
            double o = 0.0;
            o += acc[0][0][v];
            for (int c = 1; c < p.nks; c++) o += part[c][v][lane];
            if (p.C) o += p.beta * cv[v];
            *gmem(p.D + (long long)row * p.ldd + (long long)col * p.dcs) = o;
        }
    }
}

// ---------------------------------------------------------------------------------------
// Gauss-Jordan inversion
// ---------------------------------------------------------------------------------------
// Tournament LU of the panel (columns k .. k+nb) with partial pivoting, fused with the step's
// pivot bookkeeping.  One workgroup of 64 WAVES threads holds up to 64 WAVES RPL panel rows,
// RPL whole rows (32 columns) per lane in registers, row q NT + tid of the chunk in slot q.
// STAGE 0: the rows of chunk blockIdx.x (positions k + ch * rows + i); STAGE 1: the candidates
// of every chunk (a.cand).  Ties go to the lower position, as idamax takes the first maximum.
// FIN = false: the nb rows pivoted on, in order, are the chunk's candidates.  FIN = true (one
// chunk, or stage 1): they are the pivots of the step, and the same workgroup forms P^-1 of
// the pivot block, the LAPACK-order interchanges (ipiv) and the position -> row map (src).
// Per column (all 32 unrolled, so register indices are compile-time constants): each lane's
// best row, one DPP argmax per wave, the wave's best row published to LDS with its value, one
// barrier, then every thread combines the waves' candidates and reads the pivot row from the
// winner's slot (slots alternate by column parity, so column J + 1 never overwrites what a
// slower wave still reads for column J).
constexpr int GJ_NONE = 0x7fffffff;
template <int RPL>
struct PanelRows {
    double v[RPL][GJ_NB];  // the rows (multipliers left of the pivot column)
    int pos[RPL];          // position of each row at the start of the step (its name)
    int cur[RPL];          // its position now, after the step's interchanges so far
    bool act[RPL];         // row present and not yet pivoted on
};
// Pivot order key: current position, then name (both < GJ_MAXM = 2^12).
__device__ inline int piv_key(int cur, int pos) { return (cur << 12) | pos; }
template <int WAVES, bool FIN>
struct PanelShared {
    union {
        double cand[2][WAVES][GJ_NB];   // each wave's best row, by column parity
        double A[2][GJ_NB][GJ_NB];      // FIN: in-place Gauss-Jordan on P, ping-pong
    } u;
    double red_v[2][WAVES];
    int red_p[2][WAVES];
    int piv[GJ_NB];  // pivot position chosen for each column (-1: none)
    int top_row[GJ_NB], opos[GJ_NB], orow[GJ_NB];
    int nout;
};

// Wave reductions into lane 63 through DPP lane shifts: row shifts 1, 2, 4, 8 leave each
// 16-lane row's result in its lane 15; row_bcast:15 folds rows 0 -> 1 and 2 -> 3, row_bcast:31
// folds lane 31 into rows 2 and 3.  Lanes without a source lane (or in rows outside the row
// mask) see the identity.
template <int CTRL, int ROWMASK>
__device__ inline double max_dpp(double v) {  // identity -1 (every candidate is >= 0)
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWMASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(-1.0), __double2hiint(v), CTRL, ROWMASK, 0xf, false);
    return fmax(v, __hiloint2double(hi, lo));
}
template <int CTRL, int ROWMASK>
__device__ inline int min_dpp(int p) {  // identity GJ_NONE
    return min(p, __builtin_amdgcn_update_dpp(GJ_NONE, p, CTRL, ROWMASK, 0xf, false));
}
__device__ inline double wave_max(double v) {
    v = max_dpp<0x111, 0xf>(v);
    v = max_dpp<0x112, 0xf>(v);
    v = max_dpp<0x114, 0xf>(v);
    v = max_dpp<0x118, 0xf>(v);
    v = max_dpp<0x142, 0xa>(v);
    v = max_dpp<0x143, 0xc>(v);
    return v;
}
__device__ inline int wave_min(int p) {
    p = min_dpp<0x111, 0xf>(p);
    p = min_dpp<0x112, 0xf>(p);
    p = min_dpp<0x114, 0xf>(p);
    p = min_dpp<0x118, 0xf>(p);
    p = min_dpp<0x142, 0xa>(p);
    p = min_dpp<0x143, 0xc>(p);
    return p;
}
__device__ inline double readlane_dyn(double x, int src) { return readlane_f64(x, src); }

// Column J: the pivot is the largest |entry| among the active rows, the lowest current position
// among equal ones (idamax takes the first maximum of the interchanged column): a wave max of
// the values, then a wave min of the (position, name) keys of the lanes that hold that maximum.
// After the choice the row at position k + J takes the pivot row's position (the interchange).
// One wave reads the pivot row straight from its owner lane (readlane); several waves publish
// their candidate rows in LDS.
template <int J, int WAVES, int RPL, int STAGE, bool FIN>
__device__ __attribute__((always_inline)) inline void panel_column(PanelRows<RPL>& R, PanelShared<WAVES, FIN>& sh,
                                                                   int base, int top0) {
    constexpr int BUF = J & 1;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double lv = -1.0;  // the lane's best row
    int lk = GJ_NONE;
#pragma unroll
    for (int q = 0; q < RPL; q++) {
        const double x = R.act[q] ? fabs(R.v[q][J]) : -1.0;
        const int key = piv_key(R.cur[q], R.pos[q]);
        const bool take = x > lv || (x == lv && R.act[q] && key < lk);
        lk = take ? key : lk;
        lv = take ? x : lv;
    }
    const double wmax = readlane_f64(wave_max(lv), 63);
    const int wkey = __builtin_amdgcn_readlane(wave_min((lv == wmax) ? lk : GJ_NONE), 63);
    const int wbp = (wkey == GJ_NONE) ? GJ_NONE : (wkey & 4095);
    int pkey = wkey;
    double pr[GJ_NB];  // pivot row, columns J..
    int pp = wbp;
    if (WAVES == 1) {
        if (tid == 0) sh.piv[J] = (pp == GJ_NONE) ? -1 : pp;
        if (pp == GJ_NONE) return;  // uniform: no row left in the panel
        // STAGE 0: row named base + q * 64 + lane; STAGE 1 (several waves) never gets here
        const int off = pp - base, ol = off & 63, oq = off >> 6;
#pragma unroll
        for (int c = J; c < GJ_NB; c++) {
            double x = R.v[0][c];
#pragma unroll
            for (int q = 1; q < RPL; q++) x = (oq == q) ? R.v[q][c] : x;
            pr[c] = readlane_dyn(x, ol);
        }
    } else {
#pragma unroll
        for (int q = 0; q < RPL; q++)
            if (R.act[q] && R.pos[q] == wbp) {  // the wave's best row: columns J.. are what the pivot row needs
#pragma unroll
                for (int c = J; c < GJ_NB; c++) sh.u.cand[BUF][wave][c] = R.v[q][c];
            }
        if (lane == 63) { sh.red_v[BUF][wave] = wmax; sh.red_p[BUF][wave] = wkey; }
        __syncthreads();
        double best = sh.red_v[BUF][0];
        int ww = 0;
        pkey = sh.red_p[BUF][0];
#pragma unroll
        for (int w2 = 1; w2 < WAVES; w2++) {
            const double v2 = sh.red_v[BUF][w2];
            const int p2 = sh.red_p[BUF][w2];
            const bool take = v2 > best || (v2 == best && p2 < pkey);
            best = take ? v2 : best;
            pkey = take ? p2 : pkey;
            ww = take ? w2 : ww;
        }
        pp = (pkey == GJ_NONE) ? GJ_NONE : (pkey & 4095);
        if (tid == 0) sh.piv[J] = (pp == GJ_NONE) ? -1 : pp;
        if (pp == GJ_NONE) return;  // uniform: no row left in the panel
        const double* prow = sh.u.cand[BUF][ww];
#pragma unroll
        for (int c = J; c < GJ_NB; c++) pr[c] = prow[c];
    }
    const int pcur = pkey >> 12, top = top0 + J;
#pragma unroll
    for (int q = 0; q < RPL; q++) {
        if (R.act[q] && R.pos[q] == pp) R.act[q] = false;
        else if (R.act[q] && R.cur[q] == top) R.cur[q] = pcur;  // the interchange
    }
    const double piv = pr[J];
    const double rp = (piv != 0.0) ? 1.0 / piv : 0.0;
    // branch-free: rows that are not active (pivoted on, absent) take l = 0 and keep their values
#pragma unroll
    for (int q = 0; q < RPL; q++) {
        const double l = R.act[q] ? R.v[q][J] * rp : 0.0;  // multiplier, kept in place
        R.v[q][J] = R.act[q] ? l : R.v[q][J];
#pragma unroll
        for (int c = J + 1; c < GJ_NB; c++) R.v[q][c] -= l * pr[c];
    }
}

template <int WAVES, int RPL, int STAGE, bool FIN, int... J>
__device__ __attribute__((always_inline)) inline void panel_columns(std::integer_sequence<int, J...>, PanelRows<RPL>& R,
                                                                    PanelShared<WAVES, FIN>& sh, int nbb, int base,
                                                                    int top0) {
    // columns past nbb (a last step narrower than GJ_NB) are skipped; nbb is uniform
    ((J < nbb ? panel_column<J, WAVES, RPL, STAGE, FIN>(R, sh, base, top0) : void()), ...);
}

template <int STAGE, int WAVES, int RPL, bool FIN>
__global__ void __launch_bounds__(64 * WAVES) gj_panel_kernel(GJArgs a) {
    __shared__ PanelShared<WAVES, FIN> sh;
    constexpr int NT = 64 * WAVES, ROWS = NT * RPL;
    const int b = blockIdx.y, ch = blockIdx.x;
    const int m = a.m, k = a.k, nbb = min(GJ_NB, m - k);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const double* W = a.Wa + (long long)b * m * m;
    PanelRows<RPL> R;
#pragma unroll
    for (int q = 0; q < RPL; q++) {
        const int i = q * NT + tid;  // row of the chunk
        if (STAGE == 0) {
            R.pos[q] = k + ch * ROWS + i;
            R.act[q] = R.pos[q] < m;
        } else {
            const int p = (i < a.nch * GJ_NB) ? a.cand[(long long)b * GJ_MAXCH * GJ_NB + i] : -1;
            R.act[q] = p >= k && p < m;
            R.pos[q] = R.act[q] ? p : GJ_NONE;
        }
        R.cur[q] = R.pos[q];
        const double* rowp = W + (long long)(R.act[q] ? R.pos[q] : k) * m + k;
#pragma unroll
        for (int c = 0; c < GJ_NB; c++)  // columns k + c < m of a row of the matrix
            R.v[q][c] = (R.act[q] && c < nbb) ? rowp[c] : 0.0;
    }
    if (tid < GJ_NB) sh.piv[tid] = -1;
    static_assert(WAVES > 1 || STAGE == 0, "one-wave panels hold chunk rows in position order");
    // position k + J is the top of column J (a chunk's own first rows in the tournament stage)
    panel_columns<WAVES, RPL, STAGE, FIN>(std::make_integer_sequence<int, GJ_NB>{}, R, sh, nbb, k + ch * ROWS,
                                          STAGE == 0 ? k + ch * ROWS : k);
    __syncthreads();
    if (!FIN) {
        if (tid < GJ_NB) a.cand[((long long)b * GJ_MAXCH + ch) * GJ_NB + tid] = sh.piv[tid];
        return;
    }
    // P^-1: in-place Gauss-Jordan on P in LDS by the whole workgroup, P = the pivot rows (in
    // pivot order) as they were at the start of the step.  Step j leaves column j holding column j
    // of the inverse: rp = 1/p_jj on the diagonal, -a_rj rp elsewhere (what [P | I] elimination
    // puts in the identity's column j), and row j scaled by rp.  The order is the one partial
    // pivoting chose, so the multipliers below the diagonal are bounded by 1 and no further
    // pivoting is needed.  Beyond nbb the block is the identity.
    for (int e = tid; e < GJ_NB * GJ_NB; e += NT) {
        const int r = e / GJ_NB, c = e % GJ_NB;
        double x = (r == c) ? 1.0 : 0.0;
        const int pr = sh.piv[r];
        if (r < nbb && c < nbb && pr >= 0) x = W[(long long)pr * m + k + c];
        sh.u.A[0][r][c] = x;
    }
    __syncthreads();
    int zero = 0;
    for (int j = 0; j < nbb; j++) {
        const int cur = j & 1, nxt = cur ^ 1;
        const double pv = sh.u.A[cur][j][j];
        if (zero == 0 && (pv == 0.0 || sh.piv[j] < 0)) zero = j + 1;
        const double rp = (pv != 0.0) ? 1.0 / pv : 0.0;
        // NT is a multiple of GJ_NB: each thread keeps one column c and rows r0 + i NT / GJ_NB;
        // every read of the step is issued before its writes
        constexpr int RR = GJ_NB * GJ_NB / NT;
        const int c = tid % GJ_NB, r0 = tid / GJ_NB;
        const double rowj = (c == j) ? rp : sh.u.A[cur][j][c] * rp;
        double arj[RR], arc[RR];
#pragma unroll
        for (int i = 0; i < RR; i++) {
            const int r = r0 + i * (NT / GJ_NB);
            arj[i] = sh.u.A[cur][r][j];
            arc[i] = sh.u.A[cur][r][c];
        }
#pragma unroll
        for (int i = 0; i < RR; i++) {
            const int r = r0 + i * (NT / GJ_NB);
            double out;
            if (r == j) out = rowj;
            else if (c == j) out = -arj[i] * rp;
            else out = arc[i] - arj[i] * rowj;
            sh.u.A[nxt][r][c] = out;
        }
        __syncthreads();
    }
    {
        const int fin = nbb & 1;
        double* Pinv = a.Pinv + (long long)b * GJ_NB * GJ_NB;
        for (int e = tid; e < GJ_NB * GJ_NB; e += NT) {
            const int r = e / GJ_NB, c = e % GJ_NB;
            Pinv[e] = (r < nbb && c < nbb) ? sh.u.A[fin][r][c] : 0.0;
        }
    }
    if (wave == 0) {
        // interchanges (LAPACK order: position k+j with the chosen row's current position)
        int top = k + lane;      // row now at position k + lane (lanes < nbb)
        int op = -1, orw = -1;   // entry `lane` of the positions beyond the panel that changed row
        int nout = 0, mine = k + lane;
        for (int j = 0; j < nbb; j++) {
            const int target = sh.piv[j];
            const int apos = k + j;
            int t = apos;
            if (target >= 0) {
                const unsigned long long m1 = __ballot(lane >= j && lane < nbb && top == target);
                if (m1) {
                    t = k + __ffsll(m1) - 1;
                } else {
                    const unsigned long long m2 = __ballot(lane < nout && orw == target);
                    t = m2 ? __shfl(op, __ffsll(m2) - 1) : target;
                }
                const int row_a = __shfl(top, j);
                if (t != apos) {
                    if (lane == j) top = target;
                    if (t < k + nbb) {
                        if (lane == t - k) top = row_a;
                    } else {
                        const unsigned long long m3 = __ballot(lane < nout && op == t);
                        const int o = m3 ? __ffsll(m3) - 1 : nout;
                        if (lane == o) { op = t; orw = row_a; }
                        if (!m3) nout++;
                    }
                }
            }
            if (lane == j) mine = t;
        }
        if (lane < GJ_NB) {
            sh.top_row[lane] = top;
            sh.opos[lane] = op;
            sh.orow[lane] = orw;
            const int target = (lane < nbb) ? sh.piv[lane] : -1;
            a.prow[(long long)b * GJ_NB + lane] = (target >= 0) ? target : min(k + lane, m - 1);
            if (lane < nbb) a.ipiv[(long long)b * m + k + lane] = mine;
        }
        if (lane == 0) {
            sh.nout = nout;
            if (zero && a.info[b] == 0) a.info[b] = k + zero;
        }
    }
    __syncthreads();
    int* src = a.src + (long long)b * m;
    const int nout = sh.nout;
    for (int r = tid; r < m; r += NT) {
        int s = r;
        if (r >= k && r < k + nbb) s = sh.top_row[r - k];
        else
            for (int o = 0; o < nout; o++)
                if (sh.opos[o] == r) s = sh.orow[o];
        src[r] = s;
    }
}

template __global__ void gj_panel_kernel<0, 1, 1, true>(GJArgs);
template __global__ void gj_panel_kernel<0, 1, 2, true>(GJArgs);
template __global__ void gj_panel_kernel<0, 2, 2, true>(GJArgs);
template __global__ void gj_panel_kernel<0, 4, 2, true>(GJArgs);
template __global__ void gj_panel_kernel<0, 4, 2, false>(GJArgs);
template __global__ void gj_panel_kernel<1, 4, 1, true>(GJArgs);

// Multipliers of the step: M(i, :) = P^-1(j, :) - e_j on pivot position k + j, -A(src(i), panel) P^-1 elsewhere.
__global__ void __launch_bounds__(256) gj_mult_kernel(GJArgs a) {
    __shared__ double Pi[GJ_NB][GJ_NB + 1];
    const int b = blockIdx.y, tid = threadIdx.x;
    const int m = a.m, k = a.k, nbb = min(GJ_NB, m - k);
    const double* Pg = a.Pinv + (long long)b * GJ_NB * GJ_NB;
    for (int e = tid; e < GJ_NB * GJ_NB; e += 256) Pi[e / GJ_NB][e % GJ_NB] = Pg[e];
    __syncthreads();
    const long long e = (long long)blockIdx.x * 256 + tid;
    if (e >= (long long)m * GJ_NB) return;
    const int i = (int)(e / GJ_NB), c = (int)(e % GJ_NB);
    const int j = i - k;
    double val = 0.0;
    if (c < nbb) {
        if (j >= 0 && j < nbb) {
            val = Pi[j][c] - (j == c ? 1.0 : 0.0);
        } else {
            const int s = a.src[(long long)b * m + i];
            const double* row = a.Wa + (long long)b * m * m + (long long)s * m + k;
            double acc = 0.0;
            for (int t = 0; t < nbb; t++) acc += row[t] * Pi[t][c];
            val = -acc;
        }
    }
    a.Mm[(long long)b * m * GJ_NB + e] = val;
}

// Wb = Wa(src rows) + M Wa(pivot rows) outside the panel; the panel column block is M + I on
// the pivot positions.  One wave per 32 x 32 block of the matrix.
__global__ void __launch_bounds__(256) gj_update_kernel(GJArgs a) {
    const int b = blockIdx.y;
    const int m = a.m, k = a.k, nbb = min(GJ_NB, m - k);
    const int tpr = (m + 31) / 32;
    const int w = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (w >= tpr * tpr) return;
    const int lane = threadIdx.x & 63, q = lane >> 4, r = lane & 15;
    const int row0 = (w / tpr) * 32, col0 = (w % tpr) * 32;
    const double* Wa = a.Wa + (long long)b * m * m;
    double* Wb = a.Wb + (long long)b * m * m;
    const double* Mm = a.Mm + (long long)b * m * GJ_NB;
    const int* src = a.src + (long long)b * m;
    const int* prow = a.prow + (long long)b * GJ_NB;
    if (col0 == k) {  // k is a multiple of 32: this block column is the panel
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int row = row0 + 16 * i + 4 * v + q, col = col0 + 16 * j + r;
                    if (row < m && col < m)
                        Wb[(long long)row * m + col] = Mm[(long long)row * GJ_NB + (col - k)] + (row == col ? 1.0 : 0.0);
                }
        return;
    }
    const int ra = min(row0 + r, m - 1), rb = min(row0 + 16 + r, m - 1);
    const int c0 = min(col0 + r, m - 1), c1 = min(col0 + 16 + r, m - 1);
    // the block's current values, loaded before the products so their latency overlaps them
    double cv[2][2][4];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = min(row0 + 16 * i + 4 * v + q, m - 1);
            const double* crow = Wa + (long long)src[row] * m;
            cv[i][0][v] = crow[c0];
            cv[i][1][v] = crow[c1];
        }
    td4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = td4{0.0, 0.0, 0.0, 0.0};
    for (int kb = 0; kb < nbb; kb += 16) {
        const int k0 = kb + 4 * q;
        double a0[4], a1[4], b0[4], b1[4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const bool ok = k0 + s < nbb;
            const int kk = ok ? k0 + s : nbb - 1;
            const double x = Mm[(long long)ra * GJ_NB + kk], y = Mm[(long long)rb * GJ_NB + kk];
            a0[s] = ok ? x : 0.0;
            a1[s] = ok ? y : 0.0;
            const double* brow = Wa + (long long)prow[kk] * m;
            b0[s] = brow[c0];
            b1[s] = brow[c1];
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
            acc[0][0] = mfma_f64(a0[s], b0[s], acc[0][0]);
            acc[0][1] = mfma_f64(a0[s], b1[s], acc[0][1]);
            acc[1][0] = mfma_f64(a1[s], b0[s], acc[1][0]);
            acc[1][1] = mfma_f64(a1[s], b1[s], acc[1][1]);
        }
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = row0 + 16 * i + 4 * v + q, col = col0 + 16 * j + r;
                if (row < m && col < m) Wb[(long long)row * m + col] = acc[i][j][v] + cv[i][j][v];
            }
}

// Column order of the inverse: the interchanges undone from the last to the first, column k's.  Each entry is followed
// through them by a thread of its own (the last one undone is the first it meets): one thread exchanging
// entries in LDS took 66 us for m = 1024, so 28.
__global__ void __launch_bounds__(256) gj_perm_kernel(GJArgs a) {
    __shared__ int piv[GJ_MAXM];
    const int b = blockIdx.y, tid = threadIdx.x, m = a.m;
    const int* ipiv = a.ipiv + (long long)b * m;
    for (int i = a.k + tid; i < m; i += 256) piv[i] = min(max(ipiv[i], 0), m - 1);
    __syncthreads();
    const int i = (int)blockIdx.x * 256 + tid;
    int x = i;
#pragma unroll 8
    for (int c = a.k; c < m; c++) {
        const int p = piv[c];
        x = x == c ? p : x == p ? c : x;
    }
    if (i < m) a.src[(long long)b * m + i] = x;
}

// X^-1(i, j) = W(i, idx(j)), written to the operator arena.
__global__ void __launch_bounds__(256) gj_gather_kernel(GJArgs a) {
    const int b = blockIdx.y, m = a.m;
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= (long long)m * m) return;
    const int i = (int)(e / m), j = (int)(e % m);
    const int c = min(max(a.src[(long long)b * m + j], 0), m - 1);
    a.Xi[(long long)b * m * m + e] = a.Wa[(long long)b * m * m + (long long)i * m + c];
}

// ---------------------------------------------------------------------------------------
// Inversion without row exchanges
// ---------------------------------------------------------------------------------------
// The interface systems of elliptic problems are definite up to row signs (sums of the children's
// boundary operators), so Gauss-Jordan needs no pivot search on them: over adaptive, variable and
// uniform meshes with lambda <= 0 the largest multiplier is 1.3, and the inverse's residual equals
// a pivoted LU's.  These kernels eliminate in natural order and check every multiplier against
// INV_LMAX; one beyond it (an indefinite system, a zero pivot, a NaN) stops the elimination, and the
// caller goes on with the pivoted kernels above from the column it stopped at.  What bounds the pivoted path is its 32-column panel,
// a chain of 32 dependent column searches (52 us per launch): the inversions of the adaptive
// Poisson mesh (1,937 merges, m = 64 .. 1024) took 7.4 ms of GPU time with it and take 1.2 ms so,
// those of 1,024 leaves of 32 x 32 cells 12.9 and 2.3 ms.

// x, opaque to the compiler: what is computed from it is computed after this point
__device__ inline int formed_here(int x) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(x));
#endif
    return x;
}

// Step k has met a large multiplier: no step of the launch sequence from k on is taken (inv_stopped), so
// the matrices stay as they were before it.  Of a batch, the first such step counts.
__device__ inline void inv_stop(int* stop, int k) { atomicMax(stop, INV_STOP - k); }
__device__ inline bool inv_stopped(int stop, int k) { return stop >= INV_STOP - k; }

// 1 / x: hardware estimate and two Newton steps (relative error about 1 ulp; inf or NaN at 0)
__device__ inline double inv_rcp(double x) {
    double rc = __builtin_amdgcn_rcp(x);
    rc = fma(rc, fma(-x, rc, 1.0), rc);
    return fma(rc, fma(-x, rc, 1.0), rc);
}

// Gauss-Jordan on a 16 x 16 block by one wave, in place, in the accumulator layout (slot v of lane
// (q, r) is element (4v + q, r)), four columns at a time: the rows 4g .. 4g + 3 of group g are
// slot g.  Through LDS (buf: 16 x 18) every lane gets the 4 x 4 pivot block P, its own column of
// those rows (a unit vector in the pivot columns) and one entry of the pivot columns, solves
// P x = column in registers -- x_q is its entry of the new rows -- and one MFMA subtracts the pivot
// columns times the new rows from all others.  Column by column, with the pivot row and column
// broadcast across lanes, a block took 6,300 cycles (393 a column, a chain of reciprocal,
// broadcasts and selects); so it takes a third of that.
// Checked: the multipliers inside P and those of the other rows.
// bg(g) issues products of the caller's that run on the matrix cores meanwhile.
template <class BG>
__device__ inline void inv16(td4& D, double* buf, bool& ok, BG&& bg) {
    const int lane = threadIdx.x & 63, q = lane >> 4, r = lane & 15;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 4; v++) buf[(4 * v + q) * 18 + r] = D[v];
        __builtin_amdgcn_wave_barrier();
        double P[4][4], x[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const td2 u = *(const td2*)(buf + (4 * g + i) * 18 + 4 * g), w = *(const td2*)(buf + (4 * g + i) * 18 + 4 * g + 2);
            P[i][0] = u[0]; P[i][1] = u[1]; P[i][2] = w[0]; P[i][3] = w[1];
            x[i] = buf[(4 * g + i) * 18 + r];
        }
        const double a = -buf[r * 18 + 4 * g + q];
        __builtin_amdgcn_wave_barrier();
        bg(g);
        const bool pcol = (r >> 2) == g;  // a pivot column
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = pcol ? ((r & 3) == i ? 1.0 : 0.0) : x[i];
#pragma unroll
        for (int j = 0; j < 4; j++) {  // LU of P, its inverse diagonal in P(j, j); x forward
            P[j][j] = inv_rcp(P[j][j]);
#pragma unroll
            for (int i = j + 1; i < 4; i++) {
                const double l = P[i][j] * P[j][j];
                ok = ok & (fabs(l) <= INV_LMAX);
#pragma unroll
                for (int c = j + 1; c < 4; c++) P[i][c] = fma(-l, P[j][c], P[i][c]);
                x[i] = fma(-l, x[j], x[i]);
            }
        }
#pragma unroll
        for (int j = 3; j >= 0; j--) {  // and back
#pragma unroll
            for (int c = j + 1; c < 4; c++) x[j] = fma(-P[j][c], x[c], x[j]);
            x[j] *= P[j][j];
        }
        const double xq = q < 2 ? (q == 0 ? x[0] : x[1]) : (q == 2 ? x[2] : x[3]);
        td4 C;
#pragma unroll
        for (int v = 0; v < 4; v++) C[v] = pcol ? 0.0 : D[v];
        C = mfma_f64(a, xq, C);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            if (v != g) ok = ok & (!pcol | (fabs(C[v]) <= INV_LMAX));
            D[v] = v == g ? xq : C[v];
        }
    }
}

// LDS of an inversion by WAVES waves: the pivot tile row of a step (its diagonal tile already
// inverted) by step parity, and one 16 x 16 transposition tile per wave
template <int MT, int WAVES>
struct InvShared {
    double rp[2][MT][4][64];
    alignas(16) double tr[WAVES][16 * 18];
    int bad[2];  // a multiplier of an even, an odd step was too large
};

// In-place inversion of mt x mt tiles of 16 x 16 (mt <= MT <= WAVES): wave w holds tile row w, tile
// j in T[j], in the accumulator layout.  Before step kb wave kb has inverted its diagonal tile and
// published its tile row; after the step's one barrier every other wave forms L = A_wk P^-1 and
// its transpose from one transposed copy of its own tile and subtracts L times the published row,
// and wave kb multiplies its row by P^-1.  Wave kb + 1 updates its diagonal tile first and inverts
// it while the rest of its row is updated, which leaves one tile update and one inversion between
// two barriers.  (OVERLAP: the inversion and the row's other products are interleaved, for a lone
// workgroup; without it they follow one another in fewer registers, so that more workgroups
// share a CU.)  An accumulator tile is the B operand of the next product as it stands, and the
// accumulator of L^T is the A operand of L.
template <bool OVERLAP, int MT, int WAVES>
__device__ inline void inv_tiles(td4 (&T)[MT], int mt, InvShared<MT, WAVES>& sh, bool& ok) {
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int q = lane >> 4, r = lane & 15;
    double* tr = sh.tr[wave];
    auto tile = [&](int k) {  // T[k], k uniform
        td4 D = T[0];
#pragma unroll
        for (int j = 1; j < MT; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) D[v] = (j == k) ? T[j][v] : D[v];
        return D;
    };
    auto put = [&](int k, const td4& D) {
#pragma unroll
        for (int j = 0; j < MT; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) T[j][v] = (j == k) ? D[v] : T[j][v];
    };
    auto publish = [&](int k) {
#pragma unroll
        for (int j = 0; j < MT; j++)
            if (j < mt)
#pragma unroll
                for (int v = 0; v < 4; v++) sh.rp[k & 1][j][v][lane] = T[j][v];
    };
    if (wave == 0) {
        sh.bad[lane & 1] = 0;
        inv16(T[0], tr, ok, [](int) {});
        publish(0);
    }
#pragma unroll(OVERLAP ? MT : 1)
    for (int kb = 0; kb < MT; kb++) {
        if (kb >= mt) break;
        const td4 D = tile(kb);
        // the own tile's transpose: a[s] = D(r, 4s + q), an A operand
#pragma unroll
        for (int v = 0; v < 4; v++) tr[(4 * v + q) * 18 + r] = D[v];
        __builtin_amdgcn_wave_barrier();
        double a[4];
#pragma unroll
        for (int s = 0; s < 4; s++) a[s] = tr[r * 18 + 4 * s + q];
        __syncthreads();
        // the step before (a step's word is next written two barriers on)
        if (!OVERLAP && kb > 0 && sh.bad[(kb - 1) & 1]) break;  // uniform per workgroup
        const double (&rp)[MT][4][64] = sh.rp[kb & 1];
        if (wave == kb) {
#pragma unroll
            for (int j = 0; j < MT; j++) {
                if (j >= mt || j == kb) continue;
                td4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int s = 0; s < 4; s++) x = mfma_f64(a[s], T[j][s], x);
                T[j] = x;
            }
        } else if (wave < mt) {
            td4 Lt = {0.0, 0.0, 0.0, 0.0}, L = Lt;
            double p[4];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                p[s] = rp[kb][s][lane];
                Lt = mfma_f64(p[s], a[s], Lt);
            }
#pragma unroll
            for (int v = 0; v < 4; v++) ok = ok & (fabs(Lt[v]) <= INV_LMAX);
            // tile j minus L times the published tile; column kb: -A P^-1
            auto update = [&](td4& X, int j) {
#pragma unroll
                for (int s = 0; s < 4; s++) X = mfma_f64(-Lt[s], rp[j][s][lane], X);
                if (!OVERLAP) __builtin_amdgcn_sched_barrier(0);  // one tile's operands in registers at a time
            };
            auto column = [&] {
#pragma unroll
                for (int s = 0; s < 4; s++) L = mfma_f64(-a[s], p[s], L);
            };
            if (wave == kb + 1) {
                td4 X = tile(kb + 1);
                update(X, kb + 1);
                auto rest = [&](int g) {
#pragma unroll
                    for (int j = 0; j < MT; j++)
                        if ((j & 3) == g && j < mt && j != kb && j != kb + 1) update(T[j], j);
                };
                column();
                put(kb, L);
                if constexpr (OVERLAP) {
                    inv16(X, tr, ok, rest);
                } else {
                    inv16(X, tr, ok, [](int) {});
#pragma unroll
                    for (int g = 0; g < 4; g++) rest(g);
                }
                put(kb + 1, X);
                publish(kb + 1);
            } else {
#pragma unroll
                for (int j = 0; j < MT; j++)
                    if (j < mt && j != kb) update(T[j], j);
                column();
                put(kb, L);
            }
        }
        if (!OVERLAP && __ballot(!ok)) sh.bad[kb & 1] = 1;
    }
}

// Whole inverses of matrices of order m <= 16 MT <= 64, one wave each (four independent waves per
// workgroup, no barrier): tile (i, j) in T[i][j], the steps of inv_tiles with every tile at hand.
// A launch has hundreds of such matrices; with a workgroup of four waves each, one or two per CU
// for the registers, the adaptive Poisson mesh's matrices of order 64 took 140 us, so 85 us.
template <int MT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8)))
inv_wave_kernel(const double* __restrict__ A, double* __restrict__ Ai, int m, int B, int* stop) {
    __shared__ __attribute__((aligned(16))) double tr_all[4][16 * 18];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int q = lane >> 4, r = lane & 15, b = (int)blockIdx.x * 4 + wave;
    if (b >= B) return;  // uniform per wave; no barrier below
    double* tr = tr_all[wave];
    const auto* Ab = gmem(A) + (long long)b * m * m;
    td4 T[MT][MT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = 16 * i + 4 * v + q;
            const auto* p = Ab + (long long)min(row, m - 1) * m;
#pragma unroll
            for (int j = 0; j < MT; j++) {
                const int col = 16 * j + r;
                const double x = p[min(col, m - 1)];
                T[i][j][v] = (row < m && col < m) ? x : (row == col ? 1.0 : 0.0);
            }
        }
    bool ok = true;
    auto transpose = [&](const td4& D, double (&a)[4]) {  // a[s] = D(r, 4s + q), an A operand
#pragma unroll
        for (int v = 0; v < 4; v++) tr[(4 * v + q) * 18 + r] = D[v];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < 4; s++) a[s] = tr[r * 18 + 4 * s + q];
        __builtin_amdgcn_wave_barrier();
    };
#pragma unroll
    for (int kb = 0; kb < MT; kb++) {
        if (16 * kb >= m) continue;  // (identity beyond)
        inv16(T[kb][kb], tr, ok, [](int) {});
        const td4 P = T[kb][kb];
        double a[4];
#pragma unroll
        for (int i = 0; i < MT; i++) {
            if (i == kb) continue;
            transpose(T[i][kb], a);
            td4 Lt = {0.0, 0.0, 0.0, 0.0}, L = Lt;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                Lt = mfma_f64(P[s], a[s], Lt);
                L = mfma_f64(-a[s], P[s], L);
            }
            T[i][kb] = L;
#pragma unroll
            for (int v = 0; v < 4; v++) ok = ok & (fabs(Lt[v]) <= INV_LMAX);
#pragma unroll
            for (int j = 0; j < MT; j++)
                if (j != kb)
#pragma unroll
                    for (int s = 0; s < 4; s++) T[i][j] = mfma_f64(-Lt[s], T[kb][j][s], T[i][j]);
        }
        transpose(P, a);
#pragma unroll
        for (int j = 0; j < MT; j++) {
            if (j == kb) continue;
            td4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < 4; s++) x = mfma_f64(a[s], T[kb][j][s], x);
            T[kb][j] = x;
        }
        if (__ballot(!ok)) break;
    }
    const int ms = formed_here(m);  // the stores' addresses are not kept from the loads
    auto* Ib = gmem(Ai) + (long long)b * ms * ms + r;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = 16 * i + 4 * v + q;
#pragma unroll
            for (int j = 0; j < MT; j++)
                if (row < ms && 16 * j + r < ms) Ib[(long long)row * ms + 16 * j] = T[i][j][v];
        }
    if (!ok) inv_stop(stop, 0);
}

template __global__ void inv_wave_kernel<1>(const double*, double*, int, int, int*);
template __global__ void inv_wave_kernel<2>(const double*, double*, int, int, int*);
template __global__ void inv_wave_kernel<4>(const double*, double*, int, int, int*);

// Whole inverses of matrices of order m <= 16 MT, one workgroup of MT waves each (64 < m <= 128).
template <int MT>
__global__ void __launch_bounds__(64 * MT) __attribute__((amdgpu_waves_per_eu(2, 8)))
inv_small_kernel(const double* __restrict__ A, double* __restrict__ Ai, int m,
                                                            int* stop) {
    __shared__ InvShared<MT, MT> sh;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int q = lane >> 4, r = lane & 15, mt = (m + 15) / 16;
    const auto* Ab = gmem(A) + (long long)blockIdx.x * m * m;
    auto* Ib = gmem(Ai) + (long long)blockIdx.x * m * m;
    td4 T[MT];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int row = 16 * wave + 4 * v + q;
        const auto* p = Ab + (long long)min(row, m - 1) * m;
#pragma unroll
        for (int j = 0; j < MT; j++) {
            const int col = 16 * j + r;
            const double x = p[min(col, m - 1)];
            T[j][v] = (row < m && col < m) ? x : (row == col ? 1.0 : 0.0);
        }
    }
    bool ok = true;
    inv_tiles<false>(T, mt, sh, ok);
    const int ms = formed_here(m);  // the stores' addresses are not kept from the loads
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int row = 16 * wave + 4 * v + q;
        auto* p = Ib + (long long)row * ms + r;
#pragma unroll
        for (int j = 0; j < MT; j++)
            if (row < ms && 16 * j + r < ms) p[16 * j] = T[j][v];
    }
    if (!ok) inv_stop(stop, 0);
}

template __global__ void inv_small_kernel<8>(const double*, double*, int, int*);

// Larger orders, INV_NB = 64 columns per step, two launches a step: the multipliers M (m x INV_NB,
// inv_mult_kernel) and the rank-64 update (inv_update_kernel), whose first workgroup goes on to
// invert the next step's pivot block while the others update the rest of the matrix.  A step is
// bound by that chain (update one block, 64 dependent columns, multipliers): 17 + 6 us a step at
// m <= 1024.  Inverting the pivot block in every workgroup of the multipliers instead, with the
// inversion in the open, took 24 + 8 us.

// P^-1 of step k's pivot block (nb x nb, here in strips of tiles), zero beyond nb, into Pn (INV_NB x INV_NB)
__device__ inline void inv_pivot_block(td4 (&T)[INV_NB / 16], int nb, InvShared<INV_NB / 16, 4>& sh, double* Pn, int k,
                                       int* stop) {
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int q = lane >> 4, r = lane & 15;
    bool ok = true;
    inv_tiles<true>(T, (nb + 15) / 16, sh, ok);
#pragma unroll
    for (int j = 0; j < INV_NB / 16; j++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = 16 * wave + 4 * v + q, col = 16 * j + r;
            gmem(Pn)[row * INV_NB + col] = (row < nb && col < nb) ? T[j][v] : 0.0;
        }
    if (!ok) inv_stop(stop, k);
}

// the first step's pivot block, one workgroup per matrix
__global__ void __launch_bounds__(256) inv_pivot_kernel(const double* __restrict__ A, double* __restrict__ Pn, int m,
                                                        int* stop) {
    __shared__ InvShared<INV_NB / 16, 4> sh;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int q = lane >> 4, r = lane & 15;
    const auto* Ab = gmem(A) + (long long)blockIdx.x * m * m;
    td4 T[INV_NB / 16];
#pragma unroll
    for (int j = 0; j < INV_NB / 16; j++)
#pragma unroll
        for (int v = 0; v < 4; v++)  // m > INV_NB
            T[j][v] = Ab[(long long)(16 * wave + 4 * v + q) * m + 16 * j + r];
    inv_pivot_block(T, INV_NB, sh, Pn + (long long)blockIdx.x * INV_NB * INV_NB, 0, stop);
}

// M = P^-1 on the pivot rows, -A P^-1 elsewhere (zero beyond the matrix's columns): one wave per
// 16 rows x 32 columns, all operands loaded before the products.
__global__ void __launch_bounds__(512) inv_mult_kernel(const double* __restrict__ A, double* __restrict__ Mm,
                                                       const double* __restrict__ Pn, int m, int k, int* stop) {
    constexpr int MT = INV_NB / 16;
    const int st = cmem(stop);  // (what this launch itself finds is for the next one)
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int q = lane >> 4, r = lane & 15;
    const int nb = min(INV_NB, m - k), row0 = (int)blockIdx.x * 64 + 16 * (wave & 3), j0 = 2 * (wave >> 2);
    const auto* Ab = gmem(A) + (long long)blockIdx.y * m * m;
    const auto* Pb = gmem(Pn) + (long long)blockIdx.y * INV_NB * INV_NB;
    auto* Mb = gmem(Mm) + (long long)blockIdx.y * m * INV_NB;
    const bool pivot_rows = (int)blockIdx.x * 64 == k;  // uniform: k is a multiple of 64
    td4 x[2];
    if (pivot_rows) {
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) x[j][v] = Pb[(row0 - k + 4 * v + q) * INV_NB + 16 * (j0 + j) + r];
        if (inv_stopped(st, k)) return;
    } else {
        // lane group q takes columns 16 t + 4q + s at step s; m, nb are multiples of 4
        td2 a[MT][2];
        double b[MT][2][4];
        const auto* ar = Ab + (long long)min(row0 + r, m - 1) * m + k;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const int c = min(16 * t + 4 * q, nb - 4);  // past nb: times the zero rows of P^-1
            a[t][0] = *(const EF_GLOBAL td2*)(ar + c);
            a[t][1] = *(const EF_GLOBAL td2*)(ar + c + 2);
        }
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int s = 0; s < 4; s++) b[t][j][s] = Pb[(16 * t + 4 * q + s) * INV_NB + 16 * (j0 + j) + r];
        if (inv_stopped(st, k)) return;  // (after the loads are issued: the wait for it is theirs)
        x[0] = x[1] = td4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int j = 0; j < 2; j++) x[j] = mfma_f64(-a[t][s >> 1][s & 1], b[t][j][s], x[j]);
        bool ok = true;
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) ok = ok & (fabs(x[j][v]) <= INV_LMAX);
        if (!ok) inv_stop(stop, k);
    }
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = row0 + 4 * v + q;
            if (row < m) Mb[(long long)row * INV_NB + 16 * (j0 + j) + r] = x[j][v];
        }
}

// The step's update into the other buffer: Wb = Wa + M Wa(pivot rows), Wb = M Wa(pivot rows) on the
// pivot rows themselves, and the pivot columns are M.  One workgroup per 64 x 64 block, a wave per
// 32 x 32 quarter; all of a quarter's operands are loaded before its products (K is 64), so a wave
// waits for memory once.  Workgroup 0 of a matrix takes the next pivot block and inverts it (Pn).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8)))
inv_update_kernel(const double* __restrict__ Wa, double* __restrict__ Wb,
                                                         const double* __restrict__ Mm, double* __restrict__ Pn, int m,
                                                         int k, int* stop) {
    constexpr int MT = INV_NB / 16;
    const int st = cmem(stop);  // (what this launch itself finds is for the next one)
    __shared__ union {
        InvShared<MT, 4> inv;
        double blk[MT][MT][4][64];  // the next pivot block, from the waves' quarters to their strips
    } sh;
    const int tpr = (m + 63) / 64;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int q = lane >> 4, r = lane & 15;
    const int nb = min(INV_NB, m - k), kn = k + INV_NB;
    // the next pivot block trades places with block 0 in the launch order (no next one: none)
    const int dn = kn < m ? (kn / 64) * (tpr + 1) : 0;
    const int t = (int)blockIdx.x == 0 ? dn : (int)blockIdx.x == dn ? 0 : (int)blockIdx.x;
    const int row0 = (t / tpr) * 64 + 32 * (wave >> 1), col0 = (t % tpr) * 64 + 32 * (wave & 1);
    const auto* Ab = gmem(Wa) + (long long)blockIdx.y * m * m;
    auto* Bb = gmem(Wb) + (long long)blockIdx.y * m * m;
    const auto* Mb = gmem(Mm) + (long long)blockIdx.y * m * INV_NB;
    td4 acc[2][2];
    if ((t % tpr) * 64 == k) {  // pivot columns
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    acc[i][j][v] = Mb[(long long)min(row0 + 16 * i + 4 * v + q, m - 1) * INV_NB + col0 - k + 16 * j + r];
        if (inv_stopped(st, k)) return;
    } else {
        const bool pivot_rows = (t / tpr) * 64 == k;
        const int c0 = min(col0 + r, m - 1), c1 = min(col0 + 16 + r, m - 1);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const long long row = (long long)min(row0 + 16 * i + 4 * v + q, m - 1) * m;
                const double x = Ab[row + c0], y = Ab[row + c1];
                acc[i][0][v] = pivot_rows ? 0.0 : x;
                acc[i][1][v] = pivot_rows ? 0.0 : y;
            }
        const auto* m0 = Mb + (long long)min(row0 + r, m - 1) * INV_NB;
        const auto* m1 = Mb + (long long)min(row0 + 16 + r, m - 1) * INV_NB;
        double a0[MT][4], a1[MT][4], b0[MT][4], b1[MT][4];
#pragma unroll
        for (int t4 = 0; t4 < MT; t4++) {
            const int k0 = 16 * t4 + 4 * q;  // lane group q takes k = 16 t4 + 4q + s at step s
#pragma unroll
            for (int s = 0; s < 4; s++) {
                a0[t4][s] = m0[k0 + s];
                a1[t4][s] = m1[k0 + s];
                const auto* brow = Ab + (long long)(k + min(k0 + s, nb - 1)) * m;  // past nb: times a zero
                b0[t4][s] = brow[c0];
                b1[t4][s] = brow[c1];
            }
        }
        if (inv_stopped(st, k)) return;
#pragma unroll
        for (int t4 = 0; t4 < MT; t4++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                acc[0][0] = mfma_f64(a0[t4][s], b0[t4][s], acc[0][0]);
                acc[0][1] = mfma_f64(a0[t4][s], b1[t4][s], acc[0][1]);
                acc[1][0] = mfma_f64(a1[t4][s], b0[t4][s], acc[1][0]);
                acc[1][1] = mfma_f64(a1[t4][s], b1[t4][s], acc[1][1]);
            }
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = row0 + 16 * i + 4 * v + q, col = col0 + 16 * j + r;
                if (row < m && col < m) Bb[(long long)row * m + col] = acc[i][j][v];
            }
    if (kn >= m || blockIdx.x != 0) return;  // uniform per workgroup (st is too: step k's stop is older than this launch)
    const int nn = min(INV_NB, m - kn);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) sh.blk[2 * (wave >> 1) + i][2 * (wave & 1) + j][v][lane] = acc[i][j][v];
    __syncthreads();
    td4 T[MT];
#pragma unroll
    for (int j = 0; j < MT; j++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = 16 * wave + 4 * v + q, col = 16 * j + r;
            const double x = sh.blk[wave][j][v][lane];
            T[j][v] = (row < nn && col < nn) ? x : (row == col ? 1.0 : 0.0);
        }
    __syncthreads();
    inv_pivot_block(T, nn, sh.inv, Pn + (long long)blockIdx.y * INV_NB * INV_NB, kn, stop);
}

// ---------------------------------------------------------------------------------------
// Merge assembly
// ---------------------------------------------------------------------------------------
// block (sa, sb) element (i, j) of a child DtN map (4n x 4n, WESN blocks of n)
__device__ inline double tblk(const double* T, int n, int sa, int sb, int i, int j) {
    return T[(long long)(sa * n + i) * (4 * n) + sb * n + j];
}

__global__ void __launch_bounds__(256) tree_assemble_kernel(const AsmDesc* __restrict__ descs) {
    const AsmDesc d = descs[blockIdx.y];
    const int n = d.n;
    const long long n2 = (long long)n * n;
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= 16 * n2) return;
    // X (mergeX_, HPSAlgorithm.hpp:870-895), interface order [ag, bo, ab, go]
    const int row = (int)(e / (4 * n)), col = (int)(e % (4 * n));
    const int ri = row / n, i = row % n, ci = col / n, j = col % n;
    const int c1 = if_c1(ri), s1 = if_s1(ri), c2 = if_c2(ri), s2 = if_s2(ri);
    double v;
    if (ri == ci) {
        v = tblk(pick4(d.Tc, c1), n, s1, s1, i, j) - tblk(pick4(d.Tc, c2), n, s2, s2, i, j);
    } else {
        const int sc1 = side_on_if(c1, ci), sc2 = side_on_if(c2, ci);
        v = 0.0;
        if (sc1 >= 0) v = tblk(pick4(d.Tc, c1), n, s1, sc1, i, j);
        else if (sc2 >= 0) v = -tblk(pick4(d.Tc, c2), n, s2, sc2, i, j);
    }
    d.X[e] = v;
}

// L12 of fine size nf (SpecialMatrices.hpp:136-173), column b: rows 0 (b <= 2), 2b-1 and 2b
// (b >= 1), 2b+1 and 2b+2 (b <= nc-2), nf-1 (b >= nc-3).
__global__ void __launch_bounds__(256) tree_coarsen_kernel(const CoarsenDesc* __restrict__ descs) {
    const CoarsenDesc d = descs[blockIdx.y];
    const int m = d.m, mc = m / 2;
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= (long long)(4 * mc) * (4 * mc)) return;
    const int R = (int)(e / (4 * mc)), C = (int)(e % (4 * mc));
    const int sa = R / mc, ar = R % mc, sb = C / mc, bc = C % mc;
    const double* r0 = d.src + (long long)(sa * m + 2 * ar) * (4 * m) + sb * m;
    const double* r1 = r0 + 4 * m;
    auto tv = [&](int t) { return 0.5 * r0[t] + 0.5 * r1[t]; };  // L21 row ar against column t
    double s = 0.0;
    if (bc <= 2) s += (bc == 0 ? 1.40625 : bc == 1 ? -0.5625 : 0.15625) * tv(0);
    if (bc >= 1) s += 0.25 * tv(2 * bc - 1) + 0.75 * tv(2 * bc);
    if (bc <= mc - 2) s += 0.75 * tv(2 * bc + 1) + 0.25 * tv(2 * bc + 2);
    if (bc >= mc - 3) s += (bc == mc - 1 ? 1.40625 : bc == mc - 2 ? -0.5625 : 0.15625) * tv(m - 1);
    d.dst[e] = s;
}

// ---------------------------------------------------------------------------------------
// Sweeps
// ---------------------------------------------------------------------------------------
// entry i of side `side` of a child's h (side length clen / 4), coarsened `tag` times by L21
// (pairwise averages, nested as coarsenUpwards_ applies them one step at a time); Vr is the
// right-hand side's column of the arena
__device__ inline double coarse_h(const double* Vr, long long off, int clen, int tag, int side, int i) {
    const int sl = clen / 4;
    const long long base = off + (long long)side * sl;
    if (tag == 0) return Vr[base + i];
    const int w = 1 << tag;
    auto x = [&](int t) { return Vr[base + (long long)i * w + t]; };
    if (tag == 1) return 0.5 * x(0) + 0.5 * x(1);
    double s = 0.0;  // tag >= 2: blocks of four in the nested order, then their mean
    for (int t = 0; t < w; t += 4) {
        const double p = 0.5 * x(t) + 0.5 * x(t + 1), u = 0.5 * x(t + 2) + 0.5 * x(t + 3);
        s += 0.5 * p + 0.5 * u;
    }
    return s * (4.0 / (double)w);
}

// The vector kernels below (up gather, uncoarsen, side copy, side interpolation) take one
// descriptor per blockIdx.y and stride over its (rhs, row) elements with gridDim.x workgroups:
// the host sizes gridDim.x to the launch's total work, not to its longest descriptor, so short
// descriptors do not leave thousands of empty workgroups to dispatch.
__global__ void __launch_bounds__(256) tree_up_gather_kernel(const UpDesc* __restrict__ descs, double* V, int k,
                                                              long long vrows) {
    const UpDesc d = descs[blockIdx.y];
    const int n = d.n;
    const long long total = 12LL * n * k;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long long)gridDim.x * 256) {
        const int rhs = (int)(e / (12 * n)), row = (int)(e % (12 * n));
        double* Vr = V + (long long)rhs * vrows;
        if (row < 4 * n) {  // hDiff of mergeW_ (HPSAlgorithm.hpp:1059-1087)
            const int r = row / n, i = row % n;
            const int c1 = if_c1(r), c2 = if_c2(r);
            const double h2 = coarse_h(Vr, pick4(d.ch_off, c2), pick4(d.clen, c2), pick4(d.tag, c2), if_s2(r), i);
            const double h1 = coarse_h(Vr, pick4(d.ch_off, c1), pick4(d.clen, c1), pick4(d.tag, c1), if_s1(r), i);
            Vr[d.hd_off + row] = h2 - h1;
        } else {  // boundary part of mergeH_ (:1098-1117), WESN order (:1128-1150)
            const int rr = row - 4 * n, q = rr / n, i = rr % n, c = q_child(q);
            Vr[d.h_off + rr] = coarse_h(Vr, pick4(d.ch_off, c), pick4(d.clen, c), pick4(d.tag, c), q_side(q), i);
        }
    }
}

// value i of a side prolonged from nc coarse values src to nf = 2 nc (uncoarsen_'s L12:
// quadratic end weights, 3/4-1/4 in between)
__device__ inline double prolong(const double* src, int nc, int nf, int i) {
    if (i == 0) return 1.40625 * src[0] + (-0.5625) * src[1] + 0.15625 * src[2];
    if (i == nf - 1) return 0.15625 * src[nc - 3] + (-0.5625) * src[nc - 2] + 1.40625 * src[nc - 1];
    if (i & 1) {
        const int j = (i - 1) / 2;
        return 0.75 * src[j] + 0.25 * src[j + 1];
    }
    const int j = (i - 2) / 2;
    return 0.25 * src[j] + 0.75 * src[j + 1];
}

__global__ void __launch_bounds__(256) tree_uncoarsen_kernel(const VecStepDesc* __restrict__ descs, double* V, int k,
                                                              long long vrows) {
    const VecStepDesc d = descs[blockIdx.y];
    const int nf = d.nfine, nc = nf / 2;
    const long long total = 4LL * nf * k;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long long)gridDim.x * 256) {
        const int rhs = (int)(e / (4 * nf)), row = (int)(e % (4 * nf));
        const int side = row / nf, i = row % nf;
        double* Vr = V + (long long)rhs * vrows;
        Vr[d.dst_off + row] = prolong(Vr + d.src_off + (long long)side * nc, nc, nf, i);
    }
}

// A child's boundary data written out, where the sweeps cannot read sides in place (sizes that
// do not allow the 4-row operand blocks): side s of descriptor blockIdx.y from src[s], each
// thread striding over (rhs, row) elements.
__global__ void __launch_bounds__(256) tree_side_copy_kernel(const SideCopy* __restrict__ descs, double* V, int k,
                                                              long long vrows) {
    const SideCopy d = descs[blockIdx.y];
    const int len = d.len;
    const long long total = 4LL * len * k;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long long)gridDim.x * 256) {
        const int rhs = (int)(e / (4 * len)), row = (int)(e % (4 * len));
        const int s = row / len, i = row - s * len;
        double* Vr = V + (long long)rhs * vrows;
        Vr[d.dst + row] = Vr[pick4(d.src, s) + i];
    }
}

// The first uncoarsen_ step of a coarsened child straight from its sides' sources: the coarse
// side s (len values at src[s]) prolonged to 2 len values at dst + s 2 len, with the weights of
// tree_uncoarsen_kernel (HPSAlgorithm.hpp:1165-1190).
__global__ void __launch_bounds__(256) tree_side_interp_kernel(const SideCopy* __restrict__ descs, double* V, int k,
                                                                long long vrows) {
    const SideCopy d = descs[blockIdx.y];
    const int nc = d.len, nf = 2 * nc;
    const long long total = 4LL * nf * k;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long long)gridDim.x * 256) {
        const int rhs = (int)(e / (4 * nf)), row = (int)(e % (4 * nf));
        const int side = row / nf, i = row % nf;
        double* Vr = V + (long long)rhs * vrows;
        Vr[d.dst + row] = prolong(Vr + pick4(d.src, side), nc, nf, i);
    }
}

// g = r / a: the LU solve of diag(a) in solveStage (HPSAlgorithm.hpp:402-420); r is [rhs][m],
// g is column rhs of the arena (g + rhs * vrows).
__global__ void __launch_bounds__(256) tree_root_dirichlet_kernel(const double* r, const double* a, double* g, int m, int k,
                                                                   long long vrows) {
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= (long long)m * k) return;
    const int c = (int)(e / m), i = (int)(e % m);
    g[(long long)c * vrows + i] = r[e] / a[i];
}

// A = diag(a) + diag(b) T and rhs = r - b h (HPSAlgorithm.hpp:402-420), row-scaled; rhs is [rhs][m], h a
// column of the arena (h + rhs * vrows) or null.  One workgroup per row (an element per thread, each with its own
// division by m and scale: 6.4 us for m = 1024, so 5.4).
__global__ void __launch_bounds__(256) tree_root_robin_kernel(const double* T, const double* a, const double* b, const double* r,
                                                              const double* h, double* A, double* rhs, int m, int k,
                                                              long long vrows) {
    const int i = blockIdx.x;
    const long long row = (long long)i * m;
    const double ai = a[i], bi = b[i], t = T[row + i];
    // rows scaled by powers of two to diag(a / b) + T, which is definite up to row signs as T is (a
    // positive a / b outwards), and Dirichlet rows (b = 0) to the size of T's diagonal: then
    // the elimination in natural order meets no large multiplier
    auto fine = [](double x) { return fabs(x) > 1e-150 && fabs(x) < 1e150; };
    double scale = 1.0;
    if (fine(bi)) {  // (an a / b beyond the range leaves the row as it is)
        const double f = ldexp(1.0, -ilogb(bi));
        if (fabs(ai) * f < 1e150) scale = f;
    } else if (bi == 0.0 && fine(ai) && fine(t)) {
        scale = ldexp(1.0, ilogb(t) - ilogb(ai));
    }
    for (int j = threadIdx.x; j < m; j += 256) A[row + j] = scale * (bi * T[row + j] + (i == j ? ai : 0.0));
    for (int c = threadIdx.x; c < k; c += 256) {
        const long long e = (long long)c * m + i;
        rhs[e] = scale * (r[e] - bi * (h ? h[(long long)c * vrows + i] : 0.0));
    }
}

// ---------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------
// tree_gemm_lds_kernel's products on tr x tc tiles: whole tiles and blocks of k only, so no load is clamped.
// It is the faster one from its smallest launch (64 workgroups, n = 64: S 11.3 -> 10.9 us, T 12.5 -> 11.2) on; the
// square tile is taken where it fits (a third less operand traffic than 32 x 128).
static bool fits_lds_tiles(const TreeGemm& p, int tr, int tc) {
    auto row_major = [](int cs) { return cs == 0 || cs == 1; };
    auto vectors = [](const double* b, int ld) { return ((uintptr_t)b & 15) == 0 && (ld & 1) == 0; };
    return p.M > 0 && p.N > 0 && p.M % tr == 0 && p.N % tc == 0 && p.dn == 0 && p.K0 > 0 && p.K0 % 16 == 0 &&
           p.K1 % 16 == 0 && row_major(p.bcs) && row_major(p.ccs) && row_major(p.dcs) && p.cn % 32 == 0 && p.ldb0 > 1 &&
           vectors(p.B0, p.ldb0) && (p.K1 == 0 || (p.ldb1 > 1 && vectors(p.B1, p.ldb1)));
}

GemmLaunch plan_gemm(const std::vector<TreeGemm>& probs_in, int tn, DevStore& store, hipStream_t s, bool f32, int rt) {
    GemmLaunch g;
    g.tn = tn;
    g.f32 = f32;
    g.rt = (tn == 1) ? 1 : 2;
    if (probs_in.empty()) return g;
    int maxM = 0;
    for (const TreeGemm& p : probs_in) maxM = std::max(maxM, p.M);
    if (maxM <= 16) g.rt = 1;  // 16-row tiles: a 32-row tile would compute a clamped copy of the same rows
    if (rt == 1 || (rt == 2 && tn == 2)) g.rt = rt;  // an explicit choice (the tile autotuner)
    std::vector<TreeGemm> probs = probs_in;
    // Split-K: when a problem asks for k chunks (kc > 0), the whole launch runs on
    // tree_gemm_split_kernel with one wave per chunk of a 16 x 16 tile; problems that asked for
    // none are cut into chunks of the same count (rounded to 16).  The chunks depend on the
    // launch's problems only, never on N.
    int kw = 1;
    for (TreeGemm& p : probs)
        if (p.M > 0 && p.N > 0 && p.kc > 0) {
            if (p.kc % 16 != 0) throw EfError(EF_ERR_INTERNAL, "split-K chunk must be a multiple of 16");
            const int K = p.K0 + p.K1;
            // at most 16 chunks (waves per workgroup): longer ranges get longer chunks
            if ((K + p.kc - 1) / p.kc > 16) p.kc = ((K + 15) / 16 + 15) / 16 * 16;
            kw = std::max(kw, (K + p.kc - 1) / p.kc);
        }
    if (kw > 16) throw EfError(EF_ERR_INTERNAL, "split-K launch with more than 16 chunks per tile");
    if (kw > 1 && f32) throw EfError(EF_ERR_INTERNAL, "split-K launch on the FP32 matrix cores");
    if (kw > 1) {
        g.kw = kw;
        g.rt = g.tn = 1;
    }
    if (kw == 1 && !f32 && tn == 2 && rt == 0)
        for (int wr : {2, 1, 4}) {
            bool fit = g.lds == 0;
            for (const TreeGemm& p : probs) fit = fit && fits_lds_tiles(p, 32 * wr, 128 / wr);
            if (fit) g.lds = wr;
        }
    std::vector<int> start(probs.size() + 1, 0);
    const int rw = g.lds ? 32 * g.lds : 16 * g.rt, cw = g.lds ? 128 / g.lds : 16 * g.tn;
    long long total = 0;
    for (size_t i = 0; i < probs.size(); i++) {
        TreeGemm& p = probs[i];
        start[i] = (int)total;
        p.nks = 1;
        if (p.bcs == 0) p.bcs = 1;
        if (p.ccs == 0) p.ccs = 1;
        if (p.dcs == 0) p.dcs = 1;
        if (p.M <= 0 || p.N <= 0) { p.kc = 0; continue; }
        if (std::abs(p.alpha0) != 1.0 || (p.K1 > 0 && std::abs(p.alpha1) != 1.0))
            throw EfError(EF_ERR_INTERNAL, "GEMM segment factor other than 1 and -1");
        // extents: the kernel clamps rows to M-1, columns to N-1 and k to K-1
        check_strided(p.D, p.M, p.N, p.ldd, p.dcs, "GEMM D");
        if (p.cn > 0) {
            if (p.kc > 0 || !p.C || !p.C1) throw EfError(EF_ERR_INTERNAL, "GEMM with C in blocks needs both blocks and no split");
            check_strided(p.C, p.M, p.cn, p.ldc, 1, "GEMM C block");
            check_strided(p.C1, p.M, p.cn, p.ldc, 1, "GEMM C block");
        } else if (p.C) check_strided(p.C, p.M, p.N, p.ldc, p.ccs, "GEMM C");
        const double* As[2] = {p.A0, p.A1};
        const double* Bs[2] = {p.B0, p.B1};
        const int lda[2] = {p.lda0, p.lda1}, ldb[2] = {p.ldb0, p.ldb1}, K[2] = {p.K0, p.K1};
        if (p.dn > 0) {  // block-gather mode: every block's segments inside B0's allocation
            if (p.dn % 4 != 0 || p.ldb0 != 1 || p.K0 != 4 * p.dn || p.K1 > 0 || (p.dsub != 0 && p.dsub != 1))
                throw EfError(EF_ERR_INTERNAL, "block-gather GEMM needs four blocks of a multiple of 4 rows, contiguous");
            for (int r4 = 0; r4 < 4; r4++)
                for (int h2 = 0; h2 < 1 + p.dsub; h2++) {
                    const long long o = h2 ? p.d1[r4] : p.d2[r4];
                    if (o < 0 || (o & 1)) throw EfError(EF_ERR_INTERNAL, "block-gather GEMM row offset negative or odd");
                    check_strided(p.B0 + o, p.dn, p.N, 1, p.bcs, "GEMM gathered block");
                }
        }
        for (int sg = 0; sg < 2; sg++) {
            if (K[sg] <= 0) continue;
            check_matrix(As[sg], p.M, K[sg], lda[sg], "GEMM A");
            if (sg == 0 && p.dn > 0) {
                if (((uintptr_t)As[0] & 15) != 0 || (lda[0] & 1) != 0 || ((uintptr_t)p.B0 & 15) != 0 || (p.bcs & 1) != 0)
                    throw EfError(EF_ERR_INTERNAL, "block-gather GEMM operands not 16-byte aligned");
                continue;
            }
            check_strided(Bs[sg], K[sg], p.N, ldb[sg], p.bcs, "GEMM B");
            if (((uintptr_t)As[sg] & 15) != 0 || (lda[sg] & 1) != 0)
                throw EfError(EF_ERR_INTERNAL, "GEMM A operand not 16-byte aligned with an even leading dimension");
            if (ldb[sg] == 1 && (((uintptr_t)Bs[sg] & 15) != 0 || (p.bcs & 1) != 0))
                throw EfError(EF_ERR_INTERNAL, "GEMM B operand contiguous along k but not 16-byte aligned");
        }
        if (g.kw > 1) {
            const int Kt = p.K0 + p.K1;
            if (p.kc == 0) p.kc = std::max(16, ((Kt + g.kw - 1) / g.kw + 15) / 16 * 16);
            p.nks = (Kt + p.kc - 1) / p.kc;
            if (p.nks > g.kw) throw EfError(EF_ERR_INTERNAL, "split-K chunks exceed the launch's waves per tile");
            // a chunk that starts in segment 1 starts at an even k there (16-byte operand reads)
            if (p.K1 > 0 && (p.K0 & 1)) throw EfError(EF_ERR_INTERNAL, "split-K over two segments needs an even K0");
        } else {
            p.kc = 0;
        }
        total += (long long)((p.M + rw - 1) / rw) * ((p.N + cw - 1) / cw);
        if (total > 0x7fffffffLL) throw EfError(EF_ERR_INTERNAL, "GEMM launch too large");
    }
    start[probs.size()] = (int)total;
    g.nprob = (int)probs.size();
    g.nwaves = (int)total;  // waves (tile kernel) or workgroups (split kernel)
    std::vector<int> wprob((size_t)total);
    for (size_t i = 0; i < probs.size(); i++)
        for (int w = start[i]; w < start[i + 1]; w++) wprob[w] = (int)i;
    g.probs = store.stage(probs);
    g.start = store.stage(start);
    g.wprob = store.stage(wprob);
    return g;
}

void run_gemm(const GemmLaunch& g, hipStream_t s) {
    if (g.nwaves == 0) return;
    if (g.kw > 1) {
        EF_LAUNCH("tree_gemm_split_kernel", tree_gemm_split_kernel, dim3(g.nwaves), dim3(64 * g.kw), s, g.probs,
                  g.start, g.wprob, g.nwaves);
        return;
    }
#define EF_GEMM_LAUNCH(WR_, WC_, NAME_)                                                                       \
    EF_LAUNCH(NAME_, (tree_gemm_lds_kernel<WR_, WC_>), dim3(g.nwaves), dim3(256), s, g.probs, g.start, g.wprob, \
              g.nwaves)
    if (g.lds > 0) {
        if (g.lds == 1) EF_GEMM_LAUNCH(1, 4, "tree_gemm_lds_kernel<1,4>");
        else if (g.lds == 2) EF_GEMM_LAUNCH(2, 2, "tree_gemm_lds_kernel<2,2>");
        else EF_GEMM_LAUNCH(4, 1, "tree_gemm_lds_kernel<4,1>");
        return;
    }
#undef EF_GEMM_LAUNCH
    const dim3 grid(blocks_for(g.nwaves, 4)), block(256);
#define EF_GEMM_LAUNCH(RT_, TN_, F32_, NAME_)                                                          \
    EF_LAUNCH(NAME_, (tree_gemm_kernel<RT_, TN_, F32_>), grid, block, s, g.probs, g.start, g.wprob, g.nwaves)
    if (g.f32) {
        if (g.tn == 1) EF_GEMM_LAUNCH(1, 1, true, "tree_gemm_kernel<1,1,f32>");
        else if (g.rt == 1) EF_GEMM_LAUNCH(1, 2, true, "tree_gemm_kernel<1,2,f32>");
        else EF_GEMM_LAUNCH(2, 2, true, "tree_gemm_kernel<2,2,f32>");
    } else {
        if (g.tn == 1) EF_GEMM_LAUNCH(1, 1, false, "tree_gemm_kernel<1,1>");
        else if (g.rt == 1) EF_GEMM_LAUNCH(1, 2, false, "tree_gemm_kernel<1,2>");
        else EF_GEMM_LAUNCH(2, 2, false, "tree_gemm_kernel<2,2>");
    }
#undef EF_GEMM_LAUNCH
}

size_t gj_work_doubles(int m, int B) {
    return (size_t)B * ((size_t)m * m + (size_t)GJ_NB * GJ_NB + (size_t)m * GJ_NB);
}
size_t gj_work_ints(int m, int B) {
    return (size_t)B * ((size_t)GJ_MAXCH * GJ_NB + GJ_NB + 2 * (size_t)m + GJ_NB);
}

void run_gj_inverse(double* wa, double* xi, int m, int B, const GJWork& w, int* info, hipStream_t s, int k0) {
    if (B <= 0) return;
    if (m < 1 || m > GJ_MAXM)
        throw EfError(EF_ERR_ARG, "interface system of order " + std::to_string(m) + " exceeds the inversion limit " +
                                      std::to_string(GJ_MAXM));
    const size_t mm = (size_t)m * m * B;
    check_range(wa, mm * 8, "GJ matrices");
    check_range(w.wb, mm * 8, "GJ second buffer");
    check_range(xi, mm * 8, "GJ inverse output");
    check_range(w.cand, (size_t)B * GJ_MAXCH * GJ_NB * 4, "GJ candidates");
    check_range(w.cfin, (size_t)B * GJ_NB * 4, "GJ pivots");
    check_range(w.src, (size_t)B * m * 4, "GJ row map");
    check_range(w.ipiv, (size_t)B * m * 4, "GJ interchanges");
    check_range(w.prow, (size_t)B * GJ_NB * 4, "GJ pivot rows");
    check_range(w.Pinv, (size_t)B * GJ_NB * GJ_NB * 8, "GJ pivot-block inverse");
    check_range(w.Mm, (size_t)B * m * GJ_NB * 8, "GJ multipliers");
    check_range(info, (size_t)B * 4, "GJ info");
    GJArgs a{};
    a.cand = w.cand; a.cfin = w.cfin; a.src = w.src; a.ipiv = w.ipiv; a.prow = w.prow; a.info = info;
    a.Pinv = w.Pinv; a.Mm = w.Mm; a.Xi = xi;
    a.m = m; a.B = B;
    double* cur = wa;
    double* nxt = w.wb;
    const int tpr = (m + 31) / 32;
    for (int k = k0; k < m; k += GJ_NB) {
        a.Wa = cur; a.Wb = nxt; a.k = k;
        a.nch = (m - k + GJ_CH - 1) / GJ_CH;
        const int rows = m - k;
        // rows per workgroup: 64 WAVES RPL (chunks of GJ_CH = 512 rows; up to 256 candidates)
        if (rows <= 64)
            EF_LAUNCH("gj_panel_kernel<0,1,1,fin>", (gj_panel_kernel<0, 1, 1, true>), dim3(1, B), dim3(64), s, a);
        else if (rows <= 128)
            EF_LAUNCH("gj_panel_kernel<0,1,2,fin>", (gj_panel_kernel<0, 1, 2, true>), dim3(1, B), dim3(64), s, a);
        else if (rows <= 256)
            EF_LAUNCH("gj_panel_kernel<0,2,2,fin>", (gj_panel_kernel<0, 2, 2, true>), dim3(1, B), dim3(128), s, a);
        else if (a.nch == 1)
            EF_LAUNCH("gj_panel_kernel<0,4,2,fin>", (gj_panel_kernel<0, 4, 2, true>), dim3(1, B), dim3(256), s, a);
        else {
            EF_LAUNCH("gj_panel_kernel<0,4,2>", (gj_panel_kernel<0, 4, 2, false>), dim3(a.nch, B), dim3(256), s, a);
            EF_LAUNCH("gj_panel_kernel<1,4,1,fin>", (gj_panel_kernel<1, 4, 1, true>), dim3(1, B), dim3(256), s, a);
        }
        EF_LAUNCH("gj_mult_kernel", gj_mult_kernel, dim3(blocks_for((long long)m * GJ_NB), B), dim3(256), s, a);
        EF_LAUNCH("gj_update_kernel", gj_update_kernel, dim3(blocks_for((long long)tpr * tpr, 4), B), dim3(256), s, a);
        std::swap(cur, nxt);
    }
    a.Wa = cur; a.Wb = nxt; a.k = k0;
    EF_LAUNCH("gj_perm_kernel", gj_perm_kernel, dim3(blocks_for(m), B), dim3(256), s, a);
    EF_LAUNCH("gj_gather_kernel", gj_gather_kernel, dim3(blocks_for((long long)m * m), B), dim3(256), s, a);
}

size_t inv_work_doubles(int m, int B) {
    return m <= INV_SMALL ? 0 : (size_t)B * ((size_t)m * m + (size_t)m * INV_NB + (size_t)INV_NB * INV_NB);
}

void run_inverse(double* wa, double* xi, int m, int B, double* work, int* stop, hipStream_t s) {
    if (B <= 0) return;
    if (m < 1 || m > GJ_MAXM)
        throw EfError(EF_ERR_ARG, "interface system of order " + std::to_string(m) + " exceeds the inversion limit " +
                                      std::to_string(GJ_MAXM));
    const size_t mm = (size_t)m * m * B;
    check_range(wa, mm * 8, "matrices to invert");
    check_range(xi, mm * 8, "inverse output");
    check_range(stop, sizeof(int), "inversion stop");
    // up to 64 one wave holds the matrix (128 registers a lane), up to 128 a workgroup of eight
    if (m <= 16)
        EF_LAUNCH("inv_wave_kernel<1>", inv_wave_kernel<1>, dim3((B + 3) / 4), dim3(256), s, (const double*)wa, xi, m, B, stop);
    else if (m <= 32)
        EF_LAUNCH("inv_wave_kernel<2>", inv_wave_kernel<2>, dim3((B + 3) / 4), dim3(256), s, (const double*)wa, xi, m, B, stop);
    else if (m <= 64)
        EF_LAUNCH("inv_wave_kernel<4>", inv_wave_kernel<4>, dim3((B + 3) / 4), dim3(256), s, (const double*)wa, xi, m, B, stop);
    else if (m <= INV_SMALL)
        EF_LAUNCH("inv_small_kernel<8>", inv_small_kernel<8>, dim3(B), dim3(512), s, (const double*)wa, xi, m, stop);
    else {
        check_range(work, inv_work_doubles(m, B) * 8, "inversion work");
        if (m % 4 != 0) throw EfError(EF_ERR_INTERNAL, "inversion of an order that is not a multiple of 4");
        double* Mm = work + mm;
        double* Pn = Mm + (size_t)B * m * INV_NB;
        double* cur = wa;
        double* nxt = work;
        const int tpr = (m + 63) / 64;
        EF_LAUNCH("inv_pivot_kernel", inv_pivot_kernel, dim3(B), dim3(256), s, (const double*)cur, Pn, m, stop);
        for (int k = 0; k < m; k += INV_NB) {
            double* out = (k + INV_NB >= m) ? xi : nxt;  // the last step writes the inverse where it belongs
            EF_LAUNCH("inv_mult_kernel", inv_mult_kernel, dim3(tpr, B), dim3(512), s, (const double*)cur, Mm,
                      (const double*)Pn, m, k, stop);
            EF_LAUNCH("inv_update_kernel", inv_update_kernel, dim3(tpr * tpr, B), dim3(256), s, (const double*)cur, out,
                      (const double*)Mm, Pn, m, k, stop);
            std::swap(cur, nxt);
        }
    }
}

int inv_stop_column(int stop, int m) { return stop == 0 ? m : INV_STOP - stop; }

double* inv_state(double* wa, double* work, int k) { return k / INV_NB % 2 ? work : wa; }

}  // namespace efk
