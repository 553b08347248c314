// ef_patch_large.hip -- fast diagonalisation of large patches (N > 32) as batched GEMMs.
//
// Same mathematics as patch_fd_kernel (U = Q ((Q^T B Q) ./ D) Q^T, FiniteVolumeSolver.cpp
// :25-294 with constant coefficients), but the N x N arrays no longer fit one wave's
// registers: each product is a launch over a chunk of items, with HBM work buffers padded
// to Np = 16 ceil(N / 16) between them (zero padding; padded modes are zeroed by the scaling).
//   stage 0   W2 = Q^T B,   B = f - 2 c g on the edge cells (or a unit boundary column for DtN
//             chunks), folded as it is read
//   stage 1   W1 = (W2 Q) ./ D
//   stage 2   W2 = Q W1
//   stage 3   u = W2 Q^T straight to the output, or W1 = W2 Q^T and the Neumann data h / DtN
//             column from its edge cells (patch_large_out_kernel)
#include <hip/hip_runtime.h>
#include "ef_device.hpp"
#include "ef_kernels.hpp"

namespace efk {

typedef double ld4 __attribute__((ext_vector_type(4)));
typedef double ld2 __attribute__((ext_vector_type(2)));

// item t of the chunk -> (patch, rhs, DtN column or -1)
__device__ inline void large_item(const PatchLargeArgs& a, long long t, int& patch, int& rhs, int& col) {
    const long long it = a.item0 + t;
    if (a.op == PATCH_OP_DTN) {
        patch = a.patch0;
        rhs = 0;
        col = a.col0 + (int)t;
    } else {
        rhs = (int)(it / a.npatches);
        patch = (int)(it % a.npatches);
        col = -1;
    }
}

__device__ inline double large_g(const PatchLargeArgs& a, const double* g, int col, int t) {
    if (col >= 0) return (t == col) ? 1.0 : 0.0;
    return g ? g[t] : 0.0;
}

// One product of the chain, C = A B for every item (blockIdx.y), in 32 x 32 blocks of C of RT x CT tiles of
// 16 x 16 (one in a direction where the matrix ends).  The k range is summed in quarters (whole blocks of 16),
// then the quarters.  SPLIT: one workgroup per block, wave w sums quarter w, and the quarters meet in
// LDS, wave w adding up and storing tile w; otherwise one wave per block sums them one after another: the
// same bits.  Operands are read straight from memory in the v_mfma_f64_16x16x4_f64 layouts, two blocks
// ahead.  Within each block of 16 k values, lane group q takes k = kb + 4q + s at step s: an operand
// contiguous along k is read as two 16-byte vectors per lane, one contiguous along the tile as 16
// consecutive doubles per lane group and step.
// A single grid is bound by latency: one wave per block and the whole k range, with the folding, the
// scaling and the output in launches of their own, took 32 us a product at N = 512 (64 workgroups,
// 32 dependent loads; 146 us a solve), the solve so takes 59 us (15 us at the matrix cores' rate).  Stages 1
// to 3 with SPLIT keep to 128 registers: 16 grids of 512 took 493 us at three waves per SIMD, 459 us at four;
// stage 0, which holds the folding, takes 164.
// Batches that fill the chip are bound by the products' own work.  Folding every value by its own tests, and
// tiles past the matrix formed and dropped, made them slower than the separate launches (2,000 patches of
// 100^2: Neumann data 1,004 -> 1,089 us); the folding's tests now only run in blocks that touch a side: 1,011.
template <int STAGE, bool SPLIT, int RT, int CT>
__device__ inline void large_block(const PatchLargeArgs& a, int row0, int col0, double (*part)[4][4][64]) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int q = lane >> 4, r = lane & 15;
    const int Nn = a.N, Np = (Nn + 15) / 16 * 16;
    const long long t = blockIdx.y, per = (long long)Np * Np;
    int patch, rhs, col;
    large_item(a, t, patch, rhs, col);
    const long long slot = (long long)rhs * a.npatches + patch;
    const PatchCoef cf = a.coef[a.cls ? a.cls[patch] : patch];
    constexpr bool AK = STAGE != 0, BK = STAGE == 3;  // contiguous along k
    const auto* Q = gmem(a.Q);
    const auto* Ap = (STAGE == 0 || STAGE == 2) ? Q : gmem((const double*)a.W2) + t * per;
    const auto* Bp = STAGE == 2 ? gmem((const double*)a.W1) + t * per : Q;
    const bool has_f = a.f && col < 0;
    const auto* fp = has_f ? gmem(a.f) + slot * Nn * Nn : Q;  // (not read without f, or read at 0)
    const int ldf = has_f ? Nn : 0;
    const double* g = (a.g && col < 0) ? a.g + slot * 4 * Nn : nullptr;
    struct Blk {
        double a[RT][4], b[CT][4];
    };
    auto load = [&](int kb, Blk& o) {
        const int k = kb + 4 * q;
#pragma unroll
        for (int i = 0; i < RT; i++) {
            if (AK) {
                const auto* x = Ap + (long long)(row0 + 16 * i + r) * Np + k;
                const ld2 u = *(const EF_GLOBAL ld2*)x, v = *(const EF_GLOBAL ld2*)(x + 2);
                o.a[i][0] = u[0]; o.a[i][1] = u[1]; o.a[i][2] = v[0]; o.a[i][3] = v[1];
            } else {
#pragma unroll
                for (int s = 0; s < 4; s++) o.a[i][s] = Ap[(long long)(k + s) * Np + row0 + 16 * i + r];
            }
        }
#pragma unroll
        for (int j = 0; j < CT; j++) {
            const int c = col0 + 16 * j + r;
            if (BK) {
                const auto* x = Bp + (long long)c * Np + k;
                const ld2 u = *(const EF_GLOBAL ld2*)x, v = *(const EF_GLOBAL ld2*)(x + 2);
                o.b[j][0] = u[0]; o.b[j][1] = u[1]; o.b[j][2] = v[0]; o.b[j][3] = v[1];
            } else if (STAGE == 0) {  // f, zero in the padding
#pragma unroll
                for (int s = 0; s < 4; s++)
                    o.b[j][s] = fp[(unsigned)(min(k + s, Nn - 1) * ldf + (has_f ? min(c, Nn - 1) : 0))];
            } else {
#pragma unroll
                for (int s = 0; s < 4; s++) o.b[j][s] = Bp[(long long)(k + s) * Np + c];
            }
        }
    };
    // stage 0: the load's boundary terms (FiniteVolumeSolver.cpp:100-184) as its values are used
    auto fold = [&](int kb, Blk& o) {
        if (STAGE != 0) return;
        // sides that the block touches (uniform); inside, the values are f's
        const bool w = kb == 0, e = kb + 16 >= Nn, so = col0 == 0, no = col0 + 16 * CT >= Nn;
        if (has_f && !(w || e || so || no)) return;
#pragma unroll
        for (int c = 0; c < CT; c++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int i = kb + 4 * q + s, j = col0 + 16 * c + r;
                const bool in = i < Nn && j < Nn;
                double add = 0.0;
                if (w && i == 0 && in) add += cf.cx * large_g(a, g, col, W * Nn + j);
                if (e && i == Nn - 1 && in) add += cf.cx * large_g(a, g, col, E * Nn + j);
                if (so && j == 0 && in) add += cf.cy * large_g(a, g, col, S * Nn + i);
                if (no && j == Nn - 1 && in) add += cf.cy * large_g(a, g, col, N * Nn + i);
                o.b[c][s] = ((in && has_f) ? o.b[c][s] : 0.0) + -2.0 * add;
            }
    };
    ld4 acc[RT][CT], sum[RT][CT];  // sum: the quarters before, where one wave takes them all
    const ld4 zero = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < CT; j++) acc[i][j] = sum[i][j] = zero;
    auto quarter = [&] {
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int j = 0; j < CT; j++) {
                sum[i][j] += acc[i][j];
                acc[i][j] = zero;
            }
    };
    const int kc = (Np / 16 + 3) / 4 * 16;
    const int k0 = SPLIT ? min(wave * kc, Np) : 0, k1 = SPLIT ? min(k0 + kc, Np) : Np;
    Blk o[2];
    if (k0 < k1) load(k0, o[0]);
    if (k0 + 16 < k1) load(k0 + 16, o[1]);
    int next = k0 + kc;  // first block of the next quarter
    for (int kb = k0; kb < k1; kb += 32)
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int kk = kb + 16 * u;
            if (kk >= k1) break;  // uniform per wave
            if (!SPLIT && kk == next) {
                quarter();
                next += kc;
            }
            fold(kk, o[u]);
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int i = 0; i < RT; i++)
#pragma unroll
                    for (int j = 0; j < CT; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(o[u].a[i][s], o[u].b[j][s], acc[i][j], 0, 0, 0);
            if (kk + 32 < k1) load(kk + 32, o[u]);
        }
    auto put = [&](int i, int j, double x) {
        if (STAGE == 1)  // padded modes are zero
            x = (i < Nn && j < Nn) ? x / (cf.cx * a.mu[min(i, Nn - 1)] + cf.cy * a.mu[min(j, Nn - 1)] + cf.lam) : 0.0;
        if (STAGE == 3 && a.op == PATCH_OP_SOLVE) {
            if (i < Nn && j < Nn) gmem(a.out)[slot * Nn * Nn + (long long)i * Nn + j] = x;
        } else {
            gmem((STAGE & 1) ? a.W1 : a.W2)[t * per + (long long)i * Np + j] = x;
        }
    };
    if (!SPLIT) {
        quarter();
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int j = 0; j < CT; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) put(row0 + 16 * i + 4 * v + q, col0 + 16 * j + r, sum[i][j][v]);
        return;
    }
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < CT; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) part[wave][2 * i + j][v][lane] = acc[i][j][v];
    __syncthreads();
    const int ti = wave >> 1, tj = wave & 1;
    if (ti >= RT || tj >= CT) return;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        double x = 0.0;
#pragma unroll
        for (int w = 0; w < 4; w++) x += part[w][wave][v][lane];
        put(row0 + 16 * ti + 4 * v + q, col0 + 16 * tj + r, x);
    }
}

template <int STAGE, bool SPLIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(SPLIT ? (STAGE == 0 ? 3 : 4) : (STAGE <= 1 ? 2 : 3), 8)))
patch_large_gemm_kernel(PatchLargeArgs a) {
    __shared__ double part[SPLIT ? 4 : 1][4][4][64];  // [wave][tile][slot][lane]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int Np = (a.N + 15) / 16 * 16, tn = (Np + 31) / 32;
    const int bid = SPLIT ? (int)blockIdx.x : (int)blockIdx.x * 4 + wave;
    int row0 = bid / tn * 32, col0 = bid % tn * 32;
    if (STAGE == 3 && a.op != PATCH_OP_SOLVE) {  // the blocks of the edge cells: first and last rows, then columns
        if (bid >= 4 * tn - 4) return;
        const int x = bid - 2 * tn;
        row0 = (x >= 0 ? 1 + x / 2 : bid < tn ? 0 : tn - 1) * 32;
        col0 = (x >= 0 ? x % 2 * (tn - 1) : bid % tn) * 32;
    } else if (bid >= tn * tn) return;  // uniform per wave; with SPLIT no block is beyond
    const bool r1 = row0 + 16 < Np, c1 = col0 + 16 < Np;
    if (r1 && c1) large_block<STAGE, SPLIT, 2, 2>(a, row0, col0, part);
    else if (r1) large_block<STAGE, SPLIT, 2, 1>(a, row0, col0, part);
    else if (c1) large_block<STAGE, SPLIT, 1, 2>(a, row0, col0, part);
    else large_block<STAGE, SPLIT, 1, 1>(a, row0, col0, part);
}

template __global__ void patch_large_gemm_kernel<0, true>(PatchLargeArgs);
template __global__ void patch_large_gemm_kernel<1, true>(PatchLargeArgs);
template __global__ void patch_large_gemm_kernel<2, true>(PatchLargeArgs);
template __global__ void patch_large_gemm_kernel<3, true>(PatchLargeArgs);
template __global__ void patch_large_gemm_kernel<0, false>(PatchLargeArgs);
template __global__ void patch_large_gemm_kernel<1, false>(PatchLargeArgs);
template __global__ void patch_large_gemm_kernel<2, false>(PatchLargeArgs);
template __global__ void patch_large_gemm_kernel<3, false>(PatchLargeArgs);

// h, or a DtN column, from the edge cells of u: one thread per boundary position
__global__ void patch_large_out_kernel(PatchLargeArgs a) {
    const int Nn = a.N, Np = (Nn + 15) / 16 * 16;
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= (long long)a.items * 4 * Nn) return;
    const long long t = e / (4 * Nn);
    const int b = (int)(e % (4 * Nn));
    int patch, rhs, col;
    large_item(a, t, patch, rhs, col);
    const long long slot = (long long)rhs * a.npatches + patch;
    const PatchCoef cf = a.coef[a.cls ? a.cls[patch] : patch];
    const double* g = (a.g && col < 0) ? a.g + slot * 4 * Nn : nullptr;
    const int sd = b / Nn, m = b % Nn;
    int i, j;
    if (sd == W) { i = 0; j = m; }
    else if (sd == E) { i = Nn - 1; j = m; }
    else if (sd == S) { i = m; j = 0; }
    else { i = m; j = Nn - 1; }
    const double uu = a.W1[t * Np * Np + (long long)i * Np + j];
    const double dd = (sd < 2) ? cf.dx : cf.dy;
    const double sg = (sd == W || sd == S) ? 2.0 / dd : -2.0 / dd;
    const double h = sg * (uu - large_g(a, g, col, b));
    if (a.op == PATCH_OP_DTN) a.out[(long long)patch * 16 * Nn * Nn + (long long)b * 4 * Nn + col] = h;
    else a.out[slot * 4 * Nn + b] = h;
}

}  // namespace efk
