// potri.hip -- the inverse of a factor and the gradient of a Gaussian process's log marginal
// likelihood from it.
//
// With A = L L^T and X = L^{-1}, A^{-1} = X^T X, and the log-likelihood's gradient with respect to
// A is g/2 (a a^T - A^{-1}), a = A^{-1} y.  Through X that is n^3/3 flops for the inverse and n^3/3
// for the product, without the three n x n right-side solves and products of the factor's general
// adjoint (1.8 n^3, and a pass over an n x n matrix between each two of them).
//
// X is built by a tree over the 128 x 128 diagonal blocks, like a block's own inverse
// (block_inverse_kernel): a level of s blocks joins neighbours A and B of s blocks each,
//   X_BA = -X_BB (L_BA X_AA),
// two launches a level, log2(n / 128) levels, every product of a level side by side.  The diagonal
// blocks come padded with the identity, so X has np = 128 ceil(n / 128) rows, those beyond n being
// the identity's.
//
// Both X (for X_BB) and X^T (for X_AA^T and X^T X) are kept, so that every operand of every product
// is read along its columns: X in the block-lower part of V (np x (np + 128), ld np) and X^T one
// block column to the right, VT = V + 128 np, in the block-upper part: block (i, j) of X, j <= i, is
// at block column j <= i of V, and its transpose, block (j, i) of X^T, at block column i + 1 > j.
//
// Tiles are 64 x 64, a wave 32 x 32 (2 x 2 FP64 MFMA tiles): the products are triangular, so a
// tile's depth runs from 64 to the whole of it, and the deepest is launched first; with 128 x 128
// tiles a few deep ones would be left running alone.
//
// n = 4096: 640 us for X and 450 us for the gradient (36 and 51 TFLOP/s; the small levels of the tree
// are bound by one tile's latency), where the general adjoints of the solve and the factor took
// 5.0 ms; 120 systems of order 512: 310 and 230 us, before 2.4 ms.
#include "common.hpp"
#include "kernels.hpp"
#include "mfma_tile.hpp"

namespace mi {

constexpr int kPT = 64;  // tile edge
using PotriTile = WaveTile<2, 2, 7>;          // depths are multiples of 64: 16 k-steps, two rounds of the buffer
using PotriTileNeg = WaveTile<2, 2, 7, true>;

// W = (L_BA X_AA)^T for the pairs of a level of s blocks: pair p's block of 128 s x 128 s (ld 128 s)
// at W + p (128 s)^2, columns (rows of L) beyond n zero.  Operands X_AA^T from VT, k from the tile's
// own row on, and L's rows.
__global__ __launch_bounds__(256, 4) void inverse_left_kernel(const double *__restrict__ L, int64_t ldl, int64_t n,
                                                              const double *__restrict__ VT, int64_t np, int s,
                                                              double *__restrict__ W, int64_t sL, int64_t sV,
                                                              int64_t sW)
{
    L += blockIdx.z * sL;
    VT += blockIdx.z * sV;
    W += blockIdx.z * sW;
    const int nt = 2 * s;
    const int p = (int)blockIdx.x / (nt * nt), o = (int)blockIdx.x % (nt * nt), ti = o / nt, tj = o % nt;
    const int64_t S = 128 * (int64_t)s, A0 = 2 * S * p, i0 = A0 + kPT * ti, j0 = A0 + S + kPT * tj;
    if (j0 >= np) return;  // the last pair's B may be shorter
    const int w = threadIdx.x >> 6, r0 = 32 * (w >> 1), c0 = 32 * (w & 1);
    const int jv = (int)(n - j0 < kPT ? n - j0 : kPT);  // valid columns (rows of L)
    PotriTile t;
    t.zero();
    if (jv > 0) {
        t.setup(VT + i0 + i0 * np, np, r0, kPT, L + j0 + i0 * ldl, ldl, c0, jv, (int)(S - kPT * ti));
        t.run();
    }
    double *C = W + (size_t)p * S * S + kPT * ti + (int64_t)kPT * tj * S;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = c0 + t.col_of(b, r);
                C[r0 + t.row_of(a) + j * S] = j < jv ? t.acc[a][b][r] : 0.0;
            }
}

// X_BA^T = -(W X_BB^T) to VT and, unless this is the last level, X_BA to V.
__global__ __launch_bounds__(256, 4) void inverse_right_kernel(double *__restrict__ V, int64_t np, int s, bool last,
                                                               const double *__restrict__ W, int64_t sV, int64_t sW)
{
    V += blockIdx.z * sV;
    W += blockIdx.z * sW;
    const int nt = 2 * s;
    const int p = (int)blockIdx.x / (nt * nt), o = (int)blockIdx.x % (nt * nt), ti = nt - 1 - o / nt, tj = o % nt;
    const int64_t S = 128 * (int64_t)s, A0 = 2 * S * p, B0 = A0 + S, i0 = B0 + kPT * ti, j0 = A0 + kPT * tj;
    if (i0 >= np) return;
    const int w = threadIdx.x >> 6, r0 = 32 * (w >> 1), c0 = 32 * (w & 1);
    PotriTileNeg t;  // rows: X_BA's columns j0 .., columns: its rows i0 ..
    t.zero();
    t.setup(W + (size_t)p * S * S + kPT * tj, S, r0, kPT, V + i0 + B0 * np, np, c0, kPT, kPT * (ti + 1));
    t.run();
    double *VT = V + 128 * np;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t j = j0 + r0 + t.row_of(a), i = i0 + c0 + t.col_of(b, r);
                VT[j + i * np] = t.acc[a][b][r];
                if (!last) V[i + j * np] = t.acc[a][b][r];
            }
}

// G <- g/2 (a a^T - X^T X), full: the lower tiles, each stored in both triangles.
__global__ __launch_bounds__(256, 4) void gp_gradient_kernel(const double *__restrict__ VT, int64_t np, int64_t n,
                                                             const double *__restrict__ a, const double *__restrict__ g,
                                                             double *__restrict__ G, int64_t ldg, int64_t sV, int64_t sa,
                                                             int64_t sG)
{
    VT += blockIdx.z * sV;
    a += blockIdx.z * sa;
    G += blockIdx.z * sG;
    const double h = 0.5 * g[blockIdx.z];
    const int u = (int)blockIdx.x;  // tile u of the rows' order: (I, J), J <= I; the deepest rows first
    int I = (int)((__fsqrt_rn(8.0f * (float)u + 1.0f) - 1.0f) * 0.5f);
    while (I * (I + 1) / 2 > u) --I;
    while ((I + 1) * (I + 2) / 2 <= u) ++I;
    const int J = u - I * (I + 1) / 2;
    const int w = threadIdx.x >> 6, r0 = 32 * (w >> 1), c0 = 32 * (w & 1);
    if (I == J && r0 < c0) return;  // strictly upper
    const int64_t i0 = (int64_t)kPT * I, j0 = (int64_t)kPT * J;
    PotriTile t;
    t.zero();
    t.setup(VT + i0 + i0 * np, np, r0, kPT, VT + j0 + i0 * np, np, c0, kPT, (int)(np - i0));
    t.run();
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t i = i0 + r0 + t.row_of(x), j = j0 + c0 + t.col_of(b, r);
                if (i < n && j <= i) {
                    const double v = h * (a[i] * a[j] - t.acc[x][b][r]);
                    G[i + j * ldg] = v;
                    G[j + i * ldg] = v;
                }
            }
}

int64_t inverse_pairs_edge(int64_t n)
{
    const int64_t nblk = (n + kNB - 1) / kNB;
    int64_t s = 1;
    while (2 * s < nblk) s *= 2;
    return nblk > 1 ? s * kNB : 0;
}

void launch_factor_inverse(const double *L, int64_t ldl, int64_t n, double *V, double *W, hipStream_t st,
                           const Batch &bt)
{
    const int64_t nblk = (n + kNB - 1) / kNB, np = nblk * kNB;
    launch_block_inverses_to(L, ldl, n, V + kNB * np, V, np, kNB * (np + 1), st, bt.count, bt.a, bt.aux);
    for (int64_t s = 1; s < nblk; s *= 2) {
        // pairs with a B of at least one block
        const unsigned grid = (unsigned)((nblk - s + 2 * s - 1) / (2 * s) * 4 * s * s);
        hipLaunchKernelGGL(inverse_left_kernel, dim3(grid, 1, bt.count), dim3(256), 0, st, L, ldl, n, V + kNB * np, np,
                           (int)s, W, bt.a, bt.aux, bt.aux2);
        hipLaunchKernelGGL(inverse_right_kernel, dim3(grid, 1, bt.count), dim3(256), 0, st, V, np, (int)s, 2 * s >= nblk,
                           W, bt.aux, bt.aux2);
    }
}

void launch_gp_gradient(const double *V, int64_t n, const double *a, const double *g, double *G, int64_t ldg,
                        hipStream_t st, const Batch &bt)
{
    const int64_t np = (n + kNB - 1) / kNB * kNB, T = (n + kPT - 1) / kPT;
    hipLaunchKernelGGL(gp_gradient_kernel, dim3((unsigned)(T * (T + 1) / 2), 1, bt.count), dim3(256), 0, st,
                       V + kNB * np, np, n, a, g, G, ldg, bt.aux, bt.b, bt.g);
}

}  // namespace mi
