// potrf_diag.hip -- inverses of the diagonal blocks of a factor, used by the solve.
//
// The diagonal-block Cholesky itself (llt_inplace<double,Lower>::unblocked on A11,
// Eigen/src/Cholesky/LLT.h:312-336, called at :363) and the panel solve (LLT.h:364) run
// inside the fused factorization step (factor_step.hip, potrf_device.hpp):
//   * the 128 x 128 block is held in LDS and factored in 16-column panels: two waves run the
//     column loop of LLT.h:320-334 (pivot test, sqrt, scale, rank-1 update) in registers on the
//     row broadcast, which leaves the inverse of the 16 x 16 leaf too, while the other two
//     store the previous panel and bring the column after next up to date with FP64 MFMA;
//   * the pivot test is Eigen's `x <= 0 -> fail at column k` (LLT.h:327-330), so a NaN
//     pivot passes as in Eigen; the first failing column goes to `info` (LAPACK k+1); a last
//     block narrower than 128 is padded with the identity (L_pad = [L 0; 0 I]);
//   * the panel solve A21 <- A21 L11^{-T} (TriangularSolverMatrix.h:186-329) is blocked by
//     16 columns with the leaf inverses; the MFMA result layout is the operand layout of the
//     next k-step, so solved blocks feed the next MFMAs straight from registers.
// The solve's block inverses L_bb^{-1} are built after the factor from its leaf inverses or from L
// alone (block_inverse_kernel), and the couplings from them (block_coupling_kernel).
#include "leaf_device.hpp"
#include "potrf_device.hpp"

namespace mi {

// Packed lower 16 x 16 tiles of a 128 x 128 block in LDS, the diagonal included: tile (ti, tj),
// ti >= tj, at kTile (ti (ti + 1) / 2 + tj), column-major with a column every kTileLd doubles: one
// more than the rows, so that 16 lanes reading along a row hit different banks.
constexpr int kTileLd = 17, kTile = 16 * kTileLd;
__device__ __forceinline__ constexpr int tile_at(int ti, int tj) { return kTile * ((ti * (ti + 1)) / 2 + tj); }

// The MFMA operands of 16 x 16 tiles at LDS offset o: of A in a product A B (P[i][k] = A[i][k]) and
// of B (Q[j][k] = B[k][j]), k = 4s + lane/16.
__device__ __forceinline__ void tile_p(const double *S, int o, double (&p)[4])
{
    const int l = lane_id();
#pragma unroll
    for (int s = 0; s < 4; ++s) p[s] = S[o + (l & 15) + kTileLd * (4 * s + (l >> 4))];
}
__device__ __forceinline__ void tile_q(const double *S, int o, double (&q)[4])
{
    const int l = lane_id();
#pragma unroll
    for (int s = 0; s < 4; ++s) q[s] = S[o + 4 * s + (l >> 4) + kTileLd * (l & 15)];
}
// acc += A B; acc[r] is element (lane%16, 4r + lane/16).
__device__ __forceinline__ void tile_mma(const double (&p)[4], const double (&q)[4], dvec4 &acc)
{
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = mfma_f64(q[s], p[s], acc);
}
__device__ __forceinline__ void tile_put(double *S, int o, const dvec4 &acc, bool negate)
{
    const int l = lane_id();
#pragma unroll
    for (int r = 0; r < 4; ++r) S[o + (l & 15) + kTileLd * (4 * r + (l >> 4))] = negate ? -acc[r] : acc[r];
}

// One level of the tree over the diagonal: pairs of SZ-tile blocks A (tiles A0 ..) and B (tiles
// A0 + SZ ..), T = L_BA X_AA and then X_BA = -X_BB T, in place of L_BA.  A wave takes a tile row of
// T, then a tile column of X_BA, of pair w / SZ: equal shares, as X_AA and X_BB are triangular, and
// each operand tile of the row or column is read once.
template <int SZ>
__device__ __forceinline__ void inverse_level(double *S, int w)
{
    const int A0 = (w / SZ) * 2 * SZ, B0 = A0 + SZ, x = w % SZ;
    dvec4 acc[SZ];
    double p[SZ][4], q[4];
#pragma unroll
    for (int k = 0; k < SZ; ++k) tile_p(S, tile_at(B0 + x, A0 + k), p[k]);
#pragma unroll
    for (int tj = 0; tj < SZ; ++tj) {
        acc[tj] = dvec4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = tj; k < SZ; ++k) {
            tile_q(S, tile_at(A0 + k, A0 + tj), q);
            tile_mma(p[k], q, acc[tj]);
        }
    }
    // only this wave reads its tile row of L_BA
#pragma unroll
    for (int tj = 0; tj < SZ; ++tj) tile_put(S, tile_at(B0 + x, A0 + tj), acc[tj], false);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SZ; ++k) tile_q(S, tile_at(B0 + k, A0 + x), p[k]);
#pragma unroll
    for (int ti = 0; ti < SZ; ++ti) {
        acc[ti] = dvec4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k <= ti; ++k) {
            tile_p(S, tile_at(B0 + ti, B0 + k), q);
            tile_mma(q, p[k], acc[ti]);
        }
    }
    // only this wave reads its tile column of T
#pragma unroll
    for (int ti = 0; ti < SZ; ++ti) tile_put(S, tile_at(B0 + ti, A0 + x), acc[ti], true);
    __syncthreads();
}

// Step K of the inverse of a lower 16 x 16 leaf: lane c of a row of 16 holds row c of the leaf in
// v[0..15] and column c of the inverse in x[0..15].  x[K] is final after the division; rows M > K
// take L_MK x[K] away.  (Lanes c > K are left alone: their x[K] is 0, but L_MK may be infinite.)
template <int K, int M>
__device__ __forceinline__ void leaf_inverse_rows(const double (&v)[16], double (&x)[16], int c)
{
    if constexpr (M < 16) {
        double t = x[M];
        row_fnma<M, M == K + 1>(t, v[K], x[K]);
        x[M] = c <= K ? t : x[M];
        leaf_inverse_rows<K, M + 1>(v, x, c);
    }
}
template <int K>
__device__ __forceinline__ void leaf_inverse_steps(const double (&v)[16], double (&x)[16], int c)
{
    if constexpr (K < 16) {
        const double d = row_bcast<K>(v[K]);
        x[K] = c <= K ? x[K] / d : 0.0;
        leaf_inverse_rows<K, K + 1>(v, x, c);
        leaf_inverse_steps<K + 1>(v, x, c);
    }
}

// Workgroup b: X_b^T = L_bb^{-T} to Wt + b sBlk and X_b to Wx + b sBlk (ld ldw).
// A triangular inverse by a tree over the diagonal 16 x 16 leaves (the recursive form of
// LAPACK's dtrtri): from the 8 leaf inverses X_pp, three levels double the inverted diagonal
// blocks, X_BA = -X_BB (L_BA X_AA) for [A; B] of 16 + 16, 32 + 32 and 64 + 64 rows, each level's
// products over 16 x 16 tiles on FP64 MFMA, in place in LDS.  Three levels of two products each
// instead of eight dependent 16-column solve steps: the kernel is bound by one workgroup's
// latency, not by its flops.  The leaf inverses come from the factorization's panel images, or,
// without them (Wleaf null: a factor the caller kept), from the leaves, two per wave on the row
// broadcast, where a kernel of its own took as long as this one.  Beyond bs (a last block narrower
// than 128) L reads as the identity, so X is padded with the identity.
// Batched launches (every kernel of this file): system z = blockIdx.z, its pointers advanced
// by z times their strides (s*), its info at info + z.
template <typename T>
__global__ __launch_bounds__(256) void block_inverse_kernel(const T *__restrict__ L, int64_t ldl, int64_t n,
                                                            const double *__restrict__ Wleaf, double *Wt, double *Wx,
                                                            int64_t ldw, int64_t sBlk, const int *info, int64_t sL,
                                                            int64_t sWl, int64_t sWo)
{
    __shared__ double S[36 * kTile];  // the packed lower tiles
    const int64_t z = blockIdx.z;
    L += z * sL;
    Wt += z * sWo;
    Wx += z * sWo;
    if (info) info += z;
    if (factor_failed(info)) return;
    const int b = (int)blockIdx.x;
    const int64_t kb = (int64_t)b * 128;
    const int bs = (int)((n - kb) < 128 ? (n - kb) : 128);
    const T *Lb = L + kb + kb * ldl;
    const int tid = threadIdx.x, l = lane_id();
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

    // the lower tiles of L_bb: a thread takes row r, columns of parity tid / 128, all its loads in
    // flight (from clamped, in-bounds addresses) before their LDS stores
    {
        const int r = tid & 127, ch = tid >> 7, rt = r >> 4;
        double x[8];
        if (Wleaf) {
            const double *Xl = Wleaf + z * sWl + (size_t)b * kPanelDoubles + kLeafOffset;
#pragma unroll
            for (int q = 0; q < 8; ++q) x[q] = Xl[tid + 256 * q];
        }
        T v[64];
#pragma unroll
        for (int q = 0; q < 64; ++q) {
            const int c = 2 * q + ch;
            const bool in = r < bs && c <= r;
            v[q] = Lb[(in ? r : 0) + (int64_t)(in ? c : 0) * ldl];
        }
#pragma unroll
        for (int q = 0; q < 64; ++q) {
            const int c = 2 * q + ch;
            const bool in = r < bs && c <= r;
            if ((q >> 3) <= rt) S[tile_at(rt, q >> 3) + (r & 15) + kTileLd * (c & 15)] = in ? (double)v[q] : r == c ? 1.0 : 0.0;
        }
        __syncthreads();
        if (Wleaf) {  // element tid of leaf q: (tid % 16, tid / 16)
#pragma unroll
            for (int q = 0; q < 8; ++q)
                S[tile_at(q, q) + (tid & 15) + kTileLd * (tid >> 4)] = (tid >> 4) <= (tid & 15) ? x[q] : 0.0;
        } else {
            const int c = l & 15, o = tile_at(2 * w, 2 * w) + ((l >> 4) & 1) * (tile_at(2 * w + 1, 2 * w + 1) - tile_at(2 * w, 2 * w));
            double u[16], y[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                u[k] = S[o + c + kTileLd * k];
                y[k] = k == c ? 1.0 : 0.0;
            }
            leaf_inverse_steps<0>(u, y, c);
            if (l < 32) {
#pragma unroll
                for (int k = 0; k < 16; ++k) S[o + k + kTileLd * c] = y[k];
            }
        }
    }
    __syncthreads();
    inverse_level<1>(S, w);
    inverse_level<2>(S, w);
    inverse_level<4>(S, w);

    // X and X^T, zeros above and below the diagonal; two elements a store (ldw and sBlk are even)
    Wt += b * sBlk;
    Wx += b * sBlk;
#pragma unroll 8
    for (int e = tid; e < 128 * 64; e += 256) {
        const int f = 2 * (e & 63), c = e >> 6;  // elements (f, c), (f + 1, c) of X and of X^T
        dvec2 x = {0.0, 0.0}, xt = {0.0, 0.0};
        if ((f >> 4) >= (c >> 4)) {
            const double *t = S + tile_at(f >> 4, c >> 4) + (f & 15) + kTileLd * (c & 15);
            x = dvec2{t[0], t[1]};
        }
        if ((c >> 4) >= (f >> 4)) {
            const double *t = S + tile_at(c >> 4, f >> 4) + (c & 15) + kTileLd * (f & 15);
            xt = dvec2{t[0], t[kTileLd]};
        }
        *(dvec2 *)(Wx + f + ldw * c) = x;
        *(dvec2 *)(Wt + f + ldw * c) = xt;
    }
}

// Couplings of the block substitution: with them a block of the solution depends on its three
// predecessors through one product each,
//   Y_i = X_i (B_i - sum_{j<i-3} L_ij Y_j) - M3_i Y_{i-3} - M2_i Y_{i-2} - M_i Y_{i-1},
// so everything else is done before they are published (solve_couplings: none below 8 blocks,
// the third only from 16 blocks on).  Workgroup q nblk + b, distance d = 1 + q / 2: q even, M_b / M2_b / M3_b = X_b L_{b,b-d} (b >= d); q odd, N_b / N2_b / N3_b
// = X_b^T L_{b+d,b}^T (b + d < nblk).  128 x 128 each at Winv[b] + kInvM / kInvN / kInvM2 /
// kInvN2 / kInvM3 / kInvN3 (ld 128); entries of L outside the matrix read as 0.
//
// Bound by latency: a workgroup takes a 64 x 64 quadrant (blockIdx.y), a wave 32 x 32 of it, so that
// a few blocks' products still use the chip, and the k outside the triangle of X (whole chunks of 32)
// is not multiplied.  Two chunks' operands are in flight: 8 k-steps of 4 MFMAs each.
template <typename T>
__global__ __launch_bounds__(256, 2) void block_coupling_kernel(const T *__restrict__ L, int64_t ldl, int64_t n,
                                                                double *__restrict__ Winv, const int *info, int64_t sL,
                                                                int64_t sWo)
{
    const int64_t z = blockIdx.z;
    L += z * sL;
    Winv += z * sWo;
    if (info) info += z;
    if (factor_failed(info)) return;
    const int nblk = (int)((n + 127) / 128);
    const int q = (int)blockIdx.x / nblk, b = (int)blockIdx.x % nblk;
    const bool fwd = (q & 1) == 0;
    const int d = 1 + q / 2;
    if (fwd ? b < d : b + d > nblk - 1) return;
    double *Wb = Winv + (size_t)b * kInvDoubles;
    const int l = lane_id(), kl = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i0 = 64 * ((int)blockIdx.y >> 1) + 32 * (w >> 1), j0 = 64 * ((int)blockIdx.y & 1) + 32 * (w & 1);
    // P[i][k] = X_b[i][k] (forward; 0 for k > i) or X_b^T[i][k] (0 for k < i) at P + i + 128 k;
    // Q[j][k] = L[128 b + k][128 (b-d) + j] (forward; rows k < lim exist) or
    //           L[128 (b+d) + j][128 b + k] (backward; rows j < lim exist)
    const double *P = Wb + (fwd ? kInvX : 0) + i0 + (l & 15) + 128 * kl;
    const int64_t r0 = fwd ? 128 * (int64_t)b : 128 * (int64_t)(b + d);
    const int64_t c0 = fwd ? 128 * (int64_t)(b - d) : 128 * (int64_t)b;
    const int lim = (int)((n - r0) < 128 ? (n - r0) : 128);
    const int clo = fwd ? 0 : i0 / 32, chi = fwd ? i0 / 32 + 1 : 4;  // chunks of the triangle
    double pv[2][8][2];
    T qv[2][8][2];
    bool in[2][8][2];
    auto load = [&](int u, int c) {
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int k = 32 * c + 4 * s;  // + kl
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                pv[u][s][a] = P[16 * a + 128 * k];
                const int j = j0 + 16 * a + (l & 15);
                in[u][s][a] = (fwd ? k + kl : j) < lim;
                const bool i = in[u][s][a];
                qv[u][s][a] = L[fwd ? (r0 + (i ? k + kl : 0)) + (c0 + j) * ldl : (r0 + (i ? j : 0)) + (c0 + k + kl) * ldl];
            }
        }
    };
    dvec4 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int e = 0; e < 2; ++e) acc[a][e] = dvec4{0.0, 0.0, 0.0, 0.0};
    load(0, 0);
    load(1, 1);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (c >= clo && c < chi) {
#pragma unroll
            for (int s = 0; s < 8; ++s)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const double qe = in[c & 1][s][e] ? (double)qv[c & 1][s][e] : 0.0;
#pragma unroll
                    for (int a = 0; a < 2; ++a) acc[a][e] = mfma_f64(qe, pv[c & 1][s][a], acc[a][e]);
                }
        }
        if (c < 2) load(c & 1, c + 2);
    }
    double *C = Wb + (fwd ? (d == 1 ? kInvM : d == 2 ? kInvM2 : kInvM3) : (d == 1 ? kInvN : d == 2 ? kInvN2 : kInvN3));
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                C[(i0 + 16 * a + (l & 15)) + 128 * (j0 + 16 * e + 4 * r + kl)] = acc[a][e][r];
}

template <typename T>
void launch_block_inverses(const T *L, int64_t lda, int64_t n, const double *Wleaf, double *Winv, const int *info,
                           hipStream_t s, bool couplings, const Batch &bt)
{
    const unsigned nblk = (unsigned)((n + 127) / 128);
    hipLaunchKernelGGL(block_inverse_kernel<T>, dim3(nblk, 1, bt.count), dim3(256), 0, s, L, lda, n, Wleaf, Winv,
                       Winv + kInvX, (int64_t)128, kInvDoubles, info, bt.a, bt.leaf, bt.inv);
    if (couplings && solve_couplings(nblk) > 0)
        hipLaunchKernelGGL(block_coupling_kernel<T>, dim3(2 * solve_couplings(nblk) * nblk, 4, bt.count), dim3(256), 0,
                           s, L, lda, n, Winv, info, bt.a, bt.inv);
}

void launch_block_inverses_to(const double *L, int64_t lda, int64_t n, double *Wt, double *Wx, int64_t ldw,
                              int64_t stride, hipStream_t s, unsigned count, int64_t sL, int64_t sW)
{
    const unsigned nblk = (unsigned)((n + 127) / 128);
    hipLaunchKernelGGL(block_inverse_kernel<double>, dim3(nblk, 1, count), dim3(256), 0, s, L, lda, n,
                       (const double *)nullptr, Wt, Wx, ldw, stride, (const int *)nullptr, sL, (int64_t)0, sW);
}

template void launch_block_inverses<double>(const double *, int64_t, int64_t, const double *, double *, const int *,
                                            hipStream_t, bool, const Batch &);
template void launch_block_inverses<float>(const float *, int64_t, int64_t, const double *, double *, const int *,
                                           hipStream_t, bool, const Batch &);

}  // namespace mi
