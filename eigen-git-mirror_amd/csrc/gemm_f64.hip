// gemm_f64.hip -- symmetric-storage helpers: triangle transposes for uplo = 'U' and the
// symmetric L1 norm of LLT::compute.
#include "common.hpp"
#include "kernels.hpp"

namespace mi {

// ------------------------------------------------------------------------------ helpers
// W (lower) = A (upper)^T through 32x32 LDS tiles; tiles strictly above the diagonal of W
// are skipped.  Used for uplo = 'U' (LLT.h:377-399 factors the transpose).
// D may be S itself (lower -> its own upper triangle): a tile's reads and writes are separated
// by the workgroup barrier, and different tiles touch disjoint elements.
template <bool TO_LOWER, typename T>
__global__ __launch_bounds__(256) void tri_transpose_kernel(const T *S, int64_t lds_, int64_t n, T *D, int64_t ldd)
{
    // TO_LOWER: D[i][j] = S[j][i] for i >= j (D lower from S upper)
    // else    : D[j][i] = S[i][j] for i >= j (D upper from S lower)
    __shared__ T t[32][33];
    const int bi = blockIdx.x, bj = blockIdx.y;  // tile of the lower triangle (rows bi, cols bj)
    if (bj > bi) return;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
    const int64_t i0 = (int64_t)bi * 32, j0 = (int64_t)bj * 32;
    // read source block: TO_LOWER reads S[j0+.., i0+..] (upper), else S[i0+.., j0+..] (lower);
    // a thread's four loads are issued before its LDS stores (one memory round trip)
    T v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int y = ty + 8 * q;
        const int64_t rr = (TO_LOWER ? j0 : i0) + tx, cc = (TO_LOWER ? i0 : j0) + y;
        v[q] = (rr < n && cc < n) ? S[rr + cc * lds_] : T(0);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) t[ty + 8 * q][tx] = v[q];
    __syncthreads();
    for (int y = ty; y < 32; y += 8) {
        const int64_t rr = (TO_LOWER ? i0 : j0) + tx, cc = (TO_LOWER ? j0 : i0) + y;
        // element (rr, cc) of D takes source (cc, rr); keep only D's target triangle
        const bool keep = TO_LOWER ? (rr >= cc) : (rr <= cc);
        if (rr < n && cc < n && keep) D[rr + cc * ldd] = t[tx][y];
    }
}

void launch_upper_to_lower(const double *A, int64_t lda, int64_t n, double *W, int64_t ldw, hipStream_t s)
{
    const unsigned T = (unsigned)((n + 31) / 32);
    hipLaunchKernelGGL((tri_transpose_kernel<true, double>), dim3(T, T), dim3(256), 0, s, A, lda, n, W, ldw);
}

template <typename T>
void launch_upper_to_lower_t(const T *A, int64_t lda, int64_t n, T *W, int64_t ldw, hipStream_t s)
{
    const unsigned G = (unsigned)((n + 31) / 32);
    hipLaunchKernelGGL((tri_transpose_kernel<true, T>), dim3(G, G), dim3(256), 0, s, A, lda, n, W, ldw);
}
template void launch_upper_to_lower_t<float>(const float *, int64_t, int64_t, float *, int64_t, hipStream_t);

// dst (m x n, ld ldd) = src converted element by element.
template <typename S, typename D>
__global__ __launch_bounds__(256) void convert_kernel(const S *__restrict__ src, int64_t lds_, int64_t m, int64_t n,
                                                      D *__restrict__ dst, int64_t ldd)
{
    const int64_t total = m * n;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        const int64_t i = e % m, j = e / m;
        dst[i + j * ldd] = (D)src[i + j * lds_];
    }
}

template <typename S, typename D>
void launch_convert(const S *src, int64_t lds_, int64_t m, int64_t n, D *dst, int64_t ldd, hipStream_t s)
{
    const int64_t total = m * n;
    if (total == 0) return;
    const unsigned g = (unsigned)((total + 255) / 256 < 4096 ? (total + 255) / 256 : 4096);
    hipLaunchKernelGGL((convert_kernel<S, D>), dim3(g), dim3(256), 0, s, src, lds_, m, n, dst, ldd);
}
template void launch_convert<float, double>(const float *, int64_t, int64_t, int64_t, double *, int64_t, hipStream_t);
template void launch_convert<double, float>(const double *, int64_t, int64_t, int64_t, float *, int64_t, hipStream_t);

template <typename T>
void launch_lower_to_upper(const T *W, int64_t ldw, int64_t n, T *A, int64_t lda, hipStream_t s)
{
    const unsigned G = (unsigned)((n + 31) / 32);
    hipLaunchKernelGGL((tri_transpose_kernel<false, T>), dim3(G, G), dim3(256), 0, s, W, ldw, n, A, lda);
}
template void launch_lower_to_upper<double>(const double *, int64_t, int64_t, double *, int64_t, hipStream_t);
template void launch_lower_to_upper<float>(const float *, int64_t, int64_t, float *, int64_t, hipStream_t);

// Symmetric L1 norm (LLT.h:442-453): the largest column sum of |A| of the symmetric matrix, from
// one triangle, each stored element read once.  A workgroup takes a 64 x 64 tile (ti, tj) of the
// stored triangle (of its lower mirror: ti >= tj) and writes its sums along both directions:
// part[tj][64 ti + i] gets what the tile adds to the columns 64 ti.. of the symmetric matrix,
// part[ti][64 tj + j] what it adds to 64 tj.., and a diagonal tile both together -- so column c
// receives exactly one value per tile index u, part[u][c], added in that order by the second
// kernel (deterministic).  Bound by the read of the triangle (a thread's 16 loads go out
// together); n = 1024 took 228 us and n = 4001 950 us with one thread walking each row.
template <typename T>
__global__ __launch_bounds__(256) void sy_l1_tile_kernel(const T *__restrict__ A, int64_t lda, int64_t n, bool upper,
                                                         double *__restrict__ part, double *__restrict__ out)
{
    __shared__ double t[64][65];  // |element| at [second index in storage order][row in storage]
    __shared__ double red[2][4][64];
    if (blockIdx.x == 0 && threadIdx.x == 0) *out = 0.0;  // the second kernel's atomic maximum starts here
    int ti, tj;
    lower_tile((int)blockIdx.x, ti, tj);
    // storage rows r0.. (contiguous), storage columns c0..
    const int64_t r0 = 64 * (int64_t)(upper ? tj : ti), c0 = 64 * (int64_t)(upper ? ti : tj);
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    double v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int64_t r = r0 + tx, c = c0 + 16 * ty + q;
        const bool in = r < n && c < n && (upper ? r <= c : r >= c);
        const double x = (double)A[(in ? r : 0) + (in ? c : 0) * lda];
        v[q] = in ? fabs(x) : 0.0;
    }
    // along the storage rows: this thread's 16 columns, then the four waves in order
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        t[16 * ty + q][tx] = v[q];
        // a diagonal tile's column sums below take the diagonal element; the row sums skip it
        s += (ti == tj && tx == 16 * ty + q) ? 0.0 : v[q];
    }
    red[0][ty][tx] = s;
    __syncthreads();
    // along the storage columns: thread (column tx, quarter ty of the rows)
    s = 0.0;
#pragma unroll
    for (int q = 0; q < 16; ++q) s += t[tx][16 * ty + q];
    red[1][ty][tx] = s;
    __syncthreads();
    if (ty < 2) {
        const double a = (red[ty][0][tx] + red[ty][1][tx]) + (red[ty][2][tx] + red[ty][3][tx]);
        if (ti == tj) {
            red[ty][0][tx] = a;
        } else {
            // ty 0: sums of storage rows r0 + tx; ty 1: of storage columns c0 + tx
            const int64_t c = (ty == 0 ? r0 : c0) + tx;
            const int u = ty == 0 ? (int)(c0 / 64) : (int)(r0 / 64);
            if (c < n) part[(int64_t)u * n + c] = a;
        }
    }
    if (ti != tj) return;
    __syncthreads();
    if (ty == 0 && r0 + tx < n) part[(int64_t)ti * n + r0 + tx] = red[0][0][tx] + red[1][0][tx];
}

// Column sums (64 columns per workgroup, four interleaved quarters of the tile index) and
// their maximum: non-negative doubles order as their bit patterns, and a NaN sum is skipped, as
// the reference's `if (abs_col_sum > m_l1_norm)` skips it.
__global__ __launch_bounds__(256) void sy_l1_max_kernel(const double *__restrict__ part, int64_t n, double *out)
{
    __shared__ double red[4][64];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int64_t c = 64 * (int64_t)blockIdx.x + tx;
    const int T = (int)((n + 63) / 64);
    double s = 0.0;
#pragma unroll 4
    for (int u = ty; u < T; u += 4) s += part[(int64_t)u * n + (c < n ? c : n - 1)];
    red[ty][tx] = s;
    __syncthreads();
    if (ty != 0) return;
    double a = (red[0][tx] + red[1][tx]) + (red[2][tx] + red[3][tx]);
    a = c < n && a == a ? a : 0.0;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) a = fmax(a, __shfl_xor(a, d));
    if (tx == 0) atomicMax((unsigned long long *)out, (unsigned long long)__double_as_longlong(a));
}

int64_t l1norm_scratch_doubles(int64_t n) { return n * ((n + 63) / 64); }

template <typename T>
void launch_sy_l1norm(const T *A, int64_t lda, int64_t n, bool upper, double *part, double *out, hipStream_t s)
{
    const unsigned nt = (unsigned)((n + 63) / 64);
    hipLaunchKernelGGL(sy_l1_tile_kernel<T>, dim3(nt * (nt + 1) / 2), dim3(256), 0, s, A, lda, n, upper, part, out);
    hipLaunchKernelGGL(sy_l1_max_kernel, dim3(nt), dim3(256), 0, s, part, n, out);
}
template void launch_sy_l1norm<double>(const double *, int64_t, int64_t, bool, double *, double *, hipStream_t);
template void launch_sy_l1norm<float>(const float *, int64_t, int64_t, bool, double *, double *, hipStream_t);

}  // namespace mi
