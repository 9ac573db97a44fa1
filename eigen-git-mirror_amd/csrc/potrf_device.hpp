// potrf_device.hpp -- device-side pieces of the diagonal-block factor and the panel solve,
// shared by the stand-alone kernels (potrf_diag.hip) and the fused factorization step
// (factor_step.hip).  See potrf_diag.hip for the algorithms and their reference citations.
#pragma once
#include "common.hpp"
#include "kernels.hpp"
#include "leaf_device.hpp"
#include "mfma_tile.hpp"

namespace mi {

// The 128 x 128 diagonal block lives in LDS as its 36 lower 16 x 16 tiles (72 KiB instead of a
// full square), each column-major, tile (ti, tj) at 256 * (ti(ti+1)/2 + tj): so two
// workgroups fit on a CU.  sl(r, c) addresses element (r, c) for r >= c, or any element of a
// diagonal tile; an MFMA operand (16 rows of 4 consecutive columns) is then 64 consecutive
// doubles.
__device__ __forceinline__ int sl(int r, int c)
{
    const int ti = r >> 4, tj = c >> 4;
    return 256 * ((ti * (ti + 1)) / 2 + tj) + (r & 15) + 16 * (c & 15);
}
// Panel p (columns c0..c0+15 of the 128 x 128 block in S, tiled: sl), waves 0 and 1 (2 and 3
// meanwhile store the previous panel and update a later column, see potrf_in_lds).  Each row of 16
// lanes holds the whole 16 x 16 leaf in u (leaf_device.hpp), so its broadcasts need no barrier and
// no scalar registers; v holds one more row per lane, which takes the same column operations: the
// up to 112 rows below the leaf (row c0+16+64w+l), for which they are the panel solve A_ip
// L_pp^{-T}, and in the last 16 lanes of wave 1 (never a row below) the rows of the 16 x 16
// identity, which become L_pp^{-T}, i.e. column i of X_pp = L_pp^{-1} in lane 48+i, written to xleaf
// (LDS) column-major.  (With readlane broadcasts and the leaf in lanes 0..15, three waves took a panel in
// 4300 cycles; this form takes 2900, and two waves are left for the updates.)
//
// Returns the failing panel column or -1, the same in both waves.  The factored leaf is left in u:
// it is written back to S only after a barrier, since the other wave reads the unfactored leaf from
// S here and may still be doing so when one wave is done.
__device__ __forceinline__ int panel_factor2(double *S, int c0, double *xleaf, double (&u)[16])
{
    const int l = lane_id(), w = threadIdx.x >> 6;
    const int rb = c0 + 16 + 64 * w + l;
    const bool ident = w == 1 && l >= 48, below = !ident && rb < 128;
    const int r = below ? rb : c0 + (l & 15);
    double v[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) u[c] = S[sl(c0 + (l & 15), c0 + c)];
#pragma unroll
    for (int c = 0; c < 16; ++c) v[c] = S[sl(r, c0 + c)];
    if (ident) {
#pragma unroll
        for (int c = 0; c < 16; ++c) v[c] = (c == l - 48) ? 1.0 : 0.0;
    }
    const int fail = leaf_factor(u, v);
    if (fail >= 0) return fail;
    if (below) {  // rows no other wave reads before the next barrier
#pragma unroll
        for (int c = 0; c < 16; ++c) S[sl(r, c0 + c)] = v[c];
    }
    if (ident) {
#pragma unroll
        for (int c = 0; c < 16; ++c) xleaf[c + 16 * (l - 48)] = v[c];
    }
    return -1;
}

// LDS of one workgroup, shared by the two roles: the 36 lower tiles of the block for the
// factor, or the 28 strictly lower tiles of L11 plus the 8 leaf inverses for the panel solve.
constexpr int kSmem = 36 * 256;

// A (global, ld lda, valid order bs) -> S (lower part, identity beyond bs); a thread's 64 loads all
// in flight, from clamped in-bounds addresses.  T = float widens to FP64.
template <typename T>
__device__ __forceinline__ void block_to_lds(double *S, const T *__restrict__ Ab, int64_t lda, int bs)
{
    const int tid = threadIdx.x, r = tid & 127, ch = tid >> 7;
    T a[64];
#pragma unroll
    for (int q = 0; q < 64; ++q) {
        const int c = 2 * q + ch;
        const bool in = r < bs && c < bs;
        a[q] = Ab[(in ? r : 0) + (int64_t)(in ? c : 0) * lda];
    }
#pragma unroll
    for (int q = 0; q < 64; ++q) {
        const int c = 2 * q + ch;
        const bool in = r < bs && c < bs;
        if (r >= c) S[sl(r, c)] = in ? (double)a[q] : (r == c ? 1.0 : 0.0);
    }
}

template <typename T>
__device__ __forceinline__ void lds_to_block(const double *S, T *__restrict__ Ab, int64_t lda, int bs)
{
    const int tid = threadIdx.x, r = tid & 127, ch = tid >> 7;
#pragma unroll 8
    for (int q = 0; q < 64; ++q) {
        const int c = 2 * q + ch;
        if (r >= c && r < bs) Ab[r + (int64_t)c * lda] = (T)S[sl(r, c)];
    }
}

// One 16 x 16 tile of the rank-16 update in LDS: C -= Pi Pj^T (operands in registers, lane l
// k-step s: row l%16, column 4s + l/16), C at tile offset + l + 64 r.  A diagonal tile is
// updated whole: the entries above its diagonal are never read as data.
__device__ __forceinline__ void lds_tile_update(double *C, const double (&Pi)[4], const double (&Pj)[4])
{
    double old[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) old[r] = C[64 * r];
    dvec4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = mfma_f64(Pj[s], Pi[s], acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) C[64 * r] = old[r] - acc[r];
}

// Tiles (i, j), i = i0, i0 + 2, ... (NT of them), of the block in S: C[x] (the tile's elements l + 64 r)
// less its products with the panels 0 .. p, in turn, to S.  Each product's operands are read during the
// one before.
template <int NT>
__device__ __forceinline__ void column_products(double *S, int i0, int j, int p, double (&C)[3][4])
{
    const int l = lane_id();
    const double *pj = S + 256 * ((j * (j + 1)) / 2) + l;
    const double *pi[NT];
    double Pj[4], Pi[NT][4];
#pragma unroll
    for (int x = 0; x < NT; ++x) pi[x] = S + 256 * (((i0 + 2 * x) * (i0 + 2 * x + 1)) / 2) + l;
    auto operands = [&](int q) {
#pragma unroll
        for (int s = 0; s < 4; ++s) Pj[s] = pj[256 * q + 64 * s];
#pragma unroll
        for (int x = 0; x < NT; ++x)
#pragma unroll
            for (int s = 0; s < 4; ++s) Pi[x][s] = pi[x][256 * q + 64 * s];
    };
    operands(0);
    for (int q = 0; q <= p; ++q) {
        dvec4 acc[NT];
#pragma unroll
        for (int x = 0; x < NT; ++x) acc[x] = dvec4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int x = 0; x < NT; ++x) acc[x] = mfma_f64(Pj[s], Pi[x][s], acc[x]);
        operands(q < p ? q + 1 : p);
#pragma unroll
        for (int x = 0; x < NT; ++x)
#pragma unroll
            for (int r = 0; r < 4; ++r) C[x][r] -= acc[x][r];
    }
#pragma unroll
    for (int x = 0; x < NT; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[256 * (((i0 + 2 * x) * (i0 + 2 * x + 1)) / 2 + j) + l + 64 * r] = C[x][r];
}

// Image stores reach memory by themselves (agent-scope stores are written through), so publishing
// them takes the wait for them and the flag's store, no L2 writeback.
__device__ __forceinline__ void image_store(double *p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The panel flag of the launch with epoch e goes from 8 (e - 1) to 8 e: + 1 by each of two waves once
// the image's block columns below kPart1, then below kPart2, are in memory, 8 e when all of it is.
// The rows take about as long for the first part (2.8 us of MFMAs, and the image's tiles from memory)
// as the diagonal role for the rest, and are left with 12 of their 144 MFMAs a row tile when the block
// is done.  One part, two, and three with diag_helper and half tiles (syrk_tile): 41, 38 and 33 us a
// launch in FP64 at n <= 1024; factor and solve at n = 3001 1330, 1230 and 1123 us, FP32 at n = 4001
// 1979, 1850 and 1735 us.  (30 and 1057 us with the helpers' tiles in the image.)
constexpr int kPart1 = 4, kPart2 = 6;

// Where diag_helper leaves tile (i, j), i >= j, of the updated diagonal block in the panel image (lane
// order: elements l + 64 r): the places that L's tile and leaf j's inverse take when panel j is stored.
__device__ __forceinline__ constexpr int helper_tile(int i, int j)
{
    return i == j ? (int)kLeafOffset + 256 * j : 256 * ((i * (i - 1)) / 2 + j);
}

// Cholesky of the 128 x 128 lower block in S (all 256 threads), in eight 16-column panels with
// a one-panel lookahead inside the block.  After panel p is factored, with T = 7-p tile rows
// below it and their operands P_x = tile (p+1+x, p), x < T:
//   A(p): the leaf of p goes back to S; the T tiles of column p+1 get panel p's update (the
//         waves round-robin), barrier;
//   B(p): waves 0 and 1 factor panel p+1 (panel_factor2: VALU) while waves 2 and 3 store panel p
//         (its tiles and its leaf's inverse) to the panel image W and bring column p+2 up to
//         panel p on the matrix core (its tiles by panels 0 .. p), barrier.
// Column p+1 thus has every earlier panel's update before its factor, and B's products, 12 tile
// products at most, run under the column loop (1.4 us; applying panel p to all the tiles right of column
// p+1 instead took up to 21, 2.8 us).  The panels below kPart1 and kPart2 are published in B of that
// panel, a panel's time after their last store.
// Returns the first failing column or -1 (uniform); the columns after it are then factored all the same,
// to no use (a test of the failure in each panel took longer).  xs: 2 x 256 doubles of LDS, s_fail: an
// LDS int.
//
// helped: null when S holds the whole block; else S has tile columns 0 and 1 of it, and the others are
// read from the image (helper_tile), each one phase ahead, columns 2, 3 and 4 .. 7 once helped[0] and
// helped[1] have reached `epoch` (diag_helper).  Tile (i, j) is read in B(j - 3) and used in B(j - 2), so
// the panel's own tile can take its place in B(j).
__device__ __forceinline__ int potrf_in_lds(double *S, double *xs, int *s_fail, double *W, uint32_t *flag,
                                            const uint32_t *helped, uint32_t epoch, int *status)
{
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = lane_id();
    double *Xl = W + kLeafOffset;
    double lv[16];
    double next[3][4];  // waves 2 and 3: this wave's tiles (i, j), i = j + w - 2, + 2, + 4, of the next column
    auto fetch = [&](int j) {
        if (helped && (j == 2 || j == 4)) {
            uint32_t spins = 0;
            while (__hip_atomic_load(helped + (j == 4), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < epoch) {
                __builtin_amdgcn_s_sleep(1);
                if (++spins > (1u << 22)) {
                    atomicOr(status, MI_PANEL_TIMEOUT);
                    break;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");  // the loads stay behind the flag's
        }
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            const int i = j + w - 2 + 2 * x;
            if (i < 8) {
                if (helped) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) next[x][r] = coherent_load(W + helper_tile(i, j) + l + 64 * r);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) next[x][r] = S[256 * ((i * (i + 1)) / 2 + j) + l + 64 * r];
                }
            }
        }
    };
    if (tid == 0) *s_fail = -1;
    lds_barrier();
    if (w < 2) {
        const int f = panel_factor2(S, 0, xs, lv);
        if (w == 0 && l == 0 && f >= 0) *s_fail = f;
    } else {
        fetch(2);
    }
    lds_barrier();
    for (int p = 0; p < 7; ++p) {
        const int T = 7 - p;
        const int tb = p + 1;  // first trailing tile row / column
        auto operand = [&](int x, double (&P)[4]) {
            const double *src = S + 256 * (((tb + x) * (tb + x + 1)) / 2 + p) + l;
#pragma unroll
            for (int s = 0; s < 4; ++s) P[s] = src[64 * s];
        };
        // ---- A(p)
        {
            double P0[4], Pw[2][4];
            operand(0, P0);
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (w + 4 * h < T) operand(w + 4 * h, Pw[h]);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int x = w + 4 * h;
                if (x < T) lds_tile_update(S + 256 * (((tb + x) * (tb + x + 1)) / 2 + tb) + l, Pw[h], P0);
            }
        }
        if (w == 0 && l < 16) {  // the leaf of p: read by nobody until the final copy out
#pragma unroll
            for (int c = 0; c < 16; ++c) S[sl(16 * p + l, 16 * p + c)] = lv[c];
        }
        lds_barrier();
        // ---- B(p)
        if (w < 2) {
            const int f = panel_factor2(S, 16 * tb, xs + 256 * (tb & 1), lv);
            if (w == 0 && l == 0 && f >= 0 && *s_fail < 0) *s_fail = 16 * tb + f;
        } else {
            if (p == kPart1 || p == kPart2) {  // this wave's stores of the panels before p
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                if (l == 0) __hip_atomic_fetch_add(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            // column j = p + 2: tile rows i = j + w - 2, + 2, + 4 of this wave
            const int j = p + 2, i0 = j + w - 2;
            double C[3][4];
#pragma unroll
            for (int x = 0; x < 3; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r) C[x][r] = next[x][r];
            // Panel p to the image, tile rows p + 1 + w - 2, + 2, ..., and its leaf's inverse; then the next
            // column's loads.  In front of the products, so that the next phase, which waits for all of
            // them when it takes up `next`, finds them done.
            {
                double im[4][4], xi[2];
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const int i = tb + w - 2 + 2 * x;
                    if (i < 8) {
#pragma unroll
                        for (int s = 0; s < 4; ++s) im[x][s] = S[256 * ((i * (i + 1)) / 2 + p) + l + 64 * s];
                    }
                }
#pragma unroll
                for (int s = 0; s < 2; ++s) xi[s] = xs[256 * (p & 1) + (tid & 127) + 128 * s];
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const int i = tb + w - 2 + 2 * x;
                    if (i < 8) {
#pragma unroll
                        for (int s = 0; s < 4; ++s) image_store(W + 256 * ((i * (i - 1)) / 2 + p) + l + 64 * s, im[x][s]);
                    }
                }
#pragma unroll
                for (int s = 0; s < 2; ++s) image_store(Xl + 256 * p + (tid & 127) + 128 * s, xi[s]);
            }
            fetch(j + 1);
            const int nt = (9 - i0) / 2;  // this wave's tiles of the column
            if (nt == 3)
                column_products<3>(S, i0, j, p, C);
            else if (nt == 2)
                column_products<2>(S, i0, j, p, C);
            else if (nt == 1)
                column_products<1>(S, i0, j, p, C);
        }
        lds_barrier();
    }
    image_store(Xl + 256 * 7 + tid, xs[256 + tid]);
    if (w == 0 && l < 16) {  // the last leaf
#pragma unroll
        for (int c = 0; c < 16; ++c) S[sl(112 + l, 112 + c)] = lv[c];
    }
    return __builtin_amdgcn_readfirstlane(*s_fail);
}

// Row tiles of 16 per wave in the panel solve: a row role is 64 kRowTiles rows.  With one, the solve
// on the chain from panel to panel (its 144 MFMAs per row tile) and the rows' update are half as long
// as with two, and there are twice as many roles, each staging the 72 KiB panel image.  Half as long
// wins at every size: with the image stored as the block is factored (potrf_in_lds) and the deeper
// operand prefetch of the diagonal update, the FP64 factor and solve took 1437 us against 1532 at
// n = 3001 and 6282 against 6369 at n = 8192, the FP32 one 2072 against 2315 at n = 4001.
constexpr int kRowTiles = 1;

// The panel solve works on a wave's 16 RT rows x 128 columns in the FP64 MFMA result layout:
// X[t][p][r] is row 16t + lane%16, column 16p + 4r + lane/16 (t < RT row tiles, p = 0..7
// column strips).  It needs, in LDS, the 28 strictly lower tiles of L (Ls: tile (ti, tj) at
// 256 * (ti(ti-1)/2 + tj)) and the
// 8 leaf inverses (Xs, 256 doubles each, column-major): the panel image of kernels.hpp.
//
// X <- X L^{-T} in place, strip by strip (TriangularSolverMatrix.h:186-329, blocked by 16):
//   X_q <- X_q X_qq^T, then X_p <- X_p - X_q L_pq^T for the strips p > q,   X_qq = L_qq^{-1}
// with the accumulator of a solved strip used directly as the operand of the next ones (its
// layout is that of an MFMA P operand with k = 4s + lane/16).  Strips Q0 .. Q1-1 here.
template <int Q0, int Q1, int RT>
__device__ __forceinline__ void trsm_in_registers(const double *smem, dvec4 (&X)[RT][8])
{
    const int l = lane_id();
    const double *Ls = smem;
    const double *Xs = smem + kLeafOffset;
#pragma unroll
    for (int q = Q0; q < Q1; ++q) {
        dvec4 z[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t) z[t] = dvec4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const double xv = Xs[256 * q + l + 64 * s];  // X_qq[l%16][4s + l/16]
#pragma unroll
            for (int t = 0; t < RT; ++t) z[t] = mfma_f64(xv, X[t][q][s], z[t]);
        }
#pragma unroll
        for (int t = 0; t < RT; ++t) X[t][q] = z[t];
#pragma unroll
        for (int p = q + 1; p < 8; ++p) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const double lv = Ls[256 * ((p * (p - 1)) / 2 + q) + l + 64 * s];  // L[16p + l%16][16q + 4s + l/16]
#pragma unroll
                for (int t = 0; t < RT; ++t) X[t][p] = mfma_f64(-lv, z[t][s], X[t][p]);
            }
        }
    }
}

// Block columns Q0 .. Q1-1 of a published panel image (16-byte aligned) -> LDS.  COHERENT: by loads that
// are served from memory, as they stand behind no acquire; else two tiles at a time, 16 bytes per load.
template <int Q0, int Q1, bool COHERENT>
__device__ __forceinline__ void stage_panel_image(double *smem, const double *__restrict__ W)
{
    constexpr int kTiles = 28 + 8;
    constexpr auto wanted = [](int t) constexpr -> bool {  // tile t of the image: (ti, tj), then the leaves
        if (t >= 28) return t - 28 >= Q0 && t - 28 < Q1;
        int ti = 1;
        while ((ti + 1) * ti / 2 <= t) ++ti;
        const int tj = t - ti * (ti - 1) / 2;
        return tj >= Q0 && tj < Q1;
    };
    if constexpr (COHERENT) {
        double v[kTiles];
#pragma unroll
        for (int t = 0; t < kTiles; ++t)
            if (wanted(t)) v[t] = coherent_load(W + 256 * t + threadIdx.x);
#pragma unroll
        for (int t = 0; t < kTiles; ++t)
            if (wanted(t)) smem[256 * t + threadIdx.x] = v[t];
        return;
    }
    const int half = threadIdx.x >> 7, e = 2 * (threadIdx.x & 127);
    int first = -1;  // of a pair
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        if (!wanted(t)) continue;
        if (first < 0) {
            first = t;
        } else {
            const int o = 256 * (half ? t : first) + e;
            *(double2 *)(smem + o) = *(const double2 *)(W + o);
            first = -1;
        }
    }
    if (first >= 0 && half == 0) *(double2 *)(smem + 256 * first + e) = *(const double2 *)(W + 256 * first + e);
}

// Waits (thread 0) until *flag has reached `want`.  Returns the flag's value less `base` (uniform), 0 on
// a timeout, recorded as MI_PANEL_TIMEOUT.
__device__ __forceinline__ int wait_panel_flag(int *s_seen, const uint32_t *flag, uint32_t base, int want, int *status)
{
    if (threadIdx.x == 0) {
        uint32_t spins = 0;
        int seen;
        while ((seen = (int)(__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - base)) < want) {
            __builtin_amdgcn_s_sleep(2);
            if (++spins > (1u << 22)) {
                atomicOr(status, MI_PANEL_TIMEOUT);
                seen = 0;
                break;
            }
        }
        *s_seen = seen;
    }
    __syncthreads();
    return *s_seen;
}

// The rows' solve, X as in trsm_in_registers: by the panels published early while the others are being
// factored, if the block is not done yet, then by those.  A block that is done is read after an acquire
// (each wave invalidates its own view of the caches), through the L2 that the rows share; its parts by
// coherent loads, since three acquires a role cost the tiles beside them their cached operands (a batch of
// 120 systems of order 512 took 3% longer).  Returns false if the factor failed or a wait timed out.
template <int RT>
__device__ __forceinline__ bool solve_rows(double *smem, int *s_seen, dvec4 (&X)[RT][8], const double *__restrict__ W,
                                           const uint32_t *flag, uint32_t epoch, const int *info, int *status)
{
    const uint32_t base = 8 * (epoch - 1);
    int seen = wait_panel_flag(s_seen, flag, base, 2, status);
    if (seen <= 0) return false;
    if (seen >= 8) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (factor_failed(info)) return false;
        stage_panel_image<0, 8, false>(smem, W);
        __syncthreads();
        trsm_in_registers<0, 8>(smem, X);
        return true;
    }
    stage_panel_image<0, kPart1, true>(smem, W);
    __syncthreads();
    trsm_in_registers<0, kPart1>(smem, X);
    if (wait_panel_flag(s_seen, flag, base, 4, status) <= 0) return false;
    stage_panel_image<kPart1, kPart2, true>(smem, W);
    __syncthreads();
    trsm_in_registers<kPart1, kPart2>(smem, X);
    if (wait_panel_flag(s_seen, flag, base, 8, status) <= 0 || factor_failed(info)) return false;
    stage_panel_image<kPart2, 8, true>(smem, W);
    __syncthreads();
    trsm_in_registers<kPart2, 8>(smem, X);
    return true;
}

// Rows 0..64 kRowTiles - 1 of P (valid m) <- P * L^{-T} by the panel image (solve_rows).  Each wave
// owns 16 kRowTiles rows.  T = float: P is read as FP32 and widened, the arithmetic is FP64, the result
// is rounded back to FP32.  If SPLIT (a split-panel slot) is given (T = float), the rounded rows are also
// written split into split_parts BF16 parts (2 or 3), row i as row split_row0 + i of the slot
// (split_store_row; part t at split + t * split_lo).
template <typename T>
__device__ __forceinline__ void trsm_rows(double *smem, int *s_seen, T *__restrict__ P, int64_t ldp, int m,
                                          const double *__restrict__ image, const uint32_t *flag, uint32_t epoch,
                                          const int *info, int *status, __bf16 *split, int64_t split_lo,
                                          int64_t split_row0, int split_parts)
{
    const int l = lane_id(), w = threadIdx.x >> 6;
    const int row0 = 16 * kRowTiles * w;
    dvec4 X[kRowTiles][8];
#pragma unroll
    for (int t = 0; t < kRowTiles; ++t) {
        const int i = row0 + 16 * t + (l & 15);
#pragma unroll
        for (int p = 0; p < 8; ++p)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = 16 * p + 4 * r + (l >> 4);
                const double pv = (double)P[(i < m ? i : m - 1) + (int64_t)j * ldp];
                X[t][p][r] = (i < m) ? pv : 0.0;
            }
    }
    if (!solve_rows(smem, s_seen, X, image, flag, epoch, info, status)) return;
#pragma unroll
    for (int t = 0; t < kRowTiles; ++t) {
        const int i = row0 + 16 * t + (l & 15);
        if (i < m) {
#pragma unroll
            for (int p = 0; p < 8; ++p)
#pragma unroll
                for (int r = 0; r < 4; ++r) P[i + (int64_t)(16 * p + 4 * r + (l >> 4)) * ldp] = (T)X[t][p][r];
            if constexpr (sizeof(T) == 4) {
                if (split) {
                    float v[8][4];
#pragma unroll
                    for (int p = 0; p < 8; ++p)
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[p][r] = (float)X[t][p][r];
                    if (split_parts == 3)
                        split_store_row<3>(split, split_lo, split_row0 + i, v);
                    else
                        split_store_row<2>(split, split_lo, split_row0 + i, v);
                }
            }
        }
    }
}

// FP64 update of tile columns [C0, C1) of the diagonal block, A_kk - P_0 P_0^T, for tile rows W and
// 7-W, their tiles at and left of the diagonal, with acc starting from A_kk: to S for C0 = 0, to the panel
// image (helper_tile, written through) for the others.  Identity beyond bs; a diagonal tile is written
// whole, its upper entries are never read as data.
template <int W, int C0, int C1>
__device__ __forceinline__ void diag_update_f64(double *S, const double *__restrict__ Akk,
                                                const double *__restrict__ P0, int64_t lda, int bs)
{
    constexpr uint32_t kCols = ((1u << C1) - 1u) & ~((1u << C0) - 1u);
    constexpr uint32_t kActive = (((1u << (W + 1)) - 1u) & kCols) | ((((1u << (8 - W)) - 1u) & kCols) << 8);
    // registers for eight k-steps in flight with four tiles at most, for five with nine
    WaveTile<2, 8, C1 - C0 == 8 ? 5 : 8, true, kActive> t;
    const int rows[2] = {16 * W, 16 * (7 - W)};
    t.zero();
    t.load_acc(Akk, lda, rows, 0, bs, bs);
    t.setup_rows(P0, lda, rows, bs, P0, lda, 0, bs, 128);
    t.template run_fixed<32>();
    const int l = lane_id();
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const int ti = a == 0 ? W : 7 - W;
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if (t.on(a, b)) {
                double *C = S + (C0 == 0 ? 256 * ((ti * (ti + 1)) / 2 + b) : helper_tile(ti, b)) + l;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * ti + (l & 15), j = 16 * b + 4 * r + (l >> 4);
                    const double v = (i < bs && j < bs) ? t.acc[a][b][r] : (i == j ? 1.0 : 0.0);
                    if (C0 == 0)
                        C[64 * r] = v;
                    else
                        image_store(C + 64 * r, v);
                }
            }
    }
}
template <int C0, int C1>
__device__ __forceinline__ void diag_update_columns(int w, double *S, const double *__restrict__ Akk,
                                                    const double *__restrict__ P0, int64_t lda, int bs)
{
    switch (w) {
    case 0: diag_update_f64<0, C0, C1>(S, Akk, P0, lda, bs); break;
    case 1: diag_update_f64<1, C0, C1>(S, Akk, P0, lda, bs); break;
    case 2: diag_update_f64<2, C0, C1>(S, Akk, P0, lda, bs); break;
    default: diag_update_f64<3, C0, C1>(S, Akk, P0, lda, bs); break;
    }
}

// The same for FP32 storage with low-precision MFMA (the mixed-precision factorization): 64 x
// 64 wave tiles over the three lower quadrants, the old values read after the MFMAs, in two
// halves of tile rows.
template <typename T, int PREC>
__device__ __forceinline__ void diag_update_lowp(double *S, const T *__restrict__ A, int64_t lda, int64_t k0, int bs)
{
    const int w = threadIdx.x >> 6, wr = w >> 1, wc = w & 1;
    if (wr == 0 && wc == 1) return;  // strictly upper quadrant
    const T *Ck = A + k0 + k0 * lda;
    using Tile = typename TileSel<T, PREC>::type;
    Tile t;
    t.zero();
    t.setup(A + k0 + (k0 - 128) * lda, lda, wr * 64, bs, A + k0 + (k0 - 128) * lda, lda, wc * 64, bs, 128);
    t.template run_fixed<128 / Tile::KS>();
#pragma unroll
    for (int a0 = 0; a0 < 4; a0 += 2) {
        T old[2][4][4];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    int i = wr * 64 + t.row_of(a0 + a), j = wc * 64 + t.col_of(b, r);
                    i = i < bs ? i : bs - 1;
                    j = j < bs ? j : bs - 1;
                    old[a][b][r] = Ck[i + (int64_t)j * lda];
                }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = wr * 64 + t.row_of(a0 + a), j = wc * 64 + t.col_of(b, r);
                    if (i >= j) {
                        const bool in = i < bs && j < bs;
                        S[sl(i, j)] = in ? (double)old[a][b][r] - (double)t.acc[a0 + a][b][r] : (i == j ? 1.0 : 0.0);
                    }
                }
    }
}

// Helper h of the diagonal role (FP64, k0 > 0): tile columns 2, 3 (h = 0) or 4 .. 7 of A_kk - P_0 P_0^T
// to the panel image (A_kk itself stays as it is until the block is factored, also when a pivot fails), then
// helped[h] = epoch.  The update's 36 tiles are 18400 cycles of MFMA on one CU, in front
// of everything else on the chain; the diagonal role computes the 15 tiles of columns 0 and 1 and needs
// column 2 a panel's time later, column 4 three panels' time.  A tile is contiguous in the image, so stores
// and loads need no bounds: a launch at n = 1024 takes 30 us, 33 with the tiles written to A.
__device__ __forceinline__ void diag_helper(int h, const double *__restrict__ A, int64_t lda, int64_t n, int64_t k0,
                                            double *__restrict__ Wleaf, uint32_t *helped, uint32_t epoch)
{
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int bs = (int)((n - k0) < 128 ? (n - k0) : 128);
    const double *Akk = A + k0 + k0 * lda;
    const double *P0 = A + k0 + (k0 - 128) * lda;
    double *Wp = Wleaf + (size_t)(k0 / 128) * kPanelDoubles;
    if (h == 0)
        diag_update_columns<2, 4>(w, Wp, Akk, P0, lda, bs);
    else
        diag_update_columns<4, 8>(w, Wp, Akk, P0, lda, bs);
    global_barrier();  // every wave's stores are in memory
    if (threadIdx.x == 0) __hip_atomic_store(helped + h, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The panel role of one block step; g is the role from the ticket, less the nh helpers' (diag_helper):
//   role 0   : C = A_kk - P_0 P_0^T straight into LDS (with helpers its tile columns 0 and 1, the others
//              as the helpers leave them), Cholesky in LDS, the panel image (L11's strictly lower tiles
//              and the leaf inverses) to the workspace, published by `flag` in three parts, then L11
//              into A;
//   role g>0 : the g-th 64 kRowTiles rows below the block: C = A_gk - P_g P_0^T, then rows <-
//              rows * L11^{-T} with the published image as it comes, stored once.
// The diagonal role publishes even on a failing pivot, so that no waiter is left behind;
// waiters then see `info` and stop.  (LLT.h:350-366: the update of block column k by all
// earlier panels precedes its unblocked factor and the right-side solve.)
// smem: kSmem doubles of LDS; s_ok: an LDS int.  T/PREC: storage and update arithmetic
// (the diagonal factor and the panel solve are FP64 for every T).  With T = double the row
// role keeps its rows in registers from the update to the store; with T = float the update
// is rounded to FP32 storage first (as the mixed-precision trailing updates are) and read back.
template <typename T, int PREC>
__device__ __forceinline__ void panel_role(int g, int nh, double *smem, int *s_ok, T *__restrict__ A,
                                           int64_t lda, int64_t n, int64_t k0, double *__restrict__ Wleaf, int *info,
                                           uint32_t *flag, const uint32_t *helped, uint32_t epoch, int *status,
                                           __bf16 *split = nullptr, int64_t split_lo = 0)
{
    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t R0 = g == 0 ? k0 : k0 + 128 + 64 * kRowTiles * (int64_t)(g - 1);
    const int rows = (int)((n - R0) < 64 * kRowTiles ? (n - R0) : 64 * kRowTiles);
    const int bs = (int)((n - k0) < 128 ? (n - k0) : 128);
    T *Ck = A + R0 + k0 * lda;  // this role's rows of block column k0
    double *Wp = Wleaf + (size_t)(k0 / 128) * kPanelDoubles;  // the panel image

    if (g == 0) {
        __shared__ double xs[2 * 256];  // potrf_in_lds
        if (k0 > 0) {
            if constexpr (sizeof(T) == 8) {
                if (nh)
                    diag_update_columns<0, 2>(w, smem, Ck, A + k0 + (k0 - 128) * lda, lda, bs);
                else
                    diag_update_columns<0, 8>(w, smem, Ck, A + k0 + (k0 - 128) * lda, lda, bs);
            } else {
                diag_update_lowp<T, PREC>(smem, A, lda, k0, bs);
            }
        } else {
            block_to_lds(smem, Ck, lda, bs);
        }
        const uint32_t *from_helpers = nullptr;
        if constexpr (sizeof(T) == 8) from_helpers = nh ? helped : nullptr;
        const int f = potrf_in_lds(smem, xs, s_ok, Wp, flag, from_helpers, epoch, status);  // a barrier first
        if (f >= 0 && tid == 0) atomicCAS(info, 0, (int)(k0 + f + 1));
        global_barrier();  // every wave's stores of the image are in memory
        if (tid == 0) __hip_atomic_store(flag, 8 * epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (f < 0) lds_to_block(smem, Ck, lda, bs);  // read by later launches only
        return;
    }

    if constexpr (sizeof(T) == 8) {
        WaveTile<kRowTiles, 8, 3, true, 0xffffffffu, true> t;  // P_0 has all 128 rows (k0 + 128 < n)
        int r2[kRowTiles];
#pragma unroll
        for (int a = 0; a < kRowTiles; ++a) r2[a] = 16 * (kRowTiles * w + a);
        t.zero();
        t.load_acc(Ck, lda, r2, 0, rows, 128);
        if (k0 > 0) {  // C -= P_g P_0^T, P = previous panel (columns k0-128..k0-1): rows R0.. and k0..
            t.setup_rows(A + R0 + (k0 - 128) * lda, lda, r2, rows, A + k0 + (k0 - 128) * lda, lda, 0, 128, 128);
            t.template run_fixed<32>();
        }
        if (!solve_rows(smem, s_ok, t.acc, Wp, flag, epoch, info, status)) return;
        const int l = lane_id();
#pragma unroll
        for (int a = 0; a < kRowTiles; ++a) {
            const int i = r2[a] + (l & 15);
            if (i < rows) {
#pragma unroll
                for (int b = 0; b < 8; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) Ck[i + (int64_t)(16 * b + 4 * r + (l >> 4)) * lda] = t.acc[a][b][r];
            }
        }
    } else {
        if (k0 > 0) {
            const int wr = w >> 1, wc = w & 1;
            constexpr int H = 32 * kRowTiles;  // rows of a wave tile
            using Tile = typename TileSel<T, PREC, H / 16>::type;
            Tile t;
            t.zero();
            t.setup(A + R0 + (k0 - 128) * lda, lda, wr * H, rows, A + k0 + (k0 - 128) * lda, lda, wc * 64, bs, 128);
            t.template run_fixed<128 / Tile::KS>();
            t.template store<false, false>(Ck, lda, wr * H, wc * 64, rows, 128);
        }
        global_barrier();  // this role's updated rows are in L2 before other waves read them back
        trsm_rows<T>(smem, s_ok, Ck, lda, rows, Wp, flag, epoch, info, status, split, split_lo, R0,
                     PREC == kPrecBF16x6 ? 3 : 2);
    }
}

}  // namespace mi
