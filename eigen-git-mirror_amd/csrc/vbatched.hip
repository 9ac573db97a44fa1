// vbatched.hip -- thousands of independent SPD factor + solve problems of uneven order
// (0..256) in one persistent launch.
//
// Reference counterpart: a loop of LLT<MatrixXd>(A_i).solve(B_i), i.e. llt_inplace::blocked /
// unblocked (Eigen/src/Cholesky/LLT.h:312-368; below 32 columns Eigen runs the unblocked
// column loop on the whole matrix, LLT.h:345) and LLT::_solve_impl (LLT.h:483-498) per system.
//
// A system is factored by a group of W waves, W = 1, 2 or 4 by its order (n <= 64, 128, 256), in
// block columns of 64, left-looking: a wave holds its rows' part of the block column -- up to 4
// tile rows of 16 (dealt round-robin over the group's waves) x 4 tile columns -- in registers:
//   accumulate: S_ic = sum_k L_ik L_ck^T over the finished columns (the wave's rows and the
//               block's own four tile rows are read back once per block column), MFMA
//   then for each of the 4 tile columns c, right-looking inside the block:
//   subtract: C_ic = A_ic - S_ic, once all earlier columns are in S: a sum has its own rounding, not A's
//             (in single precision the products of the block's own columns, added to A one by one, made
//             the whole call's error 7.7e-7 instead of 6.1e-7)
//   leaf:   L_cc = chol(C_cc), X_cc = L_cc^{-1} in one column loop (leaf_device.hpp), by the wave
//           that owns the row; X_cc to LDS.  The next column of A is read meanwhile
//   panel:  L_ic = C_ic X_cc^T for the wave's rows below, the block's own rows to LDS
//   update: S_ic' += L_ic L_c'c^T, c' > c.
// The MFMA result layout (element r of lane l: row l%16, column kx(r, l/16)) is the operand layout of
// k-step r of the next product, so C_ic feeds C_ic X_cc^T and L_ic the update from registers.
// What used to bound this path was re-reading the system, 14 times its size (one wave per system,
// left-looking by single tile columns: 26.6 GB a launch of 20,000 systems, 5.7 TB/s beyond L2):
// with 64-column blocks held by the group a factor of 256 reads its finished columns about twice,
// and a CU has 2 to 12 systems in flight instead of 8 of any size.  20,000 systems, n ~ U[8, 256]:
// FP64 4.6 -> 3.1 ms, FP32 3.0 -> 1.9 ms; 700 systems FP64 0.60 -> 0.19 ms.  What bounds it now is
// the chain of a system's steps (about 6k cycles per 16 columns with two workgroups on a CU: leaf,
// two barriers, panel, update; then 3.5k per step of each substitution), not memory: one workgroup
// per CU takes 4.8 ms.
// The substitutions run over the same blocks: the tiles of a block are dealt over the waves, each
// sums the finished part on its own, and the block's 4 steps pass through LDS.  A partial last tile
// is padded with the identity.
#include "common.hpp"
#include "kernels.hpp"
#include "leaf_device.hpp"

namespace mi {

constexpr int kVbMaxN = 256;
constexpr int kVbMaxT = kVbMaxN / 16;
constexpr int kVbPlan = 1024;  // systems per workgroup of the plan

// Global-memory views of a system's pointers.  A pointer rebuilt from readfirstlane'd integers
// is a generic one, and generic (flat) loads count in both the vector-memory and the LDS
// counters, which the compiler can only wait on as a whole.  Global loads are counted in order.
template <typename T>
using gptr = __attribute__((address_space(1))) T *;
template <typename T>
__device__ __forceinline__ gptr<T> to_global(T *p)
{
    return (gptr<T>)p;
}
template <typename T>
__device__ __forceinline__ T load_at(gptr<const T> base, uint32_t off)
{
    return *(gptr<const T>)((__attribute__((address_space(1))) const char *)base + off);
}
// Element at a byte offset from a wave-uniform base (scalar base + 32-bit vector offset form).
template <typename T>
__device__ __forceinline__ gptr<T> elem_at(gptr<T> base, uint32_t off)
{
    return (gptr<T>)((__attribute__((address_space(1))) char *)base + off);
}

// The lane layout of a 16 x 16 tile: element r of lane (l%16, g = l/16) is column kx(r, g), the k
// index of operand k-step r (FP32 permutes k: any common order gives the same products).
// LS: padded column of a leaf (16-byte aligned).
template <typename T>
struct VbArith;
template <>
struct VbArith<double> {  // v_mfma_f64_16x16x4f64
    using acc_t = dvec4;
    static constexpr int LS = 18;
    __device__ static acc_t mma(double q, double p, acc_t c) { return mfma_f64(q, p, c); }
    __device__ static int kx(int s, int g) { return 4 * s + g; }
    __device__ static constexpr int step(int s) { return 4 * s; }  // kx(s, g) - kx(0, g)
};
template <>
struct VbArith<float> {  // v_mfma_f32_16x16x4f32
    using acc_t = fvec4;
    static constexpr int LS = 20;
    __device__ static acc_t mma(float q, float p, acc_t c) { return mfma_f32(q, p, c); }
    __device__ static int kx(int s, int g) { return 4 * g + s; }
    __device__ static constexpr int step(int s) { return s; }
};

// Workgroups per CU: FP64 holds 4 x 4 tiles in 128 registers a lane and two workgroups; FP32 fits
// three, which measured 1.96 ms against 2.40 with two (20,000 systems).  FP64 blocks of two tile
// columns with three workgroups took 6% longer (3.7 ms, 3.5 then).  The compiler spills 21 (FP64) and
// 40 (FP32) registers and 82 to 84 scalars, mostly at a system's start and end, none in the leaf.
template <typename T>
constexpr int kVbPerCu = sizeof(T) == 8 ? 2 : 3;

// One system, in the order of the queue.
struct VbDesc {
    uint64_t a, b;
    int n, lda, nrhs, ldb;
    int index, pad[3];
};
// Queue of mode c (0: groups of four waves, 1: of two, 2: single waves): systems [begin[c], end[c]),
// dealt round-robin over eight counters on lines of their own -- workgroups take from their XCD's
// counter first.  Every draw is an atomic at the memory side: at one counter they queued up for
// about 17 ns each, which alone took 140 us for 8,000 systems of order 16.
struct VbQueue {
    int begin[4], end[4];
    int pad[24];
    int next[3][8][32];  // counter x of mode c: next[c][x][0]
};

// Largest order in tiles of a group of W waves.
constexpr int vb_tm(int W) { return 4 * W; }

// LDS of a group, per tile of its largest order: X_kk by columns (before: the leaf's rows), and the
// block's own panel tiles, then Y_k^T, then X_k^T (lane order).
template <typename T>
constexpr int vb_lds_tile = 16 * VbArith<T>::LS + 256;

// Progress of a group of two waves; counts on over the systems, never reset.
struct VbSync {
    uint32_t bar[2];
    int fail, ticket[2], pad[3];
};

// Orders the LDS accesses of this wave's lanes (a wave's LDS operations execute in order).
__device__ __forceinline__ void lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A group of W waves (1, 2 or 4; a run-time scalar: one copy of the code serves all modes, and the
// kernel must stay small -- unrolled per mode and column it took 200 KB, three times the instruction
// cache, and ran at half the speed).
template <typename T>
struct VbGroup {
    using M = VbArith<T>;
    using acc_t = typename M::acc_t;
    static constexpr int LS = M::LS;

    T *X, *Y;  // LDS: X_kk at X + 16 LS k, tiles at Y + 256 k
    VbSync *sy;
    int W, w;  // waves of the group, this wave
    uint32_t bars;
    int parity;

    // Barrier of the group for its LDS data (global stores may stay in flight).  Two waves of a
    // workgroup meet through two words of LDS: each counts its barriers there and waits for the
    // other's count, which the other -- resident, being of the same workgroup -- reaches without
    // waiting for anything but earlier barriers, so the wait ends.
    __device__ __forceinline__ void barrier()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        if (W == 4) {
            __builtin_amdgcn_s_barrier();
        } else if (W == 2) {
            ++bars;
            __hip_atomic_store(&sy->bar[w], bars, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            while ((int)(__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(&sy->bar[w ^ 1], __ATOMIC_RELAXED,
                                                                               __HIP_MEMORY_SCOPE_WORKGROUP)) -
                         (int)bars) < 0)
                __builtin_amdgcn_s_sleep(0);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
    // The same after which the waves' global stores can be read by all of them.
    __device__ __forceinline__ void barrier_global()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }

    // Runs a mode's queue.  Every value that steers the loop is wave-uniform.
    __device__ __forceinline__ void run(const VbDesc *__restrict__ desc, VbQueue *queue, int mode, int *__restrict__ d_info)
    {
        const int l = lane_id();
        auto sc = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
        const int begin = sc(queue->begin[mode]), end = sc(queue->end[mode]);
        int *next = &queue->next[mode][0][0];
        int x = (int)(blockIdx.x & 7);  // the counter drawn from
        const bool draws = w == 0;
        // a ticket of counter x (valid in lane 0), and the system it stands for: when it is past the
        // end, another counter's, as long as one has systems left (counters only grow: it ends)
        auto draw = [&]() -> int { return atomicAdd(next + 32 * x, l == 0 ? 1 : 0); };
        auto settle = [&](int ticket) -> int {
            for (;;) {
                const int i = begin + x + 8 * sc(ticket);
                if (i < end) return i;
                const int v = __hip_atomic_load(next + 32 * (l & 7), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const uint32_t left = (uint32_t)__ballot(begin + (l & 7) + 8 * v < end) & 0xffu;
                if (!left) return end;
                const uint32_t turned = ((left >> x) | (left << (8 - x))) & 0xffu;  // from x on
                x = (x + __builtin_ctz(turned)) & 7;
                ticket = draw();
            }
        };
        // first pass: no system yet, only the ticket; then each pass takes one system: the loop ends
        int t = begin - 1;
        VbDesc d = desc[0];
        for (;;) {
            auto sc64 = [&](uint64_t v) {
                return ((uint64_t)(uint32_t)sc((int)(v >> 32)) << 32) | (uint32_t)sc((int)(uint32_t)v);
            };
            const bool have = t >= begin;
            const int n = have ? sc(d.n) : 0, lda = sc(d.lda), nrhs = sc(d.nrhs), ldb = sc(d.ldb), idx = sc(d.index);
            const gptr<T> A = to_global((T *)(uintptr_t)sc64(d.a)), B = to_global((T *)(uintptr_t)sc64(d.b));
            // the next ticket is drawn now, its descriptor read before the substitutions
            int tn = 0;
            if (draws) tn = draw();
            const int info = factor(n, A, lda);
            if (draws) sy->ticket[parity] = settle(tn);
            barrier_global();  // L to every wave
            tn = sc(sy->ticket[parity]);
            d = desc[tn < end ? tn : 0];
            if (info == 0 && n > 0)
                for (int c0 = 0; c0 < nrhs; c0 += 16) solve(n, A, lda, nrhs, B, ldb, c0);
            if (draws && have) d_info[idx] = info;
            barrier();  // every wave is done with this system's LDS
            if (tn >= end) return;
            parity ^= 1;
            t = tn;
        }
    }

    // C[r][c] = sum_k L[row_r, k] L[4J + c, k]^T over the k tiles [0, 4J), r < NR.
    template <int NR>
    __device__ __forceinline__ void accumulate(acc_t (&C)[4][4], gptr<const T> A, int64_t lda, int J,
                                               const uint32_t (&offp)[4], const uint32_t (&offq)[4])
    {
        constexpr int U = 4;  // k-steps in flight (16 J of them)
        T p[U][NR], q[U][4];
        const int steps = 16 * J;
        auto load = [&](int u, int s) {
            s = s < steps ? s : steps - 1;
            const gptr<const T> base = A + (int64_t)(16 * (s >> 2) + M::step(1) * (s & 3)) * lda;
#pragma unroll
            for (int r = 0; r < NR; ++r) p[u][r] = load_at<T>(base, offp[r]);
#pragma unroll
            for (int c = 0; c < 4; ++c) q[u][c] = load_at<T>(base, offq[c]);
        };
#pragma unroll
        for (int u = 0; u < U - 1; ++u) load(u, u);
        for (int s0 = 0; s0 < steps; s0 += U) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                load((u + U - 1) % U, s0 + u + U - 1);
#pragma unroll
                for (int r = 0; r < NR; ++r)
#pragma unroll
                    for (int c = 0; c < 4; ++c) C[r][c] = M::mma(q[u][c], p[u][r], C[r][c]);
                __builtin_amdgcn_sched_barrier(0);  // keeps the wait counts exact
            }
        }
    }

    // LAPACK info (uniform over the group).
    __device__ __forceinline__ int factor(const int n, const gptr<T> A, const int64_t lda)
    {
        const int l = lane_id(), li = l & 15, g = l >> 4;
        const int nt = (n + 15) >> 4;
        const T zero = (T)0, one = (T)1;
        const int kx0 = M::kx(0, g);
        auto lane_off = [&](int r) -> uint32_t { return (uint32_t)((r + (int64_t)kx0 * lda) * (int64_t)sizeof(T)); };
        for (int J = 0; 4 * J < nt; ++J) {
            const int nb = nt - 4 * J < 4 ? nt - 4 * J : 4;  // tile columns of the block
            // slot r: tile row 4J + q, q = r W + w; ns slots in use
            const int left = nt - 4 * J - w, ns = left <= 0 ? 0 : left <= W ? 1 : left <= 2 * W ? 2 : left <= 3 * W ? 3 : 4;
            acc_t C[4][4];
            uint32_t offp[4], offq[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 16 * (4 * J + r * W + w) + li, j = 16 * (4 * J + r) + li;
                offp[r] = lane_off(i < n ? i : n - 1);
                offq[r] = lane_off(j < n ? j : n - 1);
#pragma unroll
                for (int c = 0; c < 4; ++c) C[r][c] = acc_t{zero, zero, zero, zero};
            }
            if (J > 0) {
                if (ns > 2)
                    accumulate<4>(C, A, lda, J, offp, offq);
                else if (ns == 2)
                    accumulate<2>(C, A, lda, J, offp, offq);
                else if (ns == 1)
                    accumulate<1>(C, A, lda, J, offp, offq);
            }
            // A's tile column c of the block, this wave's tiles at and left of the diagonal (the strictly
            // upper part of a diagonal tile is read but never used: every lane stops at its own diagonal
            // entry).  Rows past n, rows above the diagonal and empty slots: a row that is read anyway.
            // The loads are issued in front of the barrier that ends the leaf: behind it, a launch of 20,000
            // took 0.15 ms longer in FP64; in front of the leaf, its registers spilled (6.8 ms a call against 4.8).
            auto read_column = [&](T(&a)[4][4], int c) {
                const int col = 16 * (4 * J + c);
                if (col + 16 <= n) {
                    uint32_t off[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        off[r] = r < ns && r * W + w >= c ? offp[r] : offp[0];
                        asm volatile("" : "+v"(off[r]));  // or each load gets branches of its own
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const gptr<T> base = A + (int64_t)(col + M::step(e)) * lda;
#pragma unroll
                        for (int r = 0; r < 4; ++r) a[r][e] = *elem_at(base, off[r]);
                    }
                } else {  // the last, partial tile column (its diagonal tile alone): columns past n - 1 read n - 1's
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int i = col + li, cc = col + M::kx(e, g);
                        const T x = A[(i < n ? i : n - 1) + (int64_t)(cc < n ? cc : n - 1) * lda];
#pragma unroll
                        for (int r = 0; r < 4; ++r) a[r][e] = x;
                    }
                }
            };
            // a <- A's column less S, the sum of all earlier columns' products, which is formed by itself: it
            // keeps its own rounding, not A's.  Rows past n: zero, the identity on the diagonal.
            auto subtract = [&](T(&a)[4][4], int c, int h) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int q = r * W + w;
#pragma unroll
                    for (int e = 0; e < 4; ++e) a[r][e] -= C[r][h][e];
                    if (r < ns && 16 * (4 * J + q) + 16 > n) {
                        const int i = 16 * (4 * J + q) + li;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int col = 16 * (4 * J + c) + M::kx(e, g);
                            a[r][e] = i < n && col < n ? a[r][e] : (i == col ? one : zero);
                        }
                    }
                }
            };
            // this wave's diagonal tile of the block column at hand: to LDS for the leaf
            auto give_leaf = [&](const T(&a)[4][4], int c) {
                T *xs = X + 16 * LS * (4 * J + c);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r * W + w == c) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) xs[LS * li + M::kx(e, g)] = a[r][e];
                    }
            };
            {
                T a[4][4];
                read_column(a, 0);
                subtract(a, 0, 0);
                give_leaf(a, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int e = 0; e < 4; ++e) C[r][0][e] = a[r][e];
            }
            // the column at hand is always C[.][0]; the others, sums so far, move up after each
#pragma unroll 1
            for (int c = 0; c < nb; ++c) {
                const int k = 4 * J + c, k0 = 16 * k;
                T *xs = X + 16 * LS * k;
                // ---- leaf
                T u[16];
                if (w == (c & (W - 1))) {
                    lds_order();
                    // (opaque: the identity's rows, hoisted out of the loops, would fill the registers)
                    int own = li;
                    asm volatile("" : "+v"(own));
                    T v[16];
#pragma unroll
                    for (int m = 0; m < 16; ++m) u[m] = xs[LS * li + m];
#pragma unroll
                    for (int m = 0; m < 16; ++m) v[m] = m == own ? one : zero;
                    const int f = leaf_factor(u, v);
                    __builtin_amdgcn_s_setprio(0);
                    lds_order();
                    sy->fail = f >= 0 ? k0 + f + 1 : 0;
                    if (l < 16) {
#pragma unroll
                        for (int m = 0; m < 16; ++m) xs[LS * li + m] = v[m];
                    }
                }
                T a[4][4] = {};  // the next column
                if (c + 1 < nb) read_column(a, c + 1);  // in flight during the other waves' leaf and the panel
                barrier();
                {
                    const int f = __builtin_amdgcn_readfirstlane(sy->fail);
                    if (f != 0) return f;
                }
                if (w == (c & (W - 1)) && l < 16 && k0 + l < n) {  // L_kk
                    gptr<T> p = A + (k0 + l) + (int64_t)k0 * lda;
#pragma unroll
                    for (int m = 0; m < 16; ++m, p += lda)
                        if (m <= l) *p = u[m];
                }
                // ---- panel
                T xq[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) xq[e] = xs[LS * M::kx(e, g) + li];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int q = r * W + w;
                    if (r < ns && q > c) {
                        acc_t o = {zero, zero, zero, zero};
#pragma unroll
                        for (int e = 0; e < 4; ++e) o = M::mma(xq[e], C[r][0][e], o);
                        C[r][0] = o;
                        if (q < 4) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) Y[256 * q + 64 * e + l] = o[e];
                        }
                        const int i = 16 * (4 * J + q) + li;
                        if (i < n) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) *elem_at(A + (int64_t)(k0 + M::step(e)) * lda, offp[r]) = o[e];
                        }
                    }
                }
                if (c + 1 == nb) break;
                barrier();
                // ---- update, and the columns move up
#pragma unroll
                for (int h = 1; h < 4; ++h) {  // tile column c + h
                    T pq[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) pq[e] = Y[256 * ((c + h) & 3) + 64 * e + l];
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (r < ns && c + h < nb && r * W + w >= c + h) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) C[r][h] = M::mma(pq[e], C[r][0][e], C[r][h]);
                        }
                    if (h == 1) {
                        subtract(a, c + 1, 1);
                        give_leaf(a, c + 1);
                        // The next leaf is the system's chain: until it is done, its wave goes ahead of the
                        // other workgroup's on its SIMD.  It pays where the largest systems share a CU with
                        // one other (FP64, 520 systems 203 -> 184 us, 700 202 -> 191, 850 209 -> 198; 1000
                        // 274 -> 286); 300 and 20,000 take as long without.
                        if (w == ((c + 1) & (W - 1))) __builtin_amdgcn_s_setprio(2);
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) C[r][0][e] = a[r][e];
                    C[r][1] = C[r][2];
                    C[r][2] = C[r][3];
                }
            }
            barrier_global();  // the next block reads this one's columns (and the panel tiles are free)
        }
        return 0;
    }

    // z[h] += sum over the tiles j of [j0, j1) of Y_j^T times the operand tile load(q, j) of this
    // wave's tiles h < NC, four operand tiles at a time.
    template <int NC, class Load>
    __device__ __forceinline__ void sum(acc_t (&z)[4], int j0, int j1, Load &&load)
    {
        constexpr int U = 4 / NC;
        const int l = lane_id();
        T q[U][NC][4];
        if (j0 >= j1) return;
#pragma unroll
        for (int u = 0; u < U - 1; ++u) load(q[u], j0 + u < j1 ? j0 + u : j1 - 1);
        for (int j = j0; j < j1; j += U) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                load(q[(u + U - 1) % U], j + u + U - 1 < j1 ? j + u + U - 1 : j1 - 1);
                const bool in = j + u < j1;  // past the end: times zero
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const T y = Y[256 * (in ? j + u : j0) + 64 * e + l], p = in ? y : (T)0;
#pragma unroll
                    for (int h = 0; h < NC; ++h) z[h] = M::mma(q[u][h][e], p, z[h]);
                }
            }
        }
    }

    // B[:, c0..c0+15] <- A^{-1} B with the factor in A and the X_kk in LDS, as transposed tiles (rows:
    // right-hand sides); a block's tile column c belongs to wave c % W as its tile h = c / W.
    __device__ __forceinline__ void solve(const int n, const gptr<T> A, const int64_t lda, const int nrhs,
                                          const gptr<T> B, const int64_t ldb, const int c0)
    {
        const int nbk = (((n + 15) >> 4) + 3) >> 2;
#pragma unroll 1
        for (int J = 0; J < nbk; ++J) solve_block<false>(n, A, lda, nrhs, B, ldb, c0, J);
#pragma unroll 1
        for (int J = nbk - 1; J >= 0; --J) solve_block<true>(n, A, lda, nrhs, B, ldb, c0, J);
        barrier();  // the next right-hand sides overwrite Y
    }

    // Forward:  Y_c^T = (B_c^T - sum_{j<c} Y_j^T L_cj^T) X_cc^T.
    // Backward: X_c^T = (Y_c^T - sum_{i>c} X_i^T L_ic) X_cc.
    template <bool BACK>
    __device__ __forceinline__ void solve_block(const int n, const gptr<T> A, const int64_t lda, const int nrhs,
                                                const gptr<T> B, const int64_t ldb, const int c0, const int J)
    {
        const int l = lane_id(), li = l & 15, g = l >> 4;
        const int nt = (n + 15) >> 4, nb = nt - 4 * J < 4 ? nt - 4 * J : 4;
        const T zero = (T)0;
        const int col = c0 + li;
        const bool cin = col < nrhs;
        const int64_t bcol = (int64_t)(cin ? col : c0) * ldb;
        auto clamp = [&](int i) { return i < n ? i : n - 1; };
        // operand of tile j for this wave's tile h (column 4J + c, c = h W + w): L_cj[li][k] (forward),
        // L_jc[k][li].  Only a backward j can be a partial tile (its rows past n read row n - 1).
        uint32_t off[4];
        const bool near = lda <= (1 << 20);  // 256 columns within 32-bit offsets
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const int64_t own = clamp(16 * (4 * J + h * W + w) + li), k = M::kx(0, g);
            off[h] = (uint32_t)((BACK ? k + own * lda : own + k * lda) * (int64_t)sizeof(T));
        }
        auto operand = [&](T(&q)[4], int h, int j) {
            if (near && (!BACK || 16 * j + 16 <= n)) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    q[e] = load_at<T>(A + (BACK ? (int64_t)(16 * j + M::step(e)) : (int64_t)(16 * j + M::step(e)) * lda), off[h]);
            } else {
                const int own = clamp(16 * (4 * J + h * W + w) + li);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = clamp(16 * j + M::kx(e, g));
                    q[e] = A[BACK ? k + (int64_t)own * lda : own + (int64_t)k * lda];
                }
            }
        };
        acc_t z[4];  // the sums, by themselves (see factor)
        T bv[4][4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            z[h] = acc_t{zero, zero, zero, zero};
            const int k = 4 * J + h * W + w;
            if (h * W + w < nb) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = 16 * k + M::kx(e, g);
                    if (BACK) {
                        bv[h][e] = Y[256 * k + 64 * e + l];
                    } else {
                        const T v = B[clamp(i) + bcol];
                        bv[h][e] = i < n && cin ? v : zero;
                    }
                }
            }
        }
        const int j0 = BACK ? 4 * J + 4 : 0, j1 = BACK ? nt : 4 * J;
        if (W == 4)
            sum<1>(z, j0, j1, [&](T(&q)[1][4], int j) { operand(q[0], 0, j); });
        else if (W == 2)
            sum<2>(z, j0, j1, [&](T(&q)[2][4], int j) {
                operand(q[0], 0, j);
                operand(q[1], 1, j);
            });
        // (a single wave's systems are one block: nothing to sum)
        T in[4][4];  // the operand tiles for the block's column at hand, read one column ahead
        auto needs = [&](int h, int c) -> bool { return h * W + w < nb && (BACK ? h * W + w < c : h * W + w > c); };
        auto ahead = [&](int c) {
#pragma unroll
            for (int h = 0; h < 4; ++h)
                if (needs(h, c)) operand(in[h], h, 4 * J + c);
        };
        ahead(BACK ? nb - 1 : 0);
#pragma unroll 1
        for (int s = 0; s < nb; ++s) {
            const int c = BACK ? nb - 1 - s : s, k = 4 * J + c;
            if (w == (c & (W - 1))) {
                acc_t o = {zero, zero, zero, zero}, zi = o;
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    if (h * W + w == c) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) zi[e] = bv[h][e] - z[h][e];
                    }
                const T *xs = X + 16 * LS * k;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // rows past n (forward): their sums come from copies of L's row n - 1
                    const T zz = BACK || 16 * k + M::kx(e, g) < n ? zi[e] : zero;
                    o = M::mma(xs[BACK ? LS * li + M::kx(e, g) : LS * M::kx(e, g) + li], zz, o);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = 16 * k + M::kx(e, g);
                    Y[256 * k + 64 * e + l] = !BACK || i < n ? o[e] : zero;
                    if (BACK && i < n && cin) B[i + bcol] = o[e];
                }
            }
            barrier();
            if (s + 1 < nb) {
                T y[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = Y[256 * k + 64 * e + l];
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    if (needs(h, c)) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) z[h] = M::mma(in[h][e], y[e], z[h]);
                    }
                ahead(BACK ? c - 1 : c + 1);
            }
        }
    }
};

template <typename T>
__global__ __launch_bounds__(256, kVbPerCu<T>) void vb_persistent_kernel(const VbDesc *__restrict__ desc, VbQueue *queue,
                                                               int *__restrict__ d_info)
{
    // one group of four waves, then two of two, then four single waves; a group's LDS grows with its
    // largest order, so wave w's part starts at its first wave's four tiles in every mode
    static_assert(16 * vb_lds_tile<T> * sizeof(T) + 7 * sizeof(VbSync) <= 160 * 1024 / kVbPerCu<T>, "workgroups per CU");
    __shared__ __align__(16) T lds[16 * vb_lds_tile<T>];
    __shared__ VbSync sync[7];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int i = threadIdx.x; i < (int)(sizeof(sync) / 4); i += 256) ((uint32_t *)sync)[i] = 0u;
    __syncthreads();
#pragma unroll 1
    for (int mode = 0; mode < 3; ++mode) {
        VbGroup<T> q;
        q.W = 4 >> mode;
        q.w = w & (q.W - 1);
        q.sy = &sync[mode == 0 ? 0 : mode == 1 ? 1 + (w >> 1) : 3 + w];
        const int first = w - q.w;  // the group's first wave
        q.X = lds + 4 * first * vb_lds_tile<T>;
        q.Y = q.X + 4 * q.W * 16 * VbArith<T>::LS;
        q.bars = 0;
        q.parity = 0;
        q.run(desc, queue, mode, d_info);
    }
}

// Plan: every system's arguments checked (its info set), the valid ones sorted into the queues,
// longest first within a queue (lpt: the tail of the launch stays short) or in the given order; systems of
// one bucket keep the given order in both.
// Two launches of one workgroup per kVbPlan systems: each counts its systems per bucket (tile
// count, longest first; lpt = 0: per mode), then each places its own behind the earlier workgroups'.
constexpr int kVbBuckets = kVbMaxT + 1;
__device__ __forceinline__ int vb_check(int n, int lda, int nr, int ldb)
{
    if (n < 0 || n > kVbMaxN) return -1;
    if (lda < (n > 1 ? n : 1)) return -2;
    if (nr < 0) return -3;
    if (nr > 0 && ldb < (n > 1 ? n : 1)) return -4;
    return 0;
}
// Mode of a system of nt tiles: 0: four waves, 1: two, 2: one.
__host__ __device__ constexpr int vb_mode(int nt) { return nt <= vb_tm(1) ? 2 : nt <= vb_tm(2) ? 1 : 0; }
__device__ __forceinline__ int vb_bucket(int n, int lpt)
{
    const int nt = (n + 15) / 16;
    return kVbMaxT - (lpt ? nt : vb_tm(4 >> vb_mode(nt)));  // not lpt: the bucket of the mode's largest order
}

__global__ __launch_bounds__(kVbPlan) void vb_count_kernel(int64_t batch, const int *__restrict__ d_n,
                                                           const int *__restrict__ d_lda, const int *__restrict__ d_nrhs,
                                                           const int *__restrict__ d_ldb, int *__restrict__ d_info,
                                                           int *__restrict__ hist, int lpt)
{
    __shared__ int cnt[kVbBuckets];
    const int tid = threadIdx.x;
    if (tid < kVbBuckets) cnt[tid] = 0;
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * kVbPlan + tid;
    if (i < batch) {
        const int n = d_n[i];
        const int bad = vb_check(n, d_lda[i], d_nrhs[i], d_ldb[i]);
        d_info[i] = bad;
        if (!bad) atomicAdd(&cnt[vb_bucket(n, lpt)], 1);
    }
    __syncthreads();
    if (tid < kVbBuckets) hist[(int64_t)blockIdx.x * kVbBuckets + tid] = cnt[tid];
}

template <typename T>
__global__ __launch_bounds__(kVbPlan) void vb_place_kernel(int64_t batch, const int *__restrict__ d_n,
                                                           T *const *__restrict__ d_A, const int *__restrict__ d_lda,
                                                           const int *__restrict__ d_nrhs, T *const *__restrict__ d_B,
                                                           const int *__restrict__ d_ldb, const int *__restrict__ hist,
                                                           VbDesc *__restrict__ desc, VbQueue *__restrict__ queue,
                                                           int lpt)
{
    __shared__ int total[kVbBuckets], before[kVbBuckets], start[kVbBuckets + 1], waves[kVbPlan / 64][kVbBuckets];
    const int tid = threadIdx.x;
    if (tid < kVbBuckets) total[tid] = before[tid] = 0;
    __syncthreads();
    for (int e = tid; e < (int)gridDim.x * kVbBuckets; e += kVbPlan) {
        const int wg = e / kVbBuckets, b = e % kVbBuckets, v = hist[e];
        if (v) {
            atomicAdd(&total[b], v);
            if (wg < (int)blockIdx.x) atomicAdd(&before[b], v);
        }
    }
    __syncthreads();
    if (tid == 0) {
        int s = 0;
        for (int b = 0; b < kVbBuckets; ++b) {
            start[b] = s;
            s += total[b];
        }
        start[kVbBuckets] = s;
    }
    __syncthreads();
    if (blockIdx.x == 0) {
        if (tid < 3) {  // buckets from the mode's largest order on
            queue->begin[tid] = start[kVbMaxT - vb_tm(4 >> tid)];
            queue->end[tid] = start[tid < 2 ? kVbMaxT - vb_tm(2 >> tid) : kVbBuckets];
        }
        if (tid < 3 * 8) queue->next[tid / 8][tid % 8][0] = 0;
    }
    if (tid < kVbBuckets) before[tid] += start[tid];
    const int64_t i = (int64_t)blockIdx.x * kVbPlan + tid;
    VbDesc d;
    int bucket = -1;  // none: past the end, or arguments out of range
    if (i < batch) {
        d.n = d_n[i];
        d.lda = d_lda[i];
        d.nrhs = d_nrhs[i];
        d.ldb = d_ldb[i];
        d.a = (uint64_t)(uintptr_t)d_A[i];
        d.b = (uint64_t)(uintptr_t)d_B[i];
        d.index = (int)i;
        d.pad[0] = d.pad[1] = d.pad[2] = 0;
        if (!vb_check(d.n, d.lda, d.nrhs, d.ldb)) bucket = vb_bucket(d.n, lpt);
    }
    // the systems of the bucket in front of this one: in its wave, then in the earlier waves
    const int l = lane_id(), w = tid >> 6;
    int rank = 0;
#pragma unroll
    for (int b = 0; b < kVbBuckets; ++b) {
        const uint64_t same = __ballot(bucket == b);
        if (bucket == b) rank = __popcll(same & ((1ull << l) - 1));
        if (l == b) waves[w][b] = __popcll(same);
    }
    __syncthreads();
    if (bucket < 0) return;
    for (int v = 0; v < w; ++v) rank += waves[v][bucket];
    desc[before[bucket] + rank] = d;
}

constexpr int64_t kVbQueueBytes = ((int64_t)sizeof(VbQueue) + 255) / 256 * 256;
// Bytes of the plan: the queues, the workgroups' counts and the systems in queue order.
int64_t vb_plan_bytes(int64_t batch)
{
    const int64_t wgs = (batch + kVbPlan - 1) / kVbPlan;
    return kVbQueueBytes + (wgs * kVbBuckets * 4 + 255) / 256 * 256 + batch * (int64_t)sizeof(VbDesc);
}

template <typename T>
void launch_vbatched(int64_t batch, const int *d_n, T *const *d_A, const int *d_lda, const int *d_nrhs,
                     T *const *d_B, const int *d_ldb, int *d_info, void *plan, int grid, int lpt, hipStream_t s)
{
    const unsigned wgs = (unsigned)((batch + kVbPlan - 1) / kVbPlan);
    VbQueue *queue = (VbQueue *)plan;
    int *hist = (int *)((char *)plan + kVbQueueBytes);
    VbDesc *desc = (VbDesc *)((char *)plan + kVbQueueBytes + ((int64_t)wgs * kVbBuckets * 4 + 255) / 256 * 256);
    hipLaunchKernelGGL(vb_count_kernel, dim3(wgs), dim3(kVbPlan), 0, s, batch, d_n, d_lda, d_nrhs, d_ldb, d_info,
                       hist, lpt);
    hipLaunchKernelGGL(vb_place_kernel<T>, dim3(wgs), dim3(kVbPlan), 0, s, batch, d_n, d_A, d_lda, d_nrhs, d_B, d_ldb,
                       hist, desc, queue, lpt);
    hipLaunchKernelGGL(vb_persistent_kernel<T>, dim3(grid), dim3(256), 0, s, desc, queue, d_info);
}

template void launch_vbatched<double>(int64_t, const int *, double *const *, const int *, const int *,
                                      double *const *, const int *, int *, void *, int, int, hipStream_t);
template void launch_vbatched<float>(int64_t, const int *, float *const *, const int *, const int *, float *const *,
                                     const int *, int *, void *, int, int, hipStream_t);

}  // namespace mi
