// leaf_device.hpp -- Cholesky of a 16 x 16 leaf and its inverse inside one wave, on the DPP row
// broadcast (no scalar registers, no LDS in the column loop).
//
// Every row of 16 lanes holds the whole leaf: lane l has row l % 16 in u[0..15].  A column step of
// LLT.h:320-334 (pivot test, sqrt, scale, rank-1 update) needs element c of column j on every lane
// of the row: one v_fmac_f64 with a row_newbcast operand per updated element, where a readlane
// broadcast took two v_readlane and the FMA and its scalar-register hazards.  The serial chain of a
// step is the pivot's broadcast, the reciprocal square root and one update.
#pragma once
#include "common.hpp"

namespace mi {

// x -= m(lane C of this row of 16) * y, fused.  DPP reads a register of the previous two
// instructions too early: `first` puts the wait states in front, for the statement right after m's
// last write (the statements are volatile, so the later ones stay behind it).
template <int C, bool FIRST = false>
__device__ __forceinline__ void row_fnma(double &x, double m, double y)
{
    if constexpr (FIRST)
        asm volatile("s_nop 1\n\tv_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                     : "+v"(x) : "v"(m), "v"(y), "n"(C));
    else
        asm volatile("v_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                     : "+v"(x) : "v"(m), "v"(y), "n"(C));
}
template <int C, bool FIRST = false>
__device__ __forceinline__ void row_fnma(float &x, float m, float y)
{
    if constexpr (FIRST)
        asm volatile("s_nop 1\n\tv_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                     : "+v"(x) : "v"(m), "v"(y), "n"(C));
    else
        asm volatile("v_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                     : "+v"(x) : "v"(m), "v"(y), "n"(C));
}
// Lane C's value in every lane of its row of 16.
template <int C>
__device__ __forceinline__ double row_bcast(double m)
{
    double x;
    asm volatile("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(x) : "v"(m), "n"(C));
    return x;
}
template <int C>
__device__ __forceinline__ float row_bcast(float m)
{
    float x;
    asm volatile("s_nop 1\n\tv_mov_b32_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(x) : "v"(m), "n"(C));
    return x;
}

// 1/sqrt: the hardware estimate and one Newton step, r (1.5 - (0.5 x) r r).
__device__ __forceinline__ double rsqrt_estimate(double x) { return __builtin_amdgcn_rsq(x); }
__device__ __forceinline__ float rsqrt_estimate(float x) { return __builtin_amdgcn_rsqf(x); }
template <typename T>
__device__ __forceinline__ T rsqrt_newton(T x)
{
    const T r = rsqrt_estimate(x);
    return r * ((T)1.5 - (T)0.5 * x * r * r);
}

// The updates of columns [C, E) by column J.
template <int J, int C, int E, typename T>
__device__ __forceinline__ void leaf_updates(T (&u)[16], T (&v)[16])
{
    if constexpr (C < E) {
        row_fnma<C>(u[C], u[J], u[J]);
        row_fnma<C>(v[C], u[J], v[J]);
        leaf_updates<J, C + 1, E>(u, v);
    }
}

// Column J with its pivot x on every lane.  The next column's chain -- estimate, Newton step -- is
// laid between the updates, which do not depend on it.
template <int J, typename T>
__device__ __forceinline__ void leaf_columns(T (&u)[16], T (&v)[16], T rd, int &bad)
{
    u[J] *= rd;
    v[J] *= rd;
    if constexpr (J + 1 < 16) {
        // the next pivot first: it is the loop's serial chain
        row_fnma<J + 1, true>(u[J + 1], u[J], u[J]);
        row_fnma<J + 1>(v[J + 1], u[J], v[J]);
        const T x = row_bcast<J + 1>(u[J + 1]);
        // LLT.h:327-330; a NaN pivot passes.  (A vector minimum: a scalar test would put a branch and a
        // vector-to-scalar round trip into every column, half the column's time.)
        bad = min(bad, x <= (T)0 ? J + 1 : 16);
        constexpr int N = 14 - J, C = J + 2;  // updates left, in four parts
        const T r = rsqrt_estimate(x);
        const T h = (T)0.5 * x;
        __builtin_amdgcn_sched_barrier(0);
        leaf_updates<J, C, C + N / 4>(u, v);
        __builtin_amdgcn_sched_barrier(0);
        const T hr = h * r;
        __builtin_amdgcn_sched_barrier(0);
        leaf_updates<J, C + N / 4, C + N / 2>(u, v);
        __builtin_amdgcn_sched_barrier(0);
        const T f = (T)1.5 - hr * r;
        __builtin_amdgcn_sched_barrier(0);
        leaf_updates<J, C + N / 2, C + 3 * N / 4>(u, v);
        __builtin_amdgcn_sched_barrier(0);
        const T rn = r * f;
        __builtin_amdgcn_sched_barrier(0);
        leaf_updates<J, C + 3 * N / 4, 16>(u, v);
        leaf_columns<J + 1>(u, v, rn, bad);
    }
}

// u: the leaf's rows (entries right of the diagonal: any), replicated in the four rows of lanes;
// v: rows that take the same column operations, v <- v L^{-T}.  With the identity (v[c] = c ==
// l % 16) lane l is left with column l % 16 of X = L^{-1}: v[c] = X[c][l % 16].  Returns the failing
// column or -1 (uniform); entries of u right of a lane's diagonal change but are never read.
template <typename T>
__device__ __forceinline__ int leaf_factor(T (&u)[16], T (&v)[16])
{
    const T x = row_bcast<0>(u[0]);
    int bad = x <= (T)0 ? 0 : 16;
    leaf_columns<0>(u, v, rsqrt_newton(x), bad);
    bad = __builtin_amdgcn_readfirstlane(bad);
    return bad < 16 ? bad : -1;
}

}  // namespace mi
