// quad_solve.hpp -- triangular substitution with four lanes per column.
//
// Lane s = lane & 3 of a group of four holds rows 4 t + s of a column of N
// rows in x[t].  The solved x_k reaches the other three lanes by a DPP
// broadcast, so a column takes N steps of at most N/4 fused multiply-adds (a
// thread per column: up to N - 1).  Column-oriented order, true division by
// the diagonal, as the reference's substitution kernels.
#pragma once

#include "common.hpp"

namespace rsa
{

template <int S>
__device__ __forceinline__ float quad_broadcast(float v)
{
    return __int_as_float(dpp_mov<0x55 * S>(__float_as_int(v)));
}
template <int S>
__device__ __forceinline__ double quad_broadcast(double v)
{
    return dpp_mov_d<0x55 * S>(v);
}

// 0, which the optimiser must take as computed from every x (an empty asm):
// an address it is added to is known only then, so the reads of a triangle
// that the solve of x walks through are not all issued ahead, nor the updates
// of its later rows put off with their operands kept, in registers (which
// spills).
template <typename T, int N>
__device__ __forceinline__ uint32_t after(const T (&x)[N])
{
    uint32_t zero = 0;
#pragma unroll
    for(int t = 0; t < N; ++t)
        asm volatile("" : "+v"(zero) : "v"(x[t]));
    return zero;
}

// x <- T^-1 x, T the lower (forward) or upper (backward) triangle of an N x N
// block, column-major in LDS; UNIT: its diagonal is taken as 1.  The columns
// are read in groups of G, one group ahead of the one being applied.
template <typename T, int N, bool LOWER, bool UNIT, int STEP, int G>
__device__ __forceinline__ void quad_solve_group(const T* L, int lane, T (&x)[N / 4],
                                                 const T (&cur)[G][N / 4])
{
    const int s = lane & 3;
    T next[G][N / 4];
    if constexpr(STEP + G < N)
    {
        const T* at = L + after(x) + s;
#pragma unroll
        for(int g = 0; g < G; ++g)
        {
            const int K = LOWER ? STEP + G + g : N - 1 - (STEP + G + g);
#pragma unroll
            for(int t = 0; t < N / 4; ++t)
                if(LOWER ? t >= K / 4 : t <= K / 4)
                    next[g][t] = at[K * N + 4 * t];
        }
    }
#pragma unroll
    for(int g = 0; g < G; ++g)
    {
        const int K = LOWER ? STEP + g : N - 1 - (STEP + g);
        const int o = K % 4, q = K / 4; // row K: lane o of the four, x[q]
        if constexpr(!UNIT)
        {
            // in lane o cur[g][q] is the diagonal entry
            const T y = x[q] / cur[g][q];
            x[q] = s == o ? y : x[q];
        }
        const T xk = o == 0   ? quad_broadcast<0>(x[q])
                     : o == 1 ? quad_broadcast<1>(x[q])
                     : o == 2 ? quad_broadcast<2>(x[q])
                              : quad_broadcast<3>(x[q]);
        if(LOWER ? o < 3 : o > 0)
        {
            const T y = fma_t(-cur[g][q], xk, x[q]);
            x[q] = (LOWER ? s > o : s < o) ? y : x[q];
        }
#pragma unroll
        for(int t = 0; t < N / 4; ++t)
            if(LOWER ? t > q : t < q)
                x[t] = fma_t(-cur[g][t], xk, x[t]);
    }
    if constexpr(STEP + G < N)
        quad_solve_group<T, N, LOWER, UNIT, STEP + G, G>(L, lane, x, next);
}

template <typename T, int N, bool LOWER, bool UNIT, int G = (sizeof(T) == 8 ? 2 : 4)>
__device__ __forceinline__ void quad_solve(const T* L, int lane, T (&x)[N / 4])
{
    static_assert(N % G == 0, "whole groups");
    T first[G][N / 4];
#pragma unroll
    for(int g = 0; g < G; ++g)
    {
        const int K = LOWER ? g : N - 1 - g;
#pragma unroll
        for(int t = 0; t < N / 4; ++t)
            if(LOWER ? t >= K / 4 : t <= K / 4)
                first[g][t] = L[K * N + 4 * t + (lane & 3)];
    }
    quad_solve_group<T, N, LOWER, UNIT, 0, G>(L, lane, x, first);
}

} // namespace rsa
