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
// block, column-major in LDS; UNIT: its diagonal is taken as 1.  STEP counts
// the columns done.
template <typename T, int N, bool LOWER, bool UNIT, int STEP = 0>
__device__ __forceinline__ void quad_solve(const T* L, int lane, T (&x)[N / 4])
{
    if constexpr(STEP < N)
    {
        constexpr int K = LOWER ? STEP : N - 1 - STEP;
        if constexpr(STEP % 4 == 0)
        {
            L += after(x);
        }
        const int s = lane & 3;
        const T* col = L + K * N;
        if constexpr(!UNIT)
        {
            const T y = x[K / 4] / col[K];
            x[K / 4] = s == K % 4 ? y : x[K / 4];
        }
        const T xk = quad_broadcast<K % 4>(x[K / 4]);
        if constexpr(LOWER ? K % 4 < 3 : K % 4 > 0)
        {
            const T y = fma_t(-col[K / 4 * 4 + s], xk, x[K / 4]);
            x[K / 4] = (LOWER ? s > K % 4 : s < K % 4) ? y : x[K / 4];
        }
#pragma unroll
        for(int t = LOWER ? K / 4 + 1 : 0; t < (LOWER ? N / 4 : K / 4); ++t)
            x[t] = fma_t(-col[4 * t + s], xk, x[t]);
        quad_solve<T, N, LOWER, UNIT, STEP + 1>(L, lane, x);
    }
}

} // namespace rsa
