// kron_final.hpp -- modes 1 and 0 of vectors larger than a workgroup keeps on chip, after kron_block_pass_kernel.
//
// A lane owns one position of the n^(d-2) faster elements: the n x n values there differ only in modes 0 and 1 and
// come by loads that are contiguous across the wavefront. Both modes are contracted in registers (no LDS, no
// barriers), mode 1 then mode 0, each output a fused chain over k ascending from zero as everywhere
// (kronmult_gpu/kronmult.cu:66-70). For n >= 8 a thread forms RB of the n rows of mode 1, so that the rows y[k0][RB]
// and the sums acc[r0][RB] fit the registers; the n / RB threads of one position read the same values through the
// caches.
//
// A wavefront walks `run` consecutive entries and keeps the sum of those with one output; the W wavefronts of a
// workgroup take consecutive runs of one tile and add their sums in LDS when they all end on one output. So there is
// one atomic add per element and W * run entries.
//
// What bounds it: HBM (it reads the workspace once), then registers. 2 GB of d=6 vectors, read rate: n=6 FP64 5.5 TB/s,
// n=8 4.4 (all 8 rows per thread: 1.6), n=9 3.1 (3 rows), n=10 3.7; FP32 4.7, 4.4, 3.3 (9 rows), 3.6. Two positions
// per lane in FP32 were slower (n=6 4.4). The realistic case of the reference's benchmark, d=6 n=8 FP64, 3903 entries:
// 1.8 ms here and 3.6 ms in the block pass, against 10.2 ms in two passes of three modes in LDS.
#pragma once

#include <hip/hip_runtime.h>

#include "kron_block.hpp"

namespace kronfinal
{

constexpr int kLanes = 64;
constexpr int kWaves = 4;   // wavefronts per workgroup (8: n=8 FP64 4.1 against 4.3 TB/s, fewer workgroups fit)
constexpr int kMaxRun = 8;  // entries per wavefront
// shorter runs where there are few entries: at least this many wavefronts per CU
constexpr int kWavesPerCu = 16;

// rows of mode 1 per thread (a divisor of n)
template<typename T, int N>
constexpr int rows()
{
    return N <= 7 ? N : N == 8 ? 4 : N == 9 ? (sizeof(T) == 8 ? 3 : 9) : 5;
}

template<typename T, int N, int RB>
__global__ void __launch_bounds__(kLanes *kWaves)
    kron_final_kernel(int nb, int run, int tiles, int inner, int d, T const *const *__restrict__ mats, int stride,
                      T const *const *__restrict__ ws, T *const *__restrict__ out)
{
    static_assert(N % RB == 0, "whole row blocks");
    constexpr int SB = N / RB;
    constexpr int RED = 2;  // sums per lane and step of the reduction across wavefronts
    __shared__ T red[kWaves][RED][kLanes];
    __shared__ T *last[kWaves];
    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    int const per_run = tiles * SB;
    int b = kronreg::xcd_run_index();
    int const group = b / per_run;  // of kWaves * run entries
    b -= group * per_run;
    int const tile = b / SB, r1 = (b - tile * SB) * RB;
    int const g0 = group * run * kWaves;
    if (g0 >= nb) return;
    int const e0 = g0 + wave * run < nb ? g0 + wave * run : nb;
    int const e1 = e0 + run < nb ? e0 + run : nb;
    int const pos = tile * kLanes + lane;
    bool const act = pos < inner;
    int const rd = act ? pos : inner - 1;  // a lane past the end reads the last position and adds nothing

    T acc[N][RB];
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < RB; ++j) acc[i][j] = T(0);
    T *cur = e0 < e1 ? out[e0] : nullptr;
    auto add = [&](T v, int r0, int j) {
        if (act) atomicAdd((T *)(kronreg::as_global(cur) + static_cast<size_t>(r0 * N + r1 + j) * inner + pos), v);
    };
    for (int e = e0; e < e1; ++e)
    {
        T *const dst = out[e];
        if (dst != cur)
        {
#pragma unroll
            for (int i = 0; i < N; ++i)
#pragma unroll
                for (int j = 0; j < RB; ++j)
                {
                    add(acc[i][j], i, j);
                    acc[i][j] = T(0);
                }
            cur = dst;
        }
        T const *const *A = mats + static_cast<size_t>(e) * d;
        kronreg::constant_ptr<T> A1 = kronreg::as_constant(A[1]) + r1;
        kronreg::constant_ptr<T> A0 = kronreg::as_constant(A[0]);
        kronreg::global_ptr<T const> src = kronreg::as_global(ws[e]) + rd;
        T y[N][RB];
#pragma unroll
        for (int k0 = 0; k0 < N; ++k0)
        {
            // The factors' addresses are made opaque where all their values would not fit the scalar registers:
            // they are then read again (scalar cache) instead of being kept in vector lanes (n=10 FP64 2.5 -> 3.7
            // TB/s).
            if (N * RB > 32 && k0 % 2 == 0) asm volatile("" : "+s"(A1));
            T x[N];
#pragma unroll
            for (int k1 = 0; k1 < N; ++k1) x[k1] = src[static_cast<size_t>(k0 * N + k1) * inner];
#pragma unroll
            for (int k1 = 0; k1 < N; ++k1)
#pragma unroll
                for (int j = 0; j < RB; ++j)
                    y[k0][j] = fma(x[k1], A1[j + k1 * stride], k1 == 0 ? T(0) : y[k0][j]);
        }
#pragma unroll
        for (int j = 0; j < RB; ++j)
        {
            asm volatile("" : "+s"(A0));
            T z[N];
#pragma unroll
            for (int k0 = 0; k0 < N; ++k0)
#pragma unroll
                for (int i = 0; i < N; ++i) z[i] = fma(y[k0][j], A0[i + k0 * stride], k0 == 0 ? T(0) : z[i]);
#pragma unroll
            for (int i = 0; i < N; ++i) acc[i][j] += z[i];
        }
    }
    // the wavefronts' last sums: added in LDS first where all end on one output (wavefront 0 always has entries)
    if (lane == 0) last[wave] = cur;
    __syncthreads();
    bool same = true;
#pragma unroll
    for (int w = 1; w < kWaves; ++w) same = same && (last[w] == last[0] || last[w] == nullptr);
    if (same)
    {
        cur = last[0];
#pragma unroll
        for (int q = 0; q < N * RB; q += RED)
        {
            __syncthreads();
#pragma unroll
            for (int u = 0; u < RED; ++u)
                if (q + u < N * RB) red[wave][u][lane] = acc[(q + u) / RB][(q + u) % RB];
            __syncthreads();
            if (wave < RED && q + wave < N * RB)
            {
                T s = red[0][wave][lane];
#pragma unroll
                for (int w = 1; w < kWaves; ++w) s += red[w][wave][lane];
                add(s, (q + wave) / RB, (q + wave) % RB);
            }
        }
    }
    else if (cur != nullptr)
    {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < RB; ++j) add(acc[i][j], i, j);
    }
}

} // namespace kronfinal
