// kron_final.hpp -- modes 1 and 0 of vectors larger than a workgroup keeps on chip, after kron_block_pass_kernel.
//
// A lane owns one position of the n^(d-2) faster elements: the n x n values there differ only in modes 0 and 1 and
// come by loads that are contiguous across the wavefront. Both modes are contracted in registers (no LDS, no
// barriers), mode 1 then mode 0, each output a fused chain over k ascending from zero as everywhere
// (kronmult_gpu/kronmult.cu:66-70). For n >= 8 a thread forms RB of the n rows of mode 1, so that the rows y[k0][RB]
// and the sums acc[r0][RB] fit the registers; the n / RB threads of one position read the same values through the
// caches.
//
// A wavefront walks `run` consecutive entries and keeps the sum of those with one output; the wavefronts of a workgroup
// take consecutive runs of one tile (of each of its row blocks) and add their sums in LDS when they all end on one
// output. So there is one atomic add per element and 2 or 4 runs.
//
// What bounds it: HBM (it reads the workspace once), then registers. 2 GB of d=6 vectors, read rate: n=6 FP64 6.0 TB/s,
// n=7 5.2, n=8 4.85 (all 8 rows per thread: 1.6), n=9 3.3 (3 rows), n=10 3.6; FP32 n=6 5.1, n=8 4.6, n=9 3.5 (9 rows),
// n=10 4.0. Two positions per lane in FP32 were slower (n=6 4.4). The realistic case of the reference's benchmark, d=6
// n=8 FP64, 3903 entries: 1.7 ms here and 3.55 ms in the block pass, against 10.2 ms in two passes of three modes in LDS.
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

// Runs of at least this many entries take the LONG variant. Its two differences pay where there is much to read and cost
// where the workspace still sits in the last cache level and the atomics count (both sides at the functions below).
constexpr int kLongRun = 4;

// Row blocks that share a workgroup: two blocks of one position read the same lines at about the same time there, but
// leave two runs instead of four to be summed before the atomics. d=6 n=8 FP64 1200 entries 1892 -> 1755 us, n=10 FP32
// 300 entries 975 -> 938; short runs would lose: n=8 FP64 40 entries 66 -> 77, n=10 FP64 25 entries 194 -> 222. The
// three blocks of n=9 are faster in workgroups of their own (3.3 against 2.7 TB/s).
template<int N, int RB, bool LONG>
constexpr int shared_rows()
{
    return LONG && N / RB == 2 ? 2 : 1;
}

// Reads past the caches: where one thread forms all rows each value is read once (d=6 n=6 3000 entries FP64 737 -> 717
// us, FP32 388 -> 381; n=7 FP64 d=5 346 -> 335; FP32 n=7 679 -> 690, so not there; short runs n=6 FP32 33 -> 35). Where
// row blocks share the reads it costs the cache hits (n=8 FP64 4.5 -> 3.5 TB/s).
template<typename T, int N, int RB, bool LONG>
constexpr bool past_caches()
{
    return LONG && RB == N && !(N == 7 && sizeof(T) == 4);
}

// consecutive parts of the entries that the wavefronts of one row block take
template<int N, int RB, bool LONG>
constexpr int parts()
{
    return kWaves / shared_rows<N, RB, LONG>();
}

template<typename T, int N, int RB, bool LONG>
__global__ void __launch_bounds__(kLanes *kWaves)
    kron_final_kernel(int nb, int run, int tiles, int inner, int d, T const *const *__restrict__ mats, int stride,
                      T const *const *__restrict__ ws, T *const *__restrict__ out)
{
    static_assert(N % RB == 0, "whole row blocks");
    constexpr int SHARED = shared_rows<N, RB, LONG>(), PARTS = parts<N, RB, LONG>();
    constexpr int SB = N / RB / SHARED;  // workgroups per tile
    constexpr int RED = 2;  // sums per lane and step of the reduction across wavefronts
    __shared__ T red[kWaves][RED][kLanes];
    __shared__ T *last[kWaves];
    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    int const per_run = tiles * SB;
    int b = kronreg::xcd_run_index();
    int const group = b / per_run;  // of PARTS * run entries
    b -= group * per_run;
    int const tile = b / SB;
    int const part = wave / SHARED, block = wave % SHARED;
    int const r1 = (SHARED > 1 ? block : b - tile * SB) * RB;
    int const g0 = group * run * PARTS;
    if (g0 >= nb) return;
    int const e0 = g0 + part * run < nb ? g0 + part * run : nb;
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
        auto read = [](kronreg::global_ptr<T const> p) {
            if constexpr (past_caches<T, N, RB, LONG>())
                return __builtin_nontemporal_load(p);
            else
                return *p;
        };
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
            for (int k1 = 0; k1 < N; ++k1) x[k1] = read(src + static_cast<size_t>(k0 * N + k1) * inner);
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
            if (part < RED && q + part < N * RB)
            {
                T s = red[block][part][lane];
#pragma unroll
                for (int w = 1; w < PARTS; ++w) s += red[w * SHARED + block][part][lane];
                add(s, (q + part) / RB, (q + part) % RB);
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
