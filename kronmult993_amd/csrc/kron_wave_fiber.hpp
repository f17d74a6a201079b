// kron_wave_fiber.hpp -- one wavefront per entry, each lane owning whole fibers: tensors of 81 to 625 elements, single
// batches and groups of the grouped launch.
//
// Against kron_wave.hpp (a lane forms one element per step: n values and n factor entries from LDS for n
// multiply-adds) a lane forms the n outputs of a fiber from n values and n^2 factor entries that the whole wavefront
// reads as broadcasts, 16 bytes at a time. The entry's values and factors are read into registers one entry ahead and
// staged in the wavefront's own LDS rows; a wavefront's LDS accesses complete in order, so no barriers. The factors'
// addresses are read two entries ahead, so that no load waits for another one. Steps as everywhere: one fused chain
// over k ascending from zero per output, last factor first (kronmult_gpu/kronmult.cu:66-70, :104).
//
// Each wavefront sums consecutive entries with one output in registers; kWaves wavefronts of a workgroup take
// consecutive runs, and those that end on one output add their sums in LDS before the atomics. What bounds the small
// shapes of the reference's grid (5 outputs) is the atomic adds, about 200 G/s: 4608 entries of d=3 n=6 FP32 19.5 us
// with runs of 2 in one-wavefront workgroups, 8.3 here. With four entries per output: 6000 of d=3 n=6 FP64 8.1 us
// (packed launch 11.3), FP32 5.6 (7.4); 6000 of d=3 n=7 FP64 11.4 (17.0), FP32 7.6 (13.0); 20000 of d=5 n=3 19.8
// (24.6), of d=8 n=2 19.9 (27.5); 6000 of d=4 n=5 13.5 (block sweep 14.4), FP32 8.5 (10.0).
// Outputs that no two entries share leave the sums across wavefronts nothing to do: d=4 n=3, 20000 entries FP32 10.2 us
// one element per lane, 11.4 here (with 5 outputs 78 and 26); the other shapes are within 5% or faster there too.
// Not taken here: d=3 n=5 (20000 entries 15.3 us against 13.6 one element per lane), d=6 n=3 (16.8 us against 15.6 on
// the block sweep), d=3 n=8 (18 us against 13.3 on the matrix cores).
#pragma once

#include <hip/hip_runtime.h>

#include "kron_wave.hpp"

namespace kronwave
{

constexpr int kWaves = 4;  // wavefronts per workgroup (8: 3-20% slower)

template<typename T, int D, int N>
struct FiberWave
{
    static constexpr int SIZE = wave_elems(D, N);
    static constexpr int NF = SIZE / N;
    static constexpr int F = (NF + kLanes - 1) / kLanes;  // fibers per lane
    static constexpr int NCOEF = D * N * N;
    static constexpr int XPL = (SIZE + kLanes - 1) / kLanes;
    static constexpr int CPL = (NCOEF + kLanes - 1) / kLanes;
    static constexpr int GR = 16 / static_cast<int>(sizeof(T));
    // LDS rows: the tensor in canonical order (n = 4 FP64: every row of 4 followed by 16 bytes, the fastest mode's
    // fibers then start in different banks), the factors' columns at multiples of 16 bytes
    static constexpr int PAD = (N == 4 && sizeof(T) == 8) ? GR : 0;
    static constexpr int XS = (SIZE + PAD * NF + GR - 1) / GR * GR;
    static constexpr int CP = (N + GR - 1) / GR * GR;
    static constexpr int LDS = XS + D * N * CP;

    static constexpr int pa(int e) { return PAD == 0 ? e : e + PAD * (e / N); }

    // first element of fiber lane + 64 i of the mode with stride ST (a lane past the last fiber repeats it, and
    // writes nothing)
    template<int ST>
    static __device__ __forceinline__ int fiber(int lane, int i)
    {
        int f = lane + i * kLanes;
        if (NF % kLanes != 0 && i + 1 == F && f >= NF) f = NF - 1;
        return (f / ST) * (ST * N) + f % ST;
    }
    static __device__ __forceinline__ bool active(int lane, int i)
    {
        return NF % kLanes == 0 || i + 1 < F || lane + i * kLanes < NF;
    }
    static constexpr int step(int st) { return st == 1 ? 1 : st + PAD * (st / N); }

    template<int M>
    static __device__ __forceinline__ void contract(T const *xs, T const *cs, int lane, T (&y)[F][N])
    {
        constexpr int ST = wave_elems(D - 1 - M, N);
        T x[F][N];
#pragma unroll
        for (int i = 0; i < F; ++i)
        {
            T const *p = xs + pa(fiber<ST>(lane, i));
#pragma unroll
            for (int k = 0; k < N; ++k) x[i][k] = p[k * step(ST)];
        }
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            T c[N];
#pragma unroll
            for (int r = 0; r < N; ++r) c[r] = cs[(M * N + k) * CP + r];
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int r = 0; r < N; ++r) y[i][r] = fma(x[i][k], c[r], k == 0 ? T(0) : y[i][r]);
        }
        // the sums are complete here: not moved into the branch on active lanes, which would keep every entry of the
        // factor live across it (d=3 n=6 FP64: 89 registers instead of 128)
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int r = 0; r < N; ++r) asm volatile("" : "+v"(y[i][r]));
    }
    // modes M .. 1 in place
    template<int M>
    static __device__ __forceinline__ void modes(T *xs, T const *cs, int lane)
    {
        if constexpr (M > 0)
        {
            constexpr int ST = wave_elems(D - 1 - M, N);
            T y[F][N];
            contract<M>(xs, cs, lane, y);
            wave_sync();
#pragma unroll
            for (int i = 0; i < F; ++i)
            {
                T *p = xs + pa(fiber<ST>(lane, i));
                if (active(lane, i))
#pragma unroll
                    for (int r = 0; r < N; ++r) p[r * step(ST)] = y[i][r];
            }
            wave_sync();
            modes<M - 1>(xs, cs, lane);
        }
    }

    static __device__ __forceinline__ void flush(T *cur, T const (&acc)[F][N], int lane)
    {
        kronreg::global_ptr<T> dst = kronreg::as_global(cur);
#pragma unroll
        for (int i = 0; i < F; ++i)
            if (active(lane, i))
#pragma unroll
                for (int r = 0; r < N; ++r) atomicAdd((T *)(dst + lane + i * kLanes + r * NF), acc[i][r]);
    }

    // entries [e0, e1), e0 < e1; leaves the sum of the last ones with one output, cur, in acc (zero on entry)
    static __device__ __forceinline__ void run(int e0, int e1, T const *const *__restrict__ mats, int stride,
                                               T const *const *__restrict__ in, T *const *__restrict__ out, T *xs,
                                               int lane, T (&acc)[F][N], T *&cur)
    {
        T *const cs = xs + XS;
        int const last = e1 - 1;
        T x[XPL], f[CPL];
        T const *fp[CPL];
        auto pointers = [&](int e) {
#pragma unroll
            for (int c = 0; c < CPL; ++c)
            {
                int const i = lane + c * kLanes;
                if (i < NCOEF) fp[c] = kronreg::as_global(mats)[static_cast<size_t>(e) * D + i / (N * N)];
            }
        };
        auto load = [&](int e) {
            kronreg::global_ptr<T const> src = kronreg::as_global(in[e]);
#pragma unroll
            for (int c = 0; c < CPL; ++c)
            {
                int const i = lane + c * kLanes;  // factor value i: A_m(r, k) at m n^2 + k n + r
                if (i < NCOEF) f[c] = kronreg::as_global(fp[c])[i % N + (i / N) % N * stride];
            }
#pragma unroll
            for (int j = 0; j < XPL; ++j)
                if (lane + j * kLanes < SIZE) x[j] = src[lane + j * kLanes];
        };
        pointers(e0);
        load(e0);
        pointers(e0 < last ? e0 + 1 : last);
        cur = out[e0];
        for (int e = e0; e < e1; ++e)
        {
#pragma unroll
            for (int j = 0; j < XPL; ++j)
                if (lane + j * kLanes < SIZE) xs[pa(lane + j * kLanes)] = x[j];
#pragma unroll
            for (int c = 0; c < CPL; ++c)
            {
                int const i = lane + c * kLanes;
                if (i < NCOEF) cs[(i / N) * CP + i % N] = f[c];
            }
            if (e < last)
            {
                load(e + 1);
                pointers(e + 2 < last ? e + 2 : last);
            }
            wave_sync();
            modes<D - 1>(xs, cs, lane);
            T y[F][N];
            contract<0>(xs, cs, lane, y);
            wave_sync();
            T *const dst = out[e];
            if (dst != cur)
            {
                flush(cur, acc, lane);
#pragma unroll
                for (int i = 0; i < F; ++i)
#pragma unroll
                    for (int r = 0; r < N; ++r) acc[i][r] = T(0);
                cur = dst;
            }
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int r = 0; r < N; ++r) acc[i][r] += y[i][r];
        }
    }

    // The workgroup's kWaves wavefronts (every thread comes here; cur is null for one without entries): the first
    // of those in a row that ended on one output adds their sums.
    static __device__ __forceinline__ void finish(T *cur, T (&acc)[F][N], T *rows, T **last, int wave, int lane)
    {
        T *const xs = rows + wave * LDS;
#pragma unroll
        for (int i = 0; i < F; ++i)
            if (active(lane, i))
#pragma unroll
                for (int r = 0; r < N; ++r) xs[lane + i * kLanes + r * NF] = acc[i][r];
        if (lane == 0) last[wave] = cur;
        __syncthreads();
        if (cur == nullptr || (wave > 0 && last[wave - 1] == cur)) return;
        for (int w = wave + 1; w < kWaves && last[w] == cur; ++w)
        {
            T const *const other = rows + w * LDS;
#pragma unroll
            for (int i = 0; i < F; ++i)
                if (active(lane, i))
#pragma unroll
                    for (int r = 0; r < N; ++r) acc[i][r] += other[lane + i * kLanes + r * NF];
        }
        flush(cur, acc, lane);
    }

    // entries [g0, g1) by one workgroup, consecutive runs of ceil((g1 - g0) / kWaves)
    static __device__ __forceinline__ void group(int g0, int g1, int epw, T const *const *__restrict__ mats, int stride,
                                                 T const *const *__restrict__ in, T *const *__restrict__ out, T *rows,
                                                 T **last, int wave, int lane)
    {
        int const e0 = g0 + kronruns::begin(wave, epw, g1 - g0);
        int const e1 = kronruns::end(e0, epw, g1);
        T acc[F][N];
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int r = 0; r < N; ++r) acc[i][r] = T(0);
        T *cur = nullptr;
        if (e0 < e1) run(e0, e1, mats, stride, in, out, rows + wave * LDS, lane, acc, cur);
        finish(cur, acc, rows, last, wave, lane);
    }
};

// epw: entries per workgroup, any number (its wavefronts take ceil(epw / kWaves) each, the last ones what is left)
template<typename T, int D, int N>
__global__ void __launch_bounds__(kLanes *kWaves)
    kron_wave_fiber_kernel(int nb, int epw, T const *const *__restrict__ mats, int stride,
                           T const *const *__restrict__ in, T *const *__restrict__ out)
{
    using FW = FiberWave<T, D, N>;
    __shared__ __attribute__((aligned(16))) T rows[kWaves * FW::LDS];
    __shared__ T *last[kWaves];
    int const g0 = kronreg::xcd_run_begin(epw, nb);
    if (g0 >= nb) return;
    int const g1 = kronruns::end(g0, epw, nb);
    int const wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    FW::group(g0, g1, (epw - 1) / kWaves + 1, mats, stride, in, out, rows, last, wave, static_cast<int>(threadIdx.x & 63));
}

// Shapes whose single batches run here: of the wave family, of the fiber family, of the packed family's default.
#define KRON_WAVE_FIBER_SHAPES(X) X(4, 3) X(5, 3) X(7, 2) X(8, 2) X(3, 6) X(3, 7) X(4, 5)

__host__ __device__ constexpr bool wave_fiber_shape(int d, int n)
{
#define KRON_WAVE_FIBER_IS(D, N) \
    if (d == D && n == N) return true;
    KRON_WAVE_FIBER_SHAPES(KRON_WAVE_FIBER_IS)
#undef KRON_WAVE_FIBER_IS
    return false;
}

} // namespace kronwave
