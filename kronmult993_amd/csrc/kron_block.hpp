// kron_block.hpp -- contiguous blocks of a vector swept in LDS: whole entries of 3 KB to 80 KB, and the fastest modes
// of larger ones (kron_final.hpp applies the two that are left).
//
// A block is Q consecutive sub-tensors of n^G elements. The workgroup stages it in LDS and contracts its G modes in
// place, fastest first: a thread owns whole fibers (n values that differ in one mode), at most one barrier per mode.
// n, G, Q and the workgroup size are compile-time, so every LDS address is one register plus immediate offsets.
// Every output is one fused chain over k ascending from zero, factors from the last to the first: bit-identical per
// entry to the reference's sweep (kronmult_gpu/kronmult.cu:66-70, :104).
//
// What bounds it: a workgroup's chain per entry (staging, then per mode a scalar round trip for the factor, an LDS
// round trip and a barrier) and, beside it, HBM. Hence
//   * the factors are read into scalar registers, one SGPR operand per multiply-add: as many columns as kColSgprs
//     holds one mode ahead (before the barrier that orders the mode's values), the rest at their use. 4608 entries
//     of d=5 n=5 FP64 57.7 -> 45.8 us together with the next item, of d=4 n=7 FP32 43 -> 30 us. FP32 whole entries
//     with one fiber per thread keep them in the lanes instead (LaneCols): 29.1 -> 24.7 us;
//   * the next entry's factors are brought into the L2 one entry ahead (Touch): a cold factor costs the chain two
//     trips to HBM per mode (d=5 n=5 FP64 57.7 -> 47.4 us alone, d=4 n=9 FP64 198 -> 127 us);
//   * the next block's values are read into registers while this one is swept;
//   * consecutive entries with one output are summed in registers: one atomic per element, output and run instead of
//     one per entry, which alone took 70 us of the 143 us that d=5 n=5 took with one workgroup per entry (14.4 M
//     FP64 atomic adds at about 200 G/s).
#pragma once

#include <hip/hip_runtime.h>

#include "kron_reg.hpp"

namespace kronblock
{

constexpr int ipow(int b, int e)
{
    int r = 1;
    for (int i = 0; i < e; ++i) r *= b;
    return r;
}

// Scalar registers for the factor columns that are read one mode ahead (40: d=4 n=7 FP64 51 us, 56: 46 us; more do
// not fit beside the pointers).
constexpr int kColSgprs = 56;

template<typename T, int N, int G, int Q, int P>
struct Block
{
    static constexpr int S = Q * ipow(N, G);  // elements
    static constexpr int NFIB = S / N;
    static constexpr int F = (NFIB + P - 1) / P;  // fibers per thread
    static constexpr int GR = 16 / static_cast<int>(sizeof(T));
    // LDS: canonical order; for n = 8, and n = 4 in FP64, every row of n is followed by 16 bytes, so that the fastest
    // mode's fibers, a row apart across lanes, start in different banks (other n: the row length does that by itself)
    static constexpr int PAD = N == 8 || (N == 4 && sizeof(T) == 8) ? GR : 0;
    static constexpr int LDS = S + PAD * (S / N);
    static constexpr int NGRAN = S / GR, REM = S % GR;
    static constexpr int CPT = (NGRAN + P - 1) / P;
    using V = typename kronreg::Granule<T>::type;
    // 16 bytes at an address aligned to the element: what n odd gives, and all that a caller's pointer promises
    typedef T VU __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));

    static constexpr int pa(int e) { return PAD == 0 ? e : e + PAD * (e / N); }
    // between consecutive elements of a fiber
    template<int ST>
    static constexpr int step()
    {
        return ST == 1 ? 1 : ST + PAD * (ST / N);
    }

    // ---- staging: granules c*P + t in registers, then in LDS; the last S % GR elements one by one
    V pre[CPT];
    T pre_rem;

    static __device__ __forceinline__ bool granule(int c, int t)
    {
        return NGRAN % P == 0 || c + 1 < CPT || c * P + t < NGRAN;
    }
    __device__ __forceinline__ void load(T const *src_generic, int t)
    {
        kronreg::global_ptr<T const> src = kronreg::as_global(src_generic);
#pragma unroll
        for (int c = 0; c < CPT; ++c)
            if (granule(c, t)) pre[c] = *(kronreg::global_ptr<VU const>)(src + (c * P + t) * GR);
        if (REM > 0 && t < REM) pre_rem = src[NGRAN * GR + t];
    }
    // the values of load are in the registers
    __device__ __forceinline__ void arrived()
    {
#pragma unroll
        for (int c = 0; c < CPT; ++c) asm volatile("" : "+v"(pre[c]));
        if (REM > 0) asm volatile("" : "+v"(pre_rem));
    }
    __device__ __forceinline__ void store(T *lds, int t) const
    {
#pragma unroll
        for (int c = 0; c < CPT; ++c)
            if (granule(c, t)) *reinterpret_cast<V *>(lds + pa((c * P + t) * GR)) = pre[c];
        if (REM > 0 && t < REM) lds[pa(NGRAN * GR + t)] = pre_rem;
    }

    // ---- fibers: number t + i*P of the mode with stride ST (a thread past the last one repeats it, and writes nothing)
    template<int ST>
    static __device__ __forceinline__ int fiber(int t, int i)
    {
        int f = t + i * P;
        if (NFIB % P != 0 && i + 1 == F && f >= NFIB) f = NFIB - 1;
        return (f / ST) * (ST * N) + f % ST;
    }
    static __device__ __forceinline__ bool active(int t, int i)
    {
        return NFIB % P == 0 || i + 1 < F || t + i * P < NFIB;
    }

    // The first KP columns of a factor, read ahead. The scheduling fence keeps the loads where they are written.
    static constexpr int KP = N * N * static_cast<int>(sizeof(T)) <= 4 * kColSgprs
                                  ? N
                                  : 4 * kColSgprs / (N * static_cast<int>(sizeof(T)));
    struct Cols
    {
        T c[KP][N];
        __device__ __forceinline__ void load(T const *A_generic, int stride)
        {
            kronreg::constant_ptr<T> A = kronreg::as_constant(A_generic);
#pragma unroll
            for (int k = 0; k < KP; ++k)
#pragma unroll
                for (int r = 0; r < N; ++r) c[k][r] = A[r + k * stride];
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // y = A times the thread's fibers of the mode with stride ST (cols: A's first columns)
    template<int ST>
    static __device__ __forceinline__ void contract(T const *lds, Cols const &cols, T const *A_generic, int stride,
                                                    int t, T (&y)[F][N])
    {
        constexpr int STEP = step<ST>();
        kronreg::constant_ptr<T> A = kronreg::as_constant(A_generic);
        T x[F][N];
#pragma unroll
        for (int i = 0; i < F; ++i)
        {
            T const *p = lds + pa(fiber<ST>(t, i));
#pragma unroll
            for (int k = 0; k < N; ++k) x[i][k] = p[k * STEP];
        }
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            T c[N];
#pragma unroll
            for (int r = 0; r < N; ++r) c[r] = k < KP ? cols.c[k < KP ? k : 0][r] : A[r + k * stride];
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int r = 0; r < N; ++r) y[i][r] = fma(x[i][k], c[r], k == 0 ? T(0) : y[i][r]);
        }
        // the sums are complete here: not moved into the branch on active threads, below the next columns' loads
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int r = 0; r < N; ++r) asm volatile("" : "+v"(y[i][r]));
    }

    // modes M .. 1 of the sub-tensors (cols: A[M]'s first columns on entry, A[0]'s on return)
    template<int M>
    static __device__ __forceinline__ void inner_modes(T *lds, Cols &cols, T const *const *A, int stride, int t)
    {
        if constexpr (M > 0)
        {
            constexpr int ST = ipow(N, G - 1 - M);
            constexpr int STEP = step<ST>();
            T y[F][N];
            contract<ST>(lds, cols, A[M], stride, t, y);
            cols.load(A[M - 1], stride);
#pragma unroll
            for (int i = 0; i < F; ++i)
            {
                T *p = lds + pa(fiber<ST>(t, i));
                if (active(t, i))
#pragma unroll
                    for (int r = 0; r < N; ++r) p[r * STEP] = y[i][r];
            }
            kronreg::lds_barrier();
            inner_modes<M - 1>(lds, cols, A, stride, t);
        }
    }
};

// Brings the next entry's factors into the L2: thread t reads the first or the last value of a factor column (at most
// 80 bytes, so at most two lines). The factor's address is read one entry earlier still: no load waits for another.
template<typename T, int N, int D, int P>
struct Touch
{
    static constexpr int COUNT = 2 * N * D;
    static constexpr int PER = (COUNT + P - 1) / P;
    T const *ptr[PER];
    T val[PER];
    static __device__ __forceinline__ int slot(int t, int c) { return t + c * P < COUNT ? t + c * P : COUNT - 1; }
    __device__ __forceinline__ void init(T const *const *mats, int e, int t)
    {
#pragma unroll
        for (int c = 0; c < PER; ++c)
        {
            ptr[c] = kronreg::as_global(mats)[static_cast<size_t>(e) * D + slot(t, c) / (2 * N)];
            val[c] = T(0);
        }
    }
    // reads the entry whose addresses are held, then the addresses of entry e
    __device__ __forceinline__ void next(T const *const *mats, int e, int stride, int t)
    {
#pragma unroll
        for (int c = 0; c < PER; ++c)
        {
            asm volatile("" ::"v"(val[c]));  // the previous entry's read is used, so that it is made
            int const s = slot(t, c) % (2 * N);
            val[c] = kronreg::as_global(ptr[c])[(s & 1) * (N - 1) + (s >> 1) * stride];
            ptr[c] = kronreg::as_global(mats)[static_cast<size_t>(e) * D + slot(t, c) / (2 * N)];
        }
    }
};

// FP32: the factors of an entry in the lanes and the products on the matrix cores, as LaneFactors (kron_reg.hpp), for
// any n <= 10: a factor is H = ceil(n / 4) x n blocks of four rows of one column, sixteen to a register; rows past n repeat
// the last one and their results are dropped. The values of the next entry are loaded during this one, from addresses
// read one entry earlier.
//
// Taken where a thread has one fiber. Against FMA chains with the factor columns in scalar registers, 200 / 1500 / 6000
// entries in us: d=4 n=7 5.6 / 12.3 / 31.0 -> 5.0 / 11.3 / 24.9, d=5 n=5 5.9 / 14.9 / 38.6 -> 5.5 / 14.5 / 34.6, d=4 n=6
// 16.3 -> 14.9 (6000), n=9 79 -> 67, n=10 138 -> 113, d=3 n=9 14.7 -> 12.4, n=10 18.1 -> 14.2. With two and four fibers
// the results' registers cost wavefronts (d=5 n=6 79 -> 89, d=6 n=5 220 -> 267); n = 3 gains nothing (11.5, 11.6).
template<typename T, int N, int D, int P>
constexpr bool lane_factors()
{
    return sizeof(T) == 4 && N > 4 && Block<T, N, D, 1, P>::F == 1;
}

template<typename B, int N, int D>
struct LaneCols
{
    static constexpr int H = (N + 3) / 4, V = (H * N + 15) / 16;
    float a[D][V];

    __device__ __forceinline__ void load(float const *const (&A)[D], int stride, int lane)
    {
#pragma unroll
        for (int i = 0; i < V; ++i)
        {
            int const q = i * 16 + (lane >> 2) < H * N ? i * 16 + (lane >> 2) : H * N - 1;
            int const row = 4 * (q / N) + (lane & 3);
            int const off = (row < N ? row : N - 1) + q % N * stride;
#pragma unroll
            for (int m = 0; m < D; ++m) a[m][i] = kronreg::as_global(A[m])[off];
        }
    }

    // y = factor M times the thread's fibers
    template<int M>
    __device__ __forceinline__ void contract(float const *lds, int t, float (&y)[B::F][N]) const
    {
        constexpr int ST = ipow(N, D - 1 - M);
        constexpr int STEP = B::template step<ST>();
        float x[B::F][N];
        kronreg::Quad z[B::F][H];
#pragma unroll
        for (int i = 0; i < B::F; ++i)
        {
            float const *p = lds + B::pa(B::template fiber<ST>(t, i));
#pragma unroll
            for (int k = 0; k < N; ++k) x[i][k] = p[k * STEP];
#pragma unroll
            for (int h = 0; h < H; ++h) z[i][h] = kronreg::Quad{0.f, 0.f, 0.f, 0.f};
        }
        kronreg::static_for<0, N * H>([&](auto s) {
            constexpr int k = s.value / H, h = s.value % H, q = h * N + k;
#pragma unroll
            for (int i = 0; i < B::F; ++i)
                z[i][h] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[M][q / 16], x[i][k], z[i][h], 4, q % 16, 0);
        });
        // the matrix instruction takes every lane: it stays above the branch on active threads
#pragma unroll
        for (int i = 0; i < B::F; ++i)
#pragma unroll
            for (int r = 0; r < N; ++r)
            {
                y[i][r] = z[i][r / 4][r % 4];
                asm volatile("" : "+v"(y[i][r]));
            }
    }

    template<int M>
    __device__ __forceinline__ void inner_modes(float *lds, int t) const
    {
        if constexpr (M > 0)
        {
            constexpr int ST = ipow(N, D - 1 - M);
            constexpr int STEP = B::template step<ST>();
            float y[B::F][N];
            contract<M>(lds, t, y);
#pragma unroll
            for (int i = 0; i < B::F; ++i)
            {
                float *p = lds + B::pa(B::template fiber<ST>(t, i));
                if (B::active(t, i))
#pragma unroll
                    for (int r = 0; r < N; ++r) p[r * STEP] = y[i][r];
            }
            kronreg::lds_barrier();
            inner_modes<M - 1>(lds, t);
        }
    }
};

// Whole entries of n^D elements. A workgroup walks a run of epw entries and keeps the sum of consecutive entries with
// one output in registers, in the layout of mode 0's fibers (coalesced).
template<typename T, int N, int D, int P>
__global__ void __launch_bounds__(P)
    kron_block_kernel(int nb, int epw, T const *const *__restrict__ mats, int stride, T const *const *__restrict__ in,
                      T *const *__restrict__ out)
{
    using B = Block<T, N, D, 1, P>;
    __shared__ __attribute__((aligned(16))) T lds[B::LDS];
    constexpr int ST = ipow(N, D - 1);
    int const t = threadIdx.x;
    int const e0 = kronreg::xcd_run_begin(epw, nb);
    int const e1 = kronruns::end(e0, epw, nb);
    if (e0 >= e1) return;
    B b;
    T acc[B::F][N];
#pragma unroll
    for (int i = 0; i < B::F; ++i)
#pragma unroll
        for (int r = 0; r < N; ++r) acc[i][r] = T(0);
    T *cur = out[e0];
    auto flush = [&]() {
        kronreg::global_ptr<T> dst = kronreg::as_global(cur);
#pragma unroll
        for (int i = 0; i < B::F; ++i)
        {
            int const o = B::template fiber<ST>(t, i);
            if (B::active(t, i))
#pragma unroll
                for (int r = 0; r < N; ++r) atomicAdd((T *)(dst + o + r * ST), acc[i][r]);
#pragma unroll
            for (int r = 0; r < N; ++r) acc[i][r] = T(0);
        }
    };
    int const last = e1 - 1;
    if constexpr (lane_factors<T, N, D, P>())
    {
        using LC = LaneCols<B, N, D>;
        int const lane = t & 63;
        T const *A[D];
        auto address = [&](int e) {
#pragma unroll
            for (int m = 0; m < D; ++m) A[m] = mats[static_cast<size_t>(e < last ? e : last) * D + m];
        };
        LC now, then;
        address(e0);
        now.load(A, stride, lane);
        address(e0 + 1);
        b.load(in[e0], t);
        for (int e = e0; e < e1; ++e)
        {
            T *const dst = out[e];
            if (dst != cur)
            {
                flush();
                cur = dst;
            }
            kronreg::lds_barrier();  // LDS free: every thread has read mode 0's fibers
            b.store(lds, t);
            kronreg::lds_barrier();
            then.load(A, stride, lane);
            address(e + 2);
            if (e < last) b.load(in[e + 1], t);
            now.template inner_modes<D - 1>(lds, t);
            T y[B::F][N];
            now.template contract<0>(lds, t, y);
#pragma unroll
            for (int i = 0; i < B::F; ++i)
#pragma unroll
                for (int r = 0; r < N; ++r) acc[i][r] += y[i][r];
            now = then;
        }
        flush();
        return;
    }
    else
    {
        Touch<T, N, D, P> touch;
        touch.init(mats, e0 < last ? e0 + 1 : last, t);
        b.load(in[e0], t);
        T const *A[D];
#pragma unroll
        for (int m = 0; m < D; ++m) A[m] = mats[static_cast<size_t>(e0) * D + m];
        typename B::Cols cols;
        cols.load(A[D - 1], stride);
        for (int e = e0; e < e1; ++e)
        {
            T *const dst = out[e];
            if (dst != cur)
            {
                flush();
                cur = dst;
            }
            kronreg::lds_barrier();  // LDS free: every thread has read mode 0's fibers
            b.store(lds, t);
            kronreg::lds_barrier();
            int const en = e < last ? e + 1 : last;
            T const *An[D];
#pragma unroll
            for (int m = 0; m < D; ++m) An[m] = mats[static_cast<size_t>(en) * D + m];
            touch.next(mats, en < last ? en + 1 : last, stride, t);
            if (e < last) b.load(in[en], t);
            B::template inner_modes<D - 1>(lds, cols, A, stride, t);
            T y[B::F][N];
            B::template contract<ST>(lds, cols, A[0], stride, t, y);
            cols.load(An[D - 1], stride);
#pragma unroll
            for (int i = 0; i < B::F; ++i)
#pragma unroll
                for (int r = 0; r < N; ++r) acc[i][r] += y[i][r];
#pragma unroll
            for (int m = 0; m < D; ++m) A[m] = An[m];
        }
        flush();
    }
}

// The fastest G modes of every entry: block s of entry e from in[e] to ws[e] (`items` blocks, per_entry of them in an
// entry, `run` consecutive ones per workgroup).
template<typename T, int N, int G, int Q, int P>
__global__ void __launch_bounds__(P)
    kron_block_pass_kernel(int items, int per_entry, int run, int d, T const *const *__restrict__ mats, int stride,
                           T const *const *__restrict__ in, T *const *__restrict__ ws)
{
    using B = Block<T, N, G, Q, P>;
    __shared__ __attribute__((aligned(16))) T lds[B::LDS];
    constexpr int ST = ipow(N, G - 1);
    int const t = threadIdx.x;
    int const w0 = kronreg::xcd_run_begin(run, items);
    int const w1 = kronruns::end(w0, run, items);
    if (w0 >= w1) return;
    B b;
    int e = w0 / per_entry, s = w0 - e * per_entry;
    b.load(in[e] + static_cast<size_t>(s) * B::S, t);
    T const *A[G];
#pragma unroll
    for (int m = 0; m < G; ++m) A[m] = mats[static_cast<size_t>(e) * d + (d - G) + m];
    typename B::Cols cols;
    cols.load(A[G - 1], stride);
    for (int w = w0; w < w1; ++w)
    {
        kronreg::lds_barrier();
        b.store(lds, t);
        kronreg::lds_barrier();
        int en = e, sn = s + 1;
        if (sn == per_entry)
        {
            sn = 0;
            ++en;
        }
        if (w + 1 < w1) b.load(in[en] + static_cast<size_t>(sn) * B::S, t);
        B::template inner_modes<G - 1>(lds, cols, A, stride, t);
        T y[B::F][N];
        B::template contract<ST>(lds, cols, A[0], stride, t, y);
        if (w + 1 < w1)
        {
#pragma unroll
            for (int m = 0; m < G; ++m) A[m] = mats[static_cast<size_t>(en) * d + (d - G) + m];
            cols.load(A[G - 1], stride);
        }
        kronreg::global_ptr<T> dst = kronreg::as_global(ws[e] + static_cast<size_t>(s) * B::S);
#pragma unroll
        for (int i = 0; i < B::F; ++i)
        {
            int const o = B::template fiber<ST>(t, i);
            if (B::active(t, i))
#pragma unroll
                for (int r = 0; r < N; ++r) dst[o + r * ST] = y[i][r];
        }
        e = en;
        s = sn;
    }
}

// ---- the shapes ------------------------------------------------------------------------------------------
// Whole entries, as X(D, N): the (d, n) of the reference's grid (d <= 6, n <= 10) whose vector stays on chip and
// that no other kernel takes by default.
#define KRON_BLOCK_SHAPES(X)                                                                                        \
    X(3, 9) X(3, 10) X(4, 6) X(4, 7) X(4, 9) X(4, 10) X(5, 5) X(5, 6) X(6, 3) X(6, 5)
// d=6 n=5 FP64 (125 KB) and d=4 n=10 FP64 (80 KB) take a workspace like every vector above 64 KB; the second
// still fits a workgroup's LDS, with one workgroup of 16 wavefronts per CU.
template<typename T>
constexpr bool block_shape(int d, int n)
{
    if (d == 6 && n == 5) return sizeof(T) == 4;
#define KRON_BLOCK_IS(D, N) \
    if (d == D && n == N) return true;
    KRON_BLOCK_SHAPES(KRON_BLOCK_IS)
#undef KRON_BLOCK_IS
    return false;
}

// Workgroup size: one fiber per thread, or as many as 1024 threads leave (d=5 n=5 FP64: 640 threads 45.8 us, 512
// with two fibers each 50.3, 256 with three 50.6; d=4 n=7 FP32: 384 29.7, 192 31.3).
template<int N, int D>
constexpr int block_threads()
{
    constexpr int nfib = ipow(N, D - 1);
    constexpr int per = (nfib + 1023) / 1024;
    return ((nfib + per - 1) / per + 63) / 64 * 64;
}

// Larger vectors, d = 5 or 6: this kernel takes the d - 2 fastest modes in blocks of n^4 elements.
template<typename T>
constexpr bool pass_shape(int d, int n)
{
    return (d == 6 && n == 5 && sizeof(T) == 8) || (d == 5 && n >= 7 && n <= 10) || (d == 6 && n >= 6 && n <= 10);
}

// Workgroup size of the pass. Rates (read and written, TB/s) measured with 2 GB of input, d = 6: n=5 FP64 64 threads
// 5.4 (128: 4.8); n=6 FP64 128 5.2 (256: 4.2), FP32 64 5.6 (128: 5.3); n=7 FP64 192 4.3 (384: 4.2), FP32 128 5.0
// (192: 4.7); n=8 FP64 512 4.6 (256: 3.9), FP32 256 5.2 (512: 4.6); n=9 768 4.6 / 4.4 (FP32 384: 3.9); n=10 FP64
// 1024 4.5 (512: 1.7, the columns that do not fit are read again per fiber), FP32 512 4.5 (1024: 3.9).
template<typename T, int N>
constexpr int pass_threads()
{
    bool const f64 = sizeof(T) == 8;
    return N == 5 ? 64 : N == 6 ? (f64 ? 128 : 64) : N == 7 ? (f64 ? 192 : 128) : N == 8 ? (f64 ? 512 : 256)
         : N == 9 ? 768 : (f64 ? 1024 : 512);
}

// Blocks per workgroup: one where several workgroups share a CU and hide each other's start (up to 256 threads), else
// workgroups of 128 wavefronts in total per CU, which read ahead (n=8 FP64: 16 workgroups per CU 4.7 TB/s, 8 4.5, with
// one block per workgroup 3.6; n=10 FP64 25 entries: 8 per CU 194 us, 16 210).
constexpr int kPassOneBlockThreads = 256;
constexpr int kPassWavesPerCu = 128;

} // namespace kronblock
