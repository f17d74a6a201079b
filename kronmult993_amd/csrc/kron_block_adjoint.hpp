// kron_block_adjoint.hpp -- the adjoint of whole entries on the layout of the block sweep (kron_block.hpp).
//
// Mathematics as in kron_adjoint.hpp. A thread owns one fiber of every mode. Per entry:
//   * X chain: x staged in LDS, modes d-1 .. 1 contracted in place; the fiber of mode t that the thread reads for its
//     step is X_t, and stays in registers (d n values);
//   * H chain: the cotangent is read in the layout of mode 0 (coalesced); for t = 0 .. d-1 the thread holds H_t's and
//     X_t's fiber, forms their n x n products, and contracts with A_t^T; one exchange through LDS per mode;
//   * the products are reduce-scattered across the wavefront (kron_lanes.hpp) to one value per lane, summed over
//     consecutive entries with the same gradient, published in LDS when that changes and added by one thread per
//     value after the next entry's first barrier;
//   * d x leaves through LDS in canonical order, summed over consecutive entries with the same input (which the walk
//     by input brings together, kron_order.hpp), one atomic per element.
// The factors are staged in LDS and read as broadcasts up to 256 threads, else they come through scalar registers
// (kron_block.hpp); everything an entry needs is read one entry ahead, its addresses two.
//
// What bounds it: the chain of an entry (2 d LDS exchanges, d reduce-scatters, about 900 instructions for d=4 n=4), then
// the input gradient's atomics. The general kernel (kron_adjoint.hpp) rebuilds X_t for every t, takes the products on
// matrix instructions with n of 16 rows in use (FP32), and adds every entry's gradients with atomics of their own. 8192
// entries, FP64 / FP32, general kernel -> here: d=4 n=5 with inputs of their own and 256 factor sets 191 -> 72 / 104 ->
// 37 us, as 128 x 64 element pairs 193 -> 75 / 198 -> 56; d=5 n=5 1159 -> 422 / 618 -> 237 (10 wavefronts leave it 168
// registers; the scalar factor columns spill); d=4 n=6 313 -> 248 / 189 -> 96; d=6 n=3 169 -> 87 / 260 -> 51; d=3 n=7
// pairs 125 -> 72 / 243 -> 61; against the register kernel d=5 n=4 110 -> 95 / 61 -> 53, d=4 n=8 FP32 328 -> 274. The
// input gradient alone, inputs of their own, 1100 entries: d=5 n=5 FP64 36.8 -> 29.8, 700 of d=4 n=7 FP32 13.4 -> 11.1.
#pragma once

#include <hip/hip_runtime.h>

#include "kron_block.hpp"
#include "kron_lanes.hpp"
#include "kron_order.hpp"

namespace kronblockadj
{

using kronblock::ipow;

// smallest power of two that is not below v
constexpr int pow2(int v)
{
    int p = 1;
    while (p < v) p *= 2;
    return p;
}

template<typename T, int N, int D, int P>
struct Adj
{
    using B = kronblock::Block<T, N, D, 1, P>;
    static_assert(B::F == 1, "one fiber per thread");
    static constexpr int NN = N * N;
    static constexpr int W = P / 64;
    static constexpr int C0 = pow2(NN) < 2 ? 2 : pow2(NN);  // values of the reduce-scatter, zeros from NN on
    static_assert(C0 <= 64, "one value per lane");
    static constexpr int CE = (B::S + P - 1) / P;   // canonical elements per thread
    static constexpr int RED = W * D * NN;          // published gradients
    // Factors staged in LDS, read as broadcasts, up to four wavefronts; above, the wavefronts' reads of the same
    // values would fill the LDS: scalar registers.
    static constexpr bool kCoefLds = P <= 256;
    static constexpr int GR = B::GR;
    static constexpr int CP = (N + GR - 1) / GR * GR;  // pitch of a staged column
    static constexpr int COEF = kCoefLds ? D * N * CP : 0;
    static constexpr int CPL = kCoefLds ? (D * NN + P - 1) / P : 1;
    // X_1 .. X_{d-1} in thread-private LDS slots where they would not fit the registers
    static constexpr bool kChainLds = P > 256 && sizeof(T) == 8;
    static constexpr int CHAIN = kChainLds ? (D - 1) * N * P : 0;
    static constexpr int PER = (D * NN + P - 1) / P;  // gradient values per thread

    static constexpr int st(int m) { return ipow(N, D - 1 - m); }
    static constexpr int step(int m) { return st(m) == 1 ? 1 : st(m) + B::PAD * (st(m) / N); }

    template<int M>
    static __device__ __forceinline__ void read(T const *lds, int t, T (&v)[N])
    {
        T const *p = lds + B::pa(B::template fiber<st(M)>(t, 0));
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = p[k * step(M)];
        // a thread past the last fiber holds zeros, in x and in the cotangent: its products add nothing, whatever the
        // values of the fiber that it repeats (0 times infinity would not be 0)
        if (!B::active(t, 0))
#pragma unroll
            for (int k = 0; k < N; ++k) v[k] = T(0);
    }
    template<int M>
    static __device__ __forceinline__ void write(T *lds, int t, T const (&v)[N])
    {
        T *p = lds + B::pa(B::template fiber<st(M)>(t, 0));
        if (B::active(t, 0))
#pragma unroll
            for (int k = 0; k < N; ++k) p[k * step(M)] = v[k];
    }

    // y = A x or A^T x (staged factor, or cols: A's first columns)
    template<bool TRANS>
    static __device__ __forceinline__ void apply(T const *staged, typename B::Cols const &cols, T const *A_generic,
                                                 int stride, T const (&x)[N], T (&y)[N])
    {
        kronreg::constant_ptr<T> A = kronreg::as_constant(A_generic);
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            T c[N];
#pragma unroll
            for (int r = 0; r < N; ++r)
            {
                if constexpr (kCoefLds)
                    c[r] = staged[k * CP + r];
                else
                    c[r] = k < B::KP ? cols.c[k < B::KP ? k : 0][r] : A[r + k * stride];
            }
            if constexpr (TRANS)
            {
                T acc = T(0);
#pragma unroll
                for (int r = 0; r < N; ++r) acc = fma(x[r], c[r], acc);
                y[k] = acc;
            }
            else
            {
#pragma unroll
                for (int r = 0; r < N; ++r) y[r] = fma(x[k], c[r], k == 0 ? T(0) : y[r]);
            }
        }
        // complete here, not in the branch on active threads
#pragma unroll
        for (int r = 0; r < N; ++r) asm volatile("" : "+v"(y[r]));
    }

    // one value of the reduce-scatter: lane l gets product number l >> (6 - log2 C0), summed over its wavefront
    template<int BIT, int C, int LIVE>
    static __device__ __forceinline__ T scatter(T (&q)[C0 / 2], int lane)
    {
        if constexpr (BIT == 0)
            return q[0];
        else if constexpr (C > 1)
        {
            constexpr int H = C / 2;
#pragma unroll
            for (int k = 0; k < H; ++k)
                if (k < LIVE) q[k] = kronlanes::fold<BIT>(q[k], k + H < LIVE ? q[k + H < C0 / 2 ? k + H : 0] : T(0), lane);
            return scatter<BIT / 2, H, (LIVE < H ? LIVE : H)>(q, lane);
        }
        else
        {
            q[0] = kronlanes::add<BIT>(q[0]);
            return scatter<BIT / 2, 1, 1>(q, lane);
        }
    }
    static __device__ __forceinline__ T products(T const (&h)[N], T const (&x)[N], int lane)
    {
        constexpr int H = C0 / 2;
        T q[H];
#pragma unroll
        for (int k = 0; k < H; ++k)
            if (k < NN)
                q[k] = kronlanes::fold<32>(h[k / N] * x[k % N],
                                           k + H < NN ? h[(k + H < NN ? k + H : 0) / N] * x[(k + H < NN ? k + H : 0) % N] : T(0),
                                           lane);
        return scatter<16, H, (NN < H ? NN : H)>(q, lane);
    }
    static constexpr int kLaneShift = C0 == 64 ? 0 : C0 == 32 ? 1 : C0 == 16 ? 2 : C0 == 8 ? 3 : C0 == 4 ? 4 : 5;
};

// MATS: with the factors' gradients. Without them the X chain, the products and their registers fall away, so more
// workgroups are resident.
template<typename T, int N, int D, int P, bool MATS>
__global__ void __launch_bounds__(P)
    kron_block_adjoint_kernel(int nb, int groups_shared, T const *const *__restrict__ mats, int stride,
                              T const *const *__restrict__ in, T const *const *__restrict__ gout,
                              T *const *__restrict__ gin, T *const *__restrict__ gmats)
{
    using A = Adj<T, N, D, P>;
    using B = typename A::B;
    constexpr bool kCoefLds = A::kCoefLds;
    constexpr int NN = A::NN;
    __shared__ __attribute__((aligned(16))) T lds[(B::LDS + A::GR - 1) / A::GR * A::GR + A::COEF + (MATS ? A::CHAIN : 0)];
    __shared__ T red[MATS ? A::RED : 1];
    __shared__ T *gptr_shared[D];
    T *const coef = lds + (B::LDS + A::GR - 1) / A::GR * A::GR;
    T *const chain = coef + A::COEF + threadIdx.x;
    int const t = threadIdx.x, lane = t & 63;
    int const wave = __builtin_amdgcn_readfirstlane(t >> 6);
    constexpr bool want_mats = MATS;
    bool const want_input = gin != nullptr;
    int const groups = static_cast<int>(gridDim.x);
    kronorder::Walk walk = kronorder::walk(
        gin, nb, MATS && groups_shared < groups && kronorder::shared_gradients(gmats, nb, D) ? groups_shared : groups, B::S);
    int e = walk.next();
    if (e < 0) return;
    int en = walk.next();

    T gacc[D], dx[A::CE];
#pragma unroll
    for (int m = 0; m < D; ++m) gacc[m] = T(0);
#pragma unroll
    for (int c = 0; c < A::CE; ++c) dx[c] = T(0);

    // Read one entry ahead: x (canonical granules), g (mode 0's fibers), the factors (values for the LDS, or their
    // lines and the first columns); two entries ahead: the addresses of all these, so that no load waits for another.
    // Lane m of every wavefront holds the gradient address of factor m.
    struct Addresses
    {
        T const *x, *g;
        T *gi, *gm;
        T const *f[A::CPL];
    };
    auto addresses = [&](int k) {
        Addresses a;
        a.x = want_mats ? in[k] : nullptr;
        a.g = gout[k];
        a.gi = want_input ? gin[k] : nullptr;
        a.gm = want_mats ? kronreg::as_global(gmats)[static_cast<size_t>(k) * D + (lane < D ? lane : 0)] : nullptr;
        if constexpr (kCoefLds)
        {
#pragma unroll
            for (int c = 0; c < A::CPL; ++c)
            {
                int const i = t + c * P;
                a.f[c] = kronreg::as_global(mats)[static_cast<size_t>(k) * D + (i < D * NN ? i / NN : 0)];
            }
        }
        return a;
    };
    B b;
    T g[N], fv[A::CPL];
    auto load = [&](Addresses const &a) {
        if constexpr (kCoefLds)
        {
#pragma unroll
            for (int c = 0; c < A::CPL; ++c)
            {
                int const i = t + c * P;  // A_m(r, k) at m n^2 + k n + r
                fv[c] = kronreg::as_global(a.f[c])[i < D * NN ? i % N + (i / N) % N * stride : 0];
            }
        }
        if (want_mats) b.load(a.x, t);
        kronreg::global_ptr<T const> src = kronreg::as_global(a.g) + B::template fiber<A::st(0)>(t, 0);
#pragma unroll
        for (int r = 0; r < N; ++r) g[r] = src[r * A::st(0)];
    };
    Addresses cur = addresses(e);
    load(cur);
    Addresses nxt = addresses(en >= 0 ? en : e);
    kronblock::Touch<T, N, D, P> touch;
    T const *F[D];
    typename B::Cols cols;
    if constexpr (!kCoefLds)
    {
        touch.init(mats, en >= 0 ? en : e, t);
#pragma unroll
        for (int m = 0; m < D; ++m) F[m] = mats[static_cast<size_t>(e) * D + m];
        cols.load(F[want_mats ? D - 1 : 0], stride);
    }

    unsigned pending = 0;  // modes whose gradients are published, with their addresses
    auto flush = [&]() {
        if (pending == 0) return;
#pragma unroll
        for (int c = 0; c < A::PER; ++c)
        {
            int const i = t + c * P;
            int const m = i / NN, rc = i % NN;
            if (i < D * NN && ((pending >> m) & 1u))
            {
                T s = red[i];
#pragma unroll
                for (int w = 1; w < A::W; ++w) s += red[w * D * NN + i];
                atomicAdd((T *)(kronreg::as_global(gptr_shared[m]) + rc / N + rc % N * stride), s);
            }
        }
        pending = 0;
    };

    while (e >= 0)
    {
        int const enn = en >= 0 ? walk.next() : -1;
        bool const last = en < 0;
        kronreg::lds_barrier();  // LDS free, the previous entry's gradients published
        flush();
        if (want_mats) b.store(lds, t);
        if constexpr (kCoefLds)
        {
#pragma unroll
            for (int c = 0; c < A::CPL; ++c)
            {
                int const i = t + c * P;
                if (i < D * NN) coef[(i / N) * A::CP + i % N] = fv[c];
            }
        }
        T h[N], X0[N], X[A::kChainLds ? 1 : D][N];
#pragma unroll
        for (int r = 0; r < N; ++r) h[r] = B::active(t, 0) ? g[r] : T(0);
        // modes whose gradient address changes after this entry
        unsigned const change = last ? ~0u : static_cast<unsigned>(__ballot(lane < D && cur.gm != nxt.gm));
        bool const input_changes = last || nxt.gi != cur.gi;
        kronreg::lds_barrier();
        if (want_mats && wave == 0 && lane < D && ((change >> lane) & 1u)) gptr_shared[lane] = cur.gm;
        T const *Fn[D];
        if constexpr (!kCoefLds)
        {
            int const nx = last ? e : en;
#pragma unroll
            for (int m = 0; m < D; ++m) Fn[m] = mats[static_cast<size_t>(nx) * D + m];
            touch.next(mats, enn >= 0 ? enn : nx, stride, t);
        }
        T *const gi = cur.gi;
        if (!last) load(nxt);
        cur = nxt;
        if (enn >= 0) nxt = addresses(enn);

        auto grad = [&](auto mc, T const (&x)[N]) {
            constexpr int M = decltype(mc)::value;
            gacc[M] += A::products(h, x, lane);
            if ((change >> M) & 1u)
            {
                int const idx = lane >> A::kLaneShift;
                if ((lane & ((1 << A::kLaneShift) - 1)) == 0 && idx < NN) red[(wave * D + M) * NN + idx] = gacc[M];
                gacc[M] = T(0);
                pending |= 1u << M;
            }
        };
        // modes D-1 .. 1 of x, then mode 0's fibers
        auto xchain = [&](auto self, auto mc) -> void {
            constexpr int M = decltype(mc)::value;
            if constexpr (M > 0)
            {
                T v[N], y[N];
                A::template read<M>(lds, t, v);
                A::template apply<false>(coef + M * N * A::CP, cols, kCoefLds ? nullptr : F[M], stride, v, y);
                if constexpr (!kCoefLds) cols.load(F[M - 1], stride);
#pragma unroll
                for (int r = 0; r < N; ++r)
                {
                    if constexpr (A::kChainLds)
                        chain[((M - 1) * N + r) * P] = v[r];
                    else
                        X[M][r] = v[r];
                }
                A::template write<M>(lds, t, y);
                kronreg::lds_barrier();
                self(self, std::integral_constant<int, M - 1>());
            }
            else
                A::template read<0>(lds, t, X0);
        };
        // modes M .. D-1 of the cotangent
        auto hchain = [&](auto self, auto mc) -> void {
            constexpr int M = decltype(mc)::value;
            if constexpr (M > 0) A::template read<M>(lds, t, h);
            if constexpr (want_mats)
            {
                if constexpr (M == 0)
                    grad(mc, X0);
                else if constexpr (A::kChainLds)
                {
                    T v[N];
#pragma unroll
                    for (int r = 0; r < N; ++r) v[r] = chain[((M - 1) * N + r) * P];
                    grad(mc, v);
                }
                else
                    grad(mc, X[M]);
            }
            if (M < D - 1 || want_input)
            {
                T y[N];
                A::template apply<true>(coef + M * N * A::CP, cols, kCoefLds ? nullptr : F[M], stride, h, y);
                if constexpr (!kCoefLds && M < D - 1) cols.load(F[M + 1], stride);
                if constexpr (M == 0)
                    if (want_mats) kronreg::lds_barrier();  // every thread has read X_0
                A::template write<M>(lds, t, y);
                kronreg::lds_barrier();
            }
            if constexpr (M < D - 1) self(self, std::integral_constant<int, M + 1>());
        };
        if constexpr (want_mats) xchain(xchain, std::integral_constant<int, D - 1>());
        hchain(hchain, std::integral_constant<int, 0>());
        if constexpr (!kCoefLds)
        {
            cols.load(Fn[want_mats ? D - 1 : 0], stride);
#pragma unroll
            for (int m = 0; m < D; ++m) F[m] = Fn[m];
        }
        if (want_input)
        {
            // What was read ahead has arrived before the atomics are issued: memory operations complete in order, and
            // a wait behind the branch below would be one for the atomics too.
            if (want_mats) b.arrived();
#pragma unroll
            for (int r = 0; r < N; ++r) asm volatile("" : "+v"(g[r]));
            asm volatile("" : "+v"(nxt.gm));
            if constexpr (kCoefLds)
#pragma unroll
                for (int c = 0; c < A::CPL; ++c) asm volatile("" : "+v"(fv[c]), "+v"(nxt.f[c]));
#pragma unroll
            for (int c = 0; c < A::CE; ++c)
            {
                int const i = c * P + t;
                if (B::S % P == 0 || c + 1 < A::CE || i < B::S) dx[c] += lds[B::pa(i)];
            }
            if (input_changes)
            {
                kronreg::global_ptr<T> dst = kronreg::as_global(gi);
#pragma unroll
                for (int c = 0; c < A::CE; ++c)
                {
                    int const i = c * P + t;
                    if (B::S % P == 0 || c + 1 < A::CE || i < B::S) atomicAdd((T *)(dst + i), dx[c]);
                    dx[c] = T(0);
                }
            }
        }
        e = en;
        en = enn;
    }
    kronreg::lds_barrier();
    flush();
}

// The shapes, as X(D, N). FP64 leaves d=3 n=5, d=3 n=6 and d=4 n=3 to the general kernel and d=4 n=8 to the register
// kernel: the line was drawn when the walk's search for the period took about 10 us of every call (8192 entries with
// inputs of their own 37, 50, 27 us here against 36, 45, 22; d=4 n=8 300 entries 36 against 34). Without it they take
// 26, 40, 18 us here, and d=4 n=8 477 against 501 (300 entries 35 against 34).
#define KRON_BLOCK_ADJOINT_SHAPES(X)                                                                                \
    X(3, 5) X(3, 6) X(3, 7) X(4, 3) X(4, 5) X(4, 6) X(4, 7) X(4, 8) X(5, 3) X(5, 4) X(5, 5) X(6, 2) X(6, 3)

template<typename T>
constexpr bool adjoint_shape(int d, int n)
{
    if (sizeof(T) == 8 && ((d == 3 && n < 7) || (d == 4 && (n == 3 || n == 8)))) return false;
#define KRON_BLOCK_ADJOINT_IS(D, N) \
    if (d == D && n == N) return true;
    KRON_BLOCK_ADJOINT_SHAPES(KRON_BLOCK_ADJOINT_IS)
#undef KRON_BLOCK_ADJOINT_IS
    return false;
}

} // namespace kronblockadj
