// kron_reg_adjoint2.hpp -- adjoint on the two-modes-per-phase layout of the d = 6, n = 4 forward sweep
// (kron_plan.hpp Plan<6, 4, 2>: 256 threads, 16 values per thread; phase 0 holds modes 4, 5 in registers,
// phase 1 modes 2, 3, phase 2 modes 0, 1).
//
// Same mathematics as kron_reg_adjoint.hpp: d x = H_6 with H_0 = g, H_{t+1} = A_t^T on mode t of H_t, and
// dA_t = sum over the fibers of mode t of h_f x_f^T with X_t = (A_{t+1} .. A_5 on their modes) x. Per entry:
//   * X chain: x is read from the input in the phase-0 layout (each thread 16 consecutive elements),
//     modes 5, 4 contracted, exchanged through LDS into phase 1, modes 3, 2, into phase 2: X_1 is kept,
//     mode 1 contracted: X_0;
//   * H chain, phase 2: g read in the phase-2 layout (elements j * 256 + t, coalesced); dA_0 from (H_0,
//     X_0), A_0^T, dA_1 from (H_1, X_1), A_1^T, exchange into phase 1;
//   * X_3 kept from the first pass (below), X_2 = A_3 X_3, dA_2, A_2^T, dA_3, A_3^T, exchange into phase 0;
//     X_5 = x (read again) and X_4 (kept in FP32, A_5 x in FP64), dA_4, A_4^T, dA_5, A_5^T: d x in the
//     phase-0 layout.
// The entries are walked by input (kron_order.hpp). A factor gradient's per-thread partial (16 values: its 4 fibers of
// the mode) is reduce-scattered across the wavefront in four steps (kron_lanes.hpp) to one value per lane and summed over consecutive entries that
// share the gradient pointer; when the pointer changes, two more steps, a sum over the four wavefronts in
// LDS after the next exchange's barrier and 16 atomics. d x is summed over entries that share the input gradient and leaves through one LDS
// exchange into the coalesced phase-2 layout.
//
// What bounds it: two workgroups per CU (250 registers, 66 KB of LDS in FP64) hide little of the chains' latency; the
// FMAs of a batch take 68 us. d=6 n=4, 128 x 64 pairs listed by output, FP64 / FP32: 250 / 141 us in the natural order
// (33.5 M input-gradient atomics), 195 walked by input with the sums across lanes in the vector ALU, 189 / 112 with x
// staged by LDS-DMA and the gradients' flush behind the exchanges' barriers, 172 / 101 with the period guessed instead of
// searched for; the input gradient alone 50 / 37 us, the factor gradients alone 164 / 95.
#pragma once

#include <hip/hip_runtime.h>

#include "kron_lanes.hpp"
#include "kron_order.hpp"
#include "kron_reg.hpp"

namespace kronregadj2
{

using kronreg::as_constant;
using kronreg::as_global;
using kronreg::constant_ptr;
using kronreg::global_ptr;
using kronreg::lds_barrier;

using PL = kronplan::Plan<6, 4, 2>;
constexpr int kR = PL::R;  // 16
constexpr int kP = PL::P;  // 256
constexpr int kWaves = kP / 64;

// phase holding mode m in registers, and the stride of m in the register index
constexpr int phase_of(int m) { return m >= 4 ? 0 : m >= 2 ? 1 : 2; }
constexpr int stride_of(int m) { return PL::reg_stride(m - PL::lo(phase_of(m))); }

// contract register mode M with A_M (TRANS: A_M^T); the n-term fused chain, k ascending
template<typename T, int M, bool TRANS>
__device__ __forceinline__ void contract(T (&v)[kR], T const *A_generic, int stride)
{
    constexpr int S = stride_of(M);
    constant_ptr<T> A = as_constant(A_generic);
    T a[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int k = 0; k < 4; ++k) a[r][k] = TRANS ? A[k + r * stride] : A[r + k * stride];
#pragma unroll
    for (int base = 0; base < kR; ++base)
    {
        if ((base / S) % 4 != 0) continue;
        T x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = v[base + k * S];
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            T acc = T(0);
#pragma unroll
            for (int k = 0; k < 4; ++k) acc = fma(x[k], a[r][k], acc);
            v[base + r * S] = acc;
        }
    }
}

// This thread's partial of dA_M, p[4 r + c] = sum over its 4 fibers f of h[f][r] x[f][c], reduce-scattered
// across the wavefront: after step s (lane bit 5 - s) a lane keeps the half of its values selected by that
// bit, summed with the partner lane's copy of the same half. Lane l ends with value index
// 8 b5 + 4 b4 + 2 b3 + b2 (bits of l), summed over the 16 lanes that share its bits 0..1. The first step is
// fused with the partial (values k and k + 8 formed together and folded at once, so the 16 are never live
// together).
template<typename T, int M>
__device__ __forceinline__ void partial_half(T const (&h)[kR], T const (&x)[kR], T (&q8)[8], int lane)
{
    constexpr int S = stride_of(M);
    constexpr int O = S == 4 ? 1 : 4;
#pragma unroll
    for (int k = 0; k < 8; ++k)
    {
        T lo = T(0), hi = T(0);
        int const r0 = k >> 2, c0 = k & 3, r1 = (k + 8) >> 2, c1 = (k + 8) & 3;
#pragma unroll
        for (int f = 0; f < 4; ++f)
        {
            lo = fma(h[r0 * S + f * O], x[c0 * S + f * O], lo);
            hi = fma(h[r1 * S + f * O], x[c1 * S + f * O], hi);
        }
        q8[k] = kronlanes::fold<32>(lo, hi, lane);
    }
}

template<typename T>
__device__ __forceinline__ T reduce_scatter8(T (&q8)[8], int lane)
{
    T q4[4], q2[2];
#pragma unroll
    for (int k = 0; k < 4; ++k) q4[k] = kronlanes::fold<16>(q8[k], q8[k + 4], lane);
#pragma unroll
    for (int k = 0; k < 2; ++k) q2[k] = kronlanes::fold<8>(q4[k], q4[k + 2], lane);
    return kronlanes::fold<4>(q2[0], q2[1], lane);
}

// A run's dA_M partial (one value per lane, in the order above; lanes 0..3 of each quad hold partials of one index) into
// its wavefront's row of red, index 4 r + c.
template<typename T, int M>
__device__ __forceinline__ void publish_gradient(T value, T *red, int t)
{
    int const lane = t & 63, wave = t >> 6;
    value = kronlanes::add<1>(value);
    value = kronlanes::add<2>(value);
    int const idx = ((lane >> 5) & 1) * 8 + ((lane >> 4) & 1) * 4 + ((lane >> 3) & 1) * 2 + ((lane >> 2) & 1);
    if ((lane & 3) == 0) red[(M * kWaves + wave) * 16 + idx] = value;
}

// The published gradients of the modes in `mask`, after a barrier: 16 threads per mode add the four wavefronts' rows and
// make one atomic each. The barrier is the one of the exchange that follows; the rows are written again only in the
// next entry, several barriers later. (With two barriers of its own per gradient, the d=6 batch took 195 us.)
template<typename T>
__device__ __forceinline__ void flush_gradients(unsigned mask, T *const *gA, int stride, T const *red, int t)
{
    int const m = t >> 4, i = t & 15;
    if (m < 6 && ((mask >> m) & 1u))
    {
        T s = red[m * kWaves * 16 + i];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) s += red[(m * kWaves + w) * 16 + i];
        global_ptr<T> g = as_global(gA[m]);
        atomicAdd((T *)(g + (i >> 2) + (i & 3) * stride), s);  // index 4 r + c: dA[r][c]
    }
}

// exchange the vector from the layout of phase A to that of phase B through LDS (the forward's exchange
// swizzle on both sides); between: what every thread does after the first barrier
template<typename T, int A, int B, typename F = kronreg::NoHook>
__device__ __forceinline__ void exchange(T *lds, T (&v)[kR], int t, F const &between = F())
{
    using SW = kronplan::PlanSwizzle<PL, T, 1>;
    lds_barrier();
    between();
#pragma unroll
    for (int j = 0; j < kR; ++j) lds[SW::phys(PL::elem(A, t, j))] = v[j];
    lds_barrier();
#pragma unroll
    for (int j = 0; j < kR; ++j) v[j] = lds[SW::phys(PL::elem(B, t, j))];
}

// x in the phase-0 layout: thread t holds elements 16 t .. 16 t + 15
template<typename T>
__device__ __forceinline__ void load_x(T const *src_generic, T (&v)[kR], int t)
{
    static_assert(PL::L(0) == 1, "phase 0 holds 16 consecutive elements per thread");
    global_ptr<T const> src = as_global(src_generic);
#pragma unroll
    for (int j = 0; j < kR; ++j) v[j] = src[t * kR + j];
}

// X_3 (phase-1 layout) and, in FP32, X_4 (phase-0 layout) are kept from the first pass of the X chain in
// thread-private LDS slots (element j * P + t of the buffer: each thread reads back only what it wrote, so
// no barrier) instead of being rebuilt from x; FP64 keeps X_3 only, as 64 KiB of LDS per workgroup already
// matches its two resident workgroups per CU (223 VGPRs).
template<typename T>
constexpr bool keep_x4()
{
    return sizeof(T) == 4;
}

template<typename T>
__device__ __forceinline__ void keep(T *buf, T const (&v)[kR], int t)
{
#pragma unroll
    for (int j = 0; j < kR; ++j) buf[j * kP + t] = v[j];
}
template<typename T>
__device__ __forceinline__ void restore(T const *buf, T (&v)[kR], int t)
{
#pragma unroll
    for (int j = 0; j < kR; ++j) v[j] = buf[j * kP + t];
}

// FP64: x goes through LDS, by LDS-DMA in the swizzled order of the forward sweep's staging (kron_reg.hpp), into the
// buffer that X_3 has left; there it serves X_5 and, when the next entry has the same input (the walk by input), the
// next X chain. Read straight from memory in the phase-0 layout, 16 consecutive values per thread, every load
// instruction touches 64 lines, twice per entry.
template<typename T>
constexpr bool stage_x_ok()
{
    return sizeof(T) == 8 && kronreg::Lds<T, PL>::dma_ok();
}

template<typename T>
__device__ __forceinline__ void stage_x(T *buf, T const *src, int t)
{
    if ((reinterpret_cast<uintptr_t>(src) & 15) == 0)
        kronreg::Lds<T, PL>::dma_input(buf, src, t);
    else
    {
        T tmp[kR];
        kronreg::load_input<T, PL>(src, tmp, t);
        kronreg::Lds<T, PL>::store_input(buf, tmp, t);
    }
}
__device__ __forceinline__ void stage_wait()
{
    __builtin_amdgcn_s_waitcnt(kronreg::kWaitVmcnt0);  // this wavefront's LDS-DMA loads have landed
}

// MATS: with the factors' gradients (without them only the H chain is left, in 32 KB of LDS and half the registers)
template<typename T, bool MATS>
__global__ void __launch_bounds__(kP)
    kron_reg_adjoint2_kernel(int nb, T const *const *__restrict__ mats, int stride,
                             T const *const *__restrict__ in, T const *const *__restrict__ gout,
                             T *const *__restrict__ gin, T *const *__restrict__ gmats)
{
    static_assert(PL::NPHASE == 3 && PL::elem(2, 1, 0) == 1 && PL::elem(2, 0, 1) == kP,
                  "phase 2 is element j * P + t");
    constexpr bool kKeep4 = keep_x4<T>();
    constexpr bool kStageX = stage_x_ok<T>();
    using L = kronreg::Lds<T, PL>;
    __shared__ __attribute__((aligned(16))) T lds[PL::SIZE * (MATS ? 2 + (kKeep4 ? 1 : 0) : 1)];
    __shared__ T red[MATS ? 6 * kWaves * 16 : 1];
    T *const x3buf = lds + (MATS ? 1 : 0) * PL::SIZE;
    T *const x4buf = lds + (MATS ? 2 : 0) * PL::SIZE;
    int const t = threadIdx.x;
    int const lane = t & 63;
    kronorder::Walk walk = kronorder::walk(gin, nb, static_cast<int>(gridDim.x), PL::SIZE);
    int e = walk.next();
    if (e < 0) return;
    constexpr bool want_mats = MATS;
    bool const want_input = gin != nullptr;

    T gacc[6], dxacc[kR];
#pragma unroll
    for (int m = 0; m < 6; ++m) gacc[m] = T(0);
#pragma unroll
    for (int j = 0; j < kR; ++j) dxacc[j] = T(0);

    // FP64: the next entry's cotangent is loaded while this entry runs (248 registers, still two waves per
    // SIMD; d=6 batch 273 -> 263 us). FP32 gains nothing from it (its three waves per SIMD hide the load),
    // and prefetching the input as well takes it to 180 registers and two waves (146 -> 161 us).
    constexpr bool kPreG = sizeof(T) == 8;
    T gpre[kPreG ? kR : 1];
    auto load_g = [&](int e, T (&dst)[kR]) {
        global_ptr<T const> g = as_global(gout[e]);
#pragma unroll
        for (int j = 0; j < kR; ++j) dst[j] = g[j * kP + t];
    };
    if constexpr (kPreG) load_g(e, gpre);

    unsigned pending = 0;  // modes whose gradients (of entry pending_from) are published and not yet added
    int pending_from = 0;
    T const *staged = nullptr;  // the input held in the X_3 buffer (kStageX)
    int en = -1;  // the entry after e
    for (; e >= 0; e = en)
    {
        en = walk.next();
        bool const last = en < 0;
        T const *const *A = mats + static_cast<size_t>(e) * 6;
        T h[kR], v[kR], xs[kR];
        // one dA step: partial of mode M from (h, x), run sum, published when the next entry's pointer differs
        auto grad = [&](auto mc, T const (&x)[kR]) {
            constexpr int M = decltype(mc)::value;
            T q8[8];
            partial_half<T, M>(h, x, q8, lane);
            gacc[M] += reduce_scatter8(q8, lane);
            T *const gA = gmats[static_cast<size_t>(e) * 6 + M];
            if (last || gmats[static_cast<size_t>(en) * 6 + M] != gA)
            {
                publish_gradient<T, M>(gacc[M], red, t);
                gacc[M] = T(0);
                pending |= 1u << M;
                pending_from = e;
            }
        };
        auto flush = [&]() {
            if (MATS && pending != 0)
                flush_gradients(pending, gmats + static_cast<size_t>(pending_from) * 6, stride, red, t);
            pending = 0;
        };
        // cotangent in the phase-2 layout: element j * 256 + t
        if constexpr (kPreG)
        {
#pragma unroll
            for (int j = 0; j < kR; ++j) h[j] = gpre[j];
            if (!last) load_g(en, gpre);
        }
        else
            load_g(e, h);
        if constexpr (want_mats)
        {
            if constexpr (kStageX)
            {
                if (staged != in[e])
                {
                    lds_barrier();  // every thread is done with the buffer
                    stage_x(x3buf, in[e], t);
                    staged = in[e];
                    stage_wait();
                    lds_barrier();
                }
                L::read0_dma(x3buf, v, t);
            }
            else
                load_x(in[e], v, t);
            contract<T, 5, false>(v, A[5], stride);
            if constexpr (kKeep4) keep(x4buf, v, t);  // X_4
            contract<T, 4, false>(v, A[4], stride);
            exchange<T, 0, 1>(lds, v, t, flush);  // (the previous entry's dA_4, dA_5)
            keep(x3buf, v, t);   // X_3
            contract<T, 3, false>(v, A[3], stride);
            contract<T, 2, false>(v, A[2], stride);
            exchange<T, 1, 2>(lds, v, t);
#pragma unroll
            for (int j = 0; j < kR; ++j) xs[j] = v[j];  // X_1
            contract<T, 1, false>(v, A[1], stride);      // X_0
            grad(std::integral_constant<int, 0>(), v);
        }
        contract<T, 0, true>(h, A[0], stride);  // H_1
        if constexpr (want_mats) grad(std::integral_constant<int, 1>(), xs);
        contract<T, 1, true>(h, A[1], stride);  // H_2
        exchange<T, 2, 1>(lds, h, t, flush);  // dA_0, dA_1
        if constexpr (want_mats)
        {
            restore(x3buf, v, t);
#pragma unroll
            for (int j = 0; j < kR; ++j) xs[j] = v[j];  // X_3
            contract<T, 3, false>(v, A[3], stride);      // X_2
            grad(std::integral_constant<int, 2>(), v);
        }
        contract<T, 2, true>(h, A[2], stride);  // H_3
        if constexpr (want_mats) grad(std::integral_constant<int, 3>(), xs);
        contract<T, 3, true>(h, A[3], stride);  // H_4
        exchange<T, 1, 0>(lds, h, t, [&]() {
            flush();  // dA_2, dA_3
            // every thread has read X_3: x into its buffer, for X_5 and for the next entry if it has the same input
            if constexpr (kStageX)
                if (want_mats) stage_x(x3buf, in[e], t);
        });
        if constexpr (want_mats)
        {
            if constexpr (kStageX)
            {
                stage_wait();
                lds_barrier();
                L::read0_dma(x3buf, xs, t);  // X_5
            }
            else
                load_x(in[e], xs, t);
            if constexpr (kKeep4)
                restore(x4buf, v, t);
            else
            {
#pragma unroll
                for (int j = 0; j < kR; ++j) v[j] = xs[j];
                contract<T, 5, false>(v, A[5], stride);  // X_4
            }
            grad(std::integral_constant<int, 4>(), v);
        }
        contract<T, 4, true>(h, A[4], stride);  // H_5
        if constexpr (want_mats) grad(std::integral_constant<int, 5>(), xs);
        if (want_input)
        {
            contract<T, 5, true>(h, A[5], stride);  // d x, phase-0 layout
#pragma unroll
            for (int j = 0; j < kR; ++j) dxacc[j] += h[j];
            if (last || gin[en] != gin[e])
            {
                exchange<T, 0, 2>(lds, dxacc, t);
                global_ptr<T> gi = as_global(gin[e]);
#pragma unroll
                for (int j = 0; j < kR; ++j)
                {
                    atomicAdd((T *)(gi + j * kP + t), dxacc[j]);
                    dxacc[j] = T(0);
                }
            }
        }
    }
    if (MATS && pending != 0)
    {
        lds_barrier();
        flush_gradients(pending, gmats + static_cast<size_t>(pending_from) * 6, stride, red, t);
    }
}

} // namespace kronregadj2
