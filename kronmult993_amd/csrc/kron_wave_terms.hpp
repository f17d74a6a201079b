// kron_wave_terms.hpp -- d = 6, n = 4 in FP32, mostly for several Kronecker terms: one wavefront per entry, 64 values
// per lane.
//
// The tensor's rows are the 64 settings of modes 0-2, its columns those of modes 3-5. A lane holds one row, contracts
// modes 5, 4, 3 in its registers, hands its row to the columns' lanes through LDS, and contracts modes 2, 1, 0. The
// products are LaneFactors' (kron_reg.hpp), k by k from zero as everywhere (kronmult_gpu/kronmult.cu:66-70), so
// each term's contribution is the other kernels' bit for bit. With 256 threads and 16 values each (kron_reg.hpp) a
// sweep needs two exchanges and four barriers; here it needs one exchange inside the wavefront and none.
//
// LDS: a row of 64 values is sixteen 16-byte granules, granule g of row r at g ^ (r & 15). The input is staged in
// canonical order. In the exchange, mode 3 is the fastest of a row: a lane's results of that mode lie in four
// consecutive registers, so a granule is stored as it was produced, and lane (k3, k4, k5) finds its values at granule
// 4 k4 + k5, word k3. All four access patterns are free of bank conflicts. The next entry's input is loaded into the
// registers of this one's once the last term has consumed them.
//
// Four wavefronts share a workgroup only to add the sums that they end with, where those go to one output, before the
// atomics.
//
// What bounds it: latency, with two wavefronts per SIMD (64 input values, 64 working values and 64 sums per lane); the
// matrix cores take 36 us of 24576 sweeps at their measured 135 TFLOP/s. Measured against 256 threads per entry: 8192
// entries of a 128 x 64 operator, 3 terms 70.6 -> 56.1 us, 2 terms 52.9 -> 41.5; 2048 entries, 3 terms 28.6 -> 22.2.
// Few entries, and outputs that are not shared, are faster with 256 threads (figures at the dispatch).
#pragma once

#include <hip/hip_runtime.h>

#include "kron_plan.hpp"
#include "kron_reg.hpp"

namespace kronwaveterms
{

using PL = kronplan::Plan<6, 4, 3>;  // 64 threads, 64 values each
using LF = kronreg::LaneFactors<PL>;
using kronreg::Quad;

constexpr int kWaves = 4;
constexpr int kWavesPerCu = 8;

// LDS accesses of this wavefront's lanes to each other's values: in order in hardware, kept in order by the compiler
__device__ __forceinline__ void exchange_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

__device__ __forceinline__ int granule(int row, int g)
{
    return (row * 16 + (g ^ (row & 15))) * 4;
}

// The lane index made opaque: the addresses formed from it are formed at the accesses instead of being kept in
// registers across the entries.
__device__ __forceinline__ int here(int lane)
{
    asm volatile("" : "+v"(lane));
    return lane;
}

__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
    kron_wave_terms_kernel(int nb, int nterm, int run, float const *const *__restrict__ mats, int stride,
                           float const *const *__restrict__ in, float *const *__restrict__ out)
{
    __shared__ __attribute__((aligned(16))) float all[kWaves][PL::SIZE];
    __shared__ float *last[kWaves];
    int const lane = threadIdx.x & 63;
    int const wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    int const first = kronreg::xcd_run_begin(static_cast<long>(run) * kWaves, nb);
    if (first >= nb) return;
    float *const lds = all[wave];
    int const e0 = first + kronruns::begin(wave, run, nb - first);
    int const e1 = kronruns::end(e0, run, nb);

    float acc[64];
#pragma unroll
    for (int j = 0; j < 64; ++j) acc[j] = 0.f;
    float *cur = nullptr;
    if (e0 < e1)
    {
        auto factors = [&](int term, int e) { return mats + (static_cast<size_t>(term) * nb + e) * PL::kD; };
        LF now, then;
        typename LF::Next next;
        int se = e0, st = 0;  // the sweep whose factor addresses are in `next`
        auto advance = [&]() {
            if (++st == nterm)
            {
                st = 0;
                se = se + 1 < e1 ? se + 1 : se;
            }
        };
        next.address(factors(0, e0), lane);
        next.load(now.a, stride, lane);
        advance();
        next.address(factors(st, se), lane);
        float x[64];
        kronreg::load_input<float, PL>(in[e0], x, lane);
        cur = out[e0];
        for (int e = e0; e < e1; ++e)
        {
            float *dst = out[e];
            if (dst != cur)
            {
                kronreg::flush<float, PL>(cur, acc, here(lane));
                cur = dst;
            }
            int l = here(lane);
#pragma unroll
            for (int c = 0; c < 16; ++c)
                *reinterpret_cast<Quad *>(lds + granule(c * 4 + (l >> 4), l & 15)) =
                    Quad{x[4 * c], x[4 * c + 1], x[4 * c + 2], x[4 * c + 3]};
            exchange_fence();
            l = here(lane);
#pragma unroll
            for (int q = 0; q < 16; ++q)
            {
                Quad const g = *reinterpret_cast<Quad const *>(lds + granule(l, q));
#pragma unroll
                for (int i = 0; i < 4; ++i) x[4 * q + i] = g[i];
            }
            exchange_fence();
            for (int term = 0; term < nterm; ++term)
            {
                next.load(then.a, stride, lane);
                advance();
                next.address(factors(st, se), lane);
                float v[64];
#pragma unroll
                for (int j = 0; j < 64; ++j) v[j] = x[j];
                now.template contract<5, 64, 1>(v);
                now.template contract<4, 64, 4>(v);
                now.template contract<3, 64, 16>(v);
                l = here(lane);
#pragma unroll
                for (int q = 0; q < 16; ++q)
                    *reinterpret_cast<Quad *>(lds + granule(l, q)) = Quad{v[q], v[q + 16], v[q + 32], v[q + 48]};
                exchange_fence();
                if (term + 1 == nterm && e + 1 < e1) kronreg::load_input<float, PL>(in[e + 1], x, here(lane));
                l = here(lane);
#pragma unroll
                for (int j = 0; j < 64; ++j) v[j] = lds[granule(j, l & 15) + (l >> 4)];
                exchange_fence();
                now.template contract<2, 64, 1>(v);
                now.template contract<1, 64, 4>(v);
                now.template contract<0, 64, 16>(v);
#pragma unroll
                for (int j = 0; j < 64; ++j) acc[j] += v[j];
                now = then;
            }
        }
    }
    // The wavefronts' last sums: those of neighbours with one output are added in LDS first. Each wavefront takes a
    // quarter of the elements.
    if (lane == 0) last[wave] = cur;
#pragma unroll
    for (int j = 0; j < 64; ++j) lds[j * 64 + lane] = acc[j];
    __syncthreads();
    float *dst[kWaves];
    unsigned ends = 0;  // bit w: the sum of an output ends with wavefront w
#pragma unroll
    for (int w = 0; w < kWaves; ++w) dst[w] = last[w];
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
        if (dst[w] != nullptr && (w + 1 == kWaves || dst[w + 1] != dst[w])) ends |= 1u << w;
    ends = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(ends)));
    constexpr int kPart = 64 / kWaves;
    float part[kWaves][kPart];
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
#pragma unroll
        for (int i = 0; i < kPart; ++i) part[w][i] = all[w][(wave * kPart + i) * 64 + lane];
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
    {
        if (ends >> w & 1)
        {
            kronreg::global_ptr<float> p = kronreg::as_global(dst[w]) + wave * kPart * 64 + lane;
#pragma unroll
            for (int i = 0; i < kPart; ++i) atomicAdd((float *)(p + i * 64), part[w][i]);
        }
        else if (w + 1 < kWaves)
        {
#pragma unroll
            for (int i = 0; i < kPart; ++i) part[w + 1][i] += part[w][i];
        }
    }
}

} // namespace kronwaveterms
