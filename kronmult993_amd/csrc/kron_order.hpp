// kron_order.hpp -- the order in which the workgroups of an adjoint launch walk the entries.
//
// An entry's input gradient is n^d atomic adds unless the next entry of the run adds to the same vector. A batch listed
// by output (as the forward call wants it) visits the inputs in turn: entry k and entry k + p share an input, their
// neighbours do not. The workgroup therefore looks for the first entry after 0 that shares entry 0's gradient pointer,
// p, and walks the entries k = c, c + p, c + 2p, ... column by column instead of k = 0, 1, 2, ...: every entry once in
// either order, whatever the pointers are, and the sums of shared gradients in registers when they do repeat with that
// period. d=6 n=4, 128 x 64 element pairs listed by output, FP64: 33.5 M atomic adds (about 200 G/s) become 2.1 M.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

#include "kron_reg.hpp"

namespace kronorder
{

constexpr int kScan = 4096;  // pointers looked at (16 loads per thread of a 256-thread workgroup)

struct Walk
{
    int nb, period, rows;  // the entry of column c, row r is c + r * period
    int c, r, left;        // this workgroup's next step and the number of its steps

    // the next entry, or -1 (a step past the batch, in the last row, is left out)
    __device__ __forceinline__ int next()
    {
        while (left > 0)
        {
            unsigned const k = static_cast<unsigned>(c) + static_cast<unsigned>(r) * static_cast<unsigned>(period);
            --left;
            if (++r == rows)
            {
                r = 0;
                ++c;
            }
            if (k < static_cast<unsigned>(nb)) return static_cast<int>(k);
        }
        return -1;
    }
};

// Whether a factor gradient of entry 0 is one of the entries a third and two thirds into the batch too (every wavefront
// finds the same answer; d <= 64).
template<typename T>
__device__ __forceinline__ bool shared_gradients(T *const *gmats, int nb, int d)
{
    if (gmats == nullptr) return false;
    int const lane = static_cast<int>(threadIdx.x) & 63, m = lane < d ? lane : 0;
    T *const first = kronreg::as_global(gmats)[m];
    bool const same = first == kronreg::as_global(gmats)[static_cast<size_t>(nb / 3) * d + m] ||
                      first == kronreg::as_global(gmats)[static_cast<size_t>(nb - 1 - nb / 3) * d + m];
    return __ballot(same) != 0;
}

// This workgroup's part of the batch, cut into `groups` (a multiple of 8, at most the grid) equal parts; the workgroups
// past them get none. ptr may be null (natural order). Every thread calls it.
template<typename T>
__device__ __forceinline__ Walk walk(T *const *ptr, int nb, int groups, int *shared_min)
{
    int period = 1;
    if (ptr != nullptr && nb > groups)
    {
        if (threadIdx.x == 0) *shared_min = INT_MAX;
        __syncthreads();
        T *const first = ptr[0];
        int const limit = nb < kScan ? nb : kScan;
        for (int q = 1 + static_cast<int>(threadIdx.x); q < limit; q += static_cast<int>(blockDim.x))
            if (ptr[q] == first)
            {
                atomicMin(shared_min, q);
                break;
            }
        __syncthreads();
        int const p = __builtin_amdgcn_readfirstlane(*shared_min);
        if (p != INT_MAX) period = p;
    }
    Walk w;
    w.nb = nb;
    w.period = period;
    w.rows = static_cast<int>((static_cast<long>(nb) + period - 1) / period);
    // consecutive parts on one XCD (kronreg::xcd_run_index, over `groups`)
    int const per_xcd = groups >> 3, slot = static_cast<int>(blockIdx.x >> 3);
    long const index = static_cast<long>(blockIdx.x & 7) * per_xcd + slot;
    // the steps, those past the batch among them, in parts that differ by one at most
    long const steps = static_cast<long>(w.rows) * period;
    long const v0 = slot < per_xcd ? index * steps / groups : steps;
    long const v1 = slot < per_xcd ? (index + 1) * steps / groups : steps;
    // (in scalar registers: the divisions leave them in vector registers)
    w.left = __builtin_amdgcn_readfirstlane(static_cast<int>(v1 - v0));
    w.c = __builtin_amdgcn_readfirstlane(static_cast<int>(v0 / w.rows));
    w.r = __builtin_amdgcn_readfirstlane(static_cast<int>(v0 - v0 / w.rows * w.rows));
    w.rows = __builtin_amdgcn_readfirstlane(w.rows);
    return w;
}

} // namespace kronorder
