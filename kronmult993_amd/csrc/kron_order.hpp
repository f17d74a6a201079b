// kron_order.hpp -- the order in which the workgroups of an adjoint launch walk the entries.
//
// An entry's input gradient is n^d atomic adds unless the next entry of the run adds to the same vector. A batch listed
// by output (as the forward call wants it) visits the inputs in turn: entry k and entry k + p share an input, their
// neighbours do not. The workgroup therefore guesses that p from a sample of the gradient pointers and walks the entries
// k = c, c + p, c + 2p, ... column by column instead of k = 0, 1, 2, ...: every entry once in either order, whatever the
// guess and the pointers are, and the sums of shared gradients in registers when they do repeat with that period.
// d=6 n=4, 128 x 64 element pairs listed by output, FP64: 33.5 M atomic adds (about 200 G/s) become 2.1 M.
//
// Every workgroup guesses before its first entry, so the guess costs one round trip to memory: the first 256 pointers,
// four per lane, and every 256th up to entry 4096, one per lane, compared in registers. Every distance from 1 to 4096
// is 256 (j + 1) - i for one j < 16 and one i < 256, so in a batch with a period the smallest distance between equal
// ones is the period. (A scan of the pointers from entry 1 on, a load per thread and step, was a chain of 16 to 64 round
// trips: 9 to 12 us.)
#pragma once

#include <hip/hip_runtime.h>

#include "kron_reg.hpp"

namespace kronorder
{

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

// The smallest distance between equal ones of the sampled pointers, 1 if there are none (a guess: 32 bits of the
// addresses are compared). Every wavefront finds the same answer.
template<typename T>
__device__ __forceinline__ int guess_period(T *const *ptr, int nb)
{
    constexpr int kHead = 256, kTail = 16;
    int const lane = static_cast<int>(threadIdx.x) & 63;
    auto bits = [](T *p) { return static_cast<unsigned>(reinterpret_cast<unsigned long long>(p) >> 2); };
    unsigned head[kHead / 64];
#pragma unroll
    for (int c = 0; c < kHead / 64; ++c)
        head[c] = bits(kronreg::as_global(ptr)[64 * c + lane < nb ? 64 * c + lane : 0]);
    int const at = kHead * (lane % kTail + 1);
    int const tail = static_cast<int>(bits(kronreg::as_global(ptr)[at < nb ? at : 0]));
#pragma unroll 1
    for (int j = 0; j < kTail && kHead * (j + 1) < nb; ++j)
    {
        unsigned const there = static_cast<unsigned>(__builtin_amdgcn_readlane(tail, j));
        unsigned long long same[kHead / 64];
#pragma unroll
        for (int c = 0; c < kHead / 64; ++c) same[c] = __ballot(head[c] == there);
        if ((same[0] | same[1] | same[2] | same[3]) == 0) continue;
        int i = 0;  // the last of the head's equal to this one
#pragma unroll
        for (int c = 0; c < kHead / 64; ++c) i = same[c] != 0 ? 64 * c + 63 - __builtin_clzll(same[c]) : i;
        return kHead * (j + 1) - i;
    }
    return 1;
}

// Small tensors with runs shorter than two entries stay in natural order: there is little to sum, and neighbours that
// add to one vector at the same time wait for each other. As 64-input pairs, natural / by input: 2100 entries of d=5 n=4
// FP32, 2048 workgroups, input gradient 11.4 / 17.9 us; 780 of d=6 n=4 FP32, 768 workgroups, both gradients 26.2 / 21.5,
// 1100 of d=4 n=7 FP64, input gradient 25.4 / 21.6.
constexpr int kAlwaysByInput = 2048;  // elements

// This workgroup's part of the batch, cut into `groups` (a multiple of 8, at most the grid) equal parts; the workgroups
// past them get none. ptr may be null (natural order). Every thread calls it.
template<typename T>
__device__ __forceinline__ Walk walk(T *const *ptr, int nb, int groups, int size)
{
    int period = 1;
    if (ptr != nullptr && nb > groups && (size >= kAlwaysByInput || nb / 2 >= groups)) period = guess_period(ptr, nb);
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
