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
    int nb, period, rows;  // entry of step v: v / rows + (v % rows) * period
    int v, end;            // this workgroup's next step and the end of its steps

    // the next entry, or -1 (a step past the batch, in the last row, is left out)
    __device__ __forceinline__ int next()
    {
        while (v < end)
        {
            int const c = v / rows;
            int const k = c + (v - c * rows) * period;
            ++v;
            if (k < nb) return k;
        }
        return -1;
    }
};

// `run` entries per workgroup in the natural order; ptr may be null (natural order). Every thread calls it.
template<typename T>
__device__ __forceinline__ Walk walk(T *const *ptr, int nb, int run, int *shared_min)
{
    int period = 1;
    if (ptr != nullptr && run > 1)
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
    w.rows = (nb + period - 1) / period;
    int const index = kronreg::xcd_run_index();
    int per = run;
    if (period > 1)
    {
        // steps, those past the batch among them, in equal parts
        long const steps = static_cast<long>(w.rows) * period;
        per = static_cast<int>((steps + gridDim.x - 1) / gridDim.x);
        long const v0 = static_cast<long>(index) * per;
        w.v = static_cast<int>(v0 < steps ? v0 : steps);
        w.end = static_cast<int>(v0 + per < steps ? v0 + per : steps);
        return w;
    }
    w.rows = nb;  // one column
    w.v = nb - 1 < static_cast<long>(index) * per ? nb : index * per;
    w.end = nb - w.v > per ? w.v + per : nb;
    return w;
}

} // namespace kronorder
