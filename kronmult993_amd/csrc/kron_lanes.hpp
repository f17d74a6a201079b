// kron_lanes.hpp -- sums across the lanes of a wavefront in the vector ALU (V_PERMLANE32_SWAP, V_PERMLANE16_SWAP and
// DPP), for the adjoint kernels' factor gradients. The same steps through LDS (ds_bpermute, what __shfl_xor compiles
// to) cost two LDS instructions and more selects per double.
#pragma once

#include <hip/hip_runtime.h>

namespace kronlanes
{

// Permutation that flips lane bit BIT (one of 32 .. 1) and keeps every higher bit; BIT = 4 also flips bits 1 and 0.
template<int BIT>
constexpr int dpp_ctrl()
{
    return BIT == 8 ? 0x128   // row_ror:8
         : BIT == 4 ? 0x141   // row_half_mirror
         : BIT == 2 ? 0x4e    // quad_perm:[2,3,0,1]
                    : 0xb1;   // quad_perm:[1,0,3,2]
}

template<int BIT>
__device__ __forceinline__ unsigned dpp(unsigned v)
{
    return static_cast<unsigned>(
        __builtin_amdgcn_update_dpp(0, static_cast<int>(v), dpp_ctrl<BIT>(), 0xf, 0xf, false));
}

struct Pair
{
    unsigned a, b;
};

// 32 / 16: a's upper half (of the wavefront / of every 32 lanes) and b's lower half change places
template<int BIT>
__device__ __forceinline__ Pair swap(unsigned a, unsigned b)
{
    if constexpr (BIT == 32)
    {
        auto const r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        return {static_cast<unsigned>(r[0]), static_cast<unsigned>(r[1])};
    }
    else
    {
        auto const r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        return {static_cast<unsigned>(r[0]), static_cast<unsigned>(r[1])};
    }
}

// One step of a reduce-scatter over the lanes: a lane with bit BIT clear returns lo summed with its partner's lo, a lane
// with the bit set hi summed with its partner's hi.
template<int BIT>
__device__ __forceinline__ float fold(float lo, float hi, int lane)
{
    if constexpr (BIT >= 16)
    {
        Pair const p = swap<BIT>(__float_as_uint(lo), __float_as_uint(hi));
        return __uint_as_float(p.a) + __uint_as_float(p.b);
    }
    else
    {
        bool const set = (lane & BIT) != 0;
        float const mine = set ? hi : lo, other = set ? lo : hi;
        return mine + __uint_as_float(dpp<BIT>(__float_as_uint(other)));
    }
}
template<int BIT>
__device__ __forceinline__ double fold(double lo, double hi, int lane)
{
    auto join = [](unsigned l, unsigned h) {
        return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(h) << 32) | l));
    };
    auto low = [](double v) { return static_cast<unsigned>(__double_as_longlong(v)); };
    auto high = [](double v) {
        return static_cast<unsigned>(static_cast<unsigned long long>(__double_as_longlong(v)) >> 32);
    };
    if constexpr (BIT >= 16)
    {
        Pair const l = swap<BIT>(low(lo), low(hi)), h = swap<BIT>(high(lo), high(hi));
        return join(l.a, h.a) + join(l.b, h.b);
    }
    else
    {
        bool const set = (lane & BIT) != 0;
        double const mine = set ? hi : lo, other = set ? lo : hi;
        return mine + join(dpp<BIT>(low(other)), dpp<BIT>(high(other)));
    }
}

// v summed with the partner's v
template<int BIT, typename T>
__device__ __forceinline__ T add(T v)
{
    return fold<BIT>(v, v, 0);
}

} // namespace kronlanes
