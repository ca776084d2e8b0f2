// quad.hpp -- device helpers of the marching tiles with four points per lane
// (FD step, separable SEM step).
#pragma once

#include <type_traits>
#include <utility>

#include "march.hpp"

namespace phc {

typedef float quad_f4 __attribute__((ext_vector_type(4)));

template <bool NT, typename IT>
__device__ __forceinline__ quad_f4 ldq(const float *base, IT off)
{
    if constexpr (NT) return ldo_nt<IT, quad_f4>((const quad_f4 *)base, sizeof(IT) == 4 ? off : off / 4);
    else return ldo<IT, quad_f4>((const quad_f4 *)base, sizeof(IT) == 4 ? off : off / 4);
}

template <bool NT, typename IT>
__device__ __forceinline__ void stq(float *base, IT off, quad_f4 v)
{
    if constexpr (NT) {
        sto_nt<IT, quad_f4>((quad_f4 *)base, sizeof(IT) == 4 ? off : off / 4, v);
    } else {
        if constexpr (sizeof(IT) == 4) *(quad_f4 *)((char *)base + off) = v;
        else ((quad_f4 *)base)[off / 4] = v;
    }
}

// plane(u, ib + u) for u = 0, 1, ... while ib + u < end.
template <class F, int... U>
__device__ __forceinline__ void march_turn(F &plane, int ib, int end, std::integer_sequence<int, U...>)
{
    (void)((ib + U < end && (plane(std::integral_constant<int, U>{}, ib + U), true)) && ...);
}

} // namespace phc
