// Loops whose indexes are constants, whatever the compiler unrolls, and pointers into LDS
#pragma once
#include "ds_hip.h"

#include <type_traits>
#include <utility>

namespace constants {

template <int N>
using Int = std::integral_constant<int, N>;
template <class F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) {
  (f(Int<I>{}), ...);
}
// f(Int<0>{}) .. f(Int<N - 1>{})
template <int N, class F>
__device__ __forceinline__ void each(F&& f) {
  each_of(f, std::make_integer_sequence<int, N>{});
}

typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

}  // namespace constants
