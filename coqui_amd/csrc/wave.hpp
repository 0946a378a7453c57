// Wave-wide reductions without LDS (64 lanes, gfx950), and loops over register arrays.
#pragma once

#include <hip/hip_runtime.h>

#include <utility>

namespace thcgw {

// op(x, x of the lane D away): rows of 16 or halves of 32 lanes exchanged in the vector unit
// (a shuffle through LDS adds two of its latencies to a serial step).  op is commutative, so that
// both lanes get the same bits.
template <int D, class Op>
__device__ __forceinline__ double swap_with(double x, Op op) {
  static_assert(D == 16 || D == 32, "rows of 16 or halves of 32");
  const unsigned lo = static_cast<unsigned>(__double2loint(x)), hi = static_cast<unsigned>(__double2hiint(x));
  const auto l = D == 16 ? __builtin_amdgcn_permlane16_swap(lo, lo, false, false)
                         : __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto h = D == 16 ? __builtin_amdgcn_permlane16_swap(hi, hi, false, false)
                         : __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return op(__hiloint2double(static_cast<int>(h[0]), static_cast<int>(l[0])),
            __hiloint2double(static_cast<int>(h[1]), static_cast<int>(l[1])));
}

// op(x, x of the lane N to the right in its row of 16 lanes, cyclically)
template <int N, class Op>
__device__ __forceinline__ double ror_with(double x, Op op) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0x120 + N, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0x120 + N, 0xF, 0xF, false);
  return op(x, __hiloint2double(hi, lo));
}

// over the row of 16 lanes, in every lane
template <class Op>
__device__ __forceinline__ double row_reduce(double x, Op op) {
  return ror_with<1>(ror_with<2>(ror_with<4>(ror_with<8>(x, op), op), op), op);
}

struct MaxOp {
  __device__ __forceinline__ double operator()(double a, double b) const { return fmax(a, b); }
};
struct AddOp {
  __device__ __forceinline__ double operator()(double a, double b) const { return a + b; }
};

// over the wave, in every lane
template <class Op>
__device__ __forceinline__ double wave_reduce(double x, Op op) {
  return swap_with<32>(swap_with<16>(row_reduce(x, op), op), op);
}

// x of lane N of the row of 16 lanes
template <int N>
__device__ __forceinline__ float row_bcast(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x150 + N, 0xF, 0xF, false));
}
template <int N>
__device__ __forceinline__ double row_bcast(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0x150 + N, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0x150 + N, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// f(0), ..., f(E - 1) with compile-time arguments, for register arrays whose loops the compiler
// unrolls too late or whose row is picked at run time.  A branch on such a row ends in an empty
// statement that differs from row to row and so keeps the compiler from merging the branches into one
// indexed access, which would move the array to memory.
template <class F, int... A>
__device__ __forceinline__ void each(F&& f, std::integer_sequence<int, A...>) {
  (f(std::integral_constant<int, A>{}), ...);
}

}  // namespace thcgw
