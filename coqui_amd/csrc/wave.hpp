// Wave-wide reductions without LDS (64 lanes, gfx950), and loops over register arrays.
#pragma once

#include <hip/hip_runtime.h>

#include <utility>

namespace thcgw {

// max(x, x of the lane D away): rows of 16 or halves of 32 lanes exchanged in the vector unit
// (a shuffle through LDS adds two of its latencies to a serial step)
template <int D>
__device__ __forceinline__ double swap_max(double x) {
  static_assert(D == 16 || D == 32, "rows of 16 or halves of 32");
  const unsigned lo = static_cast<unsigned>(__double2loint(x)), hi = static_cast<unsigned>(__double2hiint(x));
  const auto l = D == 16 ? __builtin_amdgcn_permlane16_swap(lo, lo, false, false)
                         : __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto h = D == 16 ? __builtin_amdgcn_permlane16_swap(hi, hi, false, false)
                         : __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return fmax(__hiloint2double(static_cast<int>(h[0]), static_cast<int>(l[0])),
              __hiloint2double(static_cast<int>(h[1]), static_cast<int>(l[1])));
}

// max(x, x of the lane N to the right in its row of 16 lanes, cyclically)
template <int N>
__device__ __forceinline__ double ror_max(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0x120 + N, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0x120 + N, 0xF, 0xF, false);
  return fmax(x, __hiloint2double(hi, lo));
}

// maximum over the wave, in every lane
__device__ __forceinline__ double wave_max(double x) {
  x = ror_max<8>(x);
  x = ror_max<4>(x);
  x = ror_max<2>(x);
  x = ror_max<1>(x);
  return swap_max<32>(swap_max<16>(x));
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
