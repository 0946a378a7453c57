// The innermost triangular solves of the blocked recursions (LU, Cholesky), complex.
#pragma once

#include "wave.hpp"

namespace thcgw {

// The four forms.  A vector is a row of T (X A = T) or a column of it (A X = T).
enum TriLeaf {
  TRI_ROW_LOWER_CONJ,  // X L^H = T, L lower with a real positive diagonal
  TRI_ROW_UPPER_UNIT,  // X U = T, U upper with a unit diagonal
  TRI_COL_LOWER,       // L X = T, L lower
  TRI_COL_UPPER_UNIT,  // U X = T, U upper with a unit diagonal
};

// Solve in place with the nb x nb (nb <= NB) triangle A, m vectors.  A vector lies across a row of
// 16 lanes, element g + 16 e in lane g, and a wave holds 4 V of them.  Step c broadcasts the
// vector's element c along the row (in the vector unit), scales it by the reciprocal of the
// diagonal and subtracts its multiples from the elements that follow; the triangle is read
// from LDS once per step for all V vectors of a lane.
//
// What bounds it: memory where there are thousands of vectors (batch x m), the chain of nb steps
// where there are few.  16 lanes per vector give a hundred rows as many waves as one thread
// per vector gives 1600, and keep a vector's elements in 8 registers instead of 128.
// A product is rounded before it is subtracted: one rounding at the size of the element, and the forms
// that hold V^-1 multiply a change in the last bits of V's factor by the condition of V.
// Against one thread per vector with the triangle read from LDS for each (per launch, order 32):
// L^H with at most 1600 rows on 4 matrices 23.3 -> 6.2 us; all leaves of the LU form on 168 matrices
// of order 200 616 -> 363 us, on 164 of order 800 4.30 -> 3.14 ms.  Order-64 leaves (100 us where two of
// order 32 take 32 each and the product between them the rest) gained 1% on the latter and lost 4%
// on order 24.
template <typename RC, int NB, int V, TriLeaf KIND>
__global__ __launch_bounds__(256) void tri_leaf_kernel(const RC* A, long sA, int lda, RC* T, long sT, int ldt, int m,
                                                       int nb) {
  using S = decltype(RC{}.x);
  constexpr int E = NB / 16;
  constexpr bool ROWS = KIND == TRI_ROW_LOWER_CONJ || KIND == TRI_ROW_UPPER_UNIT;
  constexpr bool LOWER = KIND == TRI_ROW_LOWER_CONJ || KIND == TRI_COL_LOWER;
  constexpr bool DOWN = KIND == TRI_COL_UPPER_UNIT;  // the last element is final first
  // factor[c][r]: what element c contributes to element r (zero for those before it)
  __shared__ RC factor[NB][NB + 1];
  __shared__ RC rdiag[NB];  // 1 / diagonal; for L^H the diagonal and the inverse of its square
  const int b = blockIdx.y, t = threadIdx.x, lane = t & 63, g = lane & 15;
  const RC* Ab = A + static_cast<long>(b) * sA;
  for (int q = t; q < NB * NB; q += 256) {
    const int i = q / NB, j = q % NB;
    RC a{0, 0};
    if (i < nb && j < nb && (LOWER ? i >= j : i < j)) a = Ab[static_cast<long>(i) * lda + j];
    if (LOWER && i == j) {
      if (KIND == TRI_ROW_LOWER_CONJ) {
        rdiag[i] = RC{a.x, S(1) / (a.x * a.x)};
      } else {
        const S s = S(1) / (a.x * a.x + a.y * a.y);
        rdiag[i] = RC{a.x * s, -a.y * s};
      }
      a = RC{0, 0};
    }
    if (KIND == TRI_ROW_UPPER_UNIT) factor[i][j] = a;
    else factor[j][i] = a;
  }

  const int v0 = (blockIdx.x * 4 + (t >> 6)) * 4 * V + (lane >> 4);
  RC* Tb = T + static_cast<long>(b) * sT;
  RC x[V][E];
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const long i = v0 + 4 * v, c = g + 16 * e;
      x[v][e] = (i < m && c < nb) ? Tb[ROWS ? i * ldt + c : c * ldt + i] : RC{0, 0};
    }
  __syncthreads();

  each([&](auto step) __attribute__((always_inline)) {
    constexpr int c = DOWN ? NB - 1 - step : static_cast<int>(step);
    if (c < nb) {
      RC xc[V], f[E];
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (DOWN ? e <= c / 16 : e >= c / 16) f[e] = factor[c][g + 16 * e];
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const RC s{row_bcast<c % 16>(x[v][c / 16].x), row_bcast<c % 16>(x[v][c / 16].y)};
        if (KIND == TRI_ROW_LOWER_CONJ) {
          const RC d = rdiag[c];
          xc[v] = RC{s.x * d.x * d.y, s.y * d.x * d.y};
        } else if (KIND == TRI_COL_LOWER) {
          const RC d = rdiag[c];
          xc[v] = RC{s.x * d.x - s.y * d.y, s.x * d.y + s.y * d.x};
        } else {
          xc[v] = s;
        }
      }
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (DOWN ? e <= c / 16 : e >= c / 16)
#pragma unroll
          for (int v = 0; v < V; ++v) {
            if (KIND == TRI_ROW_LOWER_CONJ) {
              x[v][e].x -= xc[v].x * f[e].x + xc[v].y * f[e].y;
              x[v][e].y -= xc[v].y * f[e].x - xc[v].x * f[e].y;
            } else {
              x[v][e].x -= fma(xc[v].x, f[e].x, -(xc[v].y * f[e].y));
              x[v][e].y -= fma(xc[v].x, f[e].y, xc[v].y * f[e].x);
            }
          }
    }
  }, std::make_integer_sequence<int, NB>{});

#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const long i = v0 + 4 * v, c = g + 16 * e;
      RC s = x[v][e];
      if (KIND == TRI_ROW_LOWER_CONJ) {
        const RC d = rdiag[c];
        s = RC{s.x * d.x * d.y, s.y * d.x * d.y};
      } else if (KIND == TRI_COL_LOWER) {
        const RC d = rdiag[c];
        s = RC{s.x * d.x - s.y * d.y, s.x * d.y + s.y * d.x};
      }
      if (i < m && c < nb) Tb[ROWS ? i * ldt + c : c * ldt + i] = s;
    }
}

// Four vectors per 16 lanes read the triangle once for all four; below 16384 vectors (4 waves per SIMD
// with one each) more waves are worth more: L^H with at most 1600 rows on 4 matrices 6.2 us with
// one, 10.4 with four; order 24 on 84 matrices 4.8 and 6.7; order 200 on 168 matrices, the narrow blocks
// below the line included, 5% less by this rule than with four everywhere.
template <TriLeaf KIND, int NB, typename RC>
void tri_leaf(hipStream_t s, const RC* A, long sA, int lda, RC* T, long sT, int ldt, int m, int nb, int batch) {
  auto go = [&](auto v) {
    constexpr int V = v;
    hipLaunchKernelGGL((tri_leaf_kernel<RC, NB, V, KIND>), dim3((m + 16 * V - 1) / (16 * V), batch), dim3(256), 0, s, A,
                       sA, lda, T, sT, ldt, m, nb);
    THCGW_HIP(hipGetLastError());
  };
  if (static_cast<long>(m) * batch > 16384) go(std::integral_constant<int, 4>{});
  else go(std::integral_constant<int, 1>{});
}

}  // namespace thcgw
