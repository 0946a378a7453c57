// Electron numbers for many chemical potentials (update_mu, scf_common.cpp:147-202): the traces
// Tr[(iw_n + mu - A)^-1] of A(n, k) = H0_k + F_k + Sigma(iw_n, k), order n <= 128, orthonormal basis.
//
// The inverse would cost 8 n^3 flops for each mu.  A does not depend on mu, so B = A^T is brought once
// to Hessenberg form by unitary reflections, B = Q H Q^H with H zero below the first subdiagonal,
// which leaves Tr[(z - A)^-1] = Tr[(z - H)^-1] = d/dz ln det(z - H).  For each mu Hyman's recurrence
// (Wilkinson, The Algebraic Eigenvalue Problem, 7.11) gives the determinant up to a factor that does
// not depend on z: with x_{n-1} = 1, the rows i = n-1 .. 1 of (z - H) x = 0 give x_{i-1}, and row 0
// leaves a number p proportional to det(z - H); differentiated along, p'/p is the trace, 8 n^2 flops.
// The reflections are backward stable.  The recurrence and its derivative round independently, with an error of
// order eps cond(z - A) for the trace, the inverse's.  N against extended precision (rms over 40 to 60 random
// H(k) + Sigma and four mu, in 1e-16 n): inverses 4.4 at any order, this 4.6 at order 8, 5.7 at 32, 6.4 at 78:
// 5e-14 there, against the mu_tol that ends the search (1e-9).  Sums of the recurrence with their rounding
// errors took 40% longer and left it at 6.9: what remains is the rounding of x and its derivative.
// Where p underflows the trace is not finite, and that mu goes to the inverses.
// Search of 34 evaluations at N_k = 64, 80 frequencies, order 78, with G(tau) at its end: 48.9 ->
// 8.2 ms.
#include "thcgw_internal.hpp"
#include "wave.hpp"

#include <type_traits>

namespace thcgw {
namespace {

__device__ __forceinline__ c128 cmul(c128 a, c128 b) { return c128{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
// c += a b
__device__ __forceinline__ void cadd(c128& c, c128 a, c128 b) {
  c.x = fma(-a.y, b.y, fma(a.x, b.x, c.x));
  c.y = fma(a.y, b.x, fma(a.x, b.y, c.y));
}
// c += conj(a) b
__device__ __forceinline__ void cadd_conj(c128& c, c128 a, c128 b) {
  c.x = fma(a.y, b.y, fma(a.x, b.x, c.x));
  c.y = fma(-a.y, b.x, fma(a.x, b.y, c.y));
}
// c -= a b
__device__ __forceinline__ void csub(c128& c, c128 a, c128 b) {
  c.x = fma(a.y, b.y, fma(-a.x, b.x, c.x));
  c.y = fma(-a.y, b.x, fma(-a.x, b.y, c.y));
}
// c -= a conj(b)
__device__ __forceinline__ void csub_conj(c128& c, c128 a, c128 b) {
  c.x = fma(-a.y, b.y, fma(-a.x, b.x, c.x));
  c.y = fma(-a.y, b.x, fma(a.x, b.y, c.y));
}
__device__ __forceinline__ c128 crecip(c128 d) {
  const double s = 1.0 / (d.x * d.x + d.y * d.y);
  return c128{d.x * s, -d.y * s};
}

// H of B = A(b)^T, one workgroup per matrix, the matrix in registers: thread (r, c) of T x T holds the
// E x E elements (r + a T, c + b T) of B.  Out[b][j][i] = H[i][j], i <= j, and rsub[b][j] = 1 / H[j][j-1]
// (subdiagonal elements below 1e-120 count as 1e-120, which changes B by no more than that).
//
// Step k reflects column k: with v = (x + x_{k+1}/|x_{k+1}| |x| e_{k+1}), x the column below its
// diagonal, and t = 2 / v^H v, B <- (1 - t v v^H) B (1 - t v v^H).  v^H B stays within the T lanes of
// a column; B v is summed in the registers, over the wave's columns and then over the waves through
// LDS.  Per step three barriers (column, partial sums, sums); the blocks of columns before k are left
// out.
//
// What bounds it: vector arithmetic, 16 fused multiply-adds per element and step where all of the matrix is
// active, with the reductions about a third of the instructions.  5120 matrices of order 78: 2.06 ms.
template <int T, int E>
__global__ __launch_bounds__(T* T) __attribute__((amdgpu_waves_per_eu(T == 32 ? 4 : E <= 3 ? 4 : 2)))
void hessenberg_kernel(const c128* H0, const c128* F, const c128* Sw, int nk, int n, c128* Out, c128* rsub) {
  constexpr int N = T * E, NW = T * T / 64;
  __shared__ c128 column[2][N], part[NW][N], sum[N], sub[N];
  const long b = blockIdx.x, m = static_cast<long>(n) * n;
  const long kofs = (b % nk) * m;
  const int t = threadIdx.x, r = t % T, c = t / T, lane = t & 63, wave = t >> 6;
  c128 v[E][E];
#pragma unroll
  for (int a = 0; a < E; ++a)
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int i = r + a * T, j = c + q * T;
      v[a][q] = c128{0.0, 0.0};
      if (i < n && j < n) {
        const long e = static_cast<long>(j) * n + i;
        const c128 h = H0 ? H0[kofs + e] : c128{0.0, 0.0};
        const c128 f = F[kofs + e], sw = Sw[b * m + e];
        v[a][q] = c128{h.x + f.x + sw.x, h.y + f.y + sw.y};
      }
    }
  auto publish = [&](auto q_tag, int cc, int buf) __attribute__((always_inline)) {
    constexpr int q = decltype(q_tag)::value;
    if (c == cc) {
#pragma unroll
      for (int a = 0; a < E; ++a) column[buf][r + a * T] = v[a][q];
      asm volatile("; column block %0" ::"n"(q));
    }
  };
  publish(std::integral_constant<int, 0>{}, 0, 0);

  auto step = [&](auto q_tag, int kk) __attribute__((always_inline)) {
    constexpr int q = decltype(q_tag)::value;
    const int k = q * T + kk;
    const c128* x = column[k & 1];
    __syncthreads();
    double s2 = 0.0;
#pragma unroll
    for (int l = 0; l < N; l += 64)
      if (lane + l < N && lane + l > k) {
        const c128 e = x[lane + l];
        s2 = fma(e.x, e.x, fma(e.y, e.y, s2));
      }
    s2 = wave_reduce(s2, AddOp{});
    const c128 alpha = x[k + 1];
    const double a2 = fma(alpha.x, alpha.x, alpha.y * alpha.y);
    if (s2 < 1e-240) {  // nothing to reflect
      if (t == 0) sub[k] = c128{0.0, 0.0};
    } else {
      const double norm = sqrt(s2), am = sqrt(a2);
      const bool zero = a2 < 1e-280;
      const double ratio = zero ? 0.0 : norm / am;
      const c128 phase_norm = zero ? c128{norm, 0.0} : c128{alpha.x * ratio, alpha.y * ratio};
      const double tau = 1.0 / fma(norm, am, s2);
      if (t == 0) sub[k] = c128{-phase_norm.x, -phase_norm.y};
      const c128 head{(zero ? 0.0 : alpha.x) + phase_norm.x, (zero ? 0.0 : alpha.y) + phase_norm.y};
      auto entry = [&](int i) __attribute__((always_inline)) {
        const c128 e = x[i];
        return i > k + 1 ? e : i == k + 1 ? head : c128{0.0, 0.0};
      };
      {  // B -= v (t v^H B), rows and columns after k
        c128 vr[E];
#pragma unroll
        for (int a = q; a < E; ++a) vr[a] = entry(r + a * T);
#pragma unroll
        for (int j = q; j < E; ++j) {
          c128 y{0.0, 0.0};
#pragma unroll
          for (int a = q; a < E; ++a) cadd_conj(y, vr[a], v[a][j]);
          y = c128{row_reduce(y.x, AddOp{}), row_reduce(y.y, AddOp{})};
          if (T == 32) y = c128{swap_with<16>(y.x, AddOp{}), swap_with<16>(y.y, AddOp{})};
          y = c128{y.x * tau, y.y * tau};
#pragma unroll
          for (int a = q; a < E; ++a) csub(v[a][j], vr[a], y);
        }
      }
      {  // B -= (t B v) v^H, every row
        c128 vc[E];
#pragma unroll
        for (int j = q; j < E; ++j) vc[j] = entry(c + j * T);
#pragma unroll
        for (int a = 0; a < E; ++a) {
          c128 z{0.0, 0.0};
#pragma unroll
          for (int j = q; j < E; ++j) cadd(z, v[a][j], vc[j]);
          if (T == 16) z = c128{swap_with<16>(z.x, AddOp{}), swap_with<16>(z.y, AddOp{})};
          z = c128{swap_with<32>(z.x, AddOp{}), swap_with<32>(z.y, AddOp{})};
          if (lane < T) part[wave][r + a * T] = z;
        }
        __syncthreads();
        if (t < N) {
          c128 z = part[0][t];
#pragma unroll
          for (int w = 1; w < NW; ++w) z = c128{z.x + part[w][t].x, z.y + part[w][t].y};
          sum[t] = c128{z.x * tau, z.y * tau};
        }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < E; ++a) {
          const c128 z = sum[r + a * T];
#pragma unroll
          for (int j = q; j < E; ++j) csub_conj(v[a][j], z, vc[j]);
        }
      }
    }
    if (kk + 1 < T) publish(q_tag, kk + 1, (k + 1) & 1);
    else if constexpr (q + 1 < E) publish(std::integral_constant<int, q + 1>{}, 0, (k + 1) & 1);
  };
  each([&](auto q_tag) __attribute__((always_inline)) {
    for (int kk = 0; kk < T && decltype(q_tag)::value * T + kk < n - 2; ++kk) step(q_tag, kk);
  }, std::make_integer_sequence<int, E>{});

  c128* Ob = Out + b * m;
#pragma unroll
  for (int a = 0; a < E; ++a)
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int i = r + a * T, j = c + q * T;
      if (i <= j && j < n) Ob[static_cast<long>(j) * n + i] = v[a][q];
      if (i == n - 1 && j == n - 2) sub[j] = v[a][q];  // the last column below its diagonal is one element
    }
  __syncthreads();
  if (t >= 1 && t < n) {
    c128 d = sub[t - 1];
    if (fabs(d.x) < 1e-120 && fabs(d.y) < 1e-120) d = c128{1e-120, 0.0};
    rsub[b * n + t] = crecip(d);
  }
}

// Tr[(iw_n + mu - H)^-1] of count Hessenberg matrices, 16 lanes per matrix (rows g + 16 e), 4 matrices per
// wave.  Step i adds column i times x_i to the sums of H x and of its derivative, of which row i
// is then complete and gives x_{i-1}.  Columns come from memory four steps ahead.
// bad[b] = 1 where the result is not finite.
//
// What bounds it: the read of H, n^2 / 2 complex numbers per matrix.  5120 matrices of order 78: 55 us,
// 4.6 TB/s, against 1.36 ms for the inverses in registers and 156 us for an elimination of z - H with
// pivoting (whose selects and divisions cost more than the read).
template <int E>
__global__ __launch_bounds__(64) void hessenberg_trace_kernel(const c128* H, const c128* rsub, const long* wn,
                                                              double beta, double mu, int nk, int n, int count,
                                                              c128* tr, int* bad) {
  constexpr int AHEAD = 4;
  const int lane = threadIdx.x, g = lane & 15, base = lane & 48;
  const int mat = blockIdx.x * 4 + (lane >> 4), b = min(mat, count - 1);
  const c128* Hb = H + static_cast<long>(b) * n * n;
  const c128* Rb = rsub + static_cast<long>(b) * n;
  const c128 z{mu, static_cast<double>(wn[b / nk]) * M_PI / beta};
  c128 hx[E], hd[E], next[AHEAD][E], rnext[AHEAD];
  auto fetch = [&](auto slot, int i, int blocks) __attribute__((always_inline)) {
    constexpr int p = decltype(slot)::value;
    const bool in = i >= 0 && i < n;
    rnext[p] = Rb[in && i > 0 ? i : n - 1];
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (e < blocks) {
        const int row = g + 16 * e;
        next[p][e] = c128{0.0, 0.0};
        if (in && row <= i) next[p][e] = Hb[static_cast<long>(i) * n + row];
      }
  };
#pragma unroll
  for (int e = 0; e < E; ++e) hx[e] = hd[e] = c128{0.0, 0.0};
  each([&](auto slot) __attribute__((always_inline)) { fetch(slot, 16 * E - 1 - slot, E); },
       std::make_integer_sequence<int, AHEAD>{});
  c128 x{1.0, 0.0}, d{0.0, 0.0}, p{0.0, 0.0}, dp{0.0, 0.0};  // x_i, its derivative; row i of (z - H) x, likewise
  each([&](auto block) __attribute__((always_inline)) {
    constexpr int q = E - 1 - block;
    for (int ii = 15; ii >= 0; ii -= AHEAD) {
      each([&](auto slot) __attribute__((always_inline)) {
        const int i = 16 * q + ii - slot;
        if (i < n) {
#pragma unroll
          for (int e = 0; e <= q; ++e) {
            cadd(hx[e], next[slot][e], x);
            cadd(hd[e], next[slot][e], d);
          }
          const int from = base + (i & 15);
          p = c128{-__shfl(hx[q].x, from), -__shfl(hx[q].y, from)};
          dp = c128{x.x - __shfl(hd[q].x, from), x.y - __shfl(hd[q].y, from)};
          cadd(p, z, x);
          cadd(dp, z, d);
          if (i > 0) {
            x = cmul(p, rnext[slot]);
            d = cmul(dp, rnext[slot]);
            const double mag = fmax(fabs(x.x), fabs(x.y));
            if (mag > 1e60) {  // a common factor, which the result does not see
              const double s = 1.0 / mag;
              x = c128{x.x * s, x.y * s};
              d = c128{d.x * s, d.y * s};
#pragma unroll
              for (int e = 0; e <= q; ++e) {
                hx[e] = c128{hx[e].x * s, hx[e].y * s};
                hd[e] = c128{hd[e].x * s, hd[e].y * s};
              }
            }
          }
        }
        fetch(slot, i - AHEAD, q + 1);
      }, std::make_integer_sequence<int, AHEAD>{});
    }
  }, std::make_integer_sequence<int, E>{});
  if (g == 0 && mat < count) {
    const c128 t = cmul(dp, crecip(p));
    tr[b] = t;
    bad[b] = !(isfinite(t.x) && isfinite(t.y));
  }
}

// out[n] = the average of tr[n, k] over k, out[nw + n].x = the number of bad ones; one wave per n
__global__ __launch_bounds__(64) void trace_sums_kernel(const c128* tr, const int* bad, int nw, int nk, c128* out) {
  const long base = static_cast<long>(blockIdx.x) * nk;
  c128 s{0.0, 0.0};
  double lost = 0.0;
  for (int k = threadIdx.x; k < nk; k += 64) {
    const c128 x = tr[base + k];
    s.x += x.x / nk;
    s.y += x.y / nk;
    lost += bad[base + k];
  }
  s = c128{wave_reduce(s.x, AddOp{}), wave_reduce(s.y, AddOp{})};
  lost = wave_reduce(lost, AddOp{});
  if (threadIdx.x == 0) {
    out[blockIdx.x] = s;
    out[nw + blockIdx.x] = c128{lost, 0.0};
  }
}

}  // namespace

bool hessenberg_fits(int no) { return no >= 1 && no <= 128; }

void hessenberg_reduce(hipStream_t s, const c128* H0, const c128* F, const c128* Sw, int nw, int nk, int no, c128* H,
                       c128* rsub) {
  THCGW_REQUIRE(hessenberg_fits(no), "hessenberg_reduce: order must be in [1, 128]");
  const long count = static_cast<long>(nw) * nk;
  THCGW_REQUIRE(count >= 1 && count < (1L << 30), "Dyson for G: too many matrices");
  auto go = [&](auto t, auto e) {
    constexpr int T = t, E = e;
    hipLaunchKernelGGL((hessenberg_kernel<T, E>), dim3(static_cast<unsigned>(count)), dim3(T * T), 0, s, H0, F, Sw, nk,
                       no, H, rsub);
    THCGW_HIP(hipGetLastError());
  };
  using std::integral_constant;
  switch ((no + 15) / 16) {
    case 1: go(integral_constant<int, 16>{}, integral_constant<int, 1>{}); break;
    case 2: go(integral_constant<int, 16>{}, integral_constant<int, 2>{}); break;
    case 3: go(integral_constant<int, 16>{}, integral_constant<int, 3>{}); break;
    case 4: go(integral_constant<int, 16>{}, integral_constant<int, 4>{}); break;
    case 5: go(integral_constant<int, 16>{}, integral_constant<int, 5>{}); break;
    case 6: go(integral_constant<int, 16>{}, integral_constant<int, 6>{}); break;
    default: go(integral_constant<int, 32>{}, integral_constant<int, 4>{}); break;
  }
}

void hessenberg_traces(hipStream_t s, const c128* H, const c128* rsub, const long* wn, double beta, double mu, int nw,
                       int nk, int no, c128* tr, int* bad, c128* sums) {
  THCGW_REQUIRE(hessenberg_fits(no), "hessenberg_traces: order must be in [1, 128]");
  const long count = static_cast<long>(nw) * nk;
  THCGW_REQUIRE(count >= 1 && count < (1L << 30), "Dyson for G: too many matrices");
  auto go = [&](auto e) {
    constexpr int E = e;
    hipLaunchKernelGGL((hessenberg_trace_kernel<E>), dim3(static_cast<unsigned>((count + 3) / 4)), dim3(64), 0, s, H, rsub,
                       wn, beta, mu, nk, no, static_cast<int>(count), tr, bad);
    THCGW_HIP(hipGetLastError());
  };
  using std::integral_constant;
  switch ((no + 15) / 16) {
    case 1: go(integral_constant<int, 1>{}); break;
    case 2: go(integral_constant<int, 2>{}); break;
    case 3: go(integral_constant<int, 3>{}); break;
    case 4: go(integral_constant<int, 4>{}); break;
    case 5: go(integral_constant<int, 5>{}); break;
    case 6: go(integral_constant<int, 6>{}); break;
    case 7: go(integral_constant<int, 7>{}); break;
    default: go(integral_constant<int, 8>{}); break;
  }
  hipLaunchKernelGGL(trace_sums_kernel, dim3(nw), dim3(64), 0, s, tr, bad, nw, nk, sums);
  THCGW_HIP(hipGetLastError());
}

}  // namespace thcgw
