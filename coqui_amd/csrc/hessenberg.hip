// Electron numbers for many chemical potentials (update_mu, scf_common.cpp:147-202): the traces
// Tr[(iw_n + mu - A)^-1] of A(n, k) = H0_k + F_k + Sigma(iw_n, k), order n <= 128, orthonormal basis.
//
// The inverse would cost 8 n^3 flops for each mu.  A does not depend on mu, so it is brought once to
// Hessenberg form by unitary reflections, A = Q H Q^H with H zero below the first subdiagonal,
// which leaves Tr[(z - A)^-1] = Tr[(z - H)^-1] = d/dz ln det(z - H), and each mu needs one
// elimination of z - H with partial pivoting (adjacent rows) that carries the derivative of the
// rows with respect to z: the trace is the sum of u'/u over the pivots, 12 n^2 flops.  Both steps are
// backward stable like the inverse.  Search of 34 evaluations at N_k = 64, 80 frequencies, order 78,
// with G(tau) at its end: 48.9 -> 11.9 ms.
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

// H of A(b) into Out (its elements (i, j), j >= i - 1), one workgroup per matrix, the matrix in registers:
// thread (r, c) of T x T holds the E x E elements (r + a T, c + b T).
//
// Step k reflects column k: with v = (x + x_{k+1}/|x_{k+1}| |x| e_{k+1}), x the column below its
// diagonal, and t = 2 / v^H v, A <- (1 - t v v^H) A (1 - t v v^H).  v^H A is summed in the
// registers, over the wave's rows and then over the waves through LDS; A v stays within the T lanes
// of a row.  Per step three barriers (column, partial sums, sums); the blocks of columns before k are
// left out.  Columns below 1e-120 in norm are taken as zero, which changes A by no more than that.
//
// What bounds it: vector arithmetic, 16 fused multiply-adds per element and step where all of the matrix is
// active, with the reductions about a third of the instructions.  5120 matrices of order 78: 2.09 ms.
template <int T, int E>
__global__ __launch_bounds__(T* T) __attribute__((amdgpu_waves_per_eu(T == 32 ? 4 : E <= 3 ? 4 : 2)))
void hessenberg_kernel(const c128* H0, const c128* F, const c128* Sw, int nk, int n, c128* Out) {
  constexpr int N = T * E, NW = T * T / 64;
  __shared__ c128 column[2][N], part[NW][N], sum[N], sub[N];
  const long b = blockIdx.x, m = static_cast<long>(n) * n;
  const long kofs = (b % nk) * m;
  const int t = threadIdx.x, r = t / T, c = t % T, lane = t & 63, wave = t >> 6;
  c128 v[E][E];
#pragma unroll
  for (int a = 0; a < E; ++a)
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int i = r + a * T, j = c + q * T;
      v[a][q] = c128{0.0, 0.0};
      if (i < n && j < n) {
        const long e = static_cast<long>(i) * n + j;
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
      {  // A -= v (t v^H A), rows and columns after k
        c128 vr[E], y[E];
#pragma unroll
        for (int a = q; a < E; ++a) vr[a] = entry(r + a * T);
#pragma unroll
        for (int j = q; j < E; ++j) {
          y[j] = c128{0.0, 0.0};
#pragma unroll
          for (int a = q; a < E; ++a) cadd_conj(y[j], vr[a], v[a][j]);
          if (T == 16) y[j] = c128{swap_with<16>(y[j].x, AddOp{}), swap_with<16>(y[j].y, AddOp{})};
          y[j] = c128{swap_with<32>(y[j].x, AddOp{}), swap_with<32>(y[j].y, AddOp{})};
          if (lane < T) part[wave][c + j * T] = y[j];
        }
        __syncthreads();
        if (t >= q * T && t < N) {
          c128 z = part[0][t];
#pragma unroll
          for (int w = 1; w < NW; ++w) z = c128{z.x + part[w][t].x, z.y + part[w][t].y};
          sum[t] = c128{z.x * tau, z.y * tau};
        }
        __syncthreads();
#pragma unroll
        for (int j = q; j < E; ++j) {
          const c128 yj = sum[c + j * T];
#pragma unroll
          for (int a = q; a < E; ++a) csub(v[a][j], vr[a], yj);
        }
      }
      {  // A -= (A v) t v^H, every row
        c128 vc[E];
#pragma unroll
        for (int j = q; j < E; ++j) vc[j] = entry(c + j * T);
#pragma unroll
        for (int a = 0; a < E; ++a) {
          c128 z{0.0, 0.0};
#pragma unroll
          for (int j = q; j < E; ++j) cadd(z, v[a][j], vc[j]);
          z = c128{row_reduce(z.x, AddOp{}), row_reduce(z.y, AddOp{})};
          if (T == 32) z = c128{swap_with<16>(z.x, AddOp{}), swap_with<16>(z.y, AddOp{})};
          z = c128{z.x * tau, z.y * tau};
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
  __syncthreads();
  c128* Ob = Out + b * m;
#pragma unroll
  for (int a = 0; a < E; ++a)
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int i = r + a * T, j = c + q * T;
      c128 x = v[a][q];
      if (j == i - 1 && j < n - 2) x = sub[j];
      if (i < n && j < n && j >= i - 1) Ob[static_cast<long>(i) * n + j] = x;
    }
}

// Tr[(iw_n + mu - H)^-1] of count Hessenberg matrices, 16 lanes per matrix (columns g + 16 e), 4 matrices
// per wave.  Step i holds row i of the elimination and its derivative; the next row of H comes from
// memory, three steps ahead.  The smaller of the two candidates for pivot i is eliminated.
// bad[b] = 1 where a pivot is zero or not finite.
//
// What bounds it: the chain of a step (pivot to the row's lanes, reciprocal, update) at 1 to 2 waves per
// SIMD and the selects that pivoting needs.  5120 matrices of order 78: 156 us, against 1.26 ms for
// the inverses in registers.
template <int E>
__global__ __launch_bounds__(64) void hessenberg_trace_kernel(const c128* H, const long* wn, double beta, double mu,
                                                              int nk, int n, int count, c128* tr, int* bad_out) {
  constexpr int AHEAD = 4;
  const int lane = threadIdx.x, g = lane & 15, base = lane & 48;
  const int mat = blockIdx.x * 4 + (lane >> 4), b = min(mat, count - 1);
  const c128* Hb = H + static_cast<long>(b) * n * n;
  const c128 z{mu, static_cast<double>(wn[b / nk]) * M_PI / beta};
  // element (i, column g + 16 e) of z - H; zero outside the matrix and below the subdiagonal
  auto element = [&](int i, int e) __attribute__((always_inline)) {
    const int j = g + 16 * e;
    const bool in = i < n && j < n && j >= i - 1;
    const c128 h = Hb[in ? static_cast<long>(i) * n + j : 0];
    return in ? c128{(j == i ? z.x : 0.0) - h.x, (j == i ? z.y : 0.0) - h.y} : c128{0.0, 0.0};
  };
  c128 r[E], d[E], next[AHEAD][E];  // row, its derivative, the rows that follow
#pragma unroll
  for (int e = 0; e < E; ++e) {
    r[e] = element(0, e);
    d[e] = c128{e == 0 && g == 0 ? 1.0 : 0.0, 0.0};
#pragma unroll
    for (int p = 0; p < AHEAD; ++p) next[p][e] = element(1 + p, e);
  }
  c128 sum{0.0, 0.0};
  bool bad = false;
  each([&](auto block) __attribute__((always_inline)) {
    constexpr int q = block;
    for (int i0 = 16 * q; i0 < 16 * q + 16 && i0 < n; i0 += AHEAD) {
#pragma unroll
      for (int p = 0; p < AHEAD; ++p) {
        const int i = i0 + p;
        if (i < n) {
          const int from = base + (i & 15);
          auto pick = [&](c128 w) __attribute__((always_inline)) {
            return c128{__shfl(w.x, from), __shfl(w.y, from)};
          };
          const c128 ri = pick(r[q]), di = pick(d[q]), mi = pick(next[p][q]);
          const bool swap = fabs(mi.x) + fabs(mi.y) > fabs(ri.x) + fabs(ri.y);
          const c128 u = swap ? mi : ri, o = swap ? ri : mi;
          const c128 du = swap ? c128{0.0, 0.0} : di, dother = swap ? di : c128{0.0, 0.0};
          if (!(isfinite(u.x) && isfinite(u.y)) || (u.x == 0.0 && u.y == 0.0)) bad = true;
          const c128 inv = crecip(u);
          cadd(sum, du, inv);
          const c128 l = cmul(o, inv);  // the multiplier and its derivative
          c128 dl = dother;
          csub(dl, l, du);
          dl = cmul(dl, inv);
#pragma unroll
          for (int e = q; e < E; ++e) {
            const c128 m = next[p][e], dm{g + 16 * e == i + 1 ? 1.0 : 0.0, 0.0};
            const c128 pr = swap ? m : r[e], pd = swap ? dm : d[e];
            c128 w = swap ? r[e] : m, dw = swap ? d[e] : dm;
            csub(w, l, pr);
            csub(dw, dl, pr);
            csub(dw, l, pd);
            r[e] = w;
            d[e] = dw;
            next[p][e] = element(i + 1 + AHEAD, e);
          }
        }
      }
    }
  }, std::make_integer_sequence<int, E>{});
  if (g == 0 && mat < count) {
    tr[b] = sum;
    bad_out[b] = bad;
  }
}

// out[n] = sum over k of tr[n, k] / N_k, in order of k; out[nw].x = number of bad traces
__global__ __launch_bounds__(256) void trace_sums_kernel(const c128* tr, const int* bad, int nw, int nk, c128* out) {
  __shared__ int nbad;
  if (threadIdx.x == 0) nbad = 0;
  __syncthreads();
  int mine = 0;
  for (int w = threadIdx.x; w < nw; w += 256) {
    c128 s{0.0, 0.0};
#pragma unroll 8
    for (int k = 0; k < nk; ++k) {
      const c128 x = tr[static_cast<long>(w) * nk + k];
      s.x += x.x / nk;
      s.y += x.y / nk;
      mine += bad[static_cast<long>(w) * nk + k];
    }
    out[w] = s;
  }
  if (mine) atomicAdd(&nbad, mine);
  __syncthreads();
  if (threadIdx.x == 0) out[nw] = c128{static_cast<double>(nbad), 0.0};
}

}  // namespace

bool hessenberg_fits(int no) { return no >= 1 && no <= 128; }

void hessenberg_reduce(hipStream_t s, const c128* H0, const c128* F, const c128* Sw, int nw, int nk, int no, c128* H) {
  THCGW_REQUIRE(hessenberg_fits(no), "hessenberg_reduce: order must be in [1, 128]");
  const long count = static_cast<long>(nw) * nk;
  THCGW_REQUIRE(count >= 1 && count < (1L << 30), "Dyson for G: too many matrices");
  auto go = [&](auto t, auto e) {
    constexpr int T = t, E = e;
    hipLaunchKernelGGL((hessenberg_kernel<T, E>), dim3(static_cast<unsigned>(count)), dim3(T * T), 0, s, H0, F, Sw, nk,
                       no, H);
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

void hessenberg_traces(hipStream_t s, const c128* H, const long* wn, double beta, double mu, int nw, int nk, int no,
                       c128* tr, int* bad, c128* sums) {
  THCGW_REQUIRE(hessenberg_fits(no), "hessenberg_traces: order must be in [1, 128]");
  const long count = static_cast<long>(nw) * nk;
  THCGW_REQUIRE(count >= 1 && count < (1L << 30), "Dyson for G: too many matrices");
  auto go = [&](auto e) {
    constexpr int E = e;
    hipLaunchKernelGGL((hessenberg_trace_kernel<E>), dim3(static_cast<unsigned>((count + 3) / 4)), dim3(64), 0, s, H, wn,
                       beta, mu, nk, no, static_cast<int>(count), tr, bad);
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
  hipLaunchKernelGGL(trace_sums_kernel, dim3(1), dim3(256), 0, s, tr, bad, nw, nk, sums);
  THCGW_HIP(hipGetLastError());
}

}  // namespace thcgw
