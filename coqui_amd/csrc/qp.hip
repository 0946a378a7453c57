// Quasiparticle equation on the device: 16 lanes per (k, n) state.
//
// Per state (solve_qp_eqn, qp_scf_common.cpp:150-311): Sigma_nn at the Pade fit frequencies
// from the diagonal Sigma_nn(tau), a Thiele continued-fraction Pade through those points (pade_t.hpp:34-168, coefficients by the
// recursion of pade_t.hpp:176-192), and the root of
//   res(e) = Re[e + i eta - Vhf_nn - Sigma_nn(e - mu + i eta)]
// by the bracketing and bisection of qp_eqn_bisection (qp_scf_common.cpp:679-728).
// The reference runs the Pade in 100-digit arithmetic; here the fit and its evaluation run
// in double-double (Hida, Li & Bailey, ARITH-15, 2001), which the tests check against a
// binary128 restatement.
#include "thcgw_internal.hpp"

namespace thcgw {
namespace {

struct dd {
  double hi, lo;
};
__device__ __forceinline__ dd two_sum(double a, double b) {
  const double s = a + b, bb = s - a;
  return {s, (a - (s - bb)) + (b - bb)};
}
__device__ __forceinline__ dd quick_two_sum(double a, double b) {
  const double s = a + b;
  return {s, b - (s - a)};
}
__device__ __forceinline__ dd two_prod(double a, double b) {
  const double p = a * b;
  return {p, fma(a, b, -p)};
}
__device__ __forceinline__ dd add(dd x, dd y) {
  dd s = two_sum(x.hi, y.hi), t = two_sum(x.lo, y.lo);
  s.lo += t.hi;
  s = quick_two_sum(s.hi, s.lo);
  s.lo += t.lo;
  return quick_two_sum(s.hi, s.lo);
}
__device__ __forceinline__ dd neg(dd x) { return {-x.hi, -x.lo}; }
__device__ __forceinline__ dd sub(dd x, dd y) { return add(x, neg(y)); }
__device__ __forceinline__ dd mul(dd x, dd y) {
  dd p = two_prod(x.hi, y.hi);
  p.lo += x.hi * y.lo + x.lo * y.hi;
  return quick_two_sum(p.hi, p.lo);
}
__device__ __forceinline__ dd mul_d(dd x, double y) {
  dd p = two_prod(x.hi, y);
  p.lo += x.lo * y;
  return quick_two_sum(p.hi, p.lo);
}
// a / y with r = 1 / y rounded: the quotient a r corrected by its remainder (Markstein, IBM J. Res. Dev.
// 34, 1990), which is a / y correctly rounded where a r is within one ulp of it and nearly so elsewhere.  The
// double-double quotient takes its remainders from these values, whatever their last bit.
__device__ __forceinline__ double quotient(double a, double y, double r) {
  const double q = a * r;
  return fma(fma(-q, y, a), r, q);
}
// x / y, r = 1 / y.hi
__device__ __forceinline__ dd div(dd x, dd y, double inv) {
  const double q1 = quotient(x.hi, y.hi, inv);
  dd r = sub(x, mul_d(y, q1));
  const double q2 = quotient(r.hi, y.hi, inv);
  r = sub(r, mul_d(y, q2));
  const double q3 = quotient(r.hi, y.hi, inv);
  return add(quick_two_sum(q1, q2), dd{q3, 0.0});
}

struct zdd {
  dd re, im;
};
__device__ __forceinline__ zdd zadd(zdd a, zdd b) { return {add(a.re, b.re), add(a.im, b.im)}; }
__device__ __forceinline__ zdd zsub(zdd a, zdd b) { return {sub(a.re, b.re), sub(a.im, b.im)}; }
__device__ __forceinline__ zdd zmul(zdd a, zdd b) {
  return {sub(mul(a.re, b.re), mul(a.im, b.im)), add(mul(a.re, b.im), mul(a.im, b.re))};
}
// the six quotients by den share one division, which costs as much as five of them
__device__ __forceinline__ zdd zdiv(zdd a, zdd b) {
  const dd den = add(mul(b.re, b.re), mul(b.im, b.im));
  const double r = 1.0 / den.hi;
  return {div(add(mul(a.re, b.re), mul(a.im, b.im)), den, r), div(sub(mul(a.im, b.re), mul(a.re, b.im)), den, r)};
}
__device__ __forceinline__ zdd zd(double re, double im) { return {dd{re, 0.0}, dd{im, 0.0}}; }

// A(w) = a_0 / (1 + a_1 (w - z_0) / (1 + a_2 (w - z_1) / (1 + ...))), z_i = i zim[i]   (pade_t.hpp:109-128)
__device__ double2 pade_eval(const QpFit& fit, const zdd* a, double wr, double wi) {
  const int n = fit.nfit;
  const zdd W = zd(wr, wi), one = zd(1.0, 0.0);
  zdd X = zmul(a[n - 1], zsub(W, zd(0.0, fit.zim[n - 2])));
  for (int f = 1; f < n - 1; ++f) {
    const int idx = n - f - 1;
    X = zdiv(zmul(a[idx], zsub(W, zd(0.0, fit.zim[idx - 1]))), zadd(one, X));
  }
  X = zdiv(a[0], zadd(one, X));
  return double2{X.re.hi + X.re.lo, X.im.hi + X.im.lo};
}

// 4 states per wave, 16 lanes each; lane l holds the points l, l + 16, ... of the fit, so that a
// column of the Thiele table is one step.  Bracketing tries 16 energies at a time and bisection the 15
// midpoints of its next four levels; both then follow the path that one trial at a time takes, with
// the same midpoints to the bit, and drop what lies beside it.
//
// What bounds it: vector instructions in double-double, n_fit divisions per trial.  The states of a system
// are too few to fill the chip with a thread each (104 waves for 6656 states), so idle lanes try ahead:
// 5 times the trials at 16 times the lanes.  6656 states, n_fit = 18: 1504 us with a thread per state and
// its tables in scratch memory, now 381 with the sums over tau (411 with six divisions per zdiv).
__global__ __launch_bounds__(64) void qp_solve_kernel(const c128* __restrict__ sig_w, const c128* __restrict__ vhf,
                                                      const double* __restrict__ E0, QpFit fit, long dim, double mu,
                                                      double eta, double tol, double* __restrict__ E_out) {
  constexpr int L = 16, PER = QP_MAX_FIT / L;
  __shared__ zdd coef[64 / L][QP_MAX_FIT];
  const int lane = threadIdx.x, l = lane & (L - 1), base = lane & ~(L - 1), own = lane / L;
  const long state = static_cast<long>(blockIdx.x) * (64 / L) + own;
  const long I = state < dim ? state : dim - 1;
  const int n = fit.nfit;
  zdd* a = coef[own];

  // Thiele coefficients a_i = g_i(z_i): g_i(z_j) = (g_{i-1}(z_{i-1}) - g_{i-1}(z_j)) / ((z_j - z_{i-1}) g_{i-1}(z_j))
  zdd g[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int j = l + L * p;
    const c128 s = j < n ? sig_w[static_cast<long>(j) * dim + I] : c128{1.0, 0.0};
    g[p] = zd(s.x, s.y);
    if (j == 0) a[0] = g[p];
  }
  __syncthreads();
  for (int i = 1; i < n; ++i) {
    const zdd gd = a[i - 1];
    const zdd zi = zd(0.0, fit.zim[i - 1]);
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int j = l + L * p;
      if (j >= i && j < n) {
        g[p] = zdiv(zsub(gd, g[p]), zmul(zsub(zd(0.0, fit.zim[j]), zi), g[p]));
        if (j == i) a[i] = g[p];
      }
    }
    __syncthreads();
  }
  const double v = vhf[I].x;
  auto res_f = [&](double e) { return e - v - pade_eval(fit, a, e - mu, eta).x; };

  // qp_eqn_bisection: bracket in steps of 0.01 Ha from the starting energy, then bisect.  The loops
  // end for the whole wave; a state that is done keeps its values.
  const double eps0 = E0[I], delta = 0.01;
  const double res0 = res_f(eps0);
  bool done = fabs(res0) < tol;
  double result = eps0;
  const bool down = res0 >= 0;
  const double sign = down ? -1.0 : 1.0;
  double edge = eps0;  // the last trial
  bool open = !done;
  for (int tried = 0; __any(open); tried += L) {
    double e = edge;
    for (int s = 0; s <= l; ++s) e += sign * delta;
    const double r = res_f(e);
    const bool more = down ? r > 0 : r < 0;  // at most 100001 trials
    const unsigned long long stop = __ballot(!more || tried + l >= 100000);
    const unsigned mine = static_cast<unsigned>(stop >> base) & 0xffffu;
    const double reached = __shfl(e, base + (mine ? __builtin_ctz(mine) : L - 1));
    if (open) {
      edge = reached;
      open = mine == 0;
    }
  }
  double e1 = down ? edge : eps0, e2 = down ? eps0 : edge;
  for (int halvings = 0; __any(!done);) {
    // node l of the tree of the next four levels (root 1, children 2 l where the residual is not
    // negative and 2 l + 1)
    double t1 = e1, t2 = e2, mid = 0.5 * (t1 + t2);
    for (int bit = 30 - __builtin_clz(l | 1); bit >= 0; --bit) {
      if ((l >> bit) & 1) t1 = mid;
      else t2 = mid;
      mid = 0.5 * (t1 + t2);
    }
    const double r = res_f(mid);
    int node = 1;
    for (int level = 0; level < 4; ++level, ++halvings) {
      const double rn = __shfl(r, base + (node & (L - 1))), mn = __shfl(mid, base + (node & (L - 1)));
      if (!done) {
        result = mn;
        if (!(fabs(rn) > tol) || halvings >= 200) done = true;
        else if (rn >= 0) e2 = mn;
        else e1 = mn;
        node = 2 * node + (rn >= 0 ? 0 : 1);
      }
    }
  }
  if (l == 0 && state < dim) E_out[state] = result;
}

// Sigma(iw_n) = Twt_ff Sigma(tau) at the fit frequencies (IAFT.hpp:55-57), a thread per (frequency, state).
// The order of the sum is part of the result: the continuation multiplies its last bits by the
// condition of the fit, and the bisection's end point moves with them.
__global__ __launch_bounds__(256) void qp_sigma_kernel(const c128* __restrict__ sig_t, const c128* __restrict__ Twt,
                                                       QpFit fit, int nt, long dim, c128* __restrict__ sig_w) {
  const long I = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
  if (I >= dim) return;
  const c128* row = Twt + static_cast<long>(fit.w[blockIdx.y]) * nt;
  double sr = 0.0, si = 0.0;
#pragma unroll 8
  for (int t = 0; t < nt; ++t) {
    const c128 T = row[t], S = sig_t[static_cast<long>(t) * dim + I];
    sr += T.x * S.x - T.y * S.y;
    si += T.x * S.y + T.y * S.x;
  }
  sig_w[static_cast<long>(blockIdx.y) * dim + I] = c128{sr, si};
}

}  // namespace

void qp_solve(hipStream_t s, const c128* sig_t, const c128* vhf, const double* E0, const c128* Twt, const QpFit& fit,
              int nt, long dim, double mu, double eta, double tol, c128* sig_w, double* E_out) {
  THCGW_REQUIRE(fit.nfit >= 2 && fit.nfit <= QP_MAX_FIT, "qp_solve: nfit must be in [2, 64]");
  if (dim <= 0) return;
  hipLaunchKernelGGL(qp_sigma_kernel, dim3(static_cast<unsigned>((dim + 255) / 256), fit.nfit), dim3(256), 0, s, sig_t,
                     Twt, fit, nt, dim, sig_w);
  THCGW_HIP(hipGetLastError());
  hipLaunchKernelGGL(qp_solve_kernel, dim3(static_cast<unsigned>((dim + 3) / 4)), dim3(64), 0, s, sig_w, vhf, E0, fit,
                     dim, mu, eta, tol, E_out);
  THCGW_HIP(hipGetLastError());
}

}  // namespace thcgw
