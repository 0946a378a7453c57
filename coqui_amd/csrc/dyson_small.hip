// The Dyson step of small orders: A = 1 - V Pi is factored and A Y = V solved in registers, one workgroup
// per matrix, with W - V = Y - V, Tr[V Pi] and ln |Re det A| (scr_coulomb_t.cpp:180-196,
// thc_rpa.icc:141-163).
//
// Gauss-Jordan elimination with partial pivoting: thread (r, c) of T x T holds the E x E elements
// (r + a T, c + b T) of D = A - 1 and of the right-hand side.  Per column: its values and one pivot
// candidate per wave are in LDS; barrier; every thread takes the same maximum; the pivot row's owners
// scale it by the pivot and publish it; barrier; rank-1 update.  Rows are not exchanged: row p_k
// of the result is row k of Y.  A pivot candidate is |Re| + |Im| with its row number in the
// lowest 7 of the 52 mantissa bits, so that one floating-point maximum yields both (lowest row on
// ties).  The division of a pivot row by its pivot is put off to the end.
//
// Accuracy.  Every update rounds its product first and then once at the size of the element.  A comes
// close to 1 and Y to V at high frequencies, where W - V and ln det are small: the ones of A are kept
// out of D and added where a value is read (a column, the pivot row), and a pivot 1 + d on the diagonal
// counts as log1p(d).  While the mean eigenvalue of -V Pi is below kWeak the right-hand side holds
// B = Y - V in the same way; beyond, Y itself, which the elimination makes smaller than V.
// Frobenius error against extended precision, LU with two triangular solves = 1: 0.4 to 0.8 at
// |V Pi| = 1, 0.9 to 1.0 at 10 and 100, 0.01 where |W - V| = 0.006 |V| (orders 8 to 96).  A^-1 formed
// by elimination and multiplied by V has 1.1 to 2.0: it was taken out for that.
//
// What bounds it: FP64 vector arithmetic and the chain of a column (barrier, maximum, reciprocal,
// barrier) for a few hundred matrices.
#include "thcgw_internal.hpp"
#include "wave.hpp"

#include <cfloat>
#include <type_traits>
#include <utility>

namespace thcgw {
namespace {

constexpr double kWeak = 0.7;

__device__ __forceinline__ c128 cmul(c128 a, c128 b) { return c128{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
// c -= a b, the product rounded before it is subtracted: one rounding at the size of c
__device__ __forceinline__ void csub(c128& c, c128 a, c128 b) {
  c.x -= fma(a.x, b.x, -(a.y * b.y));
  c.y -= fma(a.x, b.y, a.y * b.x);
}

// SOLVE: W[b] = A^-1 V - V with V's member (b0 + b) % vmod; otherwise the trace and the determinant only.
template <int T, int E, bool SOLVE>
__global__ __launch_bounds__(T* T) __attribute__((amdgpu_waves_per_eu(!SOLVE || T == 32 || E < 3 ? 4 : E == 3 ? 3 : 2)))
void dyson_small_kernel(const c128* D, const c128* V, int vmod, int b0, int n, c128* W, c128* tr, double* ldet,
                        int* info) {
  constexpr int N = T * E, NW = T * T / 64, EB = SOLVE ? E : 1;
  __shared__ c128 colv[2][N], rowv[N], scale[N], pivot[N];
  __shared__ c128 delta[N];  // element (k, k) of D before step k
  __shared__ c128 rowb[SOLVE ? N : 1], vs[SOLVE ? N : 1][SOLVE ? N : 1];
  __shared__ double key[2][NW], red[4][NW];
  __shared__ int perm[N], rowpos[N];
  __shared__ int bad;  // first zero or non-finite pivot column + 1
  const int mat = blockIdx.x;
  const long m = static_cast<long>(n) * n;
  const int r = threadIdx.x / T, c = threadIdx.x % T;

  // sums over the workgroup, in its first thread
  auto block_sum = [&](double x, double* sh) {
    x = wave_reduce(x, AddOp{});
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = x;
  };
  auto total = [&](const double* sh) {
    double x = sh[0];
    for (int q = 1; q < NW; ++q) x += sh[q];
    return x;
  };

  c128 v[E][E], b[EB][EB];
  double re = 0.0, im = 0.0;
#pragma unroll
  for (int a = 0; a < E; ++a)
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int i = r + a * T, j = c + q * T;
      const bool in = i < n && j < n;
      const long e = static_cast<long>(i) * n + j;
      v[a][q] = in ? D[mat * m + e] : c128{0.0, 0.0};
      if (i == j) {
        re -= v[a][q].x;
        im -= v[a][q].y;
      }
      if constexpr (SOLVE) {
        vs[i][j] = in ? V[((b0 + mat) % vmod) * m + e] : c128{0.0, 0.0};
      }
    }
  block_sum(re, red[0]);
  block_sum(im, red[1]);
  double part = 1.0;  // of V that is kept out of B
  if constexpr (SOLVE) {
    __syncthreads();
    part = fabs(total(red[0])) < kWeak * n ? 1.0 : 0.0;
#pragma unroll
    for (int a = 0; a < E; ++a)
#pragma unroll
      for (int q = 0; q < E; ++q) {
        const c128 u = vs[r + a * T][c + q * T];
        b[a][q] = c128{(1.0 - part) * u.x, (1.0 - part) * u.y};
      }
  }
  unsigned used = 0;  // bit a: row r + a T was a pivot row or lies outside the matrix
#pragma unroll
  for (int a = 0; a < E; ++a) used |= static_cast<unsigned>(r + a * T >= n) << a;

  // Column values of element block q of thread column cc to LDS, and the largest candidate of the
  // wave's rows.
  auto publish = [&](auto q_tag, int cc, int buf) __attribute__((always_inline)) {
    constexpr int q = decltype(q_tag)::value;
    if (r == cc && c == cc) {  // the diagonal element: its one is due
      delta[c + q * T] = v[q][q];
      v[q][q].x += 1.0;
    }
    double best = -1.0;
#pragma unroll
    for (int a = 0; a < E; ++a) {
      // fmin: a NaN or an infinity becomes a pivot by its place and is found by its value then
      const double mag = fmin(fabs(v[a][q].x) + fabs(v[a][q].y), DBL_MAX);
      const unsigned off = (used << (31 - a)) & 0x80000000u;  // negative: loses every maximum
      const unsigned lo =
          (static_cast<unsigned>(__double2loint(mag)) & ~127u) | static_cast<unsigned>(127 - (r + a * T));
      best = fmax(best, __hiloint2double(static_cast<int>(static_cast<unsigned>(__double2hiint(mag)) | off),
                                         static_cast<int>(lo)));
    }
    // 64 / T thread rows per wave, T lanes apart
    if (T == 8) best = ror_with<8>(best, MaxOp{});
    if (T <= 16) best = swap_with<16>(best, MaxOp{});
    best = swap_with<32>(best, MaxOp{});
    if (c == cc) {
#pragma unroll
      for (int a = 0; a < E; ++a) colv[buf][r + a * T] = v[a][q];
      if (r % (64 / T) == 0) key[buf][threadIdx.x >> 6] = best;
    }
  };

  if (threadIdx.x == 0) bad = 0;
  publish(std::integral_constant<int, 0>{}, 0, 0);
  auto column = [&](auto q_tag, int kk) __attribute__((always_inline)) {  // column k = q T + kk
    constexpr int q = decltype(q_tag)::value;
    const int k = q * T + kk, buf = k & 1;
    __syncthreads();
    double best = key[buf][0];
#pragma unroll
    for (int t = 1; t < NW; ++t) best = fmax(best, key[buf][t]);
    const int p = __builtin_amdgcn_readfirstlane(127 - (__double2loint(best) & 127));
    const int pr = p % T, pa = p / T;
    if (r == pr) {  // the pivot row's owners (lanes of one wave) publish row / pivot
      const c128 piv = colv[buf][p];
      const double den = 1.0 / (piv.x * piv.x + piv.y * piv.y);
      const c128 s{piv.x * den, -piv.y * den};
      used |= 1u << pa;
      each([&](auto a) __attribute__((always_inline)) {
        if (a == pa) {
#pragma unroll
          for (int j = q; j < E; ++j) rowv[c + j * T] = cmul(v[a][j], s);
          if constexpr (SOLVE) {
#pragma unroll
            for (int j = 0; j < E; ++j) {
              const c128 u = vs[p][c + j * T];
              rowb[c + j * T] = cmul(c128{fma(part, u.x, b[a][j].x), fma(part, u.y, b[a][j].y)}, s);
            }
          }
          asm volatile("; row block %0" ::"n"(decltype(a)::value));
        }
      }, std::make_integer_sequence<int, E>{});
      if (c == r && p > k) rowv[p] = c128{rowv[p].x + s.x, rowv[p].y + s.y};  // the row's own one
      if (c == 0) {
        colv[buf][p] = c128{0.0, 0.0};  // the stored row stays as it is
        scale[p] = s;
        pivot[k] = piv;
        const bool ok = isfinite(piv.x) && isfinite(piv.y) && (piv.x != 0.0 || piv.y != 0.0);
        if (!ok && bad == 0) bad = k + 1;
        perm[k] = p;
        rowpos[p] = k;
      }
    }
    __syncthreads();
    c128 w[E], wb[EB];
#pragma unroll
    for (int j = q; j < E; ++j) w[j] = rowv[c + j * T];
    if constexpr (SOLVE) {
#pragma unroll
      for (int j = 0; j < E; ++j) wb[j] = rowb[c + j * T];
    }
#pragma unroll
    for (int a = 0; a < E; ++a) {
      asm volatile("" ::: "memory");  // one row's factor at a time in registers
      const c128 f = colv[buf][r + a * T];
#pragma unroll
      for (int j = q; j < E; ++j) csub(v[a][j], f, w[j]);
      if constexpr (SOLVE) {
#pragma unroll
        for (int j = 0; j < E; ++j) csub(b[a][j], f, wb[j]);
      }
    }
    if (kk + 1 < T) publish(q_tag, kk + 1, buf ^ 1);
    else if constexpr (q + 1 < E) publish(std::integral_constant<int, q + 1>{}, 0, buf ^ 1);
  };
  each([&](auto q_tag) __attribute__((always_inline)) {
    for (int kk = 0; kk < T && decltype(q_tag)::value * T + kk < n; ++kk) column(q_tag, kk);
  }, std::make_integer_sequence<int, E>{});
  __syncthreads();
  if (threadIdx.x == 0) info[mat] = bad;

  if constexpr (SOLVE) {  // row k of W: s (V_p + B_p) - V_k, for p = k with its large parts taken out
#pragma unroll
    for (int a = 0; a < E; ++a) {
      const int i = r + a * T;
      if (i < n) {
        const int k = rowpos[i];
        const c128 s = scale[i], d = delta[k];
        const bool small_d = fabs(d.x) + fabs(d.y) < 0.5;
#pragma unroll
        for (int q = 0; q < E; ++q) {
          const int j = c + q * T;
          if (j < n) {
            const c128 u = vs[i][j], uk = vs[k][j];
            c128 x = b[a][q];
            if (k == i && small_d && part != 0.0) {
              csub(x, d, u);
              x = cmul(x, s);
            } else {
              x = cmul(c128{fma(part, u.x, x.x), fma(part, u.y, x.y)}, s);
              x = c128{x.x - uk.x, x.y - uk.y};
            }
            W[mat * m + static_cast<long>(k) * n + j] = x;
          }
        }
      }
    }
  }
  if (tr || ldet) {
    double la = 0.0, ph = 0.0;  // a swap of rows turns the phase by pi, which |Re det| does not see
    const int k = threadIdx.x;
    if (k < n) {
      const c128 p = pivot[k], d = delta[k];
      const bool near = perm[k] == k && fabs(d.x) + fabs(d.y) < 0.5;
      la = near ? 0.5 * log1p(fma(d.x, d.x, fma(d.y, d.y, 2.0 * d.x))) : log(hypot(p.x, p.y));
      ph = atan2(p.y, p.x);
    }
    block_sum(la, red[2]);
    block_sum(ph, red[3]);
    __syncthreads();
    if (threadIdx.x == 0) {
      if (tr) tr[mat] = c128{total(red[0]), total(red[1])};
      if (ldet) ldet[mat] = total(red[2]) + log(fabs(cos(total(red[3]))));
    }
  }
}

}  // namespace

// Against LU with triangular solves (about 15 launches), the whole step: 84 matrices of order 24
// 150 -> 102 us, 48 227 -> 140, 64 268 -> 177, 96 423 -> 298; 2624 of order 24 292 -> 146, 64 1000 -> 830.
// Beyond order 64 the copy of V fills the LDS of a CU with one workgroup: 336 matrices of order 80 532 ->
// 476, of order 96 646 -> 549, but 2624 of order 80 2009 -> 2420, which puts the line at about 1024.  The
// determinant alone (rpa_ec): 168 of order 80 320 -> 258, 336 379 -> 403.  The whole system counts, not the
// chunk at hand, so that chunks of any size give the same bits.
bool dyson_small_fits(int n, long total, bool solve) {
  return n >= 1 && (n <= 64 || (n <= 96 && total <= (solve ? 1024 : 256)));
}

void dyson_small(hipStream_t s, const c128* D, const c128* V, int vmod, int b0, int n, int batch, c128* W, c128* tr,
                 double* ldet, int* info) {
  THCGW_REQUIRE(n >= 1 && n <= 96, "dyson_small: order must be in [1, 96]");
  if (batch <= 0) return;
  auto go = [&](auto t, auto e) {
    constexpr int T = t, E = e;
    if (W)
      hipLaunchKernelGGL((dyson_small_kernel<T, E, true>), dim3(batch), dim3(T * T), 0, s, D, V, vmod, b0, n, W, tr,
                         ldet, info);
    else
      hipLaunchKernelGGL((dyson_small_kernel<T, E, false>), dim3(batch), dim3(T * T), 0, s, D, V, vmod, b0, n, W, tr,
                         ldet, info);
    THCGW_HIP(hipGetLastError());
  };
  using std::integral_constant;
  // One wave per matrix (T = 8), whose barriers cost nothing, from one matrix per SIMD on.
  if (n <= 32 && batch >= 1024) {
    if (n <= 16) go(integral_constant<int, 8>{}, integral_constant<int, 2>{});
    else if (n <= 24) go(integral_constant<int, 8>{}, integral_constant<int, 3>{});
    else go(integral_constant<int, 8>{}, integral_constant<int, 4>{});
    return;
  }
  switch ((n + 15) / 16) {
    case 1: go(integral_constant<int, 16>{}, integral_constant<int, 1>{}); break;
    case 2: go(integral_constant<int, 16>{}, integral_constant<int, 2>{}); break;
    case 3: go(integral_constant<int, 16>{}, integral_constant<int, 3>{}); break;
    case 4: go(integral_constant<int, 16>{}, integral_constant<int, 4>{}); break;
    default: go(integral_constant<int, 32>{}, integral_constant<int, 3>{}); break;
  }
}

}  // namespace thcgw
