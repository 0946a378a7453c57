// Batched dense LU with partial pivoting and triangular solves, complex<double>.
//
// The reference inverts (I - V Pi) with getrf + getri per (q, iW_n)
// (scr_coulomb_t.cpp:188 -> slate_ops.hpp:324-333) and takes det(I - Pi V) from the
// LU factors (thc_rpa.icc:151, slate_ops.hpp:397-403).  nda hands its C-order
// matrices to column-major LAPACK, i.e. LAPACK factors the transpose.  The same is
// done here: a row-major n x n matrix A is viewed as the column-major M = A^T and
// factored as M = P L U, which in row-major terms is
//
//     A = Lt Ut Pt,   Lt = U^T (lower, non-unit),  Ut = L^T (upper, unit diagonal),
//
// with Pt a sequence of column swaps.  Pivot rows of M are contiguous rows of A, so
// the pivot search and the rank-1 updates of the panel read contiguous memory.
//
// The factorisation is recursive (split the column panel in two, factor the left
// half, update the right half with a triangular solve and a GEMM, factor it, swap
// back) so that most flops run in the MFMA GEMM kernel with large K.  The leaves
// are 16-wide panels factored in registers by one workgroup per matrix.
#include "thcgw_internal.hpp"

#include "tri_leaf.hpp"

#include <cfloat>

namespace thcgw {
namespace {

__device__ __forceinline__ c128 cmul(c128 a, c128 b) {
  return c128{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
__device__ __forceinline__ c128 crecip(c128 d) {
  const double s = 1.0 / (d.x * d.x + d.y * d.y);
  return c128{d.x * s, -d.y * s};
}

constexpr int MAX_ORDER = 2048;

// Factor the M-column panel [j0, j0+w) over M-rows [j0, n), i.e. the A-rows [j0, j0+w)
// restricted to A-columns [j0, n).  Thread t owns the panel entries of A-columns j0 + t + s T,
// s < R, in registers.  Column swaps are applied inside the panel rows only; the caller
// applies them to the other rows.
//
// What bounds it: the chain of a column step (largest entry, barrier, pivot row to LDS, barrier,
// rank-1 update), so the workgroup is as small as the rows allow, and several share a CU.  The
// columns stay where they are until the end: who stands where is kept in LDS, and the swaps are made
// by the final stores.  A pivot candidate is |Re| + |Im| with 2047 minus the column's number in the
// lowest 11 mantissa bits, so that one floating-point maximum yields the value and the place
// (lowest column on ties).  NaN counts as zero and infinity as the largest number; what the
// pivot really holds is looked at when it has been read.  An update rounds its product first and
// then once at the size of the entry: A comes close to 1, and its two real products subtracted one after
// the other (four instructions instead of six, 1% of the panel) made W 1.3 times less accurate.
// Panels of 168 matrices of order 200, on average: 50.6 us with 1024 threads for any order, now 18.4;
// of 164 matrices of order 800: 57.5 us, now 25.2.
template <int T, int R, int W>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(T * R <= 256 ? 4 : R * W > 16 ? 2 : 4))) void getf2_panel_kernel(
    c128* A, long sA, int lda, int n, int j0, int w, int* ipiv,
                                                        int* info) {
  static_assert(T * R <= MAX_ORDER, "the candidate's index field has 11 bits");
  constexpr int NW = T / 64;
  const int b = blockIdx.x;
  c128* Ab = A + static_cast<long>(b) * sA + static_cast<long>(j0) * lda + j0;
  int* piv = ipiv + static_cast<long>(b) * n;
  const int t = threadIdx.x, m = n - j0;

  // Candidates double buffered by column parity: written before a column's first barrier, read
  // between its two; the pivot row is read after the second and rewritten after the next first.
  __shared__ double key[2][NW];
  __shared__ c128 prow[W];
  __shared__ short at[T * R], pos[T * R];  // column at a place, place of a column

  c128 v[R][W];
  unsigned used = 0;  // bit s: column t + s T was a pivot or lies outside the matrix
#pragma unroll
  for (int s = 0; s < R; ++s) {
    const int r = t + s * T;
    if (r >= m) used |= 1u << s;
    at[r] = pos[r] = static_cast<short>(r);
#pragma unroll
    for (int c = 0; c < W; ++c) v[s][c] = (r < m && c < w) ? Ab[static_cast<long>(c) * lda + r] : c128{0.0, 0.0};
  }

  int first_bad = 0;
  each([&](auto column) __attribute__((always_inline)) {
    constexpr int c = column;
    if (c < w) {
      double best = -1.0;
#pragma unroll
      for (int s = 0; s < R; ++s) {
        const double mag = fmin(fmax(fabs(v[s][c].x) + fabs(v[s][c].y), 0.0), DBL_MAX);
        const unsigned lo = (static_cast<unsigned>(__double2loint(mag)) & ~2047u) | static_cast<unsigned>(2047 - (t + s * T));
        const unsigned hi = static_cast<unsigned>(__double2hiint(mag)) | ((used << (31 - s)) & 0x80000000u);
        best = fmax(best, __hiloint2double(static_cast<int>(hi), static_cast<int>(lo)));
      }
      best = wave_reduce(best, MaxOp{});
      if ((t & 63) == 0) key[c & 1][t >> 6] = best;
      __syncthreads();
      best = key[c & 1][0];
#pragma unroll
      for (int q = 1; q < NW; ++q) best = fmax(best, key[c & 1][q]);
      const int p = __builtin_amdgcn_readfirstlane(2047 - (__double2loint(best) & 2047));
      if (t == p % T) {
        each([&](auto own) __attribute__((always_inline)) {
          constexpr int s = own;
          if (s == p / T) {
            used |= 1u << s;
#pragma unroll
            for (int cc = 0; cc < W; ++cc) prow[cc] = v[s][cc];
            asm volatile("; column %0" ::"n"(s));
          }
        }, std::make_integer_sequence<int, R>{});
      }
      __syncthreads();
      if (t == 0) {  // swap the places c and pos[p]; no other thread reads them before the end
        const int q = pos[p], o = at[c];
        piv[j0 + c] = j0 + q;
        at[q] = static_cast<short>(o);
        pos[o] = static_cast<short>(q);
        at[c] = static_cast<short>(p);
        pos[p] = static_cast<short>(c);
      }
      // scale below the pivot and update the rest of the panel.  A zero or non-finite pivot
      // is reported in info (first such column + 1), as a singular matrix.
      const c128 d = prow[c];
      const bool zero = d.x == 0.0 && d.y == 0.0;
      if (first_bad == 0 && (zero || !(isfinite(d.x) && isfinite(d.y)))) first_bad = j0 + c + 1;
      if (!zero) {
        const c128 inv = crecip(d);
#pragma unroll
        for (int s = 0; s < R; ++s)
          if (!((used >> s) & 1)) {
            const c128 l = cmul(v[s][c], inv);
            v[s][c] = l;
#pragma unroll
            for (int cc = c + 1; cc < W; ++cc) {
              const c128 u = prow[cc];
              v[s][cc].x -= fma(l.x, u.x, -(l.y * u.y));
              v[s][cc].y -= fma(l.x, u.y, l.y * u.x);
            }
          }
      }
    }
  }, std::make_integer_sequence<int, W>{});
  __syncthreads();

#pragma unroll
  for (int s = 0; s < R; ++s) {
    const int r = t + s * T;
    if (r < m) {
      const int o = pos[r];
#pragma unroll
      for (int c = 0; c < W; ++c)
        if (c < w) Ab[static_cast<long>(c) * lda + o] = v[s][c];
    }
  }
  if (t == 0 && first_bad != 0 && info[b] == 0) info[b] = first_bad;
}

__global__ void fill_int_kernel(int* p, int n, int v) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

// Apply the column swaps ipiv[k0..k1) (in order) to A-rows [r0, r1).
__global__ __launch_bounds__(256) void laswp_kernel(c128* A, long sA, int lda, int n, int r0, int r1, int k0, int k1,
                                                    const int* ipiv) {
  const int b = blockIdx.y;
  const int row = r0 + blockIdx.x * 256 + threadIdx.x;
  if (row >= r1) return;
  c128* Ar = A + static_cast<long>(b) * sA + static_cast<long>(row) * lda;
  const int* piv = ipiv + static_cast<long>(b) * n;
  for (int k = k0; k < k1; ++k) {
    const int p = piv[k];
    if (p != k && p >= 0 && p < n) {  // the panel writes pivots in [k, n); the range check guards the read
      const c128 x = Ar[k];
      Ar[k] = Ar[p];
      Ar[p] = x;
    }
  }
}

constexpr int LB = 32;  // triangular-solve leaf size

const Cplx kOne{1.0, 0.0};
const Cplx kMinusOne{-1.0, 0.0};

int split_point(int n, int unit) {
  int h = (n / 2 / unit) * unit;
  return h < unit ? unit : h;
}

// Above order 128 the recursions split at multiples of the 64-wide GEMM tile, so that no
// update product has a half-filled tile row or column at the split.
int tile_split(int n, int unit) { return split_point(n, n > 128 ? 64 : unit); }

}  // namespace

// ---- triangular solves (batched, strides between matrices) ----------------------

// X U = T, U unit upper (nb x nb), T m x nb; T is overwritten with X.
void trsm_right_upper_unit(hipStream_t s, const c128* U, long sU, int ldu, c128* T, long sT, int ldt, int m, int nb,
                           int batch) {
  if (m <= 0 || nb <= 0 || batch <= 0) return;
  if (nb <= LB) {
    tri_leaf<TRI_ROW_UPPER_UNIT, LB>(s, U, sU, ldu, T, sT, ldt, m, nb, batch);
    return;
  }
  const int n1 = tile_split(nb, LB), n2 = nb - n1;
  trsm_right_upper_unit(s, U, sU, ldu, T, sT, ldt, m, n1, batch);
  // T2 -= X1 U12
  zgemm(s, OP_N, OP_N, m, n2, n1, kMinusOne, bp(T, sT), ldt, bp(U + n1, sU), ldu, kOne, T + n1, sT, ldt, batch);
  trsm_right_upper_unit(s, U + static_cast<long>(n1) * ldu + n1, sU, ldu, T + n1, sT, ldt, m, n2, batch);
}

// L X = B, L lower non-unit n x n, B n x ncol.
void trsm_left_lower(hipStream_t s, const c128* L, long sL, int ldl, c128* B, long sB, int ldb, int n, int ncol,
                     int batch) {
  if (n <= 0 || ncol <= 0 || batch <= 0) return;
  if (n <= LB) {
    tri_leaf<TRI_COL_LOWER, LB>(s, L, sL, ldl, B, sB, ldb, ncol, n, batch);
    return;
  }
  const int n1 = tile_split(n, LB), n2 = n - n1;
  trsm_left_lower(s, L, sL, ldl, B, sB, ldb, n1, ncol, batch);
  zgemm(s, OP_N, OP_N, n2, ncol, n1, kMinusOne, bp(L + static_cast<long>(n1) * ldl, sL), ldl, bp(B, sB), ldb, kOne,
        B + static_cast<long>(n1) * ldb, sB, ldb, batch);
  trsm_left_lower(s, L + static_cast<long>(n1) * ldl + n1, sL, ldl, B + static_cast<long>(n1) * ldb, sB, ldb, n2,
                  ncol, batch);
}

// U X = B, U upper unit n x n, B n x ncol.
void trsm_left_upper_unit(hipStream_t s, const c128* U, long sU, int ldu, c128* B, long sB, int ldb, int n, int ncol,
                          int batch) {
  if (n <= 0 || ncol <= 0 || batch <= 0) return;
  if (n <= LB) {
    tri_leaf<TRI_COL_UPPER_UNIT, LB>(s, U, sU, ldu, B, sB, ldb, ncol, n, batch);
    return;
  }
  const int n1 = tile_split(n, LB), n2 = n - n1;
  trsm_left_upper_unit(s, U + static_cast<long>(n1) * ldu + n1, sU, ldu, B + static_cast<long>(n1) * ldb, sB, ldb, n2,
                       ncol, batch);
  zgemm(s, OP_N, OP_N, n1, ncol, n2, kMinusOne, bp(U + n1, sU), ldu, bp(B + static_cast<long>(n1) * ldb, sB), ldb,
        kOne, B, sB, ldb, batch);
  trsm_left_upper_unit(s, U, sU, ldu, B, sB, ldb, n1, ncol, batch);
}

// ---- LU ------------------------------------------------------------------------

namespace {
void laswp(hipStream_t s, c128* A, long sA, int lda, int n, int r0, int r1, int k0, int k1, const int* ipiv,
           int batch) {
  if (r1 <= r0 || k1 <= k0) return;
  hipLaunchKernelGGL(laswp_kernel, dim3((r1 - r0 + 255) / 256, batch), dim3(256), 0, s, A, sA, lda, n, r0, r1, k0,
                     k1, ipiv);
  THCGW_HIP(hipGetLastError());
}

template <int T, int R, int W>
void launch_panel(hipStream_t s, c128* A, long sA, int lda, int n, int j0, int w, int* ipiv, int* info, int batch) {
  hipLaunchKernelGGL((getf2_panel_kernel<T, R, W>), dim3(batch), dim3(T), 0, s, A, sA, lda, n, j0, w, ipiv, info);
  THCGW_HIP(hipGetLastError());
}

// 16 columns as long as two per thread of a 512-thread workgroup reach (128 registers hold
// 2 x 16 entries), 8 beyond.
int panel_width(int rows) { return rows <= 1024 ? 16 : 8; }

void panel(hipStream_t s, c128* A, long sA, int lda, int n, int j0, int w, int* ipiv, int* info, int batch) {
  const int rows = n - j0;
  if (rows <= 64) launch_panel<64, 1, 16>(s, A, sA, lda, n, j0, w, ipiv, info, batch);
  else if (rows <= 128) launch_panel<128, 1, 16>(s, A, sA, lda, n, j0, w, ipiv, info, batch);
  else if (rows <= 256) launch_panel<256, 1, 16>(s, A, sA, lda, n, j0, w, ipiv, info, batch);
  else if (rows <= 512) launch_panel<256, 2, 16>(s, A, sA, lda, n, j0, w, ipiv, info, batch);
  else if (rows <= 1024) launch_panel<512, 2, 16>(s, A, sA, lda, n, j0, w, ipiv, info, batch);
  else launch_panel<1024, 2, 8>(s, A, sA, lda, n, j0, w, ipiv, info, batch);
}

void getrf_rec(hipStream_t s, c128* A, long sA, int lda, int n, int j0, int w, int* ipiv, int* info, int batch) {
  const int pw = panel_width(n - j0);
  if (w <= pw) {
    panel(s, A, sA, lda, n, j0, w, ipiv, info, batch);
    return;
  }
  const int w1 = tile_split(w, pw), w2 = w - w1;
  getrf_rec(s, A, sA, lda, n, j0, w1, ipiv, info, batch);
  laswp(s, A, sA, lda, n, j0 + w1, j0 + w, j0, j0 + w1, ipiv, batch);
  c128* diag = A + static_cast<long>(j0) * lda + j0;
  c128* T = A + static_cast<long>(j0 + w1) * lda + j0;
  trsm_right_upper_unit(s, diag, sA, lda, T, sA, lda, w2, w1, batch);
  zgemm(s, OP_N, OP_N, w2, n - j0 - w1, w1, kMinusOne, bp(T, sA), lda, bp(diag + w1, sA), lda, kOne, T + w1, sA, lda,
        batch);
  getrf_rec(s, A, sA, lda, n, j0 + w1, w2, ipiv, info, batch);
  laswp(s, A, sA, lda, n, j0, j0 + w1, j0 + w1, j0 + w, ipiv, batch);
}
}  // namespace

// In-place LU of `batch` row-major n x n matrices (stride sA): A = Lt Ut Pt as described
// above.  ipiv (batch x n) receives the column swaps, info (batch) 0 or first zero pivot + 1.
void getrf_batched(hipStream_t s, c128* A, long sA, int lda, int n, int* ipiv, int* info, int batch) {
  THCGW_REQUIRE(n >= 1 && n <= MAX_ORDER, "getrf: order must be in [1, 2048]");
  hipLaunchKernelGGL(fill_int_kernel, dim3((batch + 255) / 256), dim3(256), 0, s, info, batch, 0);
  THCGW_HIP(hipGetLastError());
  getrf_rec(s, A, sA, lda, n, 0, n, ipiv, info, batch);
}

}  // namespace thcgw
