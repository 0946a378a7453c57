// Inverses of the Matsubara matrices X(n, k) = (iw_n + mu) S_k - H0_k - F_k - Sigma(iw_n, k) of
// order <= 128, one workgroup per matrix, or only the traces Tr[X^-1 S_k] that the electron
// number needs (simple_dyson.cpp:65-78,130-172).
//
// The matrix is formed in registers and inverted there in place by Gauss-Jordan elimination
// with partial pivoting: thread (r, c) of T x T holds the E x E elements (r + a T, c + b T).
// Per column: its values and one pivot candidate per wave (published at the end of the
// step before) are in LDS; barrier; every thread takes the same maximum; the pivot row's
// owners scale it by the pivot and publish it; barrier; rank-1 update.  Rows are not
// exchanged: the pivot row of column k stays where it is (row p_k), and X^-1[k][p_j] = B[p_k][j]
// at the end.  A candidate is |Re| + |Im| with its row number in the lowest 7 of the 52
// mantissa bits, so that one floating-point maximum yields both (lowest row on ties).
// The division of a pivot row by its pivot is put off to the end: row p_k is scale[p_k] times
// the stored row, whose own later updates need just its stored column values, and the identity's
// element (p_k, k) is added there too.  So no register row is picked for writing in a column step.
// An update rounds its product first and then once at the size of the element: the Frobenius error of G is
// 0.97 times that of LU with triangular solves, 1.02 with the two real products subtracted one
// after the other (which takes 5% less at order 78).
//
// What bounds it: FP64 vector arithmetic (8 n^3 flops per matrix) and two barriers per column.
// Memory traffic is one read of Sigma(iw) and one write of the inverse.  T = 16 with E = n / 16
// rounded up wastes little padding and leaves 2-8 workgroups per CU to hide the barriers; up to
// E = 6 (n <= 96) the elements fit the registers (E = 7 spills 90 of them in every column step),
// and n <= 128 takes T = 32, E = 4; many matrices of order <= 32 take T = 8, one wave each.
// N(mu) over N_k = 64 and 80 frequencies (5120 inverses with the transform and the transfer of the
// traces), batched LU with triangular solves and a row gather through memory -> this kernel:
// order 16 1.34 -> 0.15 ms, 26 2.18 -> 0.26, 52 5.17 -> 0.93, 78 9.83 -> 2.12, 96 13.2 -> 3.17,
// 104 15.5 -> 6.0, 128 20.7 -> 7.7.  At order 78 the inversion takes 1.36 ms, 14 TFLOP/s of
// vector arithmetic: two workgroups per CU (200 registers) hide half of the column step's
// chain of barrier, maximum, reciprocal, barrier; a budget of three workgroups spills (1.65 ms).
#include "thcgw_internal.hpp"
#include "wave.hpp"

#include <cfloat>
#include <type_traits>
#include <utility>

namespace thcgw {
namespace {

__device__ __forceinline__ c128 cmul(c128 a, c128 b) { return c128{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }

// INVERSE: Out = X^-1.  TRACES: tr_out = Tr[X^-1 S].
enum MatsubaraJob { INVERSE, TRACES };

template <int T, int E, MatsubaraJob JOB>
__global__ __launch_bounds__(T* T) __attribute__((amdgpu_waves_per_eu(T == 16 && E > 4 ? 2 : 4)))
void matsubara_inverse_kernel(const c128* H0, const c128* F, const c128* S, const c128* Sw, const long* wn, double beta,
                              double mu, int nk, int n, c128* Out, c128* tr_out, int* info) {
  constexpr int N = T * E, NW = T * T / 64;
  __shared__ c128 colv[2][N], rowv[N], scale[N];
  __shared__ double key[2][T * T / 64];
  __shared__ int perm[N], rowpos[N];
  __shared__ double red[2][NW];
  __shared__ int bad;  // first zero or non-finite pivot column + 1
  const long b = blockIdx.x, m = static_cast<long>(n) * n;
  const long kofs = (b % nk) * m;
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

  c128 v[E][E];
  {
    const double wi = static_cast<double>(wn[b / nk]) * M_PI / beta;
#pragma unroll
    for (int a = 0; a < E; ++a)
#pragma unroll
      for (int q = 0; q < E; ++q) {
        const int i = r + a * T, j = c + q * T;
        v[a][q] = c128{0.0, 0.0};
        if (i < n && j < n) {
          const long e = static_cast<long>(i) * n + j;
          const c128 sij = S ? S[kofs + e] : c128{i == j ? 1.0 : 0.0, 0.0};
          const c128 h = H0 ? H0[kofs + e] : c128{0.0, 0.0};
          const c128 f = F[kofs + e], sw = Sw[b * m + e];
          v[a][q] = c128{mu * sij.x - wi * sij.y - h.x - f.x - sw.x, mu * sij.y + wi * sij.x - h.y - f.y - sw.y};
        }
      }
  }
  unsigned used = 0;  // bit a: row r + a T was a pivot row or lies outside the matrix
#pragma unroll
  for (int a = 0; a < E; ++a) used |= static_cast<unsigned>(r + a * T >= n) << a;

  // Column values of element block q of thread column cc to LDS, which leaves zeros (the column
  // of the identity), and the largest candidate of the wave's rows.
  auto publish = [&](auto q_tag, int cc, int buf) __attribute__((always_inline)) {
    constexpr int q = decltype(q_tag)::value;
    double best = -1.0;
#pragma unroll
    for (int a = 0; a < E; ++a) {
      // fmin: a NaN or an infinity becomes a pivot by its place and is found by its value then
      const double mag = fmin(fabs(v[a][q].x) + fabs(v[a][q].y), DBL_MAX);
      const unsigned off = (used << (31 - a)) & 0x80000000u;  // negative: loses every maximum
      const unsigned lo = (static_cast<unsigned>(__double2loint(mag)) & ~127u) | static_cast<unsigned>(127 - (r + a * T));
      best = fmax(best, __hiloint2double(static_cast<int>(static_cast<unsigned>(__double2hiint(mag)) | off),
                                         static_cast<int>(lo)));
    }
    // 64 / T thread rows per wave, T lanes apart
    if (T == 8) best = ror_with<8>(best, MaxOp{});
    if (T <= 16) best = swap_with<16>(best, MaxOp{});
    best = swap_with<32>(best, MaxOp{});
    if (c == cc) {
#pragma unroll
      for (int a = 0; a < E; ++a) {
        colv[buf][r + a * T] = v[a][q];
        v[a][q] = c128{0.0, 0.0};
      }
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
    for (int t = 1; t < T * T / 64; ++t) best = fmax(best, key[buf][t]);
    const int p = __builtin_amdgcn_readfirstlane(127 - (__double2loint(best) & 127));
    const int pr = p % T, pa = p / T;
    if (r == pr) {  // the pivot row's owners (one wave) publish w = row / pivot
      const c128 piv = colv[buf][p];
      const double den = 1.0 / (piv.x * piv.x + piv.y * piv.y);
      const c128 s{piv.x * den, -piv.y * den};
      used |= 1u << pa;
      each([&](auto a) __attribute__((always_inline)) {
        if (a == pa) {
#pragma unroll
          for (int j = 0; j < E; ++j) rowv[c + j * T] = (j == q && c == kk) ? s : cmul(v[a][j], s);
          asm volatile("; row block %0" ::"n"(decltype(a)::value));
        }
      }, std::make_integer_sequence<int, E>{});
      if (c == 0) {
        colv[buf][p] = c128{0.0, 0.0};  // the stored row stays as it is
        scale[p] = s;
        const bool ok = isfinite(piv.x) && isfinite(piv.y) && (piv.x != 0.0 || piv.y != 0.0);
        if (!ok && bad == 0) bad = k + 1;
        perm[k] = p;
        rowpos[p] = k;
      }
    }
    __syncthreads();
    c128 w[E];
#pragma unroll
    for (int j = 0; j < E; ++j) w[j] = rowv[c + j * T];
#pragma unroll
    for (int a = 0; a < E; ++a) {
      asm volatile("" ::: "memory");  // one row's factor at a time in registers
      const c128 f = colv[buf][r + a * T];
#pragma unroll
      for (int j = 0; j < E; ++j) {
        v[a][j].x -= fma(f.x, w[j].x, -(f.y * w[j].y));
        v[a][j].y -= fma(f.x, w[j].y, f.y * w[j].x);
      }
    }
    if (kk + 1 < T) publish(q_tag, kk + 1, buf ^ 1);
    else if constexpr (q + 1 < E) publish(std::integral_constant<int, q + 1>{}, 0, buf ^ 1);
  };
  auto columns = [&](auto q_tag) __attribute__((always_inline)) {
    for (int kk = 0; kk < T && decltype(q_tag)::value * T + kk < n; ++kk) column(q_tag, kk);
  };
  columns(std::integral_constant<int, 0>{});
  if constexpr (E > 1) columns(std::integral_constant<int, 1>{});
  if constexpr (E > 2) columns(std::integral_constant<int, 2>{});
  if constexpr (E > 3) columns(std::integral_constant<int, 3>{});
  if constexpr (E > 4) columns(std::integral_constant<int, 4>{});
  if constexpr (E > 5) columns(std::integral_constant<int, 5>{});
  __syncthreads();
  if (threadIdx.x == 0) info[b] = bad;
  // the scaled rows, with the ones left out so far
#pragma unroll
  for (int a = 0; a < E; ++a) {
    const int i = r + a * T;
    if (i < n) {
      const c128 s = scale[i];
#pragma unroll
      for (int q = 0; q < E; ++q) {
        const int j = c + q * T;
        if (j < n) v[a][q] = cmul(c128{v[a][q].x + (perm[j] == i ? 1.0 : 0.0), v[a][q].y}, s);
      }
    }
  }

  if constexpr (JOB == TRACES) {  // Tr[X^-1 S] = sum over this matrix of X^-1[k][p_j] S[p_j][k]
    double re = 0.0, im = 0.0;
#pragma unroll
    for (int a = 0; a < E; ++a)
#pragma unroll
      for (int q = 0; q < E; ++q) {
        const int i = r + a * T, j = c + q * T;
        if (i < n && j < n) {
          const int row = rowpos[i], col = perm[j];
          if (S) {
            const c128 t = cmul(v[a][q], S[kofs + static_cast<long>(col) * n + row]);
            re += t.x;
            im += t.y;
          } else if (row == col) {
            re += v[a][q].x;
            im += v[a][q].y;
          }
        }
      }
    block_sum(re, red[0]);
    block_sum(im, red[1]);
    __syncthreads();
    if (threadIdx.x == 0) tr_out[b] = c128{total(red[0]), total(red[1])};
  } else {
    c128* Ob = Out + b * m;
#pragma unroll
    for (int a = 0; a < E; ++a)
#pragma unroll
      for (int q = 0; q < E; ++q) {
        const int i = r + a * T, j = c + q * T;
        if (i < n && j < n) Ob[static_cast<long>(rowpos[i]) * n + perm[j]] = v[a][q];
      }
  }
}

struct InverseArgs {
  const c128 *H0, *F, *S, *Sw;
  const long* wn;
  double beta, mu;
  int nk;
  c128 *Out, *tr;
  int* info;
};

template <MatsubaraJob JOB>
void launch_inverse(hipStream_t s, const InverseArgs& x, int n, int count) {
  auto go = [&](auto t, auto e) {
    constexpr int T = t, E = e;
    hipLaunchKernelGGL((matsubara_inverse_kernel<T, E, JOB>), dim3(count), dim3(T * T), 0, s, x.H0, x.F, x.S, x.Sw, x.wn,
                       x.beta, x.mu, x.nk, n, x.Out, x.tr, x.info);
    THCGW_HIP(hipGetLastError());
  };
  using std::integral_constant;
  // Many small matrices: one wave each (T = 8), whose barriers cost nothing.  Electron number, T = 16 -> 8, on 5120
  // matrices of order 16 163 -> 138 us, 24 249 -> 203, 32 316 -> 279; on 160 of order 16 104 -> 103,
  // 24 111 -> 113, 32 117 -> 127: the line lies at one matrix per SIMD.
  if (n <= 32 && count >= 1024) {
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
    case 5: go(integral_constant<int, 16>{}, integral_constant<int, 5>{}); break;
    case 6: go(integral_constant<int, 16>{}, integral_constant<int, 6>{}); break;
    default: go(integral_constant<int, 32>{}, integral_constant<int, 4>{}); break;
  }
}

}  // namespace

bool matsubara_inverse_fits(int no) { return no >= 1 && no <= 128; }

void matsubara_inverse(hipStream_t s, const c128* H0, const c128* F, const c128* S, const c128* Sw, const long* wn,
                       double beta, double mu, int nw, int nk, int no, c128* Out, c128* tr, int* info) {
  THCGW_REQUIRE(matsubara_inverse_fits(no), "matsubara_inverse: order must be in [1, 128]");
  THCGW_REQUIRE((Out != nullptr) != (tr != nullptr), "matsubara_inverse: either the inverses or the traces");
  const long count = static_cast<long>(nw) * nk;
  THCGW_REQUIRE(count < (1L << 30), "Dyson for G: too many matrices");
  if (count == 0) return;
  const InverseArgs x{H0, F, S, Sw, wn, beta, mu, nk, Out, tr, info};
  if (tr) launch_inverse<TRACES>(s, x, no, static_cast<int>(count));
  else launch_inverse<INVERSE>(s, x, no, static_cast<int>(count));
}

}  // namespace thcgw
