// dense_small.hip -- Cholesky + inverse and the tridiagonalisation of matrices
// up to order 192 in one workgroup, the matrix in its registers.
//
// The cooperative kernels of dense.hip and eigh.hip pay 3 to 5 us a column (or
// two grid barriers a 64-column block) for exchanges between workgroups; up to
// this order one workgroup holds the whole matrix, and a column costs one or
// two workgroup barriers.  What bounds a step is the instructions each
// wavefront issues beside the updates (a barrier and an LDS trip are 0.08 us,
// a square root and a quotient 0.05 us each), so the wavefronts are as few as
// the registers allow, and everything that depends on how far the
// factorisation has come is decided at compile time: the steps run in phases
// of 16, in which the finished row and column blocks are constants and only
// the blocks at the edge are masked per element.
//
// Element (i, j) belongs to thread (i mod RW, j mod 16), RW = threads / 16: a
// row's 16 threads are one DPP row of a wavefront, so row sums need no LDS.
// Times of one call, before (cooperative) and now: Cholesky + inverse n = 160:
// 277 -> 108 us; tridiagonalisation n = 160: 740 -> 271 us, n = 20: 68 -> 27 us.
#include <algorithm>
#include <cstdlib>
#include "chol_wg.h"
#include "context.h"

namespace qx {
namespace {

// v + (v of the lane S places on in its row of 16)
template <int S>
__device__ inline double add_ror(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x120 | S, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x120 | S, 0xf, 0xf, false);
  return v + __hiloint2double(hi, lo);
}
// sum over a row of 16 lanes, in every lane of it
__device__ inline double row_sum(double v) {
  v = add_ror<8>(v);
  v = add_ror<4>(v);
  v = add_ror<2>(v);
  return add_ror<1>(v);
}
__device__ inline double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// sum over the wavefront, in every lane
__device__ inline double wave_total(double v) {
  v = row_sum(v);
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

// ---- Cholesky and inverse ----------------------------------------------------
// S(i, j) at s[i + n j], lower triangle read; X = L^-1 row-major, X(i, j) at
// x[i n + j], zero above the diagonal; ok = {positive definite, 0}.
template <class S>
__global__ void __launch_bounds__(S::T) k_chol_inv_wg(const double* __restrict__ s, int n,
                                                      double* __restrict__ x, int* ok) {
  __shared__ CholLds<S> L;
  const int t = threadIdx.x, ti = t >> 4, tj = t & 15;
  double A[S::NR][S::NC];
#pragma unroll
  for (int r = 0; r < S::NR; ++r)
#pragma unroll
    for (int c = 0; c < S::NC; ++c) {
      const int i = ti + S::RW * r, j = tj + 16 * c;
      A[r][c] = (i < n && j < n) ? s[(size_t)max(i, j) + (size_t)n * min(i, j)] : 0.0;
      if (j == 0) L.src[0][i] = i == 0 ? 1.0 : A[r][c];
    }
  if (t == 0) L.piv[0] = A[0][0];
  bool good = true;
  chol_phase<S, 0>(A, L, n, t, ti, tj, good);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < S::NR; ++r) {
    const int i = ti + S::RW * r;
    const double il = i < n ? sqrt(L.inv[i]) : 0.0;
#pragma unroll
    for (int c = 0; c < S::NC; ++c) {
      const int j = tj + 16 * c;
      if (i < n && j < n) x[(size_t)i * n + j] = j < i ? A[r][c] * il : j == i ? il : 0.0;
    }
  }
  if (t == 0) {
    ok[0] = good ? 1 : 0;
    ok[1] = 0;
  }
}

// ---- tridiagonalisation --------------------------------------------------------
// As k_tridiag_coop: a (n x n column-major, full symmetric) -> d, e (e[i] couples
// i and i + 1, e[n - 1] = 0) and the unit reflector of step k in a(k+1 : n, k);
// n >= 3.
//
// The reflector stays unnormalised, H = I - u u^T / h with u = x - alpha e_{k+1}
// (x column k below the diagonal, h = |u|^2 / 2 = |x|^2 - alpha x_{k+1}), so the
// product with A does not wait for the norm: A u = q - alpha c with q = A x and
// c column k + 1, and u.(A u) = x.q - 2 alpha q_{k+1} + alpha^2 c_{k+1}.  Two
// barriers a step: q formed, then both sums, the square root and the quotient
// in one chain and the update A -= u w^T + w u^T, w = p / h - (u.p / 2 h^2) u.
// The columns of A keep u; the unit reflectors are scaled at the end.
template <class S>
struct TrdLds {
  double2 xc[2][S::NL];  // columns k and k + 1 below row k, zeros above
  double q[S::NL], e[S::NM], h[S::NM];
};

template <class S, int P>
__device__ inline void trd_phase(double (&A)[S::NR][S::NC], TrdLds<S>& L, int n, int t, int ti,
                                 int tj) {
  constexpr int NR = S::NR, NC = S::NC, RW = S::RW, NU = S::NU;
  constexpr int R0 = 16 * P / RW, RM = (16 * P + 16) / RW;  // first live, last masked row block
  const int lane = t & 63, ke = min(n - 2, 16 * P + 16);
  for (int k = 16 * P; k < ke; ++k) {
    const double2* X = L.xc[k & 1];
    double2* Xn = L.xc[(k & 1) ^ 1];
    const int k1 = k + 1, k2 = k + 2;
    // q = A x
    double acc[NR];
#pragma unroll
    for (int r = R0; r < NR; ++r) acc[r] = 0.0;
#pragma unroll
    for (int c = P; c < NC; ++c) {
      const double v = X[tj + 16 * c].x;
#pragma unroll
      for (int r = R0; r < NR; ++r) acc[r] += A[r][c] * v;
    }
#pragma unroll
    for (int r = R0; r < NR; ++r) acc[r] = row_sum(acc[r]);
    if (tj == 0) {
#pragma unroll
      for (int r = R0; r < NR; ++r)
        L.q[ti + RW * r] = r > RM || ti + RW * r > k ? acc[r] : 0.0;
    }
    __syncthreads();
    double sx = 0.0, sq = 0.0;
#pragma unroll
    for (int u = 16 * P / 64; u < NU; ++u) {
      const double x = X[lane + 64 * u].x;
      sx += x * x;
      sq += x * L.q[lane + 64 * u];
    }
    const double2 z1 = X[k1];
    const double q1 = L.q[k1];
    double2 zr[NR];
    double qr[NR];
#pragma unroll
    for (int r = R0; r < NR; ++r) {
      zr[r] = X[ti + RW * r];
      qr[r] = L.q[ti + RW * r];
    }
    const double nx2 = wave_total(sx), xq = wave_total(sq);
    const double rt = sqrt(nx2);
    const double alpha = z1.x >= 0.0 ? -rt : rt;
    const double h = nx2 - alpha * z1.x;
    const bool skip = !(2.0 * h > 1e-300);
    const double tau = skip ? 0.0 : 1.0 / h;
    const double al = skip ? 0.0 : alpha;
    const double gt = tau * (xq - 2.0 * al * q1 + al * al * z1.y) * tau;
    if (t == 0) {
      L.e[k] = skip ? z1.x : alpha;
      L.h[k] = skip ? 0.0 : h;
    }
    double ur[NR], fa[NR], fb[NR];
#pragma unroll
    for (int r = R0; r < NR; ++r) {
      ur[r] = zr[r].x;
      if (r <= RM) ur[r] -= ti + RW * r == k1 ? al : 0.0;
      fa[r] = -tau * ur[r];
      fb[r] = gt * ur[r] - tau * (qr[r] - al * zr[r].y);
    }
#pragma unroll
    for (int c = P; c < NC; ++c) {
      const int j = tj + 16 * c;
      const double2 z = X[j];
      double uj = z.x;
      if (c <= P + 1) uj -= j == k1 ? al : 0.0;
      const double pj = L.q[j] - al * z.y;
#pragma unroll
      for (int r = R0; r < NR; ++r) A[r][c] += fa[r] * pj + fb[r] * uj;
    }
    // columns k + 1 and k + 2 for the next step; column k is done and keeps u
    if (tj == (k1 & 15)) {
#pragma unroll
      for (int r = R0; r < NR; ++r) {
        const double v = P + 1 < NC && k1 == 16 * P + 16 ? A[r][P + 1 < NC ? P + 1 : P] : A[r][P];
        Xn[ti + RW * r].x = r > RM || ti + RW * r > k1 ? v : 0.0;
      }
    }
    if (tj == (k2 & 15)) {
#pragma unroll
      for (int r = R0; r < NR; ++r) {
        const double v = P + 1 < NC && k2 >= 16 * P + 16 ? A[r][P + 1 < NC ? P + 1 : P] : A[r][P];
        Xn[ti + RW * r].y = r > RM || ti + RW * r > k1 ? v : 0.0;
      }
    }
    const bool mine = tj == (k & 15);
#pragma unroll
    for (int r = R0; r < NR; ++r)
      A[r][P] = mine && (r > RM || ti + RW * r > k) ? ur[r] : A[r][P];
    __syncthreads();
  }
  if constexpr (P + 1 < NC)
    if (16 * (P + 1) < n - 2) trd_phase<S, P + 1>(A, L, n, t, ti, tj);
}

template <class S>
__global__ void __launch_bounds__(S::T) k_tridiag_wg(double* __restrict__ a, int n,
                                                     double* __restrict__ d,
                                                     double* __restrict__ e) {
  __shared__ TrdLds<S> L;
  const int t = threadIdx.x, ti = t >> 4, tj = t & 15;
  double A[S::NR][S::NC];
#pragma unroll
  for (int r = 0; r < S::NR; ++r)
#pragma unroll
    for (int c = 0; c < S::NC; ++c) {
      const int i = ti + S::RW * r, j = tj + 16 * c;
      A[r][c] = (i < n && j < n) ? a[(size_t)j + (size_t)n * i] : 0.0;
    }
  // the largest element is brought to [1/2, 1) by a power of two: h is a square
  // and u.(A u) a cube of the matrix's scale
  __shared__ double wmax[S::T / 64];
  double mx = 0.0;
#pragma unroll
  for (int r = 0; r < S::NR; ++r)
#pragma unroll
    for (int c = 0; c < S::NC; ++c) mx = fmax(mx, fabs(A[r][c]));
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
  if ((t & 63) == 0) wmax[t >> 6] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < S::T / 64; ++w) mx = fmax(mx, wmax[w]);
  const int sh = -__builtin_amdgcn_frexp_exp(mx);
#pragma unroll
  for (int r = 0; r < S::NR; ++r)
#pragma unroll
    for (int c = 0; c < S::NC; ++c) A[r][c] = ldexp(A[r][c], sh);
  for (int i = t; i < S::NL; i += S::T) {
    const bool in = i > 0 && i < n;
    L.xc[0][i] =
        make_double2(in ? ldexp(a[i], sh) : 0.0, in ? ldexp(a[(size_t)n + i], sh) : 0.0);
    L.xc[1][i] = make_double2(0.0, 0.0);
    L.q[i] = 0.0;
  }
  __syncthreads();
  trd_phase<S, 0>(A, L, n, t, ti, tj);
  // column n - 2 is the one published last
  for (int i = t; i < n; i += S::T)
    e[i] = ldexp(i < n - 2 ? L.e[i] : i == n - 2 ? L.xc[n & 1][n - 1].x : 0.0, -sh);
#pragma unroll
  for (int c = 0; c < S::NC; ++c) {
    const int j = tj + 16 * c;
    const double h = j < n - 2 ? L.h[j] : 0.0;
    const double inv = h > 0.0 ? 1.0 / sqrt(2.0 * h) : 0.0;
#pragma unroll
    for (int r = 0; r < S::NR; ++r) {
      const int i = ti + S::RW * r;
      if (i == j && i < n) d[i] = ldexp(A[r][c], -sh);
      if (i > j && i < n && j < n - 2) a[(size_t)i + (size_t)n * j] = A[r][c] * inv;
    }
  }
}

}  // namespace

// the orders the one-workgroup kernels take (QX_DENSE_COOP and QX_DENSE_LEGACY
// keep the cooperative and the multi-launch ones, for comparison)
bool dense_wg_ok(int n) {
  return n <= 192 && !std::getenv("QX_DENSE_COOP") && !std::getenv("QX_DENSE_LEGACY");
}

// the shape of order n: 64 VGPRs of matrix or less, 144 for the largest two
#define QX_WG_SHAPES(F) F(32, 64, 2) F(64, 128, 4) F(128, 256, 8) F(160, 512, 10) F(192, 512, 12)

int chol_inv_wg(Ctx* c, const double* s, int n, double* x, int* ok) {
#define QX_RUN(NMAX, T, NC)                                                                     \
  if (n <= NMAX) {                                                                              \
    hipLaunchKernelGGL((k_chol_inv_wg<Shape<T, NC>>), dim3(1), dim3(T), 0, c->stream, s, n, x,  \
                       ok);                                                                     \
    QX_CHECK(hipGetLastError());                                                                \
    return 0;                                                                                   \
  }
  QX_WG_SHAPES(QX_RUN)
#undef QX_RUN
  return -3;
}

int tridiag_wg(Ctx* c, double* a, int n, double* d, double* e) {
#define QX_RUN(NMAX, T, NC)                                                                   \
  if (n <= NMAX) {                                                                            \
    hipLaunchKernelGGL((k_tridiag_wg<Shape<T, NC>>), dim3(1), dim3(T), 0, c->stream, a, n, d, \
                       e);                                                                    \
    QX_CHECK(hipGetLastError());                                                              \
    return 0;                                                                                 \
  }
  QX_WG_SHAPES(QX_RUN)
#undef QX_RUN
  return -3;
}

}  // namespace qx
