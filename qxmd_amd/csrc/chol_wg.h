// chol_wg.h -- Cholesky factorisation and inverse of a matrix held in the
// registers of one workgroup, in phases of 16 columns: the whole matrix up to
// order 192 (dense_small.hip) and the 64 x 64 diagonal blocks of larger ones
// (dense.hip).
//
// Right-looking, in place: at step k element (i > k, j) holds the Schur
// complement for j > k and T(i, j) = -sum_{m < k} L(i, m) X(m, j) for j < k
// (X(k, j) = T(k, j) / L(k, k)).  One update A(i, j) -= A(i, k) / d src(j) does
// both, d the pivot, with src = column k right of k, row k left of it and 1 at
// it (where A(i, k) itself starts from 0).  Lower triangle only.
//
// A pivot counts as positive above 1e-30, the guard of rsdecmp, at every order.
// The quotients A(i, k) / d are corrected by their remainder, so that an A(i, k)
// equal to d gives one: the rows of two equal bands held here then stay equal,
// and the second one's pivot is zero or negative, never a positive rounding
// residue (n = 160: 111 us with these two FMAs a row and without).
#pragma once
#include <hip/hip_runtime.h>

namespace qx {

// one shape: T threads, orders up to 16 NC = RW NR
template <int T_, int NC_>
struct Shape {
  static constexpr int T = T_, RW = T / 16, NC = NC_, NR = 16 * NC / RW, NM = 16 * NC;
  static constexpr int NU = (NM + 63) / 64, NL = 64 * NU;
};

template <class S>
struct CholLds {
  double src[2][S::NM], piv[2], inv[S::NM];
};

template <class S, int P>
__device__ inline void chol_phase(double (&A)[S::NR][S::NC], CholLds<S>& L, int n, int t, int ti,
                                  int tj, bool& good) {
  constexpr int NR = S::NR, NC = S::NC, RW = S::RW;
  constexpr int R0 = 16 * P / RW, RM = (16 * P + 16) / RW;  // first live, last masked row block
  const int ke = min(n, 16 * P + 16);
  for (int k = 16 * P; k < ke; ++k) {
    const int q = k & 1, k1 = k + 1;
    const double* src = L.src[q];
    double* nsrc = L.src[q ^ 1];
    __syncthreads();
    const double d = L.piv[q];
    double l[NR], u[NC];
#pragma unroll
    for (int r = R0; r < NR; ++r) l[r] = src[ti + RW * r];
#pragma unroll
    for (int c = 0; c < NC; ++c) u[c] = src[tj + 16 * c];
    const bool pos = d > 1e-30;
    good = good && pos;
    const double id = pos ? 1.0 / d : 0.0;
    if (t == 0) L.inv[k] = id;
    const bool mine = tj == (k & 15);
#pragma unroll
    for (int r = R0; r < NR; ++r) {
      const double w = l[r] * id;
      l[r] = -fma(fma(-w, d, l[r]), id, w);
      if (r <= RM) l[r] = ti + RW * r > k ? l[r] : 0.0;
      A[r][P] = mine && (r > RM || ti + RW * r > k) ? 0.0 : A[r][P];
    }
#pragma unroll
    for (int r = R0; r < NR; ++r)
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (16 * c < RW * (r + 1)) A[r][c] += l[r] * u[c];
    // the next column below its pivot, the next row left of it, the pivot
    if (tj == (k1 & 15)) {
#pragma unroll
      for (int r = R0; r < NR; ++r) {
        const double v = k1 == 16 * P + 16 ? (P + 1 < NC ? A[r][P + 1 < NC ? P + 1 : P] : 0.0)
                                           : A[r][P];
        if (r > RM || ti + RW * r > k1) nsrc[ti + RW * r] = v;
        if (r <= RM && ti + RW * r == k1) L.piv[q ^ 1] = v;
      }
    }
#pragma unroll
    for (int r = R0; r <= RM && r < NR; ++r)
      if (ti + RW * r == k1) {
#pragma unroll
        for (int c = 0; c <= P + 1 && c < NC; ++c) {
          const int j = tj + 16 * c;
          if (c < P || j < k1) nsrc[j] = A[r][c];
          else if (j == k1) nsrc[j] = 1.0;
        }
      }
  }
  if constexpr (P + 1 < NC)
    if (16 * (P + 1) < n) chol_phase<S, P + 1>(A, L, n, t, ti, tj, good);
}

}  // namespace qx
