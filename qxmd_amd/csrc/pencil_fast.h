// pencil_fast.h -- device kernels of the band-apply / density pencil FFTs for
// grids whose edges each factor as NA*NB with both factors <= 16 (QX_FFT_EDGES).
//
// A line transform of length N is done in two register steps with a single
// LDS exchange between them:
//   NP ("natural -> permuted"): step A, thread b < NB: DFT_NA over the NB-strided
//       elements b + NB*a, twiddle W_N^(b*ka); step B, thread ka < NA: DFT_NB over
//       the contiguous run NB*ka + b.  Index ka + NA*kb ends up at slot kb + NB*ka.
//   PN ("permuted -> natural"): the same two steps in reverse order.
// Every inverse transform of the band-apply is NP and every forward one PN, so
// the digit-transposed intermediate order never needs a reordering pass: the
// z planes of T1/T2 and the y/x slots of a plane are kept in slot order and
// V(r) is stored pre-permuted.  In x the inverse step B, the V(r) multiply and
// the forward step B' act on the same registers.
//
// Edges: the z kernels are compiled per n3 and the plane kernels per n1 (the
// x pass is two thirds of their arithmetic).  The y edge is n1 with the same
// split (Y_CUBE: constant strides) or any edge of the table, its two radices
// picked by a workgroup-uniform switch around each y loop; one kernel per
// (n1, n2) pair would be 39^2 of them.  The switch comes with radices up to 10
// and up to 16 (YKind): the FP64 radix-16 codelet alone takes the registers
// that two blocks per CU leave.  Against the Stockham kernels of pencil.hip,
// which take the other edges: H|psi> of 240 bands on 60 x 60 x 90, mixed, 1.446
// -> 0.391 ms; of 81 bands on 27 x 56 x 56, FP64, 0.290 -> 0.150 ms.
#pragma once
#include <algorithm>
#include <type_traits>
#include "context.h"

namespace qx {

// edge, NA, NB: the products of 2, 3, 5, 7 from 16 to 128 with both factors at
// most 16, the factors as equal as the codelets allow (a row of the x pass
// keeps max(NA, NB) lanes for both steps)
#define QX_FFT_EDGES_0(F) F(16, 4, 4) F(42, 6, 7) F(72, 8, 9) F(126, 9, 14) F(50, 5, 10)
#define QX_FFT_EDGES_1(F) F(18, 3, 6) F(45, 5, 9) F(75, 5, 15) F(128, 16, 8) F(54, 6, 9)
#define QX_FFT_EDGES_2(F) F(20, 4, 5) F(48, 6, 8) F(80, 8, 10) F(120, 12, 10) F(36, 6, 6)
#define QX_FFT_EDGES_3(F) F(21, 3, 7) F(49, 7, 7) F(81, 9, 9) F(112, 8, 14) F(60, 6, 10)
#define QX_FFT_EDGES_4(F) F(24, 4, 6) F(56, 7, 8) F(84, 7, 12) F(108, 9, 12) F(35, 5, 7)
#define QX_FFT_EDGES_5(F) F(25, 5, 5) F(63, 7, 9) F(90, 9, 10) F(105, 7, 15) F(30, 6, 5)
#define QX_FFT_EDGES_6(F) F(27, 3, 9) F(64, 8, 8) F(96, 12, 8) F(32, 4, 8)
#define QX_FFT_EDGES_7(F) F(28, 4, 7) F(70, 7, 10) F(98, 7, 14) F(100, 10, 10) F(40, 5, 8)
#define QX_FFT_EDGES(F)                                                                    \
  QX_FFT_EDGES_0(F) QX_FFT_EDGES_1(F) QX_FFT_EDGES_2(F) QX_FFT_EDGES_3(F) QX_FFT_EDGES_4(F) \
  QX_FFT_EDGES_5(F) QX_FFT_EDGES_6(F) QX_FFT_EDGES_7(F)
constexpr int kFftGroups = 8;

// y edge of a plane kernel: the x edge (cube), radices <= 10, radices <= 16
enum YKind { Y_CUBE = 0, Y_R10 = 1, Y_R16 = 2 };
constexpr int y_max_radix(int yk) { return yk == Y_R16 ? 16 : 10; }

constexpr int kFastThreads = 256;
// column pairs per z block: 16, or 8 where 32 complex lines of length N would
// pass 48 KiB of static LDS
__host__ __device__ constexpr int zpairs(int N, int elem_bytes) {
  return 2 * 16 * N * elem_bytes <= 49152 ? 16 : 8;
}

__host__ __device__ inline int slot_phys(int s, int NA, int NB) { return s / NB + NA * (s % NB); }

struct FastArgs {
  int n1, n2, n3, nH, hmin, hmax, npair, ncol, nplwex, nb, bp0;
  int ya, yb;  // radices of the y edge, n2 = ya * yb
  int sa, sr;  // row strides (elements) of the plane kernel's sphere tile and x strips
  const int *pt_col, *pt_z, *pair_p0, *col_hi, *col_kmod;
  const double* kin;
  const double* tw;  // exp(+2 pi i k / n) of the x (n1), y (n2) and z (n3) edges
};

template <typename T>
__device__ inline cplx<T> twid(const cplx<T>* tw, int k, int sign) {
  cplx<T> w = tw[k];
  if (sign < 0) w.y = -w.y;
  return w;
}

// ---- line steps (one thread, line in LDS with unit stride) ----------------
// step A and A' of an NA x nb line, step B and B' of an na x NB line
template <typename T, int NA>
__device__ inline void np_stepA(cplx<T>* L, int b, int nb, const cplx<T>* tw, int sign) {
  cplx<T> v[NA];
#pragma unroll
  for (int a = 0; a < NA; ++a) v[a] = L[b + nb * a];
  Dft<T, NA>::run(v, sign);
  int k = 0;
#pragma unroll
  for (int ka = 1; ka < NA; ++ka) {
    k += b;  // b * ka
    v[ka] = cmul(v[ka], twid(tw, k, sign));
  }
#pragma unroll
  for (int ka = 0; ka < NA; ++ka) L[b + nb * ka] = v[ka];
}
template <typename T, int NB>
__device__ inline void np_stepB(cplx<T>* L, int ka, int sign) {
  cplx<T> v[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) v[b] = L[NB * ka + b];
  Dft<T, NB>::run(v, sign);
#pragma unroll
  for (int kb = 0; kb < NB; ++kb) L[NB * ka + kb] = v[kb];
}
template <typename T, int NB>
__device__ inline void pn_stepB(cplx<T>* L, int ka, const cplx<T>* tw, int sign) {
  cplx<T> v[NB];
#pragma unroll
  for (int kb = 0; kb < NB; ++kb) v[kb] = L[NB * ka + kb];
  Dft<T, NB>::run(v, sign);
  int k = 0;
#pragma unroll
  for (int b = 1; b < NB; ++b) {
    k += ka;  // b * ka
    v[b] = cmul(v[b], twid(tw, k, sign));
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) L[NB * ka + b] = v[b];
}
template <typename T, int NA>
__device__ inline void pn_stepA(cplx<T>* L, int b, int nb, int sign) {
  cplx<T> v[NA];
#pragma unroll
  for (int ka = 0; ka < NA; ++ka) v[ka] = L[b + nb * ka];
  Dft<T, NA>::run(v, sign);
#pragma unroll
  for (int a = 0; a < NA; ++a) L[b + nb * a] = v[a];
}

// f(integral_constant<int, r>) for a workgroup-uniform radix r <= MAXR of the
// edge table
template <int MAXR, typename F>
__device__ inline void with_radix(int r, F&& f) {
#define QX_CASE(R) \
  case R: f(std::integral_constant<int, R>()); break;
  switch (r) {
    QX_CASE(3) QX_CASE(4) QX_CASE(5) QX_CASE(6) QX_CASE(7) QX_CASE(8) QX_CASE(9) QX_CASE(10)
    default:
      if constexpr (MAXR > 10) {
        switch (r) { QX_CASE(12) QX_CASE(14) QX_CASE(15) QX_CASE(16) }
      }
  }
#undef QX_CASE
}

__device__ inline int mirror_col_f(int col) {
  return col == 0 ? 0 : ((col & 1) ? col + 1 : col - 1);
}

// ---- z inverse: sphere -> T1[bp][z slot][col] ------------------------------
// psi32 (optional): receives the FP32 copy of the coefficients read;
// psis (optional): their bf16 hi | lo split instead (row stride ldk, lo half
// at offset slo), the operand of the split bf16x3 KB projection
template <typename T, int NA, int NB>
__global__ void __launch_bounds__(kFastThreads) k_zinv_f(FastArgs a, const double* __restrict__ psi,
                                                         cplx<T>* __restrict__ t1,
                                                         float* __restrict__ psi32,
                                                         unsigned short* __restrict__ psis,
                                                         int ldk, long slo) {
  constexpr int N = NA * NB;
  constexpr int PB = zpairs(N, (int)sizeof(cplx<T>));
  __shared__ cplx<T> tw[N];
  __shared__ cplx<T> lines[2 * PB][N];
  const int q0 = blockIdx.x * PB, q1 = min(q0 + PB, a.npair);
  const int bp = blockIdx.y;
  const int ba = 2 * (a.bp0 + bp), bb = ba + 1;
  const int c0 = q0 == 0 ? 0 : 2 * q0 - 1, c1 = 2 * q1 - 1, ncl = c1 - c0;
  load_tw<T>(tw, a.tw + 2 * (a.n1 + a.n2), N);
  for (int i = threadIdx.x; i < ncl * N; i += blockDim.x) lines[i / N][i % N] = mk<T>(0, 0);
  __syncthreads();
  const double* pa = psi + (size_t)ba * a.nplwex;
  const double* pb = psi + (size_t)bb * a.nplwex;
  const bool hasb = bb < a.nb;
  const int p0 = a.pair_p0[q0], p1 = a.pair_p0[q1];
  for (int p = p0 + threadIdx.x; p < p1; p += blockDim.x) {
    double ar = pa[2 * p], ai = pa[2 * p + 1];
    double br = hasb ? pb[2 * p] : 0.0, bi = hasb ? pb[2 * p + 1] : 0.0;
    if (psi32) {
      float* qa = psi32 + (size_t)ba * a.nplwex;
      qa[2 * p] = (float)ar;
      qa[2 * p + 1] = (float)ai;
      if (hasb) {
        qa[a.nplwex + 2 * p] = (float)br;
        qa[a.nplwex + 2 * p + 1] = (float)bi;
      }
    }
    if (psis) {
      unsigned h, l;
      unsigned short* qa = psis + (size_t)ba * ldk + 2 * p;
      split_bf16x2((float)ar, (float)ai, h, l);
      *reinterpret_cast<unsigned*>(qa) = h;
      *reinterpret_cast<unsigned*>(qa + slo) = l;
      if (hasb) {
        split_bf16x2((float)br, (float)bi, h, l);
        *reinterpret_cast<unsigned*>(qa + ldk) = h;
        *reinterpret_cast<unsigned*>(qa + ldk + slo) = l;
      }
    }
    int col = a.pt_col[p] - c0, z = a.pt_z[p];
    if (p == 0) {
      lines[col][0] = mk<T>((T)ar, (T)br);
    } else {
      lines[col][z] = mk<T>((T)(ar - bi), (T)(ai + br));
      lines[mirror_col_f(col + c0) - c0][z == 0 ? 0 : N - z] = mk<T>((T)(ar + bi), (T)(br - ai));
    }
  }
  __syncthreads();
  for (int it = threadIdx.x; it < ncl * NB; it += blockDim.x)
    np_stepA<T, NA>(lines[it / NB], it % NB, NB, tw, +1);
  __syncthreads();
  for (int it = threadIdx.x; it < ncl * NA; it += blockDim.x)
    np_stepB<T, NB>(lines[it / NA], it % NA, +1);
  __syncthreads();
  cplx<T>* out = t1 + (size_t)bp * N * a.ncol;
  const unsigned mc = div_magic((unsigned)ncl);
  for (int i = threadIdx.x; i < ncl * N; i += blockDim.x) {
    const int zs = fdiv(i, mc), cl = i - zs * ncl;
    out[(size_t)zs * a.ncol + c0 + cl] = lines[cl][zs];
  }
}

// ---- plane: y inverse, x inverse, x V, x forward, y forward ----------------
// Row offsets in the sphere tile of the natural-x inputs b + NB a of x step A
// (lane b): row h - hmin for hmin <= h <= hmax, else row hmax - hmin + 1, which
// is kept zero, so every lane loads unconditionally; bit a of *inside is set for
// the slots inside the sphere, the ones step A' writes back.
template <int NA, int NB>
__device__ inline void x_offsets(int b, int hmin, int hmax, int sa, int (&off)[NA],
                                 unsigned* inside) {
  constexpr int N = NA * NB;
  unsigned m = 0;
#pragma unroll
  for (int a = 0; a < NA; ++a) {
    const int n = b + NB * a;
    const bool lo = n >= hmin && n <= hmax, hi = n - N >= hmin && n - N <= hmax;
    off[a] = (lo ? n - hmin : (hi ? n - N - hmin : hmax - hmin + 1)) * sa;
    m |= (lo || hi) ? 1u << a : 0u;
  }
  *inside = m;
}

// twiddles of an x-pass lane: the lane's index j is the same for every row it
// transforms (b of step A, ka of step B'), so W^(j m), m = 1 .. max(NA, NB) - 1,
// are read from the table once and kept in registers
template <int NA, int NB>
__host__ __device__ constexpr int x_ntw() {
  return (NA > NB ? NA : NB) - 1;
}
template <typename T, int NA, int NB>
__device__ inline void x_twiddles(const cplx<T>* tw, int j, cplx<T> (&w)[x_ntw<NA, NB>()]) {
  constexpr int N = NA * NB;
  int k = 0;
#pragma unroll
  for (int m = 0; m < x_ntw<NA, NB>(); ++m) {
    k += j;
    if (k >= N) k -= N;  // only lanes idle in both steps get here
    w[m] = tw[k];
  }
}

// x step A for row slot ys, inputs gathered from the sphere tile; xw: the
// lane's twiddles W^(b ka)
template <typename T, int NA, int NB>
__device__ inline void x_stepA(const cplx<T>* A, const int (&off)[NA], cplx<T>* R, int ys, int b,
                               const cplx<T> (&xw)[x_ntw<NA, NB>()]) {
  cplx<T> v[NA];
#pragma unroll
  for (int a = 0; a < NA; ++a) v[a] = A[off[a] + ys];
  Dft<T, NA>::run(v, +1);
#pragma unroll
  for (int ka = 1; ka < NA; ++ka) v[ka] = cmul(v[ka], xw[ka - 1]);
#pragma unroll
  for (int ka = 0; ka < NA; ++ka) R[b + NB * ka] = v[ka];
}

// x step A': back to natural x, the slots inside the sphere into the tile
template <typename T, int NA, int NB>
__device__ inline void x_stepAp(cplx<T>* A, const int (&off)[NA], unsigned inside,
                                const cplx<T>* R, int ys, int b) {
  cplx<T> v[NA];
#pragma unroll
  for (int ka = 0; ka < NA; ++ka) v[ka] = R[b + NB * ka];
  Dft<T, NA>::run(v, -1);
#pragma unroll
  for (int a = 0; a < NA; ++a)
    if (inside & (1u << a)) A[off[a] + ys] = v[a];
}

// LDS accesses of one wavefront are performed in issue order, so lanes of a
// wave can exchange data through LDS without a workgroup barrier; the fences
// only keep the compiler from moving LDS accesses across this point.
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kPlaneMaxThreads = 512;
constexpr int kPlaneLoads = 4;  // sphere columns held in registers per thread

// x rows a wavefront transforms at once: step A runs NB lanes per row, step B
// NA lanes per row
__host__ __device__ constexpr int plane_rows_per_wave(int NA, int NB) {
  return 64 / (NA > NB ? NA : NB);
}

// ---- y passes of a plane: nH lines of the sphere tile, line index fastest
// across lanes.  A Y_CUBE plane has the x edge's radices as constants.
template <typename T, int YK, int NA, int NB>
__device__ inline void y_inverse(cplx<T>* A, const FastArgs& a, const cplx<T>* tw) {
  const int nH = a.nH, sa = a.sa;
  const unsigned mH = div_magic((unsigned)nH);
  auto stepA = [&](auto R, int yb) {
    for (int it = threadIdx.x; it < nH * yb; it += blockDim.x) {
      const int q = fdiv(it, mH);
      np_stepA<T, decltype(R)::value>(A + (it - q * nH) * sa, q, yb, tw, +1);
    }
  };
  auto stepB = [&](auto R, int ya) {
    for (int it = threadIdx.x; it < nH * ya; it += blockDim.x) {
      const int q = fdiv(it, mH);
      np_stepB<T, decltype(R)::value>(A + (it - q * nH) * sa, q, +1);
    }
  };
  if constexpr (YK == Y_CUBE) stepA(std::integral_constant<int, NA>(), NB);
  else with_radix<y_max_radix(YK)>(a.ya, [&](auto R) { stepA(R, a.yb); });
  __syncthreads();
  if constexpr (YK == Y_CUBE) stepB(std::integral_constant<int, NB>(), NA);
  else with_radix<y_max_radix(YK)>(a.yb, [&](auto R) { stepB(R, a.ya); });
  __syncthreads();
}
template <typename T, int YK, int NA, int NB>
__device__ inline void y_forward(cplx<T>* A, const FastArgs& a, const cplx<T>* tw) {
  const int nH = a.nH, sa = a.sa;
  const unsigned mH = div_magic((unsigned)nH);
  auto stepB = [&](auto R, int ya) {
    for (int it = threadIdx.x; it < nH * ya; it += blockDim.x) {
      const int q = fdiv(it, mH);
      pn_stepB<T, decltype(R)::value>(A + (it - q * nH) * sa, q, tw, -1);
    }
  };
  auto stepA = [&](auto R, int yb) {
    for (int it = threadIdx.x; it < nH * yb; it += blockDim.x) {
      const int q = fdiv(it, mH);
      pn_stepA<T, decltype(R)::value>(A + (it - q * nH) * sa, q, yb, -1);
    }
  };
  if constexpr (YK == Y_CUBE) stepB(std::integral_constant<int, NB>(), NA);
  else with_radix<y_max_radix(YK)>(a.yb, [&](auto R) { stepB(R, a.ya); });
  __syncthreads();
  if constexpr (YK == Y_CUBE) stepA(std::integral_constant<int, NA>(), NB);
  else with_radix<y_max_radix(YK)>(a.ya, [&](auto R) { stepA(R, a.yb); });
  __syncthreads();
}

// One z plane of one band pair: y inverse over the nH sphere rows, then for
// every y slot the x line (inverse, V(r) multiply, forward) and y forward.
// The x lines are owned by wavefronts (a wave takes plane_rows_per_wave rows
// at a time through its own LDS strip), so the x pass needs no workgroup
// barrier; V(r) of a wave's next rows is loaded while the current rows are
// transformed.  LDS bank conflicts are kept down by the row strides a.sa (sphere
// tile) and a.sr (x strips), chosen on the host, and by lane maps that put the
// line (y pass) or row (x pass) index fastest across lanes.
// in, out: the columns of the plane (they may be the same ones).
template <typename T, int NA, int NB, int YK>
__device__ inline void plane_body(const FastArgs& a, const T* __restrict__ Vp, int zs,
                                  const cplx<T>* in, cplx<T>* out) {
  constexpr int N = NA * NB;  // the x edge
  constexpr int RW = plane_rows_per_wave(NA, NB);
  const int n2 = YK == Y_CUBE ? N : a.n2;
  const int NG = (n2 + RW - 1) / RW;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
  const int sa = a.sa, sr = a.sr, nH = a.nH;
  cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
  cplx<T>* twy = YK == Y_CUBE ? tw : tw + N;
  cplx<T>* A = twy + n2;                             // [nH + 1][sa], y in slot order
  cplx<T>* Rw = A + (nH + 1) * sa + wave * RW * sr;  // this wave's [RW][sr] strip

  // lane roles of the x pass (row fastest)
  const int rx = lane % RW, jx = lane / RW;
  const bool actA = jx < NB, actB = jx < NA;
  int xoff[NA];
  unsigned xin;
  x_offsets<NA, NB>(min(jx, NB - 1), a.hmin, a.hmax, sa, xoff, &xin);
  // V(r) row pieces of step B; rows past the grid and idle lanes load a valid
  // row that is not used
  const T* Vz = Vp + (size_t)zs * n2 * N + NB * min(jx, NA - 1);
  T vv[NB];  // V(r) of the wave's current rows; the next rows' are loaded once it is used
  {
    const T* row = Vz + (size_t)min(wave * RW + rx, n2 - 1) * N;
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) vv[kb] = row[kb];
  }

  // sphere columns of this plane: loads issued before the LDS fill (real and
  // imaginary parts apart: an array of FP64 pairs went through scratch memory)
  T cr[kPlaneLoads], cim[kPlaneLoads];
  int ci[kPlaneLoads];
#pragma unroll
  for (int j = 0; j < kPlaneLoads; ++j) {
    const int cl = threadIdx.x + j * blockDim.x;
    const int cc = cl < a.ncol ? cl : 0;
    cr[j] = in[cc].x;
    cim[j] = in[cc].y;
    ci[j] = cl < a.ncol ? a.col_hi[cc] * sa + a.col_kmod[cc] : -1;
  }
  load_tw<T>(tw, a.tw, N);
  if constexpr (YK != Y_CUBE) load_tw<T>(twy, a.tw + 2 * N, n2);
  for (int i = threadIdx.x; i < (nH + 1) * sa; i += blockDim.x) A[i] = mk<T>(0, 0);
  __syncthreads();
  cplx<T> xw[x_ntw<NA, NB>()];
  x_twiddles<T, NA, NB>(tw, jx, xw);
#pragma unroll
  for (int j = 0; j < kPlaneLoads; ++j)
    if (ci[j] >= 0) A[ci[j]] = mk<T>(cr[j], cim[j]);
  for (int cl = threadIdx.x + kPlaneLoads * blockDim.x; cl < a.ncol; cl += blockDim.x)
    A[a.col_hi[cl] * sa + a.col_kmod[cl]] = in[cl];
  __syncthreads();

  y_inverse<T, YK, NA, NB>(A, a, twy);

  for (int g = wave; g < NG; g += nwave) {
    const int y0 = g * RW;
    const bool row_ok = y0 + rx < n2;
    cplx<T>* Rr = Rw + rx * sr;
    if (actA && row_ok) x_stepA<T, NA, NB>(A, xoff, Rr, y0 + rx, jx, xw);
    wave_lds_sync();
    if (actB && row_ok) {
      cplx<T>* L = Rr + NB * jx;
      cplx<T> v[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) v[b] = L[b];
      Dft<T, NB>::run(v, +1);
#pragma unroll
      for (int kb = 0; kb < NB; ++kb) {
        v[kb].x *= vv[kb];
        v[kb].y *= vv[kb];
      }
      Dft<T, NB>::run(v, -1);
#pragma unroll
      for (int b = 1; b < NB; ++b) v[b] = cmul(v[b], mk<T>(xw[b - 1].x, -xw[b - 1].y));  // W^-(b jx)
#pragma unroll
      for (int b = 0; b < NB; ++b) L[b] = v[b];
    }
    if (g + nwave < NG) {
      const T* row = Vz + (size_t)min((g + nwave) * RW + rx, n2 - 1) * N;
#pragma unroll
      for (int kb = 0; kb < NB; ++kb) vv[kb] = row[kb];
    }
    wave_lds_sync();
    if (actA && row_ok) x_stepAp<T, NA, NB>(A, xoff, xin, Rr, y0 + rx, jx);
    wave_lds_sync();
  }
  __syncthreads();
  y_forward<T, YK, NA, NB>(A, a, twy);
  for (int cl = threadIdx.x; cl < a.ncol; cl += blockDim.x)
    out[cl] = A[a.col_hi[cl] * sa + a.col_kmod[cl]];
}

template <typename T, int NA, int NB, int YK>
__global__ void __launch_bounds__(kPlaneMaxThreads) k_plane_f(FastArgs a, const T* __restrict__ Vp,
                                                            const cplx<T>* __restrict__ t1,
                                                            cplx<T>* __restrict__ t2) {
  const size_t row =
      ((size_t)blockIdx.y * (YK == Y_CUBE ? NA * NB : a.n3) + blockIdx.x) * a.ncol;
  plane_body<T, NA, NB, YK>(a, Vp, blockIdx.x, t1 + row, t2 + row);
}

// ---- z forward: T2 -> split bands, x1/N, + |G|^2 psi --------------------
// kb32 (optional): an FP32 term added to the result (the KB part of H psi)
template <typename T, int NA, int NB>
__global__ void __launch_bounds__(kFastThreads) k_zfwd_f(FastArgs a, const double* __restrict__ psi,
                                                         const cplx<T>* __restrict__ t2,
                                                         double* __restrict__ out, int accumulate,
                                                         double invN,
                                                         const float* __restrict__ kb32) {
  constexpr int N = NA * NB;
  constexpr int PB = zpairs(N, (int)sizeof(cplx<T>));
  __shared__ cplx<T> tw[N];
  __shared__ cplx<T> lines[2 * PB][N];
  const int q0 = blockIdx.x * PB, q1 = min(q0 + PB, a.npair);
  const int bp = blockIdx.y;
  const int ba = 2 * (a.bp0 + bp), bb = ba + 1;
  const int c0 = q0 == 0 ? 0 : 2 * q0 - 1, c1 = 2 * q1 - 1, ncl = c1 - c0;
  load_tw<T>(tw, a.tw + 2 * (a.n1 + a.n2), N);
  const cplx<T>* in = t2 + (size_t)bp * N * a.ncol;
  const unsigned mc = div_magic((unsigned)ncl);
  for (int i = threadIdx.x; i < ncl * N; i += blockDim.x) {
    const int zs = fdiv(i, mc), cl = i - zs * ncl;
    lines[cl][zs] = in[(size_t)zs * a.ncol + c0 + cl];
  }
  __syncthreads();
  for (int it = threadIdx.x; it < ncl * NA; it += blockDim.x)
    pn_stepB<T, NB>(lines[it / NA], it % NA, tw, -1);
  __syncthreads();
  for (int it = threadIdx.x; it < ncl * NB; it += blockDim.x)
    pn_stepA<T, NA>(lines[it / NB], it % NB, NB, -1);
  __syncthreads();
  const double* pa = psi + (size_t)ba * a.nplwex;
  const double* pb = psi + (size_t)bb * a.nplwex;
  double* oa = out + (size_t)ba * a.nplwex;
  double* ob = out + (size_t)bb * a.nplwex;
  const bool hasb = bb < a.nb;
  const int p0 = a.pair_p0[q0], p1 = a.pair_p0[q1];
  for (int p = p0 + threadIdx.x; p < p1; p += blockDim.x) {
    int col = a.pt_col[p] - c0, z = a.pt_z[p];
    cplx<T> zp = lines[col][z];
    cplx<T> zm = lines[mirror_col_f(col + c0) - c0][z == 0 ? 0 : N - z];
    double Ar = 0.5 * ((double)zp.x + (double)zm.x) * invN;
    double Ai = 0.5 * ((double)zp.y - (double)zm.y) * invN;
    double Br = 0.5 * ((double)zp.y + (double)zm.y) * invN;
    double Bi = -0.5 * ((double)zp.x - (double)zm.x) * invN;
    double kin = a.kin[p];
    double r0 = kin * pa[2 * p] + Ar, r1 = kin * pa[2 * p + 1] + Ai;
    if (accumulate) { r0 += oa[2 * p]; r1 += oa[2 * p + 1]; }
    if (kb32) {
      r0 += (double)kb32[(size_t)ba * a.nplwex + 2 * p];
      r1 += (double)kb32[(size_t)ba * a.nplwex + 2 * p + 1];
    }
    oa[2 * p] = r0;
    oa[2 * p + 1] = r1;
    if (hasb) {
      double s0 = kin * pb[2 * p] + Br, s1 = kin * pb[2 * p + 1] + Bi;
      if (accumulate) { s0 += ob[2 * p]; s1 += ob[2 * p + 1]; }
      if (kb32) {
        s0 += (double)kb32[(size_t)bb * a.nplwex + 2 * p];
        s1 += (double)kb32[(size_t)bb * a.nplwex + 2 * p + 1];
      }
      ob[2 * p] = s0;
      ob[2 * p + 1] = s1;
    }
  }
}

// ---- density: y inverse, x inverse, accumulate |psi|^2 in slot order --------
// Same plane layout and lane maps as k_plane_f.  A block (z plane, group of
// band pairs) keeps its share of the plane's density in registers over all its
// band pairs (RG row groups per wavefront at most) and writes it once.
constexpr int kRhoGroups = 6;  // largest RG instantiated (2, 4 and 6 are)

// more than four row groups run with at most four wavefronts per block, which
// leaves each lane the register file's full width for the accumulators
constexpr int rho_max_threads(int RG) { return RG > 4 ? 256 : kPlaneMaxThreads; }

template <typename T, int NA, int NB, int YK, int RG>
__global__ void __launch_bounds__(rho_max_threads(RG)) k_plane_rho_f(FastArgs a,
                                                                const cplx<T>* __restrict__ t1,
                                                                int nbp_batch, int bp_per_group,
                                                                const double* __restrict__ w,
                                                                double* __restrict__ rho_part) {
  constexpr int N = NA * NB;  // the x edge
  constexpr int RW = plane_rows_per_wave(NA, NB);
  const int n2 = YK == Y_CUBE ? N : a.n2, n3 = YK == Y_CUBE ? N : a.n3;
  const int NG = (n2 + RW - 1) / RW;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
  const int sa = a.sa, sr = a.sr, nH = a.nH;
  cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
  cplx<T>* twy = YK == Y_CUBE ? tw : tw + N;
  cplx<T>* A = twy + n2;                             // [nH + 1][sa], last row zero
  cplx<T>* Rw = A + (nH + 1) * sa + wave * RW * sr;
  const int zs = blockIdx.x, grp = blockIdx.y;
  const int rx = lane % RW, jx = lane / RW;
  const bool actA = jx < NB, actB = jx < NA;
  int xoff[NA];
  unsigned xin;
  x_offsets<NA, NB>(min(jx, NB - 1), a.hmin, a.hmax, sa, xoff, &xin);
  load_tw<T>(tw, a.tw, N);
  if constexpr (YK != Y_CUBE) load_tw<T>(twy, a.tw + 2 * N, n2);
  __syncthreads();
  cplx<T> xw[x_ntw<NA, NB>()];
  x_twiddles<T, NA, NB>(tw, jx, xw);
  double acc[RG][NB];
#pragma unroll
  for (int gi = 0; gi < RG; ++gi)
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) acc[gi][kb] = 0.0;
  const int bpe = min(nbp_batch, (grp + 1) * bp_per_group);
  for (int bp = grp * bp_per_group; bp < bpe; ++bp) {
    const int ba = 2 * (a.bp0 + bp), bb = ba + 1;
    const double wa = w[ba], wb = bb < a.nb ? w[bb] : 0.0;
    __syncthreads();
    for (int i = threadIdx.x; i < (nH + 1) * sa; i += blockDim.x) A[i] = mk<T>(0, 0);
    __syncthreads();
    const cplx<T>* in = t1 + ((size_t)bp * n3 + zs) * a.ncol;
    for (int cl = threadIdx.x; cl < a.ncol; cl += blockDim.x)
      A[a.col_hi[cl] * sa + a.col_kmod[cl]] = in[cl];
    __syncthreads();
    y_inverse<T, YK, NA, NB>(A, a, twy);
#pragma unroll
    for (int gi = 0; gi < RG; ++gi) {
      const int g = wave + gi * nwave;
      if (g < NG) {
        const int y0 = g * RW;
        const bool row_ok = y0 + rx < n2;
        cplx<T>* Rr = Rw + rx * sr;
        if (actA && row_ok) x_stepA<T, NA, NB>(A, xoff, Rr, y0 + rx, jx, xw);
        wave_lds_sync();
        if (actB && row_ok) {
          const cplx<T>* L = Rr + NB * jx;
          cplx<T> v[NB];
#pragma unroll
          for (int b = 0; b < NB; ++b) v[b] = L[b];
          Dft<T, NB>::run(v, +1);
#pragma unroll
          for (int kb = 0; kb < NB; ++kb) {
            const double re = (double)v[kb].x, im = (double)v[kb].y;
            acc[gi][kb] += re * re * wa + im * im * wb;
          }
        }
        wave_lds_sync();
      }
    }
  }
  double* rp = rho_part + ((size_t)grp * n3 + zs) * n2 * N;
#pragma unroll
  for (int gi = 0; gi < RG; ++gi) {
    const int g = wave + gi * nwave, y = g * RW + rx;
    if (g < NG && y < n2 && actB) {
      double* dst = rp + (size_t)y * N + NB * jx;
#pragma unroll
      for (int kb = 0; kb < NB; ++kb) dst[kb] = acc[gi][kb];
    }
  }
}

// ---- Bloch bands (kpoint.hip): one complex band per transform, a sphere per
// k-point, the columns of a (k, band) block transformed in place ----------------
struct KFastArgs {
  FastArgs f;          // grid, y radices, strides, twiddles
  int nb, npw_max, ncol_max, kb0;
  int rpk, r0;         // band rows of a k-point in the src/dst arrays, first row used
  const int *npw, *ncol, *hmin, *hmax;  // [k]
  const int* col_p0;   // [k][ncol_max + 1]: first point of column c
  const int *col_h, *col_y;             // [k][ncol_max]: h, y index of column c
  const int *pt_z, *pt_col;             // [k][npw_max]
  const double* kin;   // [k][npw_max]: |k+G|^2
};
constexpr int kKFastCols = 16;  // columns per block of the z kernels

template <int NA, int NB>
__global__ void __launch_bounds__(kFastThreads)
    k_kzinv_f(KFastArgs a, const double* __restrict__ psi, cplx<double>* __restrict__ T) {
  constexpr int N = NA * NB;
  __shared__ cplx<double> tw[N], lines[kKFastCols][N];
  const int kb = a.kb0 + (int)blockIdx.y, k = kb / a.nb;
  const int nc = a.ncol[k], c0 = (int)blockIdx.x * kKFastCols;
  if (c0 >= nc) return;
  const int cn = min(kKFastCols, nc - c0);
  load_tw<double>(tw, a.f.tw + 2 * (a.f.n1 + a.f.n2), N);
  for (int i = threadIdx.x; i < cn * N; i += blockDim.x) lines[i / N][i % N] = mk<double>(0.0, 0.0);
  __syncthreads();
  const int* cp = a.col_p0 + (size_t)k * (a.ncol_max + 1);
  const int *pz = a.pt_z + (size_t)k * a.npw_max, *pc = a.pt_col + (size_t)k * a.npw_max;
  const double2* src = reinterpret_cast<const double2*>(
      psi + ((size_t)k * a.rpk + a.r0 + (kb - k * a.nb)) * 2 * a.npw_max);
  const int p1 = cp[c0 + cn];
  for (int p = cp[c0] + (int)threadIdx.x; p < p1; p += blockDim.x) {
    const double2 v = src[p];
    lines[pc[p] - c0][pz[p]] = mk<double>(v.x, v.y);
  }
  __syncthreads();
  for (int it = threadIdx.x; it < cn * NB; it += blockDim.x)
    np_stepA<double, NA>(lines[it / NB], it % NB, NB, tw, +1);
  __syncthreads();
  for (int it = threadIdx.x; it < cn * NA; it += blockDim.x)
    np_stepB<double, NB>(lines[it / NA], it % NA, +1);
  __syncthreads();
  cplx<double>* out = T + (size_t)blockIdx.y * N * a.ncol_max + c0;
  for (int i = threadIdx.x; i < kKFastCols * N; i += blockDim.x) {
    const int zs = i / kKFastCols, cl = i % kKFastCols;
    if (cl < cn) out[(size_t)zs * a.ncol_max + cl] = lines[cl][zs];
  }
}

template <int NA, int NB, int YK>
__global__ void __launch_bounds__(kPlaneMaxThreads)
    k_kplane_f(KFastArgs a, const double* __restrict__ Vp, cplx<double>* T) {
  const int k = (a.kb0 + (int)blockIdx.y) / a.nb;
  FastArgs f = a.f;
  f.ncol = a.ncol[k];
  f.hmin = a.hmin[k];
  f.hmax = a.hmax[k];
  f.nH = f.hmax - f.hmin + 1;
  f.col_hi = a.col_h + (size_t)k * a.ncol_max;
  f.col_kmod = a.col_y + (size_t)k * a.ncol_max;
  cplx<double>* row =
      T + ((size_t)blockIdx.y * (YK == Y_CUBE ? NA * NB : f.n3) + blockIdx.x) * a.ncol_max;
  plane_body<double, NA, NB, YK>(f, Vp, blockIdx.x, row, row);
}

template <int NA, int NB>
__global__ void __launch_bounds__(kFastThreads)
    k_kzfwd_f(KFastArgs a, const double* __restrict__ psi, const cplx<double>* __restrict__ T,
              double* __restrict__ out, double scale) {
  constexpr int N = NA * NB;
  __shared__ cplx<double> tw[N], lines[kKFastCols][N];
  const int kb = a.kb0 + (int)blockIdx.y, k = kb / a.nb;
  const int nc = a.ncol[k], np = a.npw[k];
  const size_t row = ((size_t)k * a.rpk + a.r0 + (kb - k * a.nb)) * 2 * a.npw_max;
  if (blockIdx.x == 0)  // the padding beyond npw_k stays zero
    for (int i = 2 * np + (int)threadIdx.x; i < 2 * a.npw_max; i += blockDim.x) out[row + i] = 0.0;
  const int c0 = (int)blockIdx.x * kKFastCols;
  if (c0 >= nc) return;
  const int cn = min(kKFastCols, nc - c0);
  load_tw<double>(tw, a.f.tw + 2 * (a.f.n1 + a.f.n2), N);
  const cplx<double>* in = T + (size_t)blockIdx.y * N * a.ncol_max + c0;
  for (int i = threadIdx.x; i < kKFastCols * N; i += blockDim.x) {
    const int zs = i / kKFastCols, cl = i % kKFastCols;
    if (cl < cn) lines[cl][zs] = in[(size_t)zs * a.ncol_max + cl];
  }
  __syncthreads();
  for (int it = threadIdx.x; it < cn * NA; it += blockDim.x)
    pn_stepB<double, NB>(lines[it / NA], it % NA, tw, -1);
  __syncthreads();
  for (int it = threadIdx.x; it < cn * NB; it += blockDim.x)
    pn_stepA<double, NA>(lines[it / NB], it % NB, NB, -1);
  __syncthreads();
  const int* cp = a.col_p0 + (size_t)k * (a.ncol_max + 1);
  const int *pz = a.pt_z + (size_t)k * a.npw_max, *pc = a.pt_col + (size_t)k * a.npw_max;
  const double* kin = a.kin + (size_t)k * a.npw_max;
  const double2* src = reinterpret_cast<const double2*>(psi + row);
  double2* dst = reinterpret_cast<double2*>(out + row);
  const int p1 = cp[c0 + cn];
  for (int p = cp[c0] + (int)threadIdx.x; p < p1; p += blockDim.x) {
    const cplx<double> v = lines[pc[p] - c0][pz[p]];
    const double2 c = src[p];
    dst[p] = make_double2(v.x * scale + kin[p] * c.x, v.y * scale + kin[p] * c.y);
  }
}

// ---- launch table: the kernels of one edge and precision ---------------------
constexpr int kRhoKinds = 3;  // row groups per wavefront of the density kernel: 2, 4, 6
template <typename T>
struct EdgeKernels {
  using ZInv = void (*)(FastArgs, const double*, cplx<T>*, float*, unsigned short*, int, long);
  using ZFwd = void (*)(FastArgs, const double*, const cplx<T>*, double*, int, double,
                        const float*);
  using Plane = void (*)(FastArgs, const T*, const cplx<T>*, cplx<T>*);
  using Rho = void (*)(FastArgs, const cplx<T>*, int, int, const double*, double*);
  ZInv zinv = nullptr;            // z edge
  ZFwd zfwd = nullptr;
  Plane plane[3] = {};            // x edge; by YKind
  Rho rho[3][kRhoKinds] = {};     // 6 row groups for cubes only
  // Bloch bands (FP64 only)
  void (*kzinv)(KFastArgs, const double*, cplx<double>*) = nullptr;
  void (*kzfwd)(KFastArgs, const double*, const cplx<double>*, double*, double) = nullptr;
  void (*kplane[3])(KFastArgs, const double*, cplx<double>*) = {};
};
template <typename T>
using EdgeLookup = bool (*)(int n, EdgeKernels<T>* k);
// defined by the instantiation units (pencil_inst.hip, one per group of edges)
#define QX_DECL_GROUP(g)                                  \
  bool edge_kernels_##g(int n, EdgeKernels<float>* k);    \
  bool edge_kernels_##g(int n, EdgeKernels<double>* k);
QX_DECL_GROUP(0) QX_DECL_GROUP(1) QX_DECL_GROUP(2) QX_DECL_GROUP(3)
QX_DECL_GROUP(4) QX_DECL_GROUP(5) QX_DECL_GROUP(6) QX_DECL_GROUP(7)
#undef QX_DECL_GROUP

// Bloch-band local part: launches zinv, plane, zfwd for nkb blocks of T; -3 when
// the grid or its LDS is not covered.  nH: the widest sphere's h extent.
int kp_local_fast(Ctx* c, KFastArgs a, int nH, const double* src, double* dst, double2* T,
                  int nkb);

}  // namespace qx
