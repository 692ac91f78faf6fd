// gemm_small.hip -- the contractions of gemm.hip whose output has fewer than
// 256 rows or columns: small cells, CG blocks of a few bands, the k-points of
// a mesh (batched).  FP64, or the mixed form's FP32 MFMA on FP64 operands.
// FP64 products of any size come here too when a leading dimension is odd, which
// the 16-byte rows of mfma_gemm.hip exclude (psi L^-T and the rotation of an odd
// number of bands; Gram-Schmidt of 541 bands of 43820 1.39 ms, of 540 1.24).
//
// What bounds these is latency and occupancy, not the matrix cores: 32 x 20
// outputs of 1648 plane waves are four MFMA tiles with one long sum each.  So
// nothing is staged through LDS; a wavefront loads its MFMA fragments straight
// from memory (the K index is contiguous for both operands of TN: 16 k of a
// row are one 128-byte line, four lanes of two 16-byte loads), the next
// fragments in flight during the MFMAs of the current ones, and the sum is
// split over wavefronts (added through LDS in wavefront order) and, where the
// tiles alone leave CUs idle, over workgroups (partials in a workspace, added
// in slice order by k_gs_fix): results do not depend on timing.
//
// K is split over the four wavefronts of a workgroup (their sums added through
// LDS, each wavefront adding its share of the tile) and over workgroups; more
// wavefronts per workgroup make that sum longer than what they save.  One
// launch, or two with K slices, carries the packed-sum correction, alpha, beta
// and a row scale, where a scale, an FP64-atomic product with a workgroup per
// 1024 k and a correction ran before: (32 x 20) x 1648 FP64 80 -> 8 us, (256 x
// 160) x 13134 FP64 158 -> 31 us, (384 x 240) x 19588 FP32 127 -> 77 us.
#include <algorithm>
#include "context.h"

namespace qx {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

inline unsigned cdivu(long a, long b) { return (unsigned)((a + b - 1) / b); }

template <typename T>
struct Mma;
template <>
struct Mma<double> {
  typedef d4 acc_t;
  __device__ static acc_t run(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // D(i, j): lane j + 16 (i % 4), register i / 4
  __device__ static int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <>
struct Mma<float> {
  typedef f4 acc_t;
  __device__ static acc_t run(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // D(i, j): lane j + 16 (i / 4), register i % 4
  __device__ static int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

struct GsArgs {
  int M, N, K, lda, ldb, ldc, corr;
  int ks, kper;        // K slices over workgroups, k per slice (a multiple of 16 KH)
  int tiles_m;
  long sA, sB, sC;     // batch strides
  double alpha, beta;
  const double* rscale;  // per row m of C, or null
};

// what the packed sums of TN count twice: 1 -> 0.5 A0 B0, 2 -> + A1 B1
__device__ inline double gs_corr(const GsArgs& g, const double* A, const double* B, int m, int n) {
  if (!g.corr) return 0.0;
  double c = 0.5 * A[(size_t)m * g.lda] * B[(size_t)n * g.ldb];
  if (g.corr == 2) c += A[(size_t)m * g.lda + 1] * B[(size_t)n * g.ldb + 1];
  return c;
}
__device__ inline double gs_value(const GsArgs& g, double sum, const double* A, const double* B,
                                  const double* cp, int m, int n) {
  double x = g.alpha * (sum - gs_corr(g, A, B, m, n));
  if (g.rscale) x *= g.rscale[m];
  return g.beta == 0.0 ? x : x + g.beta * *cp;
}

// four consecutive k of a row; VEC: 16-byte aligned rows
template <bool VEC>
__device__ inline void load4(const double* p, double (&r)[4]) {
  if (VEC) {
    const double2 a = *reinterpret_cast<const double2*>(p);
    const double2 b = *reinterpret_cast<const double2*>(p + 2);
    r[0] = a.x; r[1] = a.y; r[2] = b.x; r[3] = b.y;
  } else {
#pragma unroll
    for (int u = 0; u < 4; ++u) r[u] = p[u];
  }
}
template <bool VEC>
__device__ inline void load2(const double* p, double (&r)[2]) {
  if (VEC) {
    const double2 a = *reinterpret_cast<const double2*>(p);
    r[0] = a.x; r[1] = a.y;
  } else {
    r[0] = p[0]; r[1] = p[1];
  }
}

// C(m, n) = alpha sum_k A[m][k] B[n][k] ... : blockIdx.x K slice (fastest, so
// that a slice count divisible by 8 keeps a slice's workgroups on one XCD and
// its operand columns in one L2), blockIdx.y tile, blockIdx.z batch.
// BI x BJ blocks of 16 along m and n; the KH wavefronts of a workgroup share the
// slice 16 k at a time.
constexpr int KH = 4;
template <typename T, bool VEC, int BI, int BJ, int DP>
__global__ void __launch_bounds__(64 * KH, 2)
    k_gs_tn(GsArgs g, const double* __restrict__ A0, const double* __restrict__ B0,
            double* __restrict__ C0, double* __restrict__ Wp) {
  constexpr int TM = 16 * BI, TN = 16 * BJ;
  typedef typename Mma<T>::acc_t acc_t;
  __shared__ T red[KH][BI * BJ * 4][64];
  const double* A = A0 + (size_t)blockIdx.z * g.sA;
  const double* B = B0 + (size_t)blockIdx.z * g.sB;
  const int lane = threadIdx.x & 63, kh = threadIdx.x >> 6;
  const int tile = (int)blockIdx.y;
  const int m0 = (tile % g.tiles_m) * TM, n0 = (tile / g.tiles_m) * TN;
  const int r = lane & 15, q = lane >> 4;
  const int kb = (int)blockIdx.x * g.kper, ke = min(g.K, kb + g.kper);
  const double *pa[BI], *pb[BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i) pa[i] = A + (size_t)min(m0 + 16 * i + r, g.M - 1) * g.lda;
#pragma unroll
  for (int j = 0; j < BJ; ++j) pb[j] = B + (size_t)min(n0 + 16 * j + r, g.N - 1) * g.ldb;
  acc_t acc[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = (T)0;
  double a[DP][BI][4], b[DP][BJ][4];  // DP steps of 16 k in flight
  auto fetch = [&](int s, int k0) {
    const int k = k0 + 4 * q;
    if (k0 + 16 <= ke) {
#pragma unroll
      for (int i = 0; i < BI; ++i) load4<VEC>(pa[i] + k, a[s][i]);
#pragma unroll
      for (int j = 0; j < BJ; ++j) load4<VEC>(pb[j] + k, b[s][j]);
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool in = k + u < ke;
#pragma unroll
        for (int i = 0; i < BI; ++i) a[s][i][u] = in ? pa[i][k + u] : 0.0;
#pragma unroll
        for (int j = 0; j < BJ; ++j) b[s][j][u] = in ? pb[j][k + u] : 0.0;
      }
    }
  };
  constexpr int KS = 16 * KH;  // from one step of a wavefront to its next
  const int k00 = kb + 16 * kh;
#pragma unroll
  for (int s = 0; s < DP; ++s)
    if (k00 + s * KS < ke) fetch(s, k00 + s * KS);
  for (int k1 = k00; k1 < ke; k1 += DP * KS)
#pragma unroll
    for (int s = 0; s < DP; ++s) {
      const int k0 = k1 + s * KS;
      if (k0 >= ke) break;
      T fa[BI][4], fb[BJ][4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int i = 0; i < BI; ++i) fa[i][u] = (T)a[s][i][u];
#pragma unroll
        for (int j = 0; j < BJ; ++j) fb[j][u] = (T)b[s][j][u];
      }
      if (k0 + DP * KS < ke) fetch(s, k0 + DP * KS);
      // step u takes k = 4 q + u of every q; n on D's rows, m across its lanes
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < BI; ++i)
#pragma unroll
          for (int j = 0; j < BJ; ++j) acc[i][j] = Mma<T>::run(fb[j][u], fa[i][u], acc[i][j]);
    }
  const size_t slot = ((size_t)blockIdx.z * gridDim.y + tile) * g.ks + blockIdx.x;
  double* P = Wp + slot * (TM * TN);
  double* C = C0 + (size_t)blockIdx.z * g.sC;
  // every wavefront leaves its sums in LDS and adds up its share of the tile
  constexpr int ROWS = BI * BJ * 4;
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[kh][(i * BJ + j) * 4 + v][lane] = acc[i][j][v];
  __syncthreads();
  for (int row = kh; row < ROWS; row += KH) {
    double s = (double)red[0][row][lane];
#pragma unroll
    for (int h = 1; h < KH; ++h) s += (double)red[h][row][lane];
    const int i = row / (4 * BJ), j = row / 4 % BJ, v = row % 4;
    const int ml = 16 * i + r, nl = 16 * j + Mma<T>::row(lane, v), m = m0 + ml, n = n0 + nl;
    if (g.ks > 1) {
      P[nl * TM + ml] = s;
    } else if (m < g.M && n < g.N) {
      double* cp = C + (size_t)n * g.ldc + m;
      *cp = gs_value(g, s, A, B, cp, m, n);
    }
  }
}

// sums the K slices of C(m, n) in order, then the epilogue of k_gs_tn
__global__ void __launch_bounds__(256)
    k_gs_fix(GsArgs g, int tm, int tn, int tiles, const double* __restrict__ A0,
             const double* __restrict__ B0, double* __restrict__ C0,
             const double* __restrict__ Wp) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long)g.M * g.N) return;
  const int m = (int)(e % g.M), n = (int)(e / g.M);
  const int tile = m / tm + g.tiles_m * (n / tn);
  const double* w = Wp + ((size_t)blockIdx.y * tiles + tile) * g.ks * (tm * tn) +
                    (n % tn) * tm + m % tm;
  const size_t st = (size_t)tm * tn;
  double s = 0.0;
  int k = 0;
  for (; k + 8 <= g.ks; k += 8) {  // eight loads in flight, summed in slice order
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = w[(size_t)(k + u) * st];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; k < g.ks; ++k) s += w[(size_t)k * st];
  double* cp = C0 + (size_t)blockIdx.y * g.sC + (size_t)n * g.ldc + m;
  *cp = gs_value(g, s, A0 + (size_t)blockIdx.y * g.sA, B0 + (size_t)blockIdx.y * g.sB, cp, m, n);
}

// C(m, n) = alpha sum_k A[k][m] B[n][k] + beta C, one wavefront per workgroup
// and 32 G m x 16 BJ n of C.  Eight k a step: lane quarter q loads two m of each
// of the rows k = 2 q, 2 q + 1 (256 contiguous bytes per row and group of 32 m)
// and those two k of its B rows, so step s of the MFMAs takes k = 2 q + s and an
// accumulator holds the even or the odd m; C is read and written in 16-byte
// pairs of m.
template <typename T, bool VEC, int G, int BJ, int DP>
__global__ void __launch_bounds__(64, 2)
    k_gs_nn(GsArgs g, const double* __restrict__ A0, const double* __restrict__ B0,
            double* __restrict__ C0) {
  typedef typename Mma<T>::acc_t acc_t;
  const double* A = A0 + (size_t)blockIdx.z * g.sA;
  const double* B = B0 + (size_t)blockIdx.z * g.sB;
  double* C = C0 + (size_t)blockIdx.z * g.sC;
  const int lane = threadIdx.x & 63;
  const int m0 = (int)blockIdx.x * 32 * G, n0 = (int)blockIdx.y * 16 * BJ;
  const int r = lane & 15, q = lane >> 4;
  int mc[G][2];  // the lane's two m, kept inside the row (VEC: M is even)
#pragma unroll
  for (int i = 0; i < G; ++i)
#pragma unroll
    for (int e = 0; e < 2; ++e) mc[i][e] = min(m0 + 32 * i + 2 * r + e, g.M - (VEC ? 2 - e : 1));
  const double* pb[BJ];
#pragma unroll
  for (int j = 0; j < BJ; ++j) pb[j] = B + (size_t)min(n0 + 16 * j + r, g.N - 1) * g.ldb;
  acc_t acc[BJ][G][2];
#pragma unroll
  for (int j = 0; j < BJ; ++j)
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[j][i][e][v] = (T)0;
  // DP steps of 8 k in flight, as many as the registers hold.  The full steps run
  // without a branch: behind one, the compiler waits for every outstanding load,
  // and the wavefronts are too few (one a SIMD) to hide that.  Prefetches past the
  // last full step read it again.  13134 x 160 x 160 and x 256, FP32: 38 -> 28 us;
  // 5222 x 81 x 128, FP64: 18 -> 11; 19588 x 240 x 384, FP32: 85 -> 74.
  double a[DP][2][G][2], b[DP][BJ][2];
  const int nf = g.K / 8;
  auto row_pair = [&](const double* p, int i, double(&v)[2]) {
    if (VEC) {
      load2<true>(p + mc[i][0], v);
    } else {
      v[0] = p[mc[i][0]];
      v[1] = p[mc[i][1]];
    }
  };
  auto fetch = [&](int d, int t) {
    const int k = 8 * min(t, nf - 1) + 2 * q;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < G; ++i) row_pair(A + (size_t)(k + s) * g.lda, i, a[d][s][i]);
#pragma unroll
    for (int j = 0; j < BJ; ++j) load2<VEC>(pb[j] + k, b[d][j]);
  };
  T fa[2][G][2], fb[BJ][2];
  auto convert = [&](int d) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 0; i < G; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e) fa[s][i][e] = (T)a[d][s][i][e];
#pragma unroll
      for (int j = 0; j < BJ; ++j) fb[j][s] = (T)b[d][j][s];
    }
  };
  auto products = [&]() {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < BJ; ++j)
#pragma unroll
        for (int i = 0; i < G; ++i)
#pragma unroll
          for (int e = 0; e < 2; ++e)
            acc[j][i][e] = Mma<T>::run(fb[j][s], fa[s][i][e], acc[j][i][e]);
  };
  if (nf > 0) {
#pragma unroll
    for (int d = 0; d < DP; ++d) fetch(d, d);
    int t = 0;
    for (; t + DP <= nf; t += DP)
#pragma unroll
      for (int d = 0; d < DP; ++d) {
        convert(d);
        __builtin_amdgcn_sched_barrier(0);
        fetch(d, t + d + DP);
        __builtin_amdgcn_sched_barrier(0);
        products();
      }
#pragma unroll
    for (int d = 0; d < DP - 1; ++d)
      if (t + d < nf) {
        convert(d);
        products();
      }
  }
  if (8 * nf < g.K) {  // the step that K ends in
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int k = 8 * nf + 2 * q + s, kc = min(k, g.K - 1);
#pragma unroll
      for (int i = 0; i < G; ++i) {
        row_pair(A + (size_t)kc * g.lda, i, a[0][s][i]);
        if (k >= g.K) a[0][s][i][0] = a[0][s][i][1] = 0.0;
      }
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        const double v = pb[j][kc];
        b[0][j][s] = k < g.K ? v : 0.0;
      }
    }
    convert(0);
    products();
  }
#pragma unroll
  for (int j = 0; j < BJ; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int n = n0 + 16 * j + Mma<T>::row(lane, v);
      if (n >= g.N) continue;
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const int m = m0 + 32 * i + 2 * r;
        double* cp = C + (size_t)n * g.ldc + m;
        const double x = g.alpha * (double)acc[j][i][0][v], y = g.alpha * (double)acc[j][i][1][v];
        if (VEC) {
          if (m >= g.M) continue;
          double2 c = make_double2(x, y);
          if (g.beta != 0.0) {
            const double2 o = *reinterpret_cast<const double2*>(cp);
            c.x += g.beta * o.x;
            c.y += g.beta * o.y;
          }
          *reinterpret_cast<double2*>(cp) = c;
        } else {
          if (m < g.M) cp[0] = g.beta == 0.0 ? x : x + g.beta * cp[0];
          if (m + 1 < g.M) cp[1] = g.beta == 0.0 ? y : y + g.beta * cp[1];
        }
      }
    }
}

constexpr int kTarget = 512;  // workgroups of a launch with K slices (2 per CU)
constexpr int kMin = 64;      // least k of a wavefront

// the K-slice partials: kept by the context, grown to what its products need
double* workspace(Ctx* c, size_t n) {
  if (n > c->gs_len) {
    buffers_changed(c);
    if (c->d_gs) (void)hipFree(c->d_gs);  // waits for what still reads it
    c->d_gs = nullptr;
    c->gs_len = 0;
    if (hipMalloc(&c->d_gs, sizeof(double) * n) != hipSuccess) {
      (void)hipGetLastError();
      return c->d_gs = nullptr;
    }
    c->gs_len = n;
  }
  return c->d_gs;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <typename T, int BI, int BJ, int DP>
int launch_tn(Ctx* c, GsArgs g, int batch, int target, const double* A, const double* B,
              double* C) {
  constexpr int TM = 16 * BI, TN = 16 * BJ;
  g.tiles_m = (int)cdivu(g.M, TM);
  const int tiles = g.tiles_m * (int)cdivu(g.N, TN);
  // K slices: enough workgroups for the chip, at least kMin k per wavefront
  // (a multiple of 8 of them stays one: trailing slices may be empty)
  int ks = (int)std::min<long>(target / ((long)tiles * batch), g.K / (kMin * KH));
  ks = std::max(1, ks >= 8 ? ks & ~7 : ks);
  // FP32 chains: a wavefront sums in FP32, the wavefronts' and the slices' sums are
  // added in FP64.  The error grows with the chain (2080 x 100 x 13134, random
  // operands: 9.9e-7 of the result with 3284 k a chain, 5.1e-7 with 832; of one
  // sign 4.1e-7 and 1.1e-7), so a chain takes 1024 k at most, more only where the
  // output alone is many of 2048 blocks of 64 x 64 (27 MB of partials at most)
  if constexpr (sizeof(T) == 4) {
    const long blocks = (long)cdivu(g.M, 64) * cdivu(g.N, 64);
    const long chains = std::min<long>(cdivu(g.K, 1024), std::max(1L, 2048 / blocks));
    ks = std::max(ks, (int)cdivu(chains, KH));
  }
  double* W = ks > 1 ? workspace(c, (size_t)tiles * batch * ks * TM * TN) : nullptr;
  if (!W) ks = 1;  // one slice, or out of memory
  g.kper = (int)cdivu(cdivu(g.K, ks), 16 * KH) * 16 * KH;
  g.ks = ks;
  const dim3 grid(g.ks, tiles, batch);
  const bool vec = !(g.lda & 1) && !(g.ldb & 1) && !(g.sA & 1) && !(g.sB & 1) && aligned16(A) &&
                   aligned16(B);
  if (vec)
    hipLaunchKernelGGL((k_gs_tn<T, true, BI, BJ, DP>), grid, dim3(64 * KH), 0, c->stream, g, A, B,
                       C, W);
  else
    hipLaunchKernelGGL((k_gs_tn<T, false, BI, BJ, DP>), grid, dim3(64 * KH), 0, c->stream, g, A, B,
                       C, W);
  if (g.ks > 1)
    hipLaunchKernelGGL(k_gs_fix, dim3(cdivu((long)g.M * g.N, 256), batch), dim3(256), 0, c->stream,
                       g, TM, TN, tiles, A, B, C, W);
  QX_CHECK(hipGetLastError());
  return 0;
}

// (us of the candidates at M x N x K, FP64 unless marked, fix-up included)
template <typename T>
int tn(Ctx* c, const GsArgs& g, int batch, const double* A, const double* B, double* C) {
  // up to 32 tiles of 16 x 16: as many wavefronts as the sum's length feeds
  // (32 x 20 x 1648: 8.4 against 11.5 on 32 x 32 tiles; 128 x 81 x 5222, 48
  // tiles: 11.9 against 11.4; 64 products of 64 x 20 x 1672: 27 against 22)
  const long t16 = (long)cdivu(g.M, 16) * cdivu(g.N, 16) * batch;
  if (t16 <= 32) return launch_tn<T, 1, 1, 4>(c, g, batch, 1024, A, B, C);
  // 64 x 32 tiles where they are full (256 x 160 x 13134: 31 against 43); for
  // FP32, whose MFMAs ask for operands twice as fast, 64 x 64 on large outputs
  // (384 x 240 x 19588 FP32: 79 against 83, 256 x 160 x 13134 FP32: 34 against 28)
  // and, from 2^30 products on, for all that does not fit one tile of 32: each
  // column of tiles reads the long operand from memory again (both products of a
  // KB term, 32 x 32 and 64 x 64: 864 x 64 x 43820 358 and 255, 2000 x 127 x 43820
  // 1262 and 829, 700 x 127 x 13134 154 and 128; below the line 256 x 127 x 13134
  // 58 and 63, 500 x 127 x 1648 33 and 36)
  if constexpr (sizeof(T) == 4) {
    const long lo = std::min(g.M, g.N), mn = (long)g.M * g.N;
    if ((lo >= 128 && mn >= 65536) || (lo > 32 && mn * g.K >= 1L << 30))
      return launch_tn<T, 4, 4, 1>(c, g, batch, kTarget, A, B, C);
  }
  if (std::min(g.M, g.N) >= 128)
    return launch_tn<T, 4, 2, 1>(c, g, batch, kTarget, A, B, C);
  return launch_tn<T, 2, 2, 2>(c, g, batch, kTarget, A, B, C);
}

template <typename T, int G, int BJ, int DP>
int launch_nn(Ctx* c, const GsArgs& g, int batch, const double* A, const double* B, double* C) {
  const dim3 grid(cdivu(g.M, 32 * G), cdivu(g.N, 16 * BJ), batch);
  const bool vec = !(g.M & 1) && !(g.lda & 1) && !(g.ldb & 1) && !(g.ldc & 1) && !(g.sA & 1) &&
                   !(g.sB & 1) && !(g.sC & 1) && aligned16(A) && aligned16(B) && aligned16(C);
  if (vec)
    hipLaunchKernelGGL((k_gs_nn<T, true, G, BJ, DP>), grid, dim3(64), 0, c->stream, g, A, B, C);
  else
    hipLaunchKernelGGL((k_gs_nn<T, false, G, BJ, DP>), grid, dim3(64), 0, c->stream, g, A, B, C);
  QX_CHECK(hipGetLastError());
  return 0;
}

// the largest tile that gives every SIMD (4 x 256) a wavefront, else the
// smallest: A is read once per 16 BJ columns
template <typename T>
int nn(Ctx* c, const GsArgs& g, int batch, const double* A, const double* B, double* C) {
  auto waves = [&](int G, int BJ) {
    return (long)cdivu(g.M, 32 * G) * cdivu(g.N, 16 * BJ) * batch;
  };
  if (waves(2, 4) >= 1024) return launch_nn<T, 2, 4, sizeof(T) == 8 ? 1 : 2>(c, g, batch, A, B, C);
  if (waves(2, 2) >= 1024) return launch_nn<T, 2, 2, sizeof(T) == 8 ? 3 : 4>(c, g, batch, A, B, C);
  return launch_nn<T, 1, 2, 6>(c, g, batch, A, B, C);
}

}  // namespace

int gs_gemm_tn(Ctx* c, int M, int N, int K, double alpha, const double* A, int lda, const double* B,
               int ldb, double beta, double* C, int ldc, int corr, int prec, const double* rscale,
               int batch, long sA, long sB, long sC) {
  if (M <= 0 || N <= 0 || batch <= 0) return 0;
  if (K < 1) return -1;
  GsArgs g{M, N, K, lda, ldb, ldc, corr, 1, K, 1, sA, sB, sC, alpha, beta, rscale};
  return prec == PREC_FP32 ? tn<float>(c, g, batch, A, B, C) : tn<double>(c, g, batch, A, B, C);
}

int gs_gemm_nn(Ctx* c, int M, int N, int K, double alpha, const double* A, int lda, const double* B,
               int ldb, double beta, double* C, int ldc, int prec, int batch, long sA, long sB,
               long sC) {
  if (M <= 0 || N <= 0 || batch <= 0) return 0;
  if (K < 1) return -1;
  GsArgs g{M, N, K, lda, ldb, ldc, 0, 1, K, 1, sA, sB, sC, alpha, beta, nullptr};
  return prec == PREC_FP32 ? nn<float>(c, g, batch, A, B, C) : nn<double>(c, g, batch, A, B, C);
}

}  // namespace qx
