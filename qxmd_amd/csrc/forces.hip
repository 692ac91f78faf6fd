// forces.hip -- Hellmann-Feynman forces of the KB nonlocal term (kbnlpp_frc2,
// Sources/nlkbpp.f90:1878-2060, lbigmm2 / VECTOR branch), as contractions:
//   P      = slmir = 2 B^T W psi - (G = 0 terms)       (the projection of hckbpp_g)
//   F_x    = B^T (J_x psi),  (J_x psi)(G) = i G_x psi(G) in the real-packed form,
//            i.e. (Re, Im) -> (G_x Im, -G_x Re), a plain sum over the sphere
//   f(ia) += 2 sum_{p of ia, b} F_x(p, b) P(p, b) 2 occ(b) vclalp(p)
// The bands are summed before the sphere: with the weighted sum of the bands a
// projector sees, Y_p = sum_b occ(b) P(p, b) psi_b,
//   sum_b occ(b) P(p, b) F_x(p, b) = sum_G G_x (Re B_p Im Y_p - Im B_p Re Y_p)
// takes one product of the projection's size for all three directions where the
// F_x take three, and one pass over B and Y, which is bound by memory.
// 216 atoms, 864 projectors, 432 bands, 22 k waves: 3.12 ms of products and
// weighting passes -> 1.55 (at that time's product kernel 1.80).
#include <algorithm>
#include <vector>
#include "context.h"

namespace qx {

namespace {

inline unsigned cdivu(long a, long b) { return (unsigned)((a + b - 1) / b); }

// g(c, p) = reference component c at the internal wave p
__global__ void k_force_g(const double* __restrict__ gref, const int* __restrict__ perm, int np,
                          double* __restrict__ g) {
  const int p = (int)(blockIdx.x * blockDim.x + threadIdx.x), c = (int)blockIdx.y;
  if (p < np) g[(size_t)c * np + p] = gref[(size_t)c * np + perm[p]];
}

// Z(b, p) = occ(b) P(p, b): tiles of 32 x 32 transposed through LDS
__global__ void __launch_bounds__(256) k_force_z(const double* __restrict__ P,
                                                 const double* __restrict__ occ, int npj, int nb,
                                                 double* __restrict__ Z) {
  __shared__ double t[32][33];
  const int p0 = (int)blockIdx.x * 32, b0 = (int)blockIdx.y * 32;
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
  for (int j = y; j < 32; j += 8)
    if (b0 + j < nb && p0 + x < npj) t[j][x] = occ[b0 + j] * P[(size_t)(b0 + j) * npj + p0 + x];
  __syncthreads();
  for (int j = y; j < 32; j += 8)
    if (p0 + j < npj && b0 + x < nb) Z[(size_t)(p0 + j) * nb + b0 + x] = t[x][j];
}

// T(q, p, c) = sum_{G of part q} g_c (Re B_p Im Y_p - Im B_p Re Y_p): kFrcRows
// projectors per workgroup, so that the three components are read once for them
// (they stay in L2; B and Y are read once from memory), and the sphere in
// kFrcParts parts for workgroups enough to fill the memory pipes (432 rows of
// 22 k waves: 1 part 104 us, 8 parts
// 64 us = 4.8 TB/s)
constexpr int kFrcRows = 4, kFrcParts = 8;
__global__ void __launch_bounds__(256) k_force_sum(const double* __restrict__ B,
                                                   const double* __restrict__ Y,
                                                   const double* __restrict__ g, int np, int n,
                                                   int rows, int npj, double* __restrict__ T) {
  __shared__ double red[4][3 * kFrcRows];
  const int r0 = (int)blockIdx.x * kFrcRows;
  double s[kFrcRows][3] = {};
  const int per = (np + kFrcParts - 1) / kFrcParts, part = (int)blockIdx.y;
  const int pe = min(np, (part + 1) * per);
  for (int p = part * per + (int)threadIdx.x; p < pe; p += blockDim.x) {
    const double gx = g[p], gy = g[np + p], gz = g[2 * (size_t)np + p];
#pragma unroll
    for (int r = 0; r < kFrcRows; ++r) {
      const size_t o = (size_t)min(r0 + r, rows - 1) * n + 2 * (size_t)p;
      const double2 bv = *reinterpret_cast<const double2*>(B + o);
      const double2 yv = *reinterpret_cast<const double2*>(Y + o);
      const double t = bv.x * yv.y - bv.y * yv.x;
      s[r][0] += gx * t;
      s[r][1] += gy * t;
      s[r][2] += gz * t;
    }
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int r = 0; r < kFrcRows; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double v = s[r][c];
      for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
      if (lane == 0) red[wv][3 * r + c] = v;
    }
  __syncthreads();
  const int i = threadIdx.x;
  if (i < 3 * kFrcRows && r0 + i / 3 < rows)
    T[3 * ((size_t)part * npj + r0) + i] = red[0][i] + red[1][i] + red[2][i] + red[3][i];
}

// f(ia, c) += 4 sum over the atom's projectors of vclalp T
__global__ void k_force_atoms(const double* __restrict__ T, const double* __restrict__ D,
                              const int* __restrict__ p0, int natom, int npj,
                              double* __restrict__ f) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= 3 * natom) return;
  const int ia = i / 3, c = i - 3 * ia;
  double s = 0.0;
  for (int p = p0[ia]; p < p0[ia + 1]; ++p) {
    double t = 0.0;
#pragma unroll
    for (int q = 0; q < kFrcParts; ++q) t += T[3 * ((size_t)q * npj + p) + c];
    s += D[p] * t;
  }
  f[i] += 4.0 * s;
}

}  // namespace

// n doubles for the length of a force call: grown on demand and kept for the next
// MD step's (a call ends synchronised); null when out of memory
double* call_workspace(Ctx* c, size_t n) {
  if (c->frc_len < n) {
    if (c->d_frc) (void)hipFree(c->d_frc);  // waits for what still reads it
    c->d_frc = nullptr;
    c->frc_len = 0;
    if (hipMalloc(&c->d_frc, sizeof(double) * n) != hipSuccess) {
      (void)hipGetLastError();
      return c->d_frc = nullptr;
    }
    c->frc_len = n;
  }
  return c->d_frc;
}

int kb_forces(Ctx* c, const double* psi, int nb, const double* occ_host, const double* gx,
              const double* gy, const double* gz, double* fnlc_host) {
  if (c->npj == 0 || c->natom == 0) return 0;
  const int n = c->nplwex, np = c->nplw + 1, npj = c->npj;
  if (nb < 1 || nb > c->nbmax) return -1;
  if (psi == c->d_slot[2]) return -1;  // Y's place
  // projections slmir = 2 B^T psi - G0 terms
  int rc = gemm_tn(c, npj, nb, n, 2.0, c->d_B, n, psi, n, 0.0, c->d_P, npj, 2);
  if (rc) return rc;
  // projector range of each atom (projectors are atom-major)
  std::vector<int> p0(c->natom + 1, 0);
  for (int p = 0; p < npj; ++p) p0[c->proj_atom[p] + 1]++;
  for (int ia = 0; ia < c->natom; ++ia) p0[ia + 1] += p0[ia];
  // Y in chunks of equal numbers of projectors: slot 2 holds nbmax of them; a
  // context of few bands brings 128 rows of its own rather than many thin
  // products
  const int cap = npj <= c->nbmax ? npj : std::max(c->nbmax, std::min(npj, 128));
  const int nch = (npj + cap - 1) / cap, rows = (npj + nch - 1) / nch;
  const size_t own_y = rows <= c->nbmax ? 0 : (size_t)rows * n;
  // one workspace: the upload [g | occ | f | p0], then g in internal order, Z, T, Y
  const size_t o_occ = 3 * (size_t)np, o_f = o_occ + nb, o_p0 = o_f + 3 * (size_t)c->natom;
  const size_t o_g = o_p0 + (p0.size() + 1) / 2, o_z = (o_g + 3 * (size_t)np + 1) / 2 * 2;
  const size_t o_t = o_z + (size_t)npj * nb, o_y = (o_t + 3 * (size_t)npj * kFrcParts + 1) / 2 * 2;
  double* w = call_workspace(c, o_y + own_y);
  if (!w) return -3;
  QX_CHECK(hipMemcpyAsync(w, gx, sizeof(double) * np, hipMemcpyHostToDevice, c->stream));
  QX_CHECK(hipMemcpyAsync(w + np, gy, sizeof(double) * np, hipMemcpyHostToDevice, c->stream));
  QX_CHECK(hipMemcpyAsync(w + 2 * (size_t)np, gz, sizeof(double) * np, hipMemcpyHostToDevice,
                          c->stream));
  QX_CHECK(hipMemcpyAsync(w + o_occ, occ_host, sizeof(double) * nb, hipMemcpyHostToDevice,
                          c->stream));
  QX_CHECK(hipMemcpyAsync(w + o_f, fnlc_host, sizeof(double) * 3 * c->natom,
                          hipMemcpyHostToDevice, c->stream));
  QX_CHECK(hipMemcpyAsync(w + o_p0, p0.data(), sizeof(int) * p0.size(), hipMemcpyHostToDevice,
                          c->stream));
  double *g = w + o_g, *Z = w + o_z, *T = w + o_t, *Y = own_y ? w + o_y : c->d_slot[2];
  hipLaunchKernelGGL(k_force_g, dim3(cdivu(np, 256), 3), dim3(256), 0, c->stream, w, c->d_perm, np,
                     g);
  hipLaunchKernelGGL(k_force_z, dim3(cdivu(npj, 32), cdivu(nb, 32)), dim3(256), 0, c->stream,
                     c->d_P, w + o_occ, npj, nb, Z);
  for (int r0 = 0; r0 < npj; r0 += rows) {
    const int nr = std::min(rows, npj - r0);
    rc = gemm_nn(c, n, nr, nb, 1.0, psi, n, Z + (size_t)r0 * nb, nb, 0.0, Y, n);
    if (rc) return rc;
    hipLaunchKernelGGL(k_force_sum, dim3(cdivu(nr, kFrcRows), kFrcParts), dim3(256), 0, c->stream,
                       c->d_B + (size_t)r0 * n, Y, g, np, n, nr, npj, T + 3 * (size_t)r0);
  }
  hipLaunchKernelGGL(k_force_atoms, dim3(cdivu(3L * c->natom, 256)), dim3(256), 0, c->stream, T,
                     c->d_D, reinterpret_cast<const int*>(w + o_p0), c->natom, npj, w + o_f);
  QX_CHECK(hipGetLastError());
  return read_host(c, {{fnlc_host, w + o_f, sizeof(double) * 3 * c->natom}});
}

}  // namespace qx
