// pencil_fast.hip -- launches of the two-step pencil FFTs (pencil_fast.h): the
// band-apply and the density of grids whose three edges are in QX_FFT_EDGES.
#include <algorithm>
#include <array>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include "pencil_fast.h"

namespace qx {

// the two radices of each axis, in slot-order conversions
struct SlotSplit {
  int n[3], na[3], nb[3];
};
__device__ inline long slot_to_grid(const SlotSplit& f, long i) {
  const int xs = (int)(i % f.n[0]);
  const long r = i / f.n[0];
  const int ys = (int)(r % f.n[1]), zs = (int)(r / f.n[1]);
  return slot_phys(xs, f.na[0], f.nb[0]) +
         (long)f.n[0] * (slot_phys(ys, f.na[1], f.nb[1]) +
                         (long)f.n[1] * slot_phys(zs, f.na[2], f.nb[2]));
}

// sum the group partials and undo the slot permutation of all three axes
__global__ void k_rho_reduce_f(const double* __restrict__ part, int ngrp, SlotSplit f, long NN,
                               double* __restrict__ rho) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= NN) return;
  double s = 0.0;
  for (int g = 0; g < ngrp; ++g) s += part[(size_t)g * NN + i];
  rho[slot_to_grid(f, i)] = s;
}

// V_perm[zs][ys][xs] = V[phys(zs)][phys(ys)][phys(xs)]
__global__ void k_permute_v(const double* __restrict__ V, double* __restrict__ Vp,
                            float* __restrict__ Vpf, SlotSplit f, long NN) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= NN) return;
  const double v = V[slot_to_grid(f, i)];
  Vp[i] = v;
  Vpf[i] = (float)v;
}

// --------------------------------------------------------------------------
// host side
// --------------------------------------------------------------------------
bool fast_split(int n, int* na, int* nb) {
  switch (n) {
#define QX_EDGE(N, NA, NB) \
  case N: *na = NA; *nb = NB; return true;
    QX_FFT_EDGES(QX_EDGE)
#undef QX_EDGE
    default: return false;
  }
}

static bool slot_split(const Ctx* c, SlotSplit* f) {
  const int n[3] = {c->n1, c->n2, c->n3};
  for (int a = 0; a < 3; ++a) {
    f->n[a] = n[a];
    if (!fast_split(n[a], &f->na[a], &f->nb[a])) return false;
  }
  return true;
}

template <typename T>
static EdgeKernels<T> edge_kernels(int n) {
  EdgeKernels<T> k;
  using Find = bool (*)(int, EdgeKernels<T>*);
  const Find groups[kFftGroups] = {edge_kernels_0, edge_kernels_1, edge_kernels_2, edge_kernels_3,
                                   edge_kernels_4, edge_kernels_5, edge_kernels_6, edge_kernels_7};
  for (Find g : groups)
    if (g(n, &k)) break;
  return k;
}

// the grid's edges are all covered (the x pass folds h and h - n1 onto one
// natural index, so the sphere's x extent must fit in one period)
bool fast_ok(const Ctx* c) {
  SlotSplit f;
  return slot_split(c, &f) && c->pc.nH <= c->n1 && std::getenv("QX_GENERIC_FFT") == nullptr;
}

int fast_permute_v(Ctx* c) {
  SlotSplit f;
  if (!slot_split(c, &f)) return 0;
  if (!c->d_Vp) {
    buffers_changed(c);
    QX_CHECK(hipMalloc(&c->d_Vp, sizeof(double) * c->N));
    QX_CHECK(hipMalloc(&c->d_Vpf, sizeof(float) * c->N));
  }
  hipLaunchKernelGGL(k_permute_v, dim3((unsigned)((c->N + 255) / 256)), dim3(256), 0, c->stream,
                     c->d_V, c->d_Vp, c->d_Vpf, f, c->N);
  QX_CHECK(hipGetLastError());
  return 0;
}

// The plane kernels' shape: x and y edges with their radices
struct PlaneShape {
  int n1, n2, xa, xb, ya, yb, nH, rw;
  int yk;  // YKind
  size_t elem;  // bytes of a complex value
  // LDS with nwave wavefronts and row strides sa (sphere tile), sr (x strips)
  size_t lds(int sa, int sr, int nwave) const {
    return elem * ((size_t)n1 + (yk == Y_CUBE ? 0 : n2) + (size_t)(nH + 1) * sa +
                   (size_t)nwave * rw * sr);
  }
};
template <typename T>
static PlaneShape plane_shape(const Ctx* c) {
  SlotSplit f;
  (void)slot_split(c, &f);
  PlaneShape s{};
  s.n1 = c->n1; s.n2 = c->n2;
  s.xa = f.na[0]; s.xb = f.nb[0]; s.ya = f.na[1]; s.yb = f.nb[1];
  s.nH = c->pc.nH;
  s.rw = plane_rows_per_wave(s.xa, s.xb);
  s.yk = c->n1 == c->n2 && c->n2 == c->n3 ? Y_CUBE : std::max(s.ya, s.yb) <= 10 ? Y_R10 : Y_R16;
  s.elem = sizeof(cplx<T>);
  return s;
}

static FastArgs fast_args(Ctx* c, const PlaneShape& s, int nb, int bp0) {
  FastArgs a{};
  a.n1 = c->n1; a.n2 = c->n2; a.n3 = c->n3;
  a.ya = s.ya; a.yb = s.yb;
  a.nH = c->pc.nH;
  a.hmax = (c->pc.nH - 1) / 2;
  a.hmin = -a.hmax;
  a.npair = c->pc.npair;
  a.ncol = c->pc.ncol;
  a.nplwex = c->nplwex;
  a.nb = nb;
  a.bp0 = bp0;
  a.pt_col = c->d_pt_col;
  a.pt_z = c->d_pt_z;
  a.pair_p0 = c->d_pair_p0;
  a.col_hi = c->d_col_hi;
  a.col_kmod = c->d_col_kmod;
  a.kin = c->d_kin;
  a.tw = c->d_tw;
  return a;
}

constexpr size_t kCuLds = 160 * 1024;

// wavefronts per plane block: 8 unless the LDS strips would not fit
static int plane_waves(const PlaneShape& s) {
  int w = kPlaneMaxThreads / 64;
  if (const char* e = std::getenv("QX_PLANE_WAVES")) w = std::max(1, std::min(w, std::atoi(e)));
  while (w > 1 && s.lds(s.n2, s.n1, w) > kCuLds) w /= 2;
  return s.lds(s.n2, s.n1, w) <= kCuLds ? w : -1;
}

// Passes one wavefront LDS access takes when each lane moves el dwords: 64
// banks of 4 bytes serve 64/el lanes per pass, and a pass lasts as many
// cycles as the most distinct addresses one bank is asked for (lanes reading
// the same address share it).  e[l] < 0 marks an idle lane.
// (banks = 64; the variant with 32 banks serves 32/el lanes per pass)
static int lds_passes(const int* e, int el, int banks = 64) {
  int tot = 0;
  const int lpp = banks / el;
  for (int g = 0; g < 64; g += lpp) {
    int d[64], nd = 0;
    for (int l = g; l < g + lpp; ++l)
      if (e[l] >= 0)
        for (int k = 0; k < el; ++k) d[nd++] = el * e[l] + k;
    if (!nd) continue;
    std::sort(d, d + nd);
    nd = (int)(std::unique(d, d + nd) - d);
    int cnt[64] = {0}, mx = 0;
    for (int i = 0; i < nd; ++i) mx = std::max(mx, ++cnt[d[i] & (banks - 1)]);
    tot += mx;
  }
  return tot;
}

// modelled LDS passes of the accesses that depend on the sphere tile stride
// sa (y passes and the x pass's column reads/writes) ...
static long plane_cost_sa(const PlaneShape& s, int sa, int banks) {
  const int NA = s.xa, NB = s.xb, N = s.n1, nH = s.nH, hmax = (nH - 1) / 2, RW = s.rw;
  const int el = (int)s.elem / 4;
  long c = 0;
  int e[64];
  for (int step = 0; step < 2; ++step) {
    const int K = step == 0 ? s.yb : s.ya, Q = step == 0 ? s.ya : s.yb, n = nH * K;
    for (int q = 0; q < Q; ++q)
      for (int w0 = 0; w0 < n; w0 += 64) {
        for (int l = 0; l < 64; ++l) {
          const int it = w0 + l, line = it % nH, j = it / nH;
          e[l] = it < n ? line * sa + (step == 0 ? j + s.yb * q : s.yb * j + q) : -1;
        }
        c += 4 * lds_passes(e, el, banks);  // inverse and forward, read and write
      }
  }
  for (int y0 = 0; y0 < s.n2; y0 += RW)
    for (int q = 0; q < NA; ++q) {
      int e2[64];
      for (int l = 0; l < 64; ++l) {
        const int rx = l % RW, jx = l / RW, n = jx + NB * q;
        const int h = n <= hmax ? n : (n >= N - hmax ? n - N : N);
        const bool ok = jx < NB && y0 + rx < s.n2;
        // step A reads every slot (the zero row nH outside the sphere), step A'
        // writes the sphere's slots only
        e[l] = ok ? (h < N ? h + hmax : nH) * sa + y0 + rx : -1;
        e2[l] = ok && h < N ? (h + hmax) * sa + y0 + rx : -1;
      }
      c += lds_passes(e, el, banks) + lds_passes(e2, el, banks);
    }
  return c;
}

// ... and on the x strip stride sr
static long plane_cost_sr(const PlaneShape& s, int sr, int banks) {
  const int NA = s.xa, NB = s.xb, RW = s.rw, el = (int)s.elem / 4;
  long c = 0;
  int e[64];
  for (int y0 = 0; y0 < s.n2; y0 += RW) {
    for (int q = 0; q < NA; ++q) {
      for (int l = 0; l < 64; ++l) {
        const int rx = l % RW, jx = l / RW;
        e[l] = (jx < NB && y0 + rx < s.n2) ? rx * sr + jx + NB * q : -1;
      }
      c += 2 * lds_passes(e, el, banks);
    }
    for (int q = 0; q < NB; ++q) {
      for (int l = 0; l < 64; ++l) {
        const int rx = l % RW, jx = l / RW;
        e[l] = (jx < NA && y0 + rx < s.n2) ? rx * sr + NB * jx + q : -1;
      }
      c += 2 * lds_passes(e, el, banks);
    }
  }
  return c;
}

// Row strides of the plane kernel: pairs in [n2, n2+32] x [n1, n1+32] ranked by
// the modelled LDS passes, among those that keep as many blocks per CU as
// unpadded rows do; the best `keep` pairs are returned (the first is the
// model's choice).
static std::vector<std::pair<int, int>> plane_stride_ranks(const PlaneShape& s, int nwave,
                                                           int keep, int banks = 64) {
  const size_t occ0 = kCuLds / s.lds(s.n2, s.n1, nwave);
  long csr[33];
  for (int d = 0; d <= 32; ++d) csr[d] = plane_cost_sr(s, s.n1 + d, banks);
  std::vector<std::pair<long, std::pair<int, int>>> all;
  for (int da = 0; da <= 32; ++da) {
    const long ca = plane_cost_sa(s, s.n2 + da, banks);
    for (int dr = 0; dr <= 32; ++dr) {
      const size_t l = s.lds(s.n2 + da, s.n1 + dr, nwave);
      if (l > kCuLds || kCuLds / l < occ0) continue;
      all.push_back({ca + csr[dr], {s.n2 + da, s.n1 + dr}});
    }
  }
  std::stable_sort(all.begin(), all.end(),
                   [](const auto& x, const auto& y) { return x.first < y.first; });
  std::vector<std::pair<int, int>> r;
  for (const auto& x : all) {
    if ((int)r.size() >= keep) break;
    r.push_back(x.second);
  }
  if (r.empty()) r.push_back({s.n2, s.n1});
  return r;
}

// the model's stride pair (QX_PLANE_SA / QX_PLANE_SR override), kept per shape
// (all that the ranking reads: an n x n plane of a cube, of which yk is Y_CUBE,
// has one twiddle table in LDS, that of a slab two)
static void plane_strides(const PlaneShape& s, int nwave, int* psa, int* psr) {
  static std::mutex mu;
  static std::map<std::array<int, 6>, std::pair<int, int>> cache;
  const std::array<int, 6> key{s.n1, s.n2, s.yk, s.nH, (int)s.elem, nwave};
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(key);
    if (it == cache.end()) it = cache.emplace(key, plane_stride_ranks(s, nwave, 1)[0]).first;
    *psa = it->second.first;
    *psr = it->second.second;
  }
  if (const char* e = std::getenv("QX_PLANE_SA")) *psa = std::max(s.n2, std::atoi(e));
  if (const char* e = std::getenv("QX_PLANE_SR")) *psr = std::max(s.n1, std::atoi(e));
}

// Stride pairs the plane tuner times: the three best of the bank model with
// 64 banks and with 32, and a coarse grid of odd paddings (the model's
// conflict counts have not matched the measured ones, so time decides), all
// keeping the blocks per CU of unpadded rows.
static std::vector<std::pair<int, int>> plane_stride_candidates(const PlaneShape& s, int nwave) {
  std::vector<std::pair<int, int>> v = plane_stride_ranks(s, nwave, 3, 64);
  for (const auto& p : plane_stride_ranks(s, nwave, 3, 32))
    if (std::find(v.begin(), v.end(), p) == v.end()) v.push_back(p);
  const size_t occ0 = kCuLds / s.lds(s.n2, s.n1, nwave);
  for (int da : {1, 3, 5, 9, 17})
    for (int dr : {1, 5, 9, 17}) {
      const std::pair<int, int> p{s.n2 + da, s.n1 + dr};
      const size_t l = s.lds(p.first, p.second, nwave);
      if (l > kCuLds || kCuLds / l < occ0) continue;
      if (std::find(v.begin(), v.end(), p) == v.end()) v.push_back(p);
    }
  return v;
}

// mid (optional): work launched between the plane pass and the z forward pass,
// e.g. the KB contractions of the fused mixed band-apply (needs one batch)
struct FastMid {
  float* psi32;        // FP32 copy of psi, written by the z inverse pass, or
  unsigned short* psis;  // its bf16 hi | lo split (row stride ldk, lo at slo)
  int ldk;
  long slo;
  const float* kb32;   // FP32 term the z forward pass adds
  int (*run)(Ctx*, const double*, int, const FastMid&);
};

// Launch shape of the band-apply plane kernel: wavefronts per block and the
// two LDS row strides.  On the first band-apply of a shape the candidates
// (8 and 4 wavefronts, the model's three best stride pairs for each) are
// timed on the real z-pencils (k_zinv_f fills T1 first; the trial launches
// write only T2) and the fastest is kept for the process; QX_FFT_NOTUNE=1
// takes the model's choice.
struct PlaneCfg {
  int nwave = 0, sa = 0, sr = 0;
  float ms = 0.f;
};

// opt in to dynamic LDS beyond the 64 KiB default
static void plane_lds_optin(const void* fn, size_t bytes) {
  if (bytes > 65536)
    (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// blocks of the z kernels along the column pairs
template <typename T>
static unsigned zblocks(const Ctx* c) {
  const int pb = zpairs(c->n3, (int)sizeof(cplx<T>));
  return (unsigned)((c->pc.npair + pb - 1) / pb);
}

template <typename T>
static PlaneCfg plane_config(Ctx* c, const PlaneShape& s, typename EdgeKernels<T>::ZInv zinv,
                             typename EdgeKernels<T>::Plane plane, const double* psi, int nb,
                             const T* Vp, cplx<T>* t1, cplx<T>* t2, int nbb) {
  static std::mutex mu;
  static std::map<std::array<int, 4>, PlaneCfg> tuned;
  const std::array<int, 4> key{s.n1, s.n2, c->n3, s.nH};
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = tuned.find(key);
    if (it != tuned.end()) return it->second;
  }
  PlaneCfg best;
  best.nwave = plane_waves(s);
  if (best.nwave < 1) return best;
  plane_strides(s, best.nwave, &best.sa, &best.sr);
  const bool fixed = std::getenv("QX_FFT_NOTUNE") || std::getenv("QX_PLANE_WAVES") ||
                     std::getenv("QX_PLANE_SA") || std::getenv("QX_PLANE_SR");
  if (!fixed) {
    FastArgs a = fast_args(c, s, nb, 0);
    hipLaunchKernelGGL(zinv, dim3(zblocks<T>(c), nbb), dim3(kFastThreads), 0, c->stream, a, psi,
                       t1, nullptr, nullptr, 0, 0L);
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess) {
      float bms = 1e30f;
      for (int nw = kPlaneMaxThreads / 64; nw >= 4; nw /= 2) {
        if (s.lds(s.n2, s.n1, nw) > kCuLds) continue;
        for (const auto& st : plane_stride_candidates(s, nw)) {
          const size_t lp = s.lds(st.first, st.second, nw);
          if (lp > kCuLds) continue;
          plane_lds_optin(reinterpret_cast<const void*>(plane), lp);
          a.sa = st.first;
          a.sr = st.second;
          hipLaunchKernelGGL(plane, dim3(c->n3, nbb), dim3(64 * nw), lp, c->stream, a, Vp, t1, t2);
          (void)hipEventRecord(e0, c->stream);
          for (int r = 0; r < 2; ++r)
            hipLaunchKernelGGL(plane, dim3(c->n3, nbb), dim3(64 * nw), lp, c->stream, a, Vp, t1,
                               t2);
          (void)hipEventRecord(e1, c->stream);
          (void)hipEventSynchronize(e1);
          float ms = 0.f;
          (void)hipEventElapsedTime(&ms, e0, e1);
          if (std::getenv("QX_FFT_VERBOSE"))
            fprintf(stderr, "plane tune %dx%d nH=%d T%zu: %d waves, sa %d sr %d: %.4f ms\n", s.n1,
                    s.n2, s.nH, sizeof(T), nw, st.first, st.second, ms / 2);
          if (hipGetLastError() == hipSuccess && ms > 0.f && ms < bms) {
            bms = ms;
            best.nwave = nw;
            best.sa = st.first;
            best.sr = st.second;
            best.ms = ms / 2;
          }
        }
      }
      (void)hipEventDestroy(e0);
      (void)hipEventDestroy(e1);
    }
  }
  std::lock_guard<std::mutex> lk(mu);
  tuned[key] = best;
  return best;
}

// band pairs per pencil batch
template <typename T>
static int pencil_batch(const Ctx* c, int nbp) {
  const size_t per_bp = sizeof(cplx<T>) * (size_t)c->n3 * c->pc.ncol;
  return (int)std::max<size_t>(1, std::min<size_t>(c->t_bytes / per_bp, (size_t)nbp));
}

template <typename T>
static int local_fast_t(Ctx* c, const double* psi, double* out, int nb, int accumulate,
                        const FastMid* mid = nullptr) {
  const PlaneShape s = plane_shape<T>(c);
  const EdgeKernels<T> kz = edge_kernels<T>(c->n3);
  const auto plane = edge_kernels<T>(c->n1).plane[s.yk];
  if (!kz.zinv || !kz.zfwd || !plane) return -3;
  const int nbp = (nb + 1) / 2;
  const int batch = pencil_batch<T>(c, nbp);
  const unsigned gz = zblocks<T>(c);
  cplx<T>* t1 = reinterpret_cast<cplx<T>*>(c->d_t1);
  cplx<T>* t2 = reinterpret_cast<cplx<T>*>(c->d_t2);
  const T* Vp = sizeof(T) == 8 ? reinterpret_cast<const T*>(c->d_Vp)
                               : reinterpret_cast<const T*>(c->d_Vpf);
  if (mid && batch < nbp) return -3;
  const PlaneCfg cfg =
      plane_config<T>(c, s, kz.zinv, plane, psi, nb, Vp, t1, t2, std::min(batch, nbp));
  const int nwave = cfg.nwave;
  if (nwave < 1) return -3;
  const size_t lp = s.lds(cfg.sa, cfg.sr, nwave);
  if (lp > kCuLds) return -3;
  plane_lds_optin(reinterpret_cast<const void*>(plane), lp);
  for (int bp0 = 0; bp0 < nbp; bp0 += batch) {
    const int nbb = std::min(batch, nbp - bp0);
    FastArgs a = fast_args(c, s, nb, bp0);
    a.sa = cfg.sa;
    a.sr = cfg.sr;
    lt_mark(c, 1, false);
    hipLaunchKernelGGL(kz.zinv, dim3(gz, nbb), dim3(kFastThreads), 0, c->stream, a, psi, t1,
                       mid ? mid->psi32 : nullptr, mid ? mid->psis : nullptr, mid ? mid->ldk : 0,
                       mid ? mid->slo : 0L);
    hipLaunchKernelGGL(plane, dim3(c->n3, nbb), dim3(64 * nwave), lp, c->stream, a, Vp, t1, t2);
    if (mid) {  // the mid work is not part of the FFT stage's launch time
      lt_mark(c, 1, true);
      const int rc = mid->run(c, psi, nb, *mid);
      if (rc) return rc;
      lt_mark(c, 1, false, true);
    }
    hipLaunchKernelGGL(kz.zfwd, dim3(gz, nbb), dim3(kFastThreads), 0, c->stream, a, psi, t2, out,
                       accumulate, 1.0 / (double)c->N, mid ? mid->kb32 : nullptr);
    lt_mark(c, 1, true);
  }
  QX_CHECK(hipGetLastError());
  return 0;
}

int kp_local_fast(Ctx* c, KFastArgs a, int nH, const double* src, double* dst, double2* T,
                  int nkb) {
  if (!fast_ok(c) || !c->d_Vp || nH > c->n1) return -3;
  PlaneShape s = plane_shape<double>(c);
  s.nH = nH;
  const EdgeKernels<double> kz = edge_kernels<double>(c->n3);
  const auto plane = edge_kernels<double>(c->n1).kplane[s.yk];
  if (!kz.kzinv || !kz.kzfwd || !plane) return -3;
  // 8 wavefronts a block, 4 where the x pass has no more than four row groups (36 x
  // 36, 1280 (k, band) blocks, whole local part: 600 us with 8, 421 with 4).  Where
  // it has two to four, the launch blocks enough and six fit a CU, two: the other
  // blocks fill the time at the barriers, and fewer wavefronts wait for a last row
  // group.  With 4 and 2 wavefronts, 1280 (k, band) blocks, us: 20^3 121, 98; 24^3
  // 226, 146; 28^3 272, 238; 30^3 296, 240; 32^3 331, 277; 36^3 423, 409; at the
  // line, 4100 planes: 40, 37; 55, 44; 59, 55; 59, 54; 64, 59; 65, 63; at half of
  // it: 31, 28; 38, 32; 41, 40; 41, 37; 43, 40; 46, 47.  One row group (16^3): 77, 81
  int nwave = plane_waves(s);
  const int groups = (s.n2 + s.rw - 1) / s.rw;
  if (nwave == 8 && groups <= 4) nwave = 4;
  if (nwave == 4 && groups > 1 && groups <= 4 && (long)c->n3 * nkb >= 4096 &&
      6 * s.lds(s.n2, s.n1, 2) <= kCuLds)
    nwave = 2;
  if (nwave < 1) return -3;
  FastArgs f = fast_args(c, s, 0, 0);
  plane_strides(s, nwave, &f.sa, &f.sr);
  const size_t lp = s.lds(f.sa, f.sr, nwave);
  if (lp > kCuLds) return -3;
  plane_lds_optin(reinterpret_cast<const void*>(plane), lp);
  a.f = f;
  cplx<double>* t = reinterpret_cast<cplx<double>*>(T);
  const dim3 gz((unsigned)((a.ncol_max + kKFastCols - 1) / kKFastCols), nkb);
  hipLaunchKernelGGL(kz.kzinv, gz, dim3(kFastThreads), 0, c->stream, a, src, t);
  hipLaunchKernelGGL(plane, dim3(c->n3, nkb), dim3(64 * nwave), lp, c->stream, a, c->d_Vp, t);
  hipLaunchKernelGGL(kz.kzfwd, gz, dim3(kFastThreads), 0, c->stream, a, src, t, dst,
                     1.0 / (double)c->N);
  QX_CHECK(hipGetLastError());
  return 0;
}

template <typename T>
static int density_fast_t(Ctx* c, const double* psi, int nb, const double* w) {
  const PlaneShape s = plane_shape<T>(c);
  const int nwave = plane_waves(s);
  // row groups per wavefront: the fewest of 2, 4, 6 that cover the plane's rows
  const int ng_rows = (s.n2 + s.rw - 1) / s.rw;
  if (nwave < 1 || nwave * kRhoGroups < ng_rows) return -3;
  const int rk = nwave * 2 >= ng_rows ? 0 : nwave * 4 >= ng_rows ? 1 : 2;
  const int rg = rk == 2 ? kRhoGroups : 2 * (rk + 1);
  if (64 * nwave > rho_max_threads(rg)) return -3;
  const EdgeKernels<T> kz = edge_kernels<T>(c->n3);
  const auto rho = edge_kernels<T>(c->n1).rho[s.yk][rk];
  if (!kz.zinv || !rho) return -3;
  int sa, sr;
  plane_strides(s, nwave, &sa, &sr);
  const size_t lp = s.lds(sa, sr, nwave);
  if (lp > kCuLds) return -3;
  plane_lds_optin(reinterpret_cast<const void*>(rho), lp);
  const int nbp = (nb + 1) / 2;
  const int batch = pencil_batch<T>(c, nbp);
  cplx<T>* t1 = reinterpret_cast<cplx<T>*>(c->d_t1);
  const int nbatch = (nbp + batch - 1) / batch;
  const int groups_per_batch = std::max(1, c->rho_groups / nbatch);
  if (groups_per_batch * nbatch > c->rho_groups) return -4;
  int nparts = 0;
  for (int bp0 = 0; bp0 < nbp; bp0 += batch) {
    const int nbb = std::min(batch, nbp - bp0);
    FastArgs a = fast_args(c, s, nb, bp0);
    a.sa = sa;
    a.sr = sr;
    hipLaunchKernelGGL(kz.zinv, dim3(zblocks<T>(c), nbb), dim3(kFastThreads), 0, c->stream, a, psi,
                       t1, nullptr, nullptr, 0, 0L);
    int ng = std::min(groups_per_batch, nbb);
    const int per = (nbb + ng - 1) / ng;
    ng = (nbb + per - 1) / per;
    hipLaunchKernelGGL(rho, dim3(c->n3, ng), dim3(64 * nwave), lp, c->stream, a, t1, nbb, per, w,
                       c->d_rho_part + (size_t)nparts * c->N);
    nparts += ng;
  }
  SlotSplit f;
  (void)slot_split(c, &f);
  hipLaunchKernelGGL(k_rho_reduce_f, dim3((unsigned)((c->N + 255) / 256)), dim3(256), 0, c->stream,
                     c->d_rho_part, nparts, f, c->N, c->d_rho);
  QX_CHECK(hipGetLastError());
  return 0;
}

static int fused_kb_mid(Ctx* c, const double* psi, int nb, const FastMid& m) {
  return kb_mixed_f32(c, psi, m.psi32, m.psis, m.ldk, m.slo, nb, const_cast<float*>(m.kb32));
}

int hpsi_mixed_fused(Ctx* c, const double* psi, double* out, int nb) {
  if (!fast_ok(c) || !c->d_Vp || c->npj == 0 || std::getenv("QX_HPSI_UNFUSED") ||
      gemm_path() == GEMM_OWN_F32 || !use_big(c->npj, nb) ||
      !use_big(c->nplwex, nb) || (c->nplwex & 1) || (c->npj & 1))
    return -3;
  FastMid m{};
  if (gemm_path() == GEMM_OWN) {
    // the bf16 split of psi, band rows of round_up(nplwex, 64) (zero pads),
    // the lo half after room for nbmax bands, so the pads never move
    m.ldk = (c->nplwex + 63) / 64 * 64;
    m.slo = (long)c->nbmax * m.ldk;
    m.psis = mg_u16_scratch(c, 0, 2 * (size_t)m.slo);
    if (!m.psis) return -3;
  } else {
    m.psi32 = mg_f32_scratch(c, 0, (size_t)c->nplwex * nb);
    if (!m.psi32) return -3;
  }
  m.kb32 = mg_f32_scratch(c, 1, (size_t)c->nplwex * nb);
  m.run = fused_kb_mid;
  if (!m.kb32) return -3;
  return local_fast_t<float>(c, psi, out, nb, 0, &m);
}

int local_apply_fast(Ctx* c, const double* psi, double* out, int nb, int prec, int accumulate) {
  if (prec == PREC_FP32) return local_fast_t<float>(c, psi, out, nb, accumulate);
  return local_fast_t<double>(c, psi, out, nb, accumulate);
}

int density_fast(Ctx* c, const double* psi, int nb, const double* w, int prec) {
  if (prec == PREC_FP32) return density_fast_t<float>(c, psi, nb, w);
  return density_fast_t<double>(c, psi, nb, w);
}

}  // namespace qx
