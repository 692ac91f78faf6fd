// pencil_inst.hip -- instantiates the pencil FFT kernels of one group of edges
// (QX_FFT_GROUP, compiled once per group so that the groups build in parallel).
#include "pencil_fast.h"

#define QX_CAT2(a, b) a##b
#define QX_CAT(a, b) QX_CAT2(a, b)

namespace qx {

template <typename T, int NA, int NB>
static void fill(EdgeKernels<T>* k) {
  k->zinv = k_zinv_f<T, NA, NB>;
  k->zfwd = k_zfwd_f<T, NA, NB>;
  k->plane[Y_CUBE] = k_plane_f<T, NA, NB, Y_CUBE>;
  k->plane[Y_R10] = k_plane_f<T, NA, NB, Y_R10>;
  k->plane[Y_R16] = k_plane_f<T, NA, NB, Y_R16>;
  k->rho[Y_CUBE][0] = k_plane_rho_f<T, NA, NB, Y_CUBE, 2>;
  k->rho[Y_CUBE][1] = k_plane_rho_f<T, NA, NB, Y_CUBE, 4>;
  k->rho[Y_CUBE][2] = k_plane_rho_f<T, NA, NB, Y_CUBE, kRhoGroups>;
  k->rho[Y_R10][0] = k_plane_rho_f<T, NA, NB, Y_R10, 2>;
  k->rho[Y_R10][1] = k_plane_rho_f<T, NA, NB, Y_R10, 4>;
  k->rho[Y_R16][0] = k_plane_rho_f<T, NA, NB, Y_R16, 2>;
  k->rho[Y_R16][1] = k_plane_rho_f<T, NA, NB, Y_R16, 4>;
  if constexpr (sizeof(T) == 8) {
    k->kzinv = k_kzinv_f<NA, NB>;
    k->kzfwd = k_kzfwd_f<NA, NB>;
    k->kplane[Y_CUBE] = k_kplane_f<NA, NB, Y_CUBE>;
    k->kplane[Y_R10] = k_kplane_f<NA, NB, Y_R10>;
    k->kplane[Y_R16] = k_kplane_f<NA, NB, Y_R16>;
  }
}

template <typename T>
static bool lookup(int n, EdgeKernels<T>* k) {
  switch (n) {
#define QX_EDGE(N, NA, NB) \
  case N: fill<T, NA, NB>(k); return true;
    QX_CAT(QX_FFT_EDGES_, QX_FFT_GROUP)(QX_EDGE)
#undef QX_EDGE
    default: return false;
  }
}

bool QX_CAT(edge_kernels_, QX_FFT_GROUP)(int n, EdgeKernels<float>* k) { return lookup(n, k); }
bool QX_CAT(edge_kernels_, QX_FFT_GROUP)(int n, EdgeKernels<double>* k) { return lookup(n, k); }

}  // namespace qx
