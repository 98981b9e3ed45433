// sph_output.h -- the downloads' kernels: fields of the sorted state written
// as FP64 in the original particle order.
//
// Bound by HBM and the scatter of the ids: consecutive ids lie in runs of a
// cell's row, so a wavefront's stores fall in a few dozen lines.  One launch
// for all the asked fields; null pointers are left out.
#pragma once

#include "sph3d.h"

namespace arm {

template <typename R> __device__ __forceinline__ double2 slot_x(const St<R>& S, int t) { return S.xy[t]; }
template <typename R> __device__ __forceinline__ double4 slot_x(const St3<R>& S, int t) { return S.xyz[t]; }
template <typename R> struct Dim { static constexpr int n = 3; };
template <> struct Dim<double2> { static constexpr int n = 2; };
template <> struct Dim<float2> { static constexpr int n = 2; };

// Vector v of particle i of n: interleaved (apart = 0) or one array per axis.
template <typename V>
__device__ __forceinline__ void put_axes(double* __restrict__ out, const V& v, int i, int n,
                                         int apart) {
  constexpr int D = Dim<V>::n;
  const size_t at = apart ? (size_t)i : (size_t)D * i, step = apart ? (size_t)n : 1;
  out[at] = (double)v.x;
  out[at + step] = (double)v.y;
  if constexpr (D == 3) out[at + 2 * step] = (double)v.z;
}

__device__ __forceinline__ double full_rho(const KParams&, double r) { return r; }
__device__ __forceinline__ double full_rho(const KParams& K, float r) { return K.rho0 + (double)r; }

// Ghosts (ids >= nb) are left out: arm_download_ghosts gives them.
template <typename ST>
__global__ __launch_bounds__(BLOCK) void k_state_out(ST S, KParams K, int apart,
                                                     double* __restrict__ x,
                                                     double* __restrict__ v,
                                                     double* __restrict__ rho,
                                                     double* __restrict__ p,
                                                     double* __restrict__ u) {
  const int t = blockIdx.x * BLOCK + threadIdx.x;
  if (t >= K.n) return;
  const int i = S.id[t];
  if (i >= K.nb) return;
  if (x) put_axes(x, slot_x(S, t), i, K.nb, apart);
  if (v) put_axes(v, S.v[t], i, K.nb, apart);
  if (rho) rho[i] = full_rho(K, S.rho[t]);
  if (p) p[i] = (double)S.p[t];
  if (u) u[i] = S.u[t];
}

template <typename ST>
__global__ __launch_bounds__(BLOCK) void k_rates_out(ST S, KParams K, int apart,
                                                     double* __restrict__ drho,
                                                     double* __restrict__ a,
                                                     double* __restrict__ du,
                                                     double* __restrict__ av,
                                                     double* __restrict__ divv) {
  const int t = blockIdx.x * BLOCK + threadIdx.x;
  if (t >= K.n) return;
  const int i = S.id[t];
  if (i >= K.nb) return;
  if (drho) drho[i] = (double)S.drho[t];
  if (a) put_axes(a, S.a[t], i, K.nb, apart);
  if (du) du[i] = (double)S.du[t];
  if (av) put_axes(av, S.av[t], i, K.nb, apart);
  if (divv) divv[i] = (double)S.divv[t];
}

}  // namespace arm
