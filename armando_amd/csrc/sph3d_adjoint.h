// sph3d_adjoint.h -- discrete adjoint of the 3D step, for the FP64 plain
// form and the FP32 chosen form (FP32 pair arithmetic on the cell + offset
// positions, FP64 state adjoints), with the derivation of the 2D adjoint in
// sph_adjoint.h carried to three components:
//   density   drho_i = sum_j m F vr,  S_i = -sum_j m F vr (divv_i = S_i/rho_i)
//   EOS       p = Tait(rho) or c0^2 rho + p0 with the pmin clamp; psi, Q, A
//   force     G = m F (A_i Q_j + A_j Q_i + Pi),  a_i = -sum G r + g,
//             du_i = sum G vr/2 + H (u_i - u_j),  av_i = -sum eps m M W dv
//   leapfrog  time_integration.f:136-217
// r = x_i - x_j (3 components), vr = (v_i - v_j).r, grad W = F r with the
// 3D Wendland constants of KParams.  Neighbour lists and branches are those
// of the forward step.  Pair terms are gathered per particle (each pair is
// visited from both ends), so no atomics are needed.
#pragma once

#include "sph3d.h"

namespace arm {

// one recorded 3D step: the sorted state after the force pass; the density
// pass of a recorded step writes its masks here itself
template <typename R> struct Tape3 {
  using R4 = typename V4<R>::type;
  int32_t* id;
  double4* xyz;
  float4* pf;  // FP32 form: cell column + offsets of the pair arithmetic
  R4* v;
  R* rho;
  double* u;
  R* psi;
  R* divv;
  R* p;
  R* drho;
  R* du;
  R4* a;
  R4* av;
  R* rho_min;
  double* u_min;
  R4* v_min;
  uint8_t* flag;
  uint32_t* skey;
  int* cstart;
  uint32_t* nbm;  // the forward's neighbour masks (Mask3 layout, stride n)
};

__device__ __forceinline__ Pos3D tape_pos3(const Tape3<double>& T, int t) {
  const double4 q = T.xyz[t];
  return {q.x, q.y, q.z};
}
__device__ __forceinline__ Pos3F tape_pos3(const Tape3<float>& T, int t) {
  const float4 q = T.pf[t];
  return {q.w, q.x, q.y, q.z};
}

// state adjoints in id order: after the step (in), before it (out), and of
// the rates carried into the next predictor
struct AdjState3 {
  double *x, *y, *z, *vx, *vy, *vz, *rho, *u;
  double *bx, *by, *bz, *bvx, *bvy, *bvz, *brho, *bu;
  double *cax, *cay, *caz, *cdrho, *cdu;
};

// per-step scratch in sorted order.  What the reverse gathers read of a
// neighbour lies in two records, written by k3_adj_corrector: for both passes
//   rec   position (pf / xyz), (v, Q)
//   frec  (la, A), (lav, psi), (u, ldu, -, -)
// for the force pass, with Q = 1/rho, A = p/rho and la, lav, ldu the adjoints
// of the rates; k3_adj_eos puts the density pass's lt = ldrho - lS in the
// place of Q.  (One record of five vectors for both made the density pass
// fetch two and a half times its lines: 798 us
// instead of 538 at 2.2M particles in FP32.)
template <typename R> struct AdjScratch3 {
  typename V4<R>::type *rec, *frec;  // 2 and 3 vectors per particle
  R *ldrho, *lp;
  R *lQ, *lA, *lpsi, *lrhoh, *lu, *lvx, *lvy, *lvz, *lx, *ly, *lz;
  R* lus;
};

__device__ __forceinline__ float4 tape_rec3(const Tape3<float>& T, int t) { return T.pf[t]; }
__device__ __forceinline__ double4 tape_rec3(const Tape3<double>& T, int t) { return T.xyz[t]; }

template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_tape(St3<R> S, KParams K,
                                                 const uint32_t* __restrict__ skey,
                                                 const int* __restrict__ cstart, Tape3<R> T) {
  const int t = blockIdx.x * BLOCK + threadIdx.x;
  const int stride = gridDim.x * BLOCK;
  for (int c = t; c <= K.ncell; c += stride) T.cstart[c] = cstart[c];
  if (t >= K.n) return;
  T.id[t] = S.id[t];
  T.xyz[t] = S.xyz[t];
  if constexpr (sizeof(R) == 4) T.pf[t] = S.pf[t];
  T.v[t] = S.v[t];
  T.rho[t] = S.rho[t];
  T.u[t] = S.u[t];
  T.psi[t] = S.psi[t];
  T.divv[t] = S.divv[t];
  T.p[t] = S.p[t];
  T.drho[t] = S.drho[t];
  T.du[t] = S.du[t];
  T.a[t] = S.a[t];
  T.av[t] = S.av[t];
  T.rho_min[t] = S.rho_min[t];
  T.u_min[t] = S.u_min[t];
  T.v_min[t] = S.v_min[t];
  T.flag[t] = S.flag[t];
  T.skey[t] = skey[t];
}

// The lane columns of a wavefront's walk over its mask words.
struct WalkLds3 {
  uint32_t w[M3_OK][64];
  int t0[9][64];
};

// Calls visit(l, uy, uz) for every neighbour l of particle k of the taped
// step, in the forward's order: from the recorded masks when they are
// complete, in one loop over the set bits of all 27 words (a wavefront runs
// for its longest lane's neighbour count), else by testing the candidates
// again.  Wavefront s0 of NS visits its share of them (share_bits).
template <int NS, typename R, typename Visit>
__device__ __forceinline__ void for_tape_neighbours3(const Tape3<R>& T, const KParams& K, int s0,
                                                     int k, WalkLds3& L, Visit&& visit) {
  const Rows9 rw = rows3_of(K, T.skey[k], T.cstart);
  const size_t st = (size_t)K.n;
  const int lane = threadIdx.x & 63;
  if (T.nbm[M3_OK * st + k]) {
    uint32_t nz = 0u;
#pragma unroll
    for (int q = 0; q < M3_OK; ++q) {
      const uint32_t m = T.nbm[(size_t)q * st + k];
      L.w[q][lane] = m;
      nz |= (m != 0u ? 1u : 0u) << q;
    }
#pragma unroll
    for (int q = 0; q < 9; ++q) L.t0[q][lane] = rw.t0[q];
    uint32_t m = 0u;
    int tb = 0;
    R uy = (R)0, uz = (R)0;
    const uint32_t mine = share_bits<NS>(s0);
    auto enter = [&]() {
      const int w = __builtin_ctz(nz);
      nz &= nz - 1u;
      m = L.w[w][lane] & mine;
      const int row = (w * 11) >> 5;   // w / 3 for w < 27
      const int ky = (row * 11) >> 5;  // row / 3 for row < 9
      uy = row_u3<R>(K, 1 - (row - 3 * ky));
      uz = row_u3<R>(K, 1 - ky);
      tb = L.t0[row][lane] + 32 * (w - 3 * row);
    };
    while (true) {
      next_word<NS>(m, nz, enter);
      if (m == 0u) break;
      const int l = tb + (int)__builtin_ctz(m);
      m &= m - 1u;
      visit(l, uy, uz);
    }
    return;
  }
  const auto pk = tape_pos3(T, k);
  const R cut2 = cutoff2<R>(K);
  for (int row = 0; row < 9; ++row) {
    const R uy = row_u3<R>(K, 1 - row % 3), uz = row_u3<R>(K, 1 - row / 3);
    for (int l = rw.t0[row]; l < rw.t1[row]; ++l) {
      if (l == k || (l - rw.t0[row]) % NS != s0) continue;
      R d0, d1, d2;
      const R r2 = delta3(pk, tape_pos3(T, l), K, uy, uz, d0, d1, d2);
      if (!(r2 < cut2)) continue;
      visit(l, uy, uz);
    }
  }
}

// objective: jpart[block] += dt sum_{obj} f, f = p^2 (kind 0) or u^2 (kind 1)
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_objective(St3<R> S, KParams K, int kind,
                                                      const uint8_t* __restrict__ objmask,
                                                      double* __restrict__ jpart) {
  __shared__ double sh[BLOCK];
  const int i = blockIdx.x * BLOCK + threadIdx.x;
  double v = 0.0;
  if (i < K.n && objmask[S.id[i]]) {
    const double f = kind == 1 ? S.u[i] : (double)S.p[i];
    v = K.dt * f * f;
  }
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = BLOCK / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) jpart[blockIdx.x] += sh[0];
}

// 1. corrector adjoint (time_integration.f:186-217)
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_adj_corrector(Tape3<R> T, KParams K, int its,
                                                          AdjState3 L, AdjScratch3<R> W,
                                                          const uint8_t* __restrict__ objmask,
                                                          int kind, double seed) {
  const int k = blockIdx.x * BLOCK + threadIdx.x;
  if (k >= K.n) return;
  const int id = T.id[k];
  const double dt = K.dt, h2 = K.dt / 2.0;
  double lax = L.cax[id], lay = L.cay[id], laz = L.caz[id];
  double ldrho = L.cdrho[id], ldu = L.cdu[id];
  double lavx = 0, lavy = 0, lavz = 0;
  double bvx = L.vx[id], bvy = L.vy[id], bvz = L.vz[id];
  double brho = L.rho[id], bu = L.u[id];
  if (is_rate(K, id)) {
    const double c = (its != 1) ? dt : h2;
    ldrho += c * L.rho[id];
    const double ub = (its != 1) ? T.u_min[k] : T.u[k];
    const double uu = ub + c * (double)T.du[k];
    bu = 0;
    if (!(uu < 0.0)) {
      bu = L.u[id];
      ldu += c * L.u[id];
    }
    if (id < K.np) {
      const double lvtx = L.vx[id] + dt * L.x[id];
      const double lvty = L.vy[id] + dt * L.y[id];
      const double lvtz = L.vz[id] + dt * L.z[id];
      bvx = lvtx;
      bvy = lvty;
      bvz = lvtz;
      lax += c * lvtx;
      lay += c * lvty;
      laz += c * lvtz;
      if (its != 1) {
        lavx = lvtx;
        lavy = lvty;
        lavz = lvtz;
      }
    }
  }
  L.bx[id] = L.x[id];
  L.by[id] = L.y[id];
  L.bz[id] = L.z[id];
  L.bvx[id] = bvx;
  L.bvy[id] = bvy;
  L.bvz[id] = bvz;
  L.brho[id] = brho;
  L.bu[id] = bu;
  W.ldrho[k] = is_rate(K, id) ? (R)ldrho : (R)0;
  {
    using R4 = typename V4<R>::type;
    const R Q = (R)1 / dens(K, T.rho[k]);
    const R4 v = T.v[k];
    W.rec[2 * (size_t)k] = tape_rec3(T, k);
    W.rec[2 * (size_t)k + 1] = R4{v.x, v.y, v.z, Q};
    W.frec[3 * (size_t)k] = R4{(R)lax, (R)lay, (R)laz, T.p[k] * Q};
    W.frec[3 * (size_t)k + 1] = R4{(R)lavx, (R)lavy, (R)lavz, T.psi[k]};
    W.frec[3 * (size_t)k + 2] = R4{(R)T.u[k], (R)ldu, (R)0, (R)0};
  }
  W.lp[k] = (objmask[id] && kind == 0) ? (R)(seed * 2.0 * dt * (double)T.p[k]) : (R)0;
  W.lus[k] = (objmask[id] && kind == 1) ? (R)(seed * 2.0 * dt * T.u[k]) : (R)0;
}

// 2. force-pass adjoint, gathered: particle k (as i) against every
//    neighbour l (as j); accumulates k's own input adjoints.  One wavefront
//    per workgroup; a neighbour is two records (five vectors) instead of
//    thirteen scattered loads, and the pair divides by reciprocals.
//    Bound by VALU issue and the records' latency.  Measured: FP32, 2.2M
//    particles 2130 -> 1233 us; FP64, 24,874 particles 206 -> 78 us.  Contiguous
//    shares per XCD: 1384 -> 1233 us.
template <typename R, bool AV, bool AH, bool XS, int NS>
__global__ __launch_bounds__(64 * NS) void k3_adj_force(Tape3<R> T, KParams K, AdjScratch3<R> W,
                                                   double* __restrict__ alpha_part) {
  __shared__ WalkLds3 L;
  __shared__ R part[NS > 1 ? (NS - 1) * 10 : 1][64];
  __shared__ double lals[NS];
  const int lane = threadIdx.x & 63, s0 = wave_of<NS>();
  double lal = 0.0;
  const int kb = xcd_block();
  const int k = kb * 64 + lane;
  R lr_acc[3] = {0, 0, 0}, lv_acc[3] = {0, 0, 0};
  R lQ = 0, lA = 0, lpsi = 0, lu = 0;
  if (k < K.n) {
    using R4 = typename V4<R>::type;
    const R m = (R)K.mass, h = (R)K.h, invh = (R)K.invh, C1 = (R)K.C1;
    const auto pk = pos_of_rec(W.rec[2 * (size_t)k]);
    const R4 vk = W.rec[2 * (size_t)k + 1];
    const R4 ak = W.frec[3 * (size_t)k], xk = W.frec[3 * (size_t)k + 1],
             uk = W.frec[3 * (size_t)k + 2];
    const R Qk = vk.w, Ak = ak.w, psik = xk.w, lduk = uk.y;
    const R alc0 = (R)(K.av_alpha * K.c0), be = (R)K.av_beta, c0 = (R)K.c0;
    const R ave2 = (R)K.av_e2, ahe2 = (R)K.ah_e2;
    const R em = (R)(K.xsph_eps * K.mass), wn = (R)K.wnorm;
    const R iq2 = (R)(0.5 / (K.h * K.h)), c3 = (R)(3.0 * K.C1);
    const bool pa0 = K.pa_sph == 0, se = K.same_e2 != 0;
    for_tape_neighbours3<NS, R>(T, K, s0, k, L, [&](int l, R uy, R uz) {
      const R4* o = W.rec + ((unsigned)l << 1);
      const R4* f = W.frec + (((unsigned)l << 1) + (unsigned)l);
      const auto pl = pos_of_rec(o[0]);
      const R4 vl = o[1], al = f[0], xl = f[1], ul = f[2];
      R r[3];
      const R r2 = delta3(pk, pl, K, uy, uz, r[0], r[1], r[2]);
      const R q = fsqrt(r2) * invh;
      const R t = q - (R)2;
      const R t2 = t * t;
      const R F = C1 * (t2 * t);
      const R dv[3] = {vk.x - vl.x, vk.y - vl.y, vk.z - vl.z};
      const R vr = dv[0] * r[0] + dv[1] * r[1] + dv[2] * r[2];
      const R Ql = vl.w, Al = al.w;
      const R is = rcp_n(Qk + Ql);
      const R g2 = (R)2 * Ql * is;  // dM/dQk = g2 Ql/(Qk + Ql)
      const R M = Qk * g2;
      R Kc = pa0 ? (Ak * Ql + Al * Qk) : (Ak * Qk + Al * Ql);
      const R mF = m * F;
      const R Da[3] = {ak.x - al.x, ak.y - al.y, ak.z - al.z};
      const R sig = lduk + ul.y;
      const R lG = -(Da[0] * r[0] + Da[1] * r[1] + Da[2] * r[2]) + (R)0.5 * sig * vr;
      const R lK = lG * mF;
      R lM = 0, lr2 = 0, lW = 0, lvr = 0;
      R einv = 0;
      if (AV) {
        einv = rcp_n(r2 + ave2);
        const bool on = vr < (R)0;
        const R phi = on ? h * vr * einv : (R)0;  // 0: every term below is 0
        const R pc = be * phi - alc0;
        Kc += pc * phi * M;
        lM += lK * pc * phi;
        lal += (double)(lK * (-c0 * phi * M));
        const R lphi = on ? lK * (be * phi + pc) * M : (R)0;
        lvr += lphi * h * einv;
        lr2 -= lphi * phi * einv;
      }
      const R G = mF * Kc;
      lvr += (R)0.5 * sig * G;
      R lF = lG * m * Kc;
      if (pa0) {
        lA += lK * Ql;
        lQ += lK * Al;
      } else {
        lA += lK * Qk;
        lQ += lK * Ak;
      }
      if (AH) {
        const R eh = (AV && se) ? einv : rcp_n(r2 + ahe2);
        const R dl = lduk - ul.y, ps = psik + xl.w;
        const R re = r2 * eh;
        const R mMe = m * M * re;        // H = mMe ps F
        const R lH = dl * (uk.x - ul.x);
        const R lHp = lH * ps;
        lu += dl * ps * (mMe * F);
        lpsi += lH * (mMe * F);
        lF += lHp * mMe;
        lr2 += lHp * (mF * M) * ahe2 * eh * eh;
        lM += lHp * mF * re;
      }
      R ldv[3] = {lvr * r[0], lvr * r[1], lvr * r[2]};
      if (XS) {
        const R s = (R)1 - (R)0.5 * q;
        const R s2 = s * s;
        const R Wv = wn * (s2 * s2) * ((R)1 + (R)2 * q);
        const R Dv[3] = {xk.x - xl.x, xk.y - xl.y, xk.z - xl.z};
        const R lw = -em * (Dv[0] * dv[0] + Dv[1] * dv[1] + Dv[2] * dv[2]);
        const R w = em * M * Wv;
        for (int c = 0; c < 3; ++c) ldv[c] -= w * Dv[c];
        lM += lw * Wv;
        lW = lw * M * wn * (s2 * s) * ((R)-5 * q);
      }
      lQ += lM * g2 * Ql * is;
      const R lq = lF * c3 * t2 + lW;
      lr2 += lq * iq2 * rcp_n(q);
      const R r22 = (R)2 * lr2;
      for (int c = 0; c < 3; ++c) {
        lr_acc[c] += lvr * dv[c] + r22 * r[c] - G * Da[c];
        lv_acc[c] += ldv[c];
      }
    });
  }
  share_sum<NS, 10>(
      part, s0, lane,
      [&](R* v) {
        for (int c = 0; c < 3; ++c) v[c] = lr_acc[c], v[3 + c] = lv_acc[c];
        v[6] = lQ, v[7] = lA, v[8] = lpsi, v[9] = lu;
      },
      [&](const R* v) {
        for (int c = 0; c < 3; ++c) lr_acc[c] += v[c], lv_acc[c] += v[3 + c];
        lQ += v[6], lA += v[7], lpsi += v[8], lu += v[9];
      });
  if (k < K.n && s0 == 0) {
    W.lx[k] = lr_acc[0];
    W.ly[k] = lr_acc[1];
    W.lz[k] = lr_acc[2];
    W.lvx[k] = lv_acc[0];
    W.lvy[k] = lv_acc[1];
    W.lvz[k] = lv_acc[2];
    W.lQ[k] = lQ;
    W.lA[k] = lA;
    W.lpsi[k] = lpsi;
    W.lu[k] = lu + W.lus[k];
  }
  // each pair is visited from both ends: half of its alpha derivative each
  lal *= 0.5;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) lal += __shfl_down(lal, d, 64);
  if constexpr (NS > 1) {
    if (lane == 0) lals[s0] = lal;
    __syncthreads();
    lal = 0.0;
    for (int q = 0; q < NS; ++q) lal += lals[q];
  }
  if (threadIdx.x == 0) alpha_part[kb] += lal;
}

// 3. EOS and art_heat coefficient adjoint (per particle)
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_adj_eos(Tape3<R> T, KParams K, AdjScratch3<R> W) {
  const int k = blockIdx.x * BLOCK + threadIdx.x;
  if (k >= K.n) return;
  const R rho = dens(K, T.rho[k]);
  const R Q = (R)1 / rho;
  const R lp = W.lp[k] + W.lA[k] * Q;
  R lrhoe = -Q * Q * (W.lQ[k] + W.lA[k] * T.p[k]);
  const R dv = T.divv[k];
  const R dpsi = (dv < (R)0) ? (R)(-2.0 * K.g2h2) : (R)0;
  const R ldv = W.lpsi[k] * dpsi;
  W.rec[2 * (size_t)k + 1].w = W.ldrho[k] - ldv / rho;  // lt = ldrho - lS
  lrhoe += -ldv * dv / rho;
  R lrhoh = 0;
  if (is_rate(K, T.id[k]) && !(T.flag[k] & 2u)) {
    if (K.eos == 1) {
      lrhoh = lrhoe + lp * (R)K.lin_c2;
    } else {
      const R t = rho / (R)K.rho0;
      const R t2 = t * t;
      lrhoh = lrhoe + lp * (R)(7.0 * K.B / K.rho0) * (t2 * t2 * t2);
    }
  }
  W.lrhoh[k] = lrhoh;
}

// 4. density adjoint, gathered; adds to the position / velocity adjoints
//    (FP32, 2.2M particles 726 -> 538 us; FP64, 24,874 particles 73 -> 45 us)
template <typename R, int NS>
__global__ __launch_bounds__(64 * NS) void k3_adj_density(Tape3<R> T, KParams K,
                                                          AdjScratch3<R> W) {
  __shared__ WalkLds3 L;
  __shared__ R part[NS > 1 ? (NS - 1) * 6 : 1][64];
  const int lane = threadIdx.x & 63, s0 = wave_of<NS>();
  const int k0 = xcd_block() * 64 + lane;
  const bool valid = k0 < K.n;
  const int k = valid ? k0 : K.n - 1;
  using R4 = typename V4<R>::type;
  const R m = (R)K.mass, invh = (R)K.invh, C1 = (R)K.C1;
  const R c3 = (R)(1.5 * K.C1 / (K.h * K.h)) * m;  // m 3 C1 / (2 h^2)
  const auto pk = pos_of_rec(W.rec[2 * (size_t)k]);
  const R4 vk = W.rec[2 * (size_t)k + 1];
  R lr[3] = {0, 0, 0}, lv[3] = {0, 0, 0};
  for_tape_neighbours3<NS, R>(T, K, s0, k, L, [&](int l, R uy, R uz) {
    const R4* o = W.rec + ((unsigned)l << 1);
    const auto pl = pos_of_rec(o[0]);
    const R4 vl = o[1];
    R r[3];
    const R r2 = delta3(pk, pl, K, uy, uz, r[0], r[1], r[2]);
    const R lt = vk.w + vl.w;
    const R q = fsqrt(r2) * invh;
    const R t = q - (R)2;
    const R t2 = t * t;
    const R dv[3] = {vk.x - vl.x, vk.y - vl.y, vk.z - vl.z};
    const R vr = dv[0] * r[0] + dv[1] * r[1] + dv[2] * r[2];
    const R lvr = lt * m * (C1 * (t2 * t));
    const R r22 = (R)2 * (lt * vr * c3 * t2) * rcp_n(q);
    for (int c = 0; c < 3; ++c) {
      lr[c] += lvr * dv[c] + r22 * r[c];
      lv[c] += lvr * r[c];
    }
  });
  share_sum<NS, 6>(
      part, s0, lane,
      [&](R* v) {
        for (int c = 0; c < 3; ++c) v[c] = lr[c], v[3 + c] = lv[c];
      },
      [&](const R* v) {
        for (int c = 0; c < 3; ++c) lr[c] += v[c], lv[c] += v[3 + c];
      });
  if (!valid || s0 != 0) return;
  W.lx[k] += lr[0];
  W.ly[k] += lr[1];
  W.lz[k] += lr[2];
  W.lvx[k] += lv[0];
  W.lvy[k] += lv[1];
  W.lvz[k] += lv[2];
}

// 5. predictor adjoint (time_integration.f:136-154)
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_adj_predictor(Tape3<R> T, KParams K, int its,
                                                          AdjState3 L, AdjScratch3<R> W) {
  const int k = blockIdx.x * BLOCK + threadIdx.x;
  if (k >= K.n) return;
  const int id = T.id[k];
  const double h2 = K.dt / 2.0;
  const double wlvx = W.lvx[k], wlvy = W.lvy[k], wlvz = W.lvz[k];
  const double wlrho = W.lrhoh[k], wlu = W.lu[k];
  L.bx[id] += (double)W.lx[k];
  L.by[id] += (double)W.ly[k];
  L.bz[id] += (double)W.lz[k];
  L.bvx[id] += wlvx;
  L.bvy[id] += wlvy;
  L.bvz[id] += wlvz;
  L.brho[id] += wlrho;
  double cax = 0, cay = 0, caz = 0, cdrho = 0, cdu = 0;
  if (its != 1 && is_rate(K, id)) {
    cdrho = h2 * wlrho;
    if (!(T.flag[k] & 1u)) {
      L.bu[id] += wlu;
      cdu = h2 * wlu;
    }
    if (id < K.np) {
      cax = h2 * wlvx;
      cay = h2 * wlvy;
      caz = h2 * wlvz;
    }
  } else {
    L.bu[id] += wlu;
  }
  L.cax[id] = cax;
  L.cay[id] = cay;
  L.caz[id] = caz;
  L.cdrho[id] = cdrho;
  L.cdu[id] = cdu;
}

}  // namespace arm
