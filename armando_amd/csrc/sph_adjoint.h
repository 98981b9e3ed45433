// sph_adjoint.h -- discrete adjoint of the step (reverse mode), for the FP64
// plain form (R = double) and the FP32 chosen form (R = float: pair
// arithmetic in FP32 on the cell + offset positions, as the forward; the
// adjoint of the state is accumulated in FP64 like the forward's position
// and energy accumulators).
//
// Differentiates the step exactly as the forward kernels compute it:
//   density   drho_i = sum_j m F vr,  S_i = -sum_j m F vr (divv_i = S_i/rho_i)
//   EOS       p = Tait(rho) or c0^2 rho + p0, clamp p < pmin -> p = 0, rho = rho0
//   psi_i = g1 h c0 + g2 h^2 (|divv_i| - divv_i),  Q = 1/rho,  A = p/rho
//   force     G = m F (A_i Q_j + A_j Q_i + Pi),  a_i = -sum G r + g,
//             du_i = sum G vr/2 + H (u_i - u_j),  av_i = -sum eps m M W dv
//   leapfrog  time_integration.f:136-217 (predictor, corrector, v += av)
// with r = x_i - x_j, vr = (v_i - v_j).r, grad W = F r, M = 2QiQj/(Qi+Qj).
// The neighbour list and the branches (u < 0, p < pmin, vr < 0, |divv|) of
// every step are those of the forward step.
//
// Adjoint variables of the state live in id order (they survive the
// per-step reordering); per-step scratch lives in the step's sorted order.
// Pair terms are gathered per particle: a particle accumulates only the
// derivatives of its own inputs, each pair being visited from both ends, so
// no atomics are needed.  The objective is J = sum_steps dt sum_obj f,
// f = p^2 or u^2; the heat source (flag 64) adds dJ/d hs_q0 and the
// physical viscosity (flag 32: shear tensor, viscous force, tds/dt) dJ/d eta.
#pragma once

#include "sph_kernels.h"

namespace arm {

// one recorded step: the sorted state after the force pass (before the
// corrector), the keys and the cell ranges of that step
template <typename R> struct Tape {
  using R2 = typename V2<R>::type;
  int32_t* id;
  double2* xy;
  uint32_t* cxy;  // FP32 form: cell and in-cell offset of the pair arithmetic
  float2* off;
  R2* v;      // predicted (half-step) velocity
  R* rho;     // density after the EOS clamp (FP32 form: rho - rho0)
  double* u;  // predicted energy
  R* psi;
  R* divv;
  R* p;
  R* drho;
  R* du;
  R2* a;
  R2* av;
  R* rho_min;
  double* u_min;
  R2* v_min;
  uint8_t* flag;
  uint32_t* skey;
  int* cstart;
  R* tau;  // physical viscosity: (Txx, Tyy, Txy, tds) per particle, else null
  uint4* nbm;  // the density pass's neighbour masks (three rows + complete flag)
};

// adjoint variables in id order
struct AdjState {
  double *x, *y, *vx, *vy, *rho, *u;  // of the state after the step (in) ...
  double *bx, *by, *bvx, *bvy, *brho, *bu;  // ... and before it (out)
  double *cax, *cay, *cdrho, *cdu;  // of the rates carried into the next predictor
};

// What a pair of the reverse gathers reads of a particle, four vectors written
// by the corrector's adjoint: rec, two for both gathers, position, velocity,
// Q = 1/rho, A = p/rho; frec, two for the force's: the adjoints of a, av and
// du, psi and u (FP64 has a's adjoint in rec).  The EOS adjoint puts lt (the
// density pass's) in the place of Q.
template <typename R> struct Rec4;
template <> struct Rec4<float> { using type = float4; };
template <> struct Rec4<double> { using type = double4; };
template <typename R> struct AdjRec {
  R vx, vy, Q, A, lax, lay, lavx, lavy, psi, u, ldu;
};
struct PosC {  // FP32: the cell as floats, whose difference is exact
  float ox, oy, cx, cy;
};
__device__ __forceinline__ void delta(const PosC& a, const PosC& b, const KParams& K, float& dx,
                                      float& dy) {
  dx = (a.ox - b.ox) + (a.cx - b.cx) * K.cellf;
  dy = (a.oy - b.oy) + (a.cy - b.cy) * K.cellf;
}
__device__ __forceinline__ PosC rec_pos(const float4* r) { return {r[0].x, r[0].y, r[0].z, r[0].w}; }
__device__ __forceinline__ PosD rec_pos(const double4* r) { return {r[0].x, r[0].y}; }
// velocity and the word that is Q or lt
__device__ __forceinline__ void rec_vel(const float4* r, float& vx, float& vy, float& q) {
  const float4 b = r[1];
  vx = b.x, vy = b.y, q = b.z;
}
__device__ __forceinline__ void rec_vel(const double4* r, double& vx, double& vy, double& q) {
  vx = r[0].z, vy = r[0].w, q = r[1].x;
}
__device__ __forceinline__ float& rec_lt(float4* r) { return r[1].z; }
__device__ __forceinline__ double& rec_lt(double4* r) { return r[1].x; }
__device__ __forceinline__ AdjRec<float> rec_load(const float4* r, const float4* f) {
  const float4 b = r[1], c = f[0], d = f[1];
  return {b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w, d.x, d.y, d.z};
}
__device__ __forceinline__ AdjRec<double> rec_load(const double4* r, const double4* f) {
  const double4 a = r[0], b = r[1], c = f[0];
  return {a.z, a.w, b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w, f[1].x};
}
__device__ __forceinline__ void rec_store(float4* r, float4* f, const Tape<float>& T, int k,
                                          const AdjRec<float>& q) {
  const uint32_t c = T.cxy[k];
  const float2 o = T.off[k];
  r[0] = make_float4(o.x, o.y, (float)(c & 0xffffu), (float)(c >> 16));
  r[1] = make_float4(q.vx, q.vy, q.Q, q.A);
  f[0] = make_float4(q.lax, q.lay, q.lavx, q.lavy);
  f[1] = make_float4(q.psi, q.u, q.ldu, 0.f);
}
__device__ __forceinline__ void rec_store(double4* r, double4* f, const Tape<double>& T, int k,
                                          const AdjRec<double>& q) {
  const double2 x = T.xy[k];
  r[0] = double4{x.x, x.y, q.vx, q.vy};
  r[1] = double4{q.Q, q.A, q.lax, q.lay};
  f[0] = double4{q.lavx, q.lavy, q.psi, q.u};
  f[1] = double4{q.ldu, 0.0, 0.0, 0.0};
}

// per-step scratch in sorted order
template <typename R> struct AdjScratch {
  R *ldrho, *lp;
  R *lQ, *lA, *lpsi, *lrhoh, *lu, *lvx, *lvy, *lx, *ly;
  typename Rec4<R>::type *rec, *frec;  // per particle: two and two vectors of AdjRec
  R* lus;  // objective seed of the energy (ARM_OBJ_ENERGY)
  R *lTxx, *lTyy, *lTxy;  // physical viscosity: adjoint of the shear tensor
};

template <typename R>
__global__ __launch_bounds__(BLOCK) void k_tape(St<R> S, KParams K,
                                                const uint32_t* __restrict__ skey,
                                                const int* __restrict__ cstart,
                                                const uint4* __restrict__ nbm, Tape<R> T) {
  const int t = blockIdx.x * BLOCK + threadIdx.x;
  const int stride = gridDim.x * BLOCK;
  for (int c = t; c <= K.ncell; c += stride) T.cstart[c] = cstart[c];
  if (t >= K.n) return;
  T.id[t] = S.id[t];
  T.xy[t] = S.xy[t];
  if constexpr (sizeof(R) == 4) {
    T.cxy[t] = S.cxy[t];
    T.off[t] = S.off[t];
  }
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
  T.nbm[t] = nbm ? nbm[t] : make_uint4(0u, 0u, 0u, 0u);
  if (T.tau)
    for (int c = 0; c < 4; ++c) T.tau[4 * (size_t)t + c] = S.tau[4 * (size_t)t + c];
}

// objective: jpart[block] += dt sum_{obj} f over the block's particles,
// f = p^2 (kind 0) or u^2 (kind 1)
template <typename R>
__global__ __launch_bounds__(BLOCK) void k_objective(St<R> S, KParams K, int kind,
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

// 1. corrector adjoint (time_integration.f:186-217): state adjoints after
//    the step -> rate adjoints (sorted) and the direct part of the state
//    adjoints before the step (id order); the objective, scaled by the
//    incoming adjoint seed = dL/dJ, seeds lp.
template <typename R>
__global__ __launch_bounds__(BLOCK) void k_adj_corrector(Tape<R> T, KParams K, int its,
                                                         AdjState L, AdjScratch<R> W,
                                                         const uint8_t* __restrict__ objmask,
                                                         int kind, double seed) {
  const int k = blockIdx.x * BLOCK + threadIdx.x;
  if (k >= K.n) return;
  const int id = T.id[k];
  const double dt = K.dt, h2 = K.dt / 2.0;
  double lax = L.cax[id], lay = L.cay[id], ldrho = L.cdrho[id], ldu = L.cdu[id];
  double lavx = 0, lavy = 0;
  double bx = L.x[id], by = L.y[id], bvx = L.vx[id], bvy = L.vy[id];
  double brho = 0, bu = 0;
  if (!is_rate(K, id)) {
    brho = L.rho[id];
    bu = L.u[id];
  } else {
    const double c = (its != 1) ? dt : h2;
    brho = L.rho[id];
    ldrho += c * L.rho[id];
    const double ub = (its != 1) ? T.u_min[k] : T.u[k];  // its == 1: u is the state u
    const double uu = ub + c * (double)T.du[k];
    if (!(uu < 0.0)) {
      bu = L.u[id];
      ldu += c * L.u[id];
    }
    if (id < K.np) {
      const double lvtx = L.vx[id] + dt * L.x[id];
      const double lvty = L.vy[id] + dt * L.y[id];
      bvx = lvtx;
      bvy = lvty;
      lax += c * lvtx;
      lay += c * lvty;
      if (its != 1) {
        lavx = lvtx;
        lavy = lvty;
      }
    }
  }
  L.bx[id] = bx;
  L.by[id] = by;
  L.bvx[id] = bvx;
  L.bvy[id] = bvy;
  L.brho[id] = brho;
  L.bu[id] = bu;
  W.ldrho[k] = is_rate(K, id) ? (R)ldrho : (R)0;
  const R Q = (R)1 / dens(K, T.rho[k]);
  const auto v = T.v[k];
  rec_store(W.rec + 2 * (size_t)k, W.frec + 2 * (size_t)k, T, k,
            {v.x, v.y, Q, T.p[k] * Q, (R)lax, (R)lay, (R)lavx, (R)lavy, T.psi[k], (R)T.u[k],
             (R)ldu});
  W.lp[k] = (objmask[id] && kind == 0) ? (R)(seed * 2.0 * dt * (double)T.p[k]) : (R)0;
  W.lus[k] = (objmask[id] && kind == 1) ? (R)(seed * 2.0 * dt * T.u[k]) : (R)0;
}

template <typename R>
__device__ __forceinline__ void wendland_q(const KParams& K, R r2, R& q, R& F, R& Wv) {
  q = fsqrt(r2) * (R)K.invh;
  const R t = q - (R)2;
  F = (R)K.C1 * (t * t * t);
  const R s = (R)1 - (R)0.5 * q;
  Wv = (R)K.wnorm * (s * s) * (s * s) * ((R)1 + (R)2 * q);
}

template <typename R>
__device__ __forceinline__ Rows tape_rows(const KParams& K, const Tape<R>& T, int k) {
  return rows_of(K, T.skey[k], T.cstart);
}

// The neighbours l of particle k in the forward gathers' order (rows bottom
// to top, ascending position), visit(l, rx, ry, r2): from the forward's
// masks when they are complete (bit b of row r = candidate t0_r + b, walked
// in one loop over the three rows), else by testing every candidate again.
// Wavefront s0 of NS visits its share of them (share_bits).
template <int NS, typename R, typename Visit>
__device__ __forceinline__ void for_tape_neighbours(const KParams& K, const Tape<R>& T,
                                                    const typename Rec4<R>::type* rec, int s0,
                                                    int k, Visit&& visit) {
  const Rows rw = tape_rows(K, T, k);
  const uint4 nm = T.nbm[k];
  const auto pk = rec_pos(rec + 2 * (size_t)k);
  if (nm.w) {
    const uint32_t mine = share_bits<NS>(s0);
    uint32_t m0 = nm.x & mine, m1 = nm.y & mine, m2 = nm.z & mine;
    while (m0 | m1 | m2) {
      const bool s0 = m0 != 0u, s1 = !s0 && m1 != 0u;
      const uint32_t m = s0 ? m0 : (s1 ? m1 : m2);
      const int l = (s0 ? rw.t0[0] : (s1 ? rw.t0[1] : rw.t0[2])) + (int)__builtin_ctz(m);
      const uint32_t rest = m & (m - 1u);
      m0 = s0 ? rest : m0;
      m1 = s1 ? rest : m1;
      m2 = (s0 || s1) ? m2 : rest;
      R rx, ry;
      delta(pk, rec_pos(rec + ((unsigned)l << 1)), K, rx, ry);
      visit(l, rx, ry, rx * rx + ry * ry);
    }
    return;
  }
  const R cut2 = cutoff2<R>(K);
  for (int r = 0; r < 3; ++r)
    for (int l = rw.t0[r]; l < rw.t1[r]; ++l) {
      if (l == k || (l - rw.t0[r]) % NS != s0) continue;
      R rx, ry;
      delta(pk, rec_pos(rec + ((unsigned)l << 1)), K, rx, ry);
      const R r2 = rx * rx + ry * ry;
      if (!(r2 < cut2)) continue;
      visit(l, rx, ry, r2);
    }
}

// The sum over the 64 lanes of the workgroup's particles, in lane 0.
__device__ __forceinline__ double lane_sum(double v) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d, 64);
  return v;
}

// 2. force-pass adjoint, gathered: particle k (as i) against every
//    neighbour l (as j); accumulates k's own input adjoints.  64 particles a
//    workgroup, NS wavefronts (share_adj2 on the host); a neighbour is four
//    vectors of two records instead of twelve loads from as many arrays, and
//    the pair divides by reciprocals.  Bound by the records' latency.
//    Measured, FP32, 115,416 particles 28.1 -> 19.6 us (density adjoint 10.9 ->
//    9.9); the corrector's adjoint pays 3 us for the records.
template <typename R, bool AV, bool AH, bool XS, bool VI, int NS>
__global__ __launch_bounds__(64 * NS) void k_adj_force(Tape<R> T, KParams K, AdjScratch<R> W,
                                                       double* __restrict__ alpha_part,
                                                       double* __restrict__ q0_part,
                                                       double* __restrict__ eta_part) {
  constexpr int NW = VI ? 11 : 8;
  __shared__ R part[NS > 1 ? (NS - 1) * NW : 1][64];
  __shared__ double lals[NS];
  const int lane = threadIdx.x & 63, s0 = wave_of<NS>();
  // one L2 per share of the tape; the partials stay indexed by that share
  const int kb = xcd_block();
  const int k0 = kb * 64 + lane;
  const bool valid = k0 < K.n;
  const int k = valid ? k0 : K.n - 1;
  double lq0 = 0.0, lal = 0.0, leta = 0.0;
  const R m = (R)K.mass, h = (R)K.h, invh = (R)K.invh, C1 = (R)K.C1;
  const AdjRec<R> o = rec_load(W.rec + 2 * (size_t)k, W.frec + 2 * (size_t)k);
  const R Qk = o.Q, Ak = o.A;
  const R alc0 = (R)(K.av_alpha * K.c0), be = (R)K.av_beta, c0 = (R)K.c0;
  const R ave2 = (R)K.av_e2, ahe2 = (R)K.ah_e2;
  const R em = (R)(K.xsph_eps * K.mass), wn = (R)K.wnorm;
  const R iq2 = (R)(0.5 / (K.h * K.h)), c3 = (R)(3.0 * K.C1);
  const bool pa0 = K.pa_sph == 0, se = K.same_e2 != 0;
  R lx = 0, ly = 0, lvx = 0, lvy = 0, lQ = 0, lA = 0, lpsi = 0, lu = 0;
  // physical viscosity: W = c T, c = eta (pa_sph 0) or eta Q^2 (pa_sph 1)
  R Tk[3] = {0, 0, 0}, ck = 0, lWk[3] = {0, 0, 0};
  if (VI) {
    const R* tk = T.tau + 4 * (size_t)k;
    Tk[0] = tk[0];
    Tk[1] = tk[1];
    Tk[2] = tk[2];
    ck = visc_c(K, Qk);
  }
  if (valid)
    for_tape_neighbours<NS>(K, T, W.rec, s0, k, [&](int l, R rx, R ry, R r2) {
      const AdjRec<R> j = rec_load(W.rec + ((unsigned)l << 1), W.frec + ((unsigned)l << 1));
      const R q = fsqrt(r2) * invh;
      const R t = q - (R)2;
      const R t2 = t * t;
      const R F = C1 * (t2 * t);
      const R dvx = o.vx - j.vx, dvy = o.vy - j.vy;
      const R vr = dvx * rx + dvy * ry;
      const R Ql = j.Q, Al = j.A;
      const R is = rcp_n(Qk + Ql);
      const R g2 = (R)2 * Ql * is;  // dM/dQk = g2 Ql/(Qk + Ql)
      const R M = Qk * g2;
      R Kc = pa0 ? (Ak * Ql + Al * Qk) : (Ak * Qk + Al * Ql);
      const R mF = m * F;
      const R Dax = o.lax - j.lax, Day = o.lay - j.lay;
      const R sig = o.ldu + j.ldu;
      const R lG = -(Dax * rx + Day * ry) + (R)0.5 * sig * vr;
      const R lK = lG * mF;
      R lM = 0, lr2 = 0, lW = 0, lvr = 0, einv = 0;
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
      R lrx = -G * Dax, lry = -G * Day;
      if (pa0) {
        lA += lK * Ql;
        lQ += lK * Al;
      } else {
        lA += lK * Qk;
        lQ += lK * Ak;
      }
      if (AH) {
        const R eh = (AV && se) ? einv : rcp_n(r2 + ahe2);
        const R dl = o.ldu - j.ldu, ps = o.psi + j.psi;
        const R re = r2 * eh;
        const R mMe = m * M * re;  // H = mMe ps F
        const R lH = dl * (o.u - j.u);
        const R lHp = lH * ps;
        lu += dl * ps * (mMe * F);
        lpsi += lH * (mMe * F);
        lF += lHp * mMe;
        lr2 += lHp * (mF * M) * ahe2 * eh * eh;
        lM += lHp * mF * re;
      }
      R ldvx = lvr * rx, ldvy = lvr * ry;
      if (XS) {
        const R s = (R)1 - (R)0.5 * q;
        const R s2 = s * s;
        const R Wv = wn * (s2 * s2) * ((R)1 + (R)2 * q);
        const R Dvx = o.lavx - j.lavx, Dvy = o.lavy - j.lavy;
        const R lw = -em * (Dvx * dvx + Dvy * dvy);
        const R w = em * M * Wv;
        ldvx -= w * Dvx;
        ldvy -= w * Dvy;
        lM += lw * Wv;
        lW = lw * M * wn * (s2 * s) * ((R)-5 * q);
      }
      if (VI) {
        // a_k += m F S.r, S = (Q_k Q_l if pa_sph 0) (W_k + W_l); a_l gets -that
        const R* tl = T.tau + 4 * (size_t)l;
        const R cl = visc_c(K, Ql);
        R Sr[3] = {ck * Tk[0] + cl * tl[0], ck * Tk[1] + cl * tl[1], ck * Tk[2] + cl * tl[2]};
        const R qq = pa0 ? Qk * Ql : (R)1;
        const R Sx = qq * Sr[0], Sy = qq * Sr[1], Sxy = qq * Sr[2];
        lF += m * (Dax * (Sx * rx + Sxy * ry) + Day * (Sxy * rx + Sy * ry));
        lrx += mF * (Dax * Sx + Day * Sxy);
        lry += mF * (Dax * Sxy + Day * Sy);
        const R lS[3] = {mF * Dax * rx, mF * Day * ry, mF * (Dax * ry + Day * rx)};
        if (pa0) lQ += Ql * (lS[0] * Sr[0] + lS[1] * Sr[1] + lS[2] * Sr[2]);
        for (int c = 0; c < 3; ++c) lWk[c] += qq * lS[c];
      }
      lQ += lM * g2 * Ql * is;
      const R lq = lF * c3 * t2 + lW;
      lr2 += lq * iq2 * rcp_n(q);
      const R r22 = (R)2 * lr2;
      lx += lrx + (lvr * dvx + r22 * rx);
      ly += lry + (lvr * dvy + r22 * ry);
      lvx += ldvx;
      lvy += ldvy;
    });
  share_sum<NS, NW>(
      part, s0, lane,
      [&](R* v) {
        v[0] = lx, v[1] = ly, v[2] = lvx, v[3] = lvy, v[4] = lQ, v[5] = lA, v[6] = lpsi, v[7] = lu;
        if (VI)
          for (int c = 0; c < 3; ++c) v[NW - 3 + c] = lWk[c];
      },
      [&](const R* v) {
        lx += v[0], ly += v[1], lvx += v[2], lvy += v[3], lQ += v[4], lA += v[5], lpsi += v[6],
            lu += v[7];
        if (VI)
          for (int c = 0; c < 3; ++c) lWk[c] += v[NW - 3 + c];
      });
  if (valid && s0 == 0) {
    if (VI) {
      // W_k = c_k T_k and tds_k = eta/2 Q_k (Txx^2 + Tyy^2 + 2 Txy^2), added to du_k
      const R eta = (R)K.eta;
      const R tw = Tk[0] * lWk[0] + Tk[1] * lWk[1] + Tk[2] * lWk[2];
      const R tt = Tk[0] * Tk[0] + Tk[1] * Tk[1] + (R)2 * Tk[2] * Tk[2];
      const R g = o.ldu * eta * Qk;
      W.lTxx[k] = ck * lWk[0] + g * Tk[0];
      W.lTyy[k] = ck * lWk[1] + g * Tk[1];
      W.lTxy[k] = ck * lWk[2] + g * (R)2 * Tk[2];
      if (K.pa_sph == 1) lQ += (R)2 * eta * Qk * tw;
      lQ += o.ldu * (R)0.5 * eta * tt;
      leta = (double)(K.pa_sph == 0 ? tw : Qk * Qk * tw) + (double)(o.ldu * (R)0.5 * Qk * tt);
    }
    // heat source du_k += q0 E_k Q_k, E = exp(-hs_k |x_k - c|^2)
    if ((K.flags & 64) && T.id[k] < K.np) {
      const double2 xk = T.xy[k];
      const double E = heat_shape(K, xk.x, xk.y);
      lq0 = (double)o.ldu * E * (double)Qk;
      lQ += o.ldu * (R)(K.hs_q0 * E);
      const double lE = (double)o.ldu * K.hs_q0 * (double)Qk * E * (-2.0 * K.hs_k);
      lx += (R)(lE * (xk.x - K.hs_x));
      ly += (R)(lE * (xk.y - K.hs_y));
    }
    W.lx[k] = lx;
    W.ly[k] = ly;
    W.lvx[k] = lvx;
    W.lvy[k] = lvy;
    W.lQ[k] = lQ;
    W.lA[k] = lA;
    W.lpsi[k] = lpsi;
    W.lu[k] = lu + W.lus[k];
  }
  // each pair is visited from both ends: half of its alpha derivative each
  lal = lane_sum(0.5 * lal);
  if constexpr (NS > 1) {
    if (lane == 0) lals[s0] = lal;
    __syncthreads();
    lal = 0.0;
    for (int q = 0; q < NS; ++q) lal += lals[q];
  }
  lq0 = lane_sum(lq0);
  if (VI) leta = lane_sum(leta);
  if (threadIdx.x == 0) {
    alpha_part[kb] += lal;
    q0_part[kb] += lq0;
    if (VI) eta_part[kb] += leta;
  }
}

// 2b. shear-tensor adjoint (physical viscosity), gathered.  The pair term
//     H(dv, dW), dv = v_l - v_k, dW = F r, r = x_k - x_l, enters
//     T_k with m Q_l and T_l with m Q_k (H is the same from both ends), so
//     particle k collects dv, r and Q_k derivatives of lambda_H =
//     m Q_l lT_k + m Q_k lT_l.
template <typename R>
__global__ __launch_bounds__(BLOCK) void k_adj_tensor(Tape<R> T, KParams K, AdjScratch<R> W) {
  const int k = xcd_block() * BLOCK + threadIdx.x;  // one L2 per share of the tape
  if (k >= K.n) return;
  using R2 = typename V2<R>::type;
  const R m = (R)K.mass, h = (R)K.h;
  const R2 vk = T.v[k];
  const R Qk = (R)1 / dens(K, T.rho[k]);
  const R Lk[3] = {W.lTxx[k], W.lTyy[k], W.lTxy[k]};
  const R two3 = (R)(2.0 / 3.0);
  R lx = 0, ly = 0, lvx = 0, lvy = 0, lQ = 0;
  for_tape_neighbours<1>(K, T, W.rec, 0, k, [&](int l, R rx, R ry, R r2) {
    R q, F, Wv;
    wendland_q(K, r2, q, F, Wv);
    const R2 vl = T.v[l];
    const R dvx = vl.x - vk.x, dvy = vl.y - vk.y;
    const R dWx = F * rx, dWy = F * ry;
    const R a = dvx * dWx, b = dvy * dWy;
    const R H[3] = {two3 * ((R)2 * a - b), two3 * ((R)2 * b - a), dvx * dWy + dvy * dWx};
    const R Ql = (R)1 / dens(K, T.rho[l]);
    const R Ll[3] = {W.lTxx[l], W.lTyy[l], W.lTxy[l]};
    R lH[3];
    for (int c = 0; c < 3; ++c) lH[c] = m * Ql * Lk[c] + m * Qk * Ll[c];
    lQ += m * (H[0] * Ll[0] + H[1] * Ll[1] + H[2] * Ll[2]);
    const R la = two3 * ((R)2 * lH[0] - lH[1]);
    const R lb = two3 * ((R)2 * lH[1] - lH[0]);
    const R ldvx = la * dWx + lH[2] * dWy, ldvy = lb * dWy + lH[2] * dWx;
    const R ldWx = la * dvx + lH[2] * dvy, ldWy = lb * dvy + lH[2] * dvx;
    lvx -= ldvx;
    lvy -= ldvy;
    const R lF = ldWx * rx + ldWy * ry;
    const R lr2 = lF * (R)3 * (R)K.C1 * (q - (R)2) * (q - (R)2) / ((R)2 * h * h * q);
    lx += F * ldWx + (R)2 * lr2 * rx;
    ly += F * ldWy + (R)2 * lr2 * ry;
  });
  W.lx[k] += lx;
  W.ly[k] += ly;
  W.lvx[k] += lvx;
  W.lvy[k] += lvy;
  W.lQ[k] += lQ;
}

// 3. EOS and art_heat coefficient adjoint (per particle)
template <typename R>
__global__ __launch_bounds__(BLOCK) void k_adj_eos(Tape<R> T, KParams K, AdjScratch<R> W) {
  const int k = blockIdx.x * BLOCK + threadIdx.x;
  if (k >= K.n) return;
  const R rho = dens(K, T.rho[k]);
  const R Q = (R)1 / rho;
  R lp = W.lp[k] + W.lA[k] * Q;
  R lrhoe = -Q * Q * (W.lQ[k] + W.lA[k] * T.p[k]);
  const R dv = T.divv[k];  // S / rho
  const R dpsi = (dv < (R)0) ? (R)(-2.0 * K.g2h2) : (R)0;
  const R ldv = W.lpsi[k] * dpsi;
  rec_lt(W.rec + 2 * (size_t)k) = W.ldrho[k] - ldv / rho;
  lrhoe += -ldv * dv / rho;
  R lrhoh = 0;
  if (is_rate(K, T.id[k]) && !(T.flag[k] & 2u)) {
    if (K.eos == 1) {
      // linear: dp/drho = c0^2
      lrhoh = lrhoe + lp * (R)K.lin_c2;
    } else {
      // Tait: dp/drho = 7 B / rho0 (rho / rho0)^6
      const R t = rho / (R)K.rho0;
      const R t2 = t * t;
      lrhoh = lrhoe + lp * (R)(7.0 * K.B / K.rho0) * (t2 * t2 * t2);
    }
  }
  W.lrhoh[k] = lrhoh;
}

// 4. density adjoint, gathered; adds to the position / velocity adjoints
template <typename R, int NS>
__global__ __launch_bounds__(64 * NS) void k_adj_density(Tape<R> T, KParams K, AdjScratch<R> W) {
  __shared__ R part[NS > 1 ? (NS - 1) * 4 : 1][64];
  const int lane = threadIdx.x & 63, s0 = wave_of<NS>();
  const int k0 = xcd_block() * 64 + lane;  // one L2 per share of the tape
  const bool valid = k0 < K.n;
  const int k = valid ? k0 : K.n - 1;
  const R m = (R)K.mass, invh = (R)K.invh, C1 = (R)K.C1;
  const R c3 = (R)(1.5 * K.C1 / (K.h * K.h)) * m;  // m 3 C1 / (2 h^2)
  R vkx, vky, ltk;
  rec_vel(W.rec + 2 * (size_t)k, vkx, vky, ltk);
  R lx = 0, ly = 0, lvx = 0, lvy = 0;
  if (valid)
    for_tape_neighbours<NS>(K, T, W.rec, s0, k, [&](int l, R rx, R ry, R r2) {
      R vlx, vly, ltl;
      rec_vel(W.rec + ((unsigned)l << 1), vlx, vly, ltl);
      const R lt = ltk + ltl;
      const R q = fsqrt(r2) * invh;
      const R t = q - (R)2;
      const R t2 = t * t;
      const R dvx = vkx - vlx, dvy = vky - vly;
      const R vr = dvx * rx + dvy * ry;
      const R lvr = lt * m * (C1 * (t2 * t));
      const R r22 = (R)2 * (lt * vr * c3 * t2) * rcp_n(q);
      lx += lvr * dvx + r22 * rx;
      ly += lvr * dvy + r22 * ry;
      lvx += lvr * rx;
      lvy += lvr * ry;
    });
  share_sum<NS, 4>(
      part, s0, lane, [&](R* v) { v[0] = lx, v[1] = ly, v[2] = lvx, v[3] = lvy; },
      [&](const R* v) { lx += v[0], ly += v[1], lvx += v[2], lvy += v[3]; });
  if (!valid || s0 != 0) return;
  W.lx[k] += lx;
  W.ly[k] += ly;
  W.lvx[k] += lvx;
  W.lvy[k] += lvy;
}

// 5. predictor adjoint (time_integration.f:136-154): folds the rate-input
//    adjoints into the state adjoints before the step and into the carried
//    rate adjoints of the previous step
template <typename R>
__global__ __launch_bounds__(BLOCK) void k_adj_predictor(Tape<R> T, KParams K, int its,
                                                         AdjState L, AdjScratch<R> W) {
  const int k = blockIdx.x * BLOCK + threadIdx.x;
  if (k >= K.n) return;
  const int id = T.id[k];
  const double h2 = K.dt / 2.0;
  const double wlx = W.lx[k], wly = W.ly[k], wlvx = W.lvx[k], wlvy = W.lvy[k];
  const double wlrho = W.lrhoh[k], wlu = W.lu[k];
  L.bx[id] += wlx;
  L.by[id] += wly;
  L.bvx[id] += wlvx;
  L.bvy[id] += wlvy;
  L.brho[id] += wlrho;
  double cax = 0, cay = 0, cdrho = 0, cdu = 0;
  if (its != 1 && is_rate(K, id)) {
    cdrho = h2 * wlrho;
    if (!(T.flag[k] & 1u)) {
      L.bu[id] += wlu;
      cdu = h2 * wlu;
    }
    if (id < K.np) {
      cax = h2 * wlvx;
      cay = h2 * wlvy;
    }
  } else {
    L.bu[id] += wlu;
  }
  L.cax[id] = cax;
  L.cay[id] = cay;
  L.cdrho[id] = cdrho;
  L.cdu[id] = cdu;
}

}  // namespace arm
