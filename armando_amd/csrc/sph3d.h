// sph3d.h -- the WCSPH step in three dimensions for gfx950.
//
// The same routines, arguments and pair arithmetic as the 2D kernels of
// sph_kernels.h, with
//   * the hash key ix + iy nx + iz nx ny (CERNsource/link_list.f:49-99 with
//     dim = 3 is the reference's 3D grid; Code/armando.cu:3190-3317 its 27-cell
//     GPU list);
//   * the 27 neighbour cells walked as nine rows (z outer, y inner) of three
//     consecutive x-cells: in (cell, id) order each row is one contiguous
//     range [cell_start[c-1], cell_start[c+2]) of the sorted arrays;
//   * Wendland C2 in 3D: KParams.wnorm = 21/(16 pi h^3), C1 = 5 wnorm/(8 h^2)
//     (grad W = C1 (q-2)^3 (x_i - x_j) as in 2D);
//   * FP32 form: an integer cell and an FP32 in-cell offset per axis; the
//     difference of two positions per axis is
//     (off_i - off_j) + (float)(c_i - c_j) * (float)cell.  A particle keeps
//     (off_x, off_y, off_z, (float)cx) in one float4 so that a neighbour's
//     position is one 16-byte load; the y and z cell differences are those
//     of the neighbour row being walked.
// Every lane writes only its own particle: no atomics, bitwise repeatable.
#pragma once

#include "sph_kernels.h"

namespace arm {

template <typename R> struct V4;
template <> struct V4<double> { using type = double4; };
template <> struct V4<float> { using type = float4; };

// Particle state in sorted (cell, id) order (fourth vector lanes unused).
// FP64 form: xyz holds the positions, rho the density.  FP32 form: xyz holds
// the FP64 position accumulators, pf the cell + offset that the pair
// arithmetic reads, rho the perturbation rho - rho0, uf a float copy of u.
template <typename R> struct St3 {
  using R4 = typename V4<R>::type;
  int32_t* id;
  double4* xyz;
  float4* pf;
  R4* v;
  R* rho;
  double* u;
  float* uf;
  R* p;
  R* psi;
  R* drho;
  R* du;
  R4* a;
  R4* av;
  R* divv;
  R* rho_min;
  double* u_min;
  R4* v_min;
  uint8_t* flag;
};

struct Pos3D {
  double x, y, z;
};
struct Pos3F {
  float cxf, ox, oy, oz;  // cell column as float, in-cell offsets
};

__device__ __forceinline__ Pos3D load_pos3(const St3<double>& S, int t) {
  const double4 q = S.xyz[t];
  return {q.x, q.y, q.z};
}
__device__ __forceinline__ Pos3F load_pos3(const St3<float>& S, int t) {
  const float4 q = S.pf[t];
  return {q.w, q.x, q.y, q.z};
}

// The cell-difference term (float)(c_i - c_j) * cell of one axis (FP32
// form); in the row walk the y and z differences are the constants of the
// row, 1 - k % 3 and 1 - k / 3 for row k.  Unused in the FP64 form.
template <typename R> __device__ __forceinline__ R row_u3(const KParams& K, int d) {
  return (R)((float)d * K.cellf);
}
template <> __device__ __forceinline__ double row_u3<double>(const KParams&, int) { return 0.0; }

// x_i - x_j and r^2 = (dx^2 + dy^2) + dz^2, rounded step by step (no
// contraction in this module), as the oracle restates them; uy, uz are the
// row's cell terms.  The x cell columns differ by at most one, exactly
// representable, so (cxf_i - cxf_j) is the integer difference.
__device__ __forceinline__ double delta3(const Pos3D& a, const Pos3D& b, const KParams&, double,
                                         double, double& dx, double& dy, double& dz) {
  dx = a.x - b.x;
  dy = a.y - b.y;
  dz = a.z - b.z;
  double r2 = dx * dx;
  r2 = r2 + dy * dy;
  return r2 + dz * dz;
}
__device__ __forceinline__ float delta3(const Pos3F& a, const Pos3F& b, const KParams& K,
                                        float uy, float uz, float& dx, float& dy, float& dz) {
  dx = (a.ox - b.ox) + (a.cxf - b.cxf) * K.cellf;
  dy = (a.oy - b.oy) + uy;
  dz = (a.oz - b.oz) + uz;
  float r2 = dx * dx;
  r2 = r2 + dy * dy;
  return r2 + dz * dz;
}

// ------------------------------------------------------------------------
// cell keys in FP64
// ------------------------------------------------------------------------
__device__ __forceinline__ uint32_t cell_of3(const KParams& K, double x, double y, double z,
                                             int& ix, int& iy, int& iz, bool& ok) {
  const double tx = (x - K.ox) / K.cell;
  const double ty = (y - K.oy) / K.cell;
  const double tz = (z - K.oz) / K.cell;
  ok = (tx >= 0.0) && (ty >= 0.0) && (tz >= 0.0) && (tx < (double)K.nx) &&
       (ty < (double)K.ny) && (tz < (double)K.nz);
  ix = ok ? (int)tx : 0;
  iy = ok ? (int)ty : 0;
  iz = ok ? (int)tz : 0;
  ix = ix < K.nx ? ix : K.nx - 1;
  iy = iy < K.ny ? iy : K.ny - 1;
  iz = iz < K.nz ? iz : K.nz - 1;
  return (uint32_t)ix + (uint32_t)K.nx * ((uint32_t)iy + (uint32_t)K.ny * (uint32_t)iz);
}

// FP32 form: cell + offset of an FP64 position.
__device__ __forceinline__ float4 split3(const KParams& K, double4 q) {
  int ix, iy, iz;
  bool ok;
  cell_of3(K, q.x, q.y, q.z, ix, iy, iz, ok);
  const double bx = K.ox + (double)ix * K.cell;
  const double by = K.oy + (double)iy * K.cell;
  const double bz = K.oz + (double)iz * K.cell;
  return make_float4((float)(q.x - bx), (float)(q.y - by), (float)(q.z - bz), (float)ix);
}

template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_keys(St3<R> S, KParams K, KeyOut ko,
                                                 int* __restrict__ err) {
  const int s = blockIdx.x * BLOCK + threadIdx.x;
  const bool valid = s < K.n;
  uint32_t key = 0;
  int id = 0;
  if (valid) {
    const double4 q = S.xyz[s];
    int ix, iy, iz;
    bool ok;
    key = cell_of3(K, q.x, q.y, q.z, ix, iy, iz, ok);
    if (!ok) {
      atomicAdd(err, 1);
      raise_halt(K);
    }
    id = S.id[s];
    if constexpr (sizeof(R) == 4) S.pf[s] = split3(K, q);
  }
  emit_key(ko, valid, s, id, key);
}

// Permute every field from A to B (per-routine link_list).
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_reorder_all(St3<R> A, St3<R> Bs, KParams K,
                                                        const uint32_t* __restrict__ skey,
                                                        Order ord,
                                                        int* __restrict__ cstart, int fill) {
  const int p = blockIdx.x * BLOCK + threadIdx.x;
  const bool valid = p < K.n;
  if (fill) fill_cell_start(skey, p, valid, K.n, K.ncell, cstart);
  if (!valid) return;
  const int s = (int)ord.slot[p];
  const int id = A.id[s];
  const int t = ord.place(skey, cstart, p, id);
  Bs.id[t] = id;
  Bs.xyz[t] = A.xyz[s];
  if constexpr (sizeof(R) == 4) Bs.pf[t] = A.pf[s];
  Bs.v[t] = A.v[s];
  Bs.rho[t] = A.rho[s];
  const double u = A.u[s];
  Bs.u[t] = u;
  if constexpr (sizeof(R) == 4) Bs.uf[t] = (float)u;  // a rollout leaves A.uf behind
  Bs.p[t] = A.p[s];
  Bs.psi[t] = A.psi[s];
  Bs.drho[t] = A.drho[s];
  Bs.du[t] = A.du[s];
  Bs.a[t] = A.a[s];
  Bs.av[t] = A.av[s];
  Bs.divv[t] = A.divv[s];
  Bs.rho_min[t] = A.rho_min[s];
  Bs.u_min[t] = A.u_min[s];
  Bs.v_min[t] = A.v_min[s];
  Bs.flag[t] = A.flag[s];
}

// Fused reorder + leapfrog predictor (time_integration.f:136-154).
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_reorder_pred(St3<R> A, St3<R> Bs, KParams K,
                                                         const uint32_t* __restrict__ skey,
                                                         Order ord,
                                                         int* __restrict__ cstart, int predict,
                                                         int fill) {
  if (halted(K)) return;
  using R4 = typename V4<R>::type;
  const int p = blockIdx.x * BLOCK + threadIdx.x;
  const bool valid = p < K.n;
  if (fill) fill_cell_start(skey, p, valid, K.n, K.ncell, cstart);
  if (!valid) return;
  const int s = (int)ord.slot[p];
  const int id = ord.ids ? (int)ord.ids[p] : A.id[s];
  // the fields before the rank: their loads overlap its own
  const double4 q = A.xyz[s];
  R4 v = A.v[s];
  R rho = A.rho[s];
  double u = A.u[s];
  R4 a{};
  R du = (R)0, drho = (R)0;
  if (predict) {
    a = A.a[s];
    du = A.du[s];
    drho = A.drho[s];
  }
  const int t = ord.place(skey, cstart, p, id);
  Bs.id[t] = id;
  Bs.xyz[t] = q;
  if constexpr (sizeof(R) == 4) Bs.pf[t] = split3(K, q);
  uint8_t fl = 0;
  if (predict) {
    const double hdt = K.dt / 2.0;
    if (is_rate(K, id)) {
      Bs.u_min[t] = u;
      u = u + hdt * (double)du;
      if (u < 0.0) {
        u = 0.0;
        fl = 1u;
      }
      if (K.density_method == 0) {
        Bs.rho_min[t] = rho;
        rho = rho + (R)hdt * drho;
      }
    }
    if (id < K.np) {
      Bs.v_min[t] = v;
      v.x = v.x + (R)hdt * a.x;
      v.y = v.y + (R)hdt * a.y;
      v.z = v.z + (R)hdt * a.z;
    }
  }
  Bs.v[t] = v;
  Bs.rho[t] = rho;
  Bs.u[t] = u;
  if constexpr (sizeof(R) == 4) Bs.uf[t] = (float)u;
  Bs.flag[t] = fl;
  if (!is_rate(K, id)) Bs.p[t] = A.p[s];
}

// ------------------------------------------------------------------------
// neighbour rows
// ------------------------------------------------------------------------
struct Rows9 {
  int t0[9], t1[9];
};

__device__ __forceinline__ Rows9 rows3_of(const KParams& K, uint32_t key,
                                          const int* __restrict__ cstart) {
  const int nxy = K.nx * K.ny;
  const int cz = (int)key / nxy;
  const int rem = (int)key - cz * nxy;
  const int cy = rem / K.nx;
  const int cx = rem - cy * K.nx;
  const int x0 = cx > 0 ? cx - 1 : 0;
  const int x1 = cx + 1 < K.nx ? cx + 1 : K.nx - 1;
  Rows9 r;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const int rz = cz - 1 + k / 3, ry = cy - 1 + k % 3;
    if (rz < 0 || rz >= K.nz || ry < 0 || ry >= K.ny) {
      r.t0[k] = 0;
      r.t1[k] = 0;
    } else {
      const int base = (rz * K.ny + ry) * K.nx;
      r.t0[k] = cstart[base + x0];
      r.t1[k] = cstart[base + x1 + 1];
    }
  }
  return r;
}

// ------------------------------------------------------------------------
// pair arithmetic (the 2D forms with a z component)
// ------------------------------------------------------------------------
// ok = false: no neighbour, the sums keep every word.
// The constants of the pair bodies are not folded in FP32 as in 2D: with the
// products m C1, -8 C1 m and wnorm eps m / 2 rounded once, the rates of an
// 83,630-particle tank were further from FP64 (rel. L2: drho 1.56e-7 instead of
// 1.27e-7, av 1.91e-7 instead of 1.63e-7), and the dam break's velocities after
// 125 steps 1.8e-7 off instead of 1.3e-7: the rounded factors m, C1, wnorm are
// together 5e-8 to 8e-8 low, which offsets the hardware square root (1.3e-8 low
// in the mean, entering (q - 2)^3 threefold and more), while the folded ones
// are within 1e-8.  It costs nothing at 2.2M particles (force 792 us, 794
// folded; density 648 and 647), and 43.7 us instead of 40.6 of the force at 83,630.
template <typename R, bool SUM>
__device__ __forceinline__ void dens3_pair(const KParams& K, R dx, R dy, R dz, R r2, R dvx,
                                           R dvy, R dvz, Acc<R>& sum, Acc<R>& rs, bool ok = true) {
  const R q = fsqrt(r2) * (R)K.invh;
  const R tq = q - (R)2;
  const R F = (R)K.C1 * (tq * tq * tq);
  const R vcc = fmr(dvz, F * dz, fmr(dvy, F * dy, dvx * (F * dx)));
  sum.add_if((R)K.mass * vcc, ok);
  if (SUM) {
    const R s = fmr((R)-0.5, q, (R)1);
    const R s2 = s * s;
    rs.add_if((R)K.mass * ((R)K.wnorm * (s2 * s2) * fmr((R)2, q, (R)1)), ok);
  }
}

// Neighbour masks recorded by the density pass for the force pass: for row k
// of particle i, bit b of word q (q < M3_WORDS) says whether the candidate at
// sorted position t0_k + 32 q + b is a neighbour, t0_k the first position of
// the row's three cells.  Structure of arrays: word k * M3_WORDS + q of
// sorted particle i at w[(k * M3_WORDS + q) * stride + i]; word M3_OK is 1
// when every row had at most 32 M3_WORDS candidates (complete masks).
constexpr int M3_WORDS = 3;
constexpr int M3_OK = 9 * M3_WORDS;
constexpr int M3_TOTAL = M3_OK + 1;

struct Mask3 {
  uint32_t* w;
  int stride;
  __device__ __forceinline__ void put(int q, int i, uint32_t m) const {
    w[(size_t)q * stride + i] = m;
  }
  __device__ __forceinline__ uint32_t get(int q, int i) const {
    return w[(size_t)q * stride + i];
  }
};

// Neighbour data of the force pass packed per particle into one record of
// three vectors, so that a neighbour's loads fall in one or two cache lines:
// the position record of the state (FP32: pf; FP64: xyz), (v, Q = 1/rho) and
// (A = p/rho, psi, u, 0), with q_and_a's arithmetic.  Written at the end of a
// density pass with the EOS in it, whose particles hold most of it already,
// or by k3_force_pack.
template <typename R> struct Pack3 {
  using R4 = typename V4<R>::type;
  R4* rec;  // 3 per particle
};

__device__ __forceinline__ float4 pos_rec3(const St3<float>& S, int i) { return S.pf[i]; }
__device__ __forceinline__ double4 pos_rec3(const St3<double>& S, int i) { return S.xyz[i]; }
template <typename R> __device__ __forceinline__ R u3_of(const St3<R>& S, int t) {
  if constexpr (sizeof(R) == 4) return S.uf[t]; else return (R)S.u[t];
}

template <typename R>
__device__ __forceinline__ void force3_record(const St3<R>& S, const KParams& K, const Pack3<R>& P,
                                              int i) {
  using R4 = typename V4<R>::type;
  R Q, A;
  q_and_a(K, S.rho[i], S.p[i], Q, A);
  const R4 v = S.v[i];
  R4* r = P.rec + 3 * (size_t)i;
  r[0] = pos_rec3(S, i);
  r[1] = R4{v.x, v.y, v.z, Q};
  r[2] = R4{A, S.psi[i], u3_of(S, i), (R)0};
}

// ---- neighbour pre-test on the matrix cores ---------------------------------
// A particle has about 490 candidates in its nine rows, of which 68 are
// neighbours, so the candidate test dominates a density pass that makes it
// per lane (92 VALU instructions and eight 16-byte loads per lane for eight
// candidates).  Squared distances are a contraction:
//   r^2 = |x_j|^2 - 2 x_j . x_i + |x_i|^2,
// so a wavefront computes them with v_mfma_f32_16x16x4_f32, 16 candidates by
// 16 of its particles at a time: A row j = (-2x, -2y, -2z, |x|^2)_j,
// B column i = (x, y, z, 1)_i, C = |x_i|^2 - bound, and the sign of each
// result is the test (one v_alignbit per 64 of them collects it).  Positions
// are FP32 and relative to the wavefront's first cell, and the bound
// (KParams::pre3f) covers their rounding and the cancellation, so every pair
// with r < 2h passes; the survivors (about one in a thousand too many) take
// the exact test in the pair walk.
//
// The wavefront's 64 consecutive particles form four tiles of 16; two tiles
// share a row's staged candidates (in LDS, one record each) but each tests its
// own union of candidates: the lanes 16 q .. 16 q + 15 of D hold rows 4q .. 4q+3,
// and row 4q + r of step s is candidate q 4 steps + 4 s + r, so that a lane
// collects 4 steps consecutive candidates of one particle in one word.  Two
// permlane32 and two permlane16 swaps then bring a particle's four words to
// its own lane, which cuts its window [t0, t1) out of them.
//
// Bound: VALU issue (7,500 instructions a wavefront, 70 % of the launch; the
// MFMAs are busy a tenth of it).  Measured, density pass: FP32, 2,236,171-
// particle dam break 807 -> 612 us against the per-lane pre-test; FP64 (which
// tested every candidate in FP64), 83,630-particle tank 245 -> 78 us.  A
// wavefront's 64 particles staging a row at once, with the next row's loads
// ahead, took more registers and came out no faster (616 and 95 us).
constexpr int P3_CAP = 160;   // staged records of two tiles in one row (16 bytes each)
constexpr int P3_TILE = 128;  // candidates of a tile in one row, at most 4 x 32
constexpr int P3_SPAN = 12;   // cells between the first and last particle of a sweep

using f32x4 = __attribute__((ext_vector_type(4))) float;

// A particle's position relative to the corner of cell (cx0, cy, cz), for a
// candidate in row k the row's own offset included.
struct Local3 {
  float x, y, z;
};
__device__ __forceinline__ Local3 local3(const KParams& K, float4 q, int cx0, int, int, int k) {
  return {__builtin_fmaf(q.w - (float)cx0, K.cellf, q.x), q.y - row_u3<float>(K, 1 - k % 3),
          q.z - row_u3<float>(K, 1 - k / 3)};
}
__device__ __forceinline__ Local3 local3(const KParams& K, double4 q, int cx0, int cy, int cz,
                                         int) {
  return {(float)(q.x - (K.ox + (double)cx0 * K.cell)),
          (float)(q.y - (K.oy + (double)cy * K.cell)),
          (float)(q.z - (K.oz + (double)cz * K.cell))};
}

// Whether a particle sorted into cell 0 lies in it or near it, so that local3 and
// pre3f hold.  One outside the grid does not (arm_link_list sorts it into cell 0
// and returns ARM_ERR_DOMAIN; the gathers still run for a caller that goes on):
// it takes the exact test of every candidate.
__device__ __forceinline__ bool local3_holds(const KParams& K, float4 q) {
  const float c = 2.f * K.cellf;
  return fabsf(q.x) <= c && fabsf(q.y) <= c && fabsf(q.z) <= c;
}
__device__ __forceinline__ bool local3_holds(const KParams& K, double4 q) {
  const double c = 2.0 * K.cell;
  return fabs(q.x - K.ox) <= c && fabs(q.y - K.oy) <= c && fabs(q.z - K.oz) <= c;
}

// The 96-bit window [d, d + len) of the four words p of ch bits each
// (ch a multiple of 4, at most 32; len <= 96).
__device__ __forceinline__ void window3(const uint32_t* p, int ch, int d, int len, uint32_t* m) {
  const uint64_t a = (uint64_t)p[0] | ((uint64_t)p[1] << ch);
  const uint64_t b = (uint64_t)p[2] | ((uint64_t)p[3] << ch);  // from bit 2 ch on
  uint64_t lo = a | ((b << ch) << ch);
  uint64_t hi = ch ? b >> (64 - 2 * ch) : 0ull;
  if (d >= 64) {
    lo = hi;
    hi = 0ull;
    d -= 64;
  }
  lo = (lo >> d) | ((hi << 1) << (63 - d));
  hi = hi >> d;
  lo &= len >= 64 ? ~0ull : (1ull << len) - 1ull;
  const int l2 = len - 64;
  m[0] = (uint32_t)lo;
  m[1] = (uint32_t)(lo >> 32);
  m[2] = l2 <= 0 ? 0u : (uint32_t)hi & (l2 >= 32 ? ~0u : (1u << l2) - 1u);
}

// Orders a wavefront's own LDS accesses (it needs no barrier: they execute in
// order; the compiler must keep them so).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sweeps that pretest3 makes of the lanes on.
__device__ __forceinline__ int sweeps3(bool on, int cx, int row) {
  int n = 0;
  for (uint64_t todo = __ballot(on); todo; ++n) {
    const int a = __builtin_ctzll(todo);
    const int row0 = __builtin_amdgcn_readlane(row, a), cx0 = __builtin_amdgcn_readlane(cx, a);
    todo &= ~__ballot(row == row0 && cx - cx0 <= P3_SPAN);
  }
  return n;
}

// pretest3 lane by lane: the exact test of a lane's own candidates, NB at a time (in
// FP64 two: eight double4 loads of which one is a candidate took 52 us instead of 42
// on the thinnest spray below).  For wavefronts whose particles lie in many cell rows
// and have few candidates: spray, thin sheets, narrow channels.  pretest3 makes a
// sweep of nine rows for every row and 13 cells of it that the wavefront touches, one
// after the other; here they run side by side.  Measured, density pass of 300,000
// particles, FP32 (FP64), us: a sweep adds 10 (12), a hundred candidates 20 (35),
// so that lanes take less below 10 + 50 (10 + 45) candidates a sweep, FEW3:
//   spray, 0.3 / 1 / 3 per cell   sweeps 212 / 108 / 81 (239 / 124 / 97)
//                                 lanes 31 / 39 / 63 (42 / 57 / 89)
//   sheets of 2 / 3 particles     sweeps 125 / 125 (154 / 159), lanes 71 / 101 (116 / 148)
// Dense fluid has 490 candidates and one to three sweeps.
constexpr int FEW3_MAX = 288;  // beyond it no count of sweeps is looked for
template <typename R> struct Few3;
template <> struct Few3<float> { static constexpr int base = 10, sweep = 50, batch = 4; };
template <> struct Few3<double> { static constexpr int base = 10, sweep = 45, batch = 2; };
template <int NS, typename R>
__device__ __forceinline__ void pretest3_lanes(const St3<R>& S, const KParams& K, int s0, int i,
                                               bool on, const Rows9& rw,
                                               int (*__restrict__ lt)[64],
                                               uint32_t (*__restrict__ lw)[64]) {
  constexpr int NB = Few3<R>::batch;
  const int lane = threadIdx.x & 63;
  const auto pi = load_pos3(S, i);
  const R cut2 = cutoff2<R>(K);
#pragma unroll
  for (int k = 0; k < 9; ++k) {  // the rows' bounds, for a loop that is not unrolled
    if (k % NS != s0) continue;
    lt[k][lane] = rw.t0[k];
    lw[3 * k][lane] = (uint32_t)rw.t1[k];
  }
  for (int k = s0; k < 9; k += NS) {
    const int ky = (k * 11) >> 5;  // k / 3 for k < 9
    const R uy = row_u3<R>(K, 1 - (k - 3 * ky)), uz = row_u3<R>(K, 1 - ky);
    const int t0 = lt[k][lane], t1 = on ? (int)lw[3 * k][lane] : t0;
#pragma unroll
    for (int q = 0; q < M3_WORDS; ++q) {
      const int c0 = t0 + 32 * q, end = min(c0 + 32, t1);
      uint32_t m = 0u;
      for (int c = c0; c < end; c += NB) {
        uint32_t bb = 0u;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int t = min(c + b, end - 1);
          R dx, dy, dz;
          const R r2 = delta3(pi, load_pos3(S, t), K, uy, uz, dx, dy, dz);
          bb |= (r2 < cut2 && c + b < end && t != i ? 1u : 0u) << b;
        }
        m |= bb << (c - c0);
      }
      if (on) lw[3 * k + q][lane] = m;
    }
  }
}

// Mask words lw[3k + q][lane] of the nine rows (wavefront s of S: rows k = s
// modulo S) of every lane with on set (rows of at most 96 candidates), the
// particle's own bit cleared.  Called by the whole wavefront.  cx, row = cy + cz ny: the lane's cell; rec: LDS for the
// records staged of a row, P3_CAP and P3_TILE + 16 more that may be read.
template <int NS, typename R>
__device__ __forceinline__ void pretest3(const St3<R>& S, const KParams& K, int s0, int i, bool on,
                                         int cx, int row, const Rows9& rw, float4* __restrict__ rec,
                                         uint32_t (*__restrict__ lw)[64]) {
  const int* t0 = rw.t0;
  const int* t1 = rw.t1;
  const int lane = threadIdx.x & 63;
  const auto own = pos_rec3(S, i);
  const int ar = (lane & 15) >> 2, ac = lane & 3, ak = lane >> 4;
  uint64_t todo = __ballot(on);
  int span = P3_SPAN;
  while (todo) {
    // the sweep: lanes of one cell row within span cells of the first (a gap
    // of empty cells ends it; its rows hold the candidates of what lies between)
    const int a = __builtin_ctzll(todo);
    const int row0 = __builtin_amdgcn_readlane(row, a), cx0 = __builtin_amdgcn_readlane(cx, a);
    const bool in = ((todo >> lane) & 1ull) && row == row0 && cx - cx0 <= span;
    const uint64_t im = __ballot(in);
    const int cz = row0 / K.ny, cy = row0 - cz * K.ny;
    int first[4], last[4];
#pragma unroll
    for (int T = 0; T < 4; ++T) {
      const uint32_t mt = (uint32_t)(im >> (16 * T)) & 0xffffu;
      first[T] = mt ? 16 * T + __builtin_ctz(mt) : a;
      last[T] = mt ? 16 * T + 31 - __builtin_clz(mt) : -1;
    }
    const Local3 me = local3(K, own, cx0, cy, cz, 4);
    const float c = __builtin_fmaf(me.x, me.x, __builtin_fmaf(me.y, me.y, me.z * me.z)) - K.pre3f;
    float B[4];
    f32x4 C[4];
#pragma unroll
    for (int T = 0; T < 4; ++T) {
      const int src = 16 * T + (lane & 15);
      const float bx = __shfl(me.x, src, 64), by = __shfl(me.y, src, 64),
                  bz = __shfl(me.z, src, 64), cc = __shfl(c, src, 64);
      B[T] = ak == 0 ? bx : (ak == 1 ? by : (ak == 2 ? bz : 1.f));
      C[T] = f32x4{cc, cc, cc, cc};
    }
    bool fits = true;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      if (k % NS != s0) continue;
      uint32_t p[4] = {0u, 0u, 0u, 0u};
      int u0 = 0, ch = 0;  // of the lane's tile: first candidate, candidates per word
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (last[2 * h] < 0 && last[2 * h + 1] < 0) continue;
        int at[2], most = 0, U0 = 0x7fffffff, U1 = 0;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int T = 2 * h + e;
          at[e] = 0;
          if (last[T] < 0) continue;
          at[e] = __builtin_amdgcn_readlane(t0[k], first[T]);
          const int end = __builtin_amdgcn_readlane(t1[k], last[T]);
          most = max(most, end - at[e]);
          U0 = min(U0, at[e]);
          U1 = max(U1, end);
        }
        fits = fits && U1 - U0 <= P3_CAP && most <= P3_TILE;
        if (!fits) break;
        const int steps = (most + 15) >> 4;
        const int UL = U1 - U0;
        for (int q = lane; q < UL; q += 64) {
          const Local3 r = local3(K, pos_rec3(S, U0 + q), cx0, cy, cz, k);
          rec[q] = make_float4(-2.f * r.x, -2.f * r.y, -2.f * r.z,
                               __builtin_fmaf(r.x, r.x, __builtin_fmaf(r.y, r.y, r.z * r.z)));
        }
        wave_sync();
        const float* ap[2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
          ap[e] = reinterpret_cast<const float*>(rec) +
                  4 * (max(at[e] - U0, 0) + 4 * (ar * steps + steps - 1) + ac) + ak;
        for (int s = 0; s < steps; ++s) {
          f32x4 d[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            d[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(*ap[e], B[2 * h + e], C[2 * h + e], 0, 0, 0);
            ap[e] -= 16;
          }
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int r = 3; r >= 0; --r)
              p[2 * h + e] =
                  __builtin_amdgcn_alignbit(p[2 * h + e], __float_as_uint(d[e][r]), 31);
        }
        wave_sync();
        if ((lane >> 5) == h) {
          u0 = (lane >> 4) & 1 ? at[1] : at[0];
          ch = 4 * steps;
        }
      }
      if (!fits) break;
      // word T of lane group q -> word q of lane group T
      auto s2 = __builtin_amdgcn_permlane32_swap(p[0], p[2], false, false);
      p[0] = s2[0], p[2] = s2[1];
      s2 = __builtin_amdgcn_permlane32_swap(p[1], p[3], false, false);
      p[1] = s2[0], p[3] = s2[1];
      s2 = __builtin_amdgcn_permlane16_swap(p[0], p[1], false, false);
      p[0] = s2[0], p[1] = s2[1];
      s2 = __builtin_amdgcn_permlane16_swap(p[2], p[3], false, false);
      p[2] = s2[0], p[3] = s2[1];
      if (in) {
        uint32_t m[3];
        window3(p, ch, t0[k] - u0, t1[k] - t0[k], m);
        if (k == 4) {
          const int sb = i - t0[4];
          const uint32_t bit = 1u << (sb & 31);
#pragma unroll
          for (int q = 0; q < 3; ++q) m[q] &= (sb >> 5) == q ? ~bit : ~0u;
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) lw[3 * k + q][lane] = m[q];
      }
    }
    if (fits) {
      todo &= ~im;
      span = P3_SPAN;
    } else {
      // a shorter sweep; one cell's own window (at most 96) always fits
      span = span > 2 ? 2 : 0;
    }
  }
}

// Density gather of a wavefront's 64 consecutive particles: the pre-test of
// all nine rows (pretest3) into 27 mask words per lane, then one loop over a
// lane's set bits in (row, word, bit) order, two at a time so that their
// loads are in flight together, each through the exact test and the pair
// sums (a wavefront runs for its longest lane's survivor count).  The words
// are kept in the lane's own LDS column, which the staged records use
// before.  A lane with a row of more than 96 candidates, or outside the grid, tests
// and sums its candidates one by one instead, in the same order.
template <typename R, bool SUM, bool EOS, int NS>
__global__ __launch_bounds__(64 * NS) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 4 : 3))) void k3_density(St3<R> S, KParams K,
                                                 const uint32_t* __restrict__ skey,
                                                 const int* __restrict__ cstart, Mask3 nbm,
                                                 Pack3<R> P) {
  if (halted(K)) return;
  // contiguous shares per XCD (633 -> 616 us at 2.2M particles in FP32, 86 ->
  // 78 us in FP64 at 84k): the neighbour rows stay in one L2
  // staged records, then (in their place) the lanes' row starts; the reads
  // past the records end in the words
  struct Lds {
    union {
      float4 rec[NS][P3_CAP];
      int lt[9][64];
    };
    uint32_t lw[M3_OK][64];
    R part[NS > 1 ? (NS - 1) * 2 * acc_words<R>() : 1][64];
  };
  __shared__ Lds L;
  static_assert(sizeof(Lds) >= sizeof(float4) * (NS * P3_CAP + P3_TILE + 16), "reads past the records");
  const int lane = threadIdx.x & 63, s0 = wave_of<NS>();
  const int i0 = xcd_block() * 64 + lane;
  const bool valid = i0 < K.n;
  const int i = valid ? i0 : K.n - 1;
  const uint32_t key = skey[i];
  const int row = (int)(key / (uint32_t)K.nx), cx = (int)key - row * K.nx;
  const Rows9 rw = rows3_of(K, key, cstart);
  bool ok = key != 0u || local3_holds(K, pos_rec3(S, i));
  int candidates = 0;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const int len = rw.t1[k] - rw.t0[k];
    ok = ok && len <= 32 * M3_WORDS;
    candidates += len;
  }
  const bool on = valid && ok;
  // (unlikely: so that the registers of what follows stay with the sweeps)
  auto none_has = [&](int c) { return __ballot(on && candidates >= c) == 0ull; };
  if (__builtin_expect(none_has(FEW3_MAX) && none_has(Few3<R>::base + Few3<R>::sweep *
                                                      sweeps3(on, cx, row)), 0))
    pretest3_lanes<NS>(S, K, s0, i, on, rw, L.lt, L.lw);
  else
    pretest3<NS>(S, K, s0, i, on, cx, row, rw, L.rec[s0], L.lw);
  __syncthreads();
  uint32_t(*lw)[64] = L.lw;
  int(*lt)[64] = L.lt;
  uint32_t nz = 0u;  // the lane's non-empty words
  if (valid && ok) {
#pragma unroll
    for (int q = 0; q < M3_OK; ++q) nz |= (lw[q][lane] != 0u ? 1u : 0u) << q;
  }
  if (s0 == 0) {
#pragma unroll
    for (int k = 0; k < 9; ++k) lt[k][lane] = rw.t0[k];
  }
  __syncthreads();
  const auto pi = load_pos3(S, i);
  const auto vi = S.v[i];
  const R cut2 = cutoff2<R>(K);
  DensOwn<R> o;
  if (s0 == 0) dens_begin<R, SUM>(K, o);
  const uint32_t mine = share_bits<NS>(s0);
  if (valid && ok) {
    uint32_t m = 0u;
    int tb = 0, wc = 0;
    R uy = (R)0, uz = (R)0;
    // the next word: its first candidate and its row's y and z terms
    auto enter = [&]() {
      wc = __builtin_ctz(nz);
      nz &= nz - 1u;
      m = lw[wc][lane] & mine;
      const int k = (wc * 11) >> 5;  // wc / 3 for wc < 27
      const int ky = (k * 11) >> 5;  // k / 3 for k < 9
      uy = row_u3<R>(K, 1 - (k - 3 * ky));
      uz = row_u3<R>(K, 1 - ky);
      tb = lt[k][lane] + 32 * (wc - 3 * k);
    };
    while (true) {
      next_word<NS>(m, nz, enter);
      if (m == 0u) break;
      const int b0 = __builtin_ctz(m), w0 = wc, t0 = tb + b0;
      const R uy0 = uy, uz0 = uz;
      m &= m - 1u;
      next_word<NS>(m, nz, enter);
      const bool two = m != 0u;
      const int b1 = two ? __builtin_ctz(m) : b0, t1 = two ? tb + b1 : t0;
      m &= m - 1u;  // 0 stays 0
      const auto p0 = load_pos3(S, t0), p1 = load_pos3(S, t1);
      const auto v0 = S.v[t0], v1 = S.v[t1];
      R ax, ay, az, bx, by, bz;
      const R ra = delta3(pi, p0, K, uy0, uz0, ax, ay, az);
      const R rb = delta3(pi, p1, K, uy, uz, bx, by, bz);
      const bool in0 = ra < cut2, in1 = two && rb < cut2;
      dens3_pair<R, SUM>(K, ax, ay, az, ra, vi.x - v0.x, vi.y - v0.y, vi.z - v0.z, o.sum, o.rs,
                         in0);
      dens3_pair<R, SUM>(K, bx, by, bz, rb, vi.x - v1.x, vi.y - v1.y, vi.z - v1.z, o.sum, o.rs,
                         in1);
      // passed the pre-test only: out of the recorded masks
      if (!in0) atomicAnd(&lw[w0][lane], ~(1u << b0));
      if (two && !in1) atomicAnd(&lw[wc][lane], ~(1u << b1));
    }
  } else if (__builtin_expect(valid, 0)) {
    for (int k = 0; k < 9; ++k) {
      const int t0 = rw.t0[k], t1 = rw.t1[k];
      const R uy = row_u3<R>(K, 1 - k % 3), uz = row_u3<R>(K, 1 - k / 3);
      for (int t = t0; t < t1; ++t) {
        if (t == i || (t - t0) % NS != s0) continue;
        const auto pj = load_pos3(S, t);
        R dx, dy, dz;
        const R r2 = delta3(pi, pj, K, uy, uz, dx, dy, dz);
        if (!(r2 < cut2)) continue;
        const auto vj = S.v[t];
        dens3_pair<R, SUM>(K, dx, dy, dz, r2, vi.x - vj.x, vi.y - vj.y, vi.z - vj.z, o.sum, o.rs);
      }
    }
  }
  constexpr int AW = acc_words<R>();
  share_sum<NS, 2 * AW>(
      L.part, s0, lane,
      [&](R* v) {
        acc_put(v, o.sum);
        acc_put(v + AW, o.rs);
      },
      [&](const R* v) {
        acc_add(o.sum, v);
        acc_add(o.rs, v + AW);
      });
  if (!valid) return;
  if (nbm.w && ok)
#pragma unroll
    for (int q = 0; q < M3_OK; ++q)
      if (q % NS == s0) nbm.put(q, i, lw[q][lane]);
  if (s0 != 0) return;
  if (nbm.w) nbm.put(M3_OK, i, ok ? 1u : 0u);
  dens_end<R, SUM, EOS>(S, K, i, o);
  if (EOS) force3_record(S, K, P, i);
}

template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_eos(St3<R> S, KParams K) {
  const int i = blockIdx.x * BLOCK + threadIdx.x;
  if (i >= K.n) return;
  eos_point(S, K, i, is_rate(K, S.id[i]), S.rho[i], S.divv[i]);
}

// Force pass: int_force pressure part, art_visc, art_heat and av_vel in the
// Q = 1/rho, A = p/rho form of the 2D force_pair (same terms per pair).
template <typename R> struct ForceOwn3 {
  using R4 = typename V4<R>::type;
  R4 v;
  R Q, A, psi, u;
  R fx = 0, fy = 0, fz = 0, xsx = 0, xsy = 0, xsz = 0;
  Acc<R> du;
};

template <typename R>
__device__ __forceinline__ void force3_begin(const St3<R>& S, const KParams& K, int i,
                                             ForceOwn3<R>& o) {
  o.v = S.v[i];
  q_and_a(K, S.rho[i], S.p[i], o.Q, o.A);
  o.psi = S.psi[i];
  o.u = u3_of(S, i);
}

// The terms of one pair apart from their accumulation: the particle gains
// -G r, the energy rate d and -wf dv.
template <typename R> struct Terms3 {
  R G, dx, dy, dz, d, wf, dvx, dvy, dvz;
};

// SE: artificial viscosity and heat share (h eta)^2.
template <typename R, bool PRESS, bool AV, bool AH, bool XS, bool SE>
__device__ __forceinline__ Terms3<R> force3_terms(const KParams& K, const ForceOwn3<R>& o, R dx,
                                                  R dy, R dz, R r2, R vjx, R vjy, R vjz, R Qj,
                                                  R Aj, R psij, R uj) {
  Terms3<R> t;
  t.dx = dx;
  t.dy = dy;
  t.dz = dz;
  t.dvx = o.v.x - vjx;
  t.dvy = o.v.y - vjy;
  t.dvz = o.v.z - vjz;
  t.G = (R)0;
  t.d = (R)0;
  t.wf = (R)0;
  const R vr = fmr(t.dvz, dz, fmr(t.dvy, dy, t.dvx * dx));
  const R m = (R)K.mass;
  const R q = fsqrt(r2) * (R)K.invh;
  const R tq = q - (R)2;
  const R F = (R)K.C1 * (tq * tq * tq);
  const R inv_mrho = (R)2 * o.Q * Qj * frcp(o.Q + Qj);
  R coef = 0;
  if (PRESS) coef = (K.pa_sph == 0) ? fmr(o.A, Qj, Aj * o.Q) : fmr(o.A, o.Q, Aj * Qj);
  R inv_ea = 0;
  if (AV) {
    inv_ea = frcp(r2 + (R)K.av_e2);
    if (vr < (R)0) {
      const R phi = (R)K.h * vr * inv_ea;
      const R pc = fmr((R)K.av_beta, phi, -((R)K.av_alpha * (R)K.c0));
      coef = fmr(pc * phi, inv_mrho, coef);
    }
  }
  if (PRESS || AV) {
    t.G = m * F * coef;
    t.d = (R)0.5 * t.G * vr;
  }
  if (AH) {
    const R inv_eh = (AV && SE) ? inv_ea : frcp(r2 + (R)K.ah_e2);
    t.d = fmr(m * (o.psi + psij) * F * r2 * inv_mrho * inv_eh, o.u - uj, t.d);
  }
  if (XS) {
    const R s = fmr((R)-0.5, q, (R)1);
    const R s2 = s * s;
    const R w = (R)K.wnorm * (s2 * s2) * fmr((R)2, q, (R)1);
    t.wf = (R)K.eps_m * inv_mrho * w;
  }
  return t;
}

// Adds the terms of one pair when ok (else nothing), without a branch.
template <typename R, bool PRESS, bool AV, bool AH, bool XS>
__device__ __forceinline__ void force3_acc(ForceOwn3<R>& o, const Terms3<R>& t, bool ok) {
  if (PRESS || AV) {
    o.fx = ok ? fmr(-t.G, t.dx, o.fx) : o.fx;
    o.fy = ok ? fmr(-t.G, t.dy, o.fy) : o.fy;
    o.fz = ok ? fmr(-t.G, t.dz, o.fz) : o.fz;
  }
  if (PRESS || AV || AH) o.du.add_if(t.d, ok);
  if (XS) {
    o.xsx = ok ? fmr(-t.wf, t.dvx, o.xsx) : o.xsx;
    o.xsy = ok ? fmr(-t.wf, t.dvy, o.xsy) : o.xsy;
    o.xsz = ok ? fmr(-t.wf, t.dvz, o.xsz) : o.xsz;
  }
}

// The deposition heat source after the 3D force pass (fluka_heat.f:235-337),
// as k_deposition in 2D.
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_deposition(St3<R> S, KParams K) {
  if (halted(K)) return;
  const int i = blockIdx.x * BLOCK + threadIdx.x;
  if (i >= K.n || S.id[i] >= K.np) return;
  const double4 q = S.xyz[i];
  R Q, A;
  q_and_a(K, S.rho[i], S.p[i], Q, A);
  S.du[i] = S.du[i] + (R)deposition_at(K, q.x, q.y, q.z) * Q;
}

template <typename R, bool PRESS, bool XS>
__device__ __forceinline__ void force3_end(St3<R>& S, const KParams& K, int i,
                                           const ForceOwn3<R>& o) {
  using R4 = typename V4<R>::type;
  if (PRESS) {
    const int id = S.id[i];
    const bool grav = (K.flags & 16) && id < K.np;
    R4 acc;
    acc.x = o.fx + (grav ? (R)K.gx : (R)0);
    acc.y = o.fy + (grav ? (R)K.gy : (R)0);
    acc.z = o.fz + (grav ? (R)K.gz : (R)0);
    acc.w = (R)0;
    S.a[i] = acc;
    S.du[i] = o.du.get();
  }
  if (XS) {
    R4 w;
    w.x = o.xsx;
    w.y = o.xsy;
    w.z = o.xsz;
    w.w = (R)0;
    S.av[i] = w;
  }
}

__device__ __forceinline__ Pos3F pos_of_rec(float4 q) { return {q.w, q.x, q.y, q.z}; }
__device__ __forceinline__ Pos3D pos_of_rec(double4 q) { return {q.x, q.y, q.z}; }

// The records on their own (after the routines that do not write them).
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_force_pack(St3<R> S, KParams K, Pack3<R> P) {
  if (halted(K)) return;
  const int i = blockIdx.x * BLOCK + threadIdx.x;
  if (i >= K.n) return;
  force3_record(S, K, P, i);
}

// The force gather of a wavefront's 64 consecutive particles: one loop over
// every set bit of a lane's 27 mask words in (row, word, bit) order (a
// wavefront runs for its longest lane's neighbour count).  The FP32 form takes
// two neighbours at a time, whose six record loads are in flight together,
// each added in walk order; in FP64 the second one's registers cost a
// wavefront per SIMD (2.2M particles: 1507 us against 1398).  Each lane keeps its words and row starts in its own LDS column and
// a bitmap of its non-empty words.  A particle without complete masks tests
// its candidates one by one, in the same order with the same pair body.
// Contiguous shares per XCD: the packed records of the neighbour rows stay in
// one L2 (3.6x less traffic beyond L2, 915 -> 880 us in FP32 at 2.2M).
// Bound at 2.2M particles in FP32: the vector cache's tag accesses, one a cycle
// (a record load of 64 lanes touches 46 lines; three loads a neighbour keep it
// 92 % busy), so two neighbours at once leave it at 792 us.  Below that size
// latency: 83,630 particles FP32 51.6 -> 43.7 us; FP64 at 2.2M 1638 -> 1398 us.
// The records written by the density pass take 41 us there instead of a launch
// of 53 (FP64 106 of 121).
template <typename R, bool PRESS, bool AV, bool AH, bool XS, bool SE, int NS>
__global__ __launch_bounds__(64 * NS) void k3_force(
    St3<R> S, Pack3<R> P, KParams K, const uint32_t* __restrict__ skey,
    const int* __restrict__ cstart, Mask3 nbm) {
  if (halted(K)) return;
  __shared__ uint32_t lw[M3_OK][64];
  __shared__ int lt[9][64];
  __shared__ R part[NS > 1 ? (NS - 1) * (6 + acc_words<R>()) : 1][64];
  const int lane = threadIdx.x & 63, s0 = wave_of<NS>();
  const int i0 = xcd_block() * 64 + lane;
  const bool valid = i0 < K.n;
  const int i = valid ? i0 : K.n - 1;
  const auto pi = load_pos3(S, i);
  ForceOwn3<R> o;
  force3_begin(S, K, i, o);
  const Rows9 rw = rows3_of(K, skey[i], cstart);
  auto terms = [&](int t, R uy, R uz) {
    const auto* rp = P.rec + (((unsigned)t << 1) + (unsigned)t);  // 3 t, no 64-bit multiply
    const auto pj = pos_of_rec(rp[0]);
    const auto vq = rp[1];
    const auto ap = rp[2];
    R dx, dy, dz;
    const R r2 = delta3(pi, pj, K, uy, uz, dx, dy, dz);
    return force3_terms<R, PRESS, AV, AH, XS, SE>(K, o, dx, dy, dz, r2, vq.x, vq.y, vq.z, vq.w,
                                                  ap.x, ap.y, ap.z);
  };
  const bool masked = nbm.w && nbm.get(M3_OK, i);
  uint32_t nz = 0u;
  if (masked) {  // wavefronts that share the lanes write the same words
#pragma unroll
    for (int q = 0; q < M3_OK; ++q) {
      const uint32_t m = nbm.get(q, i);
      lw[q][lane] = m;
      nz |= (m != 0u ? 1u : 0u) << q;
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) lt[k][lane] = rw.t0[k];
  }
  if (valid && masked) {
    const uint32_t mine = share_bits<NS>(s0);
    uint32_t m = 0u;
    int tb = 0;
    R uy = (R)0, uz = (R)0;
    // the next word: its first candidate and its row's y and z terms
    auto enter = [&]() {
      const int w = __builtin_ctz(nz);
      nz &= nz - 1u;
      m = lw[w][lane] & mine;
      const int k = (w * 11) >> 5;   // w / 3 for w < 27
      const int ky = (k * 11) >> 5;  // k / 3 for k < 9
      uy = row_u3<R>(K, 1 - (k - 3 * ky));
      uz = row_u3<R>(K, 1 - ky);
      tb = lt[k][lane] + 32 * (w - 3 * k);
    };
    while (true) {
      next_word<NS>(m, nz, enter);
      if (m == 0u) break;
      const int ta = tb + (int)__builtin_ctz(m);
      const R ya = uy, za = uz;
      m &= m - 1u;
      if constexpr (sizeof(R) == 4 || NS > 1) {
        next_word<NS>(m, nz, enter);
        const bool two = m != 0u;
        const int tc = two ? tb + (int)__builtin_ctz(m) : ta;
        m &= m - 1u;  // 0 stays 0
        const Terms3<R> A = terms(ta, ya, za);
        const Terms3<R> B = terms(tc, uy, uz);
        force3_acc<R, PRESS, AV, AH, XS>(o, A, true);
        force3_acc<R, PRESS, AV, AH, XS>(o, B, two);
      } else {
        force3_acc<R, PRESS, AV, AH, XS>(o, terms(ta, ya, za), true);
      }
    }
  } else if (valid) {
    const R cut2 = cutoff2<R>(K);
    for (int k = 0; k < 9; ++k) {
      const R uy = row_u3<R>(K, 1 - k % 3), uz = row_u3<R>(K, 1 - k / 3);
      for (int t = rw.t0[k]; t < rw.t1[k]; ++t) {
        if (t == i || (t - rw.t0[k]) % NS != s0) continue;
        const auto pj = load_pos3(S, t);
        R dx, dy, dz;
        const R r2 = delta3(pi, pj, K, uy, uz, dx, dy, dz);
        if (!(r2 < cut2)) continue;
        force3_acc<R, PRESS, AV, AH, XS>(o, terms(t, uy, uz), true);
      }
    }
  }
  share_sum<NS, 6 + acc_words<R>()>(
      part, s0, lane,
      [&](R* v) {
        v[0] = o.fx, v[1] = o.fy, v[2] = o.fz;
        v[3] = o.xsx, v[4] = o.xsy, v[5] = o.xsz;
        acc_put(v + 6, o.du);
      },
      [&](const R* v) {
        o.fx += v[0], o.fy += v[1], o.fz += v[2];
        o.xsx += v[3], o.xsy += v[4], o.xsz += v[5];
        acc_add(o.du, v + 6);
      });
  if (valid && s0 == 0) force3_end<R, PRESS, XS>(S, K, i, o);
}

// ------------------------------------------------------------------------
// leapfrog (time_integration.f:136-154 predictor, :186-217 corrector)
// ------------------------------------------------------------------------
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_predictor(St3<R> S, KParams K) {
  const int i = blockIdx.x * BLOCK + threadIdx.x;
  if (i >= K.n) return;
  const int id = S.id[i];
  const double hdt = K.dt / 2.0;
  S.flag[i] = 0;
  if (is_rate(K, id)) {
    double u = S.u[i];
    S.u_min[i] = u;
    u = u + hdt * (double)S.du[i];
    if (u < 0.0) {
      u = 0.0;
      S.flag[i] = 1u;
    }
    S.u[i] = u;
    if constexpr (sizeof(R) == 4) S.uf[i] = (float)u;
    if (K.density_method == 0) {
      const R rho = S.rho[i];
      S.rho_min[i] = rho;
      S.rho[i] = rho + (R)hdt * S.drho[i];
    }
  }
  if (id < K.np) {
    auto v = S.v[i];
    const auto a = S.a[i];
    S.v_min[i] = v;
    v.x = v.x + (R)hdt * a.x;
    v.y = v.y + (R)hdt * a.y;
    v.z = v.z + (R)hdt * a.z;
    S.v[i] = v;
  }
}

template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_corrector(St3<R> S, KParams K, int its, int keys,
                                                      KeyOut ko, int* __restrict__ err) {
  if (halted(K)) return;
  const int i = blockIdx.x * BLOCK + threadIdx.x;
  const bool valid = i < K.n;
  uint32_t key = 0;
  int id = 0;
  if (valid) {
    id = S.id[i];
    const double dt = K.dt, hdt = K.dt / 2.0;
    double4 q = S.xyz[i];
    if (is_rate(K, id)) {
      double u;
      if (its != 1) {
        u = S.u_min[i] + dt * (double)S.du[i];
        if (K.density_method == 0) S.rho[i] = S.rho_min[i] + (R)dt * S.drho[i];
      } else {
        u = S.u[i] + hdt * (double)S.du[i];
        if (K.density_method == 0) S.rho[i] = S.rho[i] + (R)hdt * S.drho[i];
      }
      if (u < 0.0) u = 0.0;
      S.u[i] = u;
      if constexpr (sizeof(R) == 4) S.uf[i] = (float)u;
      if (id < K.np) {
        auto v = S.v[i];
        const auto a = S.a[i];
        if (its != 1) {
          const auto vm = S.v_min[i];
          const auto av = S.av[i];
          v.x = vm.x + (R)dt * a.x + av.x;
          v.y = vm.y + (R)dt * a.y + av.y;
          v.z = vm.z + (R)dt * a.z + av.z;
        } else {
          v.x = v.x + (R)hdt * a.x;
          v.y = v.y + (R)hdt * a.y;
          v.z = v.z + (R)hdt * a.z;
        }
        S.v[i] = v;
        q.x = q.x + dt * (double)v.x;
        q.y = q.y + dt * (double)v.y;
        q.z = q.z + dt * (double)v.z;
        S.xyz[i] = q;
      }
    }
    if (keys) {
      int ix, iy, iz;
      bool ok;
      key = cell_of3(K, q.x, q.y, q.z, ix, iy, iz, ok);
      if (!ok) {
      atomicAdd(err, 1);
      raise_halt(K);
    }
    }
  }
  if (keys) emit_key(ko, valid, i, id, key);
}

// ------------------------------------------------------------------------
// pair census: neighbours with larger id
// ------------------------------------------------------------------------
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_pair_count(St3<R> S, KParams K,
                                                       const uint32_t* __restrict__ skey,
                                                       const int* __restrict__ cstart,
                                                       int* __restrict__ cnt,
                                                       const int* __restrict__ offs,
                                                       int* __restrict__ out_i,
                                                       int* __restrict__ out_j) {
  const int i = blockIdx.x * BLOCK + threadIdx.x;
  if (i >= K.n) return;
  const auto pi = load_pos3(S, i);
  const int idi = S.id[i];
  const Rows9 rw = rows3_of(K, skey[i], cstart);
  const R cut2 = cutoff2<R>(K);
  int c = 0;
  const int o = offs ? offs[i] : 0;
  for (int k = 0; k < 9; ++k) {
    const R uy = row_u3<R>(K, 1 - k % 3), uz = row_u3<R>(K, 1 - k / 3);
    for (int t = rw.t0[k]; t < rw.t1[k]; ++t) {
      const int idj = S.id[t];
      if (idj <= idi) continue;
      const auto pj = load_pos3(S, t);
      R dx, dy, dz;
      const R r2 = delta3(pi, pj, K, uy, uz, dx, dy, dz);
      if (!(r2 < cut2)) continue;
      if (offs) {
        out_i[o + c] = idi;
        out_j[o + c] = idj;
      }
      ++c;
    }
  }
  if (cnt) cnt[i] = c;
}

// FP64 sums over real particles: mass, momentum x, y, z, kinetic and
// internal energy; one row of partial sums per block.
template <typename R>
__global__ __launch_bounds__(BLOCK) void k3_conserve(St3<R> S, KParams K,
                                                     double* __restrict__ part) {
  __shared__ double sh[6][BLOCK];
  const int i = blockIdx.x * BLOCK + threadIdx.x;
  double v[6] = {0, 0, 0, 0, 0, 0};
  if (i < K.n && S.id[i] < K.np) {
    const auto vel = S.v[i];
    const double vx = (double)vel.x, vy = (double)vel.y, vz = (double)vel.z;
    v[0] = K.mass;
    v[1] = K.mass * vx;
    v[2] = K.mass * vy;
    v[3] = K.mass * vz;
    v[4] = 0.5 * K.mass * (vx * vx + vy * vy + vz * vz);
    v[5] = K.mass * S.u[i];
  }
  for (int k = 0; k < 6; ++k) sh[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int s = BLOCK / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s)
      for (int k = 0; k < 6; ++k) sh[k][threadIdx.x] += sh[k][threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int k = 0; k < 6; ++k) part[blockIdx.x * 6 + k] = sh[k][0];
}

}  // namespace arm
