// sph_tiled.h -- LDS-tiled gathers of the density and force passes.
//
// A workgroup owns a segment of one cell row: a piece of up to 128
// consecutive sorted particles of the row.  Its particles are one contiguous sorted
// range, and the candidates of all of them lie in three contiguous sorted
// ranges (the cell row below, the row itself and the row above, over the
// segment's cells and one either side).  The workgroup copies those three
// ranges into LDS with coalesced loads.  Each lane then handles one
// particle, row by row:
//   A  test the row's candidates (r^2 < (2h)^2) eight at a time, reading
//      their positions from LDS with independent loads, into a 32-bit row
//      mask;
//   B  run the pair arithmetic over the set bits in ascending order, so the
//      wavefront does the expensive math only for real neighbours (one walk
//      over the three rows' masks where they are complete).
// The visiting order (rows bottom to top, ascending sorted position) and the
// arithmetic are those of the direct path, so both give identical bits.
// Rows longer than 32 candidates are handled in 32-candidate chunks (their
// masks are not recorded); when the three ranges exceed the LDS capacity the
// workgroup falls back to the direct path.
#pragma once

#include "sph_kernels.h"

namespace arm {

// ---- LDS tiles ------------------------------------------------------------
// The eight-wide neighbour test may read up to seven records past a row's end
// (their bits are masked off).  After the last row of a full tile these lie in
// the array that follows in the tile, so what the test reads is never its last
// member.  In the FP32 form a record keeps the cell column as a
// float, and the cell-row difference of a candidate row is the constant
// 1 - k of row k of the segment, so
//   dx = (off_i.x - off_j.x) + (cx_i - cx_j) cell
//   dy = (off_i.y - off_j.y) + (1 - k) cell
// are the same operations, with the same roundings, as delta() on PosF.
// Records of a tile.  A piece's three rows hold about 3 x 140 on the dam-break
// lattice, 584 at most, but up to 640 where a row has fewer particles than its
// neighbours (h = 1.7 or 1.8 dx on a lattice); a piece of more runs on the direct
// path.  FP32: 640 (ten workgroups a CU in the density pass, seven in the force),
// and 592 with the physical viscosity (five) and in the hot force gather, whose
// 18.9 KB let eight share a CU.  FP64: 600 (seven and four).  With 592 in all of
// them the passes at h = 1.8 dx, 350,000 particles, took in FP64 92 us (density) and
// 197 (force with the corrector), now 83 and 165; in FP32 64 (density), now 55.
// With the physical viscosity runs of 32 or 16 cells with smaller tiles were the
// faster form until the loads of the prologue overlapped (heated channel of 2
// million, force with the corrector: FP32 189 us on runs, 182 on pieces; FP64 377
// and 369).
template <typename R, bool VI = false> constexpr int tile_cap() {
  return sizeof(R) == 8 ? 600 : (VI ? GAP_RECORDS : 640);
}

// Byte offset 4 l of a 4-byte LDS record.  Computed out of the compiler's
// sight: otherwise it derives this address from the 16-byte records' l << 4
// with 64-bit integer multiply-adds, two of them per neighbour.
__device__ __forceinline__ uint32_t off4(int l) {
  uint32_t r;
  asm("v_lshlrev_b32 %0, 2, %1" : "=v"(r) : "v"(l));
  return r;
}

template <typename T> __device__ __forceinline__ T lds_at(const T* base, uint32_t byte_off) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + byte_off);
}

// Lane particle for tile deltas (FP32 form).
struct LaneF {
  float cxf, ox, oy;
};

// The cell-row term of row k: (float)(cy_i - cy_j) * cell with cy_i - cy_j = 1 - k.
__device__ __forceinline__ float row_uy(const KParams& K, int k) {
  return (float)(1 - k) * K.cellf;
}

__device__ __forceinline__ void tile_delta(const KParams& K, const LaneF& p, float cxj, float oxj,
                                           float oyj, float uy, float& dx, float& dy) {
  const float tx = p.ox - oxj;
  const float ux = (p.cxf - cxj) * K.cellf;
  dx = tx + ux;
  const float ty = p.oy - oyj;
  dy = ty + uy;
}

template <typename R> struct DensTile;
template <> struct DensTile<float> {
  // the neighbour test reads one 16-byte record per candidate
  float4 a[tile_cap<float>()];  // offx, offy, cell column as float, vx
  float vy[tile_cap<float>()];
  struct Raw {
    float2 o, v;
    uint32_t c;
  };
  static __device__ __forceinline__ Raw load(const St<float>& S, int t) {
    return {S.off[t], S.v[t], S.cxy[t]};
  }
  __device__ __forceinline__ void put(int l, const KParams&, const Raw& r) {
    a[l] = make_float4(r.o.x, r.o.y, (float)(r.c & 0xffffu), r.v.x);
    vy[l] = r.v.y;
  }
  __device__ __forceinline__ LaneF lane(int l) const {
    const float4 q = a[l];
    return {q.z, q.x, q.y};
  }
  __device__ __forceinline__ void delta(const KParams& K, const LaneF& p, int l, float uy,
                                        float& dx, float& dy) const {
    const float4 q = a[l];
    tile_delta(K, p, q.z, q.x, q.y, uy, dx, dy);
  }
  __device__ __forceinline__ float2 vel(int l) const {
    return make_float2(a[l].w, lds_at(vy, off4(l)));
  }
};
template <> struct DensTile<double> {
  double2 x[tile_cap<double>()], v[tile_cap<double>()];
  struct Raw {
    double2 x, v;
  };
  static __device__ __forceinline__ Raw load(const St<double>& S, int t) {
    return {S.xy[t], S.v[t]};
  }
  __device__ __forceinline__ void put(int l, const KParams&, const Raw& r) {
    x[l] = r.x;
    v[l] = r.v;
  }
  __device__ __forceinline__ PosD lane(int l) const {
    const double2 q = x[l];
    return {q.x, q.y};
  }
  __device__ __forceinline__ void delta(const KParams&, const PosD& p, int l, double, double& dx,
                                        double& dy) const {
    const double2 q = x[l];
    dx = p.x - q.x;
    dy = p.y - q.y;
  }
  __device__ __forceinline__ double2 vel(int l) const { return v[l]; }
};

// Positions of the neighbour pre-test: x and y as 16-bit fixed-point numbers of
// FIX units per cell, modulo 2^16 (a particle and its candidates are less than
// three cells apart, so their difference is exact through the wrap), in one
// 4-byte record: a candidate's test is a packed subtraction, a dot product
// against the bound and a shift of the sign into the mask, three instructions
// in either form, instead of the eight (FP32) or seven in FP64 (at half the
// rate) of a test on the staged floating-point positions.
constexpr int FIX = 4096;
using s16x2 = __attribute__((ext_vector_type(2))) short;

template <typename R> struct PreTile {
  uint32_t p[tile_cap<R>()];
  __device__ __forceinline__ void put(int l, const KParams& K,
                                      const DensTile<float>::Raw& r) {
    const uint32_t c = r.c;
    const uint32_t x = (c & 0xffffu) * FIX + (uint32_t)(int)__builtin_fmaf(r.o.x, K.fixf, 0.5f);
    const uint32_t y = (c >> 16) * FIX + (uint32_t)(int)__builtin_fmaf(r.o.y, K.fixf, 0.5f);
    p[l] = (x & 0xffffu) | (y << 16);
  }
  __device__ __forceinline__ void put(int l, const KParams& K,
                                      const DensTile<double>::Raw& r) {
    auto fix = [&](double d) {
      const double u = d * K.fix;
      return (uint32_t)(int)(u - 65536.0 * floor(u * (1.0 / 65536.0)) + 0.5);
    };
    p[l] = (fix(r.x.x - K.ox) & 0xffffu) | (fix(r.x.y - K.oy) << 16);
  }
};

// Neighbour W = c T of the physical viscosity, staged only when VI.
template <typename R, bool VI> struct TauTile {
  struct Raw {};
  static __device__ __forceinline__ Raw load(const St<R>&, int) { return {}; }
  __device__ __forceinline__ void put(int, const Raw&, R) {}
  __device__ __forceinline__ Tau3<R> get(int) const { return Tau3<R>{}; }
};
template <> struct TauTile<float, true> {
  float4 w[tile_cap<float, true>()];
  using Raw = float4;
  static __device__ __forceinline__ Raw load(const St<float>& S, int t) {
    return reinterpret_cast<const float4*>(S.tau)[t];
  }
  __device__ __forceinline__ void put(int l, const Raw& q, float c) {
    w[l] = make_float4(c * q.x, c * q.y, c * q.z, q.w);
  }
  __device__ __forceinline__ Tau3<float> get(int l) const {
    const float4 q = w[l];
    return {q.x, q.y, q.z};
  }
};
template <> struct TauTile<double, true> {
  double2 w01[tile_cap<double, true>()];
  double w2[tile_cap<double, true>()];
  struct Raw {
    double xx, yy, xy;
  };
  static __device__ __forceinline__ Raw load(const St<double>& S, int t) {
    const double* q = S.tau + 4 * (size_t)t;
    return {q[0], q[1], q[2]};
  }
  __device__ __forceinline__ void put(int l, const Raw& q, double c) {
    w01[l] = make_double2(c * q.xx, c * q.yy);
    w2[l] = c * q.xy;
  }
  __device__ __forceinline__ Tau3<double> get(int l) const {
    const double2 q = w01[l];
    return {q.x, q.y, w2[l]};
  }
};

// The particle's own viscous terms: W from its record, tds from the state.
template <typename R>
__device__ __forceinline__ void own_tau(const St<R>& S, ForceOwn<R>& o, int i, const Tau3<R>& w) {
  o.wxx = w.xx;
  o.wyy = w.yy;
  o.wxy = w.xy;
  o.tds = S.tau[4 * (size_t)i + 3];
}

// The FP32 records: offx, offy, vx, vy; Q = 1/rho, A = p/rho, psi, u; cell column
// as float.  With the shear tensor behind them the columns come last, with the spare records
// of their own (first, as without it: force of 100,000 particles 56 -> 58 us).
template <bool VI> struct ForceRecs {
  float cx[tile_cap<float>()];
  float4 a[tile_cap<float>()];
  float4 b[tile_cap<float>()];
};
template <> struct ForceRecs<true> {
  float4 a[tile_cap<float, true>() + 8];
  float4 b[tile_cap<float, true>() + 8];
  float cx[tile_cap<float, true>() + 8];
};

template <typename R, bool VI = false> struct ForceTile;
template <bool VI> struct ForceTile<float, VI> : ForceRecs<VI> {
  using ForceRecs<VI>::a;
  using ForceRecs<VI>::b;
  using ForceRecs<VI>::cx;
  TauTile<float, VI> tw;
  struct Raw {
    float2 o, v;
    float rho, p, psi, u;
    uint32_t c;
    typename TauTile<float, VI>::Raw w;
  };
  static __device__ __forceinline__ Raw load(const St<float>& S, int t) {
    return {S.off[t], S.v[t],  S.rho[t], S.p[t],
            S.psi[t], S.uf[t], S.cxy[t], TauTile<float, VI>::load(S, t)};
  }
  __device__ __forceinline__ void put(int l, const KParams& K, const Raw& r) {
    a[l] = make_float4(r.o.x, r.o.y, r.v.x, r.v.y);
    float Q, A;
    q_and_a(K, r.rho, r.p, Q, A);
    b[l] = make_float4(Q, A, r.psi, r.u);
    cx[l] = (float)(r.c & 0xffffu);
    tw.put(l, r.w, visc_c(K, Q));
  }
  // force_begin from the particle's own record
  __device__ __forceinline__ void own(const St<float>& S, const KParams& K, ForceOwn<float>& o,
                                      int i, int l) const {
    const float4 q = a[l];
    const float4 w = b[l];
    o.v = make_float2(q.z, q.w);
    o.Q = w.x;
    o.A = w.y;
    o.psi = w.z;
    o.u = w.w;
    own_factors_f32(K, o);
    if (VI) own_tau(S, o, i, tw.get(l));
  }
  __device__ __forceinline__ LaneF lane(int l) const {
    const float4 q = a[l];
    return {lds_at(cx, off4(l)), q.x, q.y};
  }
  __device__ __forceinline__ void delta(const KParams& K, const LaneF& p, int l, float uy,
                                        float& dx, float& dy) const {
    const float4 q = a[l];
    tile_delta(K, p, lds_at(cx, off4(l)), q.x, q.y, uy, dx, dy);
  }
  template <bool PRESS, bool AV, bool AH, bool XS, int PC = -1>
  __device__ __forceinline__ void pair(const KParams& K, ForceOwn<float>& o, int l, float dx,
                                       float dy, float r2) const {
    const float4 q = a[l];
    const float4 w = b[l];
    force_pair<float, PRESS, AV, AH, XS, VI, PC>(K, o, dx, dy, r2, q.z, q.w, w.x, w.y, w.z,
                                                 w.w, tw.get(l));
  }
};
template <bool VI> struct ForceTile<double, VI> {
  static constexpr int CAP = tile_cap<double, VI>();
  double2 x[CAP], v[CAP], rp[CAP], pu[CAP];  // rp = (Q, A), pu = (psi, u)
  TauTile<double, VI> tw;
  struct Raw {
    double2 x, v;
    double rho, p, psi, u;
    typename TauTile<double, VI>::Raw w;
  };
  static __device__ __forceinline__ Raw load(const St<double>& S, int t) {
    return {S.xy[t],  S.v[t], S.rho[t], S.p[t],
            S.psi[t], S.u[t], TauTile<double, VI>::load(S, t)};
  }
  __device__ __forceinline__ void put(int l, const KParams& K, const Raw& r) {
    x[l] = r.x;
    v[l] = r.v;
    double Q, A;
    q_and_a(K, r.rho, r.p, Q, A);
    rp[l] = make_double2(Q, A);
    pu[l] = make_double2(r.psi, r.u);
    tw.put(l, r.w, visc_c(K, Q));
  }
  __device__ __forceinline__ void own(const St<double>& S, const KParams&, ForceOwn<double>& o,
                                      int i, int l) const {
    o.v = v[l];
    o.Q = rp[l].x;
    o.A = rp[l].y;
    o.psi = pu[l].x;
    o.u = pu[l].y;
    if (VI) own_tau(S, o, i, tw.get(l));
  }
  __device__ __forceinline__ PosD lane(int l) const {
    const double2 q = x[l];
    return {q.x, q.y};
  }
  __device__ __forceinline__ void delta(const KParams&, const PosD& p, int l, double, double& dx,
                                        double& dy) const {
    const double2 q = x[l];
    dx = p.x - q.x;
    dy = p.y - q.y;
  }
  template <bool PRESS, bool AV, bool AH, bool XS, int PC = -1>
  __device__ __forceinline__ void pair(const KParams& K, ForceOwn<double>& o, int l, double dx,
                                       double dy, double r2) const {
    const double2 vv = v[l];
    const double2 a = rp[l];
    const double2 b = pu[l];
    force_pair<double, PRESS, AV, AH, XS, VI>(K, o, dx, dy, r2, vv.x, vv.y, a.x, a.y, b.x, b.y,
                                              tw.get(l));
  }
};

// Positions, velocities and Q = 1/rho for the shear tensor pass.
template <typename R> struct TensTile {
  DensTile<R> d;
  R q[tile_cap<R>()];
  struct Raw {
    typename DensTile<R>::Raw d;
    R rho;
  };
  static __device__ __forceinline__ Raw load(const St<R>& S, int t) {
    return {DensTile<R>::load(S, t), S.rho[t]};
  }
  __device__ __forceinline__ void put(int l, const KParams& K, const Raw& r) {
    d.put(l, K, r.d);
    q[l] = (R)1 / dens(K, r.rho);
  }
  __device__ __forceinline__ auto lane(int l) const { return d.lane(l); }
  template <typename LP>
  __device__ __forceinline__ void delta(const KParams& K, const LP& p, int l, R uy, R& dx,
                                        R& dy) const {
    d.delta(K, p, l, uy, dx, dy);
  }
};

// ---- segment geometry ------------------------------------------------------
// The piece of a workgroup: the particles [O0, O1) of cell row cy; the tile
// holds the candidate ranges of rows cy-1 .. cy+1 (rs[k], rl[k]: sorted start
// and length of row k's, lo[k]: its first tile entry).
struct Segment {
  int cy, O0, O1, x0, x1;
  int rs[3], rl[3], lo[3];
  int total;
};

struct SegArg {
  const PieceRec* tab;
  int masks;  // the density pass has recorded the neighbour masks
};

// O0 >= O1 when the workgroup has no particles.
__device__ __forceinline__ Segment segment_of(const SegArg& sa) {
  const PieceRec r = sa.tab[blockIdx.x];
  Segment g;
  g.cy = r.cy;
  g.O0 = r.O0;
  g.O1 = r.O1;
  g.x0 = r.x0;
  g.x1 = r.x1;
  g.total = r.total;
  int l = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    g.rs[k] = r.rs[k];
    g.rl[k] = r.rl[k];
    g.lo[k] = l;
    l += r.rl[k];
  }
  return g;
}

// A lane particle's cell column and its candidates [ta_k, tb_k) of row k
// (sorted positions; empty where the row has none), looked up before the tile
// is filled, so that the loads run beside the staging.
struct LaneRows {
  int cx;
  int ta[3], tb[3];
};
__device__ __forceinline__ LaneRows lane_rows(const KParams& K, const Segment& g,
                                              const int* __restrict__ cstart, uint32_t key) {
  LaneRows r;
  r.cx = (int)key - g.cy * K.nx;
  const int ca = r.cx > 0 ? r.cx - 1 : 0;
  const int cb = (r.cx + 1 < K.nx ? r.cx + 1 : K.nx - 1) + 1;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int row = (g.cy - 1 + (g.rl[k] ? k : 1)) * K.nx;
    const int a = cstart[row + ca], b = cstart[row + cb];
    r.ta[k] = g.rl[k] ? a : 0;
    r.tb[k] = g.rl[k] ? b : 0;
  }
  return r;
}

// On a grid periodic in x (PER) the particles of the first and last cell
// columns also see the column at the other end.  A piece that holds some keeps
// those cells in its tile after the rows: ranges 0 .. 2 are the last column's
// (for cells of column 0), 3 .. 5 column 0's (for the last column's).
// Particles of the seam that walked their nine cells in global memory instead
// set the time of every launch (FP64 channel of 10,000 particles: force 40 us,
// density and tensor 24 us).
template <bool PER> struct Wrap {
  static constexpr int total = 0;
  __device__ __forceinline__ Wrap(const KParams&, const Segment&, const int*) {}
};
template <> struct Wrap<true> {
  int rs[6], rl[6], lo[6];
  int total;  // 0 off the seam
  __device__ __forceinline__ Wrap(const KParams& K, const Segment& g,
                                  const int* __restrict__ cstart) {
    total = 0;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const int ry = g.cy - 1 + k % 3;
      rs[k] = rl[k] = 0;
      if ((k < 3 ? g.x0 == 0 : g.x1 == K.nx - 1) && ry >= 0 && ry < K.ny) {
        const int* e = cstart + ry * K.nx + (k < 3 ? K.nx - 1 : 0);
        rs[k] = e[0];
        rl[k] = e[1] - e[0];
      }
      lo[k] = g.total + total;
      total += rl[k];
    }
  }
};

// The lane particle as its candidates at the other end see it: sh cells on
// (the operations of delta() with a shift).
__device__ __forceinline__ LaneF image(LaneF p, int sh) {
  p.cxf = p.cxf + (float)sh;
  return p;
}
__device__ __forceinline__ PosD image(PosD p, int) { return p; }
__device__ __forceinline__ float image_dx(const KParams&, const LaneF&, float dx, int) {
  return dx;
}
__device__ __forceinline__ double image_dx(const KParams& K, const PosD&, double dx, int sh) {
  return dx + (double)sh * K.cell;
}

// Calls visit(l, dx, dy, r2) for the neighbours of a lane particle at the
// other end of the grid, after those of its own rows.
template <typename R, typename Tile, typename LP, typename Visit>
__device__ __forceinline__ void for_wrapped(const KParams& K, const Wrap<true>& W, const Tile& T,
                                            int cx, const LP& pi, Visit&& visit) {
  const bool left = cx == 0;
  if (!left && cx != K.nx - 1) return;
  const int sh = left ? K.nx : -K.nx;
  const LP p = image(pi, sh);
  const R cut2 = cutoff2<R>(K);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const R uy = (R)row_uy(K, k);
    const int l0 = left ? W.lo[k] : W.lo[3 + k];
    const int l1 = l0 + (left ? W.rl[k] : W.rl[3 + k]);
    for (int l = l0; l < l1; ++l) {
      R dx, dy;
      T.delta(K, p, l, uy, dx, dy);
      dx = image_dx(K, pi, dx, sh);
      const R r2 = dx * dx + dy * dy;
      if (r2 < cut2) visit(l, dx, dy, r2);
    }
  }
}
template <typename R, typename Tile, typename LP, typename Visit>
__device__ __forceinline__ void for_wrapped(const KParams&, const Wrap<false>&, const Tile&, int,
                                            const LP&, Visit&&) {}

// Tile entries q0 + u PIECE + lane, u < UN, of the three rows, read (load(t): the
// record of sorted position t) before any is written (put(l, record)), so that
// filling a tile waits for memory once or twice.  Past the last entry the last
// one is read and written again: no branch for the compiler to move the loads
// into.
template <int UN, typename Raw> struct Stage {
  Raw r[UN];
  template <typename Load>
  __device__ __forceinline__ void load(const Segment& g, int q0, Load&& ld) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int q = at(g, q0, u);
      int t = q + g.rs[0];
      t += q >= g.lo[1] ? g.rs[1] - g.lo[1] - g.rs[0] : 0;
      t += q >= g.lo[2] ? g.rs[2] - g.lo[2] - (g.rs[1] - g.lo[1]) : 0;
      r[u] = ld(t);
    }
  }
  template <typename Put>
  __device__ __forceinline__ void put(const Segment& g, int q0, Put&& pt) const {
#pragma unroll
    for (int u = 0; u < UN; ++u) pt(at(g, q0, u), r[u]);
  }
  static __device__ __forceinline__ int at(const Segment& g, int q0, int u) {
    return min(q0 + u * PIECE + (int)threadIdx.x, g.total - 1);
  }
};

// The batches after the first, and the seam's cells.
template <int UN, typename Raw, bool PER, typename Load, typename Put>
__device__ __forceinline__ void stage_rest(const Segment& g, const Wrap<PER>& W, Load&& ld,
                                           Put&& pt) {
  for (int q0 = UN * PIECE; q0 < g.total; q0 += UN * PIECE) {
    Stage<UN, Raw> st;
    st.load(g, q0, ld);
    st.put(g, q0, pt);
  }
  if constexpr (PER) {
    for (int q = g.total + (int)threadIdx.x; q < g.total + W.total; q += PIECE) {
      int t = 0;
#pragma unroll
      for (int k = 0; k < 6; ++k)
        if (q >= W.lo[k]) t = q - W.lo[k] + W.rs[k];  // an empty range gives way to the next
      pt(q, ld(t));
    }
  }
}

// Fills the tile (if tiled), then calls lane(i, key, rows) for the workgroup's
// particles, one lane each, and done(i, on) in all lanes (on: it has one);
// early(i) loads what else lane() needs, late(i) what depends on that.  All of
// it is read beside the tile's records: after the piece's record that takes
// two dependent loads, where a chain of staging, key and cell bounds takes six,
// most of a workgroup's life on the small tiles of 2D (720,000 particles, FP32:
// force 43.5 -> 34.3 us, density 41.8 -> 35.1; 1,972, FP64: 12.7 -> 11.5 and
// 13.0 -> 10.8).
template <int UN, typename Raw, bool PER, typename Early, typename Late, typename Load,
          typename Put, typename Lane, typename Done>
__device__ __forceinline__ void for_segment(const KParams& K, const Segment& g,
                                            const Wrap<PER>& W, const uint32_t* __restrict__ skey,
                                            const int* __restrict__ cstart, bool tiled,
                                            Early&& early, Late&& late, Load&& ld, Put&& pt,
                                            Lane&& lane, Done&& done) {
  const int i = g.O0 + (int)threadIdx.x;
  const int ic = min(i, g.O1 - 1);  // no branch, so that the loads overlap
  const uint32_t key = skey[ic];
  early(ic);
  Stage<UN, Raw> st;
  st.load(g, 0, ld);
  const LaneRows r = lane_rows(K, g, cstart, key);
  late(ic);
  if (tiled) {
    st.put(g, 0, pt);
    stage_rest<UN, Raw>(g, W, ld, pt);
  }
  __syncthreads();
  if (i < g.O1) lane(i, key, r);
  done(i, i < g.O1);
}

// The row pieces on their own (after a sort that does not build them): first the
// chunks' sums, then the table.
__global__ __launch_bounds__(ROW_CHUNK) void k_row_sums(const int* __restrict__ cstart, RowPieces rp,
                                                        Halt hl) {
  if (hl.on()) return;
  row_sums_block<ROW_CHUNK>(cstart, rp, blockIdx.x);
}
__global__ __launch_bounds__(BLOCK) void k_row_pieces(const int* __restrict__ cstart,
                                                      const uint32_t* __restrict__ skey,
                                                      RowPieces rp, Halt hl) {
  if (hl.on()) return;
  row_pieces_block<BLOCK>(cstart, skey, rp, blockIdx.x, gridDim.x);
}

// Neighbour mask of candidates l0 .. l0+len-1 (len <= 32) of row k: eight
// independent tile reads and tests per batch, no per-candidate branch; the
// bits past len and the lane's own bit are cleared afterwards.
template <typename R, typename Tile, typename LP>
__device__ __forceinline__ uint32_t row_mask(const KParams& K, const Tile& T, const LP& pi, R uy,
                                             int l0, int len, int self) {
  const R cut2 = cutoff2<R>(K);
  uint32_t m = 0;
  for (int k0 = 0; k0 < len; k0 += 8) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      R dx, dy;
      T.delta(K, pi, l0 + k0 + q, uy, dx, dy);
      const R r2 = dx * dx + dy * dy;
      m |= (r2 < cut2 ? 1u : 0u) << (k0 + q);
    }
  }
  m &= len >= 32 ? 0xffffffffu : ((1u << len) - 1u);
  const int sb = self - l0;
  if (sb >= 0 && sb < 32) m &= ~(1u << sb);
  return m;
}

// Calls visit(l, uy) for every neighbour of lane particle i, rows bottom to
// top, ascending sorted position within a row (uy: the cell-row term of the
// row).
template <typename R, typename Tile, typename LP, typename Visit>
__device__ __forceinline__ void for_neighbours(const KParams& K, const Segment& g,
                                               const LaneRows& lr, const Tile& T, const LP& pi,
                                               int i, Visit&& visit) {
  const int self = g.lo[1] + (i - g.rs[1]);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    if (g.rl[k] == 0) continue;
    const R uy = (R)row_uy(K, k);
    const int base = g.lo[k] - g.rs[k];
    for (int c0 = lr.ta[k]; c0 < lr.tb[k]; c0 += 32) {
      const int len = min(32, lr.tb[k] - c0);
      uint32_t m = row_mask<R>(K, T, pi, uy, base + c0, len, self);
      while (m) {
        const int b = __builtin_ctz(m);
        m &= m - 1;
        visit(base + c0 + b, uy);
      }
    }
  }
}

// One loop over the bits of three row masks in row order (bit b of row k:
// tile entry l_k + b), so that a wavefront runs for its longest lane's
// neighbour count rather than for the sum of the per-row maxima; the order
// of the visits, and so every sum, is that of a row-by-row walk.
template <typename R, typename Visit>
__device__ __forceinline__ void walk_masks(const KParams& K, uint32_t m0, uint32_t m1,
                                           uint32_t m2, int l0, int l1, int l2, Visit&& visit) {
  while (m0 | m1 | m2) {
    const bool s0 = m0 != 0u, s1 = !s0 && m1 != 0u;
    const uint32_t m = s0 ? m0 : (s1 ? m1 : m2);
    const int l = (s0 ? l0 : (s1 ? l1 : l2)) + (int)__builtin_ctz(m);
    const R uy = s0 ? (R)row_uy(K, 0) : (s1 ? (R)row_uy(K, 1) : (R)row_uy(K, 2));
    const uint32_t rest = m & (m - 1u);
    m0 = s0 ? rest : m0;
    m1 = s1 ? rest : m1;
    m2 = (s0 || s1) ? m2 : rest;
    visit(l, uy);
  }
}

// The same order with less work per neighbour: a lane walks one row mask at
// a time and takes the next non-empty row only when the current one is
// exhausted, so the per-neighbour step is a bit scan; the row change runs
// only in the iterations where some lane of the wavefront needs it.  Row k
// has mask m_k, first tile entry l_k and row term u_k; visit(l, u).
template <typename R, typename Visit>
__device__ __forceinline__ void walk_rows(uint32_t m0, uint32_t m1, uint32_t m2, int l0, int l1,
                                          int l2, R u0, R u1, R u2, Visit&& visit) {
  uint32_t m = m0;
  int base = l0;
  R uy = u0;
  while (true) {
    if (m == 0u) {
      const bool t1 = m1 != 0u;
      m = t1 ? m1 : m2;
      base = t1 ? l1 : l2;
      uy = t1 ? u1 : u2;
      m1 = t1 ? m2 : 0u;
      l1 = l2;
      u1 = u2;
      m2 = 0u;
      if (m == 0u) break;
    }
    const int b = (int)__builtin_ctz(m);
    m &= m - 1u;
    visit(base + b, uy);
  }
}

// The pre-test of candidates l0 .. l0+len-1 (len <= 32) of one row against
// K.fix2, a bound on (2h)^2 in units of the fixed-point positions (own: the
// lane's) that covers their rounding; the survivors (about one in two thousand
// too many) take the exact test in the walk.
template <typename R>
__device__ __forceinline__ uint32_t row_mask_pre(const KParams& K, const PreTile<R>& P, s16x2 own,
                                                 int l0, int len, int self) {
  const int bound = -K.fix2;
  uint32_t m = 0;
  for (int k0 = 0; k0 < len; k0 += 8) {
    uint32_t bb = 0u;  // the batch's bits, placed once
#pragma unroll
    for (int q = 7; q >= 0; --q) {
      const s16x2 d = own - __builtin_bit_cast(s16x2, P.p[l0 + k0 + q]);
      bb = __builtin_amdgcn_alignbit(bb, (uint32_t)__builtin_amdgcn_sdot2(d, d, bound, false), 31);
    }
    m |= bb << k0;
  }
  m &= len >= 32 ? 0xffffffffu : ((1u << len) - 1u);
  const int sb = self - l0;
  if (sb >= 0 && sb < 32) m &= ~(1u << sb);
  return m;
}

// for_neighbours of the density pass, row by row: the pre-test, then over its
// survivors the exact test (r^2 < (2h)^2 with the direct path's arithmetic)
// and the pair sums, without a branch: a survivor that fails the exact test
// adds nothing (dens_pair with ok = false) and leaves the recorded mask.
// Same visiting order and sums as for_neighbours; the exact masks in rm.
// Taken by dens_walk for a particle with a row of more than 32 candidates.
template <typename R, bool SUM, typename LP, typename V>
__device__ __forceinline__ void dens_walk_rows(const KParams& K, const Segment& g, const LaneRows& lr,
                                               const DensTile<R>& T, const PreTile<R>& P,
                                               const LP& pi, const V& vi, int i, DensOwn<R>& o,
                                               uint32_t* rm, bool* ok) {
  const int self = g.lo[1] + (i - g.rs[1]);
  const R cut2 = cutoff2<R>(K);
  const s16x2 own = __builtin_bit_cast(s16x2, P.p[self]);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    if (g.rl[k] == 0) continue;
    const R uy = (R)row_uy(K, k);
    const int ta = lr.ta[k], tb = lr.tb[k];
    const int base = g.lo[k] - g.rs[k];
    if (tb - ta > 32) *ok = false;
    for (int c0 = ta; c0 < tb; c0 += 32) {
      const int len = min(32, tb - c0);
      uint32_t m = row_mask_pre(K, P, own, base + c0, len, self);
      uint32_t w = m;
      while (w) {
        const int b = __builtin_ctz(w);
        w &= w - 1;
        const int l = base + c0 + b;
        R dx, dy;
        T.delta(K, pi, l, uy, dx, dy);
        const R r2 = dx * dx + dy * dy;
        const bool in = r2 < cut2;
        m = in ? m : (m & ~(1u << b));
        const auto vj = T.vel(l);
        dens_pair<R, SUM>(K, dx, dy, r2, vi.x - vj.x, vi.y - vj.y, o.sum, o.rs, in);
      }
      if (c0 == ta) rm[k] = m;
    }
  }
}

// The density walk: the pre-test of all three rows first, then one loop over
// the survivors of the three masks in row order (so that a wavefront runs for
// its longest lane's survivor count, not for the sum over the rows of the
// per-row maxima), each through the exact test and the pair sums without a
// branch.  Failed survivors are collected per row (fc, flushed at each row
// change) and taken out of the recorded masks.  Same visiting order and sums
// as for_neighbours; the exact masks in rm.
template <typename R, bool SUM, typename LP, typename V>
__device__ __forceinline__ void dens_walk(const KParams& K, const Segment& g, const LaneRows& lr,
                                          const DensTile<R>& T, const PreTile<R>& P,
                                          const LP& pi, const V& vi, int i, DensOwn<R>& o,
                                          uint32_t* rm, bool* ok) {
  const int self = g.lo[1] + (i - g.rs[1]);
  const s16x2 own = __builtin_bit_cast(s16x2, P.p[self]);
  uint32_t pm[3];
  int pb[3];
  bool small = true;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    pm[k] = 0u;
    pb[k] = 0;
    if (g.rl[k] == 0) continue;
    const int ta = lr.ta[k], tb = lr.tb[k];
    pb[k] = g.lo[k] - g.rs[k] + ta;
    small = small && tb - ta <= 32;
    pm[k] = row_mask_pre(K, P, own, pb[k], min(32, tb - ta), self);
  }
  if (!small) {
    dens_walk_rows<R, SUM>(K, g, lr, T, P, pi, vi, i, o, rm, ok);
    return;
  }
  const R cut2 = cutoff2<R>(K);
  uint32_t f0 = 0u, f1 = 0u, f2 = 0u, fc = 0u;  // failed survivors: rows 0..2, current row
  int kc = 0;
  uint32_t m = pm[0];
  int base = pb[0];
  R uy = (R)row_uy(K, 0);
  while (true) {
    if (m == 0u) {
      f0 |= kc == 0 ? fc : 0u;
      f1 |= kc == 1 ? fc : 0u;
      f2 |= kc == 2 ? fc : 0u;
      fc = 0u;
      const bool t1 = kc == 0 && pm[1] != 0u;
      const bool t2 = !t1 && kc < 2 && pm[2] != 0u;
      if (!(t1 || t2)) break;
      kc = t1 ? 1 : 2;
      m = t1 ? pm[1] : pm[2];
      base = t1 ? pb[1] : pb[2];
      uy = t1 ? (R)row_uy(K, 1) : (R)row_uy(K, 2);
    }
    const int b = (int)__builtin_ctz(m);
    m &= m - 1u;
    const int l = base + b;
    R dx, dy;
    T.delta(K, pi, l, uy, dx, dy);
    const R r2 = dx * dx + dy * dy;
    const bool in = r2 < cut2;
    fc |= in ? 0u : (1u << b);
    const auto vj = T.vel(l);
    dens_pair<R, SUM>(K, dx, dy, r2, vi.x - vj.x, vi.y - vj.y, o.sum, o.rs, in);
  }
  rm[0] = pm[0] & ~f0;
  rm[1] = pm[1] & ~f1;
  rm[2] = pm[2] & ~f2;
}

// The same walk driven by masks recorded by the density pass.
// (Rows outside the grid have empty masks: their entries are not looked up.)
template <typename R, typename Visit>
__device__ __forceinline__ void for_masked(const KParams& K, const Segment& g, const LaneRows& lr,
                                           uint4 nm, Visit&& visit) {
  walk_masks<R>(K, nm.x, nm.y, nm.z, g.lo[0] - g.rs[0] + lr.ta[0], g.lo[1] - g.rs[1] + lr.ta[1],
                g.lo[2] - g.rs[2] + lr.ta[2], visit);
}

// The same with walk_rows (a bit scan per neighbour, the row change only
// where a lane needs it).
template <typename R, typename Visit>
__device__ __forceinline__ void for_masked_rows(const KParams& K, const Segment& g,
                                                const LaneRows& lr, uint4 nm, Visit&& visit) {
  walk_rows(nm.x, nm.y, nm.z, g.lo[0] - g.rs[0] + lr.ta[0], g.lo[1] - g.rs[1] + lr.ta[1],
            g.lo[2] - g.rs[2] + lr.ta[2], (R)row_uy(K, 0), (R)row_uy(K, 1), (R)row_uy(K, 2),
            visit);
}

template <typename R, bool SUM, bool EOS, bool PER>
__global__ __launch_bounds__(PIECE) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 && !PER ? 8 : 1))) void k_density_tiled(St<R> S, KParams K,
                                                       const uint32_t* __restrict__ skey,
                                                       const int* __restrict__ cstart, SegArg sa,
                                                       uint4* __restrict__ nbm) {
  __shared__ struct {
    PreTile<R> P;
    DensTile<R> T;
  } L;
  PreTile<R>& P = L.P;
  DensTile<R>& T = L.T;
  const Segment g = segment_of(sa);
  if (halted(K) || g.O0 >= g.O1) return;
  const Wrap<PER> W(K, g, cstart);
  const bool tiled = g.total + W.total <= tile_cap<R>();
  using Raw = typename DensTile<R>::Raw;
  int id = 0;
  R rho = (R)0;
  for_segment<4, Raw>(
      K, g, W, skey, cstart, tiled,
      [&](int i) {
        id = S.id[i];
        if (EOS) rho = S.rho[i];
      },
      [](int) {},
      [&](int t) { return T.load(S, t); },
      [&](int l, const Raw& r) {
        T.put(l, K, r);
        P.put(l, K, r);
      },
      [&](int i, uint32_t, const LaneRows& lr) {
        if (!tiled) {
          density_direct<R, SUM, EOS, PER>(S, K, i, skey, cstart, nbm);
          return;
        }
        const int self = g.lo[1] + (i - g.rs[1]);
        const auto pi = T.lane(self);
        const auto vi = T.vel(self);
        DensOwn<R> o;
        dens_begin<R, SUM>(K, o);
        uint32_t rm[3] = {0u, 0u, 0u};
        bool ok = true;
        dens_walk<R, SUM>(K, g, lr, T, P, pi, vi, i, o, rm, &ok);
        for_wrapped<R>(K, W, T, lr.cx, pi, [&](int l, R dx, R dy, R r2) {
          const auto vj = T.vel(l);
          dens_pair<R, SUM>(K, dx, dy, r2, vi.x - vj.x, vi.y - vj.y, o.sum, o.rs);
        });
        nbm[i] = make_uint4(rm[0], rm[1], rm[2], ok ? 1u : 0u);
        dens_end<R, SUM, EOS>(S, K, i, o, id, rho);
      },
      [](int, bool) {});
}

template <typename R, bool PER>
__global__ __launch_bounds__(PIECE) void k_tensor_tiled(St<R> S, KParams K,
                                                      const uint32_t* __restrict__ skey,
                                                      const int* __restrict__ cstart, SegArg sa,
                                                      const uint4* __restrict__ nbm) {
  __shared__ TensTile<R> T;
  const Segment g = segment_of(sa);
  if (halted(K) || g.O0 >= g.O1) return;
  const Wrap<PER> W(K, g, cstart);
  const bool tiled = g.total + W.total <= tile_cap<R>();
  using Raw = typename TensTile<R>::Raw;
  uint4 nm;
  for_segment<4, Raw>(
      K, g, W, skey, cstart, tiled,
      [&](int i) {
        nm = nbm[i];
        if (!sa.masks) nm.w = 0u;
      },
      [](int) {},
      [&](int t) { return T.load(S, t); }, [&](int l, const Raw& r) { T.put(l, K, r); },
      [&](int i, uint32_t, const LaneRows& lr) {
        if (!tiled) {
          tensor_direct<R, PER>(S, K, i, skey, cstart);
          return;
        }
        const int self = g.lo[1] + (i - g.rs[1]);
        const auto pi = T.lane(self);
        const auto vi = T.d.vel(self);
        TensOwn<R> o;
        auto pair = [&](int l, R dx, R dy, R r2) {
          const auto vj = T.d.vel(l);
          tens_pair(K, o, dx, dy, r2, vj.x - vi.x, vj.y - vi.y, T.q[l]);
        };
        auto visit = [&](int l, R uy) {
          R dx, dy;
          T.delta(K, pi, l, uy, dx, dy);
          pair(l, dx, dy, dx * dx + dy * dy);
        };
        if (nm.w && sizeof(R) == 4)
          for_masked_rows<R>(K, g, lr, nm, visit);
        else if (nm.w)
          for_masked<R>(K, g, lr, nm, visit);
        else
          for_neighbours<R>(K, g, lr, T, pi, i, visit);
        for_wrapped<R>(K, W, T, lr.cx, pi, pair);
        tens_end(S, K, i, T.q[self], o);
      },
      [](int, bool) {});
}

// With M.its the workgroup also moves its particles (move_particle): the rates
// are in registers and the corrector's own values were read beside the tile, so
// the pass that read them back (14.8 us of a 115 us step of 720,000 FP32
// particles, 4.4 of 41 us with 1,972 in FP64) costs a store.
// PC: pa_sph and same_e2 fixed at compile time for the FP32 pair body
// (force_pair_f32), -1 to read them from K (k_force_hot fixes them).
template <typename R, bool PRESS, bool AV, bool AH, bool XS, bool VI, bool PER, int PC = -1>
__global__ __launch_bounds__(PIECE) void k_force_tiled(St<R> S, KParams K,
                                                     const uint32_t* __restrict__ skey,
                                                     const int* __restrict__ cstart, SegArg sa,
                                                     const uint4* __restrict__ nbm, Moved<R> M) {
  __shared__ ForceTile<R, VI> T;
  const Segment g = segment_of(sa);
  if (halted(K) || g.O0 >= g.O1) return;
  const Wrap<PER> W(K, g, cstart);
  const bool tiled = g.total + W.total <= tile_cap<R, VI>();
  using Raw = typename ForceTile<R, VI>::Raw;
  uint4 nm;
  int id = 0;
  MoveIn<R> m;
  Rates<R> rates;
  for_segment<VI ? 3 : 4, Raw>(
      K, g, W, skey, cstart, tiled,
      [&](int i) {
        nm = nbm[i];
        if (!sa.masks) nm.w = 0u;
        if (PRESS) id = S.id[i];
      },
      [&](int i) {
        if (PRESS && M.its) m = move_load(S, K, M.its, i, id);
      },
      [&](int t) { return T.load(S, t); }, [&](int l, const Raw& r) { T.put(l, K, r); },
      [&](int i, uint32_t, const LaneRows& lr) {
        if (!tiled) {
          rates = force_direct<R, PRESS, AV, AH, XS, VI, PER>(S, K, i, skey, cstart);
          return;
        }
        const int self = g.lo[1] + (i - g.rs[1]);
        const auto pi = T.lane(self);
        ForceOwn<R> o;
        T.own(S, K, o, i, self);
        auto pair = [&](int l, R dx, R dy, R r2) {
          T.template pair<PRESS, AV, AH, XS, PC>(K, o, l, dx, dy, r2);
        };
        auto visit = [&](int l, R uy) {
          R dx, dy;
          T.delta(K, pi, l, uy, dx, dy);
          pair(l, dx, dy, dx * dx + dy * dy);
        };
        if (nm.w && sizeof(R) == 4)
          for_masked_rows<R>(K, g, lr, nm, visit);  // the row-refill walk
        else if (nm.w)
          for_masked<R>(K, g, lr, nm, visit);  // FP64 (walk_rows measured 0.6 % slower here)
        else
          for_neighbours<R>(K, g, lr, T, pi, i, visit);
        for_wrapped<R>(K, W, T, lr.cx, pi, pair);
        rates = force_end<R, PRESS, XS, VI>(S, K, i, o, id);
      },
      [&](int i, bool on) {
        if (PRESS && M.its) {
          if (!XS && on) S.av[i] = {};  // no XSPH: zero, as the host's fill leaves it
          move_particle(K, M, on, i, id, m, rates);
        }
      });
}

// ---- the hot FP32 force gather ---------------------------------------------
// The dam-break flag set (pressure, artificial viscosity and heat, XSPH, no
// physical viscosity, x not periodic) with pa_sph and same_e2 fixed at
// compile time (PC), on row pieces, with 32-byte records: the record's cell
// column is not staged.  For a neighbour in row k of a lane in cell column
// cx, (cx_i - cx_j) cell is +cell, 0 or -cell as the neighbour's tile entry
// lies before the row's cell cx, in it, or after it (e1_k, e2_k: the entries
// where cells cx and cx+1 start), the exact value the FP32 delta computes.
// The smaller tile lets eight workgroups share a CU.  Particles without
// complete masks take the direct path.
struct HotForceTile {
  static constexpr int CAP = GAP_RECORDS;
  float4 a[CAP];  // offx, offy, vx, vy
  float4 b[CAP];  // Q = 1/rho, A = p/rho, psi, u
  struct Raw {
    float2 o, v;
    float rho, p, psi, u;
  };
  static __device__ __forceinline__ Raw load(const St<float>& S, int t) {
    return {S.off[t], S.v[t], S.rho[t], S.p[t], S.psi[t], S.uf[t]};
  }
  __device__ __forceinline__ void put(int l, const KParams& K, const Raw& r) {
    a[l] = make_float4(r.o.x, r.o.y, r.v.x, r.v.y);
    float Q, A;
    q_and_a(K, r.rho, r.p, Q, A);
    b[l] = make_float4(Q, A, r.psi, r.u);
  }
};

// A row of the hot walk: first tile entry of the lane's three cells, the
// entries where cells cx and cx+1 start, the row's cell-row term.
struct HotRow {
  int base, e1, e2;
  float uy;
};

// walk_rows two neighbours at a time, with the rows' cell boundaries:
// visit(la, ra, lb, rb, hb) with lb the next neighbour after la in the same
// order when hb (else lb = la, to be ignored), so that the pair arithmetic
// of two neighbours can overlap.
template <typename Visit2>
__device__ __forceinline__ void walk_rows2_hot(uint32_t m0, uint32_t m1, uint32_t m2, HotRow r0,
                                               HotRow r1, HotRow r2, Visit2&& visit) {
  uint32_t m = m0;
  HotRow r = r0;
  auto refill = [&]() {
    const bool t1 = m1 != 0u;
    m = t1 ? m1 : m2;
    r.base = t1 ? r1.base : r2.base;
    r.e1 = t1 ? r1.e1 : r2.e1;
    r.e2 = t1 ? r1.e2 : r2.e2;
    r.uy = t1 ? r1.uy : r2.uy;
    m1 = t1 ? m2 : 0u;
    r1 = r2;
    m2 = 0u;
  };
  while (true) {
    if (m == 0u) {
      refill();
      if (m == 0u) break;
    }
    const int la = r.base + (int)__builtin_ctz(m);
    const HotRow ra = r;
    m &= m - 1u;
    if (m == 0u) refill();
    const bool hb = m != 0u;
    const int lb = hb ? r.base + (int)__builtin_ctz(m) : la;
    HotRow rb;
    rb.e1 = hb ? r.e1 : ra.e1;
    rb.e2 = hb ? r.e2 : ra.e2;
    rb.uy = hb ? r.uy : ra.uy;
    m = hb ? (m & (m - 1u)) : m;
    visit(la, ra, lb, rb, hb);
  }
}

template <int PC>
__global__ __launch_bounds__(PIECE) __attribute__((amdgpu_waves_per_eu(4))) void k_force_hot(
    St<float> S, KParams K, const uint32_t* __restrict__ skey, const int* __restrict__ cstart,
    SegArg sa, const uint4* __restrict__ nbm, Moved<float> M) {
  __shared__ HotForceTile T;
  const Segment g = segment_of(sa);
  if (halted(K) || g.O0 >= g.O1) return;
  const bool tiled = g.total <= HotForceTile::CAP;
  const int i = g.O0 + (int)threadIdx.x;
  const int ic = min(i, g.O1 - 1);
  const uint32_t key = skey[ic];
  const int id = S.id[ic];
  using Raw = HotForceTile::Raw;
  Stage<4, Raw> st;  // as for_segment
  auto ld = [&](int t) { return T.load(S, t); };
  auto pt = [&](int l, const Raw& r) { T.put(l, K, r); };
  st.load(g, 0, ld);
  const int cx = (int)key - g.cy * K.nx;
  const uint4 nm = nbm[ic];
  HotRow rw[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int d = g.lo[k] - g.rs[k];
    const int* e = cstart + (g.cy - 1 + (g.rl[k] ? k : 1)) * K.nx;  // an empty row has no mask
    rw[k].base = d + e[cx > 0 ? cx - 1 : 0];
    rw[k].e1 = d + e[cx];
    rw[k].e2 = d + e[cx + 1];
    rw[k].uy = row_uy(K, k);
  }
  MoveIn<float> m;
  if (M.its) m = move_load(S, K, M.its, ic, id);
  if (tiled) {
    st.put(g, 0, pt);
    stage_rest<4, Raw>(g, Wrap<false>(K, g, cstart), ld, pt);
  }
  __syncthreads();
  Rates<float> rates;
  const bool on = i < g.O1;
  if (on && (!tiled || !nm.w || !sa.masks)) {
    rates = force_direct<float, true, true, true, true, false, false>(S, K, i, skey, cstart);
  } else if (on) {
    const int self = g.lo[1] + (i - g.rs[1]);
    const float4 qs = T.a[self];
    const float4 ws = T.b[self];
    ForceOwn<float> o;
    o.v = make_float2(qs.z, qs.w);
    o.Q = ws.x;
    o.A = ws.y;
    o.psi = ws.z;
    o.u = ws.w;
    own_factors_f32(K, o);
    const float cellf = K.cellf;
    auto terms = [&](int l, const HotRow& r) {
      const float4 q = T.a[l];
      const float4 w = T.b[l];
      const float ux = l < r.e1 ? cellf : (l < r.e2 ? 0.f : -cellf);
      const float tx = qs.x - q.x;
      const float dx = tx + ux;
      const float ty = qs.y - q.y;
      const float dy = ty + r.uy;
      return force_terms_f32<true, true, true, true, PC>(K, o, dx, dy, q.z, q.w, w.x, w.y, w.z,
                                                         w.w);
    };
    // two neighbours per step; each added in walk order
    walk_rows2_hot(nm.x, nm.y, nm.z, rw[0], rw[1], rw[2],
                   [&](int la, const HotRow& ra, int lb, const HotRow& rb, bool hb) {
                     const TermsF ta = terms(la, ra);
                     const TermsF tb = terms(lb, rb);
                     force_acc_f32<true, true, true, true>(o, ta, true);
                     // without a second neighbour G and wf are zeroed (adding
                     // -0 dx to a sum that is never -0 leaves its bits), the
                     // energy rate is skipped
                     const float gb = hb ? tb.G : 0.f, wb = hb ? tb.wf : 0.f;
                     o.fx = __builtin_fmaf(-gb, tb.dx, o.fx);
                     o.fy = __builtin_fmaf(-gb, tb.dy, o.fy);
                     o.du.add_if(tb.d, hb);
                     o.xsx = __builtin_fmaf(-wb, tb.dvx, o.xsx);
                     o.xsy = __builtin_fmaf(-wb, tb.dvy, o.xsy);
                   });
    rates = force_end<float, true, true, false>(S, K, i, o, id);
  }
  if (M.its) move_particle(K, M, on, i, id, m, rates);
}

}  // namespace arm
