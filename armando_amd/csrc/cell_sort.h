// cell_sort.h -- counting sort of particles into hash cells for gfx950.
//
// Produces the same (cell, id) order as a stable sort of the cell keys
// listed in id order, and the cell ranges as a by-product:
//   emit_key        (in the kernels that hash positions) key_by_slot[t] and
//                   count[key] += run, where a run is a group of adjacent
//                   lanes of a wavefront with the same key: one atomic per
//                   run; in sorted order most of a cell is one run
//   k_cs_scan1      exclusive scan of the counts -> cell_start[0 .. ncell]
//                   in one launch (each workgroup publishes its tile's sum
//                   and adds up those of the tiles before its own); the
//                   two-launch form k_cs_tile_sum + k_cs_tile_scan serves the
//                   allocation-free entry point and the ghost numbering
//   k_cs_scatter    every particle takes a place in its cell range (count[key]
//                   -= run restores the counters to zero); the order inside a
//                   cell is arbitrary here
//   Order::place    every particle counts the ids of its cell below its own:
//                   that rank is its place in (cell, id) order (in the reorder
//                   kernels, or in k_cs_rank)
// The counters must be zero before the keys are emitted (k_cs_zero) and are
// zero again after the scatter.  Grids of
// up to CS_TILE * CS_MAX_TILES cells are handled.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace arm {

constexpr int CS_THREADS = 256;
constexpr int CS_PER_LANE = 8;
constexpr int CS_TILE = CS_THREADS * CS_PER_LANE;  // cells per scan tile
constexpr int CS_MAX_TILES = 4096;

// Runs of equal keys in adjacent lanes of a wavefront.  All 64 lanes must
// call it.  head: first lane of its run; len: run length (valid on heads);
// hl: the head lane of this lane's run; rank: lane - hl.
struct WaveRun {
  bool head;
  int len, hl, rank;
};

__device__ __forceinline__ WaveRun wave_run(uint32_t c, bool valid) {
  const int lane = threadIdx.x & 63;
  const uint32_t prev = __shfl_up(c, 1, 64);
  const bool head = valid && (lane == 0 || prev != c);
  const uint64_t hb = __ballot(head || !valid);
  const uint64_t after = lane == 63 ? 0ull : (hb >> (lane + 1));
  const int next = after ? lane + 1 + __builtin_ctzll(after) : 64;
  const uint64_t upto = lane == 63 ? hb : (hb & ((2ull << lane) - 1ull));
  WaveRun r;
  r.head = head;
  r.len = next - lane;
  r.hl = upto ? 63 - __builtin_clzll(upto) : lane;
  r.rank = lane - r.hl;
  return r;
}

// Where the hashing kernels put the keys: indexed by id for the radix sort,
// by slot (plus the per-cell counts) for the counting sort.
struct KeyOut {
  uint32_t* key_by_id;
  uint32_t* slot_by_id;
  uint32_t* key_by_slot;
  int* count;
};

// Stores the key of slot t (particle id); nothing when every pointer of ko
// is null.  All 64 lanes of the wavefront must call it; lanes with
// valid = false only take part in the ballots.
__device__ __forceinline__ void emit_key(const KeyOut& ko, bool valid, int t, int id,
                                         uint32_t key) {
  if (ko.key_by_slot) {
    const WaveRun r = wave_run(key, valid);
    if (valid) ko.key_by_slot[t] = key;
    if (r.head) atomicAdd(&ko.count[key], r.len);
  } else if (ko.key_by_id && valid) {
    ko.key_by_id[id] = key;
    ko.slot_by_id[id] = (uint32_t)t;
  }
}

// The fused steps' halt word (see KParams::halt): the sort of step its does
// nothing once an earlier launch recorded a failure at or before its.
struct Halt {
  const int* word = nullptr;
  int its = 0;
  __device__ __forceinline__ bool on() const {
    if (!word) return false;
    const int h = *word;
    return h != 0 && its >= h;
  }
};

// Clears the per-cell counters (a fill kernel, so that it may be captured).
__global__ __launch_bounds__(CS_THREADS) void k_cs_zero(int* __restrict__ count, int ncell) {
  for (int c = blockIdx.x * CS_THREADS + threadIdx.x; c < ncell; c += gridDim.x * CS_THREADS)
    count[c] = 0;
}

// Exclusive scan of one value per lane across the workgroup (LDS, one
// wavefront-sized partial per wavefront).  Returns the lane's exclusive
// prefix; *total receives the workgroup sum.
template <int THREADS>
__device__ __forceinline__ int block_exclusive_scan(int v, int* __restrict__ wsum, int* total) {
  constexpr int NW = THREADS / 64;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  if (w == 0) {
    int s = lane < NW ? wsum[lane] : 0;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(s, d, 64);
      if (lane >= d) s += y;
    }
    if (lane < NW) wsum[lane] = s;  // inclusive prefix of the wavefront sums
  }
  __syncthreads();
  const int before = w > 0 ? wsum[w - 1] : 0;
  *total = wsum[NW - 1];
  return before + x - v;
}

// The CS_PER_LANE consecutive counters of a lane (zero past n): two 16-byte
// loads where the run lies inside the array (p comes from hipMalloc and c0
// is a multiple of CS_PER_LANE, so the loads are aligned).
static_assert(CS_PER_LANE == 8, "load8/store8 move eight counters");
__device__ __forceinline__ void load8(const int* __restrict__ p, int c0, int n, int* v) {
  if (c0 + 8 <= n) {
    const int4 a = *reinterpret_cast<const int4*>(p + c0);
    const int4 b = *reinterpret_cast<const int4*>(p + c0 + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
    v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = (c0 + k < n) ? p[c0 + k] : 0;
  }
}

__device__ __forceinline__ void store8(int* __restrict__ p, int c0, int n, const int* v) {
  if (c0 + 8 <= n) {
    *reinterpret_cast<int4*>(p + c0) = make_int4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<int4*>(p + c0 + 4) = make_int4(v[4], v[5], v[6], v[7]);
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (c0 + k < n) p[c0 + k] = v[k];
  }
}

__global__ __launch_bounds__(CS_THREADS) void k_cs_tile_sum(const int* __restrict__ count,
                                                            int ncell, int* __restrict__ tsum,
                                                            Halt hl) {
  if (hl.on()) return;
  __shared__ int wsum[CS_THREADS / 64];
  const int c0 = blockIdx.x * CS_TILE + threadIdx.x * CS_PER_LANE;
  int v[CS_PER_LANE];
  load8(count, c0, ncell, v);
  int s = 0;
#pragma unroll
  for (int k = 0; k < CS_PER_LANE; ++k) s += v[k];
  int total;
  block_exclusive_scan<CS_THREADS>(s, wsum, &total);
  if (threadIdx.x == 0) tsum[blockIdx.x] = total;
}

__global__ __launch_bounds__(CS_THREADS) void k_cs_tile_scan(const int* __restrict__ count,
                                                             int ncell, int n,
                                                             const int* __restrict__ tsum,
                                                             int* __restrict__ cstart, Halt hl) {
  if (hl.on()) return;
  __shared__ int wsum[CS_THREADS / 64];
  const int c0 = blockIdx.x * CS_TILE + threadIdx.x * CS_PER_LANE;
  int v[CS_PER_LANE];
  load8(count, c0, ncell, v);
  int s = 0;
#pragma unroll
  for (int k = 0; k < CS_PER_LANE; ++k) s += v[k];
  int part = 0;
  for (int j = threadIdx.x; j < (int)blockIdx.x; j += CS_THREADS) part += tsum[j];
  int base;
  block_exclusive_scan<CS_THREADS>(part, wsum, &base);
  __syncthreads();  // wsum is reused
  int total;
  int run = base + block_exclusive_scan<CS_THREADS>(s, wsum, &total);
  int o[CS_PER_LANE];
#pragma unroll
  for (int k = 0; k < CS_PER_LANE; ++k) {
    o[k] = run;
    run += v[k];
  }
  store8(cstart, c0, ncell, o);
  if (blockIdx.x == 0 && threadIdx.x == 0) cstart[ncell] = n;
}

// ---- single-pass scan -----------------------------------------------------
// k_cs_scan1 does the work of k_cs_tile_sum and k_cs_tile_scan in one launch:
// each workgroup publishes its tile's sum in a status word, then adds up the
// words of all the tiles before its own, read by all its lanes at once (the
// grid's workgroups run together, so the words are there within a few
// microseconds).  A word is (epoch << 32) | sum; a word of another epoch (an
// earlier sort) reads as not yet published.  The host gives every sort a new
// epoch (1 .. SCAN_EPOCH_MAX), so the words need no clearing between sorts;
// a launch replayed with the same epoch (a captured graph) would read the
// previous replay's words, so the allocation-free entry point, which a
// caller may capture, keeps the two-launch scan.
constexpr uint32_t SCAN_EPOCH_MAX = 0xffffffffu;  // the host clears the words and restarts at 1
constexpr int SCAN_SPIN_LIMIT = 1 << 14;

__global__ __launch_bounds__(CS_THREADS) void k_cs_scan1(const int* __restrict__ count, int ncell,
                                                         int n, int* __restrict__ cstart,
                                                         uint64_t* __restrict__ tstat,
                                                         uint32_t epoch, Halt hl) {
  if (hl.on()) return;
  __shared__ int wsum[CS_THREADS / 64];
  const int b = blockIdx.x;
  const int c0 = b * CS_TILE + threadIdx.x * CS_PER_LANE;
  int v[CS_PER_LANE];
  load8(count, c0, ncell, v);
  int s = 0;
#pragma unroll
  for (int k = 0; k < CS_PER_LANE; ++k) s += v[k];
  int total;
  const int pre = block_exclusive_scan<CS_THREADS>(s, wsum, &total);
  if (threadIdx.x == 0)
    __hip_atomic_store(&tstat[b], ((uint64_t)epoch << 32) | (uint32_t)total, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  // the sums of tiles 0 .. b-1; re-read while one is missing, and after
  // SCAN_SPIN_LIMIT rounds add up their counters instead (slower, the same)
  int part = 0;
  bool ready = false;
  for (int spins = 0; !ready && spins < SCAN_SPIN_LIMIT; ++spins) {
    part = 0;
    bool miss = false;
    for (int q = threadIdx.x; q < b; q += CS_THREADS) {
      const uint64_t w = __hip_atomic_load(&tstat[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      miss = miss || (uint32_t)(w >> 32) != epoch;
      part += (int)(uint32_t)w;
    }
    ready = !__syncthreads_or(miss);
  }
  if (!ready) {
    part = 0;
    for (int c = threadIdx.x; c < min(b * CS_TILE, ncell); c += CS_THREADS) part += count[c];
  }
  __syncthreads();  // wsum is reused
  int excl;
  block_exclusive_scan<CS_THREADS>(part, wsum, &excl);
  int run = excl + pre;
  int o[CS_PER_LANE];
#pragma unroll
  for (int k = 0; k < CS_PER_LANE; ++k) {
    o[k] = run;
    run += v[k];
  }
  store8(cstart, c0, ncell, o);
  if (b == 0 && threadIdx.x == 0) cstart[ncell] = n;
}

// Pieces of the cell rows, for the gathers that give each workgroup a run of
// consecutive sorted positions of one row: the sorted range of row y,
// [cstart[y nx], cstart[(y+1) nx]), cut into runs of PIECE positions from its
// start (the last one shorter).  tab[b] is all that workgroup b of a gather
// needs to begin: its particles [O0, O1) of row cy and the three ranges of
// sorted positions that hold their candidates, so that one load stands
// between the launch and the filling of the tile (a chain of five before, a
// microsecond each for every workgroup).
//
// Above a tank's free surface a row holds wall particles on either side only,
// and the row below everything between them, so that a piece over the gap needs
// more records than a gather's tile holds and its workgroup runs on the direct
// path, as long as a whole launch of the others (FP32 force of the
// 111,119-particle dam break: 28.6 us, 12.8 without; density 20.5 and 14.5).  A
// piece of more than GAP_SPAN cells whose three rows hold more than GAP_RECORDS
// particles is therefore cut at the middle of its cells, at most one of each row.
//
// The pieces of all rows come first, in row order, dealt so that the workgroups of
// one XCD take one contiguous share (neighbouring pieces, which stage the same rows,
// then share an L2); then a place for the part cut off, of every row that with its
// neighbours holds more than GAP_RECORDS particles (empty if none is); the rest of the table
// is empty.  The host bounds the places by n / PIECE + min(ny, n) +
// min(ny, 3 n / GAP_RECORDS) (piece_slots).  (The cut parts' places behind their row's
// own pieces left empty workgroups among the others, and CUs with one more than
// the rest: force of 100,000 particles, FP64, h = 2 dx, 143 -> 150 us.)
constexpr int PIECE = 128;
constexpr int GAP_SPAN = 40;      // a full piece of 2h cells spans about 20
constexpr int GAP_RECORDS = 592;  // the records of a gather's tile
struct alignas(16) PieceRec {
  int O0, O1, cy, total;  // total = rl[0] + rl[1] + rl[2]
  int rs[3], rl[3];       // sorted start and length of rows cy-1, cy, cy+1
  int x0, x1;             // cells of its first and last particle
};
// sums[c]: of rows ROW_CHUNK c .. the pieces and, from bit 32, the parts' places
// (row_sums_block)
struct RowPieces {
  PieceRec* tab = nullptr;
  uint64_t* sums = nullptr;
  int nx = 0, ny = 0, slots = 0;
};
constexpr int ROW_CHUNK = 256;
__host__ __device__ inline int row_chunks(int ny) { return (ny + ROW_CHUNK - 1) / ROW_CHUNK; }
// Bound on the places for n particles.
__host__ inline long long piece_slots(long long n, long long ny) {
  const long long cuts = 3 * n / GAP_RECORDS;
  return (n + PIECE - 1) / PIECE + (ny < n ? ny : n) + (ny < cuts ? ny : cuts);
}

// A row's sorted range, its pieces and whether a part may be cut off one.
struct RowCount {
  int a, b;
  int pieces, parts;
  __device__ __forceinline__ uint64_t both() const {
    return (uint64_t)pieces | ((uint64_t)parts << 32);
  }
};
__device__ __forceinline__ RowCount row_count(const int* __restrict__ cstart, const RowPieces& rp,
                                              int y) {
  RowCount r;
  r.a = cstart[y * rp.nx];
  r.b = cstart[(y + 1) * rp.nx];
  const int lo = cstart[max(y - 1, 0) * rp.nx], hi = cstart[min(y + 2, rp.ny) * rp.nx];
  r.pieces = (r.b - r.a + PIECE - 1) / PIECE;
  r.parts = r.pieces && hi - lo > GAP_RECORDS ? 1 : 0;
  return r;
}

// The sum of v over the wavefront, in every lane.
__device__ __forceinline__ uint64_t wave_sum(uint64_t v) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// The workgroup that takes logical block L of count: workgroup b runs on XCD
// b mod 8, and XCD x takes the x-th contiguous share of the blocks.
__device__ __forceinline__ int share_slot(int count, int L) {
  constexpr int X = 8;
  const int q = count / X, r = count - q * X;
  if (L < r * (q + 1)) return (L % (q + 1)) * X + L / (q + 1);
  const int m = L - r * (q + 1);
  return (m % q) * X + r + m / q;
}

// What the ROW_CHUNK rows of chunk c add up to, one lane per row.  They are added
// up before the table is made (beside the scatter), so that a workgroup of
// row_pieces_block reads its chunk's rows and a word for each other chunk: with
// every workgroup counting every row, ny^2 / 2 loads, the reorder of 2,400 particles
// in 60,000 rows took 2,283 us (24 now; 8 in 48 rows of as many cells in all), that
// of 1.2 million in 12,510 rows 154 us (39).
template <int THREADS>
__device__ __forceinline__ void row_sums_block(const int* __restrict__ cstart, const RowPieces& rp,
                                               int c) {
  static_assert(THREADS == ROW_CHUNK, "one lane per row");
  __shared__ uint64_t part[THREADS / 64];
  const int y = c * ROW_CHUNK + (int)threadIdx.x;
  const uint64_t v = wave_sum(y < rp.ny ? row_count(cstart, rp, y).both() : 0);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t total = 0;
    for (int w = 0; w < THREADS / 64; ++w) total += part[w];
    rp.sums[c] = total;
  }
}

// The scattered entries: id and slot of the particle at each position of
// its cell range (two arrays, so that the rank's loop reads 4 bytes per
// entry); entc = its cell.
struct Ent {
  uint32_t* id;
  uint32_t* slot;
};

// Particles in slot order; with id_of null the particle in slot t has id t.
// With row pieces (rp.tab set) the first row_chunks(ny) workgroups add up the
// rows' pieces instead.
__global__ __launch_bounds__(CS_THREADS) void k_cs_scatter(const uint32_t* __restrict__ key_by_slot,
                                                           const int32_t* __restrict__ id_of,
                                                           int n, const int* __restrict__ cstart,
                                                           int* __restrict__ count, Ent ent,
                                                           uint32_t* __restrict__ entc, Halt hl,
                                                           RowPieces rp) {
  if (hl.on()) return;
  const int rc = rp.tab ? row_chunks(rp.ny) : 0;
  if ((int)blockIdx.x < rc) {
    row_sums_block<CS_THREADS>(cstart, rp, blockIdx.x);
    return;
  }
  const int t = ((int)blockIdx.x - rc) * CS_THREADS + threadIdx.x;
  const bool valid = t < n;
  const uint32_t c = valid ? key_by_slot[t] : 0xffffffffu;
  const WaveRun r = wave_run(c, valid);
  int old = 0;
  if (r.head) old = atomicSub(&count[c], r.len);
  old = __shfl(old, r.hl, 64);
  if (!valid) return;
  const int pos = cstart[c] + old - 1 - r.rank;
  ent.id[pos] = id_of ? (uint32_t)id_of[t] : (uint32_t)t;
  ent.slot[pos] = (uint32_t)t;
  entc[pos] = c;
}

// Workgroup wg of a grid of nwg = row_blocks() lists the pieces of its share of
// the rows, one wavefront per row and one lane per piece (a lane that walked a
// row's pieces itself waited for the keys of each in turn: 32 us for a 17 us
// reorder).  rp.sums are those of all chunks, so the table needs neither atomics
// nor a cleared counter.  keys: the cell of every sorted position.
constexpr int ROWS_PER_WG = 4;
constexpr int ROW_WGS = 1024;  // at most; above 4096 rows a wavefront takes several
template <int THREADS>
__device__ __forceinline__ void row_pieces_block(const int* __restrict__ cstart,
                                                 const uint32_t* __restrict__ keys,
                                                 const RowPieces& rp, int wg, int nwg) {
  static_assert(THREADS == 64 * ROWS_PER_WG, "one wavefront per row");
  static_assert(THREADS == ROW_CHUNK, "one lane per row of a chunk");
  __shared__ uint64_t part[2][ROWS_PER_WG];
  const int nx = rp.nx, ny = rp.ny;
  const int per = (ny + nwg * ROWS_PER_WG - 1) / (nwg * ROWS_PER_WG);  // rows of a wavefront
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int y0 = (wg * ROWS_PER_WG + w) * per, y1 = min(y0 + per, ny);
  // the ranges of rows y-1 .. y+1 of the particles [p, e) of row y in cells x0 .. x1
  auto make = [&](int y, int p, int e, int x0, int x1) {
    PieceRec r{};
    const int lo = x0 > 0 ? x0 - 1 : 0, hi = (x1 + 1 < nx ? x1 + 1 : nx - 1) + 1;
    r.O0 = p;
    r.O1 = e;
    r.cy = y;
    r.x0 = x0;
    r.x1 = x1;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int ry = y - 1 + k;
      if (ry >= 0 && ry < ny) {
        r.rs[k] = cstart[ry * nx + lo];
        r.rl[k] = cstart[ry * nx + hi] - r.rs[k];
      }
      r.total += r.rl[k];
    }
    return r;
  };
  // the lane's piece of the 64 from j0 on of row y, and where it would be cut (0: not)
  struct Piece {
    PieceRec rec;
    int m;
  };
  auto piece = [&](int y, const RowCount& row, int j0) {
    Piece q{};
    const int p = row.a + (j0 + lane) * PIECE;
    if (p < row.b) {
      const int e = min(p + PIECE, row.b);
      const int x0 = (int)keys[p] - y * nx, x1 = (int)keys[e - 1] - y * nx;
      q.rec = make(y, p, e, x0, x1);
      if (x1 - x0 > GAP_SPAN && q.rec.total > GAP_RECORDS) {
        const int m = cstart[y * nx + (x0 + x1 + 1) / 2];
        q.m = m > p && m < e ? m : 0;
      }
    }
    return q;
  };
  // the first row's pieces, whose loads run beside the counting
  RowCount row{};
  Piece q{};
  if (y0 < y1) {
    row = row_count(cstart, rp, y0);
    q = piece(y0, row, 0);
  }
  // what comes before the workgroup's first row, and all
  const int first = min(wg * ROWS_PER_WG * per, ny), c0 = first / ROW_CHUNK;
  uint64_t before = 0, all = 0;
  for (int c = threadIdx.x; c < row_chunks(ny); c += THREADS) {
    const uint64_t p = rp.sums[c];
    all += p;
    before += c < c0 ? p : 0;
  }
  const int yc = c0 * ROW_CHUNK + (int)threadIdx.x;
  if (yc < first) before += row_count(cstart, rp, yc).both();
  before = wave_sum(before);
  all = wave_sum(all);
  if (lane == 0) {
    part[0][w] = before;
    part[1][w] = all;
  }
  // ... and between that and the wavefront's
  uint64_t mine = 0;
  for (int y = first + lane; y < min(y0, ny); y += 64) mine += row_count(cstart, rp, y).both();
  mine = wave_sum(mine);
  __syncthreads();
  all = 0;
#pragma unroll
  for (int k = 0; k < ROWS_PER_WG; ++k) {
    mine += part[0][k];
    all += part[1][k];
  }
  const int total = (int)(uint32_t)all;
  int base = (int)(uint32_t)mine, parts = total + (int)(mine >> 32);  // the next places
  PieceRec* slots = rp.tab;
  for (int s = total + (int)(all >> 32) + wg * THREADS + (int)threadIdx.x; s < rp.slots;
       s += nwg * THREADS)
    slots[s] = PieceRec{};
  for (int y = y0; y < y1;) {
    bool found = false;
    for (int j0 = 0; j0 < row.pieces; j0 += 64) {
      if (j0) q = piece(y, row, j0);
      const uint64_t cutters = __ballot(q.m != 0);
      if (cutters && !found) {
        found = true;
        if (lane == __builtin_ctzll(cutters)) {  // rec.total > GAP_RECORDS: the row has the place
          const PieceRec r = q.rec;
          slots[parts] = make(y, q.m, r.O1, (int)keys[q.m] - y * nx, r.x1);
          q.rec = make(y, r.O0, q.m, r.x0, (int)keys[q.m - 1] - y * nx);
        }
      }
      if (row.a + (j0 + lane) * PIECE < row.b) slots[share_slot(total, base + j0 + lane)] = q.rec;
    }
    if (!found && row.parts && lane == 0) slots[parts] = PieceRec{};
    base += row.pieces;
    parts += row.parts;
    if (++y < y1) {
      row = row_count(cstart, rp, y);
      q = piece(y, row, 0);
    }
  }
}

// Where the particle of position p of a scattered cell range goes: its rank
// by id among the cell's entries.  Eight ids are read at a time, so that a cell
// of 2D (7 particles of a 2h cell) waits for memory once and one of 3D (18)
// three times.
__device__ __forceinline__ int cell_rank(const uint32_t* __restrict__ ids,
                                         const int* __restrict__ cstart, uint32_t c, uint32_t id) {
  const int a = cstart[c], b = cstart[c + 1];
  int rank = a;
  for (int q0 = a; q0 < b; q0 += 8) {
    uint32_t o[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = ids[min(q0 + k, b - 1)];
#pragma unroll
    for (int k = 0; k < 8; ++k) rank += (q0 + k < b && o[k] < id) ? 1 : 0;
  }
  return rank;
}

// The order in which a reorder kernel takes the particles: the slot of the
// particle at position p, and where it goes.  After the counting sort's
// scatter ids is set, positions are grouped by cell and every lane ranks its
// own particle (a launch of its own, which reads all this and writes keys and
// slots for the reorder to read back, took 8.6 us of a 124 us step of 720,000
// particles and 3.4 of 42 us with 1,972); the cells of the positions are the
// sorted keys already.  After the radix sort (ids null) the order is final.
struct Order {
  const uint32_t* ids;
  const uint32_t* slot;
  __device__ __forceinline__ int place(const uint32_t* __restrict__ skey,
                                       const int* __restrict__ cstart, int p, int id) const {
    return ids ? cell_rank(ids, cstart, skey[p], (uint32_t)id) : p;
  }
};

// The ranks as a pass of their own, for the entry point that returns the order.
__global__ __launch_bounds__(CS_THREADS) void k_cs_rank(Ent ent, const uint32_t* __restrict__ entc,
                                                        int n, const int* __restrict__ cstart,
                                                        uint32_t* __restrict__ skey,
                                                        uint32_t* __restrict__ sval) {
  const int p = blockIdx.x * CS_THREADS + threadIdx.x;
  if (p >= n) return;
  const uint32_t c = entc[p];
  const int t = cell_rank(ent.id, cstart, c, ent.id[p]);
  skey[t] = c;
  sval[t] = ent.slot[p];
}

}  // namespace arm
