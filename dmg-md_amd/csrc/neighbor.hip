// neighbor.hip -- Verlet-list build for gfx950 with a device-side rebuild
// decision.
//
// Every kernel of the rebuild is launched every step and returns at once
// unless the device flag flags[kFlagRebuild] is set (by the displacement
// check in k_pack or by the host for a first call / box change).  The host
// therefore never has to read the decision back: a whole MD chunk is enqueued
// without a synchronisation.  Behaviour follows the reference's Neighbor
// class (neighbor.cu:90-134 cell list, :141-218 rows, :446-582 skin policy,
// neighbor.cuh:133-196 row order): rows hold every slot j != i with FP64
// d^2 < (rc + skin)^2, sorted ascending by slot (or by global id), plus the
// position of the centre inside each neighbour's row.
//
// Layout: rows are row-major (vl[i*MV + p]) so that a group of lanes that
// works on one centre reads and writes contiguous memory.  Build and sort run
// with kRowLanes lanes per centre (4 centres per wave), the reverse search
// with kRowLanes or, in small systems, a wavefront.
#include <algorithm>
#include <limits>
#include <type_traits>
#include "device_common.hpp"
#include "nep_math.hpp"

namespace dmgx {

namespace {

constexpr int kRowLanes = 16;  // lanes cooperating on one Verlet row
constexpr int kScanCells = 4096;  // cells per workgroup of the scan (one row of cells at least)

__global__ void k_set_flag(int* __restrict__ flag, int value) { *flag = value; }

__global__ void k_clear_moved(const int* __restrict__ go, ImageMap m)
{
  if (!*go) return;
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r < m.n_req) m.req_moved[r] = 0;
}

__global__ void k_clear_ints(int* __restrict__ p, long long n)
{
  for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < n; k += (long long)gridDim.x * blockDim.x)
    p[k] = 0;
}

// Per-step packing of positions and types into one 32-byte record per atom
// (x, y, z, type bits) so that every neighbour gather is a single 32-byte
// access; also validates the types and, unless a rebuild is forced, tests
// whether any atom moved more than skin/2 since the last rebuild
// (neighbor.cu:446-490).
__global__ __launch_bounds__(kBlock) void k_pack(DevBox b, int N, int T, const double* __restrict__ pos,
                                                 const int* __restrict__ type, const double* __restrict__ x0,
                                                 double lim2, int forced, double4* __restrict__ xq,
                                                 int* __restrict__ flags, ImageMap m)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (forced && i == 0) flags[kFlagRebuild] = kRebuildAsked | kRebuildAll;
  bool moved = false, bad = false;
  if (i < N) {
    const double x = pos[i], y = pos[N + i], z = pos[2 * N + i];
    const int t = type[i];
    bad = t < 0 || t >= T;
    xq[i] = make_double4(x, y, z, __longlong_as_double((long long)t));
    if (!forced) {
      double dx = x - x0[i], dy = y - x0[N + i], dz = z - x0[2 * N + i];
      mic(b, dx, dy, dz);
      moved = !(dist2(dx, dy, dz) <= lim2);  // NaN displacements request a rebuild too
      if (moved && m.slot_req) m.req_moved[m.slot_req[i < m.n_owned ? i : m.owner[i]]] = 1;
    }
  }
  const bool lead = (threadIdx.x & 63) == 0;
  if (__any(moved) && lead) atomicOr(&flags[kFlagRebuild], kRebuildAsked);
  if (__any(bad) && lead) atomicOr(&flags[kFlagBadType], 1);
}

// cell of every atom, its rank inside the cell, and the positions the next
// displacement checks compare against (for the slots in [a1, b1) and
// [a2, b2) whose rows this rebuild makes)
// With compacted lists (a rebuild of some requests of a batch) only the
// listed slots enter the cell list: every row it makes holds slots of its
// own request only.
__global__ void k_cell_count(const int* __restrict__ go, DevBox b, int N, const double4* __restrict__ xq,
                             int row_shift, int* __restrict__ cell_of, int* __restrict__ rank,
                             int* __restrict__ count, int* __restrict__ cursor, double* __restrict__ x0, int a1, int b1,
                             int a2, int b2, int* __restrict__ flags, ImageMap m)
{
  const int g = *go;
  if (!g) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) *cursor = 0;
  const bool listed = rebuild_listed(m);
  const int n = listed ? m.req_off[2 * m.n_req + 1] : N;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    const int i = listed ? m.lists[m.n_owned + k] : k;
    const double4 p = xq[i];
    int c[3];
    if (!cell_coords(b, p.x, p.y, p.z, c)) atomicOr(&flags[kFlagOutOfBox], 1);
    const int row = c[1] + b.nc[1] * c[2], id = c[0] + b.nc[0] * row;
    cell_of[i] = id + (row >> row_shift);  // where the scan keeps the cell's start
    rank[i] = atomicAdd(&count[id], 1);
    if (((i >= a1 && i < b1) || (i >= a2 && i < b2)) && (listed || slot_rebuilt(m, g, i))) {
      x0[i] = p.x;
      x0[N + i] = p.y;
      x0[2 * N + i] = p.z;
    }
  }
}

// Starts of the cells in cell_atoms.  A range of candidates runs along one row
// of cells, so only the cells of a row need consecutive atoms: each workgroup
// scans 2^row_shift whole rows (tile_cells cells) by itself, takes its place
// in cell_atoms from the cursor, and clears the counts for the next rebuild.
// A tile's starts are followed by its end: cell c of row r has its start at
// c + (r >> row_shift), and the next entry is the cell's end.  Bound by its
// own latency: 213,000 cells 49 -> 6.1 us against passes of one workgroup.
__global__ __launch_bounds__(1024) void k_cell_starts(const int* __restrict__ go, int ncell, int tile_cells,
                                                      int* __restrict__ count, int* __restrict__ start,
                                                      int* __restrict__ cursor)
{
  if (!*go) return;
  __shared__ int wsum[2][16];
  __shared__ int place;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = min(tile_cells, ncell - (int)blockIdx.x * tile_cells);
  int* in = count + (size_t)blockIdx.x * tile_cells;
  int* out = start + (size_t)blockIdx.x * (tile_cells + 1);
  int v[4], sum = 0;
  auto load = [&](int base) {
    sum = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = base + 4 * threadIdx.x + q;
      v[q] = k < n ? in[k] : 0;
      sum += v[q];
    }
  };
  // sum before this thread, and of the workgroup
  int flip = 0;
  auto scan = [&](int* total) {
    int x = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(x, off, 64);
      if (lane >= off) x += y;
    }
    flip ^= 1;
    if (lane == 63) wsum[flip][wave] = x;
    __syncthreads();
    int before = x - sum;
    *total = 0;
    for (int q = 0; q < 16; ++q) {
      if (q < wave) before += wsum[flip][q];
      *total += wsum[flip][q];
    }
    return before;
  };
  int all = 0, before = 0;
  for (int base = 0; base < n; base += kScanCells) {
    load(base);
    int t;
    before = scan(&t);
    all += t;
  }
  if (threadIdx.x == 0) place = atomicAdd(cursor, all);
  __syncthreads();
  int run = place;
  for (int base = 0; base < n; base += kScanCells) {
    if (n > kScanCells) {  // a row longer than the tile: its counts again
      int t;
      load(base);
      before = scan(&t);
      before += run;
      run += t;
    } else {
      before += run;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = base + 4 * threadIdx.x + q;
      if (k < n) {
        out[k] = before;
        in[k] = 0;
      }
      before += v[q];
    }
  }
  if (threadIdx.x == 0) out[n] = place + all;
}

// Count, scan and fill of a small system by one workgroup, with the cells in
// LDS: one launch instead of three, in a rebuild and in every step without
// one.  Bound by what one CU loads and stores (2.4 us per 1,000 atoms).
constexpr int kOneBlockIdBits = 14;
__global__ __launch_bounds__(1024) void k_cells_one_block(const int* __restrict__ go, DevBox b, int N, int ncell,
                                                          const double4* __restrict__ xq, int* __restrict__ cell_of,
                                                          int* __restrict__ start, double* __restrict__ x0, int a1,
                                                          int b1, int a2, int b2, int* __restrict__ flags,
                                                          int* __restrict__ atoms, double4* __restrict__ xs, ImageMap m)
{
  const int g = *go;
  if (!g) return;
  extern __shared__ int cells[];
  __shared__ int wsum[16];
  for (int k = threadIdx.x; k < ncell; k += 1024) cells[k] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < N; i += 1024) {
    const double4 p = xq[i];
    int c[3];
    if (!cell_coords(b, p.x, p.y, p.z, c)) atomicOr(&flags[kFlagOutOfBox], 1);
    const int id = c[0] + b.nc[0] * (c[1] + b.nc[1] * c[2]);
    cell_of[i] = id | atomicAdd(&cells[id], 1) << kOneBlockIdBits;
    if (((i >= a1 && i < b1) || (i >= a2 && i < b2)) && slot_rebuilt(m, g, i)) {
      x0[i] = p.x;
      x0[N + i] = p.y;
      x0[2 * N + i] = p.z;
    }
  }
  __syncthreads();
  const int per = (ncell + 1023) >> 10, c0 = min((int)threadIdx.x * per, ncell), c1 = min(c0 + per, ncell);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int sum = 0;
  for (int k = c0; k < c1; ++k) sum += cells[k];
  int x = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) wsum[wave] = x;
  __syncthreads();
  int run = x - sum;
  for (int q = 0; q < wave; ++q) run += wsum[q];
  for (int k = c0; k < c1; ++k) {
    const int v = cells[k];
    cells[k] = run;
    start[k] = run;
    run += v;
  }
  if (threadIdx.x == 0) start[ncell] = N;
  __syncthreads();
  for (int i = threadIdx.x; i < N; i += 1024) {
    const int w = cell_of[i];
    const int at = cells[w & ((1 << kOneBlockIdBits) - 1)] + (w >> kOneBlockIdBits);
    atoms[at] = i;
    xs[at] = xq[i];
  }
}

__global__ void k_cell_fill(const int* __restrict__ go, int N, const int* __restrict__ cell_of,
                            const int* __restrict__ rank, const int* __restrict__ start,
                            const double4* __restrict__ xq, int* __restrict__ atoms, double4* __restrict__ xs,
                            ImageMap m)
{
  if (!*go) return;
  const bool listed = rebuild_listed(m);
  const int n = listed ? m.req_off[2 * m.n_req + 1] : N;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    const int i = listed ? m.lists[m.n_owned + k] : k;
    const int at = start[cell_of[i]] + rank[i];
    atoms[at] = i;
    xs[at] = xq[i];
  }
}

// Offsets of each request's centres and slots in the compacted lists of the
// requests this rebuild remakes (exclusive scans over the requests, one
// workgroup), then the totals.
__global__ __launch_bounds__(1024) void k_list_scan(const int* __restrict__ go, ImageMap m)
{
  const int g = *go;
  if (!g) return;
  __shared__ int wsum[2][16];
  __shared__ int carry[2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if (threadIdx.x == 0) carry[0] = carry[1] = 0;
  __syncthreads();
  for (int base = 0; base < m.n_req; base += blockDim.x) {
    const int r = base + threadIdx.x;
    int c = 0, s = 0;
    if (r < m.n_req && ((g & kRebuildAll) || m.req_moved[r])) {
      const int4 q = m.req_range[r];
      c = q.y;
      s = q.y + q.w;
    }
    int ic = c, is = s;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int vc = __shfl_up(ic, d), vs = __shfl_up(is, d);
      if (lane >= d) {
        ic += vc;
        is += vs;
      }
    }
    if (lane == 63) {
      wsum[0][wave] = ic;
      wsum[1][wave] = is;
    }
    __syncthreads();
    int pc = carry[0], ps = carry[1];
    for (int v = 0; v < wave; ++v) {
      pc += wsum[0][v];
      ps += wsum[1][v];
    }
    if (r < m.n_req) {
      m.req_off[2 * r] = pc + ic - c;
      m.req_off[2 * r + 1] = ps + is - s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int v = 0; v < nw; ++v) {
        carry[0] += wsum[0][v];
        carry[1] += wsum[1][v];
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    m.req_off[2 * m.n_req] = carry[0];
    m.req_off[2 * m.n_req + 1] = carry[1];
  }
}

// The compacted lists: one workgroup per request
__global__ void k_list_fill(const int* __restrict__ go, ImageMap m)
{
  const int g = *go;
  if (!g) return;
  const int r = blockIdx.x;
  if (!((g & kRebuildAll) || m.req_moved[r])) return;
  const int4 q = m.req_range[r];
  int* cl = m.lists + m.req_off[2 * r];
  int* sl = m.lists + m.n_owned + m.req_off[2 * r + 1];
  for (int k = threadIdx.x; k < q.y; k += blockDim.x) {
    cl[k] = q.x + k;
    sl[k] = q.x + k;
  }
  for (int k = threadIdx.x; k < q.w; k += blockDim.x) sl[q.y + k] = q.z + k;
}

// Row key order: slot, or (global id, slot).
__device__ __forceinline__ bool key_less(const uint64_t* gid, int a, int b)
{
  if (gid) {
    const uint64_t ga = gid[a], gb = gid[b];
    if (ga != gb) return ga < gb;
  }
  return a < b;
}

// Candidate ranges of one centre: the 5x5 rows of cells around it (cell edge
// >= (rc+skin)/2, so +-2 cells cover rc+skin), each a contiguous range of
// cell_atoms, split in two where a periodic row wraps: at most 50 ranges.
constexpr int kRanges = 64;
constexpr int kRangesPerLane = kRanges / kRowLanes;
constexpr size_t kRangeLds = 2 * kRanges * sizeof(int);  // starts + prefix, per centre
// rows of at most this many entries are sorted in registers
constexpr int kSortMax = 16 * kRowLanes;

// LDS bytes of one centre's row buffers: the accepted slots, with their
// 64-bit keys where rows are keyed by global id, and the sorted row where
// the register sort may not hold it; a multiple of 8
__host__ __device__ inline size_t build_row_lds(int mv, bool keyed)
{
  return (keyed ? 16 : mv > kSortMax ? 8 : 4) * (size_t)mv;
}

// Bitonic sort of kRowLanes * E keys held E to a lane (ascending, key
// lane * E + r in register r): in-lane exchanges, and between lanes the
// mirrors and swaps that the DPP lane permutations offer.
template <class K>
__device__ __forceinline__ void exchange(K& a, K& b)
{
  const bool swap = b < a;
  const K lo = swap ? b : a, hi = swap ? a : b;
  a = lo;
  b = hi;
}
__device__ __forceinline__ void exchange(int& a, int& b)
{
  const int lo = min(a, b), hi = max(a, b);
  a = lo;
  b = hi;
}
__device__ __forceinline__ int keep(int a, int b, bool upper) { return upper ? max(a, b) : min(a, b); }
__device__ __forceinline__ uint64_t keep(uint64_t a, uint64_t b, bool upper) { return (b < a) == upper ? a : b; }

// in-lane: merge the halves of each block of S keys, the first step mirrored
template <int S, bool FLIP, int E, class K>
__device__ __forceinline__ void merge_in_lane(K (&v)[E])
{
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int o = FLIP ? r ^ (S - 1) : r ^ (S / 2);
    if (o > r) exchange(v[r], v[o]);
  }
  if constexpr (S > 2) merge_in_lane<S / 2, false>(v);
}
template <int S, int E, class K>
__device__ __forceinline__ void sort_in_lane(K (&v)[E])
{
  if constexpr (S > 2) sort_in_lane<S / 2>(v);
  if constexpr (S >= 2) merge_in_lane<S, true>(v);
}
// between lanes: key r of a lane against key r of its partner lane ...
template <int CTRL, int E, class K>
__device__ __forceinline__ void swap_step(K (&v)[E], bool upper)
{
#pragma unroll
  for (int r = 0; r < E; ++r) {
    K p = dpp_move<CTRL>(v[r]);
    v[r] = keep(v[r], p, upper);
  }
}
// ... or against key E - 1 - r of the mirrored lane
template <int CTRL, int E, class K>
__device__ __forceinline__ void mirror_step(K (&v)[E], bool upper)
{
#pragma unroll
  for (int r = 0; r < E / 2; ++r) {
    const K a = dpp_move<CTRL>(v[E - 1 - r]), b = dpp_move<CTRL>(v[r]);
    v[r] = keep(v[r], a, upper);
    v[E - 1 - r] = keep(v[E - 1 - r], b, upper);
  }
}
template <int E, class K>
__device__ __forceinline__ void sort_row(K (&v)[E], int lg)
{
  const bool b0 = lg & 1, b1 = lg & 2, b2 = lg & 4, b3 = lg & 8;
  constexpr int kX1 = 0xB1, kX2 = 0x4E, kX3 = 0x1B, kX7 = 0x141, kX15 = 0x140;  // lane ^ 1, 2, 3, 7, 15
  sort_in_lane<E>(v);
  mirror_step<kX1>(v, b0);  // two lanes
  merge_in_lane<E, false>(v);
  mirror_step<kX3>(v, b1);  // four
  swap_step<kX1>(v, b0);
  merge_in_lane<E, false>(v);
  mirror_step<kX7>(v, b2);  // eight
  swap_step<kX2>(v, b1);
  swap_step<kX1>(v, b0);
  merge_in_lane<E, false>(v);
  mirror_step<kX15>(v, b3);  // sixteen
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const K p = dpp_move<kX3>(dpp_move<kX7>(v[r]));  // lane ^ 4
    v[r] = keep(v[r], p, b2);
  }
  swap_step<kX2>(v, b1);
  swap_step<kX1>(v, b0);
  merge_in_lane<E, false>(v);
}

// sorts the n <= kRowLanes * E entries of a row and writes them out, four to
// a store (entries past n within the row's last four are not read by anyone)
template <bool KEYED, int E>
__device__ __forceinline__ void write_sorted(const int* row, const uint64_t* key, int n, int lg, bool active,
                                             int* __restrict__ out)
{
  using K = std::conditional_t<KEYED, uint64_t, int>;
  K v[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int k = r * kRowLanes + lg;
    v[r] = std::numeric_limits<K>::max();
    if (k < n) {
      if constexpr (KEYED) v[r] = key[k] << 32 | (uint32_t)row[k];
      else v[r] = row[k];
    }
  }
  sort_row(v, lg);
#pragma unroll
  for (int r = 0; r < E; r += 4) {
    const int k = lg * E + r;
    if (active && k < n)
      *reinterpret_cast<int4*>(out + k) = make_int4((int)v[r], (int)v[r + 1], (int)v[r + 2], (int)v[r + 3]);
  }
}

// the general form for longer rows and for keys that need all their bits:
// the rank of every entry among all n, then the row from its sorted copy
template <bool KEYED>
__device__ __forceinline__ void write_ranked(const int* row, const uint64_t* key, int* sorted, int n, int lg,
                                             bool active, int* __restrict__ out)
{
  for (int k = lg; k < n; k += kRowLanes) {
    const int v = row[k];
    int r = 0;
    if constexpr (KEYED) {
      const uint64_t kv = key[k];
      for (int t = 0; t < n; ++t) {
        const uint64_t kt = key[t];
        r += (kt < kv || (kt == kv && row[t] < v)) ? 1 : 0;
      }
    } else {
      // four entries per LDS read (row is 16-byte aligned: MV is a multiple of 4)
      const int4* row4 = reinterpret_cast<const int4*>(row);
      const int n4 = n >> 2;
      for (int t = 0; t < n4; ++t) {
        const int4 x = row4[t];
        r += (x.x < v) + (x.y < v) + (x.z < v) + (x.w < v);
      }
      for (int t = n4 * 4; t < n; ++t) r += row[t] < v ? 1 : 0;
    }
    sorted[r] = v;
  }
  wave_lds_sync();
  if (active)
    for (int k = lg; k < n; k += kRowLanes) out[k] = sorted[k];
}

// One kRowLanes group per centre.  The group first reads the bounds of all
// its ranges at once and prefix-sums their lengths, then streams the
// candidates as one list: candidate k is slot rs[q] + k - rp[q] of
// cell_atoms / xs (the cell-ordered copy of the positions), so a candidate
// costs two independent contiguous loads; each step tests two candidates
// per lane whose loads were issued a step earlier.  Accepted slots are compacted into LDS
// with a ballot, sorted on (key, slot) and written out as one contiguous
// row.  Rows past the capacity MV are counted but not stored; the count is
// reported through the flags.  A group lives inside one wavefront, so there
// is no workgroup barrier.
//
// Bound by vector instructions.  In an orthogonal box a range holds only the
// cells that a sphere of rc+skin around the centre reaches (84 of the 125 on
// average), and rows of up to kSortMax entries are sorted in registers: 192,000
// water atoms (143 entries a row) 316 us against 886 with every cell and rank
// sorts in LDS, 60,001 keyed rows of 90 92 against 276, 2.3 million rows of 90
// 1,570 against 2,410.  Four wavefronts per SIMD hold the sort's registers
// (five: 335, 124 and 1,480 us; six: 389, 199 and 1,950).
template <bool LISTED, bool KEYED, bool PLAIN>
__global__ __launch_bounds__(256, 4) void k_verlet_build(const int* __restrict__ go, DevBox b, int c1, int c2,
                                                      int groups, int row_shift, const double4* __restrict__ xq,
                                                      double rv2, const uint64_t* __restrict__ gid, DevWork w)
{
  const int go_word = *go;
  if (!go_word) return;
  extern __shared__ uint64_t shk[];
  const int g = threadIdx.x / kRowLanes, lg = threadIdx.x % kRowLanes;
  const int gw = g % (64 / kRowLanes);  // group inside the wavefront
  // per centre: [keys (with gid only) | row | sorted row], then the ranges
  const size_t per = build_row_lds(w.MV, KEYED) / sizeof(uint64_t);
  uint64_t* key = shk + (size_t)g * per;
  int* row = reinterpret_cast<int*>(KEYED ? key + w.MV : key);
  int* sorted = row + w.MV;
  int* rs = reinterpret_cast<int*>(shk + (size_t)groups * per) + g * 2 * kRanges;
  int* rp = rs + kRanges;
  // PLAIN: orthogonal with positive edges.  Cell edges for the trim (0: this
  // direction is not trimmed, where five periodic cells make the +-2 rows
  // reach the same atoms from both sides).  kTrim cells of slack cover the
  // rounding of the cell coordinates.
  constexpr float kTrim = 1e-3f;
  const float reach2 = (float)rv2 * (1.0f + kTrim);
  float edge[3];
  double len[3], half[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    edge[d] = b.pbc[d] && b.nc[d] < 6 ? 0.0f : (float)(b.thick[d] / b.nc[d]) * (1.0f - kTrim);
    len[d] = b.h[4 * d];
    half[d] = b.pbc[d] ? len[d] * 0.5 : std::numeric_limits<double>::infinity();
  }
  const float inv_edge_x = 1.0f / edge[0];
  // centres c1 + k, or with compacted lists the listed centres (of the
  // requests this rebuild remakes) inside [c1, c2): a pass per group of
  // `groups` centres, the grid striding over the groups
  const int ncent = LISTED ? w.map.req_off[2 * w.map.n_req] : c2 - c1;
  for (int base = blockIdx.x * groups; base < ncent; base += gridDim.x * groups) {
    const int kc = base + g;
    const int i = LISTED ? (kc < ncent ? w.map.lists[kc] : -1) : c1 + kc;
    const bool active = LISTED ? (i >= c1 && i < c2) : (i < c2 && slot_rebuilt(w.map, go_word, i));
    if (!__any(active)) continue;  // no centre of this wavefront is rebuilt
    double4 pi = make_double4(0, 0, 0, 0);
    int c[3] = {0, 0, 0};
    float f[3] = {0, 0, 0};
    if (active) {
      pi = xq[i];
      cell_coords(b, pi.x, pi.y, pi.z, c, f);
    }
    // ranges q = 2 * (5 (dz+2) + dy+2) + part, lane lg holding q in
    // [lg*kRangesPerLane, (lg+1)*kRangesPerLane); the empty ones are dropped
    int start[kRangesPerLane], count[kRangesPerLane];
    int tot = 0, some = 0;
#pragma unroll
    for (int u = 0; u < kRangesPerLane; ++u) {
      const int q = lg * kRangesPerLane + u;
      int s = 0, e = 0;
      if (active && q < 50) {
        const int r = q >> 1, part = q & 1;
        const int dz = r / 5 - 2, dy = r % 5 - 2;
        int cz = c[2] + dz, cy = c[1] + dy;
        bool ok = true;
        if (b.pbc[2]) cz = (cz + b.nc[2]) % b.nc[2];
        else ok = ok && cz >= 0 && cz < b.nc[2];
        if (b.pbc[1]) cy = (cy + b.nc[1]) % b.nc[1];
        else ok = ok && cy >= 0 && cy < b.nc[1];
        int lo0 = c[0] - 2, hi0 = c[0] + 2;
        if constexpr (PLAIN) {
          // what the row's distance in y and z leaves of the reach in x
          const float gy = fmaxf(fmaxf(dy - f[1], f[1] - dy - 1.0f) - kTrim, 0.0f) * edge[1];
          const float gz = fmaxf(fmaxf(dz - f[2], f[2] - dz - 1.0f) - kTrim, 0.0f) * edge[2];
          const float left = reach2 - gy * gy - gz * gz;
          ok = ok && left > 0.0f;
          if (edge[0] > 0.0f) {
            const float wx = sqrtf(fmaxf(left, 0.0f)) * inv_edge_x + kTrim;
            lo0 = c[0] + (int)fmaxf(floorf(f[0] - wx), -2.0f);
            hi0 = c[0] + (int)fminf(floorf(f[0] + wx), 2.0f);
          }
        }
        int lo1 = 0, hi1 = -1;
        if (b.pbc[0]) {
          if (lo0 < 0) {
            lo1 = lo0 + b.nc[0];
            hi1 = b.nc[0] - 1;
            lo0 = 0;
          } else if (hi0 >= b.nc[0]) {
            lo1 = 0;
            hi1 = hi0 - b.nc[0];
            hi0 = b.nc[0] - 1;
          }
        } else {
          lo0 = max(lo0, 0);
          hi0 = min(hi0, b.nc[0] - 1);
        }
        const int lo = part ? lo1 : lo0, hi = part ? hi1 : hi0;
        if (ok && hi >= lo) {
          const int row = cy + b.nc[1] * cz, at = b.nc[0] * row + (row >> row_shift);
          s = w.cell_start[at + lo];
          e = w.cell_start[at + hi + 1];
        }
      }
      start[u] = s;
      count[u] = e - s;
      tot += e - s;
      some += e > s ? 1 : 0;
    }
    int off = tot, at = some;
    auto scan_step = [&](int a, int t) {
      off += a;
      at += t;
    };
    scan_step(dpp_move<0x111>(off), dpp_move<0x111>(at));  // row_shr 1, 2, 4, 8: zeros come in
    scan_step(dpp_move<0x112>(off), dpp_move<0x112>(at));
    scan_step(dpp_move<0x114>(off), dpp_move<0x114>(at));
    scan_step(dpp_move<0x118>(off), dpp_move<0x118>(at));
    const int total = __shfl(off, kRowLanes - 1, kRowLanes);
    if (lg == kRowLanes - 1) rp[at] = total;
    off -= tot;
    at -= some;
#pragma unroll
    for (int u = 0; u < kRangesPerLane; ++u)
      if (count[u] > 0) {
        rs[at] = start[u] - off;
        rp[at] = off;
        off += count[u];
        ++at;
      }
    wave_lds_sync();
    // k < total lies in range q with rp[q] <= k < rp[q+1] (the last range
    // ends at total); a lane's k only grows, so q only moves forward
    int q = 0;
    auto slot_of = [&](int k) {
      while (rp[q + 1] <= k) ++q;
      return rs[q] + k;
    };
    // each step tests kBatch candidates of every lane, whose loads were issued
    // in the step before
    constexpr int kBatch = 2, kStep = kBatch * kRowLanes;
    int jn[kBatch] = {};
    double4 pn[kBatch] = {};
#pragma unroll
    for (int h = 0; h < kBatch; ++h) {
      const int k = lg + h * kRowLanes;
      if (k < total) {
        const int sl = slot_of(k);
        jn[h] = w.cell_atoms[sl];
        pn[h] = w.xs[sl];
      }
    }
    int found = 0;
    bool wide = false;  // a key of this row needs more than 32 bits
    for (int k0 = 0; __any(k0 < total); k0 += kStep) {
      int jc[kBatch];
      double4 pc[kBatch];
#pragma unroll
      for (int h = 0; h < kBatch; ++h) {
        jc[h] = jn[h];
        pc[h] = pn[h];
        const int k = k0 + kStep + lg + h * kRowLanes;
        if (k < total) {
          const int sl = slot_of(k);
          jn[h] = w.cell_atoms[sl];
          pn[h] = w.xs[sl];
        }
      }
#pragma unroll
      for (int h = 0; h < kBatch; ++h) {
        const int k = k0 + lg + h * kRowLanes;
        const int j = jc[h];
        double x = pc[h].x - pi.x, y = pc[h].y - pi.y, z = pc[h].z - pi.z;
        if constexpr (PLAIN) {  // the minimum image as mic() forms it
          x -= fabs(x) > half[0] ? copysign(len[0], x) : 0.0;
          y -= fabs(y) > half[1] ? copysign(len[1], y) : 0.0;
          z -= fabs(z) > half[2] ? copysign(len[2], z) : 0.0;
        } else {
          mic(b, x, y, z);
        }
        const bool take = k < total && j != i && dist2(x, y, z) < rv2;
        const unsigned gm = (unsigned)(__ballot(take) >> (gw * kRowLanes)) & ((1u << kRowLanes) - 1u);
        if (take) {
          const int to = found + __popc(gm & ((1u << lg) - 1u));
          if (to < w.MV) {
            row[to] = j;
            if constexpr (KEYED) {
              const uint64_t kj = gid[j];
              key[to] = kj;
              wide = wide || (kj >> 32) != 0;
            }
          }
        }
        found += __popc(gm);
      }
    }
    wave_lds_sync();
    const int n = min(found, w.MV);
    int* out = w.vl + (size_t)max(i, 0) * w.MV;
    if (__any(n > kSortMax) || (KEYED && __any(wide))) write_ranked<KEYED>(row, key, sorted, n, lg, active, out);
    else if (__any(n > 8 * kRowLanes)) write_sorted<KEYED, 16>(row, key, n, lg, active, out);
    else if (__any(n > 4 * kRowLanes)) write_sorted<KEYED, 8>(row, key, n, lg, active, out);
    else write_sorted<KEYED, 4>(row, key, n, lg, active, out);
    if (active && lg == 0) {
      w.vn[i] = found;
      if (found > w.MV) atomicMax(&w.flags[kFlagVerletOverflow], found);
    }
    wave_lds_sync();  // the next pass reuses the LDS
  }
}

// Position of the centre inside each neighbour's row (binary search on the
// row key); -1 when the neighbour has no row (outside the centre range).
// Rows are symmetric (the same FP64 test from both ends), so when both ends
// are centres and no image map is given, only the lower slot searches: it
// finds q (i in j's row) and writes the reverse entries of both directed
// edges, i -> j and j -> i; every entry is still written exactly once.  A
// lane searches kRevBatch edges of its centre in lockstep.
constexpr int kRevBatch = 4;

template <int G>
__global__ __launch_bounds__(256) void k_verlet_reverse(const int* __restrict__ go, int c1, int c2,
                                                        const uint64_t* __restrict__ gid, DevWork w)
{
  const int go_word = *go;
  if (!go_word) return;
  const bool listed = rebuild_listed(w.map);
  const int ncent = listed ? w.map.req_off[2 * w.map.n_req] : c2 - c1;
  const int lg = threadIdx.x % G;
  for (int kc = (blockIdx.x * blockDim.x + threadIdx.x) / G; kc < ncent;
       kc += gridDim.x * (blockDim.x / G)) {
  const int i = listed ? w.map.lists[kc] : c1 + kc;
  if (i < c1 || i >= c2 || (!listed && !slot_rebuilt(w.map, go_word, i))) continue;
  const int n = min(w.vn[i], w.MV);
  const int* ri = w.vl + (size_t)i * w.MV;
  const ImageMap& im = w.map;
  for (int p0 = lg; p0 < n; p0 += kRevBatch * G) {
    int t[kRevBatch], lo[kRevBatch], hi[kRevBatch], q[kRevBatch], ov[kRevBatch];
    bool own[kRevBatch];
    const int* ro[kRevBatch];
#pragma unroll
    for (int u = 0; u < kRevBatch; ++u) {
      const int p = p0 + u * G;
      // the reverse of i -> j is found in the row of j; with an image map, j
      // stands for its owner o = owner[j] shifted by S, and the reverse entry
      // is o -> (the image of i shifted by -S), one of i's own ghost slots
      int o = -1, tt = i;
      if (p < n) {
        const int j = ri[p];
        o = j;
        if (im.owner) {
          o = im.owner[j];
          const int c = im.image[j];
          if (c != image_code(0, 0, 0)) {
            // i's ghosts are stored in increasing image code
            const int want = image_neg(c);
            int lo = im.gstart[i], hi = im.gstart[i + 1] - 1;
            tt = -1;
            while (lo <= hi) {
              const int mid = (lo + hi) >> 1;
              const int v = im.image[mid];
              if (v == want) {
                tt = mid;
                break;
              }
              if (v < want) lo = mid + 1;
              else hi = mid - 1;
            }
          }
        }
      }
      const bool centre = o >= c1 && o < c2;
      const bool mine = im.owner || !centre || o > i;
      own[u] = p < n && mine;
      const bool search = own[u] && tt >= 0 && centre;
      t[u] = tt;
      ov[u] = o;
      q[u] = -1;
      lo[u] = 0;
      hi[u] = search ? min(w.vn[o], w.MV) - 1 : -1;
      ro[u] = search ? w.vl + (size_t)o * w.MV : ri;  // an in-bounds row for idle probes
    }
    bool more = true;
    while (more) {
      int v[kRevBatch];
#pragma unroll
      for (int u = 0; u < kRevBatch; ++u) v[u] = ro[u][lo[u] <= hi[u] ? (lo[u] + hi[u]) >> 1 : 0];
      more = false;
#pragma unroll
      for (int u = 0; u < kRevBatch; ++u) {
        if (lo[u] <= hi[u]) {
          const int mid = (lo[u] + hi[u]) >> 1;
          if (v[u] == t[u]) {
            q[u] = mid;
            lo[u] = hi[u] + 1;
          } else if (key_less(gid, v[u], t[u])) {
            lo[u] = mid + 1;
          } else {
            hi[u] = mid - 1;
          }
        }
        more = more || lo[u] <= hi[u];
      }
    }
#pragma unroll
    for (int u = 0; u < kRevBatch; ++u) {
      const int p = p0 + u * G;
      if (own[u]) {
        w.vrev[(size_t)i * w.MV + p] = (short)q[u];
        if (!im.owner && q[u] >= 0) w.vrev[(size_t)ov[u] * w.MV + q[u]] = (short)p;
      }
    }
  }
  }
}

inline int nblk(int n) { return (n + kBlock - 1) / kBlock; }
// workgroups of 256 lanes of a rebuild kernel, which strides over its
// centres or slots: 2,048 of them fill 256 CUs at 32 waves each, and a
// launch that finds no rebuild asked returns in about a microsecond
constexpr int kListBlocks = 2048;

// Systems up to kOneBlockAtoms atoms and kOneBlockCells cells (60 KiB of LDS)
// have their cells made by one workgroup: 4,096 atoms 11.9 us against 10.6 in
// three launches and the 4 us between them, 5,832 18 us, 11,000 29 us against
// 13; and a step without a rebuild is two launches (7 us) shorter, 82 -> 74 us
// a step of 4,096 carbon atoms.
constexpr int kOneBlockAtoms = 6144, kOneBlockCells = 15 * 1024;

// A wavefront per centre searches the reverse entries of small systems, whose
// searches are latency: 64-atom box 8.1 us against 16.5 with kRowLanes, Cu with
// vacancies 7.2 against 10.3, 4,096 carbon atoms 11.0 against 17.3, 5,832 of a
// 130-neighbour model 49 against 66 (11,000 BaTiO3 atoms 21.9 against 21.7, 60,001
// keyed rows 103 against 89).
constexpr int kWideReverse = 8192;

// LDS of one centre of the build: its row buffers and candidate ranges
size_t build_lds_per_centre(int mv, bool keyed) { return build_row_lds(mv, keyed) + kRangeLds; }

// centres per build workgroup: 16 groups of kRowLanes lanes unless the LDS
// would exceed 64 KiB
int build_groups(int mv, bool keyed)
{
  const size_t per = build_lds_per_centre(mv, keyed);
  int groups = 256 / kRowLanes;
  while (groups > 1 && per * groups > 64 * 1024) groups >>= 1;
  return groups;
}

}  // namespace

hipError_t launch_request_rebuild(DevWork& w, hipStream_t s)
{
  k_set_flag<<<1, 1, 0, s>>>(w.flags + kFlagRebuild, kRebuildAsked | kRebuildAll);
  return hipGetLastError();
}

hipError_t launch_clear_ints(int* p, long long n, hipStream_t s)
{
  if (n > 0) k_clear_ints<<<(int)std::min<long long>((n + kBlock - 1) / kBlock, 1024), kBlock, 0, s>>>(p, n);
  return hipGetLastError();
}

hipError_t launch_pack(const DevBox& b, int N, int T, const double* pos, const int* type, bool forced, DevWork& w,
                       hipStream_t s, double half_skin)
{
  const double half = half_skin > 0.0 ? half_skin : 0.5 * kSkin;
  if (N > 0)
    k_pack<<<nblk(N), kBlock, 0, s>>>(b, N, T, pos, type, w.x0, half * half, forced ? 1 : 0, w.xq, w.flags, w.map);
  else if (forced)
    k_set_flag<<<1, 1, 0, s>>>(w.flags + kFlagRebuild, kRebuildAsked | kRebuildAll);
  return hipGetLastError();
}

hipError_t launch_rebuild(const DevBox& b, int N, int c1, int c2, double rv2, const uint64_t* gid, DevWork& w,
                          hipStream_t s, const int* x0_ranges, bool capped)
{
  const int* go = w.flags + kFlagRebuild;
  const int ncell = b.nc[0] * b.nc[1] * b.nc[2];
  const int r[4] = {x0_ranges ? x0_ranges[0] : 0, x0_ranges ? x0_ranges[1] : N, x0_ranges ? x0_ranges[2] : 0,
                    x0_ranges ? x0_ranges[3] : 0};
  // the kernels stride over the centres and slots (with compacted lists,
  // the listed ones, counted on the device), so the grids may be capped
  const bool listed = rebuild_listed(w.map);
  if (listed) {
    k_list_scan<<<1, 1024, 0, s>>>(go, w.map);
    k_list_fill<<<w.map.n_req, kBlock, 0, s>>>(go, w.map);
  }
  const bool cap = capped || listed;
  const int slot_blocks = cap ? std::min(nblk(N), kListBlocks) : nblk(N);
  // the cells of small systems by one workgroup, whose LDS holds them
  int row_shift = 31;
  if (!listed && N > 0 && N <= kOneBlockAtoms && ncell <= kOneBlockCells) {
    k_cells_one_block<<<1, 1024, ncell * sizeof(int), s>>>(go, b, N, ncell, w.xq, w.cell_of, w.cell_start, w.x0, r[0],
                                                           r[1], r[2], r[3], w.flags, w.cell_atoms, w.xs, w.map);
  } else if (N > 0) {
    row_shift = 0;
    while (((long long)b.nc[0] << (row_shift + 1)) <= kScanCells) ++row_shift;
    const int rows = b.nc[1] * b.nc[2], tiles = (int)(((long long)rows + (1LL << row_shift) - 1) >> row_shift);
    int* cursor = w.cell_start + (size_t)ncell + tiles;
    k_cell_count<<<slot_blocks, kBlock, 0, s>>>(go, b, N, w.xq, row_shift, w.cell_of, w.cell_rank, w.cell_count, cursor,
                                                w.x0, r[0], r[1], r[2], r[3], w.flags, w.map);
    k_cell_starts<<<tiles, 1024, 0, s>>>(go, ncell, b.nc[0] << row_shift, w.cell_count, w.cell_start, cursor);
    k_cell_fill<<<slot_blocks, kBlock, 0, s>>>(go, N, w.cell_of, w.cell_rank, w.cell_start, w.xq, w.cell_atoms, w.xs,
                                               w.map);
  }
  if (c2 > c1) {
    const bool keyed = gid != nullptr;
    const int groups = build_groups(w.MV, keyed);
    constexpr int rows_per_block = 256 / kRowLanes;
    // build workgroups hold groups * kRowLanes lanes
    int nb = (c2 - c1 + groups - 1) / groups;
    const bool wide = c2 - c1 <= kWideReverse;
    const int reverses_per_block = wide ? 256 / 64 : rows_per_block;
    int nr = (c2 - c1 + reverses_per_block - 1) / reverses_per_block;
    if (cap) {
      nb = std::min(nb, kListBlocks * (rows_per_block / groups));
      nr = std::min(nr, kListBlocks);
    }
    const size_t lds = build_lds_per_centre(w.MV, keyed) * groups;
    const bool plain = b.ortho && b.h[0] > 0.0 && b.h[4] > 0.0 && b.h[8] > 0.0;
    const auto pick = [](auto keyed, bool listed, bool plain) {
      constexpr bool K = decltype(keyed)::value;
      return listed ? (plain ? k_verlet_build<true, K, true> : k_verlet_build<true, K, false>)
                    : (plain ? k_verlet_build<false, K, true> : k_verlet_build<false, K, false>);
    };
    const auto build = keyed ? pick(std::true_type{}, listed, plain) : pick(std::false_type{}, listed, plain);
    build<<<nb, groups * kRowLanes, lds, s>>>(go, b, c1, c2, groups, row_shift, w.xq, rv2, gid, w);
    if (wide) k_verlet_reverse<64><<<nr, 256, 0, s>>>(go, c1, c2, gid, w);
    else k_verlet_reverse<kRowLanes><<<nr, 256, 0, s>>>(go, c1, c2, gid, w);
  }
  // the request marks of this rebuild are spent
  if (w.map.slot_req && w.map.n_req > 0) k_clear_moved<<<nblk(w.map.n_req), kBlock, 0, s>>>(go, w.map);
  return hipGetLastError();
}

}  // namespace dmgx
