// dem_build.hip -- neighbour-list rebuild on the GPU.
//
// Replaces Cabana::VerletList<FullNeighborTag>::build as called at
// src/CabanaDEM_Solver.hpp:60-63,87-88 (reference paths relative to the
// ExaPhysics/CabanaDEM root).  The list is the set {j != i : dx^2+dy^2+dz^2
// <= rc^2} with the squared distance summed in x, y, z order without fused
// multiply-adds, exactly as the reference's Cabana build forms it, so the
// sets are bit-exact.
//
// Sequence (one rebuild, all stream ordered; small systems run all of it in
// one workgroup, k_rebuild_small):
//   1. k_cell_keys   cell key of every particle (tiled cell order, see
//                    dem_internal.h); per-cell arrival rank by atomic
//                    counting; optional skin-displacement check
//   2. scan          exclusive prefix over the cell counts within scan tiles,
//                    then over the tiles; clears the counts for the next
//                    rebuild
//   3. k_scatter     counting-sort scatter: slot = start[key] + rank
//   4. k_cell_order  within each cell, order by previous slot (the arrival
//                    order of step 1 is not deterministic; this makes the
//                    sort a stable, deterministic single-digit radix sort
//                    on the cell key), write the inverse permutation and the
//                    cells' starts
//   5. k_permute     gather the particle state into the new order and
//                    re-map the tracked-contact lists (j -> inv[j], re-sorted)
//   6. k_neighbors   27-cell search: for each (dz, dy) the three x-adjacent
//                    cells are one contiguous slot range; the nine ranges are
//                    visited in ascending slot order, so a row comes out in
//                    ascending j (the order the force kernel merges in).
#include "dem_internal.h"

#include <algorithm>
#include <climits>

namespace demhip {
namespace {

__device__ inline int cell_coord(double v, const Grid& g, int d) {
  double t = floor((v - g.lo[d]) / g.h[d]);
  if (!(t >= 0.0)) return 0; // below the box, or NaN
  if (t > (double)(g.nc[d] - 1)) return g.nc[d] - 1;
  return (int)t;
}

// Cell key of slot i at position p; flags a position that is not finite.
__device__ __forceinline__ int key_of(const BuildArgs& a, int i, const double4& p) {
  if (!(isfinite(p.x) && isfinite(p.y) && isfinite(p.z))) atomicOr(&a.flags->nonfinite, 1);
  // ensembles: the slot's system gives the grid and the first key
  const int sys = a.sysid ? a.sysid[i] : 0;
  const Grid& g = a.sysid ? a.grids[sys] : a.grid;
  const long base = a.sysid ? a.kbase[sys] : 0;
  const int cx = cell_coord(p.x, g, 0);
  const int cy = cell_coord(p.y, g, 1);
  const int cz = cell_coord(p.z, g, 2);
  return (int)(base + cell_key(g, cx, cy, cz));
}

// Flags slot i when it has moved more than skin/2 since the last build.
__device__ __forceinline__ void check_skin(const BuildArgs& a, int i, const double4& p) {
  const double d0 = p.x - a.xb[3 * i + 0];
  const double d1 = p.y - a.xb[3 * i + 1];
  const double d2 = p.z - a.xb[3 * i + 2];
  if (d0 * d0 + d1 * d1 + d2 * d2 > a.skin_half_sq) atomicOr(&a.flags->skin, 1);
}

// Per-cell arrival ranks with one atomic per run of equal keys in a wave:
// the slots are in the previous rebuild's cell order, so a wave's keys come
// in runs.  The run's first lane reserves the run's length and the others
// take consecutive ranks after it (any ranks that number each cell's
// particles 0 .. count - 1 will do: k_cell_order fixes the order).
__global__ __launch_bounds__(kBlock) void k_cell_keys(BuildArgs a) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const bool active = i < a.n; // the active lanes of a wave are a prefix
  int key = -1;
  double4 p = make_double4(0., 0., 0., 0.);
  if (active) {
    p = a.xr_in[i];
    key = key_of(a, i, p);
  }
  const int prev = __shfl_up(key, 1);
  const bool head = active && (lane == 0 || prev != key);
  const unsigned long long heads = __ballot(head);
  const unsigned long long below = lane == 63 ? ~0ull : ((2ull << lane) - 1); // lanes 0 .. lane
  const int hl = 63 - __clzll(heads & below); // this lane's run head (active lanes)
  const int nactive = __popcll(__ballot(active)); // with every lane of the wave executing
  int base_rank = 0;
  if (head) {
    const unsigned long long above = heads & ~below;
    const int next = above ? __ffsll((long long)above) - 1 : nactive;
    base_rank = atomicAdd(&a.cell_count[key], next - lane);
  }
  base_rank = __shfl(base_rank, hl >= 0 ? hl : 0);
  if (!active) return;
  a.key[i] = key;
  a.rank[i] = base_rank + (lane - hl);
  if (a.check_skin) check_skin(a, i, p);
}

// ---- exclusive scan of the cell counts --------------------------------------
constexpr int kScanThreads = 1024;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ inline int block_exclusive_scan(int v, int* lds, int* total) {
  const int t = threadIdx.x;
  lds[t] = v;
  __syncthreads();
  for (int off = 1; off < kScanThreads; off <<= 1) {
    int add = (t >= off) ? lds[t - off] : 0;
    __syncthreads();
    lds[t] += add;
    __syncthreads();
  }
  const int incl = lds[t];
  *total = lds[kScanThreads - 1];
  __syncthreads();
  return incl - v;
}

// Also clears `in` (the next rebuild counts into it).
__global__ __launch_bounds__(kScanThreads) void k_scan_tiles(int* in, int* out,
                                                              int* tile_sums, long count) {
  __shared__ int lds[kScanThreads];
  const long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
  int v[kScanItems];
  int s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    v[k] = (base + k < count) ? in[base + k] : 0;
    s += v[k];
  }
  int total;
  int ex = block_exclusive_scan(s, lds, &total);
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    if (base + k < count) {
      out[base + k] = ex;
      in[base + k] = 0;
    }
    ex += v[k];
  }
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

// Tile totals to tile offsets, and the build's longest row back to none.
__global__ __launch_bounds__(kScanThreads) void k_scan_top(int* tile_sums, int ntiles, DevFlags* flags) {
  __shared__ int lds[kScanThreads];
  int carry = 0;
  for (int base = 0; base < ntiles; base += kScanThreads) {
    const int t = base + (int)threadIdx.x;
    const int v = (t < ntiles) ? tile_sums[t] : 0;
    int total;
    const int ex = block_exclusive_scan(v, lds, &total);
    if (t < ntiles) tile_sums[t] = ex + carry;
    carry += total;
  }
  if (threadIdx.x == 0) flags->max_nn = 0;
}

// Start of cell c: its place in its scan tile on top of the tile's offset
// (added by the two readers instead of a pass over all cells).
__device__ __forceinline__ int start_of(const BuildArgs& a, long c) {
  return c < a.ncell ? a.cell_scan[c] + a.scan_tmp[c / kScanTile] : a.n;
}

__global__ __launch_bounds__(kBlock) void k_scatter(BuildArgs a) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.n) return;
  a.perm[start_of(a, a.key[i]) + a.rank[i]] = i;
}

// One thread per cell: insertion-sort the cell's slots by previous index
// (cells hold a handful of particles), then record old -> new and the cell's
// start.
__global__ __launch_bounds__(kBlock) void k_cell_order(BuildArgs a) {
  const long c = (long)blockIdx.x * kBlock + threadIdx.x;
  if (c > a.ncell) return;
  const int s = start_of(a, c);
  a.cell_start[c] = s;
  if (c == a.ncell) return;
  const int e = start_of(a, c + 1);
  if (e - s > kMaxCellParticles) {
    atomicOr(&a.flags->cell_overflow, 1);
    for (int q = s; q < e; ++q) a.inv[a.perm[q]] = q;
    return;
  }
  for (int q = s + 1; q < e; ++q) {
    const int v = a.perm[q];
    int r = q - 1;
    while (r >= s && a.perm[r] > v) {
      a.perm[r + 1] = a.perm[r];
      --r;
    }
    a.perm[r + 1] = v;
  }
  for (int q = s; q < e; ++q) a.inv[a.perm[q]] = q;
}

// A wave's own LDS tile: its writes before its later reads, and back.
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline void copy6(const double* src, double* dst) {
  const double2* s = reinterpret_cast<const double2*>(src);
  double2* d = reinterpret_cast<double2*>(dst);
  d[0] = s[0];
  d[1] = s[1];
  d[2] = s[2];
}

// Slot p's particle (old slot o): contact word, wall histories, bonds, group and
// external force.  inv(j): the new slot of old slot j.
template <class Inv>
__device__ __forceinline__ void permute_lists(const BuildArgs& a, int p, int o, int meta, const Inv& inv) {
  a.cmeta_out[p] = meta;
  const int wm = meta_walls(meta);
  if (wm) {
    for (int w = 0; w < DEM_MAX_WALLS; ++w)
      if (wm & (1 << w))
        for (int c = 0; c < 3; ++c)
          a.sw_out[(long)(w * 3 + c) * a.ld + p] = a.sw_in[(long)(w * 3 + c) * a.ld + o];
  }
  if (a.bonds_on) {
    // bond rows keep their slot order; partners follow the permutation
    const int nb = a.nbond_in[o];
    a.nbond_out[p] = nb;
    a.bEG_out[p] = a.bEG_in[o];
    if (a.vgroup_in) a.vgroup_out[p] = a.vgroup_in[o];
    for (int b = 0; b < nb; ++b) {
      const int j = a.bj_in[(long)b * a.ld + o];
      a.bj_out[(long)b * a.ld + p] = j >= 0 ? inv(j) : -1;
      a.bl_out[(long)b * a.ld + p] = a.bl_in[(long)b * a.ld + o];
      for (int c = 0; c < 9; ++c)
        a.bh_out[(long)(9 * b + c) * a.ld + p] = a.bh_in[(long)(9 * b + c) * a.ld + o];
    }
  } else if (a.vgroup_in) {
    a.vgroup_out[p] = a.vgroup_in[o];
  }
  if (a.fext_in)
    for (int d = 0; d < 3; ++d) a.fext_out[3l * p + d] = a.fext_in[3l * o + d];
}

// The tracked-contact list of a particle keeps its entries and histories; only
// the neighbour indices change (old j -> its new slot, id(m) for entry m) and
// the list is re-sorted by the new index.
template <class Id>
__device__ __forceinline__ void permute_contacts(const BuildArgs& a, int p, int o, int oc, const Id& id) {
  for (int m = 0; m < oc; ++m) {
    const int jm = id(m);
    int r = 0;
    for (int q = 0; q < oc; ++q) r += (id(q) < jm) ? 1 : 0;
    a.cj_out[(long)r * a.ld + p] = jm;
    for (int c = 0; c < 3; ++c)
      a.ch_out[(long)(r * 3 + c) * a.ld + p] = a.ch_in[(long)(m * 3 + c) * a.ld + o];
  }
}

__device__ __forceinline__ void permute_state(const BuildArgs& a, int p, int o, const double4& xr) {
  a.xr_out[p] = xr;
  copy6(a.uw_in + 6l * o, a.uw_out + 6l * p);
  if (a.permute_ft) copy6(a.ft_in + 6l * o, a.ft_out + 6l * p);
  a.mat_out[p] = a.mat_in[o];
  a.mI_out[p] = a.mI_in[o];
  a.id_out[p] = a.id_in[o];
  if (a.keep_xb) {
    a.xb[3 * p + 0] = xr.x;
    a.xb[3 * p + 1] = xr.y;
    a.xb[3 * p + 2] = xr.z;
  }
}

// A wave's consecutive records from its LDS tile to memory, 16 bytes a lane and
// instruction on consecutive addresses (past the caches with nt): n16 pieces.
template <int K>
__device__ __forceinline__ void store_records(const double2* st, double2* g, int n16, int lane, bool nt) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int q = k * 64 + lane;
    if (q >= n16) continue;
    const double2 v = st[q];
    if (nt) {
      __builtin_nontemporal_store(v.x, &g[q].x);
      __builtin_nontemporal_store(v.y, &g[q].y);
    } else {
      g[q] = v;
    }
  }
}

// Gather the per-particle arrays into the new order.  Everything of the
// particle is loaded before anything is stored (a store in between would wait
// for the load before it, and no load moves up over a store), and the records
// leave through LDS in whole lines, as in the fused step.  Bound: HBM, about
// 310 bytes a particle.  1M spheres 75 -> 66 us (4.7 TB/s), 4M 270 -> 232.
__global__ __launch_bounds__(kBlock) void k_permute(BuildArgs a) {
  extern __shared__ int s_j[]; // [max_c][kBlock]
  __shared__ double2 s_rec[kBlock / 64][64 * 5];
  const int tid = threadIdx.x, lane = tid & 63;
  const int p0 = blockIdx.x * kBlock + tid - lane; // the wave's first slot
  const int cnt = min(64, a.n - p0);
  const int p = p0 + lane;
  const bool act = p < a.n;
  double2* st = s_rec[tid >> 6];
  const bool nt = a.stream != 0;
  double* sx = reinterpret_cast<double*>(st + 128);
  double4 xr, mat;
  double2 u0, u1, u2, mI;
  int o = 0, id = 0, key = 0, meta = 0, oc = 0;
  if (act) {
    o = a.perm[p];
    xr = a.xr_in[o];
    const double2* uo = reinterpret_cast<const double2*>(a.uw_in + 6l * o);
    u0 = uo[0]; u1 = uo[1]; u2 = uo[2];
    mat = a.mat_in[o];
    mI = a.mI_in[o];
    id = a.id_in[o];
    key = a.key[o];
    meta = a.cmeta_in[o];
    oc = min(meta_count(meta), a.max_c); // counts are clamped on write; never index past the LDS rows
    for (int m = 0; m < oc; ++m) s_j[m * kBlock + tid] = a.inv[a.cj_in[(long)m * a.ld + o]];
    st[2 * lane] = make_double2(xr.x, xr.y);
    st[2 * lane + 1] = make_double2(xr.z, xr.w);
    st[128 + 3 * lane] = u0;
    st[128 + 3 * lane + 1] = u1;
    st[128 + 3 * lane + 2] = u2;
  }
  wave_lds_sync();
  store_records<2>(st, reinterpret_cast<double2*>(a.xr_out + p0), 2 * cnt, lane, false);
  store_records<3>(st + 128, reinterpret_cast<double2*>(a.uw_out + 6l * p0), 3 * cnt, lane, nt);
  wave_lds_sync();
  if (act) {
    st[2 * lane] = make_double2(mat.x, mat.y);
    st[2 * lane + 1] = make_double2(mat.z, mat.w);
    sx[3 * lane] = xr.x;
    sx[3 * lane + 1] = xr.y;
    sx[3 * lane + 2] = xr.z;
  }
  wave_lds_sync();
  store_records<2>(st, reinterpret_cast<double2*>(a.mat_out + p0), 2 * cnt, lane, nt);
  if (a.keep_xb) {
    double* xb = a.xb + 3l * p0;
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (k * 64 + lane < 3 * cnt) xb[k * 64 + lane] = sx[k * 64 + lane];
  }
  if (!act) return;
  a.mI_out[p] = mI;
  a.id_out[p] = id;
  a.key_sorted[p] = key;
  if (a.permute_ft) copy6(a.ft_in + 6l * o, a.ft_out + 6l * p);
  permute_lists(a, p, o, meta, [&](int j) { return a.inv[j]; });
  permute_contacts(a, p, o, oc, [&](int m) { return s_j[m * kBlock + tid]; });
}

// Minimum and maximum over the wave's 64 lanes, the same scalar in all of
// them: row shifts and row broadcasts in the VALU, where shuffles go through
// LDS six times over, each waiting for the one before (k_neighbors at 1M
// spheres, eighteen reductions a wave: 71 -> 68 us).  Every lane of the wave
// must call these.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_or(int fill, int v) {
  return __builtin_amdgcn_update_dpp(fill, v, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ int wave_max_int(int v) {
  v = max(v, dpp_or<0x111, 0xf>(INT_MIN, v)); // row_shr 1, 2, 4, 8: lane 15 of a row holds the row's
  v = max(v, dpp_or<0x112, 0xf>(INT_MIN, v));
  v = max(v, dpp_or<0x114, 0xf>(INT_MIN, v));
  v = max(v, dpp_or<0x118, 0xf>(INT_MIN, v));
  v = max(v, dpp_or<0x142, 0xa>(INT_MIN, v)); // row_bcast 15 into rows 1 and 3
  v = max(v, dpp_or<0x143, 0xc>(INT_MIN, v)); // row_bcast 31 into rows 2 and 3
  return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_min_int(int v) {
  v = min(v, dpp_or<0x111, 0xf>(INT_MAX, v));
  v = min(v, dpp_or<0x112, 0xf>(INT_MAX, v));
  v = min(v, dpp_or<0x114, 0xf>(INT_MAX, v));
  v = min(v, dpp_or<0x118, 0xf>(INT_MAX, v));
  v = min(v, dpp_or<0x142, 0xa>(INT_MAX, v));
  v = min(v, dpp_or<0x143, 0xc>(INT_MAX, v));
  return __builtin_amdgcn_readlane(v, 63);
}

// The nine slot ranges around slot p's cell `key`: three consecutive x-cells of
// one (y, z) row each, ascending by start (they never overlap), INT_MAX where
// there is none.  start(c): first slot of cell c.
template <class Start>
__device__ __forceinline__ void slot_ranges(const BuildArgs& a, int p, int key, const Start& start, int (&rs)[9],
                                            int (&re)[9]) {
  const int sys = a.sysid ? a.sysid[p] : 0;
  const Grid& g = a.sysid ? a.grids[sys] : a.grid;
  const long base = a.sysid ? a.kbase[sys] : 0;
  const int nx = g.nc[0], ny = g.nc[1], nz = g.nc[2];
  key = (int)(key - base);
  const int cx = key % nx;
  key /= nx;
  const int ly = key % g.tr;
  key /= g.tr;
  const int cz = key % nz;
  const int cy = (key / nz) * g.tr + ly;
  const int xlo = cx > 0 ? cx - 1 : 0;
  const int xhi = cx < nx - 1 ? cx + 1 : nx - 1;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const int z = cz + q / 3 - 1, y = cy + q % 3 - 1;
    const bool in = z >= 0 && z < nz && y >= 0 && y < ny;
    rs[q] = re[q] = INT_MAX;
    if (in) {
      const long k0 = base + cell_key(g, xlo, y, z);
      rs[q] = start(k0);
      re[q] = start(k0 + (xhi - xlo) + 1);
    }
  }
#pragma unroll
  for (int q = 1; q < 9; ++q)
#pragma unroll
    for (int r = q; r > 0; --r)
      if (rs[r] < rs[r - 1]) {
        int t = rs[r]; rs[r] = rs[r - 1]; rs[r - 1] = t;
        t = re[r]; re[r] = re[r - 1]; re[r - 1] = t;
      }
}

#ifndef DEM_NBR_STAGE
#define DEM_NBR_STAGE 128
#endif
constexpr int kNbrStage = DEM_NBR_STAGE; // slots of one range round staged in LDS per wave

// Cabana's full Verlet list (VerletList with FullNeighborTag, built with the
// cell list, src/CabanaDEM_Solver.hpp:60-63): j != i with |x_i - x_j|^2 <= rc^2,
// rows ascending in j.  Slot p searches the 27 cells around its own as nine
// slot ranges (three consecutive x-cells of one (y, z) row are contiguous in
// cell order), walked in ascending order.
//
// LDS-staged cell tiles: in round q every lane walks its q-th range.  The
// lanes of a wave are consecutive slots, mostly of one cell row, so their
// q-th ranges lie in one short span of slots; the wave loads that span into
// LDS once (coalesced) when it holds at most kNbrStage slots, and the lanes
// test against LDS instead of each gathering its own candidates.  Wider
// spans (a wave across a y-tile or system boundary) read from global memory.
// Either way the tested values and their order are the same.
__global__ __launch_bounds__(kBlock) void k_neighbors(BuildArgs a) {
  __shared__ double4 sx[kBlock / 64][kNbrStage];
  const int p = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const bool active = p < a.n && !a.flags->cell_overflow;
  int cnt = 0;
  long off = p; // a.nbr offset of the row's next entry: cnt * ld + p
  int rs[9], re[9];
  double4 xi = make_double4(0., 0., 0., 0.);
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    rs[q] = INT_MAX;
    re[q] = INT_MAX;
  }
  if (active) {
    xi = a.xr_out[p];
    slot_ranges(a, p, a.key_sorted[p], [&](long c) { return a.cell_start[c]; }, rs, re);
  }
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const int s = rs[q], e = re[q];
    const bool has = s != INT_MAX;
    const int lo = wave_min_int(has ? s : INT_MAX);
    const int hi = wave_max_int(has ? e : INT_MIN);
    if (lo == INT_MAX) break; // no lane has a q-th range, nor a later one
    const bool staged = hi - lo <= kNbrStage; // the same for the whole wave
    const auto within = [&](const double4& xj) {
      const double d0 = xi.x - xj.x;
      const double d1 = xi.y - xj.y;
      const double d2 = xi.z - xj.z;
      return d0 * d0 + d1 * d1 + d2 * d2 <= a.rc2;
    };
    const auto add = [&](int j) {
      if (cnt < a.max_n) a.nbr[off] = j;
      ++cnt;
      off += a.ld;
    };
    if (staged) {
      for (int t = lane; t < hi - lo; t += 64) sx[w][t] = a.xr_out[lo + t];
      wave_lds_sync();
      if (has)
        for (int j = s; j < e; ++j)
          if (j != p && within(sx[w][j - lo])) add(j);
      wave_lds_sync(); // the next round rewrites the tile
    } else if (has) {
      for (int j = s; j < e; ++j)
        if (j != p && within(a.xr_out[j])) add(j);
    }
  }
  if (active) a.nn[p] = cnt < a.max_n ? cnt : a.max_n;
  // one global atomic per wave, and only when it can raise the maximum
  const int wmax = wave_max_int(cnt);
  if (lane == 0 && wmax > 0) {
    if (wmax > *(volatile int*)&a.flags->max_nn) atomicMax(&a.flags->max_nn, wmax);
    if (wmax > a.max_n) atomicMax(&a.flags->nbr_overflow, wmax);
  }
}

// The whole rebuild of a small system in one workgroup: the sequence above with
// the counts, the sort and the positions in LDS and barriers for launches.  A
// rebuild of seven launches costs a small system 30 us and more, launch gaps
// for the most part, and by default it comes every step.
constexpr int kSmallThreads = 1024;
// Rebuilt every step, us a step with the launch sequence / one workgroup: 2
// spheres 37 / 14, 64 47 / 25, 512 58 / 40, 1,000 60 / 50, 1,728 61 / 78; in
// coarse binning too (1,000 spheres of 26 neighbours each 154 / 109, of 268
// 1065 / 560).
constexpr int kSmallMax = 1024;        // particles
constexpr int kSmallCells = 8192;      // cells, all systems

__global__ __launch_bounds__(kSmallThreads) void k_rebuild_small(BuildArgs a) {
  __shared__ double4 pos[kSmallMax];      // new order
  __shared__ int start[kSmallCells + 1];  // counts, then starts
  __shared__ int perm[kSmallMax], inv[kSmallMax], key[kSmallMax];
  __shared__ int wsum[kSmallThreads / 64];
  const int tid = threadIdx.x, T = blockDim.x, lane = tid & 63, w = tid >> 6;
  const int ncell = (int)a.ncell;
  for (int c = tid; c <= ncell; c += T) start[c] = 0;
  __syncthreads();
  static_assert(kSmallMax <= kSmallThreads, "a thread per particle");
  int rank = 0;
  if (tid < a.n) {
    const double4 p = a.xr_in[tid];
    key[tid] = key_of(a, tid, p);
    rank = atomicAdd(&start[key[tid]], 1);
    if (a.check_skin) check_skin(a, tid, p);
  }
  __syncthreads();
  { // counts -> starts: each thread a run of cells, then a scan over the threads
    const int per = (ncell + T - 1) / T, c0 = tid * per, c1 = min(ncell, c0 + per);
    int sum = 0;
    for (int c = c0; c < c1; ++c) sum += start[c];
    int incl = sum;
    for (int off = 1; off < 64; off <<= 1) {
      const int t = __shfl_up(incl, off);
      if (lane >= off) incl += t;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int run = incl - sum;
    for (int k = 0; k < w; ++k) run += wsum[k];
    for (int c = c0; c < c1; ++c) {
      const int n = start[c];
      start[c] = run;
      run += n;
    }
    if (tid == 0) start[ncell] = a.n;
  }
  __syncthreads();
  if (tid < a.n) perm[start[key[tid]] + rank] = tid;
  __syncthreads();
  for (int c = tid; c < ncell; c += T) { // within a cell by previous slot, as k_cell_order
    const int s = start[c], e = start[c + 1];
    for (int q = s + 1; q < e; ++q) {
      const int v = perm[q];
      int r = q - 1;
      while (r >= s && perm[r] > v) {
        perm[r + 1] = perm[r];
        --r;
      }
      perm[r + 1] = v;
    }
    for (int q = s; q < e; ++q) inv[perm[q]] = q;
  }
  __syncthreads();
  const int p = tid;
  const int o = p < a.n ? perm[p] : 0;
  if (p < a.n) {
    const double4 xr = a.xr_in[o];
    pos[p] = xr;
    permute_state(a, p, o, xr);
    a.key_sorted[p] = key[o];
    const auto new_slot = [&](int j) { return inv[j]; };
    const int meta = a.cmeta_in[o];
    permute_lists(a, p, o, meta, new_slot);
    permute_contacts(a, p, o, min(meta_count(meta), a.max_c), [&](int m) { return inv[a.cj_in[(long)m * a.ld + o]]; });
  }
  __syncthreads();
  int longest = 0;
  if (p < a.n) {
    int rs[9], re[9];
    slot_ranges(a, p, key[o], [&](long c) { return start[c]; }, rs, re);
    const double4 xi = pos[p];
    int cnt = 0;
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      if (rs[q] == INT_MAX) break;
      for (int j = rs[q]; j < re[q]; ++j) {
        const double4 xj = pos[j];
        const double d0 = xi.x - xj.x;
        const double d1 = xi.y - xj.y;
        const double d2 = xi.z - xj.z;
        const double dsqr = d0 * d0 + d1 * d1 + d2 * d2;
        if (j != p && dsqr <= a.rc2) {
          if (cnt < a.max_n) a.nbr[(long)cnt * a.ld + p] = j;
          ++cnt;
        }
      }
    }
    a.nn[p] = cnt < a.max_n ? cnt : a.max_n;
    longest = cnt;
  }
  longest = wave_max_int(longest);
  if (lane == 0) wsum[w] = longest;
  __syncthreads();
  for (int k = 0; k < T / 64; ++k) longest = max(longest, wsum[k]);
  if (longest > a.max_n) // the caller searches again with longer rows: k_neighbors needs the starts
    for (int c = tid; c <= ncell; c += T) a.cell_start[c] = start[c];
  if (tid == 0) {
    a.flags->max_nn = longest;
    if (longest > a.max_n) atomicMax(&a.flags->nbr_overflow, longest);
  }
}

// src/CabanaBondedDEM_Particles.hpp:118-137: bond i to every list neighbour
// j with r_ij < factor * r_i (the reference hard-codes factor 3), storing the
// partner and the initial length in the next slot.  Rows are ascending in j.
__global__ __launch_bounds__(kBlock) void k_setup_bonds(BondSetupArgs a) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.n) return;
  const double4 xi = a.xr[i];
  const double cond = a.factor * xi.w;                 // :130
  int nb = 0;
  for (int k = 0; k < a.nn[i]; ++k) {
    const int j = a.nbr[(long)k * a.ld + i];
    const double4 xj = a.xr[j];
    const double p0 = xi.x - xj.x, p1 = xi.y - xj.y, p2 = xi.z - xj.z; // :120-122
    const double r2 = p0 * p0 + p1 * p1 + p2 * p2;                      // :124
    const double rij = sqrt(r2);                                        // :126
    if (rij < cond) {                                                   // :132
      if (nb < a.max_b) {
        a.bj[(long)nb * a.ld + i] = j;                                  // :133
        a.bl[(long)nb * a.ld + i] = rij;                                // :134
        for (int c = 0; c < 9; ++c) a.bh[(long)(9 * nb + c) * a.ld + i] = 0.;
      } else {
        atomicMax(&a.flags->bond_overflow, nb + 1);
      }
      ++nb;                                                             // :135
    }
  }
  a.nbond[i] = nb < a.max_b ? nb : a.max_b;
}

__global__ void k_zero_u64(unsigned long long* p, int count) {
  if ((int)threadIdx.x < count) p[threadIdx.x] = 0ull;
}

inline unsigned nblk(long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

} // namespace

hipError_t launch_zero_u64(unsigned long long* p, int count, hipStream_t s) {
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, s, p, count);
  return hipGetLastError();
}

hipError_t launch_setup_bonds(const BondSetupArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_setup_bonds, dim3(nblk(a.n)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

bool rebuild_is_small(int n, long ncell) { return n <= kSmallMax && ncell <= kSmallCells; }

hipError_t launch_rebuild_small(const BuildArgs& a, hipStream_t s) {
  // a thread per particle, and enough of them for the cells
  const long want = std::max<long>(a.n, a.ncell / 16);
  const int threads = (int)std::min<long>(kSmallThreads, (want + 63) / 64 * 64);
  hipLaunchKernelGGL(k_rebuild_small, dim3(1), dim3(threads), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_rebuild(const BuildArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_cell_keys, dim3(nblk(a.n)), dim3(kBlock), 0, s, a);
  const int ntiles = (int)((a.ncell + kScanTile - 1) / kScanTile);
  hipLaunchKernelGGL(k_scan_tiles, dim3(ntiles), dim3(kScanThreads), 0, s, a.cell_count, a.cell_scan, a.scan_tmp,
                     a.ncell);
  hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(kScanThreads), 0, s, a.scan_tmp, ntiles, a.flags);
  hipLaunchKernelGGL(k_scatter, dim3(nblk(a.n)), dim3(kBlock), 0, s, a);
  hipLaunchKernelGGL(k_cell_order, dim3(nblk(a.ncell + 1)), dim3(kBlock), 0, s, a);
  const size_t lds = (size_t)(a.max_c > 0 ? a.max_c : 1) * kBlock * sizeof(int);
  hipLaunchKernelGGL(k_permute, dim3(nblk(a.n)), dim3(kBlock), lds, s, a);
  return hipGetLastError();
}

hipError_t launch_neighbors(const BuildArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_neighbors, dim3(nblk(a.n)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

} // namespace demhip
