// Radius graph on the device with periodic images: a cell list over the bounding box of the positions.
// Replaces radius_graph_pbc_gpu (utils/graph_utils.py:192-257: one torch_cluster.radius call per image
// shift s in {-1,0,1} on each periodic axis) and the host loop that turns the LAMMPS neighbour list into
// edges (lammps_user_mfftorch/src/USER-MFFTORCH/pair_mff_torch.cpp:597-641).
//
// The edge set is every (src i, dst j, s) with s_k in {-1,0,1} on periodic axes (0 otherwise), not
// (i == j and s == 0), and |(pos_j - pos_i) + s.cell|^2 < r^2, evaluated in double precision in that
// order with no fused multiply-adds (cell rows are the lattice vectors, as in the reference).  Edges come
// out receiver-sorted and, within a receiver, ascending in (src, s_x, s_y, s_z): a deterministic order,
// so graph preparation's stable receiver sort keeps it.
//
// Steps: bounding box and grid (cells of side >= r where the cell budget allows), atoms bucketed by cell
// (counting sort) with their positions in that order, one wave per receiver counting its neighbours over the
// image points pos_j + s.cell, a scan into the receiver CSR (the caller reads the edge count), then the same
// walk collecting the receiver's (src, s) keys in LDS, ranked there and written as edges.
#include "common.h"
#include "fsctep.h"
#include "scan.h"

namespace fsc {
namespace nbr {
namespace {

struct GridParams {
  double lo[3], hi[3], h[3];
  int32_t G[3];
  int32_t pad;
};

constexpr int KEY_IMAGES = 27;   // key = src * 27 + (sx+1)*9 + (sy+1)*3 + (sz+1)

__device__ __forceinline__ double dmul(double a, double b) { return __dmul_rn(a, b); }
__device__ __forceinline__ double dadd(double a, double b) { return __dadd_rn(a, b); }

// Block 0: the bounding box and the grid; the other blocks clear the cell counters (one launch for the three).
// Grid dimensions G_k = max(1, floor(extent_k / r)) (so cells are at least r wide), halving the largest while
// the product exceeds the cell budget.
__global__ __launch_bounds__(1024) void grid_kernel(int64_t N, const double* __restrict__ pos, double r,
                                                    int64_t cells_max, GridParams* __restrict__ g,
                                                    int32_t* __restrict__ cnt) {
  if (blockIdx.x > 0) {
    for (int64_t i = (int64_t)(blockIdx.x - 1) * 1024 + threadIdx.x; i < cells_max; i += (int64_t)(gridDim.x - 1) * 1024)
      cnt[i] = 0;
    return;
  }
  __shared__ double red[16][6];
  __shared__ double box[6];
  double v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  for (int64_t i = threadIdx.x; i < N; i += 1024) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double x = pos[3 * i + k];
      if (isfinite(x)) {
        v[k] = fmin(v[k], x);
        v[3 + k] = fmax(v[3 + k], x);
      }
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_xor(v[k], off, 64);
      v[k] = k < 3 ? fmin(v[k], o) : fmax(v[k], o);
    }
    if (lane == 0) red[wave][k] = v[k];
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    double v1 = red[0][k];
    for (int w = 1; w < 16; ++w) v1 = k < 3 ? fmin(v1, red[w][k]) : fmax(v1, red[w][k]);
    box[k] = v1;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  int64_t G[3];
  for (int k = 0; k < 3; ++k) {
    double lo = box[k], hi = box[3 + k];
    if (!(hi >= lo)) lo = hi = 0.0;   // no finite coordinate on this axis
    const double ext = hi - lo;
    double gk = floor(ext / r);
    gk = gk < 1.0 ? 1.0 : (gk > 1024.0 ? 1024.0 : gk);
    G[k] = (int64_t)gk;
    g->lo[k] = lo;
    g->hi[k] = hi;
  }
  while (G[0] * G[1] * G[2] > cells_max) {
    int m = 0;
    if (G[1] > G[m]) m = 1;
    if (G[2] > G[m]) m = 2;
    G[m] = G[m] > 1 ? G[m] / 2 : 1;
  }
  for (int k = 0; k < 3; ++k) {
    const double ext = g->hi[k] - g->lo[k];
    g->G[k] = (int32_t)G[k];
    g->h[k] = ext > 0.0 ? ext / (double)G[k] : 1.0;
  }
  g->pad = 0;
}

// Cell coordinate along axis k: floor((x - lo) / h) clamped to [0, G-1]; monotone in x, NaN -> 0.
__device__ __forceinline__ int cell_coord(const GridParams& g, int k, double x) {
  const double t = (x - g.lo[k]) / g.h[k];
  if (!(t >= 0.0)) return 0;
  if (t >= (double)(g.G[k] - 1)) return g.G[k] - 1;
  return (int)t;
}

__global__ __launch_bounds__(256) void assign_kernel(int64_t N, const double* __restrict__ pos,
                                                     const GridParams* __restrict__ gp, int32_t* __restrict__ atom_cell,
                                                     int32_t* __restrict__ cnt, int32_t* __restrict__ slot) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= N) return;
  const GridParams g = *gp;
  const int c = (cell_coord(g, 0, pos[3 * i]) * g.G[1] + cell_coord(g, 1, pos[3 * i + 1])) * g.G[2] +
                cell_coord(g, 2, pos[3 * i + 2]);
  atom_cell[i] = c;
  slot[i] = atomicAdd(cnt + c, 1);
}

// Atoms and positions in cell order (unordered within a cell: the keys are ranked at the end).
__global__ __launch_bounds__(256) void place_kernel(int64_t N, const double* __restrict__ pos,
                                                    const int32_t* __restrict__ atom_cell,
                                                    const int32_t* __restrict__ cell_start,
                                                    const int32_t* __restrict__ slot, int32_t* __restrict__ cell_atoms,
                                                    double* __restrict__ cell_pos) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= N) return;
  const int64_t o = cell_start[atom_cell[i]] + slot[i];
  cell_atoms[o] = (int32_t)i;
#pragma unroll
  for (int k = 0; k < 3; ++k) cell_pos[3 * o + k] = pos[3 * i + k];
}

struct Walk {
  const double* cell;   // [3][3], rows = lattice vectors
  const GridParams* grid;
  const int32_t* cell_start;
  const int32_t* cell_atoms;
  const double* cell_pos;   // positions in the order of cell_atoms
  int64_t N;
  int32_t pbc[3];
  double r2, reach;     // r^2 for the test; r (1 + 1e-9) for the cell range
};

// One wave visits every (i, s) within r of the receiver j at place p of the cell order (see the file
// comment).  The loops over the image shifts and the cell columns in range are uniform in the wave.  The cells
// of a column (consecutive along z) are consecutive in the cell order, so a column's candidates are one run,
// taken 64 at a time (about 40 in the three cells of side 5 at 0.1 atoms per cubic unit; a cell alone holds
// 13); the lanes test the images against the box at once, which leaves one to eight to walk.  A step's hits
// are numbered in lane order by a ballot and a prefix popcount; f(hit, key, rank) is called by every lane
// for each step with hits (rank: the hit's position among the receiver's hits so far).  Returns the number
// visited.  Count and fill at 10,000 atoms and 52 neighbours: 28 and 39 us (70 and 97 us with 16 lanes per
// receiver, cell by cell, and the keys through memory to a rank kernel); bound by the fp64 arithmetic of the
// candidates and the latency of nine columns one after the other.
template <typename F>
__device__ __forceinline__ int32_t walk_receiver(const Walk& w, int64_t p0, int lane, F&& f) {
  const GridParams& g = *w.grid;
  const int32_t j = w.cell_atoms[p0];
  const double pj[3] = {w.cell_pos[3 * p0], w.cell_pos[3 * p0 + 1], w.cell_pos[3 * p0 + 2]};
  const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
  const auto image = [&](int code, double* sv, double* p) {   // image code's shift and the receiver's image point
    const double s0 = code / 9 - 1, s1 = (code / 3) % 3 - 1, s2 = code % 3 - 1;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      sv[k] = dadd(dadd(dmul(s0, w.cell[k]), dmul(s1, w.cell[3 + k])), dmul(s2, w.cell[6 + k]));
      p[k] = pj[k] + sv[k];
    }
  };
  // lane c tests image c: no atom lies outside [lo, hi], so an image point farther than r from the box has no
  // neighbours (a non-finite one neither)
  uint64_t images;
  {
    const int code = lane < KEY_IMAGES ? lane : 0;
    bool on = lane < KEY_IMAGES && abs(code / 9 - 1) <= w.pbc[0] && abs((code / 3) % 3 - 1) <= w.pbc[1] &&
              abs(code % 3 - 1) <= w.pbc[2];
    double sv[3], p[3];
    image(code, sv, p);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (!(p[k] == p[k]) || p[k] + w.reach < g.lo[k] || p[k] - w.reach > g.hi[k]) on = false;
    images = __ballot(on);
  }
  int32_t n = 0;
  for (; images; images &= images - 1) {
    const int code = __ffsll((unsigned long long)images) - 1;
    double sv[3], p[3];
    image(code, sv, p);
    int clo[3], chi[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      clo[k] = cell_coord(g, k, p[k] - w.reach);
      chi[k] = cell_coord(g, k, p[k] + w.reach);
    }
    const bool self_image = code == KEY_IMAGES / 2;
    const int ny = chi[1] - clo[1] + 1, ncol = (chi[0] - clo[0] + 1) * ny;
    for (int c0 = 0; c0 < ncol; c0 += 64) {
      // lane c holds the bounds of column c0 + c
      const int col = c0 + lane;
      int32_t qb_l = 0, qe_l = 0;
      if (col < ncol) {
        const int c = ((clo[0] + col / ny) * g.G[1] + clo[1] + col % ny) * g.G[2];
        qb_l = w.cell_start[c + clo[2]];
        qe_l = w.cell_start[c + chi[2] + 1];
      }
      const int nc = ncol - c0 < 64 ? ncol - c0 : 64;
      for (int cc = 0; cc < nc; ++cc) {
        const int32_t qb = __builtin_amdgcn_readlane(qb_l, cc), qe = __builtin_amdgcn_readlane(qe_l, cc);
        for (int32_t q0 = qb; q0 < qe; q0 += 64) {
          const int32_t q = q0 + lane;
          bool hit = false;
          int32_t i = 0;
          if (q < qe) {
            i = w.cell_atoms[q];
            const double dx = dadd(pj[0] - w.cell_pos[3 * (int64_t)q], sv[0]);
            const double dy = dadd(pj[1] - w.cell_pos[3 * (int64_t)q + 1], sv[1]);
            const double dz = dadd(pj[2] - w.cell_pos[3 * (int64_t)q + 2], sv[2]);
            const double d2 = dadd(dadd(dmul(dx, dx), dmul(dy, dy)), dmul(dz, dz));
            hit = d2 < w.r2 && !(self_image && i == j);
          }
          const uint64_t mask = __ballot(hit);
          if (mask) {
            f(hit, (int64_t)i * KEY_IMAGES + code, n + __popcll(mask & below));
            n += __popcll(mask);
          }
        }
      }
    }
  }
  return n;
}

// Four receivers per block, in cell order: the waves that run together read the same cells.
__global__ __launch_bounds__(256) void count_kernel(Walk w, int32_t* __restrict__ deg) {
  const int64_t p = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (p >= w.N) return;
  const int lane = threadIdx.x & 63;
  const int32_t n = walk_receiver(w, p, lane, [](bool, int64_t, int32_t) {});
  if (lane == 0) deg[w.cell_atoms[p]] = n;
}

constexpr int KEY_CAP = 512;   // neighbours of a receiver whose keys are ranked in LDS (as 32-bit keys)

__device__ __forceinline__ void write_edge(int64_t o, int64_t key, int64_t j, int64_t* __restrict__ edge_src,
                                           int64_t* __restrict__ edge_dst, double* __restrict__ edge_shifts) {
  const int64_t i = key / KEY_IMAGES;
  const int code = (int)(key - i * KEY_IMAGES);
  edge_src[o] = i;
  edge_dst[o] = j;
  edge_shifts[3 * o] = (double)(code / 9 - 1);
  edge_shifts[3 * o + 1] = (double)((code / 3) % 3 - 1);
  edge_shifts[3 * o + 2] = (double)(code % 3 - 1);
}

// Ranks of the deg keys at `keys` (in memory, written by this wave), and their edges: a lane holds R keys, and all keys
// pass by through the wave's part of LDS, as Key, CAP of them at a time (padded with the largest Key, compared 16 bytes
// at a time).  Read past the L1, whose lines the segments of other receivers share.  3,000 receivers of 817 neighbours,
// count and fill: 1.98 ms with a thread an edge over keys in memory, 2.23 ms with a wave a receiver over them, 0.47 ms
// here; 2,000 of 920: 1.64, 2.38, 0.37 ms.
template <typename Key, int R>
__device__ __forceinline__ void rank_long(const int64_t* keys, int32_t deg, int lane, uint4* lds, int64_t beg, int64_t j,
                                          int64_t* __restrict__ edge_src, int64_t* __restrict__ edge_dst,
                                          double* __restrict__ edge_shifts) {
  constexpr int CAP = KEY_CAP * 4 / (int)sizeof(Key), PER = 16 / (int)sizeof(Key);
  Key* mine = reinterpret_cast<Key*>(lds);
  const auto load = [&](int32_t t) {
    return (Key)__hip_atomic_load(keys + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  for (int32_t t0 = 0; t0 < deg; t0 += 64 * R) {
    Key key[R];
    int32_t rank[R];
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int32_t t = t0 + 64 * u + lane;
      key[u] = load(t < deg ? t : deg - 1);
      rank[u] = 0;
    }
    for (int32_t c0 = 0; c0 < deg; c0 += CAP) {
      const int32_t n = deg - c0 < CAP ? deg - c0 : CAP;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the last keys are read
#pragma unroll
      for (int32_t i = lane; i < CAP; i += 64) mine[i] = i < n ? load(c0 + i) : ~Key(0);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (int32_t q = 0; PER * q < n; ++q) {
        Key o[PER];
        *reinterpret_cast<uint4*>(o) = lds[q];
#pragma unroll
        for (int u = 0; u < R; ++u)
#pragma unroll
          for (int v = 0; v < PER; ++v) rank[u] += o[v] < key[u];
      }
    }
#pragma unroll
    for (int u = 0; u < R; ++u)
      if (t0 + 64 * u + lane < deg) write_edge(beg + rank[u], (int64_t)key[u], j, edge_src, edge_dst, edge_shifts);
  }
}

// Keys of one receiver per wave, then each key's rank among them, which is its place in the receiver's
// segment.  Up to KEY_CAP keys that fit 32 bits (159 million atoms) stay in LDS, padded with the largest key
// so that they are compared four at a time; the others go through `keys` (rank_long).
__global__ __launch_bounds__(256) void fill_kernel(Walk w, const int32_t* __restrict__ dst_ptr, int64_t E, int64_t* keys,
                                                   int64_t* __restrict__ edge_src, int64_t* __restrict__ edge_dst,
                                                   double* __restrict__ edge_shifts) {
  __shared__ uint4 lkeys[4][KEY_CAP / 4];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t p = (int64_t)blockIdx.x * 4 + wave;
  if (p >= w.N) return;   // no barrier below: each wave works on its own keys
  const int lane = threadIdx.x & 63;
  const int64_t j = w.cell_atoms[p];
  const int64_t beg = dst_ptr[j], end = dst_ptr[j + 1] < E ? dst_ptr[j + 1] : E;
  if (end <= beg) return;   // no neighbours, or a segment past a caller's E: the accesses below take deg > 0
  const int32_t deg = (int32_t)(end - beg);
  // the counts came from the same walk, so rank < deg holds unless E cuts the segment: kept as a bound
  const bool small_keys = w.N < (int64_t)(UINT32_MAX / KEY_IMAGES);
  if (deg <= KEY_CAP && small_keys) {
    uint32_t* mine = reinterpret_cast<uint32_t*>(lkeys[wave]);
    if (lane < 4 && (deg & ~3) + lane < KEY_CAP) mine[(deg & ~3) + lane] = UINT32_MAX;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    walk_receiver(w, p, lane, [&](bool hit, int64_t key, int32_t rank) {
      if (hit && rank < deg) mine[rank] = (uint32_t)key;
    });
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int32_t t = lane; t < deg; t += 64) {
      const uint32_t key = mine[t];
      int32_t rank = 0;
      for (int32_t q = 0; 4 * q < deg; ++q) {
        const uint4 o = lkeys[wave][q];
        rank += (o.x < key) + (o.y < key) + (o.z < key) + (o.w < key);
      }
      write_edge(beg + rank, key, j, edge_src, edge_dst, edge_shifts);
    }
  } else {
    walk_receiver(w, p, lane, [&](bool hit, int64_t key, int32_t rank) {
      if (hit && rank < deg) __hip_atomic_store(keys + beg + rank, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    });
    __threadfence();
    if (small_keys)
      rank_long<uint32_t, 4>(keys + beg, deg, lane, lkeys[wave], beg, j, edge_src, edge_dst, edge_shifts);
    else
      rank_long<uint64_t, 2>(keys + beg, deg, lane, lkeys[wave], beg, j, edge_src, edge_dst, edge_shifts);
  }
}

int64_t cells_budget(int64_t N) {
  const int64_t c = 2 * N > 64 ? 2 * N : 64;
  return c < (int64_t(1) << 24) ? c : (int64_t(1) << 24);
}

struct NbrWs {
  int64_t cnt, grid, cell_pos, cell_start, tot, atom_cell, cell_atoms, deg, total, cells, nb;
};

NbrWs nbr_ws(int64_t N) {
  NbrWs w;
  w.cells = cells_budget(N);
  w.nb = (w.cells + 1 + SCAN_TILE - 1) / SCAN_TILE;
  int64_t o = 0;
  w.cnt = o;        o += w.cells;
  o = (o + 1) & ~int64_t(1);        // 8-byte alignment of the double fields
  w.grid = o;       o += (int64_t)(sizeof(GridParams) / 4);
  w.cell_pos = o;   o += 6 * N;
  w.cell_start = o; o += w.cells + 1;
  w.tot = o;        o += w.nb;
  w.atom_cell = o;  o += N;
  w.cell_atoms = o; o += N;
  w.deg = o;        o += N;
  w.total = o;
  return w;
}

Walk make_walk(int64_t N, const double* cell, const int32_t* pbc, double cutoff, int32_t* ws, const NbrWs& w) {
  Walk k;
  k.cell = cell;
  k.grid = reinterpret_cast<const GridParams*>(ws + w.grid);
  k.cell_start = ws + w.cell_start;
  k.cell_atoms = ws + w.cell_atoms;
  k.cell_pos = reinterpret_cast<const double*>(ws + w.cell_pos);
  k.N = N;
  for (int a = 0; a < 3; ++a) k.pbc[a] = pbc[a] ? 1 : 0;
  k.r2 = cutoff * cutoff;
  k.reach = cutoff * (1.0 + 1e-9);
  return k;
}

}  // namespace
}  // namespace nbr
}  // namespace fsc

using namespace fsc;
using namespace fsc::nbr;

extern "C" {

int fsc_neighbor_workspace(int64_t n_nodes, int64_t* workspace_ints) {
  FSC_CHECK_ARG(workspace_ints, "fsc_neighbor_workspace: null pointer");
  FSC_CHECK_ARG(n_nodes >= 0 && n_nodes < (1LL << 31) - 1, "fsc_neighbor_workspace: bad node count");
  *workspace_ints = nbr_ws(n_nodes).total;
  return 0;
}

int fsc_neighbor_count(int64_t n_nodes, const double* pos, const double* cell, const int32_t* pbc, double cutoff,
                       int32_t* dst_ptr, int32_t* workspace, hipStream_t stream) {
  FSC_CHECK_ARG(n_nodes >= 0 && n_nodes < (1LL << 31) - 1, "fsc_neighbor_count: bad node count");
  FSC_CHECK_ARG(pbc && dst_ptr && workspace && (n_nodes == 0 || (pos && cell)), "fsc_neighbor_count: null pointer");
  FSC_CHECK_ARG(cutoff > 0.0 && cutoff < 1e30, "fsc_neighbor_count: cutoff must be positive and finite");
  const int64_t N = n_nodes;
  const NbrWs w = nbr_ws(N);
  int32_t* ws = workspace;
  if (N == 0) {
    fill_i32_kernel<<<1, 256, 0, stream>>>(dst_ptr, 1, 0);
    return check_launch("fsc_neighbor_count") ? 2 : 0;
  }
  GridParams* gp = reinterpret_cast<GridParams*>(ws + w.grid);
  const int64_t fill_blocks = (w.cells + 4095) / 4096;
  grid_kernel<<<(unsigned)(1 + (fill_blocks < 255 ? fill_blocks : 255)), 1024, 0, stream>>>(N, pos, cutoff, w.cells, gp,
                                                                                           ws + w.cnt);
  int32_t* slot = ws + w.deg;   // the degrees come later
  assign_kernel<<<grid_of(N), 256, 0, stream>>>(N, pos, gp, ws + w.atom_cell, ws + w.cnt, slot);
  ScanArgs sa;
  sa.cnt[0] = sa.cnt[1] = ws + w.cnt;
  sa.out[0] = sa.out[1] = ws + w.cell_start;
  sa.tot[0] = sa.tot[1] = ws + w.tot;
  sa.n = w.cells;
  FSC_CHECK_ARG(w.nb <= SCAN_MAX_BLOCKS, "fsc_neighbor_count: too many cells for the scan");
  launch_scan(sa, 1, stream);
  place_kernel<<<grid_of(N), 256, 0, stream>>>(N, pos, ws + w.atom_cell, ws + w.cell_start, slot, ws + w.cell_atoms,
                                               reinterpret_cast<double*>(ws + w.cell_pos));
  const Walk walk = make_walk(N, cell, pbc, cutoff, ws, w);
  count_kernel<<<(unsigned)((N + 3) / 4), 256, 0, stream>>>(walk, ws + w.deg);
  // receiver CSR: exclusive scan of the degrees into dst_ptr[0..N]
  const int64_t nbn = (N + 1 + SCAN_TILE - 1) / SCAN_TILE;
  FSC_CHECK_ARG(nbn <= SCAN_MAX_BLOCKS, "fsc_neighbor_count: too many nodes for the scan");
  ScanArgs sd;
  sd.cnt[0] = sd.cnt[1] = ws + w.deg;
  sd.out[0] = sd.out[1] = dst_ptr;
  sd.tot[0] = sd.tot[1] = ws + w.cnt;   // the cell counts are dead once cell_start is built
  sd.n = N;
  launch_scan(sd, 1, stream);
  return check_launch("fsc_neighbor_count") ? 2 : 0;
}

int fsc_neighbor_fill(int64_t n_nodes, int64_t n_edges, const double* pos, const double* cell, const int32_t* pbc,
                      double cutoff, const int32_t* dst_ptr, int32_t* workspace, int32_t* fill_ws, int64_t* edge_src,
                      int64_t* edge_dst, double* edge_shifts, hipStream_t stream) {
  FSC_CHECK_ARG(n_nodes >= 0 && n_edges >= 0 && n_edges < (1LL << 31) - 1, "fsc_neighbor_fill: bad size");
  FSC_CHECK_ARG(pbc && dst_ptr && workspace, "fsc_neighbor_fill: null pointer");
  if (n_nodes == 0 || n_edges == 0) return 0;
  FSC_CHECK_ARG(pos && cell && fill_ws && edge_src && edge_dst && edge_shifts, "fsc_neighbor_fill: null pointer");
  const int64_t N = n_nodes, E = n_edges;
  const NbrWs w = nbr_ws(N);
  int64_t* keys = reinterpret_cast<int64_t*>(fill_ws);   // 2E int32, 8-byte aligned by the caller
  const Walk walk = make_walk(N, cell, pbc, cutoff, workspace, w);
  fill_kernel<<<(unsigned)((N + 3) / 4), 256, 0, stream>>>(walk, dst_ptr, E, keys, edge_src, edge_dst, edge_shifts);
  return check_launch("fsc_neighbor_fill") ? 2 : 0;
}

}  // extern "C"
