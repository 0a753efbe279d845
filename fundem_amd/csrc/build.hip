// Candidate-list builds of a step in a handful of launches, for planar or no
// periodicity and one or several systems.
//
// A build's stages each have little work (a few microseconds for 1e5 bodies),
// so what a build costs is the number of dependent launches and the longest
// chain of loads in each. Stage by stage:
//   kBuildReset   cells of the previous tables back to empty, counters to 0
//   kBuildBodies  per body: grid state, sort key; its periodic images into the
//                 ghost sets (slots reserved per workgroup), each linked into
//                 its cell; the walls' table by one workgroup
//   sort          the particle table: one workgroup ranks up to 2048 keys in
//                 LDS, more go through the radix sort; cell ranges
//   kBuildFind    sixteen lanes per particle A search every set, a row of
//                 cells per lane; A's candidates are sorted by target in LDS
//                 and left in scratch, their number in the set's counts
//   scan          the counts of all sets
//   kBuildPairs   candidates to their places in the lists, the sets each
//                 particle has pairs in (touch)
// Ghosts are in linked lists per cell, in no order, and pairs are sorted by
// target (one pair per A, target and set), so the lists are deterministic.
// Measured against a sort, a scan and two searches (count, write; one thread
// per particle) per set, 118 launches: a step of 110592 periodic particles
// that builds lists every 1.6 steps 473 -> 240 us (195 with the sweep's law
// and kBuildBodies as they are), of 216 particles (a build every 24 steps)
// 90.7 -> 69.8 us.
#include <algorithm>

#include "cull_device.hpp"
#include "fdm_device.hpp"
#include "fdm_launch.hpp"

namespace fdm {
namespace {

constexpr int kSets = 5;         // particle, wall, ghost X, Y, XY
constexpr int kFindLanes = 16;   // lanes per particle in kBuildFind
constexpr int kFindMax = 32;     // candidates of one particle and set sorted in LDS
constexpr int kSmallSort = 2048;
constexpr int kSmallWalls = 1024;
constexpr int kScanChunk = 8192;  // counts one workgroup scans in one launch

struct BuildK {
  fdm_bodies P, W;
  fdm_geometry pgeo, wgeo;
  fdm_grid pgrid, wgrid;
  fdm_hash_table ptable, wtable;
  fdm_periodic periodic;
  fdm_instances inst;
  fdm_ghosts ghosts[3];  // count NULL: no such set
  fdm_pairs sets[kSets]; // count NULL: no such set, or (particle, wall) kept
  const int* bondStart;
  double skin, maxRadius, maxBoxReach;
  int full, wallTable;
  int* touch;
  int* tmp[kSets];       // [2 * capacity] candidates: target and ghost index
  int* tmpOff;           // [5 * n] first candidate of (set, particle); -1: search again
  unsigned* status;
};

__global__ void __launch_bounds__(256) kBuildReset(BuildK k) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  auto clear = [&](const fdm_hash_table& t, long long num, bool ends) {
    const int pc = *t.prevCount;
    const long long n = pc < 0 ? num : pc;
    for (long long i = i0; i < n; i += stride) {
      const long long h = pc < 0 ? i : (long long)t.prevKey[i] - 1;
      if (h < 0 || h >= num) continue;
      t.cellStart[h] = -1;
      if (ends) t.cellEnd[h] = -1;
    }
  };
  if (k.full) clear(k.ptable, k.pgrid.num, true);
  for (int s = 0; s < 3; ++s) {
    if (!k.ghosts[s].count) continue;
    clear(k.ghosts[s].table, k.pgrid.num, false);
    if (i0 == 0) *k.ghosts[s].count = 0;
    if (i0 < 6) k.ghosts[s].cellBox[i0] = i0 < 3 ? INT_MAX : INT_MIN;
  }
}

// Stable order of n <= 2048 keys by one workgroup: a key's place is the number
// of smaller keys and of equal keys before it.
__device__ void rankSort(const unsigned* keys, int n, unsigned* outKey, int* outIndex) {
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    const unsigned mine = keys[j];
    int rank = 0;
    for (int i = 0; i < n; ++i) rank += keys[i] < mine || (keys[i] == mine && i < j) ? 1 : 0;
    outKey[rank] = mine;
    outIndex[rank] = j;
  }
}
// Half-open ranges of the cells of a sorted key list, and the keys for the
// next reset.
__device__ void markCells(const unsigned* sorted, int n, const fdm_hash_table& t, long long num) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const unsigned key = sorted[i];
    t.sortKey[i] = key;
    t.prevKey[i] = (int)key;
    const long long h = (long long)key - 1;
    if (h < 0 || h >= num) continue;
    if (i == 0 || sorted[i - 1] != key) t.cellStart[h] = i;
    if (i == n - 1 || sorted[i + 1] != key) t.cellEnd[h] = i + 1;
  }
  if (threadIdx.x == 0) *t.prevCount = n;
}

constexpr int kBodyThreads = 512;
template <bool MANY>
__global__ void __launch_bounds__(kBodyThreads) kBuildBodies(BuildK k, int particleBlocks) {
  if ((int)blockIdx.x == particleBlocks) {  // the walls' table
    __shared__ unsigned keys[kSmallWalls], sorted[kSmallWalls];
    const int W = k.W.n;
    for (int j = threadIdx.x; j < W; j += blockDim.x) {
      const int in = MANY ? k.inst.wallInstance[j] : 0;
      const fdm_grid g = MANY ? k.inst.wgrid[in] : k.wgrid;
      const V3 x = ldp(k.W.x, W, j);
      const int h = cellHash(x, g);
      k.wtable.validAtBuild[j] = bodyState(x, g);
      keys[j] = MANY ? instanceKey(h, g, k.inst.wcellOffset[in]) : (unsigned)(h + 1);
    }
    const int pc = *k.wtable.prevCount;
    const long long nc = pc < 0 ? k.wgrid.num : pc;
    for (long long i = threadIdx.x; i < nc; i += blockDim.x) {
      const long long h = pc < 0 ? i : (long long)k.wtable.prevKey[i] - 1;
      if (h < 0 || h >= k.wgrid.num) continue;
      k.wtable.cellStart[h] = -1;
      k.wtable.cellEnd[h] = -1;
    }
    __syncthreads();
    rankSort(keys, W, sorted, k.wtable.sortIndex);
    __syncthreads();
    markCells(sorted, W, k.wtable, k.wgrid.num);
    return;
  }
  // the workgroup's images of each set: their number and first slot, and the
  // box of their cells (one global atomic each per workgroup: taken per image,
  // in turn, they made up most of this kernel's time: 110592 particles 49.9 ->
  // 18.7 us, 216 particles 28.7 -> 13.7 us)
  __shared__ int cnt[3], base[3], box[3][6];
  if (threadIdx.x < 3) cnt[threadIdx.x] = 0;
  if (threadIdx.x < 18) box[threadIdx.x / 6][threadIdx.x % 6] = threadIdx.x % 6 < 3 ? INT_MAX : INT_MIN;
  __syncthreads();
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = k.P.n;
  int bits = 0, mine[3] = {0, 0, 0};
  V3 gp[3];
  fdm_grid g = k.pgrid;
  long long off = 0;
  if (i < n) {
    const int in = MANY ? k.inst.particleInstance[i] : 0;
    if (MANY) {
      g = k.inst.pgrid[in];
      off = k.inst.pcellOffset[in];
    }
    const fdm_periodic per = MANY ? k.inst.periodic[in] : k.periodic;
    const V3 x = ldp(k.P.x, n, i);
    if (k.full) {
      const int h = cellHash(x, g);
      k.ptable.validAtBuild[i] = bodyState(x, g);
      k.ptable.sortKey[i] = MANY ? instanceKey(h, g, off) : (unsigned)(h + 1);
      k.ptable.sortIndex[i] = i;
    }
    if (k.periodic.x || k.periodic.y) {
      // the images that visibilityBits counts, in the reference's order
      const WrapStages w = wrapStages(x, g, per);
      gp[0] = ghostOf(w.afterX, g, 1);
      gp[1] = ghostOf(w.afterY, g, 2);
      gp[2] = ghostOf(w.afterY, g, 3);
      if (k.periodic.x && per.x && ghostCellHash(gp[0], g) >= 0) bits |= 1;
      if (k.periodic.y && per.y && ghostCellHash(gp[1], g) >= 0) bits |= 2;
      if (k.periodic.x && k.periodic.y && per.x && per.y && ghostCellHash(gp[2], g) >= 0) bits |= 4;
      k.ghosts[k.periodic.x ? 0 : 1].atBuild[i] = bits;
    }
    const int keep = k.full ? 0
                            : k.touch[i] & (FDM_TOUCH_A(0) | FDM_TOUCH_T(0) | FDM_TOUCH_A(1) | FDM_TOUCH_BOND);
    k.touch[i] = keep | (k.full && k.bondStart && k.bondStart[i + 1] > k.bondStart[i] ? FDM_TOUCH_BOND : 0);
  }
  if (!(k.periodic.x || k.periodic.y)) return;
  // lists are built by the clamped geometric cell (monotone in the position);
  // the reference's ghost cell id decides the stencil rule
  long long cell[3] = {0, 0, 0};
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    if (!(bits >> s & 1)) continue;
    mine[s] = atomicAdd(&cnt[s], 1);
    const I3 c = clampedCell(gp[s], g);
    cell[s] = off + lin3(c, gsize(g));
    const int v[3] = {c.x, c.y, c.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      atomicMin(&box[s][a], v[a]);
      atomicMax(&box[s][3 + a], v[a]);
    }
  }
  __syncthreads();
  if (threadIdx.x < 3 && cnt[threadIdx.x] > 0) base[threadIdx.x] = atomicAdd(k.ghosts[threadIdx.x].count, cnt[threadIdx.x]);
  if (threadIdx.x >= 64 && threadIdx.x < 64 + 18) {
    const int s = (threadIdx.x - 64) / 6, a = (threadIdx.x - 64) % 6;
    if (cnt[s] > 0) {
      if (a < 3) atomicMin(&k.ghosts[s].cellBox[a], box[s][a]);
      else atomicMax(&k.ghosts[s].cellBox[a], box[s][a]);
    }
  }
  __syncthreads();
  int slot[3], next[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    if (!(bits >> s & 1)) continue;
    slot[s] = base[s] + mine[s];
    if (slot[s] >= k.ghosts[s].capacity) {
      atomicOr(k.status, FDM_STATUS_GHOST_OVERFLOW);
      bits &= ~(1 << s);
    } else {
      next[s] = atomicExch(&k.ghosts[s].table.cellStart[cell[s]], slot[s]);
    }
  }
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    if (!(bits >> s & 1)) continue;
    const fdm_ghosts& G = k.ghosts[s];
    G.realId[slot[s]] = i;
    G.pos[3 * slot[s]] = gp[s].x;
    G.pos[3 * slot[s] + 1] = gp[s].y;
    G.pos[3 * slot[s] + 2] = gp[s].z;
    G.table.hashValue[slot[s]] = ghostCellHash(gp[s], g);
    G.table.prevKey[slot[s]] = (int)(cell[s] + 1);
    G.table.sortIndex[slot[s]] = next[s];
  }
}

__global__ void __launch_bounds__(1024) kBuildSortSmall(BuildK k) {
  __shared__ unsigned keys[kSmallSort], sorted[kSmallSort];
  const int n = k.P.n;
  for (int j = threadIdx.x; j < n; j += blockDim.x) keys[j] = k.ptable.sortKey[j];
  __syncthreads();
  rankSort(keys, n, sorted, k.ptable.sortIndex);
  __syncthreads();
  markCells(sorted, n, k.ptable, k.pgrid.num);
}
__global__ void __launch_bounds__(256) kBuildMark(fdm_hash_table t, int n, long long num) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) *t.prevCount = n;
  if (i >= n) return;
  const unsigned key = t.sortKey[i];
  t.prevKey[i] = (int)key;
  const long long h = (long long)key - 1;
  if (h < 0 || h >= num) return;
  if (i == 0 || t.sortKey[i - 1] != key) t.cellStart[h] = i;
  if (i == n - 1 || t.sortKey[i + 1] != key) t.cellEnd[h] = i + 1;
}

// Whether a pair may get a node contact while its bodies move less than half
// the skin each: a necessary condition of a contact with every reach widened
// by the skin. The target's cell codes bound its level set as in the sweep:
// no contact lies nearer to A's centre than the nearest point p of the SDF
// box, nor nearer to p than the code of p's cell tells.
// Walls also take the Lipschitz bound of their level set (a plane's is 1; its
// one cell has code 0). WALL: no bounding sphere either.
template <bool SPHERE, bool WALL = false>
__device__ __forceinline__ bool acceptPair(const fdm_bodies& B, const fdm_geometry& geo, int T, V3 xT, V3 xA,
                                           double RA, double skin, double reachMax) {
  const V3 d = vsub(xA, xT);
  const double d2 = vlen2(d);
  const double far = (RA + reachMax) * kReach + skin;
  if (d2 > far * far) return false;  // before the target's own template is known
  const fdm_template t = ldu(geo.info + ldu(B.geo + T));
  const double rs = (RA + (SPHERE ? t.radius : t.boxReach)) * kReach + skin;
  if (d2 > rs * rs) return false;
  const Q4 q = {(double)B.q[T], (double)B.q[B.n + T], (double)B.q[2 * B.n + T], (double)B.q[3 * B.n + T]};
  const V3 local = qrotateT(d, q);
  const double reach = RA * kReach + skin;
  if (outsideBox(local, reach, t)) return false;
  if (WALL && lipschitzClear(local, reach, t, geo.sdf)) return false;
  if (!geo.cells) return true;
  const double u[3] = {(local.x - t.origin[0]) * t.invSpacing, (local.y - t.origin[1]) * t.invSpacing,
                       (local.z - t.origin[2]) * t.invSpacing};
  double e2 = 0.;
  int c[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double v = fmin(fmax(u[a], 0.), (double)(t.size[a] - 1));
    c[a] = min((int)v, t.size[a] - 2);
    e2 += (u[a] - v) * (u[a] - v);
  }
  const int code = geo.cells[t.cellStart + c[0] + (t.size[0] - 1) * (c[1] + (long long)(t.size[1] - 1) * c[2])];
  const double dist = (double)max(code - 1, 0) * (1.0 / FDM_CELL_UNIT), rr = reach * t.invSpacing * kReach + 1e-6;
  return e2 + dist * dist <= rr * rr;
}

// A's grid. (Opaque at each use: what is computed from a launch's one grid, as
// the periods, would otherwise be kept in registers over the loop of the sets.)
template <bool MANY>
__device__ __forceinline__ fdm_grid gridOf(const BuildK& k, int in) {
  if (MANY) return k.inst.pgrid[in];
  fdm_grid g = k.pgrid;
  asm volatile("" : "+s"(g.min.x), "+s"(g.min.y), "+s"(g.min.z), "+s"(g.max.x), "+s"(g.max.y));
  return g;
}

// Candidates of particle A in one set, by `lanes` lanes of which this is
// number `gl`: emit(target, ghost index) for each, in no order.
template <int SET, bool MANY, class Emit>
__device__ __forceinline__ void findPairs(const BuildK& k, int s, int A, V3 x, double RA, int in, int gl,
                                          int lanes, Emit emit) {
  const int n = k.P.n;
  if (SET == FDM_SET_WALL) {
    const int w0 = MANY ? k.inst.wallStart[in] : 0, w1 = MANY ? k.inst.wallStart[in + 1] : k.W.n;
    const long long num = MANY ? k.inst.wgrid[in].num : k.wgrid.num;
    for (int w = w0 + gl; w < w1; w += lanes) {
      const int h = k.wtable.hashValue[w];
      if (h < 0 || (long long)h >= num) continue;
      if (acceptPair<false, true>(k.W, k.wgeo, w, ldp(k.W.x, k.W.n, w), x, RA, k.skin, 1e300)) emit(w, w);
    }
    return;
  }
  const fdm_grid grid = gridOf<MANY>(k, in);
  const long long off = MANY ? k.inst.pcellOffset[in] : 0;
  const double reachMax = SET == FDM_SET_PARTICLE ? k.maxRadius : k.maxBoxReach;
  I3 b0, b1;
  cellRange(x, (RA + reachMax) * kReach + k.skin, grid, b0, b1);
  if (SET == FDM_SET_PARTICLE) {
    // joined with the reference's own stencil, which also covers a target
    // whose id aliases another cell in the step the lists are built
    I3 lo, hi;
    cellRange(x, RA * kReach + k.skin, grid, lo, hi);
    b0 = {min(b0.x, max(lo.x - 1, 0)), min(b0.y, max(lo.y - 1, 0)), min(b0.z, max(lo.z - 1, 0))};
    b1 = {max(b1.x, min(hi.x + 1, grid.size.x - 1)), max(b1.y, min(hi.y + 1, grid.size.y - 1)),
          max(b1.z, min(hi.z + 1, grid.size.z - 1))};
  } else {
    const int* box = k.ghosts[s - 2].cellBox;
    b0 = {max(b0.x, box[0]), max(b0.y, box[1]), max(b0.z, box[2])};
    b1 = {min(b1.x, box[3]), min(b1.y, box[4]), min(b1.z, box[5])};
  }
  const int ny = b1.y - b0.y + 1, nz = b1.z - b0.z + 1;
  if (b1.x < b0.x || ny <= 0 || nz <= 0) return;
  const I3 sz = gsize(grid);
  for (int r = gl; r < ny * nz; r += lanes) {
    const long long h0 = off + lin3({b0.x, b0.y + r % ny, b0.z + r / ny}, sz);
    if (SET == FDM_SET_PARTICLE) {
      // the cells of an x-row have consecutive ids, so the row's entries of
      // the sorted table form one range
      int m0 = INT_MAX, m1 = 0;
#pragma unroll 4
      for (int c = 0; c <= b1.x - b0.x; ++c) {
        const int cs = k.ptable.cellStart[h0 + c], ce = k.ptable.cellEnd[h0 + c];
        if (cs >= 0) {
          m0 = min(m0, cs);
          m1 = max(m1, ce);
        }
      }
      for (int m = m0; m < m1; ++m) {
        const int T = k.ptable.sortIndex[m];
        if (T > A && acceptPair<true>(k.P, k.pgeo, T, ldp(k.P.x, n, T), x, RA, k.skin, reachMax)) emit(T, T);
      }
    } else {
      const fdm_ghosts& G = k.ghosts[s - 2];
      for (int c = 0; c <= b1.x - b0.x; ++c)
        for (int m = G.table.cellStart[h0 + c]; m >= 0; m = G.table.sortIndex[m]) {
          const int T = G.realId[m];
          if (acceptPair<false>(k.P, k.pgeo, T, ldd3(G.pos + 3 * (size_t)m), x, RA, k.skin, reachMax)) emit(T, m);
        }
    }
  }
}

// Position of A that a set's detection sees: ghost contacts are detected after
// the periodic wrap.
template <bool MANY>
__device__ __forceinline__ V3 detectAt(const BuildK& k, int s, V3 x, int in) {
  if (s < 2) return x;
  return wrapPosition(x, gridOf<MANY>(k, in), MANY ? k.inst.periodic[in] : k.periodic);
}

// (four waves per SIMD instead of three, as the time is the chain of loads:
// 110592 particles 134 -> 117 us)
template <bool MANY>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) kBuildFind(BuildK k) {
  constexpr int G = 64 / kFindLanes;  // particles per wave
  struct Group {
    int n, t[kFindMax], g[kFindMax];
  };
  __shared__ Group lds[256 / kFindLanes];
  const int n = k.P.n;
  const int grp = threadIdx.x / kFindLanes, gl = threadIdx.x % kFindLanes;
  const int A = blockIdx.x * (256 / kFindLanes) + grp;
  const bool on = A < n;
  if (A == n && gl == 0)
    for (int s = 0; s < kSets; ++s)
      if (k.sets[s].count) k.sets[s].count[n] = 0;
  const int in = MANY && on ? k.inst.particleInstance[A] : 0;
  const V3 x = on ? ldp(k.P.x, n, A) : V3{0., 0., 0.};
  const double RA = on ? ldu(&k.pgeo.info[ldu(k.P.geo + A)].radius) : 0.;
  Group& L = lds[grp];
#pragma unroll 1
  for (int s = 0; s < kSets; ++s) {
    if (!k.sets[s].count) continue;
    if (gl == 0) L.n = 0;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (on) {
      const V3 xA = detectAt<MANY>(k, s, x, in);
      auto emit = [&](int T, int g) {
        const int slot = atomicAdd(&L.n, 1);
        if (slot < kFindMax) {
          L.t[slot] = T;
          L.g[slot] = g;
        }
      };
      if (s == 0) findPairs<FDM_SET_PARTICLE, MANY>(k, s, A, xA, RA, in, gl, kFindLanes, emit);
      else if (s == 1) findPairs<FDM_SET_WALL, MANY>(k, s, A, xA, RA, in, gl, kFindLanes, emit);
      else findPairs<FDM_SET_GHOST, MANY>(k, s, A, xA, RA, in, gl, kFindLanes, emit);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // the wave's share of the scratch, dealt to its particles in order
    const int c = on ? L.n : 0;
    int before = 0, all = 0;
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int cj = __shfl(c, j * kFindLanes);
      if (j < (int)(threadIdx.x % 64) / kFindLanes) before += cj;
      all += cj;
    }
    const int share = G * (k.sets[s].capacity / max(n, 1));
    const long long wave = (long long)blockIdx.x * 4 + threadIdx.x / 64;
    const long long at = wave * share + before;
    const bool fits = c <= kFindMax && all <= share && at + c <= k.sets[s].capacity;
    if (on && fits)
      for (int e = gl; e < c; e += kFindLanes) {
        int rank = 0;
        for (int j = 0; j < c; ++j) rank += L.t[j] < L.t[e] ? 1 : 0;
        k.tmp[s][2 * (at + rank)] = L.t[e];
        k.tmp[s][2 * (at + rank) + 1] = L.g[e];
      }
    if (on && gl == 0) {
      k.sets[s].count[A] = c;
      k.tmpOff[(size_t)s * n + A] = fits ? (int)at : -1;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
}

// Exclusive scan in place of every set's n + 1 counts by one workgroup each.
__global__ void __launch_bounds__(1024) kBuildScanSmall(BuildK k) {
  __shared__ int wsum[16];
  const fdm_pairs& S = k.sets[blockIdx.x];
  if (!S.count) return;
  const int n = k.P.n + 1;
  constexpr int kEach = kScanChunk / 1024;
  int v[kEach], sum = 0;
#pragma unroll
  for (int j = 0; j < kEach; ++j) {
    const int i = threadIdx.x * kEach + j;
    v[j] = i < n ? S.count[i] : 0;
    sum += v[j];
  }
  int inc = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int t = __shfl_up(inc, off, 64);
    if (laneId() >= off) inc += t;
  }
  if (laneId() == 63) wsum[threadIdx.x >> 6] = inc;
  __syncthreads();
  int run = inc - sum, total = 0;
  for (int w = 0; w < 16; ++w) {
    if (w < (int)(threadIdx.x >> 6)) run += wsum[w];
    total += wsum[w];
  }
#pragma unroll
  for (int j = 0; j < kEach; ++j) {
    const int i = threadIdx.x * kEach + j;
    if (i < n) S.count[i] = run;
    run += v[j];
  }
  if (threadIdx.x == 0) *S.total = total;
}
// The same in three launches, tiles of kTile counts (sums: [5][tiles]).
constexpr int kTile = 2048;
__device__ __forceinline__ int blockScan256(int v, int* lds, int& total) {
  int inc = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int t = __shfl_up(inc, off, 64);
    if (laneId() >= off) inc += t;
  }
  const int nw = blockDim.x >> 6;
  if (laneId() == 63) lds[threadIdx.x >> 6] = inc;
  __syncthreads();
  int before = 0;
  total = 0;
  for (int w = 0; w < nw; ++w) {
    if (w < (int)(threadIdx.x >> 6)) before += lds[w];
    total += lds[w];
  }
  __syncthreads();
  return before + inc - v;
}
__global__ void __launch_bounds__(256) kBuildScanReduce(BuildK k, int* sums) {
  __shared__ int lds[4];
  const fdm_pairs& S = k.sets[blockIdx.y];
  if (!S.count) return;
  const int n = k.P.n + 1;
  int v = 0, total;
#pragma unroll
  for (int j = 0; j < kTile / 256; ++j) {
    const int i = blockIdx.x * kTile + j * 256 + threadIdx.x;
    if (i < n) v += S.count[i];
  }
  blockScan256(v, lds, total);
  if (threadIdx.x == 0) sums[blockIdx.y * gridDim.x + blockIdx.x] = total;
}
__global__ void __launch_bounds__(1024) kBuildScanSums(BuildK k, int* sums, int tiles) {
  __shared__ int lds[16];
  const fdm_pairs& S = k.sets[blockIdx.x];
  if (!S.count) return;
  int* row = sums + (size_t)blockIdx.x * tiles;
  int carry = 0;
  for (int b = 0; b < tiles; b += 1024) {
    const int i = b + threadIdx.x;
    const int v = i < tiles ? row[i] : 0;
    int total;
    const int ex = blockScan256(v, lds, total);
    if (i < tiles) row[i] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) *S.total = carry;
}
__global__ void __launch_bounds__(256) kBuildScanApply(BuildK k, const int* sums) {
  __shared__ int lds[4];
  const fdm_pairs& S = k.sets[blockIdx.y];
  if (!S.count) return;
  const int n = k.P.n + 1;
  constexpr int kEach = kTile / 256;
  int v[kEach], sum = 0, total;
#pragma unroll
  for (int j = 0; j < kEach; ++j) {
    const int i = blockIdx.x * kTile + threadIdx.x * kEach + j;
    v[j] = i < n ? S.count[i] : 0;
    sum += v[j];
  }
  int run = blockScan256(sum, lds, total) + sums[blockIdx.y * gridDim.x + blockIdx.x];
#pragma unroll
  for (int j = 0; j < kEach; ++j) {
    const int i = blockIdx.x * kTile + threadIdx.x * kEach + j;
    if (i < n) S.count[i] = run;
    run += v[j];
  }
}

template <bool MANY>
__global__ void __launch_bounds__(256) kBuildPairs(BuildK k) {
  const int s = blockIdx.y;
  const fdm_pairs& S = k.sets[s];
  if (!S.count) return;
  const int n = k.P.n;
  const int A = blockIdx.x * blockDim.x + threadIdx.x;
  if (A == 0 && s >= 2) {
    const fdm_ghosts& G = k.ghosts[s - 2];
    const int c = min(*G.count, G.capacity);
    *G.count = c;
    *G.table.prevCount = c;
  }
  if (A >= n) return;
  const int begin = S.count[A], end = S.count[A + 1];
  if (begin == end) return;
  if (end > S.capacity) {
    // mark the slots that fit as empty so the narrow phase skips them
    for (int w = begin; w < S.capacity; ++w) S.pairA[w] = -1;
    atomicOr(k.status, FDM_STATUS_PAIR_OVERFLOW);
    return;
  }
  const int at = k.tmpOff[(size_t)s * n + A];
  if (at >= 0) {
    for (int w = begin; w < end; ++w) {
      const int2 c = reinterpret_cast<const int2*>(k.tmp[s])[at + w - begin];
      S.pairA[w] = A;
      S.pairT[w] = c.x;
      S.pairG[w] = c.y;
    }
  } else {
    // more candidates than kBuildFind could keep: search again, one lane
    const int in = MANY ? k.inst.particleInstance[A] : 0;
    const double RA = ldu(&k.pgeo.info[ldu(k.P.geo + A)].radius);
    const V3 xA = detectAt<MANY>(k, s, ldp(k.P.x, n, A), in);
    int w = begin;
    auto emit = [&](int T, int g) {
      if (w >= end) return;
      int j = w++ - 1;
      for (; j >= begin && S.pairT[j] > T; --j) {
        S.pairT[j + 1] = S.pairT[j];
        S.pairG[j + 1] = S.pairG[j];
      }
      S.pairT[j + 1] = T;
      S.pairG[j + 1] = g;
    };
    if (s == 0) findPairs<FDM_SET_PARTICLE, MANY>(k, s, A, xA, RA, in, 0, 1, emit);
    else if (s == 1) findPairs<FDM_SET_WALL, MANY>(k, s, A, xA, RA, in, 0, 1, emit);
    else findPairs<FDM_SET_GHOST, MANY>(k, s, A, xA, RA, in, 0, 1, emit);
    for (int j = begin; j < end; ++j) S.pairA[j] = A;
  }
  atomicOr(&k.touch[A], FDM_TOUCH_A(s));
  if (s != 1)
    for (int w = begin; w < end; ++w) atomicOr(&k.touch[S.pairT[w]], FDM_TOUCH_T(s));
}

// Cell codes (FDM_CELL_UNIT) of every template, a cell per thread: which cells
// hold a corner at or below a millionth of the spacing (elsewhere the
// interpolant stays positive whatever its rounding), then the squared distance
// from a cell's box to the nearest such cell's, which is a sum over the axes
// and is folded axis by axis over the sixteen cells either way. Squares of 255
// and more have one code. A grid of more than kCellsMost cells keeps all codes
// 0 (nothing is culled by them). Four launches for all templates: 16 templates
// of 31^3 cells took 4 to 20 ms on the host, by compiler and options.
constexpr long long kCellsMost = 1ll << 22;
struct CellK {
  const fdm_template* t;
  int count;
  const float* sdf;
  unsigned char* cells;
  unsigned char *squares, *folded;  // squared distances, before and after an axis
};
__device__ __forceinline__ bool cellGrid(const fdm_template& t, int c[3], long long& n) {
  for (int a = 0; a < 3; ++a) c[a] = t.size[a] - 1;
  n = (long long)c[0] * c[1] * c[2];
  return n <= kCellsMost;
}
__global__ void __launch_bounds__(256) kCellSolid(CellK k) {
  for (int g = blockIdx.y; g < k.count; g += gridDim.y) {
    const fdm_template& t = k.t[g];
    int c[3];
    long long n;
    const bool told = cellGrid(t, c, n);
    const float low = (float)(1e-6 / t.invSpacing);
    const size_t sy = t.size[0], sz = sy * t.size[1];
    for (long long e = blockIdx.x * 256ll + threadIdx.x; e < n; e += gridDim.x * 256ll) {
      bool solid = false;
      if (told) {
        const int x = (int)e % c[0], y = (int)e / c[0] % c[1], z = (int)e / c[0] / c[1];
        const float* s = k.sdf + t.sdfStart + z * sz + y * sy + x;
#pragma unroll
        for (int q = 0; q < 8; ++q) solid |= s[(q & 1) + (q & 2 ? sy : 0) + (q & 4 ? sz : 0)] <= low;
      }
      k.cells[t.cellStart + e] = solid ? 1 : 0;
    }
  }
}
// AXIS 2 leaves the codes.
template <int AXIS>
__global__ void __launch_bounds__(256) kCellFold(CellK k) {
  constexpr int kFar = 255;
  for (int g = blockIdx.y; g < k.count; g += gridDim.y) {
    const fdm_template& t = k.t[g];
    int c[3];
    long long n;
    if (!cellGrid(t, c, n)) continue;
    const int stride = AXIS == 0 ? 1 : AXIS == 1 ? c[0] : c[0] * c[1];
    unsigned char* cells = k.cells + t.cellStart;
    const unsigned char* in = (AXIS == 1 ? k.squares : k.folded) + t.cellStart;
    unsigned char* out = (AXIS == 0 ? k.squares : k.folded) + t.cellStart;
    for (long long e = blockIdx.x * 256ll + threadIdx.x; e < n; e += gridDim.x * 256ll) {
      const int i = (int)e, at = i / stride % c[AXIS];
      auto square = [&](int j) { return AXIS == 0 ? (cells[j] ? 0 : kFar) : (int)in[j]; };
      int best = square(i);
      for (int gap = 0; gap < 16 && gap * gap < best; ++gap) {
        if (at > gap) best = min(best, gap * gap + square(i - (gap + 1) * stride));
        if (at + gap + 1 < c[AXIS]) best = min(best, gap * gap + square(i + (gap + 1) * stride));
      }
      if (AXIS < 2) out[i] = (unsigned char)best;
      else cells[i] = cells[i] ? 0 : (unsigned char)(1 + (int)floor(FDM_CELL_UNIT * sqrt((double)best) * (1.0 - 1e-9)));
    }
  }
}

template <bool MANY>
int launchBuild(const BuildK& k, void* ws, size_t wsBytes, hipStream_t stream) {
  const int n = k.P.n;
  const unsigned rb = std::max<unsigned>(1, std::min<unsigned>(blocksFor(std::max(n, 1), 256), 1024));
  hipLaunchKernelGGL(kBuildReset, dim3(rb), dim3(256), 0, stream, k);
  const int pb = (int)blocksFor(n, kBodyThreads);
  hipLaunchKernelGGL(kBuildBodies<MANY>, dim3(pb + (k.wallTable ? 1 : 0)), dim3(kBodyThreads), 0, stream, k, pb);
  if (k.full) {
    if (n <= kSmallSort) {
      hipLaunchKernelGGL(kBuildSortSmall, dim3(1), dim3(1024), 0, stream, k);
    } else {
      const int r = radixSort(k.ptable.sortKey, k.ptable.sortIndex, (size_t)n, nullptr, keyBitsFor(k.pgrid.num), ws,
                              wsBytes, stream);
      if (r != FDM_OK) return r;
      hipLaunchKernelGGL(kBuildMark, dim3(blocksFor(n, 256)), dim3(256), 0, stream, k.ptable, n, k.pgrid.num);
    }
  }
  hipLaunchKernelGGL(kBuildFind<MANY>, dim3(blocksFor(n + 1, 256 / kFindLanes)), dim3(256), 0, stream, k);
  if (n + 1 <= kScanChunk) {
    hipLaunchKernelGGL(kBuildScanSmall, dim3(kSets), dim3(1024), 0, stream, k);
  } else {
    const unsigned tiles = blocksFor(n + 1, kTile);
    if (wsBytes < kSets * tiles * sizeof(int)) return FDM_EINVAL;
    int* sums = (int*)ws;
    hipLaunchKernelGGL(kBuildScanReduce, dim3(tiles, kSets), dim3(256), 0, stream, k, sums);
    hipLaunchKernelGGL(kBuildScanSums, dim3(kSets), dim3(1024), 0, stream, k, sums, (int)tiles);
    hipLaunchKernelGGL(kBuildScanApply, dim3(tiles, kSets), dim3(256), 0, stream, k, sums);
  }
  hipLaunchKernelGGL(kBuildPairs<MANY>, dim3(blocksFor(n, 256), kSets), dim3(256), 0, stream, k);
  return launchStatus();
}

}  // namespace
}  // namespace fdm

using namespace fdm;

extern "C" size_t fdm_buildListsWorkspaceBytes(size_t n) {
  return std::max(radixWorkspace(n), alignUp(kSets * (size_t)blocksFor((long long)n + 1, kTile) * sizeof(int)));
}

extern "C" int fdm_launchBuildLists(const fdm_build_args* args, void* workspace, size_t workspaceBytes,
                                    hipStream_t stream) {
  if (!args) return FDM_EINVAL;
  const fdm_build_args& g = *args;
  const int n = g.particles.n;
  if (n < 0 || g.walls.n < 0 || !(g.skin >= 0.0) || g.periodic.sector) return FDM_EINVAL;
  if (!g.sets[0] || !g.touch || !g.tmpOff || !g.status) return FDM_EINVAL;
  if (n == 0) return FDM_OK;
  if (g.walls.n > kSmallWalls && g.full) return FDM_EINVAL;
  BuildK k{};
  k.P = g.particles;
  k.W = g.walls;
  k.pgeo = g.pgeo;
  k.wgeo = g.wgeo;
  k.pgrid = g.pgrid;
  k.wgrid = g.wgrid;
  k.ptable = g.ptable;
  k.wtable = g.wtable;
  k.periodic = g.periodic;
  k.inst = g.inst;
  k.bondStart = g.bonds && g.bonds->n > 0 ? g.bonds->partStart : nullptr;
  k.skin = g.skin;
  k.maxRadius = g.maxRadius;
  k.maxBoxReach = g.maxBoxReach;
  k.full = g.full ? 1 : 0;
  k.wallTable = g.full && g.walls.n > 0;
  k.touch = g.touch;
  k.tmpOff = g.tmpOff;
  k.status = g.status;
  long long words = 0;
  for (int s = 0; s < kSets; ++s) {
    if (s >= 2) {
      const bool active = ghostSetOn(g.periodic, s - 2);
      if (!active) continue;
      if (!g.sets[s] || !g.ghosts[s - 2] || !g.ghosts[s - 2]->atBuild) return FDM_EINVAL;
      k.ghosts[s - 2] = *g.ghosts[s - 2];
    } else if (!g.sets[s] || !g.full || (s == 1 && g.walls.n == 0)) {
      continue;
    }
    k.sets[s] = *g.sets[s];
    k.tmp[s] = g.tmp + words;
    words += 2ll * k.sets[s].capacity;
  }
  if (words > g.tmpWords || (words > 0 && !g.tmp)) return FDM_EINVAL;
  return g.inst.count > 0 ? launchBuild<true>(k, workspace, workspaceBytes, stream)
                          : launchBuild<false>(k, workspace, workspaceBytes, stream);
}

extern "C" int fdm_launchCellCodes(const fdm_template* templates, int count, long long mostCells, const float* sdf,
                                   unsigned char* cells, long long totalCells, void* workspace, size_t workspaceBytes,
                                   hipStream_t stream) {
  if (count < 0 || mostCells < 0 || totalCells < mostCells) return FDM_EINVAL;
  if (count == 0) return FDM_OK;
  if (!templates || !sdf || !cells || !workspace || workspaceBytes < 2 * (size_t)totalCells) return FDM_EINVAL;
  unsigned char* w = (unsigned char*)workspace;
  const CellK k = {templates, count, sdf, cells, w, w + totalCells};
  const dim3 grid(std::max<unsigned>(1, std::min<unsigned>(blocksFor(mostCells, 256), 1024)), std::min(count, 4096));
  hipLaunchKernelGGL(kCellSolid, grid, dim3(256), 0, stream, k);
  hipLaunchKernelGGL(kCellFold<0>, grid, dim3(256), 0, stream, k);
  hipLaunchKernelGGL(kCellFold<1>, grid, dim3(256), 0, stream, k);
  hipLaunchKernelGGL(kCellFold<2>, grid, dim3(256), 0, stream, k);
  return launchStatus();
}
