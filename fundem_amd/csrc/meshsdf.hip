// Signed distance of a closed triangle mesh sampled on a background grid, or
// at a list of points (LevelSetObject::TriangleMeshParticle,
// LevelSetObjectGenerator.h:382-951, with the grid sampling of
// Base::buildGrid, LevelSetObjectGenerator.h:122-224).
//
// The reference walks a SAH-BVH for the closest point and sums the solid
// angles of all triangles for the inside test, one point at a time on the
// host. Here both reductions run over every triangle: the workgroup stages
// 256 triangles at a time in LDS (SoA) and eight lanes share a point, each
// folding every eighth triangle, before the partials are combined: a grid of
// 70k nodes then runs 560k lanes, enough to keep every SIMD of the chip busy.
// A triangle whose bounding box is farther than the lane's best distance so
// far skips the closest-point test (the BVH's pruning, per lane); the solid
// angle is needed for every triangle. The closest distance is the
// exact minimum over triangles of the FP64 point-triangle distance; ties go
// to the lowest triangle index. Compute bound (FP64 VALU), not HBM: the
// triangles are read once per workgroup from L2.
#include <algorithm>
#include <cfloat>
#include <climits>

#include "fdm_device.hpp"
#include "fdm_launch.hpp"

namespace fdm {

namespace {

constexpr int kMeshTile = 256;

// Closest point of triangle abc to p (Ericson's Voronoi-region walk), in the
// operation order of closestPointOnTriangle (LevelSetObjectGenerator.h:454-495).
__device__ __forceinline__ V3 closestOnTriangle(V3 p, V3 a, V3 b, V3 c) {
  const V3 ab = vsub(b, a), ac = vsub(c, a), ap = vsub(p, a);
  const double d1 = vdot(ab, ap), d2 = vdot(ac, ap);
  if (d1 <= 0.0 && d2 <= 0.0) return a;
  const V3 bp = vsub(p, b);
  const double d3 = vdot(ab, bp), d4 = vdot(ac, bp);
  if (d3 >= 0.0 && d4 <= d3) return b;
  const double vc = d1 * d4 - d3 * d2;
  if (vc <= 0.0 && d1 >= 0.0 && d3 <= 0.0) return vadd(a, vmul(ab, d1 / (d1 - d3)));
  const V3 cp = vsub(p, c);
  const double d5 = vdot(ab, cp), d6 = vdot(ac, cp);
  if (d6 >= 0.0 && d5 <= d6) return c;
  const double vb = d5 * d2 - d1 * d6;
  if (vb <= 0.0 && d2 >= 0.0 && d6 <= 0.0) return vadd(a, vmul(ac, d2 / (d2 - d6)));
  const double va = d3 * d6 - d5 * d4;
  if (va <= 0.0 && (d4 - d3) >= 0.0 && (d5 - d6) >= 0.0)
    return vadd(b, vmul(vsub(c, b), (d4 - d3) / ((d4 - d3) + (d5 - d6))));
  const double denom = 1.0 / (va + vb + vc);
  const double v = vb * denom, w = vc * denom;
  return vadd(vadd(a, vmul(ab, v)), vmul(ac, w));
}

// Solid angle of triangle abc seen from p (Van Oosterom and Strackee), as
// solidAngleFromPointToTriangle (LevelSetObjectGenerator.h:758-782).
__device__ __forceinline__ double solidAngle(V3 p, V3 a, V3 b, V3 c) {
  const V3 r0 = vsub(a, p), r1 = vsub(b, p), r2 = vsub(c, p);
  const double l0 = vlen(r0), l1 = vlen(r1), l2 = vlen(r2);
  if (l0 < 1e-30 || l1 < 1e-30 || l2 < 1e-30) return 0.0;
  const double num = vdot(r0, vcross(r1, r2));
  const double den = l0 * l1 * l2 + vdot(r0, r1) * l2 + vdot(r1, r2) * l0 + vdot(r2, r0) * l1;
  return 2.0 * atan2(num, den);
}

struct MeshPoints {
  // grid mode (points == nullptr): node (i, j, k) at origin + (i, j, k) h
  double ox, oy, oz, h;
  int nx, ny, nz;
  // point mode
  const double* points;  // [3*count]
  long long count;
};

__device__ __forceinline__ V3 pointOf(const MeshPoints& m, long long id) {
  if (m.points) return {m.points[3 * id], m.points[3 * id + 1], m.points[3 * id + 2]};
  const long long nxy = (long long)m.nx * m.ny;
  const int k = (int)(id / nxy);
  const long long r = id - (long long)k * nxy;
  const int j = (int)(r / m.nx);
  const int i = (int)(r - (long long)j * m.nx);
  return {m.ox + double(i) * m.h, m.oy + double(j) * m.h, m.oz + double(k) * m.h};
}

// Eight threads per point (kSlices), each folding every eighth triangle of a
// staged tile; the partials are combined in LDS. sdf (grid mode): the
// level-set value of buildGrid, value / |grad| or +-h/2 where the gradient
// vanishes. value/grad (point mode): the implicit value and gradient of
// evaluateImplicitFunctionValueAndGradient (LevelSetObjectGenerator.h:888-914).
// The closest point is the first triangle (lowest index) at the minimum
// squared distance, as a serial scan finds it. The solid angles are summed per
// slice and the slices then in order, so the sum's rounding differs from a
// serial sum; the inside decision |sum| / 4 pi > 1/2 only sees that for
// points within rounding of the surface, where the value is +-0 either way.
constexpr int kSlices = 8;
// Base::buildGrid: the signed-distance-like value from value and gradient of
// evaluateImplicitFunctionValueAndGradient; dp = node - closest point, d its
// length.
__device__ __forceinline__ void valueAndGradient(V3 dp, double d, bool inside, int positiveInside, double& val, V3& g) {
  val = inside ? -d : d;
  g = {0.0, 0.0, 0.0};
  if (d > 1e-30) {
    const V3 u = vdiv(dp, d);
    g = inside ? vneg(u) : u;
  }
  if (positiveInside) {
    val = -val;
    g = vneg(g);
  }
}
__device__ __forceinline__ double gridValue(V3 dp, double d, bool inside, int positiveInside, double h) {
  double val;
  V3 g;
  valueAndGradient(dp, d, inside, positiveInside, val, g);
  const double gn = vlen(g);
  return gn > 1e-12 ? val / gn : (val <= 0.0 ? -1.0 : 1.0) * 0.5 * h;
}
constexpr int kPointsPerBlock = kMeshTile / kSlices;

__global__ __launch_bounds__(kMeshTile) void kMeshDistance(const double* __restrict__ tri, int nt,
                                                            MeshPoints m, int positiveInside,
                                                            double* sdf, double* value,
                                                            double* grad) {
  __shared__ double sT[9][kMeshTile];
  __shared__ double sBest[kMeshTile], sSum[kMeshTile], sCp[3][kMeshTile];
  __shared__ int sIdx[kMeshTile];
  const int slice = threadIdx.x % kSlices;
  const int local = threadIdx.x / kSlices;
  const long long id = (long long)blockIdx.x * kPointsPerBlock + local;
  const bool active = id < m.count;
  const V3 p = active ? pointOf(m, id) : V3{0.0, 0.0, 0.0};
  double best = DBL_MAX;
  int bestIdx = INT_MAX;
  V3 bestCp = {0.0, 0.0, 0.0};
  double sum = 0.0;
  for (int t0 = 0; t0 < nt; t0 += kMeshTile) {
    __syncthreads();
    const int t = t0 + (int)threadIdx.x;
    if (t < nt) {
#pragma unroll
      for (int c = 0; c < 9; ++c) sT[c][threadIdx.x] = tri[9 * (size_t)t + c];
    }
    __syncthreads();
    if (!active) continue;
    const int cnt = min(kMeshTile, nt - t0);
    for (int u = slice; u < cnt; u += kSlices) {
      const V3 a = {sT[0][u], sT[1][u], sT[2][u]};
      const V3 b = {sT[3][u], sT[4][u], sT[5][u]};
      const V3 c = {sT[6][u], sT[7][u], sT[8][u]};
      // box lower bound on the distance, with a margin so that rounding
      // never skips the triangle that holds the minimum
      const double dx = fmax(fmax(fmin(fmin(a.x, b.x), c.x) - p.x, 0.0), p.x - fmax(fmax(a.x, b.x), c.x));
      const double dy = fmax(fmax(fmin(fmin(a.y, b.y), c.y) - p.y, 0.0), p.y - fmax(fmax(a.y, b.y), c.y));
      const double dz = fmax(fmax(fmin(fmin(a.z, b.z), c.z) - p.z, 0.0), p.z - fmax(fmax(a.z, b.z), c.z));
      const double box = dx * dx + dy * dy + dz * dz;
      if (box <= best * (1.0 + 1e-9)) {
        const V3 cp = closestOnTriangle(p, a, b, c);
        const double d2 = vlen2(vsub(p, cp));
        if (d2 < best) {  // triangles of a slice come in increasing index
          best = d2;
          bestIdx = t0 + u;
          bestCp = cp;
        }
      }
      sum += solidAngle(p, a, b, c);
    }
  }
  sBest[threadIdx.x] = best;
  sIdx[threadIdx.x] = bestIdx;
  sSum[threadIdx.x] = sum;
  sCp[0][threadIdx.x] = bestCp.x;
  sCp[1][threadIdx.x] = bestCp.y;
  sCp[2][threadIdx.x] = bestCp.z;
  __syncthreads();
  if (!active || slice != 0) return;
  for (int k = 1; k < kSlices; ++k) {
    const int o = threadIdx.x + k;
    const double b2 = sBest[o];
    if (b2 < best || (b2 == best && sIdx[o] < bestIdx)) {
      best = b2;
      bestIdx = sIdx[o];
      bestCp = {sCp[0][o], sCp[1][o], sCp[2][o]};
    }
    sum += sSum[o];
  }
  // evaluateImplicitFunctionValueAndGradient
  const V3 dp = vsub(p, bestCp);
  const double d = vlen(dp);
  const bool inside = fabs(sum / (4.0 * kPi)) > 0.5;
  if (sdf) {
    sdf[id] = gridValue(dp, d, inside, positiveInside, m.h);
  } else {
    double val;
    V3 g;
    valueAndGradient(dp, d, inside, positiveInside, val, g);
    value[id] = val;
    grad[3 * id] = g.x;
    grad[3 * id + 1] = g.y;
    grad[3 * id + 2] = g.z;
  }
}

// ---------------------------------------------------------------- grid path
// The same values on a grid without a solid angle per node and triangle (a
// square root each and an arctangent in FP64, some 300 instructions, made the
// kernel above take 7.5 ps per node and triangle) and without a box test per
// node and triangle:
//  - Sign: the triangles' solid angles add up to 4 pi times a whole number,
//    the winding number, if they bound a closed surface. kMeshPrep checks
//    that every directed edge has its reverse (sum of edge hashes, one 64-bit
//    word: an open mesh passes with probability 2^-64). The number is then the
//    signed count of triangles crossed by any ray from the node: the columns
//    of nodes share one ray along z each (kMeshColumns, kMeshWinding), moved
//    sideways by a 1e-4 of the spacing, as meshes like to have vertices and
//    edges on grid lines.
//  - Nodes that this does not decide for certain take the solid angles, eight
//    partial sums as above (kMeshSolid): nodes nearer to the surface than the
//    ray's shift and rounding, columns whose ray passes an edge within
//    rounding, and all nodes of an open mesh.
//  - Distance: bricks of 4 x 4 x 4 nodes, one node per lane, whose waves
//    share the triangles in chunks of 32; a chunk or triangle whose box is
//    farther than the best distance found is passed by, the chunk nearest to
//    the brick first (kMeshNearest). The chunks take the triangles in their
//    order: a mesh in no spatial order is slower, not wrong.
// Bound by FP64 VALU, and on small grids by the brick with the most triangles
// in reach. An open mesh pays for every solid angle, and on grids of few bricks
// finds the nearest triangle in the same loop (kMeshSoloBricks). Measured, a whole call of the host class: 57K nodes and 5120
// triangles 2.60 -> 0.43 ms (kernels 2.52 -> 0.33), 342K and 5120 13.1 -> 1.05
// ms, 2.4M and 5120 87 -> 3.5 ms (4.5 with the triangles shuffled), 578K and
// 20480 82 -> 3.6 ms.
constexpr int kMeshChunk = 32;
constexpr int kSolidStep = 4;  // kMeshSolid: triangles per thread between barriers
// Nodes from which eight share a workgroup in kMeshSolid (5832 nodes and 5120
// triangles 489 us with a workgroup each, 497 with eight; 8000 nodes 605 and
// 583; 1000 nodes 345 and 405).
constexpr int kSolidMany = 7168;
// Sizes between which the signs are taken from crossings: a solid angle's
// products of three lengths neither overflow nor vanish. A mesh beyond them, or
// with a coordinate that is no number, has an infinite "largest coordinate",
// under which no node counts as decided.
constexpr double kMeshLeast = 1e-20, kMeshMost = 1e90;
struct alignas(64) MeshChunk {
  double lo[3], hi[3];       // box of the triangles
  double m;                  // largest |coordinate|
  unsigned long long edges;  // sum of the directed edges' hashes minus their reverses'
};
struct MeshWork {
  const double* tri;
  int nt, nChunks;
  MeshPoints m;
  int positiveInside;
  MeshChunk* chunks;
  int* inside;          // [nodes] crossings by node, then 0 outside, 1 inside, 2 not decided
  int* column;          // [nx * ny] 1: the column's ray passes an edge
  int* list;            // nodes not decided
  int* listCount;
  double* largest;      // largest |coordinate| of triangles and grid
  int* open;            // the mesh is not closed
  double* sdf;
};
__device__ __forceinline__ unsigned long long mix64(unsigned long long x) {
  // the finaliser of SplitMix64 (Steele, Lea and Flood, OOPSLA 2014)
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
__device__ __forceinline__ unsigned long long hashVertex(V3 v) {
  // (+ 0.0: one zero)
  unsigned long long h = mix64((unsigned long long)__double_as_longlong(v.x + 0.0) + 0x9E3779B97F4A7C15ull);
  h = mix64(h + (unsigned long long)__double_as_longlong(v.y + 0.0));
  return mix64(h + 3ull * (unsigned long long)__double_as_longlong(v.z + 0.0));
}
__device__ __forceinline__ unsigned long long hashEdge(unsigned long long a, unsigned long long b) {
  return mix64(a + 5ull * b) - mix64(b + 5ull * a);
}
__device__ __forceinline__ double meshScale(const MeshPoints& m) {
  const double x = fmax(fabs(m.ox), fabs(m.ox + m.nx * m.h)), y = fmax(fabs(m.oy), fabs(m.oy + m.ny * m.h)),
               z = fmax(fabs(m.oz), fabs(m.oz + m.nz * m.h));
  return fmax(fmax(x, y), z);
}

// Boxes and edge sums of the chunks (one triangle per lane), empty counts.
__global__ void __launch_bounds__(256) kMeshPrep(MeshWork k) {
  const long long i0 = (long long)blockIdx.x * 256 + threadIdx.x, stride = (long long)gridDim.x * 256;
  for (long long i = i0; i < k.m.count; i += stride) k.inside[i] = 0;
  for (long long i = i0; i < (long long)k.m.nx * k.m.ny; i += stride) k.column[i] = 0;
  if (i0 == 0) *k.listCount = 0;
  const int lane = threadIdx.x % kMeshChunk;
  for (long long c = i0 / kMeshChunk; c < k.nChunks; c += stride / kMeshChunk) {
    const int t = (int)min(c * kMeshChunk + lane, (long long)k.nt - 1);
    const bool own = c * kMeshChunk + lane < k.nt;
    double v[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) v[q] = k.tri[9 * (size_t)t + q];
    double box[7];
    box[6] = 0.;
#pragma unroll
    for (int q = 0; q < 9; ++q)
      if (!(fabs(v[q]) <= kMeshMost)) box[6] = __builtin_inf();
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      box[a] = fmin(fmin(v[a], v[3 + a]), v[6 + a]);
      box[3 + a] = fmax(fmax(v[a], v[3 + a]), v[6 + a]);
      box[6] = fmax(box[6], fmax(fabs(box[a]), fabs(box[3 + a])));
    }
    const unsigned long long ha = hashVertex({v[0], v[1], v[2]}), hb = hashVertex({v[3], v[4], v[5]}),
                             hc = hashVertex({v[6], v[7], v[8]});
    unsigned long long e = own ? hashEdge(ha, hb) + hashEdge(hb, hc) + hashEdge(hc, ha) : 0ull;
#pragma unroll
    for (int off = kMeshChunk / 2; off > 0; off >>= 1) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        box[a] = fmin(box[a], __shfl_xor(box[a], off, 64));
        box[3 + a] = fmax(box[3 + a], __shfl_xor(box[3 + a], off, 64));
      }
      box[6] = fmax(box[6], __shfl_xor(box[6], off, 64));
      e += __shfl_xor(e, off, 64);
    }
    if (lane == 0) {
      MeshChunk& r = k.chunks[c];
      for (int a = 0; a < 3; ++a) {
        r.lo[a] = box[a];
        r.hi[a] = box[3 + a];
      }
      r.m = box[6];
      r.edges = e;
    }
  }
}

// Sum of the chunks' edge sums by a wave: zero for a closed mesh.
__device__ __forceinline__ unsigned long long edgeSum(const MeshWork& k, int lane) {
  unsigned long long e = 0ull;
  for (int c = lane; c < k.nChunks; c += 64) e += k.chunks[c].edges;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off, 64);
  return e;
}

// Triangles crossed by the columns' rays: a wave takes 8 x 8 columns, one per
// lane, and a share of the chunks. A crossing is left at the column's highest
// node below it. A triangle counts if the ray passes its three edges on one
// side for certain, is passed by if it is for certain on different sides of
// two, and otherwise leaves the column undecided. An edge function is the
// product of an edge of length l and the ray's distance to it; its rounding
// error is below 1e-15 l times the coordinates' size, a ten-thousandth of the
// tolerance.
__global__ void __launch_bounds__(256) kMeshColumns(MeshWork k, int tilesX, int tiles, int perWave) {
  const int lane = laneId();
  const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int tile = wave % tiles, c0 = wave / tiles * perWave, c1 = min(c0 + perWave, k.nChunks);
  if (c0 >= c1 || edgeSum(k, lane) != 0ull) return;  // (an open mesh takes no crossing)
  const MeshPoints& m = k.m;
  const int i0 = tile % tilesX * 8, j0 = tile / tilesX * 8;
  const int i = i0 + lane % 8, j = j0 + lane / 8;
  const bool on = i < m.nx && j < m.ny;
  const double sx = 0.618e-4 * m.h, sy = 0.414e-4 * m.h;
  const double px = m.ox + i * m.h + sx, py = m.oy + j * m.h + sy;
  const double x0 = m.ox + i0 * m.h, x1 = m.ox + (i0 + 8) * m.h, y0 = m.oy + j0 * m.h, y1 = m.oy + (j0 + 8) * m.h;
  const double pm = meshScale(m);
  const long long col = (long long)j * m.nx + i, nxy = (long long)m.nx * m.ny;
  for (int cb = c0; cb < c1; cb += 64) {
    bool near = false;
    if (cb + lane < c1) {
      const MeshChunk& r = k.chunks[cb + lane];
      const double s = 1e-9 * (r.m + pm);
      near = !(r.lo[0] > x1 + s || r.hi[0] < x0 - s || r.lo[1] > y1 + s || r.hi[1] < y0 - s);
    }
    for (unsigned long long mask = ballot64(near); mask; mask &= mask - 1ull) {
      const int c = cb + __builtin_ctzll(mask);
      // the chunk's triangles over the tile, one per lane
      const int mine = c * kMeshChunk + lane;
      bool over = false;
      if (lane < kMeshChunk && mine < k.nt) {
        const double* v = k.tri + 9 * (size_t)mine;
        const double s = 1e-9 * (k.chunks[c].m + pm);
        over = !(fmin(fmin(v[0], v[3]), v[6]) > x1 + s || fmax(fmax(v[0], v[3]), v[6]) < x0 - s ||
                 fmin(fmin(v[1], v[4]), v[7]) > y1 + s || fmax(fmax(v[1], v[4]), v[7]) < y0 - s);
      }
      for (unsigned long long tm = ballot64(over); tm; tm &= tm - 1ull) {
        const double* v = k.tri + 9 * (size_t)(c * kMeshChunk + __builtin_ctzll(tm));
        const double ax = v[0], ay = v[1], az = v[2], bx = v[3], by = v[4], bz = v[5], cx = v[6], cy = v[7], cz = v[8];
        const double big = fmax(fmax(fmax(fabs(ax), fabs(ay)), fmax(fabs(bx), fabs(by))),
                                fmax(fmax(fabs(cx), fabs(cy)), fmax(fmax(fabs(az), fabs(bz)), fabs(cz)))) + pm;
        const double ux = bx - ax, uy = by - ay, vx = cx - bx, vy = cy - by, wx = ax - cx, wy = ay - cy;
        const double f = 1e-11 * big;
        const double t0 = f * (fabs(ux) + fabs(uy)), t1e = f * (fabs(vx) + fabs(vy)), t2 = f * (fabs(wx) + fabs(wy));
        const double e0 = (px - bx) * -uy + (py - by) * ux, e1 = (px - cx) * -vy + (py - cy) * vx,
                     e2 = (px - ax) * -wy + (py - ay) * wx;
        const bool pos = e0 > t0 || e1 > t1e || e2 > t2, neg = e0 < -t0 || e1 < -t1e || e2 < -t2;
        if (!on || (pos && neg)) continue;
        const double area = e0 + e1 + e2;
        const bool sure = ((e0 > t0 && e1 > t1e && e2 > t2) || (e0 < -t0 && e1 < -t1e && e2 < -t2)) &&
                          fabs(area) > 1e3 * (t0 + t1e + t2);
        if (!sure) {
          k.column[col] = 1;
          continue;
        }
        const double z = az + (e2 * (bz - az) + e0 * (cz - az)) / area;
        const int below = (int)fmin(fmax(ceil((z - m.oz) / m.h), 0.), (double)m.nz);
        if (below > 0) atomicAdd(&k.inside[(below - 1) * nxy + col], area > 0. ? 1 : -1);
      }
    }
  }
}

// Crossings above each node, one column per lane; nothing is decided for an
// open mesh.
__global__ void __launch_bounds__(256) kMeshWinding(MeshWork k) {
  __shared__ unsigned long long edges[4];
  __shared__ double largest[4];
  unsigned long long e = 0ull;
  double big = meshScale(k.m);
  for (int c = threadIdx.x; c < k.nChunks; c += 256) {
    e += k.chunks[c].edges;
    big = fmax(big, k.chunks[c].m);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    e += __shfl_xor(e, off, 64);
    big = fmax(big, __shfl_xor(big, off, 64));
  }
  if (laneId() == 0) {
    edges[threadIdx.x >> 6] = e;
    largest[threadIdx.x >> 6] = big;
  }
  __syncthreads();
  e = edges[0] + edges[1] + edges[2] + edges[3];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    big = fmax(fmax(largest[0], largest[1]), fmax(largest[2], largest[3]));
    *k.largest = big >= kMeshLeast && big <= kMeshMost ? big : __builtin_inf();
    *k.open = e != 0ull ? 1 : 0;
  }
  const long long nxy = (long long)k.m.nx * k.m.ny, col = (long long)blockIdx.x * 256 + threadIdx.x;
  if (col >= nxy) return;
  const bool open = e != 0ull || k.column[col] != 0;
  int run = 0;
  constexpr int kAhead = 8;
  for (int z1 = k.m.nz; z1 > 0; z1 -= kAhead) {
    int v[kAhead];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) v[q] = z1 - 1 - q >= 0 ? k.inside[(z1 - 1 - q) * nxy + col] : 0;
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      run += v[q];
      if (z1 - 1 - q >= 0) k.inside[(z1 - 1 - q) * nxy + col] = open ? 2 : run != 0 ? 1 : 0;
    }
  }
}

__device__ __forceinline__ double boxDistance2(V3 p, const double* lo, const double* hi) {
  const double dx = fmax(fmax(lo[0] - p.x, 0.0), p.x - hi[0]);
  const double dy = fmax(fmax(lo[1] - p.y, 0.0), p.y - hi[1]);
  const double dz = fmax(fmax(lo[2] - p.z, 0.0), p.z - hi[2]);
  return dx * dx + dy * dy + dz * dz;
}

template <int WAVES>
__global__ void __launch_bounds__(64 * WAVES) kMeshNearest(MeshWork k, int bricksX, int bricksY, int solo) {
  __shared__ unsigned long long bound[64];  // best squared distance of the node so far
  __shared__ double sBest[WAVES][64], sCp[3][WAVES][64];
  __shared__ int sIdx[WAVES][64];
  __shared__ double startD[WAVES];
  __shared__ int startC[WAVES];
  const MeshPoints& m = k.m;
  const int lane = laneId(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.x;
  const int i0 = b % bricksX * 4, j0 = b / bricksX % bricksY * 4, k0 = b / bricksX / bricksY * 4;
  const int i = i0 + lane % 4, j = j0 + lane / 4 % 4, kk = k0 + lane / 16;
  const bool on = i < m.nx && j < m.ny && kk < m.nz;
  const V3 p = {m.ox + double(i) * m.h, m.oy + double(j) * m.h, m.oz + double(kk) * m.h};
  if (solo && *k.open) return;
  const double largest = *k.largest;
  // the brick's ball (nodes past the grid's end included)
  const V3 mid = {m.ox + (i0 + 1.5) * m.h, m.oy + (j0 + 1.5) * m.h, m.oz + (k0 + 1.5) * m.h};
  const double ball = 1.5 * 1.7320509 * m.h + 1e-9 * m.h + 1e-12 * largest;
  double best = DBL_MAX;
  int bestIdx = INT_MAX;
  V3 bestCp = {0.0, 0.0, 0.0};
  double limit = DBL_MAX;  // the least squared distance known, of any wave
  // the brick's distance within which a box may hold the nearest point of a node
  auto reach2 = [&]() __attribute__((always_inline)) {
    double far = limit;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) far = fmax(far, __shfl_xor(far, off, 64));
    const double r = (sqrt(far) + ball) * (1.0 + 1e-6);
    return r * r;
  };
  auto triangles = [&](int t0, int t1) __attribute__((always_inline)) {
    // those near the brick (one per lane), then these one by one
    const double r2 = reach2();
    bool near = false;
    if (t0 + lane < t1) {
      const double* v = k.tri + 9 * (size_t)(t0 + lane);
      const double lo[3] = {fmin(fmin(v[0], v[3]), v[6]), fmin(fmin(v[1], v[4]), v[7]), fmin(fmin(v[2], v[5]), v[8])};
      const double hi[3] = {fmax(fmax(v[0], v[3]), v[6]), fmax(fmax(v[1], v[4]), v[7]), fmax(fmax(v[2], v[5]), v[8])};
      near = !(boxDistance2(mid, lo, hi) > r2);
    }
    for (unsigned long long tm = ballot64(near); tm; tm &= tm - 1ull) {
      const int t = t0 + __builtin_ctzll(tm);
      const double* v = k.tri + 9 * (size_t)t;
      const V3 A = {v[0], v[1], v[2]}, B = {v[3], v[4], v[5]}, C = {v[6], v[7], v[8]};
      const double lo[3] = {fmin(fmin(A.x, B.x), C.x), fmin(fmin(A.y, B.y), C.y), fmin(fmin(A.z, B.z), C.z)};
      const double hi[3] = {fmax(fmax(A.x, B.x), C.x), fmax(fmax(A.y, B.y), C.y), fmax(fmax(A.z, B.z), C.z)};
      // box lower bound on the distance, with a margin so that rounding
      // never skips the triangle that holds the minimum
      if (boxDistance2(p, lo, hi) <= limit * (1.0 + 1e-9)) {
        const V3 cp = closestOnTriangle(p, A, B, C);
        const double d2 = vlen2(vsub(p, cp));
        if (d2 < best || (d2 == best && t < bestIdx)) {
          best = d2;
          bestIdx = t;
          bestCp = cp;
          limit = fmin(limit, d2);
        }
      }
    }
  };
  // the chunk nearest to the brick
  double d0 = DBL_MAX;
  int s0 = 0;
  for (int c = threadIdx.x; c < k.nChunks; c += 64 * WAVES) {
    const double d = boxDistance2(mid, k.chunks[c].lo, k.chunks[c].hi);
    if (d < d0) {
      d0 = d;
      s0 = c;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double d = __shfl_xor(d0, off, 64);
    const int c = __shfl_xor(s0, off, 64);
    if (d < d0 || (d == d0 && c < s0)) {
      d0 = d;
      s0 = c;
    }
  }
  if (lane == 0) {
    startD[wave] = d0;
    startC[wave] = s0;
  }
  if (threadIdx.x < 64) bound[threadIdx.x] = (unsigned long long)__double_as_longlong(DBL_MAX);
  __syncthreads();
  int start = startC[0];
  d0 = startD[0];
  for (int w = 1; w < WAVES; ++w)
    if (startD[w] < d0 || (startD[w] == d0 && startC[w] < start)) {
      d0 = startD[w];
      start = startC[w];
    }
  start = __builtin_amdgcn_readfirstlane(start);
  {
    const int t = start * kMeshChunk + wave * (kMeshChunk / WAVES);
    triangles(min(t, k.nt), min(t + kMeshChunk / WAVES, k.nt));
  }
  // (non-negative numbers order as their bits do)
  atomicMin(&bound[lane], (unsigned long long)__double_as_longlong(limit));
  __syncthreads();
  for (int cb = wave; cb < k.nChunks; cb += 64 * WAVES) {  // every WAVES-th chunk is this wave's
    limit = fmin(limit, __longlong_as_double((long long)*(volatile unsigned long long*)&bound[lane]));
    const double r2 = reach2();
    const int mine = cb + WAVES * lane;
    const bool near = mine < k.nChunks && mine != start &&
                      !(boxDistance2(mid, k.chunks[mine].lo, k.chunks[mine].hi) > r2);
    for (unsigned long long mask = ballot64(near); mask; mask &= mask - 1ull) {
      const int c = cb + WAVES * __builtin_ctzll(mask);
      limit = fmin(limit, __longlong_as_double((long long)*(volatile unsigned long long*)&bound[lane]));
      if (!ballot64(boxDistance2(p, k.chunks[c].lo, k.chunks[c].hi) <= limit * (1.0 + 1e-9))) continue;
      triangles(c * kMeshChunk, min((c + 1) * kMeshChunk, k.nt));
      atomicMin(&bound[lane], (unsigned long long)__double_as_longlong(limit));
    }
  }
  sBest[wave][lane] = best;
  sIdx[wave][lane] = bestIdx;
  sCp[0][wave][lane] = bestCp.x;
  sCp[1][wave][lane] = bestCp.y;
  sCp[2][wave][lane] = bestCp.z;
  __syncthreads();
  if (wave != 0 || !on) return;
  for (int w = 1; w < WAVES; ++w) {
    const double b2 = sBest[w][lane];
    if (b2 < best || (b2 == best && sIdx[w][lane] < bestIdx)) {
      best = b2;
      bestIdx = sIdx[w][lane];
      bestCp = {sCp[0][w][lane], sCp[1][w][lane], sCp[2][w][lane]};
    }
  }
  const long long id = ((long long)kk * m.ny + j) * m.nx + i;
  const double d = vlen(vsub(p, bestCp));
  const int side = k.inside[id];
  // the path to the shifted ray may cross the surface, or the ray's crossing
  // be misplaced by rounding; at distance zero both sides have one value
  const bool sure = side != 2 && d > 4e-4 * m.h + 2e-6 * largest;
  k.sdf[id] = gridValue(vsub(p, bestCp), d, sure && side == 1, k.positiveInside, m.h);
  if (!sure && d != 0.0) k.list[atomicAdd(k.listCount, 1)] = (int)id;
}

// The solid angles of NODES nodes by a workgroup: a thread takes every
// 256 / NODES-th triangle for one node, and 8 * NODES lanes add the angles,
// staged in LDS, to eight partial sums per node in the order of kMeshDistance.
// Nodes first, first + 1, ... of the list, whose sign is left; DISTANCE: of
// the grid, with the nearest triangle found in the same loop.
struct SolidSlots {
  double angle[2][kSolidStep * kMeshTile];
  unsigned long long bound[8];  // best squared distance of a node so far
};
template <int NODES, bool DISTANCE>
__device__ __forceinline__ void solidNodes(const MeshWork& k, int first, int count, SolidSlots& ws) {
  constexpr int kEach = NODES == 1 ? 1 : kSolidStep;  // triangles per thread between barriers
  constexpr int kTile = kMeshTile / NODES * kEach;
  const int node = threadIdx.x % NODES;
  const int at = min(first + node, count - 1), id = DISTANCE ? at : k.list[at];
  const V3 p = pointOf(k.m, id);
  double sum = 0.0, best = DBL_MAX;
  int buf = 0, bestIdx = INT_MAX;
  if (DISTANCE) {
    if ((int)threadIdx.x < NODES) ws.bound[threadIdx.x] = (unsigned long long)__double_as_longlong(DBL_MAX);
    __syncthreads();
  }
  for (int t0 = 0; t0 < k.nt; t0 += kTile, buf ^= 1) {
    double limit = DBL_MAX;
    if (DISTANCE) limit = __longlong_as_double((long long)*(volatile unsigned long long*)&ws.bound[node]);
#pragma unroll 1
    for (int u = 0; u < kEach; ++u) {
      const int t = t0 + (u * kMeshTile + (int)threadIdx.x) / NODES;
      double angle = 0.0;
      if (t < k.nt) {
        const double* v = k.tri + 9 * (size_t)t;
        const V3 a = {v[0], v[1], v[2]}, b = {v[3], v[4], v[5]}, c = {v[6], v[7], v[8]};
        angle = solidAngle(p, a, b, c);
        if (DISTANCE) {
          const double lo[3] = {fmin(fmin(a.x, b.x), c.x), fmin(fmin(a.y, b.y), c.y), fmin(fmin(a.z, b.z), c.z)};
          const double hi[3] = {fmax(fmax(a.x, b.x), c.x), fmax(fmax(a.y, b.y), c.y), fmax(fmax(a.z, b.z), c.z)};
          if (boxDistance2(p, lo, hi) <= limit * (1.0 + 1e-9)) {
            const double d2 = vlen2(vsub(p, closestOnTriangle(p, a, b, c)));
            if (d2 < best) {  // a thread's triangles come in increasing index
              best = d2;
              bestIdx = t;
              limit = fmin(limit, d2);
            }
          }
        }
      }
      ws.angle[buf][u * kMeshTile + threadIdx.x] = angle;
    }
    // (non-negative numbers order as their bits do)
    if (DISTANCE) atomicMin(&ws.bound[node], (unsigned long long)__double_as_longlong(limit));
    __syncthreads();
    if (threadIdx.x < kSlices * NODES)
#pragma unroll
      for (int q = 0; q < kTile / kSlices; ++q) sum += ws.angle[buf][q * kSlices * NODES + threadIdx.x];
  }
  double all = 0.0;
  if (threadIdx.x < 64) {
    all = __shfl(sum, node);
    for (int s = 1; s < kSlices; ++s) all += __shfl(sum, s * NODES + node);
  }
  const bool inside = fabs(all / (4.0 * kPi)) > 0.5;
  __syncthreads();
  if (DISTANCE) {
    double *d2 = ws.angle[0], *idx = d2 + kMeshTile;
    const int j = threadIdx.x;
    d2[j] = best;
    idx[j] = (double)bestIdx;
    __syncthreads();
    if (j < NODES && first + j < count) {
      for (int q = j + NODES; q < kMeshTile; q += NODES)
        if (d2[q] < best || (d2[q] == best && idx[q] < (double)bestIdx)) {
          best = d2[q];
          bestIdx = (int)idx[q];
        }
      V3 cp = {0.0, 0.0, 0.0};
      if (bestIdx < k.nt) {
        const double* v = k.tri + 9 * (size_t)bestIdx;
        cp = closestOnTriangle(p, {v[0], v[1], v[2]}, {v[3], v[4], v[5]}, {v[6], v[7], v[8]});
      }
      k.sdf[id] = gridValue(vsub(p, cp), vlen(vsub(p, cp)), inside, k.positiveInside, k.m.h);
    }
    __syncthreads();
  } else if ((int)threadIdx.x < NODES && first + (int)threadIdx.x < count && inside) {
    k.sdf[id] = -k.sdf[id];
  }
}

// The nodes left. A workgroup for each where they are few, as the chain of
// tiles is then the time; eight a workgroup from kSolidMany on. (With one load
// and addition after another by the eight lanes that add, and a workgroup per
// node, 57475 nodes and 5119 triangles took 3.40 ms instead of 2.18.) solo: the grid of an open mesh, which
// kMeshNearest left out. Bound by FP64 VALU (some 300 instructions an angle).
__global__ void __launch_bounds__(kMeshTile) __attribute__((amdgpu_waves_per_eu(4))) kMeshSolid(MeshWork k, int solo) {
  __shared__ SolidSlots ws;
  if (solo && *k.open) {
    const int count = (int)k.m.count;
    for (int n = 8 * blockIdx.x; n < count; n += 8 * gridDim.x) solidNodes<8, true>(k, n, count, ws);
    return;
  }
  const int count = *k.listCount;
  if (count < kSolidMany) {
    for (int n = blockIdx.x; n < count; n += gridDim.x) solidNodes<1, false>(k, n, count, ws);
  } else {
    for (int n = 8 * blockIdx.x; n < count; n += 8 * gridDim.x) solidNodes<8, false>(k, n, count, ws);
  }
}

}  // namespace
}  // namespace fdm

using namespace fdm;

namespace {
MeshPoints gridPoints(const double* origin, double spacing, const int* size) {
  MeshPoints m{};
  m.ox = origin[0];
  m.oy = origin[1];
  m.oz = origin[2];
  m.h = spacing;
  m.nx = size[0];
  m.ny = size[1];
  m.nz = size[2];
  m.count = (long long)size[0] * size[1] * size[2];
  return m;
}
}  // namespace

extern "C" int fdm_launchMeshSignedDistanceGrid(const double* triangles, int numTriangles,
                                                const double* origin, double spacing,
                                                const int* size, int positiveInside, double* sdf,
                                                hipStream_t stream) {
  if (!triangles || numTriangles <= 0 || !origin || !size || !sdf || !(spacing > 0.0))
    return FDM_EINVAL;
  if (size[0] <= 0 || size[1] <= 0 || size[2] <= 0) return FDM_EINVAL;
  const MeshPoints m = gridPoints(origin, spacing, size);
  hipLaunchKernelGGL(kMeshDistance, dim3(blocksFor(m.count, kPointsPerBlock)), dim3(kMeshTile), 0,
                     stream, triangles, numTriangles, m, positiveInside, sdf, nullptr, nullptr);
  return launchStatus();
}

namespace {
// Nodes times triangles from which the grid path's five launches pay: 34K x
// 256 (2.1 of these) 288 -> 261 us, 16K x 576 231 -> 224 us; below, the two
// take about the same.
constexpr long long kMeshGridPairs = 1ll << 22;
// Bricks below which sixteen waves share one (980 bricks: 294 -> 238 us).
constexpr unsigned kMeshFewBricks = 4096;
// Bricks below which kMeshSolid finds an open mesh's nearest triangles: some
// 1.2 ps per node and triangle on top of the angles, where the longest brick of
// kMeshNearest takes up to 60 ns per triangle, the same at 48000 nodes (324
// bricks, 20479 triangles 3.0 ms against 3.7; 980 bricks 10.2 against 9.8).
constexpr unsigned kMeshSoloBricks = 768;
bool meshGridPath(int nt, const int* size) {
  const long long count = (long long)size[0] * size[1] * size[2];
  return count < (1ll << 30) && count * nt >= kMeshGridPairs;
}
}  // namespace

extern "C" size_t fdm_meshGridWorkspaceBytes(int numTriangles, const int* size) {
  if (!size || numTriangles <= 0 || size[0] <= 0 || size[1] <= 0 || size[2] <= 0) return 0;
  if (!meshGridPath(numTriangles, size)) return 0;
  const size_t nodes = (size_t)size[0] * size[1] * size[2], cols = (size_t)size[0] * size[1];
  return alignUp(nodes * sizeof(int)) * 2 + alignUp(cols * sizeof(int)) +
         alignUp(((size_t)numTriangles + kMeshChunk - 1) / kMeshChunk * sizeof(MeshChunk)) +
         2 * alignUp(sizeof(int)) + alignUp(sizeof(double));
}

extern "C" int fdm_launchMeshSignedDistanceGridWith(const double* triangles, int numTriangles, const double* origin,
                                                    double spacing, const int* size, int positiveInside, double* sdf,
                                                    void* workspace, size_t workspaceBytes, hipStream_t stream) {
  if (!triangles || numTriangles <= 0 || !origin || !size || !sdf || !(spacing > 0.0)) return FDM_EINVAL;
  if (size[0] <= 0 || size[1] <= 0 || size[2] <= 0) return FDM_EINVAL;
  const size_t need = fdm_meshGridWorkspaceBytes(numTriangles, size);
  if (need == 0)
    return fdm_launchMeshSignedDistanceGrid(triangles, numTriangles, origin, spacing, size, positiveInside, sdf, stream);
  if (!workspace || workspaceBytes < need) return FDM_EINVAL;
  MeshWork k{};
  k.tri = triangles;
  k.nt = numTriangles;
  k.nChunks = (numTriangles + kMeshChunk - 1) / kMeshChunk;
  k.m = gridPoints(origin, spacing, size);
  k.positiveInside = positiveInside;
  k.sdf = sdf;
  const long long nxy = (long long)size[0] * size[1];
  Carve cv(workspace, workspaceBytes);
  k.inside = cv.take<int>((size_t)k.m.count);
  k.list = cv.take<int>((size_t)k.m.count);
  k.column = cv.take<int>((size_t)nxy);
  k.chunks = cv.take<MeshChunk>((size_t)k.nChunks);
  k.listCount = cv.take<int>(1);
  k.largest = cv.take<double>(1);
  k.open = cv.take<int>(1);
  if (!cv.ok) return FDM_EINVAL;
  const long long work = std::max<long long>(k.m.count, (long long)k.nChunks * kMeshChunk);
  hipLaunchKernelGGL(kMeshPrep, dim3((unsigned)std::min<long long>(blocksFor(work, 256), 4096)), dim3(256), 0, stream, k);
  const int tilesX = (size[0] + 7) / 8, tiles = tilesX * ((size[1] + 7) / 8);
  // (waves for every SIMD; at least four chunks each, so that a tile's
  // columns are set up for some work)
  const int shares = std::max(1, std::min(k.nChunks / 4, 4096 / tiles));
  const int perWave = (k.nChunks + shares - 1) / shares;
  const long long waves = (long long)tiles * ((k.nChunks + perWave - 1) / perWave);
  hipLaunchKernelGGL(kMeshColumns, dim3(blocksFor(waves, 4)), dim3(256), 0, stream, k, tilesX, tiles, perWave);
  hipLaunchKernelGGL(kMeshWinding, dim3(blocksFor(nxy, 256)), dim3(256), 0, stream, k);
  const int bx = (size[0] + 3) / 4, by = (size[1] + 3) / 4;
  // a brick's triangles are shared by sixteen waves where the grid has too few
  // bricks to fill the chip with four each: its time is then the longest
  // brick's
  const unsigned bricks = (unsigned)((long long)bx * by * ((size[2] + 3) / 4));
  const int solo = bricks < kMeshSoloBricks ? 1 : 0;
  if (bricks < kMeshFewBricks) hipLaunchKernelGGL(kMeshNearest<16>, dim3(bricks), dim3(1024), 0, stream, k, bx, by, solo);
  else hipLaunchKernelGGL(kMeshNearest<4>, dim3(bricks), dim3(256), 0, stream, k, bx, by, solo);
  hipLaunchKernelGGL(kMeshSolid, dim3(persistentBlocks(4)), dim3(kMeshTile), 0, stream, k, solo);
  return launchStatus();
}

extern "C" int fdm_launchMeshSignedDistancePoints(const double* triangles, int numTriangles,
                                                  const double* points, int numPoints,
                                                  int positiveInside, double* value, double* grad,
                                                  hipStream_t stream) {
  if (!triangles || numTriangles <= 0 || numPoints < 0 || (numPoints > 0 && (!points || !value || !grad)))
    return FDM_EINVAL;
  if (numPoints == 0) return FDM_OK;
  MeshPoints m{};
  m.points = points;
  m.count = numPoints;
  m.h = 0.0;
  hipLaunchKernelGGL(kMeshDistance, dim3(blocksFor(numPoints, kPointsPerBlock)), dim3(kMeshTile), 0,
                     stream, triangles, numTriangles, m, positiveInside, nullptr, value, grad);
  return launchStatus();
}
