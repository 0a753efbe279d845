// Contact detection and contact forces.
//
// The reference (LSParticleContactDetectionKernel.cu:4-607) runs one thread
// per surface node over the 27-cell stencil, twice (count, then write), for
// every interaction set, then one thread per contact for forces. Here:
//
//  broad phase  one thread per particle A lists the targets that any of A's
//               nodes could touch under the reference's rules, sorted by
//               target. Particle targets need |x_A - x_B| <= R_A + R_B + s,
//               ghost and wall targets need |x_A - x_T| <= R_A + (SDF box
//               reach of T) + s. A pair is dropped when the target's
//               interpolated SDF at A's centre exceeds Lip * (R_A + s) (Lip
//               bounds the gradient of the trilinear interpolant), since
//               then no node of A can reach phi <= 0. The skin s lets a list
//               serve later steps while bodies move less than s/2 (the step
//               decides on the device when to rebuild); s = 0 gives lists
//               for the current positions only.
//  narrow phase runs of one to eight candidate pairs per wavefront
//               (sweepRun). Node groups of 16 and then nodes are culled in the
//               target's frame by a code per SDF cell (how far the nearest
//               cell with phi <= 0 is); each remaining node evaluates the
//               reference's predicate exactly in FP64: stencil membership of
//               the target's cell, bounding sphere (particle targets, lower
//               index only), SDF box and -phi >= 0. The contacts' normals and
//               points stay in LDS and history records are reserved; then
//               one lane per contact takes the contact's previous spring
//               (keyed by (A, target, node)), applies the linear
//               spring-dashpot law and writes the updated spring. Forces and
//               torques are summed per pair in node order, serially, so the
//               result does not depend on the schedule. (The single-set entry
//               and law mode 2 sweep one pair per wave by 64-node chunks,
//               with the same predicate.)
//
// All culls are conservative with a relative margin of 1e-5 on reaches (a
// unit quaternion stored in FP32 scales vectors by up to 1 +- 2.4e-7), so
// they never remove a contact that the exact test would accept.
#include <algorithm>

#include "cull_device.hpp"
#include "fdm_device.hpp"
#include "fdm_launch.hpp"

namespace fdm {

struct Target {
  V3 x;       // detection position
  Q4 q;
  bool ident;  // q is exactly (1, 0, 0, 0): the rotations return their input
  fdm_template t;
  const float* sdf;
  int hash;   // hash value in the target grid
};
// Into and out of the target's frame. A rotation by the exact identity
// quaternion returns its input (up to the sign of a zero component), so it
// is skipped; the test is wave-uniform in the sweep.
__device__ __forceinline__ V3 toLocal(V3 v, const Target& tg) { return tg.ident ? v : qrotateT(v, tg.q); }
__device__ __forceinline__ V3 toWorld(V3 v, const Target& tg) { return tg.ident ? v : qrotate(tg.q, v); }


// Every kernel of this file only reads body state, templates, materials,
// candidate lists and the previous step's records: they are read through the
// constant address space (ldu), so that the wave-uniform reads of the sweep
// (one pair per wave) become scalar loads into SGPRs, issued together,
// instead of vector loads that each hold VGPRs and wait in turn.
__device__ __forceinline__ fdm_template tmplOf(const fdm_geometry& g, int geo) {
  return ldu(g.info + geo);
}
__device__ __forceinline__ fdm_material matOf(const fdm_material* m, int k) { return ldu(m + k); }
__device__ __forceinline__ V3 ldpR(const double* p, int n, int i) {
  return {ldu(p + i), ldu(p + n + i), ldu(p + 2 * n + i)};
}
__device__ __forceinline__ V3 ld3R(const fdm_real* p, int n, int i) {
  return {(double)ldu(p + i), (double)ldu(p + n + i), (double)ldu(p + 2 * n + i)};
}
__device__ __forceinline__ Q4 ld4R(const fdm_real* p, int n, int i) {
  return {(double)ldu(p + i), (double)ldu(p + n + i), (double)ldu(p + 2 * n + i),
          (double)ldu(p + 3 * n + i)};
}
__device__ __forceinline__ V3 ldd3R(const double* p) { return {ldu(p), ldu(p + 1), ldu(p + 2)}; }

// True when phi > 0 at `local` for certain on an affine (plane-wall) SDF:
// the plane's value exceeds the fit's bound on the residual and rounding.
// Such a node cannot touch, so its SDF fetch is skipped.
__device__ __forceinline__ bool planeClear(V3 local, const fdm_template& t) {
  if (!t.affine) return false;
  const double v = t.plane[3] + t.plane[0] * local.x + t.plane[1] * local.y + t.plane[2] * local.z;
  return v > t.planeSlack;
}
// The same for every point within `reach` of `local`: the plane changes by at
// most |a|_1 |d| over an offset d (|a . d| <= sum |a_i| |d_i| <= |a|_1 |d|).
// For an affine SDF this replaces the Lipschitz test without an SDF fetch.
__device__ __forceinline__ bool planeClearBall(V3 local, double reach, const fdm_template& t) {
  const double v = t.plane[3] + t.plane[0] * local.x + t.plane[1] * local.y + t.plane[2] * local.z;
  const double a1 = fabs(t.plane[0]) + fabs(t.plane[1]) + fabs(t.plane[2]);
  return v - a1 * reach > t.planeSlack;
}
// Ball test against the zero level: the plane bound for affine SDFs, the
// Lipschitz bound otherwise.
__device__ __forceinline__ bool levelClear(V3 local, double reach, const fdm_template& t, const float* sdf) {
  return t.affine ? planeClearBall(local, reach, t) : lipschitzClear(local, reach, t, sdf);
}

__device__ __forceinline__ bool cellNear(I3 t, I3 lo, I3 hi) {
  return t.x >= lo.x - 1 && t.x <= hi.x + 1 && t.y >= lo.y - 1 && t.y <= hi.y + 1 &&
         t.z >= lo.z - 1 && t.z <= hi.z + 1;
}

// ---------------------------------------------------------------- broad phase
struct BroadK {
  int set;
  fdm_bodies P;
  fdm_geometry pgeo;
  fdm_bodies W;
  fdm_geometry wgeo;
  int ghostCapacity;
  const int* ghostCount;
  const int* ghostReal;
  const double* ghostPos;
  const int* ghostBox;
  fdm_grid grid;
  fdm_hash_table table;
  fdm_pairs pairs;
  unsigned* status;
  double skin;
  double maxReach;
  const int* gate;
  fdm_instances inst;
  fdm_periodic periodic;
};

template <int SET>
__device__ __forceinline__ bool acceptCandidate(const BroadK& a, int A, V3 xA, double RA, int T,
                                                int G, V3 xT) {
  const fdm_template tT = SET == FDM_SET_WALL ? tmplOf(a.wgeo, ldu(a.W.geo + T))
                                              : tmplOf(a.pgeo, ldu(a.P.geo + T));
  const Q4 qT = SET == FDM_SET_WALL ? ld4R(a.W.q, a.W.n, T) : ld4R(a.P.q, a.P.n, T);
  const float* sdf = SET == FDM_SET_WALL ? a.wgeo.sdf : a.pgeo.sdf;
  const double reachT = SET == FDM_SET_PARTICLE ? tT.radius : tT.boxReach;
  const V3 d = vsub(xA, xT);
  const double rs = (RA + reachT) * kReach + a.skin;
  if (vlen2(d) > rs * rs) return false;
  const V3 local = qrotateT(d, qT);
  const double reach = RA * kReach + a.skin;
  // no node can enter the SDF box, or none can reach phi <= 0 inside it
  return !outsideBox(local, reach, tT) && !lipschitzClear(local, reach, tT, sdf);
}

// Visit the candidate targets of particle A; `emit(T, G)` for each.
//
// Every accepted pair satisfies a necessary condition of a node contact with
// the reach widened by the skin: a node lies within R_A of x_A, and a contact
// needs it within R_T of x_T (particle targets, sphere test) or inside T's
// SDF box, hence within the box reach of x_T (walls, ghosts). The cells
// visited cover all targets within that distance, so lists built at one step
// stay complete while bodies move less than skin/2:
//  - particles are stored under their cell id; the visited range is the
//    geometric range of A's reach plus the largest target radius, joined with
//    the reference's own stencil (one cell around A's node cells), which also
//    covers a target whose id aliases another cell in the step it is built;
//  - walls are all visited;
//  - ghosts are stored under their clamped geometric cell, which is monotone
//    in the position, so the geometric range alone suffices.
template <int SET, class Emit>
__device__ __forceinline__ void visitCandidates(const BroadK& a, int A, Emit emit) {
  const int n = a.P.n;
  const double RA = tmplOf(a.pgeo, ldu(a.P.geo + A)).radius;
  // with several instances: A's own grid, and its instance's cells and walls
  const bool many = a.inst.count > 0;
  const int in = many ? a.inst.particleInstance[A] : 0;
  // ghost contacts are detected after the periodic wrap
  const V3 xA = SET == FDM_SET_GHOST
                    ? wrapPosition(ldpR(a.P.x, n, A), many ? a.inst.pgrid[in] : a.grid,
                                   many ? a.inst.periodic[in] : a.periodic)
                    : ldpR(a.P.x, n, A);
  if (SET == FDM_SET_WALL) {
    const fdm_grid& wg = many ? a.inst.wgrid[in] : a.grid;
    const int w0 = many ? a.inst.wallStart[in] : 0;
    const int w1 = many ? a.inst.wallStart[in + 1] : a.W.n;
    for (int w = w0; w < w1; ++w) {
      const int h = a.table.hashValue[w];
      if (h < 0 || (long long)h >= wg.num) continue;
      if (acceptCandidate<SET>(a, A, xA, RA, w, w, ldpR(a.W.x, a.W.n, w))) emit(w, w);
    }
    return;
  }
  const fdm_grid& grid = many ? a.inst.pgrid[in] : a.grid;
  const long long cellOffset = many ? a.inst.pcellOffset[in] : 0;
  I3 b0, b1;
  cellRange(xA, (RA + a.maxReach) * kReach + a.skin, grid, b0, b1);
  if (SET == FDM_SET_PARTICLE) {
    I3 lo, hi;
    cellRange(xA, RA * kReach + a.skin, grid, lo, hi);
    b0 = {min(b0.x, max(lo.x - 1, 0)), min(b0.y, max(lo.y - 1, 0)), min(b0.z, max(lo.z - 1, 0))};
    b1 = {max(b1.x, min(hi.x + 1, grid.size.x - 1)), max(b1.y, min(hi.y + 1, grid.size.y - 1)),
          max(b1.z, min(hi.z + 1, grid.size.z - 1))};
  } else {
    if (*a.ghostCount <= 0) return;
    b0 = {max(b0.x, a.ghostBox[0]), max(b0.y, a.ghostBox[1]), max(b0.z, a.ghostBox[2])};
    b1 = {min(b1.x, a.ghostBox[3]), min(b1.y, a.ghostBox[4]), min(b1.z, a.ghostBox[5])};
  }
  const I3 sz = gsize(grid);
  for (int cz = b0.z; cz <= b1.z; ++cz)
    for (int cy = b0.y; cy <= b1.y; ++cy) {
      // The cells of an x-row have consecutive ids and the table is sorted by
      // cell id, so the row's entries form one range: the bounds of its
      // cells are independent loads, and the range is visited in the same
      // order as cell by cell.
      const long long h0 = cellOffset + lin3({b0.x, cy, cz}, sz);
      int s = INT_MAX, e = 0;
#pragma unroll 4
      for (int k = 0; k <= b1.x - b0.x; ++k) {
        const int cs = a.table.cellStart[h0 + k];
        const int ce = a.table.cellEnd[h0 + k];
        if (cs >= 0) {
          s = min(s, cs);
          e = max(e, ce);
        }
      }
      for (int m = s; m < e; ++m) {
        const int idx = a.table.sortIndex[m];
        if (SET == FDM_SET_PARTICLE) {
          if (idx <= A) continue;
          if (acceptCandidate<SET>(a, A, xA, RA, idx, idx, ldpR(a.P.x, n, idx))) emit(idx, idx);
        } else {
          const int j = a.ghostReal[idx];
          if (acceptCandidate<SET>(a, A, xA, RA, j, idx, ldd3R(a.ghostPos + 3 * idx)))
            emit(j, idx);
        }
      }
    }
}

template <int SET>
__global__ void kBroadCount(BroadK a) {
  if (gateOff(a.gate)) return;
  const int A = blockIdx.x * blockDim.x + threadIdx.x;
  if (A > a.P.n) return;
  if (A == a.P.n) {
    a.pairs.count[A] = 0;
    return;
  }
  int c = 0;
  visitCandidates<SET>(a, A, [&](int, int) { ++c; });
  a.pairs.count[A] = c;
}

template <int SET>
__global__ void kBroadWrite(BroadK a) {
  if (gateOff(a.gate)) return;
  const int A = blockIdx.x * blockDim.x + threadIdx.x;
  if (A >= a.P.n) return;
  const int begin = a.pairs.count[A];
  const int end = a.pairs.count[A + 1];
  if (begin == end) return;
  if (end > a.pairs.capacity) {
    // mark the slots that fit as empty so the narrow phase skips them
    for (int w = begin; w < a.pairs.capacity; ++w) a.pairs.pairA[w] = -1;
    atomicOr(a.status, FDM_STATUS_PAIR_OVERFLOW);
    return;
  }
  int w = begin;
  visitCandidates<SET>(a, A, [&](int T, int G) {
    if (w < end) {
      a.pairs.pairA[w] = A;
      a.pairs.pairT[w] = T;
      a.pairs.pairG[w] = G;
    }
    ++w;
  });
  // insertion sort of the segment by target id (lists are short)
  for (int i = begin + 1; i < end; ++i) {
    const int t = a.pairs.pairT[i], g = a.pairs.pairG[i];
    int j = i - 1;
    while (j >= begin && a.pairs.pairT[j] > t) {
      a.pairs.pairT[j + 1] = a.pairs.pairT[j];
      a.pairs.pairG[j + 1] = a.pairs.pairG[j];
      --j;
    }
    a.pairs.pairT[j + 1] = t;
    a.pairs.pairG[j + 1] = g;
  }
}

// -------------------------------------------------------------- narrow phase
// Fields shared by every interaction set of a step.
struct NarrowCommon {
  fdm_bodies P;
  fdm_geometry pgeo;
  const fdm_material* pmat;
  fdm_bodies W;
  fdm_geometry wgeo;
  const fdm_material* wmat;
  fdm_grid pgrid;
  fdm_periodic periodic;
  fdm_instances inst;
  double dt;
  int updateSprings;
  unsigned* status;
  double* dbgPoint;
  double* dbgNormal;
  double* dbgOverlap;
};

// One interaction set.
struct NarrowSet {
  int kind;           // FDM_SET_*
  int ghostMask;      // ghost sets: 1 X, 2 Y, 3 XY
  int ghostFromReal;  // ghost sets: derive positions from the real particles
  const double* ghostPos;
  const int* ghostHash;
  const double* ghostQ;    // sector images: orientation and velocity of each ghost
  const double* ghostVel;
  fdm_grid grid;
  const int* targetHash;
  fdm_pairs pairs;
  fdm_pairs prev;
  fdm_mirror mirror;
};

struct NarrowK {
  NarrowCommon c;
  NarrowSet s;
};

constexpr int kMaxSets = 5;
constexpr int kXcds = 8;  // accelerator complex dies of the MI355X, each with its own L2
struct NarrowMulti {
  NarrowCommon c;
  const int* gate;
  int nsets;
  NarrowSet s[kMaxSets];
};

// Position used for force arms: the stored position after this step's
// periodic wrap (the reference computes forces after updateGhostSpatialGrid).
__device__ __forceinline__ V3 wrappedArm(V3 x, const fdm_grid& g, const fdm_periodic& per) {
  return wrapPosition(x, g, per);
}

// The grids and periodic flags that apply to a pair whose A is `A`: its
// instance's, or the single system's.
struct PairFrame {
  const fdm_grid* pgrid;   // particle grid (wrap, ghosts, particle cell ids)
  const fdm_grid* tgrid;   // grid of the target's cell ids (the wall grid for walls)
  fdm_periodic periodic;
};
template <int SET>
__device__ __forceinline__ PairFrame pairFrame(const NarrowCommon& C, const NarrowSet& S, int A) {
  PairFrame f;
  if (C.inst.count > 0) {
    const int in = ldu(C.inst.particleInstance + A);
    f.pgrid = &C.inst.pgrid[in];
    f.tgrid = SET == FDM_SET_WALL ? &C.inst.wgrid[in] : f.pgrid;
    f.periodic = C.inst.periodic[in];
  } else {
    f.pgrid = &C.pgrid;
    f.tgrid = &S.grid;
    f.periodic = C.periodic;
  }
  return f;
}

// A's position as the set's detection sees it: stored (before this step's
// periodic wrap) for particle and wall pairs, wrapped for ghost pairs, which
// the reference detects after updateGhostSpatialGrid (LSSolver.h:1168-1171).
template <int SET>
__device__ __forceinline__ V3 detectPosA(const NarrowCommon& C, const PairFrame& f, int A) {
  const V3 x = ldpR(C.P.x, C.P.n, A);
  return SET == FDM_SET_GHOST ? wrappedArm(x, *f.pgrid, f.periodic) : x;
}
// A's orientation as the set's detection sees it: a sector turn of this
// step's wrap rotates it for ghost pairs.
template <int SET>
__device__ __forceinline__ Q4 detectQA(const NarrowCommon& C, const PairFrame& f, int A) {
  const Q4 q = ld4R(C.P.q, C.P.n, A);
  if (SET != FDM_SET_GHOST || !f.periodic.sector) return q;
  return sectorTurnQ(q, sectorWrap(ldpR(C.P.x, C.P.n, A), *f.pgrid, f.periodic).turns, f.periodic);
}
// A particle's velocity as the contact forces see it: after this step's wrap,
// which turns it in a sector (the force kernels run after
// updateGhostSpatialGrid, LSSolver.h:1170-1175).
__device__ __forceinline__ V3 forceVel(const NarrowCommon& C, const PairFrame& f, int i) {
  const V3 v = ld3R(C.P.v, C.P.n, i);
  if (!f.periodic.sector) return v;
  return sectorTurnV(v, sectorWrap(ldpR(C.P.x, C.P.n, i), *f.pgrid, f.periodic).turns, f.periodic);
}

// The reference's node predicate for one (node, target) candidate: the
// node's cell is in the target's stencil, the node is within RB of a
// particle target, inside the target's SDF box, and phi <= 0 there. The
// conjunction is evaluated with the cheapest and most selective tests first:
// the sphere, the SDF box, phi, and last the cell test (three divisions),
// which then runs for the few nodes inside the target; `tcell` is the
// target's decoded cell.
template <int SET>
__device__ __forceinline__ bool nodeHit(V3 p, const Target& tg, I3 tcell, const fdm_grid& g,
                                        double RB, Sample& s) {
  if (tg.hash < 0 || (long long)tg.hash >= g.num) return false;
  const V3 rel = vsub(p, tg.x);
  if (SET == FDM_SET_PARTICLE) {
    if (vlen2(rel) > RB * RB) return false;
  }
  int base;
  const V3 local = toLocal(rel, tg);
  if (!sdfLocate(local, tg.t, s, base)) return false;
  if (SET == FDM_SET_WALL && planeClear(local, tg.t)) return false;
  sdfCorners(tg.sdf + base, tg.t, s);
  const double ov = -trilinear(s.x, s.y, s.z, s.c);
  if (!(ov >= 0.)) return false;
  const I3 c = clampedCell(p, g);
  return abs(tcell.x - c.x) <= 1 && abs(tcell.y - c.y) <= 1 && abs(tcell.z - c.z) <= 1;
}
__device__ __forceinline__ int findPrevPair(const NarrowSet& a, int p, int A, int T, int& off) {
  // lists kept from the previous step hold the pair at the same index
  if (p < min(ldu(a.prev.total), a.prev.capacity) && ldu(a.prev.pairA + p) == A &&
      ldu(a.prev.pairT + p) == T) {
    off = ldu(a.prev.recOff + p);
    return ldu(a.prev.recCnt + p);
  }
  int lo = min(ldu(a.prev.count + A), a.prev.capacity);
  int hi = min(ldu(a.prev.count + A + 1), a.prev.capacity) - 1;
  while (lo <= hi) {
    const int mid = (lo + hi) >> 1;
    const int t = ldu(a.prev.pairT + mid);
    if (t == T) {
      off = ldu(a.prev.recOff + mid);
      return ldu(a.prev.recCnt + mid);
    }
    if (t < T) lo = mid + 1;
    else hi = mid - 1;
  }
  off = 0;
  return 0;
}

__device__ __forceinline__ V3 findPrevSpring(const NarrowSet& a, int off, int cnt, int k) {
  int lo = off, hi = off + cnt - 1;
  while (lo <= hi) {
    const int mid = (lo + hi) >> 1;
    const fdm_record r = a.prev.rec[mid];
    const int kk = r.node;
    if (kk == k) return recordSpring(r);
    if (kk < k) lo = mid + 1;
    else hi = mid - 1;
  }
  return {0., 0., 0.};
}

// The target of pair p as this step sees it: position, orientation, template,
// SDF, cell id, and the position its force arm uses.
template <int SET>
__device__ __forceinline__ void resolveTarget(const NarrowCommon& C, const NarrowSet& S, int p, int T,
                                              const PairFrame& f, Target& tg, V3& armB) {
  const int n = C.P.n;
  if (SET == FDM_SET_WALL) {
    tg.x = ldpR(C.W.x, C.W.n, T);
    tg.q = ld4R(C.W.q, C.W.n, T);
    tg.t = tmplOf(C.wgeo, ldu(C.W.geo + T));
    tg.sdf = C.wgeo.sdf;
    tg.hash = ldu(S.targetHash + T);
    armB = tg.x;
  } else if (SET == FDM_SET_PARTICLE) {
    tg.x = ldpR(C.P.x, n, T);
    tg.q = ld4R(C.P.q, n, T);
    tg.t = tmplOf(C.pgeo, ldu(C.P.geo + T));
    tg.sdf = C.pgeo.sdf;
    tg.hash = ldu(S.targetHash + T);
    armB = wrappedArm(tg.x, *f.pgrid, f.periodic);
  } else {
    if (S.ghostFromReal) {
      // no wrap happened this step: the ghost is the real particle shifted
      // by the periods, as the ghost stage computes it
      const WrapStages w = wrapStages(ldpR(C.P.x, n, T), *f.pgrid, f.periodic);
      tg.x = ghostOf(S.ghostMask == 1 ? w.afterX : w.afterY, *f.pgrid, S.ghostMask);
      tg.hash = ghostCellHash(tg.x, *f.pgrid);
    } else {
      const int G = ldu(S.pairs.pairG + p);
      tg.x = ldd3R(S.ghostPos + 3 * G);
      tg.hash = ldu(S.ghostHash + G);
    }
    if (S.ghostQ) {
      const double* gq = S.ghostQ + 4 * (size_t)S.pairs.pairG[p];
      tg.q = {gq[0], gq[1], gq[2], gq[3]};
    } else {
      tg.q = ld4R(C.P.q, n, T);
    }
    tg.t = tmplOf(C.pgeo, ldu(C.P.geo + T));
    tg.sdf = C.pgeo.sdf;
    armB = tg.x;
  }
  tg.ident = tg.q.q0 == 1.0 && tg.q.q1 == 0.0 && tg.q.q2 == 0.0 && tg.q.q3 == 0.0;
}

// Contacts staged per wave in LDS between the node sweep and the contact law.
constexpr int kMaxHits = 64;
struct HitSlots {
  double pc[3][kMaxHits];
  double nrm[3][kMaxHits];
  double ov[kMaxHits];
  int node[kMaxHits];
};

// One wave per candidate pair: chunk culls (one chunk per lane), the node
// sweep over surviving chunks (one node per lane) evaluating the reference's
// predicate, the contact geometry of every hit staged in LDS, then the
// contact law with one hit per lane and the pair sums folded in node order.
// A pair with more than kMaxHits contacts recomputes its hits chunk by chunk
// instead of staging them.
// CULL: first take a particle-level test of the pair (sphere,
// SDF box, Lipschitz bound at this step's positions) and leave empty record
// ranges when it rejects the pair.
template <int SET, bool CULL = false>
__device__ void processPair(const NarrowCommon& C, const NarrowSet& S, int p, int lane,
                           HitSlots& hs, int pool) {
  const int A = ldu(S.pairs.pairA + p);
  if (A < 0) {  // slot left empty by a capacity overflow
    if (lane == 0) {
      S.pairs.recOff[p] = 0;
      S.pairs.recCnt[p] = 0;
    }
    return;
  }
  const int T = ldu(S.pairs.pairT + p);
  const int n = C.P.n;
  const fdm_template& tA = tmplOf(C.pgeo, ldu(C.P.geo + A));
  const PairFrame fr = pairFrame<SET>(C, S, A);
  const Q4 qA = detectQA<SET>(C, fr, A);
  const V3 xA = detectPosA<SET>(C, fr, A);
  const fdm_grid& tgrid = *fr.tgrid;
  Target tg;
  V3 armB;
  resolveTarget<SET>(C, S, p, T, fr, tg, armB);
  if (CULL) {
    const double RA = tA.radius * kReach;
    const double reachT = SET == FDM_SET_PARTICLE ? tg.t.radius : tg.t.boxReach;
    const V3 d = vsub(xA, tg.x);
    const double rs = RA + reachT * kReach;
    bool keep = vlen2(d) <= rs * rs;
    if (keep) {
      const V3 local = toLocal(d, tg);
      keep = !outsideBox(local, RA, tg.t) && !levelClear(local, RA, tg.t, tg.sdf);
    }
    if (!keep) {
      if (lane == 0) {
        S.pairs.recOff[p] = 0;
        S.pairs.recCnt[p] = 0;
      }
      return;
    }
  }
  const V3 armA = SET == FDM_SET_GHOST ? xA : wrappedArm(xA, *fr.pgrid, fr.periodic);
  const double RB = tg.t.radius;
  const I3 tcell = decodeHash(tg.hash, tgrid);
  const fdm_real* nodes = C.pgeo.nodes + 3 * (size_t)tA.nodeStart;
  const float4* chunks = reinterpret_cast<const float4*>(C.pgeo.chunks) + tA.chunkStart;
  const int nChunks = tA.chunkCount;
  const unsigned long long lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));

  // chunk culls, one chunk per lane: a chunk survives unless its bounding
  // sphere fails the sphere, stencil, SDF-box or Lipschitz bound
  bool live = false;
  if (lane < nChunks) {
    const float4 ch = chunks[lane];
    const V3 cw = vadd(qrotate(qA, {(double)ch.x, (double)ch.y, (double)ch.z}), xA);
    const double rc = (double)ch.w * kReach;
    live = true;
    if (SET == FDM_SET_PARTICLE) {
      const double rr = (RB + rc) * (1.0 + 1e-9);
      if (vlen2(vsub(cw, tg.x)) > rr * rr) live = false;
    }
    if (live) {
      I3 lo, hi;
      cellRange(cw, rc, tgrid, lo, hi);
      if (!cellNear(tcell, lo, hi)) live = false;
    }
    if (live) {
      const V3 lc = toLocal(vsub(cw, tg.x), tg);
      if (outsideBox(lc, rc, tg.t) || levelClear(lc, rc, tg.t, tg.sdf)) live = false;
    }
  }
  const unsigned long long liveChunks = ballot64(live);

  // node sweep: lane c keeps chunk c's hit mask; hits in node order get LDS
  // slots holding their contact point, normal, overlap and node id
  unsigned long long myMask = 0ull;
  int total = 0;
  // the history range of the pair does not depend on the sweep: start it now
  int prevOff = 0;
  const int prevCnt = liveChunks ? findPrevPair(S, p, A, T, prevOff) : 0;
  // node coordinates of the next surviving chunk are loaded one iteration
  // ahead, so their latency overlaps the current chunk's SDF fetches
  fdm_real nx = 0, ny = 0, nz = 0;
  if (liveChunks) {
    const int k0 = __builtin_ctzll(liveChunks) * FDM_CHUNK + lane;
    if (k0 < tA.nodeCount) {
      nx = nodes[3 * k0];
      ny = nodes[3 * k0 + 1];
      nz = nodes[3 * k0 + 2];
    }
  }
  for (unsigned long long lcm = liveChunks; lcm; lcm &= lcm - 1ull) {
    const int c = __builtin_ctzll(lcm);
    const int k = c * FDM_CHUNK + lane;
    const V3 s = {(double)nx, (double)ny, (double)nz};
    const unsigned long long rest = lcm & (lcm - 1ull);
    if (rest) {
      const int k2 = __builtin_ctzll(rest) * FDM_CHUNK + lane;
      if (k2 < tA.nodeCount) {
        nx = nodes[3 * k2];
        ny = nodes[3 * k2 + 1];
        nz = nodes[3 * k2 + 2];
      }
    }
    bool hit = false;
    Sample sm;
    V3 pn;
    if (k < tA.nodeCount) {
      pn = vadd(qrotate(qA, s), xA);
      hit = nodeHit<SET>(pn, tg, tcell, tgrid, RB, sm);
    }
    const unsigned long long m = ballot64(hit);
    if (lane == c) myMask = m;
    if (hit) {
      const int slot = total + __popcll(m & lt);
      if (slot < kMaxHits) {
        const double ov = -trilinear(sm.x, sm.y, sm.z, sm.c);
        const V3 nrm = vnormalize(toWorld(gradientIntX(sm.x, sm.y, sm.z, sm.c), tg));
        const V3 pc = vadd(pn, vmul(nrm, 0.5 * ov));
        hs.pc[0][slot] = pc.x;
        hs.pc[1][slot] = pc.y;
        hs.pc[2][slot] = pc.z;
        hs.nrm[0][slot] = nrm.x;
        hs.nrm[1][slot] = nrm.y;
        hs.nrm[2][slot] = nrm.z;
        hs.ov[slot] = ov;
        hs.node[slot] = k;
      }
    }
    total += __popcll(m);
  }

  int base = 0;
  if (total > 0) {
    const int poolCap = S.pairs.recCapacity / FDM_REC_POOLS;
    if (lane == 0) base = atomicAdd(S.pairs.recTotal + pool * FDM_REC_STRIDE, total);
    base = readlaneI(base, 0);
    if (base + total > poolCap) {
      if (lane == 0) atomicOr(C.status, FDM_STATUS_RECORD_OVERFLOW);
      total = 0;
      base = 0;
    }
    base += pool * poolCap;
  }

  V3 SF = {0., 0., 0.}, STA = {0., 0., 0.}, STB = {0., 0., 0.};
  if (total > 0) {
    // material constants of the pair (contactKernel.cu:79-110,167-193,243-274)
    const int mi = ldu(C.P.mat + A);
    const fdm_material Mi = matOf(C.pmat, mi);
    const double invMi = tA.invMass;
    double kn = 0., ks = 0., effM = 0., mu, diss;
    V3 vB, wB;
    if (SET == FDM_SET_WALL) {
      const fdm_material Mw = matOf(C.wmat, ldu(C.W.mat + T));
      if (invMi > 0.) effM = 1. / invMi;
      mu = fmin(Mi.mu, Mw.mu);
      diss = Mi.e <= Mw.e ? Mi.dissipation : Mw.dissipation;
      kn = Mi.kn;
      ks = Mi.ks;
      vB = ld3R(C.W.v, C.W.n, T);
      wB = ld3R(C.W.w, C.W.n, T);
    } else {
      const fdm_material Mj = matOf(C.pmat, ldu(C.P.mat + T));
      const double invMj = tg.t.invMass;
      if (Mi.kn > 0. && Mj.kn > 0.) kn = Mi.kn * Mj.kn / (Mi.kn + Mj.kn);
      if (Mi.ks > 0. && Mj.ks > 0.) ks = Mi.ks * Mj.ks / (Mi.ks + Mj.ks);
      if (invMi > 0. || invMj > 0.) effM = 1. / (invMi + invMj);
      diss = Mi.e <= Mj.e ? Mi.dissipation : Mj.dissipation;
      mu = fmin(Mi.mu, Mj.mu);
      vB = SET == FDM_SET_GHOST && S.ghostVel
               ? ldd3R(S.ghostVel + 3 * (size_t)S.pairs.pairG[p])
               : forceVel(C, fr, T);
      wB = ld3R(C.P.w, n, T);  // a sector image keeps the real spin (contactKernel.cu:258)
    }
    const V3 vA = forceVel(C, fr, A);
    const V3 wA = ld3R(C.P.w, n, A);
    // contact law of one contact: its spring is updated in place and stored
    // with its node id as record r
    auto law = [&](V3 pc, V3 nrm, double ov, int k, int r, V3& F, V3& TA, V3& TB) {
      V3 spring = findPrevSpring(S, prevOff, prevCnt, k);
      if (C.updateSprings) {
        const V3 vc = vsub(vadd(vA, vcross(wA, vsub(pc, armA))), vadd(vB, vcross(wB, vsub(pc, armB))));
        linearContact(F, spring, vc, nrm, ov, C.dt, kn, ks, mu, diss, effM);
      }
      TA = vcross(vsub(pc, armA), F);
      TB = vcross(vsub(pc, armB), vneg(F));
      S.pairs.rec[r] = makeRecord(spring, k);
      if (C.dbgPoint) {
        C.dbgPoint[3 * r] = pc.x;
        C.dbgPoint[3 * r + 1] = pc.y;
        C.dbgPoint[3 * r + 2] = pc.z;
        C.dbgNormal[3 * r] = nrm.x;
        C.dbgNormal[3 * r + 1] = nrm.y;
        C.dbgNormal[3 * r + 2] = nrm.z;
        C.dbgOverlap[r] = ov;
      }
    };
    if (total <= kMaxHits) {
      // one staged contact per lane (the slots were written by other lanes)
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      V3 F = {0., 0., 0.}, TA = {0., 0., 0.}, TB = {0., 0., 0.};
      if (lane < total) {
        const V3 pc = {hs.pc[0][lane], hs.pc[1][lane], hs.pc[2][lane]};
        const V3 nrm = {hs.nrm[0][lane], hs.nrm[1][lane], hs.nrm[2][lane]};
        law(pc, nrm, hs.ov[lane], hs.node[lane], base + lane, F, TA, TB);
      }
      // pair sums, serially in node order
      for (int b = 0; b < total; ++b) {
        SF = vadd(SF, {readlaneD(F.x, b), readlaneD(F.y, b), readlaneD(F.z, b)});
        STA = vadd(STA, {readlaneD(TA.x, b), readlaneD(TA.y, b), readlaneD(TA.z, b)});
        STB = vadd(STB, {readlaneD(TB.x, b), readlaneD(TB.y, b), readlaneD(TB.z, b)});
      }
    } else {
      // more contacts than slots: recompute each chunk's hits
      const unsigned long long chunksWith = ballot64(myMask != 0ull);
      int running = 0;
      for (unsigned long long cw = chunksWith; cw; cw &= cw - 1ull) {
        const int c = __builtin_ctzll(cw);
        const unsigned lo32 = __builtin_amdgcn_readlane((unsigned)myMask, c);
        const unsigned hi32 = __builtin_amdgcn_readlane((unsigned)(myMask >> 32), c);
        const unsigned long long m = ((unsigned long long)hi32 << 32) | lo32;
        const bool hit = (m >> lane) & 1ull;
        const int k = c * FDM_CHUNK + lane;
        V3 F = {0., 0., 0.}, TA = {0., 0., 0.}, TB = {0., 0., 0.};
        if (hit) {
          const V3 s = {(double)nodes[3 * k], (double)nodes[3 * k + 1], (double)nodes[3 * k + 2]};
          const V3 pn = vadd(qrotate(qA, s), xA);
          Sample sm;
          nodeHit<SET>(pn, tg, tcell, tgrid, RB, sm);
          const double ov = -trilinear(sm.x, sm.y, sm.z, sm.c);
          const V3 nrm = vnormalize(toWorld(gradientIntX(sm.x, sm.y, sm.z, sm.c), tg));
          const V3 pc = vadd(pn, vmul(nrm, 0.5 * ov));
          law(pc, nrm, ov, k, base + running + __popcll(m & lt), F, TA, TB);
        }
        for (unsigned long long mm = m; mm; mm &= mm - 1ull) {
          const int b = __builtin_ctzll(mm);
          SF = vadd(SF, {readlaneD(F.x, b), readlaneD(F.y, b), readlaneD(F.z, b)});
          STA = vadd(STA, {readlaneD(TA.x, b), readlaneD(TA.y, b), readlaneD(TA.z, b)});
          STB = vadd(STB, {readlaneD(TB.x, b), readlaneD(TB.y, b), readlaneD(TB.z, b)});
        }
        running += __popcll(m);
      }
    }
  }
  if (lane == 0) {
    S.pairs.recOff[p] = base;
    S.pairs.recCnt[p] = total;
    double* f = S.pairs.sumF + 3 * (size_t)p;
    double* ta = S.pairs.sumTA + 3 * (size_t)p;
    double* tb = S.pairs.sumTB + 3 * (size_t)p;
    f[0] = SF.x; f[1] = SF.y; f[2] = SF.z;
    ta[0] = STA.x; ta[1] = STA.y; ta[2] = STA.z;
    tb[0] = STB.x; tb[1] = STB.y; tb[2] = STB.z;
    if (SET != FDM_SET_WALL && total > 0 && T != A) {
      const int pos = atomicAdd(&S.mirror.count[T], 1);
      if (pos < S.mirror.capacity) S.mirror.list[(size_t)T * S.mirror.capacity + pos] = p;
      else atomicOr(C.status, FDM_STATUS_BUCKET_OVERFLOW);
    }
  }
}

template <int SET>
__global__ void __launch_bounds__(256) kNarrow(NarrowK a) {
  __shared__ HitSlots slots[4];
  const int lane = laneId();
  const int wpb = blockDim.x >> 6;
  const int total = min(*a.s.pairs.total, a.s.pairs.capacity);
  const int stride = gridDim.x * wpb;
  HitSlots& hs = slots[threadIdx.x >> 6];
  for (int p = blockIdx.x * wpb + (threadIdx.x >> 6); p < total; p += stride)
    processPair<SET>(a.c, a.s, p, lane, hs, p % FDM_REC_POOLS);
}

// ---------------------------------------------------------------------------
// Narrow phase of several sets in one kernel: culls, exact predicate and
// contact law of runs of pairs (sweepRun).

struct NarrowScratch {
  double* hitGeom;   // [8 * hitCapacity]: contact point, normal, overlap, node id
  int hitCapacity;
  int* hitCount;     // [FDM_REC_COUNTERS] pool counters of the staged contacts
};

// ------------------------------------------------------------------- sweep
// What the culls need of one pair, in FP32 (margins below). With SDF grids:
// a point s of A's template frame has the index coordinates m s + t in the
// target's grid; a plane wall uses row 0 as its value there.
struct alignas(16) CullRec {
  float m[9], t[3];
  float centre[3], radius;   // target's centre in index coordinates, bounding radius (spacings)
  float top[3], eps;         // nodes per axis - 1; slack of an index coordinate
  float scale, planeSlack;   // spacings per length (plane walls: |gradient|)
  int size[2];               // cells per axis, x and y
  long long cells;           // first cell code; -1: a plane wall
  int groupStart, groupCount;
};
// What the exact predicate needs of one pair.
struct PairCtx {
  double qA[4], xA[3], qT[4], xT[3], ih;
  int geoA, geoT, hash, inst, ghost;
};
// What the contact law needs of one pair of a run.
struct LawRec {
  int base, first;        // first record (-1: none), first of the run's contacts
  int prevOff, prevCnt;   // the pair's records of the previous step
  int A, T;
  int staged;             // first staged contact (contacts in memory)
};
constexpr int kRunMax = 8;                  // pairs of one wave and item
constexpr int kUnitLanes = FDM_GROUP;       // groups per unit of the group cull, nodes per group
constexpr int kMaxBlocks = FDM_CHUNK * FDM_MAX_CHUNKS / (FDM_GROUP * kUnitLanes);  // units per pair
constexpr int kLiveMax = 256;
// Per-wave LDS of the sweep.
struct SweepSlots {
  CullRec cull[kRunMax];
  PairCtx ctx[kRunMax];
  // rows 0-6: point, normal and overlap of the run's hits in the order found;
  // then force and torques of its contacts in the order of their sums
  double c[9][kMaxHits];
  unsigned long long chunks[kRunMax];  // chunks of the pair holding hits
  LawRec law[kRunMax];
  int hit[kMaxHits];                                       // pair of the run << 16 | node
  int cand[64];  // nodes that passed the cell test, not yet tested exactly (same coding)
  int total[kRunMax];
  unsigned short unit[kRunMax * kMaxBlocks];  // pair << 8 | block of groups
  unsigned short live[kLiveMax];              // pair << 8 | surviving group
};
template <bool MANY>
__device__ __forceinline__ fdm_grid particleGrid(const NarrowCommon& C, int inst) {
  if (MANY) return ldu(C.inst.pgrid + inst);
  // (opaque in every run: what is computed from them, as the periods, would
  // otherwise be kept in VGPRs over the wave's whole loop)
  fdm_grid g = C.pgrid;
  asm volatile("" : "+s"(g.min.x), "+s"(g.min.y), "+s"(g.max.x), "+s"(g.max.y));
  return g;
}
// (images of a sector boundary in a kernel of their own: what turns them
// costs registers)
template <bool MANY, bool SECTOR>
__device__ __forceinline__ fdm_periodic particlePeriodic(const NarrowCommon& C, int inst) {
  fdm_periodic p = MANY ? ldu(C.inst.periodic + inst) : C.periodic;
  if (!SECTOR) p.sector = 0;
  return p;
}
template <int SET, bool MANY>
__device__ __forceinline__ fdm_grid targetGrid(const NarrowCommon& C, const NarrowSet& S, int inst) {
  if (MANY) return SET == FDM_SET_WALL ? ldu(C.inst.wgrid + inst) : ldu(C.inst.pgrid + inst);
  return S.grid;
}
__device__ __forceinline__ int lanesBelow(unsigned long long m) {  // set bits of lanes below this one
  return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}
// Inclusive sum over lanes 0 to kRunMax - 1 (lanes of one row: a row shift
// fills with zero, and no lane index is kept over the wave's loop).
__device__ __forceinline__ int runScan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);
  return v;
}
__device__ __forceinline__ float clampTo(float u, float hi) { return __builtin_amdgcn_fmed3f(u, 0.f, hi); }
// The code of the SDF cell nearest to index coordinates u (their clamped
// values in c), and the cell's indices.
__device__ __forceinline__ int cellCode(const CullRec& k, const unsigned char* cells, const float u[3],
                                        float c[3], int i[3]) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    c[a] = clampTo(u[a], k.top[a]);
    i[a] = min((int)c[a], (int)k.top[a] - 1);
  }
  return cells[k.cells + i[0] + k.size[0] * (i[1] + k.size[1] * i[2])];
}
__device__ __forceinline__ void cullPoint(const CullRec& k, float x, float y, float z, float u[3]) {
#pragma unroll
  for (int a = 0; a < 3; ++a)
    u[a] = fmaf(k.m[3 * a], x, fmaf(k.m[3 * a + 1], y, fmaf(k.m[3 * a + 2], z, k.t[a])));
}
template <int SET>
__device__ __forceinline__ bool inSphere(const CullRec& k, const float u[3], float r) {
  if (SET != FDM_SET_PARTICLE) return true;
  const float x = u[0] - k.centre[0], y = u[1] - k.centre[1], z = u[2] - k.centre[2], rr = k.radius + r;
  return fmaf(x, x, fmaf(y, y, z * z)) <= rr * rr;
}
// Whether the ball about the point s of A's frame may hold a contact of the
// pair: a contact point q lies in a cell with code 0, the point p of the SDF
// box nearest to the ball's centre has |centre - q|^2 >= |centre - p|^2 +
// |p - q|^2 (the box is convex), and |p - q| is at least the distance that
// the code of p's cell gives.
template <int SET>
__device__ __forceinline__ bool ballMayTouch(const CullRec& k, const unsigned char* cells, float4 s) {
  float u[3], c[3];
  cullPoint(k, s.x, s.y, s.z, u);
  if (SET == FDM_SET_WALL && k.cells < 0) return u[0] - k.scale * s.w <= k.planeSlack;
  const float r = fmaf(s.w, k.scale, 2.f * k.eps);
  if (!inSphere<SET>(k, u, r)) return false;
  int i[3];
  const float d = (float)max(cellCode(k, cells, u, c, i) - 1, 0) * (1.f / FDM_CELL_UNIT);
  const float ex = u[0] - c[0], ey = u[1] - c[1], ez = u[2] - c[2];
  return fmaf(ex, ex, fmaf(ey, ey, fmaf(ez, ez, d * d))) * (1.f - 1e-5f) <= r * r;
}
// The same for a node: its cell's code is 0, or it lies within the slack of a
// face of a cell next to such a cell.
template <int SET>
__device__ __forceinline__ bool nodeMayTouch(const CullRec& k, const unsigned char* cells, float4 s) {
  float u[3], c[3];
  cullPoint(k, s.x, s.y, s.z, u);
  if (SET == FDM_SET_WALL && k.cells < 0) return u[0] <= k.planeSlack;
  if (!inSphere<SET>(k, u, k.eps)) return false;
  int i[3];
  const int code = cellCode(k, cells, u, c, i);
  if (!(fmaxf(fmaxf(fabsf(u[0] - c[0]), fabsf(u[1] - c[1])), fabsf(u[2] - c[2])) <= k.eps)) return false;
  if (code != 1) return code == 0;
  float f = 1.f;
#pragma unroll
  for (int a = 0; a < 3; ++a) f = fminf(f, fminf(c[a] - (float)i[a], (float)(i[a] + 1) - c[a]));
  return f <= k.eps;
}

// The linear spring-dashpot law of one contact of a run, contact `at` of its
// pair in node order: its spring is updated and left as its record, its force
// and torques in `slot`.
template <int SET, bool MANY, bool SECTOR>
__device__ __forceinline__ void lawContact(const NarrowCommon& C, const NarrowSet& S, const PairCtx& c, const LawRec& lr,
                                           int node, int at, V3 pc, V3 nrm, double ov, SweepSlots& ws, int slot) {
  // the pair's previous contact at this place, nearly always of the same node
  fdm_record pr{};
  if (lr.prevCnt > 0) pr = ldu(S.prev.rec + lr.prevOff + min(at, lr.prevCnt - 1));
  const int n = C.P.n;
  const fdm_grid pg = particleGrid<MANY>(C, c.inst);
  const PairFrame fr = {&pg, &pg, particlePeriodic<MANY, SECTOR>(C, c.inst)};
  // material constants of the pair (contactKernel.cu:79-110,167-193,243-274)
  const fdm_material Mi = matOf(C.pmat, ldu(C.P.mat + lr.A));
  const double invMi = ldu(&C.pgeo.info[c.geoA].invMass);
  double kn = 0., ks = 0., effM = 0., mu, diss;
  V3 vB, wB;
  if (SET == FDM_SET_WALL) {
    const fdm_material Mw = matOf(C.wmat, ldu(C.W.mat + lr.T));
    if (invMi > 0.) effM = 1. / invMi;
    mu = fmin(Mi.mu, Mw.mu);
    diss = Mi.e <= Mw.e ? Mi.dissipation : Mw.dissipation;
    kn = Mi.kn;
    ks = Mi.ks;
    vB = ld3R(C.W.v, C.W.n, lr.T);
    wB = ld3R(C.W.w, C.W.n, lr.T);
  } else {
    const fdm_material Mj = matOf(C.pmat, ldu(C.P.mat + lr.T));
    const double invMj = ldu(&C.pgeo.info[c.geoT].invMass);
    if (Mi.kn > 0. && Mj.kn > 0.) kn = Mi.kn * Mj.kn / (Mi.kn + Mj.kn);
    if (Mi.ks > 0. && Mj.ks > 0.) ks = Mi.ks * Mj.ks / (Mi.ks + Mj.ks);
    if (invMi > 0. || invMj > 0.) effM = 1. / (invMi + invMj);
    diss = Mi.e <= Mj.e ? Mi.dissipation : Mj.dissipation;
    mu = fmin(Mi.mu, Mj.mu);
    vB = SECTOR && SET == FDM_SET_GHOST && S.ghostVel ? ldd3R(S.ghostVel + 3 * (size_t)c.ghost) : forceVel(C, fr, lr.T);
    wB = ld3R(C.P.w, n, lr.T);  // a sector image keeps the real spin (contactKernel.cu:258)
  }
  const V3 vA = forceVel(C, fr, lr.A);
  const V3 wA = ld3R(C.P.w, n, lr.A);
  const V3 xA = {c.xA[0], c.xA[1], c.xA[2]}, xT = {c.xT[0], c.xT[1], c.xT[2]};
  const V3 armA = SET == FDM_SET_GHOST ? xA : wrappedArm(xA, pg, fr.periodic);
  const V3 armB = SET == FDM_SET_PARTICLE ? wrappedArm(xT, pg, fr.periodic) : xT;
  V3 F = {0., 0., 0.}, spring = {0., 0., 0.};
  if (lr.prevCnt > 0) spring = pr.node == node ? recordSpring(pr) : findPrevSpring(S, lr.prevOff, lr.prevCnt, node);
  if (C.updateSprings) {
    const V3 vc = vsub(vadd(vA, vcross(wA, vsub(pc, armA))), vadd(vB, vcross(wB, vsub(pc, armB))));
    linearContact(F, spring, vc, nrm, ov, C.dt, kn, ks, mu, diss, effM);
  }
  const V3 TA = vcross(vsub(pc, armA), F), TB = vcross(vsub(pc, armB), vneg(F));
  const double v[9] = {F.x, F.y, F.z, TA.x, TA.y, TA.z, TB.x, TB.y, TB.z};
#pragma unroll
  for (int c = 0; c < 9; ++c) ws.c[c][slot] = v[c];
  const int r = lr.base + at;
  S.pairs.rec[r] = makeRecord(spring, node);
  if (C.dbgPoint) {
    C.dbgPoint[3 * r] = pc.x;
    C.dbgPoint[3 * r + 1] = pc.y;
    C.dbgPoint[3 * r + 2] = pc.z;
    C.dbgNormal[3 * r] = nrm.x;
    C.dbgNormal[3 * r + 1] = nrm.y;
    C.dbgNormal[3 * r + 2] = nrm.z;
    C.dbgOverlap[r] = ov;
  }
}

// Node sweep of a run of `np` <= kRunMax candidate pairs of one set by one
// wave: the pairs, their node groups and their nodes are culled in the
// target's frame, the remaining nodes of all the run's pairs take the
// reference's exact predicate together, and the contact law runs with one
// contact per lane, each pair's forces and torques added in node order.
//
// A pair is a chain of dependent loads (list, bodies, templates, groups,
// cell codes, nodes, cell codes, SDF corners) with little arithmetic between
// them, and each stage leaves a different number of items per pair. So a run
// goes through the stages together, each stage's items taken from a list in
// LDS and dealt to all lanes:
//  - one pair per lane: poses, bounding spheres, and the map from A's
//    template frame to the target's SDF index coordinates (one 3 x 3 matrix
//    and a shift);
//  - one node group (16 nodes) per lane, then one node per lane: placed with
//    nine multiply-adds and tested against one byte, its SDF cell's code: the
//    distance to the nearest cell in which phi can be <= 0. (A Lipschitz
//    bound of phi does not serve here: f / |grad f| is steep to 1e9 at the
//    centre of a superellipsoid.) Affine walls test the plane instead;
//  - the exact predicate (two quaternion rotations, eight SDF corners, the
//    cell stencil: some 300 FP64 instructions) for the few nodes left;
//  - the contact law from the contacts in LDS: the records are reserved by one
//    pair per lane (their atomics issued together), then one contact per lane,
//    then one component of a pair's sums per lane. As a kernel of its own with
//    a thread per pair the law was a serial chain over the pair's contacts,
//    with their geometry passed through memory. A run with more contacts than
//    the 64 slots recomputes them chunk by chunk and stages them in memory.
// Measured against one pair per wave with 64-node chunks culled by Lipschitz
// bound and swept in FP64 (and wall pairs four per wave): 254K particle pairs
// of a compressed lattice, 23 % of them in contact, 613 + 22 -> 201 us; the
// million-particle pour's 11.4K wall, 5.8K particle and 4.1K image pairs 44.3
// -> 23 us; 44.6K pairs of touching 400-node spheres 79 -> 29 us; one pair
// alone 10.7 -> 10.1 us. With the law, against the sweep and the law kernel:
// 201 + 46 -> 220 us; 23.1 + 11.7 -> 24.5 us; 216 particles, up to 20 contacts
// a pair, 11.8 + 19.5 -> 13.3 us; one pair 10.0 + 5.1 -> 11.8 us.
// Margins: reaches are widened by kReach (a unit quaternion stored in FP32
// scales vectors by up to 1 +- 2.4e-7), and index coordinates by eps, which
// covers the FP32 rounding of the map, of the nodes and of their sums (a few
// 2^-24 of the largest coordinate) and the exact predicate's own rounding.
template <int SET, bool MANY, bool SECTOR>
__device__ void sweepRun(const NarrowCommon& C, const NarrowSet& S, const NarrowScratch& X, int w0, int p0, int np,
                         int lane, SweepSlots& ws) {
  // (opaque in every run, as the grid in particleGrid)
  asm volatile("" : "+v"(lane));
  const int n = C.P.n;
  const int p = p0 + lane, w = w0 + lane;
  const fdm_geometry& tgeo = SET == FDM_SET_WALL ? C.wgeo : C.pgeo;
  auto emptyRange = [&]() __attribute__((always_inline)) {
    S.pairs.recOff[p] = 0;
    S.pairs.recCnt[p] = 0;
  };
  int units = 0;
  if (lane < np) {
    int prevOff = 0, prevCnt = -1;  // previous record range of the pair (-1: not at its index)
    ws.total[lane] = 0;
    ws.chunks[lane] = 0ull;
    const int A = ldu(S.pairs.pairA + p), T = ldu(S.pairs.pairT + p);
    // (lists kept from the previous step hold the pair at the same index:
    // these loads go along with the pair's own)
    if (p < min(ldu(S.prev.total), S.prev.capacity)) {
      const int pA = ldu(S.prev.pairA + p), pT = ldu(S.prev.pairT + p);
      prevOff = ldu(S.prev.recOff + p);
      prevCnt = ldu(S.prev.recCnt + p);
      if (pA != A || pT != T) prevCnt = -1;
    }
    ws.law[lane] = {-1, 0, prevOff, prevCnt, A, T, 0};
    if (A >= 0) {  // (below zero: a slot left empty by a capacity overflow)
      const int inst = MANY ? ldu(C.inst.particleInstance + A) : 0;
      const fdm_grid pg = particleGrid<MANY>(C, inst);
      const fdm_periodic per = particlePeriodic<MANY, SECTOR>(C, inst);
      // A's and the target's poses as the set's detection sees them
      V3 xA = ldpR(C.P.x, n, A);
      Q4 qA = ld4R(C.P.q, n, A);
      const int geoA = ldu(C.P.geo + A);
      V3 xT;
      Q4 qT;
      int hash, geoT;
      if (SET == FDM_SET_WALL) {
        xT = ldpR(C.W.x, C.W.n, T);
        qT = ld4R(C.W.q, C.W.n, T);
        geoT = ldu(C.W.geo + T);
        hash = ldu(S.targetHash + T);
      } else {
        xT = ldpR(C.P.x, n, T);
        qT = ld4R(C.P.q, n, T);
        geoT = ldu(C.P.geo + T);
        if (SET == FDM_SET_PARTICLE) hash = ldu(S.targetHash + T);
      }
      if (SET == FDM_SET_GHOST) {
        if (per.sector) {
          const SectorWrap sw = sectorWrap(xA, pg, per);
          qA = sectorTurnQ(qA, sw.turns, per);
          xA = sw.x;
        } else {
          xA = wrapStages(xA, pg, per).afterY;
        }
        if (S.ghostFromReal) {
          const WrapStages ww = wrapStages(xT, pg, per);
          xT = ghostOf(S.ghostMask == 1 ? ww.afterX : ww.afterY, pg, S.ghostMask);
          hash = ghostCellHash(xT, pg);
        } else {
          const int gi = ldu(S.pairs.pairG + p);
          ws.ctx[lane].ghost = gi;
          xT = ldd3R(S.ghostPos + 3 * (size_t)gi);
          hash = ldu(S.ghostHash + gi);
          if (SECTOR && S.ghostQ) {
            const double* gq = S.ghostQ + 4 * (size_t)gi;
            qT = {gq[0], gq[1], gq[2], gq[3]};
          }
        }
      }
      // (every template value is loaded before the sphere test, so that the
      // loads go together)
      const fdm_template* tA = C.pgeo.info + geoA;
      const fdm_template* tT = tgeo.info + geoT;
      const double RA = ldu(&tA->radius), RB = ldu(&tT->radius), reachT = ldu(&tT->boxReach);
      const int groups = ldu(&tA->groupCount), groupStart = ldu(&tA->groupStart);
      const double ih = ldu(&tT->invSpacing);
      const V3 o = {ldu(&tT->origin[0]), ldu(&tT->origin[1]), ldu(&tT->origin[2])};
      const int nx = ldu(&tT->size[0]), ny = ldu(&tT->size[1]), nz = ldu(&tT->size[2]);
      const long long cellStart = ldu(&tT->cellStart);
      const bool plane = SET == FDM_SET_WALL && ldu(&tT->affine);
      V3 a = {0., 0., 0.};
      double a3 = 0., slack = 0.;
      if (SET == FDM_SET_WALL) {
        a = {ldu(&tT->plane[0]), ldu(&tT->plane[1]), ldu(&tT->plane[2])};
        a3 = ldu(&tT->plane[3]);
        slack = ldu(&tT->planeSlack);
      }
      const V3 d = vsub(xA, xT);
      const double rs = (RA + (SET == FDM_SET_PARTICLE ? RB : reachT)) * kReach;
      if (vlen2(d) <= rs * rs) {
        units = (groups + kUnitLanes - 1) / kUnitLanes;
        PairCtx& c = ws.ctx[lane];
        c.qA[0] = qA.q0; c.qA[1] = qA.q1; c.qA[2] = qA.q2; c.qA[3] = qA.q3;
        c.xA[0] = xA.x; c.xA[1] = xA.y; c.xA[2] = xA.z;
        c.qT[0] = qT.q0; c.qT[1] = qT.q1; c.qT[2] = qT.q2; c.qT[3] = qT.q3;
        c.xT[0] = xT.x; c.xT[1] = xT.y; c.xT[2] = xT.z;
        c.geoA = geoA;
        c.geoT = geoT;
        c.hash = hash;
        c.inst = inst;
        CullRec& k = ws.cull[lane];
        k.groupStart = groupStart;
        k.groupCount = groups;
        if (plane) {
          // the plane's value at s is c0 + u . s (the rotation formula's
          // transpose is the conjugate's for any quaternion)
          const V3 ga = qrotate(qT, a);
          const V3 u = qrotateT(ga, qA);
          const double c0 = a3 + vdot(ga, d);
          const double a1 = fabs(a.x) + fabs(a.y) + fabs(a.z);
          k.m[0] = (float)u.x;
          k.m[1] = (float)u.y;
          k.m[2] = (float)u.z;
          k.t[0] = (float)c0;
          k.scale = (float)(a1 * kReach);
          k.planeSlack = (float)((slack + 2e-6 * (fabs(c0) + a1 * RA)) * kReach);
          k.cells = -1;
        } else {
          c.ih = ih;
          k.centre[0] = (float)(-o.x * ih);
          k.centre[1] = (float)(-o.y * ih);
          k.centre[2] = (float)(-o.z * ih);
          // (the pair's coordinates stay within the two reaches of the centre)
          const double span = (2. * RA + reachT) * ih;
          k.eps = (float)(1e-4 + 2e-6 * span);
          k.radius = (float)(RB * ih * kReach) + k.eps;
          k.scale = (float)(ih * kReach);
          k.top[0] = (float)(nx - 1);
          k.top[1] = (float)(ny - 1);
          k.top[2] = (float)(nz - 1);
          k.size[0] = nx - 1;
          k.size[1] = ny - 1;
          k.cells = cellStart;
        }
      }
    }
    if (units == 0) emptyRange();
  }
  // units of the group cull, pair by pair
  const int before = runScan(units);
  const int nUnits = readlaneI(before, kRunMax - 1);
  if (nUnits == 0) return;
  for (int u = 0; u < units; ++u) ws.unit[before - units + u] = (unsigned short)(lane << 8 | u);
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");

  auto quat = [](const double* q) __attribute__((always_inline)) { return Q4{q[0], q[1], q[2], q[3]}; };
  // the maps of the run's pairs, one column per lane (column 3: the shift)
  {
    const int j = lane >> 2, col = lane & 3;
    const bool has = __builtin_amdgcn_ds_bpermute(4 * j, units) > 0;
    if (has && (SET != FDM_SET_WALL || ws.cull[j].cells >= 0)) {
      const PairCtx& c = ws.ctx[j];
      CullRec& k = ws.cull[j];
      const V3 e = qrotate(quat(c.qA), {col == 0 ? 1. : 0., col == 1 ? 1. : 0., col == 2 ? 1. : 0.});
      const V3 d = vsub({c.xA[0], c.xA[1], c.xA[2]}, {c.xT[0], c.xT[1], c.xT[2]});
      const V3 l = vmul(qrotateT({col < 3 ? e.x : d.x, col < 3 ? e.y : d.y, col < 3 ? e.z : d.z}, quat(c.qT)), c.ih);
      if (col < 3) {
        k.m[col] = (float)l.x;
        k.m[3 + col] = (float)l.y;
        k.m[6 + col] = (float)l.z;
      } else {
        k.t[0] = (float)l.x + k.centre[0];
        k.t[1] = (float)l.y + k.centre[1];
        k.t[2] = (float)l.z + k.centre[2];
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  auto identity = [](Q4 q) __attribute__((always_inline)) {
    return q.q0 == 1.0 && q.q1 == 0.0 && q.q2 == 0.0 && q.q3 == 0.0;
  };
  // contact point, normal and overlap of a hit
  auto contactOf = [&](V3 pn, const Sample& sm, int j, V3& pc, V3& nrm, double& ov) __attribute__((always_inline)) {
    ov = -trilinear(sm.x, sm.y, sm.z, sm.c);
    const V3 gr = gradientIntX(sm.x, sm.y, sm.z, sm.c);
    const Q4 q = quat(ws.ctx[j].qT);
    nrm = vnormalize(identity(q) ? gr : qrotate(q, gr));
    pc = vadd(pn, vmul(nrm, 0.5 * ov));
  };
  // the exact predicate for node `id` of the run's pair j
  auto exact = [&](int j, int id, V3& pn, Sample& sm) __attribute__((always_inline)) {
    const PairCtx& c = ws.ctx[j];
    const fdm_template* tp = tgeo.info + c.geoT;
    const fdm_real* s = C.pgeo.nodes + 3 * ((size_t)ldu(&C.pgeo.info[c.geoA].nodeStart) + id);
    pn = vadd(qrotate(quat(c.qA), {(double)s[0], (double)s[1], (double)s[2]}), {c.xA[0], c.xA[1], c.xA[2]});
    Target tg;
    tg.x = {c.xT[0], c.xT[1], c.xT[2]};
    tg.q = quat(c.qT);
    tg.ident = identity(tg.q);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      tg.t.origin[a] = ldu(&tp->origin[a]);
      tg.t.size[a] = ldu(&tp->size[a]);
    }
    tg.t.invSpacing = ldu(&tp->invSpacing);
    tg.t.sdfStart = ldu(&tp->sdfStart);
    tg.t.affine = 0;
    tg.sdf = tgeo.sdf;
    tg.hash = c.hash;
    const fdm_grid tgrid = targetGrid<SET, MANY>(C, S, c.inst);
    return nodeHit<SET>(pn, tg, decodeHash(c.hash, tgrid), tgrid, ldu(&tp->radius), sm);
  };

  const float4* groups = reinterpret_cast<const float4*>(C.pgeo.groups);
  const float4* nodes = reinterpret_cast<const float4*>(C.pgeo.groupNodes);
  const int sub = lane / kUnitLanes, sl = lane % kUnitLanes;
  int iu = 0;                          // next unit
  int nlive = 0, il = 0;               // surviving groups, and the next of them
  int ncand = 0, nhit = 0;
  while (true) {
    // groups, while the list has room
    while (iu < nUnits && nlive + 64 <= kLiveMax) {
      bool live = false;
      int code = 0;
      if (iu + sub < nUnits) {
        const int un = ws.unit[iu + sub];
        const CullRec& k = ws.cull[un >> 8];
        const int g = (un & 0xFF) * kUnitLanes + sl;
        code = (un & 0xFF00) | g;
        if (g < k.groupCount) live = ballMayTouch<SET>(k, tgeo.cells, groups[k.groupStart + g]);
      }
      iu += 64 / kUnitLanes;
      const unsigned long long m = ballot64(live);
      if (live) ws.live[nlive + lanesBelow(m)] = (unsigned short)code;
      nlive += __popcll(m);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // nodes, until 64 are at hand
    bool full = false;
    while (il < nlive) {
      bool cand = false;
      int code = 0;
      if (il + sub < nlive) {
        const int lv = ws.live[il + sub];
        const CullRec& k = ws.cull[lv >> 8];
        const float4 s = nodes[FDM_GROUP * (size_t)(k.groupStart + (lv & 0xFF)) + sl];
        const int id = __float_as_int(s.w);
        code = (lv & 0xFF00) << 8 | id;
        cand = id >= 0 && nodeMayTouch<SET>(k, tgeo.cells, s);
      }
      const unsigned long long m = ballot64(cand);
      if (ncand + __popcll(m) > 64) {  // these groups again after the exact test
        full = true;
        break;
      }
      il += 64 / kUnitLanes;
      if (cand) ws.cand[ncand + lanesBelow(m)] = code;
      ncand += __popcll(m);
    }
    if (!full) {
      nlive = il = 0;
      if (iu < nUnits) continue;
    }
    if (ncand > 0) {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      bool hit = false;
      Sample sm;
      V3 pn = {0., 0., 0.};
      int code = 0;
      if (lane < ncand) {
        code = ws.cand[lane];
        hit = exact(code >> 16, code & 0xFFFF, pn, sm);
      }
      const unsigned long long m = ballot64(hit);
      if (hit) {
        const int slot = nhit + lanesBelow(m);
        if (slot < kMaxHits) {
          V3 pc, nrm;
          double ov;
          contactOf(pn, sm, code >> 16, pc, nrm, ov);
          const double v[7] = {pc.x, pc.y, pc.z, nrm.x, nrm.y, nrm.z, ov};
#pragma unroll
          for (int c = 0; c < 7; ++c) ws.c[c][slot] = v[c];
          ws.hit[slot] = code;
        }
        atomicAdd(&ws.total[code >> 16], 1);
        atomicOr(&ws.chunks[code >> 16], 1ull << ((code & 0xFFFF) / FDM_CHUNK));
      }
      nhit += __popcll(m);
      ncand = 0;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    if (!full) break;
  }

  // the record reservations and the mirror slots, one pair per lane, their
  // atomics issued together
  const bool open = units > 0;
  int total = open ? ws.total[lane] : 0;
  if (open && total == 0) emptyRange();
  if (nhit == 0) return;
  const bool has = total > 0, all = nhit <= kMaxHits;
  int base = -1, gbase = 0, mpos = 0;
  const int first = runScan(total) - total;  // first of the pair's contacts among the run's
  if (has) {
    const LawRec lr = ws.law[lane];
    const int A = lr.A, T = lr.T;
    const bool mirrored = SET != FDM_SET_WALL && T != A;
    int prevOff = lr.prevOff, prevCnt = lr.prevCnt;
    const int pool = w % FDM_REC_POOLS;
    base = atomicAdd(S.pairs.recTotal + pool * FDM_REC_STRIDE, total);
    if (!all) gbase = atomicAdd(X.hitCount + pool * FDM_REC_STRIDE, total);
    if (mirrored) mpos = atomicAdd(&S.mirror.count[T], 1);
    if (prevCnt < 0) prevCnt = findPrevPair(S, p, A, T, prevOff);
    const int cap = S.pairs.recCapacity / FDM_REC_POOLS, gcap = X.hitCapacity / FDM_REC_POOLS;
    if (base + total > cap || gbase + total > gcap) {
      atomicOr(C.status, base + total > cap ? FDM_STATUS_RECORD_OVERFLOW : FDM_STATUS_STAGING_OVERFLOW);
      total = 0;
    }
    gbase += pool * gcap;
    S.pairs.recOff[p] = total > 0 ? base + pool * cap : 0;
    S.pairs.recCnt[p] = total;
    base = total > 0 ? base + pool * cap : -1;
    // (a pair whose reservation overflowed keeps its mirror slot, with no
    // records and zero sums: the slot count and the list agree, and the
    // target's fold adds nothing stale)
    if (mirrored) {
      if (mpos < S.mirror.capacity) S.mirror.list[(size_t)T * S.mirror.capacity + mpos] = p;
      else atomicOr(C.status, FDM_STATUS_BUCKET_OVERFLOW);
      if (total == 0)
        for (int c = 0; c < 3; ++c) {
          S.pairs.sumF[3 * (size_t)p + c] = 0.;
          S.pairs.sumTB[3 * (size_t)p + c] = 0.;
        }
    }
    ws.law[lane] = {base, first, prevOff, prevCnt, A, T, gbase};
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");

  // more contacts than slots: each pair's chunks with contacts again, staged
  // in node order
  if (!all) {
    for (int j = 0; j < np; ++j) {
      if (ws.law[j].base < 0) continue;
      int at = ws.law[j].staged;
      const int count = ldu(&C.pgeo.info[ws.ctx[j].geoA].nodeCount);
      for (unsigned long long cm = ws.chunks[j]; cm; cm &= cm - 1ull) {
        const int id = __builtin_ctzll(cm) * FDM_CHUNK + lane;
        V3 pn = {0., 0., 0.};
        Sample sm;
        const bool hit = id < count && exact(j, id, pn, sm);
        const unsigned long long m = ballot64(hit);
        if (hit) {
          V3 pc, nrm;
          double ov;
          contactOf(pn, sm, j, pc, nrm, ov);
          double* g = X.hitGeom + 8 * (size_t)(at + lanesBelow(m));
          const double v[8] = {pc.x, pc.y, pc.z, nrm.x, nrm.y, nrm.z, ov, (double)id};
#pragma unroll
          for (int c = 0; c < 8; ++c) g[c] = v[c];
        }
        at += __popcll(m);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  }
  // the contact law, one contact per lane, and the pairs' sums in node order
  for (int b = 0; b < nhit; b += 64) {
    asm volatile("" : "+v"(lane));  // (as above)
    const int m = min(nhit - b, 64);
    int code = INT_MAX, at = 0;
    V3 pc = {0., 0., 0.}, nrm = {0., 0., 0.};
    double ov = 0.;
    if (all) {
      // a contact's place: the contacts of its pair at lower nodes come first
      if (lane < m) code = ws.hit[lane];
      for (int h = 0; h < m; ++h) {
        const int c = readlaneI(code, h);
        at += (c >> 16) == (code >> 16) && c < code ? 1 : 0;
      }
      pc = {ws.c[0][lane], ws.c[1][lane], ws.c[2][lane]};
      nrm = {ws.c[3][lane], ws.c[4][lane], ws.c[5][lane]};
      ov = ws.c[6][lane];
    } else if (lane < m) {
      int j = 0;
      for (int q = 1; q < np; ++q)
        if (ws.total[q] > 0 && ws.law[q].first <= b + lane) j = q;
      at = b + lane - ws.law[j].first;
      code = j << 16;
      if (ws.law[j].base >= 0) {
        const double* g = X.hitGeom + 8 * (size_t)(ws.law[j].staged + at);
        pc = {g[0], g[1], g[2]};
        nrm = {g[3], g[4], g[5]};
        ov = g[6];
        code |= (int)g[7];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (lane < m) {
      const LawRec& lr = ws.law[code >> 16];
      const int to = lr.first + at - b;
      if (lr.base >= 0) lawContact<SET, MANY, SECTOR>(C, S, ws.ctx[code >> 16], lr, code & 0xFFFF, at, pc, nrm, ov, ws, to);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    for (int t = lane; t < 9 * np; t += 64) {
      const int q = t / 9, c = t % 9;
      const LawRec lr = ws.law[q];
      if (lr.base < 0) continue;
      const int end = lr.first + ws.total[q];
      double* out = c < 3 ? S.pairs.sumF : c < 6 ? S.pairs.sumTA : S.pairs.sumTB;
      out += 3 * (size_t)(p0 + q) + c % 3;
      // (a pair's sum goes on from batch to batch)
      double acc = lr.first < b && b < end ? *out : 0.;
      for (int i = max(lr.first - b, 0); i < min(end - b, 64); ++i) acc += ws.c[c][i];
      if (end > b && lr.first < b + 64) *out = acc;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
}

// Candidate pairs of all sets in one index space: set k holds the indices
// [start[k], start[k + 1]).
struct SetStarts {
  int v[kMaxSets + 1];
};
__device__ __forceinline__ SetStarts setStarts(const NarrowMulti& a) {
  SetStarts st;
  st.v[0] = 0;
#pragma unroll
  for (int k = 0; k < kMaxSets; ++k)
    st.v[k + 1] = st.v[k] + (k < a.nsets ? min(*a.s[k].pairs.total, a.s[k].pairs.capacity) : 0);
  return st;
}

// The sweep over the candidate pairs of every set: runs of pairs of one set
// per wave (sweepRun), persistent waves, no work list. One wave per workgroup
// (waves share nothing). Runs are as long as still gives every resident wave
// one (up to 1.5 for pairs of two, 2 for four): a short list is bound by the
// latency of one run, a long one by the instructions, which a run's pairs
// share.
//
// Work assignment: workgroups are dealt to the eight XCDs in turn (workgroup
// b runs on XCD b mod 8), each XCD with an L2 of its own, and neighbouring
// candidates share bodies, templates and list lines: so each XCD takes
// stretches of 64 consecutive pairs (stretch q on XCD q mod 8), its waves
// sharing out its runs. Items are taken from the end: the image sets (whose
// box test lets many pairs through) before the wall and particle sets.
template <bool MANY, bool SECTOR>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
kSweep(NarrowMulti a, NarrowScratch x) {
  __shared__ SweepSlots slots;
  const int lane = laneId();
  const int on = gateValue(a.gate, a.s[0].pairs.total);
  const SetStarts st = setStarts(a);
  asm volatile("" ::"s"(on), "s"(st.v[kMaxSets]));  // (loaded together)
  if (!on) return;
  int shift = 0;  // log2 of the pairs of a run
  while ((1 << shift) < kRunMax &&
         (st.v[kMaxSets] >> shift) > (int)gridDim.x + ((int)gridDim.x >> 1) * shift)
    ++shift;
  const int run = 1 << shift;
  int item[kMaxSets + 1];  // first item of each set
  item[0] = 0;
#pragma unroll
  for (int q = 0; q < kMaxSets; ++q) item[q + 1] = item[q] + ((st.v[q + 1] - st.v[q] + run - 1) >> shift);
  const int items = item[kMaxSets];
  const bool byXcd = gridDim.x % kXcds == 0;
  const int xcd = byXcd ? blockIdx.x % kXcds : 0;
  const int stride = byXcd ? gridDim.x / kXcds : gridDim.x;
  const int stretch = 6 - shift;  // log2 of the runs of a stretch
  for (int i = byXcd ? blockIdx.x / kXcds : blockIdx.x;; i += stride) {
    const int r = byXcd ? ((((i >> stretch) * kXcds) + xcd) << stretch) + (i & ((1 << stretch) - 1)) : i;
    if (r >= items) break;
    const int it = items - 1 - r;
    int k = 0, i0 = 0, g0 = 0, np = st.v[1];
#pragma unroll
    for (int q = 1; q < kMaxSets; ++q)  // constant indices: the starts stay scalar
      if (it >= item[q]) {
        k = q;
        i0 = item[q];
        g0 = st.v[q];
        np = st.v[q + 1] - st.v[q];
      }
    const NarrowSet& s = a.s[k];
    const int p0 = (it - i0) << shift;
    const int len = min(run, np - p0);
    if (s.kind == FDM_SET_PARTICLE) sweepRun<FDM_SET_PARTICLE, MANY, SECTOR>(a.c, s, x, g0 + p0, p0, len, lane, slots);
    else if (s.kind == FDM_SET_WALL) sweepRun<FDM_SET_WALL, MANY, SECTOR>(a.c, s, x, g0 + p0, p0, len, lane, slots);
    else sweepRun<FDM_SET_GHOST, MANY, SECTOR>(a.c, s, x, g0 + p0, p0, len, lane, slots);
  }
}

// The pre-cull, the sweep and the contact law in one pass: one wave per
// candidate pair (WAVES waves per workgroup) whose wave then
// applies the law to its pair's contacts (one contact per lane) and folds
// the pair sums in node order (processPair); no staging, no second kernel.
template <int WAVES>
__global__ void __launch_bounds__(64 * WAVES) kCullSweepLaw(NarrowMulti a) {
  if (gateOff(a.gate)) return;
  __shared__ HitSlots slots[WAVES];
  const int lane = laneId();
  const int wave = WAVES == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const SetStarts st = setStarts(a);
  const int total = st.v[kMaxSets];
  for (int g = blockIdx.x * WAVES + wave; g < total; g += gridDim.x * WAVES) {
    int k = 0, base = 0;
#pragma unroll
    for (int q = 1; q < kMaxSets; ++q)  // constant indices: the starts stay scalar
      if (g >= st.v[q]) {
        k = q;
        base = st.v[q];
      }
    const NarrowSet& s = a.s[k];
    const int p = g - base;
    const int pool = g % FDM_REC_POOLS;
    if (s.kind == FDM_SET_PARTICLE)
      processPair<FDM_SET_PARTICLE, true>(a.c, s, p, lane, slots[wave], pool);
    else if (s.kind == FDM_SET_WALL)
      processPair<FDM_SET_WALL, true>(a.c, s, p, lane, slots[wave], pool);
    else
      processPair<FDM_SET_GHOST, true>(a.c, s, p, lane, slots[wave], pool);
  }
}

__global__ void kResetCounter(int* c) {
  for (int i = threadIdx.x; i < FDM_REC_COUNTERS; i += blockDim.x) c[i] = 0;
}

}  // namespace fdm

namespace fdm {
namespace {
fdm_tuning g_tuning = {1, 16, 256, 256, 1, 1, 0};
}
const fdm_tuning& tuning() { return g_tuning; }
}  // namespace fdm

// The shapes t asks for, zero fields taken from the process default; false
// when a field is outside the documented shapes.
static bool completeTuning(const fdm_tuning& t, fdm_tuning& n) {
  n = fdm::tuning();
  if (t.sweepWaves) n.sweepWaves = t.sweepWaves;
  if (t.sweepWavesPerCU) n.sweepWavesPerCU = t.sweepWavesPerCU;
  if (t.lawBlock) n.lawBlock = t.lawBlock;
  if (t.reduceBlock) n.reduceBlock = t.reduceBlock;
  if (t.lawMode) n.lawMode = t.lawMode;
  if (t.nodesPerLane) n.nodesPerLane = t.nodesPerLane;
  if (t.wallGroups) n.wallGroups = t.wallGroups;
  if (!(n.sweepWaves == 1 || n.sweepWaves == 2 || n.sweepWaves == 4)) return false;
  if (n.sweepWavesPerCU < 4 || n.sweepWavesPerCU > 128) return false;
  if (!(n.lawBlock == 64 || n.lawBlock == 128 || n.lawBlock == 256)) return false;
  if (n.reduceBlock < 64 || n.reduceBlock > 1024 || n.reduceBlock % 64) return false;
  if (!(n.lawMode == 1 || n.lawMode == 2)) return false;
  if (n.nodesPerLane < 1 || n.nodesPerLane > 3) return false;
  if (n.wallGroups < 0 || n.wallGroups > 2) return false;
  return true;
}


using namespace fdm;

extern "C" int fdm_launchBroadPhase(const fdm_broadphase_args* args, void* workspace,
                                    size_t workspaceBytes, hipStream_t stream) {
  if (!args) return FDM_EINVAL;
  const fdm_broadphase_args& g = *args;
  const int n = g.particles.n;
  if (n < 0) return FDM_EINVAL;
  BroadK k;
  k.set = g.set;
  k.P = g.particles;
  k.pgeo = g.pgeo;
  k.W = g.walls;
  k.wgeo = g.wgeo;
  k.ghostCapacity = g.ghosts ? g.ghosts->capacity : 0;
  k.ghostCount = g.ghosts ? g.ghosts->count : nullptr;
  k.ghostReal = g.ghosts ? g.ghosts->realId : nullptr;
  k.ghostPos = g.ghosts ? g.ghosts->pos : nullptr;
  k.ghostBox = g.ghosts ? g.ghosts->cellBox : nullptr;
  k.grid = g.grid;
  k.table = g.table;
  k.pairs = g.pairs;
  k.status = nullptr;
  k.skin = g.skin;
  k.maxReach = g.maxReach;
  k.gate = g.gate;
  k.inst = g.inst;
  k.periodic = g.periodic;
  if (g.set == FDM_SET_GHOST && !g.ghosts) return FDM_EINVAL;
  if (!(g.skin >= 0.0) || !(g.maxReach >= 0.0)) return FDM_EINVAL;
  const unsigned nb = blocksFor((long long)n + 1, 128);
  switch (g.set) {
    case FDM_SET_PARTICLE:
      hipLaunchKernelGGL(kBroadCount<FDM_SET_PARTICLE>, dim3(nb), dim3(128), 0, stream, k);
      break;
    case FDM_SET_WALL:
      hipLaunchKernelGGL(kBroadCount<FDM_SET_WALL>, dim3(nb), dim3(128), 0, stream, k);
      break;
    case FDM_SET_GHOST:
      hipLaunchKernelGGL(kBroadCount<FDM_SET_GHOST>, dim3(nb), dim3(128), 0, stream, k);
      break;
    default:
      return FDM_EINVAL;
  }
  int r = scanInts(g.pairs.count, g.pairs.count, (size_t)n + 1, false, g.pairs.total, workspace,
                   workspaceBytes, stream, g.gate);
  if (r != FDM_OK) return r;
  return launchStatus();
}

// The write half needs the status word; it is launched by the narrow-phase
// entry's companion below so that the broad-phase signature stays the
// reference-like (count, scan) pair.
extern "C" int fdm_launchBroadPhaseWrite(const fdm_broadphase_args* args, unsigned* status,
                                         hipStream_t stream) {
  if (!args) return FDM_EINVAL;
  const fdm_broadphase_args& g = *args;
  const int n = g.particles.n;
  BroadK k;
  k.set = g.set;
  k.P = g.particles;
  k.pgeo = g.pgeo;
  k.W = g.walls;
  k.wgeo = g.wgeo;
  k.ghostCapacity = g.ghosts ? g.ghosts->capacity : 0;
  k.ghostCount = g.ghosts ? g.ghosts->count : nullptr;
  k.ghostReal = g.ghosts ? g.ghosts->realId : nullptr;
  k.ghostPos = g.ghosts ? g.ghosts->pos : nullptr;
  k.ghostBox = g.ghosts ? g.ghosts->cellBox : nullptr;
  k.grid = g.grid;
  k.table = g.table;
  k.pairs = g.pairs;
  k.status = status;
  k.skin = g.skin;
  k.maxReach = g.maxReach;
  k.gate = g.gate;
  k.inst = g.inst;
  k.periodic = g.periodic;
  if (n <= 0) return FDM_OK;
  const unsigned nb = blocksFor(n, 128);
  switch (g.set) {
    case FDM_SET_PARTICLE:
      hipLaunchKernelGGL(kBroadWrite<FDM_SET_PARTICLE>, dim3(nb), dim3(128), 0, stream, k);
      break;
    case FDM_SET_WALL:
      hipLaunchKernelGGL(kBroadWrite<FDM_SET_WALL>, dim3(nb), dim3(128), 0, stream, k);
      break;
    case FDM_SET_GHOST:
      hipLaunchKernelGGL(kBroadWrite<FDM_SET_GHOST>, dim3(nb), dim3(128), 0, stream, k);
      break;
    default:
      return FDM_EINVAL;
  }
  return launchStatus();
}

namespace {

void fillCommon(NarrowCommon& k, const fdm_narrowphase_args& g) {
  k.P = g.particles;
  k.pgeo = g.pgeo;
  k.pmat = g.pmat;
  k.W = g.walls;
  k.wgeo = g.wgeo;
  k.wmat = g.wmat;
  k.pgrid = g.pgrid;
  k.periodic = g.periodic;
  k.inst = g.inst;
  k.dt = g.dt;
  k.updateSprings = g.updateSprings;
  k.status = g.status;
  k.dbgPoint = g.dbgPoint;
  k.dbgNormal = g.dbgNormal;
  k.dbgOverlap = g.dbgOverlap;
}

void fillSet(NarrowSet& k, const fdm_narrowphase_args& g) {
  k.kind = g.set;
  k.ghostMask = g.ghostMask;
  k.ghostFromReal = g.ghostFromReal;
  k.ghostPos = g.ghosts ? g.ghosts->pos : nullptr;
  k.ghostHash = g.ghosts ? g.ghosts->table.hashValue : nullptr;
  k.ghostQ = g.set == FDM_SET_GHOST && g.periodic.sector && g.ghosts ? g.ghosts->q : nullptr;
  k.ghostVel = g.set == FDM_SET_GHOST && g.periodic.sector && g.ghosts ? g.ghosts->vel : nullptr;
  k.grid = g.grid;
  k.targetHash = g.targetHash;
  k.pairs = g.pairs;
  k.prev = g.prev;
  k.mirror = g.mirror;
}

bool validSet(const fdm_narrowphase_args& g) {
  if (g.set < FDM_SET_PARTICLE || g.set > FDM_SET_GHOST) return false;
  if (g.set == FDM_SET_GHOST) {
    if (g.ghostMask < 1 || g.ghostMask > 3) return false;
    if (!g.ghostFromReal && !g.ghosts) return false;
    // sector images carry their own orientation and velocity
    if (g.periodic.sector && (g.ghostFromReal || !g.ghosts->q || !g.ghosts->vel)) return false;
  }
  if (g.periodic.sector && (g.periodic.x || g.periodic.y || g.inst.count > 0)) return false;
  return true;
}

}  // namespace

extern "C" int fdm_launchNarrowPhase(const fdm_narrowphase_args* args, hipStream_t stream) {
  if (!args || !validSet(*args)) return FDM_EINVAL;
  const fdm_narrowphase_args& g = *args;
  NarrowK k;
  fillCommon(k.c, g);
  fillSet(k.s, g);
  hipLaunchKernelGGL(kResetCounter, dim3(1), dim3(64), 0, stream, g.pairs.recTotal);
  const int blocks = persistentBlocks(4);
  switch (g.set) {
    case FDM_SET_PARTICLE:
      hipLaunchKernelGGL(kNarrow<FDM_SET_PARTICLE>, dim3(blocks), dim3(256), 0, stream, k);
      break;
    case FDM_SET_WALL:
      hipLaunchKernelGGL(kNarrow<FDM_SET_WALL>, dim3(blocks), dim3(256), 0, stream, k);
      break;
    default:
      hipLaunchKernelGGL(kNarrow<FDM_SET_GHOST>, dim3(blocks), dim3(256), 0, stream, k);
      break;
  }
  return launchStatus();
}

extern "C" int fdm_launchNarrowPhaseSets(const fdm_narrowphase_args* sets, int nsets,
                                         const fdm_narrow_workspace* ws, hipStream_t stream) {
  if (!sets || nsets < 1 || nsets > kMaxSets || !ws || !ws->hitGeom ||
      !ws->hitCount || ws->hitCapacity < FDM_REC_POOLS)
    return FDM_EINVAL;
  NarrowMulti k;
  fillCommon(k.c, sets[0]);
  k.gate = sets[0].gate;
  k.nsets = nsets;
  long long cap = 0;
  for (int i = 0; i < nsets; ++i) {
    if (!validSet(sets[i])) return FDM_EINVAL;
    fillSet(k.s[i], sets[i]);
    cap += sets[i].pairs.capacity;
  }
  if (cap > ws->workCapacity || cap >= (1ll << 28)) return FDM_EINVAL;
  for (int i = nsets; i < kMaxSets; ++i) k.s[i] = k.s[0];
  const NarrowScratch x = {ws->hitGeom, ws->hitCapacity, ws->hitCount};
  fdm_tuning tu = tuning();
  if (ws->tuning && !completeTuning(*ws->tuning, tu)) return FDM_EINVAL;
  // geometry without the culling tables of sweepRun: the kernel that culls
  // by chunk
  const fdm_geometry& pg = sets[0].pgeo;
  if (!pg.groups || !pg.groupNodes || !pg.cells || (sets[0].wgeo.num > 0 && !sets[0].wgeo.cells)) tu.lawMode = 2;
  const int sweepBlocks = std::max(1, persistentBlocks(tu.sweepWaves) * tu.sweepWavesPerCU / 32);
  if (tu.lawMode == 2) {
    if (tu.sweepWaves == 4)
      hipLaunchKernelGGL(kCullSweepLaw<4>, dim3(sweepBlocks), dim3(256), 0, stream, k);
    else if (tu.sweepWaves == 2)
      hipLaunchKernelGGL(kCullSweepLaw<2>, dim3(sweepBlocks), dim3(128), 0, stream, k);
    else
      hipLaunchKernelGGL(kCullSweepLaw<1>, dim3(sweepBlocks), dim3(64), 0, stream, k);
    return launchStatus();
  }
  const int waves = std::max(kXcds, persistentBlocks(1) * tu.sweepWavesPerCU / 32 / kXcds * kXcds);
  if (sets[0].inst.count > 0) hipLaunchKernelGGL((kSweep<true, false>), dim3(waves), dim3(64), 0, stream, k, x);
  else if (sets[0].periodic.sector) hipLaunchKernelGGL((kSweep<false, true>), dim3(waves), dim3(64), 0, stream, k, x);
  else hipLaunchKernelGGL((kSweep<false, false>), dim3(waves), dim3(64), 0, stream, k, x);
  return launchStatus();
}

extern "C" int fdm_setTuning(const fdm_tuning* t) {
  if (!t) return FDM_EINVAL;
  fdm_tuning n;
  if (!completeTuning(*t, n)) return FDM_EINVAL;
  g_tuning = n;
  return FDM_OK;
}

extern "C" int fdm_checkTuning(fdm_tuning* t) {
  if (!t) return FDM_EINVAL;
  fdm_tuning n;
  if (!completeTuning(*t, n)) return FDM_EINVAL;
  *t = n;
  return FDM_OK;
}

extern "C" void fdm_getTuning(fdm_tuning* t) {
  if (t) *t = g_tuning;
}
