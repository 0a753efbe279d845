// Device code of a step's per-body stages, shared by the kernels of
// integrate.hip and reduce.hip: the fold of a body's forces, the first half of
// a step (half-kick, drift, cell id, change flags) and the list decision.
#pragma once
#include "fdm_device.hpp"
#include "fdm_launch.hpp"

namespace fdm {

struct ReduceK {
  fdm_bodies P;
  fdm_geometry pgeo;
  fdm_pairs pp, pw, g[3];
  fdm_mirror ppm, gm[3];
  int havePW, haveG[3];
  fdm_bonds bonds;
  int haveBonds;
  V3 gravity;
  double h;
  int kick;
  int* stepCounter;
  const int* gate;
  const int* touch;
};

__device__ __forceinline__ void addRec(V3& F, V3& T, const double* f, const double* t, bool negF) {
  const V3 fv = {f[0], f[1], f[2]};
  F = vadd(F, negF ? vneg(fv) : fv);
  T = vadd(T, {t[0], t[1], t[2]});
}

// Smallest mirror entry greater than `last` (mirror lists are short and
// unordered; selection keeps the fold order independent of append order).
__device__ __forceinline__ int nextMirror(const int* list, int m, int last) {
  int best = INT_MAX;
  for (int t = 0; t < m; ++t) {
    const int v = list[t];
    if (v > last && v < best) best = v;
  }
  return best;
}

// The kernel's view of the launcher's arguments (reduce.hip).
int fillReduce(const fdm_reduce_args& g, ReduceK& k);

// Sums of up to two records, loaded together; rows of three are added in turn.
struct TwoRecs {
  double f[2][3], t[2][3];
};
__device__ __forceinline__ void loadRec(TwoRecs& r, int k, const double* f, const double* t) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    r.f[k][c] = f[c];
    r.t[k][c] = t[c];
  }
}
// Owned pairs [b, e) of a set.
__device__ __forceinline__ void addOwned(V3& F, V3& T, const fdm_pairs& s, int b, int e) {
  for (int p = b; p < e; p += 2) {
    const int q = p + 1, n0 = s.recCnt[p];
    int n1 = 0;
    TwoRecs r;
    loadRec(r, 0, s.sumF + 3 * (size_t)p, s.sumTA + 3 * (size_t)p);
    if (q < e) {
      n1 = s.recCnt[q];
      loadRec(r, 1, s.sumF + 3 * (size_t)q, s.sumTA + 3 * (size_t)q);
    }
    if (n0 > 0) addRec(F, T, r.f[0], r.t[0], false);
    if (n1 > 0) addRec(F, T, r.f[1], r.t[1], false);
  }
}

// Force and torque of particle i: its records in the canonical order (the
// header of reduce.hip). Bodies without candidate pairs or bonds are told by
// one word (touch) instead of the counts of every set. For the others this is
// a chain of dependent loads, so they are taken in rounds: the counts of all
// sets; a short mirror list as a whole; records by two, also of pairs without
// contacts, whose sums are then not added. Measured
// in kReduceStep: 216 particles 16.3 -> 14.4 us, 8192 spheres of up to twelve
// bonds 25.5 -> 20.0 us; one particle 10.3 -> 10.6 us.
__device__ __forceinline__ void foldForces(const ReduceK& a, int i, V3& F, V3& T) {
  F = {0., 0., 0.};
  T = {0., 0., 0.};
  const int touch = a.touch ? a.touch[i] : ~0;
  if (!touch) return;
  int m = 0, p0 = 0, p1 = 0, w0 = 0, w1 = 0, b0 = 0, b1 = 0;
  int gm[3] = {0, 0, 0}, g0[3] = {0, 0, 0}, g1[3] = {0, 0, 0};
  if (touch & (FDM_TOUCH_A(0) | FDM_TOUCH_T(0))) {
    m = a.ppm.count[i];
    p0 = a.pp.count[i];
    p1 = a.pp.count[i + 1];
  }
  if (a.havePW && (touch & FDM_TOUCH_A(1))) {
    w0 = a.pw.count[i];
    w1 = a.pw.count[i + 1];
  }
#pragma unroll
  for (int s = 0; s < 3; ++s)
    if (a.haveG[s] && (touch & (FDM_TOUCH_A(2 + s) | FDM_TOUCH_T(2 + s)))) {
      gm[s] = a.gm[s].count[i];
      g0[s] = a.g[s].count[i];
      g1[s] = a.g[s].count[i + 1];
    }
  if (a.haveBonds && (touch & FDM_TOUCH_BOND)) {
    b0 = a.bonds.partStart[i];
    b1 = a.bonds.partStart[i + 1];
  }
  // particle pairs: as target (partners below i), then owned (partners above)
  if (m > 0) {
    a.ppm.count[i] = 0;
    m = min(m, a.ppm.capacity);
    const int* list = a.ppm.list + (size_t)i * a.ppm.capacity;
    if (m <= 4) {
      int l[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) l[r] = r < m ? list[r] : INT_MAX;
      auto order = [](int& x, int& y) __attribute__((always_inline)) {
        const int lo = min(x, y);
        y = max(x, y);
        x = lo;
      };
      order(l[0], l[1]);
      order(l[2], l[3]);
      order(l[0], l[2]);
      order(l[1], l[3]);
      order(l[1], l[2]);
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        if (r >= m) break;
        const bool two = r + 1 < m;
        const int p = l[r], q = two ? l[r + 1] : p;
        TwoRecs x;
        loadRec(x, 0, a.pp.sumF + 3 * (size_t)p, a.pp.sumTB + 3 * (size_t)p);
        loadRec(x, 1, a.pp.sumF + 3 * (size_t)q, a.pp.sumTB + 3 * (size_t)q);
        addRec(F, T, x.f[0], x.t[0], true);
        if (two) addRec(F, T, x.f[1], x.t[1], true);
      }
    } else {
      int last = -1;
      for (int r = 0; r < m; ++r) {
        const int p = nextMirror(list, m, last);
        last = p;
        addRec(F, T, a.pp.sumF + 3 * (size_t)p, a.pp.sumTB + 3 * (size_t)p, true);
      }
    }
  }
  addOwned(F, T, a.pp, min(p0, a.pp.capacity), min(p1, a.pp.capacity));
  if (a.havePW) addOwned(F, T, a.pw, min(w0, a.pw.capacity), min(w1, a.pw.capacity));
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    const fdm_pairs& G = a.g[s];
    const fdm_mirror& M = a.gm[s];
    const int mm = min(gm[s], M.capacity);
    int own = min(g0[s], G.capacity);
    const int ownEnd = min(g1[s], G.capacity);
    if (mm <= 0 && own >= ownEnd) continue;
    const int* list = M.list + (size_t)i * M.capacity;
    int mp = mm > 0 ? nextMirror(list, mm, -1) : INT_MAX;
    int used = 0;
    while (true) {
      while (own < ownEnd && G.recCnt[own] == 0) ++own;
      const bool haveOwn = own < ownEnd;
      const bool haveMir = used < mm;
      if (!haveOwn && !haveMir) break;
      const int partnerOwn = haveOwn ? G.pairT[own] : INT_MAX;
      const int partnerMir = haveMir ? G.pairA[mp] : INT_MAX;
      if (haveOwn && partnerOwn <= partnerMir) {
        addRec(F, T, G.sumF + 3 * (size_t)own, G.sumTA + 3 * (size_t)own, false);
        ++own;
      } else {
        addRec(F, T, G.sumF + 3 * (size_t)mp, G.sumTB + 3 * (size_t)mp, true);
        ++used;
        mp = used < mm ? nextMirror(list, mm, mp) : INT_MAX;
      }
    }
    if (mm > 0) M.count[i] = 0;
  }
  if (b0 < b1) {
    const fdm_bonds& b = a.bonds;
    int n0 = b.partList[b0], n1 = b.partList[min(b0 + 1, b1 - 1)];
    for (int e = b0; e < b1; e += 2) {
      const bool two = e + 1 < b1;
      const int c0 = n0, c1 = n1;
      n0 = b.partList[min(e + 2, b1 - 1)];  // (the next bonds, a round ahead)
      n1 = b.partList[min(e + 3, b1 - 1)];
      const int k0 = c0 >> 1, k1 = c1 >> 1;
      const int on0 = b.applied[k0], on1 = b.applied[k1];
      TwoRecs x;
      loadRec(x, 0, b.outF + 3 * (size_t)k0, ((c0 & 1) ? b.outTj : b.outTi) + 3 * (size_t)k0);
      loadRec(x, 1, b.outF + 3 * (size_t)k1, ((c1 & 1) ? b.outTj : b.outTi) + 3 * (size_t)k1);
      if (on0) addRec(F, T, x.f[0], x.t[0], c0 & 1);
      if (two && on1) addRec(F, T, x.f[1], x.t[1], c1 & 1);
    }
  }
}

// Rebuild decision of one step (one thread). The displacement bound grows by
// dt times the largest motion rate, plus 1e-6 rho per step for the rounding
// of orientations to FP32 (a relative 2^-24 per component moves a point at
// distance rho by well under 1e-6 rho). Ghost lists are also rebuilt after
// a visibility change or a wrap; a wrap (positions jump by a period)
// rebuilds the next step's lists as well. One thread of one workgroup runs
// it, after every other writer of the control words has finished (earlier
// kernels of the stream); `rate` and `flags` (bit 0 grid state changed, 1
// visibility changed, 2 wrapped) add this kernel's own findings. The control
// words are read together (plain loads: the cache is fresh at kernel start),
// and the host's copy of the decision is one word, (number << 2) | rebuild
// << 1 | ghost rebuild, so it needs no ordering fence.
__device__ __forceinline__ void decideStep(const fdm_skin& s, float rateIn, int flagsIn) {
  int* c = s.ctl;
  int w[FDM_CTL_WORDS];
#pragma unroll
  for (int k = 0; k < FDM_CTL_WORDS; ++k) w[k] = c[k];
  const double disp = *s.disp;
  const float rate = fmaxf(__int_as_float(w[FDM_CTL_MAX_RATE]), rateIn);
  double d = disp + s.dt * (double)rate * (1.0 + 1e-6) + 1e-6 * s.rhoMax;
  const bool rebuild = w[FDM_CTL_FORCE] != 0 || w[FDM_CTL_PENDING] != 0 ||
                       w[FDM_CTL_VALID_CHANGED] != 0 || (flagsIn & 1) || !(2.0 * d <= s.skin);
  const bool wrapped = w[FDM_CTL_WRAPPED] != 0 || (flagsIn & 4);
  const bool ghost = rebuild || wrapped || w[FDM_CTL_GHOST_CHANGED] != 0 || (flagsIn & 2);
  if (rebuild) {
    d = 0.0;
    c[FDM_CTL_COUNT] = w[FDM_CTL_COUNT] + 1;
  }
  if (ghost) c[FDM_CTL_GHOST_COUNT] = w[FDM_CTL_GHOST_COUNT] + 1;
  *s.disp = d;
  c[FDM_CTL_REBUILD] = rebuild ? 1 : 0;
  c[FDM_CTL_REBUILD_GHOST] = ghost ? 1 : 0;
  c[FDM_CTL_KEEP] = (rebuild || ghost) ? 0 : 1;
  c[FDM_CTL_PENDING] = wrapped ? 1 : 0;
  c[FDM_CTL_MAX_RATE] = 0;
  c[FDM_CTL_FORCE] = 0;
  c[FDM_CTL_VALID_CHANGED] = 0;
  c[FDM_CTL_WRAPPED] = 0;
  c[FDM_CTL_GHOST_CHANGED] = 0;
  const int seq = w[FDM_CTL_SEQ] + 1;
  c[FDM_CTL_SEQ] = seq;
  if (s.hostDecision)
    *(volatile int*)(s.hostDecision + (seq & (FDM_DECISION_RING - 1))) =
        (int)(((unsigned)seq << 2) | (rebuild ? 2u : 0u) | (ghost ? 1u : 0u));
}

struct StepBeginK {
  fdm_step_begin_args a;
  fdm_skin s;
  float* blockRate;  // [gridDim.x] largest motion rate of each workgroup
  int* blockFlags;   // [gridDim.x] bit 0 grid state changed, 1 visibility changed, 2 wrapped
};

// One body of phase A of a step (particles, then walls). Everything it reads from the launch arguments is
// copied into registers first (selecting between argument structs by
// reference would make the compiler copy them to per-lane scratch).
// MANY: bodies of several systems (per-body grids and periodic flags); the
// single-system kernel holds its grid in scalar registers.
// REDUCED: the body's force and torque (Fr, Tr, as they would be stored) come
// from the fold of the step before, whose second half-kick is still due.
template <bool WALL, bool MANY, bool REDUCED = false>
__device__ __forceinline__ void stepBeginBody(const fdm_step_begin_args& a, int j, float& rate,
                                              int& flags, R3 Fr = {0, 0, 0}, R3 Tr = {0, 0, 0}) {
  const fdm_bodies b = WALL ? a.walls : a.particles;
  const fdm_template* tmpl = WALL ? a.wgeo.info : a.pgeo.info;
  const fdm_hash_table t = WALL ? a.wtable : a.ptable;
  const bool many = MANY;
  const int in = !many ? 0 : (WALL ? a.inst.wallInstance[j] : a.inst.particleInstance[j]);
  const fdm_grid grid =
      !many ? (WALL ? a.wgrid : a.pgrid) : (WALL ? a.inst.wgrid[in] : a.inst.pgrid[in]);
  const fdm_periodic perI = many ? a.inst.periodic[in] : a.periodic;
  const bool ghosts = !WALL && anyPeriodic(a.periodic);
  const bool kick = !WALL && a.kick;
  const int n = b.n;
  // Every input is loaded before anything is stored: the arrays may alias as
  // far as the compiler knows, so a load placed after a store could not be
  // issued before it. One round of loads (the torque only where the spin
  // changes), then the half-kick and the drift in registers with the
  // roundings of the stored state (kickOne, driftOne), then the stores.
  // (the stored FP32 values are held as loaded and widened where used)
  const int geo = b.geo[j];
  const V3 x0 = ldp(b.x, n, j);
  R3 v = ld3s(b.v, n, j), w = ld3s(b.w, n, j);
  const R4 q0 = ld4s(b.q, n, j);
  R3 F = Fr;
  if (kick && !REDUCED) F = ld3s(b.F, n, j);
  const int atBuild = t.validAtBuild[j];
  const int ghostAtBuild = ghosts ? a.ghostAtBuild[j] : 0;
  const fdm_template& tp = tmpl[geo];
  bool vNew = false, wNew = false;
  if (kick && !nearZero(tp.invMass)) {
    // particleVelocityAngularVelocityIntegrationKernel (particleIntegrationKernel.cu:3-32)
    const double h = 0.5 * a.dt;
    const V3 dv = vmul(vadd(vmul(wide(F), tp.invMass), fromD3(a.gravity)), h);
    if (REDUCED) v = narrow3(vadd(wide(v), dv));
    v = narrow3(vadd(wide(v), dv));
    vNew = true;
    if (!spinFixed(tp)) {
      const Q4 qd = wide(q0);
      const S6 I = srotate(qd, lds6(tp.inertia)), Ii = srotate(qd, lds6(tp.invInertia));
      const V3 T = REDUCED ? wide(Tr) : ld3(b.T, n, j);
#pragma unroll
      for (int k = REDUCED ? 0 : 1; k < 2; ++k) {
        const V3 wd = wide(w);
        w = narrow3(vadd(wd, vmul(smul(Ii, vsub(T, vcross(wd, smul(I, wd)))), h)));
      }
      wNew = true;
    }
  }
  V3 x = x0;
  if (vNew) st3s(b.v, n, j, v);
  if (wNew) st3s(b.w, n, j, w);
  if (a.drift) {
    // particlePositionOrientationIntegrationKernel (particleIntegrationKernel.cu:34-48)
    x = vadd(x0, vmul(wide(v), a.dt));
    stp(b.x, n, j, x);
    st4(b.q, n, j, qintegrate(wide(q0), wide(w), a.dt));
  }
  t.hashValue[j] = cellHash(x, grid);
  if (a.drift) {
    const double rho = fmax(tp.radius, tp.boxReach);
    const double r = vlen(wide(v)) + vlen(wide(w)) * rho;
    rate = (float)r * (1.0f + 1e-6f);
  }
  const int st = bodyState(x, grid);
  if (st == 2 || st != atBuild) flags |= 1;
  if (ghosts) {
    // sets exist where any instance is periodic; an instance contributes
    // only to the sets of its own periodic axes
    const int vb = visibilityBits(x, grid, a.periodic, perI);
    const int bits = vb & 7;
    for (int k = 0; k < 3; ++k)
      if (a.ghostFlag[k]) a.ghostFlag[k][j] = (bits >> k) & 1;
    if (bits != ghostAtBuild) flags |= 2;
    if (vb & 8) flags |= 4;
  }
}

// Largest motion rate and change flags of a workgroup (256 threads), on
// thread 0.
__device__ __forceinline__ void foldBlock(float& rate, int& flags) {
  __shared__ float waveMax[4];
  const int f1 = __syncthreads_or(flags & 1), f2 = __syncthreads_or(flags & 2),
            f4 = __syncthreads_or(flags & 4);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) rate = fmaxf(rate, __shfl_xor(rate, off, 64));
  if (laneId() == 0) waveMax[threadIdx.x >> 6] = rate;
  __syncthreads();
  rate = waveMax[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); ++w) rate = fmaxf(rate, waveMax[w]);
  flags = (f1 ? 1 : 0) | (f2 ? 2 : 0) | (f4 ? 4 : 0);
}

// The step's list decision by the last workgroup to arrive, without a kernel
// of its own: each workgroup folds its rate and flags into one of 64 slots
// (a cache line each) and then counts itself there, the last of a slot counts
// the slot. Only the slots' own words need ordering, so the atomics are
// relaxed, the count issued once the folds have returned (a release would
// write back the caches of eight XCDs for the body state, which only later
// kernels read). The last workgroup reads the slots, zeroes them for the next
// step, clears the counters and decides. A single workgroup decides at once.
constexpr int kFoldSlots = 64;
__device__ __forceinline__ void decideLast(const StepBeginK& k, float rate, int flags) {
  __shared__ int last;
  const int nb = gridDim.x;
  foldBlock(rate, flags);
  rate = fmaxf(rate, 0.f);  // (no number, if no body has one: as an int it would exceed every rate)
  int* fold = k.s.fold;
  const int slots = nb <= kFoldSlots ? 1 : kFoldSlots;
  if (nb > 1) {
    if (threadIdx.x == 0) {
      const int g = blockIdx.x % slots;
      const int size = nb / slots + (g < nb % slots ? 1 : 0);
      int* slot = fold + 16 * g;
      const int r0 = atomicMax(slot, __float_as_int(rate));
      const int f0 = flags ? atomicOr(slot + 1, flags) : 0;
      asm volatile("s_waitcnt vmcnt(0)" ::"v"(r0), "v"(f0) : "memory");
      int done = atomicAdd(slot + 2, 1) == size - 1 ? 1 : 0;
      if (done && slots > 1) done = atomicAdd(fold + 16 * kFoldSlots, 1) == slots - 1 ? 1 : 0;
      last = done;
    }
    __syncthreads();
    if (!last) return;
    rate = 0.f;
    flags = 0;
    if (threadIdx.x < 64) {
      if ((int)threadIdx.x < slots) {
        int* slot = fold + 16 * threadIdx.x;
        rate = __int_as_float(__hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        flags = __hip_atomic_load(slot + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int c = 0; c < 3; ++c)
          __hip_atomic_store(slot + c, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        rate = fmaxf(rate, __shfl_xor(rate, off, 64));
        flags |= __shfl_xor(flags, off, 64);
      }
      if (threadIdx.x == 0)
        __hip_atomic_store(fold + 16 * kFoldSlots, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  for (int q = 0; q < 8; ++q)
    if (k.a.clearCounters[q])
      for (int i = threadIdx.x; i < FDM_REC_COUNTERS; i += blockDim.x) k.a.clearCounters[q][i] = 0;
  if (threadIdx.x == 0) decideStep(k.s, rate, flags);
}

}  // namespace fdm
