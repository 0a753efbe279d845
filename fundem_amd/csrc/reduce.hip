// Bond forces (VBond) and the deterministic force/torque reduction.
//
// The reference adds every contact and bond contribution with double
// atomicAdds (contactKernel.cu:120-123,203-204,284-290,367-370), so its sums
// depend on scheduling. Here each particle folds its records serially in a
// fixed order: particle pairs by partner (pairs where it is the target, then
// pairs it owns), wall pairs by wall, ghost sets X, Y, XY by partner real id
// (owned before mirrored on a tie), bonds by bond id. Each record is a
// per-pair sum that the narrow phase accumulated in node order. The second
// half-kick follows in the same thread.
#include <algorithm>

#include "fdm_device.hpp"
#include "fdm_launch.hpp"
#include "step_device.hpp"

namespace fdm {

// VBond (contactKernel.cuh:138-199); returns the new bonded flag.
__device__ __forceinline__ int vbond(V3& F, V3& Mij, V3& Mji, double& sig, double& tau, V3 rbi,
                                     V3 rbj, V3 n1i, V3 n2i, V3 n3i, V3 n1j, V3 n2j, V3 n3j,
                                     double B1, double B2, double B3, double B4, double R, double D0,
                                     double st, double coh, double mub) {
  const V3 rbij = vsub(rbi, rbj);
  const double D = vlen(rbij);
  if (nearZero(D)) return 1;
  const V3 nij = vnormalize(rbij);
  const V3 e = vneg(nij);
  const V3 dn1 = vsub(n1j, n1i);
  F = vadd(vmul(e, B1 * (D - D0)), vmul(vsub(dn1, vmul(e, vdot(dn1, e))), B2 / (2 * D)));
  const V3 MTB =
      vsub(vmul(vcross(n1j, n1i), B3), vmul(vadd(vcross(n2j, n2i), vcross(n3j, n3i)), 0.5 * B4));
  Mij = vadd(vmul(vcross(e, n1i), -0.5 * B2), MTB);
  Mji = vsub(vmul(vcross(e, n1j), 0.5 * B2), MTB);
  const double Fn = vdot(F, nij);
  const V3 Fs = vsub(F, vmul(nij, Fn));
  const double Tt = vdot(MTB, nij);
  const V3 Tb = vsub(MTB, vmul(nij, Tt));
  const double A = R * R * kPi;
  const double I = A * R * R / 4.;
  const double J = 2 * I;
  sig = -Fn / A + vlen(Tb) / I * R;
  tau = vlen(Fs) / A + fabs(Tt) / J * R;
  if (st > 0. && sig > st) return 0;
  else if (coh > 0. && tau > coh - mub * sig) return 0;
  return 1;
}

// addBondedForceTorqueKernel (contactKernel.cu:293-371), results per bond.
__global__ void kBonds(fdm_bodies P, fdm_bonds b) {
  if (gateOff(b.gate)) return;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= b.n) return;
  if (b.active[k] == 0) {
    b.applied[k] = 0;
    b.maxNormalStress[k] = 0.;
    b.maxShearStress[k] = 0.;
    return;
  }
  const int n = P.n;
  const int i = b.master[k], j = b.slave[k];
  const Q4 qi = ld4(P.q, n, i), qj = ld4(P.q, n, j);
  const fdm_real* L = b.local + 24 * (size_t)k;
  auto lv = [&](int o) { return V3{(double)L[o], (double)L[o + 1], (double)L[o + 2]}; };
  const V3 n1i = qrotate(qi, lv(0)), n2i = qrotate(qi, lv(3)), n3i = qrotate(qi, lv(6));
  const V3 n1j = qrotate(qj, lv(12)), n2j = qrotate(qj, lv(15)), n3j = qrotate(qj, lv(18));
  const V3 ri = ldp(P.x, n, i), rj = ldp(P.x, n, j);
  const V3 rbi = vadd(qrotate(qi, lv(9)), ri), rbj = vadd(qrotate(qj, lv(21)), rj);
  const fdm_real* c = b.coef + 9 * (size_t)k;
  V3 F = {0., 0., 0.}, Mij = {0., 0., 0.}, Mji = {0., 0., 0.};
  double sig = b.maxNormalStress[k], tau = b.maxShearStress[k];
  const int on = vbond(F, Mij, Mji, sig, tau, rbi, rbj, n1i, n2i, n3i, n1j, n2j, n3j, c[0], c[1],
                       c[2], c[3], c[4], c[5], c[6], c[7], c[8]);
  b.active[k] = on;
  if (!on) b.breakStep[k] = b.stepIndex ? *b.stepIndex : 0;
  b.maxNormalStress[k] = sig;
  b.maxShearStress[k] = tau;
  b.applied[k] = 1;
  const V3 Ti = vadd(Mij, vcross(vsub(rbi, ri), F));
  const V3 Tj = vadd(Mji, vcross(vsub(rbj, rj), vneg(F)));
  double* of = b.outF + 3 * (size_t)k;
  double* oi = b.outTi + 3 * (size_t)k;
  double* oj = b.outTj + 3 * (size_t)k;
  of[0] = F.x; of[1] = F.y; of[2] = F.z;
  oi[0] = Ti.x; oi[1] = Ti.y; oi[2] = Ti.z;
  oj[0] = Tj.x; oj[1] = Tj.y; oj[2] = Tj.z;
}

__global__ void kReduce(ReduceK a) {
  if (gateOff(a.gate)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = a.P.n;
  if (i == 0 && a.stepCounter) *a.stepCounter += 1;  // read by the bond stage before this launch
  if (i >= n) return;
  V3 F, T;
  foldForces(a, i, F, T);
  st3(a.P.F, n, i, F);
  st3(a.P.T, n, i, T);
  if (!a.kick) return;
  // integration2ndHalf: the kick of particleIntegrationKernel.cu:3-32 with the
  // stored (FP32) force and torque
  const fdm_template& t = a.pgeo.info[a.P.geo[i]];
  const double invM = t.invMass;
  if (nearZero(invM)) return;
  const V3 Fs = roundState(F), Ts = roundState(T);
  const V3 v = ld3(a.P.v, n, i);
  st3(a.P.v, n, i, vadd(v, vmul(vadd(vmul(Fs, invM), a.gravity), a.h)));
  if (spinFixed(t)) return;
  const V3 w = ld3(a.P.w, n, i);
  const Q4 q = ld4(a.P.q, n, i);
  const V3 Iw = smul(srotate(q, lds6(t.inertia)), w);
  st3(a.P.w, n, i, vadd(w, vmul(smul(srotate(q, lds6(t.invInertia)), vsub(Ts, vcross(w, Iw))), a.h)));
}

}  // namespace fdm

using namespace fdm;

extern "C" int fdm_launchBondForces(fdm_bodies particles, fdm_bonds bonds, hipStream_t stream) {
  if (bonds.n < 0) return FDM_EINVAL;
  if (bonds.n == 0) return FDM_OK;
  hipLaunchKernelGGL(kBonds, dim3(blocksFor(bonds.n, 256)), dim3(256), 0, stream, particles, bonds);
  return launchStatus();
}

namespace fdm {
// Which sets each particle has candidate pairs in: as A from the lists'
// counts, as target (mirrored sets) from the pairs.
struct TouchK {
  int n, haveBonds;
  const int* bondStart;
  const int* count[5];  // NULL: no such set
  const int* total[5];
  const int* pairT[5];
  int capacity[5];
};
__global__ void kTouchOwn(TouchK k, int* touch) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= k.n) return;
  int t = 0;
#pragma unroll
  for (int s = 0; s < 5; ++s)
    if (k.count[s] && k.count[s][i + 1] > k.count[s][i]) t |= FDM_TOUCH_A(s);
  if (k.haveBonds && k.bondStart[i + 1] > k.bondStart[i]) t |= FDM_TOUCH_BOND;
  touch[i] = t;
}
__global__ void kTouchTargets(TouchK k, int* touch) {
  const int s = blockIdx.y;
  if (s == 1 || !k.count[s]) return;  // walls are not mirrored
  const int total = min(*k.total[s], k.capacity[s]);
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < total; p += gridDim.x * blockDim.x) {
    const int t = k.pairT[s][p];
    if (t >= 0 && t < k.n) atomicOr(&touch[t], FDM_TOUCH_T(s));
  }
}
}  // namespace fdm

extern "C" int fdm_launchTouch(const fdm_pairs* const sets[5], const fdm_bonds* bonds, int n, int* touch,
                               hipStream_t stream) {
  if (!sets || n < 0 || (n > 0 && !touch)) return FDM_EINVAL;
  if (n == 0) return FDM_OK;
  TouchK k{};
  k.n = n;
  k.haveBonds = bonds && bonds->n > 0;
  k.bondStart = k.haveBonds ? bonds->partStart : nullptr;
  for (int s = 0; s < 5; ++s)
    if (sets[s]) {
      k.count[s] = sets[s]->count;
      k.total[s] = sets[s]->total;
      k.pairT[s] = sets[s]->pairT;
      k.capacity[s] = sets[s]->capacity;
    }
  hipLaunchKernelGGL(kTouchOwn, dim3(blocksFor(n, 256)), dim3(256), 0, stream, k, touch);
  hipLaunchKernelGGL(kTouchTargets, dim3(std::min<unsigned>(blocksFor(n, 256), 256), 5), dim3(256), 0, stream,
                     k, touch);
  return launchStatus();
}

__global__ void kIncrement(int* c) {
  if (threadIdx.x == 0) *c += 1;
}

extern "C" int fdm_incrementCounter(int* counter, hipStream_t stream) {
  if (!counter) return FDM_EINVAL;
  hipLaunchKernelGGL(kIncrement, dim3(1), dim3(64), 0, stream, counter);
  return launchStatus();
}

int fdm::fillReduce(const fdm_reduce_args& g, ReduceK& k) {
  if (!g.pp || !g.ppMirror) return FDM_EINVAL;
  k = ReduceK{};
  k.P = g.particles;
  k.pgeo = g.pgeo;
  k.pp = *g.pp;
  k.ppm = *g.ppMirror;
  k.havePW = g.pw != nullptr;
  if (g.pw) k.pw = *g.pw;
  for (int s = 0; s < 3; ++s) {
    k.haveG[s] = g.ghost[s] != nullptr && g.ghostMirror[s] != nullptr;
    if (k.haveG[s]) {
      k.g[s] = *g.ghost[s];
      k.gm[s] = *g.ghostMirror[s];
    }
  }
  k.haveBonds = g.bonds != nullptr && g.bonds->n > 0;
  if (k.haveBonds) k.bonds = *g.bonds;
  k.gravity = fromD3(g.gravity);
  k.h = g.h;
  k.kick = g.kick;
  k.stepCounter = g.stepCounter;
  k.gate = g.gate;
  k.touch = g.touch;
  return FDM_OK;
}

extern "C" int fdm_launchReduceForceTorque(const fdm_reduce_args* args, hipStream_t stream) {
  if (!args) return FDM_EINVAL;
  const fdm_reduce_args& g = *args;
  ReduceK k;
  if (fillReduce(g, k) != FDM_OK) return FDM_EINVAL;
  if (g.particles.n <= 0) {
    if (g.stepCounter) hipLaunchKernelGGL(kIncrement, dim3(1), dim3(64), 0, stream, g.stepCounter);
    return launchStatus();
  }
  fdm_tuning tu = tuning();
  if (g.tuning) {
    tu = *g.tuning;
    if (fdm_checkTuning(&tu) != FDM_OK) return FDM_EINVAL;
  }
  const int rb = tu.reduceBlock;
  hipLaunchKernelGGL(kReduce, dim3(blocksFor(g.particles.n, rb)), dim3(rb), 0, stream, k);
  return launchStatus();
}
