// Kernels that read or initialise the HBM state directly: initialise, masked
// reset, state snapshot and the contact/load queries of the reference batch
// (src/cuda/extension.cu:22-50, 128-159, 175-185).
#pragma once
#include "avbd_kernels.hpp"

namespace duckhip {

template <class R, int B, int J, int CG, int CS> struct StateView {
  using State = EnvState<R, B, J, CG, CS>;
  const DeviceModel<R> &M;
  State &s;
  DUCK_HD V3<R> X(int b) const { return {s.x[0][b], s.x[1][b], s.x[2][b]}; }
  DUCK_HD Q4<R> Q(int b) const { return {s.q[0][b], s.q[1][b], s.q[2][b], s.q[3][b]}; }
  DUCK_HD V3<R> W(int b) const { return {s.w[0][b], s.w[1][b], s.w[2][b]}; }
  DUCK_HD V3<R> mv(const R (&a)[3][kMaxModelJoints], int j) const { return {a[0][j], a[1][j], a[2][j]}; }
  DUCK_HD R angle(int j) const {
    return hingeAngle(Q(M.ja[j]), Q(M.jb[j]), mv(M.axisA, j), mv(M.tangentA, j), mv(M.tangentB, j));
  }
  // Copy of the model state (kernel.cuh:383-396).
  DUCK_HD void initialize() {
    for (int b = 0; b < M.nb; ++b) {
      for (int k = 0; k < 3; ++k) {
        s.x[k][b] = M.x[k][b];
        s.v[k][b] = M.v[k][b];
        s.w[k][b] = M.w[k][b];
        s.inertia[k][b] = M.inertia[k][b];
      }
      for (int k = 0; k < 4; ++k)
        s.q[k][b] = M.q[k][b];
      s.mass[b] = M.mass[b];
    }
    for (int k = 0; k < 3; ++k)
      s.force[k] = 0;
    for (int j = 0; j < M.nj; ++j) {
      for (int k = 0; k < 7; ++k) {
        s.lambda[k][j] = 0;
        s.penalty[k][j] = k < 3 ? R(1000) : R(1);
      }
      s.lambdaF[j] = 0;
      s.penaltyF[j] = 1;
      s.target[j] = M.target[j];
      s.kp[j] = M.kp[j];
      s.maxTorque[j] = M.maxTorque[j];
      s.torque[j] = M.torque[j];
      s.frictionloss[j] = M.frictionloss[j];
      s.damping[j] = M.damping[j];
    }
    for (int k = 0; k < 8; ++k)
      s.diag[k] = 0;
    s.friction = -1;
    s.colorCount = 2;
    for (int b = 0; b < B; ++b)
      s.colors[b] = b < M.nb ? M.colors[b] : 0;
    s.modelColours = 1;
    s.drive = kDriveOther;
    s.failed = 0;
    s.ngc = 0;
    s.nsc = 0;
  }
  // Fails an imported state whose contact lists cannot be the model's (a count
  // past the list's end, a body or shape that is not there), with its lists
  // empty: every launch walks the lists by their counts and indexes by their
  // ids, in the record and, in the dense step and the queries, in memory.
  DUCK_HD void checkContacts() {
    bool ok = s.ngc >= 0 && s.ngc <= CG && s.nsc >= 0 && s.nsc <= CS;
    for (int i = 0; ok && i < s.ngc; ++i)
      ok = gcBody(s.gc[i].id) < M.nb && gcShape(s.gc[i].id) < M.ns;
    for (int i = 0; ok && i < s.nsc; ++i)
      ok = scBody(s.sc[i].id) < M.nb && scOther(s.sc[i].id) < M.nb;
    if (!ok) {
      s.failed = 1;
      s.ngc = s.nsc = 0;
    }
  }
  // Clears the claims of `drive` and `modelColours` that the blob's bytes do
  // not bear out (an imported state); keeps every true one, so that an export
  // and import of the same batch's state is the identity.
  DUCK_HD void checkStamps() {
    bool ok = true;
    if (s.drive == kDriveTarget || s.drive == kDriveMotor) {
      const bool target = s.drive == kDriveTarget;
      for (int j = 0; j < J; ++j) {
        const bool in = j < M.nj;
        ok = ok && sameBits(s.kp[j], in && target ? s.driveKp : R(0)) &&
             sameBits(s.maxTorque[j], in && target ? s.driveLimit : R(0));
        if (target)
          ok = ok && sameBits(s.torque[j], in ? M.torque[j] : R(0)) &&
               sameBits(s.frictionloss[j], in ? M.frictionloss[j] : R(0)) &&
               sameBits(s.damping[j], in ? M.damping[j] : R(0));
      }
    } else {
      ok = s.drive == kDriveOther;
    }
    if (!ok)
      s.drive = kDriveOther;
    if (s.modelColours != 0) {
      bool same = s.modelColours == 1;
      for (int b = 0; b < B; ++b)
        same = same && s.colors[b] == (b < M.nb ? M.colors[b] : 0);
      if (!same)
        s.modelColours = 0;
    }
  }
};

template <class R, int B, int J, int CG, int CS>
__global__ void initializeKernel(const DeviceModel<R> *model, unsigned char *states,
                                 long long blobBytes, int count) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= count)
    return;
  StateView<R, B, J, CG, CS> v{*model, blobAt<EnvState<R, B, J, CG, CS>>(states, blobBytes, e)};
  v.initialize();
}

template <class R, int B, int J, int CG, int CS>
__global__ void checkImportKernel(const DeviceModel<R> *model, unsigned char *states,
                                  long long blobBytes, int count) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= count)
    return;
  StateView<R, B, J, CG, CS> v{*model, blobAt<EnvState<R, B, J, CG, CS>>(states, blobBytes, e)};
  v.checkContacts();
  v.checkStamps();
}

// The model state with the hinge angles `q` and the root offset `root` into
// the masked environments: StateView::initialize's fields, the root offset and
// forward kinematics down the hinges (kernel.cuh:383-420).  ext (optional, per
// env): [friction (<0 keeps the shape friction), mass scale, vx, vy, vz] --
// batch extensions with no reference counterpart.
//
// One wave takes 64 / B environments, lane b of an environment its body b and
// hinge b, so that the blob's component rows leave as whole rows; the poses
// stay in LDS for the kinematics, one tree level of hinges at a time (a hinge
// reads only its parent body, final after the level before; hinge order where
// the model has no levels), with the operations of a walk down the hinge list.
// Bound by the levels' dependent chains: a third of 12000 environments take
// 18.4 us.  One lane per environment (a cache line per lane and store, the
// kinematics one hinge after the other through global memory) took 104 us.
template <class R, int B, int J, int CG, int CS>
__global__ __launch_bounds__(64) void resetKernel(const DeviceModel<R> *model, unsigned char *states,
                                                  long long blobBytes, int count,
                                                  const unsigned char *mask, const R *q,
                                                  const R *root, const R *ext) {
  static_assert(J <= B && 64 % B == 0 && B >= 8, "a lane per body, hinge and diagnostic");
  constexpr int G = 64 / B;
  __shared__ R pose[G][7][B], given[G][16]; // given: root offset, then ext
  const int t = threadIdx.x, lane = t % B, g = t / B;
  const int e = blockIdx.x * G + g;
  bool run = e < count && mask[e] != 0;
  if (!__any(run))
    return;
  const DeviceModel<R> &M = *model;
  const int nb = M.nb, nj = M.nj;
  auto &s = blobAt<EnvState<R, B, J, CG, CS>>(states, blobBytes, run ? e : 0);
  const bool body = run && lane < nb, joint = run && lane < nj;
  // the caller's rows, one value per lane; a value that is not finite fails
  // the environment, whose state stays as it is
  const R angle = joint ? q[size_t(e) * nj + lane] : R(0);
  const R offset = run && lane < 6 ? root[size_t(e) * 6 + lane] : R(0);
  const R extra = run && ext && lane < 5 ? ext[size_t(e) * 5 + lane] : R(0);
  const uint64_t group = (B == 64 ? ~uint64_t(0) : (uint64_t(1) << (B & 63)) - 1) << (g * B);
  const bool bad = (__ballot(!mfinite(angle) || !mfinite(offset) || !mfinite(extra)) & group) != 0;
  if (run && bad) {
    if (lane == 0)
      s.failed = 1;
    run = false;
  }
  if (lane < 8) {
    given[g][lane] = offset;
    given[g][8 + lane] = extra;
  }
  const R *row = given[g], *scale = given[g] + 8;
  // the hinge's frames, read ahead of the kinematics
  const int jc = lane < nj ? lane : 0, ja = M.ja[jc], jb = M.jb[jc];
  const V3<R> axisA{M.axisA[0][jc], M.axisA[1][jc], M.axisA[2][jc]};
  const V3<R> ra{M.ra[0][jc], M.ra[1][jc], M.ra[2][jc]}, rb{M.rb[0][jc], M.rb[1][jc], M.rb[2][jc]};
  const Q4<R> oa{M.q[0][ja], M.q[1][ja], M.q[2][ja], M.q[3][ja]};
  const Q4<R> ob{M.q[0][jb], M.q[1][jb], M.q[2][jb], M.q[3][jb]};
  const R turn = angle - M.originalAngle[jc];
  const int levels = M.jointLevels, turns = levels > 0 ? levels : nj;
  const int mine = !(run && joint) ? -1 : (levels > 0 ? M.jointLevel[jc] - 1 : lane);
  if (run && body) {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pose[g][k][lane] = M.x[k][lane];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      pose[g][3 + k][lane] = M.q[k][lane];
  }
  __syncthreads();
  // turn -1 is the root offset of body 1, by lane 1
  for (int level = -1; level < turns; ++level) {
    const bool rootTurn = level < 0 && run && lane == 1;
    if (rootTurn || (level >= 0 && mine == level)) {
      const R(&p)[7][B] = pose[g];
      const int from = rootTurn ? 1 : ja, to = rootTurn ? 1 : jb;
      const V3<R> xa{p[0][from], p[1][from], p[2][from]};
      const Q4<R> qa{p[3][from], p[4][from], p[5][from], p[6][from]};
      const V3<R> by = rootTurn ? V3<R>{row[3], row[4], row[5]} : rotate(qa, axisA) * turn;
      Q4<R> r = expmap(by) * qa;
      V3<R> x = xa + V3<R>{row[0], row[1], row[2]};
      if (!rootTurn) {
        r = normalized((r * conj(oa)) * ob);
        x = (xa + rotate(qa, ra)) - rotate(r, rb);
      }
      const R v[7] = {x.x, x.y, x.z, r.w, r.x, r.y, r.z};
#pragma unroll
      for (int k = 0; k < 7; ++k)
        pose[g][k][to] = v[k];
    }
    __syncthreads();
  }
  if (!run)
    return;
  if (body) {
    const R mass = M.mass[lane];
    const bool scaled = ext && mass > 0;
    s.mass[lane] = scaled ? mass * scale[1] : mass;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const R inertia = M.inertia[k][lane];
      s.inertia[k][lane] = scaled ? inertia * scale[1] : inertia;
      s.x[k][lane] = pose[g][k][lane];
      s.v[k][lane] = scaled ? scale[2 + k] : R(0);
      s.w[k][lane] = 0;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      s.q[k][lane] = pose[g][3 + k][lane];
  }
  if (joint) {
#pragma unroll
    for (int k = 0; k < 7; ++k) {
      s.lambda[k][lane] = 0;
      s.penalty[k][lane] = k < 3 ? R(1000) : R(1);
    }
    s.lambdaF[lane] = 0;
    s.penaltyF[lane] = 1;
    s.target[lane] = M.target[lane];
    s.kp[lane] = M.kp[lane];
    s.maxTorque[lane] = M.maxTorque[lane];
    s.torque[lane] = M.torque[lane];
    s.frictionloss[lane] = M.frictionloss[lane];
    s.damping[lane] = M.damping[lane];
  }
  s.colors[lane] = lane < nb ? M.colors[lane] : 0;
  if (lane < 8)
    s.diag[lane] = 0;
  if (lane < 3)
    s.force[lane] = 0;
  if (lane == 0) {
    s.friction = ext ? scale[0] : R(-1);
    s.colorCount = 2;
    s.modelColours = 1;
    s.drive = kDriveOther;
    s.failed = 0;
    s.ngc = 0;
    s.nsc = 0;
  }
}

// Rows of `n` consecutive environments from LDS to global memory, whole waves
// at a time (dword or 8-byte stores of 64 consecutive words, so no alignment
// beyond the word's is assumed).
template <class T>
__device__ __forceinline__ void copyRows(T *dst, const T *src, int n, int t) {
  for (int i = t; i < n; i += 64)
    dst[i] = src[i];
}

// bodies [E,B,13], joints [E,J,2], diag [E,6] (kernel.cuh:555-575).  One
// wave takes 64 / B environments, lane b of an environment its body b and
// hinge b: the blob's component rows are read by consecutive lanes, the
// output rows are formed in LDS and leave as one contiguous run.  Bound by
// launch and one memory round trip: 4.4 us at 4096 environments, 7.9 us at
// 16384.  One lane per environment (64 waves at 4096, every load and store a
// cache line per lane) took 28.6 and 33.4 us.
template <class R, int B, int J, int CG, int CS>
__global__ __launch_bounds__(64) void snapshotKernel(const DeviceModel<R> *model, unsigned char *states,
                                                     long long blobBytes, int count, R *bodies,
                                                     R *joints, R *diag) {
  static_assert(J <= B && 64 % B == 0 && B >= 6, "a lane per body, hinge and diagnostic");
  constexpr int G = 64 / B;
  __shared__ R rows[G * B * 13], angles[G * J * 2], diags[G * 6];
  const DeviceModel<R> &M = *model;
  const int t = threadIdx.x, lane = t % B, g = t / B;
  const int e0 = blockIdx.x * G, e = e0 + g, n = count - e0 < G ? count - e0 : G;
  const int nb = M.nb, nj = M.nj;
  const bool joint = e < count && lane < nj;
  const int jc = lane < nj ? lane : 0;
  const int ja = M.ja[jc], jb = M.jb[jc];
  const V3<R> axisA{M.axisA[0][jc], M.axisA[1][jc], M.axisA[2][jc]};
  const V3<R> tangentA{M.tangentA[0][jc], M.tangentA[1][jc], M.tangentA[2][jc]};
  const V3<R> tangentB{M.tangentB[0][jc], M.tangentB[1][jc], M.tangentB[2][jc]};
  if (e < count) {
    const auto &s = blobAt<EnvState<R, B, J, CG, CS>>(states, blobBytes, e);
    if (lane < nb) {
      const R row[13] = {s.x[0][lane], s.x[1][lane], s.x[2][lane], s.q[0][lane], s.q[1][lane],
                         s.q[2][lane], s.q[3][lane], s.v[0][lane], s.v[1][lane], s.v[2][lane],
                         s.w[0][lane], s.w[1][lane], s.w[2][lane]};
#pragma unroll
      for (int k = 0; k < 13; ++k)
        rows[(g * nb + lane) * 13 + k] = row[k];
    }
    constexpr int slot[5] = {kJointError, kPenetration, kContacts, kConverged, kAxisError};
#pragma unroll
    for (int k = 0; k < 5; ++k)
      if (lane == k)
        diags[g * 6 + k] = s.diag[slot[k]];
    if (lane == 5)
      diags[g * 6 + 5] = R(s.failed);
  }
  __syncthreads();
  if (joint) {
    const R *a = rows + (g * nb + ja) * 13, *b = rows + (g * nb + jb) * 13;
    const Q4<R> qa{a[3], a[4], a[5], a[6]}, qb{b[3], b[4], b[5], b[6]};
    const V3<R> wa{a[10], a[11], a[12]}, wb{b[10], b[11], b[12]};
    angles[(g * nj + lane) * 2] = hingeAngle(qa, qb, axisA, tangentA, tangentB);
    angles[(g * nj + lane) * 2 + 1] = dot(wb - wa, rotate(qa, axisA));
  }
  __syncthreads();
  copyRows(bodies + size_t(e0) * nb * 13, rows, n * nb * 13, t);
  copyRows(joints + size_t(e0) * nj * 2, angles, n * nj * 2, t);
  copyRows(diag + size_t(e0) * 6, diags, n * 6, t);
}

template <class R> DUCK_HD V3<R> selfForceWorld(const SelfContact<R> &c) {
  return ((V3<R>{c.t1[0], c.t1[1], c.t1[2]} * c.lambda[0]) +
          (V3<R>{c.t2[0], c.t2[1], c.t2[2]} * c.lambda[1])) +
         (V3<R>{c.n[0], c.n[1], c.n[2]} * c.lambda[2]);
}

// [E,B,3] contact force on each body (kernel.cuh:467-480).
template <class R, int B, int J, int CG, int CS>
__global__ void contactForcesKernel(const DeviceModel<R> *model, unsigned char *states,
                                    long long blobBytes, int count, int groundOnly, R *out) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= count)
    return;
  const DeviceModel<R> &M = *model;
  auto &s = blobAt<EnvState<R, B, J, CG, CS>>(states, blobBytes, e);
  R *o = out + size_t(e) * M.nb * 3;
  for (int i = 0; i < M.nb * 3; ++i)
    o[i] = 0;
  for (int i = 0; i < s.ngc; ++i) {
    const auto &c = s.gc[i];
    // contactWorld with the fixed basis, negated.
    V3<R> f = -((V3<R>{1, 0, 0} * c.lambda[0] + V3<R>{0, 1, 0} * c.lambda[1]) +
                V3<R>{0, 0, 1} * c.lambda[2]);
    int b = gcBody(c.id);
    o[b * 3] += f.x;
    o[b * 3 + 1] += f.y;
    o[b * 3 + 2] += f.z;
  }
  if (groundOnly)
    return;
  for (int i = 0; i < s.nsc; ++i) {
    const auto &c = s.sc[i];
    V3<R> f = -selfForceWorld(c);
    int a = scBody(c.id), b = scOther(c.id);
    o[a * 3] += f.x;
    o[a * 3 + 1] += f.y;
    o[a * 3 + 2] += f.z;
    o[b * 3] -= f.x;
    o[b * 3 + 1] -= f.y;
    o[b * 3 + 2] -= f.z;
  }
}

// [E,2] active body-body contacts and maximum depth (kernel.cuh:481-493).
template <class R, int B, int J, int CG, int CS>
__global__ void selfContactStatsKernel(const DeviceModel<R> *model, unsigned char *states,
                                       long long blobBytes, int count, R *out) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= count)
    return;
  const DeviceModel<R> &M = *model;
  auto &s = blobAt<EnvState<R, B, J, CG, CS>>(states, blobBytes, e);
  StateView<R, B, J, CG, CS> v{M, s};
  R n = 0, depthMax = 0;
  for (int i = 0; i < s.nsc; ++i) {
    const auto &c = s.sc[i];
    int a = scBody(c.id), b = scOther(c.id);
    V3<R> ra = rotate(v.Q(a), V3<R>{c.local[0], c.local[1], c.local[2]});
    V3<R> rb = rotate(v.Q(b), V3<R>{c.localB[0], c.localB[1], c.localB[2]});
    V3<R> delta = ((v.X(a) + ra) - v.X(b)) - rb;
    R cz = dot(delta, V3<R>{c.n[0], c.n[1], c.n[2]}) - M.alpha * c.c0;
    R depth = mx(R(0), -(cz + M.alpha * c.c0));
    if (c.lambda[2] < R(-1e-5) || depth > R(1e-6))
      n += 1;
    depthMax = mx(depthMax, depth);
  }
  out[2 * e] = n;
  out[2 * e + 1] = depthMax;
}

template <class R, int B, int J, int CG, int CS>
__global__ void contactCountsKernel(unsigned char *states, long long blobBytes, int count, R *out) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= count)
    return;
  auto &s = blobAt<EnvState<R, B, J, CG, CS>>(states, blobBytes, e);
  out[2 * e] = R(s.ngc);
  out[2 * e + 1] = R(s.nsc);
}

// The per-body quantities of the Newton-Euler pass.
template <class R, int B> struct RneaWork {
  V3<R> acc[B], alpha[B], force[B], moment[B], contact[B], contactMoment[B];
};

// Recursive Newton-Euler at zero joint acceleration (kernel.cuh:504-554):
// per hinge [bias, contact/limit, applied actuator torque] into o[3 j + k];
// `off` is the root COM offset of the acceleration reference point.  `work`
// holds the per-body quantities (private memory, or a caller's LDS scratch).
template <class R, int B, int J, int CG, int CS>
DUCK_HD void rneaLoadsIn(const DeviceModel<R> &M, const EnvState<R, B, J, CG, CS> &s, const R *off,
                         R *o, RneaWork<R, B> &work) {
  StateView<R, B, J, CG, CS> v{M, const_cast<EnvState<R, B, J, CG, CS> &>(s)};
  V3<R> *acc = work.acc, *alpha = work.alpha, *force = work.force, *moment = work.moment,
        *contact = work.contact, *contactMoment = work.contactMoment;
  for (int b = 0; b < M.nb; ++b)
    acc[b] = alpha[b] = force[b] = moment[b] = contact[b] = contactMoment[b] = V3<R>{0, 0, 0};
  acc[1] = cross(v.W(1), cross(v.W(1), rotate(v.Q(1), V3<R>{off[0], off[1], off[2]})));
  for (int j = 0; j < M.nj; ++j) {
    const int a = M.ja[j], b = M.jb[j];
    Q4<R> qa = v.Q(a), qb = v.Q(b);
    V3<R> axis = rotate(qa, v.mv(M.axisA, j)), ra = rotate(qa, v.mv(M.ra, j)),
          rb = rotate(qb, v.mv(M.rb, j));
    V3<R> wa = v.W(a), wb = v.W(b);
    R speed = dot(wb - wa, axis);
    alpha[b] = alpha[a] + cross(wa, axis) * speed;
    acc[b] = (((acc[a] + cross(alpha[a], ra)) + cross(wa, cross(wa, ra))) - cross(alpha[b], rb)) -
             cross(wb, cross(wb, rb));
  }
  for (int b = 1; b < M.nb; ++b) {
    Q4<R> q = v.Q(b);
    V3<R> I{s.inertia[0][b], s.inertia[1][b], s.inertia[2][b]}, w = v.W(b);
    auto inertia = [&](V3<R> u) {
      V3<R> l = rotate(conj(q), u);
      l.x *= I.x;
      l.y *= I.y;
      l.z *= I.z;
      return rotate(q, l);
    };
    force[b] = (acc[b] - V3<R>{M.gravity[0], M.gravity[1], M.gravity[2]}) * s.mass[b];
    moment[b] = inertia(alpha[b]) + cross(w, inertia(w));
  }
  for (int i = 0; i < s.ngc; ++i) {
    const auto &c = s.gc[i];
    V3<R> f = -((V3<R>{1, 0, 0} * c.lambda[0] + V3<R>{0, 1, 0} * c.lambda[1]) +
                V3<R>{0, 0, 1} * c.lambda[2]);
    int b = gcBody(c.id);
    contact[b] = contact[b] + f;
    contactMoment[b] =
        contactMoment[b] + cross(rotate(v.Q(b), V3<R>{c.local[0], c.local[1], c.local[2]}), f);
  }
  for (int i = 0; i < s.nsc; ++i) {
    const auto &c = s.sc[i];
    V3<R> f = -selfForceWorld(c);
    int a = scBody(c.id), b = scOther(c.id);
    contact[a] = contact[a] + f;
    contactMoment[a] =
        contactMoment[a] + cross(rotate(v.Q(a), V3<R>{c.local[0], c.local[1], c.local[2]}), f);
    contact[b] = contact[b] + (-f);
    contactMoment[b] = contactMoment[b] +
                       cross(rotate(v.Q(b), V3<R>{c.localB[0], c.localB[1], c.localB[2]}), -f);
  }
  for (int k = M.nj - 1; k >= 0; --k) {
    const int a = M.ja[k], b = M.jb[k];
    Q4<R> qa = v.Q(a), qb = v.Q(b);
    V3<R> axis = rotate(qa, v.mv(M.axisA, k)), rb = rotate(qb, v.mv(M.rb, k)),
          shift = v.X(b) - v.X(a);
    o[3 * k] = dot(axis, moment[b] - cross(rb, force[b]));
    o[3 * k + 1] = dot(axis, contactMoment[b] - cross(rb, contact[b])) +
                   (M.limited[k] ? -s.lambda[5][k] + s.lambda[6][k] : R(0));
    R motor = s.torque[k] - s.kp[k] * wrapAngle(v.angle(k) - s.target[k]);
    o[3 * k + 2] = s.maxTorque[k] > 0 ? clampv(motor, -s.maxTorque[k], s.maxTorque[k]) : motor;
    moment[a] = moment[a] + (moment[b] + cross(shift, force[b]));
    force[a] = force[a] + force[b];
    contactMoment[a] = contactMoment[a] + (contactMoment[b] + cross(shift, contact[b]));
    contact[a] = contact[a] + contact[b];
  }
}
template <class R, int B, int J, int CG, int CS>
DUCK_HD void rneaLoads(const DeviceModel<R> &M, const EnvState<R, B, J, CG, CS> &s, const R *off,
                       R *o) {
  RneaWork<R, B> work;
  rneaLoadsIn<R, B, J, CG, CS>(M, s, off, o, work);
}

// rneaLoadsIn split over an environment's L lanes, for a model whose hinges
// form a tree listed parent first (M.jointLevels > 0): the outward pass one
// tree level at a time (a hinge reads only its parent body, final after the
// level before), the per-body forces and the contact sums one body per lane
// (a body's contacts in list order, ground then body contacts), the inward
// pass from the deepest level: each hinge of the level writes its loads, then
// each parent adds its children's terms in decreasing hinge order.  Every
// quantity is formed by the operations of rneaLoadsIn in its order, so the
// loads are bitwise those of the sequential pass.  Every lane of the
// workgroup calls it (barriers); `valid` lanes work.  The hinges' frames are
// read once, ahead of the levels, and `jb` is the caller's LDS copy of the
// hinges' child bodies: a level then waits for LDS, not for the model in
// global memory (the fused servo substep 110.7 -> 108.4 us).  Drive: with the
// actuator column.
template <class R, int B, int J, int CG, int CS, int L, bool Drive = true>
__device__ __forceinline__ void rneaLoadsLanes(const DeviceModel<R> &M,
                                               const EnvState<R, B, J, CG, CS> &s, const R *off,
                                               R *o, RneaWork<R, B> &work, const int *jb, int lane,
                                               bool valid) {
  constexpr int BPL = (B + L - 1) / L, JPL = (J + L - 1) / L;
  StateView<R, B, J, CG, CS> v{M, const_cast<EnvState<R, B, J, CG, CS> &>(s)};
  V3<R> *acc = work.acc, *alpha = work.alpha, *force = work.force, *moment = work.moment,
        *contact = work.contact, *contactMoment = work.contactMoment;
  const int nb = M.nb, nj = M.nj, levels = M.jointLevels;
  // the lane's hinges and bodies: level, ends, child hinges (read once); a
  // hinge's world axis and child arm, formed in the outward pass, serve the
  // inward pass too (the poses do not move in between); its actuator column
  // needs no tree quantity and is written first
  int jLevel[JPL], jA[JPL], jB[JPL], bLevel[BPL];
  unsigned children[BPL];
  V3<R> jAxis[JPL], jRb[JPL], axisOf[JPL], raOf[JPL], rbOf[JPL];
  int limitedOf[JPL];
#pragma unroll
  for (int r = 0; r < JPL; ++r) {
    const int j = lane + r * L;
    const bool in = valid && j < nj;
    const int jc = in ? j : 0;
    axisOf[r] = v.mv(M.axisA, jc);
    raOf[r] = v.mv(M.ra, jc);
    rbOf[r] = v.mv(M.rb, jc);
    limitedOf[r] = M.limited[jc];
    jLevel[r] = in ? M.jointLevel[j] : -1;
    jA[r] = in ? M.ja[j] : 0;
    jB[r] = in ? M.jb[j] : 0;
    jAxis[r] = jRb[r] = V3<R>{0, 0, 0};
    if (Drive && in) {
      R motor = s.torque[j] - s.kp[j] * wrapAngle(v.angle(j) - s.target[j]);
      o[3 * j + 2] = s.maxTorque[j] > 0 ? clampv(motor, -s.maxTorque[j], s.maxTorque[j]) : motor;
    }
  }
#pragma unroll
  for (int r = 0; r < BPL; ++r) {
    const int b = lane + r * L;
    const bool in = valid && b < nb;
    bLevel[r] = in ? M.bodyLevel[b] : -1;
    children[r] = in ? M.childHinges[b] : 0u;
    if (in)
      acc[b] = alpha[b] = force[b] = moment[b] = contact[b] = contactMoment[b] = V3<R>{0, 0, 0};
  }
  __syncthreads();
  if (valid && lane == 0)
    acc[1] = cross(v.W(1), cross(v.W(1), rotate(v.Q(1), V3<R>{off[0], off[1], off[2]})));
  __syncthreads();
  for (int level = 1; level <= levels; ++level) {
#pragma unroll
    for (int r = 0; r < JPL; ++r) {
      const int j = lane + r * L;
      if (jLevel[r] != level)
        continue;
      const int a = jA[r], b = jB[r];
      Q4<R> qa = v.Q(a), qb = v.Q(b);
      V3<R> axis = rotate(qa, axisOf[r]), ra = rotate(qa, raOf[r]), rb = rotate(qb, rbOf[r]);
      V3<R> wa = v.W(a), wb = v.W(b);
      R speed = dot(wb - wa, axis);
      alpha[b] = alpha[a] + cross(wa, axis) * speed;
      acc[b] = (((acc[a] + cross(alpha[a], ra)) + cross(wa, cross(wa, ra))) - cross(alpha[b], rb)) -
               cross(wb, cross(wb, rb));
      jAxis[r] = axis;
      jRb[r] = rb;
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < BPL; ++r) {
    const int b = lane + r * L;
    if (!valid || b < 1 || b >= nb)
      continue;
    Q4<R> q = v.Q(b);
    V3<R> I{s.inertia[0][b], s.inertia[1][b], s.inertia[2][b]}, w = v.W(b);
    auto inertia = [&](V3<R> u) {
      V3<R> l = rotate(conj(q), u);
      l.x *= I.x;
      l.y *= I.y;
      l.z *= I.z;
      return rotate(q, l);
    };
    force[b] = (acc[b] - V3<R>{M.gravity[0], M.gravity[1], M.gravity[2]}) * s.mass[b];
    moment[b] = inertia(alpha[b]) + cross(w, inertia(w));
    V3<R> sum{0, 0, 0}, sumMoment{0, 0, 0};
    for (int i = 0; i < s.ngc; ++i) {
      const auto &c = s.gc[i];
      if (gcBody(c.id) != b)
        continue;
      V3<R> f = -((V3<R>{1, 0, 0} * c.lambda[0] + V3<R>{0, 1, 0} * c.lambda[1]) +
                  V3<R>{0, 0, 1} * c.lambda[2]);
      sum = sum + f;
      sumMoment = sumMoment + cross(rotate(q, V3<R>{c.local[0], c.local[1], c.local[2]}), f);
    }
    for (int i = 0; i < s.nsc; ++i) {
      const auto &c = s.sc[i];
      const int ca = scBody(c.id), cb = scOther(c.id);
      if (ca != b && cb != b)
        continue;
      V3<R> f = -selfForceWorld(c);
      if (ca == b) {
        sum = sum + f;
        sumMoment = sumMoment + cross(rotate(q, V3<R>{c.local[0], c.local[1], c.local[2]}), f);
      }
      if (cb == b) {
        sum = sum + (-f);
        sumMoment = sumMoment + cross(rotate(q, V3<R>{c.localB[0], c.localB[1], c.localB[2]}), -f);
      }
    }
    contact[b] = sum;
    contactMoment[b] = sumMoment;
  }
  __syncthreads();
  for (int level = levels; level >= 1; --level) {
#pragma unroll
    for (int r = 0; r < JPL; ++r) {
      const int k = lane + r * L;
      if (jLevel[r] != level)
        continue;
      const int b = jB[r];
      const V3<R> axis = jAxis[r], rb = jRb[r];
      o[3 * k] = dot(axis, moment[b] - cross(rb, force[b]));
      o[3 * k + 1] = dot(axis, contactMoment[b] - cross(rb, contact[b])) +
                     (limitedOf[r] ? -s.lambda[5][k] + s.lambda[6][k] : R(0));
    }
    if (level == 1)
      break; // the roots' sums feed no hinge
#pragma unroll
    for (int r = 0; r < BPL; ++r) {
      const int p = lane + r * L;
      if (bLevel[r] != level - 1)
        continue;
      // the body's child hinges in decreasing order, as the sequential pass
      for (unsigned m = children[r]; m; m &= ~(1u << (31 - __builtin_clz(m)))) {
        const int k = 31 - __builtin_clz(m);
        const int b = jb[k];
        V3<R> shift = v.X(b) - v.X(p);
        moment[p] = moment[p] + (moment[b] + cross(shift, force[b]));
        force[p] = force[p] + force[b];
        contactMoment[p] = contactMoment[p] + (contactMoment[b] + cross(shift, contact[b]));
        contact[p] = contact[p] + contact[b];
      }
    }
    __syncthreads();
  }
}

// One environment of the load query in LDS: the state as the step stages it,
// and the pass's per-body quantities.
template <class R, int B, int J, int CG, int CS> struct LoadsEnv {
  EnvState<R, B, J, CG, CS> s;
  RneaWork<R, B> work;
  R offset[3];
};

// [E,J,3] loads.  A wave takes 64 / B environments with B lanes each, as the
// fused servo substep does: the blobs staged in LDS, the pass one tree level
// at a time (rneaLoadsLanes; in hinge order on the first lane where the hinges
// are no such tree), the rows out as one contiguous run.  Bound by the levels'
// dependent chains: 13.1 us at 3001 environments.  One lane per environment,
// walking the tree through global memory, took 61 us.
template <class R, int B, int J, int CG, int CS>
__global__ __launch_bounds__(64) void generalizedLoadsKernel(const DeviceModel<R> *model,
                                                             unsigned char *states, long long blobBytes,
                                                             int count, const R *offset, R *out) {
  static_assert(J <= B && 64 % B == 0, "a lane per body and hinge");
  using State = EnvState<R, B, J, CG, CS>;
  constexpr int G = 64 / B;
  __shared__ alignas(16) LoadsEnv<R, B, J, CG, CS> envs[G];
  __shared__ R loads[G * J * 3];
  __shared__ int jb[J];
  const DeviceModel<R> &M = *model;
  const int t = threadIdx.x, lane = t % B, g = t / B;
  const int e0 = blockIdx.x * G, e = e0 + g, n = count - e0 < G ? count - e0 : G;
  const bool valid = e < count;
  const int nj = M.nj;
  auto &E = envs[g];
  loadHot<State, G>(envs, states, blobBytes, e0, count - e0, t, true);
  if (t < nj)
    jb[t] = M.jb[t];
  if (valid) {
    if (lane < 3)
      E.offset[lane] = offset[size_t(e) * 3 + lane];
    loadEnv<State>(E.s, &blobAt<State>(states, blobBytes, e), lane, B, true, false);
  }
  // every load of this wave, those straight into LDS included, has landed
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  R *o = loads + g * nj * 3;
  if (M.jointLevels > 0)
    rneaLoadsLanes<R, B, J, CG, CS, B>(M, E.s, E.offset, o, E.work, jb, lane, valid);
  else if (valid && lane == 0)
    rneaLoadsIn<R, B, J, CG, CS>(M, E.s, E.offset, o, E.work);
  __syncthreads();
  copyRows(out + size_t(e0) * nj * 3, loads, n * nj * 3, t);
}

} // namespace duckhip
