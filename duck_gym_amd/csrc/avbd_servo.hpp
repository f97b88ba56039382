// Servo substep of the BAM-actuated environment (python/duck_gym/bam_env.py:
// 307-326 with the XL330/m6 equations of python/duck_gym/actuator.py:16-77):
// the delayed-target ring buffer, the external hinge load from a zero-
// acceleration Newton-Euler pass, and the motor model, producing the
// (torque, dry-friction budget, damping) channels the next implicit step
// consumes.  One lane per environment: the supply voltage couples the joints
// of an environment through sum |previous torque|.
#pragma once
#include "../../include/duck_hip.h"
#include "avbd_queries.hpp"

namespace duckhip {

DUCK_HD float mpow(float x, float y) { return powf(x, y); }
DUCK_HD double mpow(double x, double y) { return pow(x, y); }
DUCK_HD float mexpf(float x) { return expf(x); }
DUCK_HD double mexpf(double x) { return exp(x); }

// actuator.py:44-77 for one joint.  Scalar parameters are combined in the
// order torch evaluates them: a Python float meeting a tensor is rounded to
// the tensor dtype; products of Python floats are formed in double first.
template <class R>
DUCK_HD void xl330(const DuckServo &p, R supply, R target, R position, R velocity, R previousApplied,
                   R external, R &applied, R &budget, R &damping, R &raw) {
  R speed = velocity * R(p.kd_scale);
  const double errorGain = (4096 / (2 * 3.14159265358979323846)) / (256 * 885);
  R duty = (((target - position) * R(p.kp_fw)) * R(p.kp_scale)) * R(errorGain);
  R center = (R(p.kt) * speed) / supply;
  R span = R(p.resistance * 1.75) / supply;
  R lo = center - span, hi = center + span;
  duty = duty < lo ? lo : duty; // torch.clamp(min=lo, max=hi): min(max(x, lo), hi)
  duty = duty > hi ? hi : duty;
  duty = duty < R(-1) ? R(-1) : (duty > R(1) ? R(1) : duty);
  raw = ((R(p.kt) * supply) * duty) / R(p.resistance) - (R(p.kt * p.kt) * speed) / R(p.resistance);
  R stribeck = mexpf(-mpow(mabs(velocity) / R(p.dtheta_stribeck), R(p.alpha)));
  R mot = previousApplied, ext = external;
  R quad = mabs(mot) > mabs(ext) ? R(p.load_friction_external_quad) * (ext * ext)
                                 : R(p.load_friction_motor_quad) * (mot * mot);
  budget = ((((R(p.friction_base) + stribeck * R(p.friction_stribeck)) +
              mabs(ext * R(p.load_friction_external) - mot * R(p.load_friction_motor))) +
             stribeck * mabs(ext * R(p.load_friction_external_stribeck) -
                             mot * R(p.load_friction_motor_stribeck))) +
            stribeck * quad) *
           R(p.friction_scale);
  R limit = R(p.force_limit);
  applied = raw < -limit ? -limit : (raw > limit ? limit : raw);
  damping = R(p.friction_viscous);
}

struct ServoBuffers {
  const void *target;          // [E,J] commanded target of this control step
  void *history;               // [lag+1, E, J] ring buffer of targets
  int cursor;                  // slot written this substep
  unsigned char *initialized;  // [E] ring buffer filled since the last reset
  const void *rootOffset;      // [E,3] root COM offset for the load pass
  void *previousMotor;         // [E,J] raw motor torque of the last substep (in/out)
  void *previousApplied;       // [E,J] clamped torque of the last substep (in/out)
  void *motor;                 // [E,J,3] out
  void *supply;                // [E] out, may be null
};

template <class R, int B, int J, int CG, int CS>
__global__ void servoKernel(DuckServo p, const DeviceModel<R> *model, unsigned char *states,
                            long long blobBytes, int count, ServoBuffers io) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= count)
    return;
  const DeviceModel<R> &M = *model;
  const auto &s = blobAt<EnvState<R, B, J, CG, CS>>(states, blobBytes, e);
  StateView<R, B, J, CG, CS> view{M, const_cast<EnvState<R, B, J, CG, CS> &>(s)};
  const int nj = M.nj, slots = p.lag + 1;
  const size_t row = size_t(e) * nj, plane = size_t(count) * nj;
  const R *target = static_cast<const R *>(io.target) + row;
  R *history = static_cast<R *>(io.history);
  // bam_env.py:308-314: write this substep's target, fill a fresh ring, read
  // the target `lag` substeps old.
  for (int j = 0; j < nj; ++j)
    history[size_t(io.cursor) * plane + row + j] = target[j];
  if (!io.initialized[e]) {
    for (int k = 0; k < slots; ++k)
      for (int j = 0; j < nj; ++j)
        history[size_t(k) * plane + row + j] = target[j];
    io.initialized[e] = 1;
  }
  const int delayedSlot = ((io.cursor - p.lag) % slots + slots) % slots;
  const R *delayed = history + size_t(delayedSlot) * plane + row;

  R loads[J][3];
  rneaLoads<R, B, J, CG, CS>(M, s, static_cast<const R *>(io.rootOffset) + size_t(e) * 3,
                             &loads[0][0]);
  R *prevMotor = static_cast<R *>(io.previousMotor) + row;
  R *prevApplied = static_cast<R *>(io.previousApplied) + row;
  R total = 0;
  for (int j = 0; j < nj; ++j)
    total += mabs(prevMotor[j]);
  R supply = R(p.vin) - R(p.vin_drop_gain) * total;
  supply = supply < R(p.vin_min) ? R(p.vin_min) : supply;
  R *motor = static_cast<R *>(io.motor) + row * 3;
  for (int j = 0; j < nj; ++j) {
    R position = view.angle(j);
    R velocity = dot(view.W(M.jb[j]) - view.W(M.ja[j]), rotate(view.Q(M.ja[j]), view.mv(M.axisA, j)));
    R external = -loads[j][0] + loads[j][1];
    R applied, budget, damping, raw;
    xl330(p, supply, delayed[j], position, velocity, prevApplied[j], external, applied, budget,
          damping, raw);
    motor[3 * j] = applied;
    motor[3 * j + 1] = budget;
    motor[3 * j + 2] = damping;
    prevMotor[j] = raw;
    prevApplied[j] = applied;
  }
  if (io.supply)
    static_cast<R *>(io.supply)[e] = supply;
}

// The servo substep inside the step launch (servoStepKernel): the operations
// of servoKernel on the state the launch staged in LDS, before the motor
// step.  Lanes take hinges; the environment's lanes run the load pass one
// tree level at a time (rneaLoadsLanes; for a model whose hinges are no tree
// listed parent first, the first lane runs it in hinge order), with its
// per-body quantities in the step's per-step scratch, which the step fills
// later; every lane sums the supply in servoKernel's order.  The channels
// go into `ctl`, where the motor step takes them.  A lane group that repeats
// another's environment (`own` false) forms the same channels and stores
// nothing: what it reads (loadServo) is read before the same wave's lanes
// write it.
template <class R, int B, int J, int CG, int CS, int L, int JPL, class Env>
__device__ __forceinline__ void servoPrologue(const ServoArgs<R> &sv, const DeviceModel<R> &M,
                                              const Frames<R, B, J> &F, Env &E, int e, int lane,
                                              bool own, int count, int sub, ServoIn<R, JPL> &in,
                                              R (&ctl)[JPL][3]) {
  static_assert(sizeof(RneaWork<R, B>) <= sizeof(R) * 20 * B, "the load pass fits x0 .. Iw");
  static_assert(4 * J + 3 <= 7 * J, "loads, previous torques and root offset fit c0");
  const int nj = M.nj, slots = sv.p.lag + 1;
  const size_t row = size_t(e) * nj, plane = size_t(count) * nj;
  R *loads = &E.c0[0][0], *previous = loads + 3 * J, *offset = loads + 4 * J;
  R delayed[JPL];
  // bam_env.py:308-314: this substep's target into the ring (every slot
  // of a fresh ring), the target `lag` substeps old out.  Slots that this
  // launch has written hold its target and are not read back, so no lane
  // reads what another writes.
  const int cursor = (sv.cursor + sub) % slots;
  const bool now = in.fresh || sub >= sv.p.lag;
#pragma unroll
  for (int r = 0; r < JPL; ++r) {
    const int j = lane + r * L;
    delayed[r] = in.target[r];
    if (j >= nj)
      continue;
    if (!now)
      delayed[r] = sub == 0 ? in.history[r] : sv.history[size_t((cursor + 1) % slots) * plane + row + j];
    previous[j] = mabs(in.motor[r]);
    if (own) {
      sv.history[size_t(cursor) * plane + row + j] = in.target[r];
      if (in.fresh && sub == 0)
        for (int k = 0; k < slots; ++k)
          sv.history[size_t(k) * plane + row + j] = in.target[r];
    }
  }
  if (lane < 3)
    offset[lane] = in.offset;
  if (own && lane == 0)
    sv.initialized[e] = 1;
  auto &work = *reinterpret_cast<RneaWork<R, B> *>(&E.x0[0][0]);
  if (M.jointLevels > 0) {
    rneaLoadsLanes<R, B, J, CG, CS, L, false>(M, E.s, offset, loads, work, F.b, lane, true);
  } else {
    __syncthreads();
    if (lane == 0)
      rneaLoadsIn<R, B, J, CG, CS>(M, E.s, offset, loads, work);
  }
  __syncthreads();
  R total = 0;
  for (int j = 0; j < nj; ++j)
    total += previous[j];
  R supply = R(sv.p.vin) - R(sv.p.vin_drop_gain) * total;
  supply = supply < R(sv.p.vin_min) ? R(sv.p.vin_min) : supply;
  if (own && lane == 0 && sv.supply)
    sv.supply[e] = supply;
  StateView<R, B, J, CG, CS> view{M, E.s};
  auto frame = [](const auto &a, int j) { return V3<R>{a[0][j], a[1][j], a[2][j]}; };
#pragma unroll
  for (int r = 0; r < JPL; ++r) {
    const int j = lane + r * L;
    if (j >= nj)
      continue;
    const int a = F.a[j], b = F.b[j];
    const Q4<R> qa = view.Q(a), qb = view.Q(b);
    const V3<R> axisA = frame(F.axisA, j);
    R position = hingeAngle(qa, qb, axisA, frame(F.tangentA, j), frame(F.tangentB, j));
    R velocity = dot(view.W(b) - view.W(a), rotate(qa, axisA));
    R external = -loads[3 * j] + loads[3 * j + 1];
    R applied, budget, damping, raw;
    xl330(sv.p, supply, delayed[r], position, velocity, in.applied[r], external, applied, budget,
          damping, raw);
    if (own) {
      if (sv.motor) {
        sv.motor[(row + j) * 3] = applied;
        sv.motor[(row + j) * 3 + 1] = budget;
        sv.motor[(row + j) * 3 + 2] = damping;
      }
      sv.previousMotor[row + j] = raw;
      sv.previousApplied[row + j] = applied;
    }
    in.motor[r] = raw;
    in.applied[r] = applied;
    ctl[r][0] = applied;
    ctl[r][1] = budget;
    ctl[r][2] = damping;
  }
  __syncthreads(); // the load pass's scratch is the step's
}

// torch.maximum: NaN when either operand is NaN.
template <class R> DUCK_HD R maximumNan(R a, R b) { return a != a || b != b ? R(NAN) : (a > b ? a : b); }

// The end of the servo substep, after the motor step.  On the environment's
// first lane: self_contact_stats (selfContactStatsKernel's loop) folded into
// the running maxima (bam_env.py:333-335), then refresh() (bam_env.py:128-
// 155) on the new state: gravity and velocities in the root frame and the
// mean-velocity filter (bam_env.py:343-345).  On a lane per foot: the ground
// contact force on it (contactForcesKernel's sums), its site and the
// air/contact timers.  What is read of the buffers is read first, in one
// round trip.
template <class R, int B, int J, int CG, int CS, int L, class Env>
__device__ __forceinline__ void servoEpilogue(const ServoArgs<R> &sv, const DeviceModel<R> &M, Env &E,
                                              int e, int lane) {
  static_assert(DUCK_MAX_FEET <= L, "a lane per foot");
  auto &s = E.s;
  StateView<R, B, J, CG, CS> v{M, s};
  const bool lead = lane == 0, foot = lane < sv.numFeet;
  const size_t at = size_t(e) * sv.numFeet + lane;
  R contacts = 0, penetration = 0, off[3] = {0, 0, 0}, mean[3] = {0, 0, 0}, air = 0, touch = 0;
  if (lead) {
    if (sv.selfContacts)
      contacts = sv.selfContacts[e];
    if (sv.selfPenetration)
      penetration = sv.selfPenetration[e];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      off[k] = sv.rootOffset[size_t(e) * 3 + k];
    if (sv.meanVelocity) {
#pragma unroll
      for (int k = 0; k < 3; ++k)
        mean[k] = sv.meanVelocity[size_t(e) * 3 + k];
    }
  }
  if (foot) {
    if (sv.airTime)
      air = sv.airTime[at];
    if (sv.contactTime)
      touch = sv.contactTime[at];
  }
  auto put = [](R *out, size_t i, V3<R> u) {
    if (out) {
      out[3 * i] = u.x;
      out[3 * i + 1] = u.y;
      out[3 * i + 2] = u.z;
    }
  };
  if (lead) {
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
    if (sv.selfContacts)
      sv.selfContacts[e] = maximumNan(contacts, n);
    if (sv.selfPenetration)
      sv.selfPenetration[e] = maximumNan(penetration, depthMax);
    const Q4<R> q1 = v.Q(1), root = q1 * Q4<R>{sv.rootInv[0], sv.rootInv[1], sv.rootInv[2], sv.rootInv[3]};
    const V3<R> w1 = v.W(1), v1{s.v[0][1], s.v[1][1], s.v[2][1]};
    put(sv.gravity, e, rotate(conj(root), V3<R>{0, 0, -1}));
    put(sv.angularVelocity, e, rotate(conj(root), w1));
    const V3<R> rootR = -rotate(q1, V3<R>{off[0], off[1], off[2]});
    const V3<R> origin = v1 + cross(w1, rootR);
    put(sv.originVelocity, e, origin);
    put(sv.linearVelocity, e, rotate(conj(root), origin));
    // mean_velocity_world.lerp_(origin, alpha) (bam_env.py:343-345) as
    // mean + alpha (origin - mean)
    put(sv.meanVelocity, e,
        V3<R>{mean[0] + sv.meanAlpha * (origin.x - mean[0]), mean[1] + sv.meanAlpha * (origin.y - mean[1]),
              mean[2] + sv.meanAlpha * (origin.z - mean[2])});
  }
  if (foot) {
    // (the arguments selected, not indexed by lane: indexed they would be
    // copied to scratch memory)
    int body = sv.feet[0];
    V3<R> site{sv.sites[0][0], sv.sites[0][1], sv.sites[0][2]};
#pragma unroll
    for (int f = 1; f < DUCK_MAX_FEET; ++f) {
      body = lane == f ? sv.feet[f] : body;
      site.x = lane == f ? sv.sites[f][0] : site.x;
      site.y = lane == f ? sv.sites[f][1] : site.y;
      site.z = lane == f ? sv.sites[f][2] : site.z;
    }
    V3<R> force{0, 0, 0};
    for (int i = 0; i < s.ngc; ++i) {
      const auto &c = s.gc[i];
      if (gcBody(c.id) != body)
        continue;
      V3<R> g = -((V3<R>{1, 0, 0} * c.lambda[0] + V3<R>{0, 1, 0} * c.lambda[1]) +
                  V3<R>{0, 0, 1} * c.lambda[2]);
      force.x += g.x;
      force.y += g.y;
      force.z += g.z;
    }
    put(sv.footForces, at, force);
    const V3<R> r = rotate(v.Q(body), site);
    const V3<R> vb{s.v[0][body], s.v[1][body], s.v[2][body]};
    put(sv.sitePositions, at, v.X(body) + r);
    put(sv.siteVelocities, at, vb + cross(v.W(body), r));
    const bool contact = norm(force) > R(1e-5);
    const R h = M.dt;
    if (sv.airTime)
      sv.airTime[at] = contact ? R(0) : air + h;
    if (sv.contactTime)
      sv.contactTime[at] = contact ? touch + h : R(0);
  }
}

} // namespace duckhip
