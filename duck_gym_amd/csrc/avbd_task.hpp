// Control-step kernels of the tensor VecEnv (python/duck_gym/tensor_env.py):
// action clamping and servo targets, and the observation, reward, failure,
// timeout and episode bookkeeping that the reference assembles from ~40 torch
// ops per control step (tensor_env.py:178-219, 221-391).  The root pose and
// joint state are read straight from the HBM state blob, so no [E,B,13]
// snapshot is materialised.
#pragma once
#include "../../include/duck_hip.h"
#include "avbd_queries.hpp"

namespace duckhip {

enum TaskMode { kTaskStep = 0, kTaskReset = 1 };

DUCK_HD float mexp(float x) { return expf(x); }
DUCK_HD double mexp(double x) { return exp(x); }
DUCK_HD float tsin(float x) { return sinf(x); }
DUCK_HD double tsin(double x) { return sin(x); }

// Observation widths (tensor_env.py:238-258 and the 48-wide rollout layout).
DUCK_HD int taskObsDim(const DuckTask &t, int nj) {
  if (t.kind == DUCK_TASK_STANDING)
    return 10 + 3 * nj;
  if (t.kind == DUCK_TASK_LOCOMOTION)
    return 16 + 3 * nj + (t.velocity_filter ? 2 : 0);
  return 6 + 3 * nj;
}

// The gait reference of hinge j (tensor_env.py:263-277): the episode's
// phase picks two neighbouring rows of the table of the command's direction
// (the first of the largest of +x, -x, +y, -y) and blends them linearly;
// HOME blends into that over the first second.  The operations and their
// order are torch's, in the batch dtype.
template <class R>
DUCK_HD R gaitReference(const DuckTask &t, long long episode, const R *cmd, int j, int nj) {
  const R *table = static_cast<const R *>(t.gait_table);
  const int count = t.gait_phases;
  const R ep = R(episode);
  const R phase = ep * R(t.control_dt) / R(t.gait_period);
  // torch.remainder of a non-negative phase by 1 is fmod; index < count
  // (the clamp only guards the table)
  const R index = fmod(phase, R(1)) * R(count);
  long long lo = static_cast<long long>(index);
  lo = lo < 0 ? 0 : (lo >= count ? count - 1 : lo);
  const R fraction = index - R(lo);
  const R score[4] = {cmd[0], -cmd[0], cmd[1], -cmd[1]};
  int d = 0;
  for (int k = 1; k < 4; ++k)
    d = score[k] > score[d] ? k : d;
  const R a = table[(size_t(d) * count + lo) * nj + j];
  const R b = table[(size_t(d) * count + (lo + 1) % count) * nj + j];
  const R ref = a * (R(1) - fraction) + b * fraction;
  R blend = ep * R(t.control_dt);
  blend = blend < R(0) ? R(0) : (blend > R(1) ? R(1) : blend);
  const R home = R(t.home[j]);
  return home + (ref - home) * blend;
}

// a = clamp(actions, -1, 1); target = clamp(ref + scale a, lower, upper)
// with ref = `reference`, else the gait reference (t.gait), else HOME
// (tensor_env.py:263-283).
template <class R>
__global__ void taskTargetsKernel(DuckTask t, int count, int nj, const R *actions,
                                  const R *reference, const long long *episode, const R *commands,
                                  R *clamped, R *target) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count * nj)
    return;
  int j = i % nj;
  R a = actions[i];
  // torch.clamp propagates NaN; so do these comparisons (NaN fails both).
  a = a < R(-1) ? R(-1) : (a > R(1) ? R(1) : a);
  const int e = i / nj;
  R ref = reference ? reference[i]
                    : (t.gait ? gaitReference<R>(t, episode[e], commands + size_t(e) * 2, j, nj)
                              : R(t.home[j]));
  R v = ref + R(t.action_scale) * a;
  R lo = R(t.lower[j]), hi = R(t.upper[j]);
  v = v < lo ? lo : (v > hi ? hi : v);
  clamped[i] = a;
  target[i] = v;
}

// TensorEnv.reset's inputs from the caller's random draws (tensor_env.py:
// 196-217), each value rounded per operation as the torch expressions are:
// thread i < count * nj writes q[i] = HOME + (u - 0.5) * 0.02 (HOME without
// draws); thread e < count writes the root offset (0, 0, 0.001, (v - 0.5) *
// 0.02, (v' - 0.5) * 0.02, 0) (zeros without draws) and, with a command draw
// (`selected`, or one `direction` for every env), commandsOut = mask ?
// table[direction] * speed : commands.
template <class R>
__global__ void taskResetInputsKernel(DuckTask t, int count, int nj, const unsigned char *mask,
                                      const R *jointDraws, const R *rootDraws,
                                      const long long *selected, int direction, R speed,
                                      const R *commands, R *q, R *roots, R *commandsOut) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count * nj) {
    const R home = R(t.home[i % nj]);
    q[i] = jointDraws ? home + (jointDraws[i] - R(0.5)) * R(0.02) : home;
  }
  if (i >= count)
    return;
  R *r = roots + size_t(i) * 6;
  r[0] = r[1] = r[5] = R(0);
  r[2] = rootDraws ? R(0.001) : R(0);
  r[3] = rootDraws ? (rootDraws[size_t(i) * 2] - R(0.5)) * R(0.02) : R(0);
  r[4] = rootDraws ? (rootDraws[size_t(i) * 2 + 1] - R(0.5)) * R(0.02) : R(0);
  if (selected || direction >= 0) {
    // the direction table [[1, 0], [-1, 0], [0, 1], [0, -1]]
    const int d = selected ? int(selected[i]) : direction;
    const R dx = d == 0 ? R(1) : (d == 1 ? R(-1) : R(0));
    const R dy = d == 2 ? R(1) : (d == 3 ? R(-1) : R(0));
    const bool on = mask[i] != 0;
    commandsOut[size_t(i) * 2] = on ? dx * speed : commands[size_t(i) * 2];
    commandsOut[size_t(i) * 2 + 1] = on ? dy * speed : commands[size_t(i) * 2 + 1];
  }
}

struct TaskBuffers {
  const unsigned char *mask; // reset mode: envs whose bookkeeping restarts
  void *action;              // [E,J] R: this step's clamped action (step) / current actions
  void *lastAction;          // [E,J] R: previous action; step mode overwrites it with action
  const void *commands;      // [E,2] R (locomotion, rollout)
  long long *episode;        // [E]
  void *filtered;            // [E,2] R (locomotion velocity filter)
  float *returns;            // [E]
  void *forces;              // [E,3] R (reset mode zeroes masked rows), may be null
  float *obs;                // [E,D]
  float *reward;             // [E]
  unsigned char *failed, *timeout, *done; // [E]
  void *diag;                // [E,6] R, may be null
};

// The task step and observation of [E] environments in one launch.  A wave
// takes 64 / B environments with B lanes each: lane b reads its body's
// component rows (and checks them finite), lane j forms hinge j's angle, rate,
// action terms and observation entries, lanes 0 to 2 add the three sums over
// the hinges in hinge order, lanes 0 and 1 form the two feet's terms, and
// every lane of an environment evaluates the root frame and the reward (one
// instruction stream either way); the observation rows leave as one contiguous
// run.  Every value is formed by the operations, in the order, of one lane
// going over the environment.  Bound by a few dependent chains and memory
// round trips: 7.4 us at 4096 environments, 16 us at 32768.  A lane per
// environment (64 waves at 4096, each hinge after the other) took 26 and
// 27 us.
template <class R, int B, int J, int CG, int CS>
__global__ __launch_bounds__(64) void taskKernel(DuckTask t, int mode, const DeviceModel<R> *model,
                                                 unsigned char *states, long long blobBytes, int count,
                                                 TaskBuffers io) {
  static_assert(J <= B && 64 % B == 0 && B >= 6, "a lane per body, hinge and diagnostic");
  using State = EnvState<R, B, J, CG, CS>;
  constexpr int G = 64 / B, D = 18 + 3 * J; // the widest observation row
  __shared__ R stage[G][13][B];             // x, q, v, w rows
  __shared__ R terms[G][3][J], sums[G][3], feet[G][2][2];
  __shared__ R contactZ[G][CG + CS];
  __shared__ int contactId[G][CG + CS];
  __shared__ float rows[G * D];
  const DeviceModel<R> &M = *model;
  const int lane = threadIdx.x % B, g = threadIdx.x / B;
  const int e0 = blockIdx.x * G, e = e0 + g, n = count - e0 < G ? count - e0 : G;
  const bool valid = e < count, step = mode == kTaskStep;
  const int nb = M.nb, nj = M.nj, width = taskObsDim(t, nj);
  const State &s = blobAt<State>(states, blobBytes, valid ? e : 0);
  const size_t row = size_t(valid ? e : 0), at = row * nj + lane;
  const bool joint = valid && lane < nj;
  R *actions = static_cast<R *>(io.action), *lasts = static_cast<R *>(io.lastAction);
  R *filt = io.filtered ? static_cast<R *>(io.filtered) + row * 2 : nullptr;

  // the hinge's frames, the body's rows and the caller's values
  const int jc = lane < nj ? lane : 0, ja = M.ja[jc], jb = M.jb[jc];
  const V3<R> axisA{M.axisA[0][jc], M.axisA[1][jc], M.axisA[2][jc]};
  const V3<R> tangentA{M.tangentA[0][jc], M.tangentA[1][jc], M.tangentA[2][jc]};
  const V3<R> tangentB{M.tangentB[0][jc], M.tangentB[1][jc], M.tangentB[2][jc]};
  const R home = R(t.home[jc]);
  bool finite = true;
  if (valid && lane < nb) {
    const R body[13] = {s.x[0][lane], s.x[1][lane], s.x[2][lane], s.q[0][lane], s.q[1][lane],
                        s.q[2][lane], s.q[3][lane], s.v[0][lane], s.v[1][lane], s.v[2][lane],
                        s.w[0][lane], s.w[1][lane], s.w[2][lane]};
#pragma unroll
    for (int k = 0; k < 13; ++k) {
      finite = finite && mfinite(body[k]);
      stage[g][k][lane] = body[k];
    }
  }
  const bool restart = valid && !step && io.mask && io.mask[row] != 0;
  R act = joint && !restart ? actions[at] : R(0);
  const R last = joint && step ? lasts[at] : R(0);
  R cmd[2] = {0, 0}, filtered[2] = {0, 0}, diag[6] = {0, 0, 0, 0, 0, 0};
  if (valid && io.commands) {
    cmd[0] = static_cast<const R *>(io.commands)[row * 2];
    cmd[1] = static_cast<const R *>(io.commands)[row * 2 + 1];
  }
  if (valid && filt && !restart) {
    filtered[0] = filt[0];
    filtered[1] = filt[1];
  }
  long long episode = valid && !restart ? io.episode[row] : 0;
  const float returns = valid && step ? io.returns[row] : 0.f;
  if (valid && step) {
    constexpr int slot[5] = {kJointError, kPenetration, kContacts, kConverged, kAxisError};
#pragma unroll
    for (int k = 0; k < 5; ++k)
      diag[k] = s.diag[slot[k]];
    diag[5] = R(s.failed);
  }
  if (restart) {
    // tensor_env.py:199-203: restart the episode bookkeeping of reset envs.
    if (joint)
      actions[at] = R(0);
    if (lane < 2 && filt)
      filt[lane] = R(0);
    if (lane < 3 && io.forces)
      static_cast<R *>(io.forces)[row * 3 + lane] = R(0);
    if (lane == 0) {
      io.episode[row] = 0;
      io.returns[row] = 0.f;
    }
  }
  const int ngc = valid ? (s.ngc < CG ? s.ngc : CG) : 0, nsc = valid ? (s.nsc < CS ? s.nsc : CS) : 0;
  if (step && t.load_transfer) {
    // z of contactForcesKernel's term of each contact
    for (int i = lane; i < ngc; i += B) {
      const auto &c = s.gc[i];
      contactId[g][i] = c.id;
      contactZ[g][i] = (-((V3<R>{1, 0, 0} * c.lambda[0] + V3<R>{0, 1, 0} * c.lambda[1]) +
                          V3<R>{0, 0, 1} * c.lambda[2]))
                           .z;
    }
    for (int i = lane; i < nsc; i += B) {
      contactId[g][CG + i] = s.sc[i].id;
      contactZ[g][CG + i] = (-selfForceWorld(s.sc[i])).z;
    }
  }
  const uint64_t group = ((uint64_t(1) << B) - 1) << (g * B);
  finite = (__ballot(!finite) & group) == 0;
  __syncthreads();

  auto Q = [&](int b) { return Q4<R>{stage[g][3][b], stage[g][4][b], stage[g][5][b], stage[g][6][b]}; };
  auto X = [&](int b) { return V3<R>{stage[g][0][b], stage[g][1][b], stage[g][2][b]}; };
  auto W = [&](int b) { return V3<R>{stage[g][10][b], stage[g][11][b], stage[g][12][b]}; };
  float *o = rows + g * width;
  const int heads = t.kind == DUCK_TASK_ROLLOUT ? 6 : 10;
  if (joint) {
    const Q4<R> qa = Q(ja), qb = Q(jb);
    const R d = hingeAngle(qa, qb, axisA, tangentA, tangentB) - home;
    const R rate = dot(W(jb) - W(ja), rotate(qa, axisA));
    const R da = act - last;
    terms[g][0][lane] = d * d;
    terms[g][1][lane] = act * act;
    terms[g][2][lane] = da * da;
    o[heads + lane] = float(d);
    o[heads + nj + lane] = float(R(0.1) * rate);
    o[heads + 2 * nj + lane] = float(act);
  }

  // Root frame q = q_body1 (x) conj(root_iquat) (tensor_env.py:140-142, 222).
  const int root = 1;
  const Q4<R> iq{R(t.iquat[0]), -R(t.iquat[1]), -R(t.iquat[2]), -R(t.iquat[3])};
  const Q4<R> q = Q(root) * iq;
  const V3<R> grav = rotateInv(q, V3<R>{R(0), R(0), R(-1)});
  const V3<R> vel{stage[g][7][root], stage[g][8][root], stage[g][9][root]};
  const V3<R> v = rotateInv(q, vel);
  const V3<R> w = rotateInv(q, W(root));
  const R yawC = R(1) - R(2) * (q.y * q.y + q.z * q.z);
  const R yawS = R(2) * (q.w * q.z + q.x * q.y);
  const R height = X(root).z - R(t.root_height);

  if (step && valid && lane < 2) {
    // Gait shaping (tensor_env.py:328-354), at the counter after this step:
    // lane f forms foot f's squared gap and load error.
    const int f = lane, fb = t.feet[f];
    if (t.foot_clearance) {
      // the feet's lowest collision points against a lift that peaks
      // mid-swing; the phase is float32 (an int64 counter times a float)
      const R *pts = static_cast<const R *>(t.foot_point);
      const V3<R> p = X(fb);
      const Q4<R> qf = Q(fb);
      // inverse_rotate(q, up) (tensor_env.py:21-23)
      const V3<R> up{R(0), R(0), R(1)}, u{-qf.x, -qf.y, -qf.z};
      const V3<R> tt = cross(u, up) * R(2);
      const V3<R> localUp = (up + tt * qf.w) + cross(u, tt);
      R lowest = R(0);
      for (int k = 0; k < t.foot_points; ++k) {
        const R *c = pts + (size_t(f) * t.foot_points + k) * 3;
        const R h = (c[0] * localUp.x + c[1] * localUp.y + c[2] * localUp.z) + p.z;
        lowest = k == 0 || h < lowest ? h : lowest;
      }
      float phase =
          float(episode + 1) * float(t.control_dt) / float(t.gait_period) + (f ? 0.5f : 0.0f);
      phase = fmodf(phase, 1.0f);
      float swing = (phase - 0.6f) / 0.4f;
      swing = swing < 0.0f ? 0.0f : (swing > 1.0f ? 1.0f : swing);
      const float sw = sinf(float(3.14159265358979323846) * swing);
      const R desired = R(float(t.gait_lift) * (sw * sw));
      const R gap = (lowest < R(0) ? R(0) : lowest) - desired;
      feet[g][0][f] = gap * gap;
    }
    if (t.load_transfer) {
      // vertical contact force of each foot, in body weights, against a
      // sinusoidal left/right split
      const R cycle = (R(episode) + R(1)) * R(t.control_dt) / R(t.gait_period);
      const R left = R(0.5) + R(0.5) * tsin(R(2 * 3.14159265358979323846) * (cycle - R(0.05)));
      R z = 0;
      for (int i = 0; i < ngc; ++i)
        if (gcBody(contactId[g][i]) == fb)
          z += contactZ[g][i];
      for (int i = 0; i < nsc; ++i) {
        const int id = contactId[g][CG + i];
        const R fz = contactZ[g][CG + i];
        if (scBody(id) == fb)
          z += fz;
        if (scOther(id) == fb)
          z -= fz;
      }
      R force = z / R(t.weight);
      force = force < R(0) ? R(0) : (force > R(3) ? R(3) : force);
      const R d = force - (f ? R(1) - left : left);
      feet[g][1][f] = d * d;
    }
  }
  __syncthreads();
  if (step && valid && lane < 3) {
    R sum = 0;
    for (int j = 0; j < nj; ++j)
      sum += terms[g][lane][j];
    sums[g][lane] = sum;
  }
  __syncthreads();
  if (step) {
    // Failure (tensor_env.py:294-301; the rollout task fails on a fall).
    const R cosHalf = R(cosf(0.5f)); // torch.cos of a float32 0.5
    bool failed;
    if (t.kind == DUCK_TASK_ROLLOUT)
      failed = X(root).z < R(t.fall_height);
    else
      failed = grav.z > -cosHalf || mabs(height) > R(0.04) || diag[0] > R(0.005) || diag[1] > R(0.005);
    failed = failed || diag[5] > R(0) || !finite;

    const R pose = sums[g][0], act2 = sums[g][1], dact2 = sums[g][2];
    const R tilt = grav.x * grav.x + grav.y * grav.y;
    const R w2 = dot(w, w);
    R reward;
    if (t.kind == DUCK_TASK_STANDING) {
      // tensor_env.py:302-310
      reward = R(1.5) * mexp(R(-20) * tilt) + mexp(R(-2000) * height * height) +
               R(0.5) * mexp(R(-10) * dot(v, v)) - R(0.02) * w2 - R(0.05) * pose -
               R(0.01) * act2 - R(0.02) * dact2;
    } else {
      // tensor_env.py:311-327: world-frame COM velocity against the command.
      R vx = vel.x, vy = vel.y;
      if (t.kind == DUCK_TASK_LOCOMOTION && t.velocity_filter) {
        const R alpha = R(t.velocity_alpha);
        filtered[0] = (R(1) - alpha) * filtered[0] + alpha * vx;
        filtered[1] = (R(1) - alpha) * filtered[1] + alpha * vy;
        vx = filtered[0];
        vy = filtered[1];
      }
      const R ex = vx - cmd[0], ey = vy - cmd[1];
      const R error = ex * ex + ey * ey;
      const R sigma = R(t.tracking_sigma);
      reward = R(1) * mexp(R(-20) * tilt) + mexp(R(-2000) * height * height) +
               R(t.tracking_weight) * mexp(-error / (sigma * sigma)) - R(0.1) * w2 -
               R(t.heading_weight) * (R(1) - yawC) - R(0.02) * act2 - R(0.03) * dact2;
    }
    if (t.foot_clearance)
      reward -= R(20000) * (feet[g][0][0] + feet[g][0][1]);
    if (t.load_transfer)
      reward -= R(3) * (feet[g][1][0] + feet[g][1][1]);
    reward = (failed ? R(-2) : reward) * R(t.control_dt);
    episode += 1;
    const bool timeout = episode >= t.max_episode_length && !failed;
    if (joint)
      lasts[at] = act;
    if (valid && lane == 0) {
      io.episode[row] = episode;
      io.returns[row] = returns + float(reward);
      io.reward[row] = float(reward);
      io.failed[row] = failed;
      io.timeout[row] = timeout;
      io.done[row] = failed || timeout;
      if (t.kind == DUCK_TASK_LOCOMOTION && t.velocity_filter) {
        filt[0] = filtered[0];
        filt[1] = filtered[1];
      }
    }
    if (valid && io.diag) {
#pragma unroll
      for (int k = 0; k < 6; ++k)
        if (lane == k)
          static_cast<R *>(io.diag)[row * 6 + k] = diag[k];
    }
  }

  // Observation (tensor_env.py:238-258), cast to float32: the entries before
  // and after the hinges'.
  if (valid && lane == 0) {
    int k = 0;
    o[k++] = float(grav.x);
    o[k++] = float(grav.y);
    o[k++] = float(grav.z);
    if (t.kind != DUCK_TASK_ROLLOUT) {
      o[k++] = float(v.x);
      o[k++] = float(v.y);
      o[k++] = float(v.z);
    }
    o[k++] = float(w.x);
    o[k++] = float(w.y);
    o[k++] = float(w.z);
    if (t.kind != DUCK_TASK_ROLLOUT)
      o[k++] = float(height);
    k += 3 * nj;
    if (t.kind == DUCK_TASK_LOCOMOTION) {
      // (episode * control_dt) * (2 pi / period), the factor formed in double.
      const R phase = R(episode) * R(t.control_dt) * R(2 * 3.14159265358979323846 / t.gait_period);
      o[k++] = float(cmd[0]);
      o[k++] = float(cmd[1]);
      o[k++] = float(yawC);
      o[k++] = float(yawS);
      o[k++] = float(msin(phase));
      o[k++] = float(mcos(phase));
      if (t.velocity_filter) {
        o[k++] = float(filtered[0]);
        o[k++] = float(filtered[1]);
      }
    }
  }
  __syncthreads();
  copyRows(io.obs + size_t(e0) * width, rows, n * width, threadIdx.x);
}

// The maximum of the two, NaN when either is (torch.amax).
template <class R> DUCK_HD R maxNan(R a, R b) { return a != a || b != b ? R(NAN) : (a > b ? a : b); }

// Sums (or, for the logged maxima, maxima) over the wave, on every lane.
constexpr int kTaskLogs = DUCK_TASK_LOGS;
template <class R> __device__ __forceinline__ void waveLogs(R (&v)[kTaskLogs]) {
#pragma unroll
  for (int o = 32; o > 0; o /= 2)
#pragma unroll
    for (int k = 0; k < kTaskLogs; ++k) {
      const R u = __shfl_xor(v[k], o, 64);
      v[k] = k == 1 || k == 2 ? maxNan(v[k], u) : v[k] + u;
    }
}

// The scalars that tensor_env.py:367-391 logs after a step, over all
// environments, in two launches: here a wave of 64 environments forms its
// terms (the root's pose and velocity straight from the blobs) and their sums
// and maxima as row 1 + block of `out`; taskLogReduceKernel folds the rows
// into row 0 in a fixed order, so the values do not depend on timing.  Bound by
// launch: 2 x 4 us at 4096 environments in the place of a state snapshot and
// some 50 torch launches (about 190 us of them on the stream).
template <class R, int B, int J, int CG, int CS>
__global__ __launch_bounds__(64) void taskLogKernel(DuckTask t, unsigned char *states, long long blobBytes,
                                                    int count, const unsigned char *failed, const R *diag,
                                                    const R *commands, const R *filtered, R speed,
                                                    R *out) {
  const int e = blockIdx.x * 64 + threadIdx.x;
  const bool valid = e < count;
  R v[kTaskLogs] = {0, R(-INFINITY), R(-INFINITY), 0, 0, 0, 0};
  if (valid) {
    v[0] = failed[e] ? R(1) : R(0);
    v[1] = diag[size_t(e) * 6];
    v[2] = diag[size_t(e) * 6 + 1];
  }
  if (valid && t.kind == DUCK_TASK_LOCOMOTION) {
    const auto &s = blobAt<EnvState<R, B, J, CG, CS>>(states, blobBytes, e);
    const Q4<R> q = Q4<R>{s.q[0][1], s.q[1][1], s.q[2][1], s.q[3][1]} *
                    Q4<R>{R(t.iquat[0]), -R(t.iquat[1]), -R(t.iquat[2]), -R(t.iquat[3])};
    const R vx = s.v[0][1], vy = s.v[1][1];
    const R cx = commands[size_t(e) * 2], cy = commands[size_t(e) * 2 + 1];
    const R fx = (t.velocity_filter ? filtered[size_t(e) * 2] : vx) - cx;
    const R fy = (t.velocity_filter ? filtered[size_t(e) * 2 + 1] : vy) - cy;
    const R dx = vx - cx, dy = vy - cy;
    v[3] = msqrt(dx * dx + dy * dy);
    v[4] = vx * (cx / speed) + vy * (cy / speed);
    v[5] = msqrt(fx * fx + fy * fy);
    v[6] = mabs(matan2(R(2) * (q.w * q.z + q.x * q.y), R(1) - R(2) * (q.y * q.y + q.z * q.z)));
  }
  waveLogs(v);
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < kTaskLogs; ++k)
      out[(1 + size_t(blockIdx.x)) * kTaskLogs + k] = v[k];
}

template <class R>
__global__ __launch_bounds__(64) void taskLogReduceKernel(int rows, int count, R *out) {
  R v[kTaskLogs] = {0, R(-INFINITY), R(-INFINITY), 0, 0, 0, 0};
  for (int r = threadIdx.x; r < rows; r += 64)
#pragma unroll
    for (int k = 0; k < kTaskLogs; ++k) {
      const R u = out[(1 + size_t(r)) * kTaskLogs + k];
      v[k] = k == 1 || k == 2 ? maxNan(v[k], u) : v[k] + u;
    }
  waveLogs(v);
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < kTaskLogs; ++k)
      out[k] = k == 1 || k == 2 ? v[k] : v[k] / R(count);
}

} // namespace duckhip
