"""The state snapshot, the masked reset and the load query, which give an
environment a lane per body slot (16 or 32): environment counts around a
wave's four or two, models that fill the slots and models that leave most of
them empty, against the oracle's reset kinematics, snapshot and loads."""

import numpy as np
import pytest
import torch

from duck_gym_amd import CudaBatch
from duck_gym_amd.microduck import model_text
from model_text import caterpillar, chain
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu
DT, ITER, DEV = 0.005, 10, "cuda:0"
MODELS = {
    "microduck": lambda: model_text()[0],          # 16 bodies, 14 hinges, 6 tree levels
    "pair": lambda: chain(2),                      # one body, no hinge
    "full": lambda: caterpillar(31, pairs=False),  # 32 bodies, 30 hinges, 30 levels
}


def _batch(tmp_path, which, envs, fp64):
    path = tmp_path / "model.duck"
    path.write_text(MODELS[which]())
    return CudaBatch(path, envs, DT, ITER, 0, fp64), Oracle(path, DT, ITER, fp64)


def _tolerance(fp64, levels):
    """A level is one exponential map, three quaternion products and two
    rotations (about 40 roundings of quantities of order 1)."""
    return 40 * levels * (2.0 ** -52 if fp64 else 2.0 ** -23)


@pytest.mark.parametrize("fp64", [False, True], ids=["fp32", "fp64"])
@pytest.mark.parametrize("envs", [1, 2, 3, 4, 5, 67])
@pytest.mark.parametrize("which", sorted(MODELS))
def test_masked_reset_and_snapshot(tmp_path, which, envs, fp64):
    batch, oracle = _batch(tmp_path, which, envs, fp64)
    dtype, J = batch.dtype, batch.num_joints
    rng = np.random.default_rng(envs)
    cast = lambda a: torch.tensor(a, dtype=dtype, device=DEV)  # noqa: E731
    before, state_before = batch.export_state(), batch.state()
    q, root = rng.uniform(-0.3, 0.3, (envs, J)), rng.uniform(-0.2, 0.2, (envs, 6))
    mask = rng.uniform(0, 1, envs) < 0.5
    mask[0] = True
    bad = envs - 1 if envs > 1 else None
    if bad is not None:
        mask[bad] = True
        root[bad, 3] = np.inf
    batch.reset(torch.tensor(mask, device=DEV), cast(q), cast(root))
    bodies, joints, diag = (t.cpu().double().numpy() for t in batch.state())
    after = batch.export_state()
    tol = _tolerance(fp64, max(1, J))
    for e in range(envs):
        if e == bad:
            # refused: marked failed, the pose as it was
            assert diag[e, 5] == 1
            assert np.array_equal(bodies[e], state_before[0][e].cpu().double().numpy())
        elif mask[e]:
            oracle.reset(cast(q).cpu().double().numpy()[e], cast(root).cpu().double().numpy()[e])
            ob, oj, od = oracle.snapshot()
            np.testing.assert_allclose(bodies[e], ob, atol=tol, rtol=0)
            np.testing.assert_allclose(joints[e], oj.reshape(J, 2), atol=tol, rtol=0)
            assert not diag[e].any()
        else:
            assert torch.equal(after[e], before[e])


@pytest.mark.parametrize("fp64", [False, True], ids=["fp32", "fp64"])
@pytest.mark.parametrize("envs", [1, 5, 67])
@pytest.mark.parametrize("which", sorted(MODELS))
def test_snapshot_reads_every_field(tmp_path, which, envs, fp64):
    """bodies and diagnostics are the blob's own values, bit for bit."""
    batch, _ = _batch(tmp_path, which, envs, fp64)
    rng = np.random.default_rng(envs)
    codec, raw = batch.codec(), batch.export_state().cpu().numpy()
    for e in range(envs):
        s = codec.decode(raw[e])
        for name in ("x", "q", "v", "w"):
            s[name] = rng.standard_normal(s[name].shape)
        s["diag"], s["failed"] = rng.standard_normal(8), e % 2
        codec.encode(raw[e], s)
    batch.import_state(torch.tensor(raw, device=DEV))
    bodies, joints, diag = (t.cpu().numpy() for t in batch.state())
    assert np.isfinite(joints).all()
    for e in range(envs):
        s = codec.decode(raw[e])
        assert np.array_equal(bodies[e], np.concatenate([s["x"], s["q"], s["v"], s["w"]], axis=1))
        want = [s["diag"][0], s["diag"][1], s["diag"][2], s["diag"][3], s["diag"][4], s["failed"]]
        assert np.array_equal(diag[e], np.array(want, bodies.dtype))


@pytest.mark.parametrize("fp64", [False, True], ids=["fp32", "fp64"])
@pytest.mark.parametrize("envs", [1, 5, 67])
@pytest.mark.parametrize("which", ["microduck", "full"])
def test_generalized_loads(tmp_path, which, envs, fp64):
    """Loads after a step (velocities, contacts and drive torques not zero),
    the oracle's on the same trajectory in float64; in float32 a batch of one
    environment is the reference (the same code on other lanes)."""
    batch, oracle = _batch(tmp_path, which, envs, fp64)
    single, _ = _batch(tmp_path, which, 1, fp64)
    dtype, J = batch.dtype, batch.num_joints
    rng = np.random.default_rng(envs)
    cast = lambda a: torch.tensor(a, dtype=dtype, device=DEV)  # noqa: E731
    q, root = rng.uniform(-0.1, 0.1, (envs, J)), np.zeros((envs, 6))
    target, offset = q + rng.uniform(-0.2, 0.2, (envs, J)), rng.uniform(-0.02, 0.02, (envs, 3))
    force = np.zeros((envs, 3))
    on = lambda n: torch.ones(n, dtype=torch.bool, device=DEV)  # noqa: E731
    batch.reset(on(envs), cast(q), cast(root))
    batch.step(cast(target), cast(force), 2, 8.0, 0.0)
    loads = batch.generalized_loads(cast(offset))
    for e in range(envs):
        if fp64:
            oracle.reset(q[e], root[e])
            oracle.step(target[e], force[e], 2, 8.0, 0.0)
            want = oracle.generalized_loads(offset[e]).reshape(J, 3)
            scale = max(1.0, np.abs(want).max())
            np.testing.assert_allclose(loads[e].cpu().numpy(), want, atol=1e-9 * scale, rtol=0)
        else:
            single.reset(on(1), cast(q[e:e + 1]), cast(root[e:e + 1]))
            single.step(cast(target[e:e + 1]), cast(force[:1]), 2, 8.0, 0.0)
            assert torch.equal(loads[e], single.generalized_loads(cast(offset[e:e + 1]))[0])
