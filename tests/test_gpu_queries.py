"""The state snapshot, which gives an environment a lane
per body slot (16 or 32): environment counts around a wave's four or two,
models that fill the slots and models that leave most of them empty, against the
exported state."""

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
