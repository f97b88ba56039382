"""The dense step (two waves per SIMD, for batches of more waves than the
device has SIMDs) against the full step: the same environments stepped in one
large batch and in two halves that take the full step, every live byte of the
states equal.  Models: the biped; 14 boxes in a row on the ground (56 ground
contacts, 33 of them past the dense record's 23); seven stacks of two boxes;
one body without hinges."""

import numpy as np
import pytest
import torch

from duck_gym_amd import CudaBatch
from duck_gym_amd.microduck import model_text
from model_text import caterpillar, chain

pytestmark = pytest.mark.gpu
DT, ITER, DEV = 0.005, 10, "cuda:0"
MODELS = {
    "microduck": (lambda: model_text()[0], 8),
    "row": (lambda: caterpillar(14, pairs=False), 24),
    "stacks": (lambda: caterpillar(7, pairs=False, shapes_per_segment=2), 24),
    "single": (lambda: chain(2), 0),
}


def _live(batch):
    """The exported states with the unused tails of the contact lists zeroed
    (a list that shrinks leaves its old entries there)."""
    raw = batch.export_state().cpu().numpy()
    L = batch.codec().L
    assert L["gcBytes"] == 52
    ngc = raw[:, L["ngc"]:L["ngc"] + 4].copy().view(np.int32)[:, 0]
    at = np.arange(raw.shape[1])[None]
    dead = (at >= L["gc"] + 52 * ngc[:, None]) & (at < L["gc"] + 52 * L["CG"])
    raw[dead] = 0
    return raw, ngc


@pytest.mark.parametrize("custom", [False, True], ids=["model-bodies", "own-bodies"])
@pytest.mark.parametrize("which", sorted(MODELS))
def test_dense_step_is_the_full_step(which, custom):
    text, contacts = MODELS[which][0](), MODELS[which][1]
    simds = 4 * torch.cuda.get_device_properties(0).multi_processor_count
    E = 4 * simds + 5   # one wave more than SIMDs, and a partly empty one
    cut = E // 2
    parts = [slice(0, E), slice(0, cut), slice(cut, E)]
    batches = [CudaBatch.from_text(text, p.stop - p.start, DT, ITER) for p in parts]
    full = batches[1].kernel_info()
    assert batches[0].kernel_info()["waves_per_simd"] == 2 and full["waves_per_simd"] == 1
    J, rng = batches[0].num_joints, np.random.default_rng(7)
    home = batches[0].state()[1][0, :, 0].cpu().numpy()
    q = home + rng.uniform(-0.1, 0.1, (E, J))
    root = rng.uniform(-0.05, 0.05, (E, 6)) * [0, 0, 0.1, 1, 1, 1]
    ext = np.concatenate([rng.uniform(-0.3, 1, (E, 1)), rng.uniform(0.9, 1.1, (E, 1)),
                          rng.normal(0, 0.2, (E, 3))], axis=1)
    forces = rng.uniform(-0.1, 0.1, (E, 3))

    def each(call, *arrays):
        for b, p in zip(batches, parts):
            call(b, *(torch.tensor(a[p], dtype=torch.float32, device=DEV) for a in arrays))

    def reset(b, q, root, ext):
        b.reset(torch.ones(len(q), dtype=torch.bool, device=DEV), q, root, ext if custom else None)

    each(reset, q, root, ext)
    most = 0
    for k, (substeps, kp, limit) in enumerate([(1, 8.0, 0.0), (3, 8.0, 0.0), (1, 6.0, 0.3), (2, 6.0, 0.3),
                                               (1, 6.0, 0.3)]):
        targets = home + rng.uniform(-0.3, 0.3, (E, J))
        if k == 2 and J:
            targets[3, 0], targets[E - 1, J - 1] = np.nan, np.inf  # refused: these fail
        each(lambda b, t, f: b.step(t, f, substeps, kp, limit), targets, forces)
        if k == 3:
            for b in batches:
                b.advance(1)  # the held controls: what the dense step wrote of the drive
        whole, ngc = _live(batches[0])
        halves = [_live(b)[0] for b in batches[1:]]
        assert np.array_equal(whole, np.concatenate(halves)), k
        most = max(most, int(ngc.max()))
    assert most >= contacts
    failed = batches[0].state()[2][:, 5]
    assert int(failed.sum()) == (2 if J else 0)


@pytest.mark.parametrize("dense", [False, True])
def test_imported_states_with_impossible_contact_lists_fail(dense):
    """A count past the list's end or an id of no body or shape: the
    environment fails with empty lists and stays as it was imported, in the
    full and the dense step; the others step as if it were not there, and an
    export imported again is itself."""
    text, meta = model_text()
    E = 4 * 4 * torch.cuda.get_device_properties(0).multi_processor_count + 5 if dense else 23
    batches = [CudaBatch.from_text(text, E, DT, ITER) for _ in range(2)]
    assert (batches[0].kernel_info()["waves_per_simd"] == 2) == dense
    home = torch.tensor(np.tile(meta["home"], (E, 1)), dtype=torch.float32, device=DEV)
    zero = torch.zeros(E, 6, device=DEV)
    for b in batches:
        b.reset(torch.ones(E, dtype=torch.bool, device=DEV), home, zero)
        for _ in range(3):
            b.step(home, zero[:, :3].contiguous(), 1, 8.0, 0.0)
    raw = batches[0].export_state()
    batches[0].import_state(raw)
    assert torch.equal(batches[0].export_state(), raw)
    L, host = batches[0].codec().L, raw.cpu().numpy()
    ints = lambda e, at: host[e, at:at + 4].view(np.int32)  # noqa: E731
    assert ints(0, L["ngc"])[0] > 1
    body, shape = int(batches[0].num_bodies), 63
    bad = {1: ("ngc", L["CG"] + 1), 4: ("ngc", -1), 6: ("ngc", 2**30), 9: ("nsc", L["CS"] + 1), 11: ("nsc", -7),
           13: ("body", body << 6), 17: ("shape", shape), 22: ("ngc", 2**31 - 1)}
    for e, (what, value) in bad.items():
        if what in ("ngc", "nsc"):
            ints(e, L[what])[:] = value
        else:
            ints(e, L["gc"] + L["gcBytes"] + L["gc_id"])[:] = value
    batches[0].import_state(torch.tensor(host, device=DEV))
    imported = batches[0].state()[0]
    for b in batches:
        b.step(home, zero[:, :3].contiguous(), 2, 8.0, 0.0)
        b.advance(1)
    bodies, _, diag = batches[0].state()
    failed = torch.zeros(E, dtype=torch.bool, device=DEV)
    failed[list(bad)] = True
    assert torch.equal(diag[:, 5] != 0, failed)
    assert torch.equal(bodies[failed], imported[failed])
    assert int(batches[0].contact_counts()[failed].sum()) == 0
    assert int(batches[0].contact_forces()[failed].count_nonzero()) == 0
    assert torch.equal(bodies[~failed], batches[1].state()[0][~failed])
    assert torch.equal(batches[0].export_state()[~failed], batches[1].export_state()[~failed])
