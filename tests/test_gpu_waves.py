"""Waves with fewer environments than they have room for: the lane groups left
over repeat the wave's first environment and store nothing, so an environment
steps bitwise the same with one, two or four to a wave, and a servo substep
writes every row of its outputs exactly once."""

import numpy as np
import pytest
import torch

from duck_gym_amd import CudaBatch
from duck_gym_amd.microduck import model_text
from duck_gym_amd.servo import SYNTHETIC_SUPPLY, ServoLoop, servo_params
from model_text import caterpillar

pytestmark = pytest.mark.gpu

DEV, DT, ITER = "cuda:0", 0.005, 10


def _parts(fp64):
    """A batch of four environments to a wave (the last one holding three),
    and the same environments as two to a wave (the last one alone), one to a
    wave, and three in all."""
    # own waves up to a quarter (float) or half (double) of those that fit: a
    # float workgroup takes a quarter of a compute unit, a double one half
    waves = torch.cuda.get_device_properties(0).multi_processor_count
    return [slice(0, 2 * waves + 3), slice(0, waves + 1), slice(waves + 1, 2 * waves),
            slice(2 * waves, 2 * waves + 3)]


@pytest.mark.parametrize("fp64,split,large", [(False, False, False), (True, False, False), (True, True, False),
                                              (False, False, True), (True, False, True), (True, True, True)])
def test_launches_of_several_streams_fit_the_device_together(fp64, split, large):
    """Environments get waves of their own only while two (the biped in double,
    one lane per block solve) or four such launches stay resident together;
    past that a wave is filled."""
    text = caterpillar(20, pairs=False) if large else model_text()[0]
    room, share = None, 2 if fp64 and not split and not large else 4
    for n in (4096, 1, 63, 64, 65, 100, 128, 129, 192, 193, 250, 256, 257, 500, 513, 1000, 1025):
        info = CudaBatch.from_text(text, n, DT, ITER, 0, fp64, split_solve=split).kernel_info()
        if room is None:
            cus = torch.cuda.get_device_properties(0).multi_processor_count
            room, most = cus * info["workgroups_per_cu"], info["envs_per_workgroup"]
            assert most == (2 if large else 4)
        assert info["envs_per_workgroup"] == most or share * info["workgroups_per_launch"] <= room, n
        if share * n <= room:
            assert info["envs_per_workgroup"] == 1, n


def _batches(pairs, fp64):
    text, meta = model_text(self_contact=pairs)
    parts = _parts(fp64)
    dtype = torch.float64 if fp64 else torch.float32
    batches = [CudaBatch.from_text(text, p.stop - p.start, DT, ITER, 0, fp64) for p in parts]
    assert [b.kernel_info()["envs_per_workgroup"] for b in batches] == [4, 2, 1, 1]
    rng, home = np.random.default_rng(11), np.array(meta["home"])
    E = parts[0].stop
    q, root = home + rng.uniform(-0.05, 0.05, (E, 14)), np.zeros((E, 6))
    root[:, 3:5] = rng.uniform(-0.02, 0.02, (E, 2))
    t = lambda a, p: torch.tensor(a[p], dtype=dtype, device=DEV)  # noqa: E731
    for b, p in zip(batches, parts):
        b.reset(torch.ones(p.stop - p.start, dtype=torch.bool, device=DEV), t(q, p), t(root, p))
    return batches, parts, meta, home, rng, t


def _same(outputs):
    whole, *rest = outputs
    for k, (w, *r) in enumerate(zip(whole, *rest)):
        joined = torch.cat(r)
        assert torch.equal(w, joined), (k, (w - joined).abs().max())


@pytest.mark.parametrize("pairs,fp64", [(False, False), (True, False), (False, True), (True, True)])
def test_environments_step_the_same_however_many_share_a_wave(pairs, fp64):
    batches, parts, _, home, rng, t = _batches(pairs, fp64)
    E = parts[0].stop
    for substeps in (1, 3, 1, 2):
        targets = home + rng.uniform(-0.2, 0.2, (E, 14))
        forces = rng.uniform(-0.1, 0.1, (E, 3))
        if substeps == 3:
            targets[E - 1, 2] = np.nan  # refused: that environment fails
        for b, p in zip(batches, parts):
            b.step(t(targets, p), t(forces, p), substeps, 8.0, 0.0)
        _same([b.state() for b in batches])
    assert int(batches[0].state()[2][:, 5].sum()) == 1
    motor = np.abs(rng.uniform(0, 0.1, (E, 14, 3)))
    for b, p in zip(batches, parts):
        b.step_motor(t(motor, p), t(np.zeros((E, 3)), p))
        b.advance(2)
    _same([(*b.state(), b.contact_forces(), b.contact_counts()) for b in batches])


@pytest.mark.parametrize("lag,fp64", [(0, False), (2, False), (2, True)])
def test_servo_substeps_are_the_same_however_many_share_a_wave(lag, fp64):
    batches, parts, meta, home, rng, t = _batches(True, fp64)
    feet = [meta["body_names"].index(n) for n in ("left_foot", "right_foot")]
    loops = [ServoLoop(b, servo_params(**SYNTHETIC_SUPPLY, lag=lag), home, [0.0, 0.0, 0.01],
                       root_principal_quat=meta["root_iquat"], feet=feet,
                       foot_sites=[[0.01, 0.0, -0.006]] * 2, mean_velocity_tau=0.2) for b in batches]
    for _ in range(3):
        targets = home + rng.uniform(-0.2, 0.2, (parts[0].stop, 14))
        for loop, p in zip(loops, parts):
            loop.substeps(t(targets, p), 2)
        _same([(*x.batch.state(), x.motor, x.previous_motor, x.previous_applied, x.initialized,
                x.history.transpose(0, 1), x.gravity, x.lin_vel, x.contact_force, x.site_pos,
                x.air_time, x.contact_time, x.self_contacts, x.self_penetration,
                x.mean_velocity) for x in loops])


@pytest.mark.parametrize("pairs,fp64,most", [(False, False, 0), (True, False, 48), (False, True, 0), (True, True, 320)])
def test_one_servo_substep_has_a_build_without_spills(pairs, fp64, most):
    """A single substep (duck_servo_substep, a loop with a callback) does not
    run the loop over substeps, whose spills reach 496 bytes per lane; what
    scratch memory is left holds the body-pair geometry (float: 48 bytes)."""
    b = CudaBatch.from_text(model_text(self_contact=pairs)[0], 5, DT, ITER, 0, fp64)
    one, many = b.kernel_info("servo_substep"), b.kernel_info("servo_substeps")
    assert one["scratch_bytes_per_lane"] <= most
    assert one == many if fp64 else one["vgprs"] < many["vgprs"]


@pytest.mark.parametrize("lag,fp64", [(0, False), (1, False), (2, True), (6, False)])
def test_servo_substeps_of_one_launch_are_those_of_a_launch_each(lag, fp64):
    """Histories fresh and filled, a reset between, an environment whose
    target is refused (its step fails, its servo goes on), lags below and
    above the substeps of a launch."""
    text, meta = model_text(self_contact=True)
    dtype, E = (torch.float64 if fp64 else torch.float32), 37
    home, rng = np.array(meta["home"]), np.random.default_rng(5)
    feet = [meta["body_names"].index(n) for n in ("left_foot", "right_foot")]
    t = lambda a: torch.tensor(a, dtype=dtype, device=DEV)  # noqa: E731
    every = torch.ones(E, dtype=torch.bool, device=DEV)
    loops = []
    for _ in range(2):
        b = CudaBatch.from_text(text, E, DT, ITER, 0, fp64)
        b.reset(every, t(np.tile(home, (E, 1))), t(np.zeros((E, 6))))
        loops.append(ServoLoop(b, servo_params(**SYNTHETIC_SUPPLY, lag=lag), home, [0.0, 0.0, 0.01],
                               root_principal_quat=meta["root_iquat"], feet=feet,
                               foot_sites=[[0.01, 0.0, -0.006]] * 2, mean_velocity_tau=0.2))
    some = torch.arange(E, device=DEV) % 5 == 2
    seen = []
    for k, count in enumerate((4, 1, 5, 3, 4)):
        targets = home + rng.uniform(-0.3, 0.3, (E, 14))
        if k == 2:
            targets[8, 3] = np.nan
        loops[0].substeps(t(targets), count)
        loops[1].substeps(t(targets), count, substep_callback=lambda loop: seen.append(loop.cursor))
        if k == 3:
            for loop in loops:
                loop.reset(some)
                loop.batch.reset(some, t(np.tile(home, (E, 1))), t(np.zeros((E, 6))))
        a, b = ([*x.batch.state(), x.motor, x.previous_motor, x.previous_applied, x.initialized, x.history,
                 x.gravity, x.ang_vel, x.lin_vel, x.origin_velocity, x.contact_force, x.site_pos, x.site_vel,
                 x.air_time, x.contact_time, x.self_contacts, x.self_penetration, x.mean_velocity]
                for x in loops)
        for i, (p, q) in enumerate(zip(a, b)):
            assert torch.equal(p.nan_to_num(-9.0) if p.is_floating_point() else p,
                               q.nan_to_num(-9.0) if q.is_floating_point() else q), (k, i)
        assert loops[0].cursor == loops[1].cursor
        raw = [x.batch.export_state().cpu().numpy() for x in loops]
        codec = loops[0].batch.codec()
        header = codec.L["gc"]
        assert np.array_equal(raw[0][:, :header], raw[1][:, :header]), k
    assert len(seen) == 17 and loops[0].batch.state()[2][:, 5].sum() == 1


@pytest.mark.parametrize("which,own,fp64", [("pairs", False, False), ("pairs", True, False), ("plain", False, False),
                                            ("plain", True, False), ("chain", False, False), ("chain", True, False),
                                            ("pairs", True, True), ("plain", True, True), ("chain", True, True)])
def test_servo_substeps_leave_the_blobs_of_a_launch_each(which, own, fp64):
    """Every byte of the exported states, the contact lists with the entries
    past their ends, drive channels and colours included, over falls and
    curls in which contacts come and go within a call; `own`: masses,
    friction and velocities per environment."""
    if which == "chain":
        text, home, feet, reach, curl = caterpillar(20, pairs=True), np.zeros(19), [1, 2], 1.2, 1.3
    else:
        text, meta = model_text(self_contact=which == "pairs")
        home, reach, curl = np.array(meta["home"]), 0.6, 0.0
        feet = [meta["body_names"].index(n) for n in ("left_foot", "right_foot")]
    E, J, dtype, rng = 61, len(home), torch.float64 if fp64 else torch.float32, np.random.default_rng(17)
    t = lambda a: torch.tensor(a, dtype=dtype, device=DEV)  # noqa: E731
    root, ext = np.zeros((E, 6)), np.zeros((E, 5))
    root[:, 2] = rng.uniform(0, 0.02, E)
    root[:, 3:5] = rng.uniform(-0.2, 0.2, (E, 2))
    ext[:, 0], ext[:, 1] = rng.uniform(0.3, 1, E), rng.uniform(0.9, 1.1, E)
    ext[:, 2:] = rng.normal(0, 0.3, (E, 3))
    q = home + rng.uniform(-curl, curl, (E, J))
    loops = []
    for _ in range(2):
        b = CudaBatch.from_text(text, E, DT, ITER, 0, fp64)
        b.reset(torch.ones(E, dtype=torch.bool, device=DEV), t(q), t(root), t(ext) if own else None)
        loops.append(ServoLoop(b, servo_params(**SYNTHETIC_SUPPLY, lag=1), home, [0.0, 0.0, 0.01], feet=feet,
                               foot_sites=[[0.01, 0.0, -0.006]] * 2))
    shrunk = torch.zeros(2, dtype=torch.long)
    for k in range(14):
        targets, counts = t(home + rng.uniform(-reach, reach, (E, J))), []
        loops[0].substeps(targets, 4)
        loops[1].substeps(targets, 4, lambda loop: counts.append(loop.batch.contact_counts()))
        raw = [x.batch.export_state() for x in loops]
        assert torch.equal(raw[0], raw[1]), k
        counts = torch.stack(counts)
        shrunk += (counts.amax(0) > counts[-1]).sum(0).cpu()
        if k == 6:  # another drive between: held controls, then a target launch
            for x in loops:
                x.batch.advance(1)
                x.batch.step(targets, torch.zeros(E, 3, dtype=dtype, device=DEV), 1, 8.0, 0.0)
    # lists that were longer within a call than at its end
    assert shrunk[0] > 0 and (shrunk[1] > 0 or which != "pairs"), shrunk
