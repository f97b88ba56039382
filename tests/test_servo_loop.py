"""The servo loop's host side (duck_gym_amd/servo.py) on a recording batch."""

import numpy as np
import pytest
import torch

from duck_gym_amd.servo import SYNTHETIC_SUPPLY, ServoLoop, servo_params


class _Recorder:
    """A batch on the CPU that records the servo substeps asked of it."""

    num_envs, num_joints, dt = 3, 2, 0.005
    device, dtype = "cpu", torch.float32

    def __init__(self):
        self.calls = []

    def servo_substep(self, params, target, history, cursor, *args, count=1, **kwargs):
        self.calls.append((cursor, count))


@pytest.mark.parametrize("callback", [None, lambda loop: None], ids=["plain", "callback"])
@pytest.mark.parametrize("kind", [int, np.int64, np.int32, torch.tensor, bool])
def test_servo_loop_counts_of_any_whole_type(kind, callback):
    """Any whole number counts the substeps, and the ring's cursor stays a
    Python int (a saved loop's state); a fraction is refused."""
    loop = ServoLoop(_Recorder(), servo_params(**SYNTHETIC_SUPPLY, lag=2), [0.0, 0.0], [0.0] * 3)
    target = torch.zeros(3, 2)
    count = kind(1) if kind is bool else kind(5)
    loop.substeps(target, count, callback)
    loop.substeps(target, kind(0), callback)
    assert sum(n for _, n in loop.batch.calls) == int(count)
    assert type(loop.cursor) is int and loop.cursor == int(count) % 3
    assert all(type(c) is int and type(n) is int for c, n in loop.batch.calls)
    with pytest.raises(TypeError):
        loop.substeps(target, 2.0, callback)
    assert loop.cursor == int(count) % 3
