"""GoalField.descent_yaw in one launch against the formula it fuses.

The sampler is the one `sample` uses, so the differences are the same fp32 numbers; what may
differ is atan2's last bits: two correct fp32 atan2s are within a few ulp of each other, and
360 degrees has an ulp of 3e-5, hence 1e-4 degrees.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from surfgym import goalfield

pytestmark = pytest.mark.gpu


def _field(dev, quant, shape=(9, 14, 11), cell=16.0):
    rng = np.random.default_rng(5)
    q = rng.integers(0, 3000, shape).astype(np.uint16)
    reach = 2400 * 2.0                      # some corners are not honest
    mins = np.array([-40.0, 12.5, -300.0])
    grid = q if quant else q.astype(np.float32) * np.float32(2.0)
    return goalfield.GoalField(grid, mins, cell, reach, quant=2.0 if quant else None, device=dev), mins


# a block takes 64 positions, a wave 16
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 1000])
@pytest.mark.parametrize("quant", [False, True])
def test_matches_the_samples_formula(dev, n, quant):
    field, mins = _field(dev, quant)
    rng = np.random.default_rng(n)
    p = mins + rng.uniform(-0.2, 1.2, (n, 3)) * np.array(field.dims) * field.cell
    for make in (lambda: p,
                 lambda: torch.as_tensor(p, device=dev),
                 lambda: torch.as_tensor(p, device=dev, dtype=torch.float32),
                 lambda: torch.zeros(n, 6, device=dev).index_copy_(
                     1, torch.arange(3, device=dev), torch.as_tensor(p, device=dev).float())[:, :3],
                 lambda: torch.as_tensor(p.T.copy(), device=dev).T):
        pos = make()
        got = field.descent_yaw(pos)
        assert isinstance(got, np.ndarray) == isinstance(pos, np.ndarray)
        x = np.asarray(pos.cpu() if torch.is_tensor(pos) else pos, np.float64)
        h = field.cell
        s = [field.sample(x + np.array(o)) for o in ([h, 0, 0], [-h, 0, 0], [0, h, 0], [0, -h, 0])]
        want = np.degrees(np.arctan2(-(s[2] - s[3]).astype(np.float64),
                                     -(s[0] - s[1]).astype(np.float64))) % 360.0
        diff = np.abs(np.asarray(got.cpu() if torch.is_tensor(got) else got) - want)
        assert np.minimum(diff, 360.0 - diff).max() < 1e-4


def test_no_positions_are_refused(dev):
    field, _ = _field(dev, False)
    with pytest.raises(RuntimeError):
        field.descent_yaw(np.zeros((0, 3)))
