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


def test_samples_and_yaws_run_on_the_current_stream(dev):
    """On a side stream behind the work that makes their positions, and captured into a graph,
    which a launch on any other stream would not enter: replayed on new positions, with eager calls
    between the replays."""
    field, mins = _field(dev, False)
    rng = np.random.default_rng(1)
    p = [torch.as_tensor(mins + rng.uniform(0.0, 1.0, (300, 3)) * np.array(field.dims) * field.cell, device=dev)
         for _ in range(4)]
    want = [(field.sample(x), field.descent_yaw(x)) for x in p]
    torch.cuda.synchronize()
    side = torch.cuda.Stream(dev)
    print("case goal field on a side stream", flush=True)
    with torch.cuda.stream(side):
        big = torch.randn(4096, 4096, device=dev)
        for _ in range(10):
            big = big @ big * 1e-3
        pos = p[0] + (big[0, 0] * 0.0).double().nan_to_num()
        got = field.sample(pos), field.descent_yaw(pos)
    side.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want[0]))
    pos = p[0].clone()
    graph = torch.cuda.CUDAGraph()
    print("case goal field captured", flush=True)
    with torch.cuda.graph(graph):
        out = field.sample(pos), field.descent_yaw(pos)
    for x, w in zip(p[1:], want[1:]):
        pos.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, w))
        assert torch.equal(field.sample(x), w[0])


def test_no_positions_are_refused(dev):
    field, _ = _field(dev, False)
    with pytest.raises(RuntimeError):
        field.descent_yaw(np.zeros((0, 3)))
