"""The goal-field bake's tiles and queues at their edges, against the oracle's fixpoint bit for
bit: grids of many tiles (a queue per XCD) whose sides end inside a tile, ones a tile thick along
each axis, either side of the tile count from which there are eight queues, one long enough for
several rounds of sweeps, and the quantisation of voxel counts and outputs that allow no four-voxel
stores."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import goal as ogoal
from surfgym import _sdfr, goalfield

pytestmark = pytest.mark.gpu


def _occupancy(shape, seed):
    rng = np.random.default_rng(seed)
    occ = (rng.random(shape) < 0.25).astype(np.uint8)
    # a wall to go round
    if shape[0] > 1:
        occ[shape[0] // 2, : shape[1] - 2] = 1
    else:
        occ[:, shape[1] // 2, : shape[2] - 2] = 1
    return occ


@pytest.mark.parametrize("shape", [(129, 131, 135), (128, 130, 136), (521, 523, 5), (3, 1030, 1029), (6, 7, 4099),
                                   (520, 3, 515), (515, 520, 1), (1, 512, 512), (1, 512, 504)],
                         ids=str)
def test_many_tiles_match_oracle(dev, shape):
    occ = _occupancy(shape, sum(shape))
    nz, ny, nx = shape
    occ[0:2, 0:2, 0:2] = 0
    zone = {"mins": [0.5, 0.5, 0.5], "maxs": [9.0, 9.0, 9.0]}
    lo, hi = goalfield.seed_voxel_box(zone, np.zeros(3), 8.0, (nx, ny, nz))
    print(f"case goal tiles {shape}", flush=True)
    ref = ogoal.bake(occ, 8.0, lo, hi)
    for form in (occ, torch.as_tensor(occ, device=dev), torch.as_tensor(occ * 3, device=dev) != 0):
        field = goalfield.goal_field_from_occupancy(form, np.zeros(3), zone, 8.0, device=dev)
        assert np.array_equal(field.grid_q.cpu().numpy().view(np.uint16), ref["grid_q"])
        assert np.array_equal(field.grid.cpu().numpy(), ref["grid"])
        assert np.float32(field.reach_max) == ref["reach_max"]


@pytest.mark.parametrize("nx", [1, 7, 8, 9, 15, 16, 17, 40])
def test_occupancy_rows_at_any_alignment(dev, nx):
    """Rows are read eight voxels at once: ends inside a tile, any address, any non-zero byte."""
    shape = (9, 17, nx)
    n = int(np.prod(shape))
    rng = np.random.default_rng(nx)
    occ = np.where(rng.random(shape) < 0.3, rng.choice([1, 2, 127, 128, 255], shape), 0).astype(np.uint8)
    occ[0, 0, 0] = occ[8, 16, nx - 1] = 0
    zone = {"mins": [0.5, 100.0, 50.0], "maxs": [8.0 * nx, 8.0 * 17, 8.0 * 9]}   # odd box, the last voxels in it
    lo, hi = goalfield.seed_voxel_box(zone, np.zeros(3), 8.0, shape[::-1])
    ref = ogoal.bake(occ, 8.0, lo, hi)
    for offset in (0, 1, 2, 4, 7):
        buf = torch.ones(n + 16, dtype=torch.uint8, device=dev)
        buf[offset:offset + n] = torch.as_tensor(occ, device=dev).reshape(-1)
        print(f"case goal rows nx={nx} offset={offset}", flush=True)
        field = goalfield.goal_field_from_occupancy(buf[offset:offset + n].view(shape), np.zeros(3), zone, 8.0,
                                                    device=dev)
        assert np.array_equal(field.grid_q.cpu().numpy().view(np.uint16), ref["grid_q"])
        assert field.bake_info["n_seed"] == ref["n_seed"]


@pytest.mark.parametrize("nx", [12, 13, 16])
def test_quantised_outputs_at_any_alignment(dev, nx):
    """Through the C ABI: rows that allow four-voxel stores and rows that do not, each output some
    elements into its buffer or not asked for, nothing written beside them."""
    shape = (9, 11, nx)
    occ = torch.as_tensor(_occupancy(shape, 3), device=dev)
    occ[0, 0, 0] = 0
    n = occ.numel()
    lib = _sdfr.load()
    lo = (ctypes.c_int32 * 3)(0, 0, 0)
    ref = ogoal.bake(occ.cpu().numpy(), 16.0, np.zeros(3, np.int32), np.zeros(3, np.int32))
    ws = torch.empty(int(lib.sdfr_goal_workspace_bytes(nx, 11, 9)), dtype=torch.uint8, device=dev)
    info = _sdfr.GoalInfo()
    for qs, gs in [(a, b) for a in (0, 1, 2, 3, None) for b in (0, 1, 2, 3, None) if (a, b) != (None, None)]:
        q = torch.full((n + 8,), 77, dtype=torch.int16, device=dev)
        g = torch.full((n + 8,), -1.0, dtype=torch.float32, device=dev)
        print(f"case goal alignment nx={nx} q={qs} grid={gs}", flush=True)
        rc = lib.sdfr_goal_bake(occ.data_ptr(), nx, 11, 9, 16.0, lo, lo, 1 << 20,
                                None if qs is None else q[qs:].data_ptr(), None if gs is None else g[gs:].data_ptr(),
                                ctypes.byref(info), ws.data_ptr(), ws.numel(),
                                torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        for out, s, want, guard in ((q.cpu().numpy(), qs, ref["grid_q"].view(np.int16), 77),
                                    (g.cpu().numpy(), gs, ref["grid"], -1.0)):
            if s is None:
                assert (out == guard).all()
                continue
            assert np.array_equal(out[s:s + n].reshape(shape), want)
            assert (out[:s] == guard).all() and (out[s + n:] == guard).all()


@pytest.mark.parametrize("shape", [(24, 24, 40), (17, 23, 33), (8, 8, 4), (1, 1, 36)], ids=str)
def test_tiles_without_a_free_voxel(dev, shape):
    """Whole solid tiles, which are never queued: beside the seeds, under them, and in the way."""
    occ = np.zeros(shape, np.uint8)
    occ[:8, :8, 8:16] = 1                     # a solid tile inside the seed box
    occ[8:16, 8:16, 16:24] = 1
    occ[:8, 16:24, :8] = 1
    zone = {"mins": [0.5, 0.5, 0.5], "maxs": [100.0, 30.0, 30.0]}
    nz, ny, nx = shape
    lo, hi = goalfield.seed_voxel_box(zone, np.zeros(3), 8.0, (nx, ny, nz))
    print(f"case goal solid tiles {shape}", flush=True)
    ref = ogoal.bake(occ, 8.0, lo, hi)
    field = goalfield.goal_field_from_occupancy(occ, np.zeros(3), zone, 8.0, device=dev)
    assert np.array_equal(field.grid_q.cpu().numpy().view(np.uint16), ref["grid_q"])
    assert np.array_equal(field.grid.cpu().numpy(), ref["grid"])
    assert field.bake_info["n_seed"] == ref["n_seed"]
