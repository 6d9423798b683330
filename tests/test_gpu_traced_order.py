"""The tile order of large renders on grids beyond the Infinity Cache, whose key follows a unit's
centre ray: the order only permutes the tiles, so the image is the launch order's bit for bit.

A 102 M-voxel grid (205 MB in two bytes) and one of 51 M in fp32, renders of 2^18 tiles: images of
one quad (4 tiles), one env past a whole number of keyed blocks, and eyes past the map's border."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from surfgym import vision

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("store,pinhole,surf,bf16", [("f32", False, False, False), ("f32", True, False, True),
                                                     ("f16", False, True, False), ("r16", True, False, False)])
def test_traced_order_is_the_launch_order(dev, store, pinhole, surf, bf16):
    nz, ny, nx, cell = (200 if store == "f32" else 400), 510, 505, 16.0
    z, y, x = (np.arange(k, dtype=np.float32) for k in (nz, ny, nx))
    sdf = (z * 9.0)[:, None, None] + np.abs(np.sin(y * 0.07))[:, None] * 90.0 + np.abs(np.cos(x * 0.05)) * 60.0
    mask = np.full(sdf.shape, 77, np.int8) if surf else None
    lid = vision.GpuLidar.from_grid(
        sdf, np.zeros(3, np.float32), cell, surf_nz=mask, width=27, height=7, range_units=5000.0, max_steps=40,
        near_range=1500.0, pinhole=pinhole, device=dev,
        grid_dtype={"f32": torch.float32, "f16": torch.float16, "r16": "r16"}[store])
    n = (1 << 16) + 1
    rng = np.random.default_rng(n)
    ext = np.array([nx, ny, nz]) * cell
    pose = np.concatenate([rng.uniform(-0.1, 1.1, (n, 3)) * ext, rng.uniform(-180, 180, (n, 1)),
                           rng.uniform(-80, 80, (n, 1)), rng.integers(0, 2, (n, 1))], 1).astype(np.float32)
    p = torch.as_tensor(pose, device=dev)
    images = []
    for order in ("lookahead", "lookahead", "launch"):
        print(f"case traced order {store} pinhole={pinhole} surf={surf} {order}", flush=True)
        lid.set_tile_order(order)
        out = torch.full((n, 27 * 7 * (2 if surf else 1)), -1.0, device=dev,
                         dtype=torch.bfloat16 if bf16 else torch.float32)
        lid.render(p[:, :3], p[:, 3], p[:, 4], p[:, 5], out=out)
        images.append(out)
    assert not (images[2] == -1.0).any()
    assert torch.equal(images[0], images[2]) and torch.equal(images[1], images[2])
