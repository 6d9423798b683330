"""The tiled passes of the SDF bake (edt_pack, edt_tile) at the edges of their tiles, their
16-bit squares and their LDS, and the envelope walk that longer lines keep, against scipy's
transform (oracle/edt.py) on the same occupancy.

Whole voxel distances squared are integers, so the expected value of any cell size is
sqrt(D * cell^2) in float64 rounded once to the output type, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import edt
from surfgym import vision

pytestmark = pytest.mark.gpu

# [nz, ny, nx]: blocks of 8 rows and words of 32 voxels around their edges; 509 / 510 planes,
# the last with 16-bit squares and the first with 32-bit ones; lines that need narrower tiles;
# lines past the LDS (y above 8192, z above 4096), which take the envelope walk
SHAPES = [(7, 8, 31), (8, 9, 32), (9, 7, 33), (17, 16, 1), (15, 33, 63), (24, 25, 130),
          (509, 40, 21), (510, 40, 21), (509, 530, 3), (4, 1030, 6), (3, 3000, 5), (2, 5000, 7),
          (1500, 5, 6), (2100, 4, 3), (3, 2, 1500), (4500, 3, 5), (2, 9000, 3)]
# past 4096 rows, or 2^24 voxels times planes, a block is 8 rows and not 2: either side of both
# lines, and the edges above past them; rows around the widths that 8, 16 and 32 words cover, one
# and two voxels a word; z lines that fit the LDS with blocks of 8 only
SHAPES += [(64, 64, 64), (64, 64, 65), (65, 64, 33), (7, 590, 31), (8, 513, 32), (9, 456, 34), (17, 241, 97),
           (64, 65, 1), (129, 33, 16), (129, 33, 17), (129, 33, 32), (129, 33, 65), (520, 8, 15), (520, 9, 9),
           (600, 7, 16), (600, 7, 17), (513, 9, 33), (9, 20, 16), (9, 20, 17), (9, 20, 65), (512, 8, 8),
           (600, 3, 9), (1500, 2, 3), (520, 1, 17), (4000, 1, 1), (2, 7000, 7)]


def _expected(occ, cell, dtype):
    squared = np.rint(edt.bake(occ, 1.0) ** 2)
    c = float(np.float32(cell))
    return np.sqrt(squared * (c * c)).astype(dtype)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_tile_edges_match_scipy(dev, shape):
    rng = np.random.default_rng(sum(shape))
    for density in (0.0, 0.0007, 0.05):
        occ = (rng.random(shape) < density).astype(np.uint8)
        for cell in (16.0, 24.0, 0.3):   # a power of two, exact in fp32 products, neither
            for dt, nd in ((torch.float32, np.float32), (torch.float16, np.float16)):
                print(f"case edt tiles {shape} density={density} cell={cell} {dt}", flush=True)
                got = vision.sdf_from_occupancy(occ, cell, device=dev, dtype=dt).cpu().numpy()
                assert np.array_equal(got, _expected(occ, cell, nd))


@pytest.mark.parametrize("shape", [(12, 20, 48), (12, 20, 47)], ids=str)
def test_occupancy_forms(dev, shape):
    """Any non-zero value is solid; bool, strided and misaligned device grids, other types."""
    rng = np.random.default_rng(5)
    occ = (rng.random(shape) < 0.03).astype(np.uint8) * rng.integers(1, 256, shape).astype(np.uint8)
    want = _expected((occ != 0).astype(np.uint8), 8.0, np.float32)
    o = torch.as_tensor(occ, device=dev)
    off = torch.zeros(o.numel() + 1, dtype=torch.uint8, device=dev)
    off[1:] = o.reshape(-1)
    wide = torch.zeros(shape[0], shape[1], 2 * shape[2], dtype=torch.uint8, device=dev)
    wide[:, :, ::2] = o
    forms = {"uint8": o, "bool": o != 0, "offset": off[1:].view(shape), "strided": wide[:, :, ::2],
             "float": o.float() * 0.25, "int64": o.to(torch.int64) * 256, "host bool": torch.as_tensor(occ) != 0}
    for name, form in forms.items():
        print(f"case edt form {name} {shape}", flush=True)
        got = vision.sdf_from_occupancy(form, 8.0, device=dev, dtype=torch.float32).cpu().numpy()
        assert np.array_equal(got, want), name
