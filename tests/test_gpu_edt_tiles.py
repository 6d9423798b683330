"""The tiled passes of the SDF bake (edt_pack, edt_tile) at the edges of their tiles and their
LDS, against scipy's transform (oracle/edt.py) on the same occupancy; at the largest squared
distances that 8, 16 and 32 bits hold, against the closed form of a grid with a few solid voxels;
and at outputs of any alignment.

Whole voxel distances squared are integers, so the expected value of any cell size is
sqrt(D * cell^2) in float64 rounded once to the output type, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import edt
from surfgym import _sdfr, vision

pytestmark = pytest.mark.gpu

# [nz, ny, nx]: blocks of 8 rows and words of 32 voxels around their edges; 509 / 510 planes,
# the last with 16-bit squares and the first with 32-bit ones (small distances here, large ones
# in test_large_distances); lines that need narrower tiles; lines past the LDS (y above 8192, z
# above 4096), which take the envelope walk
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


# the border is the nearest solid almost everywhere, so D reaches the square of half the shortest
# side: 255^2 at 509 planes, where distances along x of 256 and 257 are clamped to a byte; 255^2 at
# 510 planes in 32 bits; 310^2 beyond 16 bits
@pytest.mark.parametrize("shape", [(509, 511, 513), (510, 511, 513), (520, 509, 511), (620, 619, 621)], ids=str)
def test_large_distances(dev, shape):
    nz, ny, nx = shape
    axes = [torch.arange(n, device=dev, dtype=torch.int32) for n in shape]

    def border(i):   # distance along axis i to the solid layer around the grid
        return torch.minimum(axes[i] + 1, shape[i] - axes[i])

    for solids in ([], [(nz // 2, ny // 2, 40), (70, ny - 60, nx // 2), (nz // 2 + 90, 30, nx - 33)]):
        squared = torch.minimum(torch.minimum(border(0)[:, None, None], border(1)[:, None]), border(2)).square()
        occ = torch.zeros(shape, dtype=torch.uint8, device=dev)
        for p in solids:
            occ[p] = 1
            dz, dy, dx = ((axes[i] - p[i]).square() for i in range(3))
            squared = torch.minimum(squared, dz[:, None, None] + dy[:, None] + dx)
        most = int(squared.max())
        assert solids or most == ((min(shape) + 1) // 2) ** 2
        for cell in (16.0, 24.0, 0.3):
            c = float(np.float32(cell))
            for dt, nd in ((torch.float32, np.float32), (torch.float16, np.float16)):
                print(f"case edt large {shape} solids={len(solids)} cell={cell} {dt}", flush=True)
                of = torch.as_tensor(np.sqrt(np.arange(most + 1) * (c * c)).astype(nd), device=dev)
                got = vision.sdf_from_occupancy(occ, cell, device=dev, dtype=dt)
                assert torch.equal(got, of[squared])


@pytest.mark.parametrize("nx", [12, 13, 64])
def test_outputs_at_any_alignment(dev, nx):
    """Through the C ABI: outputs `shift` elements into their buffers, nothing written beside them."""
    shape = (9, 11, nx)
    rng = np.random.default_rng(nx)
    occ = (rng.random(shape) < 0.02).astype(np.uint8)
    lib = _sdfr.load()
    o = torch.as_tensor(occ, device=dev)
    n = o.numel()
    need = int(lib.sdfr_edt_workspace_bytes(nx, 11, 9))
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    for dt, nd, code in ((torch.float32, np.float32, _sdfr.F32), (torch.float16, np.float16, _sdfr.F16)):
        for shift in range(4):
            out = torch.full((n + 8,), -1.0, dtype=dt, device=dev)
            print(f"case edt alignment nx={nx} {dt} shift={shift}", flush=True)
            rc = lib.sdfr_edt(o.data_ptr(), nx, 11, 9, 16.0, out[shift:].data_ptr(), code, ws.data_ptr(), need,
                              torch.cuda.current_stream().cuda_stream)
            assert rc == 0
            got = out.cpu().numpy()
            assert np.array_equal(got[shift:shift + n].reshape(shape), _expected(occ, 16.0, nd))
            assert (got[:shift] == -1.0).all() and (got[shift + n:] == -1.0).all()


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
