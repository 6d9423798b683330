"""SDF bakes from several threads at once, each on its own stream, of grids whose tiles want
different amounts of LDS of the same kernels: the kernels' LDS attribute is one for the process,
so a call must not set it to its own size while another call's launch is on its way."""
from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

from oracle import edt
from surfgym import vision

pytestmark = pytest.mark.gpu

# y lines whose tiles take 88, 120 and 160 KB in one instantiation, z lines with 121 and 156 KB
# in another
SHAPES = [(2, 4500, 40), (2, 6144, 40), (2, 8192, 16), (770, 3, 70), (1000, 3, 70)]


def test_threads_with_different_tiles(dev):
    rng = np.random.default_rng(11)
    grids = [(rng.random(s) < 0.01).astype(np.uint8) for s in SHAPES]
    want = [edt.bake(o, 16.0).astype(np.float32) for o in grids]
    occ = [torch.as_tensor(o, device=dev) for o in grids]
    torch.cuda.synchronize()
    failed = []

    def work(i):
        try:
            stream = torch.cuda.Stream(dev)
            with torch.cuda.stream(stream):
                for _ in range(20):
                    got = vision.sdf_from_occupancy(occ[i], 16.0, device=dev, dtype=torch.float32)
                stream.synchronize()
                if not np.array_equal(got.cpu().numpy(), want[i]):
                    failed.append((SHAPES[i], "values"))
        except Exception as e:  # noqa: BLE001
            failed.append((SHAPES[i], repr(e)))

    print(f"case edt threads {SHAPES}", flush=True)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(SHAPES))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
