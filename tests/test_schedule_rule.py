"""CPU: the schedule of a new shot goes by the arrays a step moves, not by what the shot records."""
import numpy as np
import pytest

from ela3d_amd import STORAGE_FP32, STORAGE_FP64
from helpers import small_cfg


# 144^3 and FP64 120^3: one field set fits the 256 MiB cache and two do not (two passes);
# 201^3: neither does, 33^3: both do (the whole-grid step)
@pytest.mark.parametrize("n,storage,sets", [(144, STORAGE_FP32, 1), (120, STORAGE_FP64, 1), (201, STORAGE_FP32, 2),
                                            (33, STORAGE_FP32, 2)])
def test_recording_more_does_not_change_the_schedule(n, storage, sets):
    cells = n ** 3 * (8 if storage == STORAGE_FP64 else 4)
    for nrec in (1, 256, 1000, 4000):
        rec = np.full((nrec, 3), n // 2, dtype=np.int32)
        cfg = small_cfg(nx=n, ny=n, nz=n, npml=10, storage=storage, nstep=4000, receivers=rec, energy_every=2)
        one, now = cfg.replace(block=128, zseg=2).plan()["device_bytes"], cfg.plan()["device_bytes"]
        assert now == one if sets == 1 else now >= one + 9 * cells, nrec
