"""GPU: advances cut into captured runs give what eager launches give, for energy cadences and
call lengths whose runs differ from call to call (more of them than a shot keeps graphs of)."""
import numpy as np
import pytest

from ela3d_amd import SRC_EXPLOSIVE, STORAGE_FP16, STORAGE_FP32, Shot
from helpers import hetero_model, small_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [STORAGE_FP32, STORAGE_FP16])
@pytest.mark.parametrize("every,n", [(7, 50), (13, 50), (17, 21), (25, 21), (40, 33)])
def test_cadences(gpu, storage, every, n):
    cfg = small_cfg(nx=26, ny=21, nz=18, npml=3, nstep=1400, storage=storage, src_kind=SRC_EXPLOSIVE,
                    factor=1e3, energy_every=every)
    model = hetero_model(cfg, seed=13)
    out = []
    for graph in (False, True):
        with Shot(cfg.replace(use_graph=graph), *model) as s:
            for q in range(1400 // n):
                s.step(n)
                if q % 7 == 3:
                    s.sync()
            s.run()
            out.append([s.seismograms(), s.energy(), s.source_trace()] + [s.snapshot(q) for q in range(27)])
    assert out[0][1].shape[0] == 1400 // every and np.all(out[0][1] > 0)
    assert all(np.array_equal(x, y) for x, y in zip(*out))
