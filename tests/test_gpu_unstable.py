"""GPU: a shot that blows up under the whole-grid step is reported with the instability code, by
run() and by sync(), with graphs and without, wherever the non-finite value is first seen."""
import numpy as np
import pytest

from ela3d_amd import SRC_FORCE3, STORAGE_FP32, STORAGE_FP64, Ela3dError, Shot
from helpers import hetero_model, small_cfg

pytestmark = pytest.mark.gpu
E_UNSTABLE = -3


@pytest.mark.parametrize("storage,nstep", [(STORAGE_FP32, 600), (STORAGE_FP64, 2400)])
@pytest.mark.parametrize("seen_by", ["receivers", "energy", "source"])
@pytest.mark.parametrize("graph", [True, False])
def test_blow_up_has_its_code(gpu, storage, nstep, seen_by, graph):
    cfg = small_cfg(nx=40, ny=20, nz=18, npml=3, nstep=nstep, storage=storage, src_kind=SRC_FORCE3,
                    energy_every=3 if seen_by == "energy" else 0, use_graph=graph)
    if seen_by != "receivers":
        cfg = cfg.replace(receivers=np.zeros((0, 3), dtype=np.int32))
    model = hetero_model(cfg, seed=1)
    with Shot(cfg, *model) as s:
        assert s.info()["fused"] == 2
        s.run()  # a stable shot is not flagged
    cfg = cfg.replace(dt=4.0 * cfg.dt)
    with Shot(cfg, *model) as s:
        with pytest.raises(Ela3dError) as e:
            s.run()
        assert e.value.code == E_UNSTABLE
    with Shot(cfg, *model) as s:
        s.step(nstep)
        with pytest.raises(Ela3dError) as e:
            s.sync()
        assert e.value.code == E_UNSTABLE
