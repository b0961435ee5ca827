"""The model of a shot on its way in: the check names the first invalid cell whichever range
and block of the check it lies in, and padded planes arrive whole."""
import numpy as np
import pytest

import ela3d_amd
from ela3d_amd import Ela3dError, Shot
from helpers import hetero_model, homo, small_cfg


@pytest.mark.parametrize("which,value", [(0, np.inf), (0, np.nan), (0, -1.0), (1, 0.0), (1, np.nan), (1, np.inf),
                                         (2, 0.0), (2, np.inf), (2, np.nan), (2, -3.0)])
@pytest.mark.parametrize("cells", [(0, 1199), (4095, 4096), (4096, 1199999), (524288, 600000), (599999, 600001),
                                   (1199999, 1199999)])
def test_first_invalid_cell(cells, which, value):
    cfg = small_cfg(nx=120, ny=100, nz=100, nstep=2)
    model = [np.array(a, copy=True) for a in homo(cfg)]
    for q in cells:
        model[which].reshape(-1)[q] = value
    with pytest.raises(Ela3dError) as e:
        Shot(cfg, *model)
    assert e.value.code == -1 and f"model cell {cells[0]} " in str(e.value)


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(16, 12, 11), (17, 13, 9), (33, 31, 40)])  # planes of 3, 3.5 and 16 lines of 64
@pytest.mark.parametrize("storage", [0, 1, 2])
def test_model_and_fields_in_padded_planes(gpu, dims, storage):
    """A model that differs in every cell gives the step it should, and every field cell comes
    back as it was set (exactly where the storage holds it)."""
    nx, ny, nz = dims
    cfg = small_cfg(nx=nx, ny=ny, nz=nz, npml=2, nstep=4, storage=storage)
    model = hetero_model(cfg, seed=4)
    rng = np.random.default_rng(6)
    field = rng.integers(-8, 9, size=(nz, ny, nx)).astype(float)
    with Shot(cfg, *model) as s:
        s.set_field(3, field)
        assert np.array_equal(s.snapshot(3), field)
        s.set_field(3, np.zeros_like(field))
        s.run()
        a = [s.snapshot(q) for q in range(9)]
    flat = cfg.replace(block=64, zseg=1)
    with Shot(flat, *[np.asarray(m, dtype=np.float32).reshape(nz, ny, nx) for m in model]) as s:
        s.run()
        assert all(np.array_equal(x, s.snapshot(q)) for q, x in enumerate(a))
    assert ela3d_amd.device_count() > 0
