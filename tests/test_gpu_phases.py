"""GPU: stepping by phases a shot that was created with the whole-grid step."""
import numpy as np
import pytest

from ela3d_amd import SRC_EXPLOSIVE, STORAGE_FP32, STORAGE_FP64, Ela3dError, Shot, set_device_limit, set_tuning
from helpers import hetero_model, small_cfg

pytestmark = pytest.mark.gpu
E_INVALID = -1


def fields(shot):
    return [shot.snapshot(q) for q in range(27)]


#                    nx  ny  nz   what is cached for the grid once the shot is there
@pytest.mark.parametrize("dims,later", [
    ((46, 47, 28), dict(fused=1, tile=512)), ((47, 46, 28), dict(fused=1, tile=512, overlap=True)),
    ((48, 45, 28), dict(overlap=True)), ((45, 48, 28), dict(dbuf=True, merged=True)),
    ((44, 49, 28), dict(fused=2, tile=320))])
@pytest.mark.parametrize("storage", [STORAGE_FP32, STORAGE_FP64])
def test_grid_tuned_after_the_shot_was_created(gpu, dims, later, storage):
    """Phases go on in place with two passes whatever the grid was tuned to meanwhile, and the
    steps after them give the same fields bit for bit; a refused phase leaves the shot as it is."""
    cfg = small_cfg(nx=dims[0], ny=dims[1], nz=dims[2], nstep=23, storage=storage, src_kind=SRC_EXPLOSIVE,
                    energy_every=0)
    model = hetero_model(cfg, seed=6)
    with Shot(cfg.replace(block=128, zseg=2), *model) as s:
        s.run()
        ref, seis = fields(s), s.seismograms()
    with Shot(cfg, *model) as s:
        assert s.info()["fused"] == 2
        s.step(5)  # still running when the shot changes over
        set_tuning(cfg, block=128, zseg_interior=4, zseg_slab=2, **later)
        with pytest.raises(Ela3dError) as e:
            s.step_phase(2)
        assert e.value.code == E_INVALID and s.info()["fused"] == 2
        for _ in range(3):
            s.step_phase(0)
            s.step_phase(1)
        i = s.info()
        assert (i["fused"], i["dbuf"], i["overlap"], i["steps_done"]) == (0, 0, 0, 8)
        s.run()
        assert np.array_equal(s.seismograms(), seis)
        assert all(np.array_equal(x, y) for x, y in zip(ref, fields(s)))


def test_changes_over_with_graphs_in_flight(gpu):
    """A phase asked for while hundreds of replayed steps are queued runs after them."""
    cfg = small_cfg(nx=61, ny=43, nz=39, nstep=420, src_kind=SRC_EXPLOSIVE, energy_every=0)
    model = hetero_model(cfg, seed=9)
    with Shot(cfg.replace(block=128, zseg=2), *model) as s:
        s.run()
        ref, seis = fields(s), s.seismograms()
    with Shot(cfg, *model) as s:
        assert s.info()["fused"] == 2
        s.step(401)
        s.step_phase(0)
        s.step_phase(1)
        s.step(18)
        assert np.array_equal(s.seismograms(), seis)
        assert all(np.array_equal(x, y) for x, y in zip(ref, fields(s)))


@pytest.mark.parametrize("storage", [STORAGE_FP32, STORAGE_FP64])
@pytest.mark.parametrize("room", [True, False])
def test_second_field_set_is_given_back(gpu, storage, room):
    """A shot that steps by phases needs one field set and holds no more than that, except where
    there is no room to move it; either way it goes on bit for bit, checkpoints included."""
    cfg = small_cfg(nx=63, ny=31, nz=29, nstep=24, storage=storage, src_kind=SRC_EXPLOSIVE, energy_every=3)
    model = hetero_model(cfg, seed=10)
    with Shot(cfg.replace(block=128, zseg=2), *model) as s:
        one = s.info()["device_bytes"]
        s.run()
        ref, seis, trace = fields(s), s.seismograms(), s.source_trace()
    with Shot(cfg, *model) as s:
        two = s.info()["device_bytes"]
        assert s.info()["fused"] == 2 and two > one
        s.step(3)
        try:
            set_device_limit(0 if room else two + one - 1)
            s.step_phase(0)
            s.step_phase(1)
        finally:
            set_device_limit(0)
        assert s.info()["device_bytes"] == (one if room else two)
        s.run()
        assert np.array_equal(s.seismograms(), seis) and np.array_equal(s.source_trace(), trace)
        assert all(np.array_equal(x, y) for x, y in zip(ref, fields(s)))
