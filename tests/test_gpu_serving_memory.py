"""GPU: served shots whose whole-grid step wants a second field set, where memory is short."""
import numpy as np
import pytest

from ela3d_amd import Config, Server, Shot, homogeneous_model, set_device_limit

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def job(gpu):
    """(Config, model, seismograms alone, bytes with one set, bytes with two): long enough to be
    still running when the next one is submitted, with energies, so that it is not batched."""
    n = 49
    rec = np.asarray([(i, 20, 30) for i in range(4, 45, 5)], dtype=np.int32)
    cfg = Config(nx=n, ny=n, nz=n, dt=1e-3, nstep=6000, npoints_pml=6, f0=15.0, isrc=22, jsrc=25, ksrc=27,
                 receivers=rec, energy_every=10)
    model = homogeneous_model(n, n, n)
    with Shot(cfg, *model) as s:
        assert s.info()["fused"] == 2
        s.run()
        seis, two = s.seismograms(), s.info()["device_bytes"]
    one = cfg.replace(block=128, zseg=2).plan()["device_bytes"]
    assert one < two and np.any(seis)
    return cfg, model, seis, one, two


def test_device_without_room_for_the_second_set(job):
    """As ela3d_create does, the server then runs the shot with two passes in place."""
    cfg, model, seis, one, two = job
    try:
        with Server(batch_cells=0, hbm_budget_bytes=1 << 30) as srv:
            set_device_limit(one + 4096)
            info = srv.wait(srv.submit(cfg, *model))
            assert info["status"] == 0 and info["device_bytes"] == one
            assert np.array_equal(srv.result(info["ticket"])[0], seis)
    finally:
        set_device_limit(0)
