"""GPU: densities at the ends of the FP32 range.  A uniform density cancels from the velocities
of a stress source, so a run at any density has to give those of an ordinary one.  (The source's
size keeps the stresses, which go with the density, inside the normal range of FP32.)"""
import numpy as np
import pytest

from ela3d_amd import SRC_EXPLOSIVE, Config, Shot, homogeneous_model
from helpers import rel_l2

pytestmark = pytest.mark.gpu

STEPS = 40
TOL = STEPS * 4 * 2.0 ** -24  # four roundings of a velocity a step on either side


@pytest.mark.parametrize("shape", [dict(), dict(block=128, zseg=2)])  # whole-grid step, two passes
@pytest.mark.parametrize("rho,vp,factor", [(1e-38, 3000.0, 1e6), (2e-39, 3000.0, 1e6), (1e-39, 3000.0, 1e6),
                                           (1e38, 1e-3, 1e-4)])
def test_extreme_density(gpu, shape, rho, vp, factor):
    n = 33
    rec = np.asarray([(i, n // 2, n // 4) for i in range(0, n, 4)], dtype=np.int32)
    cfg = Config(nx=n, ny=n, nz=n, dt=4.8 / vp, nstep=STEPS, npoints_pml=6, f0=4e-3 * vp, vpml=vp, factor=factor,
                 src_kind=SRC_EXPLOSIVE, isrc=16, jsrc=16, ksrc=16, receivers=rec, **shape)
    out = []
    for density in (2000.0, rho):
        with Shot(cfg, *homogeneous_model(n, n, n, vp, vp / 1.7, density)) as s:
            assert s.info()["fused"] == (0 if shape else 2)
            s.run()
            out.append(s.seismograms())
    assert np.any(out[0]) and rel_l2(out[1], out[0]) <= TOL
