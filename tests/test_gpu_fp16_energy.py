"""GPU: FP16 storage keeps its energy sums to the rounding of its FP32 cell terms, which are
contracted as its updates are.  The reference values are of the version from which the FP16
results are to stay the same; a different contraction of the terms moves them by 1e-9 to 1e-7.
The terms being equal, only the order of their FP64 sum may differ: 38,000 terms, 38,000 x 2^-53."""
import numpy as np
import pytest

from ela3d_amd import SRC_EXPLOSIVE, STORAGE_FP16, Shot
from helpers import hetero_model, small_cfg

pytestmark = pytest.mark.gpu

ENERGY = [["0x1.6bec3437ae206p+17", "0x1.76c6736694074p+19"], ["0x1.41b8d08cb88f7p+27", "0x1.f648932d09bf0p+29"],
          ["0x1.e2972472f1867p+33", "0x1.67ad1ea0d09f5p+37"], ["0x1.4b5b400f4edf1p+36", "0x1.e890ca1591167p+41"],
          ["0x1.8604c54a70239p+36", "0x1.62eef7bf920f2p+42"]]


def test_energy_terms(gpu):
    cfg = small_cfg(nx=43, ny=31, nz=29, storage=STORAGE_FP16, src_kind=SRC_EXPLOSIVE, factor=1e2, nstep=60,
                    energy_every=12, block=128, zseg=2)
    with Shot(cfg, *hetero_model(cfg, seed=17)) as s:
        s.run()
        en = s.energy()
    ref = np.array([[float.fromhex(v) for v in row] for row in ENERGY])
    assert np.max(np.abs(en / ref - 1.0)) <= 38000 * 2.0 ** -53
