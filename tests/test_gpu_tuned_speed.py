"""GPU: a grid that was tuned is not slower than one that was not."""
import time

import pytest

from ela3d_amd import Config, Shot, autotune, homogeneous_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [144, 160])
def test_tuning_a_cached_grid_does_not_slow_it(gpu, n):
    """One field set of these grids fits the last-level cache and two do not: two passes in place
    take 12 % less time than the whole-grid step.  Half of that is the margin between the best
    of seven rounds of each, taken in turn (they differ by about 1 % from run to run)."""
    cfg = Config(nx=n, ny=n + 1, nz=n, dt=1e-3, nstep=20000)
    model = homogeneous_model(n, n + 1, n)
    with Shot(cfg, *model) as plain:
        assert plain.info()["fused"] == 0
        autotune(cfg, model)
        with Shot(cfg, *model) as tuned:
            best = {}
            for r in range(8):
                for s in (plain, tuned):
                    t = time.perf_counter()
                    s.step(200)
                    s.sync()
                    if r:  # the first round warms up
                        best[s] = min(best.get(s, 1e9), time.perf_counter() - t)
            print("us a step, plain and tuned:", [round(b / 200 * 1e6, 1) for b in best.values()], tuned.info())
            assert best[tuned] <= 1.06 * best[plain]


@pytest.mark.parametrize("n,every", [(81, 1), (101, 0), (101, 10), (128, 0)])
def test_tuning_a_small_grid_does_not_slow_it(gpu, n, every):
    """The whole-grid step takes 10 to 20 % less time than two passes here; margin as above."""
    cfg = Config(nx=n, ny=n + 1, nz=n + 2, dt=1e-3, nstep=20000, energy_every=every)
    model = homogeneous_model(n, n + 1, n + 2)
    with Shot(cfg, *model) as plain:
        assert plain.info()["fused"] == 2
        autotune(cfg, model)
        with Shot(cfg, *model) as tuned:
            best = {}
            for r in range(8):
                for s in (plain, tuned):
                    t = time.perf_counter()
                    s.step(320)
                    s.sync()
                    if r:
                        best[s] = min(best.get(s, 1e9), time.perf_counter() - t)
            print("us a step, plain and tuned:", [round(b / 320 * 1e6, 1) for b in best.values()], tuned.info())
            assert best[tuned] <= 1.06 * best[plain]
