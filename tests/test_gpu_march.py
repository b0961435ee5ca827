"""GPU: the whole-grid fused step (march.hip) against the oracle after one step from a
random state, at the sizes where its cut can go wrong: rows that fill a wave exactly, one
column more and one less, several x chunks, last tiles of one row, segments of one plane
and of the whole grid, layers whose edges fall inside a lane's vector.  The bars are those
of test_gpu_parity.py: 2e-6 of each field's maximum in FP32 (both sides round every
operation; the GPU contracts to FMA), 1e-12 in FP64."""
import numpy as np
import pytest

import oracle
from ela3d_amd import (COMPAT_REFERENCE, SRC_EXPLOSIVE, SRC_FORCE3, STORAGE_FP32, STORAGE_FP64, Server, Shot, set_device_limit,
                       set_tuning)
from helpers import compare_state, hetero_model, max_rel, push_state, random_state, rel_l2, small_cfg
from test_march_index import checker, run as address_check  # noqa: F401

pytestmark = pytest.mark.gpu

TOL = {STORAGE_FP32: 2e-6, STORAGE_FP64: 1e-12}
DT = {STORAGE_FP32: np.float32, STORAGE_FP64: np.float64}

#       nx  ny  nz npml tile zseg
CASES = [(29, 23, 26, 4, 384, 5), (64, 17, 19, 3, 512, 1), (65, 17, 19, 3, 192, 4), (63, 15, 13, 2, 1024, 13),
         (126, 11, 14, 3, 320, 3), (127, 12, 11, 3, 512, 2), (188, 9, 17, 1, 256, 4), (189, 11, 12, 3, 512, 5),
         (257, 13, 10, 3, 320, 10), (30, 20, 15, 0, 384, 6), (200, 9, 9, 3, 256, 9), (13, 14, 15, 5, 256, 2)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("storage", [STORAGE_FP32, STORAGE_FP64])
@pytest.mark.parametrize("variant", ["clean", "reference", "surface"])
def test_march_one_step(gpu, checker, case, storage, variant):  # noqa: F811
    nx, ny, nz, npml, tile, zseg = case
    if storage == STORAGE_FP64:
        tile = min(tile, 512)
    fs = variant == "surface"
    r = address_check(checker, (nx, ny, nz, npml), storage, tile, zseg, fs=int(fs))
    assert r is not None and r[1] == 0
    print(f"march {case} storage {storage} {variant}", flush=True)
    cfg = small_cfg(nx=nx, ny=ny, nz=nz, npml=npml, storage=storage, nstep=3, free_surface=fs,
                    compat=COMPAT_REFERENCE if variant == "reference" else 0,
                    src_kind=SRC_EXPLOSIVE if fs else SRC_FORCE3)
    set_tuning(cfg, block=128, zseg_interior=zseg, zseg_slab=2, fused=2, tile=tile)
    model = hetero_model(cfg, seed=7)
    st = random_state(cfg, seed=11, dtype=DT[storage])
    with Shot(cfg, *model) as shot:
        assert shot.info()["fused"] == 2
        push_state(shot, st)
        shot.step(1)
        shot.sync()
        seis_o, en_o, st = oracle.run(cfg, model, 1, st=st, dtype=DT[storage])
        compare_state(shot, st, TOL[storage])
        seis_g, en_g = shot.seismograms()[:1], shot.energy()[:1]
    assert max_rel(seis_g, seis_o[:1]) <= TOL[storage]
    assert np.allclose(en_g, en_o[:1], rtol=10 * TOL[storage], atol=0)


@pytest.mark.parametrize("storage", [STORAGE_FP32, STORAGE_FP64])
def test_march_cut_does_not_matter(gpu, storage):
    """Over 40 steps every cut of the grid gives the same fields bit for bit (halo cells are
    recomputed with the arithmetic of their owners), and so does the two-pass schedule."""
    cfg = small_cfg(nx=131, ny=38, nz=33, nstep=40, storage=storage, energy_every=3)
    model = hetero_model(cfg, seed=5)
    out = []
    for tile, zseg, strips in ((384, 7, 0), (256, 33, 0), (512, 1, 3), (320, 4, 2)):
        set_tuning(cfg, block=128, zseg_interior=zseg, zseg_slab=2, fused=2, tile=tile, strips=strips)
        with Shot(cfg, *model) as shot:
            assert shot.info()["fused"] == 2
            shot.run()
            out.append([shot.seismograms(), shot.energy()] + [shot.snapshot(q) for q in range(27)])
    set_tuning(cfg, block=128, zseg_interior=4, zseg_slab=2)
    with Shot(cfg, *model) as shot:
        shot.run()
        two = [shot.seismograms(), shot.energy()] + [shot.snapshot(q) for q in range(27)]
    tol = 1e-6 if storage == STORAGE_FP32 else 1e-13
    for o in out[1:] + [two]:
        for q, (x, y) in enumerate(zip(out[0], o)):
            if q != 1:
                assert np.array_equal(x, y), q
            elif o is two:  # its kinetic terms are rounded once per cell, not once per half
                assert rel_l2(x, y) <= tol
            else:
                assert np.allclose(x, y, rtol=1e-12, atol=0)


def fields(shot):
    return [shot.snapshot(q) for q in range(27)]


@pytest.mark.parametrize("storage,dims,compat,fs", [
    (STORAGE_FP32, (37, 19, 23), 0, False), (STORAGE_FP32, (66, 41, 17), COMPAT_REFERENCE, False),
    (STORAGE_FP64, (43, 18, 21), 0, True), (STORAGE_FP64, (27, 33, 16), COMPAT_REFERENCE, True)])
def test_march_by_default(gpu, tmp_path, storage, dims, compat, fs):
    """A shot of an unmeasured grid takes the whole-grid step and gives the two-pass schedule's
    fields bit for bit; their checkpoints serve each other, after odd and even steps; stepping
    by phases goes on in place; and where only one set fits, it takes two passes."""
    nx, ny, nz = dims
    cfg = small_cfg(nx=nx, ny=ny, nz=nz, npml=4, nstep=31, storage=storage, compat=compat, free_surface=fs,
                    src_kind=SRC_EXPLOSIVE, energy_every=4)
    model = hetero_model(cfg, seed=3)
    two_pass = cfg.replace(block=128, zseg=2)  # a given shape: two passes in place
    ck = [str(tmp_path / f"{n}.ck") for n in ("one", "two")]
    with Shot(two_pass, *model) as s:
        assert s.info()["fused"] == 0 and s.info()["dbuf"] == 0
        s.step(12)
        s.checkpoint(ck[0])
        one_bytes = s.info()["device_bytes"]
        s.run()
        ref, seis, en = fields(s), s.seismograms(), s.energy()
    tol = 1e-6 if storage == STORAGE_FP32 else 1e-13  # energy terms: rounding of the cell's arithmetic

    def same(s):
        s.run()
        assert all(np.array_equal(x, y) for x, y in zip(ref, fields(s)))
        assert np.array_equal(s.seismograms(), seis) and rel_l2(s.energy(), en) <= tol

    with Shot(cfg, *model) as s:
        assert s.info()["fused"] == 2 and cfg.plan()["device_bytes"] == s.info()["device_bytes"]
        s.step(7)
        s.checkpoint(ck[1])
        same(s)
    with Shot(cfg, *model) as s:
        s.step(3)
        s.restore(ck[0])
        same(s)
    with Shot(two_pass, *model) as s:
        s.restore(ck[1])
        same(s)
    with Shot(cfg, *model) as s:
        s.step(5)
        for _ in range(3):
            s.step_phase(0)
            s.step_phase(1)
        assert s.info()["steps_done"] == 8 and s.info()["fused"] == 0
        same(s)
    try:
        set_device_limit(one_bytes)
        with Shot(cfg, *model) as s:
            assert s.info()["dbuf"] == 0
            same(s)
    finally:
        set_device_limit(0)


@pytest.mark.parametrize("storage,energy_every", [(STORAGE_FP32, 0), (STORAGE_FP32, 5), (STORAGE_FP64, 3), (1, 0)])
def test_step_runs(gpu, storage, energy_every):
    """Steps replayed in runs of every length and phase, with eager steps and synchronizations
    between the replays, leave what eager launches leave: fields, samples and energies."""
    cfg = small_cfg(nx=34, ny=21, nz=18, npml=4, nstep=150, storage=storage, src_kind=SRC_EXPLOSIVE,
                    energy_every=energy_every)
    model = hetero_model(cfg, seed=8)
    with Shot(cfg.replace(use_graph=False), *model) as s:
        s.run()
        ref = [s.seismograms(), s.energy(), s.source_trace()] + fields(s)
    with Shot(cfg, *model) as s:
        for n in (1, 2, 2, 3, 16, 17, 17, 31, 2, 5, 5, 33):
            s.step(n)
            if n != 2:
                s.sync()
            s.profile(1) if n == 3 else None
        s.run()
        got = [s.seismograms(), s.energy(), s.source_trace()] + fields(s)
    assert all(np.array_equal(x, y) for x, y in zip(ref, got))


def test_turned_passes(gpu):
    """Where every other pass walks the grid backwards (more than the last-level cache, not more
    than four times that), one launch a step and two passes still agree to the bit."""
    cfg = small_cfg(nx=300, ny=110, nz=150, npml=6, nstep=7, src_kind=SRC_EXPLOSIVE, energy_every=2)
    model = hetero_model(cfg, seed=2)
    with Shot(cfg, *model) as s:
        assert s.info()["fused"] == 2
        s.run()
        a, en, seis = fields(s), s.energy(), s.seismograms()
    with Shot(cfg.replace(block=128, zseg=2), *model) as s:
        assert s.info()["fused"] == 0
        s.run()
        for q, x in enumerate(a):
            assert np.array_equal(x, s.snapshot(q)), q
        assert np.array_equal(s.seismograms(), seis) and rel_l2(s.energy(), en) <= 1e-6


@pytest.mark.parametrize("storage", [STORAGE_FP32, STORAGE_FP64])
@pytest.mark.parametrize("kind", [0, 1, 2, 3])
@pytest.mark.parametrize("cell", [(0.5, 0.5, 0.5), (0.1, 0.9, 0.2)])
def test_recording(gpu, storage, kind, cell):
    """What ends a step is recorded by the launch after it, or at a run's end by one of its own:
    samples (a receiver on the source cell, more receivers than threads), energies, source trace
    are those of the two-pass tail, whatever the runs; steps past the wavelet's end too."""
    cfg = small_cfg(nx=67, ny=19, nz=17, npml=3, nstep=47, storage=storage, src_kind=kind, energy_every=3)
    src = [int(f * n) for f, n in zip(cell, (67, 19, 17))]
    rng = np.random.default_rng(1)
    rec = np.vstack([[src], rng.integers(1, (66, 18, 16), size=(600, 3))]).astype(np.int32)
    cfg = cfg.replace(isrc=src[0], jsrc=src[1], ksrc=src[2], receivers=rec, sample_every=2)
    model = hetero_model(cfg, seed=12)
    with Shot(cfg.replace(block=128, zseg=2), *model) as s:
        s.run()
        ref, seis, en, tr = fields(s), s.seismograms(), s.energy(), s.source_trace()
    assert np.any(seis[:, 0])
    for runs, graph in (((47,), True), ((1, 2, 16, 16, 12), True), ((5, 42), False)):
        with Shot(cfg.replace(use_graph=graph), *model) as s:
            assert s.info()["fused"] == 2
            for n in runs:
                s.step(n)
            s.sync()
            assert all(np.array_equal(x, y) for x, y in zip(ref, fields(s)))
            assert np.array_equal(s.seismograms(), seis) and np.array_equal(s.source_trace(), tr)
            assert rel_l2(s.energy(), en) <= (1e-6 if storage == STORAGE_FP32 else 1e-13)


def test_recording_flags_a_blow_up(gpu):
    cfg = small_cfg(nx=40, ny=20, nz=18, npml=3, nstep=600, src_kind=SRC_FORCE3)
    cfg = cfg.replace(dt=4.0 * cfg.dt)
    with Shot(cfg, *hetero_model(cfg, seed=1)) as s:
        assert s.info()["fused"] == 2
        with pytest.raises(Exception):
            s.run()


def test_pinned_whole_grid_step_gives_way(gpu):
    """A measured or given whole-grid shape steps by phases in place too, and a shot of that grid
    that has to update in place (served in a batch, or without room for two sets) takes two passes."""
    cfg = small_cfg(nx=52, ny=22, nz=20, npml=3, nstep=24, src_kind=SRC_EXPLOSIVE, energy_every=0)
    model = hetero_model(cfg, seed=4)
    set_tuning(cfg, block=128, zseg_interior=2, zseg_slab=2, fused=2, tile=320)
    with Shot(cfg, *model) as s:
        assert s.info()["fused"] == 2 and s.info()["tile"] == 320
        s.step(3)
        s.step_phase(0)
        s.step_phase(1)
        assert s.info()["fused"] == 0 and s.info()["steps_done"] == 4
        s.run()
        seis = s.seismograms()
    with Server(max_active=3) as srv:
        tickets = [srv.submit(cfg, *model) for _ in range(3)]
        out = [srv.result(t) for t in tickets]
        assert srv.stats()["batched"] == 3
    assert all(np.array_equal(o[0], seis) for o in out)
