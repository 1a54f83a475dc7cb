"""GPU tests of the level loop's products (several levels of a column per
wavefront, row weights 64 rows at a time): ensemble widths of each kernel,
odd level counts, row lists from empty to several blocks of 64 with every
remainder, in the bucket order and in column order, against the oracle.

FP64 at the repository's 1e-10; FP32 products at its increment bound, 1e-5
RMS of the FP64 increment per call."""
import copy

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


@pytest.mark.parametrize("schedule", [1, 0])
@pytest.mark.parametrize("k,nz,cube_nz,n_obs", [
    (8, 5, 1, 30), (31, 4, 1, 400), (32, 7, 2, 2500), (33, 3, 1, 400), (64, 5, 2, 900),
    (65, 3, 1, 300), (128, 2, 1, 700), (20, 5, 3, 9000)])
def test_level_products(k, nz, cube_nz, n_obs, schedule):
    import orc
    from dida_letkf import engine, synth
    inst = synth.generate("c1", seed=k + n_obs, k=k, nlat=6, nlon=11, nz=nz, n_obs=n_obs,
                          local_dist=700.0)
    inst.cfg.vert_dist = 1.1
    inst.cfg.cube_nz = cube_nz
    ref = orc.letkf_compute(inst, want_trans=True)
    full = ref["xa"] + ref["axa"][..., None]
    inc = np.sqrt(np.mean((full - inst.xb - inst.axb[..., None]) ** 2))
    for prec in (0, 1):
        cfg = copy.copy(inst.cfg)
        cfg.precision = prec
        with engine.LetkfEngine(cfg, keep_transforms=True) as eng:
            eng.set_option(engine.OPT_SCHEDULE, schedule)
            eng.set_grid(inst.grid_lat, inst.grid_lon)
            eng.set_obs(inst.obs)
            xa, axa, rc = eng.letkf_compute(inst.xb, inst.axb)
            _, _, nobsl = eng.get_transforms()
        assert rc == 0 and np.array_equal(nobsl, ref["nobsl"])
        got = xa + axa[..., None]
        if prec == 0:
            err = np.abs(got - full).max() / np.abs(full).max()
            print(k, nz, n_obs, "p", nobsl.min(), nobsl.max(), "fp64", err, flush=True)
            assert err < 1e-10
        else:
            err = np.sqrt(np.mean((got - full) ** 2)) / inc
            print(k, nz, n_obs, "fp32 increment", err, flush=True)
            assert err < 1e-5


@pytest.mark.parametrize("k,nz,vert,n_obs", [
    (32, 9, 0.3, 6000), (20, 6, 0.26, 150), (64, 5, 0.5, 4000), (40, 7, 0.4, 3000),
    (100, 4, 0.3, 2500), (32, 12, 40.0, 3000)])
def test_level_products_support(k, nz, vert, n_obs):
    """Supports that leave most rows of a column without weight, some levels
    without any row, and one that covers every row; then the same set with one
    value that is not finite: every analysis whose row list holds that row
    keeps its background at every level, as where each row's product enters."""
    import orc
    from dida_letkf import engine, synth
    inst = synth.generate("c1", seed=k + n_obs, k=k, nlat=6, nlon=11, nz=nz, n_obs=n_obs,
                          local_dist=900.0)
    inst.cfg.vert_dist = vert
    inst.cfg.cube_nz = 1
    ref = orc.letkf_compute(inst, want_trans=True)
    full = ref["xa"] + ref["axa"][..., None]
    inc = np.sqrt(np.mean((full - inst.xb - inst.axb[..., None]) ** 2))
    # the row nearest to a column in the middle of the grid
    la, lo = np.deg2rad(inst.grid_lat[3]), np.deg2rad(inst.grid_lon[5])
    sla, slo = np.deg2rad(inst.obs.site_lat), np.deg2rad(inst.obs.site_lon)
    site = np.argmax(np.sin(la) * np.sin(sla) + np.cos(la) * np.cos(sla) * np.cos(lo - slo))
    row = int(inst.obs.site_row_ptr[site])
    for prec in (0, 1):
        cfg = copy.copy(inst.cfg)
        cfg.precision = prec
        with engine.LetkfEngine(cfg, keep_transforms=True) as eng:
            eng.set_grid(inst.grid_lat, inst.grid_lon)
            eng.set_obs(inst.obs)
            xa, axa, rc = eng.letkf_compute(inst.xb, inst.axb)
            got = xa + axa[..., None]
            assert rc == 0
            if prec == 0:
                assert np.abs(got - full).max() < 1e-10 * np.abs(full).max()
            else:
                assert np.sqrt(np.mean((got - full) ** 2)) < 1e-5 * inc
            # rc counts whole columns
            for field in ("yb", "dep"):
                obs = copy.copy(inst.obs)
                a = np.array(getattr(obs, field), copy=True)
                a.reshape(a.shape[0], -1)[row, 0] = np.nan
                setattr(obs, field, a)
                eng.set_obs(obs)
                xa2, axa2, rc2 = eng.letkf_compute(inst.xb, inst.axb)
                assert np.isfinite(xa2).all() and np.isfinite(axa2).all()
                assert rc2 > 0 and rc2 % nz == 0


@pytest.mark.parametrize("k,nz,cube_nz,tile", [(20, 4, 4, 0), (33, 3, 32, 2), (100, 2, 2, 0),
                                               (64, 5, 5, 2)])
def test_level_products_one_chunk(k, nz, cube_nz, tile):
    """A column that is one chunk of levels is localised in the vertical too (in
    each precision, with the products kernel that tiles horizontal loops asked
    for or not)."""
    import orc
    from dida_letkf import engine, synth
    inst = synth.generate("c1", seed=k, k=k, nlat=6, nlon=11, nz=nz, n_obs=900, local_dist=700.0)
    inst.cfg.vert_dist = 0.6
    inst.cfg.cube_nz = cube_nz
    ref = orc.letkf_compute(inst, want_trans=True)
    full = ref["xa"] + ref["axa"][..., None]
    inc = np.sqrt(np.mean((full - inst.xb - inst.axb[..., None]) ** 2))
    for prec in (0, 1, 2):
        got = engine.letkf_compute_nooverlap(inst, precision=prec, products_kernel=tile)
        assert got["n_flagged"] == 0
        got = got["xa"] + got["axa"][..., None]
        if prec == 0:
            assert np.abs(got - full).max() < 1e-10 * np.abs(full).max()
        else:
            assert np.sqrt(np.mean((got - full) ** 2)) < 1e-5 * inc
