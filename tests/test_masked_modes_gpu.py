"""Modes outside the 2/3 mask: their products are never formed (ProdLay), while
the state there stays and evolves.  States with energy in every mode, on grids
where the mask's edges fall differently in rows, tiles and pitches, against the
FP64 oracle; and a NaN, which reaches every mode on every path."""
import numpy as np
import pytest

import pyoracle as orc
from physics_cases import relerr
from spkmod import spk

pytestmark = pytest.mark.gpu

T = 2 * np.pi
GRIDS = [(32, 16, 4), (32, 4, 32), (64, 8, 2), (32, 32, 16), (64, 2, 8), (32, 64, 64), (128, 16, 128), (32, 128, 2)]
PHYS = {"hd": dict(), "mhd": dict(mhd=1, nu_m=3e-3), "open": dict(mhd=1, nu_m=3e-3, antialiasing=0),
        "flat": dict(mhd=1, nu_m=3e-3, with2d=1), "bouss": dict(boussinesq=1, nu_th=2e-3),
        "rkl": dict(mhd=1, nu_m=3e-3, boussinesq=1, stratification=1, strat_direction=2, N2=0.3, OmegaT2=0.5, nu_th=2e-3,
                    anisotropic_diffusion=1, reynolds_ani=50.0, supertimestepping=1, sts_mask=1 << 6, safety_sts=20),
        "strat": dict(mhd=1, nu_m=3e-3, boussinesq=1, stratification=1, strat_direction=1, N2=0.4, nu_th=2e-3)}


@pytest.fixture(scope="module")
def ctx():
    c = spk.Ctx(0)
    yield c
    c.close()


def params(grid, phys):
    return dict(dict(nx=grid[0], ny=grid[1], nz=grid[2], incompressible=1, lx=T, ly=T, lz=T, nu=2e-3, cfl=0.3,
                     t_final=1e9, toutput_flow=1e9), **PHYS[phys])


def full_state(p, seed):
    """Real noise in every field, rms 0.3: every mode of its spectrum is filled."""
    nf = 3 + 3 * p.get("mhd", 0) + p.get("boussinesq", 0)
    r = 0.3 * np.random.default_rng(seed).standard_normal((nf, p["nx"], p["ny"], p["nz"]))
    if p.get("anisotropic_diffusion"):
        r[3:6] = 0.1 * r[3:6] + np.array([1.0, 0.5, -0.7])[:, None, None, None]  # B nowhere 0
    return np.fft.rfftn(r, axes=(1, 2, 3))


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("phys", sorted(PHYS))
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "%dx%dx%d" % g)
def test_filled_spectrum_against_oracle(ctx, grid, phys, prec):
    # tolerances of test_solver_gpu.py
    p = params(grid, phys)
    u0 = full_state(p, 3)
    sim = orc.Sim(**p)
    sim.set_fields(u0)
    sim.complex2real()
    sim.compute_dfield(0)
    rhs = sim.dfields.copy()
    sim.set_fields(u0)
    sim.main_loop(3)
    sol = spk.Solver(ctx, prec, **p)
    sol.set_fields(u0)
    sol.compute_dfield()
    assert relerr(sol.get_dfields(), rhs) < {"f64": 1e-11, "f32": 3e-5}[prec]
    for fused in (0, 2):
        for points in ((4, 8) if fused else (0,)):
            sol.set_fused(fused)
            sol.set_fused_points(points)
            sol.set_fields(u0)
            sol.set_time(0.0)
            sol.main_loop(3)
            e = relerr(sol.get_fields(), sim.fields)
            assert e < {"f64": 1e-10, "f32": 2e-4}[prec], (fused, points, e)
    sol.destroy()


@pytest.mark.parametrize("grid", [(32, 16, 16), (64, 64, 2), (32, 64, 64)], ids=lambda g: "%dx%dx%d" % g)
def test_nan_reaches_every_mode_of_theta(ctx, grid):
    p = params(grid, "rkl")
    u0 = full_state(p, 5)
    u0[6, 1, 1, 0] = np.nan
    sol = spk.Solver(ctx, "f64", **p)
    sol.set_fields(full_state(p, 5))
    sol.compute_dt()
    sol.set_fields(u0)
    sol.rkl2_cycle()
    assert np.all(np.isnan(sol.get_fields()[6, 1:, :, :].real))
    sol.destroy()


@pytest.mark.parametrize("fused", [0, 2])
@pytest.mark.parametrize("grid", [(32, 16, 16), (64, 64, 2), (32, 64, 64)], ids=lambda g: "%dx%dx%d" % g)
def test_nan_reaches_every_mode(ctx, grid, fused):
    p = params(grid, "mhd")
    u0 = full_state(p, 4)
    u0[1, 1, 1, 0] = np.nan
    sol = spk.Solver(ctx, "f64", **p)
    sol.set_fused(fused)
    sol.set_fields(u0)
    sol.compute_dfield()
    assert np.all(np.isnan(sol.get_dfields()[:, 1:, :, :].real))
    sol.main_loop(1)
    assert np.all(np.isnan(sol.get_fields()[:, 1:, :, :].real))
    sol.destroy()
