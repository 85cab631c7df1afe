"""A NaN reaches every mode through tiles that hold no product: each field group of the
fused back end (velocity, magnetic, temperature alone and coupled by stratification),
both precisions and tile widths, the RKL2 flux, and batched boxes, where it stays in
its own box.  The grids have whole tiles outside the 2/3 mask at every tile width."""
import numpy as np
import pytest

from spkmod import spk
from test_masked_modes_gpu import full_state, params

pytestmark = pytest.mark.gpu

GRIDS = [(32, 64, 16), (32, 256, 2)]
# seeded field -> fields that a step makes NaN: without stratification u does not see theta
SPREAD = {"bouss": {0: (0, 1, 2, 3), 3: (3,)}, "strat": {1: range(7), 4: range(7), 6: range(7)}}


@pytest.fixture(scope="module")
def ctx():
    c = spk.Ctx(0)
    yield c
    c.close()


def is_nan(c):
    return np.isnan(c.real) & np.isnan(c.imag)


@pytest.mark.parametrize("back", ["unfused", 4, 8])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("phys,field", [(p, f) for p in SPREAD for f in SPREAD[p]])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "%dx%dx%d" % g)
def test_nan_reaches_every_mode_of_each_group(ctx, grid, phys, field, prec, back):
    p = params(grid, phys)
    u0 = full_state(p, 6)
    u0[field, 1, 1, 0] = np.nan
    sol = spk.Solver(ctx, prec, **p)
    sol.set_fused(0 if back == "unfused" else 2)
    if back != "unfused":
        sol.set_fused_points(back)
    sol.set_fields(u0)
    sol.main_loop(1)
    got = sol.get_fields()
    sol.destroy()
    for f in range(len(got)):
        if f in SPREAD[phys][field]:
            assert np.all(is_nan(got[f, 1:])), f
        else:
            assert np.all(np.isfinite(got[f])), f


@pytest.mark.parametrize("on_device", [False, True])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "%dx%dx%d" % g)
def test_nan_reaches_every_mode_of_the_conduction(ctx, grid, prec, on_device):
    p = params(grid, "rkl")
    u0 = full_state(p, 7)
    sol = spk.Solver(ctx, prec, **p)
    if on_device:
        sol.set_rkl_device(True)
    sol.set_fields(u0)
    sol.compute_dt()
    u0[4, 1, 1, 0] = np.nan  # in B: the flux alone
    sol.set_fields(u0)
    sol.rkl2_cycle()
    got = sol.get_fields()
    sol.destroy()
    assert np.all(is_nan(got[6, 1:]))
    keep = [0, 1, 2, 3, 5]
    assert np.array_equal(got[keep], u0[keep])


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_nan_stays_in_its_box(prec):
    bx = [params(g, ph) for g, ph in ((GRIDS[0], "strat"), (GRIDS[0], "rkl"), (GRIDS[1], "rkl")) for _ in range(3)]
    states = [full_state(p, 20 + i) for i, p in enumerate(bx)]
    ens = spk.Ensemble(bx, prec, lanes=2)
    assert ens.layout()["batches"] == 3
    result = []
    for bad in (None, (1, 1), (4, 4), (8, 6)):  # (box, field)
        for i, st in enumerate(states):
            st = st.copy()
            if bad and bad[0] == i:
                st[bad[1], 1, 1, 0] = np.nan
            ens.set_fields(i, st)
            ens.boxes[i].set_time(0.0)
        ens.run(2)
        result.append([ens.get_fields(i) for i in range(len(bx))])
        for i in range(len(bx)):
            if bad and bad[0] == i:
                assert np.all(is_nan(result[-1][i][:, 1:])), (bad, i)
            else:
                assert np.array_equal(result[-1][i], result[0][i]), (bad, i)
    ens.destroy()
