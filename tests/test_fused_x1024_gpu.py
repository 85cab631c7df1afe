"""The longest x lines of the fused kernel: at 4 points per thread one column a block up
to 256 blocks, two beyond; and at 8 points per thread.
Against the FP64 oracle (states and tolerances of test_masked_modes_gpu.py)."""
import numpy as np
import pytest

import pyoracle as orc
from physics_cases import relerr
from spkmod import spk
from test_masked_modes_gpu import full_state, params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("points", [4, 8])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("phys", ["mhd", "strat", "bouss"])
@pytest.mark.parametrize("ny,nz", [(2, 4), (2, 8), (128, 2), (32, 16), (2, 512)])
def test_1024_points(ny, nz, phys, prec, points):
    p = params((1024, ny, nz), phys)
    u0 = full_state(p, 9)
    sim = orc.Sim(**p)
    sim.set_fields(u0)
    sim.main_loop(2)
    ctx = spk.Ctx(0)
    sol = spk.Solver(ctx, prec, **p)
    sol.set_fused(2)
    sol.set_fused_points(points)
    sol.set_fields(u0)
    sol.main_loop(2)
    assert relerr(sol.get_fields(), sim.fields) < {"f64": 1e-10, "f32": 2e-4}[prec]
    sol.destroy()
    ctx.close()
