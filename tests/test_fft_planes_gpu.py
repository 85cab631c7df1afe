"""Transforms whose (y, z) planes fit LDS take their y and z passes as one kernel:
planes of one wavefront, of several rounds of columns and rows, the largest of each
type, and the first ones past the limit, against numpy in FP64.

Tolerance: a length-N transform of unit roundoff u has a relative L2 error below
6 u log2 N (3u per butterfly sum and product, the twiddles' own rounding)."""
import math

import numpy as np
import pytest

from spkmod import spk

pytestmark = pytest.mark.gpu

PLANES = [(16, 32), (16, 512), (32, 64), (32, 256), (64, 64), (128, 32), (128, 64), (128, 128), (256, 32), (256, 64)]


@pytest.mark.parametrize("inplace", [True, False])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("ny,nz", PLANES)
def test_plane_transforms(ny, nz, prec, inplace):
    rdt, cdt, u = {"f64": (np.float64, np.complex128, 2.0 ** -53), "f32": (np.float32, np.complex64, 2.0 ** -24)}[prec]
    nx, nb, nzh = 16, 2, nz // 2 + 1
    tol = 6 * u * math.log2(nx * ny * nz)
    r = np.random.default_rng(ny * 1000 + nz).standard_normal((nb, nx, ny, nz)).astype(rdt)
    spec = np.fft.rfftn(r.astype(np.float64), axes=(1, 2, 3))
    pad = np.full((nb, nx, ny, 2 * nzh), 7.0, rdt)
    pad[..., :nz] = r
    ctx = spk.Ctx(0)
    plan = spk.FftPlan(ctx, nx, ny, nz, prec, nb)
    d_in = ctx.alloc(pad.nbytes)
    d_out = d_in if inplace else ctx.alloc(pad.nbytes)
    d_in.upload(pad)
    plan.r2c(d_in.ptr, d_out.ptr)
    got = d_out.download(cdt, spec.shape)
    assert np.linalg.norm(got - spec) <= tol * np.linalg.norm(spec)
    if not inplace:
        assert np.array_equal(d_in.download(rdt, pad.shape), pad)

    c = spec.astype(cdt)
    ref = np.fft.irfftn(c.astype(np.complex128), s=(nx, ny, nz), axes=(1, 2, 3))
    d_in.upload(c)
    plan.c2r(d_in.ptr, d_out.ptr)
    back = d_out.download(rdt, pad.shape)
    # the input's own rounding to the type is in ref too
    assert np.linalg.norm(back[..., :nz] - ref) <= tol * np.linalg.norm(ref)
    assert np.all(back[..., nz:] == 0)
    if not inplace:
        assert np.array_equal(d_in.download(cdt, c.shape), c)
    ctx.close()
