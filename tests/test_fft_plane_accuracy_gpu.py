"""Transforms that make their y and z passes in one kernel are as accurate as the
three passes one by one (FftPlan.one_pass), against numpy in the next wider
precision.

Tolerance: the two orders of operations round differently; the ratio of their relative
L2 errors over n values scatters by about n^-1/2 (both are sums of n squares).  0.5%
is over three times that at every shape here."""
import numpy as np
import pytest
from scipy import fft

from spkmod import spk

pytestmark = pytest.mark.gpu

PLANES = [(16, 32), (16, 64), (16, 128), (16, 256), (16, 512), (32, 128), (32, 256), (64, 64), (64, 128), (128, 32)]


def err(got, ref):
    d = got.astype(ref.dtype) - ref
    return float(np.sqrt(np.sum(d.real ** 2 + d.imag ** 2) / np.sum(ref.real ** 2 + ref.imag ** 2)))


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("ny,nz", PLANES)
def test_plane_kernel_is_as_accurate_as_the_passes(ny, nz, prec):
    rdt, cdt, wide = {"f64": (np.float64, np.complex128, np.longdouble), "f32": (np.float32, np.complex64, np.float64)}[prec]
    nb, nzh = 4, nz // 2 + 1
    nx = 2 ** 17 // (ny * nz) * 2
    shape = (nb, nx, ny, nzh)
    r = np.random.default_rng(ny + nz).standard_normal((nb, nx, ny, nz)).astype(rdt)
    ref = fft.rfftn(r.astype(wide), axes=(1, 2, 3))
    pad = np.zeros(shape[:3] + (2 * nzh,), rdt)
    pad[..., :nz] = r
    ctx = spk.Ctx(0)
    plan = spk.FftPlan(ctx, nx, ny, nz, prec, nb)
    a, b = ctx.alloc(pad.nbytes), ctx.alloc(pad.nbytes)
    a.upload(pad)
    plan.r2c(a.ptr, b.ptr)
    fused = err(b.download(cdt, shape), ref)
    plan.one_pass(2, -1, a.ptr, b.ptr)
    plan.one_pass(1, -1, b.ptr, b.ptr)
    plan.one_pass(0, -1, b.ptr, b.ptr)
    assert fused <= 1.005 * err(b.download(cdt, shape), ref)

    c = ref.astype(cdt)
    n = nx * ny * nz  # one_pass leaves 1/N out
    ref = fft.irfftn(c.astype(ref.dtype), s=(nx, ny, nz), axes=(1, 2, 3))
    a.upload(c)
    plan.c2r(a.ptr, b.ptr)
    fused = err(b.download(rdt, pad.shape)[..., :nz], ref)
    plan.one_pass(0, 1, a.ptr, b.ptr)
    plan.one_pass(1, 1, b.ptr, b.ptr)
    plan.one_pass(2, 1, b.ptr, b.ptr)
    assert fused <= 1.005 * err(b.download(rdt, pad.shape)[..., :nz] / rdt(n), ref)
    ctx.close()
