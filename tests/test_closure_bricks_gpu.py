"""The closure's kernels walk a grid in 4 x 4 x 32 bricks, in an order that
depends on its size, with a halo that wraps at its faces.  A periodic 32^3 field
repeated m times along each axis has the same values at every copy of a point,
whatever brick it is in."""
import numpy as np
import pytest

from spkmod import spk

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = spk.Ctx(0)
    yield c
    c.close()


def padded(r):
    out = np.zeros(r.shape[:-1] + (r.shape[-1] + 2,))
    out[..., : r.shape[-1]] = r
    return out


def run(ctx, n, params, u, tau):
    net = spk.Closure(ctx, n)
    net.set_params(params)
    net.set_scales(0.7, [1.0, 0.5, 0.25, 2.0, 1.0, 0.5])
    du, dt, out = (ctx.alloc(c * n * n * (n + 2) * 8) for c in (3, 6, 6))
    du.upload(padded(u))
    dt.upload(padded(tau))
    out.upload(np.full(6 * n * n * (n + 2), 7.0))
    net.forward(du.ptr, out.ptr)
    loss = net.grads(du.ptr, dt.ptr)
    res = out.download(np.float64, (6, n, n, n + 2)), loss, net.get_grads()
    net.destroy()
    return res


@pytest.mark.parametrize("m", [2, 3, 4])
def test_repeated_field(ctx, m):
    rng = np.random.default_rng(17)
    params = np.zeros(sum(27 * 32 * c + 32 for c in spk.Closure.CIN), np.float32)
    for (w, b), cin in zip(spk.Closure.layer_slices(), spk.Closure.CIN):
        params[w] = rng.standard_normal(27 * 32 * cin) / np.sqrt(27 * (3 if cin == 16 else cin))
        params[b] = 0.1 * rng.standard_normal(32)
    u, tau = rng.standard_normal((3, 32, 32, 32)), rng.standard_normal((6, 32, 32, 32))
    ref, loss, grads = run(ctx, 32, params, u, tau)
    got, loss_m, grads_m = run(ctx, 32 * m, params, np.tile(u, (1, m, m, m)), np.tile(tau, (1, m, m, m)))
    # the same operations on the same values at every point, and the pads written
    assert np.array_equal(got[..., : 32 * m], np.tile(ref[..., :32], (1, m, m, m)))
    assert np.all(got[..., 32 * m:] == 0.0) and np.all(ref[..., 32:] == 0.0)
    # means over m^3 times the points: FP32 sums of up to 2^21 terms in another order
    # (2^21 eps / 2 is a bound of 0.13, sqrt(2^21) eps its statistical size 9e-5); with
    # m = 3 the loss's factor 1 / (6 P) also rounds dZ to other BF16 values, 2^-9 each,
    # unbiased over 32^3 of them
    tol = 1e-3
    assert abs(loss_m - loss) <= tol * loss
    assert np.linalg.norm(grads_m - grads) <= tol * np.linalg.norm(grads)
