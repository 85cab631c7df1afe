"""An infinity in the closure's input: layers z Phi(z) of sums with positive weights
make +inf of +inf and NaN of -inf (-inf times Phi(-inf) = 0), at every point within
four cells of it and nowhere else."""
import numpy as np
import pytest

from spkmod import spk

pytestmark = pytest.mark.gpu

N = 32


def stresses(value, at):
    rng = np.random.default_rng(7)
    params = np.zeros(sum(27 * 32 * c + 32 for c in spk.Closure.CIN), np.float32)
    for (w, b), cin in zip(spk.Closure.layer_slices(), spk.Closure.CIN):
        params[w] = rng.uniform(0.5, 1.0, 27 * 32 * cin) / (27 * cin)
    u = 0.1 * rng.standard_normal((3, N, N, N + 2))
    u[(1,) + at] = value
    ctx = spk.Ctx(0)
    net = spk.Closure(ctx, N)
    net.set_params(params)
    d_u, d_tau = ctx.alloc(u.nbytes), ctx.alloc(2 * u.nbytes)
    d_u.upload(u)
    net.forward(d_u.ptr, d_tau.ptr)
    tau = d_tau.download(np.float64, (6, N, N, N + 2))[..., :N]
    net.destroy()
    ctx.close()
    return tau


def reach(at):
    """Points within four cells of `at` along each axis of the periodic grid."""
    near = [np.minimum((np.arange(N) - a) % N, (a - np.arange(N)) % N) <= 4 for a in at]
    return near[0][:, None, None] & near[1][None, :, None] & near[2][None, None, :]


AT = [(9, 14, 13), (0, 31, 31)]


@pytest.mark.parametrize("at", AT)
def test_minus_infinity(at):
    tau, box = stresses(-np.inf, at), reach(at)
    assert np.all(np.isnan(tau[:, box]))
    assert np.all(np.isfinite(tau[:, ~box]))


@pytest.mark.parametrize("at", AT)
def test_plus_infinity(at):
    tau, box = stresses(np.inf, at), reach(at)
    assert np.all(np.isposinf(tau[:, box]))
    assert np.all(np.isfinite(tau[:, ~box]))
