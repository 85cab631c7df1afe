"""The bias gradient is a sum over every point of the grid.  One large output error and
small equal ones elsewhere, each 2^-30 of it: a running sum in single precision drops
the small ones that follow the large one.

Tolerance: 2^-24 for each rounding of a sum that holds the large term.  At 128^3 a
block adds up 16 bricks, a slice 16 blocks, the total 16 slices; the brick that holds
the large term has 32 steps, in which the small terms are 2^-21 of it together."""
import numpy as np
import pytest

from spkmod import spk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("at", [(1, 2, 5), (77, 64, 127)])
def test_small_terms_beside_a_large_one(at):
    n = 128
    ctx = spk.Ctx(0)
    net = spk.Closure(ctx, n)
    # no weights, no biases: the prediction is 0, an output's error is minus its target
    net.set_params(np.zeros(sum(27 * 32 * c + 32 for c in spk.Closure.CIN), np.float32))
    u = np.zeros((3, n, n, n + 2))
    tau = np.zeros((6, n, n, n + 2))
    tau[..., :n] = 2.0 ** -30
    tau[(slice(None),) + at] = 1.0
    d_u, d_tau = ctx.alloc(u.nbytes), ctx.alloc(tau.nbytes)
    d_u.upload(u)
    d_tau.upload(tau)
    net.grads(d_u.ptr, d_tau.ptr)
    got = net.get_grads()[spk.Closure.layer_slices()[3][1]].astype(np.float64)
    net.destroy()
    ctx.close()
    # dZ = 2 (pred - target) / (6 P) in BF16
    g = np.float32(2.0) / (np.float32(6.0) * np.float32(n ** 3))
    large = (np.frombuffer(np.float32(g).tobytes(), np.uint32).astype(np.uint64) + 0x7FFF +
             ((np.frombuffer(np.float32(g).tobytes(), np.uint32) >> 16) & 1)) >> 16 << 16
    large = float(large.astype(np.uint32).view(np.float32)[0])
    want = -large * (1.0 + (n ** 3 - 1) * 2.0 ** -30)
    tol = (16 + 16 + 16 + 1) * 2.0 ** -24 + 2.0 ** -21
    assert np.all(np.abs(got[:6] / want - 1.0) <= tol), got[:6] / want - 1.0
    assert np.all(got[6:] == 0.0)
