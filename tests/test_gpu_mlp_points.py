"""The network's cooperative value and gradient (16 points per wavefront group,
eight groups side by side, the first 256 points' activations kept) at point
counts around those edges: a few BFGS iterations against the oracle."""
import numpy as np
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


# the network amplifies a rounding difference by less than 1e3 in four
# iterations (values to 1e-13 of themselves, 1e-10 with that)
@pytest.mark.parametrize("m", [1, 15, 16, 17, 128, 129, 255, 256, 257, 400])
def test_iterations_against_oracle(orc, m):
    P = z.make_mlp_data(42, m)
    N, iters = 5, 4
    r = z.Zeus(z.Mlp(P[:m], P[m:]), -2, 2, N, iters, 2, N + 1, "mlp", 1e-8, 42, 0,
               per_start=True).per_start
    o = orc.run(orc.MLP, 321, -2, 2, N, iters, 2, N + 1, 1e-8, 42, params=P)
    assert np.array_equal(r["status"], o.status) and np.array_equal(r["iter"], o.iter)
    assert np.abs(r["fval"] - o.fval).max() <= 1e-10 * max(1e-3, np.abs(o.fval).max())
    assert np.abs(r["x"] - o.x).max() <= 1e-9
