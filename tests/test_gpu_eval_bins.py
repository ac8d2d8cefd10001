"""zeus_eval of the binned likelihood (16 lanes per point) at point counts
around a workgroup's 16 and bin counts around a team's 16."""
import numpy as np
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


# a few roundings per bin of a sum whose terms cancel by less than 1e3
@pytest.mark.parametrize("n", [1, 15, 16, 17, 300])
@pytest.mark.parametrize("bins", [1, 16, 17, 100])
def test_values_and_gradients_against_oracle(orc, n, bins):
    P = z.make_dijet(42, 2, bins)
    f, o = z.LogLikelihood.from_params(P), orc.Obj(orc.LOGLIK, 4, P)
    rng = np.random.default_rng(n + bins)
    X = np.array([0.5, 10.0, 5.0, 0.1]) * rng.uniform(0.7, 1.3, (n, 4))
    v = z.evaluate(f, X)
    va, ga = z.evaluate(f, X, "adjoint")
    vd, gd = z.evaluate(f, X, "dual")
    assert np.array_equal(v, va) and np.array_equal(v, vd)
    for i in range(n):
        fo, go = o.value_grad_adjoint(X[i])
        assert abs(v[i] - fo) <= 1e-12 * abs(fo)
        assert np.abs(ga[i] - go).max() <= 1e-12 * np.abs(go).max()
        assert np.abs(gd[i] - go).max() <= 1e-12 * np.abs(go).max()
