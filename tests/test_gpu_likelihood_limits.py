"""The binned likelihood at the limits of its forms: swarms of 16 lanes a particle
whose workgroups take several passes, and bin counts around the 16384 whose
logarithms are tabulated (beyond, power functions everywhere)."""
import numpy as np
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


# 16 particles a pass: up to 16384 particles one pass, beyond two (with a
# remainder), then four; zeus_pso_run has 64 lanes a particle.  The sums are the
# same, in the same order.
@pytest.mark.parametrize("n", [16384, 16385, 16384 + 77, 40001])
def test_passes_of_sixteen_lanes(n):
    f = z.LogLikelihood.from_params(z.make_dijet(42, 3, 19))
    want = z.pso(f, 0.0, 10.0, n, 3, 42)
    r = z.run_batch([z.Problem(f, 0.0, 10.0, n, 0, 3, 0, 1e-8, 42)], form="group",
                    group_threads=64, per_start=True)[0].per_start
    assert np.array_equal(r["x"], want[0])


# Terms that cancel by less than 1e3, 16385 of them added one by one: 2e-9 of the
# sum at most.
@pytest.mark.parametrize("bins", [16384, 16385])
def test_many_bins_against_oracle(orc, bins):
    P = z.make_dijet(42, 2, bins)
    f, o = z.LogLikelihood.from_params(P), orc.Obj(orc.LOGLIK, 4, P)
    X = np.array([0.5, 10.0, 5.0, 0.1]) * np.random.default_rng(bins).uniform(0.7, 1.3, (5, 4))
    want = [o.value_grad_adjoint(x) for x in X]
    fo = np.array([w[0] for w in want])
    go = np.array([w[1] for w in want])
    for how in ("adjoint", "dual"):
        v, g = z.evaluate(f, X, how)
        assert (np.abs(v - fo) <= 2e-9 * np.abs(fo)).all()
        assert (np.abs(g - go).max(1) <= 2e-9 * np.abs(go).max(1)).all()
    for form in ("thread", "group"):  # no iteration: value and gradient of the start
        r = z.run_batch([z.Problem(f, 0.0, 10.0, 5, 0, -1, 0, 1e-8, 42, x0=X)], form=form,
                        per_start=True)[0].per_start
        assert (np.abs(r["fval"] - fo) <= 2e-9 * np.abs(fo)).all()
        norm = np.linalg.norm(go, axis=1)
        assert (np.abs(r["gnorm"] - norm) <= 2e-9 * norm).all()
    pv = z.pso(f, 0.0, 10.0, 37, 2, 42)
    po = orc.pso(orc.LOGLIK, 4, 0.0, 10.0, 37, 2, 42, params=P)
    fin = np.isfinite(po[1])
    assert fin.any() and np.array_equal(fin, np.isfinite(pv[1]))
    assert np.allclose(pv[1][fin], po[1][fin], rtol=2e-9, atol=0)
