"""The binned likelihood in the fit: every branch of the power functions (plain,
overflow, underflow, bins outside (0, 1)) against the same sum in numpy."""
import numpy as np
import pytest
from scipy.special import gammaln

import zeus_amd as z

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["thread", "group"])
@pytest.mark.parametrize("bad", [1.0, 1.5, -0.5, 0.0, np.nan])
def test_bins_outside(bad, form):
    """0^b or a power of a negative number: no start has a value."""
    x, k = np.linspace(0.1, 0.9, 70), np.full(70, 5.0)
    x[66] = bad
    ps = z.run_batch([z.Problem(z.LogLikelihood(k, x), 0.3, 0.7, 20, 1, -1, 21, 1e-8, 3)],
                     form=form, per_start=True)[0].per_start
    assert not np.isfinite(ps["fval"]).any() and (ps["status"] > 1).all()


@pytest.mark.parametrize("form", ["thread", "group"])
@pytest.mark.parametrize("box", [1.0, 10.0, 300.0])
@pytest.mark.parametrize("n", [1, 63, 65, 130])
def test_value_at_the_result(n, box, form):
    rng = np.random.default_rng(n)
    x = rng.uniform(0.05, 0.95, n)
    k = rng.poisson(20.0, n).astype(float)
    ps = z.run_batch([z.Problem(z.LogLikelihood(k, x), 0.0, box, 200, 1, -1, 201, 1e-8, 3)],
                     form=form, per_start=True)[0].per_start
    a, b, c, d = (ps["x"][:, i:i + 1] for i in range(4))
    with np.errstate(all="ignore"):
        mean = a * np.power(1 - x, b) / np.power(x, c + d * np.log(x))
        terms = -(k * np.log(mean) - mean - gammaln(k + 1))
        want = terms.sum(1)
        scale = np.abs(terms).sum(1)
    # (a start that ended non-finite reports the value of its next point)
    both = np.isin(ps["status"], [0, 1])
    assert both.any() and np.isfinite(want[both]).all()
    # powers good to 2 ulp, exponents up to 700: 1e-13 of each term, 130 of them
    assert (np.abs(ps["fval"] - want)[both] <= 1e-11 * scale[both]).all()
