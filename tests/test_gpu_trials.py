"""Line searches of the per-workgroup form with one wavefront: the trials that
share a wavefront (5 to 16 coordinates: four, 17 to 32: two) against the same
form with four wavefronts, whose values add the same numbers in the same order
(its product with the inverse Hessian does not, so one iteration), and against
one lane per start.  Coordinates around 2^26 and beyond take the
library's general sine and cosine."""
import numpy as np
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


def solve(f, box, iters, n=67, **kw):
    r = z.run_batch([z.Problem(f, -box, box, n, iters, -1, n + 1, 1e-300, 5)], per_start=True,
                    **kw)
    return r[0].per_start


@pytest.mark.parametrize("gradient", ["adjoint", "dual"])
@pytest.mark.parametrize("box", [5.12, 2.0**27, 1e18])
def test_two_trials_a_wavefront(box, gradient):
    f = z.Rastrigin(20)
    a, b = (solve(f, box, 1, form="group", group_threads=t, gradient=gradient)
            for t in (64, 256))
    for k in a:
        assert a[k].tobytes() == b[k].tobytes(), k


@pytest.mark.parametrize("box", [3.0, 2.0**27])
@pytest.mark.parametrize("kind, dim", [(z.Rosenbrock, 10), (z.Ackley, 10),
                                       (z.Rastrigin, 20)])
@pytest.mark.parametrize("form", ["group", "team"])
def test_first_iterations(kind, dim, box, form):
    """One iteration leaves rounding no room: the first step is along -g, its
    trials alpha = 2^-t, so values differ by the order of the sum (a few ulp of
    its largest term, which a value near it shares)."""
    try:
        a = solve(kind(dim), box, 1, form=form,
                  group_threads=64 if form == "group" else 0)
    except z.capi.ZeusError:
        pytest.skip("not offered")
    b = solve(kind(dim), box, 1, form="thread")
    same = a["ls_evals"] == b["ls_evals"]
    assert same.mean() > 0.95  # a trial at the acceptance line may fall on either side
    np.testing.assert_allclose(a["fval"][same], b["fval"][same], rtol=1e-9)
