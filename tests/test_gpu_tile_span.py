"""Tile form of the BFGS: the list of directions beyond its 64 places (folded
into the explicit matrix) and steps that append the update's own vector.  A
quadratic x^T C x / 2 with eigenvalues 1 .. 1e4 takes about as many iterations
as it has dimensions: 150 are more than the list holds."""
import numpy as np
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


def spread(dim, top):
    q, _ = np.linalg.qr(np.random.default_rng(dim).standard_normal((dim, dim)))
    c = (q * np.logspace(0, np.log10(top), dim)) @ q.T
    return z.Gaussian((c + c.T) / 2)


def solve(f, form, tol, iters):
    return z.run_batch([z.Problem(f, -5.0, 5.0, 33, iters, -1, 34, tol, 11)], form=form,
                       per_start=True)[0].per_start


@pytest.mark.parametrize("dim", [32, 150])
def test_as_many_steps_as_dimensions(dim):
    f = spread(dim, 1e4)
    a, b = solve(f, "tile", 1e-6, 2000), solve(f, "group", 1e-6, 2000)
    assert (a["status"] == 1).all()
    assert dim < 150 or a["iter"].min() > 64  # the list was folded
    # the smallest eigenvalue is 1: |x| <= |C x| < tol
    assert (np.linalg.norm(a["x"], axis=1) < 1e-6).all()
    # the same method: as many iterations, but for rounding
    assert abs(a["iter"].mean() / b["iter"].mean() - 1) < 0.05


@pytest.mark.parametrize("dim", [32, 150])
def test_past_the_floor(dim):
    """tol 0: trials are rejected to the last at the rounding floor, and the
    curvature test skips updates; the value stays there."""
    a = solve(spread(dim, 10.0), "tile", 0.0, 200)
    assert (a["status"] == 0).all() and (a["iter"] == 200).all()
    # |x| at the floor is of the order 1e-7 at most (s.y < 1e-14 ends the updates)
    assert (a["fval"] >= 0).all() and (a["fval"] < 1e-12).all()
