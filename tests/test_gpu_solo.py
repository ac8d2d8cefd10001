"""Gaussian BFGS with the matrix in registers (512 threads per start, adjoint
gradient) against the per-workgroup form of 256 threads: several problems in one
call, recorded steps, early stop, more steps than the list of directions holds,
and steps past the rounding floor."""
import numpy as np
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


def spread(top, seed):
    q, _ = np.linalg.qr(np.random.default_rng(seed).standard_normal((150, 150)))
    c = (q * np.logspace(0, np.log10(top), 150)) @ q.T
    return z.Gaussian((c + c.T) / 2)


def solve(problems, threads, **kw):
    return z.run_batch(problems, form="group", group_threads=threads, per_start=True, **kw)


def problem(f, n, iters, tol, seed, required=None, **kw):
    return z.Problem(f, -5.0, 5.0, n, iters, -1, n + 1 if required is None else required, tol,
                     seed, **kw)


def test_batch_of_ragged_problems():
    ps = [problem(spread(4.0, k), n, 200, 1e-6, 7 + k) for k, n in enumerate((1, 13, 300, 2))]
    for a, b in zip(solve(ps, 512), solve(ps, 256)):
        a, b = a.per_start, b.per_start
        assert (a["status"] == 1).all() and (b["status"] == 1).all()
        # the smallest eigenvalue is 1: |x| <= |C x| < tol
        assert (np.linalg.norm(a["x"], axis=1) < 1e-6).all()
        # the same method: the same steps, but where rounding moves |g| over tol
        assert (np.abs(a["iter"] - b["iter"]) <= 1).all()
        assert (a["iter"] == b["iter"]).mean() > 0.9


def test_recorded_steps():
    f = spread(10.0, 3)
    a, b = (solve([problem(f, 3, 6, 1e-300, 5, trajectory=(6, 3))], t)[0].trajectory
            for t in (512, 256))
    assert a.keys() == b.keys()
    for k in a:
        # six steps from points of size 5: rounding of 1e-16 per operation, 150 of
        # them a sum, grows by the condition of each step (below 1e2)
        np.testing.assert_allclose(np.asarray(a[k]), np.asarray(b[k]), rtol=1e-10, atol=1e-10)


def test_early_stop():
    r = solve([problem(spread(4.0, 1), 3000, 200, 1e-6, 9, required=50)], 512)[0]
    st = r.per_start["status"]
    assert (st == 1).sum() >= 50 and set(np.unique(st)) <= {1, 2}


def test_more_steps_than_the_list_holds():
    p = [problem(spread(1e4, 2), 9, 2000, 1e-6, 11)]
    a, b = solve(p, 512)[0].per_start, solve(p, 256)[0].per_start
    assert (a["status"] == 1).all()
    assert a["iter"].min() > 64  # the list was folded
    assert (np.linalg.norm(a["x"], axis=1) < 1e-6).all()
    assert abs(a["iter"].mean() / b["iter"].mean() - 1) < 0.05


def test_past_the_floor():
    """tol 0: trials are rejected to the last at the rounding floor, and the
    curvature test skips updates; the value stays there."""
    a = solve([problem(spread(10.0, 4), 9, 200, 0.0, 11)], 512)[0].per_start
    assert (a["status"] == 0).all() and (a["iter"] == 200).all()
    # |x| at the floor is of the order 1e-7 at most (s.y < 1e-14 ends the updates)
    assert (a["fval"] >= 0).all() and (a["fval"] < 1e-12).all()


def test_where_it_is_tried():
    """Reported as the tile form; not tried where an early stop could end the
    call before the later starts have run (more starts than CUs)."""
    f = z.Gaussian(z.make_spd(42, 1, 150))
    for n, required, may in ((64, 0, True), (64, 10, True), (4096, 100, False)):
        r = z.run_batch([z.Problem(f, -5.0, 5.0, n, 10000, 10, required, 1e-8, 42)])[0]
        form, threads = z.tuned_config(z.capi.OBJ_GAUSSIAN, 150)
        assert form == z.capi.FORM_TILE
        assert may or threads != 512
        assert r.c.claimed >= min(required, n) and r.status == 1
