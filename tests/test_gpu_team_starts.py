"""Team form with more starts than fit the chip at once, alone (workgroups take
several) and beside another class (a team per start): every start's result is
that of the same start in a call of few starts, bit for bit."""
import numpy as np
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


def solve(f, points, team, beside=()):
    # ragged problems of one class, each start given
    cut = [0, 5, len(points) // 3, len(points)]
    ps = [z.Problem(f, -5.0, 5.0, b - a, 3, -1, 0, 1e-8, 1, x0=points[a:b])
          for a, b in zip(cut, cut[1:])]
    r = z.run_batch(ps + list(beside), form="team", group_threads=team, per_start=True)[:3]
    return {k: np.concatenate([q.per_start[k] for q in r]) for k in r[0].per_start}


# 256 / team teams a workgroup, two to six workgroups on each of 256 CUs
@pytest.mark.parametrize("kind, dim, team, n", [
    (z.Rastrigin, 20, 16, 8192 * 3 + 1), (z.Rastrigin, 20, 8, 16384 * 2 + 7),
    (z.Ackley, 10, 4, 41001), (z.Rosenbrock, 4, 4, 121001)])
def test_more_starts_than_fit(kind, dim, team, n):
    f = kind(dim)
    x0 = np.random.default_rng(n).uniform(-5.0, 5.0, (n, dim))
    few = 4000
    want = [solve(f, x0[i:i + few], team) for i in range(0, n, few)]
    other = z.Problem(z.Rosenbrock(10), -5.0, 5.0, 700, 3, 2, 0, 1e-8, 1)
    for beside in ((), (other,)):
        got = solve(f, x0, team, beside)
        for k in got:
            assert got[k].tobytes() == np.concatenate([w[k] for w in want]).tobytes(), k
