"""Per-start outputs of a batch: the arrays of small batches come back in one
copy per class through pinned memory, those of batches beyond 64 MiB straight
to the caller.  Start i depends on the seed and its index alone, so the first
starts of a large problem are those of a small one, bit for bit."""
import numpy as np
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


def problem(kind, dim, n, seed):
    return z.Problem(kind(dim), -5.0, 5.0, n, 3, -1, n + 1, 1e-8, seed)


def check(many, few, n):
    assert len(many) == len(few)
    for a, b in zip(many, few):
        assert a.keys() == b.keys()
        for k in a:
            x, y = np.asarray(a[k])[:n], np.asarray(b[k])[:n]
            assert x.dtype == y.dtype and x.tobytes() == y.tobytes(), k


# 1.7e6 starts of 2 dimensions are 75 MB of outputs
@pytest.mark.parametrize("big", [1001, 1_700_000])
def test_prefix_of_a_larger_batch(big):
    n = 130
    many = [problem(z.Rosenbrock, 2, big, 7), problem(z.Rastrigin, 20, 1, 8),
            problem(z.Rosenbrock, 2, n, 9)]
    few = [problem(z.Rosenbrock, 2, n, 7)] + many[1:]
    a, b = ([r.per_start for r in z.run_batch(p, form="thread", per_start=True)]
            for p in (many, few))
    check(a, b, n)
