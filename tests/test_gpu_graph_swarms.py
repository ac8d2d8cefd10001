"""Replayed graphs of batches whose counts agree (problems, starts, workgroups)
while the particles per workgroup, a launch argument of the captured PSO, do
not: each replay equals the eager result of its own batch, bit for bit."""
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


def batch(counts):
    # iterations 0: the results are the swarm's best positions
    return [z.Problem(z.Rosenbrock(50), -5.0, 5.0, n, 0, 3, 0, 1e-8, 42 + i, stream=i)
            for i, n in enumerate(counts)]


def results(probs, graph):
    r = z.run_batch(probs, form="group", group_threads=64, per_start=True, use_graph=graph)
    return [b"".join(q.per_start[k].tobytes() for k in ("x", "fval")) for q in r]


def test_batches_that_differ_in_particles_per_workgroup():
    # Four particles a workgroup while a problem has up to 1024 workgroups, eight
    # beyond.  Both: 1001 problems, 6000 starts, 1625 workgroups.
    a = batch([2500] + [4] * 500 + [3] * 500)
    b = batch([5000] + [1] * 1000)
    blocks = [sum(-(-p.N // k) for p in q) for q, k in ((a, 4), (b, 8))]
    assert blocks == [1625, 1625] and sum(p.N for p in a) == sum(p.N for p in b) == 6000
    want = [results(q, False) for q in (a, b)]
    for _ in range(3):  # captures, then replays
        for q, w in zip((a, b), want):
            assert results(q, True) == w
