"""Likelihood swarms with many particles in a launch take 16 lanes a particle,
with few 64: the same sums in the same order, so a batch of fits has the bits of
the fits one by one."""
import numpy as np
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bins", [1, 15, 17, 100])
@pytest.mark.parametrize("prng", [z.PRNGType.XORWOW, z.PRNGType.PHILOX])
def test_batch_equals_single_fits(bins, prng):
    rng = np.random.default_rng(bins)
    ps = []
    for k in range(18):  # 18 ragged problems, 4400 particles
        x, n = rng.uniform(0.1, 0.9, bins), 256 - 3 * (k % 7)
        f = z.LogLikelihood(rng.poisson(20.0, bins).astype(float), x)
        ps.append(z.Problem(f, 0.0, 5.0, n, 1, 6, n + 1, 1e-8, 11 + k, stream=k, prng=prng))
    assert sum(p.N for p in ps) >= 4096
    kw = dict(form="group", group_threads=64, per_start=True)
    for p, r in zip(ps, z.run_batch(ps, **kw)):
        one = z.run_batch([p], **kw)[0]
        assert r.fval == one.fval and r.idx == one.idx
        for key in r.per_start:
            assert r.per_start[key].tobytes() == one.per_start[key].tobytes(), key
