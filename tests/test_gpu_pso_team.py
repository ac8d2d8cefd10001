"""The team form of the PSO (several lanes per particle): the separable
objectives beyond four coordinates and the binned likelihood, at ragged start
counts, start counts that make a workgroup take several passes, and through
every entry point."""
import numpy as np
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


# Rosenbrock's value is made of + - * and the team adds its terms in serial
# order: the swarm equals the oracle's bit for bit.  16 lanes x 16 particles
# (D = 10) and 64 x 4 (D = 50) per pass; 20000 x 10 takes two passes.
@pytest.mark.parametrize("D,N", [(10, 1), (10, 17), (10, 20000), (50, 3), (50, 261), (50, 9000)])
@pytest.mark.parametrize("g", [z.PRNGType.XORWOW, z.PRNGType.PHILOX], ids=["xorwow", "philox"])
def test_rosenbrock_bitwise(orc, D, N, g):
    got = z.pso(z.Rosenbrock(D), -5, 5, N, 4, 42, prng=g)
    want = orc.pso(orc.ROSENBROCK, D, -5, 5, N, 4, 42, prng=int(g))
    for a, b in zip(got, want):
        assert np.array_equal(np.asarray(a), np.asarray(b))


# The cosines differ from the C library's by rounding (a few 1e-16 of terms up
# to 10, 20 of them); particles move by differences of pBest and gBest only,
# so positions agree to rounding as long as both sides pick the same bests.
@pytest.mark.parametrize("name,D,box", [("Rastrigin", 20, 5.12), ("Ackley", 10, 32.768)])
@pytest.mark.parametrize("N", [5, 300])
def test_trigonometric_against_oracle(orc, name, D, box, N):
    got = z.pso(getattr(z, name)(D), -box, box, N, 3, 7)
    want = orc.pso(getattr(orc, name.upper()), D, -box, box, N, 3, 7)
    assert np.abs(got[0] - want[0]).max() <= 1e-12 * box
    assert np.abs(got[1] - want[1]).max() <= 1e-12 * np.abs(want[1]).max()
    assert abs(got[3] - want[3]) <= 1e-12 * np.abs(want[1]).max()


# bins: one lane's worth, a full wavefront, a remainder, two rounds
@pytest.mark.parametrize("bins", [1, 64, 65, 100, 128])
def test_likelihood_against_oracle(orc, bins):
    P = z.make_dijet(42, 3, bins)
    got = z.pso(z.LogLikelihood.from_params(P), 0.0, 10.0, 37, 3, 42)
    want = orc.pso(orc.LOGLIK, 4, 0.0, 10.0, 37, 3, 42, params=P)
    fin = np.isfinite(want[1])
    assert np.array_equal(fin, np.isfinite(got[1]))
    assert np.abs(got[0] - want[0]).max() <= 1e-11
    assert np.allclose(got[1][fin], want[1][fin], rtol=1e-11, atol=0)


# the swarm depends on the inputs only, not on the entry point or the batch
@pytest.mark.parametrize("f,box", [(z.Rosenbrock(10), 5.0), (z.Rastrigin(20), 5.12)])
def test_entry_points_agree(f, box):
    import ctypes as C
    N, T = 700, 3
    want = z.pso(f, -box, box, N, T, 42)
    sw = z.Swarm(f, -box, box, N, 42).init()
    for t in range(1, T + 1):
        sw.step(t)
    st = sw.state()
    assert np.array_equal(st["pbest_x"], want[0]) and np.array_equal(st["pbest_val"], want[1])
    assert np.array_equal(st["gbest_x"], want[2]) and st["gbest_val"] == want[3]
    px, pv = z.DeviceArray(nbytes=8 * N * f.dim), z.DeviceArray(nbytes=8 * N)
    gx, gv = z.DeviceArray(nbytes=8 * f.dim), z.DeviceArray(nbytes=8)
    rc = z.capi.lib().zeus_pso_run_noalloc(C.byref(z.Swarm(f, -box, box, N, 42).problem),
                                           px.ptr, pv.ptr, gx.ptr, gv.ptr, None)
    assert rc == 0  # pso_iter 0 in that descriptor: the initial swarm
    assert np.array_equal(pv.to_host(), z.pso(f, -box, box, N, 0, 42)[1])
    # second problem of a batch, MAX_ITER 0: the BFGS starts are pBestX
    probs = [z.Problem(f, -box, box, n, 0, T, 0, 1e-8, 42) for n in (13, N)]
    r = z.run_batch(probs, form="group", per_start=True)[1]
    assert np.array_equal(r.per_start["x"], want[0])
