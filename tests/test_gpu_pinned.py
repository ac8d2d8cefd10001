"""The pinned buffer of the per-start outputs is given back when the calls that
follow have no use for it, and a call that wants it again gets it."""
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu


def mapped():
    with open("/proc/self/status") as fh:
        return next(int(l.split()[1]) << 10 for l in fh if l.startswith("VmSize"))


def call(n, per_start):
    return z.run_batch([z.Problem(z.Rosenbrock(2), -5.0, 5.0, n, 1, -1, 0, 1e-8, 3)],
                       form="thread", per_start=per_start)[0].per_start


def test_given_back_and_taken_again():
    want = {k: v.tobytes() for k, v in call(1_000_000, True).items()}  # 48 MB of outputs
    call(100, False)
    before = mapped()
    for _ in range(70):
        call(100, False)
    assert before - mapped() >= 40 << 20
    got = call(1_000_000, True)
    assert all(got[k].tobytes() == want[k] for k in want)
