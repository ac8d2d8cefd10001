"""The launch shape that a call reports (tuned_config) can be asked for, and a
recorded call runs the kernel that was tuned where that one records."""
import pytest

import zeus_amd as z

pytestmark = pytest.mark.gpu
SHAPE = (z.capi.OBJ_GAUSSIAN, 150)


def solve(f, n, **kw):
    rec = kw.pop("trajectory", None)
    r = z.run_batch([z.Problem(f, -5.0, 5.0, n, 10000, 10, 0, 1e-8, 42, trajectory=rec)],
                    per_start=True, **kw)[0]
    return {k: v.tobytes() for k, v in r.per_start.items()}


def test_reported_shape_can_be_asked_for():
    f = z.Gaussian(z.make_spd(42, 1, 150))
    auto = solve(f, 60)  # tunes
    auto = solve(f, 60)
    form, threads = z.tuned_config(*SHAPE)
    name = {1: "thread", 2: "group", 3: "tile", 4: "team"}[form]
    assert solve(f, 60, form=name, group_threads=threads) == auto
    assert z.tuned_config(*SHAPE) == (form, threads)
    # a workgroup per start has two names, the tile of 16 starts the other size
    one = solve(f, 60, form="tile", group_threads=512)
    assert z.tuned_config(*SHAPE) == (z.capi.FORM_TILE, 512)
    assert one == solve(f, 60, form="group", group_threads=512)
    solve(f, 60, form="tile")
    assert z.tuned_config(*SHAPE) == (z.capi.FORM_TILE, 1024)


def test_recorded_call_runs_the_tuned_kernel():
    f = z.Gaussian(z.make_spd(42, 1, 150))
    for _ in range(2):
        want = solve(f, 60)
    if z.tuned_config(*SHAPE) != (z.capi.FORM_TILE, 512):
        pytest.skip("another shape was tuned, which does not record")
    assert solve(f, 60, trajectory=(4, 2)) == want
    assert z.tuned_config(*SHAPE) == (z.capi.FORM_GROUP, 512)
