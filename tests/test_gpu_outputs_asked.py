"""zeus_run_batch with some of the per-start arrays asked for: each is the one of
the call that asks for all of them, whichever its neighbours; an array that is
not asked for is not written."""
import ctypes as C
import itertools

import numpy as np
import pytest

import zeus_amd as z
from zeus_amd import _capi as capi

pytestmark = pytest.mark.gpu
KEYS = (("status", np.int32, capi._i32p), ("iter", np.int32, capi._i32p),
        ("fval", np.float64, capi._dp), ("gnorm", np.float64, capi._dp),
        ("x", np.float64, capi._dp), ("ls_evals", np.int32, capi._i32p),
        ("grads", np.int32, capi._i32p))
PROBLEMS = [(z.Rosenbrock(2), 33), (z.Rastrigin(20), 70), (z.Rosenbrock(2), 0),
            (z.Rosenbrock(2), 131)]


def call(keys):
    P = (capi.Problem * len(PROBLEMS))()
    for i, (f, n) in enumerate(PROBLEMS):
        P[i] = capi.Problem(f.kind, f.dim, -5.0, 5.0, n, 2, -1, 0, 7 + i, 0, 0, 1e-8, None, 0,
                            None, b"f", None)
    R = (capi.Result * len(PROBLEMS))()
    bx = (C.c_double * sum(f.dim for f, _ in PROBLEMS))()
    total, coords = sum(n for _, n in PROBLEMS), sum(n * f.dim for f, n in PROBLEMS)
    out = {k: np.full(coords if k == "x" else total, -77, t) for k, t, _ in KEYS}
    so = capi.StartOutputs(*[out[k].ctypes.data_as(p) if k in keys else None
                             for k, _, p in KEYS])
    opt = capi.Options(0, capi.FORM_THREAD, 0, 0, 0, 0)
    assert capi.lib().zeus_run_batch(P, len(PROBLEMS), C.byref(opt), R, bx, C.byref(so),
                                     None) == 0
    return out


def test_arrays_asked_for():
    names = [k for k, _, _ in KEYS]
    want = call(names)
    assert all((want[k] != -77).all() for k in names)
    for r in (0, 1, 2, 6):
        for keys in itertools.combinations(names, r):
            got = call(keys)
            for k in names:
                if k in keys:
                    assert got[k].tobytes() == want[k].tobytes(), (keys, k)
                else:
                    assert (got[k] == -77).all(), (keys, k)
