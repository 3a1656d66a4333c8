"""GPU tests of single kernels and dispatch branches at the sizes where they
can go wrong: tile edges, remainders, the smallest grids.  Bars are the
rounding of the summed terms, as in the parity tests."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
import cases

pytestmark = pytest.mark.gpu


def _api():
    from parflow_amd import api
    return api


def _field(prob, rng, ghost=1e9):
    a = np.full(prob.shape, ghost)
    a[1:-1, 1:-1, 1:-1] = rng.normal(size=(prob.nz, prob.ny, prob.nx))
    return a


@pytest.mark.parametrize("shape", [(1, 1, 2), (5, 3, 2), (65, 33, 40)])
def test_reduction_results_reach_the_host(gpu, shape):
    """Sums, maxima and mixed results of two problems in turn: each call
    returns its own values (fewer blocks than threads, and more rows than
    blocks)."""
    api = _api()
    probs = [cases.hetero(*shape, seed=1), cases.hetero(7, 4, 3, seed=2)]
    gps = [api.GPUProblem(p) for p in probs]
    rng = np.random.default_rng(7)
    r, a, b = C.c_double(), C.c_double(), C.c_double()
    lib = api.lib()
    for rep in range(3):
        for prob, gp in zip(probs, gps):
            x, y = _field(prob, rng), _field(prob, rng)
            X, Y = prob.interior(x), prob.interior(y)
            dx, dy = gp.vec(x), gp.vec(y)
            api.check(lib.pfhip_vec_dot(gp.h, dx.ptr, dy.ptr, C.byref(r), None), "dot")
            assert abs(r.value - np.sum(X * Y)) <= 1e-13 * np.sum(np.abs(X * Y))
            api.check(lib.pfhip_vec_max_norm(gp.h, dx.ptr, C.byref(r), None), "max")
            assert r.value == np.max(np.abs(X))
            api.check(lib.pfhip_vec_min(gp.h, dy.ptr, C.byref(r), None), "min")
            assert r.value == np.min(Y)
            lib.pfhip_vec_dot_scsteplength.argtypes = [C.c_void_p] * 6
            api.check(lib.pfhip_vec_dot_scsteplength(gp.h, dx.ptr, dy.ptr, C.byref(a),
                                                     C.byref(b), None), "dot_scsteplength")
            assert abs(a.value - np.sum(Y * Y)) <= 1e-13 * np.sum(Y * Y)
            assert abs(b.value - np.max(np.abs(Y) / (1 + np.abs(X)))) <= 1e-15 * b.value
