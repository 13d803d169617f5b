"""A QAOA plan's term limit (n z terms and n (n - 1) / 2 zz terms, repeats
counted) is the same before and after a shot-based gradient on the plan."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n', [3, 8])
def test_term_limit_outlives_a_shot_gradient(gpu, n):
    from qradient_amd import _native
    ctx = _native.Context(0)
    plan = ctypes.c_void_p()
    _native.call('qg_qaoa_plan', ctx.handle, n, 1, _native.DTYPES['complex128'], 1, ctypes.byref(plan))
    most = n + n * (n - 1) // 2
    betas, gammas = np.array([0.3]), np.array([0.4])

    def shots(count):
        arr, k = _native.terms_array([(_native.TERM_Z, q % n, -1, 0.5) for q in range(count)])
        u = np.full((2 * (k + n), 4), 0.5)
        idx = np.empty(u.shape, dtype=np.int32)
        expec = np.empty(k + 1)
        _native.call('qg_qaoa_shift_sample', plan, arr, k, _native.dptr(betas), _native.dptr(gammas), None, arr, k,
                     _native.dptr(expec), 4, _native.dptr(u), _native.iptr(idx))
        assert abs(expec[k] - 1.0) <= 1e-12

    def grad(count):
        arr, k = _native.terms_array([(_native.TERM_Z, q % n, -1, 0.5) for q in range(count)])
        off = np.array([0, k], dtype=np.int32)
        E, g = np.empty(1), np.empty(2)
        _native.call('qg_qaoa_grad_run', plan, 1, arr, _native.iptr(off), _native.dptr(betas), _native.dptr(gammas),
                     _native.dptr(E), _native.dptr(g))

    try:
        for _ in range(2):  # the second time after both kinds of run
            for run in (shots, grad):
                with pytest.raises(ValueError):
                    run(most + 1)
                run(most)
    finally:
        _native.call('qg_plan_destroy', plan)
