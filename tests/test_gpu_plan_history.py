"""A McClean plan's passes are a function of its shape and options: a tuned plan
that held another shape or tile in between gives bitwise the results of a fresh
one."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_reshape import _case, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['complex64', 'complex128'])
@pytest.mark.parametrize('n,L,tile', [(20, 9, (12, 2)), (22, 6, (12, 2)), (22, 6, (12, 3)), (19, 6, (12, 2))])
def test_tuned_plan_forgets_what_it_held(gpu, dtype, n, L, tile):
    from qradient_amd import _native
    ctx = _native.Context(0)
    axes, angles, terms = _case(n, L, 41 * n + L)
    away = _case(15, 3, 5)

    def plan():
        h = ctypes.c_void_p()
        _native.call('qg_mcclean_plan', ctx.handle, n, L, _native.DTYPES[dtype], 0, 0, ctypes.byref(h))
        return h

    fresh, h = plan(), plan()
    try:
        _native.call('qg_plan_tune', fresh, tile[0], tile[1], 4, 4)
        E0, g0 = _run(fresh, n, L, axes, angles, terms)
        # another shape in between, then another tile
        _native.call('qg_plan_tune', h, tile[0], tile[1], 4, 4)
        _native.call('qg_plan_reshape', h, 15, 3, 0)
        _run(h, 15, 3, *away)
        _native.call('qg_plan_reshape', h, n, L, 0)
        E, g = _run(h, n, L, axes, angles, terms)
        assert E == E0 and np.array_equal(g, g0)
        _native.call('qg_plan_tune', h, 11, 2, 4, 4)
        _native.call('qg_plan_tune', h, tile[0], tile[1], 4, 4)
        E, g = _run(h, n, L, axes, angles, terms)
        assert E == E0 and np.array_equal(g, g0)
    finally:
        _native.call('qg_plan_destroy', fresh)
        _native.call('qg_plan_destroy', h)
