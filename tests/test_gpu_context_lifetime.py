"""Plans and states outlive the caller's hold on their context: an interpreter
that ends destroys a context and what was made from it in either order."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_reshape import _case, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,L', [(6, 3), (15, 3)])
def test_plan_and_state_after_their_context(gpu, n, L):
    from qradient_amd import _native
    call = _native.call
    axes, angles, terms = _case(n, L, 7 * n)
    vec = np.random.RandomState(n).standard_normal(2 << n)
    ctx, plan, state, other = (ctypes.c_void_p() for _ in range(4))
    call('qg_ctx_create', 0, None, ctypes.byref(ctx))
    call('qg_mcclean_plan', ctx, n, L, _native.DTYPES['complex128'], 0, 0, ctypes.byref(plan))
    call('qg_state_create', ctx, n, _native.DTYPES['complex128'], b'0', ctypes.byref(state))
    E0, g0 = _run(plan, n, L, axes, angles, terms)
    call('qg_state_set', state, _native.dptr(vec))
    call('qg_ctx_destroy', ctx)
    call('qg_ctx_create', 0, None, ctypes.byref(other))  # takes the memory that a freed context would leave
    try:
        E1, g1 = _run(plan, n, L, axes, angles, terms)
        assert E0 == E1 and np.array_equal(g0, g1)
        got = np.empty_like(vec)
        call('qg_state_get', state, _native.dptr(got))
        assert np.array_equal(got, vec)
    finally:
        call('qg_plan_destroy', plan)
        call('qg_state_destroy', state)
        call('qg_ctx_destroy', other)
