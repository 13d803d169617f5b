"""Expectation values of shallow large circuits: where multi-layer passes are no
fewer, the last pass takes E itself instead of leaving the state to be read once
more (2^25 amplitudes and more; below, that read is from the caches)."""
import ctypes

import numpy as np
import pytest

from oracle import statevector as sv

pytestmark = pytest.mark.gpu


# kinds of the launches: 0 forward pass, 2 with the observable
@pytest.mark.parametrize('n,L,dtype,kinds', [(25, 1, 'complex64', [0, 0, 2]), (25, 1, 'complex128', [0, 0, 2]),
                                             (28, 1, 'complex64', [0, 0, 2]), (29, 2, 'complex64', [0] * 5 + [2]),
                                             (22, 1, 'complex64', [0, 0, 2]), (25, 2, 'complex64', [0] * 4 + [2])])
@pytest.mark.parametrize('entangler', ['cnot', 'cz'])
def test_launches(gpu, n, L, dtype, kinds, entangler):
    from qradient_amd import _native
    from qradient_amd.circuit_logic import McClean
    rs = np.random.RandomState(n + L)
    axes, angles = sv.mcclean_random_params(L, n, rs)
    obs = sv.zz_chain_observable(n, rs.standard_normal(n - 1))
    c = McClean(n, obs, L, axes=axes, angles=angles, dtype=dtype, entangler=entangler)
    _native.call('qg_plan_set_profiling', c._get_plan(), 1)
    E = c.run_expec_val()
    ms, got, count = (ctypes.c_float * 64)(), (ctypes.c_int * 64)(), ctypes.c_int()
    _native.call('qg_plan_pass_times', c._get_plan(), 64, ms, got, ctypes.byref(count))
    _native.call('qg_plan_set_profiling', c._get_plan(), 0)
    Eg, _ = c.grad_run()
    c._destroy_plan()
    assert list(got[:count.value]) == kinds
    assert abs(E - Eg) <= (1e-6 if dtype == 'complex64' else 1e-12) * max(1.0, abs(Eg))
