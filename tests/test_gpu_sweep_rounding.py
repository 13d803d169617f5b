"""complex64 multi-layer forward passes round a state only where they store it.

One rounding to FP32 moves a state by at most 2^-24 of its norm, in 2^n
independent directions, so the roundings of NP passes add up to at most
2^-24 sqrt(NP) but for fluctuations of some 2^-n/2; the rotations themselves run
in FP64.  (A pass that also rounds at its ten or so exchanges is expected at
1.3 times that bound: the root mean square of a rounding is 0.41 of its bound.)"""
import ctypes

import numpy as np
import pytest

from oracle import statevector as sv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,L,tile', [(14, 12, None), (16, 20, None), (18, 12, None), (20, 12, None), (15, 16, (10, 2)),
                                      (16, 16, (13, 3))])
@pytest.mark.parametrize('entangler', ['cnot', 'cz'])
def test_one_rounding_a_pass(gpu, n, L, tile, entangler):
    from qradient_amd import _native
    from qradient_amd.circuit_logic import McClean
    rs = np.random.RandomState(17 * n + L)
    axes, angles = sv.mcclean_random_params(L, n, rs)
    obs = sv.zz_chain_observable(n, rs.standard_normal(n - 1))
    vec = {}
    for dtype in ('complex128', 'complex64'):
        c = McClean(n, obs, L, axes=axes, angles=angles, dtype=dtype, entangler=entangler)
        if tile:
            _native.call('qg_plan_tune', c._get_plan(), tile[0], tile[1], 4, 4)
        _native.call('qg_plan_set_profiling', c._get_plan(), 1)
        c.run_expec_val()
        vec[dtype] = c.final_state()
        ms, kinds, count = (ctypes.c_float * 64)(), (ctypes.c_int * 64)(), ctypes.c_int()
        _native.call('qg_plan_pass_times', c._get_plan(), 64, ms, kinds, ctypes.byref(count))
    passes = sum(k == 0 for k in kinds[:count.value])
    err = np.linalg.norm(vec['complex64'] - vec['complex128'])
    print('n={} passes={} error={:.2e}'.format(n, passes, err), flush=True)
    assert passes and err <= 2.0 ** -24 * np.sqrt(passes)
