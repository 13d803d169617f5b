"""complex64 turning forward passes round a state only where they store it.

One rounding to FP32 has a root mean square of 0.41 of its bound 2^-24 of the
state's norm, in 2^n independent directions, so the roundings of NP passes are
expected at 0.41 2^-24 sqrt(NP); 0.6 leaves room for the fluctuations of shallow
circuits.  A pass that also rounds at its exchanges, four or more, is expected at
0.9."""
import ctypes

import numpy as np
import pytest

from oracle import statevector as sv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,p', [(14, 8), (15, 3), (15, 8), (17, 6), (18, 8), (20, 4), (21, 3)])
@pytest.mark.parametrize('weights', ['unit', 'real', 'large'])
def test_one_rounding_a_pass(gpu, n, p, weights):
    from qradient_amd import _native
    from qradient_amd.circuit_logic import Qaoa
    rs = np.random.RandomState(31 * n + p)
    obs = sv.zz_chain_observable(n, np.ones(n - 1) if weights == 'unit' else rs.uniform(0.5, 2.0, n - 1))
    b, g = rs.uniform(0.1, 1.2, p), rs.uniform(0.1, 1.2, p) * (1e8 if weights == 'large' else 1.0)
    vec = {}
    for dtype in ('complex128', 'complex64'):
        c = Qaoa(n, obs, p, dtype=dtype)
        _native.call('qg_plan_set_profiling', c._get_plan(), 1)
        c.run_expec_val(b, g)
        vec[dtype] = np.empty(2 ** n, dtype=np.complex128)
        _native.call('qg_plan_get_state', c._get_plan(), vec[dtype].view(np.float64).ctypes.data_as(_native._dp))
        ms, kinds, count = (ctypes.c_float * 64)(), (ctypes.c_int * 64)(), ctypes.c_int()
        _native.call('qg_plan_pass_times', c._get_plan(), 64, ms, kinds, ctypes.byref(count))
    passes = count.value
    err = np.linalg.norm(vec['complex64'] - vec['complex128'])
    print('n={} passes={} error={:.2f}'.format(n, passes, err * 2.0 ** 24 / np.sqrt(passes)), flush=True)
    assert passes == p + 1 and err <= 0.6 * 2.0 ** -24 * np.sqrt(passes)
