"""x / y terms are measured with one amplitude per thread while the state leaves
the device idle otherwise: 16 qubits take about as long as 8 (16 amplitudes per
thread in a row: five times)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['complex64', 'complex128'])
def test_xy_terms_of_a_small_state(gpu, dtype):
    from qradient_amd import _native
    from qradient_amd.physical_components import State
    best = {}
    for n in (8, 16):
        st = State(n, '+', dtype=dtype)
        terms, count = _native.terms_array([(i % 2, i % n, 0, 1.0) for i in range(480)])
        prob = np.empty(count)
        times = []
        for _ in range(20):
            t0 = time.perf_counter()
            _native.call('qg_state_term_prob', st._h, terms, count, _native.dptr(prob))
            times.append(time.perf_counter() - t0)
        best[n] = min(times)
        # |+>: x gives 1, y gives 1/2
        assert np.allclose(prob, np.where(np.arange(480) % 2 == 0, 1.0, 0.5), atol=1e-6)
    assert best[16] <= 2.0 * best[8], best
