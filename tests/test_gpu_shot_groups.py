"""Qaoa.sample_grad_dense with more shots than one group holds: the same draws
and results as in one group, without all draws in memory at once."""
import tracemalloc

import numpy as np
import pytest

from oracle import statevector as sv

pytestmark = pytest.mark.gpu


def _circuit(n, p):
    from qradient_amd.circuit_logic import Qaoa
    obs = sv.maxcut_observable(n, [(i, (i + 1) % n) for i in range(n - 1)])
    rs = np.random.RandomState(n)
    return Qaoa(n, obs, p), rs.uniform(0.2, 1, p), rs.uniform(0.2, 1, p)


@pytest.mark.parametrize('n', [4, 14])
@pytest.mark.parametrize('exact', [True, False])
@pytest.mark.parametrize('with_ini', [False, True])
def test_groups_change_nothing(gpu, monkeypatch, n, exact, with_ini):
    from qradient_amd.circuit_logic import qaoa
    c, b, g = _circuit(n, 2)
    rs = np.random.RandomState(1)
    ini = None
    if with_ini:
        ini = rs.standard_normal(2 ** n) + 1j * rs.standard_normal(2 ** n)
        ini /= np.linalg.norm(ini)
    out = []
    for group in (1 << 24, 7 * 5, 7, 1):  # all, five, one and (less than) one circuit at a time
        monkeypatch.setattr(qaoa, 'SHOT_GROUP', group)
        np.random.seed(4)
        E, gr = c.sample_grad_dense(b, g, shot_num=7, exact_expec_val=exact, ini_state=ini)
        out.append((E, gr, np.random.random_sample()))
    for E, gr, after in out[1:]:
        assert E == out[0][0] and np.array_equal(gr, out[0][1]) and after == out[0][2]


def test_many_shots_stay_within_a_group(gpu):
    c, b, g = _circuit(4, 2)  # 28 shifted circuits
    shots = 1 << 21
    tracemalloc.start()
    try:
        _, gr = c.sample_grad_dense(b, g, shot_num=shots)
        peak = tracemalloc.get_traced_memory()[1]
    finally:
        tracemalloc.stop()
    # a group is 2^24 shots of 20 bytes (uniforms, positions, values)
    assert peak <= 1.25 * 20 * (1 << 24)
    # and the estimates are as good as their shots: C has 3 components of weight 1
    _, ref = c.grad_run(b, g)
    assert np.max(np.abs(gr - ref)) <= 8 * 28 * 3 / np.sqrt(shots)
